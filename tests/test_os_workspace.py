"""The workspace query of the output-stationary kernel against what its launch
plans need (host only): index and row order, plain and concatenated inputs,
offset splits and work balance, around the lines where the plans change."""
import ctypes
import itertools
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = ctypes.CDLL(os.path.join(ROOT, "spira_amd", "libspira_hip.so"))
F16, STORE = 0, 0


class Tuning(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("col_tile", "step_channels", "offset_splits", "offset_pack",
                                            "block_order", "row_walk", "balance_offsets", "blocks_per_cu")]


def query(T, K, cin, cout, tn):
    size = ctypes.c_size_t()
    assert LIB.spira_hip_conv_os_workspace(ctypes.c_int64(T), K, cin, cout, F16, STORE, ctypes.byref(tn),
                                           ctypes.byref(size)) == 0
    return size.value


def need(T, K, cin, cin2, cout, form, tn):
    """Bytes that a launch under the plan writes (128-row tiles)."""
    plan = (ctypes.c_int32 * 7)()
    assert LIB.spira_hip_conv_os_plan(ctypes.c_int64(T), K, cin, cin2, cout, form, STORE, ctypes.byref(tn), plan) == 0
    tile, _, splits, pack, gx, gy, _ = plan
    if splits > 1:
        return T * cout * 4
    parts = min(8, -(-K // tn.balance_offsets)) if tn.balance_offsets > 0 else 1
    if form != 2 or parts == 1 or pack > 1 or K > 128 or (cin + cin2) % 8:
        return 0
    return (gx * parts * 4 + 4 + 255) // 256 * 256 + gx * gy * parts * 128 * tile * 4


@pytest.mark.parametrize("balance", [0, 9, 14])
@pytest.mark.parametrize("tile", [0, 64, 96])
@pytest.mark.parametrize("K", [2, 8, 9, 27, 28, 125, 128, 343])
def test_query_covers_every_plan(K, tile, balance):
    tn = Tuning(col_tile=tile, balance_offsets=balance)
    rows = [1, 31, 32, 51, 52, 63, 64, 86, 101, 102, 103, 107, 127, 128, 129, 153, 154, 160, 161, 204, 205, 255, 256,
            257, 320, 321, 600]
    for r, cout in itertools.product(rows, (16, 32, 48, 64, 96, 128, 160, 256, 272, 288, 520, 544)):
        T = 128 * r
        for cin in (16, 24, 32, 64, 96, 128, 256):
            have = query(T, K, cin, cout, tn)
            for cin2, form in itertools.product((0, 8, 16, 32, 64, 128, 256), (1, 2)):
                assert need(T, K, cin, cin2, cout, form, tn) <= have, (T, K, cin, cin2, cout, form)
