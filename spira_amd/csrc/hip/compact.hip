// Sparse convolution over compacted (source, target) pairs, block by block
// (gfx950): Y[t] = epilogue(sum_k X[s(t, k)] @ W[k]) over the valid entries.
//
// A block owns BT consecutive targets and BN output channels, whose fp32 sums
// it keeps in LDS.  The kernel's offsets are taken in chunks: the block reads
// the chunk's entries for its targets and lists the valid ones per offset in
// LDS (source, target).  It then walks units of up to U pairs of one offset:
// the pairs' rows are gathered into an LDS ring (DMA, D - 1 steps ahead,
// consecutive lanes on one row), each wave multiplies them by its own slice of
// the output columns (one MFMA column per pair, weights from registers) and
// adds the products to the targets' sums.  A wave is the only writer of its
// columns, and an offset has a target at most once, so the sums need no
// atomics and are taken in offset order: the same result on every call.
//
// What it buys: the gathers, weight reads and MFMAs are done for the valid
// pairs only (rounded up to 16 per offset and block), where a voxel scene has
// a neighbour at 6 to 40 % of its offsets; and neither gathered rows nor
// products pass through memory.
//
// What bounds it: per CU, the L1's 64 bytes per clock (rows, and the weights
// of every offset once per block) and the LDS.  Measured costs per KB that
// set the layout: rows read with four or more consecutive lanes on one row 16
// to 24 clocks, in MFMA lane order 66 (one cache lookup per lane); LDS DMA 15,
// ds_read_b128 4 to 8, ds_write_b128 13, ds_add_f32 177 per 256 bytes (so the
// sums are read, added to and written, never LDS atomics).
#include "common.hpp"
#include "../../../include/spira_hip.h"

#include <algorithm>
#include <type_traits>

namespace spira_hip {

namespace compact {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Where the entry (source of target t at offset k) comes from.  The first kd
// offsets are the dense part of a hybrid map ([T, kd] rows, or without a map
// the target itself, kd = 1); the others by kind:
enum Kind { kRowsTK = 0, kRowsKT = 1, kMasks = 2 };
struct Entries {
  int kind;
  const int32_t *idx;   // kRowsTK: [T, K]; kRowsKT: [K - kd, ld]; kMasks: ranks [K - kd, ld]
  int64_t ld;
  const int32_t *list;  // kMasks: source of rank m at offset k: list[k * S + m]
  int64_t S;
  const int32_t *dense;
  int kd;
  // pairs that lost their place in idx to another pair of the same target and
  // offset: (offset, source, target, next of the block or -1) each, the first
  // of block b at heads[b]; or null
  const int4 *extra;
  const int32_t *heads;
};
constexpr int kTargets = 64;  // targets per block

struct Layer {
  const void *X;  // [S, Cin], rows of a multiple of 16 bytes
  uint32_t xbytes, rowbytes;
  const void *F;  // fp16: fragment-major weights (spira_hip_prepare_fragments)
  int ctiles, nft;  // 16-column tiles, and 64-byte fragments per input row
  int Cout;
  const void *W;  // [K, Cin, Cout] (fp32, and repeated pairs)
  uint32_t wbytes;  // of one offset
  int Cin;
  void *Y;         // [T, Cout]
  const float *scale, *shift;
  const void *residual;
  int relu;
  int vec_out;  // Y and the residual start on 16-byte boundaries
};

typedef __attribute__((address_space(3))) void lds_void_t;
constexpr uint32_t kOutOfRange = 0x80000000u;
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_t *)(const_cast<void *>(p))));
}
// LDS accesses of the unit loop are inline assembly, ordered by the explicit
// waits: beside DMA writes in flight the compiler would wait for all of them
// before each access of its own.
template <int OFF> __device__ __forceinline__ floatx4 rd16(uint32_t base) {
  floatx4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(OFF) : "memory");
  return v;
}
__device__ __forceinline__ int rd4(uint32_t base) {
  int v;
  asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(base) : "memory");
  return v;
}
template <int OFF> __device__ __forceinline__ int rd1(uint32_t base) {
  int v;
  asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(OFF) : "memory");
  return v;
}
__device__ __forceinline__ void wr16(uint32_t base, floatx4 v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(base), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <class V> __device__ __forceinline__ void pin(V &v) { asm volatile("" : "+v"(v)); }
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// One 64-byte fragment of 16 pairs times a 16-column tile of weights: the
// weights are the MFMA's A operand, so that lane l holds channels 4 (l / 16)
// .. + 3 of pair l % 16's products (one 16-byte LDS access).
__device__ __forceinline__ void mma(floatx4 &d, floatx4 w, floatx4 x, const _Float16 *) {
  d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, w), __builtin_bit_cast(half8, x), d, 0, 0, 0);
}
// (v_mfma_f32_16x16x4_f32 takes 4 channels: MFMA i multiplies element i of
// every 4-channel group)
__device__ __forceinline__ void mma(floatx4 &d, floatx4 w, floatx4 x, const float *) {
#pragma unroll
  for (int i = 0; i < 4; ++i) d = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], d, 0, 0, 0);
}

template <int I, class F> struct Unroll {
  static __device__ __forceinline__ void run(F &&f) {
    Unroll<I - 1, F>::run(f);
    f(std::integral_constant<int, I - 1>{});
  }
};
template <class F> struct Unroll<0, F> {
  static __device__ __forceinline__ void run(F &&) {}
};
template <int N, class F> __device__ __forceinline__ void unroll(F &&f) { Unroll<N, F &>::run(f); }

// NW waves x NC 16-column tiles of output; BT targets; CH offsets per chunk;
// units of U pairs, D ring stages; a step takes NF 64-byte fragments of the
// rows (PITCH bytes apart in the ring).
template <class FT, int PITCH, int NF, int NW, int NC, int BT, int CH, int U, int D, int OCC>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC))) void pair_kernel(const Entries en,
                                                                                              int64_t T, int K,
                                                                                              const Layer l) {
  constexpr int BN = 16 * NW * NC, NCK = BN / 16;
  constexpr int NT = 64 * NW;
  constexpr int EPT = (CH * BT + NT - 1) / NT;     // entries per thread and chunk
  constexpr int UT = U / 16;                       // tiles per unit
  constexpr int LPR = PITCH / 16, RPI = 64 / LPR;  // lanes per row, rows per DMA
  constexpr int IA = (U / RPI + NW - 1) / NW;      // DMAs per wave and step
  constexpr int LPS = IA + NF * NC * (sizeof(FT) == 4 ? 4 : 1);  // vector-memory loads per wave and step
  constexpr int STAGE = IA * NW * 1024;
  constexpr int MAXU = CH * ((BT + U - 1) / U);
  static_assert(BT == kTargets && BT % 64 == 0 && BT <= 128 && CH <= 32 && NT % CH == 0, "chunk shape");
  static_assert(PITCH >= NF * 64 && (D - 2) * LPS < 64 && U <= BT && U % 16 == 0, "step shape");
  // Sums: row t holds the 16-column chunks of target t (row BT takes the
  // padding pairs' products); chunk w sits at w ^ swz(t), so that 16 rows'
  // same chunk spreads over all four quarters of the banks.
  __shared__ __align__(1024) char ring[D * STAGE];
  __shared__ __align__(16) float acc[(BT + 1) * BN];
  __shared__ int32_t src_l[CH * BT];
  __shared__ uint8_t tgt_l[CH * BT];
  __shared__ int units[MAXU];  // offset << 16 | first pair << 8 | pairs
  __shared__ int cnt[CH];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  // (workgroup w goes to XCD w % 8: each XCD takes one range of targets, its
  // column tiles together, so that its L2 serves one slab of sources)
  int64_t bx;
  int by;
  {
    const int64_t G = static_cast<int64_t>(gridDim.x) * gridDim.y,
                  w = blockIdx.x + static_cast<int64_t>(blockIdx.y) * gridDim.x;
    const int64_t q = G / 8, r = G % 8, x = w % 8;
    const int64_t L = x * q + (x < r ? x : r) + w / 8;
    bx = L / gridDim.y;
    by = static_cast<int>(L % gridDim.y);
  }
  const int64_t t0 = bx * BT;
  const int nb0 = by * BN;
  const int nch = (l.nft + NF - 1) / NF;
  auto at = [](int t, int w) {
    const int z = NCK % 4 == 0 ? (t & 3) : (NCK % 4 == 2 ? (t >> 1) & 1 : 0);
    return (t * NCK + (w ^ z)) * 16;
  };
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(l.X), 0, static_cast<int>(l.xbytes), 0x00020000);
  // the wave's weight fragments: column tiles ct .. ct + NC - 1 (a tile past
  // the last repeats it; its products are not stored)
  int ct[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int c = by * NCK + wave * NC + q;
    ct[q] = c < l.ctiles ? c : l.ctiles - 1;
  }
  // the row of the ring a lane's DMA fills, and its 16-byte chunk: swizzled
  // by the row so that 16 rows' reads of one chunk hit distinct banks
  auto swz = [](int r) { return PITCH == 64 ? (r >> 2) & 3 : (PITCH == 128 ? (r >> 1) & 7 : r & 15); };
  int drow[IA];
  uint32_t dchunk[IA];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    drow[i] = (wave * IA + i) * RPI + lane / LPR;
    const int c = (lane % LPR) ^ swz(drow[i] & 15);
    dchunk[i] = c < NF * 4 ? static_cast<uint32_t>(c) * 16u : kOutOfRange;
  }
  const uint32_t ring_w = __builtin_amdgcn_readfirstlane(lds_addr(ring) + wave * IA * 1024);
  uint32_t frag_at[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) frag_at[f] = lds_addr(ring) + l16 * PITCH + (((4 * f + lq) ^ swz(l16)) * 16);
  const uint32_t src_at = lds_addr(src_l), tgt_at = lds_addr(tgt_l), units_at = lds_addr(units),
                 acc_at = lds_addr(acc) + lq * 16;

#pragma unroll 4
  for (int i = tid; i < (BT + 1) * BN / 4; i += NT) reinterpret_cast<floatx4 *>(acc)[i] = floatx4{};
#pragma unroll 1
  for (int c0 = 0; c0 < K; c0 += CH) {
    if (tid < CH) cnt[tid] = 0;
    // The chunk's entries: every load of a thread first (an entry past the end
    // reads entry 0 and is dropped), then the lists.
    int32_t ent[EPT];
    if (en.kind == kRowsTK) {
      // consecutive lanes take consecutive offsets of a row
      int kl = tid % CH, r0 = tid / CH;
      pin(r0);  // (addresses are formed here, not kept from chunk to chunk)
      const int32_t *p = en.idx + (t0 + r0) * K + c0 + kl;
      const bool kin = c0 + kl < K;
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int tl = r0 + i * (NT / CH);
        const bool in = kin && tl < BT && t0 + tl < T;
        ent[i] = *(in ? p + i * (NT / CH) * K : en.idx);
      }
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int tl = r0 + i * (NT / CH);
        if (!kin || tl >= BT || t0 + tl >= T) ent[i] = -1;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        if (ent[i] >= 0) {
          const int pos = kl * BT + atomicAdd(&cnt[kl], 1);
          src_l[pos] = ent[i];
          tgt_l[pos] = static_cast<uint8_t>(r0 + i * (NT / CH));
        }
    } else {
      // a wave takes 64 targets of one offset (k is wave-uniform)
      int w0 = wave;
      pin(w0);
      w0 = __builtin_amdgcn_readfirstlane(w0);
      auto where = [&](int i, int &kl, int &h) {
        kl = (i * NW + w0) / (BT / 64);
        h = (i * NW + w0) % (BT / 64) * 64;
        return kl < CH && c0 + kl < K;
      };
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        int kl, h;
        const bool kin = where(i, kl, h);
        const int k = c0 + kl;
        const bool in = t0 + h + lane < T;
        const int32_t *p = !kin ? nullptr : (k < en.kd ? en.dense : en.idx);
        const int64_t step = k < en.kd ? en.kd : 1;
        const int64_t o = (t0 + h) * step + (k < en.kd ? k : static_cast<int64_t>(k - en.kd) * en.ld);
        ent[i] = p ? p[in ? o + lane * step : 0] : static_cast<int32_t>(t0 + h + lane);
      }
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        int kl, h;
        if (!where(i, kl, h) || t0 + h + lane >= T) ent[i] = -1;
      }
      if (en.kind == kMasks && en.S > 0) {
        int32_t s[EPT];
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
          int kl, h;
          where(i, kl, h);
          const int k = c0 + kl;
          const bool in = k >= en.kd && ent[i] >= 0 && ent[i] < en.S;
          s[i] = en.list[in ? static_cast<int64_t>(k - en.kd) * en.S + ent[i] : 0];
        }
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
          int kl, h;
          where(i, kl, h);
          // (a rank that no source holds reads an unwritten list word)
          if (c0 + kl >= en.kd) ent[i] = ent[i] >= 0 && ent[i] < en.S && s[i] >= 0 && s[i] < en.S ? s[i] : -1;
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        int kl, h;
        if (!where(i, kl, h)) continue;
        const uint64_t m = ballot(ent[i] >= 0);
        int base = 0;
        if (lane == 0 && m) base = atomicAdd(&cnt[kl], __builtin_popcountll(m));
        const int pos = kl * BT + __builtin_amdgcn_readfirstlane(base) + lane_prefix(m);
        if (ent[i] >= 0) {
          src_l[pos] = ent[i];
          tgt_l[pos] = static_cast<uint8_t>(h + lane);
        }
      }
    }
    __syncthreads();
    // units of each offset (every wave counts them, lane = offset; wave 0 writes them)
    const int n = lane < CH ? cnt[lane] : 0;
    const int nu = (n + U - 1) / U;
    int incl = nu;
#pragma unroll
    for (int d = 1; d < CH; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    const int nunits = __builtin_amdgcn_readfirstlane(__shfl(incl, CH - 1, 64));
    if (wave == 0 && lane < CH) {
#pragma unroll 1
      for (int j = 0; j < nu; ++j)
        units[incl - nu + j] = lane << 16 | (j * U) << 8 | (n - j * U < U ? n - j * U : U);
      // the last tile padded to 16 pairs
#pragma unroll 1
      for (int j = n; j < (n + 15) / 16 * 16; ++j) tgt_l[lane * BT + j] = BT;
    }
    __syncthreads();
    const int nsteps = nunits * nch;
    if (nsteps == 0) continue;
    // Step v: unit v / nch, fragments from (v % nch) NF; each step adds its
    // products to the sums.  Steps past the last repeat it (loaded, never
    // multiplied).  nd / src: the unit of the next step to load and the lane's
    // source rows of it.  (Every LDS read of a step is waited for in the block
    // that issues it, so that no value in flight crosses a branch.)
    floatx4 wf[D][NF][NC];
    int tg[D][UT], dsc[D];
    int iunit = 0, ich = 0, nd = 0, src[IA];
    auto peek = [&](int u) {
      nd = __builtin_amdgcn_readfirstlane(u);
      const uint32_t b = src_at + ((nd >> 16) * BT + ((nd >> 8) & 255)) * 4;
#pragma unroll
      for (int i = 0; i < IA; ++i) src[i] = rd4(b + (drow[i] < (nd & 255) ? drow[i] : 0) * 4);
    };
    auto peeked = [&] {
      lds_wait();
#pragma unroll
      for (int i = 0; i < IA; ++i) pin(src[i]);
    };
    int un = rd4(units_at);
    lds_wait();
    pin(un);
    peek(un);
    peeked();
    auto issue = [&](auto S) {
      constexpr int s = decltype(S)::value;
      const int np = nd & 255, kl = nd >> 16;
      const uint32_t kb = static_cast<uint32_t>(ich * NF * 64);
      dsc[s] = np;
      const uint32_t tb = tgt_at + kl * BT + ((nd >> 8) & 255) + l16;
      unroll<UT>([&](auto I) { tg[s][decltype(I)::value] = rd1<decltype(I)::value * 16>(tb); });
      const int f0 = ich * NF;
      if (++ich == nch) {
        ich = 0;
        iunit = iunit + 1 < nunits ? iunit + 1 : iunit;
      }
      un = rd4(units_at + iunit * 4);
#pragma unroll
      for (int i = 0; i < IA; ++i) {
        const bool in = drow[i] < np && dchunk[i] != kOutOfRange && kb + dchunk[i] < l.rowbytes;
        const uint32_t o = static_cast<uint32_t>(src[i]) * l.rowbytes + kb + dchunk[i];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xr, (lds_void_t *)static_cast<uintptr_t>(ring_w + s * STAGE + i * 1024), 16, in ? o : kOutOfRange, 0, 0, 0);
      }
      lds_wait();
      pin(un);
#pragma unroll
      for (int j = 0; j < UT; ++j) pin(tg[s][j]);
      peek(un);
      if constexpr (sizeof(FT) == 4) {
        // fp32 weights as they are, so that no copy of them can be stale: the
        // lane's four channels of its column (a quarter wave on 64 bytes of a
        // row; past Cin out of the offset's range, zero; past Cout the next
        // row's values, in columns that are not stored).  20k voxels, 32 -> 32
        // 29.3 us, from fragments kept from call to call 27.9.
        const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(static_cast<const char *>(l.W) + static_cast<int64_t>(c0 + kl) * l.wbytes), 0,
            static_cast<int>(l.wbytes), 0x00020000);
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              wf[s][f][q][e] = __builtin_bit_cast(
                  float, __builtin_amdgcn_raw_buffer_load_b32(
                             wr, (((f0 + f) * 16 + lq * 4 + e) * l.Cout + ct[q] * 16 + l16) * 4, 0, 0));
      } else {
        const floatx4 *wp = static_cast<const floatx4 *>(l.F) +
                            (static_cast<int64_t>(c0 + kl) * l.ctiles * l.nft + f0) * 64 + lane;
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
          for (int f = 0; f < NF; ++f) wf[s][f][q] = wp[(ct[q] * l.nft + f) * 64];
      }
      peeked();
    };
    // the products of J + 1 tiles of stage i
    auto multiply = [&](auto I, auto J) {
      constexpr int i = decltype(I)::value, nt = decltype(J)::value + 1;
      floatx4 x[nt][NF], sum[nt][NC];
      uint32_t row[nt][NC];
      unroll<nt>([&](auto Q) {
        constexpr int j = decltype(Q)::value;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          row[j][q] = acc_at + at(tg[i][j], wave * NC + q) * 4;
          sum[j][q] = rd16<0>(row[j][q]);
        }
        unroll<NF>([&](auto F) { x[j][decltype(F)::value] = rd16<i * STAGE + j * 16 * PITCH>(frag_at[decltype(F)::value]); });
      });
      lds_wait();
#pragma unroll
      for (int j = 0; j < nt; ++j) {
#pragma unroll
        for (int f = 0; f < NF; ++f) pin(x[j][f]);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          pin(sum[j][q]);
          floatx4 d{};
#pragma unroll
          for (int f = 0; f < NF; ++f) mma(d, wf[i][f][q], x[j][f], static_cast<const FT *>(nullptr));
          wr16(row[j][q], sum[j][q] + d);
        }
      }
    };
    unroll<D - 1>(issue);
#pragma unroll 1
    for (int v = 0; v < nsteps; v += D) {
      unroll<D>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if (v + i < nsteps) {
          wait_vm<(D - 2) * LPS>();      // this wave's loads of step v + i
          __builtin_amdgcn_s_barrier();  // every wave's, and the stage issued next is read out
          issue(std::integral_constant<int, (i + D - 1) % D>{});
          const int nt = (dsc[i] + 15) >> 4;
          unroll<UT>([&](auto J) {
            if (nt == decltype(J)::value + 1) multiply(I, J);
          });
        }
      });
    }
    wait_vm<0>();
    lds_wait();
  }
  __syncthreads();
  const FT *X = static_cast<const FT *>(l.X);
  if (en.heads) {
    // repeated (offset, target) pairs, none in a map's own lists: each one's
    // product, four lanes per column (in any order).  Bound by the latency of
    // its loads: 100k voxels, fp16 64 -> 64, every 1000th / 100th / 10th of a
    // list's pairs repeated 66 / 71 / 123 us, none 48 (every block on one list,
    // a lane per column: 244 / 520 / 4483; the fused pass 81 / 81 / 85).
    const FT *W = static_cast<const FT *>(l.W);
    const int64_t xs = l.rowbytes / sizeof(FT);
    const int c0 = tid >> 2, q = tid & 3;
    int p = en.heads[bx];
    const bool any = p >= 0;
    int4 e = any ? en.extra[p] : int4{};
    while (p >= 0) {
      const int64_t k = e.x + en.kd;
      const FT *x = X + e.y * xs;
      const int tl = static_cast<int>(e.z - t0);
      p = e.w;
      if (p >= 0) e = en.extra[p];
      for (int c = c0; c < BN && nb0 + c < l.Cout; c += NT / 4) {  // (alike in the four lanes)
        const FT *w = W + k * l.Cin * l.Cout + nb0 + c;
        float v = 0.f;
#pragma unroll 8
        for (int ci = q; ci < l.Cin; ci += 4)
          v = fmaf(static_cast<float>(x[ci]), static_cast<float>(w[static_cast<int64_t>(ci) * l.Cout]), v);
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        if (q == 0) acc[at(tl, c / 16) + c % 16] += v;
      }
    }
    if (any) __syncthreads();
  }
  // output rows with the epilogue, 16 bytes per lane where rows are aligned
  constexpr int V = 16 / sizeof(FT);
  const FT *R = static_cast<const FT *>(l.residual);
  FT *Y = static_cast<FT *>(l.Y);
  auto finish = [&](float v, int n, float res) {
    if (l.scale) v *= l.scale[n];
    if (l.shift) v += l.shift[n];
    v += res;
    return l.relu ? (v > 0.f ? v : 0.f) : v;
  };
  if (l.vec_out && l.Cout % V == 0) {
    typedef FT vec __attribute__((ext_vector_type(V)));
#pragma unroll 1
    for (int i = tid; i < BT * (BN / V); i += NT) {
      const int tl = i / (BN / V), c = (i % (BN / V)) * V;
      if (t0 + tl >= T || nb0 + c >= l.Cout) continue;
      const int64_t o0 = (t0 + tl) * l.Cout + nb0 + c;
      vec r = {};
      if (R) r = *reinterpret_cast<const vec *>(R + o0);
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e)
        o[e] = static_cast<FT>(finish(acc[at(tl, c / 16) + c % 16 + e], nb0 + c + e, static_cast<float>(r[e])));
      *reinterpret_cast<vec *>(Y + o0) = o;
    }
  } else {
#pragma unroll 1
    for (int i = tid; i < BT * BN; i += NT) {
      const int tl = i / BN, c = i % BN;
      if (t0 + tl >= T || nb0 + c >= l.Cout) continue;
      const int64_t o0 = (t0 + tl) * l.Cout + nb0 + c;
      Y[o0] = static_cast<FT>(finish(acc[at(tl, c / 16) + c % 16], nb0 + c, R ? static_cast<float>(R[o0]) : 0.f));
    }
  }
}

// list[k * S + m] = s for the source mask's ranks m
__global__ __launch_bounds__(256) void mask_list_kernel(const int32_t *__restrict__ smask, int64_t n, int64_t S,
                                                        int32_t *__restrict__ list) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int32_t m = smask[i];
  if (m >= 0 && m < S) list[i / S * S + m] = static_cast<int32_t>(i % S);
}

__global__ __launch_bounds__(256) void rows_clear_kernel(int32_t *__restrict__ rows, int64_t n4, int32_t *nextra) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n4) reinterpret_cast<int4 *>(rows)[i] = make_int4(-1, -1, -1, -1);
  if (i == 0) *nextra = 0;
}

// rows[k, out] = in for the pairs of compacted row k, and with Kw > 0 the
// mirrored rows[Kw - 1 - k, in] = out (a self-mirrored centre row once); pairs
// past the last row's, or with an index outside its side (-1), are none.  A
// repeated (offset, target) goes to the list of its block of targets.
__global__ __launch_bounds__(256) void pair_rows_kernel(const int32_t *__restrict__ in_idx,
                                                        const int32_t *__restrict__ out_idx,
                                                        const int32_t *__restrict__ naddrs, int R, int64_t P, int Kw,
                                                        int64_t S, int64_t T, int64_t ld, int32_t *__restrict__ rows,
                                                        int32_t *__restrict__ heads, int4 *__restrict__ extra,
                                                        int32_t *__restrict__ nextra) {
  const int64_t p = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (p >= P || p >= naddrs[R]) return;
  int lo = 0, hi = R;  // last row with naddrs[row] <= p
  while (hi - lo > 1) {
    const int m = (lo + hi) >> 1;
    if (naddrs[m] <= p) lo = m;
    else hi = m;
  }
  auto put = [&](int k, int32_t s, int32_t t) {
    if (atomicCAS(&rows[static_cast<int64_t>(k) * ld + t], -1, s) == -1) return;
    const int at = atomicAdd(nextra, 1);
    extra[at] = make_int4(k, s, t, atomicExch(&heads[t / kTargets], at));
  };
  const int32_t a = in_idx[p], b = out_idx[p];
  if (a < 0 || a >= S || b < 0 || b >= T) return;
  put(lo, a, b);
  if (Kw > 0 && 2 * lo + 1 != Kw && b < S && a < T) put(Kw - 1 - lo, b, a);
}

// fragment-major fp16 weights: 1 KB blocks (offset k, 16-column tile c,
// fragment f), lane l's 16 bytes = input channels of quarter l / 16 of the
// fragment, output column 16 c + l % 16; zero past Cin and Cout
__global__ __launch_bounds__(256) void fragments_kernel(const _Float16 *__restrict__ W, int64_t n, int Cin, int Cout,
                                                        int ctiles, int nft, _Float16 *__restrict__ F) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;  // one lane's 16 bytes
  if (i >= n) return;
  const int lane = static_cast<int>(i & 63);
  const int64_t blk = i >> 6, k = blk / (static_cast<int64_t>(ctiles) * nft);
  const int rem = static_cast<int>(blk % (static_cast<int64_t>(ctiles) * nft));
  const int co = rem / nft * 16 + (lane & 15), ci = (rem % nft * 4 + (lane >> 4)) * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    F[i * 8 + e] = (co < Cout && ci + e < Cin) ? W[(k * Cin + ci + e) * Cout + co] : static_cast<_Float16>(0.f);
}

// Rows padded with zero channels to 16 bytes
template <class FT>
__global__ __launch_bounds__(256) void pad_rows_kernel(const FT *__restrict__ X, int64_t n, int Cin, int Cp,
                                                       FT *__restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t r = i / Cp;
  const int c = static_cast<int>(i - r * Cp);
  out[i] = c < Cin ? X[r * Cin + c] : static_cast<FT>(0.f);
}

// Shapes.  A wave per 16 output columns and 64 targets per block: four to six
// blocks share a CU, so that one block's index loads, barriers and LDS trips
// run under the others' (128 targets halve the weight reads but leave two
// blocks per CU: 64 -> 64 on a 100k-voxel LiDAR sweep 42.4 -> 44.7 us, on a
// 68k-voxel level with 9.6 pairs per target 51 -> 70 us).  Two ring stages up
// to 64 columns (three: 32 -> 32 24.6 -> 30.1 us, 64 -> 64 the same), three
// beyond.  fp32 layers wider than 64 columns take several 64-column blocks
// (128 -> 128, 20k voxels: 121 us with eight waves, 96 us; 60k 413 and 415).  16-column layers
// of more than 32 offsets take two waves, the second for the index lists
// (125 offsets, 5k voxels: 66 us with one wave, 45 us).
template <class FT, int PITCH, int NF>
static void launch_n(hipStream_t s, const Entries &en, int64_t T, int K, const Layer &l) {
#define SPIRA_PAIR_CALL(NW, CH, D, OCC)                                                                         \
  hipLaunchKernelGGL((pair_kernel<FT, PITCH, NF, NW, 1, kTargets, CH, 32, D, OCC>),                                   \
                     dim3(static_cast<unsigned>(div_up(T, kTargets)), static_cast<unsigned>(div_up(l.ctiles, NW))), \
                     dim3(64 * NW), 0, s, en, T, K, l)
  constexpr int occ4 = PITCH == 256 ? 3 : 4;  // (what the ring leaves room for)
  if (l.Cout <= 16 && K <= 32) {
    SPIRA_PAIR_CALL(1, 16, 2, 2);
  } else if (l.Cout <= 32) {
    SPIRA_PAIR_CALL(2, 32, 2, (PITCH == 256 ? 2 : 3));
  } else if constexpr (sizeof(FT) == 4) {
    SPIRA_PAIR_CALL(4, 32, 2, occ4);
  } else {
    // (96 columns of 96 channels and more: eight waves, two of them idle; 128
    // -> 96 on 90k LiDAR voxels 123 us with six, 95 with eight)
    if (l.Cout <= 64) SPIRA_PAIR_CALL(4, 32, 2, occ4);
    else if (l.Cout <= 96 && PITCH < 256) SPIRA_PAIR_CALL(6, 32, 3, 3);
    else SPIRA_PAIR_CALL(8, 32, 3, 4);
  }
#undef SPIRA_PAIR_CALL
}

static int launch(int dtype, hipStream_t s, const Entries &en, int64_t T, int K, const Layer &l) {
  // fragments per step: the largest of 4, 3, 2 and 1 that divides a row's
  // (fp32 64 -> 64 on 20k voxels: two per step 48 us, four 40 us)
  const bool f16 = dtype == SPIRA_F16;
  if (l.nft % 4 == 0) {
    if (f16) launch_n<_Float16, 256, 4>(s, en, T, K, l);
    else launch_n<float, 256, 4>(s, en, T, K, l);
  } else if (l.nft % 3 == 0) {
    if (f16) launch_n<_Float16, 256, 3>(s, en, T, K, l);
    else launch_n<float, 256, 3>(s, en, T, K, l);
  } else if (l.nft % 2 == 0) {
    if (f16) launch_n<_Float16, 128, 2>(s, en, T, K, l);
    else launch_n<float, 128, 2>(s, en, T, K, l);
  } else {
    if (f16) launch_n<_Float16, 64, 1>(s, en, T, K, l);
    else launch_n<float, 64, 1>(s, en, T, K, l);
  }
  SPIRA_HIP_LAUNCH_CHECK();
  return kOk;
}

}  // namespace compact

}  // namespace spira_hip

using namespace spira_hip;

extern "C" {

int spira_hip_conv_compact_workspace(int64_t num_sources, int64_t num_targets, int num_offsets, int64_t num_pairs,
                                     size_t *bytes) {
  // masks: the sources by rank; pairs: entry rows by target, the blocks' first
  // repeated pair, their number and the repeated pairs
  const int64_t n = std::max(num_sources, round_up(num_targets, 4)) * std::max(num_offsets, 0);
  const int64_t heads = round_up(div_up(num_targets, compact::kTargets), 4);
  *bytes = static_cast<size_t>(n + heads + 8 + 8 * std::max<int64_t>(num_pairs, 0)) * sizeof(int32_t);
  return kOk;
}

}  // extern "C"

static size_t fragments_bytes(int num_offsets, int c_in, int c_out, int dtype) {
  if (dtype != SPIRA_F16) return 0;
  return static_cast<size_t>(num_offsets) * div_up(c_out, 16) * div_up(c_in, 32) * 1024;
}

static int check_compact(int64_t num_sources, int64_t num_targets, int row_channels, int c_in, int c_out, int dtype,
                         const void *sources, const void *weights, const void *fragments) {
  SPIRA_HIP_REQUIRE(dtype == SPIRA_F16 || dtype == SPIRA_F32, "conv_compact: dtype must be fp16 or fp32");
  SPIRA_HIP_REQUIRE(c_in > 0 && c_out > 0, "conv_compact: empty channel dimension");
  const int v = dtype == SPIRA_F16 ? 8 : 4;
  SPIRA_HIP_REQUIRE(row_channels >= c_in && row_channels - c_in < v && row_channels % v == 0 &&
                        (reinterpret_cast<uintptr_t>(sources) & 15) == 0,
                    "conv_compact: source rows must be padded to 16 bytes and 16-byte aligned");
  SPIRA_HIP_REQUIRE(num_sources >= 0 && num_sources * row_channels * (16 / v) < (int64_t(1) << 31) &&
                        num_targets < (int64_t(1) << 31) - 256,
                    "conv_compact: features of one layer must stay below 2 GiB");
  SPIRA_HIP_REQUIRE(weights != nullptr && (fragments != nullptr || dtype == SPIRA_F32),
                    "conv_compact: needs the weights and, in fp16, their fragments (spira_hip_prepare_fragments)");
  SPIRA_HIP_REQUIRE((static_cast<int64_t>(c_in) + 64) * c_out * 4 < (int64_t(1) << 31),
                    "conv_compact: weights of one offset must stay below 2 GiB");
  return kOk;
}

static compact::Layer make_layer(const void *sources, int64_t num_sources, int row_channels, int c_in,
                                 const void *weights, const void *fragments, int c_out, int dtype, void *targets,
                                 const float *scale, const float *shift, const void *residual, int relu) {
  compact::Layer l{};
  const int size = dtype == SPIRA_F16 ? 2 : 4;
  l.X = sources;
  l.rowbytes = static_cast<uint32_t>(row_channels * size);
  l.xbytes = static_cast<uint32_t>(num_sources * l.rowbytes);
  l.F = fragments;
  l.ctiles = static_cast<int>(div_up(c_out, 16));
  l.nft = static_cast<int>(div_up(c_in * size, 64));
  l.Cout = c_out;
  l.W = weights;
  l.wbytes = static_cast<uint32_t>(static_cast<int64_t>(c_in) * c_out * size);
  l.Cin = c_in;
  l.Y = targets;
  l.scale = scale;
  l.shift = shift;
  l.residual = residual;
  l.relu = relu;
  auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  l.vec_out = aligned(targets) && aligned(residual);
  return l;
}

extern "C" {

int spira_hip_fragments_bytes(int num_offsets, int c_in, int c_out, int dtype, size_t *bytes) {
  *bytes = fragments_bytes(num_offsets, c_in, c_out, dtype);
  return kOk;
}

int spira_hip_prepare_fragments(const void *weights, int num_offsets, int c_in, int c_out, int dtype, void *fragments,
                                hipStream_t stream) {
  SPIRA_HIP_REQUIRE(dtype == SPIRA_F16 || dtype == SPIRA_F32, "prepare_fragments: dtype must be fp16 or fp32");
  const int64_t n = static_cast<int64_t>(fragments_bytes(num_offsets, c_in, c_out, dtype) / 16);
  if (n == 0) return kOk;
  const int ctiles = static_cast<int>(div_up(c_out, 16)), nft = static_cast<int>(div_up(c_in, 32));
  hipLaunchKernelGGL(compact::fragments_kernel, dim3(div_up(n, 256)), dim3(256), 0, stream,
                     static_cast<const _Float16 *>(weights), n, c_in, c_out, ctiles, nft,
                     static_cast<_Float16 *>(fragments));
  SPIRA_HIP_LAUNCH_CHECK();
  return kOk;
}

}  // extern "C"

extern "C" {

int spira_hip_pad_rows(const void *sources, int64_t num_sources, int c_in, int row_channels, int dtype, void *rows,
                       hipStream_t stream) {
  SPIRA_HIP_REQUIRE(dtype == SPIRA_F16 || dtype == SPIRA_F32, "pad_rows: dtype must be fp16 or fp32");
  SPIRA_HIP_REQUIRE(c_in > 0 && row_channels >= c_in, "pad_rows: bad channel counts");
  const int64_t n = num_sources * row_channels;
  if (n <= 0) return kOk;
  SPIRA_HIP_REQUIRE(n < (int64_t(1) << 31), "pad_rows: too many elements");
  if (dtype == SPIRA_F16)
    hipLaunchKernelGGL(compact::pad_rows_kernel<_Float16>, dim3(div_up(n, 256)), dim3(256), 0, stream,
                       static_cast<const _Float16 *>(sources), n, c_in, row_channels, static_cast<_Float16 *>(rows));
  else
    hipLaunchKernelGGL(compact::pad_rows_kernel<float>, dim3(div_up(n, 256)), dim3(256), 0, stream,
                       static_cast<const float *>(sources), n, c_in, row_channels, static_cast<float *>(rows));
  SPIRA_HIP_LAUNCH_CHECK();
  return kOk;
}

int spira_hip_conv_map(int64_t num_sources, int64_t num_targets, int num_offsets, const int32_t *out_in_map,
                       const void *sources, int row_channels, int c_in, const void *weights,
                       const void *fragments, int c_out, int dtype, void *targets, const float *scale, const float *shift, const void *residual, int relu,
                       hipStream_t stream) {
  if (int rc = check_compact(num_sources, num_targets, row_channels, c_in, c_out, dtype, sources, weights, fragments)) return rc;
  SPIRA_HIP_REQUIRE(num_offsets > 0 && (out_in_map || num_targets <= 0), "conv_map: no map");
  if (num_targets <= 0) return kOk;
  compact::Entries en{};
  en.kind = compact::kRowsTK;
  en.idx = out_in_map;
  en.S = num_sources;
  return compact::launch(dtype, stream, en, num_targets, num_offsets,
                         make_layer(sources, num_sources, row_channels, c_in, weights, fragments, c_out, dtype, targets,
                                    scale, shift, residual, relu));
}

int spira_hip_conv_masks(int64_t num_sources, int64_t num_targets, int num_offsets, const int32_t *source_masks,
                         const int32_t *target_masks, int dense_offsets, const int32_t *dense_map, const void *sources,
                         int row_channels, int c_in, const void *weights, const void *fragments, int c_out, int dtype, void *targets,
                         const float *scale, const float *shift, const void *residual, int relu, void *workspace,
                         size_t workspace_bytes, hipStream_t stream) {
  if (int rc = check_compact(num_sources, num_targets, row_channels, c_in, c_out, dtype, sources, weights, fragments)) return rc;
  SPIRA_HIP_REQUIRE(num_offsets >= 0 && dense_offsets >= 0 && num_offsets + dense_offsets > 0,
                    "conv_masks: no offsets");
  SPIRA_HIP_REQUIRE(dense_offsets == 0 || dense_map || (dense_offsets == 1 && num_sources == num_targets),
                    "conv_masks: without a dense map there is one dense offset and as many sources as targets");
  const int64_t n = num_sources * num_offsets;
  SPIRA_HIP_REQUIRE(workspace_bytes >= static_cast<size_t>(n) * sizeof(int32_t) && (workspace || n == 0),
                    "conv_masks: workspace too small (spira_hip_conv_compact_workspace)");
  if (num_targets <= 0) return kOk;
  auto *list = static_cast<int32_t *>(workspace);
  if (n > 0) {
    hipLaunchKernelGGL(compact::mask_list_kernel, dim3(div_up(n, 256)), dim3(256), 0, stream, source_masks, n,
                       num_sources, list);
    SPIRA_HIP_LAUNCH_CHECK();
  }
  compact::Entries en{};
  // (without masked offsets there are no ranks to look up, and no list)
  en.kind = num_offsets > 0 ? compact::kMasks : compact::kRowsKT;
  en.idx = target_masks;
  en.ld = num_targets;
  en.list = list;
  en.S = num_sources;
  en.dense = dense_map;
  en.kd = dense_offsets;
  return compact::launch(dtype, stream, en, num_targets, num_offsets + dense_offsets,
                         make_layer(sources, num_sources, row_channels, c_in, weights, fragments, c_out, dtype, targets,
                                    scale, shift, residual, relu));
}

int spira_hip_conv_pairs(int64_t num_sources, int64_t num_targets, const int32_t *in_idx, const int32_t *out_idx,
                         int rows, const int32_t *naddrs, int64_t num_pairs, int mirror_rows, int dense_offsets,
                         const int32_t *dense_map, const void *sources, int row_channels, int c_in, const void *weights,
                         const void *fragments, int c_out, int dtype, void *targets, const float *scale,
                         const float *shift, const void *residual, int relu, void *workspace, size_t workspace_bytes,
                         hipStream_t stream) {
  if (int rc = check_compact(num_sources, num_targets, row_channels, c_in, c_out, dtype, sources, weights, fragments)) return rc;
  const int K = mirror_rows > 0 ? mirror_rows : rows;
  SPIRA_HIP_REQUIRE(rows >= 0 && rows <= K && (rows >= 1 || num_pairs == 0), "conv_pairs: bad row count");
  SPIRA_HIP_REQUIRE(dense_offsets == 0 || dense_map || (dense_offsets == 1 && num_sources == num_targets),
                    "conv_pairs: without a dense map there is one dense offset and as many sources as targets");
  if (num_targets <= 0) return kOk;
  SPIRA_HIP_REQUIRE(num_pairs < (int64_t(1) << 29), "conv_pairs: too many pairs");
  const int64_t ld = round_up(num_targets, 4), n = ld * K;
  const int64_t nh = round_up(div_up(num_targets, compact::kTargets), 4);
  // (16-byte parts: the rows and the blocks' heads, cleared together, the count
  // of repeated pairs, the pairs)
  SPIRA_HIP_REQUIRE(workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
                        workspace_bytes >= static_cast<size_t>(n + nh + 4 + 8 * num_pairs) * sizeof(int32_t),
                    "conv_pairs: workspace too small (spira_hip_conv_compact_workspace) or not 16-byte aligned");
  auto *idx = static_cast<int32_t *>(workspace);
  int32_t *heads = idx + n, *nextra = heads + nh;
  auto *extra = reinterpret_cast<int4 *>(nextra + 4);
  hipLaunchKernelGGL(compact::rows_clear_kernel, dim3(div_up((n + nh) / 4, 256)), dim3(256), 0, stream, idx,
                     (n + nh) / 4, nextra);
  SPIRA_HIP_LAUNCH_CHECK();
  if (num_pairs > 0) {
    hipLaunchKernelGGL(compact::pair_rows_kernel, dim3(div_up(num_pairs, 256)), dim3(256), 0, stream, in_idx, out_idx,
                       naddrs, rows, num_pairs, mirror_rows, num_sources, num_targets, ld, idx, heads, extra, nextra);
    SPIRA_HIP_LAUNCH_CHECK();
  }
  compact::Entries en{};
  en.kind = compact::kRowsKT;
  en.idx = idx;
  en.ld = ld;
  en.S = num_sources;
  en.dense = dense_map;
  en.kd = dense_offsets;
  en.extra = extra;
  en.heads = heads;
  return compact::launch(dtype, stream, en, num_targets, K + dense_offsets,
                         make_layer(sources, num_sources, row_channels, c_in, weights, fragments, c_out, dtype, targets,
                                    scale, shift, residual, relu));
}

}  // extern "C"
