// Chained downsample over occupancy grids: every level's sorted unique keys
// from one pass over the fine keys.
//
// Level l's keys are the distinct (key & stride mask l), in key order (x, y,
// z).  One bit per cell of the level's bounding box, z fastest, in 32-bit
// words: setting the bits of all keys drops the duplicates, and reading the
// words in order gives the sorted keys, so no level waits for the one before
// and nothing is searched or sorted.  Five launches for all levels:
//   grid_box_kernel    partial bounding boxes (and the sortedness check that
//                      the callers rely on);
//   grid_clear_kernel  the levels' extents from them; clears their words;
//   grid_set_kernel    one bit per key and level (a key whose predecessor
//                      falls in the same cell skips it);
//   grid_count_kernel  set bits per block, kBlocks equal shares of a level;
//   grid_emit_kernel   each block's keys after those of the blocks before.
// Bound by the launches and, in wide scenes, by three passes over the words:
// the words taken are at most kWordsPerKey per key (and kWordsLeast: 64 MB; up
// to kWordsMost: 256 MB), so that these passes stay below the searches that
// they replace.  (A network's map build, us, by merging -> by grids: 100k
// voxels of a sweep over 3200 x 3200 x 90 cells, 6.0M words, 299 -> 239, over
// 4800 x 4800 x 90, 13.5M words, 295 -> 265.)  A box with more cells sets bit 1
// of the flag and leaves the outputs undefined; the merging chain
// (spira_hip_downsample_chain) is then the call.
#include "common.hpp"
#include "../../../include/spira_hip.h"

#include <algorithm>

namespace spira_hip {

namespace grid {

constexpr int kLevels = 8;
constexpr int kBoxBlocks = 256;
constexpr int kBlocks = 512;                            // blocks per level of the count and the emission
constexpr int64_t kWordsPerKey = 32, kWordsLeast = int64_t(1) << 24, kWordsMost = int64_t(1) << 26;
constexpr uint32_t kUnsorted = 1, kTooWide = 2;

struct Strides {
  int n;
  int shift[kLevels][3];  // log2 of the stride per axis
};
struct Level {
  uint32_t base, words;  // first word and their number (a multiple of 4)
  uint32_t x0, y0, z0;   // the box's corner, in cells (z0 a multiple of 32)
  uint32_t ny, nzw;      // cells in y, words per (x, y) column
};
struct Plan {
  int fits;
  Level lv[kLevels];
};

template <typename CT> __device__ __forceinline__ uint32_t fx(CT k) {
  return static_cast<uint32_t>((k >> Layout<CT>::XS) & Layout<CT>::XONES);
}
template <typename CT> __device__ __forceinline__ uint32_t fy(CT k) {
  return static_cast<uint32_t>((k >> Layout<CT>::YS) & Layout<CT>::YONES);
}
template <typename CT> __device__ __forceinline__ uint32_t fz(CT k) {
  return static_cast<uint32_t>(k & Layout<CT>::ZONES);
}

// Minima (0..2) and maxima (3..5) of x, y, z over the block's values.
__device__ __forceinline__ void block_box(uint32_t (&v)[6], uint32_t (*red)[6]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    v[a] = wave_min<uint32_t>(v[a]);
    v[3 + a] = wave_max<uint32_t>(v[3 + a]);
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int a = 0; a < 6; ++a) red[threadIdx.x >> 6][a] = v[a];
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      v[a] = min(v[a], red[w][a]);
      v[3 + a] = max(v[3 + a], red[w][3 + a]);
    }
}

template <typename CT>
__global__ __launch_bounds__(256) void grid_box_kernel(const CT *__restrict__ in, int64_t n,
                                                       uint32_t *__restrict__ boxes, uint32_t *__restrict__ flag) {
  __shared__ uint32_t red[4][6];
  uint32_t v[6] = {~0u, ~0u, ~0u, 0, 0, 0};
  bool down = false;
  // (four keys and their predecessors in flight per thread; past the end: the
  // last key again)
  for (int64_t i0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i0 < n; i0 += kBoxBlocks * 1024) {
    CT k[4], p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t i = min(i0 + u * (kBoxBlocks * 256), n - 1);
      k[u] = in[i];
      p[u] = in[i > 0 ? i - 1 : 0];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      down |= p[u] > k[u];
      const uint32_t f[3] = {fx<CT>(k[u]), fy<CT>(k[u]), fz<CT>(k[u])};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        v[a] = min(v[a], f[a]);
        v[3 + a] = max(v[3 + a], f[a]);
      }
    }
  }
  if (down) atomicOr(flag, kUnsorted);
  block_box(v, red);
  if (threadIdx.x == 0)
#pragma unroll
    for (int a = 0; a < 6; ++a) boxes[blockIdx.x * 6 + a] = v[a];
}

static_assert(kBoxBlocks == 256, "one thread per box");

__global__ __launch_bounds__(256) void grid_clear_kernel(const uint32_t *__restrict__ boxes, const Strides st,
                                                         int64_t cap, uint32_t *__restrict__ words,
                                                         Plan *__restrict__ plan, uint32_t *__restrict__ flag) {
  __shared__ uint32_t red[4][6];
  uint32_t v[6] = {~0u, ~0u, ~0u, 0, 0, 0};
#pragma unroll
  for (int a = 0; a < 6; ++a) v[a] = boxes[threadIdx.x * 6 + a];
  block_box(v, red);
  uint64_t base = 0;
  bool fits = true;
  for (int l = 0; l < st.n; ++l) {
    uint32_t c[3];
    uint64_t e[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      c[a] = v[a] >> st.shift[l][a];
      if (a == 2) c[a] &= ~31u;
      e[a] = static_cast<uint64_t>(v[3 + a] >> st.shift[l][a]) - c[a] + 1;
    }
    // (24, 24 and 11 bits at most: no overflow)
    const uint64_t nzw = (e[2] + 31) / 32, w = (e[0] * e[1] * nzw + 3) / 4 * 4;
    fits = fits && base + w <= static_cast<uint64_t>(cap);
    if (!fits) break;
    if (blockIdx.x == 0 && threadIdx.x == 0)
      plan->lv[l] = Level{static_cast<uint32_t>(base), static_cast<uint32_t>(w), c[0], c[1], c[2],
                          static_cast<uint32_t>(e[1]), static_cast<uint32_t>(nzw)};
    base += w;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    plan->fits = fits ? 1 : 0;
    if (!fits) atomicOr(flag, kTooWide);
  }
  if (!fits) return;
  uint4 *w4 = reinterpret_cast<uint4 *>(words);
  const int64_t n4 = static_cast<int64_t>(base / 4);
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n4; i += static_cast<int64_t>(gridDim.x) * 256)
    w4[i] = uint4{0, 0, 0, 0};
}

// The cells 2^d apart that hold a set bit of m.
__device__ __forceinline__ uint32_t coarser(uint32_t m, int d) {
  if (d >= 5) return m != 0 ? 1u : 0u;
  for (; d > 0; --d) {
    m = (m | (m >> 1)) & 0x55555555u;
    m = (m | (m >> 1)) & 0x33333333u;
    m = (m | (m >> 2)) & 0x0F0F0F0Fu;
    m = (m | (m >> 4)) & 0x00FF00FFu;
    m = (m | (m >> 8)) & 0x0000FFFFu;
  }
  return m;
}

// Neighbouring lanes mostly share a word (keys run along z), so a wave ORs
// the bits of each run of lanes and its last lane sets them; of a coarser
// level's bits only those of cells that this lane was the first to set are
// passed on.  (One atomic per key and level: 58 us for 200k keys of an indoor
// scan, many of them on the same words.)  A word's 32 cells lie in one word
// of the next level, as both start at multiples of 32.
template <typename CT>
__global__ __launch_bounds__(256) void grid_set_kernel(const CT *__restrict__ in, int64_t n, const Strides st,
                                                       const Plan *__restrict__ plan, uint32_t *__restrict__ words) {
  if (!plan->fits) return;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const CT k = in[min(i, n - 1)];
  const uint32_t x = fx<CT>(k), y = fy<CT>(k);
  uint32_t z = fz<CT>(k) >> st.shift[0][2], m, w;
  {
    const Level &lv = plan->lv[0];
    w = (((x >> st.shift[0][0]) - lv.x0) * lv.ny + ((y >> st.shift[0][1]) - lv.y0)) * lv.nzw + ((z - lv.z0) >> 5);
    m = 1u << (z & 31);
    z &= ~31u;
  }
  // OR over the run of lanes that ends here (lanes past the end repeat the
  // last key and its word)
  uint32_t wp = __shfl_up(w, 1, 64);
  bool head = lane == 0 || wp != w;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t mo = __shfl_up(m, d, 64);
    const bool ho = __shfl_up(static_cast<int>(head), d, 64) != 0;
    if (lane >= d && !head) {
      m |= mo;
      head = ho;
    }
  }
  const uint32_t wn = __shfl_down(w, 1, 64);
  if (lane != 63 && wn == w) return;
  for (int l = 0; l < st.n; ++l) {
    const Level &lv = plan->lv[l];
    if (l > 0) {
      const int d = st.shift[l][2] - st.shift[l - 1][2];
      z >>= d;
      m = coarser(m, d) << (z & 31);
      z &= ~31u;
      w = (((x >> st.shift[l][0]) - lv.x0) * lv.ny + ((y >> st.shift[l][1]) - lv.y0)) * lv.nzw + ((z - lv.z0) >> 5);
    }
    m &= ~atomicOr(&words[static_cast<int64_t>(lv.base) + w], m);
    if (m == 0) return;
  }
}

// Block b's share of a level: whole rounds of 256 words.
__device__ __forceinline__ void share(const Level &lv, uint32_t &w0, uint32_t &w1) {
  const uint32_t per = ((lv.words + kBlocks - 1) / kBlocks + 255) / 256 * 256;
  const uint64_t a = static_cast<uint64_t>(per) * blockIdx.x;
  w0 = static_cast<uint32_t>(min(a, static_cast<uint64_t>(lv.words)));
  w1 = static_cast<uint32_t>(min(a + per, static_cast<uint64_t>(lv.words)));
}
__device__ __forceinline__ uint32_t bits4(const uint4 &q) {
  return __popc(q.x) + __popc(q.y) + __popc(q.z) + __popc(q.w);
}

__global__ __launch_bounds__(256) void grid_count_kernel(const Plan *__restrict__ plan,
                                                         const uint32_t *__restrict__ words,
                                                         uint32_t *__restrict__ counts) {
  if (!plan->fits) return;
  __shared__ uint32_t red[4];
  const Level lv = plan->lv[blockIdx.y];
  uint32_t w0, w1, c = 0;
  share(lv, w0, w1);
  const uint4 *w4 = reinterpret_cast<const uint4 *>(words + lv.base);
#pragma unroll 4
  for (uint32_t i = w0 / 4 + threadIdx.x; i < w1 / 4; i += 256) c += bits4(w4[i]);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.y * kBlocks + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

template <typename CT> struct Outs {
  CT *out[kLevels];
};

template <typename CT>
__global__ __launch_bounds__(256) void grid_emit_kernel(const Plan *__restrict__ plan, const Strides st,
                                                        const uint32_t *__restrict__ words,
                                                        const uint32_t *__restrict__ counts, int64_t n,
                                                        const Outs<CT> outs, uint32_t *__restrict__ d_counts) {
  if (!plan->fits) return;
  __shared__ uint32_t before[4], wtot[2][4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l = blockIdx.y, b = blockIdx.x;
  const Level lv = plan->lv[l];
  const uint32_t *cl = counts + l * kBlocks;
  uint32_t s = 0;
  for (int t = tid; t < b; t += 256) s += cl[t];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
  if (lane == 0) before[w] = s;
  __syncthreads();
  uint32_t run = before[0] + before[1] + before[2] + before[3];
  const uint32_t own = cl[b];
  if (b == kBlocks - 1 && tid == 0) d_counts[l] = run + own;
  if (own == 0) return;
  uint32_t w0, w1;
  share(lv, w0, w1);
  const uint4 *w4 = reinterpret_cast<const uint4 *>(words + lv.base);
  CT *__restrict__ out = outs.out[l];
  const int sx = st.shift[l][0], sy = st.shift[l][1], sz = st.shift[l][2];
  // a word per thread and round, so that few cells are written one after the
  // other; four in a share of more than four rounds (sparse words, and a
  // round costs a block scan)
  const bool wide = w1 - w0 > 1024;
  const uint32_t step = wide ? 4 : 1;
  int slot = 0;
  for (uint32_t r0 = w0; r0 < w1; r0 += 256 * step, slot ^= 1) {
    const uint32_t q0 = r0 + tid * step;
    uint4 q = {0, 0, 0, 0};
    if (q0 < w1) {
      if (wide) q = w4[q0 / 4];
      else q.x = words[lv.base + q0];
    }
    const uint32_t c = bits4(q);
    uint32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) wtot[slot][w] = incl;
    __syncthreads();  // (two slots: a round's totals are read before the round after next writes them)
    uint32_t pos = run + incl - c;
    for (int v = 0; v < w; ++v) pos += wtot[slot][v];
    run += wtot[slot][0] + wtot[slot][1] + wtot[slot][2] + wtot[slot][3];
    if (c == 0) continue;
    const uint32_t bits[4] = {q.x, q.y, q.z, q.w};
    uint32_t col = q0 / lv.nzw, zw = q0 - col * lv.nzw;
    uint32_t xc = col / lv.ny, yc = col - xc * lv.ny;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > 0 && !wide) break;
      const CT xy = static_cast<CT>((static_cast<CT>(xc + lv.x0) << sx << Layout<CT>::XS) |
                                    (static_cast<CT>(yc + lv.y0) << sy << Layout<CT>::YS));
      for (uint32_t m = bits[j]; m != 0; m &= m - 1) {
        const uint32_t zc = zw * 32 + static_cast<uint32_t>(__builtin_ctz(m)) + lv.z0;
        if (pos < n) out[pos] = xy | static_cast<CT>(static_cast<CT>(zc) << sz);
        ++pos;
      }
      if (++zw == lv.nzw) {
        zw = 0;
        if (++yc == lv.ny) {
          yc = 0;
          ++xc;
        }
      }
    }
  }
}

struct Parts {
  uint32_t *words, *boxes, *counts;
  Plan *plan;
  int64_t cap;
  size_t total;
};
static Parts parts(int64_t n, int levels, void *base) {
  Parts p{};
  p.cap = std::min(std::max(n * kWordsPerKey, kWordsLeast), kWordsMost);
  char *b = static_cast<char *>(base);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *q = b ? b + off : nullptr;
    off += (bytes + 255) / 256 * 256;
    return q;
  };
  p.words = reinterpret_cast<uint32_t *>(take(static_cast<size_t>(p.cap) * 4));
  p.boxes = reinterpret_cast<uint32_t *>(take(kBoxBlocks * 6 * 4));
  p.counts = reinterpret_cast<uint32_t *>(take(static_cast<size_t>(levels) * kBlocks * 4));
  p.plan = reinterpret_cast<Plan *>(take(sizeof(Plan)));
  p.total = off;
  return p;
}

template <typename CT>
static int run(const CT *keys, int64_t n, const Strides &st, void *const *outs, uint32_t *d_counts, uint32_t *d_flag,
               const Parts &p, hipStream_t s) {
  Outs<CT> o{};
  for (int l = 0; l < st.n; ++l) o.out[l] = static_cast<CT *>(outs[l]);
  const unsigned lv = static_cast<unsigned>(st.n);
  hipLaunchKernelGGL(grid_box_kernel<CT>, dim3(kBoxBlocks), dim3(256), 0, s, keys, n, p.boxes, d_flag);
  hipLaunchKernelGGL(grid_clear_kernel, dim3(kBlocks), dim3(256), 0, s, p.boxes, st, p.cap, p.words, p.plan, d_flag);
  hipLaunchKernelGGL(grid_set_kernel<CT>, dim3(static_cast<unsigned>(div_up(n, 256))), dim3(256), 0, s, keys, n, st,
                     p.plan, p.words);
  hipLaunchKernelGGL(grid_count_kernel, dim3(kBlocks, lv), dim3(256), 0, s, p.plan, p.words, p.counts);
  hipLaunchKernelGGL(grid_emit_kernel<CT>, dim3(kBlocks, lv), dim3(256), 0, s, p.plan, st, p.words, p.counts, n, o,
                     d_counts);
  SPIRA_HIP_LAUNCH_CHECK();
  return kOk;
}

}  // namespace grid

}  // namespace spira_hip

using namespace spira_hip;

extern "C" {

int spira_hip_downsample_grid_workspace(int64_t n, int levels, size_t *bytes) {
  SPIRA_HIP_REQUIRE(n >= 0 && n < (int64_t(1) << 31) && levels >= 1 && levels <= grid::kLevels,
                    "downsample_grid: 1 to 8 levels and fewer than 2^31 keys");
  *bytes = n == 0 ? 0 : grid::parts(n, levels, nullptr).total;
  return kOk;
}

int spira_hip_downsample_grid(const void *keys, int64_t n, int key_bits, int levels, const int32_t *strides,
                              void *const *out_keys, uint32_t *d_counts, uint32_t *d_flag, void *workspace,
                              size_t workspace_bytes, hipStream_t stream) {
  SPIRA_HIP_REQUIRE(key_bits == 32 || key_bits == 64, "downsample_grid: key_bits must be 32 or 64");
  SPIRA_HIP_REQUIRE(levels >= 1 && levels <= grid::kLevels && strides && out_keys && d_counts && d_flag,
                    "downsample_grid: bad arguments");
  SPIRA_HIP_REQUIRE(n >= 1 && n < (int64_t(1) << 31) && keys, "downsample_grid: needs 1 to 2^31 - 1 keys");
  grid::Strides st{};
  st.n = levels;
  for (int l = 0; l < levels; ++l) {
    SPIRA_HIP_REQUIRE(out_keys[l] != nullptr, "downsample_grid: missing output array");
    for (int a = 0; a < 3; ++a) {
      const int32_t v = strides[3 * l + a], prev = l > 0 ? strides[3 * (l - 1) + a] : 1;
      SPIRA_HIP_REQUIRE(v > 0 && (v & (v - 1)) == 0 && v >= prev && v < (1 << 24),
                        "downsample_grid: each stride must be a power of two and a multiple of the previous one");
      st.shift[l][a] = __builtin_ctz(static_cast<unsigned>(v));
    }
  }
  SPIRA_HIP_REQUIRE(workspace != nullptr && workspace_bytes >= grid::parts(n, levels, nullptr).total,
                    "downsample_grid: workspace too small");
  const grid::Parts p = grid::parts(n, levels, workspace);
  if (key_bits == 64)
    return grid::run<uint64_t>(static_cast<const uint64_t *>(keys), n, st, out_keys, d_counts, d_flag, p, stream);
  return grid::run<uint32_t>(static_cast<const uint32_t *>(keys), n, st, out_keys, d_counts, d_flag, p, stream);
}

}  // extern "C"
