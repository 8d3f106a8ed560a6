// partition.hip -- spatial binning on gfx950: cell hash per particle, stable
// LSD radix sort of (hash, slot), cell start/end ranges. Replaces the
// reference's calculate_hashes / thrust::stable_sort_by_key / bin_particles
// (spatialpartition_inline.h:49-115, spatialpartition.cpp:77-136).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "context.hpp"
#include "device.hpp"

namespace pmpm {

thread_local char g_last_error[256] = "";
void note_error(const char *what) { snprintf(g_last_error, sizeof(g_last_error), "%s", what); }
void note_hip_error(hipError_t e, const char *what) {
  snprintf(g_last_error, sizeof(g_last_error), "%s: %s (%d)", what, hipGetErrorString(e), (int)e);
}

__global__ void zero_kernel(uint32_t *p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

int zero_fill(void *ptr, int64_t n_words, hipStream_t s) {
  if (n_words <= 0) return PMPM_OK;
  int64_t blocks = ceil_div(n_words, 256);
  if (blocks > 16384) blocks = 16384;
  PMPM_LAUNCH(zero_kernel, (::pmpm::kname("zero_kernel", {})), dim3((unsigned)blocks), dim3(256), 0, s, (uint32_t *)ptr, n_words);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

// Up to kZeroLists buffers cleared by one launch (a fill kernel, so the
// sequence stays valid inside a captured graph).
__global__ void zero_lists_kernel(ZeroLists z) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int k = 0; k < z.count; ++k)
    for (int64_t i = t; i < z.n[k]; i += stride) z.p[k][i] = 0u;
}

int zero_fill_lists(const ZeroLists &z, hipStream_t s) {
  int64_t most = 0;
  for (int k = 0; k < z.count; ++k) most = z.n[k] > most ? z.n[k] : most;
  if (most <= 0) return PMPM_OK;
  int64_t blocks = ceil_div(most, 256);
  if (blocks > 16384) blocks = 16384;
  PMPM_LAUNCH(zero_lists_kernel, (::pmpm::kname("zero_lists_kernel", {})), dim3((unsigned)blocks), dim3(256), 0, s, z);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

// bins = trunc((x - origin) * inv_h) per axis (int cast truncates toward 0, as
// Eigen's cast<int>), hash = x + y*nx + z*nx*ny. Hashes outside
// [0, num_cells_total) are clamped to num_cells_total so they sort last and
// belong to no cell. The same launch clears the cell ranges (and the `clear`
// buffers) for the range pass that follows.
template <int D>
__global__ void hash_kernel(const float *__restrict__ x, int n, pmpm_grid g, uint32_t *__restrict__ hash,
                            int32_t *__restrict__ bins, int32_t *__restrict__ cstart, int32_t *__restrict__ cend,
                            ZeroLists clear) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int64_t k = t; k < g.num_cells_total; k += stride) {
    cstart[k] = 0;
    cend[k] = 0;
  }
  for (int q = 0; q < clear.count; ++q)
    for (int64_t k = t; k < clear.n[q]; k += stride) clear.p[q][k] = 0u;
  const int i = (int)t;
  if (i >= n) return;
  int b[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const float t = __fmul_rn(__fsub_rn(x[a * n + i], g.origin[a]), g.inv_cell_size);
    b[a] = (int)t;
  }
  int64_t h = b[0];
  if (D > 1) h += (int64_t)b[1] * g.num_cells[0];
  if (D > 2) h += (int64_t)b[2] * g.num_cells[0] * g.num_cells[1];
  const uint32_t key = (h < 0 || h >= g.num_cells_total) ? (uint32_t)g.num_cells_total : (uint32_t)h;
  hash[i] = key;
  if (bins) {
#pragma unroll
    for (int a = 0; a < D; ++a) bins[a * n + i] = b[a];
  }
}

// Per-block digit histogram (digits of RB bits), digit-major layout
// hist[digit * nblocks + block]. The keys arrive nearly sorted (the previous
// step's G2P wrote the particles in cell order), so a wave's 64 consecutive
// keys hold a few runs of one digit: the head lane of each run adds the
// run's length, one LDS atomic per run instead of one per key.
template <int RB>
__global__ __launch_bounds__(kSortBlock) void radix_hist_kernel(const uint32_t *__restrict__ keys, int n, int shift,
                                                                uint32_t *__restrict__ hist, int nblocks) {
  constexpr int R = 1 << RB;
  __shared__ uint32_t h[R];
  const int t = threadIdx.x, lane = t & 63;
  for (int d = t; d < R; d += kSortBlock) h[d] = 0u;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll 4
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t i = base + (int64_t)r * kSortBlock + t;
    const bool valid = i < n;  // a prefix of the wave's lanes
    const uint32_t d = valid ? (keys[i] >> shift) & (R - 1) : 0u;
    const uint32_t prev = (uint32_t)__shfl_up((int)d, 1, 64);
    const bool head = valid && (lane == 0 || prev != d);
    const uint64_t heads = __ballot(head);
    const int nvalid = __popcll(__ballot(valid));
    if (head) {
      const uint64_t later = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
      const int next = later ? __ffsll((unsigned long long)later) - 1 : nvalid;
      atomicAdd(&h[d], (uint32_t)(next - lane));
    }
  }
  __syncthreads();
  for (int d = t; d < R; d += kSortBlock) hist[(int64_t)d * nblocks + blockIdx.x] = h[d];
}

// Exclusive scan of each digit's column hist[d][0..nblocks) (one workgroup
// per digit); the column total goes to totals[d].
__global__ __launch_bounds__(256) void scan_columns_kernel(uint32_t *__restrict__ hist, int nblocks,
                                                           uint32_t *__restrict__ totals) {
  __shared__ uint32_t part[256];
  const int t = threadIdx.x;
  uint32_t *col = hist + (int64_t)blockIdx.x * nblocks;
  const int chunk = (nblocks + 255) / 256;
  const int b = t * chunk;
  const int e = min(b + chunk, nblocks);
  uint32_t s = 0;
  for (int i = b; i < e; ++i) s += col[i];
  part[t] = s;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const uint32_t v = (t >= off) ? part[t - off] : 0u;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  uint32_t run = (t > 0) ? part[t - 1] : 0u;
  for (int i = b; i < e; ++i) {
    const uint32_t v = col[i];
    col[i] = run;
    run += v;
  }
  if (t == 255) totals[blockIdx.x] = part[255];
}

// Stable scatter of the keys [first, end) by a digit of RB bits, each digit's
// next place in base[]. Within a round of kSortBlock keys (thread order == input
// order) a lane's rank among same-digit lanes of its wave comes from RB ballots;
// per-wave counts are combined per digit in LDS (thread d owns digit d).
template <int RB> struct ScatterLds {
  uint32_t base[1 << RB];
  uint32_t wcnt[kSortBlock / 64][1 << RB];
};
template <int RB>
__device__ __forceinline__ void scatter_tile(const uint32_t *__restrict__ keys_in, const int32_t *__restrict__ vals_in,
                                    uint32_t *__restrict__ keys_out, int32_t *__restrict__ vals_out, int64_t first,
                                    int64_t end, int shift, ScatterLds<RB> &lds) {
  constexpr int R = 1 << RB, W = kSortBlock / 64;
  static_assert(R <= kSortBlock, "one digit per thread");
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = t >> 6;
  const bool owner = t < R;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int64_t r = first; r < end; r += kSortBlock) {
    if (owner) {
#pragma unroll
      for (int q = 0; q < W; ++q) lds.wcnt[q][t] = 0u;
    }
    __syncthreads();
    const int64_t i = r + t;
    const bool valid = i < end;
    const uint32_t key = valid ? keys_in[i] : 0u;
    const uint32_t d = (key >> shift) & (R - 1);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < RB; ++bit) {
      const bool on = (d >> bit) & 1u;
      const uint64_t m = __ballot(on);
      peers &= on ? m : ~m;
    }
    const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
    if (valid && rank == 0) lds.wcnt[w][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    if (owner) {
      uint32_t run = lds.base[t];
#pragma unroll
      for (int q = 0; q < W; ++q) {
        const uint32_t c = lds.wcnt[q][t];
        lds.wcnt[q][t] = run;
        run += c;
      }
      lds.base[t] = run;
    }
    __syncthreads();
    if (valid) {
      const uint32_t pos = lds.wcnt[w][d] + rank;
      keys_out[pos] = key;
      vals_out[pos] = vals_in ? vals_in[i] : (int32_t)i;
    }
    __syncthreads();
  }
}

// One radix pass: the digit bases, then the tile's scatter.
template <int RB>
__global__ __launch_bounds__(kSortBlock) void radix_scatter_kernel(
    const uint32_t *__restrict__ keys_in, const int32_t *__restrict__ vals_in, uint32_t *__restrict__ keys_out,
    int32_t *__restrict__ vals_out, int n, int shift, const uint32_t *__restrict__ hist, int nblocks,
    const uint32_t *__restrict__ totals) {
  constexpr int R = 1 << RB, W = kSortBlock / 64;
  __shared__ ScatterLds<RB> lds;
  __shared__ uint32_t wsum[W];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = t >> 6;
  const bool owner = t < R;
  // digit bases: exclusive scan of the R column totals (thread d owns digit
  // d): a shuffle scan within each wave, then the wave totals before it
  const uint32_t tot = owner ? totals[t] : 0u;
  uint32_t incl = tot;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t before = 0u;
  for (int q = 0; q < w; ++q) before += wsum[q];
  if (owner) lds.base[t] = before + incl - tot + hist[(int64_t)t * nblocks + blockIdx.x];
  const int64_t tile = (int64_t)blockIdx.x * kSortTile;
  scatter_tile<RB>(keys_in, vals_in, keys_out, vals_out, tile, min(tile + kSortTile, (int64_t)n), shift, lds);
}

// Cell ranges over the sorted hashes (spatialpartition_inline.h:85-115);
// empty cells keep the 0 of the preceding clear (spatialpartition.cpp:81-82).
// The out-of-grid particles sort last: the first of them (or the last
// particle, when there are none) writes their count.
__global__ void cell_range_kernel(const uint32_t *__restrict__ hs, int n, uint32_t ncells,
                                  int32_t *__restrict__ cstart, int32_t *__restrict__ cend,
                                  uint32_t *__restrict__ out_of_grid) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const uint32_t h = hs[j];
  if (h >= ncells) {
    if (j == 0 || hs[j - 1] < ncells) *out_of_grid = (uint32_t)(n - j);
    return;
  }
  if (j == n - 1) *out_of_grid = 0u;
  if (j == 0 || hs[j - 1] != h) cstart[h] = j;
  if (j == n - 1 || hs[j + 1] != h) cend[h] = j + 1;
}

// ---- Partition from a sorted hint ----------------------------------------
// pmpm_step hands the particles to the next partition in the previous
// partition's (cell, slot) order, and that partition's sorted keys are still
// in hash_sorted. Used as a hint h[i], they equal the new key k[i] for every
// particle that kept its cell. If h is sorted, the particles with k[i] ==
// h[i] ("stayers") are in (key, slot) order among themselves already, so only
// the others ("movers") are ordered, per cell, and the stable order is a merge
// per cell c, with S[i] = stayers before slot i:
//   first slot of c: out_start[c] = particles with key < c
//   stayer i:        out_start[c] + (S[i] - stayers with key < c) + movers of c before slot i
//   mover i:         out_start[c] + movers of c before slot i
//                    + clamp(S[i] - stayers with key < c, 0, stayers of c)
// (stayers are sorted by key, so the first S[i] of them are those before i).
//
// Four launches whatever the mover count: classify (keys, stay bits, counts
// per cell), scan (cells), movers (each into its cell's part of a list, in any
// order), place (a particle counts the movers of its cell with a smaller slot:
// a step has a handful per 1000 particles). Cells with more than kHeavyMovers
// movers get their part of the list in slot order from a workgroup that walks
// all particles, and are searched by bisection, so no particle's count takes
// more than kHeavyMovers reads. The movers used to be sorted, in one workgroup
// up to 4,096 of them and by six multi-block radix launches otherwise, which
// cost their launch also when they had nothing to do: ten launches and 50 us
// at 1.08M particles, 39 us with these four. Small scenes gain most (17k
// particles: 45 us of radix sort, 17 us).
//
// A hint that says little (the first call on new buffers, particles in another
// order, most of them in another cell) is not merged: the same launches then
// sort all particles by their keys' high and low digits ("cold"; see
// hint_scan_kernel). Per-cell counts cost such a call an atomic per particle on
// a few cache lines, and ranking within a cell the square of its particles:
// partition of 20,000 particles in random order, 8 per cell, from a zero hint 70
// -> 39 us (radix sort: 51), 2,000 per cell 302 -> 38 (29, one digit); of
// 1,000,000, 27 per cell 819 -> 90 (75), 2,000 per cell 10,500 -> 104 (69).
constexpr int kHintBlock = 256;     // particles per workgroup of classify and place
constexpr int kHintCells = 1024;    // cells per workgroup of the scan
constexpr int kHintCellBits = 10;
constexpr int kHintSlots = 4;       // cell blocks a classify workgroup sums in LDS
constexpr int kMoverBlock = 1024;   // threads of the movers pass
constexpr int kHeavyMovers = 2048;
static_assert((1 << kHintCellBits) == kHintCells, "one cell per thread in the cell scan");
// A classify workgroup is cold when over half of its particles moved; the call
// is cold when the hint is unsorted or flat or over a sixteenth of the workgroups
// are, but no more than kColdLimit (counting 256 scattered particles costs
// atomics: 1,000,000 in random order, 244 workgroups counted: classify 61 us, 32:
// 29).
constexpr uint32_t kUnsorted = 0x80000000u;
constexpr int kColdLimit = 32;
constexpr int kColdBits = 10, kColdBuckets = 1 << kColdBits;  // high digit of a cold sort
constexpr int kColdCells = 1024;    // cells of a bucket that a place workgroup counts at a time
static_assert(kMoverBlock == kSortBlock && kColdBits <= kMaxRadixBits, "the cold scatter is a radix pass");
// (a hint that is one key throughout, as new buffers' are, is told by its ends)
__device__ inline bool flat_hint(const uint32_t *__restrict__ hint, int n) { return hint[0] == hint[n - 1]; }
struct Cold {
  uint32_t limit;            // cold workgroups of a call that is still merged
  int shift, buckets;        // bucket of a key: key >> shift
  int tile, tiles;           // particles per tile of the cold sort
  uint32_t *hist;            // [tiles][kColdBuckets] particles per tile and bucket, then each bucket's first place
  uint32_t *keys;            // the particles by bucket, in slot order
  int32_t *slots;
};

// Exclusive scan over a workgroup of THREADS threads; every thread gets its
// prefix and the total. `w` holds THREADS / 64 words of LDS.
template <int THREADS, class T>
__device__ __forceinline__ T block_exclusive_scan(T v, T *w, T &total) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  T incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T u = (T)__shfl_up((unsigned long long)incl, o, 64);
    if (lane >= o) incl += u;
  }
  __syncthreads();  // w may still be read by an earlier call
  if (lane == 63) w[wv] = incl;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int q = 0; q < THREADS / 64; ++q) {
    const T x = w[q];
    before += q < wv ? x : (T)0;
    all += x;
  }
  total = all;
  return before + incl - v;
}

template <int D>
__device__ inline uint32_t cell_key(const float *__restrict__ x, int n, int i, const pmpm_grid &g, int *b) {
#pragma unroll
  for (int a = 0; a < D; ++a) b[a] = (int)__fmul_rn(__fsub_rn(x[(int64_t)a * n + i], g.origin[a]), g.inv_cell_size);
  int64_t h = b[0];
  if (D > 1) h += (int64_t)b[1] * g.num_cells[0];
  if (D > 2) h += (int64_t)b[2] * g.num_cells[0] * g.num_cells[1];
  return (h < 0 || h >= g.num_cells_total) ? (uint32_t)g.num_cells_total : (uint32_t)h;
}

// Cell key per particle (as hash_kernel), its class against the hint as a bit
// (stay[i / 64]), and the counts: per cell and per block of cells, stayers and
// movers (a run of lanes with one key and one class adds its length once);
// stayers per workgroup. *cold counts the cold workgroups (kUnsorted: the hint
// is not sorted); once the call is cold, what is left of the counting is
// skipped. Blocks past the particles only clear `clear`.
template <int D>
__global__ __launch_bounds__(kHintBlock) void hint_classify_kernel(
    const float *__restrict__ x, int n, pmpm_grid g, const uint32_t *__restrict__ hint, uint32_t *__restrict__ hash,
    int32_t *__restrict__ bins, uint32_t *__restrict__ cnt, uint32_t *__restrict__ cbt, uint32_t *__restrict__ pblk,
    uint64_t *__restrict__ stay_bits, int npb, int ncb, uint32_t *__restrict__ cold, uint32_t limit, ZeroLists clear) {
  // per-class sums for the kHintSlots blocks of cells from the workgroup's
  // first key on (one global atomic per slot and class at the end: the
  // workgroups of a stretch of particles share these counters)
  __shared__ uint32_t slot_sum[kHintSlots][2];
  // the waves' stayers, kUnsorted in the top bit (read as one word of four)
  __shared__ __attribute__((aligned(16))) uint32_t wave_stay[kHintBlock / 64];
  __shared__ uint32_t first_block, skip;
  static_assert(kHintBlock == 256, "four waves");
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int q = 0; q < clear.count; ++q)
    for (int64_t k = t; k < clear.n[q]; k += stride) clear.p[q][k] = 0u;
  if ((int)blockIdx.x >= npb) return;  // block-uniform
  const int lane = threadIdx.x & 63;
  const int i = (int)t;
  const bool valid = i < n;  // a prefix of each wave
  uint32_t key = 0u;
  bool stay = false, falls = false;
  if (valid) {
    int b[3] = {0, 0, 0};
    key = cell_key<D>(x, n, i, g, b);
    hash[i] = key;
    if (bins) {
#pragma unroll
      for (int a = 0; a < D; ++a) bins[(int64_t)a * n + i] = b[a];
    }
    const uint32_t p = hint[i];
    falls = i + 1 < n && p > hint[i + 1];
    stay = key == p;
  }
  const uint64_t bits = __ballot(stay), fall_bits = __ballot(falls);
  if (lane == 0) {
    if (valid) stay_bits[i >> 6] = bits;
    wave_stay[threadIdx.x >> 6] = (uint32_t)__popcll(bits) | (fall_bits ? kUnsorted : 0u);
  }
  if (threadIdx.x < 2 * kHintSlots) (&slot_sum[0][0])[threadIdx.x] = 0u;
  if (threadIdx.x == 0) first_block = key >> kHintCellBits;
  lds_barrier();  // (the stores above are not waited for)
  const uint4 ws = *reinterpret_cast<const uint4 *>(wave_stay);
  const uint32_t unsorted = (ws.x | ws.y | ws.z | ws.w) & kUnsorted;
  const uint32_t stayers = (ws.x + ws.y + ws.z + ws.w) & 0xffffu;
  const int movers = min(n - (int)blockIdx.x * kHintBlock, kHintBlock) - (int)stayers;
  if (__builtin_expect(movers > kHintBlock / 2 || unsorted, 0)) {  // block-uniform
    if (flat_hint(hint, n)) return;  // (the scan pass looks too)
    if (threadIdx.x == 0) {
      // (the count only grows, so a workgroup that sees it past the limit may
      // stop: the call is cold)
      bool stop = __hip_atomic_load(cold, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > limit;
      if (!stop) stop = (unsorted ? atomicOr(cold, kUnsorted) | kUnsorted : atomicAdd(cold, 1u) + 1u) > limit;
      skip = stop ? 1u : 0u;
    }
    __syncthreads();
    if (skip) return;
  }
  const uint32_t cb0 = first_block;
  const uint32_t pk = (uint32_t)__shfl_up((int)key, 1, 64);
  const int ps = __shfl_up((int)stay, 1, 64);
  const bool head = valid && (lane == 0 || pk != key || ps != (int)stay);
  const uint64_t heads = __ballot(head);
  const int nvalid = __popcll(__ballot(valid));
  if (head) {
    const uint64_t later = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
    const int next = later ? __ffsll((unsigned long long)later) - 1 : nvalid;
    const uint32_t len = (uint32_t)(next - lane);
    const int cls = stay ? 0 : 1;
    atomicAdd(&cnt[2 * (int64_t)key + cls], len);
    const uint32_t cb = key >> kHintCellBits;
    if (cb >= cb0 && cb - cb0 < (uint32_t)kHintSlots) atomicAdd(&slot_sum[cb - cb0][cls], len);
    else atomicAdd(&cbt[2 * (int64_t)cb + cls], len);
  }
  lds_barrier();
  if (threadIdx.x == 0) pblk[blockIdx.x] = stayers;
  if (threadIdx.x < 2 * kHintSlots) {
    const uint32_t v = (&slot_sum[0][0])[threadIdx.x];
    const int sl = threadIdx.x >> 1, cls = threadIdx.x & 1;
    const int64_t cb = (int64_t)cb0 + sl;
    if (v && cb < ncb) atomicAdd(&cbt[2 * cb + cls], v);
  }
}

// The stayers and movers before each block of cells, by one workgroup, for grids
// of more than kScanBlocks such blocks: on smaller ones every scan workgroup adds
// up the blocks before its own, whose reads grow with the square of the cells
// (2^24 nodes, 1,000,000 particles: partition 278 us so, 254 with this launch;
// 2^25: 574 and 419; 2^22: 82 so, 90 with it).
constexpr int kScanBlocks = 4096;
__global__ __launch_bounds__(kMoverBlock) void hint_blocks_kernel(int ncb, const uint32_t *__restrict__ cbt,
                                                                  uint32_t *__restrict__ before) {
  __shared__ uint64_t w[kMoverBlock / 64];
  uint64_t base = 0u;
  for (int b0 = 0; b0 < ncb; b0 += 4 * kMoverBlock) {  // block-uniform
    uint64_t v[4], sum = 0u, tot;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int b = b0 + 4 * (int)threadIdx.x + q;
      const uint2 u = b < ncb ? *reinterpret_cast<const uint2 *>(cbt + 2 * (int64_t)b) : make_uint2(0u, 0u);
      v[q] = ((uint64_t)u.x << 32) | u.y;
      sum += v[q];
    }
    uint64_t at = base + block_exclusive_scan<kMoverBlock, uint64_t>(sum, w, tot);
    base += tot;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int b = b0 + 4 * (int)threadIdx.x + q;
      if (b < ncb) *reinterpret_cast<uint2 *>(before + 2 * (int64_t)b) = make_uint2((uint32_t)(at >> 32), (uint32_t)at);
      at += v[q];
    }
  }
}

// Block 0: the stayers before each particle block, and whether the call is cold
// (counters[2]). Blocks 1 .. ncb: 1024 cells each (cells 0..ncells, the last
// holding the out-of-grid particles), four consecutive cells per thread: the
// exclusive scans of the stayer and mover counts give each cell's record {first
// slot, stayers before, stayers, movers}, its range (cell_start/cell_end, 0 for
// an empty cell), for the last cell the out-of-grid count (counters[0]); the
// stayer counts are cleared for the next call, the mover counts are left to the
// movers pass, and cells with many movers are listed (counters[3] of them).
//
// Cold: the particles are sorted here and in the two launches after, by the high
// digit of their keys (kColdBuckets buckets at most) and then, a workgroup per
// bucket, by cell. This pass counts each tile's particles per bucket; the movers
// pass scatters the tiles stably to the buckets (every workgroup adds up the
// tiles before its own); the place pass counts and places a bucket's particles
// cell by cell in LDS and writes the cells' ranges. No global atomics, and the
// time does not depend on the particles per cell. What the classify pass had
// counted is cleared on the way.
constexpr int kScanThreads = kHintCells / 4;
__global__ __launch_bounds__(kScanThreads) void hint_scan_kernel(int n, uint32_t ncells, int npb, int ncb,
                                                                 uint32_t *__restrict__ cnt,
                                                                 const uint32_t *__restrict__ cbt,
                                                                 uint32_t *__restrict__ pblk,
                                                                 uint32_t *__restrict__ counters,
                                                                 int4 *__restrict__ info, int32_t *__restrict__ cstart,
                                                                 int32_t *__restrict__ cend, int32_t *__restrict__ heavy,
                                                                 uint32_t heavy_cap, const uint32_t *__restrict__ hash,
                                                                 const uint32_t *__restrict__ hint,
                                                                 const uint32_t *__restrict__ before, Cold cd) {
  __shared__ uint64_t w2[kScanThreads / 64];
  __shared__ uint32_t bucket[kColdBuckets];
  const bool cold = counters[1] > cd.limit || flat_hint(hint, n);
  const int t = threadIdx.x;
  if (__builtin_expect(cold, 0)) {
    for (int tile = (int)blockIdx.x; tile < cd.tiles; tile += (int)gridDim.x) {
      for (int k = t; k < kColdBuckets; k += kScanThreads) bucket[k] = 0u;
      __syncthreads();
      const int64_t first = (int64_t)tile * cd.tile, end = min(first + cd.tile, (int64_t)n);
      for (int64_t i = first + t; i < end; i += kScanThreads) atomicAdd(&bucket[hash[i] >> cd.shift], 1u);
      __syncthreads();
      for (int k = t; k < kColdBuckets; k += kScanThreads) cd.hist[(size_t)tile * kColdBuckets + k] = bucket[k];
      __syncthreads();
    }
    if (blockIdx.x == 0 && t == 0) counters[2] = 1u;
    return;
  }
  if (blockIdx.x == 0) {
    uint32_t base = 0u;
    for (int b0 = 0; b0 < npb; b0 += 4 * kScanThreads) {
      uint32_t v[4], sum = 0u;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = b0 + 4 * t + q;
        v[q] = b < npb ? pblk[b] : 0u;
        sum += v[q];
      }
      uint64_t tot;
      uint32_t at = base + (uint32_t)block_exclusive_scan<kScanThreads, uint64_t>(sum, w2, tot);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = b0 + 4 * t + q;
        if (b < npb) pblk[b] = at;
        at += v[q];
      }
      base += (uint32_t)tot;
    }
    if (t == 0) counters[2] = 0u;
    return;
  }
  if ((int)blockIdx.x > ncb) return;  // (a cold call's tiles)
  const int b = (int)blockIdx.x - 1;
  const int64_t c0 = (int64_t)b * kHintCells + 4 * t;
  uint32_t st[4], mv[4];  // (loaded before the prefix sums' barriers)
  const bool all4 = c0 + 3 <= (int64_t)ncells;
  if (all4) {
    const uint4 u = *reinterpret_cast<const uint4 *>(cnt + 2 * c0), v = *reinterpret_cast<const uint4 *>(cnt + 2 * c0 + 4);
    st[0] = u.x; mv[0] = u.y; st[1] = u.z; mv[1] = u.w;
    st[2] = v.x; mv[2] = v.y; st[3] = v.z; mv[3] = v.w;
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool valid = c0 + q <= (int64_t)ncells;
      st[q] = valid ? cnt[2 * (c0 + q)] : 0u;
      mv[q] = valid ? cnt[2 * (c0 + q) + 1] : 0u;
    }
  }
  uint64_t pt;  // (stayers << 32) | movers of the cell blocks before this one
  if (before) {
    const uint2 v = *reinterpret_cast<const uint2 *>(before + 2 * (int64_t)b);
    pt = ((uint64_t)v.x << 32) | v.y;
  } else {
    uint64_t pp = 0u;
    for (int j = t; j < b; j += kScanThreads) {
      const uint2 v = *reinterpret_cast<const uint2 *>(cbt + 2 * j);
      pp += ((uint64_t)v.x << 32) | v.y;
    }
    (void)block_exclusive_scan<kScanThreads, uint64_t>(pp, w2, pt);
  }
  uint32_t stay_before = (uint32_t)(pt >> 32);
  uint32_t mover_before = (uint32_t)pt;
  bool any = false;
  uint64_t own = 0u;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    any = any || (st[q] | mv[q]) != 0u;
    own += ((uint64_t)st[q] << 32) | mv[q];
  }
  uint64_t tot;
  const uint64_t ex = block_exclusive_scan<kScanThreads, uint64_t>(own, w2, tot);
  stay_before += (uint32_t)(ex >> 32);
  mover_before += (uint32_t)ex;
  int s4[4], e4[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t c = c0 + q;
    const uint32_t start = stay_before + mover_before, count = st[q] + mv[q];
    s4[q] = count ? (int)start : 0;
    e4[q] = count ? (int)(start + count) : 0;
    if (c <= (int64_t)ncells) {
      if (any) *reinterpret_cast<uint2 *>(cnt + 2 * c) = make_uint2(0u, mv[q]);
      info[c] = make_int4((int)start, (int)stay_before, (int)st[q], (int)mv[q]);
      if (mv[q] > (uint32_t)kHeavyMovers) {
        const uint32_t at = atomicAdd(&counters[3], 1u);
        if (at < heavy_cap) heavy[at] = (int32_t)c;
      }
      if (c == (int64_t)ncells) counters[0] = count;
    }
    stay_before += st[q];
    mover_before += mv[q];
  }
  const bool whole = c0 + 3 < (int64_t)ncells;
  if (whole && ((reinterpret_cast<uintptr_t>(cstart) | reinterpret_cast<uintptr_t>(cend)) & 15u) == 0u) {
    *reinterpret_cast<int4 *>(cstart + c0) = make_int4(s4[0], s4[1], s4[2], s4[3]);
    *reinterpret_cast<int4 *>(cend + c0) = make_int4(e4[0], e4[1], e4[2], e4[3]);
  } else {  // (the last cells, or caller's arrays that are not 16-byte aligned)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (c0 + q < (int64_t)ncells) {
        cstart[c0 + q] = s4[q];
        cend[c0 + q] = e4[q];
      }
  }
}

// Is particle i a mover? (stay bits of the classify pass)
__device__ inline bool is_mover(const uint64_t *__restrict__ stay_bits, int i) {
  return !((stay_bits[i >> 6] >> (i & 63)) & 1ull);
}

// Each mover's slot into its cell's part of `list` ([movers with a smaller
// key] on): taken from the cell's count downward, in any order; heavy cells by
// a workgroup each, in slot order. The counts end at zero, as the next call
// needs them, and block 0 clears the per-block cell counts and the count of cold
// workgroups. Cold: the scatter of a tile to the buckets.
__global__ __launch_bounds__(kMoverBlock) void hint_movers_kernel(int n, uint32_t ncells, int ncb, int words,
                                                                  const uint32_t *__restrict__ hash,
                                                                  const uint64_t *__restrict__ stay_bits,
                                                                  const int4 *__restrict__ info,
                                                                  uint32_t *__restrict__ cnt,
                                                                  uint32_t *__restrict__ cbt,
                                                                  uint32_t *__restrict__ counters,
                                                                  const int32_t *__restrict__ heavy,
                                                                  uint32_t heavy_cap, int32_t *__restrict__ list,
                                                                  Cold cd) {
  __shared__ uint32_t w[kMoverBlock / 64];
  __shared__ ScatterLds<kColdBits> lds;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  if (blockIdx.x == 0) {
    for (int j = t; j < 2 * ncb; j += kMoverBlock) cbt[j] = 0u;
    if (t == 0) counters[1] = 0u;
  }
  // a wave takes `words` words of stay bits (at most 16); they and the count of
  // heavy cells are in flight with the flag
  const int first = ((int)blockIdx.x * (kMoverBlock / 64) + wv) * 64 * words;
  const int word = (first >> 6) + lane;
  uint32_t word_lo = 0u, word_hi = 0u;
  if (lane < words && word < (n + 63) / 64) {
    const uint2 v = reinterpret_cast<const uint2 *>(stay_bits)[word];
    word_lo = v.x;
    word_hi = v.y;
  }
  const uint32_t cold = counters[2], nheavy = min(counters[3], heavy_cap);
  asm volatile("" : "+v"(word_lo), "+v"(word_hi));
  if (__builtin_expect(cold != 0u, 0)) {
    const int tile = (int)blockIdx.x;
    if (tile >= cd.tiles) return;
    // a bucket's first place, and this tile's: thread t's bucket is t
    // (sixteen rows in flight: each is a trip to memory)
    uint32_t total = 0u, mine = 0u;
    for (int j = 0; j < cd.tiles; j += 16) {
      uint32_t v[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) v[q] = cd.hist[(size_t)min(j + q, cd.tiles - 1) * kColdBuckets + t];
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        mine += j + q < tile ? v[q] : 0u;
        total += j + q < cd.tiles ? v[q] : 0u;
      }
    }
    uint32_t all;
    const uint32_t start = block_exclusive_scan<kMoverBlock, uint32_t>(total, w, all);
    if (tile == 0) cd.hist[(size_t)cd.tiles * kColdBuckets + t] = start;
    lds.base[t] = start + mine;
    const int64_t i0 = (int64_t)tile * cd.tile;
    scatter_tile<kColdBits>(hash, nullptr, cd.keys, cd.slots, i0, min(i0 + cd.tile, (int64_t)n), cd.shift, lds);
    return;
  }
  for (uint32_t h = blockIdx.x; h < nheavy; h += gridDim.x) {  // block-uniform
    const uint32_t c = (uint32_t)heavy[h];
    if (c > ncells) continue;
    const int4 in = info[c];
    const int base = in.x - in.y;
    uint32_t done = 0u;
    for (int i0 = 0; i0 < n; i0 += 4 * kMoverBlock) {
      bool mine[4];
      uint32_t m = 0u;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = i0 + 4 * t + q;
        mine[q] = i < n && hash[i] == c && is_mover(stay_bits, i);
        m += mine[q] ? 1u : 0u;
      }
      uint32_t all;
      uint32_t at = done + block_exclusive_scan<kMoverBlock, uint32_t>(m, w, all);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (mine[q]) {
          if (at < (uint32_t)in.w) list[base + (int)at] = i0 + 4 * t + q;
          ++at;
        }
      done += all;
    }
    if (t == 0) cnt[2 * (int64_t)c + 1] = 0u;
  }
  if (first >= n) return;
  const uint64_t bits = (uint64_t)word_hi << 32 | word_lo;
  for (int q = 0; q < words; ++q) {
    const int i = first + 64 * q + lane;
    const uint64_t stay = (uint64_t)__shfl((unsigned long long)bits, q);
    const bool mover = i < n && !((stay >> lane) & 1ull);
    if (!__ballot(mover)) continue;
    if (!mover) continue;
    const uint32_t c = hash[i];
    const int4 in = info[c];
    if (in.w > kHeavyMovers) continue;
    const int at = (int)atomicSub(&cnt[2 * (int64_t)c + 1], 1u) - 1;
    if (at >= 0 && at < in.w) list[in.x - in.y + at] = i;
  }
}

// The place pass of a cold call: one bucket's particles (in slot order) counted
// per cell, the cells' ranges, and the particles to their places; kColdCells of
// the bucket's cells at a time. Each wave takes a quarter of the particles with
// counters of its own, so the waves need no barrier while they place: a lane's
// rank among its wave's particles of the same cell comes from ballots over the
// cell's bits.
struct ColdCounters {
  uint32_t next[kHintBlock / 64][kColdCells];
};
__device__ __forceinline__ void place_bucket(int bucket, int n, uint32_t ncells, const Cold &cd, uint32_t *__restrict__ cnt,
                                    uint32_t *__restrict__ counters, int32_t *__restrict__ cstart,
                                    int32_t *__restrict__ cend, uint32_t *__restrict__ hash_sorted,
                                    int32_t *__restrict__ sorted, ColdCounters &lds, uint32_t *w) {
  constexpr int W = kHintBlock / 64, F = 2;  // F: rounds whose loads are in flight together
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const uint32_t *starts = cd.hist + (size_t)cd.tiles * kColdBuckets;
  const int first = (int)starts[bucket], end = bucket + 1 < cd.buckets ? (int)starts[bucket + 1] : n;
  const int quarter = (end - first + W - 1) / W;
  const int j_first = min(first + wv * quarter, end), j_end = min(j_first + quarter, end);
  const int64_t cells_end = min((int64_t)(bucket + 1) << cd.shift, (int64_t)ncells + 1);
  uint32_t *next = lds.next[wv];
  uint32_t placed = (uint32_t)first;
  for (int64_t r0 = (int64_t)bucket << cd.shift; r0 < cells_end; r0 += kColdCells) {  // block-uniform
    const int m = (int)min(cells_end - r0, (int64_t)kColdCells);
    const uint32_t c0 = (uint32_t)r0;
    const int per = (m + kHintBlock - 1) / kHintBlock;  // cells of a thread
    __syncthreads();  // (the counters of the range before are read)
    for (int c = t; c < per * kHintBlock; c += kHintBlock)
#pragma unroll
      for (int q = 0; q < W; ++q) lds.next[q][c] = 0u;
    __syncthreads();
    for (int j = j_first + lane; j < j_end; j += 64 * F) {
      uint32_t c[F];
#pragma unroll
      for (int q = 0; q < F; ++q) c[q] = j + 64 * q < j_end ? cd.keys[j + 64 * q] - c0 : 0xffffffffu;
#pragma unroll
      for (int q = 0; q < F; ++q)
        if (c[q] < (uint32_t)m) atomicAdd(&next[c[q]], 1u);
    }
    __syncthreads();
    uint32_t sum = 0u;
    for (int c = t * per; c < (t + 1) * per; ++c)
#pragma unroll
      for (int q = 0; q < W; ++q) sum += lds.next[q][c];
    uint32_t all;
    uint32_t at = placed + block_exclusive_scan<kHintBlock, uint32_t>(sum, w, all);
    placed += all;
    for (int c = t * per; c < (t + 1) * per; ++c) {
      const uint32_t start = at;
#pragma unroll
      for (int q = 0; q < W; ++q) {
        const uint32_t count = lds.next[q][c];
        lds.next[q][c] = at;
        at += count;
      }
      if (c < m) {
        const int64_t cell = r0 + c;
        *reinterpret_cast<uint2 *>(cnt + 2 * cell) = make_uint2(0u, 0u);
        if (cell < (int64_t)ncells) {
          cstart[cell] = at > start ? (int32_t)start : 0;
          cend[cell] = at > start ? (int32_t)at : 0;
        } else {
          counters[0] = at - start;  // out-of-grid particles
        }
      }
    }
    __syncthreads();
    const int cell_bits = 32 - __clz(m - 1);  // (0 for one cell: __clz(0) is 32)
    uint32_t key[F];
    int slot[F];
    auto load = [&](int j) {
#pragma unroll
      for (int q = 0; q < F; ++q) {
        const bool valid = j + 64 * q < j_end;
        key[q] = valid ? cd.keys[j + 64 * q] : 0xffffffffu;  // (in no cell)
        slot[q] = valid ? cd.slots[j + 64 * q] : 0;
      }
    };
    load(j_first + lane);
    for (int j0 = j_first; j0 < j_end; j0 += 64 * F) {  // wave-uniform
      uint32_t k[F];
      int i[F];
#pragma unroll
      for (int q = 0; q < F; ++q) {
        k[q] = key[q];
        i[q] = slot[q];
      }
      load(j0 + 64 * F + lane);  // (the next rounds', in flight meanwhile)
#pragma unroll
      for (int q = 0; q < F; ++q) {
        const uint32_t c = k[q] - c0;
        const bool mine = c < (uint32_t)m;
        uint64_t peers = __ballot(mine);
        if (!peers) continue;
        for (int bit = 0; bit < cell_bits; ++bit) {
          const bool on = (c >> bit) & 1u;
          const uint64_t v = __ballot(on);
          peers &= on ? v : ~v;
        }
        const int rank = __popcll(peers & ((1ull << lane) - 1ull));
        const int leader = mine ? __ffsll((unsigned long long)peers) - 1 : lane;
        uint32_t pos = 0u;
        if (mine && rank == 0) {
          pos = next[c];
          next[c] = pos + (uint32_t)__popcll(peers);
        }
        wave_lds_sync();  // (the next round's leaders are other lanes)
        pos = (uint32_t)__shfl((int)pos, leader) + (uint32_t)rank;
        if (mine && pos < (uint32_t)n) {
          sorted[pos] = i[q];
          hash_sorted[pos] = k[q];
        }
      }
    }
  }
}

// The merge: each particle's place, written to sorted and hash_sorted. Block 0
// also clears the count of heavy cells for the next call. Cold: the buckets.
__global__ __launch_bounds__(kHintBlock, 8) void hint_place_kernel(int n, uint32_t ncells,
                                                                const uint32_t *__restrict__ hash,
                                                                const uint64_t *__restrict__ stay_bits,
                                                                const uint32_t *__restrict__ pofs,
                                                                const int4 *__restrict__ info,
                                                                const int32_t *__restrict__ list,
                                                                uint32_t *__restrict__ counters,
                                                                uint32_t *__restrict__ hash_sorted,
                                                                int32_t *__restrict__ sorted,
                                                                uint32_t *__restrict__ cnt, int32_t *__restrict__ cstart,
                                                                int32_t *__restrict__ cend, Cold cd) {
  // (16 KB; half of it: merged calls of 1,080,000 particles 0.2 us shorter, cold ones
  // of 4,000,000 on 1.3M nodes 180 us longer)
  __shared__ ColdCounters lds;
  __shared__ uint32_t w[kHintBlock / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int i = (int)blockIdx.x * kHintBlock + t;
  const uint32_t cold = counters[2];
  if (blockIdx.x == 0 && t == 0) counters[3] = 0u;
  uint32_t k = hash[min(i, n - 1)];
  asm volatile("" : "+v"(k));  // (or this load waits for the flag's)
  if (__builtin_expect(cold != 0u, 0)) {
    for (int b = (int)blockIdx.x; b < cd.buckets; b += (int)gridDim.x)
      place_bucket(b, n, ncells, cd, cnt, counters, cstart, cend, hash_sorted, sorted, lds, w);
    return;
  }
  if (i >= n) return;
  const int4 c = info[k];
  // stayers before this slot: those before the block, the block's waves
  // before this one, the lanes before this one
  const int w0 = (int)blockIdx.x * (kHintBlock / 64);
  uint32_t S = pofs[blockIdx.x];
  uint64_t bits = 0ull;
#pragma unroll
  for (int q = 0; q < kHintBlock / 64; ++q) {
    if (q > wv) break;
    const uint64_t v = stay_bits[w0 + q];
    if (q < wv) S += (uint32_t)__popcll(v);
    else bits = v;
  }
  S += (uint32_t)__popcll(bits & ((1ull << lane) - 1ull));
  // movers of this cell before this slot
  const int32_t *part = list + (c.x - c.y);
  int before = 0;
  if (c.w <= kHeavyMovers) {
    for (int r = 0; r < c.w; ++r) before += part[r] < i ? 1 : 0;
  } else {
    int hi = c.w;
    while (before < hi) {
      const int mid = (before + hi) >> 1;
      if (part[mid] < i) before = mid + 1;
      else hi = mid;
    }
  }
  const int own = (int)S - c.y;
  const int pos = c.x + before + ((bits >> lane) & 1ull ? own : min(max(own, 0), c.z));
  if ((unsigned)pos >= (unsigned)n) return;  // (inconsistent counts)
  sorted[pos] = i;
  hash_sorted[pos] = k;
}

// The whole partition of a small scene in one workgroup: (cell, position) of
// up to E x T particles sorted in registers (bitonic network; positions make
// the keys distinct, so the order is the stable one), lane exchanges within a
// wave, LDS between waves, and the cell ranges from the sorted keys' ends.
// Such a scene's step is a chain of launches of a few microseconds each, and
// this is one instead of four. Bound by the chain of exchanges (45 of them for
// 512 particles; 66 for 2048, of which 11 stay in a thread). Step of 960
// particles in 2D: 45 -> 38 us, of 2016 in 3D: 41 -> 36; at 4032 (8 per thread)
// the sort of one CU is the slower one (47 us against 41).
// Exchanges over up to 8 lanes are DPP moves (a ds_bpermute waits for the LDS
// pipe of the one CU).
template <int DPP> __device__ inline uint32_t dpp_move(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, DPP, 0xf, 0xf, false);
}
__device__ inline uint32_t lane_xor(uint32_t v, int m) {  // m: a constant after unrolling
  if (m == 1) return dpp_move<0xb1>(v);                     // quad_perm 1 0 3 2
  if (m == 2) return dpp_move<0x4e>(v);                     // quad_perm 2 3 0 1
  if (m == 4) return dpp_move<0x141>(dpp_move<0x1b>(v));    // quad_perm 3 2 1 0 (^3), row_half_mirror (^7)
  if (m == 8) return dpp_move<0x128>(v);                    // row_ror:8
  return (uint32_t)__shfl_xor((int)v, m);
}
__device__ inline uint32_t median(uint32_t a, uint32_t b, uint32_t c) {  // one instruction
  return max(min(a, b), min(max(a, b), c));
}
constexpr int kSmallParticles = 2048, kSmallCells = 16384, kSmallIndexBits = 12;
template <int D, int E, int T>
__global__ __launch_bounds__(T) void small_partition_kernel(const float *__restrict__ x, int n, pmpm_grid g,
                                                            uint32_t ncells, uint32_t *__restrict__ hash,
                                                            int32_t *__restrict__ bins,
                                                            uint32_t *__restrict__ hash_sorted,
                                                            int32_t *__restrict__ sorted,
                                                            int32_t *__restrict__ cell_start,
                                                            int32_t *__restrict__ cell_end,
                                                            uint32_t *__restrict__ counters, ZeroLists clear) {
  constexpr int N = E * T;
  static_assert(N <= kSmallParticles && kSmallParticles <= 1 << kSmallIndexBits, "position bits");
  struct __attribute__((aligned(E * 4))) Own { uint32_t v[E]; };
  __shared__ Own s_own[2][T];
  const int t = threadIdx.x;
  for (int q = 0; q < clear.count; ++q)
    for (int64_t k = t; k < clear.n[q]; k += T) clear.p[q][k] = 0u;
  Own a;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int i = t * E + r;
    a.v[r] = 0xffffffffu;  // past the particles: sorts last
    if (i < n) {
      int b[3] = {0, 0, 0};
      const uint32_t key = cell_key<D>(x, n, i, g, b);
      hash[i] = key;
      if (bins) {
#pragma unroll
        for (int c = 0; c < D; ++c) bins[(int64_t)c * n + i] = b[c];
      }
      a.v[r] = key << kSmallIndexBits | (uint32_t)i;
    }
  }
  for (int c = t; c < (int)ncells; c += T) {  // (the ranges of non-empty cells overwrite these below)
    cell_start[c] = 0;
    cell_end[c] = 0;
  }
  int buf = 0;
#pragma unroll
  for (int k = 2; k <= N; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      // the median with 0 is the minimum, with ~0 the maximum
      if (j >= E) {
        Own o;
        if (j >= 64 * E) {
          s_own[buf][t] = a;
          __syncthreads();
          o = s_own[buf][t ^ (j / E)];
          buf ^= 1;  // (written again two barriers on)
        } else {
#pragma unroll
          for (int r = 0; r < E; ++r) o.v[r] = lane_xor(a.v[r], j / E);
        }
        const uint32_t bound = ((t & (k / E)) == 0) == ((t & (j / E)) == 0) ? 0u : ~0u;
#pragma unroll
        for (int r = 0; r < E; ++r) a.v[r] = median(a.v[r], o.v[r], bound);
      } else {
#pragma unroll
        for (int r = 0; r < E; ++r) {
          if (r & j) continue;
          const bool up = k < E ? (r & k) == 0 : (t & (k / E)) == 0;
          const uint32_t u = a.v[r], w = a.v[r | j], bound = up ? 0u : ~0u;
          a.v[r] = median(u, w, bound);
          a.v[r | j] = median(u, w, ~bound);
        }
      }
    }
  }
  s_own[buf][t] = a;
  __syncthreads();  // (and the cleared ranges are written)
  const uint32_t before = t > 0 ? s_own[buf][t - 1].v[E - 1] : 0xffffffffu;
  const uint32_t after = t < T - 1 ? s_own[buf][t + 1].v[0] : 0xffffffffu;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int e = t * E + r;
    if (e >= n) break;
    const uint32_t key = a.v[r] >> kSmallIndexBits;
    const uint32_t prev = (r > 0 ? a.v[r - 1] : before) >> kSmallIndexBits;
    const uint32_t next = (r < E - 1 ? a.v[r + 1] : after) >> kSmallIndexBits;
    sorted[e] = (int32_t)(a.v[r] & ((1u << kSmallIndexBits) - 1u));
    hash_sorted[e] = key;
    const bool head = e == 0 || prev != key, tail = e == n - 1 || next != key;
    if (key < ncells) {
      if (head) cell_start[key] = e;
      if (tail) cell_end[key] = e + 1;
      if (e == n - 1) counters[0] = 0u;
    } else if (head) {
      counters[0] = (uint32_t)(n - e);  // out-of-grid particles
    }
  }
}

}  // namespace pmpm

using namespace pmpm;

extern "C" const char *pmpm_last_error(void) { return g_last_error; }

extern "C" int pmpm_context_create(pmpm_context **ctx) {
  if (!ctx) return PMPM_ERR_INVALID;
  pmpm_context *c = new (std::nothrow) pmpm_context();
  if (!c) return PMPM_ERR_INVALID;
  if (!hip_ok(hipGetDevice(&c->device), "hipGetDevice")) { delete c; return PMPM_ERR_HIP; }
  const char *radix_only = getenv("PMPM_PARTITION_RADIX");
  c->sort_by_hint = !(radix_only && radix_only[0] == '1');
  const char *hint_min = getenv("PMPM_PARTITION_HINT_MIN");
  if (hint_min && hint_min[0]) c->hint_min_particles = (int32_t)strtol(hint_min, nullptr, 10);
  if (!hip_ok(hipMalloc(&c->counters, kCounters * sizeof(uint32_t)), "hipMalloc")) { delete c; return PMPM_ERR_HIP; }
  c->stray_flags = reinterpret_cast<int32_t *>(c->counters + 4);
  *ctx = c;
  return PMPM_OK;
}

int pmpm::ensure_tiles(pmpm_context *ctx, const TileSizes &want) {
  TileSizes &cap = ctx->tile_cap;
  if (want.partials <= cap.partials && want.flags <= cap.flags && want.clamp <= cap.clamp && want.strays <= cap.strays)
    return PMPM_OK;
  const TileSizes to{std::max(want.partials, cap.partials), std::max(want.flags, cap.flags),
                     std::max(want.clamp, cap.clamp), std::max(want.strays, cap.strays)};
  (void)hipFree(ctx->tile_mem);
  ctx->tile_mem = ctx->partials = ctx->clamp_mask = ctx->strays = nullptr;
  ctx->tile_flags = nullptr;
  cap = TileSizes{};
  auto up = [](size_t w) { return (w + 63) / 64 * 64; };
  PMPM_HIP_CHECK(hipMalloc(&ctx->tile_mem,
                           (up(to.partials) + up(to.flags) + up(to.clamp) + to.strays) * sizeof(float)));
  ctx->partials = ctx->tile_mem;
  float *flags = ctx->partials + up(to.partials);
  ctx->tile_flags = reinterpret_cast<int32_t *>(flags);
  ctx->clamp_mask = flags + up(to.flags);
  ctx->strays = ctx->clamp_mask + up(to.clamp);
  ctx->strays_clear = false;
  cap = to;
  return PMPM_OK;
}

int pmpm::ensure_buffer(float *&buf, size_t &cap, size_t floats) {
  if (floats > cap) {
    (void)hipFree(buf);
    buf = nullptr;
    cap = 0;
    PMPM_HIP_CHECK(hipMalloc(&buf, floats * sizeof(float)));
    cap = floats;
  }
  return PMPM_OK;
}

extern "C" int pmpm_context_destroy(pmpm_context *ctx) {
  if (!ctx) return PMPM_OK;
  (void)hipFree(ctx->adj_rec);
  (void)hipFree(ctx->adj_nodes);
  (void)hipFree(ctx->adj_pb);
  (void)hipFree(ctx->tile_mem);
  (void)hipFree(ctx->hint_mem);
  (void)hipFree(ctx->keys_tmp);
  (void)hipFree(ctx->vals_tmp);
  (void)hipFree(ctx->hist);
  (void)hipFree(ctx->counters);
  delete ctx;
  return PMPM_OK;
}

// Is the partition of n particles on ncells cells from the hint? Its scan writes
// 32 bytes per cell, the radix sort's clear 8, so few particles on a large grid
// are sorted. Merged and sorted, us: 2^22 nodes, 3,000 particles 52 and 66,
// 1,000,000: 90 and 114; 2^23, 3,000: 78 and 69, 1,000,000: 143 and 122,
// 4,000,000: 196 and 298; 2^24, 1,000,000: 254 and 137, 4,000,000: 382 and 326,
// 16,000,000: 499 and 1,123; 2^26, 16,000,000: 1,395 and 1,461.
constexpr int64_t kHintNodes = 1 << 22, kHintNodesPerParticle = 3;
static bool use_hint(const pmpm_context *ctx, int n, int64_t ncells) {
  return ctx->sort_by_hint && n >= ctx->hint_min_particles && ncells <= kHintNodes + kHintNodesPerParticle * n;
}
static int reserve_hint(pmpm_context *ctx, int n, uint32_t ncells);

extern "C" int pmpm_context_reserve(pmpm_context *ctx, int32_t max_particles, int32_t max_cells) {
  if (!ctx || max_particles < 0 || max_cells < 0) return PMPM_ERR_INVALID;
  if (max_particles > ctx->cap_particles) {
    (void)hipFree(ctx->keys_tmp);
    (void)hipFree(ctx->vals_tmp);
    (void)hipFree(ctx->hist);
    ctx->keys_tmp = nullptr; ctx->vals_tmp = nullptr; ctx->hist = nullptr; ctx->cap_particles = 0;
    const size_t np = (size_t)(max_particles > 0 ? max_particles : 1);
    const size_t nblocks = (size_t)ceil_div((int64_t)np, kSortTile);
    ctx->hist_len = (size_t)kMaxRadix * nblocks + kMaxRadix;  // + digit totals
    PMPM_HIP_CHECK(hipMalloc(&ctx->keys_tmp, np * sizeof(uint32_t)));
    PMPM_HIP_CHECK(hipMalloc(&ctx->vals_tmp, np * sizeof(int32_t)));
    PMPM_HIP_CHECK(hipMalloc(&ctx->hist, ctx->hist_len * sizeof(uint32_t)));
    ctx->cap_particles = max_particles;
  }
  if (max_cells > ctx->cap_cells) ctx->cap_cells = max_cells;
  if (ctx->sort_by_hint && max_particles >= ctx->hint_min_particles && max_particles > 0 && max_cells > 0 &&
      (max_particles > kSmallParticles || max_cells > kSmallCells)) {
    // the hint partition's workspace too, for the grids it is used on, so that
    // stepping within these sizes allocates nothing
    const int64_t cells = std::min<int64_t>(max_cells, kHintNodes + kHintNodesPerParticle * max_particles);
    int rc = reserve_hint(ctx, max_particles, (uint32_t)cells);
    if (rc != PMPM_OK) return rc;
  }
  // what must be zero between calls is so when this returns, whatever stream
  // uses it first, and also if that use is only recorded (a captured graph)
  if (!ctx->counters_clear || (ctx->hint_mem && !ctx->hint_clear)) {
    ZeroLists z{};
    z.add(ctx->counters, kCounters);
    z.add(ctx->hint_mem, (int64_t)ctx->hint_zero_words);
    int rc = zero_fill_lists(z, nullptr);
    if (rc != PMPM_OK) return rc;
    PMPM_HIP_CHECK(hipStreamSynchronize(nullptr));
    ctx->counters_clear = true;
    ctx->hint_clear = ctx->hint_mem != nullptr;
  }
  return PMPM_OK;
}

int pmpm::clear_on_stream(const ZeroLists &z, bool &clear, hipStream_t s) {
  if (clear) return PMPM_OK;
  int rc = zero_fill_lists(z, s);
  if (rc != PMPM_OK) return rc;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  PMPM_HIP_CHECK(hipStreamIsCapturing(s, &capture));
  clear = capture == hipStreamCaptureStatusNone;
  return PMPM_OK;
}

// The counters of a context that was not reserved for anything yet.
static int clear_counters(pmpm_context *ctx, hipStream_t s) {
  ZeroLists z{};
  z.add(ctx->counters, kCounters);
  return clear_on_stream(z, ctx->counters_clear, s);
}

extern "C" int pmpm_context_out_of_grid(pmpm_context *ctx, pmpm_stream_t stream, int32_t *count) {
  if (!ctx || !count) return PMPM_ERR_INVALID;
  uint32_t v = 0;
  int rc = clear_counters(ctx, (hipStream_t)stream);
  if (rc != PMPM_OK) return rc;
  PMPM_HIP_CHECK(hipMemcpyAsync(&v, ctx->counters, sizeof(uint32_t), hipMemcpyDeviceToHost, (hipStream_t)stream));
  PMPM_HIP_CHECK(hipStreamSynchronize((hipStream_t)stream));
  *count = (int32_t)v;
  return PMPM_OK;
}

// LSD radix sort of (key, position) pairs by keys in [0, ncells]: n keys
// from kin, values = positions in kin; the passes alternate between (ktmp, vtmp) and (kdst,
// vdst), the last one writing (kdst, vdst). kin may alias neither.
static int radix_sort_pairs(pmpm_context *ctx, const uint32_t *kin, uint32_t *ktmp, int32_t *vtmp, uint32_t *kdst,
                            int32_t *vdst, int n, uint32_t ncells, hipStream_t s) {
  int bits = 1;
  while (bits < 32 && ((uint64_t)1 << bits) <= (uint64_t)ncells) ++bits;
  // 10-bit digits: 2 passes up to 2^20 cells (8-bit digits when one pass
  // of them covers the keys)
  const int rb = bits <= 8 ? 8 : 10;
  const int passes = (bits + rb - 1) / rb;
  const int nblocks = (int)ceil_div(n, kSortTile);
  const int32_t *vin = nullptr;  // identity on the first pass
  for (int p = 0; p < passes; ++p) {
    const bool to_dest = ((passes - 1 - p) % 2) == 0;
    uint32_t *kout = to_dest ? kdst : ktmp;
    int32_t *vout = to_dest ? vdst : vtmp;
    const int shift = p * rb;
    const int radix = 1 << rb;
    uint32_t *totals = ctx->hist + (size_t)radix * nblocks;
    if (rb == 8) {
      PMPM_LAUNCH(radix_hist_kernel<8>, (::pmpm::kname("radix_hist_kernel", {(long)(8)})), dim3(nblocks), dim3(kSortBlock), 0, s, kin, n, shift, ctx->hist, nblocks);
      PMPM_LAUNCH_CHECK();
      PMPM_LAUNCH(scan_columns_kernel, (::pmpm::kname("scan_columns_kernel", {})), dim3(radix), dim3(256), 0, s, ctx->hist, nblocks, totals);
      PMPM_LAUNCH_CHECK();
      PMPM_LAUNCH(radix_scatter_kernel<8>, (::pmpm::kname("radix_scatter_kernel", {(long)(8)})), dim3(nblocks), dim3(kSortBlock), 0, s, kin, vin, kout, vout, n,
                  shift, ctx->hist, nblocks, totals);
    } else {
      PMPM_LAUNCH(radix_hist_kernel<10>, (::pmpm::kname("radix_hist_kernel", {(long)(10)})), dim3(nblocks), dim3(kSortBlock), 0, s, kin, n, shift, ctx->hist,
                  nblocks);
      PMPM_LAUNCH_CHECK();
      PMPM_LAUNCH(scan_columns_kernel, (::pmpm::kname("scan_columns_kernel", {})), dim3(radix), dim3(256), 0, s, ctx->hist, nblocks, totals);
      PMPM_LAUNCH_CHECK();
      PMPM_LAUNCH(radix_scatter_kernel<10>, (::pmpm::kname("radix_scatter_kernel", {(long)(10)})), dim3(nblocks), dim3(kSortBlock), 0, s, kin, vin, kout, vout, n,
                  shift, ctx->hist, nblocks, totals);
    }
    PMPM_LAUNCH_CHECK();
    kin = kout;
    vin = vout;
  }
  return PMPM_OK;
}

// The per-particle part of the hint workspace, in 32-bit words: the stay bits,
// the stayers per particle block, the heavy cells, the movers by cell; each
// starts on a 256-byte boundary.
struct HintLayout {
  size_t bits, pblk, heavy, list, words;
  uint32_t heavy_cap;
};
static HintLayout hint_layout(int n) {
  auto up = [](size_t w) { return (w + 63) / 64 * 64; };
  HintLayout l;
  l.heavy_cap = (uint32_t)(n / kHeavyMovers + 1);
  l.bits = 0;
  l.pblk = l.bits + up(2 * (size_t)ceil_div(n, 64));
  l.heavy = l.pblk + up((size_t)ceil_div(n, kHintBlock));
  l.list = l.heavy + up(l.heavy_cap);
  l.words = l.list + up((size_t)n);
  return l;
}

// Grows the hint workspace to n particles on ncells cells (one allocation). The
// counts must be zero between calls: new ones are marked, and cleared by
// pmpm_context_reserve or, if they grew in a partition, by that partition on its
// stream.
static int reserve_hint(pmpm_context *ctx, int n, uint32_t ncells) {
  const size_t words = hint_layout(n).words, cells = (size_t)ncells + 1;
  if (words <= ctx->hint_part_cap && cells <= ctx->hint_cells_cap) return PMPM_OK;
  const size_t to_words = std::max(words, ctx->hint_part_cap), to_cells = std::max(cells, ctx->hint_cells_cap);
  (void)hipFree(ctx->hint_mem);
  ctx->hint_mem = nullptr;
  ctx->hint_part_cap = ctx->hint_cells_cap = 0;
  ctx->hint_clear = false;
  auto up = [](size_t w) { return (w + 63) / 64 * 64; };
  // (the blocks' counts, and where hint_blocks_kernel leaves their sums)
  const size_t blocks = (size_t)ceil_div((int64_t)to_cells, kHintCells);
  const size_t o_cbt = up(2 * to_cells), o_sums = o_cbt + up(2 * blocks), o_info = o_sums + up(2 * blocks),
               o_part = o_info + up(4 * to_cells);
  PMPM_HIP_CHECK(hipMalloc(&ctx->hint_mem, (o_part + to_words) * sizeof(uint32_t)));
  ctx->hint_cnt = ctx->hint_mem;
  ctx->hint_cbt = ctx->hint_mem + o_cbt;
  ctx->hint_sums = ctx->hint_mem + o_sums;
  ctx->hint_info = ctx->hint_mem + o_info;
  ctx->hint_part = ctx->hint_mem + o_part;
  ctx->hint_zero_words = o_sums;  // (cnt and cbt)
  ctx->hint_part_cap = to_words;
  ctx->hint_cells_cap = to_cells;
  return PMPM_OK;
}

// The one-workgroup partition (small_partition_kernel).
template <int E, int T>
static int partition_small(pmpm_context *ctx, int dim, const pmpm_grid &g, const float *x, int n, pmpm_spatial *part,
                           hipStream_t s, const ZeroLists &extra) {
#define PMPM_SMALL(D)                                                                                              \
  PMPM_LAUNCH((small_partition_kernel<D, E, T>), (::pmpm::kname("small_partition_kernel", {(long)(D)})), dim3(1),   \
              dim3(T), 0, s, x, n, g, (uint32_t)g.num_cells_total, part->hash, part->bins, part->hash_sorted,       \
              part->sorted, part->cell_start, part->cell_end, ctx->counters, extra)
  switch (dim) {
    case 1: PMPM_SMALL(1); break;
    case 2: PMPM_SMALL(2); break;
    default: PMPM_SMALL(3); break;
  }
#undef PMPM_SMALL
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

// The partition from the hint in part->hash_sorted (see hint_classify_kernel).
static int partition_by_hint(pmpm_context *ctx, int dim, const pmpm_grid &g, const float *x, int n,
                             pmpm_spatial *part, hipStream_t s, const ZeroLists &extra) {
  const uint32_t ncells = (uint32_t)g.num_cells_total;
  const int ncb = (int)ceil_div((int64_t)ncells + 1, kHintCells);
  const int npb = (int)ceil_div(n, kHintBlock);
  int rc;
  if ((rc = reserve_hint(ctx, n, ncells)) != PMPM_OK) return rc;
  if (!ctx->hint_clear) {
    ZeroLists z{};
    z.add(ctx->hint_mem, (int64_t)ctx->hint_zero_words);
    if ((rc = clear_on_stream(z, ctx->hint_clear, s)) != PMPM_OK) return rc;
  }
  const HintLayout l = hint_layout(n);
  uint32_t *base = ctx->hint_part;
  uint64_t *bits = reinterpret_cast<uint64_t *>(base + l.bits);
  uint32_t *pblk = base + l.pblk;
  int32_t *heavy = reinterpret_cast<int32_t *>(base + l.heavy), *list = reinterpret_cast<int32_t *>(base + l.list);
  uint32_t *cnt = ctx->hint_cnt, *cbt = ctx->hint_cbt;
  int4 *info = reinterpret_cast<int4 *>(ctx->hint_info);
  // a wave waits for each of its movers' chain of reads in turn: one word of
  // stay bits per wave on small scenes (16 words at 40,000 particles: 14 us,
  // one: 7), more where the waves alone would fill the chip many times over
  const int mover_words = n < (1 << 18) ? 1 : (n < (1 << 22) ? n >> 18 : 16);
  const int mover_blocks = (int)ceil_div(n, (int64_t)mover_words * kMoverBlock);
  // a cold call's buckets: as many as the high digit has, for short chains in
  // the place pass; its tiles: one per movers workgroup
  Cold cd;
  cd.limit = (uint32_t)std::min(npb / 16, kColdLimit);
  cd.shift = 0;
  while ((ncells >> cd.shift) >= (uint32_t)kColdBuckets) ++cd.shift;
  cd.buckets = (int)(ncells >> cd.shift) + 1;
  // (a movers workgroup reads every tile's counts, so their bytes grow with the
  // square of the tiles; fewer tiles are longer chains. The sum is least near the
  // cube root: movers pass of 4,000,000 particles 109 -> 80 us against tiles as
  // small as the workgroups allow)
  cd.tile = kMoverBlock * std::max({mover_words, kSortItems, (int)(n / (1024.0 * std::cbrt(2.4 * n))) + 1});
  cd.tiles = (int)ceil_div(n, cd.tile);
  cd.hist = ctx->hist;
  cd.keys = ctx->keys_tmp;
  cd.slots = ctx->vals_tmp;
  if ((size_t)(cd.tiles + 1) * kColdBuckets > ctx->hist_len) {
    note_error("partition: histogram workspace");
    return PMPM_ERR_WORKSPACE;
  }
  // classify: enough workgroups for the particles and for the clears
  int64_t words = 0;
  for (int q = 0; q < extra.count; ++q) words = extra.n[q] > words ? extra.n[q] : words;
  int64_t nb = npb;
  const int64_t nb_clear = ceil_div(words, (int64_t)kHintBlock * 4);
  if (nb_clear > nb) nb = nb_clear < 16384 ? nb_clear : (nb > 16384 ? nb : 16384);
#define PMPM_CLASSIFY(D)                                                                                               \
  PMPM_LAUNCH(hint_classify_kernel<D>, (::pmpm::kname("hint_classify_kernel", {(long)(D)})), dim3((unsigned)nb),       \
              dim3(kHintBlock), 0, s, x, n, g, part->hash_sorted, part->hash, part->bins, cnt, cbt, pblk, bits, npb, ncb, \
              ctx->counters + 1, cd.limit, extra)
  switch (dim) {
    case 1: PMPM_CLASSIFY(1); break;
    case 2: PMPM_CLASSIFY(2); break;
    default: PMPM_CLASSIFY(3); break;
  }
#undef PMPM_CLASSIFY
  PMPM_LAUNCH_CHECK();
  uint32_t *before = nullptr;
  if (ncb > kScanBlocks) {
    before = ctx->hint_sums;
    PMPM_LAUNCH(hint_blocks_kernel, (::pmpm::kname("hint_blocks_kernel", {})), dim3(1), dim3(kMoverBlock), 0, s, ncb, cbt,
                before);
    PMPM_LAUNCH_CHECK();
  }
  PMPM_LAUNCH(hint_scan_kernel, (::pmpm::kname("hint_scan_kernel", {})), dim3((unsigned)std::max(ncb + 1, cd.tiles)),
              dim3(kScanThreads), 0, s, n, ncells, npb, ncb, cnt, cbt, pblk, ctx->counters, info, part->cell_start,
              part->cell_end, heavy, l.heavy_cap, part->hash, part->hash_sorted, before, cd);
  PMPM_LAUNCH_CHECK();
  PMPM_LAUNCH(hint_movers_kernel, (::pmpm::kname("hint_movers_kernel", {})), dim3((unsigned)mover_blocks),
              dim3(kMoverBlock), 0, s, n, ncells, ncb, mover_words, part->hash, bits, info, cnt, cbt, ctx->counters, heavy,
              l.heavy_cap, list, cd);
  PMPM_LAUNCH_CHECK();
  // (a cold call of few particles: up to four buckets per workgroup)
  PMPM_LAUNCH(hint_place_kernel, (::pmpm::kname("hint_place_kernel", {})),
              dim3((unsigned)std::max(npb, std::min(cd.buckets, kColdBuckets / 4))),
              dim3(kHintBlock), 0, s, n, ncells, part->hash, bits, pblk, info, list, ctx->counters, part->hash_sorted,
              part->sorted, cnt, part->cell_start, part->cell_end, cd);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

int pmpm::partition_clearing(pmpm_context *ctx, int dim, const pmpm_grid *grid, const float *x, int n,
                             pmpm_spatial *part, hipStream_t s, const ZeroLists &extra) {
  if (!ctx || !grid_ok(grid) || !part || dim < 1 || dim > 3 || n < 0) return PMPM_ERR_INVALID;
  if (n > 0 && (!x || !part->hash || !part->hash_sorted || !part->sorted)) return PMPM_ERR_INVALID;
  if (!part->cell_start || !part->cell_end || grid->num_cells_total <= 0) return PMPM_ERR_INVALID;
  if (n > ctx->cap_particles) return PMPM_ERR_WORKSPACE;
  const pmpm_grid g = *grid;
  const uint32_t ncells = (uint32_t)g.num_cells_total;
  int rc = clear_counters(ctx, s);
  if (rc != PMPM_OK) return rc;
  if (n == 0) {
    ZeroLists z = extra;
    z.add(ctx->counters, 1);
    z.add(part->cell_start, ncells);
    z.add(part->cell_end, ncells);
    return zero_fill_lists(z, s);
  }
  if (ctx->sort_by_hint && n >= ctx->hint_min_particles && n <= kSmallParticles && ncells <= (uint32_t)kSmallCells) {
    if (n <= 512) return partition_small<1, 512>(ctx, dim, g, x, n, part, s, extra);
    if (n <= 1024) return partition_small<1, 1024>(ctx, dim, g, x, n, part, s, extra);
    return partition_small<2, 1024>(ctx, dim, g, x, n, part, s, extra);
  }
  if (use_hint(ctx, n, ncells)) return partition_by_hint(ctx, dim, g, x, n, part, s, extra);
  // enough threads for the particles, and for the clears at 4 words each
  int64_t words = ncells;
  for (int q = 0; q < extra.count; ++q) words = extra.n[q] > words ? extra.n[q] : words;
  int64_t nb = ceil_div(n, 256);
  const int64_t nb_clear = ceil_div(words, 256 * 4);
  nb = nb_clear > nb ? (nb_clear < 16384 ? nb_clear : (nb > 16384 ? nb : 16384)) : nb;
  const unsigned blocks = (unsigned)nb;
  switch (dim) {
    case 1: PMPM_LAUNCH(hash_kernel<1>, (::pmpm::kname("hash_kernel", {(long)(1)})), dim3(blocks), dim3(256), 0, s, x, n, g, part->hash, part->bins, part->cell_start, part->cell_end, extra); break;
    case 2: PMPM_LAUNCH(hash_kernel<2>, (::pmpm::kname("hash_kernel", {(long)(2)})), dim3(blocks), dim3(256), 0, s, x, n, g, part->hash, part->bins, part->cell_start, part->cell_end, extra); break;
    default: PMPM_LAUNCH(hash_kernel<3>, (::pmpm::kname("hash_kernel", {(long)(3)})), dim3(blocks), dim3(256), 0, s, x, n, g, part->hash, part->bins, part->cell_start, part->cell_end, extra); break;
  }
  PMPM_LAUNCH_CHECK();
  if ((rc = radix_sort_pairs(ctx, part->hash, ctx->keys_tmp, ctx->vals_tmp, part->hash_sorted, part->sorted, n, ncells,
                             s)) != PMPM_OK)
    return rc;
  PMPM_LAUNCH(cell_range_kernel, (::pmpm::kname("cell_range_kernel", {})), dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, s, part->hash_sorted, n, ncells,
                     part->cell_start, part->cell_end, ctx->counters);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

extern "C" int pmpm_partition(pmpm_context *ctx, int32_t dim, const pmpm_grid *grid, const float *x, int32_t n,
                              pmpm_spatial *part, pmpm_stream_t stream) {
  return partition_clearing(ctx, dim, grid, x, n, part, (hipStream_t)stream, ZeroLists{});
}
