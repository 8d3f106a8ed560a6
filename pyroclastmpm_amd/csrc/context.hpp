// context.hpp -- private definition of pmpm_context and host-side helpers
// shared by the .hip translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>
#include <string>

#include "../../include/pmpm.h"

namespace pmpm {
// Words of the P2G workspace: tile partials, tile flags, the clamp record (a byte
// per node) and the stray sums.
struct TileSizes {
  size_t partials = 0, flags = 0, clamp = 0, strays = 0;
};
}  // namespace pmpm

struct pmpm_context {
  int device = 0;
  int32_t cap_particles = 0;
  int32_t cap_cells = 0;
  uint32_t *keys_tmp = nullptr;  // radix sort ping-pong keys
  int32_t *vals_tmp = nullptr;   // radix sort ping-pong values
  uint32_t *hist = nullptr;      // [radix][blocks] digit histograms
  size_t hist_len = 0;
  // [kCounters]: out-of-grid particles, hint unsorted flag (set, kept), heavy
  // cells, stray flags (3); counters_clear: cleared since they were allocated
  uint32_t *counters = nullptr;
  bool counters_clear = false;
  // the P2G workspace, one allocation (tile_mem): tile partials (per tile, the
  // node block of each accumulated field; the grid kernel sums the tiles covering
  // a node), tile flags (1 = the tile had particles this launch), and
  // - a byte per node: the components the last grid pass's NodeDomain condition
  //   set to zero, read by the adjoint
  // - the sums of particles deposited over their own windows (mass, momentum,
  //   force per node; the adjoint scatter's fields), zero but between a pass that
  //   sets its flag (stray_flags: P2G, re-map, adjoint scatter) and the grid pass
  //   after it (strays_clear: cleared since they were allocated)
  float *tile_mem = nullptr;
  pmpm::TileSizes tile_cap;
  float *partials = nullptr;
  int32_t *tile_flags = nullptr;
  float *clamp_mask = nullptr;
  float *strays = nullptr;
  bool strays_clear = false;
  int32_t *stray_flags = nullptr;  // in counters
  // the workspace is the caller's and never grows (pmpm_step_noalloc): the
  // stray sums are then the step's node arrays, cleared before it, and without
  // room for the partials every particle is deposited over its own window
  bool fixed_workspace = false;
  // adjoint step: per-particle scatter records (15 floats, cell order) and
  // node adjoints (one record of 8 floats per node, 4 in 1D)
  float *adj_rec = nullptr;
  size_t adj_rec_cap = 0;
  float *adj_nodes = nullptr;
  size_t adj_nodes_cap = 0;
  // per-workgroup partial sums of the material parameter adjoints
  float *adj_pb = nullptr;
  size_t adj_pb_cap = 0;
  // partition from a sorted hint (the previous call's sorted keys): false
  // always runs the full radix sort (PMPM_PARTITION_RADIX=1 at creation);
  // below hint_min_particles particles the radix sort runs too
  // (PMPM_PARTITION_HINT_MIN at creation)
  bool sort_by_hint = true;
  int32_t hint_min_particles = 0;
  // its workspace, one allocation. Per cell (the last for the out-of-grid
  // particles): counts of stayers and movers, and per block of 1024 cells (both
  // zero between calls; hint_clear: cleared since they were allocated), the
  // blocks' sums, and per cell the first slot, stayers before the cell, stayers,
  // movers; then the arrays per particle (HintLayout in partition.hip)
  uint32_t *hint_mem = nullptr;
  uint32_t *hint_cnt = nullptr, *hint_cbt = nullptr, *hint_sums = nullptr, *hint_info = nullptr, *hint_part = nullptr;
  size_t hint_zero_words = 0, hint_part_cap = 0, hint_cells_cap = 0;
  bool hint_clear = false;
};

namespace pmpm {
// Grows the P2G workspace (hipMalloc on first use of a larger grid; run one step
// before capturing a graph).
int ensure_tiles(pmpm_context *ctx, const TileSizes &want);
// Grows a context-owned float buffer to at least `floats`.
int ensure_buffer(float *&buf, size_t &cap, size_t floats);
}  // namespace pmpm

namespace pmpm {

constexpr int kCounters = 8;  // words of pmpm_context::counters
constexpr int kSortBlock = 1024;  // 16 waves rank 1024 keys per round
constexpr int kSortItems = 4;
constexpr int kSortTile = kSortBlock * kSortItems;
constexpr int kMaxRadixBits = 10;  // digits of 8 bits (keys < 2^8) or 10 bits
constexpr int kMaxRadix = 1 << kMaxRadixBits;

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// A grid the kernels can address: at least one node, fewer than
// PMPM_MAX_GRID_NODES (32-bit byte offsets into the node records).
inline bool grid_ok(const pmpm_grid *g) {
  return g && g->num_cells_total > 0 && g->num_cells_total < PMPM_MAX_GRID_NODES;
}

// Records the failing HIP call of the calling thread (pmpm_last_error).
void note_hip_error(hipError_t e, const char *what);
// Records a non-HIP failure of the calling thread (pmpm_last_error).
void note_error(const char *what);
inline bool hip_ok(hipError_t e, const char *what) {
  if (e == hipSuccess) return true;
  note_hip_error(e, what);
  return false;
}

#define PMPM_HIP_CHECK(expr)                              \
  do {                                                    \
    hipError_t e_ = (expr);                               \
    if (e_ != hipSuccess) {                               \
      ::pmpm::note_hip_error(e_, #expr);                  \
      return PMPM_ERR_HIP;                                \
    }                                                     \
  } while (0)

#define PMPM_LAUNCH_CHECK()                               \
  do {                                                    \
    hipError_t e_ = hipGetLastError();                    \
    if (e_ != hipSuccess) {                               \
      ::pmpm::note_hip_error(e_, "kernel launch");        \
      return PMPM_ERR_HIP;                                \
    }                                                     \
  } while (0)

// Kernel timing (pmpm_timing_enable): a TimedRegion around a launch records
// a HIP event pair on the launch stream when the calling thread has timing on;
// the name is only formed then.
bool timing_enabled();
std::string kname(const char *base, std::initializer_list<long> targs);
class TimedRegion {
 public:
  template <class F> TimedRegion(hipStream_t s, F &&name) {
    if (timing_enabled()) start(s, name());
  }
  ~TimedRegion() {
    if (on_) finish();
  }
  TimedRegion(const TimedRegion &) = delete;
  TimedRegion &operator=(const TimedRegion &) = delete;

 private:
  void start(hipStream_t s, std::string name);
  void finish();
  bool on_ = false;
  hipStream_t s_ = nullptr;
  hipEvent_t a_ = nullptr, b_ = nullptr;
  std::string name_;
};
// hipLaunchKernelGGL with the launch timed under `name` (an expression giving
// a std::string, in parentheses) when timing is on.
#define PMPM_LAUNCH(kernel, name, grid, block, shm, stream, ...)                 \
  do {                                                                           \
    ::pmpm::TimedRegion pmpm_timed_((stream), [&]() { return std::string name; }); \
    hipLaunchKernelGGL(kernel, grid, block, shm, stream, __VA_ARGS__);           \
  } while (0)

// Fill n floats/ints with zero (a kernel, not hipMemsetAsync, so the step can
// be captured in a HIP graph).
int zero_fill(void *ptr, int64_t n_words, hipStream_t s);
constexpr int kZeroLists = 8;  // (four of a step, three of an empty partition)
struct ZeroLists {  // buffers of 32-bit words to clear in one launch
  uint32_t *p[kZeroLists];
  int64_t n[kZeroLists];
  int count;
  void add(void *ptr, int64_t words) {
    if (ptr && words > 0 && count < kZeroLists) { p[count] = (uint32_t *)ptr; n[count] = words; ++count; }
  }
};
int zero_fill_lists(const ZeroLists &z, hipStream_t s);
// Clears buffers that must be zero between a context's calls, once (`clear`),
// on the stream of the call that uses them first. A clear that is only being
// recorded into a graph does not count: the graph may not have been replayed
// when the next call comes.
int clear_on_stream(const ZeroLists &z, bool &clear, hipStream_t s);
// One step on the workspace of ctx (arguments already checked by
// step_args_ok); the body of pmpm_step.
int step_on(pmpm_context *ctx, const pmpm_params *prm, const pmpm_grid *grid, int32_t musl,
            const pmpm_particles *a, pmpm_particles *b, pmpm_spatial *part, pmpm_nodes *nodes, hipStream_t s);
// Dimension, shape function, list sizes, and the node arrays of body forces.
bool params_ok(const pmpm_params *prm);
bool step_args_ok(const pmpm_params *prm, const pmpm_grid *grid, const pmpm_particles *a, const pmpm_particles *b,
                  const pmpm_spatial *part, const pmpm_nodes *nodes);
// The P2G workspace of a step of n particles on grid g (without stray sums).
TileSizes p2g_workspace(const pmpm_params &prm, const pmpm_grid &g, int n);
// pmpm_partition whose first kernel also clears the buffers of `extra`.
int partition_clearing(pmpm_context *ctx, int dim, const pmpm_grid *grid, const float *x, int n, pmpm_spatial *part,
                       hipStream_t s, const ZeroLists &extra);

}  // namespace pmpm
