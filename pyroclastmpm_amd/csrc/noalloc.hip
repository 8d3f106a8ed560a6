// noalloc.hip -- pmpm_step_noalloc: the whole step without a context and
// without allocating. Its workspace (the radix sort's ping-pong keys, slots and
// digit histograms, the P2G tile partials and flags, the grid pass's clamp
// record, the counters) is carved out of one file-scope device array of
// PMPM_NOALLOC_SCRATCH_BYTES, which each GPU holds for the life of the process.
// Which steps fit is decided by budget_bytes.
// Every call on a GPU uses that GPU's copy: calls that overlap on one GPU race.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>

#include "context.hpp"
#include "device.hpp"

namespace pmpm {
namespace {

static __device__ __align__(256) unsigned char scratch[PMPM_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char *g_scratch[kMaxDevices] = {};

// The device address of this GPU's `scratch` (looked up once per device, with
// the device current; the array's name in host code is not that address).
int scratch_of_current_device(unsigned char **ptr) {
  int dev = 0;
  PMPM_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return PMPM_ERR_INVALID;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    PMPM_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[dev] = static_cast<unsigned char *>(p);
  }
  *ptr = g_scratch[dev];
  return PMPM_OK;
}

// Bump allocator over the scratch bytes, 256-byte aligned pieces.
struct Carver {
  size_t used = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (bytes + 255) / 256 * 256;
    return at;
  }
};

// The workspace a step is charged with: the sort's and the clamp record's own
// sizes, the partials of tiles of 256 cells (1D), 64 x 1 cells (2D; 128 x 1 for
// linear splines) or 16 x 1 x 4 cells (3D; 32 x 1 x 4 for linear splines, 8 x 1
// x 4 where larger, typed cubic) and, typed cubic in 2D and 3D, 64 records of 8
// floats per cell whose window wraps around, a byte per node and 32 lists of
// those cells. These are not the kernels' present arrays: what a caller may ask
// for must not move with their tilings. The present tiles' partials take less
// but on grids of one to five nodes along y or z, where they take up to twice as
// much (a single row of 2D cells; in 3D 1.6 times); those steps go without
// partials once the array is full (p2g_direct_kernel).
size_t budget_bytes(const pmpm_params &prm, const pmpm_grid &g, size_t n, size_t hist_len, size_t clamp_words) {
  Carver c;
  const int dim = prm.dim, span = prm.shape_fn == PMPM_SF_LINEAR ? 2 : 4;
  const bool cubic = prm.shape_fn == PMPM_SF_CUBIC && prm.node_types_built;
  size_t floats = 0, tiles = 0, wrap_floats = 0, touch = 0, list = 0;
  auto tiling = [&](int tx) {
    const size_t t = (size_t)ceil_div(g.num_cells[0], tx) * (dim > 1 ? g.num_cells[1] : 1) *
                     (dim > 2 ? ceil_div(g.num_cells[2], 4) : 1);
    const size_t f = t * (1 + 2 * dim) * (size_t)((tx + span - 1) * (dim > 1 ? span : 1) * (dim > 2 ? 3 + span : 1));
    if (f > floats) floats = f;
    if (t > tiles) tiles = t;
  };
  if (dim == 1) tiling(256);
  else tiling((dim == 2 ? 256 : 64) / span);
  if (dim == 3 && cubic) tiling(8);
  const size_t cells = dim == 3 ? (size_t)wrap_cell_count<3>(g) : (dim == 2 ? (size_t)wrap_cell_count<2>(g) : 0);
  if (cubic && prm.wrap_quirk && cells > 0) {
    wrap_floats = 8 * cells * 64;
    touch = ((size_t)g.num_cells_total + 3) / 4;
    list = 32 * (1 + cells);
  }
  for (const size_t bytes : {n * 4, n * 4, hist_len * 4, (size_t)16, floats * 4, tiles * 4, wrap_floats * 4, touch * 4,
                             list * 4, clamp_words * 4})
    (void)c.take(bytes);
  return c.used;
}

}  // namespace
}  // namespace pmpm

using namespace pmpm;

extern "C" int pmpm_step_noalloc(const pmpm_params *prm, const pmpm_grid *grid, int32_t musl,
                                 const pmpm_particles *a, pmpm_particles *b, pmpm_spatial *part, pmpm_nodes *nodes,
                                 pmpm_stream_t stream) {
  if (!step_args_ok(prm, grid, a, b, part, nodes)) return PMPM_ERR_INVALID;
  const size_t n = (size_t)(a->n > 0 ? a->n : 1);
  const size_t nblocks = (size_t)ceil_div((int64_t)n, kSortTile);
  const size_t hist_len = (size_t)kMaxRadix * nblocks + kMaxRadix;
  const TileSizes w = p2g_workspace(*prm, *grid, (int)a->n);
  Carver c;
  const size_t o_keys = c.take(n * sizeof(uint32_t));
  const size_t o_vals = c.take(n * sizeof(int32_t));
  const size_t o_hist = c.take(hist_len * sizeof(uint32_t));
  const size_t o_counters = c.take(kCounters * sizeof(uint32_t));
  const size_t o_flags = c.take(w.flags * sizeof(int32_t));
  const size_t o_clamp = c.take(w.clamp * sizeof(float));
  const size_t o_partials = c.used;
  const size_t charge = budget_bytes(*prm, *grid, n, hist_len, w.clamp);
  if (charge > (size_t)PMPM_NOALLOC_SCRATCH_BYTES || c.used > (size_t)PMPM_NOALLOC_SCRATCH_BYTES) {
    char why[200];
    snprintf(why, sizeof(why),
             "pmpm_step_noalloc: the step is charged %zu bytes of workspace, PMPM_NOALLOC_SCRATCH_BYTES is %zu "
             "(fewer particles or a smaller grid, or pmpm_step with a context)",
             charge, (size_t)PMPM_NOALLOC_SCRATCH_BYTES);
    note_error(why);
    return PMPM_ERR_WORKSPACE;
  }
  const bool tiled = o_partials + w.partials * sizeof(float) <= (size_t)PMPM_NOALLOC_SCRATCH_BYTES;
  unsigned char *base = nullptr;
  int rc = scratch_of_current_device(&base);
  if (rc != PMPM_OK) return rc;
  // a context over the scratch, which holds whatever an earlier call left; no
  // entry point below grows (allocates) anything
  pmpm_context ctx;
  PMPM_HIP_CHECK(hipGetDevice(&ctx.device));
  ctx.cap_particles = (int32_t)n;
  ctx.cap_cells = grid->num_cells_total;
  ctx.keys_tmp = reinterpret_cast<uint32_t *>(base + o_keys);
  ctx.vals_tmp = reinterpret_cast<int32_t *>(base + o_vals);
  ctx.hist = reinterpret_cast<uint32_t *>(base + o_hist);
  ctx.hist_len = hist_len;
  ctx.counters = reinterpret_cast<uint32_t *>(base + o_counters);
  ctx.counters_clear = true;  // (the radix path writes what it reads)
  ctx.sort_by_hint = false;  // the full radix sort: its workspace is all carved above
  ctx.partials = tiled ? reinterpret_cast<float *>(base + o_partials) : nullptr;
  ctx.tile_flags = reinterpret_cast<int32_t *>(base + o_flags);
  ctx.clamp_mask = reinterpret_cast<float *>(base + o_clamp);
  ctx.tile_cap = w;
  ctx.stray_flags = reinterpret_cast<int32_t *>(ctx.counters + 4);
  ctx.fixed_workspace = true;
  // (the context is a plain struct on this stack frame: nothing frees the
  // scratch pieces it points at)
  return step_on(&ctx, prm, grid, musl, a, b, part, nodes, (hipStream_t)stream);
}
