// transfer.hip -- particle/grid transfers on gfx950.
//
//   p2g_mfma_kernel   (3D) one workgroup per tile of cells, one wave per row of
//                     cells: the particles' outer products of weights and
//                     fields summed by matrix instructions into the tile's
//                     nodes, stored as a per-tile slice. Modes: P2G, MUSL
//                     re-map, adjoint scatter.
//   p2g_rows_kernel   (1D, 2D) the same passes with a lane per (cell, y node
//                     offset) that sums its nodes in registers.
//   grid_kernel       per node: sums the tile slices covering it, mass cutoff,
//                     mom_nt = mom + f dt, boundary conditions in list order,
//                     node velocities for G2P.
//   g2p_kernel        per particle (cell order): gather from the grid,
//                     FLIP/PIC update, F and volume, then the return map of the
//                     particle's material, written in cell order. MODE 1 is the
//                     MUSL first map, MODE 2 the second.
// Weights are recomputed in registers from the positions; nothing per
// particle x node is stored.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "adjoint_math.hpp"
#include "context.hpp"
#include "device.hpp"

namespace pmpm {

// Tiles whose node block covers one node, at most, per axis (y: tiles of one
// cell in small 3D scenes).
constexpr int kCoverX = 2, kCoverY = 4, kCoverZ = 2;

__device__ inline int64_t lin_index(const pmpm_grid &g, const int *b, int D) {
  int64_t h = b[0];
  if (D > 1) h += (int64_t)b[1] * g.num_cells[0];
  if (D > 2) h += (int64_t)b[2] * g.num_cells[0] * g.num_cells[1];
  return h;
}

// Per-particle weight tables for the ENTRIES nodes per axis.
template <int D, int SF> struct PW {
  static constexpr int E = Spline<SF>::ENTRIES;
  float t[3];
  int bin[3];
  int first[3];
  float N[3][4];
  float dN[3][4];
};

template <int D, int SF>
__device__ inline void particle_weights(const pmpm_params &prm, const pmpm_grid &g, const float *x, int n, int slot,
                                        PW<D, SF> &w, float *xp) {
  // all coordinates in flight before the first weight
#pragma unroll
  for (int a = 0; a < 3; ++a) xp[a] = a < D ? x[a * n + slot] : 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (a < D) {
      w.t[a] = cell_coord(xp[a], g.origin[a], g.inv_cell_size);
      w.bin[a] = (int)w.t[a];
      axis_weights<SF>(w.t[a], w.bin[a], g.num_cells[a], prm.node_types_built, g.inv_cell_size, w.first[a], w.N[a],
                       w.dN[a]);
    } else {
      w.t[a] = 0.f; w.bin[a] = 0; w.first[a] = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) { w.N[a][e] = 1.f; w.dN[a][e] = 0.f; }
    }
  }
}

// Node velocity records (pmpm_nodes.vel): NP floats per node, v_nt then dv,
// so a gather entry is one 16-byte load (two for v_nt and dv in 3D) instead
// of one load per component.
template <int D> struct NodeVel {
  static constexpr int NP = D == 3 ? 8 : 2 * D;
};
// The byte offset of a record is a 32-bit value (grids hold fewer than
// PMPM_MAX_GRID_NODES nodes), so a load is the uniform base plus one VGPR.
template <int D, bool WANT_DV>
__device__ inline void load_node_vel(const float *__restrict__ vel, int node, float *v, float *dv) {
  const char *base = reinterpret_cast<const char *>(vel);
  const uint32_t at = (uint32_t)node * (uint32_t)(NodeVel<D>::NP * sizeof(float));
  if constexpr (D == 3) {
    const float4 a = *reinterpret_cast<const float4 *>(base + at);
    v[0] = a.x; v[1] = a.y; v[2] = a.z;
    if constexpr (WANT_DV) {
      const float4 b = *reinterpret_cast<const float4 *>(base + at + 16u);
      dv[0] = a.w; dv[1] = b.x; dv[2] = b.y;
    }
  } else if constexpr (D == 2) {
    const float4 a = *reinterpret_cast<const float4 *>(base + at);
    v[0] = a.x; v[1] = a.y;
    if constexpr (WANT_DV) { dv[0] = a.z; dv[1] = a.w; }
  } else {
    const float2 a = *reinterpret_cast<const float2 *>(base + at);
    v[0] = a.x;
    if constexpr (WANT_DV) dv[0] = a.y;
  }
}
template <int D> __device__ inline void store_node_vel(float *__restrict__ vel, int node, const float *v, const float *dv) {
  if constexpr (D == 3) {
    float4 *p = reinterpret_cast<float4 *>(vel + 8 * (int64_t)node);
    p[0] = make_float4(v[0], v[1], v[2], dv[0]);
    p[1] = make_float4(dv[1], dv[2], 0.f, 0.f);
  } else if constexpr (D == 2) {
    *reinterpret_cast<float4 *>(vel + 4 * (int64_t)node) = make_float4(v[0], v[1], dv[0], dv[1]);
  } else {
    *reinterpret_cast<float2 *>(vel + 2 * (int64_t)node) = make_float2(v[0], dv[0]);
  }
}
// Where a gather reads node velocities from: the global records
// (pmpm_nodes.vel) with the grid's node strides (node (i, j, k) at
// sum id_a stride_a), or a run's node rows staged in LDS (box4 = v_nt and
// dv.x, box2 = dv.y and dv.z per node): window entry (x, sy, sz) of a
// particle at x bin b sits at (b - 1 + x - lo[0]) + sy stride[1] + sz stride[2]
// with sy, sz = 0..3 the entry's node offset + 1 along y and z.
struct NodeSrc {
  const float *vel;
  const float4 *box4;
  const float2 *box2;
  int stride[3];
  int lo[3];
};
__device__ inline NodeSrc node_src(const pmpm_grid &g, const pmpm_nodes &nodes) {
  return NodeSrc{nodes.vel, nullptr, nullptr, {1, g.num_cells[0], g.num_cells[0] * g.num_cells[1]}, {0, 0, 0}};
}
template <int D, bool WANT_DV, bool BOX>
__device__ inline void load_src(const NodeSrc &src, int node, float *v, float *dv) {
  if constexpr (BOX) {
    const float4 a = src.box4[node];
    v[0] = a.x; v[1] = a.y; v[2] = a.z;
    if constexpr (WANT_DV) {
      const float2 b = src.box2[node];
      dv[0] = a.w; dv[1] = b.x; dv[2] = b.y;
    }
  } else {
    load_node_vel<D, WANT_DV>(src.vel, node, v, dv);
  }
}

// Grid gather (1D/2D in the reference's window order, y outer, x inner; 3D in
// the separable order below). The reference skips entries outside the grid
// on any axis (usl_inline.h:281-293); here such entries get zero weights and
// a clamped, valid node index, which leaves every sum unchanged and keeps the
// loop free of branches. Nodes below the mass cutoff carry zero velocities,
// which is equivalent to skipping them.
template <int D, int SF, bool WANT_V, bool WANT_L, bool BOX = false>
__device__ inline void gather_grid(const pmpm_grid &g, const NodeSrc &src, const PW<D, SF> &w, float *vinc,
                                   float *dvinc, float *L) {
  static_assert(!BOX || D == 3, "LDS node boxes are 3D");
  constexpr int E = Spline<SF>::ENTRIES;
  constexpr int EY = D > 1 ? E : 1;
  constexpr int EZ = D > 2 ? E : 1;
  float N[3][4], dN[3][4];
  int off[3][4];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int stride = src.stride[a];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (a < D && e < E) {
        const int i = w.bin[a] + w.first[a] + e;
        const bool ok = i >= 0 && i < g.num_cells[a];
        if (BOX) off[a][e] = (a == 0 ? i - src.lo[0] : w.first[a] + 1 + e) * stride;
        else off[a][e] = min(max(i, 0), g.num_cells[a] - 1) * stride;
        N[a][e] = ok ? w.N[a][e] : 0.f;
        dN[a][e] = ok ? w.dN[a][e] : 0.f;
      } else {
        off[a][e] = 0;
        N[a][e] = 1.f;
        dN[a][e] = 0.f;
      }
    }
  }
  if constexpr (D == 3) {
    // Separable form: the weights are products of per-axis factors, so the
    // sums contract x first (a row's x nodes are adjacent records), then y,
    // then z: per row S = sum_x Nx v, Sd = sum_x dNx v; per z layer
    // U0 = sum_y Ny Sd, U1 = sum_y dNy S, U2 = sum_y Ny S; then
    // L[x][.] += Nz U0, L[y][.] += Nz U1, L[z][.] += dNz U2, v += Nz U2.
    // The next row's records are loaded while the current row is summed.
    constexpr int NR = EY * EZ;
    float rv[2][E][3], rd[2][E][3];
    auto load_row = [&](int r, int buf) {
      const int row = off[1][r % EY] + off[2][r / EY];
#pragma unroll
      for (int ex = 0; ex < E; ++ex) load_src<D, WANT_V, BOX>(src, row + off[0][ex], rv[buf][ex], rd[buf][ex]);
    };
    load_row(0, 0);
    float U0[3] = {0.f, 0.f, 0.f}, U1[3] = {0.f, 0.f, 0.f}, U2[3] = {0.f, 0.f, 0.f}, Ud[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int ey = r % EY, ez = r / EY, cb = r & 1;
      if (r + 1 < NR) load_row(r + 1, cb ^ 1);
      float Sx[3] = {0.f, 0.f, 0.f}, Sdx[3] = {0.f, 0.f, 0.f}, Sxd[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int ex = 0; ex < E; ++ex)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          Sx[b] += N[0][ex] * rv[cb][ex][b];
          if (WANT_L) Sdx[b] += dN[0][ex] * rv[cb][ex][b];
          if (WANT_V) Sxd[b] += N[0][ex] * rd[cb][ex][b];
        }
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        U2[b] += N[1][ey] * Sx[b];
        if (WANT_L) {
          U0[b] += N[1][ey] * Sdx[b];
          U1[b] += dN[1][ey] * Sx[b];
        }
        if (WANT_V) Ud[b] += N[1][ey] * Sxd[b];
      }
      if (ey == EY - 1) {  // z layer complete
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          if (WANT_L) {
            L[b] += N[2][ez] * U0[b];
            L[3 + b] += N[2][ez] * U1[b];
            L[6 + b] += dN[2][ez] * U2[b];
          }
          if (WANT_V) {
            vinc[b] += N[2][ez] * U2[b];
            dvinc[b] += N[2][ez] * Ud[b];
          }
          U0[b] = U1[b] = U2[b] = Ud[b] = 0.f;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int ey = 0; ey < EY; ++ey) {
#pragma unroll
    for (int ex = 0; ex < E; ++ex) {
      const float nxy = N[0][ex] * N[1][ey];
      const float dxy = dN[0][ex] * N[1][ey];
      const float dyx = dN[1][ey] * N[0][ex];
#pragma unroll
      for (int ez = 0; ez < EZ; ++ez) {
        const int node = off[0][ex] + off[1][ey] + off[2][ez];
        const float wgt = nxy * N[2][ez];
        float gr[3];
        gr[0] = dxy * N[2][ez];
        gr[1] = dyx * N[2][ez];
        gr[2] = (dN[2][ez] * N[0][ex]) * N[1][ey];
        float vnt[3], dv[3];
        load_node_vel<D, WANT_V>(src.vel, node, vnt, dv);
        if (WANT_V) {
#pragma unroll
          for (int a = 0; a < D; ++a) {
            dvinc[a] += wgt * dv[a];
            vinc[a] += wgt * vnt[a];
          }
        }
        if (WANT_L) {
#pragma unroll
          for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) L[3 * a + b] += gr[a] * vnt[b];
        }
      }
    }
  }
}

// Weight and gradient of one window entry with explicit node types (used when
// the node is reached through the linear-index wrap, and for materialised psi).
template <int D, int SF>
__device__ inline void entry_weight(const PW<D, SF> &w, const int *off, const int *types, float inv_h, float &wgt,
                                    float *gr) {
  float N[3] = {1.f, 1.f, 1.f}, dN[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const float frac = __fsub_rn(w.t[a], (float)w.bin[a]);
    spline_eval<SF>(__fsub_rn(frac, (float)off[a]), types[a], inv_h, N[a], dN[a]);
  }
  wgt = (N[0] * N[1]) * N[2];
  gr[0] = (dN[0] * N[1]) * N[2];
  gr[1] = (dN[1] * N[0]) * N[2];
  gr[2] = (dN[2] * N[0]) * N[1];
}

template <int D>
__device__ inline void node_ids(const pmpm_grid &g, int64_t lin, int *ids) {
  ids[0] = (int)(lin % g.num_cells[0]);
  ids[1] = (D > 1) ? (int)((lin / g.num_cells[0]) % g.num_cells[1]) : 0;
  ids[2] = (D > 2) ? (int)(lin / ((int64_t)g.num_cells[0] * g.num_cells[1])) : 0;
}

// node_ids in 32 bits (grids hold fewer than PMPM_MAX_GRID_NODES nodes).
template <int D> __device__ inline void node_ids32(const pmpm_grid &g, int lin, int *ids) {
  const uint32_t nx = (uint32_t)g.num_cells[0], row = (uint32_t)lin / nx;
  ids[0] = (int)((uint32_t)lin - row * nx);
  if (D > 1) {
    const uint32_t ny = (uint32_t)g.num_cells[1], layer = D > 2 ? row / ny : 0u;
    ids[1] = (int)(row - layer * ny);
    ids[2] = D > 2 ? (int)layer : 0;
  } else {
    ids[1] = ids[2] = 0;
  }
}

// Slow path of the scatter: every entry goes straight to global memory,
// through the linear index (wrap-around reproduced when wrap_quirk is set).
// Used for the particles that are not in the cell they are listed in (see
// p2g_stray).
// Strays: their sums, in node arrays of their own that are zero between the
// passes, and a flag the pass sets when it added something. The grid pass reads
// (and clears) them only then, so the node arrays are neither cleared before a
// step nor read by its first grid pass.
struct Strays {
  float *mass, *mom, *mom_nt;
  int32_t *flag;
};
template <int D, int SF, int MODE>
__device__ inline void scatter_entry_global(const pmpm_params &prm, const pmpm_grid &g, const Strays &nodes,
                                            int nn, const PW<D, SF> &w, const int *e, float m, const float *mv,
                                            const float A[3][3], const float *fext) {
  int nb[3] = {0, 0, 0}, off[3] = {0, 0, 0};
  bool inside = true;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    off[a] = w.first[a] + e[a];
    nb[a] = w.bin[a] + off[a];
    if (nb[a] < 0 || nb[a] >= g.num_cells[a]) inside = false;
  }
  const int64_t lin = lin_index(g, nb, D);
  if (lin < 0 || lin >= g.num_cells_total) return;
  if (!inside && !prm.wrap_quirk) return;
  int ids[3];
  node_ids<D>(g, lin, ids);
  int types[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) types[a] = cubic_node_type(ids[a], g.num_cells[a], prm.node_types_built);
  float wgt, gr[3];
  entry_weight<D, SF>(w, off, types, g.inv_cell_size, wgt, gr);
  const int node = (int)lin;
  if (MODE == 0) {
    if (wgt != 0.f) unsafeAtomicAdd(&nodes.mass[node], wgt * m);
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float pm = wgt * mv[a];
      if (pm != 0.f) unsafeAtomicAdd(&nodes.mom[a * nn + node], pm);
      float f = wgt * fext[a];
#pragma unroll
      for (int b = 0; b < D; ++b) f += A[a][b] * gr[b];
      if (f != 0.f) unsafeAtomicAdd(&nodes.mom_nt[a * nn + node], f);
    }
  } else {
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float pm = wgt * mv[a];
      if (pm != 0.f) unsafeAtomicAdd(&nodes.mom_nt[a * nn + node], pm);
    }
  }
}

// P2G of a particle that is not in the cell it is listed in: one left of the
// origin (its coordinate truncates to cell 0, its fraction is negative), or any
// other where the partition was built from other positions. This lane's y slice
// of its window goes straight to the stray sums.
template <int D, int SF, int MODE>
__device__ void p2g_stray(const pmpm_params &prm, const pmpm_grid &g, const Strays &nodes, const float *x, int n,
                          int slot, int sy, float m, const float *v, const Sym &A, const float *fext) {
  constexpr int E = Spline<SF>::ENTRIES;
  constexpr int EZ = D > 2 ? E : 1;
  if (sy >= (D > 1 ? E : 1)) return;
  PW<D, SF> w;
  float xp[3];
  particle_weights<D, SF>(prm, g, x, n, slot, w, xp);
  float mv[3] = {0.f, 0.f, 0.f}, A3[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (a < D) mv[a] = m * v[a];
#pragma unroll
    for (int b = 0; b < 3; ++b) A3[a][b] = (a < D && b < D) ? sym_at(A, a, b) : 0.f;
  }
#pragma unroll 1
  for (int ex = 0; ex < E; ++ex)
#pragma unroll 1
    for (int ez = 0; ez < EZ; ++ez) {
      const int e3[3] = {ex, sy, ez};
      scatter_entry_global<D, SF, MODE>(prm, g, nodes, g.num_cells_total, w, e3, m, mv, A3, fext);
    }
}

// The same for the adjoint scatter (MODE 2): the records' adjoints (v_pic: vpb,
// dv: dvb, L: row a from Lb + LROW a) over the entries the G2P gathered, those
// inside the grid, into the first 2 D stray arrays.
template <int D, int SF, int LROW>
__device__ void adjoint_stray(const pmpm_params &prm, const pmpm_grid &g, const Strays &nodes, const float *x, int n,
                              int slot, const float *vpb, const float *dvb, const float *Lb) {
  constexpr int E = Spline<SF>::ENTRIES, EY = D > 1 ? E : 1, EZ = D > 2 ? E : 1;
  PW<D, SF> w;
  float xp[3];
  particle_weights<D, SF>(prm, g, x, n, slot, w, xp);
#pragma unroll 1
  for (int e = 0; e < E * EY * EZ; ++e) {
    const int e3[3] = {e % E, (e / E) % EY, e / (E * EY)};
    float N[3] = {1.f, 1.f, 1.f}, dN[3] = {0.f, 0.f, 0.f};
    int id[3] = {0, 0, 0};
    bool inside = true;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      id[a] = w.bin[a] + w.first[a] + e3[a];
      inside = inside && id[a] >= 0 && id[a] < g.num_cells[a];
#pragma unroll
      for (int k = 0; k < E; ++k) {  // (picked by compares: no indexed registers)
        N[a] = e3[a] == k ? w.N[a][k] : N[a];
        dN[a] = e3[a] == k ? w.dN[a][k] : dN[a];
      }
    }
    if (!inside) continue;
    const int node = (int)lin_index(g, id, D), nn = g.num_cells_total;
    const float wgt = (N[0] * N[1]) * N[2];
    const float gr[3] = {(dN[0] * N[1]) * N[2], (dN[1] * N[0]) * N[2], (dN[2] * N[0]) * N[1]};
#pragma unroll
    for (int a = 0; a < D; ++a) {
      float v = wgt * vpb[a];
#pragma unroll
      for (int c = 0; c < D; ++c) v += gr[c] * Lb[LROW * c + a];
      unsafeAtomicAdd(&nodes.mass[(int64_t)a * nn + node], v);
      unsafeAtomicAdd(&nodes.mass[(int64_t)(D + a) * nn + node], wgt * dvb[a]);
    }
  }
}

// Fields per node of a P2G pass: MODE 0 mass, momentum, force; MODE 1 the
// re-mapped momentum; MODE 2 the adjoints of v_nt and dv.
template <int D, int MODE> constexpr int p2g_nv() { return MODE == 0 ? 1 + 2 * D : (MODE == 2 ? 2 * D : D); }

__device__ inline int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
  return v;
}

// Element i of a uniform base pointer through a 32-bit byte offset: the load
// takes its base from scalar registers and one offset register serves every
// array (a set of 2^30 particles would not fit the card, so 4 i stays below
// 2^32).
__device__ inline float ld32(const float *base, uint32_t i) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + 4u * i);
}

// Per-axis weights of one fixed span offset as polynomials of the fraction
// f = t - bin, for lanes that own one offset per axis: the coefficients are
// set once per cell (or wave) and a weight costs a few multiply-adds.
//
// Cubic: N = a0 + a1 f + a2 f^2 + a3 f^3 of node type 0-3 at span offset s
// (the piece 3 - s of the boundary-modified spline, cubic.cuh:28-197, in
// powers of f instead of r = f + 1 - s: smaller coefficients, so less
// cancellation near the spline's end than the r form).
__device__ __constant__ static const float kSpanCubic[4][4][4] = {
    {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}},
    {{1.f / 6.f, -0.5f, 0.5f, -1.f / 6.f}, {1.f, -1.f, 0.f, 1.f / 6.f}, {1.f / 6.f, 0.5f, 0.5f, -1.f / 6.f}, {0.f, 0.f, 0.f, 1.f / 6.f}},
    {{1.f / 6.f, -0.5f, 0.5f, -1.f / 6.f}, {2.f / 3.f, 0.f, -1.f, 0.5f}, {0.f, 1.f, 0.f, -1.f / 3.f}, {0.f, 0.f, 0.f, 0.f}},
    {{1.f / 6.f, -0.5f, 0.5f, -1.f / 6.f}, {2.f / 3.f, 0.f, -1.f, 0.5f}, {1.f / 6.f, 0.5f, 0.5f, -0.5f}, {0.f, 0.f, 0.f, 1.f / 6.f}}};

template <int SF> struct SpanPoly;
template <> struct SpanPoly<PMPM_SF_CUBIC> {
  float a0, a1, a2, a3, d1, d2, d3;
  // offset s, type of the node there; keep = 0 drops the offset. table:
  // kSpanCubic in LDS (a load from memory here would be a round trip per cell)
  __device__ inline void set(const float *table, int s, int type, float inv_h, float keep) {
    const float4 c = *reinterpret_cast<const float4 *>(table + 4 * (4 * type + s));
    a0 = keep * c.x; a1 = keep * c.y; a2 = keep * c.z; a3 = keep * c.w;
    d1 = inv_h * a1; d2 = inv_h * (2.f * a2); d3 = inv_h * (3.f * a3);
  }
  __device__ inline float N(float f) const { return ((a3 * f + a2) * f + a1) * f + a0; }
  __device__ inline float dN(float f) const { return (d3 * f + d2) * f + d1; }
};
// Quadratic: N = c0 + c1 b^2, dN = d1 b with b = f - e; one set for f < 1/2,
// one above. Offset s is 0 where the particle's window does not reach it.
template <> struct SpanPoly<PMPM_SF_QUADRATIC> {
  float e[2], c0[2], c1[2], d1[2];
  __device__ inline void set(const float *, int s, int, float inv_h, float keep) {
    // f < 1/2: 0.5 (f - 0.5)^2, 0.75 - f^2, 0.5 (f + 0.5)^2, 0
    // else:    0, 0.5 (f - 1.5)^2, 0.75 - (f - 1)^2, 0.5 (f - 0.5)^2
    e[0] = s == 0 ? 0.5f : (s == 2 ? -0.5f : 0.f);
    e[1] = s == 1 ? 1.5f : (s == 2 ? 1.f : 0.5f);
    const float lo = s == 3 ? 0.f : (s == 1 ? -1.f : 0.5f), hi = s == 0 ? 0.f : (s == 2 ? -1.f : 0.5f);
    c0[0] = keep * (s == 1 ? 0.75f : 0.f);
    c0[1] = keep * (s == 2 ? 0.75f : 0.f);
    c1[0] = keep * lo;
    c1[1] = keep * hi;
#pragma unroll
    for (int k = 0; k < 2; ++k) d1[k] = inv_h * (2.f * c1[k]);
  }
  __device__ inline float N(float f) const {
    const bool h = f >= 0.5f;
    const float b = f - (h ? e[1] : e[0]);
    return (h ? c1[1] : c1[0]) * (b * b) + (h ? c0[1] : c0[0]);
  }
  __device__ inline float dN(float f) const {
    const bool h = f >= 0.5f;
    return (h ? d1[1] : d1[0]) * (f - (h ? e[1] : e[0]));
  }
};
// Linear: N = c0 + c1 f; the derivative is 0 on a node (linear_eval).
template <> struct SpanPoly<PMPM_SF_LINEAR> {
  float c0, c1, d, d_at0;
  __device__ inline void set(const float *, int s, int, float inv_h, float keep) {
    const float k = s > 1 ? 0.f : keep;
    c0 = s == 0 ? k : 0.f;
    c1 = s == 0 ? -k : k;
    d = inv_h * c1;
    d_at0 = s == 0 ? 0.f : d;
  }
  __device__ inline float N(float f) const { return c1 * f + c0; }
  __device__ inline float dN(float f) const { return f == 0.f ? d_at0 : d; }
};

// All weights of an interior particle along one axis (cubic: nodes of type 3),
// and their derivatives times the cell size: SpanPoly with constant offsets.
template <int SF> __device__ inline void inner_weights(float f, float *N, float *dN) {
  if constexpr (SF == PMPM_SF_CUBIC) {
    N[0] = ((-1.f / 6.f * f + 0.5f) * f - 0.5f) * f + 1.f / 6.f;
    N[1] = (0.5f * f - 1.f) * f * f + 2.f / 3.f;
    N[2] = ((-0.5f * f + 0.5f) * f + 0.5f) * f + 1.f / 6.f;
    N[3] = 1.f / 6.f * f * f * f;
    dN[0] = (-0.5f * f + 1.f) * f - 0.5f;
    dN[1] = (1.5f * f - 2.f) * f;
    dN[2] = (-1.5f * f + 1.f) * f + 0.5f;
    dN[3] = 0.5f * f * f;
  } else {
#pragma unroll
    for (int s = 0; s < Spline<SF>::SPAN; ++s) {
      SpanPoly<SF> p;
      p.set(nullptr, s, 0, 1.f, 1.f);
      N[s] = p.N(f);
      dN[s] = p.dN(f);
    }
  }
}

// The P2G tiles of 1D and 2D scenes: CELLS x ROWS cells, one wave per row of
// CELLS cells along x, lane = (y node offset, cell).
template <int D, int SF> struct RowGeom {
  static constexpr int SPAN = Spline<SF>::SPAN, NLO = Spline<SF>::NLO;
  static constexpr int SY = D > 1 ? SPAN : 1, CELLS = 64 / SY, ROWS = D > 1 ? 4 : 1, THREADS = 64 * ROWS;
  static constexpr int NX = CELLS + SPAN - 1, NY = ROWS + SY - 1, NTN = NX * NY;  // nodes of one partial slice
};

// P2G of one tile of a 1D or 2D scene. Modes as p2g_mfma_kernel.
//
// What bounds it: latency, not bandwidth or issue. A cell's particles are a
// serial chain for its lanes (16 per cell at 4 x 4: about 70 vector
// instructions each), so the chain must read LDS only: a round stages the next
// KW particles of every cell of the row, two particles per lane, while the
// fields of the round after and the slots of the one after that are in flight.
// A lane evaluates the weights of its SPAN x node offsets and of its own y
// offset, and sums its SPAN nodes in registers; a node column's sums are
// added over the cells in LDS, phase by phase of x offset (distinct nodes
// within a phase), and over the rows when the slice is stored. Tiles of 16 x 4
// cells store 2.1 nodes per cell and a node lies in at most four of them
// (64 x 1 cells: 4.2 and eight). 398,000 particles, cubic, 402,000 nodes: P2G
// 21 us, re-map 14 us (60, and 58 with the first map fused, when each lane
// loaded its particles itself); 21,420 particles, quadratic: 8 and 7 us.
//
// Linear-index wrap-around as in p2g_mfma_kernel: a node offset outside the
// grid is a virtual node of the tile with the spline types of the node its
// linear index reaches, which the grid kernel adds. A carry out of x shifts y
// by one, so in a row that touches an x face each x offset has y weights of
// its own.
template <int D, int SF, int MODE, bool FEXT = false>
__global__ __launch_bounds__((RowGeom<D, SF>::THREADS)) void p2g_rows_kernel(
    pmpm_params prm, pmpm_grid g, pmpm_particles in, pmpm_particles out, pmpm_spatial part, Strays nodes,
    int tiles_x, float *__restrict__ partials, int32_t *__restrict__ flags, const float *__restrict__ rec) {
  using G = RowGeom<D, SF>;
  static_assert(D == 1 || D == 2, "3D passes are p2g_mfma_kernel's");
  static_assert(MODE == 0 || !FEXT, "only the P2G carries the wall force");
  constexpr int SPAN = G::SPAN, NLO = G::NLO, SY = G::SY, CELLS = G::CELLS, ROWS = G::ROWS, NX = G::NX;
  constexpr int NV = p2g_nv<D, MODE>();
  constexpr bool TYPED = SF == PMPM_SF_CUBIC;
  // a staged record: fractions, then MODE 0: m, m v, A = -V sigma (xx; yy, xy),
  // wall force; MODE 1: m v'; MODE 2: adjoints of v_pic, dv and L's columns
  constexpr int NF = MODE == 0 ? 2 * D + 1 + D * (D + 1) / 2 + (FEXT ? D : 0) : (MODE == 1 ? 2 * D : 3 * D + D * D);
  constexpr int RS = (NF + 3) / 4 * 4;
  constexpr int KW = 128 / CELLS;    // particles of a cell per round
  constexpr int CP = KW * RS + 4;    // LDS words of a cell: the 16-byte reads of 16 cells fall into distinct banks
  constexpr int WS = CELLS * CP > NV * SY * NX ? CELLS * CP : NV * SY * NX;
  __shared__ __attribute__((aligned(16))) float smem[ROWS][WS];
  __shared__ __attribute__((aligned(16))) float s_poly[TYPED ? 64 : 4];  // kSpanCubic

  const int n = in.n;
  const float inv_h = g.inv_cell_size;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lx = lane % CELLS, sy = lane / CELLS;
  const int cx0 = ((int)blockIdx.x % tiles_x) * CELLS, cy = D > 1 ? ((int)blockIdx.x / tiles_x) * ROWS + wave : 0;
  const int cx = cx0 + lx;
  int cs = 0, ce = 0;
  if (cx < g.num_cells[0] && (D < 2 || cy < g.num_cells[1])) {
    const int cell = cx + (D > 1 ? g.num_cells[0] * cy : 0);
    ce = part.cell_end[cell];
    cs = part.cell_start[cell];
  }
  if (TYPED && t < 64) s_poly[t] = (&kSpanCubic[0][0][0])[t];
  const bool none = TYPED && !prm.node_types_built;  // untyped cubic weights are zero
  if (!__syncthreads_or(ce > cs) || none) {
    if (t == 0) flags[blockIdx.x] = 0;
    return;
  }
  float *st = &smem[wave][0];
  const int most = wave_max(ce - cs);  // particles of the row's fullest cell

  struct Raw {
    int slot, cx;
    bool valid;
    float x[D], v[D], m, vol, sg[3], dv[D], Lb[D * D];
  };
  struct Where {
    uint32_t j, slot;
    bool valid;
  };
  // the two rows of this lane in a round: cell (lane + 64 r) / KW, its
  // particle lane % KW
  int rs[2], re[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int c = (lane + 64 * r) / KW;
    rs[r] = __shfl(cs, c) + lane % KW;
    re[r] = __shfl(ce, c);
  }
  auto find = [&](int k0, int r) {
    Where w;
    const int j = rs[r] + k0;
    w.valid = j < re[r];
    w.j = w.valid ? (uint32_t)j : 0u;
    w.slot = __float_as_uint(ld32(reinterpret_cast<const float *>(part.sorted), w.j));
    return w;
  };
  auto load_raw = [&](const Where &w, int r, Raw &q) {
    const uint32_t jj = w.j, slot = w.slot;
    q.valid = w.valid;
    q.slot = (int)slot;
    q.cx = cx0 + (lane + 64 * r) / KW;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const int64_t row_a = (int64_t)a * n;
      q.x[a] = ld32(in.x + row_a, slot);
      q.v[a] = MODE == 0 ? ld32(in.v + row_a, slot) : (MODE == 1 ? ld32(out.v + row_a, jj) : ld32(rec + row_a, jj));
    }
    q.m = MODE == 2 ? 1.f : ld32(in.mass, slot);
    q.vol = MODE == 0 ? ld32(in.volume, slot) : 0.f;
    if (MODE == 0) {  // xx, then yy and xy
      q.sg[0] = ld32(in.stress, slot);
      q.sg[1] = D > 1 ? ld32(in.stress + (int64_t)n, slot) : 0.f;
      q.sg[2] = D > 1 ? ld32(in.stress + 3 * (int64_t)n, slot) : 0.f;
    }
    if (MODE == 2) {
#pragma unroll
      for (int a = 0; a < D; ++a) q.dv[a] = ld32(rec + (3 + a) * (int64_t)n, jj);
#pragma unroll
      for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) q.Lb[D * a + b] = ld32(rec + (6 + 3 * a + b) * (int64_t)n, jj);
    }
  };
  // is the particle in the cell it is listed in? fr: its fractions there
  auto own_cell = [&](const Raw &q, float *fr) {
    bool own = q.valid;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float ta = cell_coord(q.x[a], g.origin[a], inv_h);
      const int ba = (int)ta;
      own = own && ta >= 0.f && ba == (a == 0 ? q.cx : cy);  // (t < 0: stray path)
      fr[a] = __fsub_rn(ta, (float)ba);
    }
    return own;
  };
  bool strays = false;  // wave-uniform: some particle is listed in another cell than its own
  auto stage_raw = [&](const Raw &q, int r) {
    float fr[D], f[RS];
    const bool own = own_cell(q, fr);
    strays = strays || __ballot(q.valid && !own) != 0ull;
#pragma unroll
    for (int k = 0; k < RS; ++k) f[k] = 0.f;
    // (a row without an own particle is zero even if the fields it loaded are
    // not finite)
    if (own) {
#pragma unroll
      for (int a = 0; a < D; ++a) f[a] = fr[a];
      if (MODE == 0) {
        f[D] = q.m;
#pragma unroll
        for (int a = 0; a < D; ++a) f[D + 1 + a] = q.m * q.v[a];
#pragma unroll
        for (int a = 0; a < D * (D + 1) / 2; ++a) f[2 * D + 1 + a] = -q.vol * q.sg[a];
        if constexpr (FEXT) {
          float fe[3] = {0.f, 0.f, 0.f};
          planar_force<D>(prm, g, q.x, q.v, q.vol, q.m, fe);
#pragma unroll
          for (int a = 0; a < D; ++a) f[2 * D + 1 + D * (D + 1) / 2 + a] = fe[a];
        }
      } else if (MODE == 1) {
#pragma unroll
        for (int a = 0; a < D; ++a) f[D + a] = q.m * q.v[a];
      } else {
#pragma unroll
        for (int a = 0; a < D; ++a) { f[D + a] = q.v[a]; f[2 * D + a] = q.dv[a]; }
#pragma unroll
        for (int a = 0; a < D * D; ++a) f[3 * D + a] = q.Lb[a];
      }
    }
    float4 *sp = reinterpret_cast<float4 *>(st + ((lane + 64 * r) / KW) * CP + (lane % KW) * RS);
#pragma unroll
    for (int k = 0; k < RS / 4; ++k) sp[k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
  };

  // this lane's y polynomial; x weights are those of interior nodes but in a
  // row with cells near an x face (typed nodes), whose weights come from the
  // table: the x type and, with a carry out of x, the y type per x offset
  const int nx = g.num_cells[0], ny = g.num_cells[1];
  const int yv = cy + NLO + sy;
  SpanPoly<SF> py;
  if (D > 1) py.set(s_poly, sy, TYPED ? cubic_node_type(yv, ny, 1) : 0, inv_h, 1.f);
  const bool faces = TYPED && __ballot(ce > cs && (cx < 3 || cx >= nx - 3)) != 0ull;  // wave-uniform
  int xt[TYPED ? SPAN : 1] = {}, yt[TYPED ? SPAN : 1] = {};
  if (TYPED && faces) {
#pragma unroll
    for (int s = 0; s < SPAN; ++s) {
      int xv = cx + NLO + s, y = yv;
      if (D > 1 && MODE != 2 && prm.wrap_quirk) {
        while (xv < 0) { xv += nx; --y; }
        while (xv >= nx) { xv -= nx; ++y; }
      }
      xt[s] = 4 * (4 * cubic_node_type(xv, nx, 1) + s);
      yt[s] = D > 1 ? 4 * (4 * cubic_node_type(y, ny, 1) + sy) : 0;
    }
  }

  float acc[SPAN][NV];
#pragma unroll
  for (int s = 0; s < SPAN; ++s)
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[s][k] = 0.f;
  const float *own = st + lx * CP;
  auto read = [&](int k, float *f) {
#pragma unroll
    for (int q = 0; q < RS / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4 *>(own + k * RS + 4 * q);
      f[4 * q] = v.x; f[4 * q + 1] = v.y; f[4 * q + 2] = v.z; f[4 * q + 3] = v.w;
    }
  };
  // the record's sums for one y weight: field k gets Nx c[k] + dNx d[k]
  auto y_products = [&](const float *f, float Ny, float dNy, float *c, float *d) {
#pragma unroll
    for (int k = 0; k < NV; ++k) c[k] = d[k] = 0.f;
    if constexpr (MODE == 0) {
      constexpr int FA = 2 * D + 1, FE = FA + D * (D + 1) / 2;
      c[0] = Ny * f[D];
#pragma unroll
      for (int a = 0; a < D; ++a) c[1 + a] = Ny * f[D + 1 + a];
      if constexpr (D == 1) {
        d[2] = f[FA];
      } else {
        d[3] = Ny * f[FA]; c[3] = dNy * f[FA + 2];
        d[4] = Ny * f[FA + 2]; c[4] = dNy * f[FA + 1];
      }
      if constexpr (FEXT) {
#pragma unroll
        for (int a = 0; a < D; ++a) c[1 + D + a] += Ny * f[FE + a];
      }
    } else if constexpr (MODE == 1) {
#pragma unroll
      for (int a = 0; a < D; ++a) c[a] = Ny * f[D + a];
    } else {
#pragma unroll
      for (int a = 0; a < D; ++a) {
        c[a] = Ny * f[D + a];
        if (D > 1) c[a] += dNy * f[3 * D + D + a];
        d[a] = Ny * f[3 * D + a];
        c[D + a] = Ny * f[2 * D + a];
      }
    }
  };
  constexpr int DLO = MODE == 0 ? 1 + D : 0, DHI = MODE == 0 ? NV : (MODE == 1 ? 0 : D);  // fields with a dNx part
  auto add = [&](int s, float Nx, float dNx, const float *c, const float *d) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      acc[s][k] += Nx * c[k];
      if (k >= DLO && k < DHI) acc[s][k] += dNx * d[k];
    }
  };
  auto product = [&](const float *f) {
    float c[NV], d[NV], Nx[SPAN], dNx[SPAN];
    float Ny = 1.f, dNy = 0.f;
    if (D > 1) {
      Ny = py.N(f[D - 1]);
      dNy = MODE == 1 ? 0.f : py.dN(f[D - 1]);
    }
    y_products(f, Ny, dNy, c, d);
#pragma unroll
    for (int k = DLO; k < DHI; ++k) d[k] *= inv_h;
    inner_weights<SF>(f[0], Nx, dNx);
#pragma unroll
    for (int s = 0; s < SPAN; ++s) add(s, Nx[s], dNx[s], c, d);
  };
  auto product_face = [&](const float *f) {
    if constexpr (TYPED) {
#pragma unroll
      for (int s = 0; s < SPAN; ++s) {
        __builtin_amdgcn_sched_barrier(0);  // (one offset's table reads at a time: registers)
        const float x = f[0], y = f[D - 1];
        const float4 p = *reinterpret_cast<const float4 *>(s_poly + xt[s]);
        const float4 q = *reinterpret_cast<const float4 *>(s_poly + yt[s]);
        const float Ny = D > 1 ? ((q.w * y + q.z) * y + q.y) * y + q.x : 1.f;
        const float dNy = D > 1 ? inv_h * ((3.f * q.w * y + 2.f * q.z) * y + q.y) : 0.f;
        float c[NV], d[NV];
        y_products(f, Ny, dNy, c, d);
        add(s, ((p.w * x + p.z) * x + p.y) * x + p.x, inv_h * ((3.f * p.w * x + 2.f * p.z) * x + p.y), c, d);
      }
    }
  };

  Raw raw[2];
  Where ahead[2] = {};
#pragma unroll
  for (int r = 0; r < 2; ++r) ahead[r] = find(0, r);
#pragma unroll
  for (int r = 0; r < 2; ++r) load_raw(ahead[r], r, raw[r]);
  if (KW < most) {
#pragma unroll
    for (int r = 0; r < 2; ++r) ahead[r] = find(KW, r);
  }
#pragma unroll 1
  for (int k0 = 0; k0 < most; k0 += KW) {  // wave-uniform
    wave_lds_sync();  // the records staged before are read
#pragma unroll
    for (int r = 0; r < 2; ++r) stage_raw(raw[r], r);
    if (k0 + KW < most) {
#pragma unroll
      for (int r = 0; r < 2; ++r) load_raw(ahead[r], r, raw[r]);
      if (k0 + 2 * KW < most) {
#pragma unroll
        for (int r = 0; r < 2; ++r) ahead[r] = find(k0 + 2 * KW, r);
      }
    }
    wave_lds_sync();
    const int rows = min(KW, most - k0);
    float f[RS], f2[RS];
    read(0, f);
    // (two records per turn, each read while the one before is summed; past
    // the last one a staged or older record is read and not used)
    if (faces) {
#pragma unroll 1
      for (int k = 0; k < rows; ++k) {
        product_face(f);
        read((k + 1) & (KW - 1), f);
      }
    } else {
#pragma unroll 1
      for (int k = 0; k + 1 < rows; k += 2) {
        read(k + 1, f2);
        product(f);
        read((k + 2) & (KW - 1), f);
        product(f2);
      }
      if (rows & 1) product(f);
    }
  }

  // sums over the row's cells, [field][y offset][x], in the staging area
  float *blk = st;
#pragma unroll
  for (int s = 0; s < SPAN; ++s) {
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float *b = blk + (k * SY + sy) * NX + lx;
      if (s == 0) {
        b[0] = acc[0][k];
        if (lx < SPAN - 1) b[CELLS] = 0.f;
      } else {
        b[s] += acc[s][k];
      }
    }
  }
  lds_barrier();
  if (t == 0) flags[blockIdx.x] = 1;
  float *slice = partials + (int64_t)blockIdx.x * NV * G::NTN;
  for (int i = t; i < G::NTN; i += G::THREADS) {
    const int ix = i % NX, iy = i / NX;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int y = iy - r;
        if (y >= 0 && y < SY) sum += smem[r][(k * SY + y) * NX + ix];
      }
      slice[k * G::NTN + i] = sum;
    }
  }
  if (strays) {
    if (lane == 0) *nodes.flag = 1;
    // as in p2g_mfma_kernel: particles listed in this row that are not in their cell
#pragma unroll 1
    for (int k0 = 0; k0 < most; k0 += KW)
#pragma unroll 1
      for (int r = 0; r < 2; ++r) {
        Raw q;
        float fr[D], fe[3] = {0.f, 0.f, 0.f};
        load_raw(find(k0, r), r, q);
        if (own_cell(q, fr) || !q.valid) continue;
        if constexpr (MODE == 2) {
          adjoint_stray<D, SF, D>(prm, g, nodes, in.x, n, q.slot, q.v, q.dv, q.Lb);
          continue;
        }
        Sym A = sym_zero();
        if (MODE == 0) {
          const float mvol = -q.vol;
          A.xx = mvol * q.sg[0];
          A.yy = mvol * q.sg[1];
          A.xy = mvol * q.sg[2];
        }
        if (FEXT) planar_force<D>(prm, g, q.x, q.v, q.vol, q.m, fe);
        float v3[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int a = 0; a < D; ++a) v3[a] = q.v[a];
#pragma unroll 1
        for (int e = 0; e < SY; ++e)
          p2g_stray<D, SF, MODE == 1 ? 1 : 0>(prm, g, nodes, in.x, n, q.slot, e, q.m, v3, A, fe);
      }
  }
}

// The matrix-core P2G of 3D scenes. Tile: CELLS x ROWS x 4 cells, one wave per
// row of CELLS cells along x.
template <int SF, int CELLS, int ROWS, int NV> struct MfmaGeom {
  static constexpr int SPAN = Spline<SF>::SPAN, NLO = Spline<SF>::NLO;
  static constexpr int TZ = 4, WAVES = TZ * ROWS, THREADS = 64 * WAVES;
  static constexpr int BX = CELLS + SPAN - 1, NY = ROWS + SPAN - 1, NZ = TZ + SPAN - 1;  // tile nodes per axis
  static constexpr int NTN = BX * NY * NZ;                                              // nodes of one partial slice
  // a wave's node columns in LDS, [field][x][4 z + y]: the field pitch is 16
  // mod 32, so the four fields x 16 nodes of a flush fall into disjoint banks,
  // and a node's y window is one 16-byte read
  static constexpr int XP = 16;
  static constexpr int BN = BX * XP;
  static_assert(BN % 32 == 16, "field pitch");
  static constexpr int CH = 64;  // particle rows staged per round, one per lane
};
typedef float v4f __attribute__((ext_vector_type(4)));

// P2G of one tile on the matrix cores (3D, every spline).
//   MODE 0: mass, momentum, force (FEXT: with planar-domain wall forces).
//   MODE 1: the MUSL re-map of m v', v' from slot j of `out` (written by the
//           first map, g2p_kernel MODE 1), weights of the old positions.
//   MODE 2: adjoint scatter of the G2P record adjoints `rec` (cell order).
// Per cell and its SPAN^3 node window, with i, j, k the x, y, z node offsets
// and p the cell's particles, v_mfma_f32_16x16x4_f32 forms
//   C1[(f, i)][(j, k)] = sum_p (Nx_i F_f)(p) (Ny_j Nz_k)(p),  F = (m, m v)
//   C2[(a, i)][(j, k)] = sum_p (dNx_i A_ax [+ Nx_i fext_a])(Ny_j Nz_k)
//                              + (Nx_i A_ay)(dNy_j Nz_k) + (Nx_i A_az)(Ny_j dNz_k),  A = -V sigma
// (usl_inline.h:114-160), four particles per instruction; MODE 2 sums
// (v_pic adjoint, dv adjoint) and the L adjoint's rows the same way. Lane l
// supplies A[l % 16][l / 16] and B[l / 16][l % 16] and receives
// D[4 (l / 16) + r][l % 16]: it evaluates the x and z weights at offset l % 4
// and the y weight at offset (l % 16) / 4 for particle l / 16, and owns field
// l / 16 of the nodes (r, j, k). The x offset being the register index, moving
// on to the next cell is a register rotation: only the leftmost node column
// leaves, and each column of the wave's row is written once, complete.
//
// 1,080,000 particles, 27 per cell, cubic: P2G 81 -> 70 us (and 32 us of
// wrap-around launches less), re-map 40 -> 36 (23), adjoint scatter 159 -> 67.
// What bounds it (P2G, 70 us there): waiting, in workgroups that do not come
// out even. Vector instructions take 26 us of issue and the matrix cores are
// busy 15 us; a workgroup's 80,896 bytes of LDS let two run per CU, so the
// column's 750 tiles with particles take the 512 places in two rounds, the
// second half full, among the 3,644 empty tiles, which hold a place for the
// length of a cell-range read; within a wave the rounds are a chain of slots,
// fields, LDS and products. Per four particles there are 4 (MODE 1: 1) matrix
// instructions of 32 cycles and about 45 vector instructions; the weights are
// evaluated from per-lane coefficients (about 20 multiply-adds) instead of
// being staged: a particle's LDS record is 20 floats written by one lane and
// read with two 16-byte broadcasts and one word. The rows of a round are the wave's particles in sorted order, each
// cell padded to a multiple of four, so a round fills its 64 lanes whatever
// the particles per cell (at 8 per cell staging cell by cell left 3 of 4
// lanes idle); the next round's fields load while a round is multiplied, the
// slots of the round after with them.
//
// Linear-index wrap-around (usl_inline.h:122-126; shapefunction.cpp:96-112):
// a node offset outside the grid stays in the tile as a virtual node, with
// the spline types of the node its linear index reaches (types matter to the
// cubic spline only), and the grid kernel adds virtual nodes to the nodes
// they reach. A carry out of x shifts the y index by one, so the x offsets
// that leave the grid (cells next to an x face) are multiplied in a pass of
// their own, with that carry's y and z types and the other x offsets' weights
// zero; the carry out of y only changes the lane's own z type.
template <int SF, int MODE, int CELLS, int ROWS, bool FEXT = false>
__global__ __launch_bounds__(256 * ROWS) void p2g_mfma_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles in,
                                                       pmpm_particles out, pmpm_spatial part, Strays nodes,
                                                       int tiles_x, int tiles_y, float *__restrict__ partials,
                                                       int32_t *__restrict__ flags, const float *__restrict__ rec) {
  constexpr int NV = p2g_nv<3, MODE>();
  using M = MfmaGeom<SF, CELLS, ROWS, NV>;
  static_assert(MODE == 0 || !FEXT, "only the P2G carries the wall force");
  static_assert(CELLS == 4 || CELLS == 8, "cells per wave");
  constexpr int SPAN = M::SPAN, NLO = M::NLO, CH = M::CH, BN = M::BN;
  constexpr bool TYPED = SF == PMPM_SF_CUBIC;
  // floats of a staged record: the fractions, then MODE 0: (m, m v) and the
  // rows of A with the wall force; MODE 1: m v'; MODE 2: dv.x, per component
  // (v_pic adjoint, L adjoint's column), then (dv.y, dv.z)
  constexpr int RS = MODE == 1 ? 8 : 20;
  __shared__ __attribute__((aligned(16))) float block[M::WAVES][NV * BN];
  __shared__ __attribute__((aligned(16))) float stage[M::WAVES][CH * RS];

  __shared__ __attribute__((aligned(16))) float s_poly[TYPED ? 64 : 4];  // kSpanCubic

  const int n = in.n;
  const float inv_h = g.inv_cell_size;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int bx = blockIdx.x % tiles_x;
  const int by = (blockIdx.x / tiles_x) % tiles_y;
  const int bz = blockIdx.x / (tiles_x * tiles_y);
  const int cx0 = bx * CELLS, cy = by * ROWS + wave / M::TZ, cz = bz * M::TZ + wave % M::TZ;  // this wave's row
  // lanes 0..CELLS-1 hold the ranges of the wave's cells
  int cs = 0, ce = 0;
  {
    const int cx = cx0 + lane;
    if (lane < CELLS && cx < g.num_cells[0] && cy < g.num_cells[1] && cz < g.num_cells[2]) {
      const int cell = cx + g.num_cells[0] * (cy + g.num_cells[1] * cz);
      ce = part.cell_end[cell];
      cs = part.cell_start[cell];
    }
  }
  if (TYPED && t < 64) s_poly[t] = (&kSpanCubic[0][0][0])[t];
  const bool none = TYPED && !prm.node_types_built;  // untyped cubic weights are zero
  if (!__syncthreads_or(ce > cs) || none) {
    if (t == 0) flags[blockIdx.x] = 0;
    return;
  }
  float *blk = &block[wave][0];
  float *st = &stage[wave][0];
  // rows of a cell: its particles, padded to a multiple of four
  const int pad = (max(ce - cs, 0) + 3) & ~3;
  int rend = pad;  // inclusive sum over the cells
#pragma unroll
  for (int o = 1; o < CELLS; o <<= 1) {
    const int u = __shfl_up(rend, o, 64);
    if (lane >= o) rend += u;
  }
  const int total = __builtin_amdgcn_readlane(rend, CELLS - 1);
  const int shift = cs - (rend - pad);  // sorted index of a row, minus the row

  // a particle's raw fields, held in registers until staged
  struct Raw {
    int slot, cx;
    bool valid;
    float x[3], v[3], m, vol;
    Sym sg;
    float dv[3], Lb[9];
  };
  // the particle of row r0 + lane: its sorted index, slot and cell (the slots
  // are fetched a round before the fields that need them)
  struct Where {
    uint32_t j, slot;
    int c;
    bool valid;
  };
  auto find = [&](int r0) {
    Where w;
    const int row = r0 + lane;
    int c = 0;  // the first cell whose rows end past this one
#pragma unroll
    for (int l = 0; l < CELLS - 1; ++l) c += __builtin_amdgcn_readlane(rend, l) <= row ? 1 : 0;
    const int j = __shfl(shift, c) + row, je = __shfl(ce, c);
    w.c = c;
    w.valid = row < total && j < je;
    w.j = w.valid ? (uint32_t)j : 0u;
    w.slot = __float_as_uint(ld32(reinterpret_cast<const float *>(part.sorted), w.j));
    return w;
  };
  auto load_raw = [&](const Where &w, Raw &r) {
    const uint32_t jj = w.j, slot = w.slot;
    r.cx = cx0 + w.c;
    r.valid = w.valid;
    r.slot = (int)slot;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int64_t row_a = (int64_t)a * n;
      r.x[a] = ld32(in.x + row_a, slot);
      r.v[a] = MODE == 0 ? ld32(in.v + row_a, slot) : (MODE == 1 ? ld32(out.v + row_a, jj) : ld32(rec + row_a, jj));
    }
    r.m = MODE == 2 ? 1.f : ld32(in.mass, slot);
    r.vol = MODE == 0 ? ld32(in.volume, slot) : 0.f;
    r.sg = sym_zero();
    if (MODE == 0) {
      const float *sg = in.stress;
      r.sg = Sym{ld32(sg, slot), ld32(sg + (int64_t)n, slot), ld32(sg + 2 * (int64_t)n, slot),
                 ld32(sg + 3 * (int64_t)n, slot), ld32(sg + 4 * (int64_t)n, slot), ld32(sg + 5 * (int64_t)n, slot)};
    }
    if (MODE == 2) {
#pragma unroll
      for (int a = 0; a < 3; ++a) r.dv[a] = ld32(rec + (3 + a) * (int64_t)n, jj);
#pragma unroll
      for (int a = 0; a < 9; ++a) r.Lb[a] = ld32(rec + (6 + a) * (int64_t)n, jj);
    }
  };
  // this lane's particle into its row of the stage (zero past the cell's
  // particles, and for a particle that is not its own cell's)
  // is the particle in the cell it is listed in? fr: its fractions there
  auto own_cell = [&](const Raw &r, float *fr) {
    bool own = r.valid;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float ta = cell_coord(r.x[a], g.origin[a], inv_h);
      const int ba = (int)ta;
      own = own && ta >= 0.f && ba == (a == 0 ? r.cx : (a == 1 ? cy : cz));
      fr[a] = __fsub_rn(ta, (float)ba);
    }
    return own;
  };
  auto minus_v_sigma = [&](const Raw &r) {
    const float mvol = -r.vol;
    return Sym{mvol * r.sg.xx, mvol * r.sg.yy, mvol * r.sg.zz, mvol * r.sg.xy, mvol * r.sg.xz, mvol * r.sg.yz};
  };
  bool strays = false;  // wave-uniform: some particle is listed in another cell than its own
  auto stage_raw = [&](const Raw &r) {
    float fr[3];
    const bool own = own_cell(r, fr);
    strays = strays || __ballot(r.valid && !own) != 0ull;
    float4 *sp = reinterpret_cast<float4 *>(st + lane * RS);
    Sym A = sym_zero();
    float fe[3] = {0.f, 0.f, 0.f};
    if (MODE == 0) {
      A = minus_v_sigma(r);
      if (FEXT && r.valid) planar_force<3>(prm, g, r.x, r.v, r.vol, r.m, fe);
    }
    // (a row without an own particle is zero even if the fields it loaded are
    // not finite)
    if (own) {
      sp[0] = make_float4(fr[0], fr[1], fr[2], MODE == 2 ? r.dv[0] : 0.f);
      if (MODE == 0) {
        sp[1] = make_float4(r.m, r.m * r.v[0], r.m * r.v[1], r.m * r.v[2]);
        sp[2] = make_float4(A.xx, A.xy, A.xz, fe[0]);
        sp[3] = make_float4(A.xy, A.yy, A.yz, fe[1]);
        sp[4] = make_float4(A.xz, A.yz, A.zz, fe[2]);
      } else if (MODE == 1) {
        sp[1] = make_float4(r.m * r.v[0], r.m * r.v[1], r.m * r.v[2], 0.f);
      } else {
#pragma unroll
        for (int a = 0; a < 3; ++a) sp[1 + a] = make_float4(r.v[a], r.Lb[a], r.Lb[3 + a], r.Lb[6 + a]);
        sp[4] = make_float4(r.dv[1], r.dv[2], 0.f, 0.f);
      }
    } else {
#pragma unroll
      for (int q = 0; q < RS / 4; ++q) sp[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };

  // lane roles in the products
  const int s1 = (lane & 15) >> 2, s2 = lane & 3, pk = lane >> 4;
  SpanPoly<SF> px, py, pz;
  // y and z weights for x carry kx (see above)
  auto set_yz = [&](int kx) {
    int ty = 0, tz = 0;
    if (TYPED) {
      int yv = cy + NLO + s1 + kx, zv = cz + NLO + s2;
      if (prm.wrap_quirk) {
        while (yv < 0) { yv += g.num_cells[1]; --zv; }
        while (yv >= g.num_cells[1]) { yv -= g.num_cells[1]; ++zv; }
      }
      ty = cubic_node_type(yv, g.num_cells[1], 1);
      tz = cubic_node_type(zv, g.num_cells[2], 1);
    }
    py.set(s_poly, s1, ty, inv_h, 1.f);
    pz.set(s_poly, s2, tz, inv_h, 1.f);
  };
  set_yz(0);

  v4f C1 = {0.f, 0.f, 0.f, 0.f}, C2 = C1;
  // what a product step reads of the stage (rows row .. row + 3): read one
  // step ahead, so that the reads' latency passes behind the step before
  struct Step {
    float4 f, A;
    float F;
  };
  const float *st_f = st + pk * RS;
  // (MODE 0: field row 3 of the force is padding and reads row 2; MODE 2: row
  // 3 is dv.x, which the fractions' word 3 holds, and C2's rows 2 and 3 are
  // padding)
  const float *st_A = st_f + (MODE == 0 ? 8 : 4) + 4 * min(s1, 2);
  const float *st_F = st_f + (MODE == 2 ? 16 : 4) + s1;
  auto read_step = [&](int row) {
    Step q;
    q.f = *reinterpret_cast<const float4 *>(st_f + row * RS);
    if (MODE != 1) q.A = *reinterpret_cast<const float4 *>(st_A + row * RS);
    q.F = st_F[row * RS];
    return q;
  };
  auto product = [&](const Step &q) {
    const float Nx = px.N(q.f.x), Ny = py.N(q.f.y), Nz = pz.N(q.f.z);
    const float b1 = Ny * Nz;
    if (MODE == 1) {
      C1 = __builtin_amdgcn_mfma_f32_16x16x4f32(Nx * q.F, b1, C1, 0, 0, 0);
      return;
    }
    const float dNx = px.dN(q.f.x), dNy = py.dN(q.f.y), dNz = pz.dN(q.f.z);
    const float b2 = dNy * Nz, b3 = Ny * dNz;
    if (MODE == 0) {
      C1 = __builtin_amdgcn_mfma_f32_16x16x4f32(Nx * q.F, b1, C1, 0, 0, 0);
      float a2 = dNx * q.A.x;
      if (FEXT) a2 += Nx * q.A.w;
      C2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, b1, C2, 0, 0, 0);
      C2 = __builtin_amdgcn_mfma_f32_16x16x4f32(Nx * q.A.y, b2, C2, 0, 0, 0);
      C2 = __builtin_amdgcn_mfma_f32_16x16x4f32(Nx * q.A.z, b3, C2, 0, 0, 0);
    } else {
      const bool v = s1 < 3;
      C1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v ? Nx * q.A.x + dNx * q.A.y : Nx * q.f.w, b1, C1, 0, 0, 0);
      C2 = __builtin_amdgcn_mfma_f32_16x16x4f32(Nx * q.F, b1, C2, 0, 0, 0);
      C1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v ? Nx * q.A.z : 0.f, b2, C1, 0, 0, 0);
      C1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v ? Nx * q.A.w : 0.f, b3, C1, 0, 0, 0);
    }
  };
  // node column lx of the wave's row is complete: out of the accumulators (linear
  // splines: the columns past the span hold products with zero weights, which
  // are not zero where a field is not finite)
  auto shifted = [](const v4f &C) {
    return v4f{C[1], SPAN > 2 ? C[2] : 0.f, SPAN > 3 ? C[3] : 0.f, 0.f};
  };
  auto flush = [&](int lx) {
    float *b = blk + lx * M::XP + 4 * s2 + s1;
    if (MODE != 1 || pk < 3) b[pk * BN] = C1[0];
    C1 = shifted(C1);
    if (MODE != 1) {
      if (pk < (MODE == 0 ? 3 : 2)) b[(4 + pk) * BN] = C2[0];
      C2 = shifted(C2);
    }
  };

  // the fields of the round to be staged next, and the slots of the one after
  Raw raw;
  Where ahead_w{};
  int next = 2 * CH;  // first row whose slots are not yet fetched
  if (total > 0) {
    load_raw(find(0), raw);
    if (CH < total) ahead_w = find(CH);
  }
  int r0 = -CH, row = 0;  // first staged row, current row
  Step cur{};
  bool inner_x = false;  // px holds the weights of the x cells [3, nx - 4], which share their node types
  const int nx = g.num_cells[0];
#pragma unroll 1
  for (int l = 0; l < CELLS; ++l) {  // wave-uniform
    const int cx = cx0 + l;
    const int end = __builtin_amdgcn_readlane(rend, l);
    if (row < end) {
      const bool inx = !TYPED || (cx >= 3 && cx < nx - 3);
      const int xv = cx + NLO + s2;  // this lane's x node
      const bool out_x = xv < 0 || xv >= nx;
      if (!inx || !inner_x) {
        px.set(s_poly, s2, TYPED ? cubic_node_type(xv, nx, 1) : 0, inv_h, TYPED && out_x ? 0.f : 1.f);
        inner_x = inx;
      }
      const bool leaves = TYPED && MODE != 2 && !inx && prm.wrap_quirk && __ballot(out_x) != 0ull;
      while (row < end) {
        if (row - r0 >= CH) {
          wave_lds_sync();  // the rows staged before are read
          stage_raw(raw);
          r0 = row;
          if (r0 + CH < total) load_raw(ahead_w, raw);
          if (next < total) ahead_w = find(next);
          next += CH;
          wave_lds_sync();
          cur = read_step(0);
        }
        const int stop = min(end, r0 + CH);
        const int first = row;
        // (two steps per turn: no register copies between cur and ahead)
        for (; row + 4 < stop; row += 8) {
          const Step ahead = read_step(row + 4 - r0);
          __builtin_amdgcn_sched_barrier(0);
          product(cur);
          cur = read_step((row + 8 - r0) & (CH - 1));
          __builtin_amdgcn_sched_barrier(0);
          product(ahead);
        }
        if (row < stop) {
          const Step ahead = read_step((row + 4 - r0) & (CH - 1));
          product(cur);
          cur = ahead;
          row += 4;
        }
        if (leaves) {
#pragma unroll 1
          for (int kx = -1; kx <= 2; ++kx) {  // (2: one-node grids only)
            const bool mine = kx != 0 && xv - kx * nx >= 0 && xv - kx * nx < nx;
            if (__ballot(mine) == 0ull) continue;
            px.set(s_poly, s2, cubic_node_type(mine ? xv - kx * nx : 0, nx, 1), inv_h, mine ? 1.f : 0.f);
            set_yz(kx);
            for (int q = first; q < stop; q += 4) product(read_step(q - r0));
          }
          px.set(s_poly, s2, cubic_node_type(xv, nx, 1), inv_h, out_x ? 0.f : 1.f);
          set_yz(0);
        }
      }
    }
    flush(l);
  }
#pragma unroll
  for (int l = 0; l < SPAN - 1; ++l) flush(CELLS + l);
  lds_barrier();
  // the waves' columns: node (ix, iy, iz) lies in the rows iy - SPAN + 1 .. iy
  // and the layers iz - SPAN + 1 .. iz; slices are stored y slowest
  if (t == 0) flags[blockIdx.x] = 1;
  float *slice = partials + (int64_t)blockIdx.x * NV * M::NTN;
  constexpr int PL = M::BX * M::NZ;  // nodes of a y plane
  for (int i = t; i < PL * NV; i += M::THREADS) {
    const int ix = i % M::BX, iz = (i / M::BX) % M::NZ, f = i / PL;
    float sum[M::NY];
#pragma unroll
    for (int y = 0; y < M::NY; ++y) sum[y] = 0.f;
#pragma unroll
    for (int w = 0; w < M::TZ; ++w) {
      const int z = iz - w;
      if (z < 0 || z >= SPAN) continue;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const float4 q = *reinterpret_cast<const float4 *>(&block[r * M::TZ + w][f * BN + ix * M::XP + 4 * z]);
        const float yj[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < SPAN; ++j) sum[r + j] += yj[j];
      }
    }
#pragma unroll
    for (int y = 0; y < M::NY; ++y) slice[f * M::NTN + y * PL + i % PL] = sum[y];
  }
  if (strays) {
    if (lane == 0) *nodes.flag = 1;
    // particles listed in this row that are not in their cell (left of the
    // origin, or a partition of other positions): deposited over their own
    // windows, straight to the stray sums. Walked again here, where the
    // registers of the products are free.
#pragma unroll 1
    for (int q0 = 0; q0 < total; q0 += 64) {
      Raw q;
      float fr[3], fe[3] = {0.f, 0.f, 0.f};
      load_raw(find(q0), q);
      if (own_cell(q, fr) || !q.valid) continue;
      if constexpr (MODE == 2) {
        adjoint_stray<3, SF, 3>(prm, g, nodes, in.x, n, q.slot, q.v, q.dv, q.Lb);
        continue;
      }
      Sym A = sym_zero();
      if (MODE == 0) A = minus_v_sigma(q);
      if (FEXT) planar_force<3>(prm, g, q.x, q.v, q.vol, q.m, fe);
#pragma unroll 1
      for (int sy = 0; sy < 4; ++sy)
        p2g_stray<3, SF, MODE == 1 ? 1 : 0>(prm, g, nodes, in.x, n, q.slot, sy, q.m, q.v, A, fe);
    }
  }
}

// P2G (MODE 0) or MUSL re-map (MODE 1) of every particle over its own window,
// straight to the stray sums: for steps whose workspace has no room for the tile
// partials (pmpm_step_noalloc). Bound by its global atomics, up to 64
// nodes of 7 fields per particle.
template <int D, int SF, int MODE>
__global__ __launch_bounds__(256) void p2g_direct_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles in,
                                                         pmpm_particles out, pmpm_spatial part, Strays nodes,
                                                         int fext) {
  const int n = in.n, j = (int)blockIdx.x * 256 + (int)threadIdx.x;
  if (j == 0) *nodes.flag = 1;
  if (j >= n) return;
  const int slot = part.sorted[j];
  if (part.hash[slot] >= (uint32_t)g.num_cells_total) return;  // (in no cell: not deposited)
  const float m = in.mass[slot];
  float x[3] = {0.f, 0.f, 0.f}, v[3] = {0.f, 0.f, 0.f}, fe[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    x[a] = in.x[(int64_t)a * n + slot];
    v[a] = MODE == 0 ? in.v[(int64_t)a * n + slot] : out.v[(int64_t)a * n + j];
  }
  Sym A = sym_zero();
  if (MODE == 0) {
    const float vol = in.volume[slot];
    const Sym s = load_sym(in.stress, n, slot);
    A = Sym{-vol * s.xx, -vol * s.yy, -vol * s.zz, -vol * s.xy, -vol * s.xz, -vol * s.yz};
    if (fext) planar_force<D>(prm, g, x, v, vol, m, fe);
  }
#pragma unroll 1
  for (int sy = 0; sy < 4; ++sy) p2g_stray<D, SF, MODE>(prm, g, nodes, in.x, n, slot, sy, m, v, A, fe);
}

// Geometry of the P2G tiles for the grid kernel's gather.
struct TileGeom {
  int tiles[3];  // tiles per axis
  int T[3];      // cells per tile per axis
  int N[3];      // nodes per tile block per axis (T + SPAN - 1)
  int nv;        // fields per node in the partials
};

// Sums the NV fields of the partial slices of the tiles whose node block
// covers node `ids`, in a fixed tile order (z, y, x ascending). The live
// flags of all candidate tiles are loaded first; then every candidate's loads
// are issued without a branch (a dead or out-of-range candidate reads tile
// 0's first entries and adds zero), so a node waits for two loads in a row,
// not one per tile. Returns whether any candidate tile was live (a node no
// live tile covers skips the loads).
// TG: the tiling's constants (the divisions then become shifts).
template <int D, int SPAN_, int CELLS_, int ROWS_> struct Tiles {
  static constexpr int SPAN = SPAN_, NLO = SPAN_ == 2 ? 0 : -1;
  static constexpr int T[3] = {CELLS_, ROWS_, D > 2 ? 4 : 1};
  static constexpr int N[3] = {CELLS_ + SPAN_ - 1, D > 1 ? ROWS_ + SPAN_ - 1 : 1, D > 2 ? 3 + SPAN_ : 1};
  static constexpr int COVER_Y = (N[1] - 1) / T[1] + 1;
  static constexpr int CELLS = T[0] * T[1] * T[2];
  static_assert((N[0] - 1) / T[0] + 1 <= kCoverX && COVER_Y <= kCoverY && (N[2] - 1) / T[2] + 1 <= kCoverZ,
                "the gather visits at most kCover tiles per axis");
};
template <int D, int NV, class TG>
__device__ inline bool gather_partials(const TileGeom &tg, const float *partials, const int32_t *flags,
                                       const int *ids, float *acc) {
  constexpr int MX = kCoverX, MY = TG::COVER_Y, MZ = D > 2 ? kCoverZ : 1;
  constexpr int MC = MX * MY * MZ, nlo = TG::NLO;
  int T[3], N[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) { T[a] = TG::T[a]; N[a] = TG::N[a]; }
  int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    // tile b covers nodes [b*T + nlo, b*T + nlo + N - 1]
    const int r = ids[a] - nlo;
    int b_hi = r / T[a];
    int b_lo = (r - N[a] + T[a]) >= 0 ? (r - N[a] + T[a]) / T[a] : 0;
    if (b_hi > tg.tiles[a] - 1) b_hi = tg.tiles[a] - 1;
    lo[a] = b_lo;
    hi[a] = b_hi;
  }
  const int ntn = N[0] * (D > 1 ? N[1] : 1) * (D > 2 ? N[2] : 1);
  bool live[MC];
  int64_t off[MC];
#pragma unroll
  for (int cz = 0; cz < MZ; ++cz)
#pragma unroll
    for (int cy = 0; cy < MY; ++cy)
#pragma unroll
      for (int cx = 0; cx < MX; ++cx) {
        const int c = (cz * MY + cy) * MX + cx;
        const int bx = lo[0] + cx, by = lo[1] + cy, bz = lo[2] + cz;
        const bool in = bx <= hi[0] && by <= hi[1] && bz <= hi[2];
        const int tile = in ? bx + tg.tiles[0] * (by + tg.tiles[1] * bz) : 0;
        live[c] = in && flags[tile] != 0;
        int li = ids[0] - (bx * T[0] + nlo);
        // (3D slices: y slowest)
        if (D == 2) li += N[0] * (ids[1] - (by * T[1] + nlo));
        if (D > 2) li += N[0] * (ids[2] - (bz * T[2] + nlo) + N[2] * (ids[1] - (by * T[1] + nlo)));
        off[c] = (int64_t)tile * NV * ntn + li;
      }
  bool any = false;
#pragma unroll
  for (int c = 0; c < MC; ++c) any = any || live[c];
  if (!any) return false;
#pragma unroll
  for (int c = 0; c < MC; ++c) {
    const float *s = partials + (live[c] ? off[c] : 0);
    float v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = s[(int64_t)k * ntn];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] += live[c] ? v[k] : 0.f;
  }
  return true;
}

// The node of thread t of a pass over all nodes (false: none): tile by tile, a
// tile's nodes in x, y, z order, so that the slice rows a wave's lanes read are
// the same or neighbours (64 nodes of one x row would read a short row of each
// of 8 or 16 slices).
template <int D, class TG>
__device__ inline bool pass_node(const pmpm_grid &g, const TileGeom &tg, int t, int *ids) {
  int b = t / TG::CELLS, l = t % TG::CELLS;
  if (b >= tg.tiles[0] * tg.tiles[1] * tg.tiles[2]) return false;
  bool in = true;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    ids[a] = (a < D - 1 ? b % tg.tiles[a] : b) * TG::T[a] + l % TG::T[a];
    b /= tg.tiles[a];
    l /= TG::T[a];
    in = in && ids[a] < g.num_cells[a];
  }
  return in;
}
// What bounds it: the slices' lines (a node reads up to 12 rows of 7 fields in
// 3D). 3,276,800 particles on 1.07M nodes 87 -> 59 us, 1,080,000 on 263,000
// 21.7 -> 18.5 us when the nodes went from x rows to tiles and the node arrays
// were no longer read.
// Per node: cutoff + forward moment (finalize), boundary conditions
// [bc_begin, bc_end) in list order, then the node velocities G2P reads.
// remap_pass: mom_nt holds the MUSL re-mapped momentum; only kinematic
// conditions apply (gravity already acted through the particle velocities).
// skip_mom_nt: mom_nt is not written (the MUSL step's first pass: nothing reads
// the forward moment but the velocity records written here, and the re-map's
// pass writes it next).
// clamp (optional): per node, the components a NodeDomain condition set to
// zero (bit a: moment, bit 3 + a: forward moment; a slip clamp counts when
// its input was not on the kept side), for the adjoint.
// 2D and 3D: the nodes the wrap-around can reach are left to the launch's
// first nwrap workgroups, four lanes per node: the node itself and the virtual
// nodes outside the grid that share its linear index (up to three on grids of
// at least three nodes along x and y) are gathered by a lane each
// and summed over the lanes in a fixed order. The workgroups after them take
// the other nodes, one lane each.
constexpr int kImageLanes = 4;
template <int D, int NV, class TG>
__device__ inline void gather_images(const pmpm_grid &g, const TileGeom &tg, const float *partials,
                                     const int32_t *flags, const int *ids, int lane, float *acc) {
  const int nx = g.num_cells[0], ny = g.num_cells[1], nz = D > 2 ? g.num_cells[2] : 1;
  constexpr int lo = TG::NLO, hi = TG::NLO + TG::SPAN - 1;
  const int kx_end = nx < 3 ? 2 : 1, ky_end = ny < 3 ? 2 : 1;
  int count = 0;
#pragma unroll 1
  for (int round = 0; round == 0 || count > kImageLanes * round; ++round) {  // (one round but on tiny grids)
    // this lane's image is picked first, so that the lanes gather together
    int mine[3] = {0, 0, 0};
    bool have = false;
    count = 0;
    for (int kx = -1; kx <= kx_end; ++kx) {
      const int vx = ids[0] + kx * nx;
      if (vx < lo || vx > nx - 1 + hi) continue;
      int qy = ids[1] - kx, qz = ids[2];
      if (D == 2) {  // (a carry out of y leaves the grid)
        if (qy < lo || qy > ny - 1 + hi) continue;
        if (count++ == kImageLanes * round + lane) {
          mine[0] = vx;
          mine[1] = qy;
          have = true;
        }
        continue;
      }
      while (qy < 0) { qy += ny; --qz; }
      while (qy >= ny) { qy -= ny; ++qz; }
      for (int ky = -1; ky <= ky_end; ++ky) {
        const int vy = qy + ky * ny, vz = qz - ky;
        if (vy < lo || vy > ny - 1 + hi || vz < lo || vz > nz - 1 + hi) continue;
        if (count++ == kImageLanes * round + lane) {
          mine[0] = vx;
          mine[1] = vy;
          mine[2] = vz;
          have = true;
        }
      }
    }
    if (have) gather_partials<D, NV, TG>(tg, partials, flags, mine, acc);
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int o = 1; o < kImageLanes; o <<= 1) acc[k] += __shfl_xor(acc[k], o);
}
// GATHER as make_tiles' `gather` (fixed per instance: it sets the fields gathered).
template <int D, int GATHER, class TG>
__global__ __launch_bounds__(256) void grid_kernel(pmpm_params prm, pmpm_grid g, pmpm_nodes nodes, int finalize, int bc_begin, int bc_end,
                            int remap_pass, TileGeom tg, const float *__restrict__ partials,
                            const int32_t *__restrict__ flags, int skip_mom_nt, uint8_t *__restrict__ clamp,
                            int nwrap, Strays strays) {
  const int nn = g.num_cells_total;
  int i, ids0[3] = {0, 0, 0};
  bool reached = false;  // a node the wrap-around can reach
  if (D > 1 && (int)blockIdx.x < nwrap) {
    const int t = (blockIdx.x * blockDim.x + threadIdx.x) / kImageLanes;
    if (t >= wrap_target_count<D>(g) || !wrap_target<D>(g, t, ids0)) return;  // (a node's lanes together)
    reached = true;
  } else {
    if (!pass_node<D, TG>(g, tg, ((int)blockIdx.x - nwrap) * (int)blockDim.x + (int)threadIdx.x, ids0)) return;
    if (D > 1 && nwrap > 0 &&
        (ids0[0] <= 1 || ids0[0] == g.num_cells[0] - 1 || (D > 2 && (ids0[1] <= 1 || ids0[1] == g.num_cells[1] - 1))))
      return;
  }
  i = ids0[0] + (D > 1 ? g.num_cells[0] * (ids0[1] + (D > 2 ? g.num_cells[1] * ids0[2] : 0)) : 0);
  // GATHER 1: mass, momentum and force are the sums gathered here; 2: the
  // momentum mom_nt is; the rest (0: all) comes from the node arrays
  float m = 0.f, P[3] = {0.f, 0.f, 0.f}, Q[3] = {0.f, 0.f, 0.f};
  if constexpr (GATHER != 1) {
    m = nodes.mass[i];
#pragma unroll
    for (int a = 0; a < D; ++a) P[a] = nodes.mom[a * nn + i];
  }
  const float P0[3] = {P[0], P[1], P[2]};
  if constexpr (GATHER == 0) {
#pragma unroll
    for (int a = 0; a < D; ++a) Q[a] = nodes.mom_nt[a * nn + i];
  } else {
    constexpr int NV = GATHER == 1 ? 1 + 2 * D : D;
    float acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = 0.f;
    if (reached) {
      if constexpr (D > 1) {
        const int lane = (int)threadIdx.x & (kImageLanes - 1);
        gather_images<D, NV, TG>(g, tg, partials, flags, ids0, lane, acc);
        if (lane != 0) return;
      }
    } else {
      gather_partials<D, NV, TG>(tg, partials, flags, ids0, acc);
    }
    if (*strays.flag) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        // (mass, momentum, force)
        float *a0 = GATHER == 1 && k == 0 ? strays.mass
                                          : (GATHER == 1 && k <= D ? strays.mom + (int64_t)(k - 1) * nn
                                                                   : strays.mom_nt + (int64_t)(GATHER == 1 ? k - 1 - D : k) * nn);
        acc[k] += a0[i];
        a0[i] = 0.f;
      }
    }
    if constexpr (GATHER == 1) {
      m = acc[0];
#pragma unroll
      for (int a = 0; a < D; ++a) {
        P[a] = acc[1 + a];
        Q[a] = acc[1 + D + a];
      }
      if (!(m <= prm.small_mass_cutoff)) nodes.mass[i] = m;  // (else written below)
    } else {
#pragma unroll
      for (int a = 0; a < D; ++a) Q[a] = acc[a];
    }
  }
  if ((finalize || remap_pass) && m <= prm.small_mass_cutoff) {
    if (finalize) {
      nodes.mass[i] = 0.f;
#pragma unroll
      for (int a = 0; a < D; ++a) nodes.mom[a * nn + i] = 0.f;
    }
#pragma unroll
    for (int a = 0; a < D; ++a) nodes.mom_nt[a * nn + i] = 0.f;
    // a body force acts whatever the node's mass (bodyforce_inline.h:41-59);
    // the gathers skip the node all the same
    for (int k = bc_begin; k < bc_end; ++k) {
      const pmpm_bc &bc = prm.bcs[k];
      if (bc.kind != PMPM_BC_BODY_FORCE || !bc.mask[i]) continue;
      if (bc.i[0] == 2) {
#pragma unroll
        for (int a = 0; a < D; ++a) nodes.mom_nt[a * nn + i] = bc.values[a * nn + i];
      } else if (!remap_pass) {
#pragma unroll
        for (int a = 0; a < D; ++a) nodes.mom[a * nn + i] += bc.values[a * nn + i];
      }
    }
    const float z[3] = {0.f, 0.f, 0.f};
    store_node_vel<D>(nodes.vel, i, z, z);
    return;
  }
  if (finalize) {
#pragma unroll
    for (int a = 0; a < D; ++a) Q[a] = P[a] + Q[a] * prm.dt;
  }
  const int *ids = ids0;
  unsigned cbits = 0u;
  for (int k = bc_begin; k < bc_end; ++k) {
    const pmpm_bc &bc = prm.bcs[k];
    if (bc.kind == PMPM_BC_GRAVITY) {
      // gravity_inline.h:46-63
      if (remap_pass || m <= 0.000000001f) continue;
#pragma unroll
      for (int a = 0; a < D; ++a) Q[a] = __fadd_rn(Q[a], __fmul_rn(__fmul_rn(bc.f[a], m), prm.dt));
    } else if (bc.kind == PMPM_BC_NODE_DOMAIN) {
      // nodedomain_inline.h:40-87: 0 fixed, 1 slip (one-sided clamp)
      if (m <= 0.00001f) continue;
#pragma unroll
      for (int a = 0; a < D; ++a) {
        if (ids[a] < 1) {
          if (bc.i[a] == 0) {
#pragma unroll
            for (int b = 0; b < D; ++b) { P[b] = 0.f; Q[b] = 0.f; }
            cbits |= 0x3fu;
          } else if (bc.i[a] == 1) {
            if (!(P[a] > 0.f)) cbits |= 1u << a;
            if (!(Q[a] > 0.f)) cbits |= 8u << a;
            P[a] = fmaxf(0.f, P[a]);
            Q[a] = fmaxf(0.f, Q[a]);
          }
        } else if (ids[a] >= g.num_cells[a] - 1) {
          if (bc.i[3 + a] == 0) {
#pragma unroll
            for (int b = 0; b < D; ++b) { P[b] = 0.f; Q[b] = 0.f; }
            cbits |= 0x3fu;
          } else if (bc.i[3 + a] == 1) {
            if (!(P[a] < 0.f)) cbits |= 1u << a;
            if (!(Q[a] < 0.f)) cbits |= 8u << a;
            P[a] = fminf(0.f, P[a]);
            Q[a] = fminf(0.f, Q[a]);
          }
        }
      }
    } else if (bc.kind == PMPM_BC_BODY_FORCE) {
      // bodyforce_inline.h:41-59: "fixed" sets the forward moments, the
      // other modes add to the moments; no mass test. The MUSL re-map pass
      // re-applies only the kinematic "fixed" mode.
      if (!bc.mask[i]) continue;
      if (bc.i[0] == 2) {
#pragma unroll
        for (int a = 0; a < D; ++a) Q[a] = bc.values[a * nn + i];
      } else if (!remap_pass) {
#pragma unroll
        for (int a = 0; a < D; ++a) P[a] = __fadd_rn(P[a], bc.values[a * nn + i]);
      }
    } else if (bc.kind == PMPM_BC_RIGID_SDF) {
      if (m <= 0.000000001f) continue;
      // box signed distance in the body frame; n = -grad(phi)
      float xn[3];
#pragma unroll
      for (int a = 0; a < D; ++a) xn[a] = g.origin[a] + (float)ids[a] * g.cell_size;
      float q[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < D; ++r) {
        float sacc = 0.f;
#pragma unroll
        for (int a = 0; a < D; ++a) sacc += bc.f[9 + a * 3 + r] * (xn[a] - bc.f[3 + a]);
        q[r] = sacc;
      }
      float d[3], out2 = 0.f, inmax = -3.0e38f;
      int amax = 0;
#pragma unroll
      for (int r = 0; r < D; ++r) {
        d[r] = fabsf(q[r]) - bc.f[r];
        if (d[r] > 0.f) out2 += d[r] * d[r];
        if (d[r] > inmax) { inmax = d[r]; amax = r; }
      }
      float gl[3] = {0.f, 0.f, 0.f}, phi;
      if (out2 > 0.f) {
        const float o = sqrtf(out2);
#pragma unroll
        for (int r = 0; r < D; ++r) gl[r] = (d[r] > 0.f ? d[r] : 0.f) * (q[r] >= 0.f ? 1.f : -1.f) / o;
        phi = o;
      } else {
#pragma unroll
        for (int r = 0; r < D; ++r) gl[r] = (r == amax) ? (q[r] >= 0.f ? 1.f : -1.f) : 0.f;
        phi = inmax;
      }
      if (!(phi < bc.f[18])) continue;
      float nrm[3];
#pragma unroll
      for (int a = 0; a < D; ++a) {
        float sacc = 0.f;
#pragma unroll
        for (int r = 0; r < D; ++r) sacc += bc.f[9 + a * 3 + r] * gl[r];
        nrm[a] = -sacc;
      }
      float rc = 0.f, rct = 0.f;
#pragma unroll
      for (int a = 0; a < D; ++a) {
        rc += (P[a] / m - bc.f[6 + a]) * nrm[a];
        rct += (Q[a] / m - bc.f[6 + a]) * nrm[a];
      }
      if (rc >= 0.f) {
#pragma unroll
        for (int a = 0; a < D; ++a) P[a] = bc.f[6 + a] * m;
      }
      if (rct >= 0.f) {
#pragma unroll
        for (int a = 0; a < D; ++a) Q[a] = bc.f[6 + a] * m;
      }
    }
  }
#pragma unroll
  for (int a = 0; a < D; ++a) {
    if (GATHER != 2 || P[a] != P0[a]) nodes.mom[a * nn + i] = P[a];  // (the re-map's pass rarely changes it)
    if (!skip_mom_nt) nodes.mom_nt[a * nn + i] = Q[a];
  }
  if (clamp) clamp[i] = (uint8_t)cbits;
  const bool live = m > prm.small_mass_cutoff;
  float vnt[3] = {0.f, 0.f, 0.f}, dv[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    vnt[a] = live ? Q[a] / m : 0.f;
    const float v = live ? P[a] / m : 0.f;
    dv[a] = vnt[a] - v;
  }
  store_node_vel<D>(nodes.vel, i, vnt, dv);
}

// MODE 0: USL G2P (usl_inline.h:245-332) + return map.
// MODE 1: MUSL first map: x, v into slot j of `out` (musl_kernels.cuh:33-60).
// MODE 2: MUSL second map: L, F, V from the re-mapped velocities + return map.
// 3D gathers read node rows staged in LDS per workgroup (see
// g2p_gather_staged); 1D/2D gathers read the node records through L2.
constexpr int kG2PThreads = 256;
// LDS node staging of the 3D G2P. A workgroup's 256 particles are
// consecutive in cell order, so they fall into a few runs: consecutive
// particles with the same y and z bins whose x bins do not decrease and stay
// within one 64-aligned block. A run's windows lie in 4 x 4 node rows (y, z
// bins - 1 .. + 2) over its x range - 1 .. + 2: at most 16 x 67 nodes. The
// runs are staged in order, as many per round as kG2PStageNodes holds (one
// round for the usual ten cells of one or two x rows at 27 particles per
// cell), and every particle gathers from LDS. A staged node is the clamped
// grid node its slot names: entries outside the grid have zero weight and
// read a finite value.
constexpr int kG2PStageNodes = 1088;  // one run of the widest x range (16 x 67 nodes) always fits
static_assert(kG2PStageNodes >= 16 * (64 + 3), "a run spans at most 64 x bins");
struct G2PRunTable {
  int y[kG2PThreads], z[kG2PThreads], x0[kG2PThreads], x1[kG2PThreads], base[kG2PThreads];
  int wave_sum[kG2PThreads / 64];
};
template <bool WANT_DV> constexpr int g2p_stage_bytes() {
  return kG2PStageNodes * (16 + (WANT_DV ? 8 : 0)) + (int)sizeof(G2PRunTable);
}

// Inclusive sum of v over the workgroup's threads in order; the total goes to
// *total. Synchronises the workgroup (wave_sum is rewritten on every call: a
// workgroup barrier must separate two calls).
__device__ inline int block_inclusive_sum(int v, int *wave_sum, int *total) {
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  if (lane == 63) wave_sum[wv] = v;
  lds_barrier();
  int before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < kG2PThreads / 64; ++k) {
    const int c = wave_sum[k];
    before += k < wv ? c : 0;
    all += c;
  }
  *total = all;
  return v + before;
}

// Gathers v_nt (and dv with WANT_DV, L with WANT_L) of the particles of lanes
// 0 .. nv - 1 (weights w) through the LDS staging `lds`
// (g2p_stage_bytes<WANT_DV>() bytes). Every thread of the workgroup calls it.
template <int D, int SF, bool WANT_DV, bool WANT_L = true>
__device__ inline void g2p_gather_staged(const pmpm_grid &g, const pmpm_nodes &nodes, const PW<D, SF> &w, int nv,
                                         char *lds, float *vinc, float *dvinc, float *L) {
  static_assert(D == 3, "3D staging");
  constexpr int CAP = kG2PStageNodes;
  float4 *box4 = reinterpret_cast<float4 *>(lds);
  float2 *box2 = reinterpret_cast<float2 *>(lds + CAP * 16);
  G2PRunTable &R = *reinterpret_cast<G2PRunTable *>(lds + CAP * (16 + (WANT_DV ? 8 : 0)));
  int *rb = reinterpret_cast<int *>(lds);  // lane bins [3][256], in box4's space before staging
  const int t = (int)threadIdx.x;
  const bool valid = t < nv;
  if (valid) {
#pragma unroll
    for (int a = 0; a < 3; ++a) rb[a * kG2PThreads + t] = w.bin[a];
  }
  lds_barrier();
  // does a run start at lane q (after lane q - 1)?
  auto starts_at = [&](int q) {
    const int p0 = rb[q - 1], q0 = rb[q];
    return rb[kG2PThreads + q - 1] != rb[kG2PThreads + q] || rb[2 * kG2PThreads + q - 1] != rb[2 * kG2PThreads + q] ||
           q0 < p0 || (q0 >> 6) != (p0 >> 6);
  };
  bool start = false, end = false;
  if (valid) {
    start = t == 0 || starts_at(t);
    end = t == nv - 1 || starts_at(t + 1);
  }
  int nruns = 0;
  const int k = block_inclusive_sum(start ? 1 : 0, R.wave_sum, &nruns) - 1;
  if (start) {
    R.y[k] = w.bin[1];
    R.z[k] = w.bin[2];
    R.x0[k] = w.bin[0];
  }
  if (end) R.x1[k] = w.bin[0];
  lds_barrier();
  const int cnt = t < nruns ? 16 * (R.x1[t] - R.x0[t] + 4) : 0;
  int all = 0;
  const int incl = block_inclusive_sum(cnt, R.wave_sum, &all);
  if (t < nruns) R.base[t] = incl - cnt;
  lds_barrier();
  const int myk = valid ? k : -1;
  for (int k0 = 0; k0 < nruns;) {
    const int b0 = R.base[k0];
    int k1 = k0 + 1;
    while (k1 < nruns && R.base[k1] + 16 * (R.x1[k1] - R.x0[k1] + 4) - b0 <= CAP) ++k1;
    const int tot = R.base[k1 - 1] + 16 * (R.x1[k1 - 1] - R.x0[k1 - 1] + 4) - b0;
    for (int q = t; q < tot; q += kG2PThreads) {
      int kk = k0;
      while (kk + 1 < k1 && R.base[kk + 1] - b0 <= q) ++kk;
      const int X = R.x1[kk] - R.x0[kk] + 4, qq = q - (R.base[kk] - b0);
      const int row = qq / X, x = qq - row * X;  // row = sz * 4 + sy
      const int ix = min(max(R.x0[kk] - 1 + x, 0), g.num_cells[0] - 1);
      const int iy = min(max(R.y[kk] - 1 + (row & 3), 0), g.num_cells[1] - 1);
      const int iz = min(max(R.z[kk] - 1 + (row >> 2), 0), g.num_cells[2] - 1);
      const uint32_t node = (uint32_t)ix + (uint32_t)g.num_cells[0] * ((uint32_t)iy + (uint32_t)g.num_cells[1] * (uint32_t)iz);
      const float4 *rec = reinterpret_cast<const float4 *>(nodes.vel + 8 * (size_t)node);
      box4[q] = rec[0];
      if (WANT_DV) {
        const float4 b = rec[1];
        box2[q] = make_float2(b.x, b.y);
      }
    }
    lds_barrier();
    if (myk >= k0 && myk < k1) {
      const int off = R.base[myk] - b0, X = R.x1[myk] - R.x0[myk] + 4;
      NodeSrc src{nodes.vel, box4 + off, box2 + off, {1, X, 4 * X}, {R.x0[myk] - 1, 0, 0}};
      gather_grid<D, SF, WANT_DV, WANT_L, true>(g, src, w, vinc, dvinc, L);
    }
    k0 = k1;
    lds_barrier();  // the next round overwrites the staging
  }
}

template <int D, int SF, int MODE>
__global__ __launch_bounds__(kG2PThreads) void g2p_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles in,
                                                          pmpm_particles out, pmpm_spatial part, pmpm_nodes nodes,
                                                          int reorder) {
  static_assert(MODE >= 0 && MODE <= 2, "G2P modes: USL (0), MUSL first map (1), MUSL second map (2)");
  constexpr bool kV = MODE != 2, kL = MODE != 1;  // what the gather sums
  const int n = in.n;
  const int j = blockIdx.x * kG2PThreads + threadIdx.x;
  const bool valid = j < n;
  if (D != 3 && !valid) return;  // the 3D workgroup synchronises below
  const int nn = g.num_cells_total;
  const int src = valid ? part.sorted[j] : 0;
  const int dst = reorder ? j : src;
  PW<D, SF> w;
  float xp[3];
  if (valid) particle_weights<D, SF>(prm, g, in.x, n, src, w, xp);
  // The USL pass loads the particle's fields before the gather, whose barriers
  // wait for LDS only: their latency passes behind it (3,276,800 particles:
  // 245 -> 223 us). The MUSL second map loads them after it: its occupancy is
  // worth more (1,080,000 particles: 65 us so, 70 us the other way).
  float v0[3] = {0.f, 0.f, 0.f}, Fo[9], vol0 = 0.f, mass = 0.f;
  int color = 0;
  uint8_t pf = 0;
  Sym s = sym_zero(), eps = sym_zero();
  auto load_fields = [&]() {
#pragma unroll
    for (int k = 0; k < D * D; ++k) Fo[k] = in.F[k * n + src];
    vol0 = in.volume0[src];
    mass = in.mass[src];
    color = in.color[src];
    pf = in.flags[src];
    s = load_sym(in.stress, n, src);
  };
  if (valid && MODE != 2) {
#pragma unroll
    for (int a = 0; a < D; ++a) v0[a] = in.v[a * n + src];
  }
  if (valid && MODE == 0) load_fields();
  float vinc[3] = {0.f, 0.f, 0.f}, dvinc[3] = {0.f, 0.f, 0.f};
  float L[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if constexpr (D == 3) {
    __shared__ __attribute__((aligned(16))) char lds[g2p_stage_bytes<kV>()];
    const int nv = min(n - (int)blockIdx.x * kG2PThreads, kG2PThreads);
    g2p_gather_staged<D, SF, kV, kL>(g, nodes, w, nv, lds, vinc, dvinc, L);
    if (!valid) return;
  } else {
    gather_grid<D, SF, kV, kL>(g, node_src(g, nodes), w, vinc, dvinc, L);
  }
  if (MODE != 2) {
    // MODE 1 writes slot j of `out` (cell order), as the second map reads it
    const int to = MODE == 1 ? j : dst;
    const float am = (float)(1.0 - (double)prm.alpha);
#pragma unroll
    for (int a = 0; a < D; ++a) {
      out.v[a * n + to] = am * vinc[a] + prm.alpha * (v0[a] + dvinc[a]);
      out.x[a * n + to] = xp[a] + prm.dt * vinc[a];
    }
    if (MODE == 1) return;
  }
  if (MODE == 2) load_fields();
  // F = (I + L dt) F, V = det(F) V0
  float Fn[9];
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = 0; b < D; ++b) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) acc += ((a == k ? 1.f : 0.f) + L[3 * a + k] * prm.dt) * Fo[k * D + b];
      Fn[a * D + b] = acc;
    }
  const float vol = det_dd<D>(Fn) * vol0;
#pragma unroll
  for (int k = 0; k < D * D; ++k) out.F[k * n + dst] = Fn[k];
  out.volume[dst] = vol;
  if (out.L) {
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int b = 0; b < D; ++b) out.L[(a * D + b) * n + dst] = L[3 * a + b];
  }
  // return map of the particle's material
  if (in.eps_e) eps = load_sym(in.eps_e, n, src);
  Sym sref = sym_zero();
  if (in.stress_ref && color < prm.num_materials && (prm.materials[color].flags & PMPM_MATF_HAS_STRESS_REF))
    sref = load_sym(in.stress_ref, n, src);
  return_map<D>(prm, color, pf, L, mass, vol, vol0, sref, s, eps);
  store_sym(out.stress, n, dst, s);
  if (out.eps_e) store_sym(out.eps_e, n, dst, eps);
  if (reorder) {
    out.mass[dst] = mass;
    out.volume0[dst] = vol0;
    out.color[dst] = (uint8_t)color;
    out.flags[dst] = pf;
    out.id[dst] = in.id[src];
    // reference stresses only matter (and only travel) when a material reads them
    bool any_ref = false;
    for (int k = 0; k < prm.num_materials; ++k) any_ref = any_ref || (prm.materials[k].flags & PMPM_MATF_HAS_STRESS_REF);
    if (any_ref && in.stress_ref && out.stress_ref) store_sym(out.stress_ref, n, dst, load_sym(in.stress_ref, n, src));
  }
}

// The return maps of the materials that run after G2P (von Mises,
// Mohr-Coulomb, modified Cam-Clay), on particle j of `out` with the L, F, V,
// stress and elastic strain G2P wrote there; the history scalars follow the
// particles into cell order here (from slot sorted[j] of `in_hist` when G2P
// reordered, from slot j in place), for every particle.
template <int D>
__global__ __launch_bounds__(256) void ext_material_kernel(pmpm_params prm, const float *__restrict__ in_hist,
                                                           pmpm_particles out, const int32_t *__restrict__ sorted,
                                                           int reorder) {
  const int n = out.n;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int src = reorder ? sorted[j] : j;
  float h0 = in_hist[src], h1 = in_hist[n + src];
  const int color = out.color[j];
  if (color < prm.num_materials && is_ext_material(prm.materials[color].kind)) {
    float L[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int b = 0; b < D; ++b) L[3 * a + b] = out.L[(a * D + b) * n + j];
    Sym s = load_sym(out.stress, n, j), eps = load_sym(out.eps_e, n, j);
    Sym sref = sym_zero();
    if (out.stress_ref && (prm.materials[color].flags & PMPM_MATF_HAS_STRESS_REF)) sref = load_sym(out.stress_ref, n, j);
    return_map_ext<D>(prm, color, L, out.volume[j], sref, s, eps, h0, h1);
    store_sym(out.stress, n, j, s);
    store_sym(out.eps_e, n, j, eps);
  }
  out.hist[j] = h0;
  out.hist[n + j] = h1;
}

// Stand-alone return map of one material from the stored velocity gradient.
template <int D>
__global__ void stress_update_kernel(pmpm_params prm, int mat_id, pmpm_particles p) {
  const int n = p.n;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int color = p.color[i];
  if (color != mat_id) return;
  float L[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = 0; b < D; ++b) L[3 * a + b] = p.L[(a * D + b) * n + i];
  Sym s = load_sym(p.stress, n, i);
  Sym eps = p.eps_e ? load_sym(p.eps_e, n, i) : sym_zero();
  Sym sref = sym_zero();
  if (p.stress_ref && (prm.materials[color].flags & PMPM_MATF_HAS_STRESS_REF)) sref = load_sym(p.stress_ref, n, i);
  return_map<D>(prm, color, p.flags[i], L, p.mass[i], p.volume[i], p.volume0[i], sref, s, eps);
  if (is_ext_material(prm.materials[color].kind)) {
    float h0 = p.hist[i], h1 = p.hist[n + i];
    return_map_ext<D>(prm, color, L, p.volume[i], sref, s, eps, h0, h1);
    p.hist[i] = h0;
    p.hist[n + i] = h1;
  }
  store_sym(p.stress, n, i, s);
  if (p.eps_e) store_sym(p.eps_e, n, i, eps);
}

// Materialised psi/dpsi in the reference's layout (shapefunction.cpp:70-142):
// window entries in the reference's table order, entries whose linear node
// index is out of range stay 0, node types of the (linear) node index.
template <int D, int SF>
__global__ void shape_function_kernel(pmpm_grid g, int types_built, const float *x, int n, float *psi, float *dpsi) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  constexpr int W = (SF == PMPM_SF_LINEAR) ? 2 : 4;
  constexpr int LO = (SF == PMPM_SF_LINEAR) ? 0 : -1;
  constexpr int NSN = (D == 1) ? W : (D == 2 ? W * W : W * W * W);
  float t[3];
  int bin[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    t[a] = cell_coord(x[a * n + i], g.origin[a], g.inv_cell_size);
    bin[a] = (int)t[a];
  }
  for (int k = 0; k < NSN; ++k) {
    int off[3] = {0, 0, 0};
    if (D == 1) off[0] = LO + k;
    else if (D == 2) { off[0] = LO + k % W; off[1] = LO + k / W; }
    else { off[2] = LO + k % W; off[0] = LO + (k / W) % W; off[1] = LO + k / (W * W); }
    int nb[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) nb[a] = bin[a] + off[a];
    const int64_t lin = lin_index(g, nb, D);
    float wgt = 0.f, gr[3] = {0.f, 0.f, 0.f};
    if (lin >= 0 && lin < g.num_cells_total) {
      int ids[3];
      node_ids<D>(g, lin, ids);
      float N[3] = {1.f, 1.f, 1.f}, dN[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int a = 0; a < D; ++a) {
        const float frac = __fsub_rn(t[a], (float)bin[a]);
        spline_eval<SF>(__fsub_rn(frac, (float)off[a]), cubic_node_type(ids[a], g.num_cells[a], types_built),
                        g.inv_cell_size, N[a], dN[a]);
      }
      if (D == 1) { wgt = N[0]; gr[0] = dN[0]; }
      else if (D == 2) { wgt = N[0] * N[1]; gr[0] = dN[0] * N[1]; gr[1] = dN[1] * N[0]; }
      else {
        wgt = N[0] * N[1] * N[2];
        gr[0] = dN[0] * N[1] * N[2];
        gr[1] = dN[1] * N[0] * N[2];
        gr[2] = dN[2] * N[0] * N[1];
      }
    }
    psi[(int64_t)i * NSN + k] = wgt;
#pragma unroll
    for (int a = 0; a < D; ++a) dpsi[((int64_t)i * NSN + k) * D + a] = gr[a];
  }
}

// ---------------------------------------------------------------------------
// host-side dispatch
// ---------------------------------------------------------------------------
#define PMPM_DISPATCH_DSF(dim, sf, FN, ...)                                       \
  switch ((dim) * 3 + (sf)) {                                                     \
    case 3: FN<1, PMPM_SF_LINEAR>(__VA_ARGS__); break;                            \
    case 4: FN<1, PMPM_SF_QUADRATIC>(__VA_ARGS__); break;                         \
    case 5: FN<1, PMPM_SF_CUBIC>(__VA_ARGS__); break;                             \
    case 6: FN<2, PMPM_SF_LINEAR>(__VA_ARGS__); break;                            \
    case 7: FN<2, PMPM_SF_QUADRATIC>(__VA_ARGS__); break;                         \
    case 8: FN<2, PMPM_SF_CUBIC>(__VA_ARGS__); break;                             \
    case 9: FN<3, PMPM_SF_LINEAR>(__VA_ARGS__); break;                            \
    case 10: FN<3, PMPM_SF_QUADRATIC>(__VA_ARGS__); break;                        \
    case 11: FN<3, PMPM_SF_CUBIC>(__VA_ARGS__); break;                            \
    default: return PMPM_ERR_INVALID;                                             \
  }

// Do virtual nodes of the tile partials land on grid nodes (the linear-index
// wrap-around, summed by the grid kernel)?
static bool wraps(const pmpm_params &prm) {
  if (!prm.wrap_quirk || prm.dim < 2) return false;
  return prm.shape_fn != PMPM_SF_CUBIC || prm.node_types_built;  // untyped cubic weights are zero
}
// The 3D P2G tiles (MfmaGeom) of a scene. A function of the grid and the
// particle count only: every pass of a step, and pmpm_step_noalloc, must agree
// on it. Small scenes take small tiles (more waves, each with a short chain of
// cells), the others larger ones (fewer nodes per cell in the slices). Small
// and large tiles, a step or adjoint step: 1,300 particles 35.5 and 37.3 us,
// 2,016: 36.5 and 38.3, 8,320: 36.6 and 38.9, 14,784: 49.9 and 51.1, 17,000:
// 73.2 and 69.8, 40,000: 46.7 and 46.4, 275,000: 101.7 and 96.0.
struct MfmaTiles { int cells, rows; };
constexpr int kSmallGridNodes = 131072, kSmallTileParticles = 16384;
static MfmaTiles mfma_tiles(const pmpm_grid &g, int n) {
  if (g.num_cells_total <= kSmallGridNodes && n <= kSmallTileParticles) return {4, 1};
  return {8, 2};
}
// Tiles of T cells and their node blocks over grid g. gather: 1: P2G (mass,
// momentum, force), 2: MUSL re-map (momentum), 3: adjoint scatter.
static TileGeom make_tiles(int dim, int sf, const pmpm_grid &g, int gather, const int *T) {
  TileGeom tg{};
  const int span = sf == PMPM_SF_LINEAR ? 2 : 4;
  for (int a = 0; a < 3; ++a) {
    tg.T[a] = a < dim ? T[a] : 1;
    tg.N[a] = a < dim ? T[a] + span - 1 : 1;
    tg.tiles[a] = a < dim ? (int)ceil_div(g.num_cells[a], T[a]) : 1;
  }
  tg.nv = gather == 2 ? dim : (gather == 3 ? 2 * dim : 1 + 2 * dim);
  return tg;
}
static TileGeom mfma_tile_geom(int sf, const pmpm_grid &g, int gather, MfmaTiles m) {
  const int T[3] = {m.cells, m.rows, 4};
  return make_tiles(3, sf, g, gather, T);
}
template <int D, int SF> TileGeom row_tile_geom(const pmpm_grid &g, int gather) {
  const int T[3] = {RowGeom<D, SF>::CELLS, RowGeom<D, SF>::ROWS, 1};
  return make_tiles(D, SF, g, gather, T);
}
// M(D, Tiles<..>) for the tiles of tg: 1D and 2D, 3D.
#define PMPM_WITH_ROWS(D, tg, M)                                                      \
  if ((tg).N[0] - (tg).T[0] == 1) {                                                   \
    M(D, Tiles<D, 2, RowGeom<D, PMPM_SF_LINEAR>::CELLS, RowGeom<D, PMPM_SF_LINEAR>::ROWS>); \
  } else {                                                                            \
    M(D, Tiles<D, 4, RowGeom<D, PMPM_SF_CUBIC>::CELLS, RowGeom<D, PMPM_SF_CUBIC>::ROWS>);   \
  }
#define PMPM_WITH_TILES3(tg, M)                      \
  if ((tg).N[0] - (tg).T[0] == 1) {                  \
    if ((tg).T[0] == 4) { M(3, Tiles<3, 2, 4, 1>); } \
    else { M(3, Tiles<3, 2, 8, 2>); }                \
  } else {                                           \
    if ((tg).T[0] == 4) { M(3, Tiles<3, 4, 4, 1>); } \
    else { M(3, Tiles<3, 4, 8, 2>); }                \
  }
// The tiles of a P2G pass over n particles (gather: TileGeom::gather, or 3 for
// the adjoint scatter).
static TileGeom tile_geom(const pmpm_params &prm, const pmpm_grid &g, int gather, int n) {
  switch (prm.dim * 3 + prm.shape_fn) {
    case 3: return row_tile_geom<1, PMPM_SF_LINEAR>(g, gather);
    case 4: return row_tile_geom<1, PMPM_SF_QUADRATIC>(g, gather);
    case 5: return row_tile_geom<1, PMPM_SF_CUBIC>(g, gather);
    case 6: return row_tile_geom<2, PMPM_SF_LINEAR>(g, gather);
    case 7: return row_tile_geom<2, PMPM_SF_QUADRATIC>(g, gather);
    case 8: return row_tile_geom<2, PMPM_SF_CUBIC>(g, gather);
    default: return mfma_tile_geom(prm.shape_fn, g, gather, mfma_tiles(g, n));
  }
}
static size_t tile_count(const TileGeom &tg) { return (size_t)tg.tiles[0] * tg.tiles[1] * tg.tiles[2]; }

template <int SF, int CELLS, int ROWS>
static void launch_p2g_mfma(const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &in,
                            const pmpm_particles &out, const pmpm_spatial &part, const Strays &strays, int mode,
                            float *partials, int32_t *flags, hipStream_t s, const float *rec) {
  const TileGeom mg = mfma_tile_geom(SF, g, mode + 1, MfmaTiles{CELLS, ROWS});
  const dim3 grid((unsigned)tile_count(mg)), block(256 * ROWS);
#define PMPM_MFMA(MODE, FEXT, ...)                                                                               \
  PMPM_LAUNCH((p2g_mfma_kernel<SF, MODE, CELLS, ROWS, FEXT>), (::pmpm::kname("p2g_mfma_kernel", {__VA_ARGS__})), \
              grid, block, 0, s, prm, g, in, out, part, strays, mg.tiles[0], mg.tiles[1], partials, flags, rec)
  if (mode == 0 && has_planar(prm)) PMPM_MFMA(0, true, (long)SF, 0L, 1L);
  else if (mode == 0) PMPM_MFMA(0, false, (long)SF, 0L);
  else if (mode == 1) PMPM_MFMA(1, false, (long)SF, 1L);
  else PMPM_MFMA(2, false, (long)SF, 2L);
#undef PMPM_MFMA
}

// mode 0: P2G, 1: MUSL first map (G2P-style) and re-map, 2: adjoint scatter of
// the records `rec` (never launched without them). 3D: the matrix-core tiles;
// 1D and 2D: tiles of rows. Without partials: every particle by itself.
template <int D, int SF>
void launch_p2g(const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &in, const pmpm_particles &out,
                const pmpm_spatial &part, const pmpm_nodes &nodes, int mode, float *partials, int32_t *flags,
                const Strays &strays, hipStream_t s, const float *rec = nullptr) {
  if (mode == 2 && !rec) return;
  if (mode == 1 && in.n > 0)
    PMPM_LAUNCH((g2p_kernel<D, SF, 1>), (::pmpm::kname("g2p_kernel", {(long)(D), (long)(SF), (long)(1)})),
                dim3((unsigned)ceil_div(in.n, kG2PThreads)), dim3(kG2PThreads), 0, s, prm, g, in, out, part, nodes, 1);
  if (!partials) {  // (the caller has cleared the tile flags)
    const dim3 grid((unsigned)ceil_div(in.n, 256)), block(256);
    if (in.n <= 0) return;
    if (mode == 0)
      PMPM_LAUNCH((p2g_direct_kernel<D, SF, 0>), (::pmpm::kname("p2g_direct_kernel", {(long)D, (long)SF, 0L})), grid,
                  block, 0, s, prm, g, in, out, part, strays, has_planar(prm) ? 1 : 0);
    else
      PMPM_LAUNCH((p2g_direct_kernel<D, SF, 1>), (::pmpm::kname("p2g_direct_kernel", {(long)D, (long)SF, 1L})), grid,
                  block, 0, s, prm, g, in, out, part, strays, 0);
    return;
  }
  if constexpr (D == 3) {
    if (mfma_tiles(g, in.n).cells == 4)
      launch_p2g_mfma<SF, 4, 1>(prm, g, in, out, part, strays, mode, partials, flags, s, rec);
    else
      launch_p2g_mfma<SF, 8, 2>(prm, g, in, out, part, strays, mode, partials, flags, s, rec);
  } else {
    const TileGeom tg = row_tile_geom<D, SF>(g, mode + 1);
    const dim3 grid((unsigned)tile_count(tg)), block(RowGeom<D, SF>::THREADS);
#define PMPM_ROWS(MODE, FEXT, ...)                                                                                 \
  PMPM_LAUNCH((p2g_rows_kernel<D, SF, MODE, FEXT>), (::pmpm::kname("p2g_rows_kernel", {(long)D, __VA_ARGS__})),    \
              grid, block, 0, s, prm, g, in, out, part, strays, tg.tiles[0], partials, flags, rec)
    if (mode == 0 && has_planar(prm)) PMPM_ROWS(0, true, (long)SF, 0L, 1L);
    else if (mode == 0) PMPM_ROWS(0, false, (long)SF, 0L);
    else if (mode == 1) PMPM_ROWS(1, false, (long)SF, 1L);
    else PMPM_ROWS(2, false, (long)SF, 2L);
#undef PMPM_ROWS
  }
}
template <int D, int SF>
void launch_g2p(const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &in, const pmpm_particles &out,
                const pmpm_spatial &part, const pmpm_nodes &nodes, int mode, int reorder, hipStream_t s) {
  const unsigned blocks = (unsigned)ceil_div(in.n, 256);
  if (mode == 0)
    PMPM_LAUNCH((g2p_kernel<D, SF, 0>), (::pmpm::kname("g2p_kernel", {(long)(D), (long)(SF), (long)(0)})), dim3(blocks), dim3(256), 0, s, prm, g, in, out, part, nodes, reorder);
  else
    PMPM_LAUNCH((g2p_kernel<D, SF, 2>), (::pmpm::kname("g2p_kernel", {(long)(D), (long)(SF), (long)(2)})), dim3(blocks), dim3(256), 0, s, prm, g, in, out, part, nodes, reorder);
}
template <int D, int SF>
void launch_shape(const pmpm_grid &g, int types_built, const float *x, int n, float *psi, float *dpsi, hipStream_t s) {
  PMPM_LAUNCH((shape_function_kernel<D, SF>), (::pmpm::kname("shape_function_kernel", {(long)(D), (long)(SF)})), dim3((unsigned)ceil_div(n, 128)), dim3(128), 0, s, g, types_built,
                     x, n, psi, dpsi);
}

// Workgroups of 256 threads of a pass over all nodes (pass_node).
static unsigned pass_blocks(const TileGeom &tg) {
  return (unsigned)ceil_div((int64_t)tile_count(tg) * tg.T[0] * tg.T[1] * tg.T[2], (int64_t)256);
}
// The stray sums of a P2G (mode 0), re-map (mode 1) or adjoint scatter (mode 2).
static Strays stray_sums(const pmpm_context *ctx, const pmpm_params &prm, const pmpm_grid &g, const pmpm_nodes &nodes,
                         int mode) {
  const int64_t nn = g.num_cells_total;
  if (ctx->fixed_workspace) return {nodes.mass, nodes.mom, nodes.mom_nt, ctx->stray_flags + mode};
  return {ctx->strays, ctx->strays + nn, ctx->strays + (1 + prm.dim) * nn, ctx->stray_flags + mode};
}
// gather: 0 = node arrays only, 1 = from the P2G tile partials, 2 = mom_nt from
// the MUSL re-map tile partials (ctx holds them) of a pass over n particles.
int launch_grid(pmpm_context *ctx, const pmpm_params &prm, const pmpm_grid &g, const pmpm_nodes &nodes, int finalize,
                int b0, int b1, int remap, int gather, hipStream_t s, int n, int skip_mom_nt = 0) {
  const TileGeom tg = tile_geom(prm, g, gather, n);
  const unsigned blocks = pass_blocks(tg);
  const Strays strays = gather ? stray_sums(ctx, prm, g, nodes, gather - 1) : Strays{};
  const float *partials = gather ? ctx->partials : nullptr;
  const int32_t *flags = gather ? ctx->tile_flags : nullptr;
  // the clamp record of a pass that applies node conditions (not the MUSL
  // re-map pass), for pmpm_adjoint_step
  uint8_t *clamp = nullptr;
  if (!remap && b1 > b0)
    clamp = nodes.clamp ? nodes.clamp : (ctx ? reinterpret_cast<uint8_t *>(ctx->clamp_mask) : nullptr);

  // with the wrap-around: the workgroups of the nodes it can reach
  const int targets = !gather || !wraps(prm) ? 0 : (prm.dim == 2 ? wrap_target_count<2>(g) : wrap_target_count<3>(g));
  const int nwrap = (int)ceil_div((int64_t)targets * kImageLanes, 256);
#define PMPM_GRID_LAUNCH(...)                                                                                          \
  PMPM_LAUNCH((grid_kernel<__VA_ARGS__>), (::pmpm::kname("grid_kernel", {(long)prm.dim}) + " gather " + std::to_string(gather)), \
              dim3(blocks + (unsigned)nwrap), dim3(256), 0, s, prm, g, nodes, finalize, b0, b1, remap, tg, partials, flags,      \
              skip_mom_nt, clamp, nwrap, strays)
#define PMPM_GRID_GATHER(D, ...)                                 \
  if (gather == 0) PMPM_GRID_LAUNCH(D, 0, __VA_ARGS__);          \
  else if (gather == 1) PMPM_GRID_LAUNCH(D, 1, __VA_ARGS__);     \
  else PMPM_GRID_LAUNCH(D, 2, __VA_ARGS__)
  if (prm.dim == 1) { PMPM_WITH_ROWS(1, tg, PMPM_GRID_GATHER) }
  else if (prm.dim == 2) { PMPM_WITH_ROWS(2, tg, PMPM_GRID_GATHER) }
  else if (prm.dim == 3) { PMPM_WITH_TILES3(tg, PMPM_GRID_GATHER) }
  else return PMPM_ERR_INVALID;
#undef PMPM_GRID_GATHER
#undef PMPM_GRID_LAUNCH
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

bool params_ok(const pmpm_params *prm) {
  if (!(prm && prm->dim >= 1 && prm->dim <= 3 && prm->shape_fn >= 0 && prm->shape_fn <= 2 &&
        prm->num_materials >= 0 && prm->num_materials <= PMPM_MAX_MATERIALS && prm->num_bcs >= 0 &&
        prm->num_bcs <= PMPM_MAX_BCS))
    return false;
  for (int k = 0; k < prm->num_bcs; ++k) {  // a body force reads its node arrays
    const pmpm_bc &bc = prm->bcs[k];
    if (bc.kind == PMPM_BC_BODY_FORCE && (!bc.values || !bc.mask || bc.i[0] < 0 || bc.i[0] > 2)) return false;
  }
  return true;
}
static bool particles_ok(const pmpm_particles *p) {
  return p && p->n >= 0 &&
         (p->n == 0 || (p->x && p->v && p->stress && p->F && p->mass && p->volume && p->volume0 && p->color &&
                        p->flags && p->id));
}

TileSizes p2g_workspace(const pmpm_params &prm, const pmpm_grid &g, int n) {
  const TileGeom tg = tile_geom(prm, g, 1, n);
  TileSizes w;
  w.flags = tile_count(tg);
  w.partials = w.flags * tg.nv * (size_t)tg.N[0] * tg.N[1] * tg.N[2];
  w.clamp = ((size_t)g.num_cells_total + 3) / 4;
  return w;
}
static int reserve_tiles(pmpm_context *ctx, const pmpm_params &prm, const pmpm_grid &g, hipStream_t s) {
  if (ctx->fixed_workspace) return ctx->partials ? PMPM_OK : zero_fill(ctx->tile_flags, (int64_t)ctx->tile_cap.flags, s);
  // (any particle count: a small grid's passes use either tiles)
  TileSizes w = p2g_workspace(prm, g, 0);
  const TileSizes large = p2g_workspace(prm, g, kSmallTileParticles + 1);
  w.partials = std::max(w.partials, large.partials);
  w.flags = std::max(w.flags, large.flags);
  w.strays = (size_t)g.num_cells_total * (1 + 2 * prm.dim);
  int rc = ensure_tiles(ctx, w);
  if (rc != PMPM_OK) return rc;
  // the stray sums are zero whenever no pass is under way
  ZeroLists z{};
  z.add(ctx->strays, (int64_t)ctx->tile_cap.strays);
  return clear_on_stream(z, ctx->strays_clear, s);
}

// Scatter into the tile partials (and the stray sums); a grid_kernel pass with
// gather = 1 completes the P2G. (zeroed: the caller has already cleared the
// stray flag)
int do_p2g(pmpm_context *ctx, const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &p,
           const pmpm_spatial &part, const pmpm_nodes &nodes, hipStream_t s, bool zeroed = false) {
  int rc = reserve_tiles(ctx, prm, g, s);
  if (rc != PMPM_OK) return rc;
  if (!zeroed && (rc = zero_fill(ctx->stray_flags, 1, s)) != PMPM_OK) return rc;
  PMPM_DISPATCH_DSF(prm.dim, prm.shape_fn, launch_p2g, prm, g, p, p, part, nodes, 0, ctx->partials, ctx->tile_flags,
                    stray_sums(ctx, prm, g, nodes, 0), s);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

// True when a material of the list runs after G2P; then the particles must
// store L, the elastic strain and the history scalars.
static bool has_ext_material(const pmpm_params &prm) {
  for (int k = 0; k < prm.num_materials; ++k)
    if (is_ext_material(prm.materials[k].kind)) return true;
  return false;
}
static bool ext_buffers_ok(const pmpm_params &prm, const pmpm_particles &p) {
  return !has_ext_material(prm) || p.n == 0 || (p.L && p.eps_e && p.hist);
}

int do_g2p(const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &in, const pmpm_particles &out,
           const pmpm_spatial &part, const pmpm_nodes &nodes, int mode, hipStream_t s) {
  if (in.n == 0) return PMPM_OK;
  if (!ext_buffers_ok(prm, in) || !ext_buffers_ok(prm, out)) return PMPM_ERR_INVALID;
  const int reorder = (out.F != in.F) ? 1 : 0;  // in place when F is updated in place
  PMPM_DISPATCH_DSF(prm.dim, prm.shape_fn, launch_g2p, prm, g, in, out, part, nodes, mode, reorder, s);
  PMPM_LAUNCH_CHECK();
  if (has_ext_material(prm)) {
    const unsigned blocks = (unsigned)ceil_div(in.n, 256);
    switch (prm.dim) {
      case 1: PMPM_LAUNCH(ext_material_kernel<1>, (std::string("ext_material_kernel<1>")), dim3(blocks), dim3(256), 0, s, prm, in.hist, out, part.sorted, reorder); break;
      case 2: PMPM_LAUNCH(ext_material_kernel<2>, (std::string("ext_material_kernel<2>")), dim3(blocks), dim3(256), 0, s, prm, in.hist, out, part.sorted, reorder); break;
      default: PMPM_LAUNCH(ext_material_kernel<3>, (std::string("ext_material_kernel<3>")), dim3(blocks), dim3(256), 0, s, prm, in.hist, out, part.sorted, reorder); break;
    }
    PMPM_LAUNCH_CHECK();
  }
  return PMPM_OK;
}

// First map (x, v into `out` in cell order) + re-map of m v into the tile
// partials; a grid_kernel pass with gather = 2 completes mom_nt.
// (zeroed: as do_p2g)
int do_musl_map(pmpm_context *ctx, const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &in,
                const pmpm_particles &out, const pmpm_spatial &part, const pmpm_nodes &nodes, hipStream_t s,
                bool zeroed = false) {
  int rc = reserve_tiles(ctx, prm, g, s);
  if (rc != PMPM_OK) return rc;
  if (!zeroed && (rc = zero_fill(ctx->stray_flags + 1, 1, s)) != PMPM_OK) return rc;
  PMPM_DISPATCH_DSF(prm.dim, prm.shape_fn, launch_p2g, prm, g, in, out, part, nodes, 1, ctx->partials,
                    ctx->tile_flags, stray_sums(ctx, prm, g, nodes, 1), s);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

}  // namespace pmpm

using namespace pmpm;

extern "C" int pmpm_shape_function(int32_t dim, int32_t shape_fn, int32_t node_types_built, const pmpm_grid *grid,
                                   const float *x, int32_t n, float *psi, float *dpsi, pmpm_stream_t stream) {
  if (!grid_ok(grid) || dim < 1 || dim > 3 || shape_fn < 0 || shape_fn > 2 || n < 0) return PMPM_ERR_INVALID;
  if (n == 0) return PMPM_OK;
  if (!x || !psi || !dpsi) return PMPM_ERR_INVALID;
  PMPM_DISPATCH_DSF(dim, shape_fn, launch_shape, *grid, node_types_built, x, n, psi, dpsi, (hipStream_t)stream);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

extern "C" int pmpm_p2g(pmpm_context *ctx, const pmpm_params *prm, const pmpm_grid *grid, const pmpm_particles *p,
                        const pmpm_spatial *part, pmpm_nodes *nodes, pmpm_stream_t stream) {
  if (!ctx || !params_ok(prm) || !grid_ok(grid) || !particles_ok(p) || !part || !nodes) return PMPM_ERR_INVALID;
  hipStream_t s = (hipStream_t)stream;
  int rc = do_p2g(ctx, *prm, *grid, *p, *part, *nodes, s);
  if (rc != PMPM_OK) return rc;
  // the reference's P2G ends with the cutoff and mom_nt = mom + f dt
  return launch_grid(ctx, *prm, *grid, *nodes, 1, 0, 0, 0, 1, s, p->n);
}

extern "C" int pmpm_grid_bc(const pmpm_params *prm, const pmpm_grid *grid, pmpm_nodes *nodes, int32_t bc_begin,
                            int32_t bc_end, int32_t remap_pass, pmpm_stream_t stream) {
  if (!params_ok(prm) || !grid_ok(grid) || !nodes) return PMPM_ERR_INVALID;
  if (bc_begin < 0 || bc_end > prm->num_bcs || bc_begin > bc_end) return PMPM_ERR_INVALID;
  return launch_grid(nullptr, *prm, *grid, *nodes, 0, bc_begin, bc_end, remap_pass ? 1 : 0, 0, (hipStream_t)stream, 0);
}

extern "C" int pmpm_g2p(const pmpm_params *prm, const pmpm_grid *grid, const pmpm_particles *in, pmpm_particles *out,
                        const pmpm_spatial *part, const pmpm_nodes *nodes, pmpm_stream_t stream) {
  if (!params_ok(prm) || !grid_ok(grid) || !particles_ok(in) || !particles_ok(out) || !part || !nodes) return PMPM_ERR_INVALID;
  if (out->n != in->n) return PMPM_ERR_INVALID;
  return do_g2p(*prm, *grid, *in, *out, *part, *nodes, 0, (hipStream_t)stream);
}

extern "C" int pmpm_musl_map(pmpm_context *ctx, const pmpm_params *prm, const pmpm_grid *grid,
                             const pmpm_particles *in, pmpm_particles *out, const pmpm_spatial *part,
                             pmpm_nodes *nodes, pmpm_stream_t stream) {
  if (!ctx || !params_ok(prm) || !grid_ok(grid) || !particles_ok(in) || !particles_ok(out) || !part || !nodes)
    return PMPM_ERR_INVALID;
  if (out->n != in->n || out->x == in->x) return PMPM_ERR_INVALID;
  hipStream_t s = (hipStream_t)stream;
  int rc = do_musl_map(ctx, *prm, *grid, *in, *out, *part, *nodes, s);
  if (rc != PMPM_OK) return rc;
  // mom_nt := re-mapped momentum (mass cutoff as P2G), node velocities
  return launch_grid(ctx, *prm, *grid, *nodes, 0, 0, 0, 1, 2, s, in->n);
}

extern "C" int pmpm_musl_g2p(const pmpm_params *prm, const pmpm_grid *grid, const pmpm_particles *in,
                             pmpm_particles *out, const pmpm_spatial *part, const pmpm_nodes *nodes,
                             pmpm_stream_t stream) {
  if (!params_ok(prm) || !grid_ok(grid) || !particles_ok(in) || !particles_ok(out) || !part || !nodes) return PMPM_ERR_INVALID;
  if (out->n != in->n) return PMPM_ERR_INVALID;
  return do_g2p(*prm, *grid, *in, *out, *part, *nodes, 2, (hipStream_t)stream);
}

extern "C" int pmpm_stress_update(const pmpm_params *prm, int32_t mat_id, pmpm_particles *p, pmpm_stream_t stream) {
  if (!params_ok(prm) || !particles_ok(p) || !p || (p->n > 0 && !p->L)) return PMPM_ERR_INVALID;
  if (mat_id < 0 || mat_id >= prm->num_materials) return PMPM_ERR_INVALID;
  if (!ext_buffers_ok(*prm, *p)) return PMPM_ERR_INVALID;
  if (p->n == 0) return PMPM_OK;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = (unsigned)ceil_div(p->n, 256);
  switch (prm->dim) {
    case 1: PMPM_LAUNCH(stress_update_kernel<1>, (::pmpm::kname("stress_update_kernel", {(long)(1)})), dim3(blocks), dim3(256), 0, s, *prm, mat_id, *p); break;
    case 2: PMPM_LAUNCH(stress_update_kernel<2>, (::pmpm::kname("stress_update_kernel", {(long)(2)})), dim3(blocks), dim3(256), 0, s, *prm, mat_id, *p); break;
    default: PMPM_LAUNCH(stress_update_kernel<3>, (::pmpm::kname("stress_update_kernel", {(long)(3)})), dim3(blocks), dim3(256), 0, s, *prm, mat_id, *p); break;
  }
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}

// ===========================================================================
// Adjoint of one USL step.
//
// Forward (per step):  P2G   m_i = sum w m,  P_i = sum w m v,  f_i = -sum V sigma grad w
//                      grid  Q_i = P_i + dt f_i, BCs, vnt_i = Q_i / m_i, dv_i = vnt_i - P_i / m_i
//                      G2P   vpic = sum w vnt, dvp = sum w dv, L = sum grad w (x) vnt,
//                            v' = (1 - a) vpic + a (v + dvp), x' = x + dt vpic,
//                            F' = (I + dt L) F, (sigma', eps') = return map
// The adjoint runs these backwards: g2p_adjoint_kernel (per particle: return
// map VJP, F, v, and the records of the PIC/FLIP/L adjoints), the adjoint
// scatter (the P2G tiles, MODE 2) of those records to the nodes,
// grid_adjoint_kernel (per node: velocities, BCs, forward moment), and
// p2g_adjoint_kernel (per particle: gather of the node adjoints into v, sigma,
// V = det(F) V0 and x, together with the position adjoint of the G2P weights
// over the same window). The weights' position dependence enters through
// grad w and its Hessian.
// ===========================================================================
namespace pmpm {

// Second derivatives of the window weights (same entries and node types as
// particle_weights).
template <int D, int SF>
__device__ inline void window_d2(const pmpm_params &prm, const pmpm_grid &g, const PW<D, SF> &w, float d2N[3][4]) {
  constexpr int E = Spline<SF>::ENTRIES;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float frac = __fsub_rn(w.t[a], (float)w.bin[a]);
    if (SF == PMPM_SF_CUBIC && a < D) {
      float N[4], dN[4];
      cubic_axis(frac, w.bin[a], g.num_cells[a], prm.node_types_built, g.inv_cell_size, N, dN, d2N[a]);
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d2N[a][e] = 0.f;
      if (a < D && e < E) {
        const int o = w.first[a] + e;
        const int type = cubic_node_type(w.bin[a] + o, g.num_cells[a], prm.node_types_built);
        d2N[a][e] = spline_d2<SF>(__fsub_rn(frac, (float)o), type, g.inv_cell_size);
      }
    }
  }
}

// Weight, gradient and Hessian (xx, yy, zz, xy, xz, yz) of one window entry
// from per-axis values.
__device__ inline void entry_derivs(const float *N, const float *dN, const float *d2N, float &wgt, float *gr,
                                    float *H) {
  wgt = (N[0] * N[1]) * N[2];
  gr[0] = (dN[0] * N[1]) * N[2];
  gr[1] = (dN[1] * N[0]) * N[2];
  gr[2] = (dN[2] * N[0]) * N[1];
  H[0] = d2N[0] * N[1] * N[2];
  H[1] = N[0] * d2N[1] * N[2];
  H[2] = N[0] * N[1] * d2N[2];
  H[3] = dN[0] * dN[1] * N[2];
  H[4] = dN[0] * N[1] * dN[2];
  H[5] = N[0] * dN[1] * dN[2];
}

// Wave sum of v (all 64 lanes take part).
__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Per particle (cell order j, state slot src): return-map VJP, F, v, x, and
// the records (vpic adjoint, FLIP adjoint, L adjoint) for the node scatter.
template <int D, int SF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 3 ? 4 : 1))) void g2p_adjoint_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles st,
                                                          pmpm_adjoint ob, pmpm_adjoint ib, pmpm_spatial part,
                                                          pmpm_nodes nodes, float *__restrict__ rec,
                                                          float *__restrict__ pbar, int32_t *stray_flag) {
  const int n = st.n;
  const int nn = g.num_cells_total;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j == 0) *stray_flag = 0;  // of the scatter that follows
  const bool valid = j < n;
  float pb[4] = {0.f, 0.f, 0.f, 0.f};
  int color = -1;
  const int src = valid ? part.sorted[j] : 0;
  PW<D, SF> w;
  float xp[3];
  if (valid) particle_weights<D, SF>(prm, g, st.x, n, src, w, xp);
  // (loaded before the gather, whose barriers wait for LDS only, at four waves
  // per SIMD: 1,080,000 particles 123 -> 110 us)
  float xo[3] = {0.f, 0.f, 0.f}, vo[3] = {0.f, 0.f, 0.f}, Fo[9], F[9], so6[6], eo6[6], s6[6], e6[6], sr6[6];
  uint8_t pf = 0;
  if (valid) {
#pragma unroll
    for (int a = 0; a < D; ++a) {
      xo[a] = ob.x[a * n + j];
      vo[a] = ob.v[a * n + j];
    }
#pragma unroll
    for (int k = 0; k < D * D; ++k) {
      Fo[k] = ob.F[k * n + j];
      F[k] = st.F[k * n + src];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      so6[k] = ob.stress[k * n + j];
      eo6[k] = ob.eps_e ? ob.eps_e[k * n + j] : 0.f;
      s6[k] = st.stress[k * n + src];
      e6[k] = st.eps_e ? st.eps_e[k * n + src] : 0.f;
      sr6[k] = 0.f;
    }
    color = st.color[src];
    pf = st.flags[src];
  }
  float vpic[3] = {0.f, 0.f, 0.f}, dvp[3] = {0.f, 0.f, 0.f};
  float L[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if constexpr (D == 3) {  // the forward G2P's gather, node rows staged in LDS
    static_assert(kG2PThreads == 256, "the workgroup of the staged gather");
    __shared__ __attribute__((aligned(16))) char lds[g2p_stage_bytes<true>()];
    const int nv = min(n - (int)blockIdx.x * kG2PThreads, kG2PThreads);
    g2p_gather_staged<D, SF, true, true>(g, nodes, w, nv, lds, vpic, dvp, L);
  } else if (valid) {
    gather_grid<D, SF, true, true>(g, node_src(g, nodes), w, vpic, dvp, L);
  }
  if (valid) {
    // return map (stress and elastic strain pass through unless updated)
    float Lb[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, sb6[6], eb6[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) { sb6[k] = 0.f; eb6[k] = 0.f; }
    bool s_through = true, e_through = true;
    if (color < prm.num_materials) {
      const pmpm_material &m = prm.materials[color];
      if (m.kind == PMPM_MAT_LINEAR_ELASTIC && (pf & PMPM_PF_ACTIVE)) {
        le_vjp<D>(m.p, prm.dt, L, s6, so6, sb6, Lb, pb);
        s_through = false;
      } else if (m.kind == PMPM_MAT_DRUCKER_PRAGER) {
        const bool history = (m.flags & PMPM_MATF_UPDATE_HISTORY) != 0;
        if (st.stress_ref && (m.flags & PMPM_MATF_HAS_STRESS_REF))
#pragma unroll
          for (int k = 0; k < 6; ++k) sr6[k] = st.stress_ref[k * n + src];
        dp_vjp_rev<D>(m.p, m.p[4], (m.flags & PMPM_MATF_VELGRAD_IS_INCREMENT) != 0, history,
                  (m.flags & PMPM_MATF_APEX_GUARD) != 0, prm.dt, L, sr6, e6, so6, eo6, eb6, Lb, pb);
        s_through = false;  // the stress is recomputed from the strain
        e_through = !history;
      }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      if (s_through) sb6[k] += so6[k];
      if (e_through) eb6[k] += eo6[k];
    }

    // F' = (I + dt L) F
    float Fb[9];
#pragma unroll
    for (int k = 0; k < D; ++k)
#pragma unroll
      for (int b = 0; b < D; ++b) {
        float acc = 0.f;
#pragma unroll
        for (int a = 0; a < D; ++a) acc += ((a == k ? 1.f : 0.f) + prm.dt * L[3 * a + k]) * Fo[a * D + b];
        Fb[k * D + b] = acc;
      }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int k = 0; k < D; ++k) {
        float acc = 0.f;
#pragma unroll
        for (int b = 0; b < D; ++b) acc += Fo[a * D + b] * F[k * D + b];
        Lb[3 * a + k] += prm.dt * acc;
      }

    // v' = (1 - a) vpic + a (v + dvp), x' = x + dt vpic
    const float al = prm.alpha, am = (float)(1.0 - (double)prm.alpha);
    float vpb[3] = {0.f, 0.f, 0.f}, dvb[3] = {0.f, 0.f, 0.f}, xb[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < D; ++a) {
      vpb[a] = am * vo[a] + prm.dt * xo[a];
      dvb[a] = al * vo[a];
      xb[a] = xo[a];
    }
    // (the position adjoint through the weights is added by p2g_adjoint_kernel,
    // which walks the same window)

#pragma unroll
    for (int a = 0; a < D; ++a) {
      ib.x[a * n + src] = xb[a];
      ib.v[a * n + src] = al * vo[a];
      rec[a * n + j] = vpb[a];
      rec[(3 + a) * n + j] = dvb[a];
    }
#pragma unroll
    for (int k = 0; k < D * D; ++k) ib.F[k * n + src] = Fb[k];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      ib.stress[k * n + src] = sb6[k];
      if (ib.eps_e) ib.eps_e[k * n + src] = eb6[k];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) rec[(6 + k) * n + j] = Lb[k];
  }
  // material parameter adjoints: the workgroup's sum per material and
  // parameter (waves in a fixed order), reduced over workgroups in a fixed
  // order by the grid adjoint pass, so the gradient does not depend on
  // scheduling
  __shared__ float wsum[4][4 * PMPM_MAX_MATERIALS];
  const int wave = threadIdx.x >> 6;
  for (int k = 0; k < prm.num_materials; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float s = wave_sum(color == k ? pb[q] : 0.f);
      if ((threadIdx.x & 63) == 0) wsum[wave][4 * k + q] = s;
    }
  __syncthreads();
  const int e = threadIdx.x;
  if (e < 4 * prm.num_materials)
    pbar[(size_t)blockIdx.x * (4 * prm.num_materials) + e] = ((wsum[0][e] + wsum[1][e]) + wsum[2][e]) + wsum[3][e];
}

// param_bar[e] += the sum over workgroups of part[b * entries + e]: one
// workgroup per entry, each lane summing a fixed stride of workgroups, then a
// fixed tree.
__device__ inline void param_bar_reduce(const float *__restrict__ part, int groups, int entries, int e,
                                        float *__restrict__ param_bar) {
  __shared__ float red[256];
  float s = 0.f;
  for (int b = threadIdx.x; b < groups; b += 256) s += part[(size_t)b * entries + e];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) param_bar[e] += red[0];
}

// Node adjoints (mass, momentum, force) as one record per node: 8 floats in
// 2D and 3D (m, P, f, padding), 4 in 1D, so a gather reads one or two
// 16-byte vectors per node instead of 1 + 2D scalars from separate arrays.
template <int D> struct NodeAdj { static constexpr int NP = D == 1 ? 4 : 8; };
template <int D>
__device__ inline void load_node_adj(const float *__restrict__ nbar, int node, float &mb, float *Pb, float *fb) {
  const char *base = reinterpret_cast<const char *>(nbar);
  const uint32_t at = (uint32_t)node * (uint32_t)(NodeAdj<D>::NP * sizeof(float));
  float r[8];
  const float4 a = *reinterpret_cast<const float4 *>(base + at);
  r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
  if constexpr (NodeAdj<D>::NP == 8) {
    const float4 b = *reinterpret_cast<const float4 *>(base + at + 16u);
    r[4] = b.x; r[5] = b.y; r[6] = b.z; r[7] = b.w;
  }
  mb = r[0];
#pragma unroll
  for (int a2 = 0; a2 < D; ++a2) {
    Pb[a2] = r[1 + a2];
    fb[a2] = r[1 + D + a2];
  }
}
template <int D>
__device__ inline void store_node_adj(float *__restrict__ nbar, int node, float mb, const float *Pb, const float *fb) {
  float r[8] = {mb, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    r[1 + a] = Pb[a];
    r[1 + D + a] = fb[a];
  }
  float4 *p = reinterpret_cast<float4 *>(nbar + (size_t)NodeAdj<D>::NP * node);
  p[0] = make_float4(r[0], r[1], r[2], r[3]);
  if constexpr (NodeAdj<D>::NP == 8) p[1] = make_float4(r[4], r[5], r[6], r[7]);
}

// Per node: adjoints of the node velocities (scattered in the tile partials)
// -> adjoints of mass, moment and force. Boundary conditions in reverse list
// order with the forward's active sets, which the forward grid pass recorded
// per node in `clamp` (components a NodeDomain condition set to zero). The
// launch's first `entries` workgroups sum the material parameters' adjoints
// that g2p_adjoint_kernel left per workgroup in `pb` (a launch of their own was
// 4 us of a small scene's 33).
template <int D, class TG>
__global__ __launch_bounds__(256) void grid_adjoint_kernel(pmpm_params prm, pmpm_grid g, pmpm_nodes nodes, TileGeom tg,
                                    const float *__restrict__ partials, const int32_t *__restrict__ flags,
                                    const uint8_t *__restrict__ clamp, float *__restrict__ nbar,
                                    const float *__restrict__ pb, int groups, int entries,
                                    float *__restrict__ param_bar, Strays strays) {
  const int nn = g.num_cells_total;
  if ((int)blockIdx.x < entries) {
    param_bar_reduce(pb, groups, entries, (int)blockIdx.x, param_bar);
    return;
  }
  int ids[3] = {0, 0, 0};
  if (!pass_node<D, TG>(g, tg, ((int)blockIdx.x - entries) * (int)blockDim.x + (int)threadIdx.x, ids)) return;
  const int i = ids[0] + (D > 1 ? g.num_cells[0] * (ids[1] + (D > 2 ? g.num_cells[1] * ids[2] : 0)) : 0);
  float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  gather_partials<D, 2 * D, TG>(tg, partials, flags, ids, acc);
  if (*strays.flag) {
#pragma unroll
    for (int k = 0; k < 2 * D; ++k) {
      acc[k] += strays.mass[(int64_t)k * nn + i];
      strays.mass[(int64_t)k * nn + i] = 0.f;
    }
  }
  const float m = nodes.mass[i];
  float mb = 0.f, Pb[3] = {0.f, 0.f, 0.f}, Qb[3] = {0.f, 0.f, 0.f}, fb[3] = {0.f, 0.f, 0.f};
  if (m > prm.small_mass_cutoff) {
    float vnt[3] = {0.f, 0.f, 0.f}, dvn[3] = {0.f, 0.f, 0.f};
    load_node_vel<D, true>(nodes.vel, i, vnt, dvn);
    const unsigned cm = clamp[i];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float vb = acc[a], db = acc[D + a];
      Qb[a] = (vb + db) / m;
      Pb[a] = -db / m;
      mb -= (vb * vnt[a] + db * dvn[a]) / m;
    }
    for (int k = prm.num_bcs - 1; k >= 0; --k) {
      const pmpm_bc &bc = prm.bcs[k];
      if (bc.kind == PMPM_BC_NODE_DOMAIN) {
        // (one NodeDomain per list: pmpm_adjoint_step checks)
#pragma unroll
        for (int a = 0; a < D; ++a) {
          if (cm & (1u << a)) Pb[a] = 0.f;
          if (cm & (8u << a)) Qb[a] = 0.f;
        }
      } else if (bc.kind == PMPM_BC_GRAVITY) {
        if (m <= 0.000000001f) continue;
        // Q += g m dt
#pragma unroll
        for (int a = 0; a < D; ++a) mb += bc.f[a] * prm.dt * Qb[a];
      }
    }
    // Q = P + dt f
#pragma unroll
    for (int a = 0; a < D; ++a) {
      Pb[a] += Qb[a];
      fb[a] = prm.dt * Qb[a];
    }
  }
  store_node_adj<D>(nbar, i, mb, Pb, fb);
}

// d det(F) / dF (row-major D x D).
template <int D> __device__ inline void cofactor(const float *F, float *C) {
  if (D == 1) { C[0] = 1.f; return; }
  if (D == 2) { C[0] = F[3]; C[1] = -F[2]; C[2] = -F[1]; C[3] = F[0]; return; }
  C[0] = F[4] * F[8] - F[5] * F[7];
  C[1] = F[5] * F[6] - F[3] * F[8];
  C[2] = F[3] * F[7] - F[4] * F[6];
  C[3] = F[2] * F[7] - F[1] * F[8];
  C[4] = F[0] * F[8] - F[2] * F[6];
  C[5] = F[1] * F[6] - F[0] * F[7];
  C[6] = F[1] * F[5] - F[2] * F[4];
  C[7] = F[2] * F[3] - F[0] * F[5];
  C[8] = F[0] * F[4] - F[1] * F[3];
}

// LDS staging of the node records the 3D adjoint P2G reads (LANES lanes per
// particle, particles consecutive in cell order): as in g2p_gather_staged, the
// workgroup's particles form runs (same y and z bins, x bins not decreasing
// and within one 32-aligned block), whose windows lie in 4 x 4 node rows over
// the run's x range - 1 .. + 2, at most 16 x 35 nodes; the runs are staged in
// rounds of at most kAdjStageNodes nodes, the node adjoint record (8 floats)
// and velocity record (8 floats) of each. A node outside the grid carries the
// adjoint of the node its linear index reaches (the wrap-around deposit's; zero
// if none, or without wrap_quirk) and zero velocities (G2P never reads it).
// gather(rec, dvz, box0, X) is called by every live thread in the round that
// holds its run: the node of window offset (ex, sy, sz) from bin - 1 is entry
// box0 + ex + X (sy + 4 sz) of rec (three float4) and dvz. Every thread of the workgroup calls this
// (barriers); `live` is false past the particles.
constexpr int kAdjStageNodes = 576;  // 16 x 36: one run always fits
static_assert(kAdjStageNodes >= 16 * (32 + 3), "a run spans at most 32 x bins");
struct AdjRunTable {
  int y[kG2PThreads], z[kG2PThreads], x0[kG2PThreads], x1[kG2PThreads], base[kG2PThreads];
  int wave_sum[kG2PThreads / 64];
};
template <int LANES, class F>
__device__ inline void adjoint_stage_rounds(const pmpm_grid &g, const pmpm_nodes &nodes,
                                            const float *__restrict__ nbar, const int *bin, bool live,
                                            bool wrap_quirk, F &&gather) {
  constexpr int CAP = kAdjStageNodes, PPB = kG2PThreads / LANES;
  // a node's 13 floats: mass and momentum adjoint, force adjoint and v.x, (v.y,
  // v.z, dv.x, dv.y); dv.z (packed so: four workgroups' staging per CU)
  __shared__ float4 s_rec[CAP * 3];
  __shared__ float s_dvz[CAP];
  __shared__ AdjRunTable R;
  static_assert(CAP * 48 >= 3 * PPB * 4, "the lane bins fit the staging");
  int(*rb)[PPB] = reinterpret_cast<int(*)[PPB]>(s_rec);  // before staging
  const int t = (int)threadIdx.x, pl = t / LANES;
  const bool lead = t % LANES == 0;  // the particle's first lane
  if (lead) {
#pragma unroll
    for (int a = 0; a < 3; ++a) rb[a][pl] = bin[a];
  }
  const int nv = __syncthreads_count(live && lead);  // live particles are a prefix
  auto starts_at = [&](int q) {
    return rb[1][q - 1] != rb[1][q] || rb[2][q - 1] != rb[2][q] || rb[0][q] < rb[0][q - 1] ||
           (rb[0][q] >> 5) != (rb[0][q - 1] >> 5);
  };
  bool start = false, end = false;
  if (live && lead) {
    start = pl == 0 || starts_at(pl);
    end = pl == nv - 1 || starts_at(pl + 1);
  }
  int nruns = 0;
  const int k = block_inclusive_sum(start ? 1 : 0, R.wave_sum, &nruns) - 1;
  if (start) {
    R.y[k] = bin[1];
    R.z[k] = bin[2];
    R.x0[k] = bin[0];
  }
  if (end) R.x1[k] = bin[0];
  lds_barrier();
  const int cnt = t < nruns ? 16 * (R.x1[t] - R.x0[t] + 4) : 0;
  int all = 0;
  const int incl = block_inclusive_sum(cnt, R.wave_sum, &all);
  if (t < nruns) R.base[t] = incl - cnt;
  lds_barrier();
  const int myk = live ? k : -1;
  const int nx = g.num_cells[0], ny = g.num_cells[1], nz = g.num_cells[2];
  for (int k0 = 0; k0 < nruns;) {  // uniform over the workgroup
    const int b0 = R.base[k0];
    int k1 = k0 + 1;
    while (k1 < nruns && R.base[k1] + 16 * (R.x1[k1] - R.x0[k1] + 4) - b0 <= CAP) ++k1;
    const int tot = R.base[k1 - 1] + 16 * (R.x1[k1 - 1] - R.x0[k1 - 1] + 4) - b0;
    for (int q = t; q < tot; q += kG2PThreads) {
      int kk = k0;
      while (kk + 1 < k1 && R.base[kk + 1] - b0 <= q) ++kk;
      const int X = R.x1[kk] - R.x0[kk] + 4, qq = q - (R.base[kk] - b0);
      const int row = qq / X, x = qq - row * X;  // row = sz * 4 + sy
      const int ix = R.x0[kk] - 1 + x, iy = R.y[kk] - 1 + (row & 3), iz = R.z[kk] - 1 + (row >> 2);
      const bool in = ix >= 0 && ix < nx && iy >= 0 && iy < ny && iz >= 0 && iz < nz;
      const int64_t lin = (int64_t)ix + (int64_t)nx * ((int64_t)iy + (int64_t)ny * (int64_t)iz);
      const bool reaches = in || (wrap_quirk && lin >= 0 && lin < g.num_cells_total);
      const size_t node = reaches ? (size_t)lin : 0;
      const float4 *ar = reinterpret_cast<const float4 *>(nbar + 8 * node);
      const float4 *vr = reinterpret_cast<const float4 *>(nodes.vel + 8 * node);
      const float4 a0 = ar[0], a1 = ar[1], v0 = vr[0], v1 = vr[1];
      // (component by component: a choice between two vectors goes through memory)
      auto keep = [](bool c, float x, float y, float z, float w) {
        return make_float4(c ? x : 0.f, c ? y : 0.f, c ? z : 0.f, c ? w : 0.f);
      };
      s_rec[3 * q] = keep(reaches, a0.x, a0.y, a0.z, a0.w);
      s_rec[3 * q + 1] = make_float4(reaches ? a1.x : 0.f, reaches ? a1.y : 0.f, reaches ? a1.z : 0.f, in ? v0.x : 0.f);
      s_rec[3 * q + 2] = keep(in, v0.y, v0.z, v0.w, v1.x);
      s_dvz[q] = in ? v1.y : 0.f;
    }
    lds_barrier();
    if (myk >= k0 && myk < k1) {
      const int off = R.base[myk] - b0, X = R.x1[myk] - R.x0[myk] + 4;
      gather(s_rec, s_dvz, off + (bin[0] - R.x0[myk]), X);
    }
    k0 = k1;
    lds_barrier();  // the next round overwrites the staging
  }
}

// Adjoint P2G of 3D scenes: p2g_adjoint_kernel's sums (below) in separable
// form, the node records staged in LDS. Per node, with the particle's factors,
//   gs = m (m_bar + v . P_bar) + v_nt . vpb + dv . dvb,  wv = L_bar v_nt - V sigma f_bar
// and the sums over the window contract x first (weights N, dN, d2N of gs, wv,
// P_bar, f_bar as each needs them), then y, then z: about 3,400 multiply-adds
// per particle instead of 4,500 with a product of three weights per entry.
// Bound by vector issue (1,080,000 particles: 225 us, of which 136 us are issue
// at three waves per SIMD; capped to 128 registers for four it spills, 272 us).
// LANES = 1: a lane per particle; 4: a lane per z layer of the window, 16: per
// row of it, for launches too small to fill the chip otherwise.
// Wrap-around entries (deposit only): a node outside the grid holds the adjoint
// of the node it reaches (see the staging), so it takes part as an ordinary
// entry wherever its weight is a product of per-axis weights: always without
// node types; with them if only x leaves the grid and the carry into y changes
// no y type, or only y leaves and the carry into z changes no z type. The
// particles of the remaining cells (the grid's edges) walk their outside
// entries one by one.
template <int SF, int LANES>
__global__ __launch_bounds__(256) void p2g_adjoint3_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles st,
                                                           pmpm_adjoint ib, pmpm_spatial part, pmpm_nodes nodes,
                                                           const float *__restrict__ nbar,
                                                           const float *__restrict__ rec) {
  constexpr int E = Spline<SF>::ENTRIES;
  constexpr bool TYPED = SF == PMPM_SF_CUBIC;
  static_assert(LANES == 1 || LANES == 4 || LANES == 16, "lanes per particle");
  const int n = st.n;
  const int j = (int)blockIdx.x * (256 / LANES) + (int)threadIdx.x / LANES, sub = (int)threadIdx.x % LANES;
  const bool live = j < n;  // a thread past the particles works on the last one and writes nothing
  const uint32_t jj = (uint32_t)(live ? j : n - 1);
  const uint32_t src = (uint32_t)part.sorted[jj];
  const float inv_h = g.inv_cell_size;
  // typed cubic: the y and z weights are formed per row from a table of the
  // span polynomials (by node type; offset 4 is past the window), which costs
  // what picking them from registers by offset would and saves 24 registers
  __shared__ __attribute__((aligned(16))) float s_poly[TYPED ? 4 * 5 * 4 : 1];
  if constexpr (TYPED) {
    if (threadIdx.x < 80) {
      const int e = (int)threadIdx.x;
      s_poly[e] = (e / 4) % 5 < 4 ? kSpanCubic[e / 20][(e / 4) % 5][e % 4] : 0.f;
    }  // (the staging's barriers come before the first use)
  }
  float t3[3], N[3][4], dN[3][4], d2N[3][4];
  int bin[3], first[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) t3[a] = cell_coord(ld32(st.x + (int64_t)a * n, src), g.origin[a], inv_h);
  bool out_axis[3] = {false, false, false};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    bin[a] = (int)t3[a];
    const float frac = __fsub_rn(t3[a], (float)bin[a]);
    first[a] = 0;
    if constexpr (TYPED) {
      first[a] = -1;
      if (a == 0) cubic_axis(frac, bin[a], g.num_cells[a], prm.node_types_built, inv_h, N[a], dN[a], d2N[a], true);
    } else {
      axis_weights<SF>(t3[a], bin[a], g.num_cells[a], 0, inv_h, first[a], N[a], dN[a]);
#pragma unroll
      for (int e = 0; e < E; ++e) d2N[a][e] = spline_d2<SF>(__fsub_rn(frac, (float)(first[a] + e)), 0, inv_h);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = bin[a] + first[a] + e;
      out_axis[a] = out_axis[a] || i < 0 || i >= g.num_cells[a];
    }
  }
  // may the outside entries take part in the separable sums?
  const bool quirk = prm.wrap_quirk != 0;
  bool joint = quirk;
  if (TYPED) {
    const bool own = t3[0] >= 0.f && t3[1] >= 0.f && t3[2] >= 0.f && bin[0] < g.num_cells[0] &&
                     bin[1] < g.num_cells[1] && bin[2] < g.num_cells[2] && g.num_cells[0] >= 4 && g.num_cells[1] >= 4;
    // (nodes bin - 2 .. bin + 3 away from the typed ones)
    const bool y_plain = bin[1] >= 4 && bin[1] <= g.num_cells[1] - 5, z_plain = bin[2] >= 4 && bin[2] <= g.num_cells[2] - 5;
    joint = quirk && own && (out_axis[0] ? !out_axis[1] && y_plain : out_axis[1] && z_plain);
  }
  const bool walk = TYPED && quirk && !joint && (out_axis[0] || out_axis[1]);
#pragma unroll
  for (int a = 0; a < (TYPED ? 1 : 3); ++a)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = bin[a] + first[a] + e;
      const bool drop = (i < 0 || i >= g.num_cells[a]) && !(joint && (a < 2 || !TYPED));
      N[a][e] = drop ? 0.f : N[a][e];
      dN[a][e] = drop ? 0.f : dN[a][e];
      d2N[a][e] = drop ? 0.f : d2N[a][e];
    }
  const float m = ld32(st.mass, src), V = ld32(st.volume, src);
  float v[3], vpb[3], dvb[3], Lb[9];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    v[a] = ld32(st.v + (int64_t)a * n, src);
    vpb[a] = ld32(rec + (int64_t)a * n, jj);
    dvb[a] = ld32(rec + (int64_t)(3 + a) * n, jj);
  }
#pragma unroll
  for (int a = 0; a < 9; ++a) Lb[a] = ld32(rec + (int64_t)(6 + a) * n, jj);
  Sym s;
  {
    const float *sg = st.stress;
    s = Sym{ld32(sg, src), ld32(sg + (int64_t)n, src), ld32(sg + 2 * (int64_t)n, src),
            ld32(sg + 3 * (int64_t)n, src), ld32(sg + 4 * (int64_t)n, src), ld32(sg + 5 * (int64_t)n, src)};
  }
  const Sym Sv{V * s.xx, V * s.yy, V * s.zz, V * s.xy, V * s.xz, V * s.yz};
  const float mv[3] = {m * v[0], m * v[1], m * v[2]};
  float xb[3] = {0.f, 0.f, 0.f}, vb[3] = {0.f, 0.f, 0.f}, G[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) G[a][b] = 0.f;
  auto pick = [](const float *a, int k) { return k == 0 ? a[0] : (k == 1 ? a[1] : (k == 2 ? a[2] : a[3])); };
  // weight, derivative and second derivative at window offset e of axis a
  auto axis_at = [&](int a, int e, float &w0, float &w1, float &w2) {
    if constexpr (TYPED) {
      const int cells = g.num_cells[a];
      const float fr = __fsub_rn(t3[a], (float)bin[a]);
      const bool left = fr < 0.f;  // t < 0: the pieces shift by one
      const float f = left ? fr + 1.f : fr;
      const int i = bin[a] - 1 + e;
      const bool out = i < 0 || i >= cells;
      const int id = a == 2 ? i : i + (i < 0 ? cells : (i >= cells ? -cells : 0));
      const int type = out && !(joint && a < 2) ? 0 : cubic_node_type(id, cells, prm.node_types_built);
      const float4 c = *reinterpret_cast<const float4 *>(&s_poly[(type * 5 + e + (left ? 1 : 0)) * 4]);
      w0 = ((c.w * f + c.z) * f + c.y) * f + c.x;
      w1 = inv_h * ((3.f * c.w * f + 2.f * c.z) * f + c.y);
      w2 = inv_h * inv_h * (6.f * c.w * f + 2.f * c.z);
    } else {
      w0 = pick(N[a], e);
      w1 = pick(dN[a], e);
      w2 = pick(d2N[a], e);
    }
  };
  // this lane's window offsets along z and y
  const int z0_lane = LANES == 1 ? 0 : (LANES == 4 ? sub : sub >> 2), z1_lane = LANES == 1 ? E : min(z0_lane + 1, E);
  const int y0_lane = LANES == 16 ? sub & 3 : 0, y1_lane = LANES == 16 ? min(y0_lane + 1, E) : E;
  adjoint_stage_rounds<LANES>(g, nodes, nbar, bin, live, quirk, [&](const float4 *nrec, const float *dvz, int box0,
                                                                   int X) {
    const int at0 = box0 + (first[0] + 1) + X * ((first[1] + 1) + 4 * (first[2] + 1));
#pragma unroll 1
    for (int sz = z0_lane; sz < z1_lane; ++sz) {
      // y-contracted sums of this layer: xb's terms by their z weight (N: yX,
      // yY; dN: yZ, zX, zY; d2N: zZ), P_bar and f_bar by theirs
      float yX = 0.f, yY = 0.f, yZ = 0.f, zX = 0.f, zY = 0.f, zZ = 0.f;
      float yP[3] = {0.f, 0.f, 0.f}, fx[3] = {0.f, 0.f, 0.f}, fy[3] = {0.f, 0.f, 0.f}, fz[3] = {0.f, 0.f, 0.f};
#pragma unroll(E > 2 || LANES == 16 ? 1 : 2)
      for (int sy = y0_lane; sy < y1_lane; ++sy) {  // (not unrolled: the next rows' records would fill the registers)
        const int at = at0 + X * (sy + 4 * sz);
        float g0 = 0.f, g1 = 0.f, wx1 = 0.f, wx2 = 0.f, wy0 = 0.f, wy1 = 0.f, wz0 = 0.f, wz1 = 0.f;
        float P0[3] = {0.f, 0.f, 0.f}, f0[3] = {0.f, 0.f, 0.f}, f1[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int ex = 0; ex < E; ++ex) {
          const float4 a0 = nrec[3 * (at + ex)], a1 = nrec[3 * (at + ex) + 1], u = nrec[3 * (at + ex) + 2];
          const float P[3] = {a0.y, a0.z, a0.w}, f[3] = {a1.x, a1.y, a1.z};
          const float vn[3] = {a1.w, u.x, u.y}, dv[3] = {u.z, u.w, dvz[at + ex]};
          float gs = m * a0.x;
#pragma unroll
          for (int a = 0; a < 3; ++a) gs += mv[a] * P[a];
#pragma unroll
          for (int a = 0; a < 3; ++a) gs += vpb[a] * vn[a];
#pragma unroll
          for (int a = 0; a < 3; ++a) gs += dvb[a] * dv[a];
          const float wx = Lb[0] * vn[0] + Lb[1] * vn[1] + Lb[2] * vn[2] - (Sv.xx * f[0] + Sv.xy * f[1] + Sv.xz * f[2]);
          const float wy = Lb[3] * vn[0] + Lb[4] * vn[1] + Lb[5] * vn[2] - (Sv.xy * f[0] + Sv.yy * f[1] + Sv.yz * f[2]);
          const float wz = Lb[6] * vn[0] + Lb[7] * vn[1] + Lb[8] * vn[2] - (Sv.xz * f[0] + Sv.yz * f[1] + Sv.zz * f[2]);
          const float n0 = N[0][ex], n1 = dN[0][ex], n2 = d2N[0][ex];
          g0 += n0 * gs; g1 += n1 * gs;
          wx1 += n1 * wx; wx2 += n2 * wx;
          wy0 += n0 * wy; wy1 += n1 * wy;
          wz0 += n0 * wz; wz1 += n1 * wz;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            P0[a] += n0 * P[a];
            f0[a] += n0 * f[a];
            f1[a] += n1 * f[a];
          }
        }
        float y0, y1, y2;
        axis_at(1, sy, y0, y1, y2);
        yX += y0 * (g1 + wx2) + y1 * wy1;
        yY += y1 * (g0 + wx1) + y2 * wy0;
        yZ += y0 * (g0 + wx1) + y1 * wy0;
        zX += y0 * wz1;
        zY += y1 * wz0;
        zZ += y0 * wz0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          yP[a] += y0 * P0[a];
          fx[a] += y0 * f1[a];
          fy[a] += y1 * f0[a];
          fz[a] += y0 * f0[a];
        }
      }
      float z0, z1, z2;
      axis_at(2, sz, z0, z1, z2);
      xb[0] += z0 * yX + z1 * zX;
      xb[1] += z0 * yY + z1 * zY;
      xb[2] += z1 * yZ + z2 * zZ;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        vb[a] += z0 * yP[a];
        G[a][0] += z0 * fx[a];
        G[a][1] += z0 * fy[a];
        G[a][2] += z1 * fz[a];
      }
    }
  });
#pragma unroll
  for (int a = 0; a < 3; ++a) vb[a] *= m;
  if (walk) {
    // outside entries one by one, with the types of the node each reaches
#pragma unroll 1
    for (int e = E * (y0_lane + E * z0_lane); e < E * (y1_lane + E * (z1_lane - 1)); ++e) {  // (z, y, x)
      const int e3[3] = {e % E, (e / E) % E, e / (E * E)};
      int nb[3];
      bool inside = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        nb[a] = bin[a] + first[a] + e3[a];
        inside = inside && nb[a] >= 0 && nb[a] < g.num_cells[a];
      }
      const int64_t lin = lin_index(g, nb, 3);
      if (inside || lin < 0 || lin >= g.num_cells_total) continue;
      int ids[3];
      node_ids32<3>(g, (int)lin, ids);
      float n3[3], d3[3], h3[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int type = cubic_node_type(ids[a], g.num_cells[a], prm.node_types_built);
        const float r = __fsub_rn(__fsub_rn(t3[a], (float)bin[a]), (float)(first[a] + e3[a]));
        spline_eval<SF>(r, type, inv_h, n3[a], d3[a]);
        h3[a] = spline_d2<SF>(r, type, inv_h);
      }
      float wgt, gr[3], H[6], mb, Pb[3], fb[3];
      entry_derivs(n3, d3, h3, wgt, gr, H);
      load_node_adj<3>(nbar, (int)lin, mb, Pb, fb);
      const float gs = m * mb + mv[0] * Pb[0] + mv[1] * Pb[1] + mv[2] * Pb[2];
      const float wv[3] = {-(Sv.xx * fb[0] + Sv.xy * fb[1] + Sv.xz * fb[2]),
                           -(Sv.xy * fb[0] + Sv.yy * fb[1] + Sv.yz * fb[2]),
                           -(Sv.xz * fb[0] + Sv.yz * fb[1] + Sv.zz * fb[2])};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        vb[a] += (m * wgt) * Pb[a];
        float hs = 0.f;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          G[a][b] += fb[a] * gr[b];
          hs += H[sym_idx(a, b)] * wv[b];
        }
        xb[a] += gr[a] * gs + hs;
      }
    }
  }
  if constexpr (LANES > 1) {  // the particle's sums over its lanes; lane 0 goes on
    auto sum_lanes = [](float u) {
#pragma unroll
      for (int o = 1; o < LANES; o <<= 1) u += __shfl_xor(u, o, 64);
      return u;
    };
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      xb[a] = sum_lanes(xb[a]);
      vb[a] = sum_lanes(vb[a]);
#pragma unroll
      for (int b = 0; b < 3; ++b) G[a][b] = sum_lanes(G[a][b]);
    }
    if (sub != 0) return;
  }
  if (!live) return;
  // M_bar = -V G, V_bar = -sigma : G
  float Vb = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) Vb -= sym_at(s, a, b) * G[a][b];
  float F[9], C[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) F[k] = ld32(st.F + (int64_t)k * n, src);
  cofactor<3>(F, C);
  const float VV = Vb * ld32(st.volume0, src);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    ib.x[(int64_t)a * n + src] += xb[a];
    ib.v[(int64_t)a * n + src] += vb[a];
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) ib.F[(int64_t)k * n + src] += VV * C[k];
  // sigma is stored symmetric: an off-diagonal component feeds both entries
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = a; b < 3; ++b)
      ib.stress[(int64_t)sym_idx(a, b) * n + src] += a == b ? -V * G[a][a] : -V * G[a][b] + -V * G[b][a];
}

// Per particle: gather of the node adjoints through the P2G window (the same
// entries as the forward deposit, linear-index wrap-around included) into the
// adjoints of v, sigma, F (through V = det(F) V0) and x, plus the position
// adjoint through the G2P weights, which walk the same window:
//   xbar_c += sum_i grad_c w (vnt . vpb + dv . dvb) + sum_ab d2w/dx_c dx_a Lb_ab vnt_b
// with vpb, dvb, Lb the records g2p_adjoint_kernel wrote. The in-grid entries
// run branch-free (clamped node, zero weights outside, as gather_grid); the
// wrap-around entries of boundary particles, which only the deposit reaches,
// take a separate compact loop. Adds to ib.
// 1D and 2D (3D: p2g_adjoint3_kernel).
template <int D, int SF, int LANES>
__global__ __launch_bounds__(256) void p2g_adjoint_kernel(pmpm_params prm, pmpm_grid g, pmpm_particles st,
                                                          pmpm_adjoint ib, pmpm_spatial part, pmpm_nodes nodes,
                                                          const float *__restrict__ nbar, const float *__restrict__ rec) {
  constexpr int E = Spline<SF>::ENTRIES;
  constexpr int EY = D > 1 ? E : 1;
  const int n = st.n;
  const int nn = g.num_cells_total;
  // LANES = 1: one lane per particle, the window's y offsets in turn;
  // LANES = 4: four consecutive lanes per particle, one y offset each, the
  // particle's sums combined by shuffles, for launches too small to fill the
  // chip otherwise.
  static_assert(D < 3 && (LANES == 1 || LANES == 4), "lanes per particle");
  const int j = (int)blockIdx.x * ((int)blockDim.x / LANES) + (int)threadIdx.x / LANES;
  const int sub0 = (int)threadIdx.x % LANES;
  if (j >= n) return;  // (all lanes of a particle together)
  const int jj = j;
  const int src = part.sorted[jj];
  PW<D, SF> w;
  float xp[3];
  particle_weights<D, SF>(prm, g, st.x, n, src, w, xp);
  float d2w[3][4];
  window_d2<D, SF>(prm, g, w, d2w);
  const float m = st.mass[src], V = st.volume[src];
  float v[3] = {0.f, 0.f, 0.f}, S[3][3];
#pragma unroll
  for (int a = 0; a < D; ++a) v[a] = st.v[a * n + src];
  const Sym s = load_sym(st.stress, n, src);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) S[a][b] = sym_at(s, a, b);
  float vpb[3] = {0.f, 0.f, 0.f}, dvb[3] = {0.f, 0.f, 0.f}, Lb[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    vpb[a] = rec[a * n + jj];
    dvb[a] = rec[(3 + a) * n + jj];
  }
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = 0; b < D; ++b) Lb[3 * a + b] = rec[(6 + 3 * a + b) * n + jj];
  // per node: the deposit adjoints (m, P, f) and, for the G2P weights, the
  // node velocities; G = sum f (x) grad w gives the stress and volume adjoints
  // after the loop
  float Sv[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) Sv[a][b] = V * S[a][b];
  float vb[3] = {0.f, 0.f, 0.f}, xb[3] = {0.f, 0.f, 0.f}, G[3][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f},
                                                                       {0.f, 0.f, 0.f}};
  // one entry's contributions (g2p = 1 adds the G2P weights' position term)
  auto entry = [&](int node, const float *N3, const float *dN3, const float *d2N3, bool g2p) {
    float wgt, gr[3], H[6];
    entry_derivs(N3, dN3, d2N3, wgt, gr, H);
    float mb, Pb[3] = {0.f, 0.f, 0.f}, fb[3] = {0.f, 0.f, 0.f};
    load_node_adj<D>(nbar, node, mb, Pb, fb);
    // gs: the weight's scalar factor; wv = L_bar v_nt - V sigma^T f_bar
    float gs = mb, wv[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < D; ++a) gs += v[a] * Pb[a];
    gs *= m;
#pragma unroll
    for (int b = 0; b < D; ++b)
#pragma unroll
      for (int a = 0; a < D; ++a) wv[b] -= Sv[a][b] * fb[a];
    if (g2p) {
      float vnt[3] = {0.f, 0.f, 0.f}, dvn[3] = {0.f, 0.f, 0.f};
      load_node_vel<D, true>(nodes.vel, node, vnt, dvn);
#pragma unroll
      for (int b = 0; b < D; ++b) gs += vnt[b] * vpb[b] + dvn[b] * dvb[b];
#pragma unroll
      for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) wv[a] += Lb[3 * a + b] * vnt[b];
    }
    const float mw = m * wgt;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      vb[a] += mw * Pb[a];
#pragma unroll
      for (int b = 0; b < D; ++b) G[a][b] += fb[a] * gr[b];
    }
#pragma unroll
    for (int c = 0; c < D; ++c) {
      float hs = 0.f;
#pragma unroll
      for (int b = 0; b < D; ++b) hs += H[sym_idx(c, b)] * wv[b];
      xb[c] += gr[c] * gs + hs;
    }
  };
  // in-grid entries
  float N[3][4], dN[3][4], d2N[3][4];
  int off[3][4];
  bool leaves = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int stride = a == 0 ? 1 : g.num_cells[0];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (a < D && e < E) {
        const int i = w.bin[a] + w.first[a] + e;
        const bool ok = i >= 0 && i < g.num_cells[a];
        leaves = leaves || !ok;
        off[a][e] = min(max(i, 0), g.num_cells[a] - 1) * stride;
        N[a][e] = ok ? w.N[a][e] : 0.f;
        dN[a][e] = ok ? w.dN[a][e] : 0.f;
        d2N[a][e] = ok ? d2w[a][e] : 0.f;
      } else {
        off[a][e] = 0;
        N[a][e] = 1.f;
        dN[a][e] = 0.f;
        d2N[a][e] = 0.f;
      }
    }
  }
  // one wrap-around entry (deposit only; the wrapped node's types)
  auto wrap_entry = [&](const int *e3) {
    int nb[3] = {0, 0, 0}, offs[3] = {0, 0, 0};
    bool inside = true;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      offs[a] = w.first[a] + e3[a];
      nb[a] = w.bin[a] + offs[a];
      inside = inside && nb[a] >= 0 && nb[a] < g.num_cells[a];
    }
    const int64_t lin = lin_index(g, nb, D);
    if (inside || lin < 0 || lin >= nn) return;
    int ids[3];
    node_ids<D>(g, lin, ids);
    float n3[3] = {1.f, 1.f, 1.f}, d3[3] = {0.f, 0.f, 0.f}, h3[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const int type = cubic_node_type(ids[a], g.num_cells[a], prm.node_types_built);
      const float r = __fsub_rn(__fsub_rn(w.t[a], (float)w.bin[a]), (float)offs[a]);
      spline_eval<SF>(r, type, g.inv_cell_size, n3[a], d3[a]);
      h3[a] = spline_d2<SF>(r, type, g.inv_cell_size);
    }
    entry((int)lin, n3, d3, h3, false);
  };
  // the window's offset along y is picked by selects, so the in-grid entries
  // stay unrolled without indexing registers at run time
  auto pick = [](const auto *a, int k) { return k == 0 ? a[0] : (k == 1 ? a[1] : (k == 2 ? a[2] : a[3])); };
  {
#pragma unroll 1
    for (int sub = sub0; sub < EY; sub += LANES) {
      const int oy = pick(off[1], sub);
      const float Ny = pick(N[1], sub), dNy = pick(dN[1], sub), d2Ny = pick(d2N[1], sub);
#pragma unroll
      for (int ex = 0; ex < E; ++ex) {
        const float n3[3] = {N[0][ex], Ny, 1.f}, d3[3] = {dN[0][ex], dNy, 0.f}, h3[3] = {d2N[0][ex], d2Ny, 0.f};
        entry(off[0][ex] + oy, n3, d3, h3, true);
      }
      if (leaves && prm.wrap_quirk) {
#pragma unroll 1
        for (int e = 0; e < E; ++e) {
          const int e3[3] = {e, D > 1 ? sub : 0, 0};
          wrap_entry(e3);
        }
      }
    }
  }
  if constexpr (LANES > 1) {  // the particle's sums over its lanes; lane 0 goes on
    auto sum_lanes = [](float v) {
#pragma unroll
      for (int o = 1; o < LANES; o <<= 1) v += __shfl_xor(v, o, 64);
      return v;
    };
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      xb[a] = sum_lanes(xb[a]);
      vb[a] = sum_lanes(vb[a]);
#pragma unroll
      for (int b = 0; b < 3; ++b) G[a][b] = sum_lanes(G[a][b]);
    }
    if (sub0 != 0) return;
  }
  // M_bar = -V G, V_bar = -sigma : G
  float Mb[3][3], Vb = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      Mb[a][b] = -V * G[a][b];
      Vb -= S[a][b] * G[a][b];
    }
  float F[9], C[9];
#pragma unroll
  for (int k = 0; k < D * D; ++k) F[k] = st.F[k * n + src];
  cofactor<D>(F, C);
  const float V0 = st.volume0[src];
#pragma unroll
  for (int a = 0; a < D; ++a) {
    ib.x[a * n + src] += xb[a];
    ib.v[a * n + src] += vb[a];
  }
#pragma unroll
  for (int k = 0; k < D * D; ++k) ib.F[k * n + src] += Vb * V0 * C[k];
  // sigma is stored symmetric: an off-diagonal component feeds both entries
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = a; b < D; ++b) ib.stress[sym_idx(a, b) * n + src] += a == b ? Mb[a][a] : Mb[a][b] + Mb[b][a];
}

// Lanes per particle of the adjoint P2G: one once that fills the chip
// (kAdjointLanesWanted), four below, sixteen while a lane's chain is what counts
// (3D, windows of 3 and 4; adjoint step, cubic: 1,152 particles 54 us with four
// and 49 with sixteen, 14,784: 55 and 52, 25,088: 62 and 70).
// PMPM_ADJOINT_P2G_LANES=1, 4 or 16 in the environment overrides the choice
// (read at every launch), so the layouts can be checked against each other.
constexpr int kAdjointLanesWanted = 256 * 4 * 64 * 3;
constexpr int kAdjointRowLanes = 16384;
inline int adjoint_p2g_lanes(int n) {
  const char *e = getenv("PMPM_ADJOINT_P2G_LANES");
  if (e) {
    const int v = atoi(e);
    if (v == 1) return 1;
    if (v == 4 || v == 16) return v;
  }
  return n >= kAdjointLanesWanted ? 1 : (n > kAdjointRowLanes ? 4 : 16);
}

template <int D, int SF>
void launch_adjoint_particles(const pmpm_params &prm, const pmpm_grid &g, const pmpm_particles &st,
                              const pmpm_adjoint &ob, const pmpm_adjoint &ib, const pmpm_spatial &part,
                              const pmpm_nodes &nodes, float *rec, float *pbar, int which, const float *nbar,
                              int32_t *stray_flag, hipStream_t s) {
  if (which == 0) {
    PMPM_LAUNCH((g2p_adjoint_kernel<D, SF>), (::pmpm::kname("g2p_adjoint_kernel", {(long)(D), (long)(SF)})), dim3((unsigned)ceil_div(st.n, 256)), dim3(256), 0, s, prm, g, st, ob, ib, part, nodes,
                       rec, pbar, stray_flag);
    return;
  }
  const int lanes = std::min(adjoint_p2g_lanes(st.n), D == 3 && SF != PMPM_SF_LINEAR ? 16 : 4);
  const dim3 grid((unsigned)ceil_div(st.n, 256 / lanes));
#define PMPM_P2G_ADJOINT(KERNEL)                                                                                 \
  PMPM_LAUNCH((KERNEL), (::pmpm::kname("p2g_adjoint_kernel", {(long)(D), (long)(SF), (long)lanes})), grid, dim3(256), 0, \
              s, prm, g, st, ib, part, nodes, nbar, rec)
  if constexpr (D == 3) {
    if (lanes == 1) { auto *k = &p2g_adjoint3_kernel<SF, 1>; PMPM_P2G_ADJOINT(*k); }
    else if (lanes == 4) { auto *k = &p2g_adjoint3_kernel<SF, 4>; PMPM_P2G_ADJOINT(*k); }
    else if constexpr (SF != PMPM_SF_LINEAR) { auto *k = &p2g_adjoint3_kernel<SF, 16>; PMPM_P2G_ADJOINT(*k); }
  } else {
    if (lanes == 1) { auto *k = &p2g_adjoint_kernel<D, SF, 1>; PMPM_P2G_ADJOINT(*k); }
    else { auto *k = &p2g_adjoint_kernel<D, SF, 4>; PMPM_P2G_ADJOINT(*k); }
  }
#undef PMPM_P2G_ADJOINT
}

}  // namespace pmpm

extern "C" int pmpm_adjoint_step(pmpm_context *ctx, const pmpm_params *prm, const pmpm_grid *grid,
                                 const pmpm_particles *state, const pmpm_adjoint *out_bar, pmpm_adjoint *in_bar,
                                 float *param_bar, int32_t recompute, pmpm_spatial *part, pmpm_nodes *nodes,
                                 pmpm_stream_t stream) {
  if (!ctx || !params_ok(prm) || !grid_ok(grid) || !particles_ok(state) || !out_bar || !in_bar || !param_bar || !part ||
      !nodes || (recompute != 0 && recompute != 1))
    return PMPM_ERR_INVALID;
  const int n = state->n;
  if (n == 0) return PMPM_OK;
  if (!out_bar->x || !out_bar->v || !out_bar->F || !out_bar->stress || !in_bar->x || !in_bar->v || !in_bar->F ||
      !in_bar->stress)
    return PMPM_ERR_INVALID;
  for (int k = 0; k < prm->num_materials; ++k) {
    const int kind = prm->materials[k].kind;
    if (kind != PMPM_MAT_LINEAR_ELASTIC && kind != PMPM_MAT_DRUCKER_PRAGER) return PMPM_ERR_UNSUPPORTED;
  }
  int walls = 0;
  for (int k = 0; k < prm->num_bcs; ++k) {
    const int kind = prm->bcs[k].kind;
    if (kind != PMPM_BC_GRAVITY && kind != PMPM_BC_NODE_DOMAIN) return PMPM_ERR_UNSUPPORTED;
    walls += kind == PMPM_BC_NODE_DOMAIN;
  }
  if (walls > 1) return PMPM_ERR_UNSUPPORTED;  // the clamp record holds one condition's set
  hipStream_t s = (hipStream_t)stream;
  const pmpm_grid &g = *grid;
  const int D = prm->dim;
  // the forward step's partition, P2G and grid update (kept by the caller
  // from its own pmpm_step when recompute == 0)
  int rc;
  if (recompute) {
    if ((rc = pmpm_partition(ctx, D, grid, state->x, n, part, stream)) != PMPM_OK) return rc;
    if ((rc = do_p2g(ctx, *prm, g, *state, *part, *nodes, s)) != PMPM_OK) return rc;
    if ((rc = launch_grid(ctx, *prm, g, *nodes, 1, 0, prm->num_bcs, 0, 1, s, n)) != PMPM_OK) return rc;
  } else if ((rc = reserve_tiles(ctx, *prm, g, s)) != PMPM_OK) {
    return rc;
  }
  if ((rc = ensure_buffer(ctx->adj_rec, ctx->adj_rec_cap, (size_t)15 * n)) != PMPM_OK) return rc;
  const size_t adj_np = D == 1 ? NodeAdj<1>::NP : NodeAdj<3>::NP;
  if ((rc = ensure_buffer(ctx->adj_nodes, ctx->adj_nodes_cap, adj_np * g.num_cells_total)) != PMPM_OK)
    return rc;
  const int groups = ceil_div(n, 256), entries = 4 * prm->num_materials;
  if ((rc = ensure_buffer(ctx->adj_pb, ctx->adj_pb_cap, (size_t)groups * entries)) != PMPM_OK) return rc;
  const Strays strays = stray_sums(ctx, *prm, g, *nodes, 2);
  // G2P adjoint (material parameter adjoints per workgroup, then summed into
  // param_bar), then the scatter of its records to the nodes
  PMPM_DISPATCH_DSF(D, prm->shape_fn, launch_adjoint_particles, *prm, g, *state, *out_bar, *in_bar, *part, *nodes,
                    ctx->adj_rec, ctx->adj_pb, 0, nullptr, strays.flag, s);
  PMPM_LAUNCH_CHECK();
  PMPM_DISPATCH_DSF(D, prm->shape_fn, launch_p2g, *prm, g, *state, *state, *part, *nodes, 2, ctx->partials,
                    ctx->tile_flags, strays, s, ctx->adj_rec);
  PMPM_LAUNCH_CHECK();
  // grid adjoint, with the forward grid pass's clamp record
  const uint8_t *clamp = nodes->clamp ? nodes->clamp : reinterpret_cast<const uint8_t *>(ctx->clamp_mask);
  const TileGeom tg = tile_geom(*prm, g, 3, n);
  const unsigned nblocks = pass_blocks(tg) + (unsigned)entries;
#define PMPM_GRID_ADJOINT(...)                                                                                   \
  PMPM_LAUNCH((grid_adjoint_kernel<__VA_ARGS__>), (::pmpm::kname("grid_adjoint_kernel", {(long)D})), dim3(nblocks), \
              dim3(256), 0, s, *prm, g, *nodes, tg, ctx->partials, ctx->tile_flags, clamp, ctx->adj_nodes, ctx->adj_pb, \
              groups, entries, param_bar, strays)
  switch (D) {
    case 1: PMPM_WITH_ROWS(1, tg, PMPM_GRID_ADJOINT) break;
    case 2: PMPM_WITH_ROWS(2, tg, PMPM_GRID_ADJOINT) break;
    default: PMPM_WITH_TILES3(tg, PMPM_GRID_ADJOINT) break;
  }
#undef PMPM_GRID_ADJOINT
  PMPM_LAUNCH_CHECK();
  // P2G adjoint
  PMPM_DISPATCH_DSF(D, prm->shape_fn, launch_adjoint_particles, *prm, g, *state, *out_bar, *in_bar, *part, *nodes,
                    ctx->adj_rec, param_bar, 1, ctx->adj_nodes, strays.flag, s);
  PMPM_LAUNCH_CHECK();
  return PMPM_OK;
}
