// Forward/backward pair of the 3D engine: J(eps) and dJ/d eps over a design box by the
// discrete adjoint (time-reversed transpose) of the engine's own update.
//
// No counterpart in the reference (it has no differentiation).  The forward map of one step
// is linear in the state (E, D, H, B) plus field-independent TF/SF and source terms, so the
// adjoint of a step is the transpose of its linear part, applied in reverse order (H, then E):
//   H cells:  plain   w = cb a;                      a unchanged
//             PML     mB = aB + kp a;  w = cbc mB;   aB <- cac mB - km a;  a <- ca5 a
//             with cb = dt / (m mu0 dx), kp = (p4 / mod) / dd5, km = (m4 / mod) / dd5 (the
//             coefficients of cell_value), a = adjoint of the cell's new value;
//   E cells:  a = aE - curl_E(w_H) first (the transpose of the H curl that read E), then the
//             same per-cell rule; aH -= curl_H(w_E) is applied at the start of the next
//             (earlier) reverse step, fused with its H transpose.
// A hard point source replaces the new value of its cell, so its adjoint is dropped.
// J = sum over the last `window` steps of the sum of Ez^2 on a monitor rectangle; its
// derivative 2 Ez is added to aEz before the reverse step of each of those steps.
// The update of an E cell depends on eps only through the averaged material m inside
// cb (1/m), so dE'/dm = -(E' - E) / m on the PML-free cells of the design box, and each of
// the two eps voxels of the average receives half of it.  E before and after every step on
// the design box comes from a trace recorded by the forward run (checkpoint_every = 0), or
// from re-running each segment of checkpoint_every steps from a snapshot of the full state.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "yee_device.h"
#include "yee_internal.h"

namespace yee {

template <typename T>
struct AdjArgs
{
  StepArgs<T> a;              // forward set-up (sizes, materials, PML tables)
  T *af[6], *ad[6];           // adjoints of E/H and of D/B
  T *w[6];                    // curl weights of the current reverse step
  uint32_t src_mask;          // hard sources (adjoint dropped at src_q)
  int64_t src_q;
  const T *mon;               // recorded Ez of the monitor rectangle at this step, [x][y] (null: none)
  int mx0, my0, mnx, mny, mz;
};

// Trace box geometry: E cells [lo, lo + n) of the three components, [comp][x][y][z].
struct TraceBox
{
  int lo[3], n[3];
  __host__ __device__ int64_t cells () const { return (int64_t) n[0] * n[1] * n[2]; }
  __host__ __device__ int64_t at (int c, int x, int y, int z) const
  {
    return ((c * (int64_t) n[0] + (x - lo[0])) * n[1] + (y - lo[1])) * n[2] + (z - lo[2]);
  }
};

// Gradient of one reverse step (adj_grad): the design voxels, E on the trace box after and before it.
template <typename T>
struct GradArgs
{
  TraceBox tb;
  const T *cur, *prev;        // null: no gradient
  int lo[3], n[3];
  double *grad;
};

// (x, y, z) of element u of a box of n cells (32-bit division where it is enough).
__device__ __forceinline__ void box_cell (const int n[3], int64_t u, int &x, int &y, int &z)
{
  if ((int64_t) n[0] * n[1] * n[2] <= (int64_t) INT32_MAX)
  {
    const uint32_t v = (uint32_t) u, r = v / (uint32_t) n[2];
    z = (int) (v - r * (uint32_t) n[2]);
    x = (int) (r / (uint32_t) n[1]);
    y = (int) (r - (uint32_t) x * (uint32_t) n[1]);
    return;
  }
  z = (int) (u % n[2]);
  y = (int) ((u / n[2]) % n[1]);
  x = (int) (u / ((int64_t) n[2] * n[1]));
}

// The adjoint D/B and PML coefficients of a special cell, loaded before any store of the
// thread (the state pointers may alias as far as the compiler knows), so that every load of a
// cell is in flight at once.
template <typename T>
struct AdjOld
{
  T ad, cac, cbc, p4, m4, ca5, dd5;
};

template <typename T, int COMP>
__device__ __forceinline__ void adj_load (const AdjArgs<T> &g, int64_t q, const int p[3], bool special, AdjOld<T> &o)
{
  if (!special) return;
  const StepArgs<T> &a = g.a;
  const size_t L = (size_t) a.tab_len;
  const T *tab = a.pml + COMP * 6 * L;
  o.ad = g.ad[COMP][q];
  const Pair<T> c = gld2 (tab + 2 * p[SigAxes<COMP>::c]);
  const Pair<T> s4 = gld2 (tab + 2 * L + 2 * p[SigAxes<COMP>::s4]);
  const Pair<T> s5 = gld2 (tab + 4 * L + 2 * p[SigAxes<COMP>::s5]);
  o.cac = c.a;
  o.cbc = c.b;
  o.p4 = s4.a;
  o.m4 = s4.b;
  o.ca5 = s5.a;
  o.dd5 = s5.b;
}

template <typename T, int COMP>
__device__ __forceinline__ T adj_cell (const AdjArgs<T> &g, int64_t q, T av, T mat, bool special, const AdjOld<T> &o)
{
  const StepArgs<T> &a = g.a;
  const T modc = COMP >= 3 ? a.mu0 : a.eps0;
  if ((g.src_mask & (1u << COMP)) && q == g.src_q) av = (T) 0;
  T w;
  if (!special)
  {
    const T cb = direct_cb (a.dt, mat, modc, a.dx);
    w = av * cb;
    g.af[COMP][q] = av;
  }
  else
  {
    const Pair<T> k = pml_factors (o.p4, o.m4, mat * modc, o.dd5);
    const T mD = o.ad + k.a * av;
    w = o.cbc * mD;
    g.ad[COMP][q] = o.cac * mD - k.b * av;
    g.af[COMP][q] = o.ca5 * av;
  }
  return w;
}

// grad(v) += sum over the six E cells whose material average contains voxel v of
// aE(c) * (-(E'(c) - E(c)) / m(c)) / 2, for design voxel u.
template <typename T>
__device__ __forceinline__ void grad_voxel (const AdjArgs<T> &g, const GradArgs<T> &d, int64_t u)
{
  if (u >= (int64_t) d.n[0] * d.n[1] * d.n[2]) return;
  const StepArgs<T> &a = g.a;
  int vx, vy, vz;
  box_cell (d.n, u, vx, vy, vz);
  vx += d.lo[0];
  vy += d.lo[1];
  vz += d.lo[2];
  const int64_t sx = a.sx;
  const int sy = a.sy;
  double acc = 0;
  // (component, cell offset along that component's axis): cells c = v and c = v - e_axis
#pragma unroll
  for (int comp = 0; comp < 3; ++comp)
  {
#pragma unroll
    for (int back = 0; back < 2; ++back)
    {
      const int cx = vx - (comp == 0 ? back : 0), cy = vy - (comp == 1 ? back : 0), cz = vz - (comp == 2 ? back : 0);
      const int64_t qc = (int64_t) cx * sx + (int64_t) cy * sy + cz;
      const int64_t step = comp == 0 ? sx : (comp == 1 ? (int64_t) sy : 1);
      const T m = avg2 (a.eps[qc], a.eps[qc + step]);
      const int64_t tix = d.tb.at (comp, cx, cy, cz);
      const T de = d.cur[tix] - d.prev[tix];
      acc += (double) g.af[comp][qc] * (-(double) de / (double) m) * 0.5;
    }
  }
  d.grad[u] += acc;
}

template <typename T>
__global__ __launch_bounds__ (256) void adj_grad (AdjArgs<T> g, GradArgs<T> d)
{
  grad_voxel (g, d, (int64_t) blockIdx.x * 256 + (int) threadIdx.x);
}

// aH -= curl_H(w_E) of the previous reverse step (the transpose of the E curl that read H;
// w_E is zero before the first one), then the transpose of this step's H update (H cells of
// [1, N-1)^3; tiles as half_cell).  The blocks past the tiles' nblk add the gradient of the reverse
// step before, which reads aE (this kernel does not touch it): a launch of its own took 5 us of the
// 59 us of a 128^3 FP32 reverse step, as did one for the monitor's source (now in adj_e).
template <typename T, int MODE>
__global__ __launch_bounds__ (256) void adj_h (AdjArgs<T> g, GradArgs<T> d, int nblk)
{
  if ((int) blockIdx.x >= nblk)
  {
    grad_voxel (g, d, (int64_t) ((int) blockIdx.x - nblk) * 256 + (int) (threadIdx.y * 64 + threadIdx.x));
    return;
  }
  const StepArgs<T> &a = g.a;
  int i, j, k;
  if (!half_cell (a, i, j, k)) return;
  const int64_t sx = a.sx;
  const int sy = a.sy;
  const int64_t q = (int64_t) i * sx + (int64_t) j * sy + k;
  const int p[3] = { i, j, k };
  const bool special = MODE != 0 && is_special (a, p, 3, MODE);
  T mx = a.mu_u, my = a.mu_u, mz = a.mu_u;
  if (a.mu)
  {
    const T *m = a.mu;
    mx = avg4 (m[q], m[q + 1], m[q + sy], m[q + sy + 1]);
    my = avg4 (m[q], m[q + 1], m[q + sx], m[q + sx + 1]);
    mz = avg4 (m[q], m[q + sy], m[q + sx], m[q + sx + sy]);
  }
  const T *ex = g.w[0], *ey = g.w[1], *ez = g.w[2];
  // the H-update stencils applied to w_E (Hx: Ey BACK/FRONT, Ez DOWN/UP; cyclic)
  const T vx[4] = { ey[q], ey[q + 1], ez[q], ez[q + sy] };
  const T vy[4] = { ez[q], ez[q + sx], ex[q], ex[q + 1] };
  const T vz[4] = { ex[q], ex[q + sy], ey[q], ey[q + sx] };
  AdjOld<T> o3 {}, o4 {}, o5 {};
  adj_load<T, 3> (g, q, p, special, o3);
  adj_load<T, 4> (g, q, p, special, o4);
  adj_load<T, 5> (g, q, p, special, o5);
  const T a3 = g.af[3][q] - curl (vx), a4 = g.af[4][q] - curl (vy), a5 = g.af[5][q] - curl (vz);
  g.w[3][q] = adj_cell<T, 3> (g, q, a3, mx, special, o3);
  g.w[4][q] = adj_cell<T, 4> (g, q, a4, my, special, o4);
  g.w[5][q] = adj_cell<T, 5> (g, q, a5, mz, special, o5);
}

// aEz += 2 Ez on the monitor rectangle (interior cells), aE -= curl_E(w_H), then the transpose of the
// E update (E cells of [1, N-1)^3).
template <typename T, int MODE>
__global__ __launch_bounds__ (256) void adj_e (AdjArgs<T> g)
{
  const StepArgs<T> &a = g.a;
  int i, j, k;
  if (!half_cell (a, i, j, k)) return;
  const int64_t sx = a.sx;
  const int sy = a.sy;
  const int64_t q = (int64_t) i * sx + (int64_t) j * sy + k;
  const int p[3] = { i, j, k };
  const bool special = MODE != 0 && is_special (a, p, 3, MODE);
  const T *wx = g.w[3], *wy = g.w[4], *wz = g.w[5];
  // the E-update stencils applied to w_H (Ex: Hz DOWN/UP, Hy BACK/FRONT; cyclic)
  const T vx[4] = { wz[q - sy], wz[q], wy[q - 1], wy[q] };
  const T vy[4] = { wx[q - 1], wx[q], wz[q - sx], wz[q] };
  const T vz[4] = { wy[q - sx], wy[q], wx[q - sy], wx[q] };
  // (averaged after the last load: averages here would wait for every load before them; backward of
  // 128^3, 160 steps: FP32 17.8 ms so, 17.6 now, FP64 37.6 and 37.1)
  T m0, mx, my, mz;
  if (a.eps)
  {
    m0 = a.eps[q];
    mx = a.eps[q + sx];
    my = a.eps[q + sy];
    mz = a.eps[q + 1];
  }
  AdjOld<T> o0 {}, o1 {}, o2 {};
  adj_load<T, 0> (g, q, p, special, o0);
  adj_load<T, 1> (g, q, p, special, o1);
  adj_load<T, 2> (g, q, p, special, o2);
  const T f0 = g.af[0][q], f1 = g.af[1][q];
  T az = g.af[2][q];
  T ex = a.eps_u, ey = a.eps_u, ez = a.eps_u;
  if (a.eps)
  {
    ex = avg2 (m0, mx);
    ey = avg2 (m0, my);
    ez = avg2 (m0, mz);
  }
  const int mi = i - g.mx0, mj = j - g.my0;
  if (g.mon && k == g.mz && mi >= 0 && mi < g.mnx && mj >= 0 && mj < g.mny) az += (T) 2 * g.mon[mi * g.mny + mj];
  const T a0 = f0 - curl (vx), a1 = f1 - curl (vy), a2 = az - curl (vz);
  g.w[0][q] = adj_cell<T, 0> (g, q, a0, ex, special, o0);
  g.w[1][q] = adj_cell<T, 1> (g, q, a1, ey, special, o1);
  g.w[2][q] = adj_cell<T, 2> (g, q, a2, ez, special, o2);
}

// Copies E of the trace box (and Ez of the monitor rectangle when mon != null).
template <typename T>
__global__ void adj_record (const T *Ex, const T *Ey, const T *Ez, int64_t sx, int sy, TraceBox tb, T *slot)
{
  const int64_t u = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nc = tb.cells ();
  if (u >= nc) return;
  int x, y, z;
  box_cell (tb.n, u, x, y, z);
  x += tb.lo[0];
  y += tb.lo[1];
  z += tb.lo[2];
  const int64_t q = (int64_t) x * sx + (int64_t) y * sy + z;
  slot[u] = Ex[q];
  slot[nc + u] = Ey[q];
  slot[2 * nc + u] = Ez[q];
}

template <typename T>
__global__ void adj_monitor (const T *Ez, int64_t sx, int sy, int64_t mz, int mx0, int my0, int mnx, int mny, T *out)
{
  const int u = (int) (blockIdx.x * blockDim.x + threadIdx.x);
  if (u >= mnx * mny) return;
  const int x = mx0 + u / mny, y = my0 + u % mny;
  out[u] = Ez[(int64_t) x * sx + (int64_t) y * sy + mz];
}

// Writes the design-box values into the eps grid.
template <typename T>
__global__ void adj_set_design (T *eps, int64_t sx, int sy, int dlo0, int dlo1, int dlo2, int dn0, int dn1, int dn2,
                                const T *vals)
{
  const int64_t u = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= (int64_t) dn0 * dn1 * dn2) return;
  const int z = dlo2 + (int) (u % dn2);
  const int y = dlo1 + (int) ((u / dn2) % dn1);
  const int x = dlo0 + (int) (u / ((int64_t) dn2 * dn1));
  eps[(int64_t) x * sx + (int64_t) y * sy + z] = vals[u];
}

struct AdjointState
{
  yee_adjoint_spec sp {};
  int T = 0;
  TraceBox tb {};
  int64_t dn[3] = { 0, 0, 0 };
  int mnx = 0, mny = 0;
  std::vector<void *> allocs;
  void *af[6] = {}, *ad[6] = {}, *w[6] = {};
  void *trace = nullptr;
  int trace_slots = 0;
  void *mon = nullptr;
  double *grad = nullptr;
  void *stage = nullptr;          // design values staging (field precision)
  std::vector<void *> snap;       // checkpoint snapshots (full state + incident grids)
  std::vector<int32_t> snap_t;
  std::vector<int> snap_cur;
  size_t snap_bytes = 0;
  bool forward_done = false;
  bool last_traced = false;   // the forward recorded the trace of the last checkpoint segment
  double J = 0;
  double fwd_ms = 0, bwd_ms = 0;
};

namespace {

int adj_alloc (yee_handle *h, void **p, size_t bytes)
{
  HIP_TRY (hipMalloc (p, bytes));
  h->adj->allocs.push_back (*p);
  HIP_TRY (hipMemsetAsync (*p, 0, bytes, h->stream));
  return YEE_OK;
}

template <typename T>
AdjArgs<T> adj_args (const yee_handle *h)
{
  AdjArgs<T> g {};
  g.a = engine_args<T> (h);
  for (int c = 0; c < 6; ++c)
  {
    g.af[c] = (T *) h->adj->af[c];
    g.ad[c] = (T *) h->adj->ad[c];
    g.w[c] = (T *) h->adj->w[c];
  }
  const int64_t *p = h->cfg.point_source_pos;
  g.src_mask = h->cfg.point_source & 0x3fu;
  g.src_q = (p[0] * h->n[1] + p[1]) * h->n[2] + p[2];
  return g;
}


template <typename T>
int record (yee_handle *h, int slot)
{
  AdjointState *s = h->adj;
  const int64_t nc = s->tb.cells ();
  T *dst = (T *) s->trace + (size_t) slot * 3 * nc;
  hipLaunchKernelGGL ((adj_record<T>), dim3 ((unsigned) ((nc + 255) / 256)), dim3 (256), 0, h->stream,
                     (const T *) h->f[h->cur][0], (const T *) h->f[h->cur][1], (const T *) h->f[h->cur][2],
                     h->n[1] * h->n[2], (int) h->n[2], s->tb, dst);
  HIP_TRY (hipGetLastError ());
  return YEE_OK;
}

template <typename T>
int monitor (yee_handle *h, int slot)
{
  AdjointState *s = h->adj;
  const int nm = s->mnx * s->mny;
  hipLaunchKernelGGL ((adj_monitor<T>), dim3 ((unsigned) ((nm + 255) / 256)), dim3 (256), 0, h->stream,
                     (const T *) h->f[h->cur][2], h->n[1] * h->n[2], (int) h->n[2], s->sp.monitor_z,
                     (int) s->sp.monitor_lo[0], (int) s->sp.monitor_lo[1], s->mnx, s->mny, (T *) s->mon + (size_t) slot * nm);
  HIP_TRY (hipGetLastError ());
  return YEE_OK;
}

// Snapshot k of the full state (fields, D/B, incident grids) and its step counter.
int snapshot (yee_handle *h, int k, bool restore)
{
  AdjointState *s = h->adj;
  const size_t grid = (size_t) h->ncell * h->wsize, inc = (size_t) h->inc_len * h->wsize;
  char *base = (char *) s->snap[k];
  if (restore)
  {
    h->t = s->snap_t[k];
    h->cur = s->snap_cur[k];
  }
  else
  {
    s->snap_t[k] = h->t;
    s->snap_cur[k] = h->cur;
  }
  size_t off = 0;
  auto move = [&] (void *state, size_t bytes) -> int {
    if (!state) return YEE_OK;
    if (restore) HIP_TRY (hipMemcpyAsync (state, base + off, bytes, hipMemcpyDeviceToDevice, h->stream));
    else HIP_TRY (hipMemcpyAsync (base + off, state, bytes, hipMemcpyDeviceToDevice, h->stream));
    off += bytes;
    return YEE_OK;
  };
  int rc;
  for (int c = 0; c < 6; ++c)
  {
    if ((rc = move (h->f[h->cur][c], grid))) return rc;
    if ((rc = move (h->d[h->cur][c], grid))) return rc;
  }
  if ((rc = move (h->einc[h->inc_cur], inc))) return rc;
  if ((rc = move (h->hinc[h->inc_cur], inc))) return rc;
  if (restore)
  {
    h->inc_t = h->hist_t = h->t;   // the next step restarts the incident rows
    // the other buffer holds the wave of later steps, and a launch of incident_steps writes it only
    // as far as the wave of its own steps reaches: the launch after that would read the rest as zeros
    for (void *p : { h->einc[1 - h->inc_cur], h->hinc[1 - h->inc_cur] })
      if (p) HIP_TRY (hipMemsetAsync (p, 0, inc, h->stream));
  }
  return YEE_OK;
}

int64_t grad_blocks (const AdjointState *s) { return (s->dn[0] * s->dn[1] * s->dn[2] + 255) / 256; }

// One reverse step.  d: the gradient that the reverse step before left to do (none: cur null), done in
// this step's H launch; on return the gradient of this step.
template <typename T>
int reverse_step (yee_handle *h, int32_t t, int slot_cur, int slot_prev, GradArgs<T> &d)
{
  AdjointState *s = h->adj;
  AdjArgs<T> g = adj_args<T> (h);
  // the interior [1, N-1)^3 in 64 x 4 tiles (half_cell)
  for (int ax = 0; ax < 3; ++ax)
  {
    g.a.run_lo[ax] = 1;
    g.a.run_hi[ax] = (int) h->n[ax] - 1;
  }
  dim3 grid;
  const dim3 block (64, 4, 1);
  if (!half_tiles (g.a, 64, 4, grid)) return fail (YEE_EINVAL, "adjoint grid too large for one launch");
  const int W = s->sp.window;
  if (t >= s->T - W)
  {
    g.mon = (const T *) s->mon + (size_t) (t - (s->T - W)) * s->mnx * s->mny;
    g.mx0 = (int) s->sp.monitor_lo[0];
    g.my0 = (int) s->sp.monitor_lo[1];
    g.mnx = s->mnx;
    g.mny = s->mny;
    g.mz = (int) s->sp.monitor_z;
  }
  dim3 hgrid = grid;
  if (d.cur) hgrid.x += (unsigned) grad_blocks (s);
  if (h->mode == 1)
  {
    hipLaunchKernelGGL ((adj_h<T, 1>), hgrid, block, 0, h->stream, g, d, (int) grid.x);
    hipLaunchKernelGGL ((adj_e<T, 1>), grid, block, 0, h->stream, g);
  }
  else
  {
    hipLaunchKernelGGL ((adj_h<T, 0>), hgrid, block, 0, h->stream, g, d, (int) grid.x);
    hipLaunchKernelGGL ((adj_e<T, 0>), grid, block, 0, h->stream, g);
  }
  const int64_t nc = s->tb.cells ();
  d.tb = s->tb;
  d.cur = (const T *) s->trace + (size_t) slot_cur * 3 * nc;
  d.prev = (const T *) s->trace + (size_t) slot_prev * 3 * nc;
  for (int ax = 0; ax < 3; ++ax)
  {
    d.lo[ax] = (int) s->sp.design_lo[ax];
    d.n[ax] = (int) s->dn[ax];
  }
  d.grad = s->grad;
  HIP_TRY (hipGetLastError ());
  return YEE_OK;
}

// The gradient that the last reverse step of a segment left, before the trace is written again or read
// out (aE is the one of that step until then).
template <typename T>
int last_gradient (yee_handle *h, GradArgs<T> &d)
{
  if (!d.cur) return YEE_OK;
  hipLaunchKernelGGL ((adj_grad<T>), dim3 ((unsigned) grad_blocks (h->adj)), dim3 (256), 0, h->stream, adj_args<T> (h), d);
  HIP_TRY (hipGetLastError ());
  d.cur = nullptr;
  return YEE_OK;
}

template <typename T>
int forward_impl (yee_handle *h, const double *design, double *J)
{
  AdjointState *s = h->adj;
  int rc;
  const int64_t nd = s->dn[0] * s->dn[1] * s->dn[2];
  {
    std::vector<T> v ((size_t) nd);
    for (int64_t u = 0; u < nd; ++u)
    {
      if (!(design[u] > 0) || !std::isfinite (design[u])) return fail (YEE_EINVAL, "design eps must be positive and finite");
      v[(size_t) u] = (T) design[u];
    }
    HIP_TRY (hipMemcpyAsync (s->stage, v.data (), (size_t) nd * sizeof (T), hipMemcpyHostToDevice, h->stream));
    hipLaunchKernelGGL ((adj_set_design<T>), dim3 ((unsigned) ((nd + 255) / 256)), dim3 (256), 0, h->stream,
                       (T *) h->mat[YEE_MAT_EPS], h->n[1] * h->n[2], (int) h->n[2], (int) s->sp.design_lo[0],
                       (int) s->sp.design_lo[1], (int) s->sp.design_lo[2], (int) s->dn[0], (int) s->dn[1], (int) s->dn[2],
                       (const T *) s->stage);
    HIP_TRY (hipGetLastError ());
    HIP_TRY (hipStreamSynchronize (h->stream));
  }
  if ((rc = engine_reset (h))) return rc;
  const int K = s->sp.checkpoint_every;
  const int W = s->sp.window;
  // with checkpoints, the last segment's trace is recorded here (the backward starts with it
  // and need not re-run it)
  const int32_t t0_last = K > 0 ? ((s->T - 1 + K - 1) / K - 1) * K : 0;
  HIP_TRY (hipEventRecord (h->ev[0], h->stream));
  for (int32_t t = 0; t < s->T; ++t)
  {
    // up to the next snapshot
    if ((rc = engine_step_once (h, std::min (K == 0 ? s->T : (t + K - 1) / K * K + 1, s->T) - t))) return rc;
    if (K == 0)
    {
      if ((rc = record<T> (h, t))) return rc;
    }
    else
    {
      if (t % K == 0 && (rc = snapshot (h, t / K, false))) return rc;
      if (t >= t0_last && (rc = record<T> (h, t - t0_last))) return rc;
    }
    if (t >= s->T - W && (rc = monitor<T> (h, t - (s->T - W)))) return rc;
  }
  HIP_TRY (hipEventRecord (h->ev[1], h->stream));
  HIP_TRY (hipEventSynchronize (h->ev[1]));
  float ms = 0;
  HIP_TRY (hipEventElapsedTime (&ms, h->ev[0], h->ev[1]));
  s->fwd_ms = ms;
  const size_t nm = (size_t) s->mnx * s->mny * W;
  std::vector<T> mon (nm);
  HIP_TRY (hipMemcpy (mon.data (), s->mon, nm * sizeof (T), hipMemcpyDeviceToHost));
  // compensated (Neumaier) sum: J is differenced by finite-difference checks, where the
  // rounding of a plain sum over millions of terms would dominate
  double acc = 0, comp = 0;
  for (size_t u = 0; u < nm; ++u)
  {
    const double v = (double) mon[u] * (double) mon[u];
    const double t = acc + v;
    comp += std::fabs (acc) >= std::fabs (v) ? (acc - t) + v : (v - t) + acc;
    acc = t;
  }
  acc += comp;
  s->J = acc;
  *J = acc;
  s->forward_done = true;
  s->last_traced = K > 0;
  return YEE_OK;
}

template <typename T>
int backward_impl (yee_handle *h, double dJ, double *grad)
{
  AdjointState *s = h->adj;
  int rc;
  const size_t grid_bytes = (size_t) h->ncell * h->wsize;
  for (int c = 0; c < 6; ++c)
  {
    if (s->af[c]) HIP_TRY (hipMemsetAsync (s->af[c], 0, grid_bytes, h->stream));
    if (s->ad[c]) HIP_TRY (hipMemsetAsync (s->ad[c], 0, grid_bytes, h->stream));
    if (s->w[c]) HIP_TRY (hipMemsetAsync (s->w[c], 0, grid_bytes, h->stream));
  }
  const int64_t nd = s->dn[0] * s->dn[1] * s->dn[2];
  HIP_TRY (hipMemsetAsync (s->grad, 0, (size_t) nd * sizeof (double), h->stream));
  HIP_TRY (hipEventRecord (h->ev[0], h->stream));
  const int K = s->sp.checkpoint_every;
  GradArgs<T> grad_d {};
  if (K == 0)
  {
    for (int32_t t = s->T - 1; t >= 1; --t)
      if ((rc = reverse_step<T> (h, t, t, t - 1, grad_d))) return rc;
    if ((rc = last_gradient (h, grad_d))) return rc;
  }
  else
  {
    const int nseg = (s->T - 1 + K - 1) / K;   // segments of steps (kK, min((k+1)K, T-1)]
    for (int k = nseg - 1; k >= 0; --k)
    {
      const int32_t t0 = k * K, t1 = std::min ((k + 1) * K, s->T - 1);
      if (!(k == nseg - 1 && s->last_traced))
      {
        if ((rc = snapshot (h, k, true))) return rc;
        if ((rc = record<T> (h, 0))) return rc;   // state after step kK
        for (int32_t t = t0 + 1; t <= t1; ++t)
        {
          if ((rc = engine_step_once (h, t1 + 1 - t))) return rc;
          if ((rc = record<T> (h, t - t0))) return rc;
        }
      }
      for (int32_t t = t1; t >= t0 + 1; --t)
        if ((rc = reverse_step<T> (h, t, t - t0, t - t0 - 1, grad_d))) return rc;
      if ((rc = last_gradient (h, grad_d))) return rc;
    }
    s->last_traced = false;   // the trace now holds segment 0
  }
  HIP_TRY (hipEventRecord (h->ev[1], h->stream));
  HIP_TRY (hipEventSynchronize (h->ev[1]));
  float ms = 0;
  HIP_TRY (hipEventElapsedTime (&ms, h->ev[0], h->ev[1]));
  s->bwd_ms = ms;
  HIP_TRY (hipMemcpy (grad, s->grad, (size_t) nd * sizeof (double), hipMemcpyDeviceToHost));
  for (int64_t u = 0; u < nd; ++u) grad[u] *= dJ;
  return YEE_OK;
}

template <typename T>
int fill_eps (yee_handle *h)
{
  // the design needs a per-cell eps grid: expand a uniform eps
  void *p = nullptr;
  int rc = engine_alloc_grid (h, &p);
  if (rc) return rc;
  std::vector<T> v ((size_t) h->ncell, (T) h->mat_u[YEE_MAT_EPS]);
  HIP_TRY (hipMemcpyAsync (p, v.data (), v.size () * sizeof (T), hipMemcpyHostToDevice, h->stream));
  HIP_TRY (hipStreamSynchronize (h->stream));
  h->mat[YEE_MAT_EPS] = p;
  return YEE_OK;
}

}  // namespace

void adjoint_free (yee_handle *h)
{
  if (!h || !h->adj) return;
  if (h->stream) (void) hipStreamSynchronize (h->stream);
  for (void *p : h->adj->allocs) (void) hipFree (p);
  for (void *p : h->adj->snap) (void) hipFree (p);
  delete h->adj;
  h->adj = nullptr;
}

}  // namespace yee

using namespace yee;

extern "C" {

int yee_adjoint_setup (yee_handle *h, const yee_adjoint_spec *sp)
{
  if (!h || !sp) return fail (YEE_EINVAL, "null argument");
  if (!h->prepared) return fail (YEE_ESTATE, "yee_prepare has not been called");
  if (h->cfg.scheme != YEE_SCHEME_DIM3 || h->mode == 2 || h->cfg.current_source || h->imag || h->fine () || h->fn_any ()
      || h->cfg.layout != 0)
    return fail (YEE_ENOTSUP, "the adjoint covers 3D E_CENTERED runs of real fields without metamaterials, current "
                              "sources, double material precision or test functions");
  const int T = h->cfg.time_steps;
  if (T < 2) return fail (YEE_EINVAL, "the adjoint needs --time-steps >= 2");
  if (sp->window < 1 || sp->window > T - 1) return fail (YEE_EINVAL, "window must be in [1, time_steps - 1]");
  if (sp->checkpoint_every < 0) return fail (YEE_EINVAL, "checkpoint_every must be >= 0");
  for (int a = 0; a < 3; ++a)
  {
    const int64_t P = h->use_pml () ? h->cfg.pml[a] : 0;
    // design voxels and their E cells (voxel - 1 .. voxel) must be direct-update cells
    if (sp->design_lo[a] < std::max<int64_t> (2, P + 1) || sp->design_hi[a] > h->n[a] - P - 2
        || sp->design_hi[a] <= sp->design_lo[a])
      return fail (YEE_EINVAL, "design box must lie inside the PML-free interior, one cell from its edge");
  }
  if (sp->monitor_z < 1 || sp->monitor_z >= h->n[2] - 1) return fail (YEE_EINVAL, "monitor plane outside the interior");
  for (int a = 0; a < 2; ++a)
    if (sp->monitor_lo[a] < 1 || sp->monitor_hi[a] > h->n[a] - 1 || sp->monitor_hi[a] <= sp->monitor_lo[a])
      return fail (YEE_EINVAL, "monitor rectangle outside the interior");
  if (h->cfg.point_source)
  {
    const int64_t *p = h->cfg.point_source_pos;
    for (int a = 0; a < 3; ++a)
      if (p[a] < 1 || p[a] >= h->n[a] - 1) return fail (YEE_EINVAL, "adjoint runs need interior point sources");
  }
  adjoint_free (h);
  h->adj = new AdjointState ();
  AdjointState *s = h->adj;
  s->sp = *sp;
  s->T = T;
  for (int a = 0; a < 3; ++a)
  {
    s->dn[a] = sp->design_hi[a] - sp->design_lo[a];
    s->tb.lo[a] = (int) sp->design_lo[a] - 1;
    s->tb.n[a] = (int) s->dn[a] + 1;
  }
  s->mnx = (int) (sp->monitor_hi[0] - sp->monitor_lo[0]);
  s->mny = (int) (sp->monitor_hi[1] - sp->monitor_lo[1]);
  int rc;
  if (!h->mat[YEE_MAT_EPS] && (rc = h->fp32 () ? fill_eps<float> (h) : fill_eps<double> (h))) return rc;
  const size_t grid = (size_t) h->ncell * h->wsize;
  for (int c = 0; c < 6; ++c)
  {
    if ((rc = adj_alloc (h, &s->af[c], grid))) return rc;
    if ((rc = adj_alloc (h, &s->w[c], grid))) return rc;
    if (h->use_pml () && (rc = adj_alloc (h, &s->ad[c], grid))) return rc;
  }
  const int K = sp->checkpoint_every;
  s->trace_slots = K == 0 ? T : K + 1;
  if ((rc = adj_alloc (h, &s->trace, (size_t) s->trace_slots * 3 * s->tb.cells () * h->wsize))) return rc;
  if ((rc = adj_alloc (h, &s->mon, (size_t) s->mnx * s->mny * sp->window * h->wsize))) return rc;
  void *g = nullptr;
  if ((rc = adj_alloc (h, &g, (size_t) (s->dn[0] * s->dn[1] * s->dn[2]) * sizeof (double)))) return rc;
  s->grad = (double *) g;
  if ((rc = adj_alloc (h, &s->stage, (size_t) (s->dn[0] * s->dn[1] * s->dn[2]) * h->wsize))) return rc;
  if (K > 0)
  {
    const int nsnap = (T - 1 + K - 1) / K + 1;
    size_t bytes = 0;
    for (int c = 0; c < 6; ++c)
    {
      if (h->f[0][c]) bytes += grid;
      if (h->d[0][c]) bytes += grid;
    }
    bytes += 2 * (size_t) h->inc_len * h->wsize;
    s->snap_bytes = bytes;
    s->snap.assign (nsnap, nullptr);
    s->snap_t.assign (nsnap, 0);
    s->snap_cur.assign (nsnap, 0);
    for (int k = 0; k < nsnap; ++k)
      if (hipMalloc (&s->snap[k], bytes) != hipSuccess) return fail (YEE_ENOMEM, "checkpoint snapshot allocation failed");
  }
  HIP_TRY (hipStreamSynchronize (h->stream));
  return YEE_OK;
}

int yee_forward (yee_handle *h, const double *design_eps, double *J)
{
  if (!h || !design_eps || !J) return fail (YEE_EINVAL, "null argument");
  if (!h->adj) return fail (YEE_ESTATE, "yee_adjoint_setup has not been called");
  return h->fp32 () ? forward_impl<float> (h, design_eps, J) : forward_impl<double> (h, design_eps, J);
}

int yee_backward (yee_handle *h, double dJ, double *grad_eps)
{
  if (!h || !grad_eps) return fail (YEE_EINVAL, "null argument");
  if (!h->adj || !h->adj->forward_done) return fail (YEE_ESTATE, "yee_forward has not been called");
  return h->fp32 () ? backward_impl<float> (h, dJ, grad_eps) : backward_impl<double> (h, dJ, grad_eps);
}

int yee_adjoint_timing (yee_handle *h, double out[2])
{
  if (!h || !out) return fail (YEE_EINVAL, "null argument");
  if (!h->adj) return fail (YEE_ESTATE, "yee_adjoint_setup has not been called");
  out[0] = h->adj->fwd_ms;
  out[1] = h->adj->bwd_ms;
  return YEE_OK;
}

}  // extern "C"
