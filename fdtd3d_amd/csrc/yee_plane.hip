// Several time steps of a 2D scheme in one launch (TMx .. TMz, TEx .. TEz, E_CENTERED, plain and PML).
//
// What bounds a 2D run: at 100^2 the two launches a step (10 us of which 2 are work), at 1403 x 977
// the passes over L2 with one cell a thread (24 us a step in FP32, 6 of them the state's bytes at
// HBM rate).  So a workgroup takes a tile, keeps it in registers and advances it by up to kPlaneSteps
// steps: a step of a cell depends on its neighbours one cell away, so a margin of as many cells
// as steps around the owned ones spoils from its ends inward and the owned ones stay exact (the
// neighbouring tiles recompute the margin).  State goes from f / d to f_n / d_n, since neighbours
// still read the old values.
//
// A tile is 64 columns (the lanes, along the contiguous axis) by NW waves of RW rows: column
// neighbours come from the next lane (DPP), row neighbours from the thread's own registers, and
// only the rows between two waves go through LDS (one write, one barrier and one read a half step).
// The coefficients of a cell are divided out once a launch.  Every cell is computed with the
// expressions of e_half_cell / tmz_e_cell in their order, so the results are the half-step
// kernels' bits.
#include <hip/hip_runtime.h>

#include "yee_device.h"
#include "yee_plane.h"

namespace yee {

// The components of a scheme and the axes of its plane: rows run along RA, columns (contiguous)
// along CA; component CC has the scheme's missing axis MA, CR lies along RA, CK along CA.  TM: CC is
// E and the others H, TE the reverse.  ODD: (RA, CA, MA) is an odd permutation of (x, y, z), which
// turns the curl's signs and the order of its two differences.
template <int SCHEME>
struct Plane
{
  static constexpr bool te = SCHEME <= YEE_SCHEME_TEZ;
  static constexpr int ma = (SCHEME - YEE_SCHEME_TEX) % 3;
  static constexpr int ra = ma == 0 ? 1 : 0, ca = ma == 2 ? 1 : 2;
  static constexpr bool odd = ma == 1;
  static constexpr int cc = (te ? 3 : 0) + ma, cr = (te ? 0 : 3) + ra, ck = (te ? 0 : 3) + ca;
  // the kernels of TEz / TMz evaluate the incident wave in 2D, the other planes in 3D
  static constexpr int dim = ma == 2 ? 2 : 3;
};

// A PML coefficient of one component over a thread's RW rows, by the axis it depends on: one value
// a lane (columns), one a row, or a constant (the missing axis).
template <typename T, int RW>
struct TileCoef
{
  T lane, row[RW];
};

// Both roles of axis pair `pair` of component comp at the cells of the thread's rows.
template <typename T, class S, int RW, int COMP, int PAIR>
__device__ __forceinline__ void tile_coef (const StepArgs<T> &a, int i0, int j, TileCoef<T, RW> &x, TileCoef<T, RW> &y)
{
  constexpr int ax = PAIR == 0 ? SigAxes<COMP>::c : (PAIR == 1 ? SigAxes<COMP>::s4 : SigAxes<COMP>::s5);
  const T *tab = a.pml + (size_t) (COMP * 3 + PAIR) * 2 * (size_t) a.tab_len;
  const int nr = S::ra == 0 ? a.nx : a.ny, nc = S::ca == 1 ? a.ny : a.nz;
  if constexpr (ax == S::ra)
  {
#pragma unroll
    for (int q = 0; q < RW; ++q)
    {
      const Pair<T> v = gld2 (tab + 2 * max (0, min (i0 + q, nr - 1)));
      x.row[q] = v.a;
      y.row[q] = v.b;
    }
  }
  else
  {
    const Pair<T> v = gld2 (tab + 2 * (ax == S::ca ? max (0, min (j, nc - 1)) : 0));
    x.lane = v.a;
    y.lane = v.b;
  }
}

template <typename T, class S, int RW, int COMP, int PAIR>
__device__ __forceinline__ T coef_at (const TileCoef<T, RW> &x, int q)
{
  constexpr int ax = PAIR == 0 ? SigAxes<COMP>::c : (PAIR == 1 ? SigAxes<COMP>::s4 : SigAxes<COMP>::s5);
  if constexpr (ax == S::ra) return x.row[q];
  else return x.lane;
}

// One component of the thread's rows: the field, D / B (PML), the factors (direct: ka = cb; PML
// cells: ka, kb the D -> field factors).
template <typename T, int RW>
struct TileComp
{
  T f[RW], d[RW], ka[RW], kb[RW];
  TileCoef<T, RW> cac, cbc, ca5;
};

// Averaged material of component COMP at cell q (e_half_cell / h_half_cell with stride 0 along the
// missing axis): rs, cs the strides of a row and a column.
template <typename T, class S, int COMP>
__device__ __forceinline__ T tile_mat (const StepArgs<T> &a, int64_t q, int64_t rs)
{
  if (a.matc[COMP]) return gld (a.matc[COMP] + q);
  const T *m = COMP < 3 ? a.eps : a.mu;
  if (!m) return COMP < 3 ? a.eps_u : a.mu_u;
  if constexpr (COMP < 3)
  {
    // 2-cell average along the component's axis (the cell itself along the missing one)
    const T e = gld (m + q);
    return avg2 (e, COMP == S::ma ? e : gld (m + q + (COMP == S::ra ? rs : 1)));
  }
  else
  {
    // 4-cell average across it
    constexpr int ax = COMP - 3;
    if constexpr (ax == S::ma) return avg4 (gld (m + q), gld (m + q + 1), gld (m + q + rs), gld (m + q + rs + 1));
    else
    {
      const T u = gld (m + q), v = gld (m + q + (ax == S::ra ? 1 : rs));
      return avg4 (u, u, v, v);
    }
  }
}

template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_load (const StepArgs<T> &a, int i0, int j, int64_t q0, int64_t rs, uint32_t in,
                                           uint32_t upd, uint32_t sp, TileComp<T, RW> &x)
{
  const T modc = COMP >= 3 ? a.mu0 : a.eps0;
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    x.f[q] = (in >> q) & 1u ? gld (a.f[COMP] + q0 + q * rs) : (T) 0;
    x.d[q] = x.ka[q] = x.kb[q] = (T) 0;
    if (PML && ((sp >> q) & 1u)) x.d[q] = gld (a.d[COMP] + q0 + q * rs);
  }
  TileCoef<T, RW> p4, m4, dd5;
  if (PML)
  {
    tile_coef<T, S, RW, COMP, 0> (a, i0, j, x.cac, x.cbc);
    tile_coef<T, S, RW, COMP, 1> (a, i0, j, p4, m4);
    tile_coef<T, S, RW, COMP, 2> (a, i0, j, x.ca5, dd5);
  }
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    if (!((upd >> q) & 1u)) continue;
    const T mat = tile_mat<T, S, COMP> (a, q0 + q * rs, rs);
    if (PML && ((sp >> q) & 1u))
    {
      const Pair<T> k = pml_factors (coef_at<T, S, RW, COMP, 1> (p4, q), coef_at<T, S, RW, COMP, 1> (m4, q), mat * modc,
                                     coef_at<T, S, RW, COMP, 2> (dd5, q));
      x.ka[q] = k.a;
      x.kb[q] = k.b;
    }
    else
    {
      x.ka[q] = direct_cb (a.dt, mat, modc, a.dx);
    }
  }
}

// Update of row q of a component from its curl (cell_value_pc: the direct or the PML expression);
// the value stays where the cell is not updated.
template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_update (TileComp<T, RW> &x, int q, T tmp, uint32_t upd, uint32_t sp)
{
  if (PML && ((sp >> q) & 1u))
  {
    const T d = x.d[q] * coef_at<T, S, RW, COMP, 0> (x.cac, q) + tmp * coef_at<T, S, RW, COMP, 0> (x.cbc, q);
    x.f[q] = x.f[q] * coef_at<T, S, RW, COMP, 2> (x.ca5, q) + d * x.ka[q] - x.d[q] * x.kb[q];
    x.d[q] = d;
  }
  else
  {
    const T v = x.f[q] * (T) 1.0 + tmp * x.ka[q];
    x.f[q] = (upd >> q) & 1u ? v : x.f[q];
  }
}

template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_store (const StepArgs<T> &a, int64_t q0, int64_t rs, uint32_t own, uint32_t sp,
                                            const TileComp<T, RW> &x)
{
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    if (!((own >> q) & 1u)) continue;
    gst (a.f_n[COMP] + q0 + q * rs, x.f[q]);
    if (PML && ((sp >> q) & 1u)) gst (a.d_n[COMP] + q0 + q * rs, x.d[q]);
  }
}

// TF/SF corrections of a tile for all its steps, filled before the first: [step][E, H][row faces:
// plane lo, hi by lane | column faces: column lo, hi by row].  The values are subtracted from one
// operand (tfsf_pair_diff); 0 where there is no correction.
template <int ROWS>
struct TileFaces
{
  double row[kPlaneSteps][2][2][64];
  double col[kPlaneSteps][2][2][ROWS];
};

// The correction of the difference along the row (ROWDIR) or column axis of half step `half` (0: E,
// 1: H) at cell (i, j) on the lo (side 0) or hi (side 1) face.
template <typename T, class S, bool ROWDIR>
__device__ double tile_face (const StepArgs<T> &a, int half, int side, int i, int j)
{
  int p[3] = { 0, 0, 0 };
  p[S::ra] = i;
  p[S::ca] = j;
  double lo = 0, hi = 0;
  if (S::te == (half == 0))
  {
    // the two components of the plane: each is differenced along one axis only
    constexpr int comp = ROWDIR ? S::ck : S::cr;
    constexpr int b = ROWDIR ? S::ra : S::ca;
    constexpr int pair = (Tab::dir[comp][0] >> 1) == b ? 0 : 1;
    tfsf_pair_diff<T, comp, pair, S::dim> (a, p[0], p[1], p[2], lo, hi);
  }
  else
  {
    constexpr int b = ROWDIR ? S::ra : S::ca;
    constexpr int pair = (Tab::dir[S::cc][0] >> 1) == b ? 0 : 1;
    tfsf_pair_diff<T, S::cc, pair, S::dim> (a, p[0], p[1], p[2], lo, hi);
  }
  // E corrects the operand across the face (lo face: hi slot), H the one on its side
  return (half == 0) == (side == 0) ? hi : lo;
}

// What a tile's steps need beside the record: its place and the values of the hard source.
template <typename T>
struct TileJob
{
  int x0, y0;          // first owned row and column
  int rows, cols;      // owned rows and columns
  int margin;          // kPlaneSteps or fewer: the most steps the margin covers
  int n;               // steps to take
};

template <typename T, class S, int RW, int NW, bool PML, bool TFSF, class Src>
__device__ __forceinline__ void tile_steps (const StepArgs<T> &a, const TileJob<T> &job, T (*xlo)[64], T (*xhi)[64],
                                            TileFaces<RW * NW> *faces, const Src &src)
{
  constexpr int ROWS = RW * NW;
  const int tid = (int) threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane (tid >> 6);
  const int nr = S::ra == 0 ? a.nx : a.ny, nc = S::ca == 1 ? a.ny : a.nz;
  const int64_t rs = S::ra == 0 ? a.sx : (int64_t) a.sy;
  const int K = job.margin;
  const int i0 = job.x0 - K + wave * RW, j = job.y0 - K + lane;   // the thread's first cell
  const int64_t q0 = (int64_t) i0 * rs + j;
  // cells in the grid, updated, PML cells, owned (bit q: row i0 + q)
  uint32_t in = 0, upd = 0, sp = 0, own = 0;
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    const int i = i0 + q;
    const bool g = i >= 0 && i < nr && j >= 0 && j < nc;
    const bool u = i >= 1 && i < nr - 1 && j >= 1 && j < nc - 1;
    const bool s = u && (i < a.slab_lo[S::ra] || i >= a.slab_hi[S::ra] || j < a.slab_lo[S::ca] || j >= a.slab_hi[S::ca]);
    const int li = i - job.x0, lj = j - job.y0;
    in |= g ? 1u << q : 0u;
    upd |= u ? 1u << q : 0u;
    sp |= s ? 1u << q : 0u;
    own |= u && li >= 0 && li < job.rows && lj >= 0 && lj < job.cols ? 1u << q : 0u;
  }
  TileComp<T, RW> C, R, K2;
  tile_load<T, S, RW, S::cc, PML> (a, i0, j, q0, rs, in, upd, sp, C);
  tile_load<T, S, RW, S::cr, PML> (a, i0, j, q0, rs, in, upd, sp, R);
  tile_load<T, S, RW, S::ck, PML> (a, i0, j, q0, rs, in, upd, sp, K2);
  // face planes of the TF/SF box as tile rows / lanes: E on L-1 and R, H on L-1 and R-1
  const int tx = job.x0 - K, ty = job.y0 - K;
  const int lo_r = a.tl[S::ra] - 1 - tx, hi_r = a.tr[S::ra] - tx, lo_c = a.tl[S::ca] - 1 - ty, hi_c = a.tr[S::ca] - ty;
  bool frow = false, fcol = false;
  if constexpr (TFSF)
  {
    frow = (lo_r >= 0 && lo_r < ROWS) || (hi_r >= 0 && hi_r <= ROWS);
    fcol = (lo_c >= 0 && lo_c < 64) || (hi_c >= 0 && hi_c <= 64);
    if (frow || fcol)
    {
      // a task is a face cell of one half step: all its reads of the incident rows are in flight
      // at once, before the first step needs one
      const int per = 2 * 64 + 2 * ROWS;
      for (int u = tid; u < job.n * 2 * per; u += 64 * NW)
      {
        const int s = u / (2 * per), half = (u / per) & 1, v = u % per;
        StepArgs<T> b = a;
        b.einc = a.einc + s * a.inc_len;
        b.hinc = a.hinc + s * a.inc_len;
        if (v < 128)
        {
          const int side = v >> 6, i = (side ? hi_r - half : lo_r) + tx, jj = ty + (v & 63);
          const bool ok = i >= 1 && i < nr - 1 && jj >= 1 && jj < nc - 1;
          faces->row[s][half][side][v & 63] = ok ? tile_face<T, S, true> (b, half, side, i, jj) : 0.0;
        }
        else
        {
          const int side = (v - 128) / ROWS, r = (v - 128) % ROWS;
          const int i = tx + r, jj = (side ? hi_c - half : lo_c) + ty;
          const bool ok = i >= 1 && i < nr - 1 && jj >= 1 && jj < nc - 1;
          faces->col[s][half][side][r] = ok ? tile_face<T, S, false> (b, half, side, i, jj) : 0.0;
        }
      }
    }
  }
  // the hard source as a row of the thread, and its lane
  const int src_q = a.src_mask ? a.src_pos[S::ra] - i0 : -1;
  const bool src_lane = a.src_mask && j == a.src_pos[S::ca];
  const bool src_row = src_q >= 0 && src_q < RW;
  // exchange of the rows between waves: the last row of the wave before (xlo: the field E reads at
  // row - 1), the first row of the next (xhi: the field H reads at row + 1)
  TileComp<T, RW> &FB = S::te ? C : K2;   // differenced backward along rows by the E half step
  TileComp<T, RW> &FF = S::te ? K2 : C;   // differenced forward along rows by the H half step
  xlo[wave + 1][lane] = FB.f[RW - 1];
  for (int s = 0; s < job.n; ++s)
  {
    __syncthreads ();
    // ---- E half step
    {
      T before = xlo[wave][lane];   // (wave 0: margin, any value)
#pragma unroll
      for (int q = 0; q < RW; ++q)
      {
        const int r = wave * RW + q;
        // operands: bm / b0 along the rows (at row - 1 and row), cm / c0 along the columns
        T bm = before, b0 = FB.f[q];
        before = b0;
        T c0 = S::te ? C.f[q] : R.f[q];
        T cm = lane_prev (c0, c0);
        T rm = bm, r0 = b0;
        if constexpr (TFSF)
        {
          if (frow)
          {
            if (r == lo_r) r0 = (T) ((double) r0 - faces->row[s][0][0][lane]);
            if (r == hi_r) rm = (T) ((double) rm - faces->row[s][0][1][lane]);
          }
          if (fcol)
          {
            const double dl = lane == lo_c ? faces->col[s][0][0][r] : 0.0, dh = lane == hi_c ? faces->col[s][0][1][r] : 0.0;
            c0 = (T) ((double) c0 - dl);
            cm = (T) ((double) cm - dh);
          }
        }
        if constexpr (!S::te)
        {
          // E_ma: d_ra H_ca - d_ca H_ra (curl: v1 - v0 - v3 + v2), odd planes the other way round
          const T tmp = S::odd ? c0 - cm - r0 + rm : r0 - rm - c0 + cm;
          tile_update<T, S, RW, S::cc, PML> (C, q, tmp, upd, sp);
        }
        else
        {
          // E_ra: + d_ca H_ma, E_ca: - d_ra H_ma (odd: the other signs)
          tile_update<T, S, RW, S::cr, PML> (R, q, S::odd ? cm - c0 : c0 - cm, upd, sp);
          tile_update<T, S, RW, S::ck, PML> (K2, q, S::odd ? r0 - rm : rm - r0, upd, sp);
        }
      }
      if (src_row)
      {
        const T v = src (s, 0);
#pragma unroll
        for (int q = 0; q < RW; ++q)
        {
          if (q != src_q || !src_lane) continue;
          if (!S::te && ((a.src_mask >> S::cc) & 1u)) C.f[q] = v;
          if (S::te && ((a.src_mask >> S::cr) & 1u)) R.f[q] = v;
          if (S::te && ((a.src_mask >> S::ck) & 1u)) K2.f[q] = v;
        }
      }
      xhi[wave][lane] = FF.f[0];
    }
    __syncthreads ();
    // ---- H half step
    {
      T after = xhi[wave + 1][lane];   // (last wave: margin, any value)
#pragma unroll
      for (int q = RW - 1; q >= 0; --q)
      {
        const int r = wave * RW + q;
        T r0 = FF.f[q], rp = after;
        after = r0;
        T c0 = S::te ? R.f[q] : C.f[q];
        T cp = lane_next (c0, c0);
        if constexpr (TFSF)
        {
          if (frow)
          {
            if (r == lo_r) r0 = (T) ((double) r0 - faces->row[s][1][0][lane]);
            if (r == hi_r - 1) rp = (T) ((double) rp - faces->row[s][1][1][lane]);
          }
          if (fcol)
          {
            const double dl = lane == lo_c ? faces->col[s][1][0][r] : 0.0;
            const double dh = lane == hi_c - 1 ? faces->col[s][1][1][r] : 0.0;
            c0 = (T) ((double) c0 - dl);
            cp = (T) ((double) cp - dh);
          }
        }
        if constexpr (!S::te)
        {
          // H_ra: - d_ca E_ma, H_ca: + d_ra E_ma (odd: the other signs)
          tile_update<T, S, RW, S::cr, PML> (R, q, S::odd ? cp - c0 : c0 - cp, upd, sp);
          tile_update<T, S, RW, S::ck, PML> (K2, q, S::odd ? r0 - rp : rp - r0, upd, sp);
        }
        else
        {
          // H_ma: d_ca E_ra - d_ra E_ca, odd planes the other way round
          const T tmp = S::odd ? rp - r0 - cp + c0 : cp - c0 - rp + r0;
          tile_update<T, S, RW, S::cc, PML> (C, q, tmp, upd, sp);
        }
      }
      if (src_row)
      {
        const T v = src (s, 1);
#pragma unroll
        for (int q = 0; q < RW; ++q)
        {
          if (q != src_q || !src_lane) continue;
          if (S::te && ((a.src_mask >> S::cc) & 1u)) C.f[q] = v;
          if (!S::te && ((a.src_mask >> S::cr) & 1u)) R.f[q] = v;
          if (!S::te && ((a.src_mask >> S::ck) & 1u)) K2.f[q] = v;
        }
      }
      xlo[wave + 1][lane] = FB.f[RW - 1];
    }
  }
  tile_store<T, S, RW, S::cc, PML> (a, q0, rs, own, sp, C);
  tile_store<T, S, RW, S::cr, PML> (a, q0, rs, own, sp, R);
  tile_store<T, S, RW, S::ck, PML> (a, q0, rs, own, sp, K2);
}

// Whether a tile holds a PML cell (uniform).
template <typename T, class S>
__device__ __forceinline__ bool tile_pml (const StepArgs<T> &a, int x0, int y0, int rows, int cols)
{
  return a.pml && (x0 < a.slab_lo[S::ra] || x0 + rows > a.slab_hi[S::ra] || y0 < a.slab_lo[S::ca] || y0 + cols > a.slab_hi[S::ca]);
}

// n steps of a single run.  Tiles are numbered along the columns and handed to the XCDs in bands.
template <typename T, int SCHEME, bool TFSF>
__global__ __launch_bounds__ (64 * kPlaneWaves) void plane_steps (StepArgs<T> a, PlaneGrid g, PlaneSource src)
{
  using S = Plane<SCHEME>;
  constexpr int RW = PLANE_RW (T), ROWS = RW * kPlaneWaves;
  __shared__ T xlo[kPlaneWaves + 1][64], xhi[kPlaneWaves + 1][64];
  extern __shared__ char dyn[];
  TileFaces<ROWS> *faces = (TileFaces<ROWS> *) dyn;
  const int b = (int) blockIdx.x, u = (b & 7) * g.per_xcd + (b >> 3);
  if (u >= g.ntile) return;   // the whole workgroup
  const int tr = u / g.ncol, tc = u - tr * g.ncol;
  TileJob<T> job;
  job.margin = g.margin;
  job.rows = ROWS - 2 * g.margin;
  job.cols = 64 - 2 * g.margin;
  job.x0 = 1 + tr * job.rows;
  job.y0 = 1 + tc * job.cols;
  job.n = g.n;
  auto value = [&] (int s, int half) { return (T) src.v[s][half]; };
  if (tile_pml<T, S> (a, job.x0 - g.margin, job.y0 - g.margin, ROWS, 64))
    tile_steps<T, S, RW, kPlaneWaves, true, TFSF> (a, job, xlo, xhi, faces, value);
  else
    tile_steps<T, S, RW, kPlaneWaves, false, TFSF> (a, job, xlo, xhi, faces, value);
}

template <typename T>
void launch_plane (int scheme, const StepArgs<T> &a, const PlaneGrid &g, const PlaneSource &src, hipStream_t stream)
{
  const dim3 grid ((unsigned) (8 * g.per_xcd)), block (64 * kPlaneWaves);
  const size_t lds = a.tfsf ? sizeof (TileFaces<PLANE_RW (T) * kPlaneWaves>) : 0;
#define YEE_PLANE(S)                                                                                              \
  case S:                                                                                                         \
    if (a.tfsf) hipLaunchKernelGGL ((plane_steps<T, S, true>), grid, block, lds, stream, a, g, src);               \
    else hipLaunchKernelGGL ((plane_steps<T, S, false>), grid, block, lds, stream, a, g, src);                     \
    break;
  switch (scheme)
  {
    YEE_PLANE (YEE_SCHEME_TEX)
    YEE_PLANE (YEE_SCHEME_TEY)
    YEE_PLANE (YEE_SCHEME_TEZ)
    YEE_PLANE (YEE_SCHEME_TMX)
    YEE_PLANE (YEE_SCHEME_TMY)
    YEE_PLANE (YEE_SCHEME_TMZ)
    default: break;
  }
#undef YEE_PLANE
}
template void launch_plane<float> (int, const StepArgs<float> &, const PlaneGrid &, const PlaneSource &, hipStream_t);
template void launch_plane<double> (int, const StepArgs<double> &, const PlaneGrid &, const PlaneSource &, hipStream_t);

}  // namespace yee
