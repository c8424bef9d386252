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
// The D -> field factors of PML cells (IEEE divisions that took 8 of the 21 us of a launch at 100^2
// FP64) come from arrays made once, by plane_factors.  Every cell is computed with the
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

// Averaged material of component COMP at byte offset o of the row that starts at cell r0
// (e_half_cell / h_half_cell with stride 0 along the missing axis); rs: cells of a row.
template <typename T, class S, int COMP>
__device__ __forceinline__ T tile_mat (const StepArgs<T> &a, int64_t r0, uint32_t o, int64_t rs)
{
  if (a.matc[COMP]) return rld (a.matc[COMP] + r0, o);
  const T *m = COMP < 3 ? a.eps : a.mu;
  if (!m) return COMP < 3 ? a.eps_u : a.mu_u;
  const T *m0 = m + r0, *m1 = m0 + rs;
  if constexpr (COMP < 3)
  {
    // 2-cell average along the component's axis (the cell itself along the missing one)
    const T e = rld (m0, o);
    return avg2 (e, COMP == S::ma ? e : (COMP == S::ra ? rld (m1, o) : rld (m0, o, 1)));
  }
  else
  {
    // 4-cell average across it
    constexpr int ax = COMP - 3;
    if constexpr (ax == S::ma) return avg4 (rld (m0, o), rld (m0, o, 1), rld (m1, o), rld (m1, o, 1));
    else
    {
      const T u = rld (m0, o), v = ax == S::ra ? rld (m0, o, 1) : rld (m1, o);
      return avg4 (u, u, v, v);
    }
  }
}

// The loads of one component (every address is clamped into the grid, so that none waits for a
// branch), then, for all three components loaded, tile_factors.
template <typename T, int RW>
struct TileRaw
{
  T mat[RW];
  Pair<T> k[RW];
};

template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_load (const StepArgs<T> &a, int i0, int j, const int64_t (&r0)[RW], uint32_t o, int64_t rs,
                                           TileComp<T, RW> &x, TileRaw<T, RW> &w)
{
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    x.f[q] = rld ((const T *) a.f[COMP] + r0[q], o);
    w.mat[q] = tile_mat<T, S, COMP> (a, r0[q], o, rs);
    if (PML)
    {
      x.d[q] = rld ((const T *) a.d[COMP] + r0[q], o);
      // (equal for the component of the missing axis)
      w.k[q].a = rld (a.pfac[COMP] + 2 * r0[q], 2 * o);
      if (COMP != S::cc) w.k[q].b = rld (a.pfac[COMP] + 2 * r0[q], 2 * o, 1);
    }
  }
  if (PML)
  {
    TileCoef<T, RW> dd5;
    tile_coef<T, S, RW, COMP, 0> (a, i0, j, x.cac, x.cbc);
    tile_coef<T, S, RW, COMP, 2> (a, i0, j, x.ca5, dd5);
  }
}

template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_factors (const StepArgs<T> &a, const bool (&in)[RW], const bool (&sp)[RW],
                                              TileComp<T, RW> &x, const TileRaw<T, RW> &w)
{
  const T modc = COMP >= 3 ? a.mu0 : a.eps0;
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    const bool s = PML && sp[q];
    x.f[q] = in[q] ? x.f[q] : (T) 0;
    x.ka[q] = direct_cb (a.dt, w.mat[q], modc, a.dx);
    if (s)
    {
      x.ka[q] = w.k[q].a;
      if (COMP != S::cc) x.kb[q] = w.k[q].b;
    }
  }
}

// Update of row q of a component from its curl (cell_value_pc: the direct or the PML expression);
// the value stays where the cell is not updated.
template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_update (TileComp<T, RW> &x, int q, T tmp, bool upd, bool sp)
{
  if (PML && sp)
  {
    const T d = x.d[q] * coef_at<T, S, RW, COMP, 0> (x.cac, q) + tmp * coef_at<T, S, RW, COMP, 0> (x.cbc, q);
    // (the missing axis has no sigma, so the two factors of its component are equal)
    const T kb = COMP == S::cc ? x.ka[q] : x.kb[q];
    x.f[q] = x.f[q] * coef_at<T, S, RW, COMP, 2> (x.ca5, q) + d * x.ka[q] - x.d[q] * kb;
    x.d[q] = d;
  }
  else
  {
    const T v = x.f[q] * (T) 1.0 + tmp * x.ka[q];
    x.f[q] = upd ? v : x.f[q];
  }
}

template <typename T, class S, int RW, int COMP, bool PML>
__device__ __forceinline__ void tile_store (const StepArgs<T> &a, int64_t q0, int64_t rs, const bool (&own)[RW],
                                            const bool (&sp)[RW], const TileComp<T, RW> &x)
{
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    if (!own[q]) continue;
    gst (a.f_n[COMP] + q0 + q * rs, x.f[q]);
    if (PML && sp[q]) gst (a.d_n[COMP] + q0 + q * rs, x.d[q]);
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

// Where a correction reads the incident wave, the same in every step: cells i1 and i1 + 1 with the
// weights p1 and p2, times the component's projection (incident_at), negated for H.
struct FacePoint
{
  int i1;
  double p1, p2, proj;
};

// The correction of operand pair PAIR of component COMP at cell p on the lo (side 0) or hi (side 1)
// face plane (tfsf_pair_diff); false where there is none.
template <typename T, int COMP, int PAIR, int DIM>
__device__ __forceinline__ bool face_point (const StepArgs<T> &a, int side, const int p[3], FacePoint &f)
{
  constexpr bool h = COMP >= 3;
  constexpr int OPP = Tab::opp[COMP][PAIR];
  const bool on = side == 0 ? tfsf_pred<T, COMP, Tab::dir[COMP][2 * PAIR], DIM> (a, p[0], p[1], p[2])
                            : tfsf_pred<T, COMP, Tab::dir[COMP][2 * PAIR + 1], DIM> (a, p[0], p[1], p[2]);
  if (!on) return false;
  // E corrects the operand across the face (lo face: the hi slot), H the one on its side
  const bool hi_slot = h ? side == 1 : side == 0;
  constexpr int lo = 2 * PAIR, hi = 2 * PAIR + 1;
  const int i = p[0] + (hi_slot ? Tab::off[COMP][hi][0] : Tab::off[COMP][lo][0]);
  const int j = p[1] + (hi_slot ? Tab::off[COMP][hi][1] : Tab::off[COMP][lo][1]);
  const int k = DIM == 3 ? p[2] + (hi_slot ? Tab::off[COMP][hi][2] : Tab::off[COMP][lo][2]) : 0;
  const double d = incident_distance<T, OPP, DIM> (a, i, j, k, h ? 0.0 : 0.5);
  const double c1 = (double) (long long) d;
  long long i1 = (long long) c1;
  if (i1 < 0) i1 = 0;
  if (i1 > a.inc_len - 2) i1 = a.inc_len - 2;
  f.i1 = (int) i1;
  f.p2 = d - c1;
  f.p1 = 1 - f.p2;
  f.proj = h ? -a.tg->proj[OPP] : a.tg->proj[OPP];
  return true;
}

// The same for the difference along the row (ROWDIR) or column axis of half step `half` (0: E, 1: H).
template <typename T, class S, bool ROWDIR>
__device__ __forceinline__ bool tile_face (const StepArgs<T> &a, int half, int side, int i, int j, FacePoint &f)
{
  int p[3] = { 0, 0, 0 };
  p[S::ra] = i;
  p[S::ca] = j;
  constexpr int b = ROWDIR ? S::ra : S::ca;
  // the component of the missing axis is differenced along both axes, the other two along one each
  constexpr int one = ROWDIR ? S::ck : S::cr;
  constexpr int pair1 = (Tab::dir[one][0] >> 1) == b ? 0 : 1, pair2 = (Tab::dir[S::cc][0] >> 1) == b ? 0 : 1;
  if (S::te == (half == 0)) return face_point<T, one, pair1, S::dim> (a, side, p, f);
  return face_point<T, S::cc, pair2, S::dim> (a, side, p, f);
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
  // cells in the grid, updated, PML cells (row i0 + q; kept as scalar lane masks)
  bool in[RW], upd[RW], sp[RW];
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    const int i = i0 + q;
    // (the last row and column are always zero: no step and no source writes them)
    const bool g = i >= 0 && i < nr - 1 && j >= 0 && j < nc - 1;
    const bool u = i >= 1 && i < nr - 1 && j >= 1 && j < nc - 1;
    const bool s = u && (i < a.slab_lo[S::ra] || i >= a.slab_hi[S::ra] || j < a.slab_lo[S::ca] || j >= a.slab_hi[S::ca]);
    in[q] = g;
    upd[q] = u;
    sp[q] = s;
  }
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
      // a thread takes a face cell of one half step: where it reads the incident wave is the same
      // in every step, and the reads of all steps are in flight at once, before the first step
      const int per = 2 * 64 + 2 * ROWS;
      for (int u = tid; u < 2 * per; u += 64 * NW)
      {
        const int half = u >= per ? 1 : 0, v = u - half * per;
        const bool rowdir = v < 128;
        const int side = rowdir ? v >> 6 : (v - 128) / ROWS;
        const int at = rowdir ? v & 63 : v - 128 - side * ROWS;   // lane, or row of the tile
        const int plane = rowdir ? (side ? hi_r - half : lo_r) : (side ? hi_c - half : lo_c);
        if (plane < 0 || plane >= (rowdir ? ROWS : 64)) continue;   // no such face in the tile
        const int i = tx + (rowdir ? plane : at), jj = ty + (rowdir ? at : plane);
        const bool ok = i >= 1 && i < nr - 1 && jj >= 1 && jj < nc - 1;
        FacePoint f {};
        const bool on = ok && (rowdir ? tile_face<T, S, true> (a, half, side, i, jj, f) : tile_face<T, S, false> (a, half, side, i, jj, f));
        const T *inc = half ? a.einc : a.hinc;
        T g0[kPlaneSteps], g1[kPlaneSteps];
#pragma unroll
        for (int s = 0; s < kPlaneSteps; ++s)
        {
          const T *r = inc + (s < job.n ? s : 0) * a.inc_len + f.i1;
          g0[s] = gld (r);
          g1[s] = gld (r + 1);
        }
#pragma unroll
        for (int s = 0; s < kPlaneSteps; ++s)
        {
          const double val = on ? ((double) g0[s] * f.p1 + (double) g1[s] * f.p2) * f.proj : 0.0;
          if (rowdir) faces->row[s][half][side][at] = val;
          else faces->col[s][half][side][at] = val;
        }
      }
    }
  }
  TileComp<T, RW> C, R, K2;
  {
    // clamped below the last row and column, whose cells no step updates (and tile_mat reads one
    // further)
    int64_t r0[RW];   // uniform: scalar registers
#pragma unroll
    for (int q = 0; q < RW; ++q) r0[q] = (int64_t) max (0, min (i0 + q, nr - 2)) * rs;
    const uint32_t o = (uint32_t) max (0, min (j, nc - 2)) * (uint32_t) sizeof (T);
    TileRaw<T, RW> wc, wr, wk;
    tile_load<T, S, RW, S::cc, PML> (a, i0, j, r0, o, rs, C, wc);
    tile_load<T, S, RW, S::cr, PML> (a, i0, j, r0, o, rs, R, wr);
    tile_factors<T, S, RW, S::cc, PML> (a, in, sp, C, wc);
    tile_load<T, S, RW, S::ck, PML> (a, i0, j, r0, o, rs, K2, wk);
    tile_factors<T, S, RW, S::cr, PML> (a, in, sp, R, wr);
    tile_factors<T, S, RW, S::ck, PML> (a, in, sp, K2, wk);
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
          tile_update<T, S, RW, S::cc, PML> (C, q, tmp, upd[q], sp[q]);
        }
        else
        {
          // E_ra: + d_ca H_ma, E_ca: - d_ra H_ma (odd: the other signs)
          tile_update<T, S, RW, S::cr, PML> (R, q, S::odd ? cm - c0 : c0 - cm, upd[q], sp[q]);
          tile_update<T, S, RW, S::ck, PML> (K2, q, S::odd ? r0 - rm : rm - r0, upd[q], sp[q]);
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
          tile_update<T, S, RW, S::cr, PML> (R, q, S::odd ? cp - c0 : c0 - cp, upd[q], sp[q]);
          tile_update<T, S, RW, S::ck, PML> (K2, q, S::odd ? r0 - rp : rp - r0, upd[q], sp[q]);
        }
        else
        {
          // H_ma: d_ca E_ra - d_ra E_ca, odd planes the other way round
          const T tmp = S::odd ? rp - r0 - cp + c0 : cp - c0 - rp + r0;
          tile_update<T, S, RW, S::cc, PML> (C, q, tmp, upd[q], sp[q]);
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
  bool own[RW];
#pragma unroll
  for (int q = 0; q < RW; ++q)
  {
    const int li = i0 + q - job.x0, lj = j - job.y0;
    own[q] = upd[q] && li >= 0 && li < job.rows && lj >= 0 && lj < job.cols;
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
// (FP32 without TF/SF: 64 VGPRs, so that a compute unit holds two tiles of 16 waves.)
template <typename T, int SCHEME, bool TFSF, int NW>
__global__ __launch_bounds__ (64 * NW, sizeof (T) == 4 && !TFSF && NW == kPlaneWaves ? 8 : 4)
void plane_steps (StepArgs<T> a, PlaneGrid g, PlaneSource src)
{
  using S = Plane<SCHEME>;
  constexpr int RW = PLANE_RW (T), ROWS = RW * NW;
  __shared__ T xlo[NW + 1][64], xhi[NW + 1][64];
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
    tile_steps<T, S, RW, NW, true, TFSF> (a, job, xlo, xhi, faces, value);
  else
    tile_steps<T, S, RW, NW, false, TFSF> (a, job, xlo, xhi, faces, value);
}

// The same for a batch of TMz simulations of different sizes: the tiles of all of them in one launch
// (bands of the table to the XCDs).  A marching wave with two steps a launch (batch_tmz_step2) moves
// each cell's state every second step, here it is every eighth (FP64: fourth): 241 -> 196 us a step
// for 64 simulations of 5.7e7 cells in FP32, 24 -> 8.8 us for 4 of 2.4e6.
template <typename T>
__global__ __launch_bounds__ (64 * BATCH_WAVES (T), 4)
void batch_plane_steps (const StepArgs<T> *sims, const int4 *tiles, int ntiles, int per_xcd, const int *state,
                        const T *src_tab, int src_len, int off, int flip, int n)
{
  using S = Plane<YEE_SCHEME_TMZ>;
  constexpr int RW = BATCH_RW (T), NW = BATCH_WAVES (T), K = BATCH_STEPS (T);
  static_assert (RW * NW - 2 * K == kBatchRows, "tile rows");
  __shared__ T xlo[NW + 1][64], xhi[NW + 1][64];
  const int b = (int) blockIdx.x, u = (b & 7) * per_xcd + (b >> 3);
  if (u >= ntiles) return;   // the whole workgroup
  const int4 td = tiles[u];
  const int t = state[2 * td.x] + off;
  // a private copy: loads through a reference could not be kept across the tile's stores
  const StepArgs<T> a = sims[2 * td.x + (state[2 * td.x + 1] ^ flip)];
  const T *st = src_tab + ((int64_t) td.x * src_len + t) * 2;
  TileJob<T> job;
  job.margin = K;
  job.rows = kBatchRows;
  job.cols = 64 - 2 * K;
  job.x0 = td.y;
  job.y0 = td.z;
  job.n = n;
  auto value = [&] (int s, int half) { return gld (st + 2 * s + half); };
  TileFaces<RW * NW> *none = nullptr;
  if (tile_pml<T, S> (a, td.y - K, td.z - K, RW * NW, 64))
    tile_steps<T, S, RW, NW, true, false> (a, job, xlo, xhi, none, value);
  else
    tile_steps<T, S, RW, NW, false, false> (a, job, xlo, xhi, none, value);
}

template <typename T>
void launch_batch_plane (const StepArgs<T> *sims, const int4 *tiles, int ntiles, const int *state, const T *src_tab,
                         int src_len, int off, int flip, int n, hipStream_t stream)
{
  const int per = (ntiles + 7) / 8;
  hipLaunchKernelGGL ((batch_plane_steps<T>), dim3 ((unsigned) (8 * (per > 0 ? per : 1))), dim3 (64 * BATCH_WAVES (T)), 0,
                     stream, sims, tiles, ntiles, per, state, src_tab, src_len, off, flip, n);
}
template void launch_batch_plane<float> (const StepArgs<float> *, const int4 *, int, const int *, const float *, int, int, int,
                                         int, hipStream_t);
template void launch_batch_plane<double> (const StepArgs<double> *, const int4 *, int, const int *, const double *, int, int,
                                          int, int, hipStream_t);

// The D/B -> field factors of the updated PML cells of one component.
template <typename T, class S, int COMP>
__device__ __forceinline__ void plane_factor (const StepArgs<T> &a, const int p[3], int64_t r0, int j, int64_t rs)
{
  const size_t L = (size_t) a.tab_len;
  const T *tab = a.pml + COMP * 6 * L;
  const Pair<T> s4 = gld2 (tab + 2 * L + 2 * p[SigAxes<COMP>::s4]);
  const Pair<T> s5 = gld2 (tab + 4 * L + 2 * p[SigAxes<COMP>::s5]);
  const Pair<T> k = pml_factors (s4.a, s4.b, tile_mat<T, S, COMP> (a, r0, (uint32_t) j * (uint32_t) sizeof (T), rs) * (COMP >= 3 ? a.mu0 : a.eps0), s5.b);
  gst ((T *) a.pfac[COMP] + 2 * (r0 + j), k.a);
  gst ((T *) a.pfac[COMP] + 2 * (r0 + j) + 1, k.b);
}

template <typename T, int SCHEME>
__global__ __launch_bounds__ (256) void plane_factors (StepArgs<T> a)
{
  using S = Plane<SCHEME>;
  const int nr = S::ra == 0 ? a.nx : a.ny, nc = S::ca == 1 ? a.ny : a.nz;
  const int64_t rs = S::ra == 0 ? a.sx : (int64_t) a.sy;
  const int64_t n = (int64_t) nr * nc;
  for (int64_t u = blockIdx.x * (int64_t) 256 + threadIdx.x; u < n; u += (int64_t) gridDim.x * 256)
  {
    const int i = (int) (u / nc), j = (int) (u - (int64_t) i * nc);
    if (i < 1 || i >= nr - 1 || j < 1 || j >= nc - 1) continue;
    if (i >= a.slab_lo[S::ra] && i < a.slab_hi[S::ra] && j >= a.slab_lo[S::ca] && j < a.slab_hi[S::ca]) continue;
    int p[3] = { 0, 0, 0 };
    p[S::ra] = i;
    p[S::ca] = j;
    plane_factor<T, S, S::cc> (a, p, i * rs, j, rs);
    plane_factor<T, S, S::cr> (a, p, i * rs, j, rs);
    plane_factor<T, S, S::ck> (a, p, i * rs, j, rs);
  }
}

template <typename T, int SCHEME>
void launch_plane_scheme (const StepArgs<T> &a, const PlaneGrid &g, const PlaneSource &src, hipStream_t stream)
{
  const dim3 grid ((unsigned) (8 * g.per_xcd)), block (64 * g.waves);
  constexpr int RW = PLANE_RW (T), NS = kPlaneWavesSmall, NL = kPlaneWaves;
  if (g.waves == NS && a.tfsf)
    hipLaunchKernelGGL ((plane_steps<T, SCHEME, true, NS>), grid, block, sizeof (TileFaces<RW * NS>), stream, a, g, src);
  else if (g.waves == NS)
    hipLaunchKernelGGL ((plane_steps<T, SCHEME, false, NS>), grid, block, 0, stream, a, g, src);
  else if (a.tfsf)
    hipLaunchKernelGGL ((plane_steps<T, SCHEME, true, NL>), grid, block, sizeof (TileFaces<RW * NL>), stream, a, g, src);
  else
    hipLaunchKernelGGL ((plane_steps<T, SCHEME, false, NL>), grid, block, 0, stream, a, g, src);
}

#define YEE_PLANES(X) X (YEE_SCHEME_TEX) X (YEE_SCHEME_TEY) X (YEE_SCHEME_TEZ) X (YEE_SCHEME_TMX) X (YEE_SCHEME_TMY) X (YEE_SCHEME_TMZ)

template <typename T>
void launch_plane (int scheme, const StepArgs<T> &a, const PlaneGrid &g, const PlaneSource &src, hipStream_t stream)
{
#define YEE_PLANE(S) case S: launch_plane_scheme<T, S> (a, g, src, stream); break;
  switch (scheme)
  {
    YEE_PLANES (YEE_PLANE)
    default: break;
  }
#undef YEE_PLANE
}

template <typename T>
void launch_plane_factors (int scheme, const StepArgs<T> &a, hipStream_t stream)
{
  const int64_t n = (int64_t) a.nx * a.ny * a.nz;
  const dim3 grid ((unsigned) (n / 256 + 1 < 4096 ? n / 256 + 1 : 4096)), block (256);
#define YEE_PLANE(S) case S: hipLaunchKernelGGL ((plane_factors<T, S>), grid, block, 0, stream, a); break;
  switch (scheme)
  {
    YEE_PLANES (YEE_PLANE)
    default: break;
  }
#undef YEE_PLANE
}

// ---------------------------------------------------------------------------------------
// Up to kIncSteps steps of a 1D run in one launch.
//
// A line has a few thousand cells at most in practice, so a step is pure latency: three launches
// took 25 us of it.  As in incident_steps, a wave owns 192 cells and keeps them with a margin of
// kIncSteps cells on either side in registers, four to a lane; neighbours come from the next lane
// (DPP), with no LDS, no barrier and no memory access between the first and the last step.  The
// coefficients of a cell are divided out once a launch, and lane s holds the TF/SF corrections of
// step s.  Operands and order are those of e_half_cell / h_half_cell.
// ---------------------------------------------------------------------------------------
template <int SCHEME>
struct Line
{
  static constexpr int ea = (SCHEME - YEE_SCHEME_EXHY) / 2;                            // Ex Ex Ey Ey Ez Ez
  static constexpr int ha = SCHEME == YEE_SCHEME_EXHY || SCHEME == YEE_SCHEME_EZHY ? 1
                            : (SCHEME == YEE_SCHEME_EXHZ || SCHEME == YEE_SCHEME_EYHZ ? 2 : 0);
  static constexpr int axis = 3 - ea - ha;
  static constexpr int ce = ea, ch = 3 + ha;
  static constexpr bool pos = axis == (ea + 1) % 3;   // curl: + d H and + d E, else both negated
};

// One component of a lane's cells.
template <typename T>
struct LineComp
{
  T f[4], d[4], k[4], cac[4], cbc[4], ca5[4];
};

template <typename T, class S, int COMP>
__device__ __forceinline__ void line_load (const StepArgs<T> &a, int first, int n, uint32_t sp, LineComp<T> &x)
{
  const T modc = COMP >= 3 ? a.mu0 : a.eps0;
  const T *m = COMP < 3 ? a.eps : a.mu;
  const size_t L = (size_t) a.tab_len;
  const T *tab = a.pml + COMP * 6 * L;
#pragma unroll
  for (int c = 0; c < 4; ++c)
  {
    const int i = max (0, min (first + c, n - 2));   // (the last cell is always zero)
    const bool in = first + c >= 0 && first + c < n - 1;
    const T f = gld (a.f[COMP] + i);
    x.f[c] = in ? f : (T) 0;
    T mat = COMP < 3 ? a.eps_u : a.mu_u;
    if (a.matc[COMP]) mat = gld (a.matc[COMP] + i);
    else if (m && COMP < 3) mat = gld (m + i);                       // 2-cell average of one cell
    else if (m) mat = avg2 (gld (m + i), gld (m + i + 1));           // 4-cell average of two
    x.k[c] = direct_cb (a.dt, mat, modc, a.dx);
    x.d[c] = x.cac[c] = x.cbc[c] = x.ca5[c] = (T) 0;
    if ((sp >> c) & 1u)
    {
      // the component's own axis is not the line's: p4 == m4 and the two factors are one
      const Pair<T> cu = gld2 (tab + 2 * (SigAxes<COMP>::c == S::axis ? i : 0));
      const Pair<T> s4 = gld2 (tab + 2 * L), s5 = gld2 (tab + 4 * L + 2 * (SigAxes<COMP>::s5 == S::axis ? i : 0));
      x.d[c] = gld (a.d[COMP] + i);
      x.cac[c] = cu.a;
      x.cbc[c] = cu.b;
      x.ca5[c] = s5.a;
      x.k[c] = pml_factors (s4.a, s4.b, mat * modc, s5.b).a;
    }
  }
}

template <typename T>
__device__ __forceinline__ void line_update (LineComp<T> &x, int c, T tmp, uint32_t upd, uint32_t sp)
{
  const T direct = x.f[c] * (T) 1.0 + tmp * x.k[c];
  const T d = x.d[c] * x.cac[c] + tmp * x.cbc[c];
  const T pml = x.f[c] * x.ca5[c] + d * x.k[c] - x.d[c] * x.k[c];
  const bool s = (sp >> c) & 1u, u = (upd >> c) & 1u;
  x.f[c] = s ? pml : (u ? direct : x.f[c]);
  x.d[c] = s ? d : x.d[c];
}

// The value of lane s (uniform).
__device__ __forceinline__ double lane_value (double v, int s)
{
  int2 w = __builtin_bit_cast (int2, v);
  w.x = __builtin_amdgcn_readlane (w.x, s);
  w.y = __builtin_amdgcn_readlane (w.y, s);
  return __builtin_bit_cast (double, w);
}

template <typename T, int SCHEME>
__global__ __launch_bounds__ (64) void line_steps (StepArgs<T> a, int steps, LineSource src)
{
  using S = Line<SCHEME>;
  const int lane = (int) threadIdx.x;
  const int n = S::axis == 0 ? a.nx : (S::axis == 1 ? a.ny : a.nz);
  const int base = 1 + (int) blockIdx.x * kIncTile - kIncSteps, first = base + 4 * lane;
  const bool mine = lane >= kIncSteps / 4 && lane < 64 - kIncSteps / 4;
  uint32_t upd = 0, sp = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c)
  {
    const int i = first + c;
    const bool u = i >= 1 && i < n - 1;
    upd |= u ? 1u << c : 0u;
    sp |= a.pml && u && (i < a.slab_lo[S::axis] || i >= a.slab_hi[S::axis]) ? 1u << c : 0u;
  }
  LineComp<T> E, H;
  line_load<T, S, S::ce> (a, first, n, sp, E);
  line_load<T, S, S::ch> (a, first, n, sp, H);
  // TF/SF: E on cells L-1 (operand H at L-1) and R (H at R-1), H on L-1 (E at L-1) and R-1 (E at R)
  const int lo = a.tl[S::axis] - 1, hi = a.tr[S::axis];
  const bool face = a.tfsf && ((lo >= base && lo < base + 256) || (hi >= base && hi <= base + 256));
  double e_lo = 0, e_hi = 0, h_lo = 0, h_hi = 0;
  if (face && lane < steps)
  {
    constexpr int pe = (Tab::dir[S::ce][0] >> 1) == S::axis ? 0 : 1, ph = (Tab::dir[S::ch][0] >> 1) == S::axis ? 0 : 1;
    StepArgs<T> b = a;
    b.einc = a.einc + lane * a.inc_len;
    b.hinc = a.hinc + lane * a.inc_len;
    double skip;
    int p[3] = { 0, 0, 0 };
    p[S::axis] = lo;
    tfsf_pair_diff<T, S::ce, pe, 3> (b, p[0], p[1], p[2], skip, e_lo);
    tfsf_pair_diff<T, S::ch, ph, 3> (b, p[0], p[1], p[2], h_lo, skip);
    p[S::axis] = hi;
    tfsf_pair_diff<T, S::ce, pe, 3> (b, p[0], p[1], p[2], e_hi, skip);
    p[S::axis] = hi - 1;
    tfsf_pair_diff<T, S::ch, ph, 3> (b, p[0], p[1], p[2], skip, h_hi);
  }
  const int at = a.src_mask ? a.src_pos[S::axis] - first : -1;   // the hard source among the lane's cells
  const bool se = (a.src_mask >> S::ce) & 1u, sh = (a.src_mask >> S::ch) & 1u;
  for (int s = 0; s < steps; ++s)
  {
    {
      T before = lane_prev (H.f[3], H.f[3]);
      const double dl = face ? lane_value (e_lo, s) : 0.0, dh = face ? lane_value (e_hi, s) : 0.0;
#pragma unroll
      for (int c = 0; c < 4; ++c)
      {
        T m = before, z = H.f[c];
        before = z;
        if (face && first + c == lo) z = (T) ((double) z - dl);
        if (face && first + c == hi) m = (T) ((double) m - dh);
        line_update (E, c, S::pos ? z - m : m - z, upd, sp);
        if (se && c == at) E.f[c] = (T) src.v[s][0];
      }
    }
    {
      T after = lane_next (E.f[0], E.f[0]);
      const double dl = face ? lane_value (h_lo, s) : 0.0, dh = face ? lane_value (h_hi, s) : 0.0;
#pragma unroll
      for (int c = 3; c >= 0; --c)
      {
        T p = after, z = E.f[c];
        after = z;
        if (face && first + c == lo) z = (T) ((double) z - dl);
        if (face && first + c == hi - 1) p = (T) ((double) p - dh);
        line_update (H, c, S::pos ? p - z : z - p, upd, sp);
        if (sh && c == at) H.f[c] = (T) src.v[s][1];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
  {
    if (!mine || !((upd >> c) & 1u)) continue;
    gst (a.f_n[S::ce] + first + c, E.f[c]);
    gst (a.f_n[S::ch] + first + c, H.f[c]);
    if ((sp >> c) & 1u)
    {
      gst (a.d_n[S::ce] + first + c, E.d[c]);
      gst (a.d_n[S::ch] + first + c, H.d[c]);
    }
  }
}

template <typename T>
void launch_line (int scheme, const StepArgs<T> &a, int n, const LineSource &src, hipStream_t stream)
{
  const int64_t cells = (int64_t) a.nx * a.ny * a.nz;
  const dim3 grid ((unsigned) ((cells - 2 + kIncTile - 1) / kIncTile)), block (64);
#define YEE_LINE(S) case S: hipLaunchKernelGGL ((line_steps<T, S>), grid, block, 0, stream, a, n, src); break;
  switch (scheme)
  {
    YEE_LINE (YEE_SCHEME_EXHY)
    YEE_LINE (YEE_SCHEME_EXHZ)
    YEE_LINE (YEE_SCHEME_EYHX)
    YEE_LINE (YEE_SCHEME_EYHZ)
    YEE_LINE (YEE_SCHEME_EZHX)
    YEE_LINE (YEE_SCHEME_EZHY)
    default: break;
  }
#undef YEE_LINE
}

template void launch_line<float> (int, const StepArgs<float> &, int, const LineSource &, hipStream_t);
template void launch_line<double> (int, const StepArgs<double> &, int, const LineSource &, hipStream_t);
template void launch_plane<float> (int, const StepArgs<float> &, const PlaneGrid &, const PlaneSource &, hipStream_t);
template void launch_plane<double> (int, const StepArgs<double> &, const PlaneGrid &, const PlaneSource &, hipStream_t);
template void launch_plane_factors<float> (int, const StepArgs<float> &, hipStream_t);
template void launch_plane_factors<double> (int, const StepArgs<double> &, hipStream_t);

}  // namespace yee
