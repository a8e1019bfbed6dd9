// Batched complex 5x5 block-pentadiagonal line solvers for gfx950.
//
// Replaces src/cpenta1bc.f, src/cpenta2bc.f (non-periodic, boundary
// wrap-around storage) and src/cpenta1p.f, src/cpenta2p.f (periodic,
// bordered).  Three stages:
//
//  1. Non-pivoted block LU.  Non-periodic lines: k_factor_chains, one wave
//     per chain of rows, the rows being updated in registers (interior rows)
//     or in an LDS window (rows next to an end; lines of 16+ rows, when there
//     are few lines, use a twisted order: two chains per line meeting in the
//     middle).  Periodic lines: k_lu_per, one wave
//     per line on a line-interleaved copy.  The storage of negated
//     multipliers and the in-pivot order follow the reference
//     (cpenta1bc.f:43-495, cpenta1p.f:46-654), including the periodic
//     factor's slot-4 placement at cpenta1p.f:284/345 unless exact is
//     requested.
//  2. k_records_rows: for non-periodic lines, turn row i's factors into the
//     records the fast solve streams:
//        forward   y_i = Linv_i b_i + N1_i y_{i-2} + N2_i y_{i-1}
//        backward  x_i = Uinv_i y_i + Q4_i x_{i+1} + Q5_i x_{i+2}
//     with Linv_i/Uinv_i the inverses of the in-block unit-lower / upper
//     factors, N = Linv * (negated multiplier block), Q = -Uinv * (upper
//     block).  Mathematically the reference's forward/back substitution
//     (cpenta1bc.f:499-847); the per-row critical path becomes one 5x5
//     matvec.  Boundary rows 0,1 and n-2,n-1 carry extra blocks, kept in a
//     per-line tail record.
//  3. k_line_solve (line_solve.hpp): one wave runs two chains of rows (a
//     twisted line's halves, or two plain lines), one component's real or
//     imaginary part per lane; three waves stream the records through an LDS
//     ring and compute the parallel parts (Linv b, Uinv y).
//  Periodic lines: k_records_per forms the same records from the bordered
//  LU plus two border blocks per row (p2: rows n-2, n-1 in column i; qp:
//  row i in columns n-2, n-1), and k_line_solve_per streams them in pairs of
//  lines with the border sums formed by the loader waves.  k_solve_lines (one lane
//  per line, the reference's substitution order on the LU working copy) is
//  kept as the order-exact solve behind lns3d_penta_solve_reference_order.
#include <algorithm>
#include <climits>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "common.hpp"
#include "line_solve.hpp"
#include "penta.hpp"

namespace lns3d {

// ---------------------------------------------------------------------------
// block addressing in the LU working copy.  Periodic lines: line-interleaved
// ([row][slot][r][c][line], one wave per line in k_lu_per); non-periodic
// lines: line-major ([line][row][slot][r][c], one wave per chain in
// k_factor_chains).  Element (r,c) of a block = p[(r*5 + c) * ldl].
template <typename T> struct Blk {
  cx<T> *p;
  __device__ __forceinline__ cx<T> &operator()(int r, int c) const { return p[(long)(r * 5 + c) * ldl]; }
  long ldl;
};

struct LineGeom {
  int n;         // unknown rows (np-1 for periodic)
  int periodic;
  int exact;
  long L;        // lines (interleave stride)
  int h = -1;    // twisted factor (non-periodic): rows 0..h+1 top-down after
                 // rows n-1..h+2 bottom-up; -1: rows in order 0..n-1
};

// the slot of column c in row i of a line, -1 if it has none: slot k holds
// column i - 2 + k, and the two rows next to an end hold the line's first or
// last five columns, wrapped.  In arithmetic: a table would be a load from
// memory for each look-up.
__device__ __forceinline__ int bc_slot(int n, int i, int c) {
  const int lo = i < 2 ? 0 : i > n - 3 ? n - 5 : i - 2;
  const int k = c - i + 2;
  return (c < lo || c > lo + 4) ? -1 : k < 0 ? k + 5 : k > 4 ? k - 5 : k;
}

// where block (row i, column c) lives; false if structurally zero
template <typename T>
__device__ __forceinline__ bool blk(const LineGeom &g, cx<T> *mat, cx<T> *per, cx<T> *per2,
                                    long line, int i, int c, Blk<T> &b) {
  b.ldl = g.L;
  const int n = g.n;
  if (!g.periodic) {
    int k = bc_slot(n, i, c);
    if (k < 0) return false;
    b.p = mat + ((line * n + i) * 5 + k) * 25;
    b.ldl = 1;
    return true;
  }
  int d = c - i;
  if (d >= -2 && d <= 2 && c >= 0 && c < n) {
    b.p = mat + ((long)(i * 5 + d + 2) * 25) * g.L + line;
    return true;
  }
  if ((c == n - 2 || c == n - 1) && i < c - 2) {
    b.p = per + ((long)(i * 2 + (c - (n - 2))) * 25) * g.L + line;
    return true;
  }
  if ((i == n - 2 || i == n - 1) && c < i - 2) {
    b.p = per2 + ((long)(c * 2 + (i - (n - 2))) * 25) * g.L + line;
    return true;
  }
  return false;
}

// rows (and columns) that a pivot on row i eliminates from / updates: the
// not yet pivoted neighbours in the pivot direction (dir +1: below, -1: above)
__device__ __forceinline__ int partners(const LineGeom &g, int i, int dir, int *cand) {
  int k = 0;
  const int hi = (g.h >= 0 && dir > 0) ? g.h + 1 : g.n - 1;   // twisted top phase stops at h+1
  for (int d = 1; d <= 4; d++) {
    int t = i + dir * d;
    if (t >= 0 && t <= hi) cand[k++] = t;
  }
  if (g.periodic)
    for (int e = g.n - 2; e < g.n; e++)
      if (e > i + 4) cand[k++] = e;
  return k;
}


// ---------------------------------------------------------------------------
// stage 1 for periodic lines, one wave per line: the bordered block LU in
// the reference's order (cpenta1p.f:46-654): pivots 0..n-1, each with its
// partner rows i+1..i+4 and the border rows n-2, n-1 (partners()), the
// storage of blk() and the fill-in placement of the shipped factor unless
// exact is requested; every element receives its operations in the
// reference's order.  Per pivot, the blocks it touches
// -- the pivot row's diagonal and right blocks, and each partner row's
// blocks in the pivot column and in the right blocks' columns (at most 49)
// -- are brought into LDS, eliminated there (the in-block steps and the
// partner steps each in two phases: multipliers, then one element per
// task), and written back.
constexpr int LUP_SLOTS = 49;    // 0 D, 1..6 right blocks, 7 + 7a + b partner a (b 0: pivot column)
__global__ __launch_bounds__(64) void k_lu_per(LineGeom g, cx<double> *mat, cx<double> *per, cx<double> *per2) {
  using T = double;
  __shared__ cx<T> blkv[LUP_SLOTS][25];
  __shared__ cx<T> *bptr[LUP_SLOTS];      // the slots' blocks in HBM (null: no such block)
  __shared__ cx<T> mlt[6][5];
  const long line = blockIdx.x;
  const int lane = threadIdx.x;
  const int n = g.n, np = n + 1;
  const long L = g.L;
  // bordered fill-in storage (cpenta1p.f:53-78)
  for (long e = lane; e < (long)np * 50; e += 64) {
    per[e * L + line] = cx<T>{0, 0};
    per2[e * L + line] = cx<T>{0, 0};
  }
  __builtin_amdgcn_s_waitcnt(0);
  wave_sync();
  if (lane < 25) {
    const int e = lane;
    per[((long)(0 * 2 + 0) * 25 + e) * L + line] = mat[((long)(0 * 5 + 0) * 25 + e) * L + line];
    per[((long)(0 * 2 + 1) * 25 + e) * L + line] = mat[((long)(0 * 5 + 1) * 25 + e) * L + line];
    per[((long)(1 * 2 + 1) * 25 + e) * L + line] = mat[((long)(1 * 5 + 0) * 25 + e) * L + line];
    per2[((long)(0 * 2 + 0) * 25 + e) * L + line] = mat[((long)((n - 2) * 5 + 4) * 25 + e) * L + line];
    per2[((long)(0 * 2 + 1) * 25 + e) * L + line] = mat[((long)((n - 1) * 5 + 3) * 25 + e) * L + line];
    per2[((long)(1 * 2 + 1) * 25 + e) * L + line] = mat[((long)((n - 1) * 5 + 4) * 25 + e) * L + line];
  }
  __builtin_amdgcn_s_waitcnt(0);
  wave_sync();
  for (int i = 0; i < n; i++) {
    // candidates a = 0..5: rows / columns i+1..i+4 in the line, then the
    // border rows / columns n-2, n-1 beyond i+4 (partners(), dir +1)
    auto cand = [&](int a) {
      const int t = a < 4 ? i + 1 + a : n - 6 + a;
      const bool ok = a < 4 ? t <= n - 1 : t > i + 4;
      return ok ? t : -1;
    };
    // where slot k lives in HBM (false: no such block); uniform over the wave
    auto where = [&](int k, Blk<T> &B) -> bool {
      if (k == 0) return blk(g, mat, per, per2, line, i, i, B);
      if (k <= 6) {
        const int c = cand(k - 1);
        return c >= 0 && blk(g, mat, per, per2, line, i, c, B);
      }
      const int a = (k - 7) / 7, bb = (k - 7) % 7, t = cand(a);
      Blk<T> Lb;
      if (t < 0 || !blk(g, mat, per, per2, line, t, i, Lb)) return false;   // not a partner
      if (bb == 0) { B = Lb; return true; }
      Blk<T> U;
      const int c = cand(bb - 1);
      if (c < 0 || !blk(g, mat, per, per2, line, i, c, U)) return false;    // no right block there
      if (!blk(g, mat, per, per2, line, t, c, B)) return false;
      if (!g.exact && i == n - 6 && t == n - 4 && c == n - 2)             // cpenta1p.f:284, 345
        B.p = mat + ((long)(t * 5 + 3) * 25) * L + line;
      return true;
    };
    // the slots' addresses, one lane per slot, then the blocks into LDS (all
    // loads in flight at once)
    if (lane < LUP_SLOTS) {
      Blk<T> B;
      bptr[lane] = where(lane, B) ? B.p : nullptr;
    }
    wave_sync();
    constexpr int PER_LANE = (LUP_SLOTS * 25 + 63) / 64;
    cx<T> tmp[PER_LANE];
#pragma unroll
    for (int r = 0; r < PER_LANE; r++) {
      const int e = r * 64 + lane, k = e / 25, el = e % 25;
      const cx<T> *bp = e < LUP_SLOTS * 25 ? bptr[k] : nullptr;
      tmp[r] = bp ? bp[(long)el * L] : cx<T>{0, 0};
    }
#pragma unroll
    for (int r = 0; r < PER_LANE; r++) {
      const int e = r * 64 + lane;
      if (e < LUP_SLOTS * 25) blkv[e / 25][e % 25] = tmp[r];
    }
    wave_sync();
    // slot existence, uniform: right blocks and partners
    unsigned uok = 0, pok = 0;
#pragma unroll
    for (int u = 0; u < 6; u++) {
      if (bptr[1 + u]) uok |= 1u << u;
      if (bptr[7 + 7 * u]) pok |= 1u << u;
    }
    cx<T> *D = blkv[0];
    // in-block LU of D, its row operations applied to the right blocks
    for (int nc = 0; nc < 4; nc++) {
      if (lane < 4 - nc) {
        const int l = nc + 1 + lane;
        const cx<T> mult = -cdiv(D[l * 5 + nc], D[nc * 5 + nc]);
        mlt[0][l] = mult;
        D[l * 5 + nc] = mult;
      }
      wave_sync();
      const int nt = (4 - nc) * 5 * 7;          // tasks (l, q, b): b 0 D (q > nc), 1 + u right block u
      for (int tk = lane; tk < nt; tk += 64) {
        const int l = nc + 1 + tk / 35, q = (tk / 7) % 5, b = tk % 7;
        const cx<T> mult = mlt[0][l];
        if (b == 0) {
          if (q > nc) D[l * 5 + q] = cfma(mult, D[nc * 5 + q], D[l * 5 + q]);
        } else if (uok >> (b - 1) & 1) {
          cx<T> *U = blkv[b];
          U[l * 5 + q] = cfma(mult, U[nc * 5 + q], U[l * 5 + q]);
        }
      }
      wave_sync();
    }
    // partner rows: the block in the pivot column becomes the multipliers,
    // the partner's blocks in the right blocks' columns are updated
    for (int nc = 0; nc < 5; nc++) {
      if (lane < 30) {
        const int a = lane / 5, m = lane % 5;
        if (pok >> a & 1) {
          cx<T> *Lb = blkv[7 + 7 * a];
          const cx<T> fact = crecip(D[nc * 5 + nc]);
          const cx<T> mult = -(Lb[m * 5 + nc] * fact);
          mlt[a][m] = mult;
          Lb[m * 5 + nc] = mult;
        }
      }
      wave_sync();
      const int nt = 6 * 5 * 5 * 7;             // tasks (a, m, q, b)
      for (int tk = lane; tk < nt; tk += 64) {
        const int a = tk / 175, m = (tk / 35) % 5, q = (tk / 7) % 5, b = tk % 7;
        if (!(pok >> a & 1)) continue;
        const cx<T> mult = mlt[a][m];
        cx<T> *Lb = blkv[7 + 7 * a];
        if (b == 0) {
          if (q > nc) Lb[m * 5 + q] = cfma(mult, D[nc * 5 + q], Lb[m * 5 + q]);
        } else if (uok >> (b - 1) & 1) {
          cx<T> *Dst = blkv[7 + 7 * a + b];
          Dst[m * 5 + q] = cfma(mult, blkv[b][nc * 5 + q], Dst[m * 5 + q]);
        }
      }
      wave_sync();
    }
    // write the blocks back; the next pivot reads them after the stores
#pragma unroll
    for (int r = 0; r < PER_LANE; r++) {
      const int e = r * 64 + lane, k = e / 25, el = e % 25;
      cx<T> *bp = e < LUP_SLOTS * 25 ? bptr[k] : nullptr;
      if (bp) bp[(long)el * L] = blkv[k][el];
    }
    __builtin_amdgcn_s_waitcnt(0);
    wave_sync();
  }
}

// ---------------------------------------------------------------------------
// periodic (and reference-order) solve, one lane per line, in place on the
// rhs array: element (row i, comp m) of line l at rhs[(l*sL + i*sR)*5 + m]
template <typename T>
__global__ void k_solve_lines(LineGeom g, const cx<T> *mat_, const cx<T> *per_, const cx<T> *per2_,
                              double2 *rhs, long sL, long sR) {
  long line = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (line >= g.L) return;
  cx<T> *mat = const_cast<cx<T> *>(mat_), *per = const_cast<cx<T> *>(per_),
        *per2 = const_cast<cx<T> *>(per2_);
  const int n = g.n;
  auto X = [&](int i, int d) -> double2 & { return rhs[(line * sL + (long)i * sR) * 5 + d]; };
  int cand[8];
  for (int i = 0; i < n; i++) {
    Blk<T> D;
    blk(g, mat, per, per2, line, i, i, D);
    cx<T> x[5];
    for (int d = 0; d < 5; d++) x[d] = cx<T>{(T)X(i, d).x, (T)X(i, d).y};
    for (int nc = 0; nc < 4; nc++)
      for (int l = nc + 1; l < 5; l++) x[l] = cfma(D(l, nc), x[nc], x[l]);
    for (int d = 0; d < 5; d++) X(i, d) = make_double2(x[d].re, x[d].im);
    int nc_ = partners(g, i, 1, cand);
    for (int a = 0; a < nc_; a++) {
      Blk<T> Lb;
      int t = cand[a];
      if (!blk(g, mat, per, per2, line, t, i, Lb)) continue;
      for (int m = 0; m < 5; m++) {
        cx<T> acc = cx<T>{(T)X(t, m).x, (T)X(t, m).y};
        for (int nc = 0; nc < 5; nc++) acc = cfma(Lb(m, nc), x[nc], acc);
        X(t, m) = make_double2(acc.re, acc.im);
      }
    }
  }
  for (int i = n - 1; i >= 0; i--) {
    Blk<T> D;
    blk(g, mat, per, per2, line, i, i, D);
    cx<T> acc[5];
    for (int d = 0; d < 5; d++) acc[d] = cx<T>{(T)X(i, d).x, (T)X(i, d).y};
    int nc_ = partners(g, i, 1, cand);
    for (int a = 0; a < nc_; a++) {
      Blk<T> U;
      int c = cand[a];
      if (!blk(g, mat, per, per2, line, i, c, U)) continue;
      cx<T> xc[5];
      for (int d = 0; d < 5; d++) xc[d] = cx<T>{(T)X(c, d).x, (T)X(c, d).y};
      for (int m = 0; m < 5; m++)
        for (int q = 0; q < 5; q++) acc[m] = cfma(-U(m, q), xc[q], acc[m]);
    }
    for (int m = 4; m >= 0; m--) {
      for (int q = m + 1; q < 5; q++) acc[m] = cfma(-D(m, q), acc[q], acc[m]);
      acc[m] = cdiv(acc[m], D(m, m));
    }
    for (int d = 0; d < 5; d++) X(i, d) = make_double2(acc[d].re, acc[d].im);
  }
  if (g.periodic)
    for (int d = 0; d < 5; d++) X(n, d) = X(0, d);
}

// ---------------------------------------------------------------------------
// stage 2: records for the fast non-periodic solve
// fwd[(line*n + i)*60 + ...]: 50 complex of N2 and N1, a component's rows as
//                           20 reals (rec_pos); 50 + k -> strict lower of
//                           Linv, k = l*(l-1)/2 + q
// bwd[(line*n + i)*66 + ...] (one complex of padding): Q4 and Q5 likewise;
//                           50 + k -> upper of Uinv (row-major, incl. diagonal)
// tail[line*150 + ...]: 0 row n-2 N(col n-5); 25 row n-1 N(col n-5);
//                       50 row n-1 N(col n-4); 75 row 0 Q(col 3);
//                       100 row 0 Q(col 4); 125 row 1 Q(col 4)   ([m][q])
// Records of (line, chain row)s: eight per workgroup, 32 lanes each (a row
// and its inverses in LDS; lane (m, q) = (l / 5, l % 5) of lanes 0..24 forms
// entry (m, q) of a block).  The row's five LU blocks are read with
// consecutive lanes on consecutive entries; with flags, the line's flag is set
// on the way if one of them is unhealthy (a pass of its own over the factors
// took 58 us at 257 lines of 513 rows).
template <typename TF, typename TR>
__global__ __launch_bounds__(256) void k_records_rows(LineGeom g, const cx<TF> *mat, cx<TR> *fwd, cx<TR> *bwd,
                                                      cx<TR> *tail, int *flags) {
  __shared__ cx<TF> rowb[8][125];
  __shared__ cx<TF> Lis[8][25], Uis[8][25];
  const int n = g.n;
  const int grp = threadIdx.x >> 5, gl = threadIdx.x & 31;
  const long idx0 = (long)blockIdx.x * 8 + grp;
  const bool valid = idx0 < g.L * n;
  const long idx = valid ? idx0 : g.L * n - 1;        // idle groups repeat the last row, store nothing
  const long line = idx / n;
  const int jj = (int)(idx - line * n);
  const bool tw = g.h >= 0;
  const int nchain = tw ? 2 : 1;
  // chain t: rows in elimination order; t = 1 runs bottom-up (row n-1-j)
  const int t = (tw && jj >= g.h + 2) ? 1 : 0;
  const int j = t == 0 ? jj : jj - (g.h + 2);
  const int len = tw ? (t == 0 ? g.h + 2 : n - g.h - 2) : n;
  const int dir = t == 0 ? 1 : -1;
  const int i = t == 0 ? j : n - 1 - j;
  cx<TF> *rb = rowb[grp];
  const cx<TF> *src = mat + ((line * n + i) * 125);
  bool bad = false;                // the row's share of the line's health (k_check_factor)
  for (int e = gl; e < 125; e += 32) {
    const cx<TF> x = src[e];
    rb[e] = x;
    bad |= !(isfinite(x.re) && isfinite(x.im)) || (e / 25 == 2 && e % 25 % 6 == 0 && x.re == 0 && x.im == 0);
  }
  if (flags && bad) flags[line] = 1;
  const int m = gl / 5, q = gl % 5;
  const bool act = gl < 25;
  const int sd = bc_slot(n, i, i) * 25;
  if (act) Lis[grp][gl] = cx<TF>{TF(m == q), 0};
  wave_sync();
  // Linv: the in-block elimination steps applied to I
#pragma unroll
  for (int nc = 0; nc < 4; nc++) {
    if (act && m > nc && q <= nc) Lis[grp][gl] = cfma(rb[sd + m * 5 + nc], Lis[grp][nc * 5 + q], Lis[grp][gl]);
    wave_sync();
  }
  // Uinv by back substitution on identity columns (lane c < 5: column c)
  if (gl < 5) {
    const int c = gl;
    cx<TF> u[5];
#pragma unroll
    for (int r = 0; r < 5; r++) u[r] = cx<TF>{0, 0};
#pragma unroll
    for (int mm = 4; mm >= 0; mm--)
      if (mm <= c) {
        cx<TF> acc = cx<TF>{TF(mm == c), 0};
#pragma unroll
        for (int k = mm + 1; k < 5; k++)
          if (k <= c) acc = cfma(-rb[sd + mm * 5 + k], u[k], acc);
        u[mm] = cdiv(acc, rb[sd + mm * 5 + mm]);
      }
#pragma unroll
    for (int r = 0; r < 5; r++) Uis[grp][r * 5 + c] = u[r];
  }
  wave_sync();
  const cx<TF> *Li = Lis[grp], *Ui = Uis[grp];
  // entry (m, q) of Linv * M(i, col) (a multiplier block), zero if col has none
  auto Nent = [&](int col) {
    cx<TF> acc{0, 0};
    const int sl = (col >= 0 && col < n) ? bc_slot(n, i, col) : -1;
    if (sl >= 0)
      for (int k = 0; k <= m; k++) acc = cfma(Li[m * 5 + k], rb[sl * 25 + k * 5 + q], acc);
    return cx<TR>{(TR)acc.re, (TR)acc.im};
  };
  // entry (m, q) of -Uinv * U(i, col), col pivoted after i
  auto Qent = [&](int col) {
    cx<TF> acc{0, 0};
    const bool later = !(tw && t == 0 && col >= g.h + 2);
    const int sl = (later && col >= 0 && col < n) ? bc_slot(n, i, col) : -1;
    if (sl >= 0)
      for (int k = m; k < 5; k++) acc = cfma(Ui[m * 5 + k], rb[sl * 25 + k * 5 + q], acc);
    return cx<TR>{(TR)-acc.re, (TR)-acc.im};
  };
  cx<TR> *F = fwd + idx * 60;
  cx<TR> *B = bwd + idx * 66;
  cx<TR> *Tl = tail + (line * nchain + t) * 150;
  if (valid && act) {
    auto put = [&](cx<TR> *rec, int older, cx<TR> v) {
      TR *w = reinterpret_cast<TR *>(rec) + m * 20 + rec_pos(older, q);
      w[0] = v.re;
      w[10] = v.im;
    };
    put(F, 0, Nent(i - dir));
    put(F, 1, Nent(i - 2 * dir));
    put(B, 0, Qent(i + dir));
    put(B, 1, Qent(i + 2 * dir));
    // forward blocks of the chain's last two rows outside the band: columns
    // n-5, n-4 (plain) or the bottom chain's last rows h+2, h+3 (twisted);
    // the bottom chain of a twisted factor has none (zeros)
    const bool fw_tail = !(tw && t == 1);
    const int x0 = !fw_tail ? -1 : (tw ? g.h + 2 : n - 5), x1 = !fw_tail ? -1 : (tw ? g.h + 3 : n - 4);
    if (j == (fw_tail ? len - 2 : 0)) Tl[m * 5 + q] = Nent(x0);
    if (j == (fw_tail ? len - 1 : 0)) { Tl[25 + m * 5 + q] = Nent(x0); Tl[50 + m * 5 + q] = Nent(x1); }
    // backward blocks of the chain's first two rows: columns 3, 4 counted
    // along the chain
    const int c3 = t == 0 ? 3 : n - 4, c4 = t == 0 ? 4 : n - 5;
    if (j == 0) { Tl[75 + m * 5 + q] = Qent(c3); Tl[100 + m * 5 + q] = Qent(c4); }
    if (j == 1) Tl[125 + m * 5 + q] = Qent(c4);
  }
  if (valid && gl < 10) {            // strict lower of Linv, row-major
    const int l = gl < 1 ? 1 : gl < 3 ? 2 : gl < 6 ? 3 : 4, c = gl - l * (l - 1) / 2;
    F[50 + gl] = cx<TR>{(TR)Li[l * 5 + c].re, (TR)Li[l * 5 + c].im};
  }
  if (valid && gl < 16) {            // upper of Uinv incl. diagonal, row-major; then the pad
    if (gl < 15) {
      const int r = gl < 5 ? 0 : gl < 9 ? 1 : gl < 12 ? 2 : gl < 14 ? 3 : 4;
      const int c = r + gl - (5 * r - r * (r - 1) / 2);
      B[50 + gl] = cx<TR>{(TR)Ui[r * 5 + c].re, (TR)Ui[r * 5 + c].im};
    } else {
      B[65] = cx<TR>{0, 0};
    }
  }
}

// ---------------------------------------------------------------------------
// A wave's elimination of one interior pivot row of a chain in registers.
//
// The pivot's window is 15 x 15: rows v..v+2 and columns v..v+2 as scalars.
// Lane 16 g + j holds column j (15 idle) of row 0 and of the four rows
//   slot 0: 1 + g;   slots 1-3: 5 + g + 4 (slot - 1)  (15 and 16 do not exist)
// so that a row's 15 entries sit in one 16-lane row, where the multiplier of
// column k reaches them as the DPP operand of the multiply-adds
// (row_newbcast:k).  Pivot row k > 0 is passed from group k - 1 to the others
// by v_permlane16/32_swap.  Every entry gets the operations of the generic
// path in the same order: the in-block multipliers by cdiv, the partner rows'
// by the pivot's reciprocal, then its updates by columns 0..4.
template <int K> __device__ __forceinline__ double row_bcast(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x150 + K, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x150 + K, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// the value of 16-lane row G in all four
template <int G> __device__ __forceinline__ double group_bcast(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  auto one = [](unsigned w) {
    const auto a = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const unsigned y = G < 2 ? a[0] : a[1];
    const auto c = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    return G % 2 == 0 ? c[0] : c[1];
  };
  const unsigned lo = one((unsigned)b), hi = one((unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// fact = -1 / d and m = -a / d for a pivot d that all lanes hold: Smith's
// algorithm with the wave's one branch, its quotients by reciprocals of the
// denominators, corrected with their remainders (Markstein).  The denominators
// lie between the pivot's larger part and twice that; near the ends of the
// range they are divided by in full.
__device__ __forceinline__ double pivot_recip(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double quotient(double a, double b, double y) {     // a / b, y = 1 / b
  const double q = a * y;
  return fma(fma(-b, q, a), y, q);
}
__device__ __forceinline__ void pivot_div(cx<double> d, cx<double> a, cx<double> &fact, cx<double> &m) {
  const bool by_re = __any(fabs(d.re) >= fabs(d.im));
  const double big = by_re ? fabs(d.re) : fabs(d.im);
  if (__builtin_expect(__any(!(big > 0x1p-400 && big < 0x1p400)), 0)) {
    fact = -crecip(d);
    m = -cdiv(a, d);
  } else if (by_re) {
    const double r = quotient(d.im, d.re, pivot_recip(d.re)), den = fma(d.im, r, d.re), y = pivot_recip(den);
    fact = cx<double>{quotient(-1, den, y), quotient(r, den, y)};
    m = cx<double>{quotient(fma(-a.im, r, -a.re), den, y), quotient(fma(a.re, r, -a.im), den, y)};
  } else {
    const double r = quotient(d.re, d.im, pivot_recip(d.im)), den = fma(d.re, r, d.im), y = pivot_recip(den);
    fact = cx<double>{quotient(-r, den, y), quotient(1, den, y)};
    m = cx<double>{quotient(fma(-a.re, r, -a.im), den, y), quotient(fma(-a.im, r, a.re), den, y)};
  }
}

struct PivotWindow {
  cx<double> top;        // row 0
  cx<double> s[4];       // slots 0-3

  template <int K> __device__ __forceinline__ void step(int j, int g) {
    cx<double> p = K == 0 ? top : cx<double>{group_bcast<(K + 3) % 4>(s[0].re), group_bcast<(K + 3) % 4>(s[0].im)};
    cx<double> fact, m;
    pivot_div(cx<double>{row_bcast<K>(p.re), row_bcast<K>(p.im)}, s[0], fact, m);
    // column K becomes the multipliers
    if (j == K) {
      if (K < 4 && g >= K) s[0] = m;
#pragma unroll
      for (int t = 1; t < 4; t++) s[t] = cmul(s[t], fact);
    }
    // columns up to K, and in the block the rows up to the pivot, are final:
    // they are updated by zeros
    if (j <= K) p = cx<double>{0, 0};
    cx<double> p0 = p;
    if (g < K) p0 = cx<double>{0, 0};
    // Lane K keeps its value throughout, so a slot is its own multiplier; the
    // order leaves the two wait states between a write and its DPP read.
#define LNS3D_PIV(ACC, M, P) "v_fmac_f64_dpp %" ACC ", " M ", %" P " row_newbcast:%12 row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n"
        LNS3D_PIV("0", "%0", "8") LNS3D_PIV("2", "%2", "10") LNS3D_PIV("4", "%4", "10") LNS3D_PIV("6", "%6", "10")
        LNS3D_PIV("1", "%0", "9") LNS3D_PIV("3", "%2", "11") LNS3D_PIV("5", "%4", "11") LNS3D_PIV("7", "%6", "11")
        LNS3D_PIV("0", "-%1", "9") LNS3D_PIV("2", "-%3", "11") LNS3D_PIV("4", "-%5", "11") LNS3D_PIV("6", "-%7", "11")
        LNS3D_PIV("1", "%1", "8") LNS3D_PIV("3", "%3", "10") LNS3D_PIV("5", "%5", "10") LNS3D_PIV("7", "%7", "10")
        : "+&v"(s[0].re), "+&v"(s[0].im), "+&v"(s[1].re), "+&v"(s[1].im), "+&v"(s[2].re), "+&v"(s[2].im),
          "+&v"(s[3].re), "+&v"(s[3].im)
        : "v"(p0.re), "v"(p0.im), "v"(p.re), "v"(p.im), "n"(K));
#undef LNS3D_PIV
  }
};

// The rows of a chain between its ends: pivots [vs, ve), chain row v at line
// row v (dir 1) or n - 1 - v (dir -1).  The window moves down its diagonal
// through the LDS array mx: an elimination leaves its trailing 10 x 10 there,
// the 125 entries that the next window adds come from memory, read two pivots
// ahead, and the 125 entries that are final go back, gathered in mx so that
// two stores of whole blocks take them.  mx holds the first window on entry
// and, in its first 10 rows and columns, the trailing part on return.  Entries
// of rows and columns from zero_from on count as zero when they are first
// read.  A chain is serial, so its time is latency: per pivot five divisions
// in a row, the exchange through LDS, the multiply-adds of one wave.  Every
// load and store of memory is unconditional (idle lanes repeat another's), so
// that the wait for a window's entries counts past the stores in between.
// 257 twisted lines of 513 rows: 1770 -> 680 us (562 to 706), 2.6 us a pivot;
// one line of 2000 rows, with import and records, 5.86 -> 1.88 ms for a chain
// of 1000 pivots.  A pivot's 450 vector instructions take 1.0 us
constexpr int MX_OUT = 17 * 16, MX_SIZE = MX_OUT + 125;     // 17 rows of 16, the final entries
__device__ __forceinline__ void eliminate_interior(cx<double> *mx, cx<double> *lul, int n, int dir, int vs, int ve,
                                                   int zero_from, int lane) {
  const int j = min(lane & 15, 14), g = lane >> 4;           // lane 15 of a row repeats column 14
  // block (v + dr, v + dc) of chain rows: its place in the line
  auto place = [&](int v, int dr, int dc) {
    return (dir > 0 ? v + dr : n - 1 - v - dr) * 125 + (2 + dir * (dc - dr)) * 25;
  };
  // this lane's two entries of what window v adds to window v - 1, and of
  // what is final after pivot v
  struct Entry { int from, at, low; } fr[2];      // low: the smaller of row and column
  int fin[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int e = min(lane + 64 * h, 124), b = e / 25, in = e % 25;
    const int dr = min(b, 2), dc = b < 2 ? 2 : b - 2;
    fr[h] = Entry{place(0, dr, dc) + in, (dr * 5 + in / 5) * 16 + dc * 5 + in % 5, min(dr, dc)};
    fin[h] = place(0, max(b - 2, 0), b < 3 ? b : 0) + in;
  }
  auto fetch = [&](int v, cx<double> (&x)[2]) {
#pragma unroll
    for (int h = 0; h < 2; h++) x[h] = lul[fr[h].from + dir * v * 125];
  };
  // where this lane's entries go after a pivot: row 0 and slot 0 are final;
  // of slots 1-3 columns 0-4 are, the rest moves up the diagonal
  const int out0 = MX_OUT + (j / 5) * 25 + j % 5;
  int to[4];
#pragma unroll
  for (int t = 1; t < 4; t++) {
    const int r = 1 + g + 4 * t;
    to[t] = r > 14 ? 15 * 16 + j : j < 5 ? MX_OUT + 75 + (r - 5) * 5 + j : (r - 5) * 16 + j - 5;
  }
  auto put_final = [&](int v, const cx<double> (&x)[2]) {
#pragma unroll
    for (int h = 0; h < 2; h++) lul[fin[h] + dir * v * 125] = x[h];
  };
  // pivot v, with next the entries of window v + 1; those of window v + 2 are
  // read into after.  Two sets in turn, as a copy from one to another
  // would wait for the loads and the stores before them
  auto pivot = [&](int v, cx<double> (&next)[2], cx<double> (&after)[2]) {
    PivotWindow w;
    w.top = mx[j];
    w.s[0] = mx[(1 + g) * 16 + j];
#pragma unroll
    for (int t = 1; t < 4; t++) w.s[t] = mx[(1 + g + 4 * t) * 16 + j];
    cx<double> done[2];
#pragma unroll
    for (int h = 0; h < 2; h++) done[h] = mx[MX_OUT + min(lane + 64 * h, 124)];
    fetch(min(v + 2, ve - 1), after);
    w.step<0>(j, g);
    if (v > vs) put_final(v - 1, done);      // behind the first column, when they have come from LDS
    w.step<1>(j, g);
    w.step<2>(j, g);
    w.step<3>(j, g);
    w.step<4>(j, g);
    wave_sync();
    mx[out0] = w.top;
    mx[out0 + 5 * (1 + g)] = w.s[0];
#pragma unroll
    for (int t = 1; t < 4; t++) mx[to[t]] = w.s[t];
#pragma unroll
    for (int h = 0; h < 2; h++)                                // after the last pivot nothing reads these
      mx[fr[h].at] = v + 1 + fr[h].low >= zero_from ? cx<double>{0, 0} : next[h];
    wave_sync();
  };
  cx<double> f1[2], f2[2];
  fetch(min(vs + 1, ve - 1), f1);
  wave_sync();
  for (int v = vs; v < ve; v += 2) {
    pivot(v, f1, f2);
    if (v + 1 < ve) pivot(v + 1, f2, f1);
  }
  const cx<double> last[2] = {mx[MX_OUT + lane], mx[MX_OUT + min(lane + 64, 124)]};
  put_final(ve - 1, last);
}

// ---------------------------------------------------------------------------
// stage 1 for non-periodic lines: block LU with one wave per chain, interior
// rows by eliminate_interior, the others with the rows v..v+4 of the chain in
// an LDS window.  A plain factor is one chain
// (rows 0..n-1).  The twisted factor runs two chains concurrently, rows
// 0..h-1 top-down and rows n-1..h+2 bottom-up (the bottom one in reversed
// indices, where the band looks the same); both update the 2x2 block of
// rows/columns h, h+1, the top chain in place and the bottom chain into a
// scratch copy that starts at zero.  Once both are done the two are summed
// and rows h, h+1 are eliminated.  Inside a pivot the elimination follows
// cpenta1bc.f:43-495: in-block LU with negated multipliers stored below the
// diagonal, its row operations applied to the pivot row's right blocks, then
// each partner row's block in the pivot column turned into multipliers and
// the partner's blocks updated.
constexpr int FW = 5;

// TW: twisted lines, two chains.  A plain line has one and half the LDS: ten
// of its workgroups fit a CU, where four did with the LDS of two chains (a
// factor with its import and records, us: 1300 lines of 7 rows 330 -> 191,
// 2000 of 12 393 -> 244, 20000 of 33 4920 -> 2914; with rows updated task by
// task in LDS, before, these took 241, 362 and 6666).
template <bool TW>
__global__ __launch_bounds__(TW ? 128 : 64) void k_factor_chains(LineGeom g, cx<double> *lu, cx<double> *mid) {
  using T = double;
  __shared__ cx<T> win[TW ? 2 : 1][FW][125];
  __shared__ cx<T> mx[TW ? 2 : 1][MX_SIZE];
  const int wave = TW ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, lane = threadIdx.x & 63;
  const long line = blockIdx.x;
  const int n = g.n, h = g.h;
  constexpr bool tw = TW;
  cx<T> *lul = lu + line * n * 125;
  cx<T> *midl = mid ? mid + line * 4 * 25 : nullptr;
  // one chain on window w, chain direction tt, pivots [v0, v1), rows above
  // lim never touched
  auto chain = [&](int w, int tt, int v0, int v1, int lim, bool preloaded) {
    auto real = [&](int v) { return tt == 0 ? v : n - 1 - v; };
    auto slot = [&](int vr, int vc) {
      if (vr < 0 || vc < 0 || vr >= n || vc >= n) return -1;
      return bc_slot(n, real(vr), real(vc));
    };
    auto B = [&](int vr, int sl) -> cx<T> * { return &win[w][vr % FW][sl * 25]; };
    auto middle = [&](int vr, int vc) {
      int r = real(vr), c = real(vc);
      return tw && (r == h || r == h + 1) && (c == h || c == h + 1);
    };
    // a row into the window: entries e = lane, lane + 64 (x0, x1) of row vr
    auto put_row = [&](int vr, cx<T> x0, cx<T> x1) {
#pragma unroll
      for (int h2 = 0; h2 < 2; h2++) {
        const int e = lane + 64 * h2;
        if (e >= 125) continue;
        cx<T> x = h2 == 0 ? x0 : x1;
        if (tt == 1 && tw && (real(vr) == h || real(vr) == h + 1)) {   // bottom chain: middle blocks start at zero
          int sl = e / 25;
          for (int vc = vr - 4; vc <= vr + 4; vc++)
            if (slot(vr, vc) == sl && middle(vr, vc)) x = cx<T>{0, 0};
        }
        win[w][vr % FW][e] = x;
      }
    };
    // rows v.. up to lim into the window, all loads before the first use
    auto load_window = [&](int v) {
      cx<T> x[FW][2];
#pragma unroll
      for (int r = 0; r < FW; r++) {
        const cx<T> *src = lul + (long)real(min(v + r, lim)) * 125;
        x[r][0] = src[lane];
        x[r][1] = src[min(lane + 64, 124)];
      }
#pragma unroll
      for (int r = 0; r < FW; r++)
        if (v + r <= lim) put_row(v + r, x[r][0], x[r][1]);
    };
    // write back a row: all slots (pivot rows) or the chain's share
    auto store_row = [&](int vr, bool all) {
      cx<T> *dst = lul + (long)real(vr) * 125;
      if (all) {
        for (int e = lane; e < 125; e += 64) dst[e] = win[w][vr % FW][e];
        return;
      }
      for (int e = lane; e < 125; e += 64) {
        const int sl = e / 25;
        int vcol = -1;
        for (int vc = vr - 4; vc <= vr + 4; vc++)
          if (slot(vr, vc) == sl) vcol = vc;
        if (vcol < 0) continue;
        const int c = real(vcol);
        if (middle(vr, vcol)) {
          if (tt == 0) dst[e] = win[w][vr % FW][e];
          else midl[((real(vr) - h) * 2 + (c - h)) * 25 + (e % 25)] = win[w][vr % FW][e];
        } else if ((tt == 0 && c <= h + 1) || (tt == 1 && c >= h + 2)) {
          dst[e] = win[w][vr % FW][e];
        }
      }
    };
    if (!preloaded) load_window(v0);
    wave_sync();
    // Pivots from 2 on whose partner rows v+1 and v+2 are interior rows of the
    // line (and the chain's): the blocks right of them are columns v+1, v+2,
    // and they go through registers.  The rows beside them keep the window.
    const int vfast = min(v1, min(lim - 1, n - 5));
    for (int v = v0; v < v1; v++) {
      if (v == 2 && v0 < 2 && vfast > 2) {
        for (int e = lane; e < 225; e += 64) {
          const int r = e / 15, c = e % 15;
          mx[w][r * 16 + c] = B(v + r / 5, slot(v + r / 5, v + c / 5))[(r % 5) * 5 + c % 5];
        }
        // multipliers already formed in these rows
        for (int e = lane; e < 75; e += 64) {
          const int b = e / 25, vr = v + b / 2, vc = v - 2 + (b + 1) / 2, sl = slot(vr, vc);
          lul[(long)real(vr) * 125 + sl * 25 + e % 25] = B(vr, sl)[e % 25];
        }
        wave_sync();
        eliminate_interior(mx[w], lul, n, tt == 0 ? 1 : -1, v, vfast, tt == 1 && tw ? lim - 1 : n, lane);
        __threadfence_block();
        v = vfast;
        load_window(v);
        wave_sync();
        for (int e = lane; e < 100; e += 64) {
          const int r = e / 10, c = e % 10;
          B(v + r / 5, slot(v + r / 5, v + c / 5))[(r % 5) * 5 + c % 5] = mx[w][r * 16 + c];
        }
        wave_sync();
        if (v == v1) break;
      }
      // row v+5 comes into the window when row v leaves it; its loads are
      // issued now, so that they arrive while row v is eliminated
      const bool pf_ok = v + FW <= lim;
      cx<T> pf0, pf1;
      {
        const cx<T> *src = lul + (long)real(pf_ok ? v + FW : v) * 125;
        pf0 = src[lane];
        pf1 = lane + 64 < 125 ? src[lane + 64] : cx<T>{0, 0};
      }
      // Blocks right of the pivot (columns uc, slots us) and partner rows pr;
      // filled and read with constant indices only, so that they stay in
      // registers (a run-time index puts a local array in scratch).  Every
      // loop over columns and tasks stays rolled, and a task decodes to an
      // entry of whole blocks: this code runs four to eight times a chain, and
      // its cost is fetching it (unrolled 200 of 660 us at 257 lines of 513)
      cx<T> *D = B(v, slot(v, v));
      int uc[4] = {0, 0, 0, 0}, us[4] = {0, 0, 0, 0}, pr[4] = {0, 0, 0, 0}, nu = 0, nparts = 0;
#pragma unroll
      for (int d = 1; d <= 4; d++) {
        const int vc = v + d;
        const int su = vc <= lim ? slot(v, vc) : -1;
        const bool hp = vc <= lim && slot(vc, v) >= 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if (su >= 0 && nu == i) { uc[i] = vc; us[i] = su; }
          if (hp && nparts == i) pr[i] = vc;
        }
        nu += su >= 0;
        nparts += hp;
      }
      auto pick = [](const int (&a)[4], int i) { return i == 0 ? a[0] : i == 1 ? a[1] : i == 2 ? a[2] : a[3]; };
      // in-block LU of D, its row operations applied to the right blocks
#pragma unroll 1
      for (int nc = 0; nc < 4; nc++) {
        const int l = nc + 1 + lane;
        if (l < 5) D[l * 5 + nc] = -cdiv(D[l * 5 + nc], D[nc * 6]);
        wave_sync();
#pragma unroll 1
        for (int k = lane; k < (1 + nu) * 25; k += 64) {
          const int b = k / 25, e = k % 25, l = e / 5, q = e % 5;
          cx<T> *X = b == 0 ? D : B(v, pick(us, b - 1));
          if (l > nc && (b > 0 || q > nc)) X[e] = cfma(D[l * 5 + nc], X[nc * 5 + q], X[e]);
        }
        wave_sync();
      }
      // partner rows: the block in the pivot column becomes the multipliers
#pragma unroll 1
      for (int nc = 0; nc < 5; nc++) {
        if (lane < nparts * 5) {
          const int p = pick(pr, lane / 5);
          cx<T> *x = B(p, slot(p, v)) + (lane % 5) * 5 + nc;
          *x = -(*x * crecip(D[nc * 6]));
        }
        wave_sync();
#pragma unroll 1
        for (int k = lane; k < nparts * (1 + nu) * 25; k += 64) {
          const int pp = k / ((1 + nu) * 25), b = k / 25 - pp * (1 + nu), e = k % 25, q = e % 5, p = pick(pr, pp);
          cx<T> *Lb = B(p, slot(p, v));
          const int sdst = b == 0 ? slot(p, v) : slot(p, pick(uc, b - 1));
          if (sdst < 0 || (b == 0 && q <= nc)) continue;      // no such block (does not occur in the band); final
          const cx<T> *X = b == 0 ? D : B(v, pick(us, b - 1));
          cx<T> *x = B(p, sdst) + e;
          *x = cfma(Lb[e - q + nc], X[nc * 5 + q], *x);
        }
        wave_sync();
      }
      // row v is final: write it back and bring in row v+5
      store_row(v, true);
      wave_sync();
      if (pf_ok) put_row(v + FW, pf0, pf1);
      wave_sync();
    }
    // rows the chain updated but did not pivot
    for (int vr = v1; vr <= min(v1 + FW - 1, lim); vr++) store_row(vr, !tw);
  };
  // the chain of this wave, and then the two rows between the chains; one call
  // site, so that the code exists once
  int tt = tw ? wave : 0, v0 = 0, v1 = !tw ? n : wave == 0 ? h : n - h - 2, lim = !tw ? n - 1 : wave == 0 ? h + 1 : n - 1 - h;
  for (bool middle_rows = false;; middle_rows = true) {
    chain(tt, tt, v0, v1, lim, middle_rows);
    if (!tw || middle_rows) return;
    __syncthreads();
    if (wave != 0) return;
    // rows h, h+1 with both chains' updates of their 2x2 middle block summed,
    // then their elimination
    for (int rr = h; rr <= h + 1; rr++)
      for (int e = lane; e < 125; e += 64) win[0][rr % FW][e] = lul[(long)rr * 125 + e];
    wave_sync();
    for (int e = lane; e < 100; e += 64) {
      const int b = e / 25, r = h + b / 2, c = h + b % 2;
      cx<T> &x = win[0][r % FW][bc_slot(n, r, c) * 25 + e % 25];
      x = x + midl[e];
    }
    wave_sync();
    v0 = h;
    v1 = h + 2;
    lim = h + 1;
  }
}

// ---------------------------------------------------------------------------
// periodic lines (cpenta1p.f / cpenta2p.f): records from the bordered LU of
// k_lu_per and a streaming solve.  The LU's band gives the same recurrence
// as non-periodic lines; the border (rows n-2, n-1 in every column: per2;
// columns n-2, n-1 in every row: per) becomes two more per-row records:
//   p2[row c] = (Linv_{n-2} per2(n-2,c), Linv_{n-1} per2(n-1,c)): the forward
//     contributions of y_c to the last two rows;
//   qp[row i] = (-Uinv_i per(i,n-2), -Uinv_i per(i,n-1)): the backward terms
//     in x_{n-2}, x_{n-1}, which are known first, folded into d_i.
__device__ __forceinline__ void inblock_inverses(const Blk<double> &D, cx<double> (&Li)[5][5],
                                                 cx<double> (&Ui)[5][5]) {
  for (int r = 0; r < 5; r++)
    for (int c = 0; c < 5; c++) { Li[r][c] = cx<double>{double(r == c), 0}; Ui[r][c] = cx<double>{0, 0}; }
  for (int nc = 0; nc < 4; nc++)
    for (int l = nc + 1; l < 5; l++)
      for (int c = 0; c <= nc; c++) Li[l][c] = cfma(D(l, nc), Li[nc][c], Li[l][c]);
  for (int c = 0; c < 5; c++)
    for (int m = c; m >= 0; m--) {
      cx<double> acc = cx<double>{double(m == c), 0};
      for (int q = m + 1; q <= c; q++) acc = cfma(-D(m, q), Ui[q][c], acc);
      Ui[m][c] = cdiv(acc, D(m, m));
    }
}

__device__ __noinline__ void records_per_row(LineGeom g, cx<double> *mat, cx<double> *per, cx<double> *per2,
                                             cx<double> *fwd, cx<double> *bwd, cx<double> *p2,
                                             cx<double> *qp, long idx) {
  const int n = g.n;
  const long line = idx / n;
  const int i = (int)(idx - line * n);
  Blk<double> D, M;
  cx<double> Li[5][5], Ui[5][5];
  blk(g, mat, per, per2, line, i, i, D);
  inblock_inverses(D, Li, Ui);
  cx<double> *F = fwd + idx * 60, *B = bwd + idx * 66, *P2 = p2 + idx * 50, *QP = qp + idx * 50;
  // entry (m, q) of a block of the recurrence (rec_pos), of a border block
  auto in_record = [](cx<double> *rec, int older) {
    return [=](int m, int q, cx<double> v) {
      double *w = reinterpret_cast<double *>(rec) + m * 20 + rec_pos(older, q);
      w[0] = v.re;
      w[10] = v.im;
    };
  };
  auto in_block = [](cx<double> *dst) { return [=](int m, int q, cx<double> v) { dst[m * 5 + q] = v; }; };
  auto lmul = [&](const cx<double> (&A)[5][5], int row, int col, auto put) {
    bool ok = col >= 0 && col < n && blk(g, mat, per, per2, line, row, col, M);
    for (int m = 0; m < 5; m++)
      for (int q = 0; q < 5; q++) {
        cx<double> acc{0, 0};
        if (ok)
          for (int k = 0; k <= m; k++) acc = cfma(A[m][k], M(k, q), acc);
        put(m, q, acc);
      }
  };
  auto umul = [&](int col, auto put) {
    bool ok = col >= 0 && col < n && blk(g, mat, per, per2, line, i, col, M);
    for (int m = 0; m < 5; m++)
      for (int q = 0; q < 5; q++) {
        cx<double> acc{0, 0};
        if (ok)
          for (int k = m; k < 5; k++) acc = cfma(Ui[m][k], M(k, q), acc);
        put(m, q, cx<double>{-acc.re, -acc.im});
      }
  };
  // band blocks only (columns i-1, i-2 / i+1, i+2 within the line)
  lmul(Li, i, i >= 1 ? i - 1 : -1, in_record(F, 0));
  lmul(Li, i, i >= 2 ? i - 2 : -1, in_record(F, 1));
  for (int l = 1, k = 0; l < 5; l++)
    for (int q = 0; q < l; q++, k++) F[50 + k] = Li[l][q];
  umul(i + 1 < n ? i + 1 : -1, in_record(B, 0));
  umul(i + 2 < n ? i + 2 : -1, in_record(B, 1));
  for (int m = 0, k = 0; m < 5; m++)
    for (int q = m; q < 5; q++, k++) B[50 + k] = Ui[m][q];
  B[65] = cx<double>{0, 0};
  // border columns of row i (per exists for i < col-2)
  umul(i < n - 4 ? n - 2 : -1, in_block(QP));
  umul(i < n - 3 ? n - 1 : -1, in_block(QP + 25));
  // border rows in column i (per2 exists for i < row-2), with those rows' Linv
  cx<double> Lb[5][5], Ub[5][5];
  blk(g, mat, per, per2, line, n - 2, n - 2, D);
  inblock_inverses(D, Lb, Ub);
  lmul(Lb, n - 2, i < n - 4 ? i : -1, in_block(P2));
  blk(g, mat, per, per2, line, n - 1, n - 1, D);
  inblock_inverses(D, Lb, Ub);
  lmul(Lb, n - 1, i < n - 3 ? i : -1, in_block(P2 + 25));
}

__global__ __launch_bounds__(128) void k_records_per(LineGeom g, cx<double> *mat, cx<double> *per, cx<double> *per2,
                              cx<double> *fwd, cx<double> *bwd, cx<double> *p2, cx<double> *qp) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < g.L * g.n) records_per_row(g, mat, per, per2, fwd, bwd, p2, qp, idx);
}

// ---------------------------------------------------------------------------
// layout conversions between the reference's arrays and the working copy
// ref mat (5,5,5,...) element (slot k, r, c) of (line l, row i) at
//   ((i*sRm + l*sLm) * 125 + k + 5r + 25c)
// Periodic lines keep the line index fastest.
__global__ void k_import_mat(const double2 *ref, cx<double> *lu, int n, long L, long sLm, long sRm) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;   // over (i, k, r, c, line)
  long total = (long)n * 125 * L;
  if (idx >= total) return;
  long line = idx % L;
  long e = idx / L;            // (i*5 + k)*25 + r*5 + c
  int c = e % 5, r = (e / 5) % 5, k = (e / 25) % 5;
  long i = e / 125;
  double2 v = ref[(i * sRm + line * sLm) * 125 + k + 5 * r + 25 * c];
  lu[idx] = cx<double>{v.x, v.y};
}
// Non-periodic lines: a block row's 125 entries are consecutive on both sides,
// so IMP rows a workgroup are read in order and leave in order, transposed in
// LDS between.  Bound by memory, 4000 B a row: 257 lines of 513 rows (528 MB)
// 437 us with reads of one entry per 2000 B, 95 us (5.6 TB/s) so.
constexpr int IMP = 16;
__global__ __launch_bounds__(256) void k_import_rows(const double2 *ref, double2 *lu, int n, int rows, long sLm, long sRm) {
  __shared__ double2 buf[IMP * 125];
  const int row0 = blockIdx.x * IMP, count = min(IMP, rows - row0) * 125;
  constexpr int PER = (IMP * 125 + 255) / 256;
  double2 v[PER];
#pragma unroll
  for (int t = 0; t < PER; t++) {
    const int e = min((int)threadIdx.x + 256 * t, count - 1), row = row0 + e / 125;
    v[t] = ref[((row % n) * sRm + (row / n) * sLm) * 125 + e % 125];
  }
#pragma unroll
  for (int t = 0; t < PER; t++) {
    const int e = threadIdx.x + 256 * t, in = e % 125, k = in % 5, r = (in / 5) % 5, c = in / 25;
    if (e < count) buf[e - in + k * 25 + r * 5 + c] = v[t];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < PER; t++) {
    const int e = threadIdx.x + 256 * t;
    if (e < count) lu[(long)row0 * 125 + e] = buf[e];
  }
}

// Factor health (the reference has no pivoting and no check: a zero pivot
// spreads Inf/NaN through its line, src/cpenta1bc.f:80-82 fact = one/pivot).
// One flag per line: set when an entry of the line's factors is not finite
// or a pivot (diagonal of the slot-3 block) is zero.  a holds total complex
// values; line-major arrays hold per_line values per line, interleaved ones
// put the line index fastest (stride L).
template <typename T>
__global__ void k_check_factor(const cx<T> *a, long total, long L, int line_major, long per_line,
                               int pivots, int *flag) {
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    const cx<T> x = a[idx];
    const long line = line_major ? idx / per_line : idx % L;
    const long e = line_major ? idx % per_line : idx / L;     // ((row*5 + slot)*25 + 5r + c)
    bool bad = !(isfinite(x.re) && isfinite(x.im));
    if (pivots && (e / 25) % 5 == 2 && (e % 25) % 6 == 0 && x.re == T(0) && x.im == T(0)) bad = true;
    if (bad) flag[line] = 1;
  }
}
__global__ void k_zero_i32(int *x, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0;
}

// ---------------------------------------------------------------------------
// host side
constexpr unsigned LDS_PER_CU = 160 * 1024;
static int grid_for(long n, int b) { return (int)((n + b - 1) / b); }

static int check_launch_grid(long total) { return (int)std::min<long>(grid_for(total, 256), 4096); }

static int clear_flags(PentaPlan *pl, hipStream_t s) {
  if (!pl->flags) LNS3D_CHECK(hipMalloc(&pl->flags, (size_t)pl->L * sizeof(int)));
  hipLaunchKernelGGL(k_zero_i32, dim3(grid_for(pl->L, 256)), dim3(256), 0, s, (int *)pl->flags, pl->L);
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

int penta_check_launch(PentaPlan *pl, hipStream_t s) {
  if (!pl->periodic) return 0;       // k_records_rows has checked them
  const int rc = clear_flags(pl, s);
  if (rc) return rc;
  const long L = pl->L;
  const long tl = (long)pl->np * 125 * L, tp = (long)pl->np * 50 * L;
  hipLaunchKernelGGL(k_check_factor<double>, dim3(check_launch_grid(tl)), dim3(256), 0, s,
                     (const cx<double> *)pl->lu, tl, L, 0, 0L, 1, (int *)pl->flags);
  hipLaunchKernelGGL(k_check_factor<double>, dim3(check_launch_grid(tp)), dim3(256), 0, s,
                     (const cx<double> *)pl->per, tp, L, 0, 0L, 0, (int *)pl->flags);
  hipLaunchKernelGGL(k_check_factor<double>, dim3(check_launch_grid(tp)), dim3(256), 0, s,
                     (const cx<double> *)pl->per2, tp, L, 0, 0L, 0, (int *)pl->flags);
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

// records of a plan whose LU another plan holds (the complex-float records
// of the refined step): their entries, per line
int penta_check_records_launch(PentaPlan *pl, hipStream_t s) {
  if (!pl->prec) return 0;
  const int rc = clear_flags(pl, s);
  if (rc) return rc;
  const long n = pl->n, L = pl->L;
  const long tf = n * 60 * L, tb = n * 66 * L;
  hipLaunchKernelGGL(k_check_factor<float>, dim3(check_launch_grid(tf)), dim3(256), 0, s,
                     (const cx<float> *)pl->fwd, tf, L, 1, n * 60, 0, (int *)pl->flags);
  hipLaunchKernelGGL(k_check_factor<float>, dim3(check_launch_grid(tb)), dim3(256), 0, s,
                     (const cx<float> *)pl->bwd, tb, L, 1, n * 66, 0, (int *)pl->flags);
  if (pl->periodic) {         // the border records, rounded too
    const long tq = n * 50 * L;
    hipLaunchKernelGGL(k_check_factor<float>, dim3(check_launch_grid(tq)), dim3(256), 0, s,
                       (const cx<float> *)pl->p2, tq, L, 1, n * 50, 0, (int *)pl->flags);
    hipLaunchKernelGGL(k_check_factor<float>, dim3(check_launch_grid(tq)), dim3(256), 0, s,
                       (const cx<float> *)pl->qp, tq, L, 1, n * 50, 0, (int *)pl->flags);
  }
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

int penta_check_result(PentaPlan *pl, hipStream_t s, long *bad_lines, long *first_bad) {
  *bad_lines = 0;
  *first_bad = -1;
  if (!pl->flags) return 0;
  std::vector<int> f((size_t)pl->L);
  LNS3D_CHECK(hipMemcpyAsync(f.data(), pl->flags, f.size() * sizeof(int), hipMemcpyDeviceToHost, s));
  LNS3D_CHECK(hipStreamSynchronize(s));
  for (long l = 0; l < pl->L; l++)
    if (f[l]) {
      if (*first_bad < 0) *first_bad = l;
      ++*bad_lines;
    }
  return 0;
}

static std::mutex g_tune_mu;
static std::map<std::tuple<int, long, int>, int> g_tuned;

// Twisted lines (two chains per line, one line per workgroup) under 512 lines:
// there the chain's length is what a solve takes.  From 512 on plain lines (two
// per workgroup) where the caller may ask for the reference's substitution
// order, which needs factors in row order; else twisted lines from 160 rows on.
// Measured, plain / twisted us: 511 lines of 65 rows 18 / 15, of 129 34 / 27,
// 513 of 65 19 / 18, of 257 80 / 67, 1025 of 65 33 / 39, of 129 65 / 72, of 144
// 72 / 80, of 160 89 / 86, of 257 142 / 128, 1500 of 144 88 / 95, of 160
// 109 / 102.
int penta_variant_for(int n, long lines, int prec, bool row_order) {
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(std::make_tuple(n, lines, prec));
    if (it != g_tuned.end()) return it->second;
  }
  const bool tw = n >= 16 && (lines < 512 || (!row_order && n >= 160));
  return tw ? PENTA_TWISTED : PENTA_PLAIN1;
}

int penta_tune_set(int n, long lines, int prec, int variant) {
  if (variant < -1 || variant >= PENTA_NVARIANT)
    return set_error(__FILE__, __LINE__, "line-solve variant out of range");
  std::lock_guard<std::mutex> lk(g_tune_mu);
  if (variant < 0) g_tuned.erase(std::make_tuple(n, lines, prec));
  else g_tuned[std::make_tuple(n, lines, prec)] = variant;
  return 0;
}

int penta_plan_create(PentaPlan *pl, int periodic, int exact, int n_rows, long lines, int prec, bool row_order) {
  const int n = periodic ? n_rows - 1 : n_rows;
  return penta_plan_create_variant(pl, periodic, exact, n_rows, lines, prec,
                                   periodic ? PENTA_PLAIN1 : penta_variant_for(n, lines, prec, row_order));
}

// what a plan holds on the device
namespace {
struct PlanBytes {
  size_t lu, per, fwd, bwd, tail, mid, border;   // per: each of per, per2; border: each of p2, qp
};
}  // namespace
static PlanBytes plan_bytes(int periodic, int n_rows, long lines, int prec, bool tw) {
  const size_t es = prec ? sizeof(cx<float>) : sizeof(cx<double>), z = sizeof(cx<double>);
  const size_t L = (size_t)lines, np = (size_t)n_rows, n = periodic ? np - 1 : np;
  PlanBytes b{};
  b.lu = np * 125 * L * z;
  b.fwd = n * 60 * L * es;
  b.bwd = n * 66 * L * es;
  if (periodic) {
    // complex-float plans take their records from a complex-double plan
    // (penta_records_narrow): no bordered LU of their own
    if (!prec) b.per = np * 50 * L * z;
    b.border = n * 50 * L * es;
  } else {
    b.tail = 150 * L * (tw ? 2 : 1) * es;
    if (tw) b.mid = 100 * L * z;
  }
  return b;
}

size_t penta_plan_bytes(int periodic, int n_rows, long lines, int prec, bool row_order, bool own_lu) {
  const int n = periodic ? n_rows - 1 : n_rows;
  const bool tw = !periodic && n >= 16 && penta_twisted(penta_variant_for(n, lines, 0, row_order));
  const PlanBytes b = plan_bytes(periodic, n_rows, lines, prec, tw);
  return (own_lu ? b.lu : 0) + 2 * b.per + b.fwd + b.bwd + b.tail + b.mid + 2 * b.border + (size_t)lines * sizeof(int);
}

int penta_plan_create_variant(PentaPlan *pl, int periodic, int exact, int n_rows, long lines, int prec,
                              int variant) {
  pl->periodic = periodic;
  pl->exact = exact;
  pl->np = n_rows;
  pl->n = periodic ? n_rows - 1 : n_rows;
  pl->L = lines;
  pl->prec = prec;
  if (pl->n < 7 || lines < 1) return set_error(__FILE__, __LINE__, "line length must be >= 7 unknowns");
  if (penta_twisted(variant) && pl->n < 16) variant = PENTA_PLAIN1;
  pl->variant = periodic ? PENTA_PLAIN1 : variant;
  pl->h = (!periodic && penta_twisted(pl->variant)) ? (pl->n - 1) / 2 : -1;
  const PlanBytes b = plan_bytes(periodic, n_rows, lines, prec, pl->h >= 0);
  LNS3D_CHECK(hipMalloc(&pl->lu, b.lu));
  pl->per = pl->per2 = nullptr;
  pl->fwd = pl->bwd = pl->tail = pl->mid = pl->p2 = pl->qp = pl->flags = nullptr;
  if (b.per) {
    LNS3D_CHECK(hipMalloc(&pl->per, b.per));
    LNS3D_CHECK(hipMalloc(&pl->per2, b.per));
  }
  LNS3D_CHECK(hipMalloc(&pl->fwd, b.fwd));
  LNS3D_CHECK(hipMalloc(&pl->bwd, b.bwd));
  if (b.border) {
    LNS3D_CHECK(hipMalloc(&pl->p2, b.border));
    LNS3D_CHECK(hipMalloc(&pl->qp, b.border));
  }
  if (b.tail) LNS3D_CHECK(hipMalloc(&pl->tail, b.tail));
  if (b.mid) LNS3D_CHECK(hipMalloc(&pl->mid, b.mid));
  return 0;
}

void penta_plan_destroy(PentaPlan *pl) {
  if (pl->lu) (void)hipFree(pl->lu);
  if (pl->per) (void)hipFree(pl->per);
  if (pl->per2) (void)hipFree(pl->per2);
  if (pl->fwd) (void)hipFree(pl->fwd);
  if (pl->bwd) (void)hipFree(pl->bwd);
  if (pl->tail) (void)hipFree(pl->tail);
  if (pl->mid) (void)hipFree(pl->mid);
  if (pl->p2) (void)hipFree(pl->p2);
  if (pl->qp) (void)hipFree(pl->qp);
  if (pl->flags) (void)hipFree(pl->flags);
  pl->lu = pl->per = pl->per2 = pl->fwd = pl->bwd = pl->tail = pl->mid = pl->p2 = pl->qp = nullptr;
  pl->flags = nullptr;
}

int penta_import(PentaPlan *pl, const void *ref_mat, long sLm, long sRm, hipStream_t s) {
  if (pl->periodic) {
    hipLaunchKernelGGL(k_import_mat, dim3(grid_for((long)pl->np * 125 * pl->L, 256)), dim3(256), 0, s,
                       (const double2 *)ref_mat, (cx<double> *)pl->lu, pl->np, pl->L, sLm, sRm);
  } else {
    const long rows = pl->np * pl->L;
    if (rows > INT_MAX) return set_error(__FILE__, __LINE__, "penta_import: more rows than an index holds");
    hipLaunchKernelGGL(k_import_rows, dim3(grid_for(rows, IMP)), dim3(256), 0, s, (const double2 *)ref_mat,
                       (double2 *)pl->lu, pl->np, (int)rows, sLm, sRm);
  }
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

static int records_launch(PentaPlan *pl, int *flags, hipStream_t s) {
  if (pl->periodic) return set_error(__FILE__, __LINE__, "records are for non-periodic lines");
  LineGeom g{pl->n, pl->periodic, pl->exact, pl->L, pl->h};
  const int nb = grid_for(pl->L * (long)pl->n, 8);
  if (pl->prec)
    hipLaunchKernelGGL((k_records_rows<double, float>), dim3(nb), dim3(256), 0, s, g,
                       (const cx<double> *)pl->lu, (cx<float> *)pl->fwd, (cx<float> *)pl->bwd,
                       (cx<float> *)pl->tail, flags);
  else
    hipLaunchKernelGGL((k_records_rows<double, double>), dim3(nb), dim3(256), 0, s, g,
                       (const cx<double> *)pl->lu, (cx<double> *)pl->fwd, (cx<double> *)pl->bwd,
                       (cx<double> *)pl->tail, flags);
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

int penta_factor_records_only(PentaPlan *pl, hipStream_t s) { return records_launch(pl, nullptr, s); }

__global__ void k_narrow(const cx<double> *src, cx<float> *dst, long count) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const cx<double> a = src[t];
  dst[t] = cx<float>{(float)a.re, (float)a.im};
}

int penta_records_narrow(PentaPlan *dst, const PentaPlan *src, hipStream_t s) {
  if (!dst->periodic || !src->periodic || !dst->prec || src->prec || dst->n != src->n || dst->L != src->L)
    return set_error(__FILE__, __LINE__, "penta_records_narrow: a complex-float and a complex-double periodic plan of one shape");
  const long n = src->n, L = src->L;
  const void *from[4] = {src->fwd, src->bwd, src->p2, src->qp};
  void *to[4] = {dst->fwd, dst->bwd, dst->p2, dst->qp};
  const long count[4] = {n * 60 * L, n * 66 * L, n * 50 * L, n * 50 * L};
  for (int k = 0; k < 4; k++)
    hipLaunchKernelGGL(k_narrow, dim3(grid_for(count[k], 256)), dim3(256), 0, s, (const cx<double> *)from[k],
                       (cx<float> *)to[k], count[k]);
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

int penta_factor(PentaPlan *pl, hipStream_t s) {
  LineGeom g{pl->n, pl->periodic, pl->exact, pl->L, pl->h};
  if (pl->periodic && pl->prec)
    return set_error(__FILE__, __LINE__, "periodic complex-float plans take their records from a complex-double plan");
  if (pl->periodic) {
    hipLaunchKernelGGL(k_lu_per, dim3((unsigned)pl->L), dim3(64), 0, s, g,
                       (cx<double> *)pl->lu, (cx<double> *)pl->per, (cx<double> *)pl->per2);
    LNS3D_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_records_per, dim3(grid_for(pl->L * (long)pl->n, 128)), dim3(128), 0, s, g,
                       (cx<double> *)pl->lu, (cx<double> *)pl->per, (cx<double> *)pl->per2,
                       (cx<double> *)pl->fwd, (cx<double> *)pl->bwd, (cx<double> *)pl->p2,
                       (cx<double> *)pl->qp);
    LNS3D_CHECK(hipGetLastError());
    return 0;
  }
  const bool tw = pl->h >= 0;
  hipLaunchKernelGGL(tw ? k_factor_chains<true> : k_factor_chains<false>, dim3((unsigned)pl->L), dim3(tw ? 128 : 64),
                     0, s, g, (cx<double> *)pl->lu, (cx<double> *)pl->mid);
  LNS3D_CHECK(hipGetLastError());
  const int rc = clear_flags(pl, s);
  return rc ? rc : records_launch(pl, (int *)pl->flags, s);
}

// Forms of the line solve: rows of a chunk and buffers of its ring, and
// whether the right-hand sides stay in LDS.  Resident right-hand sides spare
// the forward result's way to memory and back (160 of 2320 B per row); longer
// chunks spare barriers (complex float, whose chunks are half the bytes);
// small rings let more workgroups share a CU.
enum { LINES_RES6, LINES_RING6, LINES_RES3, LINES_RING3, LINES_RES12, LINES_RING12 };
template <int R_, int NBUF_, bool RES_> struct LineForm {
  static constexpr int R = R_, NBUF = NBUF_;
  static constexpr bool RES = RES_;
};
// f(T{}, LineForm, TW) with the types of a form
template <typename F> static auto with_line_form(int form, int prec, bool tw, F f) {
  auto fam = [&](auto t, auto lf) {
    return tw ? f(t, lf, std::true_type()) : f(t, lf, std::false_type());
  };
  switch (form) {
    case LINES_RES6: return prec ? fam(float{}, LineForm<6, 4, true>()) : fam(double{}, LineForm<6, 4, true>());
    case LINES_RES3: return fam(double{}, LineForm<3, 4, true>());
    case LINES_RING3: return fam(double{}, LineForm<3, 5, false>());
    case LINES_RES12: return fam(float{}, LineForm<12, 4, true>());
    case LINES_RING12: return fam(float{}, LineForm<12, 4, false>());
    default: return prec ? fam(float{}, LineForm<6, 4, false>()) : fam(double{}, LineForm<6, 4, false>());
  }
}
// the same for periodic lines, which have six of them
template <typename F> static auto with_per_form(int form, int prec, F f) {
  switch (form) {
    case LINES_RES6: return prec ? f(float{}, LineForm<6, 4, true>()) : f(double{}, LineForm<6, 4, true>());
    case LINES_RES3: return f(double{}, LineForm<3, 4, true>());
    case LINES_RES12: return f(float{}, LineForm<12, 4, true>());
    case LINES_RING12: return f(float{}, LineForm<12, 4, false>());
    default: return f(double{}, LineForm<6, 4, false>());
  }
}
static unsigned line_lds(int form, int prec, bool tw, int n, bool per = false) {
  if (per)
    return with_per_form(form, prec, [&](auto t, auto lf) {
      return LineSolve<decltype(t), lf.R, lf.NBUF, false, lf.RES, true>::lds_bytes(n);
    });
  return with_line_form(form, prec, tw, [&](auto t, auto lf, auto TW) {
    return LineSolve<decltype(t), lf.R, lf.NBUF, TW.value, lf.RES>::lds_bytes(n);
  });
}

// workgroups of a form that a CU holds.  The LDS is given out in pieces of 1280
// bytes: three workgroups of 53,664 bytes share a CU, of 53,824 bytes two
// (1025 plain lines of 157 and 158 rows, LINES_RES3: 80 and 128 us).
static int cu_fit(int form, int prec, bool tw, int n, bool per = false) {
  constexpr unsigned PIECE = 1280;
  return (int)(LDS_PER_CU / ((line_lds(form, prec, tw, n, per) + PIECE - 1) / PIECE * PIECE));
}

// The form for `lines` lines of n rows solved by one launch.  What matters is
// how many workgroups share a CU (256 CUs, LDS_PER_CU of LDS each): while all
// lines run at once a solve takes as long as its chain, so one or two per CU
// take the form with the shortest step; more lines stream at the memory's
// rate and take the form that moves least.  Measured at lines x rows, us
// (complex double unless said):
//   twisted  RES6 / RING6: 65x129 19 / 20, 127x384 43 / 44, 256x1025 117 / 124,
//            257x257 36 / 37; 1025 lines of 257: RES6 120, RES3 126, RING3 132;
//            513 of 257: RES3 63, RES6 75; 700 of 600: RING3 189, RING6 207
//   plain    1025 of 65: RES3 33, RES6 41; 513 of 257: RING6 73, RING3 79;
//            1025 of 257: RING3 133, RING6 151; where three workgroups of RES3
//            don't fit, RES6 / RING3: 1300 of 163 106 / 103, 2000 of 163
//            124 / 148, 3000 of 170 194 / 229
//            twisted, RES3 / RES6: all at once 513 of 160 39 / 50, 769 of 129
//            43 / 50; not, 1025 of 96 56 / 59, of 129 72 / 70, of 200 105 / 103
//   complex float, twisted: 257x1025 RING12 85, RING6 101; 127x384 RES12 35,
//            RES6 41; 1025 of 257: RES6 74, RING6 83
//   complex float, RES6 / RES12: 257 twisted lines of 65 rows 9.6 / 10.6, of
//            96 13.1 / 13.1, of 129 16.1 / 15.4; plain, of 33 7.9 / 7.9, of 65
//            13.0 / 11.7, of 96 17.8 / 17.0
//   complex float, more than two workgroups a CU, RES6 / RING6 / RING12:
//            all at once with RES6, plain 1500 of 129 50 / 55 / 68; only with
//            RING6, plain 1025 of 200 90 / 59 / 81, 1600 of 158 84 / 71 / 78,
//            twisted 513 of 384 93 / 59 / 84, 769 of 200 59 / 45 / 55; with
//            neither, plain 2500 of 158 98 / 120 / 116, of 257 178 / 190 / 169,
//            3000 of 200 156 / 160 / 151
static int line_form(int variant, int n, long lines, int prec, bool tw) {
  auto fit = [&](int form) { return cu_fit(form, prec, tw, n); };
  const long wg = tw ? lines : (lines + 1) / 2;
  auto at_once = [&](int form) { return wg <= 256L * fit(form); };
  const int need = wg <= 256 ? 1 : wg <= 512 ? 2 : 3;      // to run all at once, up to three
  // variants that pin a form
  const int small = prec ? (fit(LINES_RES6) >= 2 ? LINES_RES6 : LINES_RING6) : (fit(LINES_RES3) >= 3 ? LINES_RES3 : LINES_RING3);
  switch (variant) {
    case PENTA_PLAIN2: case PENTA_TWISTED_PAIRS: return LINES_RING6;
    case PENTA_PLAIN3: case PENTA_TWISTED_HALF: return small;
    case PENTA_PLAIN4: return prec ? LINES_RING12 : LINES_RING3;
    default: break;
  }
  if (need < 3) {
    if (prec && n >= (tw ? 96 : 60)) return fit(LINES_RES12) >= need ? LINES_RES12 : LINES_RING12;
    return fit(LINES_RES6) >= need ? LINES_RES6 : LINES_RING6;
  }
  if (prec) {
    if (at_once(LINES_RES6)) return LINES_RES6;
    if (at_once(LINES_RING6)) return LINES_RING6;
    return fit(LINES_RES6) >= 3 ? LINES_RES6 : LINES_RING12;
  }
  if (fit(LINES_RES3) >= 3 && (!tw || n < 128 || at_once(LINES_RES3))) return LINES_RES3;
  return (tw || wg > 768) && fit(LINES_RES6) >= 2 ? LINES_RES6 : LINES_RING3;
}

// The form of periodic lines, two per workgroup: resident right-hand sides
// where they fit (they spare 160 of 3920 bytes a row), with one workgroup per
// CU the longer chunks, from about 48 rows on in complex float; with more
// workgroups than CUs the shorter chunks while two of them fit a CU (up to
// about 85 rows, complex float 120; the prologues of short lines overlap then).
// Measured at lines x rows, us:
//   complex double, RES6 / RES3 / RING6: 257 of 33 12 / 16 / 15, 1025 of 33
//            41 / 38 / 52, of 65 70 / 73 / 82, of 100 100 / 136 / 113
//   complex float, RES12 / RES6 / RING12: 257 of 24 12 / 10 / 15, of 48
//            14.5 / 14.4 / 20, of 65 16 / 18 / 23, 513 of 100 46 / 30 / 65,
//            of 129 58 / 63 / 77, of 300 - / 145 / 161
static int per_form(int n, long lines, int prec) {
  auto fit = [&](int form) { return cu_fit(form, prec, false, n, true); };
  const int res = prec ? LINES_RES12 : LINES_RES6, small = prec ? LINES_RES6 : LINES_RES3;
  if ((lines + 1) / 2 > 256 && fit(small) >= 2) return small;
  if (prec && n < 48) return LINES_RES6;
  if (fit(res) >= 1) return res;
  if (prec && fit(LINES_RES6) >= 1) return LINES_RES6;
  return prec ? LINES_RING12 : LINES_RING6;
}

// a kernel's dynamic LDS above the default 64 KB has to be asked for
template <typename K> static int allow_lds(K k, unsigned lds) {
  if (lds > 64 * 1024)
    LNS3D_CHECK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_PER_CU));
  return 0;
}

static int launch_line_solve(const PentaPlan *pl, const void *in, void *rhs, long sL, long sR, hipStream_t s) {
  const bool tw = pl->h >= 0;
  const int form = line_form(pl->variant, pl->n, pl->L, pl->prec, tw);
  return with_line_form(form, pl->prec, tw, [&](auto t, auto lf, auto TW) {
    using T = decltype(t);
    auto k = k_line_solve<T, lf.R, lf.NBUF, TW.value, lf.RES>;
    const unsigned lds = line_lds(form, pl->prec, tw, pl->n);
    const int rc = allow_lds(k, lds);
    if (rc) return rc;
    const long wg = tw ? pl->L : (pl->L + 1) / 2;
    hipLaunchKernelGGL(k, dim3((unsigned)wg), dim3(256), lds, s, pl->n, pl->h, pl->L,
                       (const cx<T> *)pl->fwd, (const cx<T> *)pl->bwd, (const cx<T> *)pl->tail, (const double2 *)in,
                       (double2 *)rhs, sL, sR);
    return 0;
  });
}

static int launch_per_solve(const PentaPlan *pl, const void *in, void *rhs, long sL, long sR, hipStream_t s) {
  const int form = per_form(pl->n, pl->L, pl->prec);
  return with_per_form(form, pl->prec, [&](auto t, auto lf) {
    using T = decltype(t);
    auto k = k_line_solve_per<T, lf.R, lf.NBUF, lf.RES>;
    const unsigned lds = line_lds(form, pl->prec, false, pl->n, true);
    const int rc = allow_lds(k, lds);
    if (rc) return rc;
    hipLaunchKernelGGL(k, dim3((unsigned)((pl->L + 1) / 2)), dim3(256), lds, s, pl->n, pl->L, (const cx<T> *)pl->fwd,
                       (const cx<T> *)pl->bwd, (const cx<T> *)pl->p2, (const cx<T> *)pl->qp, (const double2 *)in,
                       (double2 *)rhs, sL, sR);
    return 0;
  });
}

int penta_solve(PentaPlan *pl, void *rhs, long sL, long sR, hipStream_t s, const void *in) {
  if (!in) in = rhs;
  const int rc = pl->periodic ? launch_per_solve(pl, in, rhs, sL, sR, s) : launch_line_solve(pl, in, rhs, sL, sR, s);
  if (rc) return rc;
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// batches: one launch solves the lines of many plans of one solve kernel.
// Workgroup b belongs to member k with off[k] <= b < off[k + 1]; the member's
// item holds its plan's records and its two right-hand sides.
__device__ __forceinline__ int batch_member(const int *off, int count) {
  int lo = 0, hi = count;
  const int b = (int)blockIdx.x;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

template <typename T, int R, int NBUF, bool TW, bool RES>
__global__ __launch_bounds__(256, 2) void kb_line_solve(const PentaBatchItem *items, const int *off, int count,
                                                       int which) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  const int k = batch_member(off, count);
  const PentaBatchItem &b = items[k];
  LineSolve<T, R, NBUF, TW, RES>::run(sm, (long)blockIdx.x - off[k], b.n, b.h, b.L, (const cx<T> *)b.fwd,
                                      (const cx<T> *)b.bwd, (const cx<T> *)b.tail, b.in[which], b.rhs[which], b.sL, b.sR);
}

template <typename T, int R, int NBUF, bool RES>
__global__ __launch_bounds__(256, 2) void kb_line_solve_per(const PentaBatchItem *items, const int *off, int count,
                                                           int which) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  const int k = batch_member(off, count);
  const PentaBatchItem &b = items[k];
  LineSolve<T, R, NBUF, false, RES, true>::run(sm, (long)blockIdx.x - off[k], b.n, -1, b.L, (const cx<T> *)b.fwd,
                                               (const cx<T> *)b.bwd, nullptr, b.in[which], b.rhs[which], b.sL, b.sR,
                                               (const cx<T> *)b.p2, (const cx<T> *)b.qp);
}

// lines per workgroup of a batch group's solve kernel
static int group_lines(const PentaBatchGroup &g) { return g.tw ? 1 : 2; }

int stage_upload(void *dev, const void *src, size_t bytes, std::vector<TableUpload> &ups) {
  void *h = nullptr;
  LNS3D_CHECK(hipHostMalloc(&h, bytes, hipHostMallocDefault));
  memcpy(h, src, bytes);
  ups.push_back(TableUpload{dev, h, bytes});
  return 0;
}

int penta_batch_build(const PentaPlan *const *plans, const double2 *const *in0, double2 *const *rhs0,
                      double2 *const *rhs1, const long *sL, const long *sR, int count,
                      std::vector<PentaBatchGroup> &out, std::vector<TableUpload> &ups) {
  out.clear();
  long lines = 0;              // solved by one launch or another at a time
  for (int k = 0; k < count; k++) lines += plans[k]->L;
  // members that share a kernel: by form, family and precision
  std::map<std::tuple<int, int, int, int>, std::vector<int>> by;   // (form, periodic, twisted, precision)
  for (int k = 0; k < count; k++) {
    const PentaPlan *pl = plans[k];
    const bool tw = pl->h >= 0;
    if (pl->periodic) by[{per_form(pl->n, lines, pl->prec), 1, 0, pl->prec}].push_back(k);
    else by[{line_form(pl->variant, pl->n, lines, pl->prec, tw), 0, tw, pl->prec}].push_back(k);
  }
  for (auto &kv : by) {
    // longest lines first: their workgroups start in the first wave and the
    // short ones fill in behind them
    std::stable_sort(kv.second.begin(), kv.second.end(),
                     [&](int a, int b) { return plans[a]->n > plans[b]->n; });
    PentaBatchGroup g;
    g.form = std::get<0>(kv.first);
    g.per = std::get<1>(kv.first);
    g.tw = std::get<2>(kv.first);
    g.prec = std::get<3>(kv.first);
    g.count = (int)kv.second.size();
    std::vector<PentaBatchItem> items;
    std::vector<int> off(1, 0);
    for (int k : kv.second) {
      const PentaPlan *pl = plans[k];
      PentaBatchItem it;
      it.n = pl->n;
      it.h = pl->h;
      it.L = pl->L;
      it.fwd = pl->fwd;
      it.bwd = pl->bwd;
      it.tail = pl->tail;
      it.p2 = pl->p2;
      it.qp = pl->qp;
      it.in[0] = in0[k];
      it.in[1] = rhs1[k];
      it.rhs[0] = rhs0[k];
      it.rhs[1] = rhs1[k];
      it.sL = sL[k];
      it.sR = sR[k];
      items.push_back(it);
      const long wg = (pl->L + group_lines(g) - 1) / group_lines(g);
      g.lds = std::max(g.lds, line_lds(g.form, g.prec, g.tw, pl->n, g.per));
      if ((long)off.back() + wg > 0x7fffffffL) return set_error(__FILE__, __LINE__, "batch too large");
      off.push_back(off.back() + (int)wg);
    }
    g.blocks = off.back();
    LNS3D_CHECK(hipMalloc(&g.items, items.size() * sizeof(PentaBatchItem)));
    out.push_back(g);             // freed with the groups from here on
    LNS3D_CHECK(hipMalloc(&out.back().off, off.size() * sizeof(int)));
    int rc = stage_upload(g.items, items.data(), items.size() * sizeof(PentaBatchItem), ups);
    if (!rc) rc = stage_upload(out.back().off, off.data(), off.size() * sizeof(int), ups);
    if (rc) return rc;
  }
  return 0;
}

void penta_batch_free(std::vector<PentaBatchGroup> &groups) {
  for (auto &g : groups) {
    if (g.items) (void)hipFree(g.items);
    if (g.off) (void)hipFree(g.off);
  }
  groups.clear();
}

static int launch_batch_group(const PentaBatchGroup &g, int which, hipStream_t s) {
  const auto *it = (const PentaBatchItem *)g.items;
  const dim3 grid((unsigned)g.blocks), blk(256);
  auto launch = [&](auto k) {
    const int rc = allow_lds(k, g.lds);
    if (rc) return rc;
    hipLaunchKernelGGL(k, grid, blk, g.lds, s, it, g.off, g.count, which);
    return 0;
  };
  if (g.per)
    return with_per_form(g.form, g.prec, [&](auto t, auto lf) {
      return launch(kb_line_solve_per<decltype(t), lf.R, lf.NBUF, lf.RES>);
    });
  return with_line_form(g.form, g.prec, g.tw, [&](auto t, auto lf, auto TW) {
    return launch(kb_line_solve<decltype(t), lf.R, lf.NBUF, TW.value, lf.RES>);
  });
}

int penta_batch_solve(const std::vector<PentaBatchGroup> &groups, int which, hipStream_t s) {
  for (const auto &g : groups) {
    const int rc = launch_batch_group(g, which, s);
    if (rc) return rc;
    LNS3D_CHECK(hipGetLastError());
  }
  return 0;
}

int penta_solve_reference_order(PentaPlan *pl, void *rhs, long sL, long sR, hipStream_t s) {
  if (pl->h >= 0)
    return set_error(__FILE__, __LINE__, "reference-order solve needs factors in row order (this plan is twisted)");
  LineGeom g{pl->n, pl->periodic, pl->exact, pl->L};
  hipLaunchKernelGGL(k_solve_lines<double>, dim3(grid_for(pl->L, 64)), dim3(64), 0, s, g,
                     (const cx<double> *)pl->lu, (const cx<double> *)pl->per,
                     (const cx<double> *)pl->per2, (double2 *)rhs, sL, sR);
  LNS3D_CHECK(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// autotuner: synthetic diagonally dominant lines of the requested shape,
// every solve variant factored and timed, the fastest kept for the shape
__global__ void k_fill_synthetic(cx<double> *lu, long total, unsigned seed) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  unsigned x = (unsigned)(idx * 2654435761u) ^ seed;
  x ^= x >> 13; x *= 0x5bd1e995u; x ^= x >> 15;
  double a = ((x & 0xffff) / 65536.0 - 0.5) * 0.1, b = ((x >> 16) / 65536.0 - 0.5) * 0.1;
  const int e = (int)(idx % 125), k = e / 25, r = (e / 5) % 5, c = e % 5;
  if (k == 2 && r == c) a += 3.0;
  lu[idx] = cx<double>{a, b};
}

int penta_tune(int n, long lines, int prec, int *variant, float *times_ms) {
  float best = 1e30f;
  int bestv = -1;
  hipStream_t s;
  LNS3D_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  hipEvent_t e0, e1;
  LNS3D_CHECK(hipEventCreate(&e0));
  LNS3D_CHECK(hipEventCreate(&e1));
  void *rhs = nullptr;
  LNS3D_CHECK(hipMalloc(&rhs, (size_t)n * lines * 5 * sizeof(double2)));
  LNS3D_CHECK(hipMemsetAsync(rhs, 0, (size_t)n * lines * 5 * sizeof(double2), s));
  int rc = 0;
  for (int v = 0; v < PENTA_NVARIANT && !rc; v++) {
    if (times_ms) times_ms[v] = -1.0f;
    if (penta_twisted(v) && n < 16) continue;
    PentaPlan pl;
    rc = penta_plan_create_variant(&pl, 0, 0, n, lines, prec, v);
    if (!rc) {
      long total = (long)n * 125 * lines;
      hipLaunchKernelGGL(k_fill_synthetic, dim3(grid_for(total, 256)), dim3(256), 0, s,
                         (cx<double> *)pl.lu, total, 12345u);
      rc = penta_factor(&pl, s);
    }
    if (!rc) rc = penta_solve(&pl, rhs, n, 1, s);      // warm-up
    if (!rc) {
      (void)hipEventRecord(e0, s);
      for (int k = 0; k < 3 && !rc; k++) rc = penta_solve(&pl, rhs, n, 1, s);
      (void)hipEventRecord(e1, s);
      (void)hipEventSynchronize(e1);
      float ms = 0;
      (void)hipEventElapsedTime(&ms, e0, e1);
      ms /= 3;
      if (times_ms) times_ms[v] = ms;
      if (ms < best) { best = ms; bestv = v; }
    }
    (void)hipStreamSynchronize(s);
    penta_plan_destroy(&pl);
  }
  (void)hipFree(rhs);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipStreamDestroy(s);
  if (rc) return rc;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[std::make_tuple(n, lines, prec)] = bestv;
  }
  if (variant) *variant = bestv;
  return 0;
}

}  // namespace lns3d
