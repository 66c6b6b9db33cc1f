// Batched uneven cell-block LU, inverse and block-Jacobi sweep (BlockJacobi.cs:63-197,
// IMatrixExtensions.InvertInPlace:2128-2230 -> LAPACK DGETRF/DGETRI semantics).
//
// Every form follows DGETF2: partial pivoting picks the first row with the largest
// |a| in the column, as LAPACK's idamax does (a NaN in the diagonal position is never
// beaten); a zero pivot sets INFO = j+1 (1-based) and the factorisation continues.
// Pivots are stored 1-based (ipiv).  Blocks up to 20 DOF keep their rows in registers
// (several blocks per wavefront), 21..128 DOF one block per workgroup in registers,
// larger ones (Schwarz blocks) are blocked: panels in registers up to 1024 DOF where the
// caller keeps the pivots, in global memory otherwise.
//
// Blocks of different size share a launch (each wave reads its own size), so a whole
// block-Jacobi set of uneven XDG blocks (10x10 and 20x20) is one kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/bosss_hip.h"
#include "devbuf.hpp"

namespace bosss {

constexpr int LU_MAXN = 128;

template <typename Real>
__device__ __forceinline__ void wave_argmax(Real& v, int& idx) {
  // reduce (|a|, index) over the 64 lanes; ties keep the smaller index
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    Real ov = __shfl_xor(v, o, 64);
    int oi = __shfl_xor(idx, o, 64);
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
}

// Shared state of the register-tile kernel.  The row placement (pos, lrow) is kept once per
// wavefront: each wavefront applies every exchange to its own copy, so a column step needs one
// workgroup barrier (publishing the column and the pivot) and no wavefront reads a copy that
// another one is still writing.
template <int RA>
struct TileLDS {
  double col[2][16 * RA], row[2][16 * RA], pv[2];
  int pos[4][16 * RA], lrow[4][16 * RA], piv[16 * RA], p[2];
};

// Loads block g (n x n, row-major) into the register tile and resets the row bookkeeping.
template <int RA>
__device__ __forceinline__ void tile_load(double (&a)[RA][RA], const double* __restrict__ g, int n, TileLDS<RA>& L) {
  const int tid = threadIdx.x, tc = tid >> 4, tr = tid & 15;
#pragma unroll
  for (int x = 0; x < RA; x++)
#pragma unroll
    for (int y = 0; y < RA; y++) {
      const int r = tr + 16 * x, c = tc + 16 * y;
      a[x][y] = 0.0;
      if (r < n && c < n) a[x][y] = g[(int64_t)r * n + c];
    }
  for (int i = tid; i < 4 * 16 * RA; i += 256) {
    const int w = i / (16 * RA), r = i - w * 16 * RA;
    L.pos[w][r] = r;
    L.lrow[w][r] = r;
  }
  __syncthreads();
}

// Column steps 0..n-1 of getf2 on the register
// tile.  Returns INFO (first zero pivot, 1-based).  L.piv[j] receives the
// position of step j's pivot row, L.pos / L.lrow the final row placement (every wavefront's copy).
//
// One barrier per step: the 16 threads holding column j publish it and the pivot (row, value);
// after the barrier the thread of each 16-lane group that holds the pivot row's entries of the
// group's columns c = tc + 16 y publishes them in row[][c], which only that group reads back.
// Column group tc lives in wavefront tc / 4 and the LDS accesses of one wavefront complete in
// order, so this exchange needs no workgroup barrier; lane 0 of each wavefront applies the row
// exchange to that wavefront's copy of the placement.
template <int RA>
__device__ __forceinline__ int tile_eliminate(double (&a)[RA][RA], int n, TileLDS<RA>& L) {
  const int tid = threadIdx.x, tc = tid >> 4, tr = tid & 15, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int* pos = L.pos[w];
  int* lrow = L.lrow[w];
  unsigned used = 0;   // bit x: row tr + 16 x is in a position <= j
  int inf = 0;
  for (int j = 0; j < n; j++) {
    const int k = j & 1, jc = j & 15, jy = j >> 4;
    if (tc == jc) {
      // the 16 threads holding column j: publish it, find the pivot among the unused rows
      double best = -1.0, bval = 0.0;
      int bpos = 1 << 30, bp = -1;
#pragma unroll
      for (int yy = 0; yy < RA; yy++)
        if (yy == jy) {
#pragma unroll
          for (int x = 0; x < RA; x++) {
            const int r = tr + 16 * x;
            const double v0 = a[x][yy];
            if (r < n) {
              L.col[k][r] = v0;
              const int ps = pos[r];
              if (ps >= j) {
                double v = fabs(v0);
                if (ps == j && v != v) v = (double)INFINITY;   // idamax: a NaN first element is never beaten
                if (v > best || (v == best && ps < bpos)) { best = v; bpos = ps; bp = r; bval = v0; }
              }
            }
          }
        }
#pragma unroll
      for (int o = 8; o >= 1; o >>= 1) {
        const double ov = __shfl_xor(best, o, 16), oval = __shfl_xor(bval, o, 16);
        const int opos = __shfl_xor(bpos, o, 16), op = __shfl_xor(bp, o, 16);
        if (ov > best || (ov == best && opos < bpos)) { best = ov; bpos = opos; bp = op; bval = oval; }
      }
      if (tr == 0) {
        if (bp < 0) { bp = lrow[j]; bval = L.col[k][bp]; }   // no comparable candidate (all NaN): position j
        L.p[k] = bp;
        L.pv[k] = bval;
      }
    }
    __syncthreads();
    const int p = __builtin_amdgcn_readfirstlane(L.p[k]);
    const double pv = L.pv[k];
    if (tid == 0) L.piv[j] = pos[p];
    if (!(pv != 0.0)) {   // zero pivot (NaN passes, as in DGETF2)
      if (!inf) inf = j + 1;
      const int r0 = lrow[j];   // no exchange: the row in position j is done all the same
      if (tr == (r0 & 15)) used |= 1u << (r0 >> 4);
      continue;
    }
    if (lane == 0) {   // read by this wavefront's lanes from the next step on
      const int q = pos[p], rj = lrow[j];
      pos[p] = j; pos[rj] = q; lrow[j] = p; lrow[q] = rj;
    }
    const int pc = p & 15, px = __builtin_amdgcn_readfirstlane(p >> 4);
    const double pinv = 1.0 / pv;
    if (tr == pc) {   // the pivot row's entries of the group's columns tc + 16 y
#pragma unroll
      for (int xx = 0; xx < RA; xx++)
        if (xx == px) {
#pragma unroll
          for (int y = 0; y < RA; y++) {
            const int c = tc + 16 * y;
            L.row[k][c] = a[xx][y];
          }
        }
    }
    __builtin_amdgcn_wave_barrier();
    double u[RA];
#pragma unroll
    for (int y = 0; y < RA; y++) u[y] = L.row[k][tc + 16 * y];
    // rows after the pivot in factor order: multiplier into column j, columns > j updated
#pragma unroll
    for (int x = 0; x < RA; x++) {
      const int r = tr + 16 * x;
      if (r < n && r != p && !((used >> x) & 1u)) {
        const double l = L.col[k][r] * pinv;
#pragma unroll
        for (int y = 0; y < RA; y++)
          if (tc + 16 * y > j) a[x][y] -= l * u[y];
        if (tc == jc) {
#pragma unroll
          for (int yy = 0; yy < RA; yy++)
            if (yy == jy) a[x][yy] = l;
        }
      }
    }
    if (tr == pc) used |= 1u << px;
  }
  return inf;
}

// Writes the factors back in position order (row pos[r]).
template <int RA>
__device__ __forceinline__ void tile_store(const double (&a)[RA][RA], double* __restrict__ g, int n, const TileLDS<RA>& L) {
  const int tid = threadIdx.x, tc = tid >> 4, tr = tid & 15;
#pragma unroll
  for (int x = 0; x < RA; x++) {
    const int r = tr + 16 * x;
    if (r < n) {
      const int64_t row = (int64_t)L.pos[0][r] * n;
#pragma unroll
      for (int y = 0; y < RA; y++) {
        const int c = tc + 16 * y;
        if (c < n) g[row + c] = a[x][y];
      }
    }
  }
}

// Blocks of 21..16 RA DOF (the 100-DOF cell blocks of p = 3 Euler, up to 128): one workgroup of
// 256 threads per block, the whole block in registers.  Thread (tc, tr) = (tid >> 4, tid & 15)
// holds rows tr + 16 x and columns tc + 16 y (x, y < RA), in the block's original row order:
// row exchanges are bookkeeping only, pos[r] is the position (row of the factors) that physical
// row r has been given and lrow[] its inverse.  Each column step: the 16 threads holding column j
// find the pivot among the rows not yet used (largest |a|, ties to the smaller position, a NaN in
// position j never beaten: getf2's IDAMAX in getf2's row order) with shuffles inside their 16-lane
// group and publish the column; the threads holding the pivot row publish it to their own
// 16-lane groups; every thread updates its entries.  Factors, pivots and INFO are getf2's, operation for operation (multiplier a * (1 / pivot),
// then the rank-one update of the columns after j).
// Register columns and rows are picked with wavefront-uniform branches, so no register array is
// indexed dynamically.
template <int RA>
__global__ void __launch_bounds__(256) k_block_lu_tile(int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                       double* __restrict__ A, int32_t* __restrict__ ipiv,
                                                       const int64_t* __restrict__ pivoff, int32_t* __restrict__ info) {
  __shared__ TileLDS<RA> L;
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax || n > 16 * RA) {   // size outside what the launch was sized for: report, touch nothing
    if (threadIdx.x == 0 && info) info[b] = -1;
    return;
  }
  double* g = A + off[b];
  double a[RA][RA];
  tile_load<RA>(a, g, n, L);
  const int inf = tile_eliminate<RA>(a, n, L);
  __syncthreads();
  tile_store<RA>(a, g, n, L);
  if (ipiv)
    for (int i = threadIdx.x; i < n; i += 256) ipiv[pivoff[b] + i] = L.piv[i] + 1;
  if (threadIdx.x == 0 && info) info[b] = inf;
}

// Inverse of blocks of 21..128 DOF, blocked: Gauss-Jordan on panels of four columns, the rest of
// the block updated by one rank-4 product per panel on v_mfma_f64_16x16x4f64.
//
// One workgroup of four wavefronts per block, the block in registers as 16 x 16 accumulator tiles:
// wavefront w holds tile columns w and w + 4 (TR tile rows each), rows in their original places
// (row exchanges are bookkeeping, as in the register-tile form).  Per panel the wavefront that holds
// its four columns runs in-place Gauss-Jordan on them, lane l with rows l and l + 64: pivots are
// getf2's (largest |a| among the rows not yet used, ties to the smaller position, a NaN in position j
// never beaten) on columns updated by the earlier panels.  The other columns then receive the same four
// steps: the scaled pivot rows u_0 .. u_3 are formed one after the other (u_k = (a_pk - sum_i<k f_i(p_k) u_i)
// / pivot k, f_i(r) the entry of row r in column i before step i) and all rows take -sum_k f_k(r) u_k, a
// pivot row from zero on and with 1 in its own step.  Same operations in the same order as column by
// column; the rank-4 form X = -A_RJ A_PJ^-1, A += X A_P has larger coefficients and measured 1.8 times
// the error.  One barrier per panel (X, F double-buffered): pivot rows are exchanged inside the
// wavefront that owns their columns.
//
// Bound: the latency of the panel's four column steps, which one wavefront runs; three workgroups per
// CU overlap it (100 DOF: two waves per SIMD 1.27 ms, three 0.92 ms).  4000 blocks of 100 DOF: 1.61 ms
// column by column in a register tile (260 vector and 34 LDS instructions per wavefront and column),
// 0.92 ms here; 32 DOF 134 -> 122 us, 64 DOF 0.43 -> 0.31 ms, 128 DOF 2.77 -> 1.50 ms.  The results
// are those of the column-by-column form to the bit.
// A zero pivot stops it and the block is factored from its original values instead (LU and INFO).
typedef double gj_f64x4 __attribute__((ext_vector_type(4)));

// Maximum over the 64 lanes of values that are not NaN, the same in every lane.
__device__ __forceinline__ double wave_max(double v) {
  auto step = [](double x, auto ctrl, auto mask) {
    union { double d; int i[2]; } u, t;
    u.d = x;
    t.i[0] = __builtin_amdgcn_update_dpp(u.i[0], u.i[0], decltype(ctrl)::value, decltype(mask)::value, 0xf, false);
    t.i[1] = __builtin_amdgcn_update_dpp(u.i[1], u.i[1], decltype(ctrl)::value, decltype(mask)::value, 0xf, false);
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(t.d));   // fmax() would quiet both operands first
    return r;
  };
  v = step(v, std::integral_constant<int, 0x111>(), std::integral_constant<int, 0xf>());   // row_shr:1
  v = step(v, std::integral_constant<int, 0x112>(), std::integral_constant<int, 0xf>());   // row_shr:2
  v = step(v, std::integral_constant<int, 0x114>(), std::integral_constant<int, 0xf>());   // row_shr:4
  v = step(v, std::integral_constant<int, 0x118>(), std::integral_constant<int, 0xf>());   // row_shr:8
  v = step(v, std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xa>());   // row_bcast:15
  v = step(v, std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xc>());   // row_bcast:31
  union { double d; int i[2]; } r;
  r.d = v;
  r.i[0] = __builtin_amdgcn_readlane(r.i[0], 63);
  r.i[1] = __builtin_amdgcn_readlane(r.i[1], 63);
  return r.d;
}
// Maximum of lanes 0..7, in every lane.
__device__ __forceinline__ double wave_max8(double v) {
  auto step = [](double x, auto ctrl) {
    union { double d; int i[2]; } u, t;
    u.d = x;
    t.i[0] = __builtin_amdgcn_update_dpp(u.i[0], u.i[0], decltype(ctrl)::value, 0xf, 0xf, false);
    t.i[1] = __builtin_amdgcn_update_dpp(u.i[1], u.i[1], decltype(ctrl)::value, 0xf, 0xf, false);
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(t.d));
    return r;
  };
  v = step(v, std::integral_constant<int, 0x111>());
  v = step(v, std::integral_constant<int, 0x112>());
  v = step(v, std::integral_constant<int, 0x114>());
  union { double d; int i[2]; } r;
  r.d = v;
  r.i[0] = __builtin_amdgcn_readlane(r.i[0], 7);
  r.i[1] = __builtin_amdgcn_readlane(r.i[1], 7);
  return r.d;
}
__device__ __forceinline__ double wave_read(double v, int lane) {   // lane: wavefront-uniform
  union { double d; int i[2]; } u;
  u.d = v;
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], lane);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], lane);
  return u.d;
}

template <int TR>
struct PanelLDS {
  double X[2][16 * TR][4];       // the panel before and after its column steps
  double F[2][16 * TR][4];       // coefficient of pivot row k in every row's update
  double tri[2][4][4];           // [k][i < k]: pivot row k's entry in column i before step i; [k][k]: 1 / pivot k
  double row[4][4][32];          // per wavefront: the four pivot rows at its columns
  int pos[16 * TR], row_at[16 * TR], piv[16 * TR], p[2][4], stop[2];
};

// Column steps j0 .. j0 + nb - 1 (nb <= 4) on the panel in X, by one wavefront.  Returns 0 or
// INFO at a zero pivot; p[k] receives the pivot row of step k, F and tri its update (see gj_blocked).
template <int TR>
__device__ __forceinline__ int gj_panel(double (*X)[4], double (*F)[4], double (*tri)[4], int n, int j0, int nb, int* pos_, int* piv, int* p_) {
  const int lane = threadIdx.x & 63;
  const int r1 = lane + 64 < 16 * TR ? lane + 64 : 16 * TR - 1;   // rows of this lane; lanes past the tile hold no second row
  const bool in0 = lane < n, in1 = lane + 64 < 16 * TR && lane + 64 < n;
  double v[2][4], f[2][4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    f[0][k] = f[1][k] = 0.0;
    v[0][k] = lane < 16 * TR ? X[lane < 16 * TR ? lane : 0][k] : 0.0;
    v[1][k] = X[r1][k];
  }
  int pos0 = lane < 16 * TR ? pos_[lane < 16 * TR ? lane : 0] : -1, pos1 = in1 ? pos_[r1] : -1;
#pragma unroll
  for (int jj = 0; jj < 4; jj++) {
    if (jj >= nb) break;
    const int j = j0 + jj;
    auto cand = [&](double x, int ps, bool in) {
      double c = fabs(x);
      if (c != c) c = ps == j ? (double)INFINITY : -1.0;   // idamax: a NaN first element is never beaten, any other never chosen
      return in && ps >= j ? c : -1.0;
    };
    const double c0 = cand(v[0][jj], pos0, in0), c1 = cand(v[1][jj], pos1, in1);
    const double best = wave_max(c0 > c1 ? c0 : c1);
    // rows holding the maximum (the row in position j always qualifies for best >= 0); ties to the smaller position
    unsigned long long m0 = __ballot(c0 == best), m1 = __ballot(c1 == best);
    int p = m0 ? __builtin_ctzll(m0) : 64 + __builtin_ctzll(m1);
    int q = p < 64 ? __builtin_amdgcn_readlane(pos0, p) : __builtin_amdgcn_readlane(pos1, p - 64);
    if (__builtin_popcountll(m0) + __builtin_popcountll(m1) > 1) {
      while (m0) {
        const int r = __builtin_ctzll(m0), ps = __builtin_amdgcn_readlane(pos0, r);
        m0 &= m0 - 1;
        if (ps < q) { q = ps; p = r; }
      }
      while (m1) {
        const int r = __builtin_ctzll(m1), ps = __builtin_amdgcn_readlane(pos1, r);
        m1 &= m1 - 1;
        if (ps < q) { q = ps; p = 64 + r; }
      }
    }
    p = __builtin_amdgcn_readfirstlane(p);
    q = __builtin_amdgcn_readfirstlane(q);
    const int pl = p & 63;
    double u[4];
#pragma unroll
    for (int k = 0; k < 4; k++) u[k] = wave_read(p < 64 ? v[0][k] : v[1][k], pl);
    if (!(u[jj] != 0.0)) return j + 1;   // NaN passes, as in DGETF2
    // exchange of positions: the row in position j goes to the pivot row's place
    if (pos0 == j) pos0 = q;
    if (pos1 == j) pos1 = q;
    if (lane == pl) { if (p < 64) pos0 = j; else pos1 = j; }
    const double pinv = 1.0 / u[jj];
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (i < jj) {
        const double t = wave_read(p < 64 ? f[0][i] : f[1][i], pl);
        if (lane == 0) tri[jj][i] = -t;
      }
    if (lane == 0) { piv[j] = q; p_[jj] = p; tri[jj][jj] = pinv; }
#pragma unroll
    for (int k = 0; k < 4; k++) u[k] = k == jj ? pinv : u[k] * pinv;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const bool self = lane == pl && (p >> 6) == h;
      const double m = v[h][jj];
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i < jj) f[h][i] = self ? 0.0 : f[h][i];
      f[h][jj] = self ? 1.0 : -m;
      v[h][jj] = 0.0;
#pragma unroll
      for (int k = 0; k < 4; k++) v[h][k] = self ? u[k] : v[h][k] - m * u[k];
    }
  }
  if (lane < 16 * TR) {
    pos_[lane] = pos0;
#pragma unroll
    for (int k = 0; k < 4; k++) { X[lane][k] = v[0][k]; F[lane][k] = f[0][k]; }
  }
  if (lane + 64 < 16 * TR) {
    if (in1) pos_[r1] = pos1;
#pragma unroll
    for (int k = 0; k < 4; k++) { X[r1][k] = v[1][k]; F[r1][k] = f[1][k]; }
  }
  return 0;
}

// In-place inverse of the n x n block g, n <= 16 TR; returns 0, or INFO with g untouched.
template <int TR>
__device__ __forceinline__ int gj_blocked(double* __restrict__ g, int n, PanelLDS<TR>& L) {
  constexpr int TC = (TR + 3) / 4;      // tile columns of a wavefront: w, w + 4
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  gj_f64x4 a[TC][TR];
#pragma unroll
  for (int c = 0; c < TC; c++)
#pragma unroll
    for (int t = 0; t < TR; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = 16 * t + grp + 4 * r, cc = 16 * (w + 4 * c) + col;
        a[c][t][r] = row < n && cc < n ? g[(int64_t)row * n + cc] : 0.0;
      }
  for (int i = tid; i < 16 * TR; i += 256) L.pos[i] = i;
  __syncthreads();
  for (int j0 = 0, k = 0; j0 < n; j0 += 4, k ^= 1) {
    const int nb = n - j0 < 4 ? n - j0 : 4;
    const int tc = j0 >> 4, cs = tc >> 2, c4 = (j0 & 15) >> 2;   // tile column of the panel, its slot, the lanes' column group
    double (*X)[4] = L.X[k];
    if ((tc & 3) == w) {
      const int kc = col & 3;
      if ((col >> 2) == c4) {
#pragma unroll
        for (int c = 0; c < TC; c++)
          if (c == cs) {
#pragma unroll
            for (int t = 0; t < TR; t++)
#pragma unroll
              for (int r = 0; r < 4; r++) X[16 * t + grp + 4 * r][kc] = a[c][t][r];
          }
      }
      __builtin_amdgcn_wave_barrier();
      const int inf = gj_panel<TR>(X, L.F[k], L.tri[k], n, j0, nb, L.pos, L.piv, L.p[k]);
      if (lane == 0) L.stop[k] = inf;
    }
    __syncthreads();
    const int stop = __builtin_amdgcn_readfirstlane(L.stop[k]);
    if (stop) return stop;
    // pivot rows at this wavefront's columns: out to LDS, zero in the tiles
    double (*P)[32] = L.row[w];
    for (int q = 0; q < nb; q++) {
      const int p = __builtin_amdgcn_readfirstlane(L.p[k][q]);
#pragma unroll
      for (int t = 0; t < TR; t++)
        if (t == (p >> 4)) {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (r == ((p >> 2) & 3)) {
              const bool mine = grp == (p & 3);
              if constexpr (TR == 7) {   // at three waves per SIMD the selects below spill (100 DOF: +8 %; other sizes -5 %)
                if (mine)
#pragma unroll
                  for (int c = 0; c < TC; c++) { P[q][16 * c + col] = a[c][t][r]; a[c][t][r] = 0.0; }
              } else {
#pragma unroll
                for (int c = 0; c < TC; c++) {
                  if (mine) P[q][16 * c + col] = a[c][t][r];
                  a[c][t][r] = mine ? 0.0 : a[c][t][r];
                }
              }
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
    double b[TC], x[TR], tri[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int i = 0; i <= q; i++) tri[q][i] = q < nb ? L.tri[k][q][i] : 0.0;
#pragma unroll
    for (int c = 0; c < TC; c++) {
      double u[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {      // steps past nb have tri = 0
        u[q] = q < nb ? P[q][16 * c + col] : 0.0;
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (i < q) u[q] -= tri[q][i] * u[i];
        u[q] *= tri[q][q];
      }
      b[c] = grp == 0 ? u[0] : grp == 1 ? u[1] : grp == 2 ? u[2] : u[3];
    }
#pragma unroll
    for (int t = 0; t < TR; t++) x[t] = L.F[k][16 * t + col][grp];
#pragma unroll
    for (int c = 0; c < TC; c++)
      if (w + 4 * c < TR)
#pragma unroll
        for (int t = 0; t < TR; t++) a[c][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], b[c], a[c][t], 0, 0, 0);
    if ((tc & 3) == w && (col >> 2) == c4 && (col & 3) < nb) {   // the panel's own columns
#pragma unroll
      for (int c = 0; c < TC; c++)
        if (c == cs) {
#pragma unroll
          for (int t = 0; t < TR; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) a[c][t][r] = X[16 * t + grp + 4 * r][col & 3];
        }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // X[pos[r]][row placed in position c] = a[r][c]
  for (int i = tid; i < n; i += 256) L.row_at[L.pos[i]] = i;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TR; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 16 * t + grp + 4 * r;
      if (row < n) {
        const int64_t o = (int64_t)L.pos[row] * n;
#pragma unroll
        for (int c = 0; c < TC; c++) {
          const int cc = 16 * (w + 4 * c) + col;
          if (cc < n) g[o + L.row_at[cc]] = a[c][t][r];
        }
      }
    }
  return 0;
}

template <int TR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TR <= 4 ? 4 : TR == 7 ? 3 : 2))) k_block_inverse(int nblk, int nmax, const int32_t* __restrict__ nsz,
                                                                const int64_t* __restrict__ off, double* __restrict__ A,
                                                                int32_t* __restrict__ ipiv, const int64_t* __restrict__ pivoff,
                                                                int32_t* __restrict__ info) {
  __shared__ union { PanelLDS<TR> panel; TileLDS<TR> tile; } L;
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax || n > 16 * TR) {   // size outside what the launch was sized for: report, touch nothing
    if (threadIdx.x == 0 && info) info[b] = -1;
    return;
  }
  double* g = A + off[b];
  int inf = gj_blocked<TR>(g, n, L.panel);
  const int* piv = L.panel.piv;
  if (inf) {   // singular: factor the original block (LU and INFO, no inverse)
    __syncthreads();
    double a[TR][TR];
    tile_load<TR>(a, g, n, L.tile);
    inf = tile_eliminate<TR>(a, n, L.tile);
    __syncthreads();
    tile_store<TR>(a, g, n, L.tile);
    piv = L.tile.piv;
  }
  if (ipiv)
    for (int i = threadIdx.x; i < n; i += 256) ipiv[pivoff[b] + i] = piv[i] + 1;
  if (threadIdx.x == 0 && info) info[b] = inf;
}

// Small blocks (n <= 20: the 10- and 20-DOF cell blocks of XDG and p <= 2 scalar operators): G lanes
// per block (G = 16 or 32, so 64 / G blocks per wavefront), lane r of a group holds row r of its
// block in registers for the whole factorisation.  Row exchanges are bookkeeping, as in the
// workgroup-tile form: each lane carries the position its row has been given.  The pivot is the
// unused row with the largest |a| (ties to the smaller position, a NaN in position j never beaten,
// any other NaN never chosen: IDAMAX in getf2's row order), found by a shuffle argmax inside the
// group; the pivot row goes to the group's LDS slot and every lane reads it back (a group is part
// of one wavefront, whose LDS operations complete in order: no barrier).  LU: getf2's operations
// in getf2's order (multiplier a * (1 / pivot), rank-one update of the columns after j) on the
// rows after the pivot in position order.  Inverse: Gauss-Jordan in place, written out with both
// permutations applied; a zero pivot makes the group factor its block from the original values
// instead (LU and INFO).  The step loop is unrolled, so column j is a register index known at
// compile time.  No lane returns early: every shuffle has all lanes of its group taking part.
template <typename Real, int G, int NM, bool GJ>
__device__ __forceinline__ int rows_eliminate(Real (&a)[NM], int r, int n, int& pos, Real* row_slot, int* pr, int* pp, int base) {
  int inf = 0;
  bool dead = false;   // Gauss-Jordan stops at a zero pivot
#pragma unroll
  for (int j = 0; j < NM; j++) {
    if (j < n && !dead) {   // uniform over the group
      Real v = Real(-1);
      if (r < n && pos >= j) {
        v = fabs(a[j]);
        if (pos == j && v != v) v = Real(INFINITY);   // idamax: a NaN first element is never beaten
        if (!(v >= Real(0))) v = Real(-1);              // any other NaN is never a candidate
      }
      int key = v >= Real(0) ? (pos << 6) | r : 0x7fffffff;   // position first (unique), then the lane
#pragma unroll
      for (int o = G / 2; o >= 1; o >>= 1) {
        const Real ov = __shfl_xor(v, o, 64);
        const int ok = __shfl_xor(key, o, 64);
        if (ov > v || (ov == v && ok < key)) { v = ov; key = ok; }
      }
      // the row in position j is always a candidate (|a| >= 0, or a NaN made infinite), so key is set
      const int p = key & 63, ps = key >> 6;
      const Real apj = __shfl(a[j], base + p, 64);
      if (r == 0) { pr[j] = p; pp[j] = ps; }
      if (!(apj != Real(0))) {   // zero pivot (NaN passes, as in DGETF2)
        if (!inf) inf = j + 1;
        if (GJ) dead = true;
        continue;                // no exchange: the row in position j is done all the same
      }
      if (r == p) pos = j;
      else if (pos == j) pos = ps;
      const Real pinv = Real(1) / apj;
      if (r == p) {
#pragma unroll
        for (int c = 0; c < NM; c++) row_slot[c] = GJ ? (c == j ? pinv : a[c] * pinv) : a[c];
      }
      __builtin_amdgcn_wave_barrier();
      if (GJ) {
        const Real f = a[j];
        a[j] = Real(0);          // becomes -f / pivot through the update
#pragma unroll
        for (int c = 0; c < NM; c++) a[c] -= f * row_slot[c];
        if (r == p) {
#pragma unroll
          for (int c = 0; c < NM; c++) a[c] = row_slot[c];
        }
      } else if (pos > j) {      // rows after the pivot in position order
        const Real l = a[j] * pinv;
        a[j] = l;
#pragma unroll
        for (int c = j + 1; c < NM; c++) a[c] -= l * row_slot[c];
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  return inf;
}

template <typename Real, int G, int NM>
__global__ void __launch_bounds__(256) k_block_lu_rows(int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                       Real* __restrict__ A, int32_t* __restrict__ ipiv, const int64_t* __restrict__ pivoff,
                                                       int32_t* __restrict__ info, int want_inverse) {
  __shared__ Real s_row[256 / G][NM];
  __shared__ int s_pr[256 / G][NM], s_pp[256 / G][NM];   // per step: pivot row (physical), its position before the exchange
  const int r = threadIdx.x % G, grp = threadIdx.x / G;   // row of the block this lane holds, group in the workgroup
  const int b = blockIdx.x * (256 / G) + grp;
  const int base = (threadIdx.x & 63) - r;             // first lane of the group in the wavefront
  const bool inb = b < nblk;
  const int n0 = inb ? nsz[b] : 0;
  if (inb && (n0 <= 0 || n0 > nmax) && r == 0 && info) info[b] = -1;   // size outside the launch: report
  const bool ok = inb && n0 > 0 && n0 <= nmax;
  const int n = ok ? n0 : 0;
  Real* g = ok ? A + off[b] : A;
  Real a[NM];
#pragma unroll
  for (int c = 0; c < NM; c++) a[c] = (r < n && c < n) ? g[(size_t)r * n + c] : Real(0);
  int pos = r, inf = 0;
  bool inverse = false;
  if (want_inverse) {
    inf = rows_eliminate<Real, G, NM, true>(a, r, n, pos, s_row[grp], s_pr[grp], s_pp[grp], base);
    inverse = inf == 0;
    if (!inverse) {   // singular (uniform over the group): factor the original block, LU and INFO
#pragma unroll
      for (int c = 0; c < NM; c++) a[c] = (r < n && c < n) ? g[(size_t)r * n + c] : Real(0);
      pos = r;
    }
  }
  if (!inverse) inf = rows_eliminate<Real, G, NM, false>(a, r, n, pos, s_row[grp], s_pr[grp], s_pp[grp], base);
  __builtin_amdgcn_wave_barrier();
  if (ok && r < n) {
    Real* out = g + (size_t)pos * n;
    if (inverse) {
#pragma unroll
      for (int c = 0; c < NM; c++)
        if (c < n) out[s_pr[grp][c]] = a[c];   // X[pos[r]][row placed in position c] = a[r][c]
    } else {
#pragma unroll
      for (int c = 0; c < NM; c++)
        if (c < n) out[c] = a[c];
    }
    if (ipiv) ipiv[pivoff[b] + r] = s_pp[grp][r] + 1;
  }
  if (ok && r == 0 && info) info[b] = inf;
}

// Blocks above LU_MAXN (the multi-cell blocks of Schwarz smoothers, up to LU_BIG_MAXN), pivots not kept or above
// LU_REG_MAXN: in place in global memory, blocked (see the blocked forms below); the pivot search is getf2's:
// the first row with the largest |a| in the column (workgroup argmax, ties to the smaller row).
constexpr int LU_BIG_MAXN = 4096;
// the two-launch-per-panel form takes over for blocks of at least LU_SPLIT_MINN when the batch
// has fewer than LU_SPLIT_MAXBLK blocks (fewer blocks than CUs leave the one-workgroup form idle)
constexpr int LU_SPLIT_MINN = 512;
constexpr int LU_SPLIT_MAXBLK = 256;
// Returns the pivot row and, in act, whether the pivot is non-zero.  Thread 0 reads the pivot
// entry before the final barrier, so every thread decides on the same value even though the
// row swap that follows overwrites it (NaN counts as non-zero, as in DGETF2).
template <typename Real, int NT = 256>
__device__ __forceinline__ int lu_pivot_wg(const Real* a, int n, int j, Real* sv, int* si, int* s_piv, int* s_act, bool& act) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  Real best = Real(-1);
  int bi = n;
  for (int i = j + t; i < n; i += NT) {
    Real v = fabs(a[(size_t)i * n + j]);
    if (i == j && v != v) v = Real(INFINITY);   // idamax: a NaN first element is never beaten
    if (v > best || (v == best && i < bi)) { best = v; bi = i; }
  }
  wave_argmax(best, bi);
  if (lane == 0) { sv[w] = best; si[w] = bi; }
  __syncthreads();
  if (t == 0) {
    Real bv = sv[0];
    int bx = si[0];
    for (int k = 1; k < NT / 64; k++)
      if (sv[k] > bv || (sv[k] == bv && si[k] < bx)) { bv = sv[k]; bx = si[k]; }
    *s_piv = bx < n ? bx : j;   // no comparable candidate (all NaN): the diagonal, as idamax
    *s_act = a[(size_t)*s_piv * n + j] != Real(0);
  }
  __syncthreads();
  act = *s_act != 0;
  return *s_piv;
}

template <typename Real, int NT = 256>
__device__ __forceinline__ void lu_swap_rows(Real* a, int n, int r1, int r2) {
  for (int c = threadIdx.x; c < n; c += NT) {
    const Real x = a[(size_t)r1 * n + c];
    a[(size_t)r1 * n + c] = a[(size_t)r2 * n + c];
    a[(size_t)r2 * n + c] = x;
  }
}

// Blocked forms for blocks above 128 DOF (right-looking, panel width LU_NB): getf2 on the
// LU_NB columns of a panel with whole-row exchanges -- getf2's pivots, exchanges and scaling, the
// rank-1 updates applied to the panel columns only --, then U12 = L11^-1 A12 by forward
// substitution (each element gets getf2's updates in getf2's order), then the trailing update
// A22 -= L21 U12 as one rank-LU_NB product on v_mfma_f64_16x16x4f64.  Pivots, INFO and the
// factors of the panel rows are getf2's; the trailing elements receive the same products summed
// in the matrix units' order (rounding).  A column whose pivot is zero is skipped by getf2
// (no scaling, no update): its L entries count as zero in the solve and the product (zmask).
constexpr int LU_NB = 32;
typedef double lu_f64x4 __attribute__((ext_vector_type(4)));

// Panel [k0, k0 + nb) of block a (n x n, row-major), one workgroup.  Returns the panel's zero-pivot
// mask (bit jj: column k0 + jj) and sets inf to the first zero pivot (1-based) if it is still 0.
template <typename Real, int NT = 256>
__device__ __forceinline__ unsigned lu_panel(Real* a, int n, int k0, int nb, int32_t* ipiv_b, int& inf, Real* sv, int* si, int* s_piv, int* s_act) {
  const int t = threadIdx.x;
  const int kend = k0 + nb;
  unsigned zmask = 0;
  for (int j = k0; j < kend; j++) {
    bool act;
    const int p = lu_pivot_wg<Real, NT>(a, n, j, sv, si, s_piv, s_act, act);
    if (t == 0 && ipiv_b) ipiv_b[j] = p + 1;
    if (!act) {
      if (!inf) inf = j + 1;
      zmask |= 1u << (j - k0);
      __syncthreads();
      continue;
    }
    if (p != j) lu_swap_rows<Real, NT>(a, n, j, p);
    __syncthreads();
    const Real inv = Real(1) / a[(size_t)j * n + j];
    for (int i = j + 1 + t; i < n; i += NT) a[(size_t)i * n + j] *= inv;
    __syncthreads();
    const int w = kend - j - 1;   // panel columns right of j
    if (w > 0)
      for (int e = t; e < (n - j - 1) * w; e += NT) {
        const int i = j + 1 + e / w, c = j + 1 + e % w;
        a[(size_t)i * n + c] -= a[(size_t)i * n + j] * a[(size_t)j * n + c];
      }
    __syncthreads();
  }
  return zmask;
}

// U12 = L11^-1 A12 for the columns c = k0 + LU_NB + c_begin, + c_step, ... (one column per thread;
// only full panels have columns to their right).  sL: LU_NB x LU_NB staging of L11 (zero-pivot
// columns as zero), filled by the calling workgroup.
template <typename Real>
__device__ __forceinline__ void lu_trsm(Real* a, int n, int k0, unsigned zmask, int c_begin, int c_step, Real* sL) {
  for (int e = threadIdx.x; e < LU_NB * LU_NB; e += blockDim.x) {
    const int i = e / LU_NB, q = e % LU_NB;
    sL[e] = (q < i && !((zmask >> q) & 1u)) ? a[(size_t)(k0 + i) * n + k0 + q] : Real(0);
  }
  __syncthreads();
#pragma unroll 1
  for (int c = k0 + LU_NB + c_begin; c < n; c += c_step) {
    Real* pc = a + (size_t)k0 * n + c;
    Real u[LU_NB];
#pragma unroll
    for (int i = 0; i < LU_NB; i++) u[i] = pc[i * n];
    // column-oriented: u[i] -= L[i][q] u[q] for q = 0, 1, ... -- per element the order of getf2's steps
#pragma unroll
    for (int q = 0; q < LU_NB - 1; q++) {
      asm volatile("" ::: "memory");   // L11 is read column by column in each pass, not hoisted out of the loop over c
      const Real uq = u[q];
#pragma unroll
      for (int i = q + 1; i < LU_NB; i++) u[i] -= sL[i * LU_NB + q] * uq;
    }
#pragma unroll
    for (int i = 1; i < LU_NB; i++) pc[i * n] = u[i];
  }
}

// A22 -= L21 U12 on 16 x 16 tiles of the trailing matrix (rows and columns >= k0 + LU_NB, full
// panels only): each wavefront takes the tile rows ti = r_begin, + r_step, ... and keeps that
// row's L21 operands in registers while it walks the tile columns.
template <typename Real>
__device__ __forceinline__ void lu_trail(Real* a, int n, int k0, unsigned zmask, int r_begin, int r_step) {
  const int k1 = k0 + LU_NB, m = n - k1;
  if (m <= 0) return;
  const int T = (m + 15) / 16;
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const Real* U = a + (size_t)k0 * n;            // U12 rows k0 .. k0 + LU_NB - 1
#pragma unroll 1
  for (int ti = r_begin; ti < T; ti += r_step) {
    const int r0 = k1 + 16 * ti;
    Real av[LU_NB / 4];
#pragma unroll
    for (int kk = 0; kk < LU_NB / 4; kk++) {
      const int q = 4 * kk + grp;                           // panel column this lane supplies
      const int row = r0 + col;                             // A row this lane supplies
      av[kk] = (row < n && !((zmask >> q) & 1u)) ? -a[(size_t)row * n + k0 + q] : Real(0);
    }
#pragma unroll 1
    for (int tj = 0; tj < T; tj++) {
      const int c = k1 + 16 * tj + col;
      lu_f64x4 acc;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = r0 + grp + 4 * r;
        acc[r] = (row < n && c < n) ? a[(size_t)row * n + c] : Real(0);
      }
#pragma unroll
      for (int kk = 0; kk < LU_NB / 4; kk++) {
        const Real bv = c < n ? U[(4 * kk + grp) * n + c] : Real(0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[kk], bv, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = r0 + grp + 4 * r;
        if (row < n && c < n) a[(size_t)row * n + c] = acc[r];
      }
    }
  }
}

// One workgroup per block, every panel in turn.
template <typename Real>
__global__ void __launch_bounds__(256) k_block_lu_blocked(int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                          Real* __restrict__ A, int32_t* __restrict__ ipiv, const int64_t* __restrict__ pivoff,
                                                          int32_t* __restrict__ info) {
  __shared__ Real sv[4];
  __shared__ int si[4];
  __shared__ int s_piv, s_act;
  __shared__ Real sL[LU_NB * LU_NB];
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax) {
    if (threadIdx.x == 0 && info) info[b] = -1;
    return;
  }
  Real* a = A + off[b];
  int32_t* ipiv_b = ipiv ? ipiv + pivoff[b] : nullptr;
  int inf = 0;
  for (int k0 = 0; k0 < n; k0 += LU_NB) {
    const int nb = n - k0 < LU_NB ? n - k0 : LU_NB;
    const unsigned zmask = lu_panel(a, n, k0, nb, ipiv_b, inf, sv, si, &s_piv, &s_act);
    if (k0 + nb < n) {   // a full panel with columns to its right
      lu_trsm(a, n, k0, zmask, (int)threadIdx.x, 256, sL);
      __syncthreads();
      lu_trail(a, n, k0, zmask, (int)(threadIdx.x >> 6), 4);
      __syncthreads();
    }
  }
  if (threadIdx.x == 0 && info) info[b] = inf;
}

// The same for few large blocks, two launches per panel.  k_lu_panel (one workgroup per block)
// factors the panel and solves U12; st[b] holds the block's INFO so far (-1: invalid size),
// st[nblk + b] the panel's zero-pivot mask.  k_lu_trail spreads the trailing product of every
// block over gridDim.x workgroups per block.
constexpr int LU_PANEL_THREADS = 512;   // few blocks: the panel's column steps get 8 wavefronts
template <typename Real>
__global__ void __launch_bounds__(LU_PANEL_THREADS) k_lu_panel(int k0, int nblk, int nmax, const int32_t* __restrict__ nsz,
                                                               const int64_t* __restrict__ off, Real* __restrict__ A,
                                                               int32_t* __restrict__ ipiv, const int64_t* __restrict__ pivoff,
                                                               int32_t* __restrict__ st) {
  __shared__ Real sv[LU_PANEL_THREADS / 64];
  __shared__ int si[LU_PANEL_THREADS / 64];
  __shared__ int s_piv, s_act;
  __shared__ Real sL[LU_NB * LU_NB];
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (k0 == 0 && threadIdx.x == 0) st[b] = (n <= 0 || n > nmax) ? -1 : 0;
  if (n <= 0 || n > nmax || k0 >= n) return;
  Real* a = A + off[b];
  int inf = k0 == 0 ? 0 : st[b];
  const int nb = n - k0 < LU_NB ? n - k0 : LU_NB;
  const unsigned zmask = lu_panel<Real, LU_PANEL_THREADS>(a, n, k0, nb, ipiv ? ipiv + pivoff[b] : nullptr, inf, sv, si, &s_piv, &s_act);
  if (k0 + nb < n) lu_trsm(a, n, k0, zmask, (int)threadIdx.x, LU_PANEL_THREADS, sL);
  if (threadIdx.x == 0) { st[b] = inf; st[nblk + b] = (int32_t)zmask; }
}

template <typename Real>
__global__ void __launch_bounds__(256) k_lu_trail(int k0, int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                  Real* __restrict__ A, const int32_t* __restrict__ st) {
  const int b = blockIdx.y;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax || k0 + LU_NB >= n) return;
  lu_trail(A + off[b], n, k0, (unsigned)st[nblk + b], (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), (int)(gridDim.x * 4));
}

__global__ void k_lu_info(int nblk, const int32_t* __restrict__ st, int32_t* __restrict__ info) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < nblk) info[b] = st[b];
}


// Blocks of 129..LU_REG_MAXN DOF whose pivots the caller keeps: the panel in registers, two launches
// per panel and nothing else kept between them (a zero-pivot column is one whose diagonal is zero).
//
// k_lu_panel_reg: one workgroup of 512 threads per block, thread t holds the panel rows k0 + t and
// k0 + 512 + t (32 columns each).  A column step is a wavefront maximum, one exchange of the eight
// wavefront winners and one of the pivot row through LDS (two barriers), and the rank-one update of
// the panel in registers; the panel's columns are walked in four groups of eight that rotate through
// the same registers, so the loop body stays small.  Operations and order are getf2's.
// k_lu_update: one workgroup per 32 columns outside the panel applies the panel's 32 row exchanges
// (as one permutation, every value read before any is written), and to the right of the panel the
// solve with L11 and the product A22 -= L21 U12 on the matrix units.
//
// Bound: the latency of the column steps (1.5 us each at 500 rows, 0.8 us below 256; 4.6 us in the form
// that searches, swaps and updates in global memory, k_lu_panel).  48 blocks of 200..540 DOF, factored:
// 3.4 ms before, 1.3 ms here; 300 of 200 1.07 -> 0.58 ms, 300 of 1024 67 -> 22 ms; factors and pivots the
// same to the bit.  Measured and not kept: the panel rows turned through LDS for coalesced access
// (48 -> 56 us per panel), exchanged rows moved between threads instead of their positions (64 us).
constexpr int LU_REG_MAXN = 1024, LU_COLS = 32;

template <int THREADS>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) k_lu_panel_reg(int k0, int nblk, int nmax, const int32_t* __restrict__ nsz,
                                                          const int64_t* __restrict__ off, double* __restrict__ A,
                                                          int32_t* __restrict__ piv, const int64_t* __restrict__ pivoff) {
  constexpr int W = THREADS / 64;
  static_assert(W == 4 || W == 8, "the winners of the wavefronts are reduced over eight lanes");
  __shared__ double s_val[2][8];
  __shared__ int s_pos[2][8];
  __shared__ __align__(16) double s_piv[2][LU_NB];
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax || k0 >= n || n - k0 > 2 * THREADS) return;   // (the launch's thread count covers nmax)
  double* a = A + off[b] + k0;
  int32_t* pb = piv + pivoff[b] + k0;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nb = n - k0 < LU_NB ? n - k0 : LU_NB;
  // rows stay with their threads; pos is the position (row of the factors) the exchanges have given them
  int pos[2] = {k0 + t, k0 + THREADS + t};
  const bool two = k0 + THREADS < n, in[2] = {pos[0] < n, pos[1] < n};
  double v[2][LU_NB];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < LU_NB; c++) v[h][c] = in[h] && c < nb ? a[(size_t)pos[h] * n + c] : 0.0;
  if (t < 16) { s_val[t >> 3][t & 7] = -1.0; s_pos[t >> 3][t & 7] = 1 << 30; }
  __syncthreads();
#pragma unroll 1
  for (int s = 0; s < LU_NB / 8; s++) {
#pragma unroll
    for (int jj = 0; jj < 8; jj++) {
      const int jl = 8 * s + jj, j = k0 + jl, k = jj & 1;
      if (jl < nb) {
        auto cand = [&](double x, int ps, bool ok) {
          double c = fabs(x);
          if (c != c) c = ps == j ? (double)INFINITY : -1.0;   // idamax: a NaN first element is never beaten, any other never chosen
          return ok && ps >= j ? c : -1.0;
        };
        const double c0 = cand(v[0][jj], pos[0], in[0]), c1 = two ? cand(v[1][jj], pos[1], in[1]) : -1.0;
        const double best = wave_max(c0 > c1 ? c0 : c1);
        // smallest position among the rows holding the maximum
        auto first = [&](unsigned long long m, int ps) {
          int r = 1 << 30;
          for (; m; m &= m - 1) r = std::min(r, __builtin_amdgcn_readlane(ps, __builtin_ctzll(m)));
          return r;
        };
        if (best >= 0.0) {
          int q = first(__ballot(c0 == best), pos[0]);
          if (two) q = std::min(q, first(__ballot(c1 == best), pos[1]));
          if (lane == 0) { s_val[k][w] = best; s_pos[k][w] = q; }
        } else if (lane == 0) {
          s_val[k][w] = -1.0;
        }
        __syncthreads();
        const double bv = s_val[k][lane & 7];
        const int bp = s_pos[k][lane & 7];
        const int q = __builtin_amdgcn_readfirstlane(first(__ballot(bv == wave_max8(bv)) & 0xff, bp));   // the row in position j always takes part
        if (pos[0] == q)
#pragma unroll
          for (int c = 0; c < LU_NB; c++) s_piv[k][c] = v[0][c];
        if (two && pos[1] == q)
#pragma unroll
          for (int c = 0; c < LU_NB; c++) s_piv[k][c] = v[1][c];
        if (t == 0) pb[jl] = q + 1;
        __syncthreads();
        const double pv = s_piv[k][jj];
        if (pv != 0.0) {   // NaN passes, as in DGETF2; a zero pivot leaves the column as it is
#pragma unroll
          for (int h = 0; h < 2; h++) pos[h] = pos[h] == q ? j : (pos[h] == j ? q : pos[h]);
          const double inv = 1.0 / pv;
          const bool act[2] = {in[0] && pos[0] > j, in[1] && pos[1] > j};
          double l[2];
#pragma unroll
          for (int h = 0; h < 2; h++) {
            l[h] = v[h][jj] * inv;
            if (act[h]) v[h][jj] = l[h];
          }
#pragma unroll
          for (int g = 0; g < LU_NB / 8; g++)
            if (g == 0 || s < LU_NB / 8 - g) {   // column groups still to be factored
              double u[8];
#pragma unroll
              for (int c = 0; c < 8; c++) u[c] = s_piv[k][8 * g + c];
              if (act[0])
#pragma unroll
                for (int c = g == 0 ? jj + 1 : 0; c < 8; c++) v[0][8 * g + c] -= l[0] * u[c];
              if (two && act[1])
#pragma unroll
                for (int c = g == 0 ? jj + 1 : 0; c < 8; c++) v[1][8 * g + c] -= l[1] * u[c];
            }
        }
      }
    }
    // the next eight columns move to the front
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const double x = v[h][c];
        v[h][c] = v[h][c + 8];
        v[h][c + 8] = v[h][c + 16];
        v[h][c + 16] = v[h][c + 24];
        v[h][c + 24] = x;
      }
  }
#pragma unroll
  for (int h = 0; h < 2; h++)
    if (in[h])
#pragma unroll
      for (int c = 0; c < LU_NB; c++)
        if (c < nb) a[(size_t)pos[h] * n + c] = v[h][c];
}

__global__ void __launch_bounds__(256, 3) k_lu_update(int k0, int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                   double* __restrict__ A, const int32_t* __restrict__ piv, const int64_t* __restrict__ pivoff) {
  __shared__ double sU[LU_NB][LU_COLS + 1], sL[LU_NB][LU_NB];
  __shared__ int s_src[LU_NB], s_dst[LU_NB];
  __shared__ unsigned s_zero;
  const int b = blockIdx.y;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || n > nmax || n > LU_REG_MAXN || k0 >= n) return;
  const int nb = n - k0 < LU_NB ? n - k0 : LU_NB, k1 = k0 + LU_NB, nleft = k0 / LU_COLS;
  const bool right = (int)blockIdx.x >= nleft;
  const int c0 = right ? k1 + ((int)blockIdx.x - nleft) * LU_COLS : (int)blockIdx.x * LU_COLS;
  if (c0 >= n) return;
  double* a = A + off[b];
  const int32_t* pb = piv + pivoff[b] + k0;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  if (w == 0) {
    // where the exchanges take each row involved: lane d < 32 follows panel row k0 + d, lane 32 + q the row of pivot q
    const int q = lane & 31, pq = q < nb ? pb[q] - 1 : k0 + q, orig = lane < 32 ? k0 + lane : pq;
    int loc = orig;
#pragma unroll
    for (int i = 0; i < LU_NB; i++) {
      const int p = __builtin_amdgcn_readlane(pq, i), j = k0 + i;
      loc = loc == j ? p : (loc == p ? j : loc);
    }
    if (lane < 32) s_dst[lane] = loc;
    if (loc >= k0 && loc < k1) s_src[loc - k0] = orig;
    const bool z = q < nb && a[(size_t)(k0 + q) * n + k0 + q] == 0.0;
    const unsigned long long zm = __ballot(z);
    if (lane == 0) s_zero = (unsigned)zm;
  }
  __syncthreads();
  // exchanges: thread (column, part) moves four of the panel rows
  const int c = c0 + (t & 31), part = t >> 5;
  const bool in = c < n;
  double top[4], old[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int d = 4 * part + i;
    top[i] = in && d < nb ? a[(size_t)s_src[d] * n + c] : 0.0;
    old[i] = in && d < nb ? a[(size_t)(k0 + d) * n + c] : 0.0;
  }
  const unsigned zmask = s_zero;
  if (right)
    for (int e = t; e < LU_NB * LU_NB; e += 256) {
      const int i = e / LU_NB, q = e % LU_NB;
      sL[q][i] = (q < i && !((zmask >> q) & 1u)) ? a[(size_t)(k0 + i) * n + k0 + q] : 0.0;   // column q of L11
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int d = 4 * part + i;
    if (in && d < nb) {
      if (s_dst[d] >= k1) a[(size_t)s_dst[d] * n + c] = old[i];
      if (!right && s_src[d] != k0 + d) a[(size_t)(k0 + d) * n + c] = top[i];
    }
  }
  if (!right) return;   // (the block is uniform in this)
  // U12 = L11^-1 A12, four rows after the other: per element the order of getf2's steps
#pragma unroll 1
  for (int qb = 0; qb < LU_NB / 4; qb++) {
    if (part == qb) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int i = q + 1; i < 4; i++) top[i] -= sL[4 * qb + q][4 * qb + i] * top[q];
        sU[4 * qb + q][t & 31] = top[q];
      }
    }
    __syncthreads();
    if (part > qb) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const double uq = sU[4 * qb + q][t & 31];
#pragma unroll
        for (int i = 0; i < 4; i++) top[i] -= sL[4 * qb + q][4 * part + i] * uq;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (in) a[(size_t)(k0 + 4 * part + i) * n + c] = top[i];
  const int col = lane & 15, grp = lane >> 4;
  double u[2][LU_NB / 4];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int kk = 0; kk < LU_NB / 4; kk++) u[h][kk] = sU[4 * kk + grp][16 * h + col];
#pragma unroll 1
  for (int r0 = k1 + 16 * w; r0 < n; r0 += 128) {   // tile rows r0 and r0 + 64, their loads together
    double l[2][LU_NB / 4];
    gj_f64x4 acc[2][2];
#pragma unroll
    for (int g = 0; g < 2; g++) {
#pragma unroll
      for (int kk = 0; kk < LU_NB / 4; kk++) {
        const int q = 4 * kk + grp, r = r0 + 64 * g + col;
        l[g][kk] = r < n && !((zmask >> q) & 1u) ? -a[(size_t)r * n + k0 + q] : 0.0;
      }
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int r = r0 + 64 * g + grp + 4 * i, cc = c0 + 16 * h + col;
          acc[g][h][i] = r < n && cc < n ? a[(size_t)r * n + cc] : 0.0;
        }
    }
#pragma unroll
    for (int kk = 0; kk < LU_NB / 4; kk++)
#pragma unroll
      for (int g = 0; g < 2; g++)
#pragma unroll
        for (int h = 0; h < 2; h++) acc[g][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(l[g][kk], u[h][kk], acc[g][h], 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int r = r0 + 64 * g + grp + 4 * i, cc = c0 + 16 * h + col;
          if (r < n && cc < n) a[(size_t)r * n + cc] = acc[g][h][i];
        }
  }
}

// INFO of the factored blocks: the first zero on the diagonal (1-based), 0, or -1 for an invalid size.
__global__ void __launch_bounds__(64) k_lu_first_zero(int nblk, int nmax, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                      const double* __restrict__ A, int32_t* __restrict__ info) {
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  int inf = n <= 0 || n > nmax ? -1 : 0;
  for (int j0 = 0; j0 < n && !inf; j0 += 64) {
    const int j = j0 + (int)threadIdx.x;
    const unsigned long long z = __ballot(j < n && A[off[b] + (int64_t)j * n + j] == 0.0);
    if (z) inf = j0 + __builtin_ctzll(z) + 1;
  }
  if (threadIdx.x == 0) info[b] = inf;
}

// x_b <- LU_b \ x_b   (getrs with the 1-based pivots), two kernels that each take their block sizes; any size.
//
// Up to SOLVE_SMALL DOF: one wavefront per block, lane l holds x_l and x_64+l in registers.  The
// substitutions run column by column; the finished x_j reaches the other lanes as a scalar and the
// factor's columns, which do not depend on it, are loaded ahead.  The forward sweep adds the terms of a
// row in getrs' order (k = 0 .. i-1), the backward sweep from the last column.
//
// Up to LU_BIG_MAXN, the largest x that LDS holds: one workgroup per block, x in LDS, SOLVE_T columns at a time: one wavefront solves the diagonal
// tile, staged in LDS, then every wavefront subtracts the finished entries from groups of 64 rows, lane
// by lane in the same order.  The factor does not depend on x, so the next tile and every wavefront's
// first group are loaded (coalesced, turned in LDS) while the diagonal tile is solved.
//
// Above (factors that were made elsewhere): one wavefront per block, x in place (solve_in_memory).
//
// Bound: the 2 n dependent steps of the diagonal tiles, half of them with a division.  48 blocks of
// 200..540 DOF: 1.67 ms by one wavefront per block walking the factor's columns in memory, 0.20 ms here;
// 300 of 128 DOF 0.135 -> 0.062 ms, 31000 of 10 DOF 88 -> 79 us, of 10 and 20 mixed 171 -> 119 us (the wide kernel's
// workgroups that find a small block and return are within these).  Measured and not kept: lane partial sums of the rows (0.20 ms too, and
// other rounding), the division by a Newton step on a reciprocal (0.23 ms).
constexpr int SOLVE_SMALL = 128, SOLVE_T = 64, SOLVE_WAVES = 8;

// One wavefront, lane l owns the rows l (mod 64) of x and is the only one to write them; column by column,
// the finished x_j reaches the other lanes by a shuffle from its owner.
__device__ void solve_in_memory(int n, const double* __restrict__ L, const int32_t* __restrict__ pv, double* x) {
  const int lane = threadIdx.x;
  if (lane == 0)
    for (int j = 0; j < n; j++) {
      const int p = pv[j] - 1;
      if (p != j) { const double t = x[j]; x[j] = x[p]; x[p] = t; }
    }
  __syncthreads();   // the interchanged entries are read by their owners below
  for (int j = 0; j < n; j++) {
    double xj = lane == (j & 63) ? x[j] : 0.0;
    xj = __shfl(xj, j & 63, 64);
    for (int i = lane + (lane <= j ? ((j - lane) / 64 + 1) * 64 : 0); i < n; i += 64) x[i] -= L[(size_t)i * n + j] * xj;
  }
  for (int j = n - 1; j >= 0; j--) {
    double xj = 0.0;
    if (lane == (j & 63)) {
      xj = x[j] / L[(size_t)j * n + j];
      x[j] = xj;
    }
    xj = __shfl(xj, j & 63, 64);
    for (int i = lane; i < j; i += 64) x[i] -= L[(size_t)i * n + j] * xj;
  }
}

__global__ void __launch_bounds__(64) k_block_solve(int nblk, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                    const double* __restrict__ LU, const int32_t* __restrict__ ipiv,
                                                    const int64_t* __restrict__ pivoff, const int64_t* __restrict__ xoff,
                                                    double* __restrict__ x) {
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= 0 || (n > SOLVE_SMALL && n <= LU_BIG_MAXN)) return;
  if (n > LU_BIG_MAXN) {
    solve_in_memory(n, LU + off[b], ipiv + pivoff[b], x + xoff[b]);
    return;
  }
  const int lane = threadIdx.x;
  const double* L = LU + off[b];
  const int32_t* pv = ipiv + pivoff[b];
  double* xb = x + xoff[b];
  const int r[2] = {lane, lane + 64};
  double v[2];
  int p[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    v[h] = r[h] < n ? xb[r[h]] : 0.0;
    p[h] = r[h] < n ? pv[r[h]] - 1 : r[h];
  }
  auto entry = [&](int j) { return j < 64 ? wave_read(v[0], j) : wave_read(v[1], j - 64); };   // j: uniform
  auto set = [&](int j, double y) {
    if (lane == (j & 63)) { if (j < 64) v[0] = y; else v[1] = y; }
  };
#pragma unroll
  for (int h = 0; h < 2; h++)
    for (unsigned long long m = __ballot(p[h] != r[h]); m; m &= m - 1) {   // exchanges, in order
      const int j = 64 * h + __builtin_ctzll(m), q = __builtin_amdgcn_readlane(p[h], j & 63);
      const double xj = entry(j), xq = entry(q);
      set(j, xq);
      set(q, xj);
    }
  // columns in batches whose loads are issued together (rows and columns clamped into the block)
  constexpr int B = 8;
  const double* row[2] = {L + (size_t)(r[0] < n ? r[0] : n - 1) * n, L + (size_t)(r[1] < n ? r[1] : n - 1) * n};
  const bool two = n > 64;
  for (int j0 = 0; j0 < n; j0 += B) {
    double l[2][B];
#pragma unroll
    for (int i = 0; i < B; i++) {
      const int j = j0 + i < n ? j0 + i : n - 1;
      l[0][i] = row[0][j];
      if (two) l[1][i] = row[1][j];
    }
#pragma unroll
    for (int i = 0; i < B; i++) {
      const int j = j0 + i;
      if (j < n) {
        const double xj = entry(j);
        if (r[0] > j) v[0] -= l[0][i] * xj;
        if (two && r[1] > j) v[1] -= l[1][i] * xj;
      }
    }
  }
  for (int j0 = n - 1; j0 >= 0; j0 -= B) {
    double u[2][B];
#pragma unroll
    for (int i = 0; i < B; i++) {
      const int j = j0 - i > 0 ? j0 - i : 0;
      u[0][i] = row[0][j];
      u[1][i] = two ? row[1][j] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < B; i++) {
      const int j = j0 - i;
      if (j >= 0) {
        const double xj = entry(j) / (j < 64 ? wave_read(u[0][i], j) : wave_read(u[1][i], j - 64));
        set(j, xj);
        if (r[0] < j) v[0] -= u[0][i] * xj;
        if (two && r[1] < j) v[1] -= u[1][i] * xj;
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 2; h++)
    if (r[h] < n) xb[r[h]] = v[h];
}

__global__ void __launch_bounds__(64 * SOLVE_WAVES) k_block_solve_wide(int nblk, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                                       const double* __restrict__ LU, const int32_t* __restrict__ ipiv,
                                                                       const int64_t* __restrict__ pivoff, const int64_t* __restrict__ xoff,
                                                                       double* __restrict__ x) {
  constexpr int NT = 64 * SOLVE_WAVES, TE = SOLVE_T * SOLVE_T / NT;
  __shared__ double xs[LU_BIG_MAXN];
  __shared__ double tile[SOLVE_T][SOLVE_T + 1];
  __shared__ double turn[SOLVE_WAVES][64][17];
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  if (n <= SOLVE_SMALL || n > LU_BIG_MAXN) return;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const double* L = LU + off[b];
  const int32_t* pv = ipiv + pivoff[b];
  double* xb = x + xoff[b];
  for (int i = t; i < n; i += NT) xs[i] = xb[i];
  double next[TE];        // this thread's entries of the next diagonal tile
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int i = 0; i < TE; i++) {
      const int e = t + NT * i, r = k0 + e / SOLVE_T, c = k0 + e % SOLVE_T;
      next[i] = r < n && c < n ? L[(size_t)r * n + c] : 0.0;
    }
  };
  load_tile(0);
  __syncthreads();
  if (w == 0)
    for (int j0 = 0; j0 < n; j0 += 64) {   // exchanges, in order; rows that stay are skipped
      const int p = j0 + lane < n ? pv[j0 + lane] - 1 : j0 + lane;
      for (unsigned long long m = __ballot(p != j0 + lane); m; m &= m - 1) {
        const int i = __builtin_ctzll(m), q = __builtin_amdgcn_readlane(p, i);
        if (lane == 0) { const double y = xs[j0 + i]; xs[j0 + i] = xs[q]; xs[q] = y; }
      }
    }
  const int T = (n + SOLVE_T - 1) / SOLVE_T;
#pragma unroll 1
  for (int step = 0; step < 2 * T; step++) {
    const bool lower = step < T;
    const int k0 = SOLVE_T * (lower ? step : 2 * T - 1 - step), k1 = k0 + SOLVE_T < n ? k0 + SOLVE_T : n, m = k1 - k0;
    const int ra = lower ? k1 : 0, rb = lower ? n : k0;   // rows the finished entries are subtracted from
    // (the last reader of the tile, the solve below, is a barrier behind)
#pragma unroll
    for (int i = 0; i < TE; i++) {
      const int e = t + NT * i;
      tile[e / SOLVE_T][e % SOLVE_T] = next[i];
    }
    // columns k0 .. k1 of rows base .. base + 63, four rows of 16 columns per load
    double pre[4][16];
    auto load_rows = [&](int base) {
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int r = base + 4 * i + (lane >> 4), c = k0 + 16 * s + (lane & 15);
          pre[s][i] = r < rb && c < k1 ? L[(size_t)r * n + c] : 0.0;
        }
    };
    if (ra + 64 * w < rb) load_rows(ra + 64 * w);
    if (step + 1 < 2 * T) load_tile(SOLVE_T * (step + 1 < T ? step + 1 : 2 * T - 2 - step));
    __syncthreads();
    if (w == 0) {
      double v = lane < m ? xs[k0 + lane] : 0.0;
      if (lower) {
#pragma unroll 8
        for (int j = 0; j < m; j++) {
          const double l = tile[lane][j], xj = wave_read(v, j);
          if (lane > j) v -= l * xj;
        }
      } else {
        const double d = tile[lane][lane];
#pragma unroll 8
        for (int j = m - 1; j >= 0; j--) {
          const double u = tile[lane][j];
          if (lane == j) v = v / d;
          const double xj = wave_read(v, j);
          if (lane < j) v -= u * xj;
        }
      }
      if (lane < m) xs[k0 + lane] = v;
    }
    __syncthreads();
    for (int base = ra + 64 * w; base < rb; base += NT) {
      if (base != ra + 64 * w) load_rows(base);
      const int r = base + lane;
      double y = r < rb ? xs[r] : 0.0;
      double (*T2)[17] = turn[w];
#pragma unroll
      for (int ss = 0; ss < 4; ss++) {
        auto part = [&](const double (&p)[16], int s) {
#pragma unroll
          for (int i = 0; i < 16; i++) T2[4 * i + (lane >> 4)][lane & 15] = p[i];
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int q = 0; q < 16; q++) {
            const int j = lower ? q : 15 - q;
            if (16 * s + j < m) y -= T2[lane][j] * xs[k0 + 16 * s + j];
          }
          __builtin_amdgcn_wave_barrier();
        };
        if (lower) part(pre[ss], ss);
        else part(pre[3 - ss], 3 - ss);
      }
      if (r < rb) xs[r] = y;
    }
  }
  __syncthreads();
  for (int i = t; i < n; i += NT) xb[i] = xs[i];
}

// y_b <- alpha * Ainv_b x_b + beta * y_b   (block-diagonal apply with explicit inverses, one wave per block)
template <typename Real>
__global__ void __launch_bounds__(64) k_block_gemv(int nblk, const int32_t* __restrict__ nsz, const int64_t* __restrict__ off,
                                                   const Real* __restrict__ Ainv, const int64_t* __restrict__ xoff, Real alpha,
                                                   const Real* __restrict__ xin, Real beta, Real* __restrict__ y) {
  const int b = blockIdx.x;
  if (b >= nblk) return;
  const int n = nsz[b];
  const Real* M = Ainv + off[b];
  const Real* xb = xin + xoff[b];
  Real* yb = y + xoff[b];
  for (int i = threadIdx.x; i < n; i += 64) {
    Real a = 0;
    for (int k = 0; k < n; k++) a += M[i * n + k] * xb[k];
    yb[i] = alpha * a + (beta != Real(0) ? beta * yb[i] : Real(0));
  }
}

}  // namespace bosss

using namespace bosss;

namespace bosss {
int ctx_device_stream(bosss_ctx* ctx, int* device, hipStream_t* stream);
}

namespace {
thread_local std::string g_lu_err;

// With a context, launch on its device (the stream argument must belong to that device);
// without one, on the calling thread's current device.
int select_device(bosss_ctx* ctx) {
  if (!ctx) return BOSSS_OK;
  int dev = 0;
  hipStream_t st = nullptr;
  if (bosss::ctx_device_stream(ctx, &dev, &st) != BOSSS_OK) { g_lu_err = "bad context"; return BOSSS_ERR_ARG; }
  if (hipSetDevice(dev) != hipSuccess) { g_lu_err = "hipSetDevice failed"; return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}
}

// ---- scratch of the allocation-free factorisation (bosss_hip_block_lu_noalloc_dev) ----
// The split form keeps two status words per block between its launches.  The no-alloc entry
// point takes them from this file-scope array instead of a per-call allocation: every device the
// library runs on holds its own copy (8 KiB) until the process ends, and every call on one device
// shares it, so calls that overlap on one device race.  Every word a call reads it has written
// itself earlier in the same call (k_lu_panel writes a block's words before k_lu_trail and the
// next k_lu_panel read them), so nothing needs clearing between calls.
constexpr int LU_NOALLOC_MAXBLK = 1024;
static __device__ __align__(256) int32_t scratch[2 * LU_NOALLOC_MAXBLK];

namespace {
constexpr int LU_NOALLOC_MAXDEV = 64;
std::mutex g_scratch_mu;
int32_t* g_scratch_ptr[LU_NOALLOC_MAXDEV] = {};   // device address of each device's copy of scratch

// The address of the current device's copy of scratch, looked up once per device (a host-side
// name of a __device__ array is not a device address; hipGetSymbolAddress gives that device's).
int scratch_on_current_device(int32_t** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) { g_lu_err = std::string("hipGetDevice: ") + hipGetErrorString(e); return BOSSS_ERR_HIP; }
  if (dev < 0 || dev >= LU_NOALLOC_MAXDEV) { g_lu_err = "device index out of range for the scratch table"; return BOSSS_ERR_ARG; }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      g_lu_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return BOSSS_ERR_HIP;
    }
    g_scratch_ptr[dev] = static_cast<int32_t*>(p);
  }
  *out = g_scratch_ptr[dev];
  return BOSSS_OK;
}
}  // namespace

// Argument checks shared by the factorisation entry points (selects ctx's device).
static int lu_check_args(bosss_ctx* ctx, int32_t nmax, const int32_t* n, const int64_t* off, const double* A, const int32_t* ipiv,
                         const int64_t* pivoff) {
  if (int rc = select_device(ctx)) return rc;
  if (!n || !off || !A || (ipiv && !pivoff)) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  if (nmax <= 0 || nmax > LU_BIG_MAXN) { g_lu_err = "block size out of range (1..4096)"; return BOSSS_ERR_ARG; }
  return BOSSS_OK;
}

// Blocks up to LU_MAXN, in registers: up to 20 DOF several blocks per wavefront, 21..128 one workgroup per block.
static int lu_launch_reg(int nblk, int nmax, const int32_t* n, const int64_t* off, double* A, int32_t* ipiv, const int64_t* pivoff,
                         int32_t* info, int want_inverse, hipStream_t s) {
  if (nmax <= 20) {
    // rows in registers, 64 / G blocks per wavefront (larger rows would not fit one lane's
    // registers: those blocks take the workgroup-tile kernel)
    if (nmax <= 16)
      hipLaunchKernelGGL((k_block_lu_rows<double, 16, 16>), dim3((unsigned)((nblk + 15) / 16)), dim3(256), 0, s, nblk, nmax, n, off, A,
                         ipiv, pivoff, info, want_inverse);
    else
      hipLaunchKernelGGL((k_block_lu_rows<double, 32, 20>), dim3((unsigned)((nblk + 7) / 8)), dim3(256), 0, s, nblk, nmax, n, off, A,
                         ipiv, pivoff, info, want_inverse);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
    return BOSSS_OK;
  }
  // 21..128: one workgroup per block, the block in registers
  const dim3 grid((unsigned)nblk), blk(256);
#define LU_TILE(RA)                                                                                                     \
  if (want_inverse)                                                                                                     \
    hipLaunchKernelGGL(k_block_inverse<RA>, grid, blk, 0, s, nblk, nmax, n, off, A, ipiv, pivoff, info);                \
  else                                                                                                                  \
    hipLaunchKernelGGL(k_block_lu_tile<RA>, grid, blk, 0, s, nblk, nmax, n, off, A, ipiv, pivoff, info);
  if (nmax <= 32) {
    LU_TILE(2)
  } else if (nmax <= 64) {
    LU_TILE(4)
  } else if (nmax <= 112) {
    LU_TILE(7)
  } else {
    LU_TILE(8)
  }
#undef LU_TILE
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

// Blocks of 129..LU_REG_MAXN DOF, panels in registers; piv: the caller's pivots.
static int lu_launch_panels(int nblk, int nmax, const int32_t* n, const int64_t* off, double* A, int32_t* piv, const int64_t* pivoff,
                            int32_t* info, hipStream_t s) {
  for (int k0 = 0; k0 < nmax; k0 += LU_NB) {
    if (nmax - k0 <= 512) hipLaunchKernelGGL(k_lu_panel_reg<256>, dim3(nblk), dim3(256), 0, s, k0, nblk, nmax, n, off, A, piv, pivoff);
    else hipLaunchKernelGGL(k_lu_panel_reg<512>, dim3(nblk), dim3(512), 0, s, k0, nblk, nmax, n, off, A, piv, pivoff);
    const int chunks = k0 / LU_COLS + (std::max(0, nmax - k0 - LU_NB) + LU_COLS - 1) / LU_COLS;
    if (chunks) hipLaunchKernelGGL(k_lu_update, dim3(chunks, nblk), dim3(256), 0, s, k0, nblk, nmax, n, off, A, piv, pivoff);
  }
  if (info) hipLaunchKernelGGL(k_lu_first_zero, dim3(nblk), dim3(64), 0, s, nblk, nmax, n, off, A, info);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

// The split form (two launches per panel) with its per-block status words st[2 nblk] in device
// memory the caller provides; queued on s, not synchronised.
static hipError_t lu_launch_split(int nblk, int nmax, const int32_t* n, const int64_t* off, double* A, int32_t* ipiv,
                                  const int64_t* pivoff, int32_t* info, int32_t* st, hipStream_t s) {
  for (int k0 = 0; k0 < nmax; k0 += LU_NB) {
    hipLaunchKernelGGL(k_lu_panel<double>, dim3(nblk), dim3(LU_PANEL_THREADS), 0, s, k0, nblk, nmax, n, off, A, ipiv, pivoff, st);
    const int m = nmax - k0 - LU_NB;   // trailing size of the largest block
    if (m > 0) hipLaunchKernelGGL(k_lu_trail<double>, dim3((unsigned)((m + 63) / 64), nblk), dim3(256), 0, s, k0, nblk, nmax, n, off, A, st);
  }
  if (info) hipLaunchKernelGGL(k_lu_info, dim3((nblk + 255) / 256), dim3(256), 0, s, nblk, st, info);
  return hipGetLastError();
}

extern "C" {

// Host-side error text of the block routines (the context-level message lives in bosss_hip.hip).
const char* bosss_hip_block_last_error(void) { return g_lu_err.c_str(); }

int bosss_hip_block_lu_dev(bosss_ctx* ctx, int nblk, int32_t nmax, const int32_t* n, const int64_t* off, double* A,
                           int32_t* ipiv, const int64_t* pivoff, int32_t* info, int32_t want_inverse, void* stream) {
  if (nblk <= 0) return BOSSS_OK;
  if (int rc = lu_check_args(ctx, nmax, n, off, A, ipiv, pivoff)) return rc;
  if (nmax <= LU_MAXN) return lu_launch_reg(nblk, nmax, n, off, A, ipiv, pivoff, info, want_inverse, (hipStream_t)stream);
  if (want_inverse) { g_lu_err = "inverses are limited to blocks of 128 DOF"; return BOSSS_ERR_UNSUPPORTED; }
  hipStream_t s = (hipStream_t)stream;
  // Panels in registers up to LU_REG_MAXN DOF (two rows a thread).  They keep no state but the pivots, so a
  // call without ipiv takes the forms below, as larger blocks do; a grid's y extent bounds the batch.
  if (nmax <= LU_REG_MAXN && ipiv && nblk <= 65535) return lu_launch_panels(nblk, nmax, n, off, A, ipiv, pivoff, info, s);
  if (nmax >= LU_SPLIT_MINN && nblk < LU_SPLIT_MAXBLK) {
    // few large blocks: two launches per panel, the trailing update over many workgroups
    int32_t* st = nullptr;
    hipError_t e = hipMalloc((void**)&st, 2 * (size_t)nblk * sizeof(int32_t));
    if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
    e = lu_launch_split(nblk, nmax, n, off, A, ipiv, pivoff, info, st, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);   // st is freed next
    (void)hipFree(st);
    if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
    return BOSSS_OK;
  }
  hipLaunchKernelGGL(k_block_lu_blocked<double>, dim3(nblk), dim3(256), 0, s, nblk, nmax, n, off, A, ipiv, pivoff, info);
  hipError_t eb = hipGetLastError();
  if (eb != hipSuccess) { g_lu_err = hipGetErrorString(eb); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

int bosss_hip_block_lu_noalloc_dev(bosss_ctx* ctx, int nblk, int32_t nmax, const int32_t* n, const int64_t* off, double* A,
                                   int32_t* ipiv, const int64_t* pivoff, int32_t* info, int32_t want_inverse, void* stream) {
  if (nblk <= 0) return BOSSS_OK;
  if (int rc = lu_check_args(ctx, nmax, n, off, A, ipiv, pivoff)) return rc;
  if (nmax <= LU_MAXN) return lu_launch_reg(nblk, nmax, n, off, A, ipiv, pivoff, info, want_inverse, (hipStream_t)stream);
  if (want_inverse) { g_lu_err = "inverses are limited to blocks of 128 DOF"; return BOSSS_ERR_UNSUPPORTED; }
  if (nblk > LU_NOALLOC_MAXBLK) {
    g_lu_err = "bosss_hip_block_lu_noalloc_dev: " + std::to_string(nblk) + " blocks above " + std::to_string(LU_MAXN) +
               " DOF exceed its scratch (at most " + std::to_string(LU_NOALLOC_MAXBLK) + " per call)";
    return BOSSS_ERR_ARG;
  }
  if (nmax <= LU_REG_MAXN && ipiv) return lu_launch_panels(nblk, nmax, n, off, A, ipiv, pivoff, info, (hipStream_t)stream);
  int32_t* st = nullptr;
  if (int rc = scratch_on_current_device(&st)) return rc;
  hipError_t e = lu_launch_split(nblk, nmax, n, off, A, ipiv, pivoff, info, st, (hipStream_t)stream);
  if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

int bosss_hip_block_solve_dev(bosss_ctx* ctx, int nblk, const int32_t* n, const int64_t* off, const double* LU, const int32_t* ipiv,
                              const int64_t* pivoff, const int64_t* xoff, double* x, void* stream) {
  if (nblk <= 0) return BOSSS_OK;
  if (int rc = select_device(ctx)) return rc;
  if (!n || !off || !LU || !ipiv || !pivoff || !xoff || !x) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  hipLaunchKernelGGL(k_block_solve, dim3(nblk), dim3(64), 0, (hipStream_t)stream, nblk, n, off, LU, ipiv, pivoff, xoff, x);
  hipLaunchKernelGGL(k_block_solve_wide, dim3(nblk), dim3(64 * SOLVE_WAVES), 0, (hipStream_t)stream, nblk, n, off, LU, ipiv, pivoff, xoff, x);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

int bosss_hip_block_gemv_dev(bosss_ctx* ctx, int nblk, const int32_t* n, const int64_t* off, const double* Ainv, const int64_t* xoff,
                             double alpha, const double* x, double beta, double* y, void* stream) {
  if (nblk <= 0) return BOSSS_OK;
  if (int rc = select_device(ctx)) return rc;
  if (!n || !off || !Ainv || !xoff || !x || !y) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  hipLaunchKernelGGL(k_block_gemv<double>, dim3(nblk), dim3(64), 0, (hipStream_t)stream, nblk, n, off, Ainv, xoff, alpha, x, beta, y);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { g_lu_err = hipGetErrorString(e); return BOSSS_ERR_HIP; }
  return BOSSS_OK;
}

// ---- host-pointer forms: the arrays are host memory, copied to the device and back on the
//      context's stream; the call returns with the results in the host arrays.
static int host_batch_check(bosss_ctx* ctx, int nblk, const int32_t* n, const int64_t* off, hipStream_t* s) {
  if (!ctx) { g_lu_err = "ctx is NULL (host-pointer calls copy on the context's stream)"; return BOSSS_ERR_ARG; }
  int dev = 0;
  if (bosss::ctx_device_stream(ctx, &dev, s) != BOSSS_OK) { g_lu_err = "bad context"; return BOSSS_ERR_ARG; }
  if (int rc = select_device(ctx)) return rc;
  if (!n || !off) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  for (int b = 0; b < nblk; b++)
    if (n[b] < 0 || off[b] < 0) { g_lu_err = "negative block size or offset"; return BOSSS_ERR_ARG; }
  return BOSSS_OK;
}
static int host_fail(hipError_t e, const char* what) {
  g_lu_err = std::string(what) + ": " + hipGetErrorString(e);
  return BOSSS_ERR_HIP;
}

int bosss_hip_block_lu(bosss_ctx* ctx, int nblk, int32_t nmax, const int32_t* n, const int64_t* off, double* A, int32_t* ipiv,
                       const int64_t* pivoff, int32_t* info, int32_t want_inverse) {
  if (nblk <= 0) return BOSSS_OK;
  hipStream_t s = nullptr;
  if (int rc = host_batch_check(ctx, nblk, n, off, &s)) return rc;
  if (!A || (ipiv && !pivoff)) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  const int64_t na = batch_extent(nblk, off, [&](int b) { return (int64_t)n[b] * n[b]; });
  const int64_t np = ipiv ? batch_extent(nblk, pivoff, [&](int b) { return (int64_t)n[b]; }) : 0;
  DevArrays d(s);
  const int32_t* dn = d.in(n, nblk);
  const int64_t* doff = d.in(off, nblk);
  double* dA = d.in((const double*)A, na);
  int32_t* dpiv = ipiv ? d.in((const int32_t*)ipiv, np) : nullptr;
  const int64_t* dpo = ipiv ? d.in(pivoff, nblk) : nullptr;
  int32_t* dinfo = info ? d.out<int32_t>(nblk) : nullptr;
  if (d.error() != hipSuccess) return host_fail(d.error(), "block_lu staging");
  if (int rc = bosss_hip_block_lu_dev(ctx, nblk, nmax, dn, doff, dA, dpiv, dpo, dinfo, want_inverse, s)) return rc;
  d.back(A, (const double*)dA, na);
  if (ipiv) d.back(ipiv, (const int32_t*)dpiv, np);
  if (info) d.back(info, (const int32_t*)dinfo, nblk);
  if (hipError_t e = d.finish()) return host_fail(e, "block_lu");
  return BOSSS_OK;
}

int bosss_hip_block_solve(bosss_ctx* ctx, int nblk, const int32_t* n, const int64_t* off, const double* LU, const int32_t* ipiv,
                          const int64_t* pivoff, const int64_t* xoff, double* x) {
  if (nblk <= 0) return BOSSS_OK;
  hipStream_t s = nullptr;
  if (int rc = host_batch_check(ctx, nblk, n, off, &s)) return rc;
  if (!LU || !ipiv || !pivoff || !xoff || !x) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  const int64_t na = batch_extent(nblk, off, [&](int b) { return (int64_t)n[b] * n[b]; });
  const int64_t np = batch_extent(nblk, pivoff, [&](int b) { return (int64_t)n[b]; });
  const int64_t nx = batch_extent(nblk, xoff, [&](int b) { return (int64_t)n[b]; });
  DevArrays d(s);
  const int32_t* dn = d.in(n, nblk);
  const int64_t* doff = d.in(off, nblk);
  const double* dLU = d.in(LU, na);
  const int32_t* dpiv = d.in(ipiv, np);
  const int64_t* dpo = d.in(pivoff, nblk);
  const int64_t* dxo = d.in(xoff, nblk);
  double* dx = d.in((const double*)x, nx);
  if (d.error() != hipSuccess) return host_fail(d.error(), "block_solve staging");
  if (int rc = bosss_hip_block_solve_dev(ctx, nblk, dn, doff, dLU, dpiv, dpo, dxo, dx, s)) return rc;
  d.back(x, (const double*)dx, nx);
  if (hipError_t e = d.finish()) return host_fail(e, "block_solve");
  return BOSSS_OK;
}

int bosss_hip_block_gemv(bosss_ctx* ctx, int nblk, const int32_t* n, const int64_t* off, const double* Ainv, const int64_t* xoff,
                         double alpha, const double* x, double beta, double* y) {
  if (nblk <= 0) return BOSSS_OK;
  hipStream_t s = nullptr;
  if (int rc = host_batch_check(ctx, nblk, n, off, &s)) return rc;
  if (!Ainv || !xoff || !x || !y) { g_lu_err = "NULL argument"; return BOSSS_ERR_ARG; }
  const int64_t na = batch_extent(nblk, off, [&](int b) { return (int64_t)n[b] * n[b]; });
  const int64_t nx = batch_extent(nblk, xoff, [&](int b) { return (int64_t)n[b]; });
  DevArrays d(s);
  const int32_t* dn = d.in(n, nblk);
  const int64_t* doff = d.in(off, nblk);
  const double* dAi = d.in(Ainv, na);
  const int64_t* dxo = d.in(xoff, nblk);
  const double* dx = d.in(x, nx);
  double* dy = d.in((const double*)y, nx);
  if (d.error() != hipSuccess) return host_fail(d.error(), "block_gemv staging");
  if (int rc = bosss_hip_block_gemv_dev(ctx, nblk, dn, doff, dAi, dxo, alpha, dx, beta, dy, s)) return rc;
  d.back(y, (const double*)dy, nx);
  if (hipError_t e = d.finish()) return host_fail(e, "block_gemv");
  return BOSSS_OK;
}

}  // extern "C"
