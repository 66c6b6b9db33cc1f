// Operator kernels of the linear, constant-coefficient scalar forms (SIP, upwind + SIP) on
// axis-aligned cells, in modal space.
//
// The integrands of these forms are products of two polynomials of the basis, the Gauss rule with
// p + 1 points per direction integrates them exactly, and the basis is the tensor product of
// normalised Legendre polynomials truncated at total degree p.  So no quadrature node is needed:
//   * the reference derivative d/dxi_d maps coefficients to coefficients with the 1D matrix
//     D[a'][a] = int L'_a' L_a = sqrt((2a+1)(2a'+1)) for a < a', a' - a odd (11 entries per
//     direction for the 20 modes of p = 3), and its transpose is the test with d/dxi_d;
//   * the trace on the face xi_d = s (s = +-1) has the face-mode coefficients sum_a s^a l_a u_abc,
//     l_a = L_a(1) = sqrt(a + 1/2), its outward derivative sum_a s^a m_a u_abc times invJ_d, with
//     m_a = L'_a(1) = l_a a (a+1) / 2; the face modes are orthonormal, so the numerical flux acts on
//     these coefficients one by one, and the test with a trace or an outward derivative is the
//     transpose of the same sums.
// The adjoint is the transposed chain with the face terms of both rows collected.
//
// One thread owns one cell: coefficients, result and face traces in registers, all tables literals.
// A wavefront's 64 cells are consecutive, so its loads sweep whole cache lines.
//
// Bound: HBM and L2 traffic (own and 2D neighbour coefficients, one store), where the nodal kernels
// of dg_tensor.hpp are bound by their dense contractions.  Upwind + SIP p = 3 residual at 64^3, FP64:
// a call takes 522 us with the nodal kernel, 51 us here (the kernel 47; 84 MB of coefficients in and out, 31 MB of
// metrics); FP32 adjoint at 45 x 37 x 29: 65 -> 11 us.  Measured and not kept: all faces
// unrolled (448 registers, 60 us), neighbour coefficients gathered through an LDS tile (67 us: the
// lane exchange of the cell indices costs more than the scattered lines), results stored without
// the tile (55 us), three wavefronts per SIMD (100 us, spills).
#pragma once
#include <hip/hip_runtime.h>

#include "dg_tensor.hpp"

namespace bosss {

constexpr double ct_sqrt(double x) {
  double r = x > 1.0 ? x : 1.0;
  for (int i = 0; i < 64; i++) r = 0.5 * (r + x / r);
  return r;
}

// Modes of total degree <= P (by degree, then lexicographic exponents), and for each direction the
// face mode a mode's other exponents belong to.
template <int D_, int P_>
struct Modal {
  static constexpr int D = D_, P = P_, N = tdeg_count(D, P), NT = D == 3 ? (P + 1) * (P + 2) / 2 : P + 1;
  struct Table {
    int e[N][3];      // exponents
    int t[3][N];      // face mode of mode n on the faces of direction d
    int lower[3][N][2];   // modes with exponent e_d - 1 and e_d - 3, or -1
    double l[P + 1], m[P + 1], d[P + 1][2];   // L_a(1), L'_a(1), D[a][a-1], D[a][a-3]
    constexpr Table() : e(), t(), lower(), l(), m(), d() {
      int n = 0;
      for (int deg = 0; deg <= P; deg++)
        for (int a = 0; a <= deg; a++)
          for (int b = 0; b <= deg - a; b++) {
            const int c = deg - a - b;
            if (D == 2 && c != 0) continue;
            e[n][0] = a; e[n][1] = b; e[n][2] = c;
            n++;
          }
      for (int k = 0; k < D; k++)
        for (int i = 0; i < N; i++) {
          const int u = e[i][k == 0 ? 1 : 0], v = D == 3 ? e[i][k == 2 ? 1 : 2] : 0;
          t[k][i] = D == 3 ? (u + v) * (u + v + 1) / 2 + v : u;
          for (int q = 0; q < 2; q++) {
            lower[k][i][q] = -1;
            for (int j = 0; j < N; j++) {
              bool same = e[j][k] == e[i][k] - 1 - 2 * q;
              for (int o = 0; o < 3; o++) if (o != k && e[j][o] != e[i][o]) same = false;
              if (same) lower[k][i][q] = j;
            }
          }
        }
      for (int a = 0; a <= P; a++) {
        l[a] = ct_sqrt(a + 0.5);
        m[a] = l[a] * (a * (a + 1) / 2);
        d[a][0] = a >= 1 ? ct_sqrt((2.0 * a + 1) * (2.0 * a - 1)) : 0.0;
        d[a][1] = a >= 3 ? ct_sqrt((2.0 * a + 1) * (2.0 * a - 5)) : 0.0;
      }
    }
  };
  static constexpr Table T = Table();
  static_assert(P <= 4, "D[a'][a] is listed for a' - a = 1 and 3");
};

// Axis-aligned geometry in cell-fastest arrays (made at grid upload).
struct AxisGrid {
  const double* iJ;     // [D][J]   diagonal of the inverse Jacobian
  const double* sqrtg;  // [NF][J]
  const int* nb;        // [NF][J]
};

template <typename Real>
struct MArgs {
  int J, nxcd;
  const double *detJ, *scaling, *lenscale;
  AxisGrid g;
  FormParams fp;
  double alpha, beta;
  const Real *U, *X;
  Real *R, *out;
};

// Direction and side of local face f (Cube / Square.Faces: -x, +x, +y, -y, +z, -z).
__host__ __device__ constexpr int face_dir(int f) { return f / 2; }
__host__ __device__ constexpr bool face_upper(int f) { return f == 1 || f == 2 || f == 4; }

// Coefficients of one cell, consecutive in memory: each lane's loads walk its own lines.
template <int N, typename Real>
__device__ __forceinline__ void load_cell(const Real* __restrict__ x, int cell, Real (&u)[N]) {
  const Real* q = x + (size_t)cell * N;
#pragma unroll
  for (int n = 0; n < N; n++) u[n] = q[n];
}

// Results of the wavefront's cells through an LDS tile (row c: cell of lane c, LD = N | 1 apart, so
// the column writes are free of bank conflicts) to whole-line stores.
template <int N, typename Real>
struct CellTile {
  static constexpr int LD = N | 1;
  Real* t;
  int lane;
  __device__ __forceinline__ CellTile(Real* tile) : t(tile), lane(threadIdx.x) {}
  // o[first + c][k] <- al * r + be * old for the cells c < count (be = 0: the old value is not read)
  __device__ __forceinline__ void store(Real* __restrict__ o, int first, int count, const Real (&r)[N], Real al, Real be) const {
#pragma unroll
    for (int n = 0; n < N; n++) t[lane * LD + n] = al * r[n];
    __builtin_amdgcn_wave_barrier();
    Real* p = o + (size_t)first * N;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int e = 64 * i + lane, c = e / N, k = e - c * N;
      if (c < count) {
        const Real v = t[c * LD + k];
        p[e] = be != Real(0) ? be * p[e] + v : v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
};

// r <- A x (ADJ: A^T x) of cell j.
template <int D, int P, typename Real, bool ADV, bool ADJ>
__device__ __forceinline__ void modal_apply(const MArgs<Real>& a, int j, const Real* __restrict__ x, Real (&r)[Modal<D, P>::N]) {
  typedef Modal<D, P> M;
  constexpr int N = M::N, NT = M::NT;
  const int J = a.J;
  const Real sc = Real(a.scaling[j]), detJ = Real(a.detJ[j]), nu = Real(a.fp.nu);
  const Real pbd = Real(a.fp.penalty_base * a.fp.penalty_deg), cown = Real(1.0 / a.lenscale[j]);
  Real u[N];
  load_cell<N>(x, j, u);
#pragma unroll
  for (int n = 0; n < N; n++) { u[n] *= sc; r[n] = Real(0); }

  // volume: with q = D_d u,  forward  D_d^T (-vel u - nu iJ q) iJ,  adjoint  iJ (-vel q - nu iJ D_d^T q)
#pragma unroll
  for (int k = 0; k < D; k++) {
    const Real iJ = Real(a.g.iJ[(size_t)k * J + j]);
    const Real w = detJ * iJ, cd = -nu * iJ * w, cv = ADV ? Real(-a.fp.vel[k]) * w : Real(0);
    Real q[N];
#pragma unroll
    for (int n = 0; n < N; n++) q[n] = Real(0);
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (M::T.lower[k][n][h] >= 0) q[M::T.lower[k][n][h]] += Real(M::T.d[M::T.e[n][k]][h]) * u[n];
    if (ADV && ADJ) {
#pragma unroll
      for (int n = 0; n < N; n++) r[n] += cv * q[n];
    }
#pragma unroll
    for (int n = 0; n < N; n++) q[n] = cd * q[n] + ((ADV && !ADJ) ? cv * u[n] : Real(0));
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (M::T.lower[k][n][h] >= 0) r[n] += Real(M::T.d[M::T.e[n][k]][h]) * q[M::T.lower[k][n][h]];
  }

  // Faces, both sides of a direction in one loop body (the side is a sign on the odd exponents): the
  // traces of both sides are accumulated into their jump and the sum of their outward derivatives,
  // the flux acts on the face modes, the transposed traces add it to r.  The loop is not unrolled and
  // the directions are kept apart: hoisting the loads of all faces costs more registers than there are.
  const Real half = Real(0.5) * nu;
#pragma unroll
  for (int k = 0; k < D; k++) {
    const Real iJ = Real(a.g.iJ[(size_t)k * J + j]);
#pragma unroll 1
    for (int side = 0; side < 2; side++) {
      asm volatile("" ::: "memory");
      const int f = 2 * k + side;
      const Real s = (k == 0) == (side == 1) ? Real(1) : Real(-1);   // outward direction: +1 upper, -1 lower
      const int nbr = a.g.nb[(size_t)f * J + j];
      const bool has = nbr >= 0;
      const int cn = has ? nbr : j;
      Real p[N];
      load_cell<N>(x, cn, p);
      const Real sg = Real(a.g.sqrtg[(size_t)f * J + j]);
      const Real scn = has ? Real(a.scaling[cn]) : Real(0), iJn = Real(a.g.iJ[(size_t)k * J + cn]);
      Real mu = pbd * cown;
      if (has) { const Real mo = pbd * Real(1.0 / a.lenscale[cn]); mu = mo > mu ? mo : mu; }
      Real v[NT], jump[NT], g[NT];   // own trace, own - neighbour trace, own + neighbour outward derivative
#pragma unroll
      for (int t = 0; t < NT; t++) { v[t] = Real(0); jump[t] = Real(0); g[t] = Real(0); }
      const Real gs = iJn * scn;
#pragma unroll
      for (int n = 0; n < N; n++) {
        const int t = M::T.t[k][n], e = M::T.e[n][k];
        const Real l = (e & 1) ? s * Real(M::T.l[e]) : Real(M::T.l[e]), m = (e & 1) ? s * Real(M::T.m[e]) : Real(M::T.m[e]);
        v[t] += l * u[n];
        if (e > 0) g[t] += (iJ * m) * u[n];
        // the neighbour's face is its other side: odd exponents change sign; its outward derivative
        // seen along the own normal is the negative one
        if (e & 1) { jump[t] += (l * scn) * p[n]; g[t] += (m * gs) * p[n]; }
        else { jump[t] -= (l * scn) * p[n]; if (e > 0) g[t] -= (m * gs) * p[n]; }
      }
      const Real vel = ADV ? s * Real(a.fp.vel[k]) : Real(0);   // velocity . n
      const Real cp = (has ? mu : Real(2) * mu) * nu, cg = has ? half : nu;
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const Real un = -jump[t];        // neighbour trace (0 on the boundary)
        jump[t] += v[t];
        Real fv = cg * g[t] - cp * jump[t];   // coefficient of the test trace
        if (ADV) {
          if (ADJ) fv += (vel > Real(0) || (!has && vel == Real(0))) ? vel * jump[t] : Real(0);
          else if (has) fv += vel > Real(0) ? vel * v[t] : vel * un;
          else fv += vel >= Real(0) ? vel * v[t] : Real(0);
        }
        v[t] = sg * fv;
        g[t] = (sg * iJ * cg) * jump[t];      // coefficient of the test's outward derivative
      }
#pragma unroll
      for (int n = 0; n < N; n++) {
        const int t = M::T.t[k][n], e = M::T.e[n][k];
        const Real l = (e & 1) ? s * Real(M::T.l[e]) : Real(M::T.l[e]), m = (e & 1) ? s * Real(M::T.m[e]) : Real(M::T.m[e]);
        r[n] += l * v[t];
        if (e > 0) r[n] += m * g[t];
      }
    }
  }
#pragma unroll
  for (int n = 0; n < N; n++) r[n] *= sc;
}

// FWD: R <- beta R + alpha A U (or, with JVP, out <- A X); ADJ: out <- A^T X.
template <int D, int P, typename Real, bool ADV, bool FWD, bool JVP, bool ADJ>
__global__ void __launch_bounds__(64) k_modal(MArgs<Real> a) {
  constexpr int N = Modal<D, P>::N;
  __shared__ Real smem[64 * CellTile<N, Real>::LD];
  const CellTile<N, Real> tile(smem);
  const int first = xcd_block(a.nxcd, 0) * 64, count = min(64, a.J - first);
  const int j = min(first + (int)threadIdx.x, a.J - 1);   // lanes past the last cell repeat it
  Real r[N];
  if (FWD) {
    modal_apply<D, P, Real, ADV, false>(a, j, JVP ? a.X : a.U, r);
    if (JVP) tile.store(a.out, first, count, r, Real(1), Real(0));
    else tile.store(a.R, first, count, r, Real(a.alpha), Real(a.beta));
  }
  if (ADJ) {
    modal_apply<D, P, Real, ADV, true>(a, j, a.X, r);
    tile.store(a.out, first, count, r, Real(1), Real(0));
  }
}

}  // namespace bosss
