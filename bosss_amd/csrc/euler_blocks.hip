// Diagonal blocks of the Euler Jacobian, dR_j/dU_j + shift I per cell, from moments of the pointwise
// flux Jacobians; 3D alone.
//
// With A_e(x) = detJ sc^2 sum_d invJ[e][d] dF_d/dU the 5 x 5 Jacobian at a node, the
// volume part of entry ((v, n), (w, m)) is sum_e sum_k w_k d_e phi_n A_e,vw phi_m.  d_e phi_n is a short
// combination of modes of degree < p, and the product of two modes a short combination of Legendre
// products of degree <= 2 p - 1 (one to four terms), so the entry is a short combination of the moments
// sum_k w_k psi_l A_e,vw.  The same holds on the faces: a trace is s^a l_a times a face mode (s = +-1 the
// side), and the products of face modes have degree <= 2 p.  The Gauss sums are the ones of the
// pointwise form, node by node; only their order changes.
//
// One workgroup per cell: states at the nodes, Jacobians by dual numbers (one thread per node and
// seed), moments as an MFMA product [moments x nodes] [nodes x Jacobian entries], then every thread combines the
// entries (n, m) it owns for all V^2 pairs.  At p = 3 a cell costs about 0.7 M multiply-adds in
// the moments and 0.1 M in the combination.
//
// Bound: latency between its barriers at two workgroups per CU (vector issue about a quarter, matrix
// units a seventh, LDS a third of the time).  20^3 cells, p = 3 (640 MB of blocks): 17.4 ms by probing
// (one Jacobian-vector product over the whole grid per column and two passes over the blocks), 1.18 ms
// here.  Measured and not kept: the moment matrices in registers (1.61 ms, spills).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

#include "dg_tensor.hpp"
#include "euler_blocks.hpp"

namespace bosss {

template <int P_, int K1_>
struct EB {
  static constexpr int D = 3, P = P_, K1 = K1_, K2 = K1 + 2, V = D + 2, N = tdeg_count(D, P), NT = V * N;
  static constexpr int KV = ipow(K1, D), KE = ipow(K1, D - 1);
  static constexpr int LV = tdeg_count(D, 2 * P - 1), LF = tdeg_count(2, 2 * P);   // moments per pair
  static constexpr int KSV = (KV + 3) / 4, KSF = (KE + 3) / 4;      // MFMA k-steps
  static constexpr int RV = (LV + 15) / 16, RF = (LF + 15) / 16;    // 16-row tiles
  static constexpr int VV = V * V, CT = (VV + 15) / 16;             // Jacobian entries, 16-column tiles
  // tile of a wavefront: row tile w with all column tiles, or one (row, column) tile per wavefront
  static constexpr bool WIDE = RV * CT > 4;
  static_assert(RV <= 4 && (WIDE || RV * CT <= 4) && RF * CT <= 4, "at most four wavefronts share the moment tiles");
  static constexpr int WI = (N * N + 63) / 64;                       // wavefront-sized groups of entries
  static_assert(WI <= 8, "two groups per wavefront");
  // strides: a node row of Jacobian entries (volume; faces, both sides), 2 mod 32 so the 16 columns x 2
  // nodes a half wavefront reads as an MFMA operand lie in different banks; a moment row
  static constexpr int GS = (4 * KSV + 29) / 32 * 32 + 2, GF = (8 * KSF + 29) / 32 * 32 + 2, MS = (VV + 1) & ~1;
  static constexpr int NG = VV * (GS > GF ? GS : GF) > N * NT ? VV * (GS > GF ? GS : GF) : N * NT;   // also the store staging
  static constexpr int NM = (LV > 2 * LF ? LV : 2 * LF) * MS;
  static constexpr int NS = V * KV > 4 * V * KE ? V * KV : 4 * V * KE;
  // uploaded doubles
  static constexpr int O_L = 0, O_AV = (P + 1) * K2, O_AF = O_AV + RV * KSV * 64, O_C = O_AF + RF * KSF * 64;
  // uploaded ints
  static constexpr int I_OFF = 0, I_ORD = 2 * D * WI + 1, I_IDX = I_ORD + 64 * WI;
  static constexpr int LDS = (P + 1) * K2 + 3 * NT + NS + NG + 1 + NM;   // doubles
};

// Nested 1D sums of one variable at the node with 1D indices q (L: [P+1][K2]).
template <class E>
__device__ __forceinline__ double node_value(const double* L, const double* u, const int (&q)[3]) {
  constexpr int P = E::P;
  double s[P + 1];
#pragma unroll
  for (int a = 0; a <= P; a++) s[a] = 0.0;
  // modes by degree, then lexicographic: mode n has exponents (a, b, c)
  int n = 0;
#pragma unroll
  for (int deg = 0; deg <= P; deg++)
#pragma unroll
    for (int a = 0; a <= deg; a++) {
      double t = 0.0;
#pragma unroll
      for (int b = 0; b <= deg - a; b++) {
        t += u[n] * (L[b * E::K2 + q[1]] * L[(deg - a - b) * E::K2 + q[2]]);
        n++;
      }
      s[a] += t;
    }
  double r = 0.0;
#pragma unroll
  for (int a = 0; a <= P; a++) r += s[a] * L[a * E::K2 + q[0]];
  return r;
}

// acc[slot][pair] += coef * moment over the term lists of one phase.
template <class E>
__device__ __forceinline__ void add_terms(const EulerBlockArgs& a, int phase, int w, int lane, const double* M, double (&acc)[2][E::VV]) {
#pragma unroll
  for (int slot = 0; slot < 2; slot++) {
    const int wi = slot == 0 ? w : 7 - w;   // groups are sorted by length: a long one and a short one
    if (wi >= E::WI) continue;
    const int t0 = a.ints[E::I_OFF + phase * E::WI + wi], t1 = a.ints[E::I_OFF + phase * E::WI + wi + 1];
    const double* pc = a.real + E::O_C + lane;
    const int32_t* pi = a.ints + E::I_IDX + lane;
    double c = t0 < t1 ? pc[t0 * 64] : 0.0;
    int ix = t0 < t1 ? pi[t0 * 64] : 0;
    for (int t = t0; t < t1; t++) {      // the next term is loaded while this one's moments are read
      const int tn = t + 1 < t1 ? t + 1 : t;
      const double cn = pc[tn * 64];
      const int in = pi[tn * 64];
      const double* m = M + ix;
#pragma unroll
      for (int v = 0; v < E::VV; v++) acc[slot][v] += c * m[v];
      c = cn;
      ix = in;
    }
  }
}

template <class Form, int P, int K1, typename Real>
__global__ void __launch_bounds__(256, 2) k_euler_blocks(EulerBlockArgs a) {
  typedef EB<P, K1> E;
  typedef Dual<1, double> T;
  constexpr int D = E::D, V = E::V, N = E::N, NT = E::NT, VV = E::VV, KV = E::KV, KE = E::KE, CTW = E::WIDE ? E::CT : 1;
  extern __shared__ __align__(16) double smem[];
  double* L = smem;
  double* uo = L + (P + 1) * E::K2;      // own coefficients, then both neighbours of a direction
  double* st = uo + 3 * NT;              // states at nodes
  double* G = st + E::NS;
  if ((G - smem) & 1) G++;
  double* M = G + E::NG + (E::NG & 1);
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < (P + 1) * E::K2; i += 256) L[i] = a.real[E::O_L + i];

  const int rtv = E::WIDE ? w : w / E::CT, ctv = E::WIDE ? 0 : w % E::CT;
  const int rtf = w / E::CT, ctf = w % E::CT;
  const bool hasv = rtv < E::RV, hasf = rtf < E::RF;
  // left operands of this wavefront's row tiles (L2: holding them costs the registers of the Jacobians)
  const double* av = a.real + E::O_AV + (size_t)(hasv ? rtv : 0) * E::KSV * 64 + lane;
  const double* af = a.real + E::O_AF + (size_t)(hasf ? rtf : 0) * E::KSF * 64 + lane;

  const Real* U = static_cast<const Real*>(a.U);
  for (int j = blockIdx.x; j < a.J; j += gridDim.x) {
    const double sc = a.scaling[j];
    double iJ[D][D];
#pragma unroll
    for (int e = 0; e < D; e++)
#pragma unroll
      for (int d = 0; d < D; d++) iJ[e][d] = a.invJ[((size_t)j * D + e) * D + d];
    double acc[2][VV];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int v = 0; v < VV; v++) acc[s][v] = 0.0;
    __syncthreads();                     // the previous cell's staging and coefficients are read
    for (int i = tid; i < NT; i += 256) uo[i] = sc * (double)U[(size_t)j * NT + i];
    __syncthreads();
    for (int i = tid; i < V * KV; i += 256) {
      const int v = i / KV, k = i - v * KV;
      int q[3];
      vol_axes<D, K1>(k, q);
      st[v * KV + k] = node_value<E>(L, uo + v * N, q);
    }
    // ---------------------------------------------------------------- volume, one reference direction at a time
    const double wv = a.detJ[j] * sc * sc;
#pragma unroll 1
    for (int e = 0; e < D; e++) {
      double ie[D];
#pragma unroll
      for (int d = 0; d < D; d++) ie[d] = wv * a.invJ[((size_t)j * D + e) * D + d];
      __syncthreads();
      for (int i = tid; i < V * 4 * E::KSV; i += 256) {
        const int k = i % (4 * E::KSV), c = i / (4 * E::KSV);   // node, seed variable
        T Uq[V], GU[V][D], F[V][D];
#pragma unroll
        for (int v = 0; v < V; v++) {
          Uq[v] = dconst<1, double>(st[v * KV + (k < KV ? k : 0)]);
          Uq[v].d[0] = v == c ? 1.0 : 0.0;
#pragma unroll
          for (int d = 0; d < D; d++) GU[v][d] = Uq[v];
        }
        Form::template volume<D, T, double>(a.fp, Uq, GU, F);
#pragma unroll
        for (int v = 0; v < V; v++) {
          double s = 0.0;
#pragma unroll
          for (int d = 0; d < D; d++) s += ie[d] * F[v][d].d[0];
          G[(v * V + c) * E::GS + k] = k < KV ? s : 0.0;
        }
      }
      __syncthreads();
      if (hasv) {
        const double* g[CTW];
        f64x4 m[CTW];
#pragma unroll
        for (int ct = 0; ct < CTW; ct++) {
          const int pr = (ctv + ct) * 16 + col;
          g[ct] = G + (pr < VV ? pr : 0) * E::GS + grp;
          m[ct] = acc_zero<double>();
        }
#pragma unroll 8
        for (int k = 0; k < E::KSV; k++) {
          const double x = av[64 * k];
#pragma unroll
          for (int ct = 0; ct < CTW; ct++) m[ct] = MM<double>::mma(x, g[ct][4 * k], m[ct]);
        }
#pragma unroll
        for (int ct = 0; ct < CTW; ct++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int l = rtv * 16 + MM<double>::row(grp, r), pr = (ctv + ct) * 16 + col;
            if (l < E::LV && pr < VV) M[l * E::MS + pr] = m[ct][r];
          }
      }
      __syncthreads();
      add_terms<E>(a, e, w, lane, M, acc);
    }
    // ---------------------------------------------------------------- faces, both sides of a direction together
#pragma unroll 1
    for (int d = 0; d < D; d++) {
      const int fs[2] = {d == 0 ? 0 : 2 * d + 1, d == 0 ? 1 : 2 * d};   // lower and upper face of the direction
      __syncthreads();
      for (int i = tid; i < 2 * NT; i += 256) {
        const int side = i / NT, k = i - side * NT;
        const int nb = a.cf.nb[(size_t)j * (2 * D) + fs[side]];
        const int cn = nb >= 0 ? nb : j;
        uo[NT + i] = a.scaling[cn] * (double)U[(size_t)cn * NT + k];
      }
      __syncthreads();
      for (int i = tid; i < 4 * V * KE; i += 256) {
        const int k = i % KE, v = (i / KE) % V, h = i / (KE * V);   // h: 2 side + (0 own, 1 neighbour)
        const int f = fs[h >> 1];
        int q[3];
        face_axes<D, K1>((h & 1) ? a.cf.pair[f] : f, k, q);
        st[i] = node_value<E>(L, uo + ((h & 1) ? 1 + (h >> 1) : 0) * NT + v * N, q);
      }
      __syncthreads();
      for (int i = tid; i < 2 * V * 4 * E::KSF; i += 256) {
        const int k = i % (4 * E::KSF), c = (i / (4 * E::KSF)) % V, side = i / (4 * E::KSF * V);
        const int f = fs[side], kn = k < KE ? k : 0;
        const double sg = a.cf.sqrtg[(size_t)j * (2 * D) + f] * sc * sc;
        double nrm[D];
#pragma unroll
        for (int x = 0; x < D; x++) nrm[x] = a.cf.normal[((size_t)j * (2 * D) + f) * D + x];
        T Uo[V], Un[V], Go[V][D], fo[V], go[V][D], fn[V], gn[V][D];
#pragma unroll
        for (int v = 0; v < V; v++) {
          Uo[v] = dconst<1, double>(st[((2 * side) * V + v) * KE + kn]);
          Uo[v].d[0] = v == c ? 1.0 : 0.0;
          Un[v] = dconst<1, double>(st[((2 * side + 1) * V + v) * KE + kn]);
#pragma unroll
          for (int x = 0; x < D; x++) Go[v][x] = Uo[v];
        }
        Form::template inner<D, T, double>(a.fp, nrm, 0.0, Uo, Un, Go, Go, fo, go, fn, gn);
#pragma unroll
        for (int v = 0; v < V; v++) G[(v * V + c) * E::GF + side * 4 * E::KSF + k] = k < KE ? sg * fo[v].d[0] : 0.0;
      }
      __syncthreads();
      if (hasf) {
        const int pr = ctf * 16 + col;
        const double* g = G + (pr < VV ? pr : 0) * E::GF + grp;
        f64x4 lo = acc_zero<double>(), up = acc_zero<double>();
#pragma unroll
        for (int k = 0; k < E::KSF; k++) {
          const double x = af[64 * k];
          lo = MM<double>::mma(x, g[4 * k], lo);
          up = MM<double>::mma(x, g[4 * (E::KSF + k)], up);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int l = rtf * 16 + MM<double>::row(grp, r);
          if (l < E::LF && pr < VV) {
            M[l * E::MS + pr] = up[r] + lo[r];                 // even total exponent along the direction
            M[(E::LF + l) * E::MS + pr] = up[r] - lo[r];       // odd
          }
        }
      }
      __syncthreads();
      add_terms<E>(a, D + d, w, lane, M, acc);
    }
    // ---------------------------------------------------------------- store, one variable's rows at a time
    double* out = a.blocks + (size_t)j * NT * NT;
#pragma unroll
    for (int o = 0; o < V; o++) {
      __syncthreads();
#pragma unroll
      for (int slot = 0; slot < 2; slot++) {
        const int wi = slot == 0 ? w : 7 - w;
        if (wi >= E::WI) continue;
        const int nm = a.ints[E::I_ORD + wi * 64 + lane];      // entry (n, m), -1: none
        if (nm < 0) continue;
        const int n = nm / N, m = nm - n * N;
#pragma unroll
        for (int v = 0; v < V; v++) {
          if (a.transposed) G[m * NT + v * N + n] = acc[slot][v * V + o];
          else G[n * NT + v * N + m] = acc[slot][o * V + v];
        }
      }
      __syncthreads();
      for (int i = tid; i < N * NT; i += 256) {
        const int r = i / NT, q = i - r * NT;
        out[(size_t)o * N * NT + i] = a.alpha * G[i] + (q == o * N + r ? a.shift : 0.0);
      }
    }
  }
}

// ---------------------------------------------------------------- host tables, in extended precision, rounded once
// (a rounding error of a coefficient is the same in every cell: with tables in double the p = 2 blocks
// were 5 % further from 64-bit exact, now they are 6 % nearer than by probing).  The normalisation sqrt(a + 1/2) of the basis is the rounded
// one of the other kernels' tables, so that these blocks are the derivative of their residual.
typedef long double ext;
static ext rounded_norm(int a) { return (ext)std::sqrt(a + 0.5); }
static ext norm_ratio(const std::vector<int>& e, int D) {   // of a mode: rounded over exact normalisation
  ext r = 1.0L;
  for (int d = 0; d < D; d++) r *= rounded_norm(e[d]) / std::sqrt(e[d] + 0.5L);
  return r;
}
// Product of normalised Legendre polynomials: L_a L_b = sum_c T[a][b][c] L_c (Adams' formula).
static ext legendre_product(int a, int b, int c) {
  if (c > a + b || c < std::abs(a - b) || ((a + b + c) & 1)) return 0.0L;
  auto A = [](int r) { ext v = 1.0L; for (int i = 1; i <= r; i++) v *= (2.0L * i - 1.0L) / i; return v; };
  const int r = (a + b - c) / 2;
  const ext t = A(r) * A(a - r) * A(b - r) / A(a + b - r) * (2.0L * c + 1.0L) / (2.0L * (a + b - r) + 1.0L);
  return t * std::sqrt((2.0L * a + 1.0L) * (2.0L * b + 1.0L) / (2.0L * (2.0L * c + 1.0L)));
}

static std::vector<std::vector<int>> total_degree(int D, int p) {   // by degree, then lexicographic
  std::vector<std::vector<int>> e;
  for (int deg = 0; deg <= p; deg++)
    for (int a = 0; a <= deg; a++) {
      for (int b = 0; b <= deg - a; b++) {
        if (D == 2 && a + b != deg) continue;
        e.push_back({a, b, D == 3 ? deg - a - b : 0});
      }
    }
  return e;
}

static ext legendre(int n, ext x) {   // normalised
  ext p0 = 1.0L, p1 = x;
  if (n == 0) p1 = 1.0L;
  for (int k = 1; k < n; k++) { const ext p2 = ((2 * k + 1) * x * p1 - k * p0) / (k + 1); p0 = p1; p1 = p2; }
  return std::sqrt(n + 0.5L) * p1;
}

void euler_block_tables(int P, int K1, const std::vector<double>& nodes, EulerBlockTables& t) {
  const int D = 3, K2 = K1 + 2;
  const auto modes = total_degree(D, P), vol = total_degree(D, 2 * P - 1), face = total_degree(D - 1, 2 * P);
  const int N = (int)modes.size(), LV = (int)vol.size(), LF = (int)face.size(), V = D + 2, MS = (V * V + 1) & ~1;
  int KE = 1;
  for (int d = 0; d + 1 < D; d++) KE *= K1;
  const int KV = KE * K1;
  // Gauss rule: Newton steps from the nodes in double
  std::vector<ext> x(nodes.begin(), nodes.end()), w(K1);
  for (int q = 0; q < K1; q++)
    for (int it = 0; it < 3; it++) {
      ext p0 = 1.0L, p1 = x[q];
      for (int k = 1; k < K1; k++) { const ext p2 = ((2 * k + 1) * x[q] * p1 - k * p0) / (k + 1); p0 = p1; p1 = p2; }
      const ext d = K1 * (x[q] * p1 - p0) / (x[q] * x[q] - 1.0L);
      w[q] = 2.0L / ((1.0L - x[q] * x[q]) * d * d);
      x[q] -= p1 / d;
    }
  for (int a = 0; a <= P; a++)
    for (int q = 0; q < K2; q++) t.real.push_back((double)(legendre(a, q < K1 ? x[q] : (q == K1 ? -1.0L : 1.0L)) * (rounded_norm(a) / std::sqrt(a + 0.5L))));
  // moment matrices in MFMA order: [row tile][k-step][lane], lane = row % 16 + 16 (node % 4)
  auto moments = [&](const std::vector<std::vector<int>>& e, int KN, int dim) {
    const int R = ((int)e.size() + 15) / 16, KS = (KN + 3) / 4;
    for (int rt = 0; rt < R; rt++)
      for (int ks = 0; ks < KS; ks++)
        for (int lane = 0; lane < 64; lane++) {
          const int l = rt * 16 + lane % 16;
          int k = ks * 4 + lane / 16;
          ext v = 0.0L;
          if (l < (int)e.size() && k < KN) {
            v = 1.0L;
            for (int d = 0; d < dim; d++) { v *= w[k % K1] * legendre(e[l][d], x[k % K1]); k /= K1; }
          }
          t.real.push_back((double)v);
        }
  };
  moments(vol, KV, D);
  moments(face, KE, D - 1);
  // terms of every entry in every phase: volume directions, then face directions
  typedef std::vector<std::pair<int, ext>> Terms;   // (moment row * MS, coefficient)
  std::vector<std::vector<Terms>> terms(2 * D, std::vector<Terms>(N * N));
  auto add = [&](Terms& ts, int l, ext c) {
    if (c == 0.0L) return;
    for (auto& q : ts)
      if (q.first == l * MS) { q.second += c; return; }
    ts.push_back({l * MS, c});
  };
  for (int n = 0; n < N; n++)
    for (int m = 0; m < N; m++)
      for (int e = 0; e < D; e++) {
        const ext norm = norm_ratio(modes[n], D) * norm_ratio(modes[m], D);
        for (int a = modes[n][e] - 1; a >= 0; a -= 2) {   // d_e phi_n over the modes with exponent a
          const ext de = std::sqrt((2.0L * modes[n][e] + 1.0L) * (2.0L * a + 1.0L));
          for (int l = 0; l < LV; l++) {
            ext c = norm * de;
            for (int d = 0; d < D; d++) c *= legendre_product(d == e ? a : modes[n][d], modes[m][d], vol[l][d]);
            add(terms[e][n * N + m], l, c);
          }
        }
        // face coordinates (s0, s1): the tangential axes in the order the node index runs over them
        const int s0 = e == 0 ? 2 : 0, s1 = e == 2 ? 1 : (e == 0 ? 1 : 2);
        const int odd = (modes[n][e] + modes[m][e]) & 1;
        for (int l = 0; l < LF; l++) {
          ext c = norm * std::sqrt((modes[n][e] + 0.5L) * (modes[m][e] + 0.5L)) * legendre_product(modes[n][s0], modes[m][s0], face[l][0]);
          c *= legendre_product(modes[n][s1], modes[m][s1], face[l][1]);
          add(terms[D + e][n * N + m], odd * LF + l, c);
        }
      }
  // entries by descending number of terms, in groups of 64: a group runs to its longest list
  std::vector<int> order(N * N), total(N * N, 0);
  for (int i = 0; i < N * N; i++) {
    order[i] = i;
    for (int ph = 0; ph < 2 * D; ph++) total[i] += (int)terms[ph][i].size();
  }
  std::stable_sort(order.begin(), order.end(), [&](int p, int q) { return total[p] > total[q]; });
  const int WI = (N * N + 63) / 64;
  order.resize(64 * WI, -1);
  std::vector<int32_t> offs(1, 0), idx;
  std::vector<double> coef;
  for (int ph = 0; ph < 2 * D; ph++)
    for (int wi = 0; wi < WI; wi++) {
      size_t len = 0;
      for (int i = 0; i < 64; i++)
        if (order[wi * 64 + i] >= 0) len = std::max(len, terms[ph][order[wi * 64 + i]].size());
      for (size_t k = 0; k < len; k++)
        for (int i = 0; i < 64; i++) {
          const int en = order[wi * 64 + i];
          const bool in = en >= 0 && k < terms[ph][en].size();
          idx.push_back(in ? terms[ph][en][k].first : 0);
          coef.push_back(in ? (double)terms[ph][en][k].second : 0.0);
        }
      offs.push_back(offs.back() + (int32_t)len);
    }
  t.real.insert(t.real.end(), coef.begin(), coef.end());
  t.ints = offs;
  t.ints.insert(t.ints.end(), order.begin(), order.end());
  t.ints.insert(t.ints.end(), idx.begin(), idx.end());
}

template <class Form, int P, int K1>
static void launch_blocks(bool fp32, int num_cu, const EulerBlockArgs& a, hipStream_t s) {
  typedef EB<P, K1> E;
  const size_t lds = (size_t)(E::LDS + 2) * sizeof(double);
  const dim3 grid((unsigned)std::min(a.J, 2 * num_cu));   // two workgroups per CU (registers), each walking its cells
  if (fp32) hipLaunchKernelGGL((k_euler_blocks<Form, P, K1, float>), grid, dim3(256), lds, s, a);
  else hipLaunchKernelGGL((k_euler_blocks<Form, P, K1, double>), grid, dim3(256), lds, s, a);
}
template <int P, int K1>
static void launch_form(bool hllc, bool fp32, int num_cu, const EulerBlockArgs& a, hipStream_t s) {
  if (hllc) launch_blocks<FormEuler<3, true>, P, K1>(fp32, num_cu, a, s);
  else launch_blocks<FormEuler<3, false>, P, K1>(fp32, num_cu, a, s);
}

bool has_euler_blocks(int D, int P, int K1) { return D == 3 && ((P == 2 && K1 == 4) || (P == 3 && K1 == 5)); }

void launch_euler_blocks(bool hllc, int P, bool fp32, int num_cu, const EulerBlockArgs& a, hipStream_t s) {
  if (P == 2) launch_form<2, 4>(hllc, fp32, num_cu, a, s);
  else launch_form<3, 5>(hllc, fp32, num_cu, a, s);
}

}  // namespace bosss
