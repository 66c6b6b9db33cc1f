// Operator matrix of the linear, constant-coefficient scalar forms (SIP, upwind + SIP) by direct
// combination of reference matrices.
//
// On an affine cell every block of the matrix is a short linear combination
//     block(j, s)[n][m] = sum_t coef_t(j) T_t[n][m]
// of reference matrices T_t that depend on the basis and the quadrature alone:
//   volume   C_e    = sum_k w_k d_e phi_n phi_m          K_ee' = sum_k w_k d_e phi_n d_e' phi_m
//   face f   M  = sum_k w_k psi_n chi_m    G_e = sum_k w_k psi_n d_e chi_m    H_e = sum_k w_k d_e psi_n chi_m
// with psi the trace of the row cell on its face f and chi the trace of the column cell on its side
// of it (chi = psi for the diagonal block).  The coefficients are the derivatives of the pointwise
// form (the same FormX::volume / inner / boundary the residual kernels evaluate, on dual numbers)
// times the cell's metrics.  So the matrix is written once, entry by entry, where the coloured
// probing runs one Jacobian-vector product over the whole grid per colour and mode.
//
// Bound: the store of the matrix.  24^3 cells, p = 3 (310 MB): 12.6 ms by probing (260 probes of
// 49 us), 0.131 ms here (2.4 TB/s).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "dg_kernels.hpp"
#include "forms.hpp"
#include "assemble_linear.hpp"

namespace bosss {

// Coefficients of one cell: LinShape<D>::NC doubles, first those of the diagonal block (volume,
// then the own-own part of every face), then the own-neighbour part of every face.
// One thread per (cell, part): part 0 the volume, 1 + f face f.
template <class Form, int D>
__global__ void __launch_bounds__(256) k_linear_coefs(LinArgs a, double* __restrict__ coef) {
  typedef LinShape<D> LS;
  constexpr int NF = 2 * D;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t j = i / (1 + NF);
  if (j >= a.J) return;
  const int part = (int)(i - j * (1 + NF));
  double* c = coef + j * LS::NC;
  double iJ[D][D];
#pragma unroll
  for (int e = 0; e < D; e++)
#pragma unroll
    for (int d = 0; d < D; d++) iJ[e][d] = a.invJ[j * D * D + e * D + d];
  const double sc = a.scaling[j];
  if (part == 0) {
    typedef Dual<1 + D, double> T;
    T U[1], G[1][D], F[1][D];
    U[0] = dconst<1 + D, double>(0.0);
    U[0].d[0] = 1.0;
#pragma unroll
    for (int d = 0; d < D; d++) { G[0][d] = dconst<1 + D, double>(0.0); G[0][d].d[1 + d] = 1.0; }
    Form::template volume<D, T, double>(a.fp, U, G, F);
    const double w = a.detJ[j] * sc * sc;
#pragma unroll
    for (int e = 0; e < D; e++) {
      double s = 0.0;
#pragma unroll
      for (int d = 0; d < D; d++) s += iJ[e][d] * F[0][d].d[0];
      c[LS::O_C + e] = w * s;
#pragma unroll
      for (int e2 = 0; e2 < D; e2++) {
        double t = 0.0;
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
          for (int d2 = 0; d2 < D; d2++) t += iJ[e][d] * F[0][d].d[1 + d2] * iJ[e2][d2];
        c[LS::O_K + e * D + e2] = w * t;
      }
    }
    return;
  }
  const int f = part - 1;
  const int nb = a.nb[j * NF + f];
  const bool has_nb = nb >= 0;
  const int64_t cn = has_nb ? nb : j;
  double n[D];
#pragma unroll
  for (int d = 0; d < D; d++) n[d] = a.normal[(j * NF + f) * D + d];
  const double pbd = a.fp.penalty_base * a.fp.penalty_deg;
  double mu = pbd * (1.0 / a.lenscale[j]);
  if (has_nb) { const double mo = pbd * (1.0 / a.lenscale[cn]); mu = mo > mu ? mo : mu; }
  constexpr int M = 2 + 2 * D;   // seeds: own value, neighbour value, own gradient, neighbour gradient
  typedef Dual<M, double> T;
  T Uo[1], Un[1], Go[1][D], Gn[1][D], fo[1], go[1][D], fn[1], gn[1][D];
  Uo[0] = dconst<M, double>(0.0); Uo[0].d[0] = 1.0;
  Un[0] = dconst<M, double>(0.0); Un[0].d[1] = 1.0;
#pragma unroll
  for (int d = 0; d < D; d++) {
    Go[0][d] = dconst<M, double>(0.0); Go[0][d].d[2 + d] = 1.0;
    Gn[0][d] = dconst<M, double>(0.0); Gn[0][d].d[2 + D + d] = 1.0;
  }
  if (has_nb) Form::template inner<D, T, double>(a.fp, n, mu, Uo, Un, Go, Gn, fo, go, fn, gn);
  else Form::template boundary<D, T, double>(a.fp, n, mu, Uo, Go, fo, go);
  const double woo = a.sqrtg[j * NF + f] * sc * sc;
  const double won = has_nb ? a.sqrtg[j * NF + f] * sc * a.scaling[cn] : 0.0;
  double* coo = c + LS::O_FACE + f * LS::NTF;
  double* con = c + LS::NT0 + f * LS::NTF;
  coo[0] = woo * fo[0].d[0];
  con[0] = has_nb ? won * fo[0].d[1] : 0.0;
#pragma unroll
  for (int e = 0; e < D; e++) {
    double go_ = 0.0, gn_ = 0.0, ho = 0.0, hn = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      go_ += fo[0].d[2 + d] * iJ[e][d];
      gn_ += fo[0].d[2 + D + d] * a.invJ[cn * D * D + e * D + d];
      ho += go[0][d].d[0] * iJ[e][d];
      hn += go[0][d].d[1] * iJ[e][d];
    }
    coo[1 + e] = woo * go_;
    coo[1 + D + e] = woo * ho;
    con[1 + e] = has_nb ? won * gn_ : 0.0;
    con[1 + D + e] = has_nb ? won * hn : 0.0;
  }
}

// acc over the tables of one block kind: NTAB table entries stay in registers while the thread
// walks its cells; the coefficients are wave-uniform (scalar loads).
template <int NTAB>
__device__ __forceinline__ void linear_blocks(int J, int c0, int c1, int step, int64_t NC, int o_coef, int NN, int e, bool live,
                                              const double* __restrict__ tab, const double* __restrict__ coef, double alpha, double beta,
                                              double shift, int64_t stride, double* __restrict__ out) {
  double t[NTAB];
#pragma unroll
  for (int k = 0; k < NTAB; k++) t[k] = tab[(size_t)k * NN + e];
  for (int j = c0; j < c1; j += step) {
    const double* c = coef + (int64_t)j * NC + o_coef;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NTAB; k++) s += c[k] * t[k];
    if (live) {
      double* o = out + (int64_t)j * stride;
      *o = alpha * s + shift + (beta != 0.0 ? beta * *o : 0.0);
    }
  }
}

// Blocks of slot s = blockIdx.y (0 the diagonal) of the cells of chunk blockIdx.x.  Thread (sub, e):
// entry e of the N x N block, of every sub-th cell; NP = N^2 rounded up to whole wavefronts, so a
// wavefront works on one cell at a time.  Slots without a column cell become beta * old.
template <int D>
__global__ void __launch_bounds__(512) k_linear_assemble(int J, int N, int NP, int chunk, int S, const double* __restrict__ tables,
                                                         const double* __restrict__ coef, double alpha,
                                                         double beta, double shift, int transposed, double* __restrict__ blocks) {
  typedef LinShape<D> LS;
  const int NN = N * N, nsub = blockDim.x / NP;
  const int sub = __builtin_amdgcn_readfirstlane(threadIdx.x / NP);
  const int e0 = threadIdx.x - sub * NP, e = e0 < NN ? e0 : NN - 1;
  const bool live = e0 < NN;
  const int s = blockIdx.y;
  const int c0 = blockIdx.x * chunk + sub, c1 = min(J, (int)(blockIdx.x + 1) * chunk);
  const int r = e / N, q = e - r * N;
  const double sh = (s == 0 && r == q) ? shift : 0.0;
  double* out = blocks + (int64_t)s * NN + (transposed ? q * N + r : e);
  const int64_t stride = (int64_t)S * NN;
  if (s == 0) {
    linear_blocks<LS::NT0>(J, c0, c1, nsub, LS::NC, 0, NN, e, live, tables, coef, alpha, beta, sh, stride, out);
  } else {
    // a boundary face has zero coefficients: its slot becomes beta * old
    linear_blocks<LS::NTF>(J, c0, c1, nsub, LS::NC, LS::NT0 + (s - 1) * LS::NTF, NN, e, live,
                           tables + (size_t)(LS::NT0 + (s - 1) * LS::NTF) * NN, coef, alpha, beta, 0.0, stride, out);
  }
}

// Reference matrices, in the order of the coefficients (host, from the uploaded tables).
void linear_reference_matrices(int D, int N, int Kv, int Ke, const int* pair, const double* vw, const double* phi, const double* dphi,
                               const double* fw, const double* trace, const double* dtrace, std::vector<double>& T) {
  const int NF = 2 * D, NTF = 1 + 2 * D, NT0 = D + D * D + NF * NTF, NN = N * N;
  T.assign((size_t)(NT0 + NF * NTF) * NN, 0.0);
  for (int e = 0; e < D; e++)
    for (int n = 0; n < N; n++)
      for (int m = 0; m < N; m++) {
        double c = 0.0, k2[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < Kv; k++) {
          const double wn = vw[k] * dphi[((size_t)k * N + n) * D + e];
          c += wn * phi[(size_t)k * N + m];
          for (int e2 = 0; e2 < D; e2++) k2[e2] += wn * dphi[((size_t)k * N + m) * D + e2];
        }
        T[(size_t)e * NN + n * N + m] = c;
        for (int e2 = 0; e2 < D; e2++) T[(size_t)(D + e * D + e2) * NN + n * N + m] = k2[e2];
      }
  for (int f = 0; f < NF; f++)
    for (int other = 0; other < 2; other++) {
      const int g = other ? pair[f] : f;
      const size_t base = (size_t)(other ? NT0 + f * NTF : D + D * D + f * NTF);
      for (int n = 0; n < N; n++)
        for (int m = 0; m < N; m++) {
          double mm = 0.0, gg[3] = {0.0, 0.0, 0.0}, hh[3] = {0.0, 0.0, 0.0};
          for (int k = 0; k < Ke; k++) {
            const double pn = fw[k] * trace[((size_t)f * Ke + k) * N + n], pm = trace[((size_t)g * Ke + k) * N + m];
            mm += pn * pm;
            for (int e = 0; e < D; e++) {
              gg[e] += pn * dtrace[(((size_t)g * Ke + k) * N + m) * D + e];
              hh[e] += fw[k] * dtrace[(((size_t)f * Ke + k) * N + n) * D + e] * pm;
            }
          }
          T[base * NN + n * N + m] = mm;
          for (int e = 0; e < D; e++) {
            T[(base + 1 + e) * NN + n * N + m] = gg[e];
            T[(base + 1 + D + e) * NN + n * N + m] = hh[e];
          }
        }
    }
}

int64_t linear_coefs_per_cell(int D) { return D == 2 ? LinShape<2>::NC : LinShape<3>::NC; }

template <class Form, int D>
static void launch_linear(const LinArgs& a, int N, int S, const double* tables, double* coef, double alpha,
                          double beta, double shift, int transposed, double* blocks, hipStream_t s) {
  const int64_t nt = (int64_t)a.J * (1 + 2 * D);
  hipLaunchKernelGGL((k_linear_coefs<Form, D>), dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, s, a, coef);
  // Chunks of 32 cells: the 3.2 KB tables of a block kind (54 of them for the diagonal) are read
  // once per chunk from L2, against 32 blocks written; 32 still gives a few workgroups per CU and slot.
  const int NP = (N * N + 63) / 64 * 64, nsub = NP >= 256 ? 1 : 256 / NP, chunk = 32;
  hipLaunchKernelGGL((k_linear_assemble<D>), dim3((unsigned)((a.J + chunk - 1) / chunk), S), dim3(NP * nsub), 0, s, a.J, N, NP, chunk, S,
                     tables, coef, alpha, beta, shift, transposed, blocks);
}

void launch_linear_assemble(bool advection, int D, const LinArgs& a, int N, int S, const double* tables, double* coef,
                            double alpha, double beta, double shift, int transposed, double* blocks, hipStream_t s) {
  if (advection) {
    if (D == 2) launch_linear<FormAdvDiff, 2>(a, N, S, tables, coef, alpha, beta, shift, transposed, blocks, s);
    else launch_linear<FormAdvDiff, 3>(a, N, S, tables, coef, alpha, beta, shift, transposed, blocks, s);
  } else {
    if (D == 2) launch_linear<FormSIP, 2>(a, N, S, tables, coef, alpha, beta, shift, transposed, blocks, s);
    else launch_linear<FormSIP, 3>(a, N, S, tables, coef, alpha, beta, shift, transposed, blocks, s);
  }
}

}  // namespace bosss
