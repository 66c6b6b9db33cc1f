// Direct assembly of the linear scalar forms (assemble_linear.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "forms.hpp"

namespace bosss {

// Reference matrices and their per-cell coefficients, in this order: C_e (D), K_ee' (D^2), then per
// face M, G_e, H_e (1 + 2 D) of the diagonal block; then per face M, G_e, H_e of the neighbour block.
template <int D>
struct LinShape {
  static constexpr int NF = 2 * D, NTF = 1 + 2 * D;
  static constexpr int O_C = 0, O_K = D, O_FACE = D + D * D;
  static constexpr int NT0 = O_FACE + NF * NTF;   // tables of the diagonal block
  static constexpr int NC = NT0 + NF * NTF;
};

struct LinArgs {
  int J;
  const double *detJ, *invJ, *scaling, *lenscale, *sqrtg, *normal;
  const int* nb;
  FormParams fp;
};

void linear_reference_matrices(int D, int N, int Kv, int Ke, const int* pair, const double* vw, const double* phi, const double* dphi,
                               const double* fw, const double* trace, const double* dtrace, std::vector<double>& T);
int64_t linear_coefs_per_cell(int D);
// blocks[j][s] <- alpha * (matrix block) + beta * old (+ shift on the diagonal of s = 0) for s < S;
// S = 1 writes the diagonal blocks alone.  transposed stores every block transposed.
void launch_linear_assemble(bool advection, int D, const LinArgs& a, int N, int S, const double* tables, double* coef,
                            double alpha, double beta, double shift, int transposed, double* blocks, hipStream_t s);

}  // namespace bosss
