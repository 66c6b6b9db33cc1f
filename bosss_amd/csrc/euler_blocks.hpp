// Direct diagonal blocks of the Euler Jacobian (euler_blocks.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "dg_kernels.hpp"

namespace bosss {

// Host tables of one (D, P, K1), made once per operator: `real` and `ints` are uploaded as they are.
struct EulerBlockTables {
  std::vector<double> real;    // 1D values, volume and face moment matrices in MFMA order, term coefficients
  std::vector<int32_t> ints;   // term list offsets, entry order, term indices
};
void euler_block_tables(int D, int P, int K1, const std::vector<double>& nodes, EulerBlockTables& t);   // nodes: 1D Gauss nodes

struct EulerBlockArgs {
  int J;
  const double *detJ, *invJ, *scaling;
  CellFaces cf;
  FormParams fp;
  const double* real;
  const int32_t* ints;
  const void* U;
  double alpha, shift;
  int transposed;
  double* blocks;
};

// blocks[j] <- alpha dR_j/dU_j + shift I (stored transposed if asked).  Returns false where no kernel
// is built for (D, P, K1).
bool launch_euler_blocks(bool hllc, int D, int P, int K1, bool fp32, int num_cu, const EulerBlockArgs& a, hipStream_t s);

}  // namespace bosss
