// Direct diagonal blocks of the Euler Jacobian (euler_blocks.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "dg_kernels.hpp"

namespace bosss {

// Host tables of one (P, K1), made once per operator: `real` and `ints` are uploaded as they are.
struct EulerBlockTables {
  std::vector<double> real;    // 1D values, volume and face moment matrices in MFMA order, term coefficients
  std::vector<int32_t> ints;   // term list offsets, entry order, term indices
};
void euler_block_tables(int P, int K1, const std::vector<double>& nodes, EulerBlockTables& t);   // nodes: 1D Gauss nodes

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

// Whether the kernel is built for these operators: 3D.  The 24 columns of the 2D p = 2 blocks cost little by
// probing, and by moments they measured 12 % further from 64-bit exact (7.1e-16 against 6.3e-16; 3D p = 2 8.5e-16
// against 9.0e-16, p = 3 1.4e-15 against 1.7e-15).
bool has_euler_blocks(int D, int P, int K1);

// blocks[j] <- alpha dR_j/dU_j + shift I (stored transposed if asked).
void launch_euler_blocks(bool hllc, int P, bool fp32, int num_cu, const EulerBlockArgs& a, hipStream_t s);

}  // namespace bosss
