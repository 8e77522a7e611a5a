// Set-up of the fused transfers of the AMG levels (amg_cycle.h): values of
// sparse products on a given pattern.
#include "mpet_ops.h"
#include <stdio.h>

namespace mpet {

// One thread per entry of C: its row of X is walked in order and each
// partner is found in Y's sorted row by bisection.  Set-up only (once per
// level and solver): 25 M-nonzero A times the P1 embedding takes ~2 ms.
__global__ void __launch_bounds__(256)
product_values_kernel(long long nnz, const int* __restrict__ row, const int* __restrict__ col,
                      const int* __restrict__ Xrp, const int* __restrict__ Xci,
                      const double* __restrict__ Xv, const int* __restrict__ Yrp,
                      const int* __restrict__ Yci, const double* __restrict__ Yv,
                      double* __restrict__ out) {
  const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
  if (k >= nnz) return;
  const int r = row[k], c = col[k];
  double s = 0.0;
  for (int j = Xrp[r]; j < Xrp[r + 1]; ++j) {
    const int m = Xci[j];
    const int hi = Yrp[m + 1];
    const int p = lower_bound_i32(Yci, Yrp[m], hi, c);
    if (p < hi && Yci[p] == c) s += Xv[j] * Yv[p];
  }
  out[k] = s;
}

}  // namespace mpet

using namespace mpet;

extern "C" int mpet_product_values(int64_t nnz, const int32_t* row, const int32_t* col,
                                   const int32_t* X_rp, const int32_t* X_ci, const double* X_v,
                                   const int32_t* Y_rp, const int32_t* Y_ci, const double* Y_v,
                                   double* out, hipStream_t stream) {
  if (nnz < 0 || (nnz > 0 && (!row || !col || !X_rp || !Y_rp || !out))) {
    mpet_set_error("mpet_product_values: invalid argument");
    return ERR_INVALID;
  }
  if (nnz == 0) return OK;
  const long long blocks = (nnz + 255) / 256;
  hipLaunchKernelGGL(product_values_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     (long long)nnz, row, col, X_rp, X_ci, X_v, Y_rp, Y_ci, Y_v, out);
  return hipGetLastError() == hipSuccess ? OK : ERR_HIP;
}
