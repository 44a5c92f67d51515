// Gaussian elimination of a small linear system by four lanes that share it.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

namespace mole {

// Row echelon form with partial pivoting of A y = b (A n x n by rows, y holding
// b), both shared by the lanes sub = 0..3: every lane searches the pivot, then
// the lanes take the columns of the row swap (y is column n) and the rows below
// the pivot in turn.  sync() orders the lanes' accesses; each of them calls it
// 3 `steps` times, steps >= n (systems that run side by side may differ in n).
// The search reads what the swap of another lane writes, so it has a sync() of
// its own behind it.
template <class Sync>
__host__ __device__ inline void eliminate_by_lanes(double *A, double *y, int n, int steps, int sub, Sync sync) {
#pragma unroll 1
  for (int p = 0; p < steps; ++p) {
    int piv = p;
    if (p < n) {
      double best = fabs(A[p * n + p]);
      for (int r = p + 1; r < n; ++r) {
        const double v = fabs(A[r * n + p]);
        if (v > best) {
          best = v;
          piv = r;
        }
      }
    }
    sync();
    if (p < n && piv != p)
      for (int k = p + sub; k <= n; k += 4) {
        double *u = k < n ? A + p * n + k : y + p, *v = k < n ? A + piv * n + k : y + piv;
        const double t = *u;
        *u = *v;
        *v = t;
      }
    sync();
    if (p < n) {
      const double app = A[p * n + p], yp = y[p];
      for (int r = p + 1 + sub; r < n; r += 4) {
        const double f = A[r * n + p] / app;
        int k = p + 1;
        for (; k + 2 <= n; k += 2) {
          const double a0 = A[p * n + k], a1 = A[p * n + k + 1], b0 = A[r * n + k], b1 = A[r * n + k + 1];
          A[r * n + k] = fma(-f, a0, b0);
          A[r * n + k + 1] = fma(-f, a1, b1);
        }
        if (k < n) A[r * n + k] = fma(-f, A[p * n + k], A[r * n + k]);
        y[r] = fma(-f, yp, y[r]);
      }
    }
    sync();
  }
}

}  // namespace mole
