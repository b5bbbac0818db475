// xs_batch.h -- persistent batched CG kernels (xs_batch.hip).
#pragma once
#include <hip/hip_runtime.h>

void xs_batch_prep(hipStream_t s, int n, const int *rp, const int *ci, const double *v,
                   double *dinv, float *dinv32, float *v32, int *bad);
void xs_batch_prep64(hipStream_t s, int n, const int *rp, const int *ci, const double *v,
                     double *dinv, unsigned *queue);
// rows of a system that k_batch_res can keep on one CU
#define BT_RES_ROWS 25600
// and in its form with two workgroups on a CU
#define BT_RES_SMALL 4096
// diagonal slots per row of its copy of the matrix: 5-point systems
#define BT_RES_ND 5
// N rows and nnz entries in the whole batch (N is the stride of the vectors
// in w64 / w32 and of the diagonal slots); order == nullptr: systems are
// taken in index order.  A system whose rows or columns fall outside its
// bounds gets iters = -1 and relres = NaN.
struct xs_batch_args {
  int N = 0, nnz = 0;
  const int *order = nullptr, *sys_ptr = nullptr, *rp = nullptr, *ci = nullptr;
  const double *v = nullptr;
  const float *v32 = nullptr;
  // diagonal slots of every system: BT_RES_ND slabs of N values in FP64 and
  // FP32, offsets off[sys * XS_DIA_MAX + k]; null = CSR
  const int *off = nullptr;
  const double *dv = nullptr;
  const float *dv32 = nullptr;
  const double *dinv = nullptr;
  const float *dinv32 = nullptr;
  const double *b = nullptr;
  double *x = nullptr;
  double *w64 = nullptr;   // 6 N (FP64; k_batch_res uses 2 N)
  float *w32 = nullptr;    // 6 N (FP32)
  double tol = 0.0, inner_tol = 0.0;
  int maxiter = 0;
  unsigned *queue = nullptr;
  int *iters = nullptr;
  double *relres = nullptr;
};
// the systems of more than minrows rows (by k_batch_res: and at most maxrows, no
// more than BT_RES_ROWS); false: the launch was refused.  Rows outside the
// batch are reported by xs_batch_res with minrows = 0.
void xs_batch_cg(hipStream_t s, int grid, int nsys, int minrows, int precision,
                 const xs_batch_args &P);
bool xs_batch_res(hipStream_t s, int grid, int nsys, int minrows, int maxrows, int precision,
                  const xs_batch_args &P);
// diagonal slots: the offsets of every system (stat[0] = the most of one,
// stat[1] = 1 when one has too many or unsorted rows; both 0 before), then
// the slabs
void xs_batch_offsets(hipStream_t s, int nsys, const int *sys_ptr, const int *rp, const int *ci,
                      int *off, int *stat);
void xs_batch_dia(hipStream_t s, int nsys, int N, const int *sys_ptr, const int *off,
                  const int *rp, const int *ci, const double *v, double *dv, float *dv32);
