// xs_batch_create of the library's own source over the simulated runtime: the
// kernels are stand-ins that do what the host code reads back.  Arguments: the
// null stream's lateness, the diagonal offsets of a system, a zero pivot's row
// (-1: none), and the bytes of device memory; prints the status, whether the
// solve is given diagonal slots, and whether the FP32 CSR values are there.
#include <cstdio>
#include <vector>

#include "../../xsolver_amd/csrc/xs_batch_host.cpp"

static int nd, bad_row, slots = -1, v32 = -1;

void xs_batch_offsets(hipStream_t s, int, const int *, const int *, const int *, int *, int *stat) {
  sim_push(s, [=] {
    if (nd > stat[0]) stat[0] = nd;   // the kernel's atomicMax
    if (nd > XS_DIA_MAX && stat[1] < 1) stat[1] = 1;
  });
}
void xs_batch_dia(hipStream_t, int, int, const int *, const int *, const int *, const int *,
                  const double *, double *, float *) {}
void xs_batch_prep(hipStream_t s, int, const int *, const int *, const double *, double *, float *,
                   float *, int *bad) {
  sim_push(s, [=] {
    if (bad_row >= 0 && bad_row + 1 < *bad) *bad = bad_row + 1;   // atomicMin
  });
}
void xs_batch_prep64(hipStream_t, int, const int *, const int *, const double *, double *, unsigned *) {}
void xs_batch_cg(hipStream_t, int, int, int, int, const xs_batch_args &) {}
bool xs_batch_res(hipStream_t, int, int nsys, int, int, int, const xs_batch_args &P) {
  slots = P.dv != nullptr && P.dv32 != nullptr;
  v32 = P.v32 != nullptr;
  for (int q = 0; q < nsys; ++q) {
    P.iters[q] = 1;
    P.relres[q] = 0.0;
  }
  return true;
}

int main(int argc, char **argv) {
  if (argc != 5) return 2;
  sim_late = atoi(argv[1]);
  nd = atoi(argv[2]);
  bad_row = atoi(argv[3]);
  sim_alloc_left = atol(argv[4]);
  const int nsys = 3, n = 3 * 1000;
  std::vector<int> sp{0, 1000, 2000, n}, rp(n + 1), ci(n);
  for (int i = 0; i <= n; ++i) rp[i] = i;
  for (int i = 0; i < n; ++i) ci[i] = i;
  std::vector<double> v(n, 1.0), b(n, 1.0), x(n, 0.0);
  xs_batch *bt = nullptr;
  const int rc = xs_batch_create(&bt, nsys, sp.data(), rp.data(), ci.data(), v.data());
  if (rc == XS_OK && xs_batch_solve(bt, b.data(), x.data(), 1e-8, 10, 0) != XS_OK) return 3;
  xs_batch_destroy(bt);
  printf("%d %d %d\n", rc, slots, v32);
  return 0;
}
