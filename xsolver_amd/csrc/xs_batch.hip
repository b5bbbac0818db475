// xs_batch.hip -- many independent systems in one persistent launch.
//
// The systems are the diagonal blocks of one block-diagonal CSR matrix
// (sys_ptr[s]..sys_ptr[s+1] are the rows of system s, with columns in the
// same range).  Each workgroup takes systems from an atomic queue (largest
// first, a longest-processing-time order) and runs preconditioned CG with
// Jacobi (hip/Solver/xsolver_cg.cpp:16-74) on it to convergence with
// workgroup barriers only: every system stops at its own iteration count
// (per-system convergence), and no kernel is launched per iteration.
// Precision 1 runs one FP32 CG recurrence (FP32 values, vectors, SpMV) with
// FP64 reliable updates: the FP64 residual b - A x replaces the FP32 one at
// every 1e-2 drop and decides convergence.
// Two kernels: k_batch_res keeps a system's vectors on the chip (systems of
// up to BT_RES_ROWS rows), k_batch_cg keeps them in memory (larger ones).
// No reference counterpart (the reference solves one system per call).
#include <climits>
#include <type_traits>
#include <utility>

#include "xs_device.h"
#include "xs_batch.h"

#define BT_THREADS 1024
#define BT_WAVES (BT_THREADS / XS_WAVE)

template <class T>
__device__ __forceinline__ T bt_wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, XS_WAVE);
  return v;
}

// workgroup sum of two values (double accumulation)
template <int NT = BT_THREADS>
__device__ __forceinline__ void bt_sum2(double &a, double &b, double (*red)[2]) {
  const int lane = threadIdx.x & (XS_WAVE - 1), w = threadIdx.x / XS_WAVE;
  a = bt_wave_sum(a);
  b = bt_wave_sum(b);
  __syncthreads();
  if (lane == 0) { red[w][0] = a; red[w][1] = b; }
  __syncthreads();
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int q = 0; q < NT / XS_WAVE; ++q) { s0 += red[q][0]; s1 += red[q][1]; }
  a = s0;
  b = s1;
}

// Rows of a thread: r0 + threadIdx.x, then every BT_THREADS.  Each thread's
// loads are serial chains (row pointer -> column -> gather; or the operands
// of an update, behind the previous element's stores, which may alias them
// as far as the compiler knows), so the loops below take two rows (four
// elements) per step with every load of the step issued before any store:
// the same arithmetic in the same order, half (a quarter of) the chains.

// A row's first W entries, loaded branch-free and masked (a masked slot
// reads column r, value ignored).
template <int W, class TV, class TX>
struct bt_rowbuf {
  int e0, e1;
  int c[W];
  TV a[W];
  TX g[W];
  __device__ __forceinline__ void load(int r, const int *__restrict__ rp, const int *__restrict__ ci,
                                       const TV *__restrict__ v) {
    e0 = rp[r];
    e1 = rp[r + 1];
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const int e = min(e0 + k, max(e1 - 1, 0));
      const int cc = ci[e];
      c[k] = e0 + k < e1 ? cc : r;
      a[k] = v[e];
    }
  }
  __device__ __forceinline__ void gather(const TX *x) {
#pragma unroll
    for (int k = 0; k < W; ++k) g[k] = x[c[k]];
  }
  // sum_e v[e] x[ci[e]] in CSR order
  __device__ __forceinline__ TX sum() const {
    TX s = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const TX t = s + (TX)a[k] * g[k];
      s = e0 + k < e1 ? t : s;
    }
    return s;
  }
};

// f(row, (A x)_row) for the thread's rows of [r0, r1), in order, two rows per
// step: each row's first W entries in the window, any further ones after
// them in a loop (rows longer than W are rare), so the sum keeps CSR order.
template <int W, class TV, class TX, class F>
__device__ __forceinline__ void bt_rows(int r0, int r1, const int *__restrict__ rp,
                                        const int *__restrict__ ci, const TV *__restrict__ v,
                                        const TX *x, F &&f) {
  auto tail = [&](const bt_rowbuf<W, TV, TX> &R, TX s) {
    for (int e = R.e0 + W; e < R.e1; ++e) s += (TX)v[e] * x[ci[e]];
    return s;
  };
  for (int r = r0 + threadIdx.x; r < r1; r += 2 * BT_THREADS) {
    const int rb = r + BT_THREADS;
    const bool vb = rb < r1;
    bt_rowbuf<W, TV, TX> A, B;
    A.load(r, rp, ci, v);
    B.load(vb ? rb : r, rp, ci, v);
    A.gather(x);
    B.gather(x);
    f(r, tail(A, A.sum()));
    if (vb) f(rb, tail(B, B.sum()));
  }
}

// y = A p over rows [r0, r1) and sum p.y
template <int W, class TV, class TX>
__device__ __forceinline__ double bt_spmv_dot(int r0, int r1, const int *__restrict__ rp,
                                              const int *__restrict__ ci,
                                              const TV *__restrict__ v, const TX *p, TX *y) {
  double acc = 0.0;
  bt_rows<W, TV, TX>(r0, r1, rp, ci, v, p, [&](int r, TX s) {
    y[r] = s;
    acc += (double)s * (double)p[r];
  });
  return acc;
}

// CG + Jacobi on rows [r0, r1) for A d = rhs from d = 0 (FP32 or FP64);
// stops when ||r|| <= tol * ||rhs||.  Returns iterations (barrier-uniform).
template <int W, class TV, class TX>
__device__ int bt_cg(int r0, int r1, const int *__restrict__ rp, const int *__restrict__ ci,
                     const TV *__restrict__ v, const TX *__restrict__ dinv, const TX *rhs, TX *d,
                     TX *r, TX *z, TX *p, TX *q, double tol, int maxit, double (*red)[2]) {
  constexpr int U = 4;   // elements per step of the update loops
  double tau = 0.0, rr = 0.0;
  for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) {
    const TX ri = rhs[i];
    const TX zi = dinv[i] * ri;
    d[i] = 0;
    r[i] = ri;
    z[i] = zi;
    p[i] = zi;
    tau += (double)ri * (double)zi;
    rr += (double)ri * (double)ri;
  }
  bt_sum2(tau, rr, red);
  const double res0 = sqrt(rr);
  if (res0 == 0.0) return 0;
  int it = 0;
  while (it < maxit) {
    __syncthreads();
    double sigma = bt_spmv_dot<W, TV, TX>(r0, r1, rp, ci, v, p, q), dummy = 0.0;
    bt_sum2(sigma, dummy, red);
    const TX alpha = (TX)(tau / sigma);
    double tn = 0.0, rn = 0.0;
    for (int i0 = r0 + threadIdx.x; i0 < r1; i0 += U * BT_THREADS) {
      TX pv[U], qv[U], rv[U], dv[U], di[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = min(i0 + k * BT_THREADS, r1 - 1);
        pv[k] = p[i];
        qv[k] = q[i];
        rv[k] = r[i];
        dv[k] = d[i];
        di[k] = dinv[i];
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = i0 + k * BT_THREADS;
        if (i < r1) {
          d[i] = dv[k] + alpha * pv[k];
          const TX ri = rv[k] - alpha * qv[k];
          r[i] = ri;
          const TX zi = di[k] * ri;
          z[i] = zi;
          tn += (double)zi * (double)ri;
          rn += (double)ri * (double)ri;
        }
      }
    }
    bt_sum2(tn, rn, red);
    const TX beta = (TX)(tn / tau);
    tau = tn;
    ++it;
    if (!(sqrt(rn) > tol * res0)) break;   // also stops on NaN
    for (int i0 = r0 + threadIdx.x; i0 < r1; i0 += U * BT_THREADS) {
      TX zv[U], pv[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = min(i0 + k * BT_THREADS, r1 - 1);
        zv[k] = z[i];
        pv[k] = p[i];
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = i0 + k * BT_THREADS;
        if (i < r1) p[i] = zv[k] + beta * pv[k];
      }
    }
  }
  __syncthreads();
  return it;
}

// 1 when every row of [r0, r1) has row pointers inside [0, nnz] and every
// column inside [r0, r1) (block-diagonal pattern), else 0; workgroup-uniform.
template <int NT>
__device__ int bt_pattern_ok(int r0, int r1, int N, int nnz, const int *__restrict__ rp,
                             const int *__restrict__ ci, double (*red)[2]) {
  double bad = 0.0, dummy = 0.0;
  if (r0 < 0 || r1 > N || r1 <= r0) bad = 1.0;
  else
    for (int i = r0 + threadIdx.x; i < r1; i += NT) {
      const int e0 = rp[i], e1 = rp[i + 1];
      if (e0 < 0 || e1 < e0 || e1 > nnz) { bad = 1.0; continue; }
      for (int e = e0; e < e1; ++e)
        if (ci[e] < r0 || ci[e] >= r1) bad = 1.0;
    }
  bt_sum2<NT>(bad, dummy, red);
  return bad == 0.0;
}

// ||r|| / ||b - A x0|| from the squares; NaN when the base is not finite (a
// NaN or an infinity in b, x0 or A, or a norm that overflows): such a system
// has no residual to speak of and has not converged
__device__ __forceinline__ double bt_relres(double rn, double bb) {
  return isfinite(bb) ? (bb > 0.0 ? sqrt(rn / bb) : 0.0) : __builtin_nan("");
}

// One system on rows [r0, r1): FP64 CG from x0 (PREC 0), or FP32 CG with
// FP64 reliable updates (PREC 1).
#define BT_W 6   // row window of the SpMV (FP64: the register budget of 1024-thread groups)
template <int PREC>
__device__ void bt_system(int r0, int r1, int N, const int *__restrict__ rp,
                          const int *__restrict__ ci, const double *__restrict__ v,
                          const float *__restrict__ v32, const double *__restrict__ dinv,
                          const float *__restrict__ dinv32, const double *__restrict__ b,
                          double *__restrict__ x, double *__restrict__ w64,
                          float *__restrict__ w32, double tol, int maxiter, double inner_tol,
                          double (*red)[2], int &it, double &rel) {
  constexpr int W = BT_W;
  it = 0;
  rel = 0.0;
  if (PREC == 0) {
    // FP64 CG from x0 (the workspace holds r, z, p, q, rhs, d)
    double *r = w64, *z = w64 + N, *p = z + N, *q = p + N;
    double *rhs = q + N, *d = rhs + N;
    double bb = 0.0, dummy = 0.0;   // ||b - A x0||^2: the base of tol and relres
    bt_rows<W, double, double>(r0, r1, rp, ci, v, x, [&](int i, double ax) {
      const double t = b[i] - ax;
      rhs[i] = t;
      bb += t * t;
    });
    bt_sum2(bb, dummy, red);
    it = bt_cg<W, double, double>(r0, r1, rp, ci, v, dinv, rhs, d, r, z, p, q, tol, maxiter, red);
    double rn = 0.0, dm = 0.0;
    for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) x[i] += d[i];
    __syncthreads();
    bt_rows<W, double, double>(r0, r1, rp, ci, v, x, [&](int i, double ax) {
      const double t = b[i] - ax;
      rn += t * t;
    });
    bt_sum2(rn, dm, red);
    rel = bt_relres(rn, bb);
  } else {
    // One FP32 CG recurrence (FP32 values, vectors and SpMV) with reliable
    // updates: whenever its residual has dropped by inner_tol since the last
    // replacement, or claims convergence, the FP32 correction d is added to
    // the FP64 x, the FP64 residual b - A x replaces the FP32 one and decides
    // convergence; the search direction is kept (no restart, so the
    // iteration count stays near the FP64 CG's).
    constexpr int U = 4;
    float *r = w32, *z = w32 + N, *p = z + N, *q = p + N, *d = q + N;
    double rn64 = 0.0, dm = 0.0;
    bt_rows<W, double, double>(r0, r1, rp, ci, v, x, [&](int i, double ax) {
      const double t = b[i] - ax;
      r[i] = (float)t;
      rn64 += t * t;
    });
    bt_sum2(rn64, dm, red);
    const double bb = rn64;   // ||b - A x0||^2: the base of tol and relres
    rel = bt_relres(bb, bb);
    if (!isfinite(bb) || bb == 0.0) return;  // nothing to solve for, or x0 solves it (rel 0)
    double rref = sqrt(bb), tau = 0.0, t2 = 0.0;
    for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) {
      const float ri = r[i], zi = dinv32[i] * ri;
      z[i] = zi;
      p[i] = zi;
      d[i] = 0.0f;
      tau += (double)zi * (double)ri;
    }
    bt_sum2(tau, t2, red);
    rel = 1.0;
    bool fresh = true;   // x and rel hold the last FP64 residual
    while (it < maxiter) {
      __syncthreads();
      double sigma = bt_spmv_dot<W, float, float>(r0, r1, rp, ci, v32, p, q), dummy = 0.0;
      bt_sum2(sigma, dummy, red);
      const float alpha = (float)(tau / sigma);
      double tn = 0.0, rn = 0.0;
      for (int i0 = r0 + threadIdx.x; i0 < r1; i0 += U * BT_THREADS) {
        float pv[U], qv[U], rv[U], dv[U], di[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int i = min(i0 + k * BT_THREADS, r1 - 1);
          pv[k] = p[i];
          qv[k] = q[i];
          rv[k] = r[i];
          dv[k] = d[i];
          di[k] = dinv32[i];
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int i = i0 + k * BT_THREADS;
          if (i < r1) {
            d[i] = dv[k] + alpha * pv[k];
            const float ri = rv[k] - alpha * qv[k];
            r[i] = ri;
            const float zi = di[k] * ri;
            z[i] = zi;
            tn += (double)zi * (double)ri;
            rn += (double)ri * (double)ri;
          }
        }
      }
      bt_sum2(tn, rn, red);
      ++it;
      fresh = false;
      const double rnorm = sqrt(rn);
      if (!(rnorm > inner_tol * rref) || !(rnorm > tol * sqrt(bb))) {
        // reliable update: x += d, r = b - A x in FP64
        __syncthreads();
        for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) {
          x[i] += (double)d[i];
          d[i] = 0.0f;
        }
        __syncthreads();
        rn64 = 0.0;
        bt_rows<W, double, double>(r0, r1, rp, ci, v, x, [&](int i, double ax) {
          const double t = b[i] - ax;
          r[i] = (float)t;
          rn64 += t * t;
        });
        bt_sum2(rn64, dm, red);
        fresh = true;
        rel = sqrt(rn64 / bb);
        if (!(rel >= tol)) break;   // converged (or NaN)
        rref = sqrt(rn64);
        tn = 0.0;
        for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) {
          const float ri = r[i], zi = dinv32[i] * ri;
          z[i] = zi;
          tn += (double)zi * (double)ri;
        }
        bt_sum2(tn, dm, red);
      }
      const float beta = (float)(tn / tau);
      tau = tn;
      for (int i0 = r0 + threadIdx.x; i0 < r1; i0 += U * BT_THREADS) {
        float zv[U], pv[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int i = min(i0 + k * BT_THREADS, r1 - 1);
          zv[k] = z[i];
          pv[k] = p[i];
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int i = i0 + k * BT_THREADS;
          if (i < r1) p[i] = zv[k] + beta * pv[k];
        }
      }
    }
    if (!fresh) {   // out of iterations: x and relres with the last correction
      __syncthreads();
      for (int i = r0 + threadIdx.x; i < r1; i += BT_THREADS) x[i] += (double)d[i];
      __syncthreads();
      rn64 = 0.0;
      bt_rows<W, double, double>(r0, r1, rp, ci, v, x, [&](int i, double ax) {
        const double t = b[i] - ax;
        rn64 += t * t;
      });
      bt_sum2(rn64, dm, red);
      rel = sqrt(rn64 / bb);
    }
  }
}

// N: rows of the whole batch (the workspace stride); nnz: entries of the
// whole batch.  A system whose rows or pattern fall outside those bounds is
// not solved: iters = -1, relres = NaN.  Systems of at most minrows rows are
// left to k_batch_res.
template <int PREC>
__global__ __launch_bounds__(BT_THREADS) void k_batch_cg(
    int nsys, int N, int nnz, int minrows, const int *__restrict__ order,
    const int *__restrict__ sys_ptr, const int *__restrict__ rp, const int *__restrict__ ci,
    const double *__restrict__ v, const float *__restrict__ v32, const double *__restrict__ dinv,
    const float *__restrict__ dinv32, const double *__restrict__ b, double *__restrict__ x,
    double *__restrict__ w64, float *__restrict__ w32, double tol, int maxiter,
    double inner_tol, unsigned *queue, int *iters, double *relres) {
  __shared__ double red[BT_WAVES][2];
  __shared__ int s_sys;
  for (;;) {
    if (threadIdx.x == 0) {
      const unsigned t = atomicAdd(queue, 1u);
      s_sys = t < (unsigned)nsys ? (order ? order[t] : (int)t) : -1;
    }
    __syncthreads();
    const int sys = s_sys;
    __syncthreads();
    if (sys < 0) break;
    const int r0 = sys_ptr[sys], r1 = sys_ptr[sys + 1];
    // (a pattern that is not a system's is reported by k_batch_res)
    if (r0 < 0 || r1 > N || r1 - r0 <= minrows) continue;   // workgroup-uniform
    int it = 0;
    double rel = 0.0;
    if (!bt_pattern_ok<BT_THREADS>(r0, r1, N, nnz, rp, ci, red)) {
      it = -1;
      rel = __builtin_nan("");
    } else {
      bt_system<PREC>(r0, r1, N, rp, ci, v, v32, dinv, dinv32, b, x, w64, w32, tol, maxiter,
                      inner_tol, red, it, rel);
    }
    if (threadIdx.x == 0) {
      iters[sys] = it;
      relres[sys] = rel;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Resident form: a workgroup of RS_THREADS threads keeps the system it works
// on in its CU.  A thread owns the rows t, t + 512, ... (up to R of them) and
// holds their r, q = A p (z = D^-1 r once q is used) and, where it fits, the
// correction d in registers; p is in LDS.  What bounds the form with the
// vectors in memory (k_batch_cg): ~172 bytes per row and iteration, and for
// the largest systems of a batch the serial time of one workgroup streaming
// them (160 x 160 rows: 155 us per iteration, 62 ms for 401 iterations, the
// whole batch's time).  Here an iteration reads the matrix and 1/a_ii only
// (48 bytes per row of a 5-point system in diagonal slots; 16 more for d in
// systems beyond 32 rows per thread).  512 systems of 32^2 to 160^2 rows:
// FP64 63.5 -> 26.6 ms, FP32 40.4 -> 12.3 ms; the 160^2 system alone 99 -> 51
// us per iteration (FP64), 66 -> 22 (FP32), now bound by the loads one CU has
// in flight; 256 of 128^2 rows 119 -> 46 us (4.45 TB/s).
//
// Batches in which some system has more than BT_RES_ND offsets, or rows that
// do not ascend, are read from the CSR arrays (KB = 1: fewer loads in flight).
// k_batch_cg against that form, ms: 512 7-point systems of 16^3 rows 3.13 and
// 1.27 (FP32 2.11 and 1.21), 256 of 8^3 to 29^3 10.3 and 8.9 (6.4 and 6.3), 64 of
// 20^3 to 29^3 8.5 and 8.3 (5.9 and 6.0), one of 29^3 6.0 and 6.1 (4.5 and 4.5);
// 256 9-point systems of 32^2 to 160^2 18.1 and 13.7 (10.9 and 9.2); the 512
// systems above with one 9-point system among them 85 and 68 (46 and 35).
//
// 512 threads with 256 registers each: the registers of a CU hold 512 KB
// either way, and 8 waves that each have 20 loads in flight reach what one CU
// can draw.  LDS holds the first RS_LDS_ROWS entries of p (FP64; all of them
// in FP32); the rest of p and, beyond 32 rows per thread, d go through the
// workspace.
// The arithmetic and its order depend on a system's rows alone, not on the
// variant: sums of a row in column order by fused multiply-adds, partial sums
// per thread in row order, then lanes, then waves.
// ---------------------------------------------------------------------------
#define RS_THREADS 512
#define RS_WAVES (RS_THREADS / XS_WAVE)
#define RS_RMAX 50                                   // rows per thread
#define RS_LDS_K 39                                  // FP64: rows per thread whose p is in LDS
#define RS_LDS_ROWS (RS_LDS_K * RS_THREADS)          // 19968 x 8 B = 156 KB of the CU's 160
static_assert(BT_RES_ROWS == RS_RMAX * RS_THREADS && BT_RES_SMALL == 8 * RS_THREADS,
              "capacity of the resident forms");

// f(0), f(1), ..., f(N - 1) with constant arguments: loops over register
// arrays that are unrolled whatever their size
template <class F, int... K>
__device__ __forceinline__ void rs_each_seq(F &&f, std::integer_sequence<int, K...>) {
  (f(std::integral_constant<int, K>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void rs_each(F &&f) {
  rs_each_seq(f, std::make_integer_sequence<int, N>{});
}

// The thread's number as a value the compiler cannot follow: a pass over the
// rows that starts from it computes its addresses and loads its operands
// itself.  Otherwise the addresses, the matrix and 1/a_ii, which no iteration
// changes, are all moved ahead of the iteration loop and spilled.
__device__ __forceinline__ int rs_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

__device__ __forceinline__ double rs_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float rs_fma(float a, float b, float c) { return fmaf(a, b, c); }

// workgroup sum of two values; the caller alternates the two buffers of red,
// so that one barrier per sum is enough
__device__ __forceinline__ void rs_sum2(double &a, double &b, double (*red)[2]) {
  const int lane = threadIdx.x & (XS_WAVE - 1), w = threadIdx.x / XS_WAVE;
  a = bt_wave_sum(a);
  b = bt_wave_sum(b);
  if (lane == 0) { red[w][0] = a; red[w][1] = b; }
  __syncthreads();
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int q = 0; q < RS_WAVES; ++q) { s0 += red[q][0]; s1 += red[q][1]; }
  a = s0;
  b = s1;
}

// Row sums of KB rows at once, every load before any sum.  Diagonal slots: ND
// slabs of ld values (slot k of row r = entry (r, r + off[k]) or 0).
template <int ND_, class TV>
struct rs_dia {
  static constexpr int ND = ND_;
  static constexpr bool CSR = false;
  const TV *v;      // at the system's first row
  size_t ld;
  int off[ND_];
  template <int KB, class TX, class G>
  __device__ __forceinline__ void sums(const int (&i)[KB], int m, G &&g, TX (&s)[KB]) const {
    TV a[KB][ND];
#pragma unroll
    for (int k = 0; k < KB; ++k)
#pragma unroll
      for (int e = 0; e < ND; ++e) a[k][e] = v[e * ld + i[k]];
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      s[k] = 0;
#pragma unroll
      for (int e = 0; e < ND; ++e)
        s[k] = rs_fma((TX)a[k][e], g(min(max(i[k] + off[e], 0), m - 1)), s[k]);
    }
  }
};

// The same from the CSR arrays: the first BT_W entries of every row at once,
// the rest of longer rows in a loop.
template <class TV>
struct rs_csr {
  static constexpr int ND = BT_W;
  static constexpr bool CSR = true;
  const int *rp, *ci;
  const TV *v;
  int r0;
  template <int KB, class TX, class G>
  __device__ __forceinline__ void sums(const int (&i)[KB], int m, G &&g, TX (&s)[KB]) const {
    bt_rowbuf<BT_W, TV, TX> B[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) B[k].load(r0 + i[k], rp, ci, v);
#pragma unroll
    for (int k = 0; k < KB; ++k)
#pragma unroll
      for (int e = 0; e < BT_W; ++e) B[k].g[e] = g(B[k].c[e] - r0);
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      s[k] = 0;
#pragma unroll
      for (int e = 0; e < BT_W; ++e) {
        const TX t = rs_fma((TX)B[k].a[e], B[k].g[e], s[k]);
        s[k] = B[k].e0 + e < B[k].e1 ? t : s[k];
      }
      for (int e = B[k].e0 + BT_W; e < B[k].e1; ++e) s[k] = rs_fma((TX)v[e], g(ci[e] - r0), s[k]);
    }
  }
};

// p of the system: entries below cap in LDS, the others in memory (HYB)
template <class T, bool HYB>
struct rs_p {
  T *l, *g;
  __device__ __forceinline__ T operator()(int c) const {
    if (HYB && c >= RS_LDS_ROWS) return g[c];
    return l[c];
  }
  template <int K>   // i = a thread's K-th row
  __device__ __forceinline__ void set(int i, T x) {
    if constexpr (HYB && K >= RS_LDS_K) g[i] = x;
    else l[i] = x;
  }
  template <int K>
  __device__ __forceinline__ T own(int i) const {
    if constexpr (HYB && K >= RS_LDS_K) return g[i];
    else return l[i];
  }
};

// f(k, i, s) for the thread's rows i = t + 512 k < m, s = row i's sum over g,
// KB rows per step
template <int R, int KB, class TX, class M, class G, class F>
__device__ __forceinline__ void rs_rows(const M &A, int m, G &&g, F &&f) {
  const int t = rs_tid();
  rs_each<(R + KB - 1) / KB>([&](auto step) {
    constexpr int k0 = decltype(step)::value * KB;
    if (k0 * RS_THREADS >= m) return;   // uniform
    int i[KB];
    TX s[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) i[k] = min(t + (k0 + k) * RS_THREADS, m - 1);
    A.template sums<KB, TX>(i, m, g, s);
    rs_each<KB>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      if constexpr (k0 + k < R)
        if (t + (k0 + k) * RS_THREADS < m) f(std::integral_constant<int, k0 + k>{}, i[k], s[k]);
    });
  });
}

// One system of m rows at r0.  PREC 0: FP64 CG + Jacobi on A d = b - A x0,
// x = x0 + d; PREC 1: FP32 CG with FP64 reliable updates (bt_system).  A:
// the matrix in T for the CG, A64 in FP64 for the residuals.  wp / wd: the
// system's part of the workspace for p (HYB) and d.
template <int PREC, int R, class T, class M, class M64>
__device__ void rs_system(const M &A, const M64 &A64, int m, const T *__restrict__ dinv,
                          const double *__restrict__ b, double *x, T *wp, T *wd, T *lp, double tol,
                          int maxiter, double inner_tol, double (*red)[RS_WAVES][2], int &it,
                          double &rel) {
  constexpr bool F64 = sizeof(T) == 8;
  constexpr bool HYB = F64 && R > RS_LDS_K;
  constexpr bool DREG = !F64 || R <= 32;
  // rows per step of the products: the loads in flight against the registers
  constexpr int KB = M::CSR ? 1 : F64 ? 2 : 4;
  constexpr int U = F64 && R > 8 ? 2 : 4;   // and of the updates
  rs_p<T, HYB> p{lp, wp};
  T r[R], q[R], d[DREG ? R : 1];
  int rb = 0;   // the reduction buffer in use
  auto sum2 = [&](double &a, double &c) {
    rs_sum2(a, c, red[rb]);
    rb ^= 1;
  };
  it = 0;
  rel = 0.0;
  double rn = 0.0, tau = 0.0, none = 0.0;
  // f(k, i) for the thread's rows i = t + 512 k < m
  auto own_rows = [&](auto &&f) {
    const int t = rs_tid();
    rs_each<R>([&](auto k) {
      constexpr int K = decltype(k)::value;
      if (K * RS_THREADS >= m) return;   // uniform
      const int i = t + K * RS_THREADS;
      if (i < m) f(k, i);
    });
  };
  // r = b - A x in FP64, rn = its square norm
  auto residual = [&](bool store) {
    rn = 0.0;
    rs_rows<R, 1, double>(A64, m, [&](int c) { return x[c]; }, [&](auto k, int i, double s) {
      const double e = b[i] - s;
      if (store) r[decltype(k)::value] = (T)e;
      rn += e * e;
    });
    sum2(rn, none);
  };
  residual(true);
  const double bb = rn;   // the base of tol and relres
  rel = bt_relres(bb, bb);
  if ((PREC == 1 && !isfinite(bb)) || bb == 0.0) return;   // nothing to solve for, or x0 solves it (rel 0)
  const double res0 = sqrt(bb);
  double rref = res0;     // PREC 1: the last FP64 residual
  bool fresh = true;      // PREC 1: x and rel hold it
  own_rows([&](auto kc, int i) {
    constexpr int k = decltype(kc)::value;
    const T z = dinv[i] * r[k];
    p.template set<k>(i, z);
    if constexpr (DREG) d[k] = 0;
    else wd[i] = 0;
    tau += (double)r[k] * (double)z;
  });
  sum2(tau, none);   // (its barrier also publishes p)
  rel = 1.0;
  while (it < maxiter) {
    double sigma = 0.0;
    rs_rows<R, KB, T>(A, m, [&](int c) { return p(c); }, [&](auto k, int i, T s) {
      q[decltype(k)::value] = s;
      sigma += (double)s * (double)p.template own<decltype(k)::value>(i);
    });
    sum2(sigma, none);
    const T alpha = (T)(tau / sigma);
    double tn = 0.0;
    rn = 0.0;
    const int t = rs_tid();
    rs_each<(R + U - 1) / U>([&](auto step) {
      constexpr int k0 = decltype(step)::value * U;
      if (k0 * RS_THREADS >= m) return;   // uniform
      T di[U], dv[U], pv[U];
      rs_each<U>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr (k0 + k < R) {
          const int i = min(t + (k0 + k) * RS_THREADS, m - 1);
          di[k] = dinv[i];
          if constexpr (!DREG) dv[k] = wd[i];
          pv[k] = p.template own<k0 + k>(i);
        }
      });
      rs_each<U>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr (k0 + k < R) {
          const int i = t + (k0 + k) * RS_THREADS;
          if (i < m) {
            if constexpr (DREG) d[k0 + k] = rs_fma(alpha, pv[k], d[k0 + k]);
            else wd[i] = rs_fma(alpha, pv[k], dv[k]);
            const T ri = rs_fma(-alpha, q[k0 + k], r[k0 + k]);
            const T zi = di[k] * ri;
            r[k0 + k] = ri;
            q[k0 + k] = zi;
            tn += (double)zi * (double)ri;
            rn += (double)ri * (double)ri;
          }
        }
      });
    });
    sum2(tn, rn);
    ++it;
    fresh = false;
    const double rnorm = sqrt(rn);
    if (PREC == 0) {
      if (!(rnorm > tol * res0)) break;   // also stops on NaN
    } else if (!(rnorm > inner_tol * rref) || !(rnorm > tol * res0)) {
      // reliable update: x += d, then the FP64 residual
      own_rows([&](auto kc, int i) {
        constexpr int k = DREG ? decltype(kc)::value : 0;
        x[i] += (double)d[k];
        d[k] = 0;
      });
      __syncthreads();
      residual(true);
      fresh = true;
      rel = sqrt(rn / bb);
      if (!(rel >= tol)) break;   // converged (or NaN)
      rref = sqrt(rn);
      tn = 0.0;
      own_rows([&](auto kc, int i) {
        constexpr int k = decltype(kc)::value;
        const T zi = dinv[i] * r[k];
        q[k] = zi;
        tn += (double)zi * (double)r[k];
      });
      sum2(tn, none);
    }
    const T beta = (T)(tn / tau);
    tau = tn;
    own_rows([&](auto kc, int i) {
      constexpr int k = decltype(kc)::value;
      p.template set<k>(i, rs_fma(beta, p.template own<k>(i), q[k]));
    });
    __syncthreads();
  }
  if (PREC == 1 && fresh) return;
  // x with the correction, and its FP64 residual
  own_rows([&](auto kc, int i) {
    if constexpr (DREG) x[i] += (double)d[decltype(kc)::value];
    else x[i] += (double)wd[i];
  });
  __syncthreads();
  residual(false);
  rel = bt_relres(rn, bb);
}

// Systems of more than minrows and at most maxrows rows, from the queue.  ND:
// BT_RES_ND diagonal slots (xs_batch_dia), or 0 = CSR.  BIG = 0: at most 8 rows
// per thread (BT_RES_SMALL per system) with registers for two workgroups on a
// CU; 1: up to RS_RMAX.
template <int PREC, int ND, int BIG>
__global__ __launch_bounds__(RS_THREADS, BIG ? 2 : 4) void k_batch_res(
    int nsys, int minrows, int maxrows, const xs_batch_args P) {
  typedef typename std::conditional<PREC == 0, double, float>::type T;
  extern __shared__ __align__(16) unsigned char rs_lds[];
  __shared__ double red[2][RS_WAVES][2];
  __shared__ int s_sys;
  T *lp = reinterpret_cast<T *>(rs_lds);
  for (;;) {
    if (threadIdx.x == 0) {
      const unsigned t = atomicAdd(P.queue, 1u);
      s_sys = t < (unsigned)nsys ? (P.order ? P.order[t] : (int)t) : -1;
    }
    __syncthreads();
    const int sys = __builtin_amdgcn_readfirstlane(s_sys);
    __syncthreads();
    if (sys < 0) break;
    const int r0 = P.sys_ptr[sys], r1 = P.sys_ptr[sys + 1], m = r1 - r0;
    // the others' systems; rows outside the batch are reported by the launch
    // with minrows = 0
    const bool inside = r0 >= 0 && r1 <= P.N;
    if (inside ? (m > maxrows || (minrows > 0 && m <= minrows)) : minrows > 0) continue;
    int it = 0;
    double rel = 0.0;
    if (ND == 0 && !bt_pattern_ok<RS_THREADS>(r0, r1, P.N, P.nnz, P.rp, P.ci, red[1])) {   // (the sums of rs_system start with red[0])
      it = -1;
      rel = __builtin_nan("");
    } else {
      const T *dinv = (PREC == 0 ? (const T *)P.dinv : (const T *)P.dinv32) + r0;
      T *wp = (PREC == 0 ? (T *)P.w64 : (T *)P.w32) + r0, *wd = wp + P.N;
#define RS_RUN(R)                                                                               \
  rs_system<PREC, R, T>(A, A64, m, dinv, P.b + r0, P.x + r0, wp, wd, lp, P.tol, P.maxiter,      \
                        P.inner_tol, red, it, rel)
      if constexpr (ND > 0) {
        rs_dia<ND, T> A;
        rs_dia<ND, double> A64;
        A.v = (PREC == 0 ? (const T *)P.dv : (const T *)P.dv32) + r0;
        A64.v = P.dv + r0;
        A.ld = A64.ld = (size_t)P.N;
#pragma unroll
        for (int k = 0; k < ND; ++k)
          A.off[k] = A64.off[k] =
              __builtin_amdgcn_readfirstlane(P.off[(size_t)sys * XS_DIA_MAX + k]);
        if (!BIG) RS_RUN(8);
        else if (m <= 32 * RS_THREADS) RS_RUN(32);
        else RS_RUN(RS_RMAX);
      } else {
        const rs_csr<T> A{P.rp, P.ci, PREC == 0 ? (const T *)P.v : (const T *)P.v32, r0};
        const rs_csr<double> A64{P.rp, P.ci, P.v, r0};
        if (!BIG) RS_RUN(8);
        else if (m <= 32 * RS_THREADS) RS_RUN(32);
        else RS_RUN(RS_RMAX);
      }
#undef RS_RUN
    }
    if (threadIdx.x == 0) {
      P.iters[sys] = it;
      P.relres[sys] = rel;
    }
    __syncthreads();
  }
}

// Distinct column - row offsets of each system (a workgroup per system),
// ascending in off[sys * XS_DIA_MAX ..], the unused ones 0; stat[0] = the
// most that a system has, stat[1] = 1 when one has more than XS_DIA_MAX or a
// row's columns do not ascend.
__global__ __launch_bounds__(256) void k_batch_offsets(int nsys, const int *__restrict__ sys_ptr,
                                                       const int *__restrict__ rp,
                                                       const int *__restrict__ ci,
                                                       int *__restrict__ off, int *stat) {
  __shared__ int tab[XS_DIA_MAX];
  __shared__ int bad;
  const int s = blockIdx.x;
  if (threadIdx.x < XS_DIA_MAX) tab[threadIdx.x] = INT_MIN;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  for (int r = sys_ptr[s] + threadIdx.x; r < sys_ptr[s + 1]; r += 256)
    for (int e = rp[r]; e < rp[r + 1]; ++e)
      if ((e > rp[r] && ci[e] <= ci[e - 1]) || !dia_insert(tab, ci[e] - r)) {
        bad = 1;
        break;
      }
  __syncthreads();
  if (threadIdx.x != 0) return;
  int nd = 0;
  for (int a = 0; a < XS_DIA_MAX; ++a) {   // ascending insertion, free slots (INT_MIN) left out
    const int v = tab[a];
    if (v == INT_MIN) continue;
    int q = nd++;
    for (; q > 0 && off[s * XS_DIA_MAX + q - 1] > v; --q)
      off[s * XS_DIA_MAX + q] = off[s * XS_DIA_MAX + q - 1];
    off[s * XS_DIA_MAX + q] = v;
  }
  for (int a = nd; a < XS_DIA_MAX; ++a) off[s * XS_DIA_MAX + a] = 0;
  atomicMax(&stat[0], nd);
  if (bad) atomicMax(&stat[1], 1);
}

// slot k of row r = entry (r, r + off[k]) or 0 in dv[k * N + r] (FP64) and
// dv32 (FP32)
__global__ __launch_bounds__(256) void k_batch_dia(int N, const int *__restrict__ sys_ptr,
                                                   const int *__restrict__ off,
                                                   const int *__restrict__ rp,
                                                   const int *__restrict__ ci,
                                                   const double *__restrict__ v,
                                                   double *__restrict__ dv,
                                                   float *__restrict__ dv32) {
  const int s = blockIdx.x;
  int o[BT_RES_ND];
#pragma unroll
  for (int k = 0; k < BT_RES_ND; ++k) o[k] = off[s * XS_DIA_MAX + k];
  for (int r = sys_ptr[s] + threadIdx.x; r < sys_ptr[s + 1]; r += 256) {
    double slot[BT_RES_ND];
#pragma unroll
    for (int k = 0; k < BT_RES_ND; ++k) slot[k] = 0.0;
    for (int e = rp[r]; e < rp[r + 1]; ++e) {
      const int d = ci[e] - r;
      bool done = false;   // a padding slot repeats offset 0: the first match takes the entry
#pragma unroll
      for (int k = 0; k < BT_RES_ND; ++k)
        if (!done && o[k] == d) {
          slot[k] = v[e];
          done = true;
        }
    }
#pragma unroll
    for (int k = 0; k < BT_RES_ND; ++k) {
      dv[(size_t)k * N + r] = slot[k];
      dv32[(size_t)k * N + r] = (float)slot[k];
    }
  }
}

void xs_batch_offsets(hipStream_t s, int nsys, const int *sys_ptr, const int *rp, const int *ci,
                      int *off, int *stat) {
  hipLaunchKernelGGL(k_batch_offsets, dim3(nsys), dim3(256), 0, s, nsys, sys_ptr, rp, ci, off, stat);
}

void xs_batch_dia(hipStream_t s, int nsys, int N, const int *sys_ptr, const int *off,
                  const int *rp, const int *ci, const double *v, double *dv, float *dv32) {
  hipLaunchKernelGGL(k_batch_dia, dim3(nsys), dim3(256), 0, s, N, sys_ptr, off, rp, ci, v, dv,
                     dv32);
}

__global__ void k_batch_prep(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                             const double *__restrict__ v, double *__restrict__ dinv,
                             float *__restrict__ dinv32, float *__restrict__ v32, int *bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double d = 0.0;
  for (int e = rp[i]; e < rp[i + 1]; ++e) {
    if (ci[e] == i) d = v[e];
    if (v32) v32[e] = (float)v[e];
  }
  if (d == 0.0) atomicMin(bad, i + 1);
  dinv[i] = 1.0 / d;
  dinv32[i] = (float)(1.0 / d);
}

// FP64 Jacobi set-up only (1/a_ii; a zero or missing diagonal gives inf,
// which the CG turns into a non-finite relres for that system), and the three
// work-queue counters cleared by the same launch (thread 0), so a caller
// under graph capture records kernels only.
__global__ void k_batch_prep64(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                               const double *__restrict__ v, double *__restrict__ dinv,
                               unsigned *queue) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3) queue[i] = 0u;
  if (i >= n) return;
  double d = 0.0;
  for (int e = rp[i]; e < rp[i + 1]; ++e)
    if (ci[e] == i) d = v[e];
  dinv[i] = 1.0 / d;
}

void xs_batch_prep64(hipStream_t s, int n, const int *rp, const int *ci, const double *v,
                     double *dinv, unsigned *queue) {
  hipLaunchKernelGGL(k_batch_prep64, dim3((n + 255) / 256), dim3(256), 0, s, n, rp, ci, v, dinv,
                     queue);
}

void xs_batch_prep(hipStream_t s, int n, const int *rp, const int *ci, const double *v,
                   double *dinv, float *dinv32, float *v32, int *bad) {
  hipLaunchKernelGGL(k_batch_prep, dim3((n + 255) / 256), dim3(256), 0, s, n, rp, ci, v, dinv,
                     dinv32, v32, bad);
}

// LDS of k_batch_res for systems of at most maxrows rows
static size_t res_lds(int maxrows, size_t es) {
  size_t rows = ((size_t)maxrows + RS_THREADS - 1) / RS_THREADS * RS_THREADS;
  if (es == 8 && rows > RS_LDS_ROWS) rows = RS_LDS_ROWS;
  return rows * es;
}

template <int PREC, int ND, int BIG>
static bool res_launch(hipStream_t s, int grid, int nsys, int minrows, int maxrows, size_t lds,
                       const xs_batch_args &P) {
  if (lds > 65536 &&
      hipFuncSetAttribute(reinterpret_cast<const void *>(&k_batch_res<PREC, ND, BIG>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return false;
  hipLaunchKernelGGL((k_batch_res<PREC, ND, BIG>), dim3(grid), dim3(RS_THREADS), lds, s, nsys,
                     minrows, maxrows, P);
  return true;
}

template <int PREC, int ND>
static bool res_launch(hipStream_t s, int grid, int nsys, int minrows, int maxrows,
                       const xs_batch_args &P) {
  const size_t lds = res_lds(maxrows, PREC == 0 ? 8 : 4);
  return maxrows <= BT_RES_SMALL ? res_launch<PREC, ND, 0>(s, grid, nsys, minrows, maxrows, lds, P)
                                 : res_launch<PREC, ND, 1>(s, grid, nsys, minrows, maxrows, lds, P);
}

bool xs_batch_res(hipStream_t s, int grid, int nsys, int minrows, int maxrows, int precision,
                  const xs_batch_args &P) {
  if (nsys <= 0) return true;
  if (maxrows > BT_RES_ROWS) maxrows = BT_RES_ROWS;
#define RS_GO(ND_) (precision == 0 ? res_launch<0, ND_>(s, grid, nsys, minrows, maxrows, P) \
                                   : res_launch<1, ND_>(s, grid, nsys, minrows, maxrows, P))
  return P.dv ? RS_GO(BT_RES_ND) : RS_GO(0);
#undef RS_GO
}

void xs_batch_cg(hipStream_t s, int grid, int nsys, int minrows, int precision,
                 const xs_batch_args &P) {
  if (nsys <= 0) return;
#define BT_GO(PR)                                                                              \
  hipLaunchKernelGGL(k_batch_cg<PR>, dim3(grid), dim3(BT_THREADS), 0, s, nsys, P.N, P.nnz,     \
                     minrows, P.order, P.sys_ptr, P.rp, P.ci, P.v, P.v32, P.dinv, P.dinv32,    \
                     P.b, P.x, P.w64, P.w32, P.tol, P.maxiter, P.inner_tol, P.queue, P.iters,  \
                     P.relres)
  if (precision == 0) BT_GO(0);
  else BT_GO(1);
#undef BT_GO
}
