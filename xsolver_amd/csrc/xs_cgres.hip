// xs_cgres.hip -- CG with Jacobi (or no) preconditioner on a matrix with few
// diagonals, the whole solve in one launch.
//
// What bounds the launch-per-kernel loop on such systems: three kernels per
// iteration whose work takes a fraction of a launch (256 x 256 rows, 5
// points: 16.7 us per iteration, 14.5 of them inside kernels that move 4 MB
// of cached data).  Measured against it, us per iteration: 33 x 33 rows 15.9
// -> 2.5, 256 x 256 15.7 -> 5.8, 512 x 512 18.1 -> 7.7, 1000 x 1000 33 -> 16.
// What is left is, in one workgroup, the barriers, reductions and divisions of
// an iteration, and beyond that the two round trips between workgroups.  Here
// every workgroup owns a run of consecutive rows and
// keeps them for the whole solve: the matrix's diagonal slots, 1/a_ii, x, r
// and q in registers (R rows per thread), p in LDS together with the p of the
// rows within the matrix's reach on both sides (the halo).  Up to 512 R rows
// fit one workgroup, and nothing crosses workgroups; larger systems run on a
// cooperative grid and meet twice per iteration, in the two inner products.
//
// Exchange between workgroups: every 8-byte word carries half of a value and
// the sequence number of the exchange, written and polled with relaxed
// agent-scope atomics, so a word says by itself whether it is the awaited one:
// no fence, no flag beside the data, no reset.  A word is overwritten at the
// earliest by the exchange after the next one of the other kind, which its
// writer enters only after every reader has answered with a value computed
// from it.  The inner products are summed from all workgroups' partials by
// every workgroup in the same order, so all hold the same scalars and stop at
// the same iteration; the halo's p is updated from the owners' z by the same
// operations as the owners', so both hold the same bits.
// Waits are bounded (XS_SPIN_LIMIT): past the limit the flag is raised and NaN
// is used, which ends every workgroup's loop.
//
// Sums of a row in slot (column) order as k_spmv_dia; the recurrence is
// hip/Solver/xsolver_cg.cpp:16-74.
#include "xs_device.h"
#include "xs_cgres.h"

#define CR_THREADS 512
#define CR_WAVES (CR_THREADS / XS_WAVE)
static_assert(CR_MAX_WG * 2 <= CR_THREADS, "one thread polls one partial");

// total of the wave's values in every lane (cross-lane adds on the DPP path)
__device__ __forceinline__ double cr_wave_total(double v) {
  v += dpp_d<0x111, 0xF>(v, 0.0);   // row_shr:1, 2, 4, 8
  v += dpp_d<0x112, 0xF>(v, 0.0);
  v += dpp_d<0x114, 0xF>(v, 0.0);
  v += dpp_d<0x118, 0xF>(v, 0.0);
  v += dpp_d<0x142, 0xA>(v, 0.0);   // row_bcast:15, row_bcast:31
  v += dpp_d<0x143, 0xC>(v, 0.0);
  return wave_readlane_f64(v, XS_WAVE - 1);
}

__device__ __forceinline__ void cr_store(unsigned long long *w, double v, unsigned tag) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned long long t = (unsigned long long)tag << 32;
  __hip_atomic_store(w, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(w + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long cr_load(const unsigned long long *w) {
  return __hip_atomic_load(const_cast<unsigned long long *>(w), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
// the value with that sequence number, polled for; a, b: the words as loaded
// before
__device__ __forceinline__ double cr_wait(const unsigned long long *w, unsigned tag, unsigned *err,
                                          unsigned long long a, unsigned long long b) {
  unsigned polls = 0;
  for (;;) {
    if ((unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag)
      return __longlong_as_double((long long)((b << 32) | (a & 0xffffffffull)));
    if (++polls > XS_SPIN_LIMIT) {
      atomicOr(err, 1u);
      return __longlong_as_double(0x7FF8000000000000ll);
    }
    a = cr_load(w);
    b = cr_load(w + 1);
  }
}
__device__ __forceinline__ double cr_wait(const unsigned long long *w, unsigned tag,
                                          unsigned *err) {
  return cr_wait(w, tag, err, cr_load(w), cr_load(w + 1));
}

// ND slots (an unused one: offset 0 and zero values), R rows per thread
template <int ND, int R, bool MULTI>
__global__ __launch_bounds__(CR_THREADS, 2) void k_cg_res(const xs_cgres_args A) {
  extern __shared__ __align__(16) double cr_p[];   // p of the rows [r0 - B, r0 + 512 R + B)
  __shared__ double part[2][CR_WAVES][2];
  const int t = threadIdx.x, w = t / XS_WAVE, lane = t & (XS_WAVE - 1);
  const int n = A.n, B = A.reach, rows = CR_THREADS * R;
  const int r0 = (int)blockIdx.x * rows, m = min(rows, n - r0);
  unsigned seq = 0;
  // sums of two values over the grid (MULTI: slot pair of this exchange);
  // ahead(): called between sending the partials and waiting for the others'
  auto sum2 = [&](double &a, double &b, auto &&ahead) {
    a = cr_wave_total(a);
    b = cr_wave_total(b);
    if (lane == 0) { part[0][w][0] = a; part[0][w][1] = b; }
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int q = 0; q < CR_WAVES; ++q) { a += part[0][q][0]; b += part[0][q][1]; }
    if (!MULTI) {
      __syncthreads();   // part is written again by the next sum
      return;
    }
    ++seq;
    unsigned long long *slots = A.slots + (seq & 1) * (CR_MAX_WG * 4);
    const int G = (int)gridDim.x;
    if (t == 0) {
      cr_store(slots + 2 * blockIdx.x, a, seq);
      cr_store(slots + 2 * (CR_MAX_WG + blockIdx.x), b, seq);
    }
    // thread g of the lower (upper) half takes the first (second) value of
    // workgroup g
    const int g = t & (CR_THREADS / 2 - 1), half = t / (CR_THREADS / 2);
    const unsigned long long *slot = slots + 2 * (half * CR_MAX_WG + g);
    unsigned long long pa = 0, pb = 0;
    if (g < G) {
      pa = cr_load(slot);
      pb = cr_load(slot + 1);
    }
    ahead();
    double v = g < G ? cr_wait(slot, seq, A.err, pa, pb) : 0.0;
    v = cr_wave_total(v);
    if (lane == 0) part[1][w][0] = v;
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int q = 0; q < CR_WAVES / 2; ++q) {
      a += part[1][q][0];
      b += part[1][CR_WAVES / 2 + q][0];
    }
  };
  // the halo's p: p_j <- z_j + beta p_j (first: z_j) from the owners' z.  The
  // words of a thread's first halo row are asked for while the sum of the
  // partials is waited for (halo_ahead): the owners sent them before.
  unsigned long long ha = 0, hb = 0;
  auto halo_row = [&](int h, int &l) -> int {   // window position and row, -1: outside
    l = h < B ? h : h + rows;
    const int j = r0 - B + l;
    return h < 2 * B && j >= 0 && j < n ? j : -1;
  };
  auto halo_ahead = [&]() {
    int l;
    const int j = halo_row(t, l);
    if (j >= 0) {
      ha = cr_load(A.z + 2 * (size_t)j);
      hb = cr_load(A.z + 2 * (size_t)j + 1);
    }
  };
  auto halo = [&](double beta, bool first, unsigned tag) {
    if (!MULTI) return;
    for (int h = t; h < 2 * B; h += CR_THREADS) {
      int l;
      const int j = halo_row(h, l);
      if (j < 0) continue;                      // stays 0
      const unsigned long long *zw = A.z + 2 * (size_t)j;
      const double z = h == t ? cr_wait(zw, tag, A.err, ha, hb) : cr_wait(zw, tag, A.err);
      cr_p[l] = first ? z : fma(beta, cr_p[l], z);
    }
  };
  auto nothing = [] {};
  auto publish = [&](int i, double z, unsigned tag) {   // rows that some halo holds
    if (MULTI && (i < B || i >= rows - B)) cr_store(A.z + 2 * (size_t)(r0 + i), z, tag);
  };

  double a[R][ND], di[R], x[R], r[R], q[R];
  int off[ND];
#pragma unroll
  for (int e = 0; e < ND; ++e) off[e] = e < A.nd ? A.off.o[e] : 0;
  for (int l = t; l < rows + 2 * B; l += CR_THREADS) cr_p[l] = 0.0;
  __syncthreads();
  // r = b - A x0, z = D^-1 r
  double tau = 0.0, rr = 0.0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * CR_THREADS, row = r0 + i;
    x[k] = r[k] = q[k] = 0.0;
    di[k] = 0.0;
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < ND; ++e) {
      a[k][e] = (i < m && e < A.nd) ? A.dv[(size_t)e * A.ld + row] : 0.0;
      if (i < m) s = fma(a[k][e], A.x[min(max(row + off[e], 0), n - 1)], s);
    }
    if (i < m) {
      di[k] = A.dinv ? A.dinv[row] : 1.0;
      x[k] = A.x[row];
      r[k] = A.b[row] - s;
      const double z = di[k] * r[k];
      q[k] = z;
      cr_p[B + i] = z;
      publish(i, z, 1u);
      tau += r[k] * z;
      rr += r[k] * r[k];
    }
  }
  sum2(tau, rr, halo_ahead);
  const double res0 = sqrt(rr);
  double resl = res0;
  int done = 0, it = 0;
  if (!isfinite(res0)) done = 2;
  else if (res0 == 0.0 || res0 <= A.abstol) done = 1;
  const bool lead = blockIdx.x == 0 && t == 0;
  if (lead && A.resvec) A.resvec[0] = res0;
  if (!done) halo(0.0, true, 1u);
  __syncthreads();
  while (!done && it < A.maxiter) {
    double sigma = 0.0, none = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int i = B + t + k * CR_THREADS;
      double s = 0.0;
#pragma unroll
      for (int e = 0; e < ND; ++e) s = fma(a[k][e], cr_p[i + off[e]], s);
      q[k] = s;
      sigma += cr_p[i] * s;   // rows past the end: p and the slots are 0
    }
    sum2(sigma, none, nothing);
    const double alpha = tau / sigma;
    double tn = 0.0;
    rr = 0.0;
    ++it;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int i = t + k * CR_THREADS;
      x[k] = fma(alpha, cr_p[B + i], x[k]);
      r[k] = fma(-alpha, q[k], r[k]);
      const double z = di[k] * r[k];
      q[k] = z;
      if (i < m) publish(i, z, (unsigned)it + 1u);
      tn += z * r[k];
      rr += r[k] * r[k];
    }
    sum2(tn, rr, halo_ahead);
    resl = sqrt(rr);
    if (lead && A.resvec) A.resvec[it] = resl;
    if (!isfinite(resl)) done = 2;
    else if (resl / res0 < A.tol || resl <= A.abstol) done = 1;
    if (done) break;
    const double beta = tn / tau;
    tau = tn;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int i = B + t + k * CR_THREADS;
      cr_p[i] = fma(beta, cr_p[i], q[k]);
    }
    halo(beta, false, (unsigned)it + 1u);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * CR_THREADS;
    if (i < m) A.x[r0 + i] = x[k];
  }
  if (lead) {
    A.st->sc[S_RES0] = res0;
    A.st->sc[S_RESL] = resl;
    A.st->iter = it;
    A.st->done = done;
  }
}

__global__ void k_cr_clear(unsigned long long *p, size_t len) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < len;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0ull;
}

// Rows per thread and workgroups.  One workgroup up to 4096 rows: nothing
// crosses workgroups (64 x 63 rows: 2.6 us per iteration; 64 x 65 rows in 5
// workgroups: 4.2).  Beyond, few workgroups: an exchange costs more the more
// workgroups poll, local work little (us per iteration with R = 2 / 4 / 8:
// 70^2 rows 4.0 / 4.1 / 4.7, 128^2 4.8 / 4.2 / 4.3, 256^2 6.6 / 6.0 / 5.8,
// 512^2 13.3 / 9.4 / 7.7).  A thread polls for its halo rows one after another,
// so a far reach costs what the launches do: the loop of kernels against one
// launch, 37^3 rows 17.0 and 9.6, 48^3 17.1 and 12.1, 64^3 18.7 and 17.0, 70^3
// (reach 4900) 22.3 and 21.5, 72^3 (5184) 22.7 and 22.9, 80^3 25.5 and 27.0,
// 86^3 27.9 and 32.0; 5000 x 30 rows 18.1 and 16.9, 7000 x 40 19.9 and 23.0.
#define CR_MAX_REACH (10 * CR_THREADS)   // 20 halo rows a thread
static_assert((8 * CR_THREADS + 2 * CR_MAX_REACH) * sizeof(double) <= CR_LDS_MAX, "the window of p");
static bool cr_shape(int n, int reach, int &R, int &G) {
  for (int r : {2, 4, 8})
    if (n <= r * CR_THREADS) { R = r; G = 1; return true; }
  if (reach > CR_MAX_REACH) return false;
  for (int r : {2, 4, 8}) {
    const int g = (n + r * CR_THREADS - 1) / (r * CR_THREADS);
    if (g <= (r < 8 ? 8 : CR_MAX_WG)) {
      R = r;
      G = g;
      return true;
    }
  }
  return false;
}

size_t xs_cgres_words(int n, int reach) {
  int R, G;
  if (!cr_shape(n, reach, R, G)) return 0;
  return CR_MAX_WG * 8 + (G > 1 ? 2 * (size_t)n : 0);
}

template <int ND, int R, bool MULTI>
static bool cr_launch(hipStream_t s, int G, const xs_cgres_args &A) {
  const size_t lds = (size_t)(R * CR_THREADS + 2 * A.reach) * sizeof(double);
  const void *f = reinterpret_cast<const void *>(&k_cg_res<ND, R, MULTI>);
  if (lds > 65536 &&
      hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return false;
  if (!MULTI) {
    hipLaunchKernelGGL((k_cg_res<ND, R, MULTI>), dim3(1), dim3(CR_THREADS), lds, s, A);
    return hipGetLastError() == hipSuccess;
  }
  // a cooperative grid: every workgroup is resident, or the launch is refused
  xs_cgres_args arg = A;
  void *args[] = {&arg};
  if (hipLaunchCooperativeKernel(f, dim3(G), dim3(CR_THREADS), args, (unsigned)lds, s) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}

int xs_cgres(hipStream_t s, const xs_cgres_args &A) {
  int R, G;
  if (!(A.dv && A.b && A.x && A.st && A.slots && A.err && A.nd > 0 && A.nd <= XS_DIA_MAX) ||
      !cr_shape(A.n, A.reach, R, G))
    return 0;
  if (G > 1) {
    const size_t len = CR_MAX_WG * 8 + 2 * (size_t)A.n;
    hipLaunchKernelGGL(k_cr_clear, dim3((unsigned)((len + 1023) / 1024)), dim3(256), 0, s, A.slots, len);
  }
#define CR_M(ND, R_) (G > 1 ? cr_launch<ND, R_, true>(s, G, A) : cr_launch<ND, R_, false>(s, 1, A))
#define CR_R(ND) (R == 2 ? CR_M(ND, 2) : R == 4 ? CR_M(ND, 4) : CR_M(ND, 8))
  return (A.nd <= 5 ? CR_R(5) : CR_R(XS_DIA_MAX)) ? G : 0;
#undef CR_R
#undef CR_M
}
