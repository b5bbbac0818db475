// xs_cgres.h -- CG solve in one launch (xs_cgres.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "xs_internal.h"

#define CR_MAX_WG 256
#define CR_LDS_MAX (150 * 1024)   // LDS window of p: own rows and halo

struct xs_cgres_args {
  int n = 0, ld = 0, nd = 0, reach = 0;   // reach: largest |column - row|
  xs_dia_offs off{};
  const double *dv = nullptr;     // diagonal slots, nd slabs of ld values
  const double *dinv = nullptr;   // 1/a_ii, null = no preconditioner
  const double *b = nullptr;
  double *x = nullptr;            // x0 in, solution out
  double tol = 0.0, abstol = 0.0;
  int maxiter = 0;
  xs_state *st = nullptr;         // S_RES0, S_RESL, iter, done
  double *resvec = nullptr;
  unsigned *err = nullptr;        // raised if a wait expires
  unsigned long long *slots = nullptr;   // 8 CR_MAX_WG words, then z
  unsigned long long *z = nullptr;       // slots + 8 CR_MAX_WG: 2 words per row
};
// words of the exchange buffer for a system of n rows; 0: not for this kernel
size_t xs_cgres_words(int n, int reach);
// the whole solve: its workgroups, or 0 when the system or the device does
// not allow it (nothing has been launched that touches x)
int xs_cgres(hipStream_t s, const xs_cgres_args &A);
