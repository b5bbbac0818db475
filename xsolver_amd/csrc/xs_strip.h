// xs_strip.h -- triangular solves over chains of row groups (xs_strip.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#define ST_MAX_WAVES 8  // chains (waves) per workgroup, at most: 4 or 8
#define ST_RING 32      // steps whose values a wave keeps in LDS
#define ST_MAXQ 3       // entries of a row outside its group, at most

// Source of an entry's value, one int: a code >= 0 names a value of the same
// workgroup's chains, its place in their rings ((wave * ST_RING + step %
// ST_RING) * 64 + lane) and, from ST_STEP_SHIFT, its step; ST_NONE: no entry;
// ST_PREV: this lane's value of the step before; ST_IDLE (of the first entry):
// no row in this lane; any other negative code c: row ~c, read from memory.
#define ST_NONE 0x7fffffff
#define ST_PREV 0x7ffffffe
#define ST_IDLE (-2147483647 - 1)
#define ST_STEP_SHIFT 14                                 // ring places fit below
#define ST_MAX_STEPS ((1 << (31 - ST_STEP_SHIFT)) - 1)   // the last names no step
#define ST_SEQ_SHIFT 9                                   // a place's wave times four
#define ST_LDS 4               // from this bit of carry's second: entries of the workgroup's other chains
#define ST_MEM 8               // and entries read from memory
#define ST_MAX_ROWS (1 << 28)  // 32-bit byte offsets
static_assert(ST_RING * 64 == 1 << (ST_SEQ_SHIFT + 2) && ST_MAX_WAVES * ST_RING * 64 <= 1 << ST_STEP_SHIFT &&
              (ST_MAX_WAVES & (ST_MAX_WAVES - 1)) == 0, "code layout");

// A code's ring place and the step counter of its wave as byte offsets into
// the LDS arrays of a workgroup of W waves.  Codes that name no ring place
// (their values are not used) give places in the arrays too: a step reads them
// for all its lanes.
template <int W>
__host__ __device__ constexpr unsigned st_ring_byte(int code) {
  return ((unsigned)code << 3) & (W * ST_RING * 64 * 8 - 1);
}
template <int W>
__host__ __device__ constexpr unsigned st_seq_byte(int code) {
  return ((unsigned)code >> ST_SEQ_SHIFT) & ((W - 1) * 4);
}

// One triangle.  Positions count along the solve (L: rows ascending, U:
// descending).  Chain c owns the slots [cptr[c], cptr[c + 1]), a group of at
// most 64 consecutive positions each, base + step * stride the first.
struct xs_strip {
  int n = 0, Q = 0, nchains = 0, nslots = 0, stride = 0, waves = 0;
  bool ready = false, tried = false, vals = false;   // pattern built / refused; values current
  int *cptr = nullptr;     // nchains + 1
  int *cbase = nullptr;    // first position of each chain
  // per slot and lane: Q codes; Q values and the coefficient of the position
  // before.  carry[slot]: source of the position before a group that continues
  // the chain of rows across a group boundary (ST_NONE: none); its place among
  // lane 0's entries, with the bits from ST_LDS on.
  int *code = nullptr;
  int2 *carry = nullptr;
  double *val = nullptr;
  int *vpos = nullptr;     // where the values sit in the factor (-1: 0)
};

// Host analysis of a triangle's pattern: groups (maximal runs of positions
// that each depend on the one before, cut at 64), their chains, and whether
// the solve can run over them.  False: the general solve is used.
struct xs_strip_plan {
  int Q = 0, stride = 0;
  std::vector<int> gstart;            // first position of each group, then n
  std::vector<int> gchain, gstep;     // chain and step of each group
  std::vector<int> cptr, cbase;
};
bool xs_strip_analyse(int n, const int *rp, const int *ci, const int *dpos, bool upper,
                      xs_strip_plan &P);

void xs_strip_free(xs_strip &S);
// device arrays from the plan (rp, ci, dpos: the pattern on the device);
// 0 = built, else a status of the C interface
int xs_strip_build(hipStream_t s, int n, const int *rp, const int *ci, const int *dpos, bool upper,
                   const xs_strip_plan &P, xs_strip &S);
void xs_strip_values(hipStream_t s, const double *lu, xs_strip &S);
// x = T^-1 b; x holds the sentinel in every entry (xs_fill_sentinel); dinv
// null: unit diagonal.  The bits of k_trsv's scan path.
void xs_strip_solve(hipStream_t s, const xs_strip &S, bool upper, const double *dinv,
                    const double *b, double *x, unsigned *tickets, const struct xs_state *st);
