// xs_strip.hip -- exact triangular solves of narrow factors (ILU(0) of 5- and
// 7-point grids) over chains of row groups.
//
// What bounds k_trsv there is one thing: a dependency between two groups of
// 64 rows costs a trip through memory at agent scope, 0.8-1 us, and a solve
// has as many of them in sequence as the group graph is deep (512 x 512 grid:
// 520 levels, 420 us; 128^3: 256 levels, 265 us; the bytes alone would take 3
// and 21 us).  Here a wave owns a chain of groups, each the neighbour of the
// last at one fixed distance (a column block of a 2D grid from line to line,
// a line of a 3D grid from plane to plane), and a workgroup the chains next
// to each other:
//  * the value a row needs from its own chain's last group is in a register;
//  * values of the other chains of the workgroup pass through LDS: a wave
//    writes the group it solved into its ring of ST_RING groups, then its step
//    counter, and a reader takes the counter, the value and the counter again
//    (LDS operations of a wave run in order): the first must be past the step,
//    the second not yet where the ring place is written again -- if it is, the
//    value is read from memory, where every row is also published;
//  * only values from other workgroups go through memory, asked for two steps
//    ahead; what does not depend on other rows is asked for eight steps ahead.
// A step is then bound by its own instructions (178 of a wave by the counters,
// 107 of them VALU, and an LDS round trip: 0.52 us), not by a memory access.  L
// of a 512 x 512 grid 421 -> 270 us, 1000 x 1000 871 -> 526, 64 x 64 56 -> 33;
// of a 7-point grid 128^3 262 -> 233, 100^3 210 -> 185, 64^3 129 -> 96, 24^3
// 290 -> 37.
// Chains depend on lower chains only (checked when the chains are formed) and
// workgroups take them in that order by ticket, so the earliest unfinished
// chain never waits: every wait ends.  Waits are bounded as in k_trsv.
//
// The values are those of k_trsv's scan path bit for bit: products rounded on
// their own, summed by the same tree in the same order, the affine scan
// composed over the same groups -- where the groups are the same; a group here
// ends at every row that does not depend on the one before, which only
// shortens scans of independent parts.
#include "xs_device.h"
#include "xs_strip.h"

#include "../../include/xsolver_c.h"

#include <algorithm>
#include <unordered_map>

#define ST_DEP 2     // steps ahead: values from memory
#define ST_STA 8     // steps ahead: codes, factor values, b and 1/u_ii
#define ST_PACE 12   // steps ahead of the next chain

struct st_args {
  int n, nchains, stride;
  const int *cptr, *cbase, *code;
  const int2 *carry;
  const double *val;
};

template <int Q>
struct st_static {       // a step's operands that do not depend on others
  double v[Q + 1], b, di;
  int c[Q];
  int2 cc;
};
template <int Q>
struct st_dyn {          // and those of other workgroups' rows
  unsigned long long g[Q + 1];
};

template <bool UPPER, bool DIAG, int Q, int W>
__global__ __launch_bounds__(W *XS_WAVE) void k_strip(const st_args S,
                                                             const double *__restrict__ dinv,
                                                             const double *__restrict__ b,
                                                             double *x, unsigned *tickets,
                                                             const xs_state *st) {
#pragma clang fp contract(off)
  if (st != nullptr && st->done) return;
  __shared__ double ring_[W * ST_RING * XS_WAVE];
  __shared__ int seq_[W];
  __shared__ unsigned s_ticket;
  // LDS pointers by type: volatile accesses through generic ones stay flat
  // accesses, which count as memory loads too and make every wait one for all
  // of them
  typedef __attribute__((address_space(3))) volatile double lds_double;
  typedef __attribute__((address_space(3))) volatile int lds_int;
  typedef __attribute__((address_space(3))) volatile char lds_char;
  lds_double *const ring = (lds_double *)ring_;
  lds_int *const seq = (lds_int *)seq_;
  unsigned *err = tickets + 4;
  const int lane = threadIdx.x & (XS_WAVE - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / XS_WAVE));
  if (threadIdx.x == 0) s_ticket = atomicAdd(&tickets[0], 1u);
  if (threadIdx.x < W) seq[threadIdx.x] = 0;
  __syncthreads();
  const int c = __builtin_amdgcn_readfirstlane((int)s_ticket) * W + w;
  if (c < S.nchains) {
    const int slot0 = S.cptr[c], steps = S.cptr[c + 1] - slot0, base = S.cbase[c];
    st_static<Q> sa[ST_STA];
    st_dyn<Q> dy[ST_DEP];
    // addresses as a uniform base and a 32-bit byte offset per lane
    const unsigned l8r = 8u * (UPPER ? XS_WAVE - 1 - lane : lane);
    auto at = [](const void *p, size_t uni, unsigned off) { return (const char *)p + uni + off; };
    // the step's first row (its last if UPPER)
    auto first_of = [&](int step) {
      const int p = base + step * S.stride;
      return UPPER ? S.n - XS_WAVE - p : p;
    };
    // 0, but not to the compiler: a uniform load would go to a scalar register
    // at once, by a wait for it
    unsigned vzero = 0;
    asm volatile("" : "+v"(vzero));
    auto load_static = [&](int step, st_static<Q> &z) {
      const int sn = min(step, steps - 1);
      const size_t sl = slot0 + sn;
      const char *pv = (const char *)(S.val + sl * (Q + 1) * XS_WAVE), *pc = (const char *)(S.code + sl * Q * XS_WAVE);
      if (Q == 1) {
        const double2 v2 = *(const double2 *)(pv + 16u * lane);
        z.v[0] = v2.x;
        z.v[Q] = v2.y;
        z.c[0] = *(const int *)(pc + 4u * lane);
      } else if (Q == 3) {
        const double2 va = *(const double2 *)(pv + 32u * lane), vb = *(const double2 *)(pv + 32u * lane + 16u);
        z.v[0] = va.x; z.v[1] = va.y; z.v[2 % (Q + 1)] = vb.x; z.v[Q] = vb.y;
#pragma unroll
        for (int e = 0; e < Q; ++e) z.c[e] = *(const int *)(pc + 4u * (Q * lane + e));
      } else {
#pragma unroll
        for (int e = 0; e <= Q; ++e) z.v[e] = *(const double *)(pv + 8u * ((Q + 1) * lane + e));
        const int2 c2 = *(const int2 *)(pc + 8u * lane);
        z.c[0] = c2.x;
        z.c[Q - 1] = c2.y;
      }
      z.cc = *(const int2 *)((const char *)(S.carry + sl) + vzero);
      // lanes past the group read other rows' values, never used
      const unsigned r = 8u * (unsigned)min(max(first_of(sn) + (UPPER ? XS_WAVE - 1 - lane : lane), 0), S.n - 1);
      z.b = *(const double *)at(b, 0, r);
      z.di = DIAG ? *(const double *)at(dinv, 0, r) : 1.0;
    };
    auto load_dyn = [&](const st_static<Q> &z, st_dyn<Q> &d) {
      // a code's row when its value comes from memory
#pragma unroll
      for (int e = 0; e <= Q; ++e) {
        const int cd = e < Q ? z.c[e < Q ? e : 0] : z.cc.x;
        if (cd < 0 && cd != ST_IDLE) d.g[e] = ld_relaxed((const double *)at(x, 0, 8u * (unsigned)~cd));
      }
    };
    double xprev = 0.0;
    // The next chain's length, for the pace below (0: there is none here).
    const int next = w + 1 < W && c + 1 < S.nchains ? S.cptr[c + 2] - S.cptr[c + 1] : 0;
    auto solve = [&](int step, const st_static<Q> &z, st_dyn<Q> &d) {
      const int behind = seq[(w + 1) & (W - 1)];
      const bool live = step < steps, act = z.c[0] != ST_IDLE && live;   // live: uniform
      int code[Q + 1];
      double val[Q + 1];
#pragma unroll
      for (int e = 0; e < Q; ++e) {
        code[e] = act ? z.c[e] : ST_NONE;
        val[e] = z.v[e];
      }
      code[Q] = lane == 0 && live ? z.cc.x : ST_NONE;
      val[Q] = z.v[Q];
      // Values that are there: the whole step runs without a branch and waits
      // for no load but its own.  (Only the path below touches registers that
      // a load ahead may still be filling.)
      double xv[Q + 1];
      bool ok = true;
      // (a code that names no ring place reads one all the same)
      auto take = [&](int cd, int &ps, double &v, int &f1, int &f2) {
        lds_int *const sq = (lds_int *)((lds_char *)seq + st_seq_byte<W>(cd));
        lds_double *const rg = (lds_double *)((lds_char *)ring + st_ring_byte<W>(cd));
        ps = cd >> ST_STEP_SHIFT;
        f1 = *sq;
        v = *rg;
        f2 = *sq;
        return cd >= 0 && cd < ST_PREV;
      };
      const int kind = live ? __builtin_amdgcn_readfirstlane(z.cc.y) : 0;
#pragma unroll
      for (int e = 0; e <= Q; ++e) {
        xv[e] = xprev;
        if (kind >> (ST_LDS + e) & 1) {   // uniform, as the next
          int ps, f1, f2;
          double v;
          const bool lds = take(code[e], ps, v, f1, f2);
          xv[e] = lds ? v : xv[e];
          const bool there = ((int)(f1 > ps) & (int)(f2 < ps + ST_RING)) != 0;
          ok = ((int)ok & ((int)(!lds) | (int)there)) != 0;
        }
        if (kind >> (ST_MEM + e) & 1) {
          const bool mem = code[e] < 0, got = d.g[e] != XS_SENTINEL;
          xv[e] = mem ? __longlong_as_double((long long)d.g[e]) : xv[e];
          ok = ((int)ok & ((int)(!mem) | (int)got)) != 0;
        }
      }
      if (!__all(ok)) {
        // Values of this workgroup's chains first: nothing here waits for a
        // memory access, so a chain close behind its neighbour loses an LDS
        // round trip and no more.
        unsigned polls = 0;
        unsigned over = 0;   // a bit per entry whose ring place is (being) written again
        for (;;) {
          bool late = false;
#pragma unroll
          for (int e = 0; e <= Q; ++e) {
            int ps, f1, f2;
            double v;
            const bool lds = take(code[e], ps, v, f1, f2);
            const bool there = lds && f1 > ps, kept = f2 < ps + ST_RING;
            xv[e] = there && kept ? v : xv[e];
            over |= there && !kept ? 1u << e : 0u;
            late |= lds && !there;
          }
          if (!__any(late)) break;
          if (++polls > XS_SPIN_LIMIT) {   // bounded: flag it, continue with NaN
            if (late) atomicOr(err, 1u);
#pragma unroll
            for (int e = 0; e <= Q; ++e)
              if (late && code[e] >= 0 && code[e] < ST_PREV) xv[e] = __longlong_as_double(0x7FF8000000000000ll);
            break;
          }
        }
        unsigned wait = over;
#pragma unroll
        for (int e = 0; e <= Q; ++e)
          if ((kind >> (ST_MEM + e) & 1) && code[e] < 0 && d.g[e] == XS_SENTINEL) wait |= 1u << e;
        if (__any((int)wait)) {
          // what comes from memory: rows of other workgroups, overrun places
          int row[Q + 1];
#pragma unroll
          for (int e = 0; e <= Q; ++e) {
            row[e] = ~code[e];
            if ((over >> e) & 1u) {
              const int cp = (c & ~(W - 1)) + (code[e] / (ST_RING * XS_WAVE) & (W - 1));
              const int p = S.cbase[cp] + (code[e] >> ST_STEP_SHIFT) * S.stride + (code[e] & (XS_WAVE - 1));
              row[e] = UPPER ? S.n - 1 - p : p;
            }
          }
          polls = 0;
          for (;;) {
            unsigned long long u[Q + 1];
#pragma unroll
            for (int e = 0; e <= Q; ++e) u[e] = (wait >> e) & 1u ? ld_relaxed(x + row[e]) : 0ull;
#pragma unroll
            for (int e = 0; e <= Q; ++e)
              if (((wait >> e) & 1u) && u[e] != XS_SENTINEL) {
                xv[e] = __longlong_as_double((long long)u[e]);
                wait &= ~(1u << e);
              }
            if (!__any((int)wait)) break;
            if (++polls > XS_SPIN_LIMIT) {
              if (wait) atomicOr(err, 1u);
#pragma unroll
              for (int e = 0; e <= Q; ++e)
                if ((wait >> e) & 1u) xv[e] = __longlong_as_double(0x7FF8000000000000ll);
              break;
            }
          }
        }
      }
      // the products in solve order and k_trsv's sum of a batch of four
      double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int e = 0; e < Q; ++e) p[e] = code[e] != ST_NONE ? val[e] * xv[e] : 0.0;
      // the carry: last, or in the place of a third entry that lane 0 lacks
      // (elsewhere its place changes no sum)
      const double pc = code[Q] != ST_NONE ? val[Q] * xv[Q] : 0.0;
      const bool third = Q == 3 && (kind & 3) == 2 && code[Q] != ST_NONE;
      if (Q == 3) p[2] = third ? pc : p[2];
      p[Q] = third ? 0.0 : pc;
      const double acc = (act ? z.b : 0.0) - ((p[0] + p[2]) + (p[1] + p[3]));
      double cv[1] = {act ? z.di * acc : 0.0};
      double m = act && lane > 0 ? -z.di * z.v[Q] : 0.0;
      wave_affine_scan<1>(cv, m);
      xprev = cv[0];
      if (live) {
        ring[(w * ST_RING + (step & (ST_RING - 1))) * XS_WAVE + lane] = xprev;
        if (lane == 0) seq[w] = step + 1;
      }
      if (act) st_ready((double *)const_cast<char *>(at(x, 0, 8u * (unsigned)first_of(step) + l8r)), xprev);
      // A chain with less to do than the next runs away from it, and the next
      // would find the ring overrun and read memory from then on.  So a chain
      // far ahead loses a little time; it never waits for what comes after it.
      if (min(step, next) > behind + ST_PACE)
        for (int t = 0; t < 4 && min(step, next) > seq[(w + 1) & (W - 1)] + ST_PACE; ++t)
          __builtin_amdgcn_s_sleep(2);
    };
#pragma unroll
    for (int k = 0; k < ST_STA - ST_DEP; ++k) load_static(k, sa[k]);
    // in the loop's order, so that its waits count the same loads on entry
#pragma unroll
    for (int k = 0; k < ST_DEP; ++k) {
      load_dyn(sa[k], dy[k]);
      load_static(k + ST_STA - ST_DEP, sa[k + ST_STA - ST_DEP]);
    }
    // whole blocks of steps, those past the end as if idle: a way out in the
    // middle would have the waits of all the others count its loads
    for (int s0 = 0; s0 < steps; s0 += ST_STA) {
#pragma unroll
      for (int k = 0; k < ST_STA; ++k) {
        const int step = s0 + k;
        solve(step, sa[k], dy[k % ST_DEP]);
        load_dyn(sa[(k + ST_DEP) % ST_STA], dy[k % ST_DEP]);
        load_static(step + ST_STA, sa[k]);
      }
    }
  }
  trsv_retire(tickets);
}

// slots of the triangle: a wave per slot
template <bool UPPER>
__global__ __launch_bounds__(256) void k_strip_fill(int n, int Q, int nslots, int waves,
                                                    const int *__restrict__ rp,
                                                    const int *__restrict__ ci,
                                                    const int *__restrict__ dpos,
                                                    const int *__restrict__ sgroup,
                                                    const int *__restrict__ gstart,
                                                    const int *__restrict__ gchain,
                                                    const int *__restrict__ gstep,
                                                    const int *__restrict__ grp,
                                                    int *__restrict__ code, int *__restrict__ vpos,
                                                    int2 *__restrict__ carry) {
  const int slot = blockIdx.x * (256 / XS_WAVE) + threadIdx.x / XS_WAVE;
  const int lane = threadIdx.x & (XS_WAVE - 1);
  if (slot >= nslots) return;
  const int g = sgroup[slot], p0 = gstart[g], len = gstart[g + 1] - p0, c = gchain[g];
  const int p = p0 + lane;
  int mp = -1, cc = ST_NONE, kk = 0, e = 0;
  unsigned lds = 0, mem = 0;   // entries of other chains
  // entry t of the row in solve order
  const int r = UPPER ? n - 1 - p : p;
  int cnt = 0, e0 = 0;
  if (lane < len) {
    e0 = UPPER ? rp[r + 1] - 1 : rp[r];
    cnt = UPPER ? rp[r + 1] - 1 - dpos[r] : dpos[r] - rp[r];
  }
  auto source = [&](int q) {   // position q's value
    const int gq = grp[q], cq = gchain[gq], sq = gstep[gq], lq = q - gstart[gq];
    if (cq == c && sq == gstep[g] - 1 && lq == lane) return ST_PREV;
    if (cq / waves == c / waves) return ((cq % waves) * ST_RING + (sq & (ST_RING - 1))) * XS_WAVE + lq | sq << ST_STEP_SHIFT;
    return ~(UPPER ? n - 1 - q : q);
  };
  for (int t = 0; t < cnt; ++t) {
    const int f = UPPER ? e0 - t : e0 + t;
    const int q = UPPER ? n - 1 - ci[f] : ci[f];
    if (q == p - 1 && (lane > 0 || t == cnt - 1)) {
      // the position before: inside the group the scan's, for lane 0 the
      // carry from the group it continues
      mp = f;
      if (lane == 0) { cc = source(q); kk = e; }
    } else if (e < Q) {
      const int cd = source(q);
      if (cd < 0) mem |= 1u << e;
      else if (cd != ST_PREV) lds |= 1u << e;
      code[((size_t)slot * XS_WAVE + lane) * Q + e] = cd;
      vpos[((size_t)slot * XS_WAVE + lane) * (Q + 1) + e] = f;
      ++e;
    }
  }
  for (; e < Q; ++e) {
    code[((size_t)slot * XS_WAVE + lane) * Q + e] = lane < len || e > 0 ? ST_NONE : ST_IDLE;
    vpos[((size_t)slot * XS_WAVE + lane) * (Q + 1) + e] = -1;
  }
  vpos[((size_t)slot * XS_WAVE + lane) * (Q + 1) + Q] = mp;
  for (int k = 0; k < Q; ++k) {
    if (__any((int)(lds >> k & 1u))) kk |= 1 << (ST_LDS + k);
    if (__any((int)(mem >> k & 1u))) kk |= 1 << (ST_MEM + k);
  }
  if (cc != ST_NONE && cc != ST_PREV) kk |= 1 << (cc < 0 ? ST_MEM + Q : ST_LDS + Q);
  if (lane == 0) carry[slot] = make_int2(cc, kk);
}

__global__ __launch_bounds__(256) void k_strip_vals(size_t len, const int *__restrict__ pos,
                                                    const double *__restrict__ lu,
                                                    double *__restrict__ out) {
  const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
  if (i < len) out[i] = pos[i] >= 0 ? lu[pos[i]] : 0.0;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
// Chains pay off where the groups are wide (a wave's lanes) and the chains
// long (what they replace): 64 x 64 and 24^3 grids, whose groups have 64 and
// 24 lanes, run 1.7 and 8 times as fast as by k_trsv (33 against 56 us, 37
// against 291).  A matrix without such a structure keeps k_trsv.
#define ST_MIN_GROUP 16
#define ST_MIN_CHAIN 8
// On 3D grids whose lines are blocks of several groups, the chains of a line
// fill half a workgroup or more, and a value passes through memory every line
// or two; k_trsv has no more levels than lines, planes and blocks of a line.
// Unless there are many lines, that is less (us, k_trsv against chains): 200 x
// 20 x 20 48 and 52, 320 x 12 x 12 32 and 37, 256 x 40 x 40 91 and 95, 500 x 30
// x 30 80 and 89, 320 x 64 x 64 147 and 157, 200 x 80 x 80 180 and 185; 256 x
// 100 x 20 119 and 111, 200 x 128 x 50 196 and 179, 200^3 782 and 517; with
// three blocks 130 x 20 x 20 47.3 and 46.9, 150 x 40 x 40 91 and 85, 160^3 423
// and 330.  (It loses where a line ends in a group of one row, which it runs
// together with the next line's: 257 x 40 x 40 169 and 101.)
#define ST_LINE_BLOCKS 4
#define ST_MIN_LINES 90
// A workgroup of four chains has a SIMD for each; one of eight has half as many
// places where a value goes through memory (about 2.5 us later) instead of
// LDS.  L by four and by eight, us: 512 x 512 grid (8 chains of 512 steps) 270
// and 294, 1000 x 1000 (16 of 1000) 526 and 581; 128^3 (256 of 128) 272 and
// 233, 100^3 216 and 186, 64^3 103 and 96.
#define ST_FOUR 4

bool xs_strip_analyse(int n, const int *rp, const int *ci, const int *dpos, bool upper,
                      xs_strip_plan &P) {
  P = xs_strip_plan();
  if (n > ST_MAX_ROWS) return false;
  auto row = [&](int p) { return upper ? n - 1 - p : p; };
  auto cnt = [&](int r) { return upper ? rp[r + 1] - 1 - dpos[r] : dpos[r] - rp[r]; };
  // position of the t-th entry of row r in solve order
  auto dep = [&](int r, int t) {
    return upper ? n - 1 - ci[rp[r + 1] - 1 - t] : ci[rp[r] + t];
  };
  std::vector<int> grp(n);
  int run = 0, blocks = 0;   // groups of this line of rows, of the longest
  bool single = false;       // some group has one row
  for (int p = 0; p < n; ++p) {
    const int r = row(p), m = cnt(r);
    const bool chain = m > 0 && dep(r, m - 1) == p - 1;
    const int gs = P.gstart.empty() ? 0 : P.gstart.back();
    const bool first = P.gstart.empty() || !chain || p - gs == XS_WAVE;
    if (first) {
      single |= p - gs == 1;
      P.gstart.push_back(p);
      run = chain ? run + 1 : 1;
      blocks = std::max(blocks, run);
    }
    // entries outside the group (the position before apart): few, and none
    // inside it
    const int ext = chain ? m - 1 : m;
    if (ext > ST_MAXQ) return false;
    if (ext > 0 && dep(r, ext - 1) >= P.gstart.back()) return false;
    P.Q = std::max(P.Q, ext);
    grp[p] = (int)P.gstart.size() - 1;
  }
  const int G = (int)P.gstart.size();
  if ((long)G * ST_MIN_GROUP > n) return false;
  P.Q = std::max(P.Q, 1);
  // the chains' stride: the commonest distance from a group's first position
  // to its farthest dependency, where that is a group's first position too
  std::unordered_map<int, int> hist;
  std::vector<int> far(G, -1);
  for (int g = 0; g < G; ++g) {
    const int p = P.gstart[g], r = row(p);
    if (cnt(r) == 0) continue;
    const int q = dep(r, 0);
    if (P.gstart[grp[q]] != q) continue;
    far[g] = q;
    hist[p - q]++;
  }
  int best = 0;
  for (auto &h : hist)
    if (h.second > best || (h.second == best && h.first > P.stride)) { best = h.second; P.stride = h.first; }
  if (!best) return false;
  P.gchain.resize(G);
  P.gstep.resize(G);
  std::vector<int> len;
  std::vector<char> taken(G, 0);
  for (int g = 0; g < G; ++g) {
    const int d = far[g] >= 0 && P.gstart[g] - far[g] == P.stride ? grp[far[g]] : -1;
    if (d >= 0 && !taken[d]) {
      taken[d] = 1;
      P.gchain[g] = P.gchain[d];
      P.gstep[g] = P.gstep[d] + 1;
      len[P.gchain[g]]++;
    } else {
      P.gchain[g] = (int)len.size();
      P.gstep[g] = 0;
      len.push_back(1);
      P.cbase.push_back(P.gstart[g]);
    }
    if (P.gstep[g] >= ST_MAX_STEPS) return false;
  }
  const int C = (int)len.size();
  if ((long)C * ST_MIN_CHAIN > G) return false;
  if (P.Q >= 2 && blocks >= ST_LINE_BLOCKS && C < ST_MIN_LINES * blocks && !single) return false;
  // every dependency on another chain points to a lower one
  for (int p = 0; p < n; ++p) {
    const int r = row(p), m = cnt(r), c = P.gchain[grp[p]];
    for (int t = 0; t < m; ++t)
      if (P.gchain[grp[dep(r, t)]] > c) return false;
  }
  P.cptr.assign(C + 1, 0);
  for (int c = 0; c < C; ++c) P.cptr[c + 1] = P.cptr[c] + len[c];
  P.gstart.push_back(n);
  return true;
}

void xs_strip_free(xs_strip &S) {
  for (void *p : {(void *)S.cptr, (void *)S.cbase, (void *)S.code, (void *)S.val,
                  (void *)S.vpos, (void *)S.carry})
    if (p) (void)hipFree(p);
  S = xs_strip();
}

int xs_strip_build(hipStream_t s, int n, const int *rp, const int *ci, const int *dpos, bool upper,
                   const xs_strip_plan &P, xs_strip &S) {
  xs_strip_free(S);
  const int G = (int)P.gstart.size() - 1, C = (int)P.cptr.size() - 1;
  S.n = n;
  S.Q = P.Q;
  S.nchains = C;
  S.nslots = G;
  S.stride = P.stride;
  S.waves = G / C >= ST_FOUR * C ? 4 : 8;
  int *tmp = nullptr;   // sgroup, gstart, gchain, gstep, grp
  const size_t lanes = (size_t)G * XS_WAVE, ent = lanes * (S.Q + 1);
  const size_t tlen = (size_t)G + (G + 1) + G + G + n;
  auto get = [](auto **p, size_t len) {
    return hipMalloc((void **)p, sizeof(**p) * len) == hipSuccess;
  };
  if (!(get(&S.cptr, C + 1) && get(&S.cbase, C) && get(&S.code, lanes * S.Q) &&
        get(&S.val, ent) && get(&S.vpos, ent) && get(&S.carry, G) && get(&tmp, tlen))) {
    (void)hipGetLastError();
    if (tmp) (void)hipFree(tmp);
    xs_strip_free(S);
    return XS_ERR_MEMORY;
  }
  std::vector<int> h(tlen);
  int *sgroup = h.data(), *gstart = sgroup + G, *gchain = gstart + G + 1, *gstep = gchain + G,
      *grp = gstep + G;
  std::copy(P.gstart.begin(), P.gstart.end(), gstart);
  std::copy(P.gchain.begin(), P.gchain.end(), gchain);
  std::copy(P.gstep.begin(), P.gstep.end(), gstep);
  for (int g = 0; g < G; ++g) {
    sgroup[P.cptr[P.gchain[g]] + P.gstep[g]] = g;
    for (int p = P.gstart[g]; p < P.gstart[g + 1]; ++p) grp[p] = g;
  }
  bool ok = hipMemcpyAsync(tmp, h.data(), sizeof(int) * tlen, hipMemcpyHostToDevice, s) == hipSuccess &&
            hipMemcpyAsync(S.cptr, P.cptr.data(), sizeof(int) * (C + 1), hipMemcpyHostToDevice, s) == hipSuccess &&
            hipMemcpyAsync(S.cbase, P.cbase.data(), sizeof(int) * C, hipMemcpyHostToDevice, s) == hipSuccess;
  if (ok) {
    int *d = tmp;
    const int *dsg = d, *dgs = d + G, *dgc = dgs + G + 1, *dgt = dgc + G, *dgr = dgt + G;
    const dim3 grid((G + 3) / 4), blk(256);
    if (upper)
      hipLaunchKernelGGL(k_strip_fill<true>, grid, blk, 0, s, n, S.Q, G, S.waves, rp, ci, dpos, dsg,
                         dgs, dgc, dgt, dgr, S.code, S.vpos, S.carry);
    else
      hipLaunchKernelGGL(k_strip_fill<false>, grid, blk, 0, s, n, S.Q, G, S.waves, rp, ci, dpos, dsg,
                         dgs, dgc, dgt, dgr, S.code, S.vpos, S.carry);
  }
  ok = ok && hipGetLastError() == hipSuccess && hipStreamSynchronize(s) == hipSuccess;
  (void)hipFree(tmp);
  if (!ok) {
    xs_strip_free(S);
    return XS_ERR_DEVICE;
  }
  S.ready = true;
  return XS_OK;
}

void xs_strip_values(hipStream_t s, const double *lu, xs_strip &S) {
  XS_GUARD(S.ready && lu);
  const size_t ent = (size_t)S.nslots * XS_WAVE * (S.Q + 1);
  hipLaunchKernelGGL(k_strip_vals, dim3((unsigned)((ent + 255) / 256)), dim3(256), 0, s, ent, S.vpos, lu, S.val);
  S.vals = true;
}

void xs_strip_solve(hipStream_t s, const xs_strip &S, bool upper, const double *dinv,
                    const double *b, double *x, unsigned *tickets, const xs_state *st) {
  XS_GUARD(S.ready && S.vals && b && x && tickets && S.Q >= 1 && S.Q <= ST_MAXQ);
  const st_args A{S.n, S.nchains, S.stride, S.cptr, S.cbase, S.code, S.carry, S.val};
  const dim3 grid((S.nchains + S.waves - 1) / S.waves), blk(S.waves * XS_WAVE);
#define ST_GO(U, D, Q_, W) hipLaunchKernelGGL((k_strip<U, D, Q_, W>), grid, blk, 0, s, A, dinv, b, x, tickets, st)
#define ST_W(U, D, Q_) do { if (S.waves == 4) ST_GO(U, D, Q_, 4); else ST_GO(U, D, Q_, 8); } while (0)
#define ST_Q(U, D) do { if (S.Q == 1) ST_W(U, D, 1); else if (S.Q == 2) ST_W(U, D, 2); else ST_W(U, D, 3); } while (0)
  if (upper) { if (dinv) ST_Q(true, true); else ST_Q(true, false); }
  else { if (dinv) ST_Q(false, true); else ST_Q(false, false); }
#undef ST_Q
#undef ST_W
#undef ST_GO
}
