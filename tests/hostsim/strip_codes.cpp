// Where the source codes of the chain solves (xs_strip.h) point in the LDS
// arrays of a workgroup of W waves: every place inside them, and that of a
// code which names one exactly there.  Prints the number of faults.
#include <cstdio>

#include "../../xsolver_amd/csrc/xs_strip.h"

template <int W>
static long faults() {
  long bad = 0;
  auto inside = [&](int code) {
    const unsigned r = st_ring_byte<W>(code), q = st_seq_byte<W>(code);
    bad += r % 8 != 0 || r + 8 > W * ST_RING * 64 * 8 || q % 4 != 0 || q + 4 > W * 4;
  };
  for (long c = -2147483648l; c <= 2147483647l; c += 13) inside((int)c);
  for (int c : {ST_NONE, ST_PREV, ST_IDLE, -1, ~(ST_MAX_ROWS - 1)}) inside(c);
  for (int w = 0; w < W; ++w)
    for (int step : {0, 1, ST_RING - 1, ST_RING, 511, ST_MAX_STEPS - 1})
      for (int lane = 0; lane < 64; ++lane) {   // as k_strip_fill writes them
        const int place = (w * ST_RING + (step & (ST_RING - 1))) * 64 + lane;
        const int code = place | step << ST_STEP_SHIFT;
        inside(code);
        bad += code < 0 || code >= ST_PREV || st_ring_byte<W>(code) != 8u * place ||
               st_seq_byte<W>(code) != 4u * w || code >> ST_STEP_SHIFT != step;
      }
  return bad;
}

int main() {
  printf("%ld\n", faults<4>() + faults<8>());
  return 0;
}
