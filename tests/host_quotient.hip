// host_quotient.hip -- the FP64 step's quotient and square root
// (cable_amd/csrc/cbm_physics.h) on the CPU, from estimates as rough as the
// hardware's, against IEEE division and square root (tests/test_quotient.py).
//
//   host_quotient SEED COUNT BITS
//
// draws COUNT operands of each kind from SEED, starts from estimates off by
// up to 2^-BITS and prints the quotients, constant quotients and roots that
// differ from IEEE's.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../cable_amd/csrc/cbm_physics.h"

using namespace cbm;

namespace {
uint64_t state;
uint64_t bits64() {  // xorshift64*
  state ^= state >> 12;
  state ^= state << 25;
  state ^= state >> 27;
  return state * 0x2545F4914F6CDD1Dull;
}
// sign, exponent in +-lim, and a mantissa that is random, sparse, or next to
// a power of two in turn (all ones left out: see refine_reciprocal)
double operand(int lim, int kind) {
  uint64_t m = bits64() >> 12;
  if (kind == 1) m &= bits64() & bits64() & bits64();
  if (kind == 2) m = (bits64() & 1) ? (1ull << 52) - 2 - (bits64() & 3) : (bits64() & 3);
  const uint64_t e = 1023 + (int64_t)(bits64() % (2 * lim + 1)) - lim;
  const uint64_t u = (bits64() & (1ull << 63)) | e << 52 | m;
  double x;
  memcpy(&x, &u, 8);
  return x;
}
double rough(double exact, int bits) {
  return exact * (1.0 + ldexp(((double)(bits64() >> 11) * 0x1p-52 - 1.0), -bits));
}
}  // namespace

int main(int argc, char **argv) {
  if (argc != 4) return 2;
  state = strtoull(argv[1], nullptr, 10) * 2654435761ull + 1;
  const long count = atol(argv[2]);
  const int b = atoi(argv[3]);
  long q = 0, c = 0, s = 0;
  for (long i = 0; i < count; i++) {
    const double n = operand(300, i % 3), d = operand(300, (i / 3) % 3), x = fabs(n);
    q += corrected_quotient(n, d, refine_reciprocal(d, rough(1.0 / d, b))) != n / d;
    c += corrected_quotient(n, d, 1.0 / d) != n / d;
    s += refined_root(x, rough(1.0 / sqrt(x), b)) != sqrt(x);
  }
  printf("%ld %ld %ld\n", q, c, s);
  return 0;
}
