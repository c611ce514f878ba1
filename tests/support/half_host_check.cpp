// rgmath::half_bits against fp16_bits(round_fp16(x)) on the f32 bit patterns
// i = j * stride (stride 1: all 2^32).  Prints "<checked> <mismatches> <first>".
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "../../rustgears_amd/csrc/devmath.h"

int main(int argc, char** argv) {
  const uint64_t stride = argc > 1 ? strtoull(argv[1], nullptr, 0) : 7;
  uint64_t checked = 0, bad = 0;
  uint32_t first = 0;
  for (uint64_t i = 0; i < (1ull << 32); i += stride) {
    const float x = rgmath::bitsf((uint32_t)i);
    checked++;
    if (rgmath::half_bits(x) != rgmath::fp16_bits(rgmath::round_fp16(x)) && !bad++) first = (uint32_t)i;
  }
  printf("%llu %llu %08x\n", (unsigned long long)checked, (unsigned long long)bad, first);
  return bad != 0;
}
