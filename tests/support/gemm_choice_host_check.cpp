// choose_gemm for each "M Mpad Npad Kpad" of the arguments: "bm bn splits" a line.
#include <cstdio>
#include <cstdlib>

#include "../../rustgears_amd/csrc/gemm_choice.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    const rgnpu::GemmChoice g = rgnpu::choose_gemm(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2]), atoll(argv[i + 3]));
    printf("%d %d %d\n", g.bm, g.bn, g.splits);
  }
}
