// Every slot of ad_slot.hpp's map on the host: argv[1] holds the fitted coefficients (doubles).
#include <stdio.h>

#include <hip/hip_runtime.h>

inline double __fma_rn(double a, double b, double c) { return fma(a, b, c); }
#define __restrict__

#include "../../mbx_amd/csrc/ad_slot.hpp"
#define MBXG_SYM_SPACE static
#include SYM_INC

#define CAT_(a, b) a##b
#define CAT(a, b) CAT_(a, b)

int main(int, char** argv) {
    static double coef[4096];
    FILE* f = fopen(argv[1], "rb");
    if (!f || fread(coef, 8, 4096, f) == 0) return 2;
    for (int q = 0; q < CAT(kNSlot_, NAME); ++q)
        printf("%a\n", mbxg::ad_slot(CAT(kSymRow_, NAME), CAT(kSymK_, NAME), CAT(kSymW_, NAME), CAT(kSymLow_, NAME),
                                     CAT(kNRow_, NAME), q, coef));
    return 0;
}
