// The gradient table of scatter.hpp on the host: for every first atom on the command line, where the values
// of a monomer that starts there end up ("first atom, value index, values from the gradient's start").
// argv[1]: entries that other monomers take first (128: the table is full, device atomics directly).
#include <stdio.h>
#include <stdlib.h>

#include "../../mbx_amd/csrc/scatter.hpp"

int main(int argc, char** argv) {
    double* const grad = (double*)((size_t)1 << 44);  // never read or written
    for (int k = 2; k < argc; ++k) {
        static mbxg::GradTable<128, 9> T;
        const int taken = atoi(argv[1]);
        std::vector<int> first_atom(taken + 1);
        for (int m = 0; m < taken; ++m) first_atom[m] = 3 * m;
        first_atom[taken] = (int)atoll(argv[k]);
        mbxg::table_init(T);
        added().clear();
        for (int m = 0; m <= taken; ++m) {
            double g[9];
            for (int c = 0; c < 9; ++c) g[c] = 16.0 * m + c;
            mbxg::table_add_runs<9>(T, true, m, g, grad, first_atom.data());
        }
        mbxg::table_flush(T, grad);
        for (const Added& a : added())
            if (a.v >= 16.0 * taken) printf("%s %d %lld\n", argv[k], (int)(a.v - 16.0 * taken), (long long)(a.at - grad));
    }
    return 0;
}
