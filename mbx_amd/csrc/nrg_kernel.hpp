// MB-nrg families (CH4-H2O 2B, CH4-CH4 2B, CH4-H2O-H2O 3B): shared pieces.
//
// A holder is described as data (gen/holder_<name>.inc, generated from the holder's text):
// its monomers in argument order, its sites (real atoms in that order, plus the water's two
// lone-pair sites when it builds them), and its variables, each a function of one site pair:
//   form 0  exp(k (d - r))         tools/variable.cpp:49-64   (v_exp0)
//   form 1  exp(k (d - r)) / r     tools/variable.cpp:87-106  (v_coul0)
//   form 2  exp(-k r)              tools/variable.cpp:68-83   (v_exp)
// The polynomials are the blocked ones of poly_kernel.hpp, a translation unit each.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gen/poly_support.hpp"

namespace mbxg {

struct NrgVar {
    int form;
    double k, d;
    int s1, s2;
};

}  // namespace mbxg
