// Enough of HIP's device language for g++ to build scatter.hpp and run it on the host: one thread, one
// wavefront of one active lane.  Device-memory atomics are recorded instead of done.
#pragma once
#include <math.h>
#include <stddef.h>

#include <utility>
#include <vector>

#define __device__
#define __global__
#define __forceinline__ inline

struct Dim {
    int x;
};
static const Dim threadIdx = {0}, blockDim = {1};

inline int __ffsll(long long v) { return __builtin_ffsll(v); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline unsigned long long __ballot(bool v) { return v ? 1 : 0; }
inline int __double2loint(double) { return 0; }
inline int __double2hiint(double) { return 0; }
inline double __hiloint2double(int, int) { return 0.0; }
#define __builtin_amdgcn_update_dpp(old, v, ctrl, rows, banks, bound) (v)
#define __builtin_amdgcn_readlane(v, lane) (v)
#define __builtin_amdgcn_ds_atomic_fadd_f64(p, v) (*(p) += (v))

inline int atomicCAS(int* p, int old, int v) {
    const int was = *p;
    if (was == old) *p = v;
    return was;
}
inline int atomicAdd(int* p, int v) {
    const int was = *p;
    *p += v;
    return was;
}

struct Added {
    double* at;
    double v;
};
inline std::vector<Added>& added() {
    static std::vector<Added> a;
    return a;
}
inline void unsafeAtomicAdd(double* p, double v) { added().push_back({p, v}); }
