// Gradient scatter for the chain-rule stages: "reduce in LDS, then atomics".
//
// A block of n-mers touches far fewer distinct monomers than it has n-mer slots (the evaluated
// lists are grouped by query monomer, and partners are its near neighbours).  Each lane adds
// its per-monomer atom gradients into a small open-addressing table in LDS keyed by monomer
// (LDS FP64 atomics); after a barrier the table is flushed to the global gradient with one
// set of device atomics per distinct monomer.  If the table fills, the lane falls back to
// device atomics directly, so the result never depends on the table size.
//
// These kernels are bound by the atomics and by the latency around them, not by arithmetic.  What helped,
// measured on the 2B chain rules (32 beads of 57 CH4 + 513 H2O: MB-pol / CH4-H2O; 2048; 6859 waters):
// before 97 / 122; 23; 43 us, with the entries' values flushed by consecutive lanes from a list of the
// occupied entries (no loads from memory, some eight cache lines a wavefront instead of 64), tables at
// most half full and the query monomer's values summed across the wavefront 57 / 65; 18; 26 us.  CH4-H2O-H2O
// 370 -> 315 us.  Device atomics without the table: 193 / 119; 40 us.
#pragma once

#include <hip/hip_runtime.h>

#include "mbxg_device.hpp"

namespace mbxg {

template <int TB, int NA>
struct GradTable {
    double val[TB * NA];
    int key[TB];    // monomer, -1: free
    int first[TB];  // its first atom (three values an atom: scaled by three it needs more than 32 bits)
    int used[TB];   // the occupied entries * 32 + their numbers of values, in the order they were taken
    int count;
};

// LDS FP64 add.  The pointer is cast to the LDS address space: through a generic one unsafeAtomicAdd
// becomes a flat atomic, which also waits for the device memory path.
__device__ __forceinline__ void lds_add(double* p, double v) {
    __builtin_amdgcn_ds_atomic_fadd_f64((__attribute__((address_space(3))) double*)p, v);
}

template <int TB, int NA>
__device__ __forceinline__ void table_init(GradTable<TB, NA>& T) {
    for (int i = threadIdx.x; i < TB; i += blockDim.x) T.key[i] = -1;
    for (int i = threadIdx.x; i < TB * NA; i += blockDim.x) T.val[i] = 0.0;
    if (threadIdx.x == 0) T.count = 0;
}

// The entry of monomer `mon`, whose cnt values start at atom `first`; -1: the table is full.
template <int TB, int NA>
__device__ __forceinline__ int table_entry(GradTable<TB, NA>& T, int mon, int cnt, int first) {
    unsigned h = ((unsigned)mon * 2654435761u) % TB;
    for (int probe = 0; probe < TB; ++probe) {
        int k = __atomic_load_n(&T.key[h], __ATOMIC_RELAXED);
        if (k == -1) {
            k = atomicCAS(&T.key[h], -1, mon);
            if (k == -1) {  // taken here
                T.first[h] = first;
                T.used[atomicAdd(&T.count, 1)] = (int)h * 32 + cnt;
                return h;
            }
        }
        if (k == mon) return h;
        h = (h + 1) % TB;
    }
    return -1;
}

// Add cnt (<= NA) values for monomer `mon`, whose first atom is `first`; device atomics if the table is full.
template <int TB, int NA>
__device__ __forceinline__ void table_add(GradTable<TB, NA>& T, int mon, const double* g, int cnt, double* grad,
                                          int first) {
    const int h = table_entry(T, mon, cnt, first);
#pragma unroll
    for (int c = 0; c < NA; ++c)
        if (c < cnt) {
            if (h >= 0)
                lds_add(&T.val[h * NA + c], g[c]);
            else
                unsafeAtomicAdd(grad + 3 * (size_t)first + c, g[c]);
        }
}

// The sum of a run: lanes `in`'s CNT values added across the wavefront, value c left in lane c.
template <int CNT>
__device__ __forceinline__ double run_sum(bool in, const double* g) {
    const int lane = threadIdx.x & 63;
    double mine = 0.0;
#pragma unroll
    for (int c = 0; c < CNT; ++c) {
        const double v = wave_sum(in ? g[c] : 0.0);
        if (lane == c) mine = v;
    }
    return mine;
}

// The evaluate lists are grouped by query monomer, so one slot of an n-mer has the same monomer in runs
// of lanes, where 64 atomics on one address would be done one after the other.  table_add_runs
// adds every active lane's CNT values for its monomer `mon` (the other lanes' values are zeros); all lanes
// of the wavefront have to arrive together.  A run's values are summed across the wavefront first and
// added once, one lane per value; lanes left after kRuns runs, and short runs, add for themselves.
constexpr int kRuns = 3;      // a wavefront of a long list spans two query monomers, seldom three
constexpr int kRunLanes = 8;  // a run's sum costs about as much as eight lanes on one address

// One run of the lanes in `left`: sets mq and in, takes the run's lanes out of left; false: none worth it.
__device__ __forceinline__ bool next_run(bool act, int mon, unsigned long long& left, int& mq, bool& in) {
    mq = __builtin_amdgcn_readlane(mon, __ffsll((long long)left) - 1);
    in = act && mon == mq;
    const unsigned long long same = __ballot(in) & left;
    if (__popcll(same) < kRunLanes) return false;
    left &= ~same;
    return true;
}

template <int CNT, int TB, int NA>
__device__ __forceinline__ void table_add_runs(GradTable<TB, NA>& T, bool act, int mon, const double* g, double* grad,
                                               const int* first_atom) {
    const int lane = threadIdx.x & 63;
    unsigned long long left = __ballot(act);
    int mq;
    bool in;
#pragma nounroll
    for (int run = 0; run < kRuns && left; ++run) {
        if (!next_run(act, mon, left, mq, in)) break;
        const double mine = run_sum<CNT>(in, g);
        const int first = first_atom[mq];
        int h = 0;
        if (lane == 0) h = table_entry(T, mq, CNT, first);
        h = __builtin_amdgcn_readlane(h, 0);
        if (lane < CNT) {
            if (h >= 0)
                lds_add(&T.val[h * NA + lane], mine);
            else
                unsafeAtomicAdd(grad + 3 * (size_t)first + lane, mine);
        }
    }
    if (act && ((left >> lane) & 1)) table_add(T, mon, g, CNT, grad, first_atom[mon]);
}

// One slot of an n-mer whose query monomer may be in any slot (`query`: this lane's is in this one).
template <int CNT, int TB, int NA>
__device__ __forceinline__ void table_add_slot(GradTable<TB, NA>& T, bool act, bool query, int mon, const double* g,
                                               double* grad, const int* first_atom) {
    if (__ballot(act && query))
        table_add_runs<CNT>(T, act, mon, g, grad, first_atom);
    else if (act)
        table_add(T, mon, g, CNT, grad, first_atom[mon]);
}

// After a barrier: the occupied entries into the gradient, one device atomic per value, consecutive threads
// on consecutive values, so a wavefront's atomics fall on some eight cache lines instead of one line per
// lane, and nothing is loaded from memory on the way.
template <int TB, int NA>
__device__ __forceinline__ void table_flush(const GradTable<TB, NA>& T, double* grad) {
    const int n = T.count * NA;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int e = i / NA, c = i - e * NA, u = T.used[e], h = u >> 5;
        if (c < (u & 31)) unsafeAtomicAdd(grad + 3 * (size_t)T.first[h] + c, T.val[h * NA + c]);
    }
}

}  // namespace mbxg
