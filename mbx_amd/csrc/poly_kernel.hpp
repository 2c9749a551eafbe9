// The polynomial stage: one lane per n-mer, variables in, gradient and value out.
//
// It runs as its own kernel so the register allocator sees nothing but the generated
// straight-line polynomial (x and g arrays plus a few trie temporaries); the variable and
// chain-rule stages, whose exp/sqrt code the instruction selector freely interleaves, would
// otherwise push the polynomial past the register file.  (k_mbpol_fused, mbpol_fused.hip, runs them in one
// kernel with barriers between.)
//
// The polynomial is evaluated in symmetry-adapted coordinates (mbx_amd/gen/symmetry.py): sums and
// differences of the variables that exchanges of like sites permute.  In them a fraction of the
// monomials survives (MB-pol 3B 6,773 of 33,525: 20.0k FP64 operations a trimer for value and
// gradient instead of 72.5k; 2B 7.2k instead of 27.5k; CH4-H2O-H2O 14.3k instead of 63.0k; a fifth of them
// carries what rounding the coefficients left, without which energies have an error that grows with the
// system), which is what bounds these kernels: at full occupancy they run at 95-99% of the FP64 issue slots, alone on
// the chip at one wavefront's serial length.  The transform (SYM, in place on the registers, its own
// transpose) costs one to three additions a variable each way.  Whole steps, before and after with this
// change alone (and a third of the present second coefficients): 2048 waters 632 -> 354 us, 6859 waters
// 1592 -> 762 us, 32 beads of 57 CH4 + 513 H2O 4.24 -> 2.81 ms, six waters 284 -> 206 us.
//
// Layout: xs and gs are variable-major ("SoA"), entry (j, t) at j*ld + t, so a wavefront's 64
// lanes read and write 64 consecutive doubles per variable.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gen/poly_support.hpp"

namespace mbxg {

typedef void (*poly_eg_part_fn)(int, int, mbxg_cptr, const double*, double*, double*);
typedef void (*poly_e_part_fn)(int, int, mbxg_cptr, const double*, double*);
typedef void (*poly_sym_fn)(double*);

// The generated polynomial comes in Q pieces (linear: value and gradient are sums over the
// pieces).  A block holds 64 n-mers and P = blockDim.x / 64 wavefronts (P divides Q); wavefront
// w evaluates pieces w, w + P, ... for the block's 64 n-mers, and the P partial results are
// summed through LDS in a fixed order by wavefront 0, kRedChunk gradient components at a time.
// Splitting one n-mer's work over P wavefronts multiplies the number of wavefronts by P at 1/P
// of the length each, so the last round of wavefronts on the machine is short (less idle
// tail).  Dynamic LDS: poly_lds_bytes(P).  The pieces' values meet in LDS and are
// added in one order for every P (poly_value), so energies do not depend on the split.
constexpr int kRedChunk = 12;
constexpr int kPolyParts = 8;
constexpr size_t poly_lds_bytes(int P) { return ((size_t)(P - 1) * kRedChunk + kPolyParts) * 64 * sizeof(double); }

// The value from the pieces' shares e[64 * piece].
__device__ __forceinline__ double poly_value(const double* e) {
    return ((e[0] + e[4 * 64]) + (e[2 * 64] + e[6 * 64])) + ((e[64] + e[5 * 64]) + (e[3 * 64] + e[7 * 64]));
}

// One block's work: 64 n-mers of group `grp`, P = blockDim.x / 64 wavefronts.
template <int NV, int Q, poly_eg_part_fn PART, poly_sym_fn SYM>
__device__ __forceinline__ void poly_eg_group(int grp, const double* __restrict__ xs, int n, int ld,
                                              uint64_t coef_addr, double* __restrict__ gs, double* __restrict__ ps,
                                              double* red) {
    const int P = blockDim.x >> 6;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t = grp * 64 + lane;
    if (grp * 64 >= n) return;  // the whole block is past the end (uniform per block)
    const bool active = t < n;
    const mbxg_cptr C = (mbxg_cptr)coef_addr;
    double x[NV], g[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        x[j] = active ? xs[(size_t)j * ld + t] : 0.0;
        g[j] = 0.0;
    }
    SYM(x);
    double* es = red + (size_t)(P - 1) * kRedChunk * 64 + lane;
    PART(wv, P, C, x, g, es);
    if (P > 1) {
#pragma unroll
        for (int c0 = 0; c0 < NV; c0 += kRedChunk) {
            if (wv > 0) {
                double* r = red + (size_t)(wv - 1) * kRedChunk * 64 + lane;
#pragma unroll
                for (int j = c0; j < c0 + kRedChunk && j < NV; ++j) r[(j - c0) * 64] = g[j];
            }
            __syncthreads();
            if (wv == 0) {
                for (int v = 1; v < P; ++v) {
                    const double* r = red + (size_t)(v - 1) * kRedChunk * 64 + lane;
#pragma unroll
                    for (int j = c0; j < c0 + kRedChunk && j < NV; ++j) g[j] += r[(j - c0) * 64];
                }
            }
            __syncthreads();
        }
    }
    if (wv == 0 && active) {
        SYM(g);
#pragma unroll
        for (int j = 0; j < NV; ++j) gs[(size_t)j * ld + t] = g[j];
        ps[t] = poly_value(es);
    }
}

// Energy and gradient, WPE waves per SIMD: x and g take 4 registers a variable and the trie some 24, so
// 4 up to 26 variables, 3 up to 36 (MB-pol: at most 168 VGPRs), 2 up to 58 (CH4-H2O-H2O: 55), 1 for the
// 66 of the water 4B polynomial.
constexpr int poly_max_split(int wpe) { return wpe == 1 ? 4 : 8; }  // a block's wavefronts have to fit one CU

template <int NV, int Q, poly_eg_part_fn PART, poly_sym_fn SYM, int WPE>
__global__ void __launch_bounds__(64 * poly_max_split(WPE)) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    k_poly_eg(const double* __restrict__ xs, const int* __restrict__ n_dev, int cap, int ld, uint64_t coef_addr,
              double* __restrict__ gs, double* __restrict__ ps) {
    extern __shared__ double red[];  // poly_lds_bytes(P)
    poly_eg_group<NV, Q, PART, SYM>(blockIdx.x, xs, min(*n_dev, cap), ld, coef_addr, gs, ps, red);
}

// Two polynomials in one launch: blocks [0, nb_a) evaluate polynomial A (groups of 64 n-mers in
// order), the rest polynomial B.  Blocks are dispatched in index order, so B's blocks take the
// slots that A's last blocks leave idle.  Both use blockDim.x / 64 wavefronts per group.
struct PolyJob {
    const double* xs;
    const int* n_dev;
    int cap, ld;
    uint64_t coef_addr;
    double* gs;
    double* ps;
};

template <int NVA, int QA, poly_eg_part_fn PA, poly_sym_fn SA, int NVB, int QB, poly_eg_part_fn PB, poly_sym_fn SB>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(3, 3)))
    k_poly_eg_pair(PolyJob A, PolyJob B, int nb_a) {
    extern __shared__ double red[];
    if ((int)blockIdx.x < nb_a)
        poly_eg_group<NVA, QA, PA, SA>(blockIdx.x, A.xs, min(*A.n_dev, A.cap), A.ld, A.coef_addr, A.gs, A.ps, red);
    else
        poly_eg_group<NVB, QB, PB, SB>(blockIdx.x - nb_a, B.xs, min(*B.n_dev, B.cap), B.ld, B.coef_addr, B.gs, B.ps, red);
}

// One polynomial over several n-mer lists with their own coefficients, in one launch: the further
// families that share a structure hold a few hundred n-mers each, so a launch a family is all latency.
constexpr int kMaxPolyLists = 5;
struct PolyList {
    const double* xs;
    uint64_t coef_addr;
    double* gs;
    double* ps;
    int n, ld;
};
struct PolyLists {
    PolyList list[kMaxPolyLists];
    int count;
};

template <int NV, int Q, poly_eg_part_fn PART, poly_sym_fn SYM, int WPE>
__global__ void __launch_bounds__(64 * poly_max_split(WPE)) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    k_poly_eg_lists(PolyLists J) {
    extern __shared__ double red[];
    int grp = blockIdx.x, k = 0;
    while (k < J.count - 1 && grp >= (J.list[k].n + 63) / 64) grp -= (J.list[k++].n + 63) / 64;
    const PolyList& L = J.list[k];
    poly_eg_group<NV, Q, PART, SYM>(grp, L.xs, L.n, L.ld, L.coef_addr, L.gs, L.ps, red);
}

template <int NV, int Q, poly_eg_part_fn PEG, poly_sym_fn SYM, int WPE>
hipError_t launch_poly_eg_lists(const PolyLists& J, int P, hipStream_t st) {
    int groups = 0;
    for (int k = 0; k < J.count; ++k) groups += (J.list[k].n + 63) / 64;
    if (groups == 0) return hipSuccess;
    if (P > poly_max_split(WPE)) P = poly_max_split(WPE);
    hipLaunchKernelGGL((k_poly_eg_lists<NV, Q, PEG, SYM, WPE>), dim3(groups), dim3(64 * P), poly_lds_bytes(P), st, J);
    return hipGetLastError();
}

// Energy only.
template <int NV, int Q, poly_e_part_fn PART, poly_sym_fn SYM>
__global__ void __launch_bounds__(512) k_poly_e(const double* __restrict__ xs, const int* __restrict__ n_dev, int cap,
                                                int ld, uint64_t coef_addr, double* __restrict__ ps) {
    extern __shared__ double red[];  // [kPolyParts][64]
    const int P = blockDim.x >> 6;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t = blockIdx.x * 64 + lane;
    const int n = min(*n_dev, cap);
    if (blockIdx.x * 64 >= n) return;
    const bool active = t < n;
    const mbxg_cptr C = (mbxg_cptr)coef_addr;
    double x[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) x[j] = active ? xs[(size_t)j * ld + t] : 0.0;
    SYM(x);
    PART(wv, P, C, x, red + lane);
    if (P > 1) __syncthreads();
    if (wv == 0 && active) ps[t] = poly_value(red + lane);
}

// Launch helpers: P wavefronts per 64 n-mers (P in {1, 2, 4, 8}, dividing Q; the widest polynomials
// take 4 at most).
template <int NV, int Q, poly_eg_part_fn PEG, poly_sym_fn SYM, int WPE>
hipError_t launch_poly_eg(const double* xs, const int* n_dev, int cap, int ld, const double* coef, double* gs,
                          double* ps, int P, hipStream_t st) {
    if (cap <= 0) return hipSuccess;
    if (P != 1 && P != 2 && P != 4 && P != 8) return hipErrorInvalidValue;
    if (P > poly_max_split(WPE)) P = poly_max_split(WPE);
    hipLaunchKernelGGL((k_poly_eg<NV, Q, PEG, SYM, WPE>), dim3((cap + 63) / 64), dim3(64 * P), poly_lds_bytes(P), st, xs,
                       n_dev, cap, ld, (uint64_t)(uintptr_t)coef, gs, ps);
    return hipGetLastError();
}

template <int NV, int Q, poly_eg_part_fn PEG, poly_e_part_fn PE, poly_sym_fn SYM, int WPE = 3>
hipError_t launch_poly(const double* xs, const int* n_dev, int cap, int ld, const double* coef, int do_grads,
                       double* gs, double* ps, int P, hipStream_t st) {
    if (cap <= 0) return hipSuccess;
    if (do_grads) return launch_poly_eg<NV, Q, PEG, SYM, WPE>(xs, n_dev, cap, ld, coef, gs, ps, P, st);
    if (P != 1 && P != 2 && P != 4 && P != 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_poly_e<NV, Q, PE, SYM>), dim3((cap + 63) / 64), dim3(64 * P),
                       kPolyParts * 64 * sizeof(double), st, xs, n_dev, cap, ld, (uint64_t)(uintptr_t)coef, ps);
    return hipGetLastError();
}

}  // namespace mbxg
