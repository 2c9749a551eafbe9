// The whole MB-pol 3B and 2B evaluation with gradients in one launch: variables, polynomial, chain rule,
// switch, virial and gradient scatter of 64 trimers or dimers a block (the trimers' blocks first).
// Restates x2o::x3b_v2x::eval and x2o::x2b_v9x::eval (potential/3b/x3b-v2x.cpp:1403-1806,
// potential/2b/x2b-v9x.cpp:1514-1820) as the stage kernels do (eval_mbpol3b.hip, eval_mbpol2b.hip,
// poly_mbpol*.hip, mbpol3b_chain.hpp), which stay for energies alone and for the separate launches.
//
// Four wavefronts share a block's 64 n-mers through LDS.  Each of the first ones loads a monomer; every
// wavefront computes every fourth variable, evaluates two of the eight pieces of the polynomial, sums every
// fourth component of the gradient over the wavefronts, and runs the chain rule of its variables, for which
// an exponential needs only y_j = x_j dP/dx_j; then each of the first
// wavefronts gathers one monomer's gradient and scatters it while the last one has done the switch, energy
// and virial.  With the polynomial down to 20.0k operations a trimer (poly_kernel.hpp) the stages around it
// count: as launches of their own the variables take 27 us at 2048 waters, the 2B chain rule 20, the 3B chain
// rule 35, the polynomials 132.  Nothing of an n-mer but its energy goes through memory here.  This launch
// against those four, us: 6 waters 32 / 62, 256 waters 48 / 84, 617 waters 77 / 112, 2048 waters 192 / 214, 6859
// waters 548 / 521 (the registers of all stages in one kernel spill some 340 B a lane).
//
// Four is fixed, for every size: the gradient's order of summation and with it the results do not depend on
// how many n-mers there are, and it is the best or close to it over the range (a first form, with fewer second
// coefficients, at split 1 / 2 / 4 / 8, us: 6 waters 82 / 56 / 40 / 39, 256 waters 95 / 76 / 57 / 77, 617
// 105 / 85 / 87 / 135).
//
// Each variable is its own uniform branch, which also keeps the compiler from computing all square roots
// and exponentials at once (some 500 registers).
#include "gen/poly_mbpol_2b.inc"
#include "gen/poly_mbpol_3b.inc"
#include "mbpol2b_dev.hpp"
#include "mbpol3b_chain.hpp"
#include "mbxg_kernels.hpp"
#include "poly_kernel.hpp"

namespace mbxg {

namespace {

constexpr int kWaves = kFusedSplit;
constexpr int kExchange = 7;  // components an exchange round

// LDS of a block, rows of 64 doubles: 51 KB, three blocks (three wavefronts per SIMD) a CU.
//   kX  the variables, then the gradient, then y; then the site gradients gathered; then the scatter table
//   kR  the exchange [kWaves][kExchange]; then the virials [monomer][6]
//   kW  the sites' coordinates (2B: 18 + 12 of the M-sites)
//   kE  the pieces' values; then the switch and its derivatives
constexpr int kX = 0, kR = 36, kW = kR + kWaves * kExchange, kE = kW + 30, kRows = kE + kPolyParts;
typedef GradTable<128, 9> FusedTable;
static_assert(sizeof(FusedTable) <= kR * 64 * sizeof(double), "the table fits the variables' place");
static_assert(3 * kRows * 64 * sizeof(double) <= 160 * 1024, "three blocks a CU");

// Sum g (this wavefront's share of the gradient, in adapted coordinates, in the order of poly_eg_group) over
// the wavefronts into g of all of them.  The sums go to the variables' place.
template <int NV>
__device__ __forceinline__ void exchange_gradient(double* g, double* L, int wv) {
    double* X = L + kX * 64;
    double* R = L + kR * 64;
#pragma unroll
    for (int c0 = 0; c0 < NV; c0 += kExchange) {
#pragma unroll
        for (int j = c0; j < c0 + kExchange && j < NV; ++j) R[(wv * kExchange + j - c0) * 64] = g[j];
        __syncthreads();
#pragma unroll
        for (int j = c0; j < c0 + kExchange && j < NV; ++j)
            if ((j & 3) == wv) {
                const double* r = R + (j - c0) * 64;
                X[j * 64] = ((r[0] + r[kExchange * 64]) + r[2 * kExchange * 64]) + r[3 * kExchange * 64];
            }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) g[j] = X[j * 64];
}

// Round s of gathering the site gradients: every wavefront's N values v to wavefront s, summed into out.
template <int N>
__device__ __forceinline__ void gather(const double* v, double* out, int s, double* L, int wv) {
    static_assert(kWaves * N <= kW, "the round fits the variables' and the exchange's place");
    double* G = L;
#pragma unroll
    for (int c = 0; c < N; ++c) G[(wv * N + c) * 64] = v[c];
    __syncthreads();
    if (wv == s)
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const double* r = G + c * 64;
            out[c] = ((r[0] + r[N * 64]) + r[2 * N * 64]) + r[3 * N * 64];
        }
    __syncthreads();
}

// The end, after the gather: wavefront s < ORDER holds its monomer's coordinates w and gradient gd.
template <int ORDER>
__device__ __forceinline__ void finish_nmers(const FusedJob& J, const NmerCtx& N, int grp, bool act, int mon,
                                             const double* w, double* gd, double e, double* L, double* lds, int wv) {
    const int lane = threadIdx.x & 63, t = grp * 64 + lane;
    FusedTable& T = *reinterpret_cast<FusedTable*>(lds + kX * 64);
    table_init(T);
    if (wv < ORDER) {
        const int va[6] = {0, 0, 0, 1, 1, 2}, vb[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
        for (int q = 0; q < 6; ++q) {  // -sum_atoms w_a g_b
            double acc = 0.0;
#pragma unroll
            for (int at = 0; at < 3; ++at) acc -= w[3 * at + va[q]] * gd[3 * at + vb[q]];
            L[(kR + 6 * wv + q) * 64] = acc;
        }
        if (!act)
#pragma unroll
            for (int i = 0; i < 9; ++i) gd[i] = 0.0;
    }
    __syncthreads();
    if (wv == 0)
        table_add_runs<9>(T, act, mon, gd, J.grad, N.first_atom);  // the query monomer
    else if (wv < ORDER && act)
        table_add(T, mon, gd, 9, J.grad, N.first_atom[mon]);
    if (wv == kWaves - 1) {
        double vir[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            double v = L[(kR + q) * 64] + L[(kR + 6 + q) * 64];
            if (ORDER == 3) v += L[(kR + 12 + q) * 64];
            vir[q] = act ? v : 0.0;
        }
        if (act) {
            J.e_out[t] = e;
            if (J.vir_out)
#pragma unroll
                for (int q = 0; q < 6; ++q) J.vir_out[(size_t)q * J.ld + t] = vir[q];
        }
        double* out = J.partials + (size_t)grp * kPartials;
        e = wave_sum(act ? e : 0.0);
        if (lane == 0) out[0] = e;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const double v = wave_sum(vir[q]);
            if (lane == 0) out[1 + q] = v;
        }
    }
    __syncthreads();
    table_flush(T, J.grad);
}

// Monomer `mon`'s nine coordinates, imaged next to the point q0 (which is its own first atom's for monomer 1).
__device__ __forceinline__ void load_monomer(const NmerCtx& N, int mon, const double* q0, bool image, double* w) {
    const double* a = N.xyz + 3 * (size_t)N.first_atom[mon];
#pragma unroll
    for (int j = 0; j < 9; ++j) w[j] = a[j];
    if (image && N.periodic) {
        double v[3];
        image_vector(*N.box, q0[0], q0[1], q0[2], w[0], w[1], w[2], v);
#pragma unroll
        for (int j = 0; j < 9; ++j) w[j] -= v[j % 3];
    }
}

__device__ __forceinline__ void fused_trimers(const FusedJob& J, const NmerCtx& N, int grp, double* lds) {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n = min(*J.n_dev, J.cap);
    if (grp * 64 >= n) return;  // uniform
    const bool act = grp * 64 + lane < n;
    const int t = min(grp * 64 + lane, n - 1);  // lanes past the end repeat the last trimer
    double* L = lds + lane;
    int mon = -1;
    if (wv < 3) {
        mon = J.list[3 * t + wv];
        double w[9];
        load_monomer(N, mon, N.xyz + 3 * (size_t)N.first_atom[J.list[3 * t]], wv > 0, w);
#pragma unroll
        for (int j = 0; j < 9; ++j) L[(kW + 9 * wv + j) * 64] = w[j];
    }
    __syncthreads();
    {
        double w[27];
#pragma unroll
        for (int j = 0; j < 27; ++j) w[j] = L[(kW + j) * 64];
        static_for<36>([&](auto I) {
            constexpr int j = decltype(I)::value;
            if ((j & 3) == wv) {
                const int st = kVar3[j].set, a1 = kVar3[j].a1, a2 = kVar3[j].a2;
                const double d0 = w[3 * a1] - w[3 * a2], d1 = w[3 * a1 + 1] - w[3 * a2 + 1],
                             d2 = w[3 * a1 + 2] - w[3 * a2 + 2];
                L[(kX + j) * 64] = exp(-kset(st) * (sqrt(d0 * d0 + d1 * d1 + d2 * d2) - dset(st)));
            }
        });
    }
    __syncthreads();
    {
        double x[36], g[36];
#pragma unroll
        for (int j = 0; j < 36; ++j) {
            x[j] = L[(kX + j) * 64];
            g[j] = 0.0;
        }
        poly_mbpol_3b_sym(x);
        poly_mbpol_3b_parts(wv, kWaves, (mbxg_cptr)J.coef_addr, x, g, L + kE * 64);
        double own[9];  // this wavefront's variables
#pragma unroll
        for (int i = 0; i < 9; ++i) own[i] = 4 * i + wv < 36 ? L[(kX + 4 * i + wv) * 64] : 0.0;
        __syncthreads();  // every wavefront has read the variables and left its pieces' values
        exchange_gradient<36>(g, L, wv);
        poly_mbpol_3b_sym(g);
        __syncthreads();
        static_for<36>([&](auto I) {  // y_j = x_j dP/dx_j into their place
            constexpr int j = decltype(I)::value;
            if ((j & 3) == wv) L[(kX + j) * 64] = own[j / 4] * g[j];
        });
    }
    double w[27], gd[27];
#pragma unroll
    for (int j = 0; j < 27; ++j) {
        w[j] = L[(kW + j) * 64];
        gd[j] = 0.0;
    }
    static_for<36>([&](auto I) {  // g_var (x3b-v2x.cpp:63-76): -k x dP/dx (p1 - p2) / r
        constexpr int j = decltype(I)::value;
        if ((j & 3) == wv) {
            const int st = kVar3[j].set, a1 = kVar3[j].a1, a2 = kVar3[j].a2;
            const double d0 = w[3 * a1] - w[3 * a2], d1 = w[3 * a1 + 1] - w[3 * a2 + 1],
                         d2 = w[3 * a1 + 2] - w[3 * a2 + 2];
            const double gg = -kset(st) * L[(kX + j) * 64] * rsqrt(d0 * d0 + d1 * d1 + d2 * d2);
            gd[3 * a1] += gg * d0;
            gd[3 * a1 + 1] += gg * d1;
            gd[3 * a1 + 2] += gg * d2;
            gd[3 * a2] -= gg * d0;
            gd[3 * a2 + 1] -= gg * d1;
            gd[3 * a2 + 2] -= gg * d2;
        }
    });
    double e = 0.0;
    if (wv == 3) {  // the switch and what its derivatives put on the pairs
        const double P3 = poly_value(L + kE * 64);
        double dab[3], dac[3], dbc[3], rab, rac, rbc, sab, sac, sbc, gab, gac, gbc;
        const double s = switches(w, dab, dac, dbc, rab, rac, rbc, sab, sac, sbc, gab, gac, gbc);
        L[kE * 64] = s;
        L[(kE + 1) * 64] = gab * ((sac + sbc) * P3 / rab);
        L[(kE + 2) * 64] = gac * ((sab + sbc) * P3 / rac);
        L[(kE + 3) * 64] = gbc * ((sab + sac) * P3 / rbc);
        e = s * P3;
    }
    __syncthreads();  // y has been read
    double own[9];
#pragma unroll
    for (int s = 0; s < 3; ++s) gather<9>(gd + 9 * s, own, s, L, wv);
    double wm[9];
    if (wv < 3) {
        const double s = L[kE * 64], gab = L[(kE + 1) * 64], gac = L[(kE + 2) * 64], gbc = L[(kE + 3) * 64];
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            wm[j] = L[(kW + 9 * wv + j) * 64];
            own[j] *= s;
        }
        // pairs ab, ac, bc: +d on the first monomer's oxygen, -d on the second's
        const double f1 = wv == 0 ? gab : wv == 1 ? gab : gac, f2 = wv == 0 ? gac : gbc;
        const int o1 = wv == 0 ? 1 : 0, o2 = wv == 2 ? 1 : 2;
#pragma unroll
        for (int c = 0; c < 3; ++c)
            own[c] += f1 * (wm[c] - L[(kW + 9 * o1 + c) * 64]) + f2 * (wm[c] - L[(kW + 9 * o2 + c) * 64]);
    }
    finish_nmers<3>(J, N, grp, act, mon, wm, own, e, L, lds, wv);
}

__device__ __forceinline__ void fused_dimers(const FusedJob& J, const NmerCtx& N, int grp, double* lds) {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n = min(*J.n_dev, J.cap);
    if (grp * 64 >= n) return;
    const bool act = grp * 64 + lane < n;
    const int t = min(grp * 64 + lane, n - 1);
    double* L = lds + lane;
    int mon = -1;
    if (wv < 2) {
        mon = J.list[2 * t + wv];
        double w[15], oh1[3], oh2[3];
        load_monomer(N, mon, N.xyz + 3 * (size_t)N.first_atom[J.list[2 * t]], wv > 0, w);
        msites(w, 0, 3, 4, oh1, oh2);
#pragma unroll
        for (int j = 0; j < 9; ++j) L[(kW + 9 * wv + j) * 64] = w[j];
#pragma unroll
        for (int j = 0; j < 6; ++j) L[(kW + 18 + 6 * wv + j) * 64] = w[9 + j];
    }
    __syncthreads();
    {
        double s[30];
#pragma unroll
        for (int j = 0; j < 30; ++j) s[j] = L[(kW + j) * 64];
        static_for<31>([&](auto I) {
            constexpr int j = decltype(I)::value;
            if ((j & 3) == wv) {
                double gg, d0, d1, d2;
                L[(kX + j) * 64] = var2(kVar2[j], s, gg, d0, d1, d2);
            }
        });
    }
    __syncthreads();
    {
        double x[31], g[31];
#pragma unroll
        for (int j = 0; j < 31; ++j) {
            x[j] = L[(kX + j) * 64];
            g[j] = 0.0;
        }
        poly_mbpol_2b_sym(x);
        poly_mbpol_2b_parts(wv, kWaves, (mbxg_cptr)J.coef_addr, x, g, L + kE * 64);
        double own[8];  // this wavefront's variables
#pragma unroll
        for (int i = 0; i < 8; ++i) own[i] = 4 * i + wv < 31 ? L[(kX + 4 * i + wv) * 64] : 0.0;
        __syncthreads();
        exchange_gradient<31>(g, L, wv);
        poly_mbpol_2b_sym(g);
        __syncthreads();
        static_for<31>([&](auto I) {  // y_j = x_j dP/dx_j into their place
            constexpr int j = decltype(I)::value;
            if ((j & 3) == wv) L[(kX + j) * 64] = own[j / 4] * g[j];
        });
    }
    double s[30], xg[30];
#pragma unroll
    for (int i = 0; i < 30; ++i) {
        s[i] = L[(kW + i) * 64];
        xg[i] = 0.0;
    }
    static_for<31>([&](auto I) {  // d x / d (p1 - p2) = -(k, or k + 1/r for the Coulomb form) x / r
        constexpr int j = decltype(I)::value;
        if ((j & 3) == wv) {
            const int s1 = kVar2[j].s1, s2 = kVar2[j].s2;
            const double d0 = s[3 * s1] - s[3 * s2], d1 = s[3 * s1 + 1] - s[3 * s2 + 1], d2 = s[3 * s1 + 2] - s[3 * s2 + 2];
            const double rinv = rsqrt(d0 * d0 + d1 * d1 + d2 * d2), k = kval(kVar2[j].k);
            const double gg = -(kVar2[j].kind == 1 ? k + rinv : k) * L[(kX + j) * 64] * rinv;
            xg[3 * s1] += gg * d0;
            xg[3 * s1 + 1] += gg * d1;
            xg[3 * s1 + 2] += gg * d2;
            xg[3 * s2] -= gg * d0;
            xg[3 * s2 + 1] -= gg * d1;
            xg[3 * s2 + 2] -= gg * d2;
        }
    });
    double e = 0.0;
    if (wv == 3) {
        const double P2 = poly_value(L + kE * 64);
        const double d0 = s[0] - s[9], d1 = s[1] - s[10], d2 = s[2] - s[11];
        const double rOO = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
        double gsw;
        const double sw = switch2(rOO, gsw);
        L[kE * 64] = sw;
        L[(kE + 1) * 64] = gsw * (P2 / rOO);
        e = sw * P2;
    }
    __syncthreads();
    double own[15], wm[9];
#pragma unroll
    for (int q = 0; q < 2; ++q) {  // monomer q's atoms and its two M-sites
        double v[15];
#pragma unroll
        for (int j = 0; j < 15; ++j) v[j] = xg[j < 9 ? 9 * q + j : 18 + 6 * q + j - 9];
        gather<15>(v, own, q, L, wv);
    }
    if (wv < 2) {
        double oh1[3], oh2[3];
#pragma unroll
        for (int j = 0; j < 9; ++j) wm[j] = L[(kW + 9 * wv + j) * 64];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            oh1[i] = wm[3 + i] - wm[i];
            oh2[i] = wm[6 + i] - wm[i];
        }
        msite_grads(oh1, oh2, own + 9, own + 12, own);
        const double sw = L[kE * 64], gsc = L[(kE + 1) * 64];
#pragma unroll
        for (int j = 0; j < 9; ++j) own[j] *= sw;
#pragma unroll
        for (int c = 0; c < 3; ++c) own[c] += gsc * (wm[c] - L[(kW + 9 * (1 - wv) + c) * 64]);
    }
    finish_nmers<2>(J, N, grp, act, mon, wm, own, e, L, lds, wv);
}

__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(3, 3)))
    k_mbpol_fused(FusedJob A, FusedJob B, int nb_a, NmerCtx N) {
    __shared__ double lds[kRows * 64];
    if ((int)blockIdx.x < nb_a)
        fused_trimers(A, N, blockIdx.x, lds);
    else
        fused_dimers(B, N, blockIdx.x - nb_a, lds);
}

}  // namespace

hipError_t launch_mbpol_fused(const FusedJob& trimers, const FusedJob& dimers, const NmerCtx& N, hipStream_t st) {
    const int nb3 = (trimers.cap + 63) / 64, nb2 = (dimers.cap + 63) / 64;
    if (nb3 + nb2 == 0) return hipSuccess;
    hipLaunchKernelGGL(k_mbpol_fused, dim3(nb3 + nb2), dim3(64 * kWaves), 0, st, trimers, dimers, nb3, N);
    return hipGetLastError();
}

}  // namespace mbxg
