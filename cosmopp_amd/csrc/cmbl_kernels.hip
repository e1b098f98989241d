// HIP kernels of the map-level likelihood for gfx950 (CDNA4, wave64, FP64).
//
// Stages of one likelihood + gradient evaluation (all FP64):
//   k_pre     packed a_lm (almToVector layout, source/cmb_gibbs.cpp:320-357)
//             -> m-major B_l N_lm a_lm, and the prior partial sums
//   k_synth   Legendre synthesis (the a_lm -> ring Fourier part of HEALPix
//             alm2map): per (m, ring pair) parity sums E_m, O_m
//   k_ring    per ring pair: phase fold + inverse ring DFT -> map s,
//             r = d - s, w r, chi^2 partial (source/cmb_gibbs.cpp:381-387),
//             forward ring DFT + unfold -> Psi_m (map2alm's ring part with
//             ring weight Npix/4pi, source/cmb_gibbs.cpp:390-391)
//   k_adj     adjoint Legendre: u_lm = sum_rings lambda_lm Psi_m
//   k_post    gradient assembly into the packed layout
//   k_final   deterministic -2lnL reduction
#include <atomic>
#include <cstdlib>

#include "cmbl_device.hpp"
#include "cmbl_internal.hpp"

namespace cmbl {

// ================================================================== helpers

__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmulc(double2 a, double2 b)  // a * conj(b)
{
    return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// e^{i pi q / n} for integer q (argument reduced exactly modulo 2n)
__device__ __forceinline__ double2 cis_pi_frac(long q, long n)
{
    const long two_n = 2 * n;
    long r = q % two_n;
    if (r < 0) r += two_n;
    double s, c;
    sincospi((double)r / (double)n, &s, &c);
    return make_double2(c, s);
}

// Ordering point for LDS data exchanged inside one wavefront.  The Legendre
// kernels run one wavefront per workgroup and the LDS executes the operations
// of a wavefront in issue order, so a store is visible to every later load of
// the same wavefront: the compiler only must not move memory operations across
// this point.  Unlike __syncthreads() it costs no lgkmcnt(0) wait.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Compile-time loops: every index is a constant when the accumulators are laid
// out, so they stay in registers (a runtime loop, even one that is unrolled
// later, left them in scratch).
template <class F, int... I>
__device__ __forceinline__ void for_each_map(std::integer_sequence<int, I...>, F&& f)
{
    (f(std::integral_constant<int, I>{}), ...);
}

// acc += c x (or -= c x), c taken from lane N of the lane's row of 16.  The
// rows hold the same 16 coefficients, so one register pair feeds 16 steps.  A
// DPP operand must not have been written by the VALU in the last two wait
// states, which the compiler does not see to for operands of an asm: every c
// passes dpp_ready() after its last copy and before its first use.
template <int N, bool NEG>
__device__ __forceinline__ void fmac_row(double& acc, double c, double x)
{
    if (NEG)
        asm("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(c), "v"(x), "n"(N));
    else
        asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(c), "v"(x), "n"(N));
}

__device__ __forceinline__ void dpp_ready(double& c) { asm volatile("s_nop 1" : "+v"(c)); }

// Global-address-space views of device memory: loads and stores through them
// compile to global_* instructions (counted by vmcnt only) rather than flat_*
// ones, whose lgkmcnt share makes every LDS wait also wait for memory, and
// which the compiler must order after earlier LDS and global stores.
typedef __attribute__((address_space(1))) double gdouble;
typedef const __attribute__((address_space(1))) double gcdouble;
typedef double __attribute__((ext_vector_type(2))) dvec2;
// Wave-uniform coefficients through the scalar cache.
typedef const __attribute__((address_space(4))) double scdouble;

// Views of double2 arrays in global memory (16-byte loads and stores).
struct GCView2 {
    const __attribute__((address_space(1))) dvec2* p;
    __device__ __forceinline__ double2 operator[](long i) const
    {
        const dvec2 v = p[i];
        return make_double2(v.x, v.y);
    }
    __device__ __forceinline__ GCView2 operator+(long k) const { return GCView2{p + k}; }
};
struct GView2 {
    __attribute__((address_space(1))) dvec2* p;
    struct Ref {
        __attribute__((address_space(1))) dvec2* q;
        __device__ __forceinline__ void operator=(double2 a) const
        {
            dvec2 v;
            v.x = a.x;
            v.y = a.y;
            *q = v;
        }
        __device__ __forceinline__ operator double2() const
        {
            const dvec2 v = *q;
            return make_double2(v.x, v.y);
        }
    };
    __device__ __forceinline__ Ref operator[](long i) const { return Ref{p + i}; }
    __device__ __forceinline__ GView2 operator+(long k) const { return GView2{p + k}; }
};

__device__ __forceinline__ gcdouble* gview(const double* p) { return (gcdouble*)p; }
__device__ __forceinline__ gdouble* gview(double* p) { return (gdouble*)p; }
__device__ __forceinline__ GCView2 gview(const double2* p)
{
    return GCView2{(const __attribute__((address_space(1))) dvec2*)p};
}
__device__ __forceinline__ GView2 gview(double2* p) { return GView2{(__attribute__((address_space(1))) dvec2*)p}; }

// Element i of an array below 4 GB: a uniform base and a 32-bit byte offset, one
// address register and no 64-bit arithmetic per lane.
__device__ __forceinline__ double2 ld_at(const double2* base, unsigned i)
{
    const dvec2 v = *(const __attribute__((address_space(1))) dvec2*)((const __attribute__((address_space(1))) char*)base +
                                                                     (i << 4));
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ double ld_at(const double* base, unsigned i)
{
    return *(gcdouble*)((const __attribute__((address_space(1))) char*)base + (i << 3));
}

// ================================================================== k_pre / k_post
// The packed parameter vector (almToVector: l-major, index l^2 + 2m - 1 + c)
// and the m-major device arrays (alm, Nrm, upart: index moff(L, m) + l - m)
// are transposes of each other over (l, m).  Both kernels work on kLM x kLM
// tiles of the triangle m <= l <= L, one tile per block, and transpose through
// LDS so that each side is read or written in its own contiguous order.
constexpr int kLM = 32;

__device__ __forceinline__ void tile_of(int b, int& tl, int& tm)
{
    int t = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while (t * (t + 1) / 2 > b) --t;
    while ((t + 1) * (t + 2) / 2 <= b) ++t;
    tl = t;
    tm = b - t * (t + 1) / 2;
}

// Packed index of (l, m, c) (c = 0 real, 1 imaginary), -1 for the absent Im a_l0.
__device__ __forceinline__ long packed_index(int l, int m, int c)
{
    const long li = (long)l * l;
    if (m == 0) return c == 0 ? li : -1;
    return li + 2 * m - 1 + c;
}

// alm = B_l N_lm a_lm (m-major) from the packed x, and the prior partial sum
// of the tile: sum invcl_l (|a_l0|^2 + 2 sum_m>0 |a_lm|^2).
__device__ __forceinline__ void pre_tile(const MapDesc& md, const double* __restrict__ x, int tile)
{
    __shared__ double T[kLM][2 * kLM + 1];
    __shared__ double sh[4];
    const int L = md.L;
    int tl, tm;
    tile_of(tile, tl, tm);
    const int l0 = tl * kLM, m0 = tm * kLM;
    // all loads of a thread are issued before their first use (entries
    // outside the triangle read entry 0 and are dropped)
    constexpr int kX = kLM * 2 * kLM / 256, kE = kLM * kLM / 256;
    double xv[kX];
#pragma unroll
    for (int e = 0; e < kX; ++e) {
        const int i = threadIdx.x + 256 * e;
        const int lr = i / (2 * kLM), c = i % (2 * kLM);
        const int l = l0 + lr, m = m0 + (c >> 1);
        const long pi = (l <= L && m <= l) ? packed_index(l, m, c & 1) : -1;
        xv[e] = gview(x)[pi >= 0 ? pi : 0];
        xv[e] = pi >= 0 ? xv[e] : 0.0;
    }
    double sc[kE], ic[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const int i = threadIdx.x + 256 * e;
        const int l = l0 + i % kLM, m = m0 + i / kLM;
        const bool ok = l <= L && m <= l;
        sc[e] = gview(md.beam)[ok ? l : 0] * gview(md.Nrm)[ok ? moff(L, m) + (l - m) : 0];
        ic[e] = gview(md.invcl)[ok ? l : 0];
    }
#pragma unroll
    for (int e = 0; e < kX; ++e) {
        const int i = threadIdx.x + 256 * e;
        T[i / (2 * kLM)][i % (2 * kLM)] = xv[e];
    }
    __syncthreads();
    double pr = 0.0;
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const int i = threadIdx.x + 256 * e;
        const int mr = i / kLM, lr = i % kLM;
        const int l = l0 + lr, m = m0 + mr;
        if (l <= L && m <= l) {
            const double re = T[lr][2 * mr], im = T[lr][2 * mr + 1];
            md.alm[aoff(L, m) + (l - m)] = make_double2(sc[e] * re, sc[e] * im);
            pr += ic[e] * ((m == 0) ? re * re : 2.0 * (re * re + im * im));
        }
    }
    const double t = block_sum<256>(pr, sh);
    if (threadIdx.x == 0) md.prior[tile] = t;
}

__global__ __launch_bounds__(256) void k_pre(const MapDesc* __restrict__ md_, const double* __restrict__ x)
{
    pre_tile(*md_, x, blockIdx.x);
}

// Map of block b in a batched launch (wave-uniform, at most kBatchGroup steps).
__device__ __forceinline__ int batch_map(const BatchArgs& a, int b)
{
    int i = 0;
    while (i + 1 < a.n && a.tile0[i + 1] <= b) ++i;
    return i;
}

__global__ __launch_bounds__(256) void k_pre_b(const MapDesc* __restrict__ mds, const BatchArgs a)
{
    const int i = batch_map(a, blockIdx.x);
    pre_tile(mds[i], a.x[i], blockIdx.x - a.tile0[i]);
}

// u = N_lm B_l sum_rb upart (fixed order) -> the packed output of `mode`
// (PostMode): the gradient forms kPostGrad / kPostLike, or the Gibbs forms in
// the HEALPix complex-a_lm convention (no factor 2 for m >= 1).  kPostAddAlm
// scales by c instead of B_l and adds to g.
__device__ __forceinline__ void post_tile(const MapDesc& md, const double* __restrict__ x, double* __restrict__ g,
                                          int mode, double c, int tile)
{
    __shared__ double T[kLM][2 * kLM + 1];
    const int L = md.L;
    int tl, tm;
    tile_of(tile, tl, tm);
    const int l0 = tl * kLM, m0 = tm * kLM;
    constexpr int kE = kLM * kLM / 256;  // elements per thread
    // every load of the thread's elements is issued before the sums (entries
    // outside the triangle read entry 0 and are dropped)
    long k[kE];
    bool ok[kE];
    double sc[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const int i = threadIdx.x + 256 * e;
        const int l = l0 + i % kLM, m = m0 + i / kLM;
        ok[e] = l <= L && m <= l;
        k[e] = ok[e] ? moff(L, m) + (l - m) : 0;
        const double s = (mode == kPostAddAlm || mode == kPostQuad) ? c : gview(md.beam)[ok[e] ? l : 0];
        sc[e] = gview(md.Nrm)[k[e]] * s;
    }
    const GCView2 u = gview(reinterpret_cast<const double2*>(md.upart));
    const long stride = md.nalm;  // double2 per ring block
    double ur[kE], ui[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) ur[e] = ui[e] = 0.0;
    // eight partials of two elements in flight per thread, added in
    // ring-block order
#pragma unroll
    for (int e0 = 0; e0 < kE; e0 += 2) {
        int rb = 0;
        for (; rb + 8 <= md.nrb5; rb += 8) {
            double2 v[2][8];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int j = 0; j < 8; ++j) v[e][j] = u[k[e0 + e] + (rb + j) * stride];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    ur[e0 + e] += v[e][j].x;
                    ui[e0 + e] += v[e][j].y;
                }
        }
        for (; rb < md.nrb5; ++rb) {
            double2 v[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) v[e] = u[k[e0 + e] + rb * stride];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                ur[e0 + e] += v[e].x;
                ui[e0 + e] += v[e].y;
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const int i = threadIdx.x + 256 * e;
        const int mr = i / kLM, lr = i % kLM;
        T[lr][2 * mr] = ok[e] ? ur[e] * sc[e] : 0.0;
        T[lr][2 * mr + 1] = ok[e] ? ui[e] * sc[e] : 0.0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kLM * 2 * kLM; i += 256) {
        const int lr = i / (2 * kLM), c2 = i % (2 * kLM);
        const int l = l0 + lr, m = m0 + (c2 >> 1);
        const long pi = (l <= L && m <= l) ? packed_index(l, m, c2 & 1) : -1;
        if (pi < 0) continue;
        const double u = T[lr][c2];
        switch (mode) {
        case kPostGrad: g[pi] = (m == 0) ? u : 2.0 * u; break;
        case kPostLike:
            g[pi] = (m == 0) ? -2.0 * u + 2.0 * md.invcl[l] * x[pi] : -4.0 * u + 4.0 * md.invcl[l] * x[pi];
            break;
        case kPostGibbs: g[pi] = x[pi] + u; break;
        case kPostAlm:
        case kPostQuad: g[pi] = u; break;
        default: g[pi] += u; break;  // kPostAddAlm
        }
    }
}

__global__ __launch_bounds__(256) void k_post(const MapDesc* __restrict__ md_, const double* __restrict__ x,
                                              double* __restrict__ g, int mode, double c)
{
    post_tile(*md_, x, g, mode, c, blockIdx.x);
}

__global__ __launch_bounds__(256) void k_post_b(const MapDesc* __restrict__ mds, const BatchArgs a, int mode)
{
    const int i = batch_map(a, blockIdx.x);
    post_tile(mds[i], a.x[i], a.g[i], mode, 0.0, blockIdx.x - a.tile0[i]);
}

// y_p = x_p / d_l over the packed layout (l = floor(sqrt(p))): the Gibbs
// preconditioner (source/cmb_gibbs.cpp:407-423 divides every a_lm by d_l).
// y may be x (in place).
__global__ __launch_bounds__(256) void k_ldiv(double* y, const double* x, const double* __restrict__ dl, int L)
{
    const long n = (long)(L + 1) * (L + 1);
    for (long p = blockIdx.x * 256L + threadIdx.x; p < n; p += (long)gridDim.x * 256L) {
        long l = (long)sqrt((double)p);
        while (l * l > p) --l;
        while ((l + 1) * (l + 1) <= p) ++l;
        y[p] = x[p] / dl[l];
    }
}

// ================================================================== spin-2 synthesis
// alm2map_pol (HEALPix; called at source/likelihood.cpp:585 and
// source/c_matrix_generator.cpp:577-578): T = sum a^T Y, and with
// W_lm = (2Y_lm + -2Y_lm)/2 = F1_lm(theta) e^{i m phi},
// X_lm = (2Y_lm - -2Y_lm)/2 = F2_lm(theta) e^{i m phi},
//   Q = -sum (a^E W + i a^B X),   U = -sum (a^B W - i a^E X).
// With kappa_l = 2 / sqrt((l-1) l (l+1) (l+2)), q_lm = sqrt((2l+1)/(2l-1) (l^2 - m^2)),
// c = cos(theta), s2 = sin^2(theta) and lambda_lm = Y_lm(theta, 0):
//   F1_lm = kappa_l [-((l - m^2)/s2 + l(l-1)/2) lambda_lm + c q_lm lambda_{l-1,m} / s2]
//   F2_lm = kappa_l (m/s2) [-(l-1) c lambda_lm + q_lm lambda_{l-1,m}].
// The sums over l of a field need three scalar Legendre
// sums of one recursion,
//   S1 = sum kappa a g lambda_l,  g = (m^2 - l) / s2 - l (l - 1) / 2,
//   S2 = sum kappa q a lambda_{l-1}  (coefficients shifted by one l),
//   S3 = sum (l - 1) kappa a lambda_l:
//   sum_l a F1 = S1 + c S2/s2,   sum_l a F2 = m (S2 - c S3)/s2.
// k_synth_pol runs the recursion once per (m, ring block) for the T sum and
// the six field sums and forms Q_m, U_m per ring in its epilogue.

// Record of (l, m) (m-major with padded rows, kPolRec doubles): complex N a^T;
// N kappa_l a^E, the same of B; N kappa_{l+1} q_{l+1,m} a^E_{l+1,m}, B;
// (l - 1) N kappa_l a^E, B.
__global__ __launch_bounds__(256) void k_pre_pol(const MapDesc* __restrict__ md_, const double* __restrict__ t,
                                                 const double* __restrict__ e, const double* __restrict__ b,
                                                 double2* __restrict__ rec)
{
    __shared__ double T[3][kLM + 1][2 * kLM + 1];
    const MapDesc& md = *md_;
    const int L = md.L;
    int tl, tm;
    tile_of(blockIdx.x, tl, tm);
    const int l0 = tl * kLM, m0 = tm * kLM;
    // rows l0 .. l0 + kLM: the extra row feeds the shifted coefficients
    for (int i = threadIdx.x; i < (kLM + 1) * 2 * kLM; i += 256) {
        const int lr = i / (2 * kLM), c = i % (2 * kLM);
        const int l = l0 + lr, m = m0 + (c >> 1);
        const long pi = (l <= L && m <= l) ? packed_index(l, m, c & 1) : -1;
        T[0][lr][c] = pi >= 0 ? t[pi] : 0.0;
        T[1][lr][c] = pi >= 0 ? e[pi] : 0.0;
        T[2][lr][c] = pi >= 0 ? b[pi] : 0.0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kLM * kLM; i += 256) {
        const int mr = i / kLM, lr = i % kLM;
        const int l = l0 + lr, m = m0 + mr;
        if (l > L || m > l) continue;
        const long k = moff(L, m) + (l - m);
        const double nr = md.Nrm[k];
        const double fl = l, m2 = (double)m * m;
        const double ck = l >= 2 ? nr * 2.0 / sqrt((fl - 1.0) * fl * (fl + 1.0) * (fl + 2.0)) : 0.0;
        const double l1 = fl + 1.0;
        const double dk = (l + 1 <= L && l + 1 >= 2)
                              ? nr * 2.0 / sqrt((l1 - 1.0) * l1 * (l1 + 1.0) * (l1 + 2.0)) *
                                    sqrt((2.0 * l1 + 1.0) / (2.0 * l1 - 1.0) * (l1 * l1 - m2))
                              : 0.0;
        double2* o = rec + (aoff(L, m) + (l - m)) * (kPolRec / 2);
        const double e0 = ck * T[1][lr][2 * mr], e1 = ck * T[1][lr][2 * mr + 1];
        const double b0 = ck * T[2][lr][2 * mr], b1 = ck * T[2][lr][2 * mr + 1];
        o[0] = make_double2(nr * T[0][lr][2 * mr], nr * T[0][lr][2 * mr + 1]);
        o[1] = make_double2(e0, e1);
        o[2] = make_double2(b0, b1);
        o[3] = make_double2(dk * T[1][lr + 1][2 * mr], dk * T[1][lr + 1][2 * mr + 1]);
        o[4] = make_double2(dk * T[2][lr + 1][2 * mr], dk * T[2][lr + 1][2 * mr + 1]);
        o[5] = make_double2((fl - 1.0) * e0, (fl - 1.0) * e1);
        o[6] = make_double2((fl - 1.0) * b0, (fl - 1.0) * b1);
    }
}

// ================================================================== MASTER coupling
// Mode-coupling matrix of a mask with pseudo spectrum W (source/master.cpp:180-215):
//   M[l1][l2] = (2 l2 + 1) / (4 pi) sum_{l3 <= L} (2 l3 + 1) W_l3 (l1 l2 l3; 0 0 0)^2.
// The symbol's closed form, with g = (l1 + l2 + l3) / 2 and h(n) = (2n)! / (4^n n!^2),
//   (l1 l2 l3; 0 0 0)^2 = h(g - l1) h(g - l2) h(g - l3) / ((2g + 1) h(g)),
// makes the sum of the pair l2, l1 = l2 + d, over l3 = d + 2 t, t <= l2,
//   sum_t F_d(t) h(l2 - t) k(l2 + d + t),  F_d(t) = (2 l3 + 1) W_l3 h(t) h(d + t),
//   k(g) = 1 / ((2g + 1) h(g)):
// two FP64 instructions per term and no division in the loop.

// C(2n, n), an integer below 2^53 for n <= 28.
struct CentralBinomials {
    double c[29];
    constexpr CentralBinomials() : c{}
    {
        unsigned long long v = 1;
        c[0] = 1.0;
        for (unsigned long long n = 1; n <= 28; ++n) {
            v = v * (2 * (2 * n - 1)) / n;
            c[n] = (double)v;
        }
    }
};
__constant__ const CentralBinomials kCentral;

// h(n) = s r, r = 1 / sqrt(pi (n + 1/4)), with the series s of Gamma(n + 1/2) /
// Gamma(n + 1) in u = 1 / (n + 1/4)^2 (its next term is below 1e-17 from n = 29);
// h(n < 0) = 0.
__device__ __forceinline__ double central_series(double r)
{
    const double v = 3.141592653589793 * (r * r), u = v * v;
    return fma(u, fma(u, fma(u, fma(u, 180323.0 / 134217728.0, -671.0 / 524288.0), 21.0 / 8192.0), -1.0 / 64.0), 1.0);
}
__device__ __forceinline__ double central_h(int n)
{
    if (n < 29) return n < 0 ? 0.0 : ldexp(kCentral.c[n], -2 * n);
    const double r = rsqrt(3.141592653589793 * (n + 0.25));
    return central_series(r) * r;
}
__device__ __forceinline__ double central_k(int g)
{
    if (g < 29) return ldexp(1.0, 2 * g) / ((2.0 * g + 1.0) * kCentral.c[g]);
    const double y = 3.141592653589793 * (g + 0.25), r = rsqrt(y);
    return y * r / ((2.0 * g + 1.0) * central_series(r));
}

// A workgroup takes kCoupD distances d (a wave each) and 64 kCoupR degrees l2,
// kCoupR consecutive ones per lane: when t advances, a lane's h and k move on by
// one degree, so a step reads one new value of each from LDS for kCoupR terms.
// Both are stored by degree modulo kCoupR, which puts the lanes of a read on
// consecutive doubles.  F comes through the DPP operand, 16 steps per row of
// lanes.  Bound by FP64 issue (a product and a sum per term; LDS reads take
// about as long).  The results cross LDS so that the stores of both triangles
// write runs of kCoupD entries.
// lmax 1535: 994 -> 75 us (a recursion over l3 with a division per term before;
// kCoupD 8 3% more, 16 8%; kCoupR 2 8%, 8 three times, out of registers; a bound
// of four waves per SIMD, which spills: the same).  Two thirds of
// that is issue, 128 + 22 instructions per 16 steps, and the tables.
constexpr int kCoupR = 4;
constexpr int kCoupD = 4;
constexpr int kCoupL = 64 * kCoupR;  // degrees l2 of a workgroup
constexpr int kCoupT = 512;          // steps t per staging of the tables
constexpr int kCoupS = (kCoupL + kCoupT) / kCoupR + 4;  // entries of one residue

// 16 steps: F of step s in lane s of each row; ho and ko[c] index the lane's next
// values in hC and kD (indices: pointers in an array would lose that they are LDS).  TRI: some lanes' sums end here; step s ends the sum of degree
// index kCoupR q + s of the block, whose value is kept in end.
template <bool TRI>
__device__ __forceinline__ void coupling_steps(double (&acc)[kCoupR], double (&end)[kCoupR], double (&hv)[kCoupR],
                                               double (&kv)[kCoupR], double F, const double* hC, int ho,
                                               const double* kD, const int (&ko)[kCoupR], int q, int lane)
{
    for_each_map(std::make_integer_sequence<int, 16>{}, [&](auto si) {
        constexpr int s = decltype(si)::value;
        constexpr int hs = (kCoupR * 16 - s) % kCoupR;  // slot of degree index 0; degree r: (r - s) mod kCoupR
        constexpr int ks = (kCoupR - 1 + s) % kCoupR;   // slot of degree index kCoupR - 1; r: (r + s) mod kCoupR
        hv[hs] = hC[ho + hs * kCoupS - (s + hs) / kCoupR];
        kv[ks] = kD[ko[s % kCoupR] + s / kCoupR];
#pragma unroll
        for (int r = 0; r < kCoupR; ++r)
            fmac_row<s, false>(acc[r], F, hv[(r - s + 16 * kCoupR) % kCoupR] * kv[(r + s) % kCoupR]);
        if (TRI) end[s % kCoupR] = lane == q + s / kCoupR ? acc[s % kCoupR] : end[s % kCoupR];
    });
}

__global__ __launch_bounds__(64 * kCoupD, 3) void k_coupling(int L, const double* __restrict__ W, double* __restrict__ M)
{
    constexpr int kTab = 2 * kCoupR * kCoupS + 2 * kCoupT + kCoupD, kOut = kCoupD * (kCoupL + 1);
    __shared__ double lds[kTab > kOut ? kTab : kOut];
    double* hC = lds;                    // h(l2 - t)
    double* kD = hC + kCoupR * kCoupS;   // k(l2 + d + t)
    double* hA = kD + kCoupR * kCoupS;   // h(t)
    double* hB = hA + kCoupT;            // h(d + t)
    const int d0 = kCoupD * blockIdx.y, b = kCoupL * blockIdx.x;
    if (b > L - d0) return;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int d = d0 + w;
    // steps of the workgroup and of this wave
    auto steps = [&](int dd) { return dd > L ? 0 : min(b + kCoupL - 1, (L - dd) / 2) + 1; };
    const int n0 = steps(d0), nw = (steps(d) + 15) & ~15;
    double acc[kCoupR], end[kCoupR];
#pragma unroll
    for (int r = 0; r < kCoupR; ++r) acc[r] = end[r] = 0.0;
    for (int t0 = 0; t0 < n0; t0 += kCoupT) {
        const int nt = min(kCoupT, (n0 - t0 + 15) & ~15);  // staged steps
        __syncthreads();
        // hC: degree index i <-> l2 - t = b - t0 - nt + i; kD: l2 + d + t = b + d0 + t0 + i
        for (int i = tid; i < kCoupL + nt; i += 64 * kCoupD) hC[(i % kCoupR) * kCoupS + i / kCoupR] = central_h(b - t0 - nt + i);
        for (int i = tid; i < kCoupL + nt + kCoupD; i += 64 * kCoupD)
            kD[(i % kCoupR) * kCoupS + i / kCoupR] = central_k(b + d0 + t0 + i);
        for (int i = tid; i < nt; i += 64 * kCoupD) hA[i] = central_h(t0 + i);
        for (int i = tid; i < nt + kCoupD; i += 64 * kCoupD) hB[i] = central_h(d0 + t0 + i);
        __syncthreads();
        const int ne = min(nt, nw - t0);
        if (ne <= 0) continue;
        int ho = nt / kCoupR + lane, ko[kCoupR];
#pragma unroll
        for (int c = 0; c < kCoupR; ++c) {
            const int i = kCoupR - 1 + w + c;
            ko[c] = (i % kCoupR) * kCoupS + i / kCoupR + lane;
        }
        double hv[kCoupR], kv[kCoupR];
        // the first step's values but the ones it reads itself
#pragma unroll
        for (int r = 1; r < kCoupR; ++r) hv[r] = hC[ho + r * kCoupS];
#pragma unroll
        for (int r = 0; r < kCoupR - 1; ++r) {
            const int i = r + w;
            kv[r] = kD[(i % kCoupR) * kCoupS + i / kCoupR + lane];
        }
        const int j = lane & 15;
        auto weight = [&](int t) { const int l3 = d + 2 * (t0 + t); return l3 <= L ? (2.0 * l3 + 1.0) * W[l3] : 0.0; };
        double f = weight(j);
        for (int t = 0; t < ne; t += 16) {
            // past L the weight is zero, and so is F whatever the tables hold
            double F = f * (hA[t + j] * hB[w + t + j]);
            f = t + 16 < ne ? weight(t + 16 + j) : 0.0;
            dpp_ready(F);
            const int q = (t0 + t - b) / kCoupR;
            if (t0 + t < b)
                coupling_steps<false>(acc, end, hv, kv, F, hC, ho, kD, ko, q, lane);
            else
                coupling_steps<true>(acc, end, hv, kv, F, hC, ho, kD, ko, q, lane);
            ho -= 16 / kCoupR;
#pragma unroll
            for (int c = 0; c < kCoupR; ++c) ko[c] += 16 / kCoupR;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kCoupR; ++r) {
        const int i = kCoupR * lane + r;
        lds[w * (kCoupL + 1) + i] = b + i < nw ? end[r] : acc[r];
    }
    __syncthreads();
    const double inv4pi = 0.25 / 3.141592653589793;
    // row l2: the entries l1 = l2 + d0 .. of this workgroup
    for (int u = tid; u < kCoupL * kCoupD; u += 64 * kCoupD) {
        const int i = u / kCoupD, e = u % kCoupD, l2 = b + i, l1 = l2 + d0 + e;
        if (l1 <= L) M[(long)l2 * (L + 1) + l1] = (2.0 * l1 + 1.0) * inv4pi * lds[e * (kCoupL + 1) + i];
    }
    // row l1: the entries l2 = l1 - d0 - e
    for (int u = tid; u < (kCoupL + kCoupD - 1) * kCoupD; u += 64 * kCoupD) {
        const int e = kCoupD - 1 - u % kCoupD, i = u / kCoupD - e, l2 = b + i, l1 = l2 + d0 + e;
        if (i >= 0 && i < kCoupL && l1 <= L) M[(long)l1 * (L + 1) + l2] = (2.0 * l2 + 1.0) * inv4pi * lds[e * (kCoupL + 1) + i];
    }
}

// NEST <-> RING reordering of a map: out[i] = in[pixel of i in the other
// scheme].  Writes are coalesced, reads gathered.
__global__ __launch_bounds__(256) void k_reorder(const double* __restrict__ in, double* __restrict__ out, long nside,
                                                 int to_ring)
{
    const long npix = 12 * nside * nside;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < npix; i += (long)gridDim.x * 256L)
        out[i] = in[to_ring ? ring_to_nest(nside, i) : nest_to_ring(nside, i)];
}

// ================================================================== Legendre stages
//
// One wavefront (= one workgroup) per work item: degree m of one ring block
// of one map.  Lane `lane` handles ring pairs p_k = rb*64*K + k*64 + lane,
// k < K.  The recurrence mu_l = A_lm x mu_{l-1} - mu_{l-2} runs in registers,
// starting from the state precomputed at set-up for the item's first live l.
//
// Its odd members (l - m odd) are carried divided by x = cos theta, which
// takes x out of every second step,
//   odd:  mu_l / x = A_lm mu_{l-1} - mu_{l-2} / x
//   even: mu_l     = A_lm x^2 (mu_{l-1} / x) - mu_{l-2},
// so a pair of l-steps costs 3 FP64 instructions instead of 4; the sums over
// odd l - m are multiplied by x once, at the end (synthesis) or in their
// inputs (adjoint).  x^2 is rounded, and that one relative error, the same at
// every step, would be a phase error growing with l: of the eight even steps
// of every 16 l-steps the first takes x^2 plus eight times the rounding error
// (rounded again: Ring::ya), and of every eighth 16 also eight times what that
// rounding left (yb), so that the mean multiplier is x^2 to 2^-60 and the
// phase never drifts by more than a few steps' rounding.  From start states
// that are right to the last place (CaptureState) the error against higher
// precision is that of the plain recurrence (by ring 0.8 to 1.25 times; whole
// results, nside 64 to 1024: 0.93 to 1.07 times).
// The wave-uniform coefficients (A_lm and, for the synthesis, B_l N_lm a_lm)
// come through the scalar cache, or from a row of 16 lanes, a step group ahead:
// read from LDS by every wave they kept its port (128 bytes per clock) as busy
// as the multipliers (2.45 ns per instruction and SIMD, scalar operands 2.1).
// Lanes whose scale count is > 0 are negligible (|lambda| < 2^-100): the wave
// runs a "scaled" path with rescale checks until every lane is live, then a
// check-free path of 3.5 FP64 VALU operations per (l, ring pair).
//
// nside 1024 / lmax 2048: synthesis 527 -> 408, adjoint 650 -> 531 us.

template <int K>
__device__ __forceinline__ bool all_live(const int (&sc)[K])
{
    int ok = 1;
#pragma unroll
    for (int k = 0; k < K; ++k) ok &= (sc[k] == 0);
    return __all(ok);
}
template <int K>
__device__ __forceinline__ bool rescale(double (&mu1)[K], double (&mu2)[K], int (&sc)[K])
{
    int need = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) need |= (sc[k] > 0) & (fabs(mu1[k]) > kScaleHi);
    if (!__any(need)) return false;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (sc[k] > 0 && fabs(mu1[k]) > kScaleHi) {
            mu1[k] *= kScaleDn;
            mu2[k] *= kScaleDn;
            sc[k] -= 1;
        }
    }
    return true;
}

// x^2 of a ring pair and its corrected values, from x = cos theta.
struct Ring {
    double y, ya, yb;
    __device__ __forceinline__ explicit Ring(double x)
    {
        y = x * x;
        const double d = fma(x, x, -y);
        ya = fma(8.0, d, y);
        yb = fma(8.0, fma(8.0, d, y - ya), ya);
    }
};

// Recurrence state of k_scan.
template <int K>
struct LegState {
    double mu1[K], mu2[K];  // mu_l, mu_{l-1}
    int sc[K];
};

// -------------------------------------------------------------- synthesis
template <int K>
struct SynAcc {
    double er[K], ei[K], orr[K], oi[K];
};

// Synthesis state of a lane's K ring pairs.  With step q = l - l0 of the item,
// the recurrence runs in place on v_q = s_q mu_{l0 + q}, s = + + - - + + - -
// from q = 0 (v_-1 = -mu_{l0-1}), which turns mu_q = c mu_{q-1} - mu_{q-2} into
//   u += c w (q odd),  w -= c u (q even),
// u holding the odd and w the even members.
template <int K>
struct SynState {
    double y[K], ya[K], yb[K];  // x^2 and its corrected values (Ring)
    double u[K], w[K];
    int sc[K];
    bool all;
};

// Steps J + 1 + q, q = Q0 .. Q1 - 1 (J a multiple of 4), of the 16 whose A the
// lanes hold, with scalar coefficients r, i of the G maps; x multiplies the
// steps of even l - m.  P1: parity of the odd steps' l - m.
template <int K, int G, bool P1, int J, int Q0, int Q1, int NS>
__device__ __forceinline__ void syn_steps(SynState<K>& st, SynAcc<K> (&ac)[G], const double (&x)[K], double A,
                                          const double (&r)[G][NS], const double (&i)[G][NS])
{
    for_each_map(std::make_integer_sequence<int, Q1 - Q0>{}, [&](auto qi) {
        constexpr int q = Q0 + decltype(qi)::value, j = J + q;
        constexpr bool qodd = (j & 1) == 0;       // step q = j + 1 of the item's 16
        constexpr bool odd = qodd ? P1 : !P1;     // parity of l - m
        constexpr bool minus = ((j + 1) & 2) != 0;  // s_q
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double& n = qodd ? st.u[k] : st.w[k];
            const double& p = qodd ? st.w[k] : st.u[k];
            fmac_row<j, !qodd>(n, A, odd ? p : x[k] * p);
        }
        for_each_map(std::make_integer_sequence<int, G>{}, [&](auto gi) {
            constexpr int g = decltype(gi)::value;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const double nu = minus ? -(qodd ? st.u[k] : st.w[k]) : (qodd ? st.u[k] : st.w[k]);
                if (odd) {
                    ac[g].orr[k] = fma(nu, r[g][q], ac[g].orr[k]);
                    ac[g].oi[k] = fma(nu, i[g][q], ac[g].oi[k]);
                } else {
                    ac[g].er[k] = fma(nu, r[g][q], ac[g].er[k]);
                    ac[g].ei[k] = fma(nu, i[g][q], ac[g].ei[k]);
                }
            }
        });
    });
}

// Rescale check after a row of eight steps while some lane is scaled: lanes
// above 2^900 drop by 2^-1000; a lane whose count reaches 0 clears its sums.
// Scaled lanes (count > 0) accumulate like live ones: their scaled mu
// (|mu| < 2^950 between checks) makes meaningless sums, which are cleared when
// the lane turns live and never stored while it is scaled, so the result
// equals gating each term by the lane's state at the last check, without the
// multiplies.  Eight steps multiply |mu| by at most prod (A_l + 1) < 2^50 up to
// the largest lmax, 8192 (2^49.5 at m = 8184; A_{m+1} = sqrt(2m + 3) is the
// largest factor), so from 2^900 nothing overflows between checks.  A lane
// below 2^-100 at one check is below 2^-50 at the next, where it joins: the
// terms it leaves out are below 2^-50 of lambda's O(1).
template <int K, int G>
__device__ __forceinline__ void syn_rescale(SynState<K>& st, SynAcc<K> (&ac)[G])
{
    int need = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) need |= (st.sc[k] > 0) & (fabs(st.w[k]) > kScaleHi);
    if (!__any(need)) return;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool r = st.sc[k] > 0 && fabs(st.w[k]) > kScaleHi;
        st.w[k] = r ? st.w[k] * kScaleDn : st.w[k];
        st.u[k] = r ? st.u[k] * kScaleDn : st.u[k];
        st.sc[k] -= r ? 1 : 0;
        const bool join = r && st.sc[k] == 0;
        for_each_map(std::make_integer_sequence<int, G>{}, [&](auto gi) {
            constexpr int g = decltype(gi)::value;
            ac[g].er[k] = join ? 0.0 : ac[g].er[k];
            ac[g].ei[k] = join ? 0.0 : ac[g].ei[k];
            ac[g].orr[k] = join ? 0.0 : ac[g].orr[k];
            ac[g].oi[k] = join ? 0.0 : ac[g].oi[k];
        });
    }
    st.all = all_live<K>(st.sc);
}

// Scalar loads of NS coefficients of the G maps.
template <int G, int NS>
__device__ __forceinline__ void syn_coef(scdouble* const (&a)[G], long o, double (&r)[G][NS], double (&i)[G][NS])
{
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            r[g][q] = a[g][2 * (o + q)];
            i[g][q] = a[g][2 * (o + q) + 1];
        }
}

// A group of NS steps on coefficients r, i; the next group's (nr, ni, at o of
// the rows) are loaded after the first step, whose wait would otherwise cover
// them: scalar loads return out of order, so any wait for one waits for all
// (and nothing else in the loop, such as LDS, may share their counter).
template <int K, int G, bool P1, int J, int NS>
__device__ __forceinline__ void syn_group(SynState<K>& st, SynAcc<K> (&ac)[G], const double (&x)[K], double A,
                                          const double (&r)[G][NS], const double (&i)[G][NS], scdouble* const (&a)[G],
                                          long o, double (&nr)[G][NS], double (&ni)[G][NS])
{
    // x is for the group's first even step (q = 0 or 1)
    syn_steps<K, G, P1, J, 0, 1, NS>(st, ac, x, A, r, i);
    __builtin_amdgcn_sched_barrier(0);
    syn_coef<G, NS>(a, o, nr, ni);
    syn_steps<K, G, P1, J, 1, 2, NS>(st, ac, x, A, r, i);
    syn_steps<K, G, P1, J, 2, NS, NS>(st, ac, st.y, A, r, i);
    __builtin_amdgcn_sched_barrier(0);
}

// 16 steps (two rows of eight) from step o of the rows; SCALED: a rescale
// check after each row.  xa multiplies the first even step (Ring).
template <int K, int G, bool P1, bool SCALED, int NS>
__device__ __forceinline__ void syn_block(SynState<K>& st, SynAcc<K> (&ac)[G], const double (&xa)[K], double A,
                                          scdouble* const (&a)[G], long o, double (&xr)[G][NS], double (&xi)[G][NS])
{
    double yr[G][NS], yi[G][NS];
    dpp_ready(A);
    if constexpr (NS == 8) {
        syn_group<K, G, P1, 0, NS>(st, ac, xa, A, xr, xi, a, o + 8, yr, yi);
        if (SCALED) syn_rescale<K, G>(st, ac);
        syn_group<K, G, P1, 8, NS>(st, ac, st.y, A, yr, yi, a, o + 16, xr, xi);
    } else {
        syn_group<K, G, P1, 0, NS>(st, ac, xa, A, xr, xi, a, o + 4, yr, yi);
        syn_group<K, G, P1, 4, NS>(st, ac, st.y, A, yr, yi, a, o + 8, xr, xi);
        if (SCALED) syn_rescale<K, G>(st, ac);
        syn_group<K, G, P1, 8, NS>(st, ac, st.y, A, xr, xi, a, o + 12, yr, yi);
        syn_group<K, G, P1, 12, NS>(st, ac, st.y, A, yr, yi, a, o + 16, xr, xi);
    }
    if (SCALED) syn_rescale<K, G>(st, ac);
}

// Steps l0 + 1 .. L in blocks of 16 (the rows of a are zero past L and A is
// loaded as zero there, so the last block needs no remainder): with rescale
// checks until every lane is live, then without.  A of the next block is
// loaded while a block runs.
template <int K, int G, bool P1>
__device__ __forceinline__ void syn_run(SynState<K>& st, SynAcc<K> (&ac)[G], gcdouble* __restrict__ A,
                                        scdouble* const (&a)[G], int l0, int L, int lane)
{
    constexpr int NS = G == 1 ? 8 : 4, PER = kSynChunk / 16;
    const int nblk = (L - l0 + 15) / 16;
    int l = l0 + 1 + (lane & 15);
    double A0 = l <= L ? A[l] : 0.0;
    double xr[G][NS], xi[G][NS];
    long o = l0 + 1;
    syn_coef<G, NS>(a, o, xr, xi);
    int b = 0;
    for (; b < nblk && !st.all; ++b, o += 16) {
        l += 16;
        const double A1 = l <= L ? A[l] : 0.0;
        double xa[K];
#pragma unroll
        for (int k = 0; k < K; ++k) xa[k] = b % PER == 0 ? st.yb[k] : st.ya[k];
        syn_block<K, G, P1, true, NS>(st, ac, xa, A0, a, o, xr, xi);
        A0 = A1;
    }
    while (b < nblk) {
        if (b % PER == 0) {
            l += 16;
            const double A1 = l <= L ? A[l] : 0.0;
            syn_block<K, G, P1, false, NS>(st, ac, st.yb, A0, a, o, xr, xi);
            A0 = A1;
            ++b;
            o += 16;
        }
        const int e = min(nblk, b / PER * PER + PER);
        for (; b < e; ++b, o += 16) {
            l += 16;
            const double A1 = l <= L ? A[l] : 0.0;
            syn_block<K, G, P1, false, NS>(st, ac, st.ya, A0, a, o, xr, xi);
            A0 = A1;
        }
    }
}

// Legendre synthesis of G maps of one geometry (G > 1: the recurrence runs
// once for them; item.map is then a row of gmaps).
template <int K, int G>
__global__ __launch_bounds__(64) void k_synth(const WorkItem* __restrict__ items, const MapDesc* __restrict__ maps,
                                              const int* __restrict__ gmaps)
{
    const WorkItem it = items[blockIdx.x];
    if (it.mcnt == 0) return;
    const MapDesc* mds[G];
#pragma unroll
    for (int g = 0; g < G; ++g) mds[g] = maps + (G == 1 ? it.map : gmaps[G * it.map + g]);
    const MapDesc& md = *mds[0];
    const int L = md.L;
    const int lane = threadIdx.x;
    const int m = it.m0;
    const int l0 = it.lfirst;
    gcdouble* __restrict__ A = (gcdouble*)(md.A + (moff(L, m) - m));
    scdouble* a[G];
#pragma unroll
    for (int g = 0; g < G; ++g) a[g] = (scdouble*)(mds[g]->alm + (aoff(L, m) - m));

    SynState<K> st;
    SynAcc<K> ac[G];
    int p[K];
    const bool odd0 = ((l0 - m) & 1) != 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        p[k] = it.rb * 64 * K + k * 64 + lane;
        const long q = (long)m * md.npair_pad + p[k];
        const Ring c(md.ring_x[p[k]]);
        st.y[k] = c.y;
        st.ya[k] = c.ya;
        st.yb[k] = c.yb;
        st.w[k] = md.s1_cur[q];
        st.u[k] = -md.s1_prev[q];
        st.sc[k] = md.s1_k[q];
    }
    st.all = all_live<K>(st.sc);
    // the item's first l, its parity by value
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const double ar = a[g][2 * (long)l0], ai = a[g][2 * (long)l0 + 1];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            ac[g].er[k] = odd0 ? 0.0 : st.w[k] * ar;
            ac[g].ei[k] = odd0 ? 0.0 : st.w[k] * ai;
            ac[g].orr[k] = odd0 ? st.w[k] * ar : 0.0;
            ac[g].oi[k] = odd0 ? st.w[k] * ai : 0.0;
        }
    }
    if (odd0)
        syn_run<K, G, false>(st, ac, A, a, l0, L, lane);
    else
        syn_run<K, G, true>(st, ac, A, a, l0, L, lane);
    // lanes still scaled at L store zeros
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (p[k] < md.npair) {
                const bool z = st.sc[k] != 0;
                const double x = md.ring_x[p[k]];
                double2* dst = reinterpret_cast<double2*>(mds[g]->P + ((long)p[k] * (L + 1) + m) * 4);
                dst[0] = make_double2(z ? 0.0 : ac[g].er[k], z ? 0.0 : ac[g].ei[k]);
                dst[1] = make_double2(z ? 0.0 : x * ac[g].orr[k], z ? 0.0 : x * ac[g].oi[k]);
            }
        }
}

// -------------------------------------------------------------- fused spin-2 synthesis
//
// One ring pair per lane: recurrence 1.5, T 2, field sums 12 and g 3 FP64
// instructions per l, which bound it.  The 14 coefficients of a step are
// wave-uniform; 16 steps of them sit in one row of 16 lanes, one step per lane,
// loaded a block ahead, and feed the sums through the DPP operand (fmac_row).
// Read from LDS instead they kept its read port busy longer than the multiplier
// (8 KB per wave and step), and scalar loads, of which only one step fits the
// scalar registers ahead, waited for memory.  nside 512 / lmax 1024, scalar
// loads 620, two ring pairs per lane (half the waves) 399, this form 330 us;
// with four sums per field (no g), two ring pairs and LDS 476 us.

// Sums of a ring pair by parity of l - m (0: even), one per number of a
// record: T (re, im), then S1, S2, S3 at 2, 6, 10, each E.re, E.im, B.re, B.im.
struct PolAcc {
    double v[2][kPolRec];
};

// The coefficients of 16 l-steps, one step per lane of a row of 16: A, the
// records, l - m^2 and l (l - 1) / 2.
struct PolRow {
    double A, c[kPolRec], e, h;
    __device__ __forceinline__ void load(gcdouble* Am, gcdouble* R, int l, int L)
    {
        A = l <= L ? Am[l] : 0.0;
#pragma unroll
        for (int i = 0; i < kPolRec; ++i) c[i] = R[(long)l * kPolRec + i];
    }
    // to be called before a row's first use (the c may just have been copied)
    __device__ __forceinline__ void ready(int l, double m2)
    {
        const double fl = l;
        e = fl - m2;
        h = 0.5 * (fl * (fl - 1.0));
#pragma unroll
        for (int i = 0; i < kPolRec; i += 7)
            asm volatile("" : "+v"(c[i]), "+v"(c[i + 1]), "+v"(c[i + 2]), "+v"(c[i + 3]), "+v"(c[i + 4]),
                              "+v"(c[i + 5]), "+v"(c[i + 6]));
        asm volatile("s_nop 1" : "+v"(A), "+v"(e), "+v"(h));
    }
};

// c of lane N of the lane's row of 16.
template <int N>
__device__ __forceinline__ double mov_row(double c)
{
    double r;
    asm("v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(c), "n"(N));
    return r;
}

// Step J + 1 of a block of 16 as in syn_steps (the recurrence and the T sums
// are those of k_synth, operation by operation).
template <bool P1, int J>
__device__ __forceinline__ void pol_step(SynState<1>& st, PolAcc& ac, double x, double is2, const PolRow& r)
{
    constexpr bool qodd = (J & 1) == 0, odd = qodd ? P1 : !P1, minus = ((J + 1) & 2) != 0;
    double& v = qodd ? st.u[0] : st.w[0];
    const double& p = qodd ? st.w[0] : st.u[0];
    fmac_row<J, !qodd>(v, r.A, odd ? p : x * p);
    double(&a)[kPolRec] = ac.v[odd];
    fmac_row<J, minus>(a[0], r.c[0], v);
    fmac_row<J, minus>(a[1], r.c[1], v);
    double g = mov_row<J>(r.h);  // -g
    fmac_row<J, false>(g, r.e, is2);
    g *= v;
#pragma unroll
    for (int i = 2; i < kPolRec; ++i) fmac_row<J, minus>(a[i], r.c[i], i < 6 ? g : v);
}

// syn_rescale for the spin-2 sums.
__device__ __forceinline__ void pol_rescale(SynState<1>& st, PolAcc& ac)
{
    const bool r = st.sc[0] > 0 && fabs(st.w[0]) > kScaleHi;
    if (!__any(r)) return;
    st.w[0] = r ? st.w[0] * kScaleDn : st.w[0];
    st.u[0] = r ? st.u[0] * kScaleDn : st.u[0];
    st.sc[0] -= r ? 1 : 0;
    const bool join = r && st.sc[0] == 0;
#pragma unroll
    for (int i = 0; i < kPolRec; ++i) {
        ac.v[0][i] = join ? 0.0 : ac.v[0][i];
        ac.v[1][i] = join ? 0.0 : ac.v[1][i];
    }
    st.all = all_live<1>(st.sc);
}

// A block of 16 steps; xa multiplies the first even step (Ring).
template <bool P1, bool SCALED>
__device__ __forceinline__ void pol_block(SynState<1>& st, PolAcc& ac, double xa, double is2, const PolRow& r)
{
    for_each_map(std::make_integer_sequence<int, 16>{}, [&](auto ji) {
        constexpr int j = decltype(ji)::value;
        pol_step<P1, j>(st, ac, j < 2 ? xa : st.y[0], is2, r);
        if (SCALED && (j & 7) == 7) pol_rescale(st, ac);
    });
}

// syn_run for the spin-2 sums: the same blocks, x^2 corrections and checks.
template <bool P1>
__device__ __forceinline__ void pol_run(SynState<1>& st, PolAcc& ac, gcdouble* __restrict__ A,
                                        gcdouble* __restrict__ R, double is2, double m2, int l0, int L, int lane)
{
    constexpr int PER = kSynChunk / 16;
    const int nblk = (L - l0 + 15) / 16;
    int l = l0 + 1 + (lane & 15);
    PolRow r0, r1;
    r0.load(A, R, min(l, L + 16), L);
    int b = 0;
    auto run = [&](auto scaled, PolRow& r, PolRow& n) {
        r.ready(l, m2);
        l += 16;
        n.load(A, R, min(l, L + 16), L);
        pol_block<P1, decltype(scaled)::value>(st, ac, b % PER == 0 ? st.yb[0] : st.ya[0], is2, r);
        ++b;
    };
    while (b < nblk && !st.all) {
        run(std::true_type{}, r0, r1);
        r0 = r1;
    }
    // two blocks at a time: their rows change places without copies
    while (b < nblk) {
        run(std::false_type{}, r0, r1);
        if (b >= nblk) break;
        run(std::false_type{}, r1, r0);
    }
}

// One block of 64 ring pairs (blockIdx.y) of a (m, ring block) item of the
// synthesis work list, from the item's first l: T, Q, U parity sums of its
// ring pairs into pt, pq, pu ([pair][m] (E.re, E.im, O.re, O.im), the form the
// ring stage reads; Q and U as ((north + south)/2, (north - south)/2)).
__global__ __launch_bounds__(64) void k_synth_pol(const WorkItem* __restrict__ items, const MapDesc* __restrict__ maps,
                                                  const double2* __restrict__ rec, double* __restrict__ pt,
                                                  double* __restrict__ pq, double* __restrict__ pu)
{
    const WorkItem it = items[blockIdx.x];
    if (it.mcnt == 0) return;
    const MapDesc& md = maps[it.map];
    const int L = md.L;
    const int lane = threadIdx.x;
    const int m = it.m0;
    const int l0 = it.lfirst;
    gcdouble* __restrict__ A = (gcdouble*)(md.A + (moff(L, m) - m));
    gcdouble* __restrict__ R = (gcdouble*)(rec + (aoff(L, m) - m) * (kPolRec / 2));

    const int p = (it.rb * (int)gridDim.y + (int)blockIdx.y) * 64 + lane;
    const long q = (long)m * md.npair_pad + p;
    const double x = md.ring_x[p], is2 = 1.0 / md.ring_s2[p];
    const bool odd0 = ((l0 - m) & 1) != 0;
    SynState<1> st;
    PolAcc ac;
    const Ring c(x);
    st.y[0] = c.y;
    st.ya[0] = c.ya;
    st.yb[0] = c.yb;
    st.w[0] = md.s1_cur[q];
    st.u[0] = -md.s1_prev[q];
    st.sc[0] = md.s1_k[q];
    st.all = all_live<1>(st.sc);
    const double m2 = (double)m * m;
    // the item's first l, its parity by value
    {
        const double fl = l0, h = 0.5 * (fl * (fl - 1.0));
        const double g = st.w[0] * fma(fl - m2, is2, h);
#pragma unroll
        for (int i = 0; i < kPolRec; ++i) {
            const double t = (i >= 2 && i < 6 ? g : st.w[0]) * R[(long)l0 * kPolRec + i];
            ac.v[0][i] = odd0 ? 0.0 : t;
            ac.v[1][i] = odd0 ? t : 0.0;
        }
    }
    if (odd0)
        pol_run<false>(st, ac, A, R, is2, m2, l0, L, lane);
    else
        pol_run<true>(st, ac, A, R, is2, m2, l0, L, lane);
    // epilogue: north (E + O at c) and south (E - O at -c); lanes still scaled
    // at L store zeros
    if (p >= md.npair) return;
    const double fm = m;
    const long o = ((long)p * (L + 1) + m) * 4;
    const bool z = st.sc[0] != 0;
    double e[kPolRec], d[kPolRec];
#pragma unroll
    for (int i = 0; i < kPolRec; ++i) {
        e[i] = z ? 0.0 : ac.v[0][i];
        d[i] = z ? 0.0 : x * ac.v[1][i];
    }
    *reinterpret_cast<double4*>(pt + o) = make_double4(e[0], e[1], d[0], d[1]);
    double W[2][2][2], X[2][2][2];  // [field][north/south][re/im]
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const double sg = s ? -1.0 : 1.0;  // south: E - O, c -> -c
            const double ch = sg * x;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int b = 2 + 2 * f + r;
                const double S1 = e[b] + sg * d[b], S2 = e[b + 4] + sg * d[b + 4];  // S1: its negative
                const double S3 = e[b + 8] + sg * d[b + 8];
                W[f][s][r] = ch * is2 * S2 - S1;
                X[f][s][r] = fm * is2 * (S2 - ch * S3);
            }
        }
    }
    // Q = -(W_E + i X_B), U = -(W_B - i X_E)
    double Q[2][2], U[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        Q[s][0] = -(W[0][s][0] - X[1][s][1]);
        Q[s][1] = -(W[0][s][1] + X[1][s][0]);
        U[s][0] = -(W[1][s][0] + X[0][s][1]);
        U[s][1] = -(W[1][s][1] - X[0][s][0]);
    }
    *reinterpret_cast<double4*>(pq + o) = make_double4(0.5 * (Q[0][0] + Q[1][0]), 0.5 * (Q[0][1] + Q[1][1]),
                                                       0.5 * (Q[0][0] - Q[1][0]), 0.5 * (Q[0][1] - Q[1][1]));
    *reinterpret_cast<double4*>(pu + o) = make_double4(0.5 * (U[0][0] + U[1][0]), 0.5 * (U[0][1] + U[1][1]),
                                                       0.5 * (U[0][0] - U[1][0]), 0.5 * (U[0][1] - U[1][1]));
}

// -------------------------------------------------------------- adjoint
// u_lm = sum over ring pairs of lambda_lm Psi_m.  One wavefront takes one
// degree m of a block of 64 K ring pairs, lane j holding the pairs 64 k + j,
// and walks l in rows of eight steps; each lane adds its K products per step
// and the row's 16 sums (8 steps, real and imaginary) are then reduced over
// the 64 lanes and stored as the block's partial u.
//
// What bounds it: FP64 VALU issue, 3.5 instructions per (l, ring pair) plus
// about 60 issue slots per row for the reduction, whatever K: K = 8 halves
// the reduction's share against K = 4 (28 K against 60 slots per row).  Its
// 512-pair blocks would start all their pairs at the earliest live l of the
// block; instead each group k of 64 pairs joins at the row of its own first
// live l (AdjItem::row), so the skipped range is that of 64-pair blocks.  The
// registers of K = 8 (about 200) allow two waves per SIMD, enough here: eight
// independent chains per wave.  The recurrence coefficients are wave-uniform
// and come through the scalar cache a row ahead; LDS carries the reduction
// tile and the ring constants.

// A lane's ring-stage inputs Psi_m (even and odd parts, the odd one times x)
// of its K ring pairs.  Lanes whose scale count is > 0 hold
// zeros, so that the same step serves the scaled and the live path: their
// scaled mu (|mu| < 2^950 between rescale checks) times 0 contributes exactly
// 0.  A lane that turns live loads its inputs at the rescale check where its
// count reaches 0.
template <int K>
struct AdjState {
    double y[K];           // x^2
    double mu1[K], mu2[K]; // mu_{l-1}, mu_{l-2} before step l, odd ones divided by x
    double per[K], pei[K], por[K], poi[K];
    int sc[K];
};

template <int K>
__device__ __forceinline__ void adj_load_in(AdjState<K>& st, int k, const AdjItem& it, int lane)
{
    const int p = it.p0 + k * 64 + lane;
    double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
    if (p < it.npair) {
        gcdouble* src = gview(it.Q) + (long)p * 4 * (it.L + 1);
        const double x = gview(it.x)[p];
        v0 = src[0];
        v1 = src[1];
        v2 = x * src[2];
        v3 = x * src[3];
    }
    // one unconditional store per field: stores in both arms of a branch
    // would be merged through a pointer and keep the inputs in memory
    st.per[k] = v0;
    st.pei[k] = v1;
    st.por[k] = v2;
    st.poi[k] = v3;
}

// Rescale check of the groups k >= K - KA: lanes above 2^900 drop by 2^-1000;
// a lane whose count reaches 0 loads its inputs.  Returns whether all are live.
// (Checking only the groups that still hold scaled lanes, by a branch each,
// made the register allocator copy the state at every merge: 40 more VGPRs at
// K = 8, spills, 115 against 105 us at nside 512.)
template <int K, int KA>
__device__ __forceinline__ bool adj_rescale(AdjState<K>& st, const AdjItem& it, int lane)
{
    int need = 0;
#pragma unroll
    for (int k = K - KA; k < K; ++k) need |= (st.sc[k] > 0) & (fabs(st.mu1[k]) > kScaleHi);
    if (__any(need)) {
#pragma unroll
        for (int k = K - KA; k < K; ++k) {
            if (st.sc[k] > 0 && fabs(st.mu1[k]) > kScaleHi) {
                st.mu1[k] *= kScaleDn;
                st.mu2[k] *= kScaleDn;
                st.sc[k] -= 1;
                if (st.sc[k] == 0) adj_load_in<K>(st, k, it, lane);
            }
        }
    }
    int ok = 1;
#pragma unroll
    for (int k = K - KA; k < K; ++k) ok &= (st.sc[k] == 0);
    return __all(ok);
}

// Rows of eight steps.  Steps 2p and 2p + 1 are folded as soon as both exist,
// once over lane pairs (j, j + 32) with permlane32 swaps (fold_pair): z[2p + c]
// then holds step 2p in lanes 0..31 and step 2p + 1 in lanes 32..63 (c = 0
// real, 1 imaginary).  tile_store puts lane L's four (re, im) records as
// records (q, L & 31), q = 2p + (L >> 5), at index 33 q + (L & 31); tile_load
// gives lane j the records (j & 7, 4 (j >> 3) + r), r < 4 (the skew of one
// record per q puts the eight lanes of a read on distinct banks); finish_row
// sums them and completes the sum over the eight lanes that share j & 7
// (distances 32, 16, 8): the real part ends in lanes 0..31, the imaginary part
// in lanes 32..63.  A permlane swap costs about 1.2 to 1.6 FP64 issue slots, so
// the tile carries the second fold: 20 swaps per row instead of 28, for 4 KB of
// LDS traffic each way.
constexpr int kAdjTile = 33 * 7 + 32;  // records of the row tile

struct AdjRed {
    double2* tile;
    gdouble* dst;  // output row, dst[2 l], dst[2 l + 1]
    int l, lend, lane;
    __device__ __forceinline__ void tile_store(const double (&z)[8])
    {
        double2* t = tile + 33 * (lane >> 5) + (lane & 31);
#pragma unroll
        for (int p = 0; p < 4; ++p) t[66 * p] = make_double2(z[2 * p], z[2 * p + 1]);
        wave_sync();
    }
    __device__ __forceinline__ void tile_load(double2 (&t4)[4]) const
    {
        const double2* t = tile + 33 * (lane & 7) + 4 * (lane >> 3);
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[r] = t[r];
    }
    __device__ __forceinline__ void finish_row(const double2 (&t4)[4])
    {
        const double re = (t4[0].x + t4[1].x) + (t4[2].x + t4[3].x);
        const double im = (t4[0].y + t4[1].y) + (t4[2].y + t4[3].y);
        double s = swap32_add(re, im);
        s = swap16_add(s, s);
        s = ror_add<8>(s);
        // four lanes hold each value and store it
        const int lr = l + (lane & 7);
        if (lr <= lend) dst[2 * (long)lr + (lane >> 5)] = s;
        l += 8;
    }
};

// Step j of a row on the groups k >= K - KA, returning the lane's sums.  Rows
// start at even l - m, so j's parity is that of l - m.
template <int K, int KA>
__device__ __forceinline__ void adj_step(AdjState<K>& st, bool odd, double A, const double (&y)[K], double& sr,
                                         double& si)
{
    sr = 0.0;
    si = 0.0;
#pragma unroll
    for (int k = K - KA; k < K; ++k) {
        const double nu = fma(odd ? A : A * y[k], st.mu1[k], -st.mu2[k]);
        st.mu2[k] = st.mu1[k];
        st.mu1[k] = nu;
        sr = fma(nu, odd ? st.por[k] : st.per[k], sr);
        si = fma(nu, odd ? st.poi[k] : st.pei[k], si);
    }
}

// Rows r .. rend - 1 with KA groups; SCALED: with a rescale check after each
// row, until every lane is live.  a holds row r's coefficients; a row loads
// the next one's after its first step (scalar loads return out of order: the
// wait before that step would otherwise cover them), and reads the previous
// row's tile there, which it finishes halfway.  What eight steps can
// multiply |mu| by, and what a lane that joins at a row's end leaves out, is as
// in syn_rescale.
template <int K, int KA, bool SCALED>
__device__ __forceinline__ bool adj_rows(AdjState<K>& st, AdjRed& rd, const AdjItem& it, scdouble* A, double (&a)[8],
                                         const double* yl, int& r, int rend, bool all)
{
    double2 t4[4];
    bool pend = false;
    const int lane = rd.lane;
    // multipliers of a row's first step: x^2, in every second row its
    // corrected values (Ring)
    double y0[K];
    auto load_y0 = [&](int row) {
        const double* src = yl + ((row & 1) ? 0 : (row & 15) ? 64 * K : 128 * K) + lane;
#pragma unroll
        for (int k = K - KA; k < K; ++k) y0[k] = src[64 * k];
    };
    load_y0(r);
    while (r < rend && !(SCALED && all)) {
        double z[8], are, aim, bre, bim, an[8];
        adj_step<K, KA>(st, false, a[0], y0, are, aim);
        __builtin_amdgcn_sched_barrier(0);
        if (pend) rd.tile_load(t4);
#pragma unroll
        for (int q = 0; q < 8; ++q) an[q] = A[8 * (long)(r + 1) + q];
        adj_step<K, KA>(st, true, a[1], st.y, bre, bim);
        z[0] = swap32_add(are, bre);
        z[1] = swap32_add(aim, bim);
        adj_step<K, KA>(st, false, a[2], st.y, are, aim);
        adj_step<K, KA>(st, true, a[3], st.y, bre, bim);
        z[2] = swap32_add(are, bre);
        z[3] = swap32_add(aim, bim);
        if (pend) rd.finish_row(t4);
        adj_step<K, KA>(st, false, a[4], st.y, are, aim);
        __builtin_amdgcn_sched_barrier(0);
        load_y0(r + 1);
        adj_step<K, KA>(st, true, a[5], st.y, bre, bim);
        z[4] = swap32_add(are, bre);
        z[5] = swap32_add(aim, bim);
        adj_step<K, KA>(st, false, a[6], st.y, are, aim);
        adj_step<K, KA>(st, true, a[7], st.y, bre, bim);
        z[6] = swap32_add(are, bre);
        z[7] = swap32_add(aim, bim);
        rd.tile_store(z);
        pend = true;
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = an[q];
        ++r;
        if (SCALED) all = adj_rescale<K, KA>(st, it, lane);
    }
    if (pend) {
        rd.tile_load(t4);
        rd.finish_row(t4);
        wave_sync();
    }
    return all;
}

// The rows in which KA groups of ring pairs run, then those with more.
template <int K, int KA>
__device__ __forceinline__ void adj_phase(AdjState<K>& st, AdjRed& rd, const AdjItem& it, scdouble* A, double (&a)[8],
                                          const double* yl, int& r)
{
    const int rend = KA < K ? it.row[K - KA - 1] : it.nrow;
    if (r < rend) {
        int ok = 1;
#pragma unroll
        for (int k = K - KA; k < K; ++k) ok &= (st.sc[k] == 0);
        bool all = __all(ok);
        if (!all) all = adj_rows<K, KA, true>(st, rd, it, A, a, yl, r, rend, all);
        if (r < rend) adj_rows<K, KA, false>(st, rd, it, A, a, yl, r, rend, all);
    }
    if constexpr (KA < K) adj_phase<K, KA + 1>(st, rd, it, A, a, yl, r);
}

template <int K>
__global__ __launch_bounds__(64, K == 8 ? 2 : K == 4 ? 3 : 4) void k_adj(const AdjItem* __restrict__ items)
{
    __shared__ double2 tile[kAdjTile];
    __shared__ double yl[3 * K * 64];
    const AdjItem it = items[blockIdx.x];
    if (it.nrow == 0) return;
    const int lane = threadIdx.x;
    AdjState<K> st;
    const auto sv = gview(it.st) + lane;
    const __attribute__((address_space(1))) int* sk = (const __attribute__((address_space(1))) int*)it.sk + lane;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double2 v = sv[64 * k];
        st.mu2[k] = v.x;
        st.mu1[k] = v.y;
        st.sc[k] = sk[64 * k];
        const Ring c(gview(it.x)[it.p0 + 64 * k + lane]);
        st.y[k] = c.y;
        yl[64 * k + lane] = c.y;
        yl[64 * (K + k) + lane] = c.ya;
        yl[64 * (2 * K + k) + lane] = c.yb;
        adj_load_in<K>(st, k, it, lane);
    }
    // lanes still scaled start from zero inputs
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool z = st.sc[k] != 0;
        st.per[k] = z ? 0.0 : st.per[k];
        st.pei[k] = z ? 0.0 : st.pei[k];
        st.por[k] = z ? 0.0 : st.por[k];
        st.poi[k] = z ? 0.0 : st.poi[k];
    }
    wave_sync();
    AdjRed rd;
    rd.tile = tile;
    rd.dst = (gdouble*)it.u;
    rd.l = it.l0;
    rd.lend = it.lend;
    rd.lane = lane;
    scdouble* A = (scdouble*)(it.A + it.l0);
    double a[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) a[q] = A[q];
    int r = 0;
    adj_phase<K, 1>(st, rd, it, A, a, yl, r);
}

// -------------------------------------------------------------- Legendre stages on the matrix cores
//
// Maps of one geometry share lambda_lm(theta), so the Legendre sums of a group
// of up to kSynG = 8 such maps are matrix products with 16 columns c = (map,
// re / im), done by v_mfma_f64_16x16x4f64: lane layout A[i][k] from lane
// i + 16 k, B[k][j] from lane j + 16 k, D[i][j] in lane j + 16 (i % 4),
// register i / 4.  The recurrence of each 64 ring pairs runs once for the group
// into an LDS tile of kMmaSteps l-steps.  FP64 matrix and vector instructions
// share the multipliers (a mixture takes the sum of both times), so the gain is
// the shared recurrence and, in the adjoint, the sum over ring pairs inside
// the instruction: 16 maps of nside 256 / lmax 512 take 158 us against 285 us
// map by map (k_adj<8>), the synthesis 134 against 160 us in pairs.
constexpr int kMmaSteps = 32;
constexpr int kMmaRow = 65;   // adjoint tile row: the 16 rows of one parity start 4 banks apart
constexpr int kMmaRowS = 72;  // synthesis tile row: rows two apart start 32 banks apart

typedef double dbl4 __attribute__((ext_vector_type(4)));

// Rescale check of a scaled lane (every 8 steps), without branches.
__device__ __forceinline__ void mma_rescale(double& mu1, double& mu2, int& sc, double& g, bool& all)
{
    const bool r = sc > 0 && fabs(mu1) > kScaleHi;
    mu1 = r ? mu1 * kScaleDn : mu1;
    mu2 = r ? mu2 * kScaleDn : mu2;
    sc -= r ? 1 : 0;
    g = sc == 0 ? 1.0 : 0.0;
    all = __all(sc == 0);
}

// kMmaSteps recurrence steps of one ring pair into tile column `lane`: row s
// holds lambda at l = c0 + s.  SCALED: times the gate, rescale checks every 8
// steps.  Coefficients are read from LDS eight steps ahead of their use.
// The matrix-core kernels run the recursion in its plain form, mu_l = A_l x
// mu_{l-1} - mu_{l-2} (the states' odd values times x): between matrix
// instructions the products A_l x are free, and the divided form with its
// direct coefficients was slower (8 maps, nside 256: synthesis 134 and 141 us,
// adjoint 158 and 163 us).
template <bool SCALED, int RS>
__device__ __forceinline__ void mma_fill(double* __restrict__ T, const double* __restrict__ cA, int lane, double x,
                                         double& mu1, double& mu2, int& sc, double& g, bool& all)
{
    double c[8], cn[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = cA[u];
#pragma unroll
    for (int s8 = 0; s8 < kMmaSteps; s8 += 8) {
        if (s8 + 8 < kMmaSteps) {
#pragma unroll
            for (int u = 0; u < 8; ++u) cn[u] = cA[s8 + 8 + u];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double nu = fma(c[u] * x, mu1, -mu2);
            mu2 = mu1;
            mu1 = nu;
            T[(s8 + u) * RS + lane] = SCALED ? mu1 * g : mu1;
        }
        if (SCALED) mma_rescale(mu1, mu2, sc, g, all);
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = cn[u];
    }
}

// The synthesis' first tile: row 0 is the start state itself, later rows advance.
__device__ __forceinline__ void mma_fill_first(double* __restrict__ T, const double* __restrict__ cA, int lane,
                                               double x, double& mu1, double& mu2, int& sc, double& g, bool& all)
{
#pragma unroll
    for (int s = 0; s < kMmaSteps; ++s) {
        if (s > 0) {
            const double nu = fma(cA[s] * x, mu1, -mu2);
            mu2 = mu1;
            mu1 = nu;
        }
        T[s * kMmaRowS + lane] = mu1 * g;
        if ((s & 7) == 7) mma_rescale(mu1, mu2, sc, g, all);
    }
}

// A wave's first tile of the adjoint: rows below its first row r0 (even) are
// zero, later rows advance from (mu_{l-2}, mu_{l-1}) at row r0.
__device__ __forceinline__ void mma_fill_from(double* __restrict__ T, const double* __restrict__ cA, int lane, int r0,
                                              double x, double& mu1, double& mu2, int& sc, double& g, bool& all)
{
#pragma unroll
    for (int s = 0; s < kMmaSteps; ++s) {
        const bool adv = s >= r0;
        const double nu = fma(cA[s] * x, mu1, -mu2);
        mu2 = adv ? mu1 : mu2;
        mu1 = adv ? nu : mu1;
        T[s * kMmaRow + lane] = adv ? mu1 * g : 0.0;
        if ((s & 7) == 7) mma_rescale(mu1, mu2, sc, g, all);
    }
}

// Shared adjoint: U[l][c] = sum_p Lambda[l][p] Psi[p][c] for one (m, block of 64
// ring pairs) per wave; the 16 rows of one parity of a tile are the A operands
// and the Psi of the block's ring pairs stay in registers as B operands for
// the whole item.  A workgroup is kMmaWaves waves on consecutive blocks of
// one m, each starting at its own first live l (even l - m) on a common grid
// of tiles; their products are added in LDS in wave order, so one partial per
// kMmaWaves blocks goes to memory.
__global__ __launch_bounds__(64 * kMmaWaves, 2) void k_adj_mma(const WorkItem* __restrict__ items,
                                                               const MmaSub* __restrict__ subs,
                                                               const MapDesc* __restrict__ maps,
                                                               const int* __restrict__ groups)
{
    __shared__ double T[kMmaWaves][kMmaSteps * kMmaRow];
    __shared__ double sA[2][kMmaSteps];
    const WorkItem it = items[blockIdx.x];
    if (it.mcnt == 0) return;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int* __restrict__ gm = groups + kSynG * it.map;
    const MapDesc& md = maps[gm[0]];
    const int L = md.L;
    const int m = it.m0;
    const int l0 = it.lfirst;  // the earliest start of the workgroup's blocks, even l - m
    const long base = moff(L, m) - m;
    gcdouble* __restrict__ A = (gcdouble*)(md.A + base);
    const MmaSub& sub = subs[it.sub];
    const int lfw = sub.lf[w];             // this wave's first l, -1: no live item
    const int rb = it.rb * kMmaWaves + w;  // this wave's 64-pair block
    double* __restrict__ Tw = T[w];

    // the recurrence of ring pair rb * 64 + lane, from the wave's start state
    // (a wave without a live item may lie past the ring tables)
    double x = 0.0, mu1 = 0.0, mu2 = 0.0;
    int sc = 1;
    if (lfw >= 0) {
        x = md.ring_x[rb * 64 + lane];
        const double2 v = sub.st[w][lane];
        mu2 = v.x;
        mu1 = v.y * x;  // l - m odd
        sc = sub.sk[w][lane];
    }
    double g = sc == 0 ? 1.0 : 0.0;
    bool all = __all(sc == 0);

    // B operands: B[k][j] = Psi of ring pair rb * 64 + 4 b + k, column j =
    // (map j / 2 of the group, re / im j % 2); a group's empty columns (entry
    // -1) hold zeros and are not stored
    const int j = lane & 15, kq = lane >> 4;
    const int mapj = gm[j >> 1];
    const MapDesc& mj = maps[mapj >= 0 ? mapj : gm[0]];
    double bE[16], bO[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) bE[b] = bO[b] = 0.0;
    if (lfw >= 0 && mapj >= 0) {
        const long row = 4 * (long)(L + 1);
        // padding pairs (past npair) read the last ring pair's row and are
        // zeroed afterwards, so that all loads are issued together
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const int pp = min(rb * 64 + 4 * b + kq, md.npair - 1);
            gcdouble* src = (gcdouble*)(mj.Q + (long)pp * row + 4 * (long)m + (j & 1));
            bE[b] = src[0];
            bO[b] = src[2];
        }
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const bool pad = rb * 64 + 4 * b + kq >= md.npair;
            bE[b] = pad ? 0.0 : bE[b];
            bO[b] = pad ? 0.0 : bO[b];
        }
    }
    // this workgroup's partial (kMmaWaves blocks), written by wave 0
    gdouble* __restrict__ dst = (gdouble*)(mj.upart + 2 * ((long)it.rb * md.nalm + base) + (j & 1));

    // coefficients of the current tile in sA[buf], of the next one in tA
    const int t = threadIdx.x;
    double tA = 0.0;
    if (t < kMmaSteps) {
        sA[0][t] = (l0 + t <= L) ? A[l0 + t] : 0.0;
        tA = (l0 + kMmaSteps + t <= L) ? A[l0 + kMmaSteps + t] : 0.0;
    }
    __syncthreads();
    int buf = 0;
    for (int c0 = l0; c0 <= L; c0 += kMmaSteps) {
        const int n2 = c0 + 2 * kMmaSteps;
        // tile rows past L hold finite values that no stored output uses
        const bool active = lfw >= 0 && lfw < c0 + kMmaSteps;
        if (active) {
            if (lfw >= c0)
                mma_fill_from(Tw, sA[buf], lane, lfw - c0, x, mu1, mu2, sc, g, all);
            else if (all)
                mma_fill<false, kMmaRow>(Tw, sA[buf], lane, x, mu1, mu2, sc, g, all);
            else
                mma_fill<true, kMmaRow>(Tw, sA[buf], lane, x, mu1, mu2, sc, g, all);
        }
        wave_sync();
        dbl4 dE = {0.0, 0.0, 0.0, 0.0}, dO = {0.0, 0.0, 0.0, 0.0};
        if (active) {
            // the ring-pair sums, 16 l-rows of each parity (even rows first)
            const double* tE = Tw + 2 * j * kMmaRow + kq;
            const double* tO = tE + kMmaRow;
            double aE[16], aO[16];
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                aE[b] = tE[4 * b];
                aO[b] = tO[4 * b];
            }
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                dE = __builtin_amdgcn_mfma_f64_16x16x4f64(aE[b], bE[b], dE, 0, 0, 0);
                dO = __builtin_amdgcn_mfma_f64_16x16x4f64(aO[b], bO[b], dO, 0, 0, 0);
            }
        }
        // waves 1.. hand their sums to wave 0 through their own tile (its
        // A operands are in registers; LDS runs a wave's operations in order)
        if (w > 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Tw[r * 64 + lane] = dE[r];
                Tw[(4 + r) * 64 + lane] = dO[r];
            }
        }
        __syncthreads();
        if (w == 0) {
#pragma unroll
            for (int v = 1; v < kMmaWaves; ++v) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    dE[r] += T[v][r * 64 + lane];
                    dO[r] += T[v][(4 + r) * 64 + lane];
                }
            }
            // row i = kq + 4 r of each parity: l = c0 + 2 i (+ 1)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int lE = c0 + 2 * (kq + 4 * r);
                if (mapj >= 0 && lE <= L) dst[2 * (long)lE] = dE[r];
                if (mapj >= 0 && lE + 1 <= L) dst[2 * (long)lE + 2] = dO[r];
            }
        }
        if (t < kMmaSteps) {
            sA[buf ^ 1][t] = tA;
            tA = (n2 + t <= L) ? A[n2 + t] : 0.0;
        }
        __syncthreads();
        buf ^= 1;
    }
}

// -------------------------------------------------------------- shared synthesis on the matrix cores
//
// The synthesis of a group of up to kSynG = 8 maps of one geometry (a smaller
// group leaves columns empty) as matrix products: for a block of 64 ring
// pairs, P[p][c] = sum_l Lambda[l][p] a_l[c] per parity, c = (map, re / im),
// accumulated over the item's l range in registers.  Each lane runs the
// recurrence of one ring pair (once for the group) into an LDS tile of
// kMmaSteps l-steps; an instruction takes 16 ring pairs by 4
// l-steps of one parity (A, read across the tile's rows) times those 4
// l-steps' a_lm of the 8 maps (B, from global memory, a tile ahead).  A tile
// is 2 parities x 4 groups of 4 l-steps x 4 blocks of 16 pairs = 32
// instructions; the item's sums (E, O per pair and map) are stored once at
// its end.  No sums cross waves, so a workgroup is one wave; an item of K
// ring pairs per lane runs as K workgroups, all from the item's first l.
template <int K>
__global__ __launch_bounds__(64, 2) void k_synth_mma(const WorkItem* __restrict__ items,
                                                     const MapDesc* __restrict__ maps, const int* __restrict__ groups)
{
    __shared__ double T[kMmaSteps * kMmaRowS];
    __shared__ double sA[2][kMmaSteps];
    const WorkItem it = items[blockIdx.x / K];
    if (it.mcnt == 0) return;
    const int w = blockIdx.x % K;
    const int* __restrict__ gm = groups + kSynG * it.map;
    const MapDesc& md = maps[gm[0]];
    const int L = md.L;
    const int m = it.m0;
    const int l0 = it.lfirst;
    const int lane = threadIdx.x;
    const long base = moff(L, m) - m;
    gcdouble* __restrict__ A = (gcdouble*)(md.A + base);
    const int pbase = it.rb * 64 * K + 64 * w;  // this wave's 64 ring pairs

    // the recurrence of ring pair pbase + lane, from the item's start state
    const long q = (long)m * md.npair_pad + pbase + lane;
    const double x = md.ring_x[pbase + lane];
    double mu1 = md.s1_cur[q], mu2 = md.s1_prev[q];
    if ((l0 - m) & 1)
        mu1 *= x;
    else
        mu2 *= x;
    int sc = md.s1_k[q];
    double g = sc == 0 ? 1.0 : 0.0;
    bool all = __all(sc == 0);

    // B operands: B[k][j] = a_l of column j = (map j / 2, re / im j % 2) at
    // the k-th l-step of a group; empty columns hold zeros and are not stored
    const int j = lane & 15, kq = lane >> 4;
    const int mapj = gm[j >> 1];
    gcdouble* __restrict__ aj = (gcdouble*)(maps[mapj >= 0 ? mapj : gm[0]].alm + (aoff(L, m) - m)) + (j & 1);
    auto load_b = [&](int c0, double(&bE)[4], double(&bO)[4]) {
        const int sE = (c0 - m) & 1;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const int lE = c0 + sE + 2 * (4 * h + kq), lO = c0 + (sE ^ 1) + 2 * (4 * h + kq);
            const double e = aj[2 * (long)min(lE, L)], o = aj[2 * (long)min(lO, L)];
            bE[h] = (mapj >= 0 && lE <= L) ? e : 0.0;
            bO[h] = (mapj >= 0 && lO <= L) ? o : 0.0;
        }
    };
    double bE[4], bO[4], nE[4], nO[4];
    load_b(l0, bE, bO);

    dbl4 dE[4], dO[4];
#pragma unroll
    for (int pb = 0; pb < 4; ++pb) dE[pb] = dO[pb] = dbl4{0.0, 0.0, 0.0, 0.0};

    // coefficients of the current tile in sA[buf], of the next one in tA
    double tA = 0.0;
    if (lane < kMmaSteps) {
        sA[0][lane] = (l0 + lane <= L) ? A[l0 + lane] : 0.0;
        tA = (l0 + kMmaSteps + lane <= L) ? A[l0 + kMmaSteps + lane] : 0.0;
    }
    wave_sync();
    int buf = 0;
    for (int c0 = l0; c0 <= L; c0 += kMmaSteps) {
        const int n2 = c0 + 2 * kMmaSteps;
        if (c0 + kMmaSteps <= L) load_b(c0 + kMmaSteps, nE, nO);
        // tile rows past L hold finite values whose B operands are zero
        if (c0 == l0)
            mma_fill_first(T, sA[buf], lane, x, mu1, mu2, sc, g, all);
        else if (all)
            mma_fill<false, kMmaRowS>(T, sA[buf], lane, x, mu1, mu2, sc, g, all);
        else
            mma_fill<true, kMmaRowS>(T, sA[buf], lane, x, mu1, mu2, sc, g, all);
        wave_sync();
        const int sE = (c0 - m) & 1;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const double* tE = T + (sE + 2 * (4 * h + kq)) * kMmaRowS + j;
            const double* tO = T + ((sE ^ 1) + 2 * (4 * h + kq)) * kMmaRowS + j;
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                dE[pb] = __builtin_amdgcn_mfma_f64_16x16x4f64(tE[16 * pb], bE[h], dE[pb], 0, 0, 0);
                dO[pb] = __builtin_amdgcn_mfma_f64_16x16x4f64(tO[16 * pb], bO[h], dO[pb], 0, 0, 0);
            }
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            bE[h] = nE[h];
            bO[h] = nO[h];
        }
        if (lane < kMmaSteps) {
            sA[buf ^ 1][lane] = tA;
            tA = (n2 + lane <= L) ? A[n2 + lane] : 0.0;
        }
        wave_sync();
        buf ^= 1;
    }
    // D[i][j] lands in lane j + 16 (i % 4), register i / 4: ring pair
    // pbase + 16 pb + kq + 4 r
    if (mapj >= 0) {
        gdouble* __restrict__ P = (gdouble*)maps[mapj].P;
#pragma unroll
        for (int pb = 0; pb < 4; ++pb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int pair = pbase + 16 * pb + kq + 4 * r;
                if (pair < md.npair) {
                    const long o = ((long)pair * (L + 1) + m) * 4 + (j & 1);
                    P[o] = dE[pb][r];
                    P[o + 2] = dO[pb][r];
                }
            }
    }
}

// -------------------------------------------------------------- set-up passes
// All run the scaled recurrence from the seed lambda_mm.

// The start states' recurrence (odd members divided by cos theta = c) carries
// each value as a sum hi + lo and c^2 = y + d exactly: a start state's error is
// that of every l after it.  (Plain doubles cannot hold the correction of y: the
// fma that adds it to mu_{l-2} rounds it away, and its drift grew with l.)
template <int K>
struct CaptureState {
    double h1[K], e1[K], h2[K], e2[K];  // mu_l and mu_{l-1}, hi and lo
    int sc[K];
};

// hi + lo of q + b + lo
__device__ __forceinline__ void two_sum(double q, double b, double lo, double& hi, double& e)
{
#pragma clang fp contract(off)
    const double s = q + b, t = s - q;
    const double r = ((q - (s - t)) + (b - t)) + lo;
    hi = s + r;
    e = r - (hi - s);
}

template <int K>
__device__ __forceinline__ void capture_step(CaptureState<K>& st, const double (&c)[K], bool odd, double Al)
{
#pragma clang fp contract(off)  // q is rounded before the sum
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double p = st.h1[k], e = st.e1[k];
        if (!odd) {
            const double y = c[k] * c[k], d = fma(c[k], c[k], -y);
            p = y * st.h1[k];
            e = fma(y, st.h1[k], -p) + fma(y, st.e1[k], d * st.h1[k]);
        }
        const double q = Al * p;
        const double f = fma(Al, p, -q) + Al * e;
        double h, l;
        two_sum(q, -st.h2[k], f - st.e2[k], h, l);
        st.h2[k] = st.h1[k];
        st.e2[k] = st.e1[k];
        st.h1[k] = h;
        st.e1[k] = l;
        // as rescale()
        const bool r = st.sc[k] > 0 && fabs(h) > kScaleHi;
        const double f2 = r ? kScaleDn : 1.0;
        st.h1[k] *= f2;
        st.e1[k] *= f2;
        st.h2[k] *= f2;
        st.e2[k] *= f2;
        st.sc[k] -= r ? 1 : 0;
    }
}

// k_scan: first l at which each ring pair becomes live (L+1 if never).
template <int K>
__global__ __launch_bounds__(64) void k_scan(const WorkItem* __restrict__ items, const MapDesc* __restrict__ maps,
                                             int* __restrict__ lstart)
{
    const WorkItem it = items[blockIdx.x];
    const MapDesc& md = maps[it.map];
    const int L = md.L;
    const int npad = md.npair_pad;
    const int lane = threadIdx.x;
    for (int mi = 0; mi < it.mcnt; ++mi) {
        const int m = it.m0 + mi;
        const double* __restrict__ A = md.A + moff(L, m) - m;
        LegState<K> st;
        double x[K];
        int p[K], ls[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            p[k] = it.rb * 64 * K + k * 64 + lane;
            x[k] = md.ring_x[p[k]];
            st.mu1[k] = md.seed_v[(long)m * npad + p[k]];
            st.sc[k] = md.seed_k[(long)m * npad + p[k]];
            st.mu2[k] = 0.0;
            ls[k] = st.sc[k] == 0 ? m : L + 1;
        }
        bool all = all_live<K>(st.sc);
        int l = m;
        while (!all && l < L) {
            ++l;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const double nu = fma(A[l] * x[k], st.mu1[k], -st.mu2[k]);
                st.mu2[k] = st.mu1[k];
                st.mu1[k] = nu;
            }
            if (rescale<K>(st.mu1, st.mu2, st.sc)) {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (st.sc[k] == 0 && ls[k] > L) ls[k] = l + 1;
                all = all_live<K>(st.sc);
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) lstart[(long)m * npad + p[k]] = ls[k];
    }
}

// k_capture: the state (mu_{l-1}, mu_l, scale count) at l = item.lfirst.
template <int K>
__global__ __launch_bounds__(64) void k_capture(const WorkItem* __restrict__ items, const MapDesc* __restrict__ maps,
                                                double* __restrict__ prev, double* __restrict__ cur,
                                                int* __restrict__ kout)
{
    const WorkItem it = items[blockIdx.x];
    if (it.mcnt == 0) return;
    const MapDesc& md = maps[it.map];
    const int L = md.L;
    const int npad = md.npair_pad;
    const int lane = threadIdx.x;
    const int m = it.m0;
    const double* __restrict__ A = md.A + moff(L, m) - m;
    CaptureState<K> st;
    int p[K];
    double c[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        p[k] = it.rb * 64 * K + k * 64 + lane;
        c[k] = md.ring_x[p[k]];
        st.h1[k] = md.seed_v[(long)m * npad + p[k]];
        st.sc[k] = md.seed_k[(long)m * npad + p[k]];
        st.e1[k] = st.h2[k] = st.e2[k] = 0.0;
    }
    for (int l = m + 1; l <= it.lfirst; ++l) capture_step<K>(st, c, ((l - m) & 1) != 0, A[l]);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const long q = (long)m * npad + p[k];
        prev[q] = st.h2[k];
        cur[q] = st.h1[k];
        kout[q] = st.sc[k];
    }
}

// k_adj_capture: the adjoint's start states of 64 ring pairs of degree m at the
// row starts l (even l - m) of a run of entries, by l: (mu_{l-2}, mu_{l-1}) and
// the scale count; (-mu_m, 0) at l = m, from which the first step gives mu_m.
// The recurrence runs once for the run (its entries are the segments of one
// group; once for each of them, from l = m, took up to eight times the steps).
__global__ __launch_bounds__(64) void k_adj_capture(const AdjCap* __restrict__ caps, const int* __restrict__ runs,
                                                    double2* __restrict__ st, int* __restrict__ sk,
                                                    const MapDesc* __restrict__ md_)
{
    const MapDesc& md = *md_;
    const int i0 = runs[blockIdx.x], i1 = runs[blockIdx.x + 1];
    const int L = md.L, m = caps[i0].m, p = caps[i0].p0 + threadIdx.x;
    const double* __restrict__ A = md.A + moff(L, m) - m;
    CaptureState<1> s;
    const double x[1] = {md.ring_x[p]};
    s.h1[0] = md.seed_v[(long)m * md.npair_pad + p];
    s.sc[0] = md.seed_k[(long)m * md.npair_pad + p];
    s.e1[0] = s.h2[0] = s.e2[0] = 0.0;
    int l = m + 1;
    for (int i = i0; i < i1; ++i) {
        const AdjCap c = caps[i];
        for (; l < c.l; ++l) capture_step<1>(s, x, ((l - m) & 1) != 0, A[l]);
        const long q = 64L * c.at + threadIdx.x;
        st[q] = c.l == m ? make_double2(-s.h1[0], 0.0) : make_double2(s.h2[0], s.h1[0]);
        sk[q] = s.sc[0];
    }
}

// ================================================================== ring stage
//
// One workgroup per ring pair.  The north and south rings of a pair share
// nph = n and phi0, so they travel as the real and imaginary parts of one
// complex sequence of length n held in LDS:
//   synthesis: Z_k = G_N,k + i G_S,k  ->  inverse DFT  ->  s_N + i s_S
//   adjoint:   f_N + i f_S  ->  forward DFT  ->  Y, split into H_N, H_S.
// Power-of-two n uses the FFT directly; other n (the polar rings, n = 4i)
// use Bluestein's chirp-z with a power-of-two length M >= 2n-1.  All
// transforms take and return natural order.  The phase of the first pixel,
// phi0 = pi/n, enters per Fourier bin: e^{i pi m/n} = e^{i pi k/n} (-1)^j for
// m = k + j n.
//
// LDS layout: element e of a sequence lives at zp(e) = e + e/16, one spare
// slot per 16 values, so the stride-16 accesses of the FFT passes fall on
// distinct banks.

__device__ __forceinline__ int zp(int e) { return e + (e >> 4); }

__device__ __forceinline__ double2 tw_get(const double2* __restrict__ tw, int t, int sign)
{
    double2 w = ld_at(tw, t);
    if (sign > 0) w.y = -w.y;
    return w;
}

// x e^{SIGN 2 pi i j / 16}, j = 0..7 (cos, sin of pi j / 8 as literals).
template <int SIGN>
__device__ __forceinline__ double2 tw16(double2 x, int j)
{
    constexpr double C1 = 0.9238795325112867, S1 = 0.3826834323650898, R2 = 0.7071067811865476;
    double c, sn;
    switch (j) {
    case 0: return x;
    case 4: return SIGN > 0 ? make_double2(-x.y, x.x) : make_double2(x.y, -x.x);
    case 1: c = C1; sn = S1; break;
    case 2: c = R2; sn = R2; break;
    case 3: c = S1; sn = C1; break;
    case 5: c = -S1; sn = C1; break;
    case 6: c = -R2; sn = R2; break;
    default: c = -C1; sn = S1; break;
    }
    sn *= SIGN;
    return make_double2(x.x * c - x.y * sn, x.x * sn + x.y * c);
}

// In-register R-point DFT (R <= 16), radix-2 decimation in frequency:
// natural order in, u[bitrev(q)] = sum_r u_r e^{SIGN 2 pi i r q / R} out.
// HALF: inputs r >= R / 2 are zero (and not read).
template <int R, int SIGN, bool HALF = false>
__device__ __forceinline__ void dft_reg(double2 (&u)[R])
{
    if (HALF) {
#pragma unroll
        for (int a = 0; a < R / 2; ++a) u[a + R / 2] = tw16<SIGN>(u[a], a * (16 / R));
    }
#pragma unroll
    for (int s = HALF ? R / 4 : R / 2; s >= 1; s /= 2) {
#pragma unroll
        for (int blk = 0; blk < R; blk += 2 * s) {
#pragma unroll
            for (int a = 0; a < s; ++a) {
                const double2 x0 = u[blk + a], x1 = u[blk + a + s];
                u[blk + a] = cadd(x0, x1);
                u[blk + a + s] = tw16<SIGN>(csub(x0, x1), a * (8 / s));
            }
        }
    }
}

template <int LR>
__device__ __forceinline__ constexpr int brev_c(int q)
{
    int r = 0;
    for (int b = 0; b < LR; ++b) r |= ((q >> b) & 1) << (LR - 1 - b);
    return r;
}

// One Stockham pass of radix R over M points with p = product of the radices
// already applied: butterfly i (k = i mod p) reads x[i + r M/R], twiddles by
// e^{SIGN 2 pi i r k/(p R)}, transforms, and writes y[(i - k) R + k + q p].
// Every thread loads all its butterflies before the first barrier and stores
// after it, so the pass works in place.  The twiddle loads (from the table in
// global memory, mostly L2 hits) are issued first, so their latency runs
// alongside the LDS loads and the barrier instead of after them.
constexpr int kLogMaxFFT = 13;
static_assert((1 << kLogMaxFFT) == kMaxFFT, "twiddle table length");

// Pointwise factors of a Bluestein transform fused into the first and last
// pass of its two FFTs: kFuseChirpIn multiplies each loaded input by the
// chirp (inputs at n and beyond are zero and not read), kFuseFilt each output
// by the chirp filter, kFuseChirpOut each output by 1/M and the chirp (outputs
// at n and beyond are not stored).  As M >= 2 n, the upper half of the first
// pass' inputs and of the last pass' outputs are such: their share of the
// butterflies is left out.  OS is the sign of the ring transform: for
// OS > 0 the chirps are conjugated and the filter is read reversed and
// conjugated.
enum { kFuseNone = 0, kFuseChirpIn = 1, kFuseFilt = 2, kFuseChirpOut = 3 };
struct BsFuse {
    const double2* chirp;
    const double2* filt;
    int n;
    double inv;  // 1 / M
};

// The tables hold half of each sequence: the chirp of even length n has
// c_{n-j} = c_j ((n - j)^2 = j^2 mod 2n), and the filter, the FFT of a
// sequence even in j (b_{M-j} = b_j), has F_{M-r} = F_r; entries 0..n/2 and
// 0..M/2 are stored.
template <int OS>
__device__ __forceinline__ double2 bs_chirp(BsFuse f, int j)
{
    double2 c = ld_at(f.chirp, min(j, f.n - j));
    if (OS > 0) c.y = -c.y;
    return c;
}

template <int OS>
__device__ __forceinline__ double2 bs_filt(BsFuse f, int r, int M)
{
    double2 g = ld_at(f.filt, min(r, M - r));
    if (OS > 0) g.y = -g.y;  // F_{M-r} conjugated, F_{M-r} = F_r
    return g;
}

template <int R, int LR, int SIGN, int MAXM, int PRE = kFuseNone, int POST = kFuseNone, int OS = -1>
__device__ __forceinline__ void stockham_pass(double2* Z, int M, int p, int lp, const double2* __restrict__ tw,
                                              BsFuse fz = BsFuse{})
{
    constexpr int NT = ring_threads(MAXM);
    constexpr int B = (MAXM / R + NT - 1) / NT;  // butterflies per thread, at most
    const int tid = threadIdx.x;
    const int nb = M / R;
    double2 u[B][R];
    double2 w1v[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int i = tid + b * NT;
        const int k = i & (p - 1);
        w1v[b] = make_double2(1.0, 0.0);
        if (i < nb && k) w1v[b] = tw_get(tw, k << (kLogMaxFFT - lp - LR), SIGN);  // k kMaxFFT / (p R)
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int i = tid + b * NT;
        if (i < nb) {
            if (PRE == kFuseChirpIn) {
                // chirps first (global loads in flight), then the LDS loads
#pragma unroll
                for (int r = 0; r < R / 2; ++r) {
                    const int e = i + r * nb;
                    u[b][r] = e < fz.n ? bs_chirp<OS>(fz, e) : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int r = 0; r < R / 2; ++r) {
                    const int e = i + r * nb;
                    if (e < fz.n) u[b][r] = cmul(Z[zp(e)], u[b][r]);
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) u[b][r] = Z[zp(i + r * nb)];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int i = tid + b * NT;
        if (i < nb) {
            const int k = i & (p - 1);
            if (k) {
                const double2 w1 = w1v[b];
                double2 w = w1;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    u[b][r] = cmul(u[b][r], w);
                    if (r + 1 < R) w = cmul(w, w1);
                }
            }
            dft_reg<R, SIGN, PRE == kFuseChirpIn>(u[b]);
            const int j = (i - k) * R + k;
#pragma unroll
            for (int q = 0; q < (POST == kFuseChirpOut ? R / 2 : R); ++q) {
                const int e = j + q * p;
                double2 v = u[b][brev_c<LR>(q)];
                if (POST == kFuseFilt) {
                    v = cmul(v, bs_filt<OS>(fz, e, M));
                } else if (POST == kFuseChirpOut) {
                    if (e >= fz.n) continue;
                    v = cmul(make_double2(v.x * fz.inv, v.y * fz.inv), bs_chirp<OS>(fz, e));
                }
                Z[zp(e)] = v;
            }
        }
    }
    __syncthreads();
}

// stockham_pass over two transforms of length M = 2^logM side by side in
// LDS (transform t at Z[t M ..)): butterfly g belongs to transform g / (M/R).
template <int R, int LR, int SIGN, int MAXM>
__device__ __forceinline__ void stockham_pass_two(double2* Z, int logM, int p, int lp, const double2* __restrict__ tw)
{
    constexpr int NT = ring_threads(MAXM);
    constexpr int B = (MAXM / R + NT - 1) / NT;  // butterflies per thread, at most (2 M <= MAXM)
    const int tid = threadIdx.x;
    const int lnb = logM - LR;  // log2 of the butterflies per transform
    const int nb = 1 << lnb;
    double2 u[B][R];
    double2 w1v[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * NT;
        const int i = g & (nb - 1);
        const int k = i & (p - 1);
        w1v[b] = make_double2(1.0, 0.0);
        if (g < 2 * nb && k) w1v[b] = tw_get(tw, k << (kLogMaxFFT - lp - LR), SIGN);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * NT;
        if (g < 2 * nb) {
            const int base = (g >> lnb) << logM;
            const int i = g & (nb - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) u[b][r] = Z[zp(base + i + r * nb)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * NT;
        if (g < 2 * nb) {
            const int base = (g >> lnb) << logM;
            const int i = g & (nb - 1);
            const int k = i & (p - 1);
            if (k) {
                const double2 w1 = w1v[b];
                double2 w = w1;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    u[b][r] = cmul(u[b][r], w);
                    if (r + 1 < R) w = cmul(w, w1);
                }
            }
            dft_reg<R, SIGN>(u[b]);
            const int j = (i - k) * R + k;
#pragma unroll
            for (int q = 0; q < R; ++q) Z[zp(base + j + q * p)] = u[b][brev_c<LR>(q)];
        }
    }
    __syncthreads();
}

// fft() of two transforms of length M = 2^logM side by side (2 M <= MAXM).
template <int SIGN, int MAXM>
__device__ void fft_two(double2* Z, int logM, const double2* __restrict__ tw)
{
    int p = 1, lp = 0, rem = logM;
    for (; rem >= 3; rem -= 3, p <<= 3, lp += 3) stockham_pass_two<8, 3, SIGN, MAXM>(Z, logM, p, lp, tw);
    if (rem == 2)
        stockham_pass_two<4, 2, SIGN, MAXM>(Z, logM, p, lp, tw);
    else if (rem == 1)
        stockham_pass_two<2, 1, SIGN, MAXM>(Z, logM, p, lp, tw);
}

// Unnormalised DFT of Z[0..M) in place, natural order in and out:
// Z_q <- sum_r Z_r e^{SIGN 2 pi i r q / M}, M = 2^logM <= MAXM <= kMaxFFT, M >= 2.
// Radix-8 passes, then one radix-4/2 pass for the remaining factor.  MAXM
// bounds the butterflies per thread and so the registers.
template <int SIGN, int MAXM>
__device__ void fft(double2* Z, int M, int logM, const double2* __restrict__ tw)
{
    // radix 8: one butterfly per thread at M = 8 x threads, within the 128
    // VGPRs that four waves per SIMD allow (radix 16 spills there)
    constexpr int LR = 3;
    int p = 1, lp = 0, rem = logM;
    for (; rem >= LR; rem -= LR, p <<= LR, lp += LR) stockham_pass<1 << LR, LR, SIGN, MAXM>(Z, M, p, lp, tw);
    if (rem == 2)
        stockham_pass<4, 2, SIGN, MAXM>(Z, M, p, lp, tw);
    else if (rem == 1)
        stockham_pass<2, 1, SIGN, MAXM>(Z, M, p, lp, tw);
}

// The FFT of fft() with pointwise factors fused into its first (PRE) and last
// (POST) pass; M >= 8.
template <int SIGN, int MAXM, int PRE, int POST, int OS>
__device__ void fft_fused(double2* Z, int M, int logM, const double2* __restrict__ tw, BsFuse fz)
{
    if (logM == 3) {
        stockham_pass<8, 3, SIGN, MAXM, PRE, POST, OS>(Z, M, 1, 0, tw, fz);
        return;
    }
    stockham_pass<8, 3, SIGN, MAXM, PRE, kFuseNone, OS>(Z, M, 1, 0, tw, fz);
    int p = 8, lp = 3, rem = logM - 3;
    for (; rem > 3; rem -= 3, p <<= 3, lp += 3) stockham_pass<8, 3, SIGN, MAXM>(Z, M, p, lp, tw);
    if (rem == 3)
        stockham_pass<8, 3, SIGN, MAXM, kFuseNone, POST, OS>(Z, M, p, lp, tw, fz);
    else if (rem == 2)
        stockham_pass<4, 2, SIGN, MAXM, kFuseNone, POST, OS>(Z, M, p, lp, tw, fz);
    else
        stockham_pass<2, 1, SIGN, MAXM, kFuseNone, POST, OS>(Z, M, p, lp, tw, fz);
}

// Bluestein DFT of z[0..n) (natural order; M >= 2n, so M >= 8): result in
// natural order in z[0..n).  chirp[j] = e^{-i pi j^2/n}, j <= n/2; filt =
// FFT_M of e^{+i pi j^2/n} (wrapped), entries 0..M/2.  For SIGN > 0 the chirps
// are conjugated and the filter is read reversed and conjugated.  The chirp
// products, the zero padding, the filter product and the final chirp and 1/M
// ride on the first and last passes of the two FFTs.
template <int SIGN, int MAXM>
__device__ void bluestein(double2* z, int n, int M, int logM, const double2* __restrict__ chirp,
                          const double2* __restrict__ filt, const double2* __restrict__ tw)
{
    const BsFuse fz{chirp, filt, n, ldexp(1.0, -logM)};  // 1 / M, M = 2^logM
    fft_fused<-1, MAXM, kFuseChirpIn, kFuseFilt, SIGN>(z, M, logM, tw, fz);
    fft_fused<+1, MAXM, kFuseNone, kFuseChirpOut, SIGN>(z, M, logM, tw, fz);
}

// Length-n DFT in LDS (natural order): the FFT for power-of-two n, Bluestein otherwise.
template <int SIGN, int MAXM>
__device__ __forceinline__ void ring_dft(double2* Z, int n, int M, int logM, bool pow2, const double2* chirp,
                                         const double2* filt, const double2* __restrict__ tw)
{
    if (pow2)
        fft<SIGN, MAXM>(Z, n, logM, tw);
    else
        bluestein<SIGN, MAXM>(Z, n, M, logM, chirp, filt, tw);
}

// Alias sums of Fourier bin k over the parity rows (E, O) of a ring pair:
// sum_j (-1)^{j shift} F_{k+jn} + sum_{j>=1} (-1)^{j shift} conj(F_{jn-k}),
// for j = r, r+R, r+2R, ... (one thread group of R).
__device__ __forceinline__ void fold_aliases(const double2* __restrict__ row, int L, int n, int k, int r, int R,
                                             bool shifted, double2& gN, double2& gS)
{
    gN = make_double2(0.0, 0.0);
    gS = make_double2(0.0, 0.0);
    for (int j = r; k + (long)j * n <= L; j += R) {
        const int mm = k + j * n;
        const double2 e = row[2 * mm], o = row[2 * mm + 1];
        const double sg = (shifted && (j & 1)) ? -1.0 : 1.0;
        gN.x += sg * (e.x + o.x);
        gN.y += sg * (e.y + o.y);
        gS.x += sg * (e.x - o.x);
        gS.y += sg * (e.y - o.y);
    }
    for (int j = 1 + r; (long)j * n - k <= L; j += R) {
        const int mm = j * n - k;
        const double2 e = row[2 * mm], o = row[2 * mm + 1];
        const double sg = (shifted && (j & 1)) ? -1.0 : 1.0;
        gN.x += sg * (e.x + o.x);
        gN.y -= sg * (e.y + o.y);
        gS.x += sg * (e.x - o.x);
        gS.y -= sg * (e.y - o.y);
    }
}

// e^{i pi (k0 + t D) / n} for t = 0, 1, 2, ...: the first two factors from
// sincospi, each later term by one complex multiply (a thread's bins and
// samples step by a fixed D; the rounding grows by about an ulp per step, over
// at most 16 steps).  A phase by sincospi costs a 64-bit remainder, an FP64
// division and the polynomial, about a hundred instructions.
struct PhaseSeq {
    double2 cur, step;
    __device__ __forceinline__ void init(long k0, long D, long n)
    {
        cur = cis_pi_frac(k0, n);
        step = cis_pi_frac(D, n);
    }
    __device__ __forceinline__ double2 next()
    {
        const double2 c = cur;
        cur = cmul(cur, step);
        return c;
    }
};

// Bin of the packed pair spectrum (natural order): phase ph = e^{i pi k/n}
// (bin k) for shifted rings, no south ring at the equator.
__device__ __forceinline__ void fold_store(double2* Z, int slot, double2 ph, bool shifted, bool no_south,
                                           double2 gN, double2 gS)
{
    if (no_south) gS = make_double2(0.0, 0.0);
    if (shifted) {
        gN = cmul(gN, ph);
        gS = cmul(gS, ph);
    }
    Z[zp(slot)] = make_double2(gN.x - gS.y, gN.y + gS.x);
}

// Unfold bin k and its mirror n - k of Y into Q (the aliases m = k + j n,
// j = r, r + R, ...): Psi_X,m = e^{-i pi k/n} (-1)^j H_X,k; ph = e^{i pi k/n}
// (used for shifted rings).
__device__ __forceinline__ void unfold_bin(double2* qrow, int L, int n, int k, int r, int R, bool shifted,
                                           double2 ph, double2 y, double2 z2)
{
    const double2 yc = make_double2(z2.x, -z2.y);
    double2 hN = make_double2(0.5 * (y.x + yc.x), 0.5 * (y.y + yc.y));
    double2 hS = make_double2(0.5 * (y.y - yc.y), -0.5 * (y.x - yc.x));
    if (shifted) {
        ph.y = -ph.y;
        hN = cmul(hN, ph);
        hS = cmul(hS, ph);
    }
    const double2 pe = cadd(hN, hS), po = csub(hN, hS);
    auto q = gview(qrow);
    for (int j = r; k + (long)j * n <= L; j += R) {
        const int mm = k + j * n;
        const double sg = (shifted && (j & 1)) ? -1.0 : 1.0;
        q[2 * mm] = make_double2(sg * pe.x, sg * pe.y);
        q[2 * mm + 1] = make_double2(sg * po.x, sg * po.y);
    }
}

// Y_k of a split ring from its two half transforms: SE (global scratch) and
// Z (LDS), Y_k = E_{k mod h} + w O_{k mod h}, w = e^{-2 pi i k/n}.
__device__ __forceinline__ double2 split_bin(const double2* SE, const double2* Z, int k, int h, double2 w)
{
    const int kk = k % h;
    return cadd(gview(SE)[kk], cmul(Z[zp(kk)], w));
}

// A ring pair whose length-n Bluestein transform would not fit in LDS (n = 4i
// with 2n - 1 > kMaxFFT): each direction splits into two length-h = n/2 DFTs
// over the even and odd samples, each done by Bluestein in LDS, the first kept
// in global scratch while the second runs (decimation in time):
//   synthesis  s_j = E_j + w^j O_j,  s_{j+h} = E_j - w^j O_j,  w = e^{2 pi i/n},
//              E, O = inverse DFT_h of the even / odd bins;
//   analysis   Y_k = FE_{k mod h} + w^{-k} FO_{k mod h},
//              FE, FO = DFT_h of the even / odd samples.
// Scratch per ring: SE[h] (a half transform) and SF[n] (weighted residual).
template <int MODE, int MAXM>
__device__ void ring_split(const MapDesc& md, int p, int n, int M, int logM, bool shifted, long oN, long oS,
                           double* __restrict__ map_out, const double* __restrict__ map_in,
                           const double2* __restrict__ tw, double2* Z, double* sh)
{
    const int L = md.L;
    constexpr int NT = ring_threads(MAXM);
    const int tid = threadIdx.x;
    const int h = n >> 1;
    const double2* filt = md.bs_filt + md.ring_bsofs[p];
    const double2* chirp = md.bs_chirp + md.ring_chofs[p];
    double2* SE = md.ring_scr + md.ring_scrofs[p];
    double2* SF = SE + h;

    if (MODE != kRingAna) {
        const double2* row = reinterpret_cast<const double2*>(md.P + (long)p * (L + 1) * 4);
        for (int r = 0; r < 2; ++r) {
            PhaseSeq ps;
            if (shifted) ps.init(2 * tid + r, 2 * NT, n);
            for (int kk = tid; kk < h; kk += NT) {
                const int k = 2 * kk + r;
                double2 gN, gS;
                fold_aliases(row, L, n, k, 0, 1, shifted, gN, gS);
                fold_store(Z, kk, shifted ? ps.next() : make_double2(1.0, 0.0), shifted, oS < 0, gN, gS);
            }
            __syncthreads();
            bluestein<+1, MAXM>(Z, h, M, logM, chirp, filt, tw);
            if (r == 0) {
                for (int j = tid; j < h; j += NT) SE[j] = Z[zp(j)];
                __syncthreads();
            }
        }
        double chi = 0.0;
        PhaseSeq tw2;  // e^{2 pi i j / n}
        tw2.init(2 * tid, 2 * NT, n);
        for (int j = tid; j < h; j += NT) {
            const double2 e = SE[j];
            const double2 o = cmul(Z[zp(j)], tw2.next());
            const double2 sv[2] = {cadd(e, o), csub(e, o)};
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const long t = j + half * h;
                const double2 v = sv[half];
                if (MODE == kRingSyn) {
                    map_out[oN + t] = v.x;
                    if (oS >= 0) map_out[oS + t] = v.y;
                } else if (MODE == kRingWeight) {
                    SF[t] = make_double2(md.w[oN + t] * v.x, oS >= 0 ? md.w[oS + t] * v.y : 0.0);
                } else {
                    const double rN = md.d[oN + t] - v.x;
                    const double fN = md.w[oN + t] * rN;
                    chi = fma(fN, rN, chi);
                    double fS = 0.0;
                    if (oS >= 0) {
                        const double rS = md.d[oS + t] - v.y;
                        fS = md.w[oS + t] * rS;
                        chi = fma(fS, rS, chi);
                    }
                    SF[t] = make_double2(fN, fS);
                }
            }
        }
        if (MODE == kRingSyn) return;
        if (MODE == kRingLike) {
            const double t = block_sum<NT>(chi, sh);
            if (tid == 0) md.chi[p] = t;
        } else {
            __syncthreads();
        }
    }

    for (int r = 0; r < 2; ++r) {
        for (int j = tid; j < h; j += NT) {
            const long t = 2 * j + r;
            Z[zp(j)] = (MODE == kRingAna) ? make_double2(map_in[oN + t], oS >= 0 ? map_in[oS + t] : 0.0) : SF[t];
        }
        __syncthreads();
        bluestein<-1, MAXM>(Z, h, M, logM, chirp, filt, tw);
        if (r == 0) {
            for (int j = tid; j < h; j += NT) SE[j] = Z[zp(j)];
            __syncthreads();
        }
    }

    double2* qrow = reinterpret_cast<double2*>(md.Q + (long)p * (L + 1) * 4);
    PhaseSeq wk, pk;  // e^{2 pi i k/n} and e^{i pi k/n}
    wk.init(2 * tid, 2 * NT, n);
    if (shifted) pk.init(tid, NT, n);
    for (int k = tid; k < n && k <= L; k += NT) {
        const int nk = (k == 0) ? 0 : n - k;
        const double2 a = wk.next();  // e^{-2 pi i (n-k)/n} = a, e^{-2 pi i k/n} = conj(a)
        const double2 ph = shifted ? pk.next() : make_double2(1.0, 0.0);
        unfold_bin(qrow, L, n, k, 0, 1, shifted, ph, split_bin(md.ring_scr + md.ring_scrofs[p], Z, k, h,
                                                                 make_double2(a.x, -a.y)),
                   split_bin(md.ring_scr + md.ring_scrofs[p], Z, nk, h, a));
    }
}

// Two power-of-two rings of length n = MAXM / 2 in one workgroup (each longer
// than its map's lmax and unsplit; the pair of a RingItem with pair2 >= 0):
// ring r's spectrum and samples live at Z[r n ..), a thread holds CNT / 2
// samples of each, and every step is the single ring's (one-alias fold,
// transform, residual or weights, transform, unfold) with the two transforms
// side by side.  Rings of half the launch's length would otherwise leave half
// of their workgroup's threads idle in every FFT pass.
constexpr int clog2(int v) { return v <= 1 ? 0 : 1 + clog2(v / 2); }

template <int MODE, int MAXM>
__device__ void ring_two(const RingItem& it, const MapDesc* __restrict__ maps, double* __restrict__ map_out,
                         const double* __restrict__ map_in, const double2* __restrict__ tw, double2* Z, double* sh)
{
    constexpr int NT = ring_threads(MAXM);
    constexpr int n = MAXM / 2;
    constexpr int logn = clog2(n);
    constexpr int CNT = MAXM / NT;  // samples per thread, both rings
    constexpr int CH = CNT / 2;     // per ring
    static_assert(CNT % 2 == 0 && (1 << logn) == n, "two rings per workgroup");
    const int tid = threadIdx.x;
    const MapDesc* mdr[2] = {&maps[it.map], &maps[it.map2]};
    const int pr[2] = {it.pair, it.pair2};
    bool shf[2];
    long oN[2], oS[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        shf[r] = mdr[r]->ring_shift[pr[r]] != 0;
        oN[r] = mdr[r]->ring_ofsN[pr[r]];
        oS[r] = mdr[r]->ring_ofsS[pr[r]];
    }

    if (MODE != kRingAna) {
        // fold, n > L: at most the alias k and the mirror n - k per bin
        double2 e[CNT], o[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int L = mdr[r]->L;
            auto rw = gview(reinterpret_cast<const double2*>(mdr[r]->P + (long)pr[r] * (L + 1) * 4));
            const int k = tid + (t - r * CH) * NT;
            const int m = k <= L ? k : n - k;
            if (k <= L || (k >= 1 && n - k <= L)) {
                e[t] = rw[2 * m];
                o[t] = rw[2 * m + 1];
            }
        }
        PhaseSeq ps;
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int L = mdr[r]->L;
            auto rw = gview(reinterpret_cast<const double2*>(mdr[r]->P + (long)pr[r] * (L + 1) * 4));
            const int k = tid + (t - r * CH) * NT;
            if (t % CH == 0 && shf[r]) ps.init(tid, NT, n);
            const double sg = shf[r] ? -1.0 : 1.0;  // (-1)^{j shift} at j = 1
            const double2 ph = shf[r] ? ps.next() : make_double2(1.0, 0.0);
            double2 gN = make_double2(0.0, 0.0), gS = make_double2(0.0, 0.0);
            const bool mirror = k >= 1 && n - k <= L;
            if (k <= L) {
                gN.x += 1.0 * (e[t].x + o[t].x);
                gN.y += 1.0 * (e[t].y + o[t].y);
                gS.x += 1.0 * (e[t].x - o[t].x);
                gS.y += 1.0 * (e[t].y - o[t].y);
                if (mirror) {
                    e[t] = rw[2 * (n - k)];
                    o[t] = rw[2 * (n - k) + 1];
                }
            }
            if (mirror) {
                gN.x += sg * (e[t].x + o[t].x);
                gN.y -= sg * (e[t].y + o[t].y);
                gS.x += sg * (e[t].x - o[t].x);
                gS.y -= sg * (e[t].y - o[t].y);
            }
            fold_store(Z, r * n + k, ph, shf[r], oS[r] < 0, gN, gS);
        }
        __syncthreads();
        fft_two<+1, MAXM>(Z, logn, tw);
    }

    if (MODE == kRingSyn) {
        gdouble* out = gview(map_out);
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int j = tid + (t - r * CH) * NT;
            const double2 v = Z[zp(r * n + j)];
            out[oN[r] + j] = v.x;
            if (oS[r] >= 0) out[oS[r] + j] = v.y;
        }
        return;
    }

    if (MODE == kRingLike) {
        double dN[CNT], wN[CNT], dS[CNT], wS[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            gcdouble* dd = gview(mdr[r]->d);
            gcdouble* ww = gview(mdr[r]->w);
            const int j = tid + (t - r * CH) * NT;
            dN[t] = dd[oN[r] + j];
            wN[t] = ww[oN[r] + j];
            if (oS[r] >= 0) {
                dS[t] = dd[oS[r] + j];
                wS[t] = ww[oS[r] + j];
            }
        }
        double chi[2] = {0.0, 0.0};
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int j = tid + (t - r * CH) * NT;
            const double2 v = Z[zp(r * n + j)];
            const double rN = dN[t] - v.x;
            const double fN = wN[t] * rN;
            chi[r] = fma(fN, rN, chi[r]);
            double fS = 0.0;
            if (oS[r] >= 0) {
                const double rS = dS[t] - v.y;
                fS = wS[t] * rS;
                chi[r] = fma(fS, rS, chi[r]);
            }
            Z[zp(r * n + j)] = make_double2(fN, fS);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const double c = block_sum<NT>(chi[r], sh);
            if (tid == 0) mdr[r]->chi[pr[r]] = c;
        }
    } else if (MODE == kRingWeight) {
        double wN[CNT], wS[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            gcdouble* ww = gview(mdr[r]->w);
            const int j = tid + (t - r * CH) * NT;
            wN[t] = ww[oN[r] + j];
            wS[t] = oS[r] >= 0 ? ww[oS[r] + j] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int j = tid + (t - r * CH) * NT;
            const double2 v = Z[zp(r * n + j)];
            Z[zp(r * n + j)] = make_double2(wN[t] * v.x, oS[r] >= 0 ? wS[t] * v.y : 0.0);
        }
        __syncthreads();
    } else {  // kRingAna
        gcdouble* in = gview(map_in);
        double2 mv[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int j = tid + (t - r * CH) * NT;
            mv[t] = make_double2(in[oN[r] + j], oS[r] >= 0 ? in[oS[r] + j] : 0.0);
        }
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int r = t / CH;
            const int j = tid + (t - r * CH) * NT;
            Z[zp(r * n + j)] = mv[t];
        }
        __syncthreads();
    }
    fft_two<-1, MAXM>(Z, logn, tw);

    // unfold, one alias per bin (n > L)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int L = mdr[r]->L;
        double2* qrow = reinterpret_cast<double2*>(mdr[r]->Q + (long)pr[r] * (L + 1) * 4);
        PhaseSeq ps;
        if (shf[r]) ps.init(tid, NT, n);
        for (int k = tid; k < n; k += NT) {
            const double2 ph = shf[r] ? ps.next() : make_double2(1.0, 0.0);
            if (k > L) continue;
            const int nk = (k == 0) ? 0 : n - k;
            unfold_bin(qrow, L, n, k, 0, 1, shf[r], ph, Z[zp(r * n + k)], Z[zp(r * n + nk)]);
        }
    }
}

// Ring kernels up to M = 4096 are held to four waves per SIMD (128 VGPRs):
// two workgroups of 512 threads, or four of 256 up to M = 2048, per CU.
template <int MODE, int MAXM>
__global__ __launch_bounds__(ring_threads(MAXM), MAXM > 4096 ? 1 : 4) void k_ring(const RingItem* __restrict__ items,
                                                       const MapDesc* __restrict__ maps,
                                                       double* __restrict__ map_out,
                                                       const double* __restrict__ map_in,
                                                       const double2* __restrict__ tw)
{
    constexpr int NT = ring_threads(MAXM);
    extern __shared__ double2 Z[];
    __shared__ double sh[NT / 64];
    const RingItem it = items[blockIdx.x];
    if constexpr (MAXM <= 4096) {
        if (it.pair2 >= 0) {
            ring_two<MODE, MAXM>(it, maps, map_out, map_in, tw, Z, sh);
            return;
        }
    }
    const MapDesc& md = maps[it.map];
    const int L = md.L;
    const int p = it.pair;
    const int n = md.ring_nph[p];
    const int M = md.ring_M[p];
    int logM = 0;
    while ((1 << logM) < M) ++logM;
    const bool pow2 = (M == n);
    const bool shifted = md.ring_shift[p] != 0;
    const long oN = md.ring_ofsN[p];
    const long oS = md.ring_ofsS[p];
    if (md.ring_scrofs[p] >= 0) {
        ring_split<MODE, MAXM>(md, p, n, M, logM, shifted, oN, oS, map_out, map_in, tw, Z, sh);
        return;
    }
    const double2* filt = pow2 ? nullptr : md.bs_filt + md.ring_bsofs[p];
    const double2* chirp = pow2 ? nullptr : md.bs_chirp + md.ring_chofs[p];
    const int tid = threadIdx.x;
    constexpr int CNT = (MAXM + NT - 1) / NT;  // ring samples per thread, at most
    gdouble* out = gview(map_out);
    gcdouble* in = gview(map_in);
    gcdouble* dd = gview(md.d);
    gcdouble* ww = gview(md.w);
    // for n < NT the aliases of each bin are split over R thread
    // groups (reads stay coalesced over k), partial sums added in fixed order
    const int R = n < NT ? NT / n : 1;

    if (MODE != kRingAna) {
        const double2* row = reinterpret_cast<const double2*>(md.P + (long)p * (L + 1) * 4);
        // fold: Z_k = G_N,k + i G_S,k
        if (R == 1 && n > L) {
            // at most the alias k (k <= L) and the mirror n - k (n - k <= L)
            // per bin, and both only where n - L <= k <= L: one load per bin
            // issued for every bin of the thread before the sums, the rare
            // second one where the sums need it
            auto rw = gview(row);
            double2 e[CNT], o[CNT];
#pragma unroll
            for (int t = 0; t < CNT; ++t) {
                const int k = tid + t * NT;
                const int m = k <= L ? k : n - k;
                if (k < n && (k <= L || (k >= 1 && n - k <= L))) {
                    e[t] = rw[2 * m];
                    o[t] = rw[2 * m + 1];
                }
            }
            const double sg = shifted ? -1.0 : 1.0;  // (-1)^{j shift} at j = 1
            PhaseSeq ps;
            if (shifted) ps.init(tid, NT, n);
#pragma unroll
            for (int t = 0; t < CNT; ++t) {
                const int k = tid + t * NT;
                if (k >= n) continue;
                const double2 ph = shifted ? ps.next() : make_double2(1.0, 0.0);
                double2 gN = make_double2(0.0, 0.0), gS = make_double2(0.0, 0.0);
                const bool mirror = k >= 1 && n - k <= L;
                if (k <= L) {
                    gN.x += 1.0 * (e[t].x + o[t].x);
                    gN.y += 1.0 * (e[t].y + o[t].y);
                    gS.x += 1.0 * (e[t].x - o[t].x);
                    gS.y += 1.0 * (e[t].y - o[t].y);
                    if (mirror) {
                        e[t] = rw[2 * (n - k)];
                        o[t] = rw[2 * (n - k) + 1];
                    }
                }
                if (mirror) {
                    gN.x += sg * (e[t].x + o[t].x);
                    gN.y -= sg * (e[t].y + o[t].y);
                    gS.x += sg * (e[t].x - o[t].x);
                    gS.y -= sg * (e[t].y - o[t].y);
                }
                fold_store(Z, k, ph, shifted, oS < 0, gN, gS);
            }
        } else if (R == 1) {
            PhaseSeq ps;
            if (shifted) ps.init(tid, NT, n);
            for (int k = tid; k < n; k += NT) {
                double2 gN, gS;
                fold_aliases(row, L, n, k, 0, 1, shifted, gN, gS);
                fold_store(Z, k, shifted ? ps.next() : make_double2(1.0, 0.0), shifted, oS < 0, gN, gS);
            }
        } else {
            double2 gN = make_double2(0.0, 0.0), gS = make_double2(0.0, 0.0);
            if (tid < R * n) {
                fold_aliases(row, L, n, tid % n, tid / n, R, shifted, gN, gS);
                Z[zp(2 * tid)] = gN;
                Z[zp(2 * tid + 1)] = gS;
            }
            __syncthreads();
            if (tid < n) {
                gN = make_double2(0.0, 0.0);
                gS = make_double2(0.0, 0.0);
                for (int r = 0; r < R; ++r) {
                    gN = cadd(gN, Z[zp(2 * (r * n + tid))]);
                    gS = cadd(gS, Z[zp(2 * (r * n + tid) + 1)]);
                }
            }
            __syncthreads();
            if (tid < n)
                fold_store(Z, tid, shifted ? cis_pi_frac(tid, n) : make_double2(1.0, 0.0), shifted, oS < 0, gN, gS);
        }
        __syncthreads();
        ring_dft<+1, MAXM>(Z, n, M, logM, pow2, chirp, filt, tw);
    }

    if (MODE == kRingSyn) {
        for (int j = tid; j < n; j += NT) {
            const double2 v = Z[zp(j)];
            out[oN + j] = v.x;
            if (oS >= 0) out[oS + j] = v.y;
        }
        return;
    }

    // per-pixel inputs of the thread's samples, all loaded before use
    if (MODE == kRingLike) {
        double dN[CNT], wN[CNT], dS[CNT], wS[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j < n) {
                dN[t] = dd[oN + j];
                wN[t] = ww[oN + j];
                if (oS >= 0) {
                    dS[t] = dd[oS + j];
                    wS[t] = ww[oS + j];
                }
            }
        }
        double chi = 0.0;
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j >= n) continue;
            const double2 v = Z[zp(j)];
            const double rN = dN[t] - v.x;
            const double fN = wN[t] * rN;
            chi = fma(fN, rN, chi);
            double fS = 0.0;
            if (oS >= 0) {
                const double rS = dS[t] - v.y;
                fS = wS[t] * rS;
                chi = fma(fS, rS, chi);
            }
            Z[zp(j)] = make_double2(fN, fS);
        }
        const double t = block_sum<NT>(chi, sh);
        if (tid == 0) md.chi[p] = t;
    } else if (MODE == kRingWeight) {
        double wN[CNT], wS[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j < n) {
                wN[t] = ww[oN + j];
                wS[t] = oS >= 0 ? ww[oS + j] : 0.0;
            }
        }
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j >= n) continue;
            const double2 v = Z[zp(j)];
            Z[zp(j)] = make_double2(wN[t] * v.x, oS >= 0 ? wS[t] * v.y : 0.0);
        }
        __syncthreads();
    } else {  // kRingAna: load the map to analyse
        double2 mv[CNT];
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j < n) mv[t] = make_double2(in[oN + j], oS >= 0 ? in[oS + j] : 0.0);
        }
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int j = tid + t * NT;
            if (j < n) Z[zp(j)] = mv[t];
        }
        __syncthreads();
    }
    ring_dft<-1, MAXM>(Z, n, M, logM, pow2, chirp, filt, tw);

    // unfold, with the aliases of bin k split over R thread groups as in the fold
    double2* qrow = reinterpret_cast<double2*>(md.Q + (long)p * (L + 1) * 4);
    if (R == 1) {
        PhaseSeq ps;
        if (shifted) ps.init(tid, NT, n);
        for (int k = tid; k < n; k += NT) {
            const double2 ph = shifted ? ps.next() : make_double2(1.0, 0.0);
            if (k > L) continue;
            const int nk = (k == 0) ? 0 : n - k;
            unfold_bin(qrow, L, n, k, 0, 1, shifted, ph, Z[zp(k)], Z[zp(nk)]);
        }
    } else if (tid < R * n) {  // R n <= NT: one (bin, group) per thread
        const int k = tid % n, r = tid / n;
        if (k <= L) {
            const int nk = (k == 0) ? 0 : n - k;
            unfold_bin(qrow, L, n, k, r, R, shifted, shifted ? cis_pi_frac(k, n) : make_double2(1.0, 0.0), Z[zp(k)],
                       Z[zp(nk)]);
        }
    }
}

// The ring stage of maps whose transforms all have at most kSmallFFT points
// (nside <= 128): a launch of some hundred workgroups, bound by the latency of
// one.  So, against k_ring: radix-4 passes, which keep four times as many
// threads busy as radix 8 on a chain half as long, between two LDS buffers, one
// barrier each; twiddles, chirps, filters and pixels loaded at the start, at
// once with the parity sums, into LDS or the registers of the thread that uses
// them in both directions (Bluestein's chirp products move to the steps that
// write and read the samples, where thread k holds c_k = c_{n-k}).
// us per call by events, before and after: nside 8 17.1 / 12.9, 32 19.1 / 14.2, 64
// 20.3 / 15.5, 128 24.4 / 18.5 (an empty kernel: 5).
constexpr int kSmallFFT = 1024;
constexpr int kSmallT = 256;

// DFT of the M = 2^logM points of a (those from nin on are zero), natural order
// in and out, by way of b; returns the buffer that holds it.  sign: +-1; filt:
// times f[q], its imaginary part times conj, at point tid + q M / 4.  (Signs by
// value: each copy of the code is fetched once and run once.)
__device__ __forceinline__ double2* small_fft(double2* a, double2* b, int M, int logM, int nin, const double2* tw,
                                              double sign, bool filt, const double2 (&f)[4], double conj)
{
    const int i = threadIdx.x;
    const double2 zero = make_double2(0.0, 0.0);
    int p = 1, lp = 0;
    if (logM & 1) {
        const int nb = M / 2;  // at most kSmallT: logM <= 9
        if (i < nb) {
            const double2 x0 = i < nin ? a[zp(i)] : zero, x1 = i + nb < nin ? a[zp(i + nb)] : zero;
            b[zp(2 * i)] = cadd(x0, x1);
            b[zp(2 * i + 1)] = csub(x0, x1);
        }
        __syncthreads();
        double2* t = a;
        a = b;
        b = t;
        nin = M;
        p = 2;
        lp = 1;
    }
    const int nb = M / 4;
    for (; p < M; p <<= 2, lp += 2) {
        if (i < nb) {
            double2 u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) u[r] = i + r * nb < nin ? a[zp(i + r * nb)] : zero;
            const int k = i & (p - 1);
            if (p > 1) {
                double2 w1 = tw[k << (logM - 2 - lp)];  // e^{-2 pi i k / (4 p)}
                w1.y *= -sign;
                const double2 w2 = cmul(w1, w1);
                u[1] = cmul(u[1], w1);
                u[2] = cmul(u[2], w2);
                u[3] = cmul(u[3], cmul(w2, w1));
            }
            const double2 s0 = cadd(u[0], u[2]), d0 = csub(u[0], u[2]), s1 = cadd(u[1], u[3]), d1 = csub(u[1], u[3]);
            const double2 e1 = make_double2(-sign * d1.y, sign * d1.x);
            double2 y[4] = {cadd(s0, s1), cadd(d0, e1), csub(s0, s1), csub(d0, e1)};
            const int j = (i - k) * 4 + k;
            const bool last = filt && 4 * p == M;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (last) y[q] = cmul(y[q], make_double2(f[q].x, conj * f[q].y));
                b[zp(j + q * p)] = y[q];
            }
        }
        __syncthreads();
        double2* t = a;
        a = b;
        b = t;
        nin = M;
    }
    return a;
}

// The ring's DFT of that sign: the FFT for power-of-two n, else Bluestein's two,
// whose filter is conjugated for the + sign.  Z: data and result, Y: the other
// buffer.
__device__ __forceinline__ void small_dft(double2*& Z, double2*& Y, int n, int M, int logM, const double2* tw,
                                          double sign, const double2 (&f)[4])
{
    const bool pow2 = M == n;
    for (int h = pow2 ? 1 : 0; h < 2; ++h) {
        double2* r = small_fft(Z, Y, M, logM, h == 0 ? n : M, tw, pow2 ? sign : h == 0 ? -1.0 : 1.0, h == 0, f, -sign);
        if (r != Z) {
            Y = Z;
            Z = r;
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(kSmallT) void k_ring_small(const RingItem* __restrict__ items,
                                                        const MapDesc* __restrict__ maps,
                                                        double* __restrict__ map_out,
                                                        const double* __restrict__ map_in,
                                                        const double2* __restrict__ tw)
{
    // rings of up to 2 NT samples: 4 nside, and below 512 where the transform is longer
    constexpr int NT = kSmallT, CNT = 2, kZ = kSmallFFT + kSmallFFT / 16;
    __shared__ double2 Zs[2 * kZ];
    __shared__ double2 tws[kSmallFFT / 4];
    __shared__ double sh[NT / 64];
    const RingItem it = items[blockIdx.x];
    const MapDesc& md = maps[it.map];
    const int tid = threadIdx.x;
    const int L = md.L;
    const int p = it.pair;
    const int n = md.ring_nph[p];
    const int M = md.ring_M[p];
    const int logM = 31 - __builtin_clz(M);
    const bool pow2 = (M == n);
    const bool shifted = md.ring_shift[p] != 0;
    const long oN = md.ring_ofsN[p];
    const long oS = md.ring_ofsS[p];
    // aliases of a bin over R groups of threads as in k_ring; k1: the thread's
    // first bin and (where it is below n) sample
    const int R = n < NT ? NT / n : 1;
    const int k1 = R > 1 ? tid % n : tid;

    const double2 one = make_double2(1.0, 0.0);
    double2 f[4] = {one, one, one, one}, c[CNT];
    double dN[CNT], wN[CNT], dS[CNT], wS[CNT];
    double2 twv = one;
    if (tid < M / 4) twv = ld_at(tw, tid << (kLogMaxFFT - logM));
    if (!pow2) {
        const BsFuse fz{md.bs_chirp + md.ring_chofs[p], md.bs_filt + md.ring_bsofs[p], n, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (tid < M / 4) f[q] = bs_filt<-1>(fz, tid + q * (M / 4), M);
#pragma unroll
        for (int t = 0; t < CNT; ++t)
            if (k1 + t * NT < n) c[t] = bs_chirp<-1>(fz, k1 + t * NT);
    }
#pragma unroll
    for (int t = 0; t < CNT; ++t) {
        const int j = tid + t * NT;
        dN[t] = wN[t] = dS[t] = wS[t] = 0.0;
        if (t * NT < n && j < n && MODE != kRingSyn) {
            if (MODE == kRingLike) dN[t] = ld_at(md.d + oN, j);
            if (MODE == kRingAna)
                dN[t] = ld_at(map_in + oN, j);
            else
                wN[t] = ld_at(md.w + oN, j);
            if (oS >= 0) {
                if (MODE == kRingLike) dS[t] = ld_at(md.d + oS, j);
                if (MODE == kRingAna)
                    dS[t] = ld_at(map_in + oS, j);
                else
                    wS[t] = ld_at(md.w + oS, j);
            }
        }
    }
    PhaseSeq phase;
    if (shifted) phase.init(k1, NT, n);
    if (tid < M / 4) tws[tid] = twv;
    double2 *Z = Zs, *Y = Zs + kZ;

    if (MODE != kRingAna) {
        const double2* row = reinterpret_cast<const double2*>(md.P + (long)p * (L + 1) * 4);
        if (R == 1) {
            PhaseSeq ps = phase;
#pragma unroll
            for (int t = 0; t < CNT; ++t) {
                const int k = tid + t * NT;
                if (k >= n) continue;
                double2 gN, gS;
                fold_aliases(row, L, n, k, 0, 1, shifted, gN, gS);
                fold_store(Z, k, shifted ? ps.next() : one, shifted, oS < 0, gN, gS);
                if (!pow2) Z[zp(k)] = cmulc(Z[zp(k)], c[t]);
            }
        } else {
            double2 gN, gS;
            if (tid < R * n) {
                fold_aliases(row, L, n, k1, tid / n, R, shifted, gN, gS);
                Y[zp(2 * tid)] = gN;
                Y[zp(2 * tid + 1)] = gS;
            }
            __syncthreads();
            if (tid < n) {
                gN = gS = make_double2(0.0, 0.0);
                for (int r = 0; r < R; ++r) {
                    gN = cadd(gN, Y[zp(2 * (r * n + tid))]);
                    gS = cadd(gS, Y[zp(2 * (r * n + tid) + 1)]);
                }
                fold_store(Z, tid, phase.cur, shifted, oS < 0, gN, gS);
                if (!pow2) Z[zp(tid)] = cmulc(Z[zp(tid)], c[0]);
            }
        }
        __syncthreads();
        small_dft(Z, Y, n, M, logM, tws, 1.0, f);
    }

    const double inv = ldexp(1.0, -logM);
    double chi = 0.0;
#pragma unroll
    for (int t = 0; t < CNT; ++t) {
        const int j = tid + t * NT;
        if (j >= n) continue;
        double2 v = make_double2(dN[t], dS[t]);  // kRingAna
        if (MODE != kRingAna) {
            v = Z[zp(j)];
            if (!pow2) v = cmulc(make_double2(v.x * inv, v.y * inv), c[t]);
        }
        if (MODE == kRingSyn) {
            map_out[oN + j] = v.x;
            if (oS >= 0) map_out[oS + j] = v.y;
            continue;
        }
        if (MODE == kRingLike) {
            const double rN = dN[t] - v.x, fN = wN[t] * rN;
            chi = fma(fN, rN, chi);
            double fS = 0.0;
            if (oS >= 0) {
                const double rS = dS[t] - v.y;
                fS = wS[t] * rS;
                chi = fma(fS, rS, chi);
            }
            v = make_double2(fN, fS);
        } else if (MODE == kRingWeight) {
            v = make_double2(wN[t] * v.x, oS >= 0 ? wS[t] * v.y : 0.0);
        }
        Z[zp(j)] = pow2 ? v : cmul(v, c[t]);
    }
    if (MODE == kRingSyn) return;
    if (MODE == kRingLike) {
        const double t = block_sum<NT>(chi, sh);
        if (tid == 0) md.chi[p] = t;
    } else {
        __syncthreads();
    }
    small_dft(Z, Y, n, M, logM, tws, -1.0, f);

    // unfold
    double2* qrow = reinterpret_cast<double2*>(md.Q + (long)p * (L + 1) * 4);
    auto bin = [&](int k, int t, int r, double2 ph) {
        if (k > L) return;
        double2 y = Z[zp(k)], z2 = Z[zp(k == 0 ? 0 : n - k)];
        if (!pow2) {
            y = cmul(make_double2(y.x * inv, y.y * inv), c[t]);
            z2 = cmul(make_double2(z2.x * inv, z2.y * inv), c[t]);
        }
        unfold_bin(qrow, L, n, k, r, R, shifted, ph, y, z2);
    };
    if (R == 1) {
#pragma unroll
        for (int t = 0; t < CNT; ++t) {
            const int k = tid + t * NT;
            if (k < n) bin(k, t, 0, shifted ? phase.next() : one);
        }
    } else if (tid < R * n) {
        bin(k1, 0, tid / n, phase.cur);
    }
}

// Bluestein set-up for one ring pair of Bluestein length n (nph, or nph/2 for
// a split ring; even): chirp[j] = e^{-i pi j^2/n} for j <= n/2 and filt =
// FFT_M of b_j = e^{+i pi j^2/n} for |j| < n wrapped mod M, entries 0..M/2 (the
// rest follow by symmetry).
__global__ __launch_bounds__(ring_threads(kMaxFFT)) void k_bluestein_setup(const int* __restrict__ pairs,
                                                                  const MapDesc* __restrict__ md_,
                                                                  double2* __restrict__ filt_out,
                                                                  double2* __restrict__ chirp_out,
                                                                  const double2* __restrict__ tw)
{
    extern __shared__ double2 Z[];
    const MapDesc& md = *md_;
    const int p = pairs[blockIdx.x];
    const int n = md.ring_scrofs[p] >= 0 ? md.ring_nph[p] / 2 : md.ring_nph[p];  // Bluestein length
    const int M = md.ring_M[p];
    int logM = 0;
    while ((1 << logM) < M) ++logM;
    for (int j = threadIdx.x; j < M; j += blockDim.x) {
        int jj = -1;
        if (j < n)
            jj = j;
        else if (j > M - n)
            jj = M - j;
        Z[zp(j)] = jj >= 0 ? cis_pi_frac(((long)jj * jj) % (2L * n), n) : make_double2(0.0, 0.0);
    }
    double2* ch = chirp_out + md.ring_chofs[p];
    for (int j = threadIdx.x; j <= n / 2; j += blockDim.x) {
        double2 c = cis_pi_frac(((long)j * j) % (2L * n), n);
        c.y = -c.y;
        ch[j] = c;
    }
    __syncthreads();
    fft<-1, kMaxFFT>(Z, M, logM, tw);
    double2* dst = filt_out + md.ring_bsofs[p];
    for (int j = threadIdx.x; j <= M / 2; j += blockDim.x) dst[j] = Z[zp(j)];
}

// ================================================================== k_final
// One block: -2lnL = sum_pairs chi + sum_blocks prior, fixed order.
__device__ __forceinline__ void final_map(const MapDesc& md, double* __restrict__ f)
{
    __shared__ double sh[16];
    double a = 0.0;
    for (int i = threadIdx.x; i < md.npair; i += 1024) a += md.chi[i];
    for (int i = threadIdx.x; i < md.nprior; i += 1024) a += md.prior[i];
    const double t = block_sum<1024>(a, sh);
    if (threadIdx.x == 0) {
        *f = t;
        if (!isfinite(t)) *md.nonfinite = 1;
    }
}

__global__ __launch_bounds__(1024) void k_final(const MapDesc* __restrict__ md_, double* __restrict__ f)
{
    final_map(*md_, f);
}

// one block per map of the group
__global__ __launch_bounds__(1024) void k_final_b(const MapDesc* __restrict__ mds, const BatchArgs a)
{
    final_map(mds[blockIdx.x], a.f + blockIdx.x);
}

// ================================================================== BLAS-1

// y and x may be the same vector (in-place scaling y = c y, y += c y).
__global__ void k_vec(int op, double* y, const double* x, double c, long n)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        switch (op) {
        case kVecCopy: y[i] = c * x[i]; break;
        case kVecSet: y[i] = c; break;
        case kVecAxpy: y[i] = fma(c, x[i], y[i]); break;
        case kVecMul: y[i] *= x[i]; break;
        case kVecDiv: y[i] /= x[i]; break;
        case kVecPow: y[i] = pow(y[i], c); break;
        }
    }
}

__global__ __launch_bounds__(256) void k_dot_part(const double* __restrict__ x, const double* __restrict__ y, long n,
                                                  double* __restrict__ part)
{
    __shared__ double sh[4];
    double a = 0.0;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) a = fma(x[i], y[i], a);
    const double t = block_sum<256>(a, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ __launch_bounds__(1024) void k_dot_final(const double* __restrict__ part, int np, double* __restrict__ out)
{
    __shared__ double sh[16];
    double a = 0.0;
    for (int i = threadIdx.x; i < np; i += 1024) a += part[i];
    const double t = block_sum<1024>(a, sh);
    if (threadIdx.x == 0) *out = t;
}

// ================================================================== launchers

// Raise a kernel's dynamic-LDS limit to kMaxLds once per device (function
// attributes belong to a device; one bit per device id in `done`).
static int allow_dynamic_lds(const void* fn, std::atomic<unsigned long long>& done)
{
    int dev = 0;
    CMBL_HIP(hipGetDevice(&dev));
    const unsigned long long bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return CMBL_OK;
    CMBL_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
    done.fetch_or(bit, std::memory_order_acq_rel);
    return CMBL_OK;
}

int lm_tiles(int L)
{
    const int nt = (L + kLM) / kLM;
    return nt * (nt + 1) / 2;
}

int launch_pre(const MapDesc& md, const MapDesc* d_md, const double* d_x, hipStream_t s)
{
    hipLaunchKernelGGL(k_pre, dim3(lm_tiles(md.L)), dim3(256), 0, s, d_md, d_x);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

template <int K>
static int synth_k(const WorkItem* items, int n, const MapDesc* d_maps, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    hipLaunchKernelGGL((k_synth<K, 1>), dim3(n), dim3(64), 0, s, items, d_maps, (const int*)nullptr);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}
int launch_adj(int K, const AdjItem* items, int n, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    switch (K) {
    case 1: hipLaunchKernelGGL(k_adj<1>, dim3(n), dim3(64), 0, s, items); break;
    case 2: hipLaunchKernelGGL(k_adj<2>, dim3(n), dim3(64), 0, s, items); break;
    case 4: hipLaunchKernelGGL(k_adj<4>, dim3(n), dim3(64), 0, s, items); break;
    case 8: hipLaunchKernelGGL(k_adj<8>, dim3(n), dim3(64), 0, s, items); break;
    default: return fail(CMBL_ERR_ARG, "unsupported rings-per-lane K");
    }
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}
int launch_adj_mma(const WorkItem* items, const MmaSub* subs, int n, const MapDesc* d_maps, const int* d_groups,
                   hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    hipLaunchKernelGGL(k_adj_mma, dim3(n), dim3(64 * kMmaWaves), 0, s, items, subs, d_maps, d_groups);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}
int launch_synth_mma(int K, const WorkItem* items, int n, const MapDesc* d_maps, const int* d_groups, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    if (K == 1)
        hipLaunchKernelGGL(k_synth_mma<1>, dim3(n), dim3(64), 0, s, items, d_maps, d_groups);
    else if (K == 2)
        hipLaunchKernelGGL(k_synth_mma<2>, dim3(2 * n), dim3(64), 0, s, items, d_maps, d_groups);
    else
        return fail(CMBL_ERR_ARG, "unsupported rings-per-lane K for the matrix-core synthesis");
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}
template <int K>
static int scan_k(const WorkItem* items, int n, const MapDesc* d_maps, int* d_lstart, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    hipLaunchKernelGGL(k_scan<K>, dim3(n), dim3(64), 0, s, items, d_maps, d_lstart);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_synth_pairs(int K, const WorkItem* items, int n, const MapDesc* d_maps, const int* d_groups, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    switch (K) {
    case 1: hipLaunchKernelGGL((k_synth<1, 2>), dim3(n), dim3(64), 0, s, items, d_maps, d_groups); break;
    case 2: hipLaunchKernelGGL((k_synth<2, 2>), dim3(n), dim3(64), 0, s, items, d_maps, d_groups); break;
    default: return fail(CMBL_ERR_ARG, "unsupported shared-synthesis shape");
    }
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_synth(int K, const WorkItem* items, int n, const MapDesc* d_maps, hipStream_t s)
{
    switch (K) {
    case 1: return synth_k<1>(items, n, d_maps, s);
    case 2: return synth_k<2>(items, n, d_maps, s);
    case 4: return synth_k<4>(items, n, d_maps, s);
    case 8: return synth_k<8>(items, n, d_maps, s);
    }
    return fail(CMBL_ERR_ARG, "unsupported rings-per-lane K");
}
template <int K>
static int capture_k(const WorkItem* items, int n, const MapDesc* d_maps, double* prev, double* cur, int* kk,
                     hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    hipLaunchKernelGGL(k_capture<K>, dim3(n), dim3(64), 0, s, items, d_maps, prev, cur, kk);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}
int launch_capture(int K, const WorkItem* items, int n, const MapDesc* d_maps, double* prev, double* cur, int* kk,
                   hipStream_t s)
{
    switch (K) {
    case 1: return capture_k<1>(items, n, d_maps, prev, cur, kk, s);
    case 2: return capture_k<2>(items, n, d_maps, prev, cur, kk, s);
    case 4: return capture_k<4>(items, n, d_maps, prev, cur, kk, s);
    case 8: return capture_k<8>(items, n, d_maps, prev, cur, kk, s);
    }
    return fail(CMBL_ERR_ARG, "unsupported rings-per-lane K");
}

int launch_adj_capture(const AdjCap* caps, const int* runs, int nruns, double2* st, int* sk, const MapDesc* d_md,
                       hipStream_t s)
{
    if (nruns <= 0) return CMBL_OK;
    hipLaunchKernelGGL(k_adj_capture, dim3(nruns), dim3(64), 0, s, caps, runs, st, sk, d_md);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_scan(int K, const WorkItem* items, int n, const MapDesc* d_maps, int* d_lstart, hipStream_t s)
{
    switch (K) {
    case 1: return scan_k<1>(items, n, d_maps, d_lstart, s);
    case 2: return scan_k<2>(items, n, d_maps, d_lstart, s);
    case 4: return scan_k<4>(items, n, d_maps, d_lstart, s);
    case 8: return scan_k<8>(items, n, d_maps, d_lstart, s);
    }
    return fail(CMBL_ERR_ARG, "unsupported rings-per-lane K");
}

template <int MODE, int MAXM>
static int ring_mm(const RingItem* items, int n, const MapDesc* d_maps, int lds, double* out, const double* in,
                   const double2* tw, hipStream_t s)
{
    static std::atomic<unsigned long long> lds_set{0};
    CMBL_TRY(allow_dynamic_lds((const void*)k_ring<MODE, MAXM>, lds_set));
    hipLaunchKernelGGL((k_ring<MODE, MAXM>), dim3(n), dim3(ring_threads(MAXM)), lds, s, items, d_maps, out, in, tw);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

// One instantiation per transform-length class (the classes' LDS sizes):
// the bound on the transform length bounds the registers of the FFT passes.
template <int MODE>
static int ring_m(const RingItem* items, int n, const MapDesc* d_maps, int lds, double* out, const double* in,
                  const double2* tw, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    if (lds > kMaxLds) return fail(CMBL_ERR_ARG, "ring transform longer than the LDS FFT");
    if (lds <= lds_bytes(kSmallFFT)) {
        hipLaunchKernelGGL(k_ring_small<MODE>, dim3(n), dim3(kSmallT), 0, s, items, d_maps, out, in, tw);
        CMBL_HIP(hipGetLastError());
        return CMBL_OK;
    }
    if (lds > lds_bytes(4096)) return ring_mm<MODE, 8192>(items, n, d_maps, lds, out, in, tw, s);
    if (lds > lds_bytes(2048)) return ring_mm<MODE, 4096>(items, n, d_maps, lds, out, in, tw, s);
    return ring_mm<MODE, 2048>(items, n, d_maps, lds, out, in, tw, s);
}

int launch_ring(int mode, const RingItem* items, int n, const MapDesc* d_maps, int lds, double* out,
                const double* in, const double2* tw, hipStream_t s)
{
    switch (mode) {
    case kRingLike: return ring_m<kRingLike>(items, n, d_maps, lds, out, in, tw, s);
    case kRingSyn: return ring_m<kRingSyn>(items, n, d_maps, lds, out, in, tw, s);
    case kRingAna: return ring_m<kRingAna>(items, n, d_maps, lds, out, in, tw, s);
    case kRingWeight: return ring_m<kRingWeight>(items, n, d_maps, lds, out, in, tw, s);
    }
    return fail(CMBL_ERR_ARG, "bad ring mode");
}

int launch_bluestein_setup(const MapDesc* d_md, const int* d_pairs, int npairs_bs, double2* d_out,
                           double2* d_chirp, int lds, const double2* tw, hipStream_t s)
{
    if (npairs_bs <= 0) return CMBL_OK;
    static std::atomic<unsigned long long> lds_set{0};
    CMBL_TRY(allow_dynamic_lds((const void*)k_bluestein_setup, lds_set));
    hipLaunchKernelGGL(k_bluestein_setup, dim3(npairs_bs), dim3(ring_threads(kMaxFFT)), lds, s, d_pairs, d_md, d_out, d_chirp,
                       tw);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_post(const MapDesc& md, const MapDesc* d_md, const double* d_x, double* d_g, int mode, hipStream_t s,
                double c)
{
    hipLaunchKernelGGL(k_post, dim3(lm_tiles(md.L)), dim3(256), 0, s, d_md, d_x, d_g, mode, c);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_coupling(const double* w, int L, double* M, hipStream_t s)
{
    hipLaunchKernelGGL(k_coupling, dim3(L / kCoupL + 1, L / kCoupD + 1), dim3(64 * kCoupD), 0, s, L, w, M);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_pre_pol(const MapDesc& md, const MapDesc* d_md, const double* t, const double* e, const double* b,
                   double2* d_rec, hipStream_t s)
{
    hipLaunchKernelGGL(k_pre_pol, dim3(lm_tiles(md.L)), dim3(256), 0, s, d_md, t, e, b, d_rec);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_synth_pol(int K, const WorkItem* items, int n, const MapDesc* d_md, const double2* d_rec, double* d_pt,
                     double* d_pq, double* d_pu, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    hipLaunchKernelGGL(k_synth_pol, dim3(n, K), dim3(64), 0, s, items, d_md, d_rec, d_pt, d_pq, d_pu);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_reorder(const double* in, double* out, long nside, int to_ring, hipStream_t s)
{
    const long npix = 12 * nside * nside;
    const int blocks = (int)std::min<long>((npix + 255) / 256, 8192);
    hipLaunchKernelGGL(k_reorder, dim3(blocks), dim3(256), 0, s, in, out, nside, to_ring);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_ldiv(double* y, const double* x, const double* dl, int L, hipStream_t s)
{
    const long n = (long)(L + 1) * (L + 1);
    const int blocks = (int)std::min<long>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_ldiv, dim3(blocks), dim3(256), 0, s, y, x, dl, L);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_pre_batch(const MapDesc* d_mds, const BatchArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_pre_b, dim3(a.tile0[a.n]), dim3(256), 0, s, d_mds, a);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_post_batch(const MapDesc* d_mds, const BatchArgs& a, int mode, hipStream_t s)
{
    hipLaunchKernelGGL(k_post_b, dim3(a.tile0[a.n]), dim3(256), 0, s, d_mds, a, mode);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_final_batch(const MapDesc* d_mds, const BatchArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_final_b, dim3(a.n), dim3(1024), 0, s, d_mds, a);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_final(const MapDesc* d_md, double* d_f, hipStream_t s)
{
    hipLaunchKernelGGL(k_final, dim3(1), dim3(1024), 0, s, d_md, d_f);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_vec(int op, double* y, const double* x, double c, long n, hipStream_t s)
{
    if (n <= 0) return CMBL_OK;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_vec, dim3((unsigned)blocks), dim3(256), 0, s, op, y, x, c, n);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

int launch_dot(const double* x, const double* y, long n, double* d_out, double* d_work, hipStream_t s)
{
    const int np = kDotParts;
    hipLaunchKernelGGL(k_dot_part, dim3(np), dim3(256), 0, s, x, y, n, d_work);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(1024), 0, s, d_work, np, d_out);
    CMBL_HIP(hipGetLastError());
    return CMBL_OK;
}

}  // namespace cmbl
