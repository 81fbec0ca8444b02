// Device kernels of the GPE step.  Every transform pass is a row pass
// (TR rows of N points along x per workgroup) or a column pass (TC columns
// of N points along y per workgroup); pointwise physics is fused into the
// passes so that each field round trip to HBM carries as much work as
// possible.  See vk_cfg.hpp for the layouts.
#pragma once
#include "vk_cfg.hpp"

// optional occupancy request for the pass kernels (waves per SIMD), and for
// the P2/P4 column passes alone
#ifdef VK_WAVES
#define VK_OCC __attribute__((amdgpu_waves_per_eu(VK_WAVES)))
#else
#define VK_OCC
#endif
#ifdef VK_COL_WAVES
#define VK_COCC __attribute__((amdgpu_waves_per_eu(VK_COL_WAVES)))
#else
#define VK_COCC VK_OCC
#endif
// P4 at 4 waves per SIMD (<= 128 VGPRs: two 512-thread workgroups per CU)
// is 9% faster than at the compiler's choice of 134-181 VGPRs
#ifndef VK_P4_WAVES
#define VK_P4_WAVES 4
#endif
#if VK_P4_WAVES > 0
#define VK_P4OCC(C) __attribute__((amdgpu_waves_per_eu(is_lat<C>::value ? 1 : VK_P4_WAVES)))
#else
#define VK_P4OCC(C) VK_COCC
#endif
#ifdef VK_P1_WAVES
#define VK_P1OCC __attribute__((amdgpu_waves_per_eu(VK_P1_WAVES)))
#else
#define VK_P1OCC VK_OCC
#endif
// P3 without particles or with real-space ones (PM 0, 4) at 4 waves per SIMD
// (<= 128 VGPRs; LAT shapes, one wave per SIMD, as they come)
#ifndef VK_P3_WAVES
#define VK_P3_WAVES 4
#endif
#define VK_P3OCC(C, PM) __attribute__((amdgpu_waves_per_eu(!is_lat<C>::value && ((PM) == 0 || (PM) == 4) ? VK_P3_WAVES : 1)))

namespace vk {

// ----------------------------------------------------------------------------
// thread <-> data mapping helpers
// ----------------------------------------------------------------------------

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Row passes remap so that each XCD takes a contiguous run of row
// blocks: neighbouring row blocks share 128-byte lines of the panel layout,
// and those lines then stay in one L2.
__device__ __forceinline__ int xcd_remap(int b, int nb)
{
    return (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
}

#define VK_ROW_SETUP(C)                                                    \
    constexpr int N = C::N, S = C::S, T = C::T, TC = C::TC, TR = C::TR;    \
    constexpr int NP = C::NP;                                              \
    (void)NP;                                                              \
    extern __shared__ double lds[];                                        \
    const int u = tid_of<C>();                                             \
    const int q_ = u % (TR * TC);                                          \
    const int rr = q_ / TC, c = q_ % TC, pidx0 = u / (TR * TC);            \
    const int t = TC * pidx0 + c;                                          \
    const int y = xcd_remap(blk_, nblk_) * TR + rr;                       \
    double* lg = lds + rr * C::ROWRS;

#define VK_COL_SETUP(C, PEXPR)                                             \
    constexpr int N = C::N, S = C::S, T = C::T, TC = C::TC;                \
    constexpr int NP = C::NP;                                              \
    (void)NP;                                                              \
    extern __shared__ double lds[];                                        \
    const int u = tid_of<C>();                                             \
    const int c = u % TC, t = u / TC;                                      \
    const int p = (PEXPR);                                                 \
    const int kx = p * TC + c;                                             \
    double* lg = lds + c * C::COLRS;

// Column-pass setup for G columns per workgroup (G divides TC).  For
// G < TC the TC/G workgroups of a panel are siblings placed on one XCD:
// blocks come in groups of 8*TC/G covering 8 panels, and blocks b and b + 8
// (consecutive on one XCD under round-robin dispatch) share a panel.  Blocks
// past NPAN panels return here, before any barrier.
#define VK_COL_SETUP_G(C, G, B, PEXPR, NPAN)                                \
    constexpr int N = C::N, S = C::S, T = C::T, TC = C::TC;                \
    constexpr int NP = C::NP;                                              \
    (void)NP;                                                              \
    constexpr int GS_ = TC / (G);                                          \
    extern __shared__ double lds[];                                        \
    int pb_ = (B), hh_ = 0;                                                \
    if constexpr (GS_ > 1) {                                               \
        const int r_ = pb_ % (8 * GS_);                                    \
        hh_ = r_ / 8;                                                      \
        pb_ = pb_ / (8 * GS_) * 8 + r_ % 8;                                \
        if (pb_ >= (NPAN)) return;                                         \
    }                                                                      \
    const int p = (PEXPR);                                                 \
    const int u = tid_of<C>();                                             \
    const int cl_ = u % (G), t = u / (G);                                  \
    const int c = hh_ * (G) + cl_;                                         \
    const int kx = p * TC + c;                                             \
    double* lg = lds + cl_ * C::COLRS;

// panel holding kx = t + T*s in a row pass
#define VK_PANEL(s) (pidx0 + (T / TC) * (s))

__device__ __forceinline__ cplx czero() { return mk(0.0, 0.0); }

// ----------------------------------------------------------------------------
// Generic transform passes (set/get, diagnostics, conformance hook)
// ----------------------------------------------------------------------------

// x-space rows -> FFT along x -> H, all panels.
template <class C>
__device__ __forceinline__ void row_fwd_body(int blk_, int nblk_, const cplx* __restrict__ X, cplx* __restrict__ H,
                                             const cplx* __restrict__ tw)
{
    VK_ROW_SETUP(C)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
    const cplx* xr = X + (size_t)y * N;
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = xr[t + T * s];
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) H[hoff<C>(VK_PANEL(s), y, c)] = v[s];
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_OCC k_row_fwd(const cplx* __restrict__ X, cplx* __restrict__ H,
                                                     const cplx* __restrict__ tw)
{
    row_fwd_body<C>(blockIdx.x, gridDim.x, X, H, tw);
}

// H column -> FFT along y -> K, all panels.  op 1: dealias.
template <class C, int G = C::TC>
__device__ __forceinline__ void col_fwd_body(int b, const cplx* __restrict__ H, cplx* __restrict__ K,
                                             const cplx* __restrict__ tw, int op)
{
    VK_COL_SETUP_G(C, G, b, pb_, C::NP)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = H[hoff<C>(p, t + T * s, c)];
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
    const int kxs = ksg(kx, N);
    cplx* kr = K + (size_t)kx * N;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int ky = t + T * s;
        cplx a = v[s];
        if (op == 1 && kmasked(kxs, ksg(ky, N), N)) a = czero();
        kr[ky] = a;
    }
}

template <class C, int G = C::TC>
__global__ void __launch_bounds__(G * C::T) VK_OCC k_col_fwd(const cplx* __restrict__ H, cplx* __restrict__ K,
                                                     const cplx* __restrict__ tw, int op)
{
    col_fwd_body<C, G>(blockIdx.x, H, K, tw, op);
}

// panels a column pass over pmode covers (0 all, 1 retained)
#define VK_NPAN(C, g, pmode) ((pmode) == 0 ? C::NP : (g).Pp + (g).Pn)

// K row -> op -> unnormalised inverse FFT along y -> H.
// op 0: as is; 2: times i*ky.
template <class C, int G = C::TC>
__device__ __forceinline__ void col_inv_body(int b, const cplx* __restrict__ K, cplx* __restrict__ H,
                                             const cplx* __restrict__ tw, Geo g, int pmode, int op)
{
    VK_COL_SETUP_G(C, G, b, panel_of_block(pb_, C::NP, g, pmode), VK_NPAN(C, g, pmode))
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
    const cplx* kr = K + (size_t)kx * N;
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = conjc(kr[t + T * s]);
    if (op == 2) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const double kys = ksg(t + T * s, N);
            v[s] = mk(kys * v[s].y, -kys * v[s].x);
        }
    }
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) H[hoff<C>(p, t + T * s, c)] = conjc(v[s]);
}

template <class C, int G = C::TC>
__global__ void __launch_bounds__(G * C::T) VK_OCC k_col_inv(const cplx* __restrict__ K, cplx* __restrict__ H,
                                                     const cplx* __restrict__ tw, Geo g, int pmode, int op)
{
    col_inv_body<C, G>(blockIdx.x, K, H, tw, g, pmode, op);
}

// H row (panels of mode pload) -> unnormalised inverse FFT along x -> times
// scale -> X.
template <class C>
__device__ __forceinline__ void row_inv_body(int blk_, int nblk_, const cplx* __restrict__ H, cplx* __restrict__ X,
                                             const cplx* __restrict__ tw, Geo g, int pload, double scale)
{
    VK_ROW_SETUP(C)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
    const brsrc rH = mkbuf(H, N);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int pp = VK_PANEL(s);
        v[s] = bld(rH, boff(hoff<C>(pp, y, c), panel_stored(pp, NP, g, pload)));
    }
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = conjc(v[s]);
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
    cplx* xr = X + (size_t)y * N;
#pragma unroll
    for (int s = 0; s < S; ++s) xr[t + T * s] = rmul(scale, conjc(v[s]));
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_OCC k_row_inv(const cplx* __restrict__ H, cplx* __restrict__ X,
                                                     const cplx* __restrict__ tw, Geo g, int pload, double scale)
{
    row_inv_body<C>(blockIdx.x, gridDim.x, H, X, tw, g, pload, scale);
}

// zero a field
__global__ void k_zero(cplx* __restrict__ K, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) K[i] = czero();
}

// zero the dealiased modes of a k-space field (all N^2 entries)
__global__ void k_dealias(cplx* __restrict__ K, int N)
{
    const size_t n2 = (size_t)N * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x) {
        const int kx = (int)(i / N), ky = (int)(i % N);
        if (kmasked(ksg(kx, N), ksg(ky, N), N)) K[i] = czero();
    }
}

// ----------------------------------------------------------------------------
// Fused RK4 / ARGLE passes
// ----------------------------------------------------------------------------

// Sums over a row of nv <= 8 values per point group: thread t of the row's T
// holds x[]; out[i] = the sum over t in a fixed tree (neighbour pairs, then
// pairs of pairs, ...), the same in every workgroup shape.  sh: nv * T
// doubles of LDS of this row.  Every thread of the workgroup calls it.
template <int NV, int T>
__device__ __forceinline__ void row_sum(const double (&x)[NV], double* sh, int t, double* __restrict__ out)
{
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NV; ++i) sh[i * T + t] = x[i];
#pragma unroll
    for (int h = 1; h < T; h *= 2) {
        lds_barrier();
        if (t % (2 * h) == 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) sh[i * T + t] += sh[i * T + t + h];
        }
    }
    lds_barrier();
    if (t == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) out[i] = sh[i * T];
    }
}

// P1 after its loads: v holds the conjugated Hpsi row points of this thread
// (NORM: the row's sum of |psi|^2 goes to nsum[y])
template <class C, bool XS, bool NORM = false, class W>
__device__ __forceinline__ void p1_core(cplx (&v)[C::S], double* lg, int t, int y, int pidx0, int c,
                                        cplx* __restrict__ Hrho, const W& w_, const Geo& g,
                                        double scale, cplx* __restrict__ Xpsi, double* __restrict__ nsum = nullptr)
{
    constexpr int N = C::N, S = C::S, T = C::T, TC = C::TC;
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
    if constexpr (XS) {
        cplx* xr = Xpsi + (size_t)y * N;
#pragma unroll
        for (int s = 0; s < S; ++s) xr[t + T * s] = rmul(scale, conjc(v[s]));
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const double a = scale * v[s].x, b = scale * v[s].y;   // conj does not change |.|
        v[s] = mk(a * a + b * b, 0.0);
    }
    double ns[1] = {0.0};
    if constexpr (NORM) {
#pragma unroll
        for (int s = 0; s < S; ++s) ns[0] += v[s].x;
    }
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int pp = VK_PANEL(s);
        if (pp < g.Pp) Hrho[hoff<C>(pp, y, c)] = v[s];
    }
    if constexpr (NORM) row_sum<1, T>(ns, lg, t, nsum + y);
}

// P1 (row): psi row from Hpsi (inverse along x, times 1/N^2), rho = |psi|^2,
// forward along x, keep kx >= 0 retained panels (rho is real).  The psi row
// is stored in x-space (Xpsi[y*N + x]) for P3, which then needs no transform
// of its own for psi; the diagnostics do without (XS false).
template <class C, bool XS = true, bool NORM = false>
__device__ __forceinline__ void p1_body(int blk_, int nblk_, const cplx* __restrict__ Hpsi, cplx* __restrict__ Hrho,
                                                const cplx* __restrict__ tw, Geo g, int psi_pmode,
                                                double scale, cplx* __restrict__ Xpsi,
                                                double* __restrict__ nsum = nullptr)
{
    VK_ROW_SETUP(C)
    cplx v[S];
    const brsrc rH = mkbuf(Hpsi, N);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int pp = VK_PANEL(s);
        v[s] = bld(rH, boff(hoff<C>(pp, y, c), panel_stored(pp, NP, g, psi_pmode)));
    }
    const auto w_ = twiddles<C>(tw, t);
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = conjc(v[s]);   // a panel not stored loads as zero
    p1_core<C, XS, NORM>(v, lg, t, y, pidx0, c, Hrho, w_, g, scale, Xpsi, nsum);
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_P1OCC k_p1x(const cplx* __restrict__ Hpsi, cplx* __restrict__ Hrho,
                                                 const cplx* __restrict__ tw, Geo g, int psi_pmode,
                                                 double scale, cplx* __restrict__ Xpsi)
{
    p1_body<C>(blockIdx.x, gridDim.x, Hpsi, Hrho, tw, g, psi_pmode, scale, Xpsi);
}

// Retained-panel geometry of a size, at compile time (as the host computes
// it), and the LDS slots of the prefetching P1: the points s of a thread
// whose panel can be stored get a 16-byte slot per lane and wave; points
// whose stored lanes are disjoint share a slot (at 4096^2: 11 slots for the
// 12 point indices with stored panels).
struct P1Slots {
    int slot[16];
    int nslot;
};
template <class C> constexpr int geo_pp()
{
    constexpr int M = C::N / 3, pp = (M + 1 + C::TC - 1) / C::TC, pn = (M + C::TC - 1) / C::TC;
    return pp + pn > C::NP ? C::NP : pp;
}
template <class C> constexpr int geo_pn()
{
    constexpr int M = C::N / 3, pp = (M + 1 + C::TC - 1) / C::TC, pn = (M + C::TC - 1) / C::TC;
    return pp + pn > C::NP ? 0 : pn;
}
template <class C> constexpr P1Slots p1_slots()
{
    static_assert(C::S <= 16 && C::T / C::TC <= 128, "slot map sized for S <= 16, T/TC <= 128");
    P1Slots m{};
    unsigned long long occ[16][2] = {};
    m.nslot = 0;
    for (int s = 0; s < C::S; ++s) {
        unsigned long long b[2] = {0ull, 0ull};
        bool any = false;
        for (int q = 0; q < C::T / C::TC; ++q) {
            const int p = q + (C::T / C::TC) * s;
            if (p < geo_pp<C>() || p >= C::NP - geo_pn<C>()) {
                b[q / 64] |= 1ull << (q % 64);
                any = true;
            }
        }
        m.slot[s] = -1;
        if (!any) continue;
        for (int k = 0; k < m.nslot; ++k)
            if (!(occ[k][0] & b[0]) && !(occ[k][1] & b[1])) {
                m.slot[s] = k;
                break;
            }
        if (m.slot[s] < 0) m.slot[s] = m.nslot++;
        occ[m.slot[s]][0] |= b[0];
        occ[m.slot[s]][1] |= b[1];
    }
    return m;
}
template <class C> constexpr size_t p1p_lds()
{
    return (size_t)C::TR * C::ROWRS * sizeof(double) + (size_t)p1_slots<C>().nslot * C::ROWT * sizeof(cplx);
}

// P1 of an RK4 stage (retained panels) on the psi-row path, persistent: each
// workgroup walks row blocks of its XCD's contiguous range (XCD x = block %
// 8 owns [x R/8, (x+1) R/8), its workgroups stride through it) and loads the
// next block's Hpsi points into LDS with asynchronous global->LDS copies
// while it transforms the current one.  Every workgroup runs the same fixed
// number of iterations (the host checks that the blocks divide evenly).
template <class C>
__global__ void __launch_bounds__(C::ROWT) k_p1xp(const cplx* __restrict__ Hpsi, cplx* __restrict__ Hrho,
                                                  const cplx* __restrict__ tw, Geo g, double scale,
                                                  cplx* __restrict__ Xpsi)
{
    constexpr P1Slots SM = p1_slots<C>();
    constexpr int N = C::N, S = C::S, T = C::T, TC = C::TC, TR = C::TR, NP = C::NP;
    constexpr int NW = C::ROWT / 64;
    static_assert(C::ROWT % 64 == 0, "whole waves");
    extern __shared__ double lds[];
    const int u = threadIdx.x;
    const int q_ = u % (TR * TC);
    const int rr = q_ / TC, c = q_ % TC, pidx0 = u / (TR * TC);
    const int t = TC * pidx0 + c;
    double* lg = lds + rr * C::ROWRS;
    cplx* buf = reinterpret_cast<cplx*>(lds + TR * C::ROWRS);
    const int lane = u % 64, wv = u / 64;
    const int R8 = (N / TR) / 8, G8 = gridDim.x / 8;
    const int xcd = blockIdx.x % 8, j = blockIdx.x / 8;
    const int K = R8 / G8;
    auto prefetch = [&](int blk) {
        const int yy = blk * TR + rr;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (SM.slot[s] < 0) continue;
            const int pp = pidx0 + (T / TC) * s;
            if (pp < g.Pp || pp >= NP - g.Pn)
                __builtin_amdgcn_global_load_lds(
                    (const void*)(Hpsi + hoff<C>(pp, yy, c)),
                    (__attribute__((address_space(3))) void*)(buf + (SM.slot[s] * NW + wv) * 64), 16, 0, 0);
        }
    };
    prefetch(xcd * R8 + j);
    for (int k = 0; k < K; ++k) {
        const int y = (xcd * R8 + j + k * G8) * TR + rr;
        // this wave's copies have landed (vmcnt), and every wave's (barrier)
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        cplx v[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int pp = pidx0 + (T / TC) * s;
            v[s] = (SM.slot[s] >= 0 && (pp < g.Pp || pp >= NP - g.Pn))
                       ? conjc(buf[(SM.slot[s] * NW + wv) * 64 + lane])
                       : czero();
        }
        // all reads are done before the next copies overwrite the slots
        __syncthreads();
        if (k + 1 < K) prefetch(xcd * R8 + j + (k + 1) * G8);
        p1_core<C, true>(v, lg, t, y, pidx0, c, Hrho, tw, g, scale, Xpsi);
    }
}

// P2 (column, kx >= 0 retained panels): forward along y, dealias
// (P_G), inverse along y, in place.  flags & 1: also the particle
// potential column HV = IFFT_y(KV); flags & 2: store the dealiased
// rho-hat row into K-space Krho (for the particle force).
// FL >= 0: the flags as a compile-time constant (flags is then ignored).
template <class C, int G = C::TC, int FL = -1>
__device__ __forceinline__ void p2_body(int blk_, int nblk_, cplx* __restrict__ Hrho, cplx* __restrict__ HV,
                                                const cplx* __restrict__ KV, cplx* __restrict__ Krho,
                                                const cplx* __restrict__ tw, Geo g, int flags_)
{
    const int flags = FL >= 0 ? FL : flags_;
    VK_COL_SETUP_G(C, G, blk_, pb_, g.Pp)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = Hrho[hoff<C>(p, t + T * s, c)];
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int ky = t + T * s;
        const bool m = kmasked(kx, ksg(ky, N), N);
        if (m) v[s] = czero();
        else if (flags & 2) Krho[(size_t)kx * N + ky] = v[s];
        v[s] = conjc(v[s]);
    }
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) Hrho[hoff<C>(p, t + T * s, c)] = conjc(v[s]);
    if (flags & 1) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int ky = t + T * s;
            v[s] = kmasked(kx, ksg(ky, N), N) ? czero() : conjc(KV[(size_t)kx * N + ky]);
        }
        fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
        for (int s = 0; s < S; ++s) HV[hoff<C>(p, t + T * s, c)] = conjc(v[s]);
    }
}

template <class C, int G = C::TC, int FL = -1>
__global__ void __launch_bounds__(G * C::T) VK_COCC k_p2(cplx* __restrict__ Hrho, cplx* __restrict__ HV,
                                                const cplx* __restrict__ KV, cplx* __restrict__ Krho,
                                                const cplx* __restrict__ tw, Geo g, int flags)
{
    p2_body<C, G, FL>(blockIdx.x, gridDim.x, Hrho, HV, KV, Krho, tw, g, flags);
}

// deterministic workgroup sum of NV values per thread; result valid in
// thread 0.  sh must hold NV * (blockDim/64) doubles.
template <int NV>
__device__ __forceinline__ void block_sum(double (&x)[NV], double* sh)
{
    if (blockDim.x < 64) {
        // partial wave: no cross-lane shuffles over inactive lanes
        const int nt = blockDim.x;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NV; ++i) sh[i * nt + threadIdx.x] = x[i];
        __syncthreads();
        if (threadIdx.x == 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                double s = 0.0;
                for (int k = 0; k < nt; ++k) s += sh[i * nt + k];
                x[i] = s;
            }
        }
        __syncthreads();
        return;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x[i] += __shfl_xor(x[i], o, 64);
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) sh[i * nw + w] = x[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double s = 0.0;
            for (int k = 0; k < nw; ++k) s += sh[i * nw + k];
            x[i] = s;
        }
    }
    __syncthreads();
}

// Real-space particle terms for P3 (used when the particle potential's
// spectrum is negligible beyond the dealias radius, so that the reference's
// spectral translation IFFT(exp(-i k.q) Vhat) equals V(x - q) to far below
// FP64 roundoff; see the host-side selection).
// V and its gradient factor into one function of x and one of y per particle,
// tabulated over the window by k_wtab whenever the positions change.  P3 with
// the sines and exponentials in its point loop took 17.5 us at 512^2 with 8
// particles (229 VGPRs and 162 us at 4096^2 with 32); from the tables 10.9 us
// (at most 128 VGPRs, 138 us at 4096^2 with 32 and without any).
struct P3Part {
    const int4* win;     // per particle: first column and count of its window, first row and count
    const double2* tx;   // [particle][k < N]: ex, -ex X dX/dx / d^2, ex = exp(-X^2 / (2 d^2))
    const double2* ty;   // the same in y, times V0
    double* ppart;       // per row block, wave and particle: sum rho_raw * dV/dx, dV/dy
    unsigned char* phit; // per row block and particle: 1 if the window reaches the block
    int np;
    const double* vx;    // static potential on the grid (PM 8)
};

// minimum-image displacement in [-pi, pi)
__device__ __forceinline__ double pwrap(double a)
{
    const double tp = 6.283185307179586476925;
    return a - tp * rint(a * (1.0 / tp));
}

// periodic coordinate of src/gpe_particle.f90:46-50 (c = pi/L = 1/2):
// X = (1/c)(s + s^3/6 + s^5/40), s = sin(c a); also dX/da
__device__ __forceinline__ void pcoord(double a, double& X, double& dX)
{
    double sn, cs;
    sincos(0.5 * a, &sn, &cs);
    const double s2 = sn * sn;
    X = 2.0 * (sn + (1.0 / 6.0) * (s2 * sn) + (1.0 / 40.0) * (s2 * s2 * sn));
    dX = (1.0 + 0.5 * s2 + 0.125 * s2 * s2) * cs;
}

// Advective ARGLE terms (src/gpe.f90:78-81,91-94,114-146): tg adds the
// Taylor-Green velocity u = (sin x cos y, -cos x sin y) as
// -i u.grad psi - |u|^2 psi / (4 alpha); (vx, vy) the constant counterflow
// -i v.grad psi.  c4 = 1/(4 alpha); sc normalises the gradient transforms.
struct AdvArgs {
    int tg;
    double vx, vy, c4, sc;
    // a caller-supplied velocity field in place of the Taylor-Green one
    // (x-space, x fastest), when ux is set
    const double* ux;
    const double* uy;
};

// P3 (row): rho_d (+ i V) row from the kx >= 0 halves (Hermitian), psi row
// as P1 stored it (x-space, scaled), N = (gs*rho_d + V) * psi, forward along
// x -> HN.  gs = +-g/N^2, vs = +-1/N^2 (RK4 +, ARGLE -).
// PM (particle mode, compile time): 0 none; 1 spectral potential (HV); 4
// real-space potential of moving particles + force partial sums; 8 static
// potential from the grid array.
// vsign: +1 RK4, -1 ARGLE.
// ADV: advective ARGLE; grad psi from the rows of i kx Hpsi and of Hdy =
// IFFT_y(i ky kpsi), two more transforms.
template <class C, int PM, bool ADV = false>
__device__ __forceinline__ void p3_body(int blk_, int nblk_, const cplx* __restrict__ Hrhod, const cplx* __restrict__ HV,
                                                const cplx* __restrict__ Xpsi, cplx* __restrict__ HN,
                                                const cplx* __restrict__ tw, Geo g, int store_pmode, double gs,
                                                double vs, double vsign, P3Part pa,
                                                const cplx* __restrict__ Hpsi = nullptr,
                                                const cplx* __restrict__ Hdy = nullptr, AdvArgs aa = AdvArgs{})
{
    constexpr int flags = PM;
    VK_ROW_SETUP(C)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
    const int Kp = TC * g.Pp;
    // particle windows staged after the transform regions during the first
    // transform, read back as broadcasts
    int4* ql = reinterpret_cast<int4*>(lds + TR * C::ROWRS);
    if constexpr ((flags & 4) != 0) {
        for (int i = threadIdx.x; i < pa.np; i += blockDim.x) ql[i] = pa.win[i];
        // a one-wave workgroup's transform has no barrier
        if constexpr (C::ROWT <= 64) lds_barrier();
    }
    // kx >= 0 columns are stored; kx < 0 ones are the conjugates of N - kx
    const brsrc rR = mkbuf(Hrhod, N);
    cplx bv[(flags & 1) ? S : 1];
    cplx xv[is_lat<C>::value ? S : 1];
    double sv[(flags & 8) ? S : 1];
    if constexpr (is_lat<C>::value) {
#pragma unroll
        for (int s = 0; s < S; ++s) xv[s] = (Xpsi + (size_t)y * N)[t + T * s];
    }
    if constexpr ((flags & 8) != 0) {
#pragma unroll
        for (int s = 0; s < S; ++s) sv[(flags & 8) ? s : 0] = pa.vx[(size_t)y * N + t + T * s];
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int kxi = t + T * s;
        const bool neg = kxi >= Kp;
        const int km = neg ? N - kxi : kxi;
        const unsigned o = boff(hoff<C>(km / TC, y, km % TC), kxi < Kp || kxi > N - Kp);
        v[s] = bld(rR, o);
        if constexpr ((flags & 1) != 0) bv[(flags & 1) ? s : 0] = bld(mkbuf(HV, N), o);
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const bool neg = t + T * s > N - Kp;
        cplx a = v[s], b = czero();
        if constexpr ((flags & 1) != 0) b = bv[(flags & 1) ? s : 0];
        if (neg) {
            a = conjc(a);
            b = conjc(b);
        }
        v[s] = conjc(mk(a.x - b.y, a.y + b.x));   // a + i b, conj for the inverse
    }
    fft_fwd<N, S, C::SPLIT, PM == 4>(v, lg, t, w_);
    // v[s].x = rho_d (unnormalised); v[s].y = -V (unnormalised, flags & 1).
    double f[S];   // the real factor g rho_d + V
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if constexpr ((flags & 1) != 0) f[s] = gs * v[s].x + vs * (-v[s].y);
        else f[s] = gs * v[s].x;
    }
    if constexpr ((flags & 8) != 0) {
#pragma unroll
        for (int s = 0; s < S; ++s) f[s] += vsign * sv[(flags & 8) ? s : 0];
    }
    if constexpr ((flags & 4) != 0) {
        // real-space particle potential added into f; force partials
        const int blk = xcd_remap(blk_, nblk_);
        const int yb = blk * TR;
        // The particle loop has no workgroup barrier: every wave tests the
        // windows itself (one lane per particle, a ballot gives the hit set,
        // the same in every wave), reduces its force partials with lane
        // shuffles and writes them per wave; the per-block hit flags tell
        // the reduction which entries were written.
        constexpr int WV = C::ROWT < 64 ? C::ROWT : 64;   // lanes of a wave in use
        constexpr int NW = (C::ROWT + 63) / 64;            // waves per workgroup
        const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;
        const brsrc rX = mkbuf_bytes(pa.tx, pa.np * N * 16);
        for (int base = 0; base < pa.np; base += WV) {
            const int pq = base + lane;
            bool hit = false;
            if (lane < WV && pq < pa.np) {
                const int4 w = ql[pq];
                for (int r2 = 0; r2 < TR; ++r2) hit |= ((yb + r2 - w.z) & (N - 1)) < w.w;
                if (wv == 0) pa.phit[(size_t)blk * pa.np + pq] = hit ? 1 : 0;
            }
            // hit particles in increasing order (uniform over the wave)
            for (unsigned long long m = __ballot(hit); m != 0ull; m &= m - 1ull) {
                const int pp = base + __builtin_ctzll(m);
                const int4 w = ql[pp];
                double fr[2] = {0.0, 0.0};
                const int ky = (y - w.z) & (N - 1);
                const bool row = ky < w.w;
                const double2 wy = pa.ty[(size_t)pp * N + (row ? ky : 0)];
                // LAT shapes: a window spans several of a thread's points, all
                // its loads at once; else (window narrower than the thread
                // stride T) mostly one, skipped by the waves outside
                cplx wx[is_lat<C>::value ? S : 1];
                if constexpr (is_lat<C>::value) {
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        const int k = (t + T * s - w.x) & (N - 1);
                        wx[s] = bld(rX, boff((size_t)pp * N + k, row && k < w.y));
                    }
                }
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const int k = (t + T * s - w.x) & (N - 1);
                    if (is_lat<C>::value || (row && k < w.y)) {
                        const cplx a = is_lat<C>::value ? wx[is_lat<C>::value ? s : 0] : bld(rX, boff((size_t)pp * N + k, true));
                        f[s] += vsign * (a.x * wy.x);
                        fr[0] += v[s].x * (a.y * wy.x);
                        fr[1] += v[s].x * (a.x * wy.y);
                    }
                }
#pragma unroll
                for (int o = WV / 2; o > 0; o >>= 1) {
                    fr[0] += __shfl_xor(fr[0], o, WV);
                    fr[1] += __shfl_xor(fr[1], o, WV);
                }
                if (lane == 0) {
                    double* q = pa.ppart + (((size_t)blk * NW + wv) * pa.np + pp) * 2;
                    q[0] = fr[0];
                    q[1] = fr[1];
                }
            }
        }
    }
    // Taylor-Green u at (x, y) from the twiddle table: tw[k] = e^{-2 pi i k/N}
    const double cy_ = tw[y].x, sy_ = -tw[y].y;
    if constexpr (ADV) {
        if (aa.ux) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const size_t i = (size_t)y * N + t + T * s;
                const double ux = aa.ux[i], uy = aa.uy[i];
                f[s] -= aa.c4 * (ux * ux + uy * uy);
            }
        } else if (aa.tg) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const cplx e = tw[t + T * s];
                const double ux = -e.y * cy_, uy = -e.x * sy_;
                f[s] -= aa.c4 * (ux * ux + uy * uy);
            }
        }
    }
    const cplx* xr = Xpsi + (size_t)y * N;
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = rmul(f[s], is_lat<C>::value ? xv[is_lat<C>::value ? s : 0] : xr[t + T * s]);
    if constexpr (ADV) {
        // -i (u + v).grad psi, one gradient component at a time
        cplx w[S];
#pragma unroll 1
        for (int comp = 0; comp < 2; ++comp) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int pp = VK_PANEL(s);
                cplx a = czero();
                if (panel_stored(pp, NP, g, 0)) {
                    if (comp == 0) {
                        a = Hpsi[hoff<C>(pp, y, c)];
                        const double kk = (double)ksg(t + T * s, N);
                        a = mk(-kk * a.y, kk * a.x);   // i kx
                    } else {
                        a = Hdy[hoff<C>(pp, y, c)];
                    }
                }
                w[s] = conjc(a);
            }
            fft_fwd<N, S, C::SPLIT, PM == 4>(w, lg, t, w_);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const cplx e = tw[t + T * s];
                double uf;
                if (aa.ux) uf = (comp == 0 ? aa.ux : aa.uy)[(size_t)y * N + t + T * s];
                else uf = aa.tg ? (comp == 0 ? -e.y * cy_ : -e.x * sy_) : 0.0;
                const double u = uf + (comp == 0 ? aa.vx : aa.vy);
                const cplx d = rmul(aa.sc, conjc(w[s]));   // d psi / dx_comp
                v[s] = cadd(v[s], mk(u * d.y, -u * d.x));  // -i u d
            }
        }
    }
    fft_fwd<N, S, C::SPLIT, PM == 4>(v, lg, t, w_);
    // branch-free buffer stores (an unstored panel gets the out-of-range
    // offset and is dropped): conditional stores made the compiler sink the
    // last butterfly into one branch per store (P3 0.191 -> 0.187 ms)
    const brsrc rN = mkbuf(HN, N);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int pp = VK_PANEL(s);
        bst(rN, boff(hoff<C>(pp, y, c), panel_stored(pp, NP, g, store_pmode)), v[s]);
    }
}

template <class C, int PM>
__global__ void __launch_bounds__(C::ROWT) VK_OCC k_p3a(const cplx* __restrict__ Hrhod, const cplx* __restrict__ HV,
                                                 const cplx* __restrict__ Hpsi, const cplx* __restrict__ Xpsi,
                                                 const cplx* __restrict__ Hdy, cplx* __restrict__ HN,
                                                 const cplx* __restrict__ tw, Geo g, double gs, double vs,
                                                 double vsign, P3Part pa, AdvArgs aa)
{
    p3_body<C, PM, true>(blockIdx.x, gridDim.x, Hrhod, HV, Xpsi, HN, tw, g, 0, gs, vs, vsign, pa, Hpsi, Hdy, aa);
}

template <class C, int PM>
__global__ void __launch_bounds__(C::ROWT) VK_P3OCC(C, PM) k_p3x(const cplx* __restrict__ Hrhod, const cplx* __restrict__ HV,
                                                 const cplx* __restrict__ Xpsi, cplx* __restrict__ HN,
                                                 const cplx* __restrict__ tw, Geo g, int store_pmode, double gs,
                                                 double vs, double vsign, P3Part pa)
{
    p3_body<C, PM>(blockIdx.x, gridDim.x, Hrhod, HV, Xpsi, HN, tw, g, store_pmode, gs, vs, vsign, pa);
}

struct RKArgs {
    cplx pref;      // (1 - i disp)/i
    double alpha, omega;
    double wacc;    // dt/6 (stages 1,4) or dt/6*2 (stages 2,3)
    double cstep;   // dt/2, dt/2, dt, - for stages 1..3
    double r1;      // stage 2: str2 after stage 1 = r1 (K2 - K0), r1 = (dt/6)/(dt/2)
    double r3;      // stage 4: str2 after stage 3 = K1 + r3 (K2 - K0), r3 = (dt/3)/dt
    int stage;
};

// P4 (column, retained panels both signs): forward along y -> N-hat;
// RHS = pref*((alpha k^2 - omega) psi_s-hat + N-hat) on the retained disk;
// RK4 accumulation and stage update (src/gpe.f90:366-487);
// inverse along y of the new kpsi -> Hpsi.
// K0 = str1 (= kpsi at step start), K1 = str2, K2 = stage kpsi.  Stages 1
// and 3 do not store str2: the term they would add, (dt/6) rhs1 or
// (dt/3) rhs3, equals r (K2 - K0) with the K2 they write, and the next
// stage rebuilds it from arrays it reads anyway (two fewer field writes
// and one fewer field read per step; each costs one rounding of K2, ~1 ulp
// of kpsi).  The stage is a compile-time constant, and the K accesses of
// the dealiased modes go to the out-of-range offset (loads read zero,
// stores are dropped), so the loads of all points are issued back to back.
// G < TC: G of a panel's TC columns per workgroup (sibling workgroups of a
// panel on one XCD, as in P2).
template <class C, int STAGE, int G = C::TC>
__device__ __forceinline__ void p4_body(int blk_, int nblk_, const cplx* __restrict__ HN, cplx* __restrict__ Hpsi,
                                                cplx* __restrict__ K0, cplx* __restrict__ K1,
                                                cplx* __restrict__ K2, const cplx* __restrict__ tw,
                                                Geo g, RKArgs a)
{
    VK_COL_SETUP_G(C, G, blk_, panel_of_block(pb_, C::NP, g, 1), g.Pp + g.Pn)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = HN[hoff<C>(p, t + T * s, c)];
    const int kxs = ksg(kx, N);
    const size_t rowo = (size_t)kx * N;
    const brsrc r0 = mkbuf(K0, N), r1 = mkbuf(K1, N), r2 = mkbuf(K2, N);
    // LAT: the K operands before the transform (their latency overlaps it)
    constexpr bool LAT = is_lat<C>::value;
    cplx k0v[LAT ? S : 1], k1v[LAT && STAGE >= 3 ? S : 1], k2v[LAT && STAGE >= 2 ? S : 1];
    if constexpr (LAT) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int ky = t + T * s;
            const unsigned o = boff(rowo + ky, !kmasked(kxs, ksg(ky, N), N));
            k0v[s] = bld(r0, o);
            if constexpr (STAGE >= 2) k2v[s] = bld(r2, o);
            if constexpr (STAGE >= 3) k1v[s] = bld(r1, o);
        }
    }
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int ky = t + T * s;
        const int kys = ksg(ky, N);
        const bool keep = !kmasked(kxs, kys, N);
        const unsigned o = boff(rowo + ky, keep);
        const double kr2 = (double)(kxs * kxs + kys * kys);
        const cplx s1 = LAT ? k0v[LAT ? s : 0] : bld(r0, o);
        const cplx ps = STAGE == 1 ? s1 : LAT ? k2v[LAT ? s : 0] : bld(r2, o);
        const cplx lin = rmul(a.alpha * kr2 - a.omega, ps);
        const cplx rhs = cmul(a.pref, cadd(lin, v[s]));
        const cplx inc = rmul(a.wacc, rhs);
        cplx acc = inc, kn;
        if constexpr (STAGE == 2) acc = cadd(rmul(a.r1, csub(ps, s1)), inc);
        else if constexpr (STAGE == 3) acc = cadd(LAT ? k1v[LAT ? s : 0] : bld(r1, o), inc);
        else if constexpr (STAGE == 4) acc = cadd(cadd(LAT ? k1v[LAT ? s : 0] : bld(r1, o), rmul(a.r3, csub(ps, s1))), inc);
        if constexpr (STAGE < 4) {
            if constexpr (STAGE == 2) bst(r1, o, acc);
            kn = cadd(s1, rmul(a.cstep, rhs));
            bst(r2, o, kn);
        } else {
            kn = cadd(s1, acc);
            bst(r0, o, kn);
        }
        v[s] = conjc(keep ? kn : czero());
    }
    fft_fwd<N, S, C::SPLIT, true>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) Hpsi[hoff<C>(p, t + T * s, c)] = conjc(v[s]);
}

template <class C, int STAGE, int G = C::TC>
__global__ void __launch_bounds__(G * C::T) VK_P4OCC(C) k_p4(const cplx* __restrict__ HN, cplx* __restrict__ Hpsi,
                                                cplx* __restrict__ K0, cplx* __restrict__ K1,
                                                cplx* __restrict__ K2, const cplx* __restrict__ tw,
                                                Geo g, RKArgs a)
{
    p4_body<C, STAGE, G>(blockIdx.x, gridDim.x, HN, Hpsi, K0, K1, K2, tw, g, a);
}

struct ArgleArgs {
    double alpha, omega, dt;
    int want_res;
    // SGLE (src/gpe.f90:200-217): sqrt(dt) times the transform of Hn (dealiased) is
    // added to the numerator, omega is this step's chemical potential and,
    // for ktrunc2 > 0, modes with k^2 > ktrunc2 are zeroed
    const cplx* Hn;        // noise rows transformed along x, retained panels
    const double* nsum;    // P1's row sums of |psi|^2
    double* om;            // [0] before this step, [1] of this step
    double sdt, ktrunc2, dvol, nuN, L2;
    Geo g;
};

// finiteT_adhoc_chempot (src/gpe.f90:226-266): norm = sum_x |psi|^2 dvol,
// omega - dt (nuN/L^2)(norm - L^2).  Every workgroup sums the rows in the same
// order (N doubles from L2) instead of waiting for a launch of its own.
template <int N, int BD> __device__ __forceinline__ double chempot_step(const ArgleArgs& a, double* lds)
{
    static_assert(N % BD == 0, "whole rounds of the workgroup");
    double q[N / BD], x[1] = {0.0};
    const double om = a.om[0];
#pragma unroll
    for (int i = 0; i < N / BD; ++i) q[i] = a.nsum[threadIdx.x + i * BD];
#pragma unroll
    for (int i = 0; i < N / BD; ++i) x[0] += q[i];
    block_sum<1>(x, lds);
    if (threadIdx.x == 0) lds[0] = om - a.dt * (a.nuN / a.L2) * (x[0] * a.dvol - a.L2);
    __syncthreads();
    const double o = lds[0];
    __syncthreads();
    return o;
}

// ARGLE A4 (column, all panels): forward along y -> N-hat; implicit update
// kpsi = (kpsi + dt*(N-hat + omega*kpsi))/(1 + alpha*k^2*dt) on every mode
// (src/gpe.f90:195-197, no dealiasing of the result); residual partial
// sums; inverse along y of the new kpsi -> Hpsi.  SG: SGLE; the noise column
// is transformed here too.  G < TC: G of a panel's
// columns per workgroup (the host keeps NP a multiple of 8 then, so that
// every workgroup writes its residual partials).
template <class C, int G = C::TC, bool SG = false>
__device__ __forceinline__ void a4_body(int blk_, int nblk_, const cplx* __restrict__ HN, cplx* __restrict__ Hpsi,
                                                cplx* __restrict__ K0, const cplx* __restrict__ tw,
                                                ArgleArgs a, double* __restrict__ part)
{
    VK_COL_SETUP_G(C, G, blk_, pb_, C::NP)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = HN[hoff<C>(p, t + T * s, c)];
    const int kxs = ksg(kx, N);
    const size_t rowo = (size_t)kx * N;
    constexpr bool LAT = is_lat<C>::value;
    cplx k0v[LAT ? S : 1];
    if constexpr (LAT) {
#pragma unroll
        for (int s = 0; s < S; ++s) k0v[s] = K0[rowo + t + T * s];
    }
    cplx nz[SG ? S : 1];
    double omega = a.omega;
    if constexpr (SG) {
        const bool on = panel_stored(p, NP, a.g, 1);   // every mode of the others is masked
#pragma unroll
        for (int s = 0; s < S; ++s) nz[s] = on ? a.Hn[hoff<C>(p, t + T * s, c)] : czero();
        omega = chempot_step<N, G * T>(a, lds);
        if (blk_ == 0 && threadIdx.x == 0) a.om[1] = omega;
        if (on) fft_fwd<N, S, C::SPLIT>(nz, lg, t, w_);
    }
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
    double r[2] = {0.0, 0.0};
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int ky = t + T * s;
        const int kys = ksg(ky, N);
        const size_t o = rowo + ky;
        const cplx old = LAT ? k0v[LAT ? s : 0] : K0[o];
        const double kr2 = (double)(kxs * kxs + kys * kys);
        const cplx t1 = cadd(v[s], rmul(omega, old));
        const double t2 = 1.0 + a.alpha * kr2 * a.dt;
        cplx num = cadd(old, rmul(a.dt, t1));
        if constexpr (SG) num = cadd(num, kmasked(kxs, kys, N) ? czero() : rmul(a.sdt, nz[s]));
        cplx nw = mk(num.x / t2, num.y / t2);
        if constexpr (SG) {
            if (a.ktrunc2 > 0.0 && kr2 > a.ktrunc2) nw = czero();
        }
        K0[o] = nw;
        if (a.want_res) {
            const double dx = nw.x - old.x, dy = nw.y - old.y;
            r[0] += dx * dx + dy * dy;
            r[1] += old.x * old.x + old.y * old.y;
        }
        v[s] = conjc(nw);
    }
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) Hpsi[hoff<C>(p, t + T * s, c)] = conjc(v[s]);
    if (a.want_res) {
        block_sum<2>(r, lds);
        if (threadIdx.x == 0) {
            part[2 * blk_] = r[0];
            part[2 * blk_ + 1] = r[1];
        }
    }
}

template <class C, int G = C::TC, bool SG = false>
__global__ void __launch_bounds__(G * C::T) VK_OCC k_a4(const cplx* __restrict__ HN, cplx* __restrict__ Hpsi,
                                                cplx* __restrict__ K0, const cplx* __restrict__ tw,
                                                ArgleArgs a, double* __restrict__ part)
{
    a4_body<C, G, SG>(blockIdx.x, gridDim.x, HN, Hpsi, K0, tw, a, part);
}

// fixed-order reduction of nb partial records of nv doubles -> out[nv]
__device__ __forceinline__ void reduce_fixed_body(const double* __restrict__ part, int nb, int nv,
                                                  double* __restrict__ out)
{
    __shared__ double sh[1024];
    for (int i = 0; i < nv; ++i) {
        double x = 0.0;
        for (int b = threadIdx.x; b < nb; b += blockDim.x) x += part[(size_t)b * nv + i];
        double xx[1] = {x};
        block_sum<1>(xx, sh);
        if (threadIdx.x == 0) out[i] = xx[0];
        __syncthreads();
    }
}

__global__ void k_reduce_fixed(const double* __restrict__ part, int nb, int nv, double* __restrict__ out)
{
    reduce_fixed_body(part, nb, nv, out);
}

// ----------------------------------------------------------------------------
// Diagnostics (src/diagnostics.f90:54-426)
// ----------------------------------------------------------------------------

struct DiagArgs {
    double alpha, omega, g, smlnum;
    int N;
    int has_v;
};

// Row pass of the diagnostics (src/diagnostics.f90:54-317): from the rows of
// Hpsi, Hdy = IFFT_y(i ky kpsi), Hrhod (and HV) the x-space psi, d_x psi,
// d_y psi, P_G rho (and V), never stored; per row the sums
//   0 momx 1 momy 2 egrad 3 echem 4 eintr 5 eppot 6 norm   (rsum[y][8])
// and the transforms along x of two pairs of real fields, packed as complex
// ones, on the retained panels: H1: w_x + i q_x, H2: w_y + i q_y with
//   w = 2 alpha Im(psi* grad psi)/(|psi| + smlnum),
//   q = Re(psi* grad psi)/(|psi| + smlnum)
// (this pairing lets each direction's pair go before the next one's gradient
// is formed; w_x with w_y would hold 64 registers more and spill 240).
// Six transforms per row.  4096^2: 0.8 GB against the 5.4 GB of separate
// transforms and a pointwise pass over x-space arrays (1.5 ms).  0.42 ms, bound
// by the transforms (0.05 ms each at full occupancy): with the directions
// unrolled and index arithmetic shared by the transforms 96 registers spilled,
// 0.56 ms.
template <class C>
__device__ __forceinline__ void diag_row_body(int blk_, int nblk_, const cplx* __restrict__ Hpsi,
                                              const cplx* __restrict__ Hdy, const cplx* __restrict__ Hrhod,
                                              const cplx* __restrict__ HV, cplx* __restrict__ H1,
                                              cplx* __restrict__ H2, const cplx* __restrict__ tw, Geo g, int pl,
                                              double scale, const DiagArgs& a, double* __restrict__ rsum)
{
    VK_ROW_SETUP(C)
    const auto w_ = twiddles<C>(tw, t);
    cplx v[S], ps[S];
    const brsrc rH = mkbuf(Hpsi, N), rD = mkbuf(Hdy, N), rR = mkbuf(Hrhod, N);
    // Offsets are formed anew for each load and store phase (from an opaque
    // copy of the panel index), not kept across the transforms.
    auto again = [&](int q) {
        if constexpr (!is_lat<C>::value) asm volatile("" : "+v"(q));
        return q;
    };
    double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    // a row of a field stored on the panels of mode pl, conjugated for the
    // inverse; dx: times i kx
    auto load = [&](brsrc rb, bool dx) {
        const int p0 = again(pidx0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int pp = p0 + (T / TC) * s;
            v[s] = bld(rb, boff(hoff<C>(pp, y, c), panel_stored(pp, NP, g, pl)));
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            cplx z = v[s];
            if (dx) {
                const double kk = (double)ksg(t + T * s, N);
                z = mk(-kk * z.y, kk * z.x);
            }
            v[s] = conjc(z);
        }
    };
    load(rH, false);
    fft_fwd<N, S, C::SPLIT>(v, lg, again(t), w_);
#pragma unroll
    for (int s = 0; s < S; ++s) ps[s] = rmul(scale, conjc(v[s]));
    // P_G rho + i V from the kx >= 0 halves
    const int Kp = TC * g.Pp, t0 = again(t);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int kxi = t0 + T * s;
        const int km = kxi >= Kp ? N - kxi : kxi;
        const unsigned o = boff(hoff<C>(km / TC, y, km % TC), kxi < Kp || kxi > N - Kp);
        cplx z = bld(rR, o);
        cplx zv = a.has_v ? bld(mkbuf(HV, N), o) : czero();
        if (kxi > N - Kp) {
            z = conjc(z);
            zv = conjc(zv);
        }
        v[s] = conjc(mk(z.x - zv.y, z.y + zv.x));
    }
    fft_fwd<N, S, C::SPLIT>(v, lg, again(t), w_);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const double pr = scale * v[s].x, ap2 = ps[s].x * ps[s].x + ps[s].y * ps[s].y;
        acc[3] += a.omega * ap2;
        acc[4] += 0.5 * a.g * fabs(pr) * ap2;
        if (a.has_v) acc[5] += (-scale * v[s].y) * pr;
        acc[6] += ap2;
    }
    auto direction = [&](int dir) {
        load(dir == 0 ? rH : rD, dir == 0);
        fft_fwd<N, S, C::SPLIT>(v, lg, again(t), w_);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const cplx d = rmul(scale, conjc(v[s]));
            const cplx z = cmul(conjc(ps[s]), d);
            acc[dir] += z.y;
            acc[2] += a.alpha * (d.x * d.x + d.y * d.y);
            double px = ps[s].x;
            if constexpr (!is_lat<C>::value) asm volatile("" : "+v"(px));   // formed twice, not kept
            const double inv = 1.0 / (sqrt(px * px + ps[s].y * ps[s].y) + a.smlnum);
            v[s] = mk(2.0 * a.alpha * (z.y * inv), z.x * inv);
            // one point's square root and division at a time
            if constexpr (!is_lat<C>::value) __builtin_amdgcn_sched_barrier(0);
        }
        fft_fwd<N, S, C::SPLIT>(v, lg, again(t), w_);
        const brsrc ro = mkbuf(dir == 0 ? H1 : H2, N);
        const int p0 = again(pidx0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int pp = p0 + (T / TC) * s;
            bst(ro, boff(hoff<C>(pp, y, c), panel_stored(pp, NP, g, 1)), v[s]);
        }
    };
    if constexpr (is_lat<C>::value) {
        direction(0);
        direction(1);
    } else {
#pragma unroll 1
        for (int dir = 0; dir < 2; ++dir) direction(dir);   // rolled, nothing spills
    }
    row_sum<7, T>(acc, lg, t, rsum + 8 * (size_t)y);
}

struct SpecArgs {
    double alpha, g, enorm;
    int N, nshell;
};

// shells that hold retained modes: 0 .. spec_shells - 1, nint(|k|) of the
// dealias radius N/3
__host__ __device__ constexpr int spec_shells(int N) { return (N + 1) / 3 + 1; }

// largest ky >= 0 of column kx in a shell <= m: kx^2 + ky^2 <= m (m + 1)
// (src/diagnostics.f90:341-343 by the integer identity m(m-1) < k^2 <=
// m(m+1)); -1 if there is none
__device__ __forceinline__ int shell_end(int m, int kx)
{
    const int r = m * (m + 1) - kx * kx;
    return r < 0 ? -1 : (int)sqrt((double)r);
}

// Column pass of the spectra (src/diagnostics.f90:320-402): the columns kx
// and -kx of H1 and H2 (kx >= 0 panels), transformed along y and separated
// into the transforms of the real fields by their symmetry, with rho-hat and
// kpsi give the terms of every mode of the two columns; a mode and its mirror
// share the first five.  The shells of a column are runs of ky, so each
// shell's sum is one thread's, in order of |ky|; part[kx][6][spec_shells],
// entries m >= kx, summed over the columns by spec_reduce_body.
// 4096^2: 0.6 GB in order, 0.28 ms, against a gather of 16-byte values by shell
// lists (0.42 ms) after eight transforms.
template <class C, int G = C::TC>
__device__ __forceinline__ void diag_col_body(int b, cplx* __restrict__ H1, const cplx* __restrict__ H2,
                                              const cplx* __restrict__ K0, const cplx* __restrict__ Krho,
                                              const cplx* __restrict__ tw, Geo g, double* __restrict__ part)
{
    VK_COL_SETUP_G(C, G, b, pb_, g.Pp)
    const auto w_ = twiddles<C>(tw, t);
    const bool live = kx <= g.M;
    const int km = (N - kx) & (N - 1);
    constexpr int MS = spec_shells(N);
    const double mult = kx > 0 ? 2.0 : 1.0;
    double* pk = part + (size_t)kx * 6 * MS;
    // val of every ky of this column into its shells of spectrum q
    auto bin = [&](const double (&val)[S], int q) {
        lds_barrier();
#pragma unroll
        for (int s = 0; s < S; ++s) lg[t + T * s] = val[s];
        lds_barrier();
        if (live)
            for (int m = kx + t; m < MS; m += T) {
                const int hi = shell_end(m, kx);
                double x = 0.0;
                for (int k = m > 0 ? shell_end(m - 1, kx) + 1 : 0; k <= hi; ++k) x += k > 0 ? lg[k] + lg[N - k] : lg[0];
                pk[q * MS + m] = x;
            }
    };
    auto again = [&](int q) {   // index arithmetic formed anew per transform
        if constexpr (!is_lat<C>::value) asm volatile("" : "+v"(q));
        return q;
    };
    cplx v[S], um[S];
    // the transforms of the two real fields packed in H: v, um
    auto pair = [&](const cplx* H) {
        const brsrc rb = mkbuf(H, N);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            v[s] = bld(rb, boff(hoff<C>(p, t + T * s, c), live));
            um[s] = bld(rb, boff(hoff<C>(km / TC, t + T * s, km % TC), live));
        }
        fft_fwd<N, S, C::SPLIT>(v, lg, again(t), w_);
        lds_barrier();
        fft_fwd<N, S, C::SPLIT>(um, lg, again(t), w_);
        lds_barrier();
        // um at -ky
#pragma unroll
        for (int s = 0; s < S; ++s) lg[t + T * s] = um[s].x;
        lds_barrier();
#pragma unroll
        for (int s = 0; s < S; ++s) um[s].x = lg[(N - t - T * s) & (N - 1)];
        lds_barrier();
#pragma unroll
        for (int s = 0; s < S; ++s) lg[t + T * s] = um[s].y;
        lds_barrier();
#pragma unroll
        for (int s = 0; s < S; ++s) {
            um[s].y = -lg[(N - t - T * s) & (N - 1)];
            const cplx z = v[s], m = um[s];
            v[s] = mk(0.5 * (z.x + m.x), 0.5 * (z.y + m.y));
            um[s] = mk(0.5 * (z.y - m.y), -0.5 * (z.x - m.x));
        }
    };
    auto sq = [](cplx z) { return z.x * z.x + z.y * z.y; };
    double e[3][S];
    // w_x, q_x: w_x waits in its column of H1, this workgroup's alone
    const brsrc r1 = mkbuf(H1, N);
#pragma unroll
    for (int s = 0; s < S; ++s) e[2][s] = 0.0;
    auto direction = [&](int dir) {
        pair(dir == 0 ? H1 : H2);
#pragma unroll
        for (int s = 0; s < S; ++s) e[2][s] += mult * sq(um[s]);
        if (dir == 0) {
#pragma unroll
            for (int s = 0; s < S; ++s) bst(r1, boff(hoff<C>(p, t + T * s, c), live), v[s]);
            lds_barrier();
        }
    };
    if constexpr (is_lat<C>::value) {
        direction(0);
        direction(1);
    } else {
#pragma unroll 1
        for (int dir = 0; dir < 2; ++dir) direction(dir);
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const bool use = live && !kmasked(kx, ksg(t + T * s, N), N);
        if (!use) e[2][s] = 0.0;
        um[s] = bld(r1, boff(hoff<C>(p, t + T * s, c), live));
    }
    bin(e[2], 3);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int ky = ksg(t + T * s, N);
        const bool use = live && !kmasked(kx, ky, N);
        const double kxd = kx, kyd = ky, kr2 = kxd * kxd + kyd * kyd;
        const double ik2 = kr2 > 0.0 ? 1.0 / kr2 : 0.0;
        // compressible part k (k.w)/k^2, and the rest
        const cplx wx = um[s], wy = v[s];
        const cplx dv = rmul(ik2, mk(kxd * wx.x + kyd * wy.x, kxd * wx.y + kyd * wy.y));
        const cplx c1 = rmul(kxd, dv), c2 = rmul(kyd, dv);
        e[0][s] = use ? mult * (sq(wx) + sq(wy)) : 0.0;
        e[1][s] = use ? mult * (sq(csub(wx, c1)) + sq(csub(wy, c2))) : 0.0;
        e[2][s] = use ? mult * (sq(c1) + sq(c2)) : 0.0;
    }
    bin(e[0], 0);
    bin(e[1], 1);
    bin(e[2], 2);
    const brsrc rk = mkbuf(K0, N), rr = mkbuf(Krho, N);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int k = t + T * s;
        const bool use = live && !kmasked(kx, ksg(k, N), N);
        e[1][s] = mult * sq(bld(rr, boff((size_t)kx * N + k, use)));
        e[2][s] = sq(bld(rk, boff((size_t)kx * N + k, use))) +
                  sq(bld(rk, boff((size_t)km * N + ((N - k) & (N - 1)), use && kx > 0)));
    }
    bin(e[1], 4);
    bin(e[2], 5);
}

// The column partials of diag_col_body and the row sums of diag_row_body to
// the results: block (bx, q < 6): 64 shells of spectrum q over the columns,
// out[8 + q (nshell + 1) + m]; block (0, 6): the 8 sums over the rows, out[0..7].
// Fixed order: 16 interleaved partial sums, added in turn.
constexpr int SPEC_G = 16;
__device__ __forceinline__ void spec_reduce_body(const double* __restrict__ part, const double* __restrict__ rsum,
                                                 const SpecArgs& a, double* __restrict__ out)
{
    __shared__ double sh[SPEC_G][64];
    const int l = threadIdx.x % 64, w = threadIdx.x / 64, q = blockIdx.y;
    const int MS = spec_shells(a.N), M = a.N / 3;
    double x = 0.0;
    if (q == 6) {
        if (blockIdx.x > 0) return;
        // lane l: value l % 8 of the rows l / 8 + 8 w + 128 i
        if (l % 8 < 7)
            for (int y = l / 8 + 8 * w; y < a.N; y += 8 * SPEC_G) x += rsum[8 * (size_t)y + l % 8];
        sh[w][l] = x;
        __syncthreads();
        if (threadIdx.x < 8) {
            double s = 0.0;
            for (int k = 0; k < SPEC_G; ++k)
                for (int j = 0; j < 8; ++j) s += sh[k][8 * j + threadIdx.x];
            out[threadIdx.x] = threadIdx.x < 7 ? s : 0.0;
        }
        return;
    }
    const int m = blockIdx.x * 64 + l;
    if (m < MS) {
        const int last = m < M ? m : M;
#pragma unroll 4
        for (int kx = w; kx <= last; kx += SPEC_G) x += part[((size_t)kx * 6 + q) * MS + m];
    }
    sh[w][l] = x;
    __syncthreads();
    if (w == 0 && m <= a.nshell) {
        double s = sh[0][l];
#pragma unroll
        for (int k = 1; k < SPEC_G; ++k) s += sh[k][l];
        // factors of spec_gp (:394-399)
        const double f = q < 3 ? 0.5 : q == 3 ? 2.0 * (a.alpha * a.alpha) : q == 4 ? 0.5 * a.g * 2.0 * a.alpha : 1.0;
        out[8 + q * (a.nshell + 1) + m] = a.enorm * s * f;
    }
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) k_p1d(const cplx* __restrict__ Hpsi, cplx* __restrict__ Hrho,
                                                 const cplx* __restrict__ tw, Geo g, int psi_pmode, double scale)
{
    p1_body<C, false>(blockIdx.x, gridDim.x, Hpsi, Hrho, tw, g, psi_pmode, scale, nullptr);
}

// waves per SIMD: two (<= 256 VGPRs) with 16 points per thread, with 8 what
// whole workgroups fill (T/256 waves per SIMD each); the LAT shapes one
#define VK_DIAGOCC(C) \
    __attribute__((amdgpu_waves_per_eu(is_lat<C>::value ? 1 : C::S == 16 ? 2 : C::T == 512 ? 4 : 3)))

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_DIAGOCC(C)
k_diag_row(const cplx* __restrict__ Hpsi, const cplx* __restrict__ Hdy, const cplx* __restrict__ Hrhod,
           const cplx* __restrict__ HV, cplx* __restrict__ H1, cplx* __restrict__ H2, const cplx* __restrict__ tw,
           Geo g, int pl, double scale, DiagArgs a, double* __restrict__ rsum)
{
    diag_row_body<C>(blockIdx.x, gridDim.x, Hpsi, Hdy, Hrhod, HV, H1, H2, tw, g, pl, scale, a, rsum);
}

template <class C, int G>
__global__ void __launch_bounds__(G * C::T) VK_DIAGOCC(C)
k_diag_col(cplx* __restrict__ H1, const cplx* __restrict__ H2, const cplx* __restrict__ K0,
           const cplx* __restrict__ Krho, const cplx* __restrict__ tw, Geo g, double* __restrict__ part)
{
    diag_col_body<C, G>(blockIdx.x, H1, H2, K0, Krho, tw, g, part);
}

__global__ void __launch_bounds__(64 * SPEC_G) k_spec_reduce(const double* __restrict__ part,
                                                             const double* __restrict__ rsum, SpecArgs a,
                                                             double* __restrict__ out)
{
    spec_reduce_body(part, rsum, a, out);
}

// ----------------------------------------------------------------------------
// Batched forms for many fields of one size (the ensemble's diagnostics):
// blockIdx.y selects the field's pointers, blockIdx.x is the block within
// the field, as in the single-field launch
// ----------------------------------------------------------------------------

struct BPair {
    const cplx* src;
    cplx* dst;
};

template <class C>
__global__ void __launch_bounds__(C::COLT) VK_OCC k_col_inv_b(const BPair* __restrict__ P, const cplx* __restrict__ tw,
                                                       Geo g, int pmode, int op)
{
    const BPair q = P[blockIdx.y];
    col_inv_body<C>(blockIdx.x, q.src, q.dst, tw, g, pmode, op);
}

// one field's diagnostics operands
struct DiagB {
    const cplx *Hpsi, *K0;
    cplx *Hd, *Hrho, *Krho, *H1, *H2;
    double *rsum, *part, *out;
    DiagArgs da;
    SpecArgs sa;
};

template <class C>
__global__ void __launch_bounds__(C::COLT) VK_OCC k_diag_dy_b(const DiagB* __restrict__ D, const cplx* __restrict__ tw,
                                                              Geo g, int pl)
{
    const DiagB& d = D[blockIdx.y];
    col_inv_body<C>(blockIdx.x, d.K0, d.Hd, tw, g, pl, 2);
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_OCC k_p1d_b(const DiagB* __restrict__ D, const cplx* __restrict__ tw,
                                                          Geo g, int pl, double scale)
{
    const DiagB& d = D[blockIdx.y];
    p1_body<C, false>(blockIdx.x, gridDim.x, d.Hpsi, d.Hrho, tw, g, pl, scale, nullptr);
}

template <class C>
__global__ void __launch_bounds__(C::COLT) VK_OCC k_p2d_b(const DiagB* __restrict__ D, const cplx* __restrict__ tw,
                                                          Geo g)
{
    const DiagB& d = D[blockIdx.y];
    p2_body<C, C::TC, 2>(blockIdx.x, gridDim.x, d.Hrho, nullptr, nullptr, d.Krho, tw, g, 2);
}

template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_DIAGOCC(C)
k_diag_row_b(const DiagB* __restrict__ D, const cplx* __restrict__ tw, Geo g, int pl, double scale)
{
    const DiagB& d = D[blockIdx.y];
    diag_row_body<C>(blockIdx.x, gridDim.x, d.Hpsi, d.Hd, d.Hrho, nullptr, d.H1, d.H2, tw, g, pl, scale, d.da, d.rsum);
}

template <class C, int G>
__global__ void __launch_bounds__(G * C::T) VK_DIAGOCC(C)
k_diag_col_b(const DiagB* __restrict__ D, const cplx* __restrict__ tw, Geo g)
{
    const DiagB& d = D[blockIdx.y];
    diag_col_body<C, G>(blockIdx.x, d.H1, d.H2, d.K0, d.Krho, tw, g, d.part);
}

__global__ void __launch_bounds__(64 * SPEC_G) k_spec_reduce_b(const DiagB* __restrict__ D)
{
    const DiagB& d = D[blockIdx.z];
    spec_reduce_body(d.part, d.rsum, d.sa, d.out);
}

// ----------------------------------------------------------------------------
// Particles (src/gpe_particle.f90)
// ----------------------------------------------------------------------------

// V(x,y) = V0 exp(-r^2/(2 d^2)), r from the periodic coordinate
// (1/c)(s + s^3/6 + s^5/40), s = sin(c x), c = pi/L  (:34-56)
__global__ void k_pot_x(cplx* __restrict__ X, int N, double dx, double c1, double V0, double d)
{
    const size_t n2 = (size_t)N * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x) {
        const int ix = (int)(i % N), iy = (int)(i / N);
        const double x = ix * dx, y = iy * dx;
        const double sx = sin(c1 * x), sy = sin(c1 * y);
        const double sx2 = sx * sx, sy2 = sy * sy;
        const double xp = (1.0 / c1) * (sx + (1.0 / 6.0) * (sx2 * sx) + (1.0 / 40.0) * (sx2 * sx2 * sx));
        const double yp = (1.0 / c1) * (sy + (1.0 / 6.0) * (sy2 * sy) + (1.0 / 40.0) * (sy2 * sy2 * sy));
        const double rp = sqrt(xp * xp + yp * yp);
        X[i] = mk(V0 * exp(-(rp * rp) / (2.0 * (d * d))), 0.0);
    }
}

struct WTab {
    double V0, d, W;     // potential height, width, window radius
    int4* win;
    double2 *tx, *ty;
};

// Windows and factor tables of the real-space particle potential (P3Part):
// particle p covers the columns x with |x dx - qx| <= W (minimum image, all N
// when the window spans the period), from column win.x on; V(x, y) =
// tx.x ty.x, dV/dx = tx.y ty.x, dV/dy = tx.x ty.y.  Positions that are not
// finite get empty windows.  One direction of one particle at coordinate q,
// by nt threads.
__device__ __forceinline__ void window_table(const WTab& w, int p, int dir, double q, int N, int tid, int nt)
{
    const double dx = 6.283185307179586476925 / N;
    const double c = q / dx, r = w.W / dx;
    int n = 0, first = 0;
    if (fabs(c) < 1e15) {
        const double lo = ceil(c - r), hi = floor(c + r);
        n = (int)fmin(fmax(hi - lo + 1.0, 0.0), (double)N);
        first = (int)(lo - N * floor(lo / N)) & (N - 1);
    }
    if (tid == 0) {
        int* o = reinterpret_cast<int*>(w.win + p) + 2 * dir;
        o[0] = first;
        o[1] = n;
    }
    const double inv2d2 = 1.0 / (2.0 * (w.d * w.d)), invd2 = 1.0 / (w.d * w.d), a = dir ? w.V0 : 1.0;
    double2* tab = (dir ? w.ty : w.tx) + (size_t)p * N;
    for (int k = tid; k < n; k += nt) {
        double X, dX;
        pcoord(pwrap(((first + k) & (N - 1)) * dx - q), X, dX);
        const double e = a * exp(-(X * X) * inv2d2);
        tab[k] = make_double2(e, -e * X * dX * invd2);
    }
}

__global__ void k_wtab(const double* __restrict__ pos, int N, WTab w)
{
    window_table(w, blockIdx.x, blockIdx.y, pos[2 * blockIdx.x + blockIdx.y], N, threadIdx.x, blockDim.x);
}

// V on the grid from the tables (particles in increasing order)
__global__ void k_potfield(const int4* __restrict__ win, const double2* __restrict__ tx, const double2* __restrict__ ty,
                           int np, int N, double* __restrict__ V)
{
    const size_t n2 = (size_t)N * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i & (N - 1)), y = (int)(i / N);
        double v = 0.0;
        for (int p = 0; p < np; ++p) {
            const int4 w = win[p];
            const int kx = (x - w.x) & (N - 1), ky = (y - w.z) & (N - 1);
            if (kx < w.y && ky < w.w) v += tx[(size_t)p * N + kx].x * ty[(size_t)p * N + ky].x;
        }
        V[i] = v;
    }
}

// EX[p*N + i] = exp(-i kx(i) qx_p), EY[p*N + i] = exp(-i ky(i) qy_p)
__global__ void k_ptab(const double* __restrict__ pos, cplx* __restrict__ EX, cplx* __restrict__ EY,
                       int np, int N)
{
    const int n = np * N;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int pp = i / N, k = i % N;
        const double kk = (double)ksg(k, N);
        double sx, cx, sy, cy;
        sincos(kk * pos[2 * pp], &sx, &cx);
        sincos(kk * pos[2 * pp + 1], &sy, &cy);
        EX[i] = mk(cx, -sx);
        EY[i] = mk(cy, -sy);
    }
}

// KV(kx,ky) = Vhat(kx,ky) * sum_p EX_p(kx) EY_p(ky) on the unmasked modes of
// rows kx in [0, nrows) (nrows = N: all rows)   (:334-349, separable)
__global__ void k_kv(const cplx* __restrict__ Vhat, const cplx* __restrict__ EX, const cplx* __restrict__ EY,
                     cplx* __restrict__ KV, int np, int N)
{
    extern __shared__ double dsh[];
    cplx* ex = reinterpret_cast<cplx*>(dsh);
    const int kx = blockIdx.x;
    for (int pp = threadIdx.x; pp < np; pp += blockDim.x) ex[pp] = EX[(size_t)pp * N + kx];
    __syncthreads();
    const int kxs = ksg(kx, N);
    for (int ky = threadIdx.x; ky < N; ky += blockDim.x) {
        const int kys = ksg(ky, N);
        if (kmasked(kxs, kys, N)) continue;
        cplx sacc = czero();
        for (int pp = 0; pp < np; ++pp) sacc = cadd(sacc, cmul(ex[pp], EY[(size_t)pp * N + ky]));
        const size_t o = (size_t)kx * N + ky;
        KV[o] = cmul(sacc, Vhat[o]);
    }
}

// Force partial sums for rows kx: for each particle p (PG particles per
// block in blockIdx.y), B_p = sum_ky A conj(EY_p(ky)), By_p = sum_ky ky A
// conj(EY_p(ky)) with A = rhohat_d(k) * conj(Vhat(k)) = rhohat_d(k) Vhat(-k)
// (V real).  out: fpart[((kx*np)+p)*4 + {ReB, ImB, ReBy, ImBy}]
template <int PG>
__global__ void k_force_rows(const cplx* __restrict__ Krho, const cplx* __restrict__ Vhat,
                             const cplx* __restrict__ EY, double* __restrict__ fpart, int np, int N)
{
    __shared__ double sh[4 * PG * 4];
    const int kx = blockIdx.x, p0 = blockIdx.y * PG;
    const int kxs = ksg(kx, N);
    double acc[4 * PG];
#pragma unroll
    for (int i = 0; i < 4 * PG; ++i) acc[i] = 0.0;
    for (int ky = threadIdx.x; ky < N; ky += blockDim.x) {
        const int kys = ksg(ky, N);
        if (kmasked(kxs, kys, N)) continue;
        const size_t o = (size_t)kx * N + ky;
        const cplx A = cmul(Krho[o], conjc(Vhat[o]));
#pragma unroll
        for (int j = 0; j < PG; ++j) {
            const int pp = p0 + j;
            if (pp < np) {
                const cplx z = cmul(A, conjc(EY[(size_t)pp * N + ky]));
                acc[4 * j + 0] += z.x;
                acc[4 * j + 1] += z.y;
                acc[4 * j + 2] += (double)kys * z.x;
                acc[4 * j + 3] += (double)kys * z.y;
            }
        }
    }
    block_sum<4 * PG>(acc, sh);
    if (threadIdx.x == 0)
        for (int j = 0; j < PG; ++j)
            if (p0 + j < np)
                for (int k = 0; k < 4; ++k) fpart[((size_t)kx * np + p0 + j) * 4 + k] = acc[4 * j + k];
}

struct PartArgs {
    int nblk, nw;             // real space: row blocks and waves per block
    int np, N, nrows, half;   // rows kx in [0,nrows); half: weight 2 for kx>0
    double coef;              // 2 alpha dvol / N^2
    double rf;                // short-range factor 384 dE pi^12 r0^12 / L^12
    double dt, mass;
    int stage;                // 1..4 RK4 stage; 0: forces only (diagnostics)
    double efac;              // 64 dE pi^12 r0^12 / L^12 (diagnostic energy)
};

// Particle forces and one RK4 stage of gp_particle_motion_rk4
// (src/gpe_particle.f90:219-324, 378-531), one workgroup of PSTEP_T threads.
// Fluid force F_j = -2 alpha dvol Re sum_x d_j rho V_p
//   = (2 alpha dvol/N^2) Im sum_k k_j rhohat_d(k) Vhat(-k) e^{i k.q_p}.
// The reference advances the particles one at a time, so the short-range
// force on particle ip sees the particles q < ip at their new positions and
// q > ip at their old ones.  A particle's new position depends only on the
// state at the start of the stage (tpos, its velocity, the earlier stages'
// kq), so all new positions are formed first; the forces then run one
// particle per wave, each with the lane order and shuffle tree of the
// one-wave form (lane l sums q = l, l + 64, ...), from positions in LDS.
// st: pos(2np) vel(2np) fext(2np) tpos tvel ku[4](2np) kq[4](2np) frc(2np)
//     then diag[5] = {eobj_kin, esrep, momx, momy, -}
constexpr int PSTEP_T = 512;
__global__ void __launch_bounds__(PSTEP_T) k_pstep(const double* __restrict__ fpart, const cplx* __restrict__ EX,
                                                   double* __restrict__ st, PartArgs a)
{
    __shared__ double fl[2 * 256];
    __shared__ double po[2 * 256];   // positions at the start of the stage
    __shared__ double pn[2 * 256];   // positions after the stage
    __shared__ double ff[2 * 256];   // total force
    const int np = a.np;
    double* pos = st;
    double* vel = st + 2 * np;
    double* fext = st + 4 * np;
    double* tpos = st + 6 * np;
    double* tvel = st + 8 * np;
    double* ku = st + 10 * np;   // [4][2np]
    double* kq = st + 18 * np;   // [4][2np]
    double* frc = st + 26 * np;
    double* dg = st + 28 * np;
    const int tid = threadIdx.x, lane = tid % 64, wv = tid / 64;
    constexpr int NW = PSTEP_T / 64;
    // fluid forces, fixed order over rows
    for (int pp = tid; pp < np; pp += PSTEP_T) {
        double bx = 0.0, by = 0.0;
        for (int kx = 0; kx < a.nrows; ++kx) {
            const double* f = fpart + ((size_t)kx * np + pp) * 4;
            const double w = (a.half && kx > 0) ? 2.0 : 1.0;
            const cplx e = conjc(EX[(size_t)pp * a.N + kx]);   // e^{+i kx qx}
            const double kxd = (double)ksg(kx, a.N);
            const cplx B = cmul(e, mk(f[0], f[1]));
            const cplx By = cmul(e, mk(f[2], f[3]));
            bx += w * kxd * B.y;
            by += w * By.y;
        }
        fl[2 * pp] = a.coef * bx;
        fl[2 * pp + 1] = a.coef * by;
    }
    // start-of-stage positions, and the new positions
    // (stage 1 first saves tpos, tvel)
    for (int i = tid; i < 2 * np; i += PSTEP_T) {
        const double q = pos[i], u = vel[i];
        if (a.stage == 1) { tpos[i] = q; tvel[i] = u; }
        po[i] = q;
        double qn = q;
        if (a.stage > 0) {
            const double kqv = a.dt * u;
            const double tp = a.stage == 1 ? q : tpos[i];
            if (a.stage <= 2) qn = tp + 0.5 * kqv;
            else if (a.stage == 3) qn = tp + kqv;
            else qn = tp + (1.0 / 6.0) * (kq[i] + 2.0 * kq[2 * np + i] + 2.0 * kq[4 * np + i] + kqv);
        }
        pn[i] = qn;
    }
    __syncthreads();
    // short-range forces, one particle per wave
    for (int ip = wv; ip < np; ip += NW) {
        double sx = 0.0, sy = 0.0;
        const double px = po[2 * ip], py = po[2 * ip + 1];
        for (int qq = lane; qq < np; qq += 64) {
            if (qq == ip) continue;
            const double* P = (a.stage > 0 && qq < ip) ? pn : po;
            const double x = px - P[2 * qq], y = py - P[2 * qq + 1];
            const double b = -3.0 + cos(x) + cos(y);
            const double b2 = b * b, b4 = b2 * b2;
            const double den = b4 * b2 * b;
            sx += -a.rf * sin(x) / den;
            sy += -a.rf * sin(y) / den;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            sx += __shfl_xor(sx, o, 64);
            sy += __shfl_xor(sy, o, 64);
        }
        if (np == 1) { sx = 0.0; sy = 0.0; }
        if (lane == 0) {
            ff[2 * ip] = fl[2 * ip] + sx + fext[2 * ip];
            ff[2 * ip + 1] = fl[2 * ip + 1] + sy + fext[2 * ip + 1];
        }
    }
    __syncthreads();
    // stage update of every particle
    for (int i = tid; i < 2 * np; i += PSTEP_T) {
        const double F = ff[i];
        frc[i] = F;
        if (a.stage > 0) {
            const int sidx = a.stage - 1;
            const double kuv = a.dt * F / a.mass;
            const double u = vel[i];
            ku[sidx * 2 * np + i] = kuv;
            kq[sidx * 2 * np + i] = a.dt * u;
            const double tv = a.stage == 1 ? u : tvel[i];
            if (a.stage <= 2) vel[i] = tv + 0.5 * kuv;
            else if (a.stage == 3) vel[i] = tv + kuv;
            else vel[i] = tv + (1.0 / 6.0) * (ku[i] + 2.0 * ku[2 * np + i] + 2.0 * ku[4 * np + i] + kuv);
            pos[i] = pn[i];
        }
    }
    if (a.stage == 0 && wv == 0) {
        // particle energies and momentum (src/diagnostics.f90:210-239)
        double ek = 0.0, es = 0.0, mx = 0.0, my = 0.0;
        for (int i1 = lane; i1 < np; i1 += 64) {
            ek += vel[2 * i1] * vel[2 * i1] + vel[2 * i1 + 1] * vel[2 * i1 + 1];
            mx += a.mass * vel[2 * i1];
            my += a.mass * vel[2 * i1 + 1];
            for (int i2 = 0; i2 < np; ++i2) {
                if (i1 == i2) continue;
                const double x = po[2 * i1] - po[2 * i2], y = po[2 * i1 + 1] - po[2 * i2 + 1];
                const double b = -3.0 + cos(x) + cos(y);
                const double b2 = b * b;
                es += a.efac / (b2 * b2 * b2);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            ek += __shfl_xor(ek, o, 64);
            es += __shfl_xor(es, o, 64);
            mx += __shfl_xor(mx, o, 64);
            my += __shfl_xor(my, o, 64);
        }
        if (lane == 0) {
            dg[0] = 0.5 * a.mass * ek;
            dg[1] = np == 1 ? 0.0 : 0.5 * es;
            dg[2] = mx;
            dg[3] = my;
        }
    }
}

// One RK4 stage of the particles on the real-space path, one workgroup per
// particle: its fluid force (coef times the sum over the row blocks whose
// window flag is set, in a fixed order, of the wave partials of P3), its
// short-range force, its update, and the window tables of its new position.
// Another particle's new position depends only on the state at the start of
// the stage (see k_pstep), so every workgroup forms the ones it needs itself:
// the stage reads positions and velocities from `cur` and writes them to
// `nxt` (pos(2np) vel(2np) each; four stages end where they began).
// Separate force, update and table kernels took 12 us of a 512^2 stage; this
// one 6.
struct PStage {
    const double* ppart;
    const unsigned char* phit;
    const double* cur;
    double *nxt, *st;
    PartArgs a;
    WTab w;
};

template <int NT>
__device__ __forceinline__ void pstage_body(int p, const PStage& q)
{
    static_assert(NT >= 64, "whole waves");
    __shared__ double sh[4 * NT / 64];
    __shared__ double pnew[2];
    const double *ppart = q.ppart, *cur = q.cur;
    const unsigned char* phit = q.phit;
    double *nxt = q.nxt, *st = q.st;
    const PartArgs& a = q.a;
    const WTab& w = q.w;
    const int np = a.np, tid = threadIdx.x;
    const double *pos = cur, *vel = cur + 2 * np;
    double* fext = st + 4 * np;
    double* tpos = st + 6 * np;
    double* tvel = st + 8 * np;
    double* ku = st + 10 * np;   // [4][2np]
    double* kq = st + 18 * np;   // [4][2np]
    double* frc = st + 26 * np;
    auto newpos = [&](int i) {
        const double q = pos[i], kqv = a.dt * vel[i], tp = a.stage == 1 ? q : tpos[i];
        if (a.stage <= 2) return tp + 0.5 * kqv;
        if (a.stage == 3) return tp + kqv;
        return tp + (1.0 / 6.0) * (kq[i] + 2.0 * kq[2 * np + i] + 2.0 * kq[4 * np + i] + kqv);
    };
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (tid < 64) {
        const double px = pos[2 * p], py = pos[2 * p + 1];
        for (int q = tid; q < np; q += 64) {
            if (q == p) continue;
            const double x = px - (q < p ? newpos(2 * q) : pos[2 * q]);
            const double y = py - (q < p ? newpos(2 * q + 1) : pos[2 * q + 1]);
            const double b = -3.0 + cos(x) + cos(y);
            const double b2 = b * b, b4 = b2 * b2;
            const double den = b4 * b2 * b;
            acc[2] += -a.rf * sin(x) / den;
            acc[3] += -a.rf * sin(y) / den;
        }
    }
    for (int b = tid; b < a.nblk; b += NT) {
        if (!phit[(size_t)b * np + p]) continue;
        for (int v = 0; v < a.nw; ++v) {
            acc[0] += ppart[(((size_t)b * a.nw + v) * np + p) * 2];
            acc[1] += ppart[(((size_t)b * a.nw + v) * np + p) * 2 + 1];
        }
    }
    block_sum<4>(acc, sh);
    if (tid == 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int i = 2 * p + c;
            const double F = a.coef * acc[c] + acc[2 + c] + fext[i];
            frc[i] = F;
            const double u = vel[i], kuv = a.dt * F / a.mass;
            const double qn = newpos(i);
            if (a.stage == 1) {
                tpos[i] = pos[i];
                tvel[i] = u;
            }
            const int sidx = a.stage - 1;
            const double tv = a.stage == 1 ? u : tvel[i];
            ku[sidx * 2 * np + i] = kuv;
            kq[sidx * 2 * np + i] = a.dt * u;
            double un;
            if (a.stage <= 2) un = tv + 0.5 * kuv;
            else if (a.stage == 3) un = tv + kuv;
            else un = tv + (1.0 / 6.0) * (ku[i] + 2.0 * ku[2 * np + i] + 2.0 * ku[4 * np + i] + kuv);
            nxt[i] = qn;
            nxt[2 * np + i] = un;
            pnew[c] = qn;
        }
    }
    __syncthreads();
    constexpr int H = NT / 2;
    window_table(w, p, tid / H, pnew[tid / H], a.N, tid % H, H);
}

template <int NT> __global__ void __launch_bounds__(NT) k_pstage(PStage q) { pstage_body<NT>(blockIdx.x, q); }

// P4 with the particles' update, which it does not touch, as the first
// workgroups of its launch (a multiple of eight, so that P4's keep their XCDs).
// us per step with a launch of its own for the update, then so: 128^2 with 8
// particles 119 and 105, 512^2 162 and 141, 1024^2 221 and 195, with 64 268 and
// 239.
template <class C, int STAGE, int G>
__global__ void __launch_bounds__(G * C::T) VK_OCC k_p4_part(const cplx* __restrict__ HN, cplx* __restrict__ Hpsi,
                                                     cplx* __restrict__ K0, cplx* __restrict__ K1,
                                                     cplx* __restrict__ K2, const cplx* __restrict__ tw, Geo g,
                                                     RKArgs a, PStage q)
{
    const int n = (q.a.np + 7) / 8 * 8;
    if ((int)blockIdx.x < n) {
        if ((int)blockIdx.x < q.a.np) pstage_body<G * C::T>(blockIdx.x, q);
        return;
    }
    p4_body<C, STAGE, G>(blockIdx.x - n, gridDim.x - n, HN, Hpsi, K0, K1, K2, tw, g, a);
}

// ----------------------------------------------------------------------------
// SGLE (src/gpe.f90:149-217, 226-266)
// ----------------------------------------------------------------------------

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC 2011): ten rounds of two 32x32->64 multiplications
// and a Weyl-sequence key schedule; counter c, key k.
__host__ __device__ inline void philox4x32_10(unsigned c[4], unsigned k0, unsigned k1)
{
    for (int r = 0; r < 10; ++r) {
        const unsigned long long p0 = 0xD2511F53ull * c[0], p1 = 0xCD9E8D57ull * c[2];
        const unsigned hi0 = (unsigned)(p0 >> 32), lo0 = (unsigned)p0;
        const unsigned hi1 = (unsigned)(p1 >> 32), lo1 = (unsigned)p1;
        const unsigned n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// Two independent standard normals at grid point i for noise draw `step`
// (counter (i, 0, step_lo, step_hi), key = seed): uniforms from 53-bit
// fractions of the 64-bit words, u1 in (0, 1], u2 in [0, 1), then the
// Box-Muller transform.  The reference draws its pair with the polar method
// from Fortran's RANDOM_NUMBER; only the distribution is the same.
__device__ __forceinline__ void sgle_normals(unsigned long long i, unsigned long long step, unsigned long long seed,
                                             double* v1, double* v2)
{
    unsigned c[4] = {(unsigned)i, (unsigned)(i >> 32), (unsigned)step, (unsigned)(step >> 32)};
    philox4x32_10(c, (unsigned)seed, (unsigned)(seed >> 32));
    const unsigned long long a = ((unsigned long long)c[1] << 32) | c[0];
    const unsigned long long b = ((unsigned long long)c[3] << 32) | c[2];
    const double u1 = (double)((a >> 11) + 1) * 0x1.0p-53;
    const double u2 = (double)(b >> 11) * 0x1.0p-53;
    const double rr = sqrt(-2.0 * log(u1));
    double sn, cs;
    sincospi(2.0 * u2, &sn, &cs);
    *v1 = rr * cs;
    *v2 = rr * sn;
}

// X = the standard normals of noise draw `step`
__global__ void k_sgle_noise(cplx* __restrict__ X, int N, unsigned long long step, unsigned long long seed)
{
    const size_t n2 = (size_t)N * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x) {
        double v1, v2;
        sgle_normals(i, step, seed, &v1, &v2);
        X[i] = mk(v1, v2);
    }
}

struct NoiseArgs {
    const cplx* X;   // the caller's standard normals, or null: draw `step` of seed
    cplx* H;
    unsigned long long step, seed;
    double invsq, sigma;   // 1/sqrt(dvol), then noisesigma (src/gpe.f90:163)
    double* om;
};

// The noise rows of one SGLE step: standard normals, scaled, transformed along
// x, retained panels stored.
template <class C>
__device__ __forceinline__ void noise_row_body(int blk_, int nblk_, const cplx* __restrict__ tw, Geo g,
                                               const NoiseArgs& a)
{
    VK_ROW_SETUP(C)
    const auto w_ = twiddles<C>(tw, t);
    if (blk_ == 0 && threadIdx.x == 0) a.om[0] = a.om[1];
    cplx v[S];
    if (a.X) {
        const cplx* xr = a.X + (size_t)y * N;
#pragma unroll
        for (int s = 0; s < S; ++s) v[s] = rmul(a.sigma, rmul(a.invsq, xr[t + T * s]));
    } else {
        // the generator in a loop, its points passed on through this thread's
        // own LDS slots (unrolled, it would be S copies of log and sincos)
        constexpr int Q = S / 2;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll 1
            for (int s = 0; s < Q; ++s) {
                double v1, v2;
                sgle_normals((size_t)y * N + t + T * (h * Q + s), a.step, a.seed, &v1, &v2);
                const cplx z = rmul(a.sigma, rmul(a.invsq, mk(v1, v2)));
                lg[s * T + t] = z.x;
                lg[N / 2 + s * T + t] = z.y;
            }
#pragma unroll
            for (int s = 0; s < Q; ++s) v[h * Q + s] = mk(lg[s * T + t], lg[N / 2 + s * T + t]);
        }
        lds_barrier();
    }
    fft_fwd<N, S, C::SPLIT>(v, lg, t, w_);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int pp = VK_PANEL(s);
        if (panel_stored(pp, NP, g, 1)) a.H[hoff<C>(pp, y, c)] = v[s];
    }
}

// P1 of an SGLE step with its norm sums, and the noise rows, which need
// nothing of it, as the first half of the same launch: P1's loads and the
// generator's arithmetic then share the CUs (25 us together at 1024^2, where
// the generator's 13, the noise rows' 11 and P1's 12 ran one after another).
// With A4 taking the noise columns and the norm, an SGLE step is 4 launches
// of 9 and moves no noise through k-space: 128^2 32.0 to 21.9 us, 512^2 56.0
// to 44.8, 1024^2 88.4 to 64.8, 4096^2 1160 to 960.
template <class C>
__global__ void __launch_bounds__(C::ROWT) VK_OCC k_p1_noise(const cplx* __restrict__ Hpsi, cplx* __restrict__ Hrho,
                                                     const cplx* __restrict__ tw, Geo g, double scale,
                                                     cplx* __restrict__ Xpsi, double* __restrict__ nsum, NoiseArgs a)
{
    const int nb = gridDim.x / 2;
    if ((int)blockIdx.x < nb) noise_row_body<C>(blockIdx.x, nb, tw, g, a);
    else p1_body<C, true, true>(blockIdx.x - nb, nb, Hpsi, Hrho, tw, g, 0, scale, Xpsi, nsum);
}

// ----------------------------------------------------------------------------
// Vortex initial condition and the imposed vortex velocity
// ----------------------------------------------------------------------------

// Padé-core vortex product: amplitude prod_j sqrt(rho(r_j/xi)), r_j the
// minimum-image distance; phase sum_j q_j sum_{|m|<=nimg}
// arg(sin((x-x_j)/2 + i(y-y_j-2 pi m)/2)) - (sum_j q_j x_j) y/(2 pi), which
// is 2 pi-periodic in x and y for zero net charge up to exp(-2 pi nimg).
__host__ __device__ inline void ic_point(double x, double y, int nv, const double* xs, const double* ys,
                                         const int* qs, double xi, int nimg, double* out)
{
    const double pi = 3.14159265358979323846;
    const double a1 = 11.0 / 32.0, a2 = 11.0 / 384.0, b1 = 1.0 / 3.0;
    double amp = 1.0, pr = 1.0, pim = 0.0, lin = 0.0;
    for (int j = 0; j < nv; ++j) {
        double dxp = x - xs[j], dyp = y - ys[j];
        double wx = dxp - 2.0 * pi * floor(dxp / (2.0 * pi) + 0.5);
        double wy = dyp - 2.0 * pi * floor(dyp / (2.0 * pi) + 0.5);
        double r2 = (wx * wx + wy * wy) / (xi * xi);
        double rho = r2 * (a1 + a2 * r2) / (1.0 + b1 * r2 + a2 * r2 * r2);
        amp *= sqrt(rho);
        lin += qs[j] * xs[j];
        const double sX = sin(0.5 * dxp), cX = cos(0.5 * dxp);
        for (int m = -nimg; m <= nimg; ++m) {
            const double Y = 0.5 * (dyp - 2.0 * pi * m);
            double zr = sX * cosh(Y), zi = cX * sinh(Y);
            const double h = sqrt(zr * zr + zi * zi);
            if (h > 0.0) { zr /= h; zi /= h; } else { zr = 1.0; zi = 0.0; }
            if (qs[j] < 0) zi = -zi;
            const double nr = pr * zr - pim * zi, ni = pr * zi + pim * zr;
            pr = nr;
            pim = ni;
        }
        const double hn = sqrt(pr * pr + pim * pim);
        pr /= hn;
        pim /= hn;
    }
    const double th = -lin * y / (2.0 * pi);
    const double c = cos(th), s = sin(th);
    out[0] = amp * (pr * c - pim * s);
    out[1] = amp * (pr * s + pim * c);
}

// Imposed velocity of a vortex configuration for the advective ARGLE:
// u = 2 alpha rho0 grad(theta0), the current of the Padé product ansatz
// (rho0 = prod_j rho(r_j/xi), theta0 its phase), smooth and zero in the
// cores.  grad arg(sin((X + i Y_m)/2)) = (-sinh Y_m, sin X)/(2 (cosh Y_m -
// cos X)), summed over the nimg images Y_m = Y - 2 pi m and the vortices
// with their charges, minus (sum_j q_j x_j)/(2 pi) along y from the linear
// phase term.
__host__ __device__ inline void vortex_velocity_point(double x, double y, int nv, const double* xs,
                                                      const double* ys, const int* qs, double xi, int nimg,
                                                      double alpha, double* ux, double* uy)
{
    const double pi = 3.14159265358979323846;
    const double a1 = 11.0 / 32.0, a2 = 11.0 / 384.0, b1 = 1.0 / 3.0;
    double rho = 1.0, gx = 0.0, gy = 0.0, lin = 0.0;
    for (int j = 0; j < nv; ++j) {
        const double dxp = x - xs[j], dyp = y - ys[j];
        const double wx = dxp - 2.0 * pi * floor(dxp / (2.0 * pi) + 0.5);
        const double wy = dyp - 2.0 * pi * floor(dyp / (2.0 * pi) + 0.5);
        const double r2 = (wx * wx + wy * wy) / (xi * xi);
        rho *= r2 * (a1 + a2 * r2) / (1.0 + b1 * r2 + a2 * r2 * r2);
        lin += qs[j] * xs[j];
        const double sX = sin(dxp), cX = cos(dxp);
        for (int m = -nimg; m <= nimg; ++m) {
            const double Ym = dyp - 2.0 * pi * m;
            const double den = cosh(Ym) - cX;
            if (den > 0.0) {
                gx += qs[j] * (-0.5 * sinh(Ym) / den);
                gy += qs[j] * (0.5 * sX / den);
            }
        }
    }
    gy -= lin / (2.0 * pi);
    *ux = 2.0 * alpha * rho * gx;
    *uy = 2.0 * alpha * rho * gy;
}

__global__ void k_vortex_velocity(double* __restrict__ UX, double* __restrict__ UY, int N, int nv,
                                  const double* __restrict__ xs, const double* __restrict__ ys,
                                  const int* __restrict__ qs, double xi, int nimg, double alpha)
{
    const size_t n2 = (size_t)N * N;
    const double dx = 2.0 * 3.14159265358979323846 / N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x)
        vortex_velocity_point((int)(i % N) * dx, (int)(i / N) * dx, nv, xs, ys, qs, xi, nimg, alpha, UX + i, UY + i);
}

__global__ void k_ic(cplx* __restrict__ X, int N, int nv, const double* __restrict__ xs,
                     const double* __restrict__ ys, const int* __restrict__ qs, double xi, int nimg)
{
    const size_t n2 = (size_t)N * N;
    const double dx = 2.0 * 3.14159265358979323846 / N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n2; i += (size_t)gridDim.x * blockDim.x) {
        const int ix = (int)(i % N), iy = (int)(i / N);
        double o[2];
        ic_point(ix * dx, iy * dx, nv, xs, ys, qs, xi, nimg, o);
        X[i] = mk(o[0], o[1]);
    }
}

}  // namespace vk
