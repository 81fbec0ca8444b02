// Host side of the vikshobha library: handle, pipelines, C ABI.
//
// One RK4 stage (src/gpe.f90:357-492 around gpe_rhs :498-671) is four
// passes over HBM:
//   P1 row   : psi(y,.) = IFFT_x Hpsi ; rho = |psi|^2 ; Hrho = FFT_x rho
//   P2 column: rho-hat = FFT_y Hrho ; P_G ; Hrho_d = IFFT_y
//   P3 row   : rho_d, V, psi rows ; N = (g rho_d + V) psi ; HN = FFT_x N
//   P4 column: N-hat = FFT_y HN ; RHS, RK4 accumulation ; Hpsi = IFFT_y kpsi
// kpsi is dealiased, so only |kx| <= N/3 columns are stored and moved;
// rho, rho_d and V are real, so only their kx >= 0 halves are moved.
#include "vk_ens.hpp"
#include "vk_target.hpp"
#include "vikshobha.h"

#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <type_traits>
#include <vector>

using vk::cplx;
using vk::Geo;

namespace {
thread_local std::string g_err;
}

// Scratch of the allocation-free entry point vk_fft2d_noalloc: one
// half-spectral field (the row pass output the column pass reads) of the
// largest size that entry point accepts, VK_NOALLOC_MAX_N^2 complex doubles
// = 16 MiB.  Every GPU the library runs on holds its own copy until the
// process ends.  Host code never passes this name to a kernel: its device
// address on each device is looked up once, in vk_gpe_create with that
// device current (scratch_setup), and kept in g_scratch_ptr.
#define VK_NOALLOC_MAX_N 1024
#define VK_MAX_DEVICES 64
static __device__ __align__(256) double2 scratch[(size_t)VK_NOALLOC_MAX_N * VK_NOALLOC_MAX_N];

// shared with the other translation units of the library (vk_last_error)
int vk_set_error(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

namespace {

int fail(int code, const std::string& msg) { return vk_set_error(code, msg); }

#define HIPCHK(x)                                                                          \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess) return fail(VK_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

enum PassKind { PK_P1 = 0, PK_P2, PK_P3, PK_P4, PK_PART, PK_ARG4, PK_OTHER, PK_COUNT };
const char* kPassNames[PK_COUNT] = {"p1_rho_row", "p2_dealias_col", "p3_nonlin_row", "p4_rk4_col",
                                    "particles", "argle_update_col", "other"};

bool masked_host(int kx, int ky, int N) { return 9LL * ((long long)kx * kx + (long long)ky * ky) >= (long long)N * N; }

std::mutex g_scratch_mu;
cplx* g_scratch_ptr[VK_MAX_DEVICES] = {};

// device address of `scratch` on device dev, which must be current; looked
// up on the first handle created on that device and kept
int scratch_setup(int dev)
{
    if (dev < 0 || dev >= VK_MAX_DEVICES) return fail(VK_ERR_UNSUPPORTED, "device index beyond the library's table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev]) return 0;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return fail(VK_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<cplx*>(ptr);
    return 0;
}

}  // namespace

struct vk_gpe {
    vk_gpe_params p{};
    int N = 0;
    int nshell = 0;
    Geo geo{};
    int NP = 0, TC = 0;
    hipStream_t stream = nullptr;
    hipStream_t pstream = nullptr;     // particle update, overlapped with P4/P1/P2
    hipEvent_t ev_p3 = nullptr, ev_ps = nullptr;
    cplx* tw = nullptr;
    // state and RK4/ARGLE work fields
    cplx *K0 = nullptr, *K1 = nullptr, *K2 = nullptr, *Hpsi = nullptr, *Hrho = nullptr, *HN = nullptr;
    // x-space field: psi rows from P1 to P3 within a step, and between steps the
    // staging of the x-space transforms (all on the handle's stream)
    cplx* Xs = nullptr;
    int dev = 0;        // device the handle was created on
    int ncu = 0;        // compute units of the device
    int p1pf = 0;       // RK4 P1 as the persistent prefetching kernel (4096^2)
    int tr1_p1 = 0, tr1_p3 = 0;   // RK4 P1 / P3 (psi-row path) with one row per workgroup
    // advective ARGLE (Taylor-Green and/or counterflow); Hdy = IFFT_y(i ky kpsi)
    int adv_tg = 0;
    double adv_vx = 0.0, adv_vy = 0.0;
    cplx* Hdy = nullptr;
    // caller-supplied advection velocity (replaces the Taylor-Green field)
    double *Ux = nullptr, *Uy = nullptr;
    int adv_field = 0;
    // SGLE (GPE_SGLE): the caller's normals (or the generator's, on request), the
    // chemical potential before and after a step on the device, the row sums of
    // |psi|^2, the draw counter of the generator
    int sgle = 0;
    double sg_beta = 0.0, sg_nuN = 0.0, sg_ktrunc = 0.0;
    unsigned long long sg_seed = 0, sg_draw = 0;
    cplx* Xn = nullptr;
    double *omega_dev = nullptr, *npart = nullptr;
    cplx *HV = nullptr, *KV = nullptr, *Krho = nullptr, *Vhat = nullptr, *EX = nullptr, *EY = nullptr;
    double* pst2 = nullptr;   // real-space path: positions and velocities after RK4 stages 1 and 3
    int side_busy = 0;        // a particle update is queued on pstream
    double *fpart = nullptr, *pst = nullptr, *part = nullptr, *dsum = nullptr;
    unsigned char* phit = nullptr;   // real-space path: window flags per row block and particle
    int4* pwin = nullptr;            // real-space path: windows and factor tables of the positions,
    double2 *ptx = nullptr, *pty = nullptr;
    double* Vx = nullptr;            // and the potential on the grid for ARGLE
    int vx_valid = 0;   // Vx belongs to the current positions
    int hstate = 0;   // 0: Hpsi stale, 1: Hpsi = IFFT_y K0 on all panels, 2: K0 dealiased, Hpsi on retained panels,
                      // 3: K0 dealiased, Hpsi on the retained panels of the single-field shape svar (layout CfgE<N, svar>)
    int kv_valid = 0;
    int have_part = 0;
    int np_cap = 0;     // particle buffers are sized for this many particles
    int rs_part = 0;   // particle potential and force evaluated in real space inside P3
    // diagnostics
    cplx* Kd0 = nullptr;
    cplx* Hd = nullptr;
    double* hres = nullptr;   // pinned: sums and spectra of the last call
    int diag_ready = 0;
    // ensemble shape variant of this member (CfgE<N, ens_var>) and its
    // panel geometry; Hpsi holds that variant's layout only between the
    // ensemble's preparation and the member's next single-field access
    int ens_var = 0;
    Geo geo_v{};
    // transform shape of the single field: 0 (CfgS<N>; bit for bit a default
    // ensemble member), 1 (CfgE<N, 1>, stepped as an ensemble of one with the
    // member table below)
    int svar = 0;
    Geo geo_s{};
    vk::EnsReal* e1R = nullptr;
    int* e1map[3] = {};
    int* e1off[3] = {};
    int e1nblk[3] = {};
    size_t e1lds[4] = {};
    // timing
    bool timing = false;
    std::vector<hipEvent_t> ev;
    std::vector<int> evkind;
    size_t evn = 0;
};

namespace {

size_t f2(const vk_gpe* h) { return (size_t)h->N * h->N; }

// A field made on first use, zero: cleared by a kernel on the stream of the
// kernels that follow, which is non-blocking (a clear on the default stream
// could land after them)
int make_field(vk_gpe* h, cplx** p, hipStream_t st)
{
    if (*p) return 0;
    HIPCHK(hipMalloc(p, f2(h) * sizeof(cplx)));
    hipLaunchKernelGGL(vk::k_zero, dim3(1024), dim3(256), 0, st, *p, f2(h));
    return 0;
}

template <int N> using CfgN = vk::CfgS<N>;
// The same panel layout with one row per row-pass workgroup (256 threads)
// instead of TR rows: more, smaller workgroups per CU at the cost of half
// as long row pieces of the panels.
template <class C> using CfgTR1 = vk::CfgT<C::N, C::S, C::TC, 1, C::SPLIT>;

template <class F>
int dispatch(int N, F&& f)
{
    switch (N) {
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
    case 256: return f(std::integral_constant<int, 256>{});
    case 512: return f(std::integral_constant<int, 512>{});
    case 1024: return f(std::integral_constant<int, 1024>{});
    case 2048: return f(std::integral_constant<int, 2048>{});
    case 4096: return f(std::integral_constant<int, 4096>{});
    default: return fail(VK_ERR_UNSUPPORTED, "N must be a power of two in [32, 4096]");
    }
}

void ev_begin(vk_gpe* h)
{
    if (!h->timing) return;
    if (h->evn + 2 > h->ev.size()) {
        for (int i = 0; i < 64; ++i) {
            hipEvent_t e;
            if (hipEventCreate(&e) == hipSuccess) h->ev.push_back(e);
        }
    }
    hipEventRecord(h->ev[h->evn], h->stream);
}
void ev_end(vk_gpe* h, int kind)
{
    if (!h->timing) return;
    hipEventRecord(h->ev[h->evn + 1], h->stream);
    h->evkind.push_back(kind);
    h->evn += 2;
}

std::mutex g_lds_mu;
std::map<const void*, size_t> g_lds_max;   // dynamic-LDS limit set per kernel so far

template <class Kern>
void set_lds(Kern k, size_t bytes)
{
    // the limit only grows: a kernel whose LDS depends on a runtime size
    // (P3 with np particles) may be launched larger than at its first use
    if (bytes <= 65536) return;
    std::lock_guard<std::mutex> lk(g_lds_mu);
    size_t& cur = g_lds_max[(const void*)k];
    if (bytes > cur) {
        hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        cur = bytes;
    }
}

template <class C, class Kern, class... A>
void row_launch_x(vk_gpe* h, int kind, size_t extra, Kern k, A... args)
{
    const size_t lds = (size_t)C::TR * C::ROWRS * sizeof(double) + extra;
    set_lds(k, lds);
    ev_begin(h);
    hipLaunchKernelGGL(k, dim3(C::N / C::TR), dim3(C::ROWT), lds, h->stream, args...);
    ev_end(h, kind);
}

template <class C, class Kern, class... A>
void row_launch(vk_gpe* h, int kind, Kern k, A... args)
{
    row_launch_x<C>(h, kind, 0, k, args...);
}

// P3 stages the particle windows after its transform regions
size_t p3_extra(const vk_gpe* h) { return (size_t)std::max(h->p.np, 1) * sizeof(int4); }

// P2 columns per workgroup.  P2 covers only the kx >= 0 panels.  At
// 4096^2 one column per workgroup (1366 workgroups) is the fastest: with
// 2-column panels 4% faster than whole panels, with 4-column panels
// 0.0697 against 0.0707 ms for two columns; at 2048^2 one column is 10%
// slower than whole panels.  Results are bitwise the same either way.
#ifndef VK_P2_COLS_4096
#define VK_P2_COLS_4096 1
#endif
// The LAT shapes have their own.
template <class C> constexpr int p2_cols()
{
    if constexpr (vk::is_lat<C>::value) return C::G;
    else return C::N == 4096 ? VK_P2_COLS_4096 : C::TC;
}
// P4 columns per workgroup at 4096^2 (0: whole panels).  Two of the four
// columns of a panel in a 512-thread workgroup: 0.170 ms against 0.189 for
// whole panels (1024 threads, one workgroup per CU) and 0.193 for one.
#ifndef VK_P4_COLS_4096
#define VK_P4_COLS_4096 2
#endif
template <class C> constexpr int p4_cols()
{
    if constexpr (vk::is_lat<C>::value) return C::G;
    else return C::N == 4096 && VK_P4_COLS_4096 > 0 ? VK_P4_COLS_4096 : C::TC;
}

// column pass with G columns per workgroup over npan panels
template <class C, int G, class Kern, class... A>
void colg_launch(vk_gpe* h, int kind, int npan, Kern k, A... args)
{
    constexpr int GS = C::TC / G;
    const size_t lds = (size_t)G * C::COLRS * sizeof(double);
    set_lds(k, lds);
    const int grid = GS == 1 ? npan : (npan + 7) / 8 * 8 * GS;
    ev_begin(h);
    hipLaunchKernelGGL(k, dim3(grid), dim3(G * C::T), lds, h->stream, args...);
    ev_end(h, kind);
}

// P4 after the workgroups of the particles' update
template <class C, int G, class Kern>
void p4_part_launch(vk_gpe* h, Kern k, const vk::RKArgs& a, const vk::PStage& q)
{
    constexpr int GS = C::TC / G;
    const size_t lds = (size_t)G * C::COLRS * sizeof(double);
    set_lds(k, lds);
    const int npan = h->geo.Pp + h->geo.Pn, grid = GS == 1 ? npan : (npan + 7) / 8 * 8 * GS;
    hipLaunchKernelGGL(k, dim3((h->p.np + 7) / 8 * 8 + grid), dim3(G * C::T), lds, h->stream, (const cplx*)h->HN,
                       h->Hpsi, h->K0, h->K1, h->K2, (const cplx*)h->tw, h->geo, a, q);
}

// the flags (last argument, 0..3) select a compile-time instantiation
template <class C>
void p2_launch(vk_gpe* h, cplx* Hrho, cplx* HV, const cplx* KV, cplx* Krho, const cplx* tw, Geo g, int flags)
{
    constexpr int G = p2_cols<C>();
    auto go = [&](auto k) { colg_launch<C, G>(h, PK_P2, h->geo.Pp, k, Hrho, HV, KV, Krho, tw, g, flags); };
    if (flags == 0) go(vk::k_p2<C, G, 0>);
    else if (flags == 1) go(vk::k_p2<C, G, 1>);
    else if (flags == 2) go(vk::k_p2<C, G, 2>);
    else go(vk::k_p2<C, G, 3>);
}

// The persistent prefetching P1 (vk::k_p1xp) runs at 4096^2 when the
// runtime panel geometry is the one its LDS slot map was built for and the
// row blocks split evenly over one workgroup per CU in XCD groups of 8.
#ifndef VK_P1_PREFETCH
#define VK_P1_PREFETCH 1
#endif
// the persistent prefetching P1 fits this handle and device (4096^2, a CU
// count whose row blocks divide evenly over the XCDs)
int p1_prefetch_fits(const vk_gpe* h)
{
    if (!VK_P1_PREFETCH || h->N != 4096) return 0;
    using C = CfgN<4096>;
    static_assert(vk::p1p_lds<C>() <= 160 * 1024, "prefetch buffer exceeds LDS");
    const int g8 = h->ncu / 8, r8 = (C::N / C::TR) / 8;
    return h->ncu > 0 && h->ncu % 8 == 0 && r8 % g8 == 0 && h->geo.Pp == vk::geo_pp<C>() &&
           h->geo.Pn == vk::geo_pn<C>();
}

int p1_prefetch_ok(const vk_gpe* h)
{
    // the plain P1, whose loads are all in flight at once, is faster; the
    // prefetching kernel runs when VK_P1_PREFETCH=1 (tests compare the two)
    const char* on = std::getenv("VK_P1_PREFETCH");
    return on && on[0] == '1' && p1_prefetch_fits(h);
}

template <class C>
void p1p_launch(vk_gpe* h, double sc)
{
    if constexpr (C::N == 4096) {
        auto k = vk::k_p1xp<C>;
        const size_t lds = vk::p1p_lds<C>();
        set_lds(k, lds);
        ev_begin(h);
        hipLaunchKernelGGL(k, dim3(h->ncu), dim3(C::ROWT), lds, h->stream, (const cplx*)h->Hpsi, h->Hrho,
                           (const cplx*)h->tw, h->geo, sc, h->Xs);
        ev_end(h, PK_P1);
    }
}

int ncols(const vk_gpe* h, int pmode)
{
    return pmode == 0 ? h->NP : h->geo.Pp + h->geo.Pn;
}

double scale_of(const vk_gpe* h) { return 1.0 / ((double)h->N * (double)h->N); }

// ---- generic 2D transforms ------------------------------------------------

int fwd2d(vk_gpe* h, const cplx* X, cplx* Hs, cplx* K, int op_col)
{
    return dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        row_launch<C>(h, PK_OTHER, vk::k_row_fwd<C>, X, Hs, (const cplx*)h->tw);
        constexpr int G = p4_cols<C>();
        colg_launch<C, G>(h, PK_OTHER, h->NP, vk::k_col_fwd<C, G>, (const cplx*)Hs, K, (const cplx*)h->tw, op_col);
        return 0;
    });
}

int col_inv(vk_gpe* h, const cplx* K, cplx* Hs, int pmode, int op)
{
    return dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        constexpr int G = p4_cols<C>();
        colg_launch<C, G>(h, PK_OTHER, ncols(h, pmode), vk::k_col_inv<C, G>, K, Hs, (const cplx*)h->tw, h->geo, pmode,
                          op);
        return 0;
    });
}

int row_inv(vk_gpe* h, const cplx* Hs, cplx* X, int pload, double scale)
{
    return dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        row_launch<C>(h, PK_OTHER, vk::k_row_inv<C>, Hs, X, (const cplx*)h->tw, h->geo, pload, scale);
        return 0;
    });
}

int dealias_k(vk_gpe* h, cplx* K)
{
    hipLaunchKernelGGL(vk::k_dealias, dim3(1024), dim3(256), 0, h->stream, K, h->N);
    return 0;
}

// ---- state management -------------------------------------------------------

int ensure_any(vk_gpe* h)
{
    if (h->hstate == 0 || h->hstate == 3) {
        int rc = col_inv(h, h->K0, h->Hpsi, 0, 0);
        if (rc) return rc;
        h->hstate = 1;
    }
    return 0;
}

int ensure_rk4(vk_gpe* h)
{
    if (h->hstate != 2) {
        dealias_k(h, h->K0);
        int rc = col_inv(h, h->K0, h->Hpsi, 1, 0);
        if (rc) return rc;
        h->hstate = 2;
    }
    return 0;
}

int ensure_full(vk_gpe* h)
{
    if (h->hstate != 1) {
        int rc = col_inv(h, h->K0, h->Hpsi, 0, 0);
        if (rc) return rc;
        h->hstate = 1;
    }
    return 0;
}

// ---- particles ----------------------------------------------------------------

double ipow(double x, int n)
{
    double r = 1.0;
    for (int i = 0; i < n; ++i) r *= x;
    return r;
}

vk::PartArgs part_args(const vk_gpe* h, int nrows, int half, int stage, int nblk = 0, int nw = 0)
{
    const double pi = 4.0 * std::atan(1.0);
    const double L = 2.0 * pi;
    const double dx = L / h->N;
    vk::PartArgs a{};
    a.np = h->p.np;
    a.N = h->N;
    a.nrows = nrows;
    a.half = half;
    a.coef = 2.0 * h->p.alpha * (dx * dx) / ((double)h->N * (double)h->N);
    const double dE = (double)0.062f;         // src/gpe_particle.f90:395, default-real literal
    const double r0 = 4.0 * h->p.xi;         // :396
    a.rf = 384.0 * dE * ipow(pi, 12) * ipow(r0, 12) / ipow(L, 12);
    a.efac = 64.0 * dE * ipow(pi, 12) * ipow(r0, 12) / ipow(L, 12);
    a.dt = h->p.dt;
    a.mass = h->p.mass;
    a.stage = stage;
    a.nblk = nblk;
    a.nw = nw;
    return a;
}

// Window radius (in the minimum-image displacement a) of the real-space
// particle potential.  The potential depends on the periodic coordinate
// X(a) = 2(s + s^3/6 + s^5/40), s = sin(a/2), which saturates at
// X(pi) = 2.383 near the half box, so V at the edge a = 10 d is
// V0 exp(-X(10 d)^2/(2 d^2)), not V0 exp(-50).  The 10 d window is kept when
// that is below exp(-45) (3e-20) of the peak (X(a) = a - O(a^5) for small
// a, so narrow potentials keep it); otherwise the window covers the whole
// period (any radius >= pi does).
double real_space_window(double d)
{
    const double pi = 4.0 * std::atan(1.0);
    const double a = std::min(10.0 * d, pi);
    const double s = std::sin(0.5 * a), s2 = s * s;
    const double X = 2.0 * (s + (1.0 / 6.0) * (s2 * s) + (1.0 / 40.0) * (s2 * s2 * s));
    if (10.0 * d < pi && X * X / (2.0 * d * d) >= 45.0) return 10.0 * d;
    return 4.0;
}

vk::P3Part p3part(const vk_gpe* h)
{
    vk::P3Part q{};
    if (h->p.np > 0 && h->have_part) {
        q.win = h->pwin;
        q.tx = h->ptx;
        q.ty = h->pty;
        q.ppart = h->fpart;
        q.phit = h->phit;
        q.np = h->p.np;
        q.vx = h->Vx;
    }
    return q;
}

vk::WTab wtab(const vk_gpe* h)
{
    return vk::WTab{h->p.V0, h->p.d, real_space_window(h->p.d), h->pwin, h->ptx, h->pty};
}

// The particles have been set: windows and tables of their positions now, not
// in the next step, so that they follow the positions for every later step,
// also one that was recorded before (steps move them along themselves)
void particles_moved(vk_gpe* h)
{
    h->kv_valid = h->vx_valid = 0;
    if (h->rs_part)
        hipLaunchKernelGGL(vk::k_wtab, dim3(h->p.np, 2), dim3(128), 0, h->stream, (const double*)h->pst, h->N, wtab(h));
}

// ARGLE never moves the particles: their potential on the grid, once per set
// of positions
int particle_field(vk_gpe* h)
{
    if (h->vx_valid) return 0;
    if (!h->Vx) HIPCHK(hipMalloc(&h->Vx, f2(h) * sizeof(double)));
    hipLaunchKernelGGL(vk::k_potfield, dim3(std::min((int)(f2(h) / 256), 4096)), dim3(256), 0, h->stream,
                       (const int4*)h->pwin, (const double2*)h->ptx, (const double2*)h->pty, h->p.np, h->N, h->Vx);
    h->vx_valid = 1;
    return 0;
}

// Real-space particle path in P3: valid when the Gaussian's spectrum beyond
// the dealias radius, exp(-(N/3 d)^2 / 2), is below 1e-20 of its peak (and
// the aliasing beyond N/2 smaller still), so the reference's spectral
// translation equals the analytic V(x - q) to far below FP64 roundoff.
int use_real_space(const vk_gpe_params& p)
{
    if (p.np <= 0 || p.d <= 0.0) return 0;
    const double kd = (p.N / 3.0) * p.d;
    return 0.5 * kd * kd > 46.0;
}

// KV on rows [0, nrows) from the current positions
int particle_kv(vk_gpe* h, int nrows)
{
    const int np = h->p.np;
    ev_begin(h);
    hipLaunchKernelGGL(vk::k_ptab, dim3((np * h->N + 255) / 256), dim3(256), 0, h->stream, (const double*)h->pst,
                       h->EX, h->EY, np, h->N);
    hipLaunchKernelGGL(vk::k_kv, dim3(nrows), dim3(256), (size_t)np * sizeof(cplx), h->stream,
                       (const cplx*)h->Vhat, (const cplx*)h->EX, (const cplx*)h->EY, h->KV, np, h->N);
    ev_end(h, PK_PART);
    return 0;
}

int particle_forces(vk_gpe* h, const cplx* Krho, int nrows, int half, int stage)
{
    const int np = h->p.np;
    constexpr int PG = 8;
    ev_begin(h);
    hipLaunchKernelGGL(vk::k_force_rows<PG>, dim3(nrows, (np + PG - 1) / PG), dim3(256), 0, h->stream, Krho,
                       (const cplx*)h->Vhat, (const cplx*)h->EY, h->fpart, np, h->N);
    hipLaunchKernelGGL(vk::k_pstep, dim3(1), dim3(vk::PSTEP_T), 0, h->stream, (const double*)h->fpart, (const cplx*)h->EX,
                       h->pst, part_args(h, nrows, half, stage));
    ev_end(h, PK_PART);
    return 0;
}

// Particle stage update from the real-space block partials written by P3; the
// next P3 needs its window tables.  From 2048^2 on it runs on a side stream
// while P4, P1, P2 proceed (0.1 ms of passes hide it); below, the two event
// waits would cost more than the update itself (6 us), and it goes with P4
// (vk::k_p4_part) where P4's workgroups are whole waves.
vk::PStage pstage_args(vk_gpe* h, int nblk, int nw, int stage)
{
    double *cur = stage % 2 ? h->pst : h->pst2, *nxt = stage % 2 ? h->pst2 : h->pst;
    return vk::PStage{h->fpart, h->phit, cur, nxt, h->pst, part_args(h, 0, 0, stage, nblk, nw), wtab(h)};
}

template <int NT>
int particle_step_rs(vk_gpe* h, int nblk, int nw, int stage)
{
    const bool side = !h->timing && h->pstream && h->N >= 2048;
    hipStream_t st = side ? h->pstream : h->stream;
    if (side) {
        hipEventRecord(h->ev_p3, h->stream);
        hipStreamWaitEvent(h->pstream, h->ev_p3, 0);
    }
    ev_begin(h);
    hipLaunchKernelGGL(vk::k_pstage<NT>, dim3(h->p.np), dim3(NT), 0, st, pstage_args(h, nblk, nw, stage));
    ev_end(h, PK_PART);
    if (side) {
        hipEventRecord(h->ev_ps, h->pstream);
        h->side_busy = 1;
    }
    return 0;
}

// order the main stream after the last side-stream particle update
void join_particles(vk_gpe* h)
{
    if (!h->side_busy) return;
    hipStreamWaitEvent(h->stream, h->ev_ps, 0);
    h->side_busy = 0;
}

// ---- RK4 / ARGLE -----------------------------------------------------------------

int ens1_step(vk_gpe* h);
vk::EnsReal single_entry(const vk_gpe* h);
int prep_rk4(vk_gpe* h);

int rk4_step(vk_gpe* h)
{
    if (h->svar) return ens1_step(h);
    return dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        const double sc = scale_of(h);
        const double dt = h->p.dt, oney6 = 1.0 / 6.0;
        const int parts = h->have_part && h->p.np > 0;
        const int rs = parts && h->rs_part;
        const int Kp = C::TC * h->geo.Pp;
        h->vx_valid = 0;
        const vk::P3Part pa = p3part(h);
        vk::RKArgs a{};
        a.pref = make_double2(-h->p.disp, -1.0);   // (1 - i disp)/i
        a.alpha = h->p.alpha;
        a.omega = h->p.omega;
        for (int stage = 1; stage <= 4; ++stage) {
            if (parts && !rs) particle_kv(h, Kp);
            constexpr bool VAR = C::N >= 2048;   // sizes with row-pass variants
            using C1 = std::conditional_t<VAR, CfgTR1<C>, C>;
            if (h->p1pf)
                p1p_launch<C>(h, sc);
            else if (VAR && h->tr1_p1)
                row_launch<C1>(h, PK_P1, vk::k_p1x<C1>, (const cplx*)h->Hpsi, h->Hrho, (const cplx*)h->tw, h->geo, 1,
                               sc, h->Xs);
            else
                row_launch<C>(h, PK_P1, vk::k_p1x<C>, (const cplx*)h->Hpsi, h->Hrho, (const cplx*)h->tw, h->geo, 1, sc,
                              h->Xs);
            p2_launch<C>(h, h->Hrho, h->HV, (const cplx*)h->KV, h->Krho,
                          (const cplx*)h->tw, h->geo, (parts && !rs) ? 3 : 0);
            if (parts && !rs) particle_forces(h, h->Krho, Kp, 1, stage);
            if (rs) join_particles(h);   // positions from the previous stage
            if (VAR && h->tr1_p3) {
                auto k3 = !parts ? vk::k_p3x<C1, 0> : (rs ? vk::k_p3x<C1, 4> : vk::k_p3x<C1, 1>);
                row_launch_x<C1>(h, PK_P3, p3_extra(h), k3, (const cplx*)h->Hrho, (const cplx*)h->HV,
                                 (const cplx*)h->Xs, h->HN, (const cplx*)h->tw, h->geo, 1, h->p.g * sc, sc, 1.0, pa);
            } else {
                auto k3 = !parts ? vk::k_p3x<C, 0> : (rs ? vk::k_p3x<C, 4> : vk::k_p3x<C, 1>);
                row_launch_x<C>(h, PK_P3, p3_extra(h), k3, (const cplx*)h->Hrho, (const cplx*)h->HV,
                                (const cplx*)h->Xs, h->HN, (const cplx*)h->tw, h->geo, 1, h->p.g * sc, sc, 1.0, pa);
            }
            constexpr int G4 = p4_cols<C>();
            // up to 1024^2 the particles' update goes with P4 (timed passes: alone)
            constexpr bool WITH_P4 = !VAR && G4 * C::T >= 64;
            constexpr int PT = WITH_P4 ? G4 * C::T : 256;
            const bool with_p4 = WITH_P4 && rs && !h->timing;
            if (rs && !with_p4) {
                if (VAR && h->tr1_p3) particle_step_rs<PT>(h, C::N, (C1::ROWT + 63) / 64, stage);
                else particle_step_rs<PT>(h, C::N / C::TR, (C::ROWT + 63) / 64, stage);
            }
            a.stage = stage;
            a.wacc = (stage == 1 || stage == 4) ? dt * oney6 : dt * oney6 * 2.0;
            a.cstep = stage == 3 ? dt : dt * 0.5;
            a.r1 = (dt * oney6) / (dt * 0.5);
            a.r3 = (dt * oney6 * 2.0) / dt;
            if constexpr (WITH_P4) {
                if (with_p4) {
                    auto kp = stage == 1 ? vk::k_p4_part<C, 1, G4> : stage == 2 ? vk::k_p4_part<C, 2, G4>
                                         : stage == 3 ? vk::k_p4_part<C, 3, G4> : vk::k_p4_part<C, 4, G4>;
                    p4_part_launch<C, G4>(h, kp, a, pstage_args(h, C::N / C::TR, (C::ROWT + 63) / 64, stage));
                    continue;
                }
            }
            auto k4 = stage == 1 ? vk::k_p4<C, 1, G4> : stage == 2 ? vk::k_p4<C, 2, G4>
                                                      : stage == 3 ? vk::k_p4<C, 3, G4> : vk::k_p4<C, 4, G4>;
            colg_launch<C, G4>(h, PK_P4, h->geo.Pp + h->geo.Pn, k4, (const cplx*)h->HN, h->Hpsi, h->K0, h->K1,
                               h->K2, (const cplx*)h->tw, h->geo, a);
        }
        if (rs) join_particles(h);
        h->kv_valid = 0;
        return 0;
    });
}

int argle_step(vk_gpe* h, int want_res, const double* noise = nullptr)
{
    if (noise) HIPCHK(hipMemcpyAsync(h->Xn, noise, f2(h) * sizeof(cplx), hipMemcpyDefault, h->stream));
    return dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        const double sc = scale_of(h);
        const int parts = h->have_part && h->p.np > 0;
        const int rs = parts && h->rs_part;
        // the obstacles' potential: from the grid up to 1024^2; from 2048^2 on from
        // the windows, as RK4 (with 8 obstacles 4096^2 745 us a step from the grid,
        // whose 134 MB P3 would read, and 702 so)
        constexpr bool GRID = C::N < 2048;
        constexpr int PMR = GRID ? 8 : 4;
        if (GRID && rs) {
            int rc = particle_field(h);
            if (rc) return rc;
        }
        const vk::P3Part pa = p3part(h);
        if (parts && !rs && !h->kv_valid) {
            particle_kv(h, C::TC * h->geo.Pp);
            h->kv_valid = 1;
        }
        const bool adv = h->adv_tg || h->adv_field || h->adv_vx != 0.0 || h->adv_vy != 0.0;
        constexpr int GC = p4_cols<C>();
        if (adv)   // i ky kpsi -> Hdy (all columns)
            colg_launch<C, GC>(h, PK_OTHER, h->NP, vk::k_col_inv<C, GC>, (const cplx*)h->K0, h->Hdy,
                               (const cplx*)h->tw, h->geo, 0, 2);
        const double L = 8.0 * std::atan(1.0), dvol = (L / h->N) * (L / h->N);
        if (h->sgle) {
            // this step's noise (the caller's normals, or the generator's next
            // draw; src/gpe.f90:150-164) and P1
            const vk::NoiseArgs na{noise ? h->Xn : nullptr, h->Hd, h->sg_draw, h->sg_seed, 1.0 / std::sqrt(dvol),
                                   std::sqrt((1.0 / (2.0 * h->p.alpha)) * h->sg_beta), h->omega_dev};
            if (!noise) h->sg_draw++;
            const size_t lds = (size_t)C::TR * C::ROWRS * sizeof(double);
            auto k = vk::k_p1_noise<C>;
            set_lds(k, lds);
            ev_begin(h);
            hipLaunchKernelGGL(k, dim3(2 * (C::N / C::TR)), dim3(C::ROWT), lds, h->stream, (const cplx*)h->Hpsi,
                               h->Hrho, (const cplx*)h->tw, h->geo, sc, h->Xs, h->npart, na);
            ev_end(h, PK_P1);
        } else {
            row_launch<C>(h, PK_P1, vk::k_p1x<C>, (const cplx*)h->Hpsi, h->Hrho, (const cplx*)h->tw, h->geo, 0, sc,
                          h->Xs);
        }
        p2_launch<C>(h, h->Hrho, h->HV, (const cplx*)h->KV, h->Krho,
                      (const cplx*)h->tw, h->geo, (parts && !rs) ? 1 : 0);
        if (adv) {
            const vk::AdvArgs aa{h->adv_tg, h->adv_vx, h->adv_vy, 0.25 / h->p.alpha, sc,
                                 h->adv_field ? (const double*)h->Ux : nullptr,
                                 h->adv_field ? (const double*)h->Uy : nullptr};
            row_launch_x<C>(h, PK_P3, p3_extra(h),
                            !parts ? vk::k_p3a<C, 0> : (rs ? vk::k_p3a<C, PMR> : vk::k_p3a<C, 1>), (const cplx*)h->Hrho,
                            (const cplx*)h->HV, (const cplx*)h->Hpsi, (const cplx*)h->Xs, (const cplx*)h->Hdy, h->HN,
                            (const cplx*)h->tw, h->geo, -h->p.g * sc, -sc, -1.0, pa, aa);
        } else {
            auto k3 = !parts ? vk::k_p3x<C, 0> : (rs ? vk::k_p3x<C, PMR> : vk::k_p3x<C, 1>);
            row_launch_x<C>(h, PK_P3, p3_extra(h), k3, (const cplx*)h->Hrho, (const cplx*)h->HV, (const cplx*)h->Xs,
                            h->HN, (const cplx*)h->tw, h->geo, 0, -h->p.g * sc, -sc, -1.0, pa);
        }
        vk::ArgleArgs a{h->p.alpha, h->p.omega, h->p.dt, want_res};
        if (h->sgle) {
            a.Hn = h->Hd;
            a.nsum = h->npart;
            a.om = h->omega_dev;
            a.dvol = dvol;
            a.nuN = h->sg_nuN;
            a.L2 = L * L;
            a.g = h->geo;
            a.sdt = std::sqrt(h->p.dt);
            a.ktrunc2 = h->sg_ktrunc > 0.0 ? h->sg_ktrunc * h->sg_ktrunc : 0.0;
        }
        // the columns per workgroup of P4 (two of four at 4096^2)
        constexpr int GA = p4_cols<C>();
        static_assert(GA == C::TC || C::NP % 8 == 0, "column groups need whole groups of 8 panels");
        colg_launch<C, GA>(h, PK_ARG4, h->NP, h->sgle ? vk::k_a4<C, GA, true> : vk::k_a4<C, GA>, (const cplx*)h->HN, h->Hpsi, h->K0,
                           (const cplx*)h->tw, a, h->part);
        if (want_res)
            hipLaunchKernelGGL(vk::k_reduce_fixed, dim3(1), dim3(256), 0, h->stream, (const double*)h->part,
                               h->NP * (C::TC / GA), 2, h->dsum);
        return 0;
    });
}

// ---- diagnostics ---------------------------------------------------------------

int diag_setup(vk_gpe* h, hipStream_t st)
{
    if (h->diag_ready) return 0;
    int rc = make_field(h, &h->Hd, st);
    if (rc) return rc;
    h->diag_ready = 1;
    return 0;
}

// Scratch of the diagnostics: fields that hold nothing between steps.  K2
// (2 N^2 doubles) takes the spectra's column partials and the row sums.
double* diag_part(const vk_gpe* h) { return reinterpret_cast<double*>(h->K2); }
double* diag_rsum(const vk_gpe* h)
{
    return diag_part(h) + (size_t)(h->N / 3 + 1) * 6 * vk::spec_shells(h->N);
}
size_t diag_results(const vk_gpe* h) { return 8 + 6 * (size_t)(h->nshell + 1); }
vk::SpecArgs spec_args(const vk_gpe* h)
{
    const double en = 1.0 / ((double)h->N * (double)h->N);
    return vk::SpecArgs{h->p.alpha, h->p.g, en * en, h->N, h->nshell};
}
vk::DiagArgs diag_args(const vk_gpe* h, int has_v)
{
    return vk::DiagArgs{h->p.alpha, h->p.omega, h->p.g, (double)1e-30f, h->N, has_v};
}

// the diagnostics' device work on h->stream: the energy sums and the six
// spectra to out (8 + 6 (nshell + 1) doubles the device can write), particle
// diagnostics in the particle state
int diag_launch(vk_gpe* h, double* out)
{
    int rc = diag_setup(h, h->stream);
    if (rc) return rc;
    if ((rc = ensure_any(h))) return rc;
    const double sc = scale_of(h);
    const int pl = h->hstate == 2 ? 1 : 0;
    const int parts = h->have_part && h->p.np > 0;
    const int Kp = h->TC * h->geo.Pp;
    cplx *H1 = h->HN, *H2 = h->Xs;
    if ((rc = col_inv(h, h->K0, h->Hd, pl, 2))) return rc;   // i ky kpsi
    if (parts) particle_kv(h, Kp);
    rc = dispatch(h->N, [&](auto n) {
        using C = CfgN<decltype(n)::value>;
        using C1 = std::conditional_t<(C::N >= 2048), CfgTR1<C>, C>;
        const cplx* tw = h->tw;
        row_launch<C1>(h, PK_OTHER, vk::k_p1d<C1>, (const cplx*)h->Hpsi, h->Hrho, tw, h->geo, pl, sc);
        p2_launch<C>(h, h->Hrho, h->HV, (const cplx*)h->KV, h->Krho, tw, h->geo, parts ? 3 : 2);
        row_launch<C1>(h, PK_OTHER, vk::k_diag_row<C1>, (const cplx*)h->Hpsi, (const cplx*)h->Hd, (const cplx*)h->Hrho,
                       (const cplx*)h->HV, H1, H2, tw, h->geo, pl, sc, diag_args(h, parts), diag_rsum(h));
        using CC = std::conditional_t<(C::N >= 256), vk::CfgD<C::N, true>, C>;
        constexpr int G = CC::G;
        colg_launch<CC, G>(h, PK_OTHER, h->geo.Pp, vk::k_diag_col<CC, G>, H1, (const cplx*)H2,
                          (const cplx*)h->K0, (const cplx*)h->Krho, tw, h->geo, diag_part(h));
        return 0;
    });
    if (rc) return rc;
    hipLaunchKernelGGL(vk::k_spec_reduce, dim3(h->nshell / 64 + 1, 7), dim3(64 * vk::SPEC_G), 0, h->stream,
                       (const double*)diag_part(h), (const double*)diag_rsum(h), spec_args(h), out);
    if (parts) particle_forces(h, h->Krho, Kp, 1, 0);
    return 0;
}

// the diagnostics from the sums s[8], the spectra sp[6 (nshell + 1)] and
// the particle diagnostics dg[4] of diag_launch
void diag_final(const vk_gpe* h, const double* s, const double* sp, const double* dg, double* scal, double* spec,
                double* pscal)
{
    const double pi = 4.0 * std::atan(1.0);
    const int parts = h->have_part && h->p.np > 0;
    const double L = 2.0 * pi, dx = L / h->N, dvol = dx * dx, L2 = L * L, al = h->p.alpha;
    // final factors (src/diagnostics.f90:105-106,189-207,244)
    const double egrad = 2.0 * al * s[2] * dvol / L2;
    const double echem = 2.0 * al * s[3] * dvol / L2;
    const double eintr = 2.0 * al * s[4] * dvol / L2;
    if (scal) {
        scal[0] = egrad;
        scal[1] = echem;
        scal[2] = eintr;
        scal[3] = egrad + eintr;
        scal[4] = s[6] * dvol;
        scal[5] = 2.0 * al * s[0] * dvol / L2;
        scal[6] = 2.0 * al * s[1] * dvol / L2;
        scal[7] = sp[5 * (h->nshell + 1) + 0];
    }
    if (spec) std::memcpy(spec, sp, sizeof(double) * 6 * (h->nshell + 1));
    if (pscal) {
        for (int i = 0; i < 5; ++i) pscal[i] = 0.0;
        if (parts) {
            pscal[0] = 2.0 * al * s[5] * dvol / L2;
            pscal[1] = dg[0];
            pscal[2] = dg[1];
            pscal[3] = dg[2];
            pscal[4] = dg[3];
        }
    }
}

int diagnostics(vk_gpe* h, double* scal, double* spec, double* pscal)
{
    // results in pinned memory, which the last kernel writes
    if (!h->hres) HIPCHK(hipHostMalloc((void**)&h->hres, diag_results(h) * sizeof(double)));
    int rc = diag_launch(h, h->hres);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    double dg[4] = {};
    if (h->have_part && h->p.np > 0)
        HIPCHK(hipMemcpy(dg, h->pst + 28 * h->p.np, sizeof(dg), hipMemcpyDeviceToHost));
    diag_final(h, h->hres, h->hres + 8, dg, scal, spec, pscal);
    return 0;
}

}  // namespace

// =============================================================================
// C ABI
// =============================================================================

extern "C" {

const char* vk_last_error(void) { return g_err.c_str(); }
const char* vk_version(void) { return "vikshobha-mi355x 0.1 (gfx950)"; }

int vk_nshell(int N)
{
    const float a = 1.414f * (float)N;   // default-real literal (src/mod_grid.f90:77)
    return (int)((double)a / 2.0) + 1;
}

int vk_gpe_params_init(vk_gpe_params* p, int N, double dt, double xi_in, double csound, double rho_avg, double disp)
{
    if (!p || N < 32) return fail(VK_ERR_ARG, "params_init: bad arguments");
    std::memset(p, 0, sizeof(*p));
    const double pi = 4.0 * std::atan(1.0);
    const double L = 2.0 * pi;
    const double dx = L / N;
    p->N = N;
    p->dt = dt;
    p->xi = xi_in * dx;
    p->alpha = csound * p->xi * std::sqrt(rho_avg / 2.0);
    p->g = (csound * csound) / (2.0 * p->alpha);
    p->omega = p->g;
    p->disp = disp;
    p->mass = 1.0;
    p->force_dealias = 1;
    return 0;
}

int vk_gpe_create(vk_gpe** out, const vk_gpe_params* p)
{
    if (!out || !p) return fail(VK_ERR_ARG, "create: null argument");
    *out = nullptr;
    const int N = p->N;
    if (N < 32 || N > 4096 || (N & (N - 1))) return fail(VK_ERR_UNSUPPORTED, "N must be a power of two in [32, 4096]");
    if (p->np < 0 || p->np > 256) return fail(VK_ERR_ARG, "np must be in [0, 256]");
    if (p->np > 0 && !p->force_dealias)
        return fail(VK_ERR_UNSUPPORTED, "force_dealias=0 (no dealiasing of rho-hat in the particle force) is not implemented");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(VK_ERR_HIP, "no ROCm device available");
    vk_gpe* h = new vk_gpe();
    h->p = *p;
    h->N = N;
    h->nshell = vk_nshell(N);
    int TC = 0;
    dispatch(N, [&](auto n) { TC = CfgN<decltype(n)::value>::TC; return 0; });
    h->TC = TC;
    h->NP = N / TC;
    const int M = N / 3;
    h->geo.M = M;
    h->geo.Pp = (M + 1 + TC - 1) / TC;
    h->geo.Pn = (M + TC - 1) / TC;
    h->rs_part = use_real_space(*p);
    h->np_cap = p->np;
    if (h->geo.Pp + h->geo.Pn > h->NP) { h->geo.Pp = h->NP; h->geo.Pn = 0; }
    auto cleanup = [&](int rc) { vk_gpe_destroy(h); return rc; };
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(VK_ERR_HIP, "hipStreamCreate failed"));
    const size_t fb = f2(h) * sizeof(cplx);
    cplx** bufs[] = {&h->K0, &h->K1, &h->K2, &h->Hpsi, &h->Hrho, &h->HN};
    for (auto b : bufs) {
        if (hipMalloc(b, fb) != hipSuccess || hipMemset(*b, 0, fb) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "hipMalloc failed (fields)"));
    }
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&h->ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "device attribute query failed"));
        h->dev = dev;
        if (int rc = scratch_setup(dev)) return cleanup(rc);
        h->p1pf = p1_prefetch_ok(h);
        const char* t1 = std::getenv("VK_P1_TR1");
        const char* t3 = std::getenv("VK_P3_TR1");
        // Measured defaults (4-column panels: 64-byte row pieces), ms per step
        // with 32 particles / without: at 2048^2 one row per workgroup in P1
        // and P3, 0.551 / 0.513 (four rows in P3 0.575 / 0.533, in both 0.637 /
        // 0.588); at 4096^2 one row in P1 and two in P3, 2.019 / 1.997 (one in
        // both 2.087 / 2.038, two in both 2.064 / 2.026).
        // VK_P1_TR1 / VK_P3_TR1 = 0 or 1 override; vk_gpe_autotune_rows
        // times every pair on the device at hand.
        h->tr1_p1 = t1 ? t1[0] == '1' : (N == 4096 || N == 2048);
        h->tr1_p3 = t3 ? t3[0] == '1' : N == 2048;
    }
    if (hipMalloc(&h->Xs, fb) != hipSuccess) return cleanup(fail(VK_ERR_HIP, "hipMalloc failed (psi rows)"));
    if (hipMalloc(&h->tw, sizeof(cplx) * N) != hipSuccess) return cleanup(fail(VK_ERR_HIP, "hipMalloc tw"));
    // twiddles w_k = exp(-2 pi i k/N): long-double sin/cos on the first
    // octant, exact quadrant/octant symmetries elsewhere
    {
        std::vector<double2> tw(N);
        const long double pil = 3.141592653589793238462643383279502884L;
        for (int k = 0; k < N; ++k) {
            const int q = N / 4, quad = k / q;
            int a = k % q, flip = 0;
            if (2 * a > q) { a = q - a; flip = 1; }
            const long double t = 2.0L * pil * (long double)a / (long double)N;
            long double c = cosl(t), s = sinl(t);
            if (flip) { long double tmp = c; c = s; s = tmp; }
            for (int i = 0; i < quad; ++i) { long double tmp = c; c = -s; s = tmp; }
            tw[k] = make_double2((double)c, -(double)s);
        }
        if (hipMemcpy(h->tw, tw.data(), sizeof(double2) * N, hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "twiddle upload"));
    }
    // residual partials: one pair per ARGLE column workgroup (at most one per column)
    if (hipMalloc(&h->part, sizeof(double) * 2 * N) != hipSuccess) return cleanup(fail(VK_ERR_HIP, "hipMalloc part"));
    if (hipMalloc(&h->dsum, sizeof(double) * 8) != hipSuccess) return cleanup(fail(VK_ERR_HIP, "hipMalloc dsum"));
    if (p->np > 0) {
        const int np = p->np;
        cplx** pb[] = {&h->HV, &h->KV, &h->Krho, &h->Vhat};
        for (auto b : pb) {
            if (hipMalloc(b, fb) != hipSuccess || hipMemset(*b, 0, fb) != hipSuccess)
                return cleanup(fail(VK_ERR_HIP, "hipMalloc failed (particles)"));
        }
        // force partials: spectral path 4 per row kx and particle; real-space
        // path 2 per row block, wave and particle
        size_t rows = 0, nw = 0;
        dispatch(N, [&](auto n) {
            using C = CfgN<decltype(n)::value>;
            rows = C::N;                      // one row per block at most
            nw = (C::ROWT + 63) / 64;
            return 0;
        });
        const size_t nfp = std::max((size_t)4 * np * N, 2 * rows * nw * np);
        if (hipMalloc(&h->EX, sizeof(cplx) * np * N) != hipSuccess ||
            hipMalloc(&h->EY, sizeof(cplx) * np * N) != hipSuccess ||
            hipMalloc(&h->fpart, sizeof(double) * nfp) != hipSuccess ||
            hipMalloc(&h->phit, rows * np) != hipSuccess ||
            hipMalloc(&h->pst2, sizeof(double) * 4 * np) != hipSuccess ||
            hipMalloc(&h->pwin, sizeof(int4) * np) != hipSuccess ||
            hipMalloc(&h->ptx, sizeof(double2) * np * N) != hipSuccess ||
            hipMalloc(&h->pty, sizeof(double2) * np * N) != hipSuccess ||
            hipMalloc(&h->pst, sizeof(double) * (30 * np + 8)) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "hipMalloc failed (particle tables)"));
        if (hipMemset(h->pst, 0, sizeof(double) * (30 * np + 8)) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "hipMemset failed (particle state)"));
        if (hipStreamCreateWithFlags(&h->pstream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&h->ev_p3, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&h->ev_ps, hipEventDisableTiming) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "particle stream/events"));
    } else {
        // P2/P3 take these pointers even when unused
        h->HV = h->Hrho;
        h->KV = h->K1;
        h->Krho = h->K1;
    }
    if (hipDeviceSynchronize() != hipSuccess) return cleanup(fail(VK_ERR_HIP, "create: device sync"));
    *out = h;
    return 0;
}

void vk_gpe_destroy(vk_gpe* h)
{
    if (!h) return;
    if (h->stream) hipStreamSynchronize(h->stream);
    cplx* fields[] = {h->K0, h->K1, h->K2, h->Hpsi, h->Hrho, h->HN, h->tw, h->Hd, h->Xs, h->Hdy, h->Xn};
    for (auto f : fields) if (f) hipFree(f);
    for (double* f : {h->Ux, h->Uy, h->omega_dev, h->npart}) if (f) hipFree(f);
    if (h->np_cap > 0) {
        cplx* pf[] = {h->HV, h->KV, h->Krho, h->Vhat, h->EX, h->EY};
        for (auto f : pf) if (f) hipFree(f);
        if (h->fpart) hipFree(h->fpart);
        if (h->phit) hipFree(h->phit);
        if (h->pst2) hipFree(h->pst2);
        if (h->pwin) hipFree(h->pwin);
        if (h->ptx) hipFree(h->ptx);
        if (h->pty) hipFree(h->pty);
        if (h->Vx) hipFree(h->Vx);
        if (h->pst) hipFree(h->pst);
    }
    if (h->Kd0) hipFree(h->Kd0);
    if (h->hres) hipHostFree(h->hres);
    if (h->part) hipFree(h->part);
    if (h->dsum) hipFree(h->dsum);
    if (h->e1R) hipFree(h->e1R);
    for (int k = 0; k < 3; ++k) { if (h->e1map[k]) hipFree(h->e1map[k]); if (h->e1off[k]) hipFree(h->e1off[k]); }
    for (auto e : h->ev) hipEventDestroy(e);
    if (h->pstream) { hipStreamSynchronize(h->pstream); hipStreamDestroy(h->pstream); }
    if (h->ev_p3) hipEventDestroy(h->ev_p3);
    if (h->ev_ps) hipEventDestroy(h->ev_ps);
    if (h->stream) hipStreamDestroy(h->stream);
    delete h;
}

static int sgle_sync_omega(vk_gpe* h);
static int ensure_hdy(vk_gpe* h);

static int need_hd(vk_gpe* h) { return make_field(h, &h->Hd, h->stream); }

static int set_from_xs(vk_gpe* h, int flags)
{
    int rc = fwd2d(h, h->Xs, h->Hd, h->K0, 0);
    if (rc) return rc;
    h->hstate = 0;
    if (flags & VK_SYNC_DEALIAS) {
        if ((rc = ensure_rk4(h))) return rc;
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    return 0;
}

int vk_gpe_set_psi(vk_gpe* h, const double* psi, int flags)
{
    if (!h || !psi) return fail(VK_ERR_ARG, "set_psi: null argument");
    int rc = need_hd(h);
    if (rc) return rc;
    // stream-ordered: a device-to-device hipMemcpy does not block the host and
    // is not ordered against this non-blocking stream
    HIPCHK(hipMemcpyAsync(h->Xs, psi, f2(h) * sizeof(cplx), hipMemcpyDefault, h->stream));
    return set_from_xs(h, flags);
}

int vk_gpe_set_kpsi(vk_gpe* h, const double* kpsi)
{
    if (!h || !kpsi) return fail(VK_ERR_ARG, "set_kpsi: null argument");
    HIPCHK(hipMemcpyAsync(h->K0, kpsi, f2(h) * sizeof(cplx), hipMemcpyDefault, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    h->hstate = 0;
    return 0;
}

// whether a kernel on the handle's stream may write `bytes` at p
static bool kernel_target(const vk_gpe* h, const void* p, size_t bytes)
{
    hipPointerAttribute_t a;
    hipDeviceptr_t base = nullptr;
    size_t n = 0;
    if (hipPointerGetAttributes(&a, p) == hipSuccess && a.type == hipMemoryTypeDevice &&
        hipMemGetAddressRange(&base, &n, const_cast<void*>(p)) == hipSuccess)
        return vk::kernel_writable((uintptr_t)p, bytes, vk::Target{true, a.device, (uintptr_t)base, n}, h->dev);
    (void)hipGetLastError();
    return false;
}

// psi goes straight into a caller's device buffer (16 us a 128..512^2 field
// instead of 35 with a copy and a wait between); other memory through Xs
int vk_gpe_get_psi(vk_gpe* h, double* psi, double* kpsi)
{
    if (!h) return fail(VK_ERR_ARG, "get_psi: null handle");
    int rc;
    if (psi) {
        const size_t bytes = f2(h) * sizeof(cplx);
        // an error of the steps queued so far: kernel_target's query leaves and
        // clears one of its own for host memory
        HIPCHK(hipGetLastError());
        const bool direct = kernel_target(h, psi, bytes);
        if (!direct && (rc = need_hd(h))) return rc;
        if ((rc = ensure_any(h))) return rc;
        cplx* x = direct ? reinterpret_cast<cplx*>(psi) : h->Xs;
        if ((rc = row_inv(h, h->Hpsi, x, h->hstate == 2 ? 1 : 0, scale_of(h)))) return rc;
        HIPCHK(hipGetLastError());
        if (!direct) HIPCHK(hipMemcpyAsync(psi, x, bytes, hipMemcpyDefault, h->stream));
        HIPCHK(hipStreamSynchronize(h->stream));
    }
    if (kpsi) {
        HIPCHK(hipMemcpyAsync(kpsi, h->K0, f2(h) * sizeof(cplx), hipMemcpyDefault, h->stream));
        HIPCHK(hipStreamSynchronize(h->stream));
    }
    return 0;
}

int vk_gpe_rk4_steps_async(vk_gpe* h, int nsteps)
{
    if (!h || nsteps < 0) return fail(VK_ERR_ARG, "rk4_steps: bad arguments");
    int rc = prep_rk4(h);
    if (rc) return rc;
    for (int i = 0; i < nsteps; ++i)
        if ((rc = rk4_step(h))) return rc;
    return 0;
}

int vk_gpe_rk4_steps(vk_gpe* h, int nsteps)
{
    int rc = vk_gpe_rk4_steps_async(h, nsteps);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    return 0;
}

int vk_gpe_argle_steps(vk_gpe* h, int nsteps, double* residual)
{
    if (!h || nsteps < 0) return fail(VK_ERR_ARG, "argle_steps: bad arguments");
    int rc = ensure_full(h);
    if (rc) return rc;
    for (int i = 0; i < nsteps; ++i)
        if ((rc = argle_step(h, residual && i == nsteps - 1))) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    if ((rc = sgle_sync_omega(h))) return rc;
    if (residual && nsteps > 0) {
        double r[2];
        HIPCHK(hipMemcpy(r, h->dsum, sizeof(r), hipMemcpyDeviceToHost));
        *residual = std::sqrt(r[0]) / (h->p.dt * std::sqrt(r[1]));
    }
    return 0;
}

int vk_gpe_argle_until(vk_gpe* h, double tol, int max_steps, int check_every, int* steps_out, double* residual)
{
    if (!h || max_steps < 0 || check_every <= 0 || tol <= 0.0) return fail(VK_ERR_ARG, "argle_until: bad arguments");
    int rc = ensure_full(h);
    if (rc) return rc;
    int done = 0;
    double res = INFINITY;
    while (done < max_steps) {
        const int n = std::min(check_every, max_steps - done);
        for (int i = 0; i < n; ++i)
            if ((rc = argle_step(h, i == n - 1))) return rc;
        done += n;
        double r[2];
        HIPCHK(hipMemcpyAsync(r, h->dsum, sizeof(r), hipMemcpyDeviceToHost, h->stream));
        HIPCHK(hipStreamSynchronize(h->stream));
        res = std::sqrt(r[0]) / (h->p.dt * std::sqrt(r[1]));
        if (!(res > tol)) break;   // converged (or NaN: stop and report)
    }
    HIPCHK(hipGetLastError());
    if ((rc = sgle_sync_omega(h))) return rc;
    if (steps_out) *steps_out = done;
    if (residual) *residual = res;
    return 0;
}

int vk_gpe_diagnostics(vk_gpe* h, double* scal, double* spec, double* pscal)
{
    if (!h) return fail(VK_ERR_ARG, "diagnostics: null handle");
    return diagnostics(h, scal, spec, pscal);
}

// particle_potential (src/gpe_particle.f90:3-90): V of one particle at the
// origin on the grid, forward transform, dealias -> Vhat
static int particle_potential(vk_gpe* h)
{
    const double pi = 4.0 * std::atan(1.0);
    const double L = 2.0 * pi, dx = L / h->N, c1 = 2 * pi / (2.0 * L);
    hipLaunchKernelGGL(vk::k_pot_x, dim3(1024), dim3(256), 0, h->stream, h->Xs, h->N, dx, c1, h->p.V0, h->p.d);
    int rc = fwd2d(h, h->Xs, h->Hd, h->Vhat, 1);
    if (rc) return rc;
    h->have_part = 1;
    return 0;
}

int vk_gpe_particles_set(vk_gpe* h, const double* pos, const double* vel, const double* fext)
{
    if (!h) return fail(VK_ERR_ARG, "particles_set: null handle");
    const int np = h->p.np;
    if (np <= 0) return fail(VK_ERR_STATE, "particles_set: handle created with np = 0");
    int rc = need_hd(h);
    if (rc) return rc;
    // steps queued by vk_gpe_rk4_steps_async read and write the particle
    // state (the side-stream updates are joined into h->stream at the end of
    // every step): the copies go on h->stream, after them
    if (pos) HIPCHK(hipMemcpyAsync(h->pst, pos, sizeof(double) * 2 * np, hipMemcpyDefault, h->stream));
    if (vel) HIPCHK(hipMemcpyAsync(h->pst + 2 * np, vel, sizeof(double) * 2 * np, hipMemcpyDefault, h->stream));
    if (fext) HIPCHK(hipMemcpyAsync(h->pst + 4 * np, fext, sizeof(double) * 2 * np, hipMemcpyDefault, h->stream));
    if (!h->have_part && (rc = particle_potential(h))) return rc;
    particles_moved(h);
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    return 0;
}

}  // extern "C"

// accessors for the library's other translation units (not part of the C ABI)
cplx* vk_internal_kpsi(vk_gpe* h) { return h ? h->K0 : nullptr; }
int vk_internal_N(const vk_gpe* h) { return h ? h->N : 0; }
hipStream_t vk_internal_stream(const vk_gpe* h) { return h ? h->stream : nullptr; }

extern "C" {

int vk_gpe_set_advection(vk_gpe* h, int taylor_green, double vnx, double vny)
{
    if (!h || (taylor_green != 0 && taylor_green != 1) || !std::isfinite(vnx) || !std::isfinite(vny))
        return fail(VK_ERR_ARG, "set_advection: taylor_green must be 0 or 1 and the velocity finite");
    HIPCHK(hipStreamSynchronize(h->stream));
    if (taylor_green || vnx != 0.0 || vny != 0.0) {
        int rc = ensure_hdy(h);
        if (rc) return rc;
    }
    h->adv_tg = taylor_green;
    h->adv_vx = vnx;
    h->adv_vy = vny;
    return 0;
}

static int ensure_hdy(vk_gpe* h) { return make_field(h, &h->Hdy, h->stream); }

static int ensure_field_bufs(vk_gpe* h)
{
    if (!h->Ux) HIPCHK(hipMalloc(&h->Ux, f2(h) * sizeof(double)));
    if (!h->Uy) HIPCHK(hipMalloc(&h->Uy, f2(h) * sizeof(double)));
    return ensure_hdy(h);
}

int vk_gpe_set_advection_field(vk_gpe* h, const double* ux, const double* uy)
{
    if (!h || (!ux) != (!uy)) return fail(VK_ERR_ARG, "set_advection_field: both components or neither");
    HIPCHK(hipStreamSynchronize(h->stream));
    if (!ux) {
        h->adv_field = 0;
        return 0;
    }
    int rc = ensure_field_bufs(h);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(h->Ux, ux, f2(h) * sizeof(double), hipMemcpyDefault, h->stream));
    HIPCHK(hipMemcpyAsync(h->Uy, uy, f2(h) * sizeof(double), hipMemcpyDefault, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    h->adv_field = 1;
    return 0;
}

int vk_gpe_set_vortex_advection(vk_gpe* h, int nv, const double* xs, const double* ys, const int* qs, int nimg)
{
    if (!h || nv <= 0 || !xs || !ys || !qs || nimg < 0) return fail(VK_ERR_ARG, "set_vortex_advection: bad arguments");
    for (int j = 0; j < nv; ++j)
        if (qs[j] != 1 && qs[j] != -1) return fail(VK_ERR_ARG, "set_vortex_advection: charges must be +-1");
    int rc = ensure_field_bufs(h);
    if (rc) return rc;
    double* d = nullptr;
    HIPCHK(hipMalloc(&d, sizeof(double) * 2 * nv + sizeof(int) * nv));
    HIPCHK(hipMemcpy(d, xs, sizeof(double) * nv, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d + nv, ys, sizeof(double) * nv, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d + 2 * nv, qs, sizeof(int) * nv, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(vk::k_vortex_velocity, dim3(1024), dim3(256), 0, h->stream, h->Ux, h->Uy, h->N, nv,
                       (const double*)d, (const double*)(d + nv), (const int*)(d + 2 * nv), h->p.xi, nimg,
                       h->p.alpha);
    const hipError_t e = hipStreamSynchronize(h->stream);
    hipFree(d);
    HIPCHK(e);
    HIPCHK(hipGetLastError());
    h->adv_field = 1;
    return 0;
}

int vk_vortex_velocity_host(int N, int nv, const double* xs, const double* ys, const int* qs, double xi,
                            double alpha, int nimg, double* ux, double* uy)
{
    if (N <= 0 || nv <= 0 || !xs || !ys || !qs || !ux || !uy || nimg < 0)
        return fail(VK_ERR_ARG, "vortex_velocity_host: bad arguments");
    const double dx = 2.0 * 3.14159265358979323846 / N;
    for (int j = 0; j < N; ++j)
        for (int i = 0; i < N; ++i)
            vk::vortex_velocity_point(i * dx, j * dx, nv, xs, ys, qs, xi, nimg, alpha, ux + (size_t)j * N + i,
                                      uy + (size_t)j * N + i);
    return 0;
}

int vk_gpe_set_sgle(vk_gpe* h, int on, double oneybeta, double nuN, double chempot0, double ktrunc,
                    unsigned long long seed)
{
    if (!h || (on != 0 && on != 1) || !(oneybeta >= 0.0) || !std::isfinite(nuN) || !std::isfinite(chempot0) ||
        !std::isfinite(ktrunc) || !std::isfinite(oneybeta))
        return fail(VK_ERR_ARG, "set_sgle: on must be 0 or 1, oneybeta >= 0 and the parameters finite");
    HIPCHK(hipStreamSynchronize(h->stream));
    if (!on) {
        h->sgle = 0;
        return 0;
    }
    int rc = need_hd(h);
    if (rc) return rc;
    if (!h->Xn) HIPCHK(hipMalloc(&h->Xn, f2(h) * sizeof(cplx)));
    if (!h->omega_dev) HIPCHK(hipMalloc(&h->omega_dev, 2 * sizeof(double)));
    if (!h->npart) HIPCHK(hipMalloc(&h->npart, sizeof(double) * h->N));
    const double om[2] = {chempot0, chempot0};   // before the last step, after it
    HIPCHK(hipMemcpy(h->omega_dev, om, sizeof(om), hipMemcpyHostToDevice));
    h->p.omega = chempot0;
    h->sgle = 1;
    h->sg_beta = oneybeta;
    h->sg_nuN = nuN;
    h->sg_ktrunc = ktrunc;
    h->sg_seed = seed;
    h->sg_draw = 0;
    return 0;
}

// the chemical potential the SGLE steps have reached, into the handle's
// parameters (RK4 after SGLE runs at it, as the reference's omega_chem)
static int sgle_sync_omega(vk_gpe* h)
{
    if (!h->sgle) return 0;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipMemcpy(&h->p.omega, h->omega_dev + 1, sizeof(double), hipMemcpyDeviceToHost));
    if (h->e1R) {
        const vk::EnsReal x = single_entry(h);
        HIPCHK(hipMemcpy(h->e1R, &x, sizeof(x), hipMemcpyHostToDevice));
    }
    return 0;
}

int vk_gpe_get_chempot(vk_gpe* h, double* omega)
{
    if (!h || !omega) return fail(VK_ERR_ARG, "get_chempot: null argument");
    int rc = sgle_sync_omega(h);
    if (rc) return rc;
    *omega = h->p.omega;
    return 0;
}

int vk_gpe_argle_step_noise(vk_gpe* h, const double* noise_xy, double* residual)
{
    if (!h || !noise_xy) return fail(VK_ERR_ARG, "argle_step_noise: null argument");
    if (!h->sgle) return fail(VK_ERR_STATE, "argle_step_noise: SGLE is off (vk_gpe_set_sgle)");
    int rc = ensure_full(h);
    if (rc) return rc;
    if ((rc = argle_step(h, residual != nullptr, noise_xy))) return rc;
    if ((rc = sgle_sync_omega(h))) return rc;
    HIPCHK(hipGetLastError());
    if (residual) {
        double r[2];
        HIPCHK(hipMemcpy(r, h->dsum, sizeof(r), hipMemcpyDeviceToHost));
        *residual = std::sqrt(r[0]) / (h->p.dt * std::sqrt(r[1]));
    }
    return 0;
}

int vk_sgle_noise(vk_gpe* h, unsigned long long draw, double* out_xy)
{
    if (!h || !out_xy) return fail(VK_ERR_ARG, "sgle_noise: null argument");
    if (!h->sgle) return fail(VK_ERR_STATE, "sgle_noise: SGLE is off (vk_gpe_set_sgle)");
    hipLaunchKernelGGL(vk::k_sgle_noise, dim3(1024), dim3(256), 0, h->stream, h->Xn, h->N, draw, h->sg_seed);
    HIPCHK(hipMemcpyAsync(out_xy, h->Xn, f2(h) * sizeof(cplx), hipMemcpyDefault, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    return 0;
}

int vk_gpe_set_dt(vk_gpe* h, double dt)
{
    if (!h || !(dt > 0.0) || !std::isfinite(dt)) return fail(VK_ERR_ARG, "set_dt: dt must be positive and finite");
    HIPCHK(hipStreamSynchronize(h->stream));
    h->p.dt = dt;
    if (h->e1R) {
        const vk::EnsReal x = single_entry(h);
        HIPCHK(hipMemcpy(h->e1R, &x, sizeof(x), hipMemcpyHostToDevice));
    }
    return 0;
}

int vk_gpe_set_obstacles(vk_gpe* h, int np, const double* pos, double V0, double d)
{
    if (!h) return fail(VK_ERR_ARG, "set_obstacles: null handle");
    if (np < 0 || np > h->np_cap)
        return fail(VK_ERR_ARG, "set_obstacles: np must be in [0, np of the params the handle was created with]");
    if (np > 0 && (!pos || !(d > 0.0) || !std::isfinite(V0)))
        return fail(VK_ERR_ARG, "set_obstacles: positions, d > 0 and a finite V0 are required");
    int rc = need_hd(h);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    h->p.np = np;
    h->p.V0 = V0;
    h->p.d = d;
    h->rs_part = use_real_space(h->p);
    h->have_part = 0;
    if (np == 0) return 0;
    std::vector<double> st(30 * (size_t)np + 8, 0.0);
    std::copy(pos, pos + 2 * np, st.begin());
    HIPCHK(hipMemcpyAsync(h->pst, st.data(), sizeof(double) * st.size(), hipMemcpyHostToDevice, h->stream));
    if ((rc = particle_potential(h))) return rc;
    particles_moved(h);
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    return 0;
}

int vk_gpe_particles_get(vk_gpe* h, double* pos, double* vel, double* frc)
{
    if (!h) return fail(VK_ERR_ARG, "particles_get: null handle");
    const int np = h->p.np;
    if (np <= 0) return fail(VK_ERR_STATE, "particles_get: handle created with np = 0");
    HIPCHK(hipStreamSynchronize(h->stream));
    if (pos) HIPCHK(hipMemcpy(pos, h->pst, sizeof(double) * 2 * np, hipMemcpyDeviceToHost));
    if (vel) HIPCHK(hipMemcpy(vel, h->pst + 2 * np, sizeof(double) * 2 * np, hipMemcpyDeviceToHost));
    if (frc) HIPCHK(hipMemcpy(frc, h->pst + 26 * np, sizeof(double) * 2 * np, hipMemcpyDeviceToHost));
    return 0;
}

int vk_fft2d(vk_gpe* h, int dir, const double* in, double* out)
{
    if (!h || !in || !out || (dir != -1 && dir != 1)) return fail(VK_ERR_ARG, "fft2d: bad arguments");
    int rc = need_hd(h);
    if (rc) return rc;
    if (!h->Kd0) HIPCHK(hipMalloc(&h->Kd0, f2(h) * sizeof(cplx)));
    const size_t fb = f2(h) * sizeof(cplx);
    if (dir < 0) {
        HIPCHK(hipMemcpyAsync(h->Xs, in, fb, hipMemcpyHostToDevice, h->stream));
        if ((rc = fwd2d(h, h->Xs, h->Hd, h->Kd0, 0))) return rc;
        HIPCHK(hipStreamSynchronize(h->stream));
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpy(out, h->Kd0, fb, hipMemcpyDeviceToHost));
    } else {
        HIPCHK(hipMemcpy(h->Kd0, in, fb, hipMemcpyHostToDevice));
        if ((rc = col_inv(h, h->Kd0, h->Hd, 0, 0))) return rc;
        if ((rc = row_inv(h, h->Hd, h->Xs, 0, scale_of(h)))) return rc;
        HIPCHK(hipStreamSynchronize(h->stream));
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpy(out, h->Xs, fb, hipMemcpyDeviceToHost));
    }
    return 0;
}

// The transforms of vk_fft2d between caller-owned device buffers, with the
// half-spectral intermediate in the static scratch instead of library
// memory: no allocation of any kind.  Stream-ordered on the handle's stream
// (returns once the launches are queued).
int vk_fft2d_noalloc(vk_gpe* h, int dir, const double* in, double* out)
{
    if (!h || !in || !out || (dir != -1 && dir != 1) || (const void*)in == (const void*)out)
        return fail(VK_ERR_ARG, "fft2d_noalloc: bad arguments (distinct device buffers, dir = -1 or +1)");
    if (h->N > VK_NOALLOC_MAX_N)
        return fail(VK_ERR_UNSUPPORTED, "fft2d_noalloc: N = " + std::to_string(h->N) + " exceeds the " +
                                            std::to_string(VK_NOALLOC_MAX_N) + "^2 scratch");
    for (const void* q : {(const void*)in, (const void*)out}) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, q) != hipSuccess || a.type != hipMemoryTypeDevice) {
            (void)hipGetLastError();
            return fail(VK_ERR_ARG, "fft2d_noalloc: in and out must be device memory");
        }
    }
    cplx* H = g_scratch_ptr[h->dev];
    if (!H) return fail(VK_ERR_STATE, "fft2d_noalloc: scratch not set up on this device");
    const cplx* ci = reinterpret_cast<const cplx*>(in);
    cplx* co = reinterpret_cast<cplx*>(out);
    int rc;
    if (dir < 0) rc = fwd2d(h, ci, H, co, 0);
    else if (!(rc = col_inv(h, ci, H, 0, 0))) rc = row_inv(h, H, co, 0, scale_of(h));
    if (rc) return rc;
    HIPCHK(hipGetLastError());
    return 0;
}

int vk_ic_vortices_host(int N, int nv, const double* xs, const double* ys, const int* qs, double xi, int nimg,
                        double* psi)
{
    if (N < 2 || nv < 0 || !psi || (nv > 0 && (!xs || !ys || !qs))) return fail(VK_ERR_ARG, "ic: bad arguments");
    const double dx = 2.0 * 3.14159265358979323846 / N;
    for (int iy = 0; iy < N; ++iy)
        for (int ix = 0; ix < N; ++ix) vk::ic_point(ix * dx, iy * dx, nv, xs, ys, qs, xi, nimg, psi + 2 * ((size_t)iy * N + ix));
    return 0;
}

int vk_gpe_set_ic_vortices(vk_gpe* h, int nv, const double* xs, const double* ys, const int* qs, int nimg, int flags)
{
    if (!h || nv < 0 || (nv > 0 && (!xs || !ys || !qs))) return fail(VK_ERR_ARG, "set_ic_vortices: bad arguments");
    int rc = need_hd(h);
    if (rc) return rc;
    double *dx = nullptr, *dy = nullptr;
    int* dq = nullptr;
    const int n = nv > 0 ? nv : 1;
    HIPCHK(hipMalloc(&dx, sizeof(double) * n));
    HIPCHK(hipMalloc(&dy, sizeof(double) * n));
    HIPCHK(hipMalloc(&dq, sizeof(int) * n));
    if (nv > 0) {
        HIPCHK(hipMemcpy(dx, xs, sizeof(double) * nv, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(dy, ys, sizeof(double) * nv, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(dq, qs, sizeof(int) * nv, hipMemcpyHostToDevice));
    }
    hipLaunchKernelGGL(vk::k_ic, dim3(2048), dim3(256), 0, h->stream, h->Xs, h->N, nv, (const double*)dx,
                       (const double*)dy, (const int*)dq, h->p.xi, nimg);
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    hipFree(dx);
    hipFree(dy);
    hipFree(dq);
    return set_from_xs(h, flags);
}

void* vk_gpe_stream(vk_gpe* h) { return h ? (void*)h->stream : nullptr; }

int vk_pass_kinds(void) { return PK_COUNT; }
const char* vk_pass_name(int kind) { return (kind >= 0 && kind < PK_COUNT) ? kPassNames[kind] : "?"; }

int vk_gpe_pass_times(vk_gpe* h, int nsteps, double* ms_out, int nkinds)
{
    if (!h || nsteps <= 0 || !ms_out) return fail(VK_ERR_ARG, "pass_times: bad arguments");
    int rc = prep_rk4(h);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    h->timing = true;
    h->evn = 0;
    h->evkind.clear();
    for (int i = 0; i < nsteps && !rc; ++i) rc = rk4_step(h);
    h->timing = false;
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipGetLastError());
    std::vector<double> sum(PK_COUNT, 0.0);
    std::vector<int> cnt(PK_COUNT, 0);
    for (size_t i = 0; i < h->evkind.size(); ++i) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, h->ev[2 * i], h->ev[2 * i + 1]));
        sum[h->evkind[i]] += ms;
        cnt[h->evkind[i]]++;
    }
    for (int k = 0; k < nkinds && k < PK_COUNT; ++k) ms_out[k] = cnt[k] ? sum[k] / cnt[k] : 0.0;
    return 0;
}

int vk_gpe_set_row_variants(vk_gpe* h, int p1, int p3)
{
    if (!h || p1 < 0 || p1 > 2 || p3 < 0 || p3 > 1) return fail(VK_ERR_ARG, "set_row_variants: bad arguments");
    if (h->N < 2048) return fail(VK_ERR_UNSUPPORTED, "set_row_variants: the row-pass variants exist for N >= 2048 only");
    if (p1 == 2 && !p1_prefetch_fits(h))
        return fail(VK_ERR_UNSUPPORTED, "set_row_variants: the prefetching P1 does not fit this size or device");
    HIPCHK(hipStreamSynchronize(h->stream));
    h->p1pf = p1 == 2;
    h->tr1_p1 = p1 == 1;
    h->tr1_p3 = p3;
    return 0;
}

int vk_gpe_get_row_variants(vk_gpe* h, int* p1, int* p3)
{
    if (!h) return fail(VK_ERR_ARG, "get_row_variants: null");
    if (p1) *p1 = h->p1pf ? 2 : (h->tr1_p1 ? 1 : 0);
    if (p3) *p3 = h->tr1_p3;
    return 0;
}

int vk_gpe_autotune_rows(vk_gpe* h, int nsteps, int* choice, double* ms_out)
{
    if (!h || nsteps <= 0) return fail(VK_ERR_ARG, "autotune_rows: bad arguments");
    if (h->N < 2048) return fail(VK_ERR_UNSUPPORTED, "autotune_rows: the row-pass variants exist for N >= 2048 only");
    int rc = ensure_rk4(h);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    // save the state: kpsi, its y-inverse, the particle state
    const size_t nf = f2(h), npst = h->pst ? (size_t)30 * h->np_cap + 8 : 0;
    cplx* sv = nullptr;
    double* sp = nullptr;
    HIPCHK(hipMalloc(&sv, 2 * nf * sizeof(cplx)));
    if (npst && hipMalloc(&sp, npst * sizeof(double)) != hipSuccess) {
        hipFree(sv);
        return fail(VK_ERR_HIP, "autotune_rows: hipMalloc");
    }
    auto release = [&]() { hipFree(sv); if (sp) hipFree(sp); };
    auto copy = [&](bool save) -> int {
        HIPCHK(hipMemcpyAsync(save ? sv : h->K0, save ? h->K0 : sv, nf * sizeof(cplx), hipMemcpyDeviceToDevice,
                              h->stream));
        HIPCHK(hipMemcpyAsync(save ? sv + nf : h->Hpsi, save ? h->Hpsi : sv + nf, nf * sizeof(cplx),
                              hipMemcpyDeviceToDevice, h->stream));
        if (npst)
            HIPCHK(hipMemcpyAsync(save ? sp : h->pst, save ? h->pst : sp, npst * sizeof(double),
                                  hipMemcpyDeviceToDevice, h->stream));
        HIPCHK(hipStreamSynchronize(h->stream));
        return 0;
    };
    if ((rc = copy(true))) { release(); return rc; }
    hipEvent_t a = nullptr, b = nullptr;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) {
        release();
        return fail(VK_ERR_HIP, "autotune_rows: events");
    }
    const int keep1 = h->p1pf ? 2 : (h->tr1_p1 ? 1 : 0), keep3 = h->tr1_p3;
    double best = 1e300;
    int b1 = keep1, b3 = keep3;
    for (int p1 = 0; p1 <= 2 && !rc; ++p1)
        for (int p3 = 0; p3 <= 1 && !rc; ++p3) {
            if (ms_out) ms_out[2 * p1 + p3] = -1.0;
            if (p1 == 2 && !p1_prefetch_fits(h)) continue;
            h->p1pf = p1 == 2;
            h->tr1_p1 = p1 == 1;
            h->tr1_p3 = p3;
            if ((rc = vk_gpe_rk4_steps_async(h, 1))) break;   // warm
            if (hipEventRecord(a, h->stream) != hipSuccess) { rc = fail(VK_ERR_HIP, "autotune_rows: event"); break; }
            if ((rc = vk_gpe_rk4_steps_async(h, nsteps))) break;
            if (hipEventRecord(b, h->stream) != hipSuccess || hipEventSynchronize(b) != hipSuccess) {
                rc = fail(VK_ERR_HIP, "autotune_rows: event");
                break;
            }
            float ms = 0.f;
            hipEventElapsedTime(&ms, a, b);
            const double per = ms / nsteps;
            if (ms_out) ms_out[2 * p1 + p3] = per;
            if (per < best) { best = per; b1 = p1; b3 = p3; }
        }
    hipEventDestroy(a);
    hipEventDestroy(b);
    h->p1pf = b1 == 2;
    h->tr1_p1 = b1 == 1;
    h->tr1_p3 = b3;
    // the starting state back, also after a failed trial (whose error code
    // is the one returned)
    hipStreamSynchronize(h->stream);
    const int rc2 = copy(false);
    if (!rc) rc = rc2;
    release();
    if (rc) return rc;
    h->hstate = 2;
    h->kv_valid = h->vx_valid = 0;
    if (h->have_part && h->p.np > 0) particles_moved(h);
    if (choice) { choice[0] = b1; choice[1] = b3; }
    return 0;
}

double vk_gpe_pass_bytes(vk_gpe* h, int kind)
{
    if (!h) return 0.0;
    const double F = 16.0 * (double)h->N * (double)h->N;
    const double fp = (double)(h->geo.Pp * h->TC) / h->N;                        // kx >= 0 half columns
    const double fr = (double)((h->geo.Pp + h->geo.Pn) * h->TC) / h->N;         // retained columns
    // retained disk modes
    long long disk = 0;
    for (int kx = -h->N / 2; kx < h->N / 2; ++kx)
        for (int ky = -h->N / 2; ky < h->N / 2; ++ky)
            if (!masked_host(kx, ky, h->N)) ++disk;
    const double D = 16.0 * (double)disk;
    switch (kind) {
    case PK_P1: return F * (fr + fp + 1.0);   // + psi rows written for P3
    case PK_P2: return F * 2.0 * fp;
    case PK_P3: return F * (fp + 1.0 + fr);    // psi rows
    // K accesses per mode, stages 1-4: K0 read + K2 write; K0, K2 read + K1,
    // K2 write; K0, K2 read + K2 write (str2 is not read in stage 3); K0, K1,
    // K2 read + K0 write
    case PK_P4: return F * (fr + fr) + D * (2 + 4 + 3 + 4) / 4.0;
    default: return 0.0;
    }
}

}  // extern "C"

// =============================================================================
// Ensemble of independent realizations (batched launches, graph replay)
// =============================================================================

struct vk_ens {
    std::vector<vk_gpe*> h;
    hipStream_t stream = nullptr;
    vk::EnsReal* dR = nullptr;
    // block maps: 0 row passes (P1, P3), 1 P2, 2 P4; per-size maps for mode 1
    int* dmap[3] = {};
    int* doff[3] = {};
    int nblk[3] = {};
    std::vector<int> sizes;                       // distinct N
    std::map<int, std::vector<int>> size_reals;   // N -> realization ids
    std::map<int, std::array<int*, 6>> smaps;     // N -> {map0, off0, map1, off1, map2, off2}
    std::map<int, std::array<int, 3>> snblk;
    size_t lds[4] = {};                           // max dynamic LDS per pass
    // 0: one launch per pass for all sizes; 1: one per size; 2: per realization;
    // 3: one persistent launch per step (all passes, grid barriers between)
    int mode = 0;
    int use_graph = 1;
    hipGraphExec_t gexec[4] = {};
    unsigned* dbar = nullptr;   // the persistent step's barrier counters
    int* derr = nullptr;        // set by a barrier wait that ran out of time
    int pgrid = 0;              // persistent grid: resident workgroups, multiple of 8
    size_t plds = 0;
    long long plimit = 0;       // barrier wait limit in wall-clock ticks
    double* hstage = nullptr;   // pinned staging of every member's diagnostics
    double* dstage = nullptr;   // the same on the device
    size_t nstage = 0;
    void* dtab = nullptr;       // operand tables of the batched diagnostics
    void* htab = nullptr;       // their pinned host staging
    size_t ntab = 0;
    int synced = 0;
    std::map<int, int> var;                       // N -> shape variant
};

namespace {

// panel geometry of panel width TC (as vk_gpe_create computes it)
Geo geo_of(int N, int TC)
{
    Geo g{};
    const int NP = N / TC, M = N / 3;
    g.M = M;
    g.Pp = (M + 1 + TC - 1) / TC;
    g.Pn = (M + TC - 1) / TC;
    if (g.Pp + g.Pn > NP) { g.Pp = NP; g.Pn = 0; }
    return g;
}

// call f with the shape type of (N, var)
template <class F>
int dispatch_var(int N, int var, F&& f)
{
    switch (N * 2 + var) {
    case 256: return f(vk::CfgE<128, 0>{});
    case 512: return f(vk::CfgE<256, 0>{});
    case 513: return f(vk::CfgE<256, 1>{});
    case 1024: return f(vk::CfgE<512, 0>{});
    case 1025: return f(vk::CfgE<512, 1>{});
    case 2048: return f(vk::CfgE<1024, 0>{});
    case 2049: return f(vk::CfgE<1024, 1>{});
    default: return fail(VK_ERR_UNSUPPORTED, "no such ensemble shape");
    }
}

template <class C> void ens_lds(size_t* l)
{
    l[0] = std::max(l[0], (size_t)C::TR * C::ROWRS * sizeof(double));
    l[1] = std::max(l[1], (size_t)C::TC * C::COLRS * sizeof(double));
    l[2] = std::max(l[2], (size_t)C::TR * C::ROWRS * sizeof(double) + 16);   // f in registers (psi rows)
    l[3] = std::max(l[3], (size_t)C::TC * C::COLRS * sizeof(double));
}

// Block maps for the realizations in ids: for pass kinds 0 (row passes),
// 1 (P2) and 2 (P4), map[b] = realization of block b (runs contiguous, in
// ids order) and off[2r], off[2r+1] = [start, end) of r's run.
int build_maps(const std::vector<vk_gpe*>& hs, const std::vector<int>& ids, int** dmap, int** doff, int* nblk)
{
    for (int k = 0; k < 3; ++k) {
        std::vector<int> map;
        std::vector<int> se(2 * hs.size(), 0);
        for (int r : ids) {
            const vk_gpe* h = hs[r];
            int TR = 0;
            dispatch_var(h->N, h->ens_var, [&](auto c) { TR = decltype(c)::TR; return 0; });
            const Geo& gv = h->ens_var ? h->geo_v : h->geo;
            const int nb = k == 0 ? h->N / TR : (k == 1 ? gv.Pp : gv.Pp + gv.Pn);
            se[2 * r] = (int)map.size();
            for (int b = 0; b < nb; ++b) map.push_back(r);
            se[2 * r + 1] = (int)map.size();
        }
        nblk[k] = (int)map.size();
        HIPCHK(hipMalloc(&dmap[k], sizeof(int) * std::max<size_t>(1, map.size())));
        HIPCHK(hipMalloc(&doff[k], sizeof(int) * se.size()));
        HIPCHK(hipMemcpy(dmap[k], map.data(), sizeof(int) * map.size(), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(doff[k], se.data(), sizeof(int) * se.size(), hipMemcpyHostToDevice));
    }
    return 0;
}

vk::EnsReal ens_entry(const vk_gpe* h)
{
    vk::EnsReal x{};
    x.N = h->N;
    x.var = h->ens_var;
    x.g = h->ens_var ? h->geo_v : h->geo;
    x.K0 = h->K0; x.K1 = h->K1; x.K2 = h->K2; x.Hpsi = h->Hpsi; x.Hrho = h->Hrho; x.HN = h->HN; x.Xs = h->Xs;
    x.tw = h->tw;
    x.alpha = h->p.alpha;
    x.omega = h->p.omega;
    x.sc = scale_of(h);
    x.gsc = h->p.g * x.sc;
    x.dt = h->p.dt;
    x.pref = make_double2(-h->p.disp, -1.0);
    return x;
}

// the same in the single-field shape svar
vk::EnsReal single_entry(const vk_gpe* h)
{
    vk::EnsReal x = ens_entry(h);
    x.var = h->svar;
    x.g = h->svar ? h->geo_s : h->geo;
    return x;
}

int make_single_table(vk_gpe* h)
{
    // the table and block maps of the single-field shape svar (build_maps
    // and ens_entry read the member shape fields, borrowed here)
    const int keep_var = h->ens_var;
    const Geo keep_geo = h->geo_v;
    h->ens_var = h->svar;
    h->geo_v = h->geo_s;
    const vk::EnsReal x = single_entry(h);
    for (int k = 0; k < 3; ++k) {
        if (h->e1map[k]) { hipFree(h->e1map[k]); h->e1map[k] = nullptr; }
        if (h->e1off[k]) { hipFree(h->e1off[k]); h->e1off[k] = nullptr; }
    }
    std::vector<vk_gpe*> hs{h};
    int rc = 0;
    if (!h->e1R && hipMalloc(&h->e1R, sizeof(vk::EnsReal)) != hipSuccess) rc = fail(VK_ERR_HIP, "hipMalloc e1R");
    if (!rc && hipMemcpy(h->e1R, &x, sizeof(x), hipMemcpyHostToDevice) != hipSuccess) rc = fail(VK_ERR_HIP, "e1R copy");
    if (!rc) rc = build_maps(hs, std::vector<int>{0}, h->e1map, h->e1off, h->e1nblk);
    h->ens_var = keep_var;
    h->geo_v = keep_geo;
    if (rc) return rc;
    for (auto& l : h->e1lds) l = 0;
    dispatch_var(h->N, h->svar, [&](auto c) { ens_lds<decltype(c)>(h->e1lds); return 0; });
    set_lds(vk::k_ens_p1, h->e1lds[0]);
    set_lds(vk::k_ens_p2, h->e1lds[1]);
    set_lds(vk::k_ens_p3, h->e1lds[2]);
    set_lds(vk::k_ens_p4, h->e1lds[3]);
    for (auto k : {vk::k_ens_p4s<1>, vk::k_ens_p4s<2>, vk::k_ens_p4s<3>, vk::k_ens_p4s<4>}) set_lds(k, h->e1lds[3]);
    return 0;
}

// Before RK4 steps: K0 dealiased and Hpsi = IFFT_y(K0) on the retained
// panels in the layout the steps use: the single-field shape's for the
// one-member ensemble path (hstate 3 with svar = 1), else Cfg<N>'s
// (hstate 2).
int prep_rk4(vk_gpe* h)
{
    if (!h->svar) return ensure_rk4(h);
    if (h->hstate == 3) return 0;
    int rc = ensure_rk4(h);
    if (rc) return rc;
    rc = dispatch_var(h->N, h->svar, [&](auto c) {
        using C = decltype(c);
        const size_t lds = (size_t)C::TC * C::COLRS * sizeof(double);
        set_lds(vk::k_col_inv<C>, lds);
        hipLaunchKernelGGL(vk::k_col_inv<C>, dim3(h->geo_s.Pp + h->geo_s.Pn), dim3(C::COLT), lds, h->stream,
                           (const cplx*)h->K0, h->Hpsi, (const cplx*)h->tw, h->geo_s, 1, 0);
        return 0;
    });
    if (rc) return rc;
    h->hstate = 3;
    return 0;
}

// the ensemble P4 of one stage: a kernel per stage, or one kernel taking
// the stage at run time (VK_ENS_P4_RUNTIME_STAGE=1)
#ifndef VK_ENS_P4_RUNTIME_STAGE
#define VK_ENS_P4_RUNTIME_STAGE 0
#endif
void ens_p4_launch(hipStream_t st, int nb, size_t lds, const vk::EnsReal* R, const int* m, const int* o, int stage)
{
    if (VK_ENS_P4_RUNTIME_STAGE) {
        hipLaunchKernelGGL(vk::k_ens_p4, dim3(nb), dim3(256), lds, st, R, m, o, stage);
        return;
    }
    auto k = stage == 1 ? vk::k_ens_p4s<1> : stage == 2 ? vk::k_ens_p4s<2> : stage == 3 ? vk::k_ens_p4s<3>
                                                                                   : vk::k_ens_p4s<4>;
    hipLaunchKernelGGL(k, dim3(nb), dim3(256), lds, st, R, m, o);
}

// launch the four passes of every stage over the given block maps
void ens_passes(hipStream_t st, const vk::EnsReal* R, int* const* m, int* const* o, const int* nb, const size_t* lds,
                vk_gpe* th)
{
    for (int stage = 1; stage <= 4; ++stage) {
        if (th) ev_begin(th);
        hipLaunchKernelGGL(vk::k_ens_p1, dim3(nb[0]), dim3(256), lds[0], st, R, (const int*)m[0], (const int*)o[0]);
        if (th) ev_end(th, PK_P1), ev_begin(th);
        hipLaunchKernelGGL(vk::k_ens_p2, dim3(nb[1]), dim3(256), lds[1], st, R, (const int*)m[1], (const int*)o[1]);
        if (th) ev_end(th, PK_P2), ev_begin(th);
        hipLaunchKernelGGL(vk::k_ens_p3, dim3(nb[0]), dim3(256), lds[2], st, R, (const int*)m[0], (const int*)o[0]);
        if (th) ev_end(th, PK_P3), ev_begin(th);
        ens_p4_launch(st, nb[2], lds[3], R, (const int*)m[2], (const int*)o[2], stage);
        if (th) ev_end(th, PK_P4);
    }
}

int ens1_step(vk_gpe* h)
{
    ens_passes(h->stream, h->e1R, h->e1map, h->e1off, h->e1nblk, h->e1lds, h);
    h->kv_valid = 0;
    return 0;
}

}  // namespace

namespace {

// shape variant per (N, GPU model) chosen by vk_ens_autotune_shapes in this
// process
std::mutex g_shape_mu;
std::map<std::pair<int, std::string>, int> g_shape_cache;

std::string gpu_model()
{
    int dev = 0;
    hipDeviceProp_t pr{};
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&pr, dev) != hipSuccess) return "?";
    return std::string(pr.gcnArchName);
}

int cached_shape(int N)
{
    std::lock_guard<std::mutex> lk(g_shape_mu);
    auto it = g_shape_cache.find({N, gpu_model()});
    return it == g_shape_cache.end() ? 0 : it->second;
}

void set_member_variant(vk_ens* e, int N, int v)
{
    e->var[N] = v;
    for (int r : e->size_reals[N]) {
        vk_gpe* h = e->h[r];
        h->ens_var = v;
        int TC = 0;
        dispatch_var(N, v, [&](auto c) { TC = decltype(c)::TC; return 0; });
        h->geo_v = geo_of(N, TC);
    }
}

// (re)build the member table, the block maps of all launch modes and drop
// captured graphs (after a shape change)
int ens_rebuild(vk_ens* e)
{
    for (auto& g : e->gexec)
        if (g) { hipGraphExecDestroy(g); g = nullptr; }
    for (int k = 0; k < 3; ++k) {
        if (e->dmap[k]) { hipFree(e->dmap[k]); e->dmap[k] = nullptr; }
        if (e->doff[k]) { hipFree(e->doff[k]); e->doff[k] = nullptr; }
    }
    for (auto& kv : e->smaps) for (auto p : kv.second) if (p) hipFree(p);
    e->smaps.clear();
    e->snblk.clear();
    const int nreal = (int)e->h.size();
    std::vector<vk::EnsReal> R(nreal);
    for (int r = 0; r < nreal; ++r) R[r] = ens_entry(e->h[r]);
    if (!e->dR) HIPCHK(hipMalloc(&e->dR, sizeof(vk::EnsReal) * nreal));
    HIPCHK(hipMemcpy(e->dR, R.data(), sizeof(vk::EnsReal) * nreal, hipMemcpyHostToDevice));
    std::vector<int> all(nreal);
    for (int r = 0; r < nreal; ++r) all[r] = r;
    int rc = build_maps(e->h, all, e->dmap, e->doff, e->nblk);
    if (rc) return rc;
    for (int N : e->sizes) {
        std::array<int*, 6> m{};
        int* dm[3];
        int* dof[3];
        std::array<int, 3> nb{};
        if ((rc = build_maps(e->h, e->size_reals[N], dm, dof, nb.data()))) return rc;
        for (int k = 0; k < 3; ++k) { m[2 * k] = dm[k]; m[2 * k + 1] = dof[k]; }
        e->smaps[N] = m;
        e->snblk[N] = nb;
    }
    e->synced = 0;
    return 0;
}

// Hpsi = IFFT_y(K0) on the retained panels of shape (N, var)
int col_inv_var(vk_gpe* h, int var)
{
    return dispatch_var(h->N, var, [&](auto c) {
        using C = decltype(c);
        const Geo& g = var ? h->geo_v : h->geo;
        const size_t lds = (size_t)C::TC * C::COLRS * sizeof(double);
        set_lds(vk::k_col_inv<C>, lds);
        hipLaunchKernelGGL(vk::k_col_inv<C>, dim3(g.Pp + g.Pn), dim3(C::COLT), lds, h->stream, (const cplx*)h->K0,
                           h->Hpsi, (const cplx*)h->tw, g, 1, 0);
        return 0;
    });
}

// Diagnostics of the members hs (all of size C::N, all with Hpsi in layout
// pl: 1 retained panels, 0 all panels) as batched launches on stream st:
// the single-field pipeline (diag_launch) with blockIdx.y selecting the
// member.  Its sums run per row, column and shell, whatever the workgroup
// shape, so each member gets bit for bit its single-field result.  Member
// i's sums and spectra go to out[i].
// tab: device memory for the operand table, ens_diag_tab_bytes(hs.size());
// htab: pinned host memory of the same size, not rewritten before the
// stream has passed the copy.
size_t ens_diag_tab_bytes(size_t n) { return n * sizeof(vk::DiagB); }

// columns per workgroup of the ensemble's spectra pass
template <class C, class CC> constexpr int diag_cols()
{
    if constexpr (C::N >= 256) return CC::G;
    else return C::TC;
}

template <class C>
int ens_diag_group(const std::vector<vk_gpe*>& hs, int pl, hipStream_t st, void* tab, void* htab,
                   const std::vector<double*>& out)
{
    const int n = (int)hs.size();
    const vk_gpe* h0 = hs[0];
    const Geo g = h0->geo;
    const cplx* tw = h0->tw;   // the same table in every member of this size
    const double sc = scale_of(h0);
    vk::DiagB* db = static_cast<vk::DiagB*>(htab);
    for (int i = 0; i < n; ++i) {
        const vk_gpe* h = hs[i];
        db[i] = vk::DiagB{h->Hpsi, h->K0, h->Hd, h->Hrho, h->Krho, h->HN, h->Xs, diag_rsum(h), diag_part(h), out[i],
                          diag_args(h, 0), spec_args(h)};
    }
    const vk::DiagB* dd = static_cast<const vk::DiagB*>(tab);
    HIPCHK(hipMemcpyAsync(tab, htab, ens_diag_tab_bytes(n), hipMemcpyHostToDevice, st));
    const size_t rl = (size_t)C::TR * C::ROWRS * sizeof(double), cl = (size_t)C::TC * C::COLRS * sizeof(double);
    set_lds(vk::k_p1d_b<C>, rl);
    set_lds(vk::k_diag_row_b<C>, rl);
    set_lds(vk::k_diag_dy_b<C>, cl);
    set_lds(vk::k_p2d_b<C>, cl);
    using CC = std::conditional_t<(C::N >= 256), vk::CfgD<C::N, false>, C>;
    constexpr int GC = diag_cols<C, CC>(), GS = C::TC / GC;
    const size_t ccl = (size_t)GC * CC::COLRS * sizeof(double);
    set_lds(vk::k_diag_col_b<CC, GC>, ccl);
    const dim3 rg(C::N / C::TR, n), rb(C::ROWT), cb(C::COLT);
    hipLaunchKernelGGL(vk::k_diag_dy_b<C>, dim3(pl == 1 ? g.Pp + g.Pn : C::NP, n), cb, cl, st, dd, tw, g, pl);
    hipLaunchKernelGGL(vk::k_p1d_b<C>, rg, rb, rl, st, dd, tw, g, pl, sc);
    hipLaunchKernelGGL(vk::k_p2d_b<C>, dim3(g.Pp, n), cb, cl, st, dd, tw, g);
    hipLaunchKernelGGL(vk::k_diag_row_b<C>, rg, rb, rl, st, dd, tw, g, pl, sc);
    hipLaunchKernelGGL((vk::k_diag_col_b<CC, GC>), dim3(GS == 1 ? g.Pp : (g.Pp + 7) / 8 * 8 * GS, n), dim3(GC * CC::T),
                       ccl, st, dd, tw, g);
    hipLaunchKernelGGL(vk::k_spec_reduce_b, dim3(h0->nshell / 64 + 1, 7, n), dim3(64 * vk::SPEC_G), 0, st, dd);
    return 0;
}

}  // namespace

extern "C" {

int vk_ens_create(vk_ens** out, int nreal, const vk_gpe_params* params)
{
    if (!out || nreal <= 0 || !params) return fail(VK_ERR_ARG, "ens_create: bad arguments");
    *out = nullptr;
    for (int r = 0; r < nreal; ++r) {
        const int N = params[r].N;
        if (N != 128 && N != 256 && N != 512 && N != 1024)
            return fail(VK_ERR_UNSUPPORTED, "ensemble members must have N in {128, 256, 512, 1024}");
        if (params[r].np != 0) return fail(VK_ERR_UNSUPPORTED, "ensemble members carry no particles");
    }
    vk_ens* e = new vk_ens();
    auto cleanup = [&](int rc) { vk_ens_destroy(e); return rc; };
    for (int r = 0; r < nreal; ++r) {
        vk_gpe* h = nullptr;
        int rc = vk_gpe_create(&h, &params[r]);
        if (rc) return cleanup(rc);
        e->h.push_back(h);
        e->size_reals[h->N].push_back(r);
    }
    for (auto& kv : e->size_reals) e->sizes.push_back(kv.first);
    if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(VK_ERR_HIP, "ens stream"));
    // LDS limits for every shape a member may take
    for (int N : e->sizes)
        for (int v = 0; v <= 1; ++v)
            if (vk::has_variant(N, v)) dispatch_var(N, v, [&](auto c) { ens_lds<decltype(c)>(e->lds); return 0; });
    set_lds(vk::k_ens_p1, e->lds[0]);
    set_lds(vk::k_ens_p2, e->lds[1]);
    set_lds(vk::k_ens_p3, e->lds[2]);
    set_lds(vk::k_ens_p4, e->lds[3]);
    for (auto k : {vk::k_ens_p4s<1>, vk::k_ens_p4s<2>, vk::k_ens_p4s<3>, vk::k_ens_p4s<4>}) set_lds(k, e->lds[3]);
    // the persistent step: as many workgroups as the device holds at once
    {
        e->plds = *std::max_element(e->lds, e->lds + 4);
        set_lds(vk::k_ens_step, e->plds);
        int dev = 0, per_cu = 0, ncu = 0, rate_khz = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, vk::k_ens_step, 256, e->plds) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "ens_create: device attributes"));
        e->pgrid = (per_cu * ncu) / 8 * 8;
        e->plimit = (long long)std::max(rate_khz, 1000) * 1000;   // one second
        if (hipMalloc(&e->dbar, sizeof(unsigned) * vk::kEnsStepBarriers) != hipSuccess ||
            hipMalloc(&e->derr, sizeof(int)) != hipSuccess || hipMemset(e->derr, 0, sizeof(int)) != hipSuccess)
            return cleanup(fail(VK_ERR_HIP, "ens_create: barrier memory"));
    }
    // shapes an earlier autotuning picked for this size on this GPU model
    for (int N : e->sizes) {
        const int v = cached_shape(N);
        if (v > 0) set_member_variant(e, N, v);
    }
    int rc = ens_rebuild(e);
    if (rc) return cleanup(rc);
    *out = e;
    return 0;
}

void vk_ens_destroy(vk_ens* e)
{
    if (!e) return;
    if (e->stream) hipStreamSynchronize(e->stream);
    for (auto g : e->gexec) if (g) hipGraphExecDestroy(g);
    for (int k = 0; k < 3; ++k) { if (e->dmap[k]) hipFree(e->dmap[k]); if (e->doff[k]) hipFree(e->doff[k]); }
    for (auto& kv : e->smaps) for (auto p : kv.second) if (p) hipFree(p);
    if (e->dR) hipFree(e->dR);
    if (e->dbar) hipFree(e->dbar);
    if (e->derr) hipFree(e->derr);
    if (e->hstage) hipHostFree(e->hstage);
    if (e->dstage) hipFree(e->dstage);
    if (e->dtab) hipFree(e->dtab);
    if (e->htab) hipHostFree(e->htab);
    for (auto h : e->h) vk_gpe_destroy(h);
    if (e->stream) hipStreamDestroy(e->stream);
    delete e;
}

}  // extern "C"

namespace {

// After the stream has drained: fail if a persistent step's barrier wait ran
// out of time (a workgroup was not resident; that step's results are
// invalid).  The flag is cleared for later steps.
int ens_check_barrier(vk_ens* e)
{
    int err = 0;
    HIPCHK(hipMemcpy(&err, e->derr, sizeof(int), hipMemcpyDeviceToHost));
    if (!err) return 0;
    hipLaunchKernelGGL(vk::k_zero_u32, dim3(1), dim3(64), 0, e->stream, reinterpret_cast<unsigned*>(e->derr), 1);
    return fail(VK_ERR_STATE, "ensemble mode 3: a grid barrier timed out (workgroups not co-resident); state invalid");
}

// one RK4 step of every realization on the ensemble stream
int ens_step_launch(vk_ens* e)
{
    if (e->mode == 2) {
        // per realization: the single-field kernels, one launch per pass each
        for (auto h : e->h) {
            hipStream_t keep = h->stream;
            h->stream = e->stream;
            int rc = rk4_step(h);
            h->stream = keep;
            if (rc) return rc;
        }
        return 0;
    }
    if (e->mode == 3) {
        if (e->pgrid < 8) return fail(VK_ERR_UNSUPPORTED, "ensemble: the device holds too few workgroups for mode 3");
        vk::EnsStepArgs A{};
        // one group per member size, blocks numbered over the sizes ascending
        if ((int)e->sizes.size() > vk::kEnsMaxGroups) return fail(VK_ERR_UNSUPPORTED, "ensemble: too many sizes");
        int base[3] = {};
        for (int N : e->sizes) {
            vk::EnsGroup& G = A.grp[A.ngrp++];
            G.key = N * 2 + (e->var.count(N) ? e->var[N] : 0);
            const auto& m = e->smaps[N];
            const auto& nb = e->snblk[N];
            for (int k = 0; k < 3; ++k) {
                G.map[k] = m[2 * k];
                G.off[k] = m[2 * k + 1];
                G.nblk[k] = nb[k];
                G.base[k] = base[k];
                base[k] += nb[k];
            }
        }
        A.bar = e->dbar;
        A.err = e->derr;
        A.limit = e->plimit;
        // no more workgroups than the largest pass has blocks: a small
        // ensemble's barriers then wait for few arrivals
        const int most = std::max(base[0], std::max(base[1], base[2]));
        const int grid = std::min(e->pgrid, (most + 7) / 8 * 8);
        hipLaunchKernelGGL(vk::k_zero_u32, dim3(1), dim3(64), 0, e->stream, e->dbar, vk::kEnsStepBarriers);
        hipLaunchKernelGGL(vk::k_ens_step, dim3(grid), dim3(256), e->plds, e->stream, (const vk::EnsReal*)e->dR, A);
        return 0;
    }
    struct Grp { int* m[3]; int* o[3]; int nb[3]; };
    std::vector<Grp> gs;
    if (e->mode == 0) {
        gs.push_back({{e->dmap[0], e->dmap[1], e->dmap[2]}, {e->doff[0], e->doff[1], e->doff[2]},
                      {e->nblk[0], e->nblk[1], e->nblk[2]}});
    } else {
        for (int N : e->sizes) {
            auto& m = e->smaps[N];
            auto& nb = e->snblk[N];
            gs.push_back({{m[0], m[2], m[4]}, {m[1], m[3], m[5]}, {nb[0], nb[1], nb[2]}});
        }
    }
    if (gs.size() == 1) {
        ens_passes(e->stream, e->dR, gs[0].m, gs[0].o, gs[0].nb, e->lds, nullptr);
        return 0;
    }
    // one launch per size, sizes interleaved pass by pass
    for (int stage = 1; stage <= 4; ++stage) {
        for (auto& g : gs)
            hipLaunchKernelGGL(vk::k_ens_p1, dim3(g.nb[0]), dim3(256), e->lds[0], e->stream,
                               (const vk::EnsReal*)e->dR, (const int*)g.m[0], (const int*)g.o[0]);
        for (auto& g : gs)
            hipLaunchKernelGGL(vk::k_ens_p2, dim3(g.nb[1]), dim3(256), e->lds[1], e->stream,
                               (const vk::EnsReal*)e->dR, (const int*)g.m[1], (const int*)g.o[1]);
        for (auto& g : gs)
            hipLaunchKernelGGL(vk::k_ens_p3, dim3(g.nb[0]), dim3(256), e->lds[2], e->stream,
                               (const vk::EnsReal*)e->dR, (const int*)g.m[0], (const int*)g.o[0]);
        for (auto& g : gs)
            ens_p4_launch(e->stream, g.nb[2], e->lds[3], (const vk::EnsReal*)e->dR, (const int*)g.m[2],
                          (const int*)g.o[2], stage);
    }
    return 0;
}

// Every member's Hpsi = IFFT_y(K0) in its shape's layout (the one-launch
// modes), or in the single-field layout (one launch per member).  A member
// of shape variant 1 then marks its Hpsi stale for the single-field entry
// points (hstate 0), which rebuild it in their layout on access.
int ens_prepare(vk_ens* e)
{
    if (e->synced) return 0;
    for (auto h : e->h) {
        int rc = ensure_rk4(h);
        if (rc) return rc;
        if (e->mode != 2 && h->ens_var) {
            if ((rc = col_inv_var(h, h->ens_var))) return rc;
            h->hstate = 0;
        }
        HIPCHK(hipStreamSynchronize(h->stream));
    }
    e->synced = 1;
    return 0;
}

int ens_steps_async(vk_ens* e, int nsteps)
{
    int rc = ens_prepare(e);
    if (rc) return rc;
    if (e->use_graph) {
        hipGraphExec_t& ge = e->gexec[e->mode];
        if (!ge) {
            hipGraph_t g;
            HIPCHK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
            rc = ens_step_launch(e);
            hipError_t ce = hipStreamEndCapture(e->stream, &g);
            if (rc) return rc;
            HIPCHK(ce);
            HIPCHK(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
            HIPCHK(hipGraphDestroy(g));
        }
        for (int i = 0; i < nsteps; ++i) HIPCHK(hipGraphLaunch(ge, e->stream));
    } else {
        for (int i = 0; i < nsteps; ++i)
            if ((rc = ens_step_launch(e))) return rc;
    }
    return 0;
}

}  // namespace

extern "C" {

int vk_ens_size(vk_ens* e) { return e ? (int)e->h.size() : 0; }
void* vk_ens_stream(vk_ens* e) { return e ? (void*)e->stream : nullptr; }

static int ens_member(vk_ens* e, int r, vk_gpe** h)
{
    if (!e || r < 0 || r >= (int)e->h.size()) return fail(VK_ERR_ARG, "ensemble: bad realization index");
    HIPCHK(hipStreamSynchronize(e->stream));
    *h = e->h[r];
    return 0;
}

int vk_ens_set_psi(vk_ens* e, int r, const double* psi, int flags)
{
    vk_gpe* h;
    int rc = ens_member(e, r, &h);
    if (rc) return rc;
    e->synced = 0;
    return vk_gpe_set_psi(h, psi, flags);
}

int vk_ens_set_ic_vortices(vk_ens* e, int r, int nv, const double* xs, const double* ys, const int* qs, int nimg,
                           int flags)
{
    vk_gpe* h;
    int rc = ens_member(e, r, &h);
    if (rc) return rc;
    e->synced = 0;
    return vk_gpe_set_ic_vortices(h, nv, xs, ys, qs, nimg, flags);
}

int vk_ens_get_psi(vk_ens* e, int r, double* psi, double* kpsi)
{
    vk_gpe* h;
    int rc = ens_member(e, r, &h);
    if (rc) return rc;
    if (h->ens_var && psi) e->synced = 0;   // psi rebuilds Hpsi in the single-field layout
    return vk_gpe_get_psi(h, psi, kpsi);
}

int vk_ens_diagnostics(vk_ens* e, int r, double* scal, double* spec, double* pscal)
{
    vk_gpe* h;
    int rc = ens_member(e, r, &h);
    if (rc) return rc;
    if (h->ens_var) e->synced = 0;
    return vk_gpe_diagnostics(h, scal, spec, pscal);
}

int vk_ens_diagnostics_all(vk_ens* e, double* scal, double* spec)
{
    if (!e) return fail(VK_ERR_ARG, "ens_diagnostics_all: null");
    HIPCHK(hipStreamSynchronize(e->stream));
    const size_t nreal = e->h.size();
    std::vector<size_t> offs(nreal + 1, 0);
    for (size_t r = 0; r < nreal; ++r) offs[r + 1] = offs[r] + diag_results(e->h[r]);
    const size_t need = offs[nreal];
    if (need > e->nstage) {
        if (e->hstage) hipHostFree(e->hstage);
        if (e->dstage) hipFree(e->dstage);
        e->hstage = nullptr;
        e->dstage = nullptr;
        e->nstage = 0;
        HIPCHK(hipHostMalloc((void**)&e->hstage, need * sizeof(double)));
        HIPCHK(hipMalloc(&e->dstage, need * sizeof(double)));
        e->nstage = need;
    }
    for (auto h : e->h) {
        int rc = diag_setup(h, e->stream);
        if (rc) return rc;
    }
    // groups of one size and one Hpsi state, batched launches on the
    // ensemble stream, each group's operand tables in its own part of dtab
    std::map<std::pair<int, int>, std::vector<int>> groups;
    for (size_t r = 0; r < nreal; ++r) groups[{e->h[r]->N, e->h[r]->hstate}].push_back((int)r);
    // per group: the ensure table (one pair per member), then the group's
    // tables; pinned staging in the same layout, so no copy waits
    auto ens_bytes = [](size_t n) { return (n * sizeof(vk::BPair) + 255) / 256 * 256; };
    size_t tabb = 0;
    for (auto& kv : groups)
        tabb += ens_bytes(kv.second.size()) + (ens_diag_tab_bytes(kv.second.size()) + 255) / 256 * 256;
    if (tabb > e->ntab) {
        if (e->dtab) hipFree(e->dtab);
        if (e->htab) hipHostFree(e->htab);
        e->dtab = nullptr;
        e->htab = nullptr;
        e->ntab = 0;
        HIPCHK(hipMalloc(&e->dtab, tabb));
        HIPCHK(hipHostMalloc(&e->htab, tabb));
        e->ntab = tabb;
    }
    size_t toff = 0;
    for (auto& kv : groups) {
        std::vector<vk_gpe*> hs;
        std::vector<double*> res;
        for (int r : kv.second) {
            hs.push_back(e->h[r]);
            res.push_back(e->dstage + offs[r]);
        }
        char* etab = static_cast<char*>(e->dtab) + toff;
        char* ehtab = static_cast<char*>(e->htab) + toff;
        toff += ens_bytes(hs.size());
        char* tab = static_cast<char*>(e->dtab) + toff;
        char* htab = static_cast<char*>(e->htab) + toff;
        toff += (ens_diag_tab_bytes(hs.size()) + 255) / 256 * 256;
        int rc = dispatch_var(kv.first.first, 0, [&](auto shape) {
            using C = decltype(shape);
            if (kv.first.second == 0) {
                // Hpsi stale (a member in its second shape): IFFT_y(K0) on
                // all panels in the single-field layout, as ensure_any does
                vk::BPair* pr = reinterpret_cast<vk::BPair*>(ehtab);
                for (size_t i = 0; i < hs.size(); ++i) pr[i] = vk::BPair{hs[i]->K0, hs[i]->Hpsi};
                HIPCHK(hipMemcpyAsync(etab, ehtab, hs.size() * sizeof(vk::BPair), hipMemcpyHostToDevice, e->stream));
                const size_t cl = (size_t)C::TC * C::COLRS * sizeof(double);
                set_lds(vk::k_col_inv_b<C>, cl);
                hipLaunchKernelGGL(vk::k_col_inv_b<C>, dim3(C::NP, (int)hs.size()), dim3(C::COLT), cl, e->stream,
                                   (const vk::BPair*)etab, (const cplx*)hs[0]->tw, hs[0]->geo, 0, 0);
                for (auto h : hs) h->hstate = 1;
            }
            return ens_diag_group<C>(hs, hs[0]->hstate == 2 ? 1 : 0, e->stream, tab, htab, res);
        });
        if (rc) return rc;
        for (auto h : hs)
            if (h->ens_var) e->synced = 0;   // Hpsi now in the single-field layout
    }
    HIPCHK(hipMemcpyAsync(e->hstage, e->dstage, need * sizeof(double), hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    HIPCHK(hipGetLastError());
    const double dg[4] = {};
    size_t so = 0;
    for (size_t r = 0; r < nreal; ++r) {
        const vk_gpe* h = e->h[r];
        const size_t ns = 6 * (size_t)(h->nshell + 1);
        diag_final(h, e->hstage + offs[r], e->hstage + offs[r] + 8, dg, scal ? scal + 8 * r : nullptr,
                   spec ? spec + so : nullptr, nullptr);
        so += ns;
    }
    return 0;
}

void vk_ens_forget_shapes(void)
{
    std::lock_guard<std::mutex> lk(g_shape_mu);
    g_shape_cache.clear();
}

int vk_ens_set_shape(vk_ens* e, int N, int var)
{
    if (!e || !e->size_reals.count(N) || !vk::has_variant(N, var))
        return fail(VK_ERR_ARG, "ens_set_shape: no members of that size, or no such shape for it");
    HIPCHK(hipStreamSynchronize(e->stream));
    set_member_variant(e, N, var);
    return ens_rebuild(e);
}

int vk_ens_get_shape(vk_ens* e, int N, int* var)
{
    if (!e || !var || !e->size_reals.count(N)) return fail(VK_ERR_ARG, "ens_get_shape: bad arguments");
    *var = e->var.count(N) ? e->var[N] : 0;
    return 0;
}

int vk_ens_rk4_steps_async(vk_ens* e, int nsteps)
{
    if (!e || nsteps < 0) return fail(VK_ERR_ARG, "ens_rk4_steps: bad arguments");
    return ens_steps_async(e, nsteps);
}

int vk_ens_rk4_steps(vk_ens* e, int nsteps)
{
    int rc = vk_ens_rk4_steps_async(e, nsteps);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(e->stream));
    HIPCHK(hipGetLastError());
    return ens_check_barrier(e);
}

int vk_ens_set_mode(vk_ens* e, int mode, int use_graph)
{
    if (!e || mode < 0 || mode > 3) return fail(VK_ERR_ARG, "ens_set_mode: bad arguments");
    HIPCHK(hipStreamSynchronize(e->stream));
    if (mode != e->mode) e->synced = 0;   // the per-member mode uses the single-field layout
    e->mode = mode;
    e->use_graph = use_graph ? 1 : 0;
    return 0;
}

int vk_ens_get_mode(vk_ens* e, int* mode, int* use_graph)
{
    if (!e) return fail(VK_ERR_ARG, "ens_get_mode: null");
    if (mode) *mode = e->mode;
    if (use_graph) *use_graph = e->use_graph;
    return 0;
}

// Autotuner: times every (launch mode, graph) schedule over nsteps steps from
// the current state, restores the state, keeps the fastest.  ms_out[8]:
// ms per step for modes 0..3 x {graph, direct}.
int vk_ens_autotune(vk_ens* e, int nsteps, double* ms_out)
{
    if (!e || nsteps <= 0) return fail(VK_ERR_ARG, "ens_autotune: bad arguments");
    int rc = ens_prepare(e);
    if (rc) return rc;
    // save the state (kpsi and its y-inverse); K1/K2 are rewritten by stage 1
    std::vector<cplx*> save;
    for (auto h : e->h) {
        cplx* b = nullptr;
        HIPCHK(hipMalloc(&b, 2 * f2(h) * sizeof(cplx)));
        HIPCHK(hipMemcpyAsync(b, h->K0, f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
        HIPCHK(hipMemcpyAsync(b + f2(h), h->Hpsi, f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
        save.push_back(b);
    }
    hipEvent_t a, b;
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    double best = 1e300;
    int bm = 0, bg = 1;
    for (int m = 0; m < 4; ++m)
        for (int gph = 1; gph >= 0; --gph) {
            if (m != e->mode) e->synced = 0;
            e->mode = m;
            e->use_graph = gph;
            // warm: capture, graph upload on the first replays
            if ((rc = ens_steps_async(e, 3))) return rc;
            HIPCHK(hipEventRecord(a, e->stream));
            if ((rc = ens_steps_async(e, nsteps))) return rc;
            HIPCHK(hipEventRecord(b, e->stream));
            HIPCHK(hipEventSynchronize(b));
            if (ens_check_barrier(e)) {   // mode 3 not co-resident here: not a candidate
                if (ms_out) ms_out[2 * m + (1 - gph)] = -1.0;
                continue;
            }
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, a, b));
            const double per = ms / nsteps;
            if (ms_out) ms_out[2 * m + (1 - gph)] = per;
            if (per < best) { best = per; bm = m; bg = gph; }
        }
    if (bm != e->mode) e->synced = 0;
    e->mode = bm;
    e->use_graph = bg;
    for (size_t i = 0; i < e->h.size(); ++i) {
        vk_gpe* h = e->h[i];
        HIPCHK(hipMemcpyAsync(h->K0, save[i], f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
        HIPCHK(hipMemcpyAsync(h->Hpsi, save[i] + f2(h), f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
    }
    HIPCHK(hipStreamSynchronize(e->stream));
    for (auto p : save) hipFree(p);
    hipEventDestroy(a);
    hipEventDestroy(b);
    return 0;
}

// Shape autotuner: for each member size with a second shape (8 points per
// thread instead of 16), times whole-ensemble steps in the current launch
// mode with either shape for that size (the other sizes as chosen so far,
// sizes ascending), restoring kpsi before every trial, and keeps the faster
// one.  The choice is remembered per (N, GPU model) for ensembles created
// later in the process.  vars_out[i], ms_out[2i], ms_out[2i+1]: the chosen
// shape and the ms/step of shapes 0 and 1 for the i-th distinct size
// (ascending; -1 where a size has one shape).
int vk_ens_autotune_shapes(vk_ens* e, int nsteps, int* vars_out, double* ms_out)
{
    if (!e || nsteps <= 0) return fail(VK_ERR_ARG, "ens_autotune_shapes: bad arguments");
    if (e->mode == 2) return fail(VK_ERR_STATE, "ens_autotune_shapes: the per-member mode has one shape");
    HIPCHK(hipStreamSynchronize(e->stream));
    std::vector<cplx*> save;
    for (auto h : e->h) {
        cplx* p = nullptr;
        HIPCHK(hipMalloc(&p, f2(h) * sizeof(cplx)));
        HIPCHK(hipMemcpyAsync(p, h->K0, f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
        save.push_back(p);
    }
    auto restore = [&]() -> int {
        for (size_t i = 0; i < e->h.size(); ++i) {
            vk_gpe* h = e->h[i];
            HIPCHK(hipMemcpyAsync(h->K0, save[i], f2(h) * sizeof(cplx), hipMemcpyDeviceToDevice, e->stream));
            h->hstate = 0;
        }
        e->synced = 0;
        return 0;
    };
    hipEvent_t a, b;
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    int rc = 0;
    for (size_t i = 0; i < e->sizes.size() && !rc; ++i) {
        const int N = e->sizes[i];
        if (vars_out) vars_out[i] = 0;
        if (ms_out) ms_out[2 * i] = ms_out[2 * i + 1] = -1.0;
        if (!vk::has_variant(N, 1)) continue;
        double t[2] = {0.0, 0.0};
        for (int v = 0; v <= 1 && !rc; ++v) {
            set_member_variant(e, N, v);
            if ((rc = ens_rebuild(e)) || (rc = restore()) || (rc = ens_steps_async(e, 1))) break;
            if (hipEventRecord(a, e->stream) != hipSuccess) { rc = fail(VK_ERR_HIP, "event"); break; }
            if ((rc = ens_steps_async(e, nsteps))) break;
            if (hipEventRecord(b, e->stream) != hipSuccess || hipEventSynchronize(b) != hipSuccess) {
                rc = fail(VK_ERR_HIP, "event");
                break;
            }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, a, b);
            t[v] = ms / nsteps;
        }
        if (rc) break;
        const int best = t[1] < t[0] ? 1 : 0;
        set_member_variant(e, N, best);
        if ((rc = ens_rebuild(e))) break;
        if (vars_out) vars_out[i] = best;
        if (ms_out) { ms_out[2 * i] = t[0]; ms_out[2 * i + 1] = t[1]; }
        std::lock_guard<std::mutex> lk(g_shape_mu);
        g_shape_cache[{N, gpu_model()}] = best;
    }
    if (!rc) rc = restore();
    HIPCHK(hipStreamSynchronize(e->stream));
    for (auto p : save) hipFree(p);
    hipEventDestroy(a);
    hipEventDestroy(b);
    return rc;
}

}  // extern "C"

// single-field transform shape (defined here, after the ensemble helpers it uses)
extern "C" {

int vk_gpe_set_shape(vk_gpe* h, int var)
{
    if (!h || (var != 0 && var != 1)) return fail(VK_ERR_ARG, "set_shape: bad arguments");
    if (h->np_cap > 0 || h->N < 128 || h->N > 1024 || !vk::has_variant(h->N, var))
        return fail(VK_ERR_UNSUPPORTED, "set_shape: shapes exist for N in {256, 512, 1024} without particles");
    HIPCHK(hipStreamSynchronize(h->stream));
    if (var == h->svar) return 0;
    if (h->hstate == 3) h->hstate = 0;   // Hpsi in the old shape's layout
    h->svar = var;
    int TC = 0;
    dispatch_var(h->N, var, [&](auto c) { TC = decltype(c)::TC; return 0; });
    h->geo_s = var ? geo_of(h->N, TC) : h->geo;
    return make_single_table(h);
}

int vk_gpe_get_shape(vk_gpe* h, int* var)
{
    if (!h || !var) return fail(VK_ERR_ARG, "get_shape: bad arguments");
    *var = h->svar;
    return 0;
}

}  // extern "C"
