// Fourier neural operator for the ARGLE warm start: forward, backward and
// Adam on the GPU.  Activations and accumulation are FP32, weights are BF16
// (FP32 master copies are kept for the optimizer).  No reference counterpart:
// the reference prepares ARGLE states from an analytic ansatz only
// (src/initial_config.f90, restart_from_argle_data).
//
// Network (per sample, N x N grid, planes [b][c][y][x], x fastest):
//   z0 = Wp x + bp                                    (lift, cin -> C)
//   u_{l+1} = W_l z_l + b_l + K_l z_l,  z_{l+1} = gelu(u_{l+1}) for l < L-1,
//   z_L = u_L
//   h = Q1 z_L + bq1 (C -> P),  out = Q2 gelu(h) + bq2 (P -> 2)
// Spectral convolution K z = E(R . D z):
//   D z (kx, ky) = sum_{x,y} z e^{-2 pi i (kx x + ky y)/N},  kx in [0,M),
//                  ky in [-M, M)  (index j = ky mod 2M)
//   (R . X)_o = s(kx) sum_i X_i R_io,  s(0) = 1/N^2, s(kx>0) = 2/N^2
//   E(Y)(x, y) = Re sum_{kx,ky} Y e^{+2 pi i (kx x + ky y)/N}
// Adjoints used by the backward pass (du = dL/du_{l+1}, real):
//   dR_io = s sum_b D(du_o) conj(X_i)
//   dz_i  = W^T du + Re sum_m [s sum_o D(du_o) conj(R_io)] e^{ik.x}
// Only 2 M^2 of the N^2 modes are kept, so D and E are separable sums over
// e^{-2 pi i k x/N} tables instead of full transforms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "vikshobha.h"

int vk_set_error(int code, const std::string& msg);   // vk_gpe.hip (vk_last_error)

namespace {

#define FCHK(x)                                                                                            \
    do {                                                                                                   \
        hipError_t e_ = (x);                                                                               \
        if (e_ != hipSuccess) return vk_set_error(VK_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

typedef float2 c32;

__host__ __device__ inline float bf2f(uint16_t h)
{
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}
__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest, ties to even (finite inputs)
    return (uint16_t)(u >> 16);
}

// Phi(x) = (1 + erf(x/sqrt 2))/2 as exp2(t P(t))/2, t = |x|: log2 erfc(t/sqrt 2)
// divided by t is smooth, so one polynomial (degree 9, weighted minimax fit
// on [0, 6]) and one exp2 serve every x without a branch.  In FP32, absolute
// error of Phi 3.5e-8 for x < 0 and 6.5e-8 for x > 0, where the rounding of 1 - e
// (half an FP32 ulp of 1, 3e-8) adds; relative error 5.6e-6 in the tail to x = -5.
// P's leading coefficient is negative, so |x| -> inf gives 0 or 1.
__device__ __forceinline__ float phi_cdf(float x)
{
    const float t = fabsf(x);
    float p = -2.6835729813894552e-08f;
    p = fmaf(p, t, 8.12881606235977e-07f);
    p = fmaf(p, t, -1.052355304431135e-05f);
    p = fmaf(p, t, 7.409366645662003e-05f);
    p = fmaf(p, t, -0.00027201727040192f);
    p = fmaf(p, t, -1.542872901961795e-05f);
    p = fmaf(p, t, 0.0069657554272513356f);
    p = fmaf(p, t, -0.052454154921228756f);
    p = fmaf(p, t, -0.45921661787979434f);
    p = fmaf(p, t, -1.1511046520970696f);
    const float e = 0.5f * __builtin_amdgcn_exp2f(p * t);
    return x >= 0.f ? 1.0f - e : (x < 0.f ? e : 0.5f + x);   // NaN takes the last form
}
__device__ __forceinline__ float gelu(float x) { return x * phi_cdf(x); }
// gelu(x) and its derivative Phi(x) + x phi(x)
__device__ __forceinline__ void gelu2(float x, float& g, float& d)
{
    const float c = phi_cdf(x);
    const float pdf = 0.39894228040143268f * __builtin_amdgcn_exp2f(-0.72134752044448170f * x * x);
    g = x * c;
    d = fmaf(x, pdf, c);
}

constexpr int CIN_MAX = 4;
constexpr int P_MAX = 64;
constexpr int L_MAX = 8;

typedef float f4 __attribute__((ext_vector_type(4)));

// D += A B, one 16 x 16 x 4 FP32 matrix instruction.  Lane l holds
// A[l%16][l/16], B[l/16][l%16] and D[4 (l/16) + r][l%16], r = 0..3.
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// order this wave's LDS accesses (the data of one lane is read by others of
// the same wave; a wave's LDS operations execute in order)
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// Row kernels.  A workgroup of up to 8 waves takes one grid row (b, y) at a
// time, all channels of it; a wave takes 64-column chunks of the row.  The
// pointwise channel map and the spectral inverse along x are one matrix
// product per chunk,
//   s[c][x] = [W | Re Bk, Im Bk][c][k] * [z; F][k][x],  k < C + 2M,
// and the truncated transform along x of the result,
//   A[c][kx] = sum_x z[c][x] e^{-2 pi i kx x/N},
// is a second one whose sums run over the chunk and then over the waves.
// Both run on the FP32 matrix instructions (FP32 products and sums).  The
// columns of a chunk are numbered x = 4 n + nt (n = l % 16, nt = 0..3), so
// that a lane's four B values and its four D values of a channel are one
// float4 of memory, and a product's k index is 16 kg + 4 (l/16) + j, so that
// D feeds the next product's B without a move.  The second product needs the
// chunk transposed across lanes: through a wave-private LDS tile, row stride
// 68 floats (every b128 access spreads over all 64 banks).
// Activations are stored once per layer, before gelu; readers apply gelu.
// ---------------------------------------------------------------------------

// Most waves of a row workgroup: 4 (several workgroups per CU run past each
// other's barriers: layers 3.02 ms a step against 3.06 with 8), 8 where the
// projection is trained (its LDS allows 8 waves per CU either way: 0.76
// against 0.88 ms).
constexpr int ROW_W = 4, ROW_W_TRAIN = 8;
#define ROW_OCC(n) __attribute__((amdgpu_waves_per_eu(n)))
constexpr int TLD = 68;         // floats per tile row

template <int C, int M> struct Row {
    static constexpr int CP = C < 16 ? 16 : C;          // channel rows padded to the matrix tile
    static constexpr int MT = CP / 16;
    static constexpr int K = C + 2 * M;
    static constexpr int KG = K / 16;
    static constexpr int NT = 2 * M < 16 ? 1 : 2 * M / 16;   // column tiles of the transform along x
    static constexpr int WLD = K + 4;
    static constexpr int QLD = CP + 4;
    static_assert(K % 16 == 0 && (C >= 16 || K == 16), "tile shapes");
};

struct RowArgs {
    const float* x;             // input planes [b][cin][N][N]
    const float* z;             // forward: u of the layer below (gelu applied here); backward: dL/du of the layer above
    const uint16_t *Wp, *bp;    // lift
    const uint16_t *W, *bias;   // pointwise map of the layer
    const c32* Bk;              // spectral part, inverse along y done: [b][c][y][kx]
    const float* FT;            // [2M][N]: Re, Im of e^{-2 pi i kx x/N}, x fastest
    const f4* FP;               // the same as B operands of the transform along x
    float* u;                   // forward: u of this layer; backward: dL/du of the layer below
    const float* uprev;         // backward: u of the layer below
    c32* A;                     // transform along x of gelu(u) (forward) or of dL/du (backward)
    int N, rows, cin;
    // head
    const uint16_t *Q1, *bq1, *Q2, *bq2;
    int P;
    float* out;
    const float* tgt;
    float inv_n;
    double* loss;               // per workgroup
    float* part;                // per workgroup: weight-gradient partial sums of this kernel
    int pstride;                // floats per workgroup in part
};

// transform along x of the chunk in the wave's tile
template <int C, int M>
__device__ __forceinline__ void dft_chunk(const float* ts, const f4* __restrict__ FP, int ch, int lane,
                                          f4 (&da)[Row<C, M>::MT][Row<C, M>::NT])
{
    using R = Row<C, M>;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        f4 a[R::MT];
#pragma unroll
        for (int mt = 0; mt < R::MT; ++mt)
            a[mt] = *reinterpret_cast<const f4*>(ts + (mt * 16 + lane % 16) * TLD + 16 * s + 4 * (lane / 16));
#pragma unroll
        for (int nt = 0; nt < R::NT; ++nt) {
            const f4 b = FP[((ch * 4 + s) * R::NT + nt) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt) da[mt][nt] = mfma(a[mt][j], b[j], da[mt][nt]);
        }
    }
}

// D layout -> wave tile
template <int MT>
__device__ __forceinline__ void tile_put(float* ts, int lane, const f4 (&d)[MT][4])
{
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f4*>(ts + (mt * 16 + 4 * (lane / 16) + r) * TLD + 4 * (lane % 16)) =
                f4{d[mt][0][r], d[mt][1][r], d[mt][2][r], d[mt][3][r]};
}

// sum over the workgroup's waves (in wave order) of the transforms along x,
// then to A; every thread of the workgroup takes part
template <int C, int M>
__device__ __forceinline__ void dft_store(float* tiles, int lane, int wv, int nw, int b, int y, int N,
                                          const f4 (&da)[Row<C, M>::MT][Row<C, M>::NT], c32* __restrict__ A)
{
    using R = Row<C, M>;
    constexpr int NC = R::NT * 16;
    float* ts = tiles + wv * R::CP * TLD;
    wave_lds_fence();
#pragma unroll
    for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < R::NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) ts[(mt * 16 + 4 * (lane / 16) + r) * NC + nt * 16 + lane % 16] = da[mt][nt][r];
    __syncthreads();
    for (int e = threadIdx.x; e < C * 2 * M; e += blockDim.x) {
        const int c = e / (2 * M), n = e % (2 * M);
        float s = 0.f;
        for (int w = 0; w < nw; ++w) s += tiles[w * R::CP * TLD + c * NC + n];
        reinterpret_cast<float*>(A)[(((size_t)b * C + c) * N + y) * (2 * M) + n] = s;
    }
    __syncthreads();
}

// Bk of row (b, y) into the weight rows' columns C..K-1
template <int C, int M>
__device__ __forceinline__ void load_bk(float* Wl, const c32* __restrict__ Bk, int b, int y, int N)
{
    using R = Row<C, M>;
    const float* f = reinterpret_cast<const float*>(Bk);
    for (int i = threadIdx.x; i < C * 2 * M; i += blockDim.x) {
        const int c = i / (2 * M), k = i % (2 * M);
        Wl[c * R::WLD + C + k] = f[(((size_t)b * C + c) * N + y) * (2 * M) + k];
    }
}

// lift of input planes xin at one channel
__device__ __forceinline__ f4 lift4(const float* wl, const f4 (&xin)[CIN_MAX])
{
    f4 s = {wl[CIN_MAX], wl[CIN_MAX], wl[CIN_MAX], wl[CIN_MAX]};
#pragma unroll
    for (int q = 0; q < CIN_MAX; ++q) s += wl[q] * xin[q];
    return s;
}

// lift weights and biases of every channel to LDS, [channel][CIN_MAX + 1]
template <int C, int CP>
__device__ __forceinline__ void load_lift(float* ll, const RowArgs& a)
{
    for (int i = threadIdx.x; i < CP * (CIN_MAX + 1); i += blockDim.x) {
        const int c = i / (CIN_MAX + 1), q = i % (CIN_MAX + 1);
        ll[i] = c >= C ? 0.f : (q == CIN_MAX ? bf2f(a.bp[c]) : (q < a.cin ? bf2f(a.Wp[c * a.cin + q]) : 0.f));
    }
}

// z0 = lift(x) and its transform along x (z0 itself is not stored: the
// first layer and its backward rebuild it from the planes)
template <int C, int M>
__global__ void __launch_bounds__(64 * ROW_W) k_lift_dft(RowArgs a)
{
    using R = Row<C, M>;
    extern __shared__ float sm[];
    float* tiles = sm;
    const int N = a.N, nw = blockDim.x / 64, lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    float* ll = tiles + nw * R::CP * TLD;
    float* ts = tiles + wv * R::CP * TLD;
    const size_t NN = (size_t)N * N;
    load_lift<C, R::CP>(ll, a);
    __syncthreads();
    for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
        const int b = row / N, y = row % N;
        f4 da[R::MT][R::NT] = {};
        for (int ch = wv; ch < N / 64; ch += nw) {
            const int x0 = ch * 64 + 4 * (lane % 16);
            f4 xin[CIN_MAX] = {};
#pragma unroll
            for (int q = 0; q < CIN_MAX; ++q)
                if (q < a.cin) xin[q] = *reinterpret_cast<const f4*>(a.x + ((size_t)b * a.cin + q) * NN + (size_t)y * N + x0);
            wave_lds_fence();
#pragma unroll
            for (int i = 0; i < R::CP / 4; ++i) {
                const int c = 4 * i + lane / 16;
                *reinterpret_cast<f4*>(ts + c * TLD + 4 * (lane % 16)) = lift4(ll + c * (CIN_MAX + 1), xin);
            }
            wave_lds_fence();
            dft_chunk<C, M>(ts, a.FP, ch, lane, da);
        }
        dft_store<C, M>(tiles, lane, wv, nw, b, y, N, da, a.A);
    }
}

// s = [W | Bk] [z; F] for one chunk: B operands of z from zv(k) (a float4 of
// channel k at this lane's columns), of F from the table
template <int C, int M, class ZV>
__device__ __forceinline__ void chunk_gemm(const float* Wl, const float* __restrict__ FT, int N, int x0, int lane,
                                           f4 (&acc)[Row<C, M>::MT][4], ZV&& zv)
{
    using R = Row<C, M>;
#pragma unroll
    for (int kg = 0; kg < R::KG; ++kg) {
        f4 w[R::MT];
#pragma unroll
        for (int mt = 0; mt < R::MT; ++mt)
            w[mt] = *reinterpret_cast<const f4*>(Wl + (mt * 16 + lane % 16) * R::WLD + 16 * kg + 4 * (lane / 16));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 16 * kg + 4 * (lane / 16) + j;
            f4 bv;
            if constexpr (C >= 16) {
                if (16 * kg < C) bv = zv(kg, j, k);
                else bv = *reinterpret_cast<const f4*>(FT + (size_t)(k - C) * N + x0);
            } else {
                if (k < C) bv = zv(kg, j, k);
                else bv = *reinterpret_cast<const f4*>(FT + (size_t)(k - C) * N + x0);
            }
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt) acc[mt][nt] = mfma(w[mt][j], bv[nt], acc[mt][nt]);
        }
    }
}

// sum over the 16 lanes of a row (row_ror 8, 4, 2, 1), in every lane
__device__ __forceinline__ float row16_sum(float x)
{
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x124, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x122, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x121, 0xf, 0xf, true));
    return x;
}

enum { TAIL_LAYER = 0, TAIL_INFER = 1, TAIL_TRAIN = 2 };

// LDS of the row kernels, in floats
template <int C, int M> size_t fwd_lds(int nw, bool head)
{
    using R = Row<C, M>;
    return (size_t)nw * R::CP * TLD + R::CP * R::WLD + R::CP + R::CP * (CIN_MAX + 1) +
           (head ? P_MAX * R::QLD + 3 * P_MAX + 4 : 0);
}
// the projection's weight gradients of a wave, in LDS between chunks: per 16
// hidden rows dQ1 as D tiles, then dbq1 and the two rows of dQ2
template <int C, int M> constexpr int dq_words() { return P_MAX / 16 * (Row<C, M>::MT * 64 * 4 + 3 * 16); }

// Forward layer.  LIFT: the layer's input is z0 = lift(x), otherwise
// gelu(a.z).  TAIL_LAYER: store u and the transform along x of gelu(u).
// TAIL_INFER: the projection h = Q1 u + bq1, out = Q2 gelu(h) + bq2 from the
// accumulators, out stored.  TAIL_TRAIN: also the loss, the projection's
// backward (dL/du stored, its transform along x) and the projection's weight
// gradients.
// Batch 8, 512^2, 32 channels, 16 modes: one layer reads and writes 268 MB
// (0.11 ms at the copy rate) and does 13 GFLOP on the matrix cores (0.09 ms):
// 0.284 ms, against 0.43 ms for separate x-transform and pointwise kernels
// that stored gelu(u) too; the sums of a wave's phases (loads, two products,
// two gelus) bound it, not one of them (without the transform 0.21, without
// gelu 0.27 ms).  TAIL_TRAIN: 0.76 ms, against 2.5 ms for the kernels that
// stored the hidden units.
template <int C, int M, bool LIFT, int TAIL>
__global__ void __launch_bounds__(64 * (TAIL == TAIL_TRAIN ? ROW_W_TRAIN : ROW_W)) ROW_OCC(TAIL == TAIL_TRAIN ? 2 : 3)
k_layer(RowArgs a)
{
    using R = Row<C, M>;
    extern __shared__ float sm[];
    const int N = a.N, nw = blockDim.x / 64, lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    const int n16 = lane % 16, g = lane / 16;
    float* tiles = sm;
    float* Wl = tiles + nw * R::CP * TLD;
    float* bs = Wl + R::CP * R::WLD;
    float* ll = bs + R::CP;
    float* Ql = ll + R::CP * (CIN_MAX + 1);
    float* bq = Ql + P_MAX * R::QLD;
    float* q2 = bq + P_MAX;           // [2][P_MAX], then bq2
    float* ts = tiles + wv * R::CP * TLD;
    const size_t NN = (size_t)N * N;
    for (int i = threadIdx.x; i < R::CP * C; i += blockDim.x) {
        const int c = i / C, k = i % C;
        Wl[c * R::WLD + k] = c < C ? bf2f(a.W[c * C + k]) : 0.f;
    }
    if constexpr (C < R::CP)
        for (int i = threadIdx.x; i < (R::CP - C) * 2 * M; i += blockDim.x)
            Wl[(C + i / (2 * M)) * R::WLD + C + i % (2 * M)] = 0.f;
    for (int i = threadIdx.x; i < R::CP; i += blockDim.x) bs[i] = i < C ? bf2f(a.bias[i]) : 0.f;
    if constexpr (LIFT) load_lift<C, R::CP>(ll, a);
    const int pm = (a.P + 15) / 16;   // 16-row tiles of the projection
    if constexpr (TAIL != TAIL_LAYER) {
        for (int i = threadIdx.x; i < P_MAX * R::CP; i += blockDim.x) {
            const int p = i / R::CP, c = i % R::CP;
            Ql[p * R::QLD + c] = p < a.P && c < C ? bf2f(a.Q1[p * C + c]) : 0.f;
        }
        for (int i = threadIdx.x; i < P_MAX; i += blockDim.x) {
            bq[i] = i < a.P ? bf2f(a.bq1[i]) : 0.f;
            q2[i] = i < a.P ? bf2f(a.Q2[i]) : 0.f;
            q2[P_MAX + i] = i < a.P ? bf2f(a.Q2[a.P + i]) : 0.f;
        }
        if (threadIdx.x < 2) q2[2 * P_MAX + threadIdx.x] = bf2f(a.bq2[threadIdx.x]);
    }
    // the projection's weight gradients over all rows of this workgroup
    // in this wave's LDS slots (in registers they would spill)
    constexpr int QW = R::MT * 64 * 4 + 3 * 16;   // words per 16 hidden rows
    float* dq = q2 + 2 * P_MAX + 4 + wv * dq_words<C, M>();
    if constexpr (TAIL == TAIL_TRAIN)
        for (int i = lane; i < dq_words<C, M>(); i += 64) dq[i] = 0.f;
    float dbq2[2] = {0.f, 0.f};
    double lacc = 0.0;

    for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
        const int b = row / N, y = row % N;
        __syncthreads();
        load_bk<C, M>(Wl, a.Bk, b, y, N);
        __syncthreads();
        f4 da[R::MT][R::NT] = {};
        for (int ch = wv; ch < N / 64; ch += nw) {
            const int x0 = ch * 64 + 4 * n16;
            const size_t ro = (size_t)y * N + x0;
            f4 acc[R::MT][4];
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = *reinterpret_cast<const f4*>(bs + mt * 16 + 4 * g);
            if constexpr (LIFT) {
                f4 xin[CIN_MAX] = {};
#pragma unroll
                for (int q = 0; q < CIN_MAX; ++q)
                    if (q < a.cin) xin[q] = *reinterpret_cast<const f4*>(a.x + ((size_t)b * a.cin + q) * NN + ro);
                chunk_gemm<C, M>(Wl, a.FT, N, x0, lane, acc,
                                 [&](int, int, int k) { return lift4(ll + k * (CIN_MAX + 1), xin); });
            } else {
                f4 zin[R::MT][4];
                const float* zp = a.z + (size_t)b * C * NN + ro;
#pragma unroll
                for (int kg = 0; kg < R::MT; ++kg)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int k = 16 * kg + 4 * g + j;
                        zin[kg][j] = *reinterpret_cast<const f4*>(zp + (size_t)(k < C ? k : 0) * NN);
                    }
                chunk_gemm<C, M>(Wl, a.FT, N, x0, lane, acc, [&](int kg, int j, int) {
                    f4 v = zin[kg < R::MT ? kg : 0][j];
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = gelu(v[i]);
                    return v;
                });
            }
            if constexpr (TAIL == TAIL_LAYER) {
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int c = mt * 16 + 4 * g + r;
                        if (C >= 16 || c < C)
                            *reinterpret_cast<f4*>(a.u + ((size_t)b * C + c) * NN + ro) =
                                f4{acc[mt][0][r], acc[mt][1][r], acc[mt][2][r], acc[mt][3][r]};
                    }
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[mt][nt][r] = gelu(acc[mt][nt][r]);
                wave_lds_fence();
                tile_put<R::MT>(ts, lane, acc);
                wave_lds_fence();
                dft_chunk<C, M>(ts, a.FP, ch, lane, da);
            } else {
                // projection, 16 hidden rows at a time
                auto hidden = [&](int pt, f4 (&h)[4]) {
#pragma unroll
                    for (int nt = 0; nt < 4; ++nt) h[nt] = *reinterpret_cast<const f4*>(bq + pt * 16 + 4 * g);
#pragma unroll
                    for (int mt = 0; mt < R::MT; ++mt) {
                        const f4 w = *reinterpret_cast<const f4*>(Ql + (pt * 16 + n16) * R::QLD + 16 * mt + 4 * g);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int nt = 0; nt < 4; ++nt) h[nt] = mfma(w[r], acc[mt][nt][r], h[nt]);
                    }
                };
                f4 o0 = {}, o1 = {};
                for (int pt = 0; pt < pm; ++pt) {
                    f4 h[4];
                    hidden(pt, h);
                    const f4 qa = *reinterpret_cast<const f4*>(q2 + pt * 16 + 4 * g);
                    const f4 qb = *reinterpret_cast<const f4*>(q2 + P_MAX + pt * 16 + 4 * g);
#pragma unroll
                    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float gv = gelu(h[nt][r]);
                            o0[nt] = fmaf(qa[r], gv, o0[nt]);
                            o1[nt] = fmaf(qb[r], gv, o1[nt]);
                        }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o0[i] += __shfl_xor(o0[i], 16, 64);
                    o1[i] += __shfl_xor(o1[i], 16, 64);
                    o0[i] += __shfl_xor(o0[i], 32, 64);
                    o1[i] += __shfl_xor(o1[i], 32, 64);
                }
                o0 += q2[2 * P_MAX];
                o1 += q2[2 * P_MAX + 1];
                const size_t oo = (size_t)b * 2 * NN + ro;
                if constexpr (TAIL == TAIL_INFER) {
                    if (g == 0) *reinterpret_cast<f4*>(a.out + oo) = o0;
                    if (g == 1) *reinterpret_cast<f4*>(a.out + oo + NN) = o1;
                } else {
                    const f4 e0 = o0 - *reinterpret_cast<const f4*>(a.tgt + oo);
                    const f4 e1 = o1 - *reinterpret_cast<const f4*>(a.tgt + oo + NN);
                    if (g == 0) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) lacc += (double)e0[i] * e0[i] + (double)e1[i] * e1[i];
                    }
                    const f4 d0 = 2.f * e0 * a.inv_n, d1 = 2.f * e1 * a.inv_n;
                    dbq2[0] += (d0[0] + d0[1]) + (d0[2] + d0[3]);   // the same in the four lane groups
                    dbq2[1] += (d1[0] + d1[1]) + (d1[2] + d1[3]);
                    // u of this chunk as B operands with the sum over x
                    wave_lds_fence();
                    tile_put<R::MT>(ts, lane, acc);
                    wave_lds_fence();
                    f4 zf[R::MT][4];
#pragma unroll
                    for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                        for (int s = 0; s < 4; ++s)
                            zf[mt][s] = *reinterpret_cast<const f4*>(ts + (mt * 16 + n16) * TLD + 16 * s + 4 * g);
                    f4 dz[R::MT][4] = {};
#pragma unroll 1
                    for (int pt = 0; pt < pm; ++pt) {
                        f4 h[4];
                        hidden(pt, h);
                        float* dp = dq + pt * QW;
                        const f4 qa = *reinterpret_cast<const f4*>(q2 + pt * 16 + 4 * g);
                        const f4 qb = *reinterpret_cast<const f4*>(q2 + P_MAX + pt * 16 + 4 * g);
                        f4 s1 = {}, sa = {}, sb = {};
#pragma unroll
                        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                float gv, gd;
                                gelu2(h[nt][r], gv, gd);
                                sa[r] = fmaf(d0[nt], gv, sa[r]);
                                sb[r] = fmaf(d1[nt], gv, sb[r]);
                                const float dh = (qa[r] * d0[nt] + qb[r] * d1[nt]) * gd;
                                s1[r] += dh;
                                h[nt][r] = dh;
                            }
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            s1[r] = row16_sum(s1[r]);
                            sa[r] = row16_sum(sa[r]);
                            sb[r] = row16_sum(sb[r]);
                        }
                        if (n16 == 0) {
                            f4* d = reinterpret_cast<f4*>(dp + R::MT * 256) + g;
                            d[0] += s1;
                            d[4] += sa;
                            d[8] += sb;
                        }
                        // dz = Q1^T dh
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int mt = 0; mt < R::MT; ++mt) {
                                const float w = Ql[(pt * 16 + 4 * g + r) * R::QLD + 16 * mt + n16];
#pragma unroll
                                for (int nt = 0; nt < 4; ++nt) dz[mt][nt] = mfma(w, h[nt][r], dz[mt][nt]);
                            }
                        // dQ1 += dh u^T over the chunk's columns
                        wave_lds_fence();
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            *reinterpret_cast<f4*>(ts + (4 * g + r) * TLD + 4 * n16) = f4{h[0][r], h[1][r], h[2][r], h[3][r]};
                        wave_lds_fence();
                        f4 q1[R::MT];
#pragma unroll
                        for (int mt = 0; mt < R::MT; ++mt) q1[mt] = *reinterpret_cast<const f4*>(dp + mt * 256 + 4 * lane);
#pragma unroll
                        for (int s = 0; s < 4; ++s) {
                            const f4 av = *reinterpret_cast<const f4*>(ts + n16 * TLD + 16 * s + 4 * g);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
#pragma unroll
                                for (int mt = 0; mt < R::MT; ++mt) q1[mt] = mfma(av[j], zf[mt][s][j], q1[mt]);
                        }
#pragma unroll
                        for (int mt = 0; mt < R::MT; ++mt) *reinterpret_cast<f4*>(dp + mt * 256 + 4 * lane) = q1[mt];
                    }
#pragma unroll
                    for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int c = mt * 16 + 4 * g + r;
                            if (C >= 16 || c < C)
                                *reinterpret_cast<f4*>(a.u + ((size_t)b * C + c) * NN + ro) =
                                    f4{dz[mt][0][r], dz[mt][1][r], dz[mt][2][r], dz[mt][3][r]};
                        }
                    wave_lds_fence();
                    tile_put<R::MT>(ts, lane, dz);
                    wave_lds_fence();
                    dft_chunk<C, M>(ts, a.FP, ch, lane, da);
                }
            }
        }
        if constexpr (TAIL != TAIL_INFER) dft_store<C, M>(tiles, lane, wv, nw, b, y, N, da, a.A);
    }
    if constexpr (TAIL == TAIL_TRAIN) {
        // this workgroup's partial sums: dQ1[P][C], dbq1[P], dQ2[2][P],
        // dbq2[2], summed over the waves in wave order; the loss
        float* pb = a.part + (size_t)blockIdx.x * a.pstride;
        dbq2[0] = row16_sum(dbq2[0]);
        dbq2[1] = row16_sum(dbq2[1]);
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) lacc += __shfl_xor(lacc, o, 64);
        auto wave_sum = [&](int n, int off) {
            __syncthreads();
            for (int e = threadIdx.x; e < n; e += blockDim.x) {
                float s = 0.f;
                for (int w = 0; w < nw; ++w) s += tiles[w * R::CP * TLD + e];
                pb[off + e] = s;
            }
            __syncthreads();
        };
        for (int pt = 0; pt < pm; ++pt) {
            const int np = min(16, a.P - 16 * pt);
            __syncthreads();
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt) {
                const f4 q1 = *reinterpret_cast<const f4*>(dq + pt * QW + mt * 256 + 4 * lane);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * mt + n16 < C) ts[(4 * g + r) * C + 16 * mt + n16] = q1[r];
            }
            wave_sum(np * C, 16 * pt * C);
        }
        __syncthreads();
        for (int i = lane; i < 3 * a.P; i += 64) {
            const int k = i / a.P, p = i % a.P;
            ts[i] = dq[(p / 16) * QW + R::MT * 256 + 16 * k + p % 16];
        }
        if (lane == 0) {
            ts[3 * a.P] = dbq2[0];
            ts[3 * a.P + 1] = dbq2[1];
        }
        wave_sum(3 * a.P + 2, a.P * C);
        double* dl = reinterpret_cast<double*>(tiles);
        if (lane == 0) dl[wv] = lacc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int w = 0; w < nw; ++w) s += dl[w];
            a.loss[blockIdx.x] = s * a.inv_n;
        }
    }
}

template <int C, int M> size_t bwd_lds(int nw)
{
    using R = Row<C, M>;
    return (size_t)nw * R::CP * TLD + R::CP * R::WLD + R::CP * (CIN_MAX + 1);
}

// Backward layer.  a.z = dL/du of this layer's output; per row
//   s = W^T du + Re(Bk conj F),  dL/du_below = s gelu'(u_below)
// with dW += du z^T (z = gelu(u_below), or lift(x) for the first layer) and
// db += du; the first layer instead ends in the lift's gradients from s.
// 0.30 ms at batch 8, 512^2, 32 channels (0.8 GB: 0.17 ms at the copy rate),
// against 0.32 + 1.6 ms for the pointwise kernel and its outer products.
template <int C, int M, bool LIFT>
__global__ void __launch_bounds__(64 * ROW_W) ROW_OCC(2) k_layer_bwd(RowArgs a)
{
    using R = Row<C, M>;
    extern __shared__ float sm[];
    const int N = a.N, nw = blockDim.x / 64, lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    const int n16 = lane % 16, g = lane / 16;
    float* tiles = sm;
    float* Wl = tiles + nw * R::CP * TLD;
    float* ll = Wl + R::CP * R::WLD;
    float* ts = tiles + wv * R::CP * TLD;
    const size_t NN = (size_t)N * N;
    for (int i = threadIdx.x; i < R::CP * C; i += blockDim.x) {
        const int c = i / C, k = i % C;
        Wl[c * R::WLD + k] = c < C ? bf2f(a.W[k * C + c]) : 0.f;   // transposed
    }
    if constexpr (C < R::CP)
        for (int i = threadIdx.x; i < (R::CP - C) * 2 * M; i += blockDim.x)
            Wl[(C + i / (2 * M)) * R::WLD + C + i % (2 * M)] = 0.f;
    if constexpr (LIFT) load_lift<C, R::CP>(ll, a);
    f4 dw[R::MT][R::MT] = {};
    f4 db[R::MT] = {};
    f4 dwp[LIFT ? CIN_MAX : 1][R::MT] = {}, dbp[LIFT ? R::MT : 1] = {};
    for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
        const int b = row / N, y = row % N;
        __syncthreads();
        load_bk<C, M>(Wl, a.Bk, b, y, N);
        __syncthreads();
        f4 da[R::MT][R::NT] = {};
        for (int ch = wv; ch < N / 64; ch += nw) {
            const int x0 = ch * 64 + 4 * n16;
            const size_t ro = (size_t)y * N + x0;
            f4 du[R::MT][4], uv[R::MT][4];
            f4 xin[CIN_MAX] = {};
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = 16 * mt + 4 * g + j;
                    const size_t o = ((size_t)b * C + (k < C ? k : 0)) * NN + ro;
                    du[mt][j] = *reinterpret_cast<const f4*>(a.z + o);
                    if constexpr (!LIFT) uv[mt][j] = *reinterpret_cast<const f4*>(a.uprev + o);
                }
            if constexpr (LIFT) {
#pragma unroll
                for (int q = 0; q < CIN_MAX; ++q)
                    if (q < a.cin) xin[q] = *reinterpret_cast<const f4*>(a.x + ((size_t)b * a.cin + q) * NN + ro);
            }
            if constexpr (C < R::CP) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * g + j >= C) du[0][j] = f4{0.f, 0.f, 0.f, 0.f};
            }
            // du as A operands with the sum over x
            wave_lds_fence();
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    *reinterpret_cast<f4*>(ts + (16 * mt + 4 * g + j) * TLD + 4 * n16) = du[mt][j];
                    db[mt][j] += (du[mt][j][0] + du[mt][j][1]) + (du[mt][j][2] + du[mt][j][3]);
                }
            wave_lds_fence();
            f4 df[R::MT][4];
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    df[mt][s] = *reinterpret_cast<const f4*>(ts + (mt * 16 + n16) * TLD + 16 * s + 4 * g);
            f4 acc[R::MT][4] = {};
            chunk_gemm<C, M>(Wl, a.FT, N, x0, lane, acc, [&](int kg, int j, int) { return du[kg < R::MT ? kg : 0][j]; });
            // z of the layer below, and dL/du below in place of s
            wave_lds_fence();
#pragma unroll
            for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = 16 * mt + 4 * g + j;
                    f4 zv;
                    if constexpr (LIFT) {
                        zv = lift4(ll + k * (CIN_MAX + 1), xin);
                        const f4 s = {acc[mt][0][j], acc[mt][1][j], acc[mt][2][j], acc[mt][3][j]};
                        dbp[LIFT ? mt : 0][j] += (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
                        for (int q = 0; q < CIN_MAX; ++q) {
                            const f4 t = s * xin[q];
                            dwp[LIFT ? q : 0][mt][j] += (t[0] + t[1]) + (t[2] + t[3]);
                        }
                    } else {
#pragma unroll
                        for (int nt = 0; nt < 4; ++nt) {
                            float gv, gd;
                            gelu2(uv[mt][j][nt], gv, gd);
                            zv[nt] = gv;
                            acc[mt][nt][j] *= gd;
                        }
                    }
                    *reinterpret_cast<f4*>(ts + k * TLD + 4 * n16) = zv;
                }
            wave_lds_fence();
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                f4 zf[R::MT];
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt)
                    zf[mt] = *reinterpret_cast<const f4*>(ts + (mt * 16 + n16) * TLD + 16 * s + 4 * g);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int mo = 0; mo < R::MT; ++mo)
#pragma unroll
                        for (int mi = 0; mi < R::MT; ++mi) dw[mo][mi] = mfma(df[mo][s][j], zf[mi][j], dw[mo][mi]);
            }
            if constexpr (!LIFT) {
#pragma unroll
                for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int c = mt * 16 + 4 * g + r;
                        if (C >= 16 || c < C)
                            *reinterpret_cast<f4*>(a.u + ((size_t)b * C + c) * NN + ro) =
                                f4{acc[mt][0][r], acc[mt][1][r], acc[mt][2][r], acc[mt][3][r]};
                    }
                wave_lds_fence();
                tile_put<R::MT>(ts, lane, acc);
                wave_lds_fence();
                dft_chunk<C, M>(ts, a.FP, ch, lane, da);
            }
        }
        if constexpr (!LIFT) dft_store<C, M>(tiles, lane, wv, nw, b, y, N, da, a.A);
    }
    // partial sums: dW[C][C], db[C], and for the first layer dWp[C][cin], dbp[C]
    float* pb = a.part + (size_t)blockIdx.x * a.pstride;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1)
#pragma unroll
        for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                db[mt][r] += __shfl_xor(db[mt][r], o, 64);
                if constexpr (LIFT) {
                    dbp[LIFT ? mt : 0][r] += __shfl_xor(dbp[LIFT ? mt : 0][r], o, 64);
#pragma unroll
                    for (int q = 0; q < CIN_MAX; ++q) dwp[LIFT ? q : 0][mt][r] += __shfl_xor(dwp[LIFT ? q : 0][mt][r], o, 64);
                }
            }
    __syncthreads();
#pragma unroll
    for (int mo = 0; mo < R::MT; ++mo)
#pragma unroll
        for (int mi = 0; mi < R::MT; ++mi)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                ts[(16 * mo + 4 * g + r) * R::CP + 16 * mi + n16] = dw[mo][mi][r];
    __syncthreads();
    for (int e = threadIdx.x; e < C * C; e += blockDim.x) {
        float s = 0.f;
        for (int w = 0; w < nw; ++w) s += tiles[w * R::CP * TLD + (e / C) * R::CP + e % C];
        pb[e] = s;
    }
    __syncthreads();
    if (n16 == 0) {
#pragma unroll
        for (int mt = 0; mt < R::MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = 16 * mt + 4 * g + r;
                if (c < C) {
                    ts[c] = db[mt][r];
                    if constexpr (LIFT) {
                        for (int q = 0; q < a.cin; ++q) ts[C + c * a.cin + q] = 0.f;
#pragma unroll
                        for (int q = 0; q < CIN_MAX; ++q)
                            if (q < a.cin) ts[C + c * a.cin + q] = dwp[LIFT ? q : 0][mt][r];
                        ts[C + C * a.cin + c] = dbp[LIFT ? mt : 0][r];
                    }
                }
            }
    }
    __syncthreads();
    const int nv = C + (LIFT ? C * a.cin + C : 0);
    for (int e = threadIdx.x; e < nv; e += blockDim.x) {
        float s = 0.f;
        for (int w = 0; w < nw; ++w) s += tiles[w * R::CP * TLD + e];
        pb[C * C + e] = s;
    }
}

// X[q][kx][j] = sum_y A[q][y][kx] G[y][j] for 16/M planes q per workgroup:
// complex products as FP32 matrix instructions over the real and imaginary
// columns, the 16 waves each a sixteenth of the rows y, summed in wave order.
// 8 us for 32 planes of 512 rows, 11 for 256 (launch and latency bound); one
// thread per (kx, j) walking all rows took 148 and 184 us: a serial chain.
constexpr int DY_W = 16;
template <int M>
__global__ void __launch_bounds__(64 * DY_W) k_dfty(const c32* __restrict__ A, const c32* __restrict__ G,
                                                    c32* __restrict__ X, int N)
{
    constexpr int PL = 16 / M, NT = M / 4;
    __shared__ float red[DY_W][16][4 * M];
    const int lane = threadIdx.x % 64, wv = threadIdx.x / 64, i = lane % 16, g = lane / 16;
    const int q0 = blockIdx.x * PL;
    const c32* Aq = A + (size_t)(q0 + i / M) * N * M + i % M;
    f4 acc[NT] = {};
    const int yb = wv * (N / DY_W);
#pragma unroll 8
    for (int s = 0; s < N / DY_W / 4; ++s) {
        const int y = yb + 4 * s + g;
        const c32 av = Aq[(size_t)y * M];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int n = nt * 16 + i, ri = n / (2 * M);
            const c32 gv = G[(size_t)y * 2 * M + n % (2 * M)];
            acc[nt] = mfma(av.x, ri ? gv.y : gv.x, acc[nt]);
            acc[nt] = mfma(av.y, ri ? gv.x : -gv.y, acc[nt]);
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wv][4 * g + r][nt * 16 + i] = acc[nt][r];
    __syncthreads();
    float* Xf = reinterpret_cast<float*>(X);
    for (int e = threadIdx.x; e < 16 * 4 * M; e += 64 * DY_W) {
        const int rr = e / (4 * M), n = e % (4 * M);
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < DY_W; ++w) s += red[w][rr][n];
        Xf[(((size_t)q0 * M + rr) * 2 * M + n % (2 * M)) * 2 + n / (2 * M)] = s;
    }
}

// Mode mixing and the inverse along y in one launch.  A workgroup forms the
// 2 M^2 modes of one output channel,
//   forward: Y[b][o][m] = s(m) sum_i X[b][i][m] R[i][o][m]
//   adjoint: Y[b][i][m] = s(m) sum_o X[b][o][m] conj(R[i][o][m])
// in LDS, and from them its share (blockIdx.z) of the rows
//   Bk[q][y][kx] = sum_j Y[q][kx][j] conj(G[y][j])
// as matrix products over (re, im) pairs.  7.5 us at batch 1, 15 at batch 8
// (512 rows, 32 channels), against 18 and 83 us for the two steps apart.
template <int C, int M>
__global__ void __launch_bounds__(512) k_mix_inv(const c32* __restrict__ X, const uint16_t* __restrict__ R,
                                                 const c32* __restrict__ G, c32* __restrict__ Bk, int N, int adjoint,
                                                 float inv_n2)
{
    constexpr int NM = 2 * M * M, NS = 512 / NM, YLD = 4 * M + 4, NT = 2 * M < 16 ? 1 : 2 * M / 16;
    __shared__ c32 ps[NS][NM];
    __shared__ __align__(16) float Ys[16 * YLD];
    const int o = blockIdx.x, b = blockIdx.y;
    {
        const int m = threadIdx.x % NM, part = threadIdx.x / NM;
        float yr = 0.f, yi = 0.f;
#pragma unroll 8
        for (int i = part; i < C; i += NS) {
            const size_t ridx = adjoint ? (((size_t)o * C + i) * NM + m) : (((size_t)i * C + o) * NM + m);
            const float rr = bf2f(R[2 * ridx]);
            const float ri = adjoint ? -bf2f(R[2 * ridx + 1]) : bf2f(R[2 * ridx + 1]);
            const c32 x = X[((size_t)b * C + i) * NM + m];
            yr += x.x * rr - x.y * ri;
            yi += x.x * ri + x.y * rr;
        }
        ps[part][m] = make_float2(yr, yi);
    }
    __syncthreads();
    if (threadIdx.x < NM) {
        const int m = threadIdx.x;
        float yr = 0.f, yi = 0.f;
#pragma unroll
        for (int p = 0; p < NS; ++p) {
            yr += ps[p][m].x;
            yi += ps[p][m].y;
        }
        const float s = (m / (2 * M) == 0 ? 1.f : 2.f) * inv_n2;
        float* d = Ys + (m / (2 * M)) * YLD + 2 * (m % (2 * M));
        d[0] = s * yr;
        d[1] = s * yi;
    }
    __syncthreads();
    const int lane = threadIdx.x % 64, wv = threadIdx.x / 64, n16 = lane % 16, g = lane / 16;
    const float* Gf = reinterpret_cast<const float*>(G);
    float* Bf = reinterpret_cast<float*>(Bk) + ((size_t)b * C + o) * N * (2 * M);
    const int ny = N / 16 / gridDim.z;          // row tiles of this workgroup
    const int t0 = blockIdx.z * ny;
    for (int t = t0 + wv; t < t0 + ny; t += 8) {
        f4 acc[NT] = {};
#pragma unroll
        for (int kg = 0; kg < M / 4; ++kg) {
            const f4 av = *reinterpret_cast<const f4*>(Gf + (size_t)(t * 16 + n16) * (4 * M) + 16 * kg + 4 * g);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int n = nt * 16 + n16, kx = n / 2 < M ? n / 2 : 0;
                const f4 v = *reinterpret_cast<const f4*>(Ys + kx * YLD + 16 * kg + 4 * g);
                const f4 bv = n % 2 ? f4{v[1], -v[0], v[3], -v[2]} : v;
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[nt] = mfma(av[j], bv[j], acc[nt]);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (nt * 16 + n16 < 2 * M) Bf[(size_t)(t * 16 + 4 * g + r) * (2 * M) + nt * 16 + n16] = acc[nt][r];
    }
}

// Weight gradients out of the row kernels' per-workgroup partial sums, and
// the loss: FP64 sums over the workgroups in a fixed order.  Value v of a
// record goes to g[v + shift of its segment].
constexpr int RED_SEG = 2 * L_MAX + 8;
struct RedArgs {
    const float* part;
    int nblk, nval, nseg;
    int nblk_head, head;        // workgroups of the projection's kernel, its first value
    int start[RED_SEG + 1];     // first value of each segment, then nval
    long dst[RED_SEG];          // offset of each segment in the gradient
    float* g;
    const double* loss;
    double* loss_out;
};
constexpr int RED_G = 16;
__global__ void __launch_bounds__(64 * RED_G) k_reduce_grad(RedArgs a)
{
    __shared__ double sh[RED_G][64];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int v = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (v < a.nval) {
#pragma unroll 8
        for (int k = w; k < (v < a.head ? a.nblk : a.nblk_head); k += RED_G) s += (double)a.part[(size_t)k * a.nval + v];
    }
    sh[w][lane] = s;
    __syncthreads();
    if (w == 0 && v < a.nval) {
#pragma unroll
        for (int k = 1; k < RED_G; ++k) s += sh[k][lane];
        int seg = 0;
        while (seg + 1 < a.nseg && v >= a.start[seg + 1]) ++seg;
        a.g[a.dst[seg] + v - a.start[seg]] = (float)s;
    }
    if (blockIdx.x == 0) {
        __syncthreads();
        double l = 0.0;
        for (int k = threadIdx.x; k < a.nblk_head; k += 64 * RED_G) l += a.loss[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
        if (lane == 0) sh[0][w] = l;
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = 0.0;
            for (int k = 0; k < RED_G; ++k) t += sh[0][k];
            *a.loss_out = t;
        }
    }
}

// dR[i][o][m] = s(m) sum_b Yb[b][o][m] conj(X[b][i][m])   (Yb = D du)
template <int C, int M>
__global__ void k_rgrad(const c32* __restrict__ Yb, const c32* __restrict__ X, float* __restrict__ dR, int B,
                        float inv_n2)
{
    constexpr int NM = 2 * M * M;
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (t >= (size_t)C * C * NM) return;
    const int m = (int)(t % NM), o = (int)((t / NM) % C), i = (int)(t / ((size_t)NM * C));
    float gr = 0.f, gi = 0.f;
    for (int b = 0; b < B; ++b) {
        const c32 yb = Yb[((size_t)b * C + o) * NM + m], x = X[((size_t)b * C + i) * NM + m];
        gr += yb.x * x.x + yb.y * x.y;
        gi += yb.y * x.x - yb.x * x.y;
    }
    const float s = (m / (2 * M) == 0 ? 1.f : 2.f) * inv_n2;
    dR[2 * t] = s * gr;
    dR[2 * t + 1] = s * gi;
}

// Adam on the FP32 masters, refreshed BF16 copies
__global__ void k_adam(float* __restrict__ w, uint16_t* __restrict__ wb, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v, size_t n, float lr, float b1, float b2,
                       float eps, float c1, float c2)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wn = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wn;
    wb[i] = f2bf(wn);
}

// masters rounded to BF16, BF16 copies
__global__ void k_to_bf16(float* __restrict__ w, uint16_t* __restrict__ wb, size_t n)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint16_t h = f2bf(w[i]);
    wb[i] = h;
    w[i] = bf2f(h);
}

__global__ void k_fill0(float* __restrict__ p, size_t n)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

// planar FP32 (re, im) planes -> interleaved FP64 psi; real_only drops Im;
// base (may be null) is added to Re psi
__global__ void k_to_psi(const float* __restrict__ out, const float* __restrict__ base, double* __restrict__ psi,
                         size_t NN, int real_only)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= NN) return;
    psi[2 * i] = (double)out[i] + (base ? (double)base[i] : 0.0);
    psi[2 * i + 1] = real_only ? 0.0 : (double)out[NN + i];
}

// Periodic coordinate of the particle potential (src/gpe_particle.f90:31-45):
// X(dx) = (1/c)(s + s^3/6 + s^5/40), s = sin(c dx), c = 1/2 on the 2 pi box
__device__ inline double pcoord(double d)
{
    const double s = sin(0.5 * d), s2 = s * s;
    return 2.0 * (s + s * s2 * (1.0 / 6.0) + s * s2 * s2 * (1.0 / 40.0));
}

// Input planes of one sample: x[0] = sum_v q_v exp(-r_v^2 / (2 sigma^2)),
// x[1] = (V0 / vnorm) sum_p exp(-r_p^2 / (2 d^2)), r from pcoord per axis,
// and with cin >= 3 x[2] = sqrt(max(0, (omega - V)/g)) (Thomas-Fermi).
// src: xv[nv], yv[nv], qv[nv] (as doubles), pos[2*nobs]
__global__ void k_features(const double* __restrict__ src, int nv, int nobs, int N, double sigma, double amp,
                           double d, double vnorm, double omega, double g, int cin, float* __restrict__ x)
{
    const size_t NN = (size_t)N * N;
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= NN) return;
    const double h = 2.0 * 3.14159265358979323846 / N;
    const double px = (double)(i % N) * h, py = (double)(i / N) * h;
    const double* xv = src;
    const double* yv = src + nv;
    const double* qv = src + 2 * nv;
    const double* pos = src + 3 * nv;
    const double is2 = 0.5 / (sigma * sigma), id2 = 0.5 / (d * d);
    double c = 0.0, v = 0.0;
    for (int k = 0; k < nv; ++k) {
        const double X = pcoord(px - xv[k]), Y = pcoord(py - yv[k]);
        c += qv[k] * exp(-(X * X + Y * Y) * is2);
    }
    for (int k = 0; k < nobs; ++k) {
        const double X = pcoord(px - pos[2 * k]), Y = pcoord(py - pos[2 * k + 1]);
        v += exp(-(X * X + Y * Y) * id2);
    }
    x[i] = (float)c;
    x[NN + i] = (float)(amp * v);
    if (cin >= 3) x[2 * NN + i] = (float)sqrt(fmax(0.0, (omega - vnorm * amp * v) / g));
    for (int k = 3; k < cin; ++k) x[k * NN + i] = 0.f;
}

// Thomas-Fermi guess from the potential plane: psi = sqrt(max(0, (omega - V)/g)), V = vnorm x[1]
__global__ void k_tf(const float* __restrict__ x, size_t NN, double omega, double g, double vnorm,
                     double* __restrict__ psi)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= NN) return;
    const double V = vnorm * (double)x[NN + i];
    psi[2 * i] = sqrt(fmax(0.0, (omega - V) / g));
    psi[2 * i + 1] = 0.0;
}

unsigned nblk(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

constexpr int FEAT_MAXV = 4096, FEAT_MAXO = 256;

}  // namespace

// ------------------------------------------------------------------ host --

struct vk_fno {
    int N = 0, cin = 0, C = 0, M = 0, L = 0, P = 0, B = 0;
    hipStream_t st = nullptr;
    size_t np = 0;
    size_t oWp = 0, obp = 0, oR[L_MAX] = {}, oW[L_MAX] = {}, ob[L_MAX] = {}, oQ1 = 0, obq1 = 0, oQ2 = 0, obq2 = 0;
    float *w = nullptr, *g = nullptr, *am = nullptr, *av = nullptr;
    uint16_t* wb = nullptr;
    c32* G = nullptr;
    float *FT = nullptr;      // the x table planar, [2M][N]
    f4 *FP = nullptr;         // the x table as B operands of the transform along x
    float *x = nullptr, *tgt = nullptr, *out = nullptr;
    float *u[L_MAX + 1] = {};   // u[1..L-1]; the last layer's stays in registers
    c32 *A = nullptr, *X[L_MAX] = {}, *Bk = nullptr, *Yb = nullptr;
    float *dz = nullptr, *du = nullptr;
    float* part = nullptr;    // per row workgroup: weight-gradient partial sums
    double* lpart = nullptr;  // the same for the loss, then the loss
    int nval = 0;             // partial sums per workgroup
    double* psi = nullptr;
    double* fsrc = nullptr;   // staging for the feature builder
    long step = 0;
    size_t NN() const { return (size_t)N * N; }
    int NM() const { return 2 * M * M; }
};

namespace {

// Row workgroups: a wave per 64 columns up to `most`, and as many
// workgroups as 16 waves per CU of 256 CUs are.
int row_waves(int N, int most) { return std::min(most, N / 64); }
int row_grid(int N, int rows, int most) { return std::min(rows, 4096 / row_waves(N, most)); }

int fno_alloc(vk_fno* f)
{
    const size_t NN = f->NN(), B = f->B, C = f->C, NM = f->NM();
    size_t o = 0;
    f->oWp = o, o += C * f->cin;
    f->obp = o, o += C;
    for (int l = 0; l < f->L; ++l) {
        f->oR[l] = o, o += 2 * C * C * NM;
        f->oW[l] = o, o += C * C;
        f->ob[l] = o, o += C;
    }
    f->oQ1 = o, o += (size_t)f->P * C;
    f->obq1 = o, o += f->P;
    f->oQ2 = o, o += 2 * (size_t)f->P;
    f->obq2 = o, o += 2;
    f->np = o;
    FCHK(hipMalloc(&f->w, o * 4));
    FCHK(hipMalloc(&f->g, o * 4));
    FCHK(hipMalloc(&f->am, o * 4));
    FCHK(hipMalloc(&f->av, o * 4));
    FCHK(hipMalloc(&f->wb, o * 2));
    FCHK(hipMemset(f->w, 0, o * 4));
    FCHK(hipMemset(f->wb, 0, o * 2));
    FCHK(hipMemset(f->g, 0, o * 4));
    FCHK(hipMemset(f->am, 0, o * 4));
    FCHK(hipMemset(f->av, 0, o * 4));
    FCHK(hipMalloc(&f->x, B * f->cin * NN * 4));
    FCHK(hipMalloc(&f->tgt, B * 2 * NN * 4));
    FCHK(hipMalloc(&f->out, B * 2 * NN * 4));
    for (int l = 1; l < f->L; ++l) FCHK(hipMalloc(&f->u[l], B * C * NN * 4));
    FCHK(hipMalloc(&f->A, B * C * f->N * f->M * 8));
    for (int l = 0; l < f->L; ++l) FCHK(hipMalloc(&f->X[l], B * C * NM * 8));
    FCHK(hipMalloc(&f->Yb, B * C * NM * 8));
    FCHK(hipMalloc(&f->Bk, B * C * f->N * f->M * 8));
    FCHK(hipMalloc(&f->dz, B * C * NN * 4));
    FCHK(hipMalloc(&f->du, B * C * NN * 4));
    FCHK(hipMalloc(&f->psi, NN * 16));
    FCHK(hipMalloc(&f->fsrc, (3 * FEAT_MAXV + 2 * FEAT_MAXO) * sizeof(double)));
    f->nval = (int)(f->L * (C * C + C) + C * f->cin + C + f->P * C + 3 * f->P + 2);
    const size_t ngrid = row_grid(f->N, f->B * f->N, ROW_W);   // the larger of the two
    FCHK(hipMalloc(&f->part, ngrid * f->nval * 4));
    FCHK(hipMalloc(&f->lpart, (ngrid + 1) * 8));
    // e^{-2 pi i k x / N}; the phase index k*x is reduced mod N exactly
    std::vector<c32> F((size_t)f->N * f->M), G((size_t)f->N * 2 * f->M);
    const double pi = 3.14159265358979323846;
    for (int x = 0; x < f->N; ++x) {
        for (int k = 0; k < f->M; ++k) {
            const double a = -2.0 * pi * (double)(((long)k * x) % f->N) / f->N;
            F[(size_t)x * f->M + k] = make_float2((float)cos(a), (float)sin(a));
        }
        for (int j = 0; j < 2 * f->M; ++j) {
            const long ky = j < f->M ? j : j - 2 * f->M;
            const long kk = ((ky * x) % f->N + f->N) % f->N;
            const double a = -2.0 * pi * (double)kk / f->N;
            G[(size_t)x * 2 * f->M + j] = make_float2((float)cos(a), (float)sin(a));
        }
    }
    // the x table planar, and as the lanes of the transform along x read it:
    // [chunk][s][column tile][lane] float4 over j, x = 64 chunk + 16 s +
    // 4 (lane/16) + j, column 2 kx + (re, im) = 16 tile + lane%16
    const int M2 = 2 * f->M, nt = std::max(1, M2 / 16);
    std::vector<float> FT((size_t)M2 * f->N), FP((size_t)f->N / 16 * nt * 64 * 4, 0.f);
    auto fv = [&](int x, int n) { const c32 e = F[(size_t)x * f->M + n / 2]; return n % 2 ? e.y : e.x; };
    for (int x = 0; x < f->N; ++x)
        for (int n = 0; n < M2; ++n) FT[(size_t)n * f->N + x] = fv(x, n);
    for (int t = 0; t < f->N / 16; ++t)
        for (int k = 0; k < nt; ++k)
            for (int l = 0; l < 64; ++l)
                for (int j = 0; j < 4; ++j)
                    if (16 * k + l % 16 < M2)
                        FP[(((size_t)t * nt + k) * 64 + l) * 4 + j] = fv(16 * t + 4 * (l / 16) + j, 16 * k + l % 16);
    FCHK(hipMalloc(&f->FT, FT.size() * 4));
    FCHK(hipMalloc(&f->FP, FP.size() * 4));
    FCHK(hipMalloc(&f->G, G.size() * 8));
    FCHK(hipMemcpy(f->FT, FT.data(), FT.size() * 4, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(f->FP, FP.data(), FP.size() * 4, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(f->G, G.data(), G.size() * 8, hipMemcpyHostToDevice));
    return 0;
}

template <int C, int M>
struct Net {
    static float inv_n2(const vk_fno* f) { return 1.0f / ((float)f->N * (float)f->N); }

    static void dfty(vk_fno* f, c32* X, int nb)
    {
        hipLaunchKernelGGL(k_dfty<M>, dim3(nb * C * M / 16), dim3(64 * DY_W), 0, f->st, (const c32*)f->A,
                           (const c32*)f->G, X, f->N);
    }

    // modes mixed and inverted along y: enough workgroups for half the CUs,
    // a row tile (16 rows) per wave at least
    static void mix_inv(vk_fno* f, const c32* X, int l, int nb, int adjoint)
    {
        int ys = 1;
        while (ys < 4 && nb * C * ys < 128 && (f->N / 16) % (2 * ys) == 0) ys *= 2;
        hipLaunchKernelGGL((k_mix_inv<C, M>), dim3(C, nb, ys), dim3(512), 0, f->st, X, f->wb + f->oR[l],
                           (const c32*)f->G, f->Bk, f->N, adjoint, inv_n2(f));
    }

    static RowArgs args(const vk_fno* f, int nb)
    {
        RowArgs a{};
        a.x = f->x;
        a.Wp = f->wb + f->oWp, a.bp = f->wb + f->obp;
        a.Bk = f->Bk, a.FT = f->FT, a.FP = f->FP, a.A = f->A;
        a.N = f->N, a.rows = nb * f->N, a.cin = f->cin;
        a.Q1 = f->wb + f->oQ1, a.bq1 = f->wb + f->obq1, a.Q2 = f->wb + f->oQ2, a.bq2 = f->wb + f->obq2;
        a.P = f->P, a.out = f->out, a.tgt = f->tgt;
        a.inv_n = 1.0f / (float)((size_t)nb * 2 * f->NN());
        a.loss = f->lpart;
        a.pstride = f->nval;
        return a;
    }

    template <class K>
    static int row_launch(vk_fno* f, K k, size_t lds_floats, const RowArgs& a, int most = ROW_W)
    {
        const size_t lds = lds_floats * 4;
        if (lds > 65536) FCHK(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k, dim3(row_grid(f->N, a.rows, most)), dim3(64 * row_waves(f->N, most)), lds, f->st, a);
        return 0;
    }

    // partial sums of layer l's row kernel in a workgroup's record, the
    // lift's after layer 0's and the projection's last
    static int rec(const vk_fno* f, int l) { return l * (C * C + C) + (l > 0 ? C * f->cin + C : 0); }

    static int forward(vk_fno* f, int nb, bool train)
    {
        const int nw = row_waves(f->N, ROW_W), nt = row_waves(f->N, ROW_W_TRAIN);
        int rc = row_launch(f, k_lift_dft<C, M>, (size_t)nw * Row<C, M>::CP * TLD + Row<C, M>::CP * (CIN_MAX + 1), args(f, nb));
        for (int l = 0; l < f->L && !rc; ++l) {
            dfty(f, f->X[l], nb);
            mix_inv(f, f->X[l], l, nb, 0);
            RowArgs a = args(f, nb);
            a.W = f->wb + f->oW[l], a.bias = f->wb + f->ob[l];
            a.z = f->u[l];
            const size_t lds = fwd_lds<C, M>(nw, l == f->L - 1);
            if (l < f->L - 1) {
                a.u = f->u[l + 1];
                rc = l == 0 ? row_launch(f, k_layer<C, M, true, TAIL_LAYER>, lds, a)
                            : row_launch(f, k_layer<C, M, false, TAIL_LAYER>, lds, a);
            } else if (train) {
                a.u = f->dz;
                a.part = f->part + rec(f, f->L);
                const size_t lds = fwd_lds<C, M>(nt, true) + (size_t)nt * dq_words<C, M>();
                rc = l == 0 ? row_launch(f, k_layer<C, M, true, TAIL_TRAIN>, lds, a, ROW_W_TRAIN)
                            : row_launch(f, k_layer<C, M, false, TAIL_TRAIN>, lds, a, ROW_W_TRAIN);
            } else {
                rc = l == 0 ? row_launch(f, k_layer<C, M, true, TAIL_INFER>, lds, a)
                            : row_launch(f, k_layer<C, M, false, TAIL_INFER>, lds, a);
            }
        }
        return rc;
    }

    // after forward(train): f->dz = dL/du_L, f->A its transform along x, the
    // projection's gradients and the loss in partial sums
    static int backward(vk_fno* f, int nb)
    {
        const int nw = row_waves(f->N, ROW_W);
        float *dcur = f->dz, *dnext = f->du;
        int rc = 0;
        for (int l = f->L - 1; l >= 0 && !rc; --l) {
            dfty(f, f->Yb, nb);
            hipLaunchKernelGGL((k_rgrad<C, M>), dim3(nblk((size_t)C * C * 2 * M * M, 256)), dim3(256), 0, f->st,
                               (const c32*)f->Yb, (const c32*)f->X[l], f->g + f->oR[l], nb, inv_n2(f));
            mix_inv(f, f->Yb, l, nb, 1);
            RowArgs a = args(f, nb);
            a.W = f->wb + f->oW[l];
            a.z = dcur, a.u = dnext, a.uprev = f->u[l];
            a.part = f->part + rec(f, l);
            rc = l == 0 ? row_launch(f, k_layer_bwd<C, M, true>, bwd_lds<C, M>(nw), a)
                        : row_launch(f, k_layer_bwd<C, M, false>, bwd_lds<C, M>(nw), a);
            std::swap(dcur, dnext);
        }
        if (rc) return rc;
        RedArgs d{};
        d.part = f->part, d.nblk = row_grid(f->N, nb * f->N, ROW_W), d.nval = f->nval;
        d.nblk_head = row_grid(f->N, nb * f->N, ROW_W_TRAIN), d.head = rec(f, f->L);
        d.g = f->g, d.loss = f->lpart, d.loss_out = f->lpart + row_grid(f->N, f->B * f->N, ROW_W);
        int at = 0;
        auto seg = [&](size_t dst, int n) { d.start[d.nseg] = at; d.dst[d.nseg++] = (long)dst; at += n; };
        for (int l = 0; l < f->L; ++l) {
            seg(f->oW[l], C * C);
            seg(f->ob[l], C);
            if (l == 0) {
                seg(f->oWp, C * f->cin);
                seg(f->obp, C);
            }
        }
        seg(f->oQ1, f->P * C);
        seg(f->obq1, f->P);
        seg(f->oQ2, 2 * f->P);
        seg(f->obq2, 2);
        d.start[d.nseg] = at;
        hipLaunchKernelGGL(k_reduce_grad, dim3(nblk(f->nval, 64)), dim3(64 * RED_G), 0, f->st, d);
        return 0;
    }
};

typedef int (*fwd_fn)(vk_fno*, int, bool);
typedef int (*bwd_fn)(vk_fno*, int);

int dispatch(const vk_fno* f, fwd_fn* fw, bwd_fn* bw)
{
    if (f->C == 32 && f->M == 16) {
        *fw = Net<32, 16>::forward, *bw = Net<32, 16>::backward;
    } else if (f->C == 16 && f->M == 8) {
        *fw = Net<16, 8>::forward, *bw = Net<16, 8>::backward;
    } else if (f->C == 8 && f->M == 4) {
        *fw = Net<8, 4>::forward, *bw = Net<8, 4>::backward;
    } else {
        return vk_set_error(VK_ERR_UNSUPPORTED, "fno: (width, modes) must be (32,16), (16,8) or (8,4)");
    }
    return 0;
}

int load_input(vk_fno* f, const float* x, int nb)
{
    FCHK(hipMemcpyAsync(f->x, x, (size_t)nb * f->cin * f->NN() * 4, hipMemcpyDefault, f->st));
    return 0;
}

}  // namespace

extern "C" {

int vk_fno_create(vk_fno** out, int N, int cin, int width, int modes, int layers, int proj, int batch)
{
    if (!out) return vk_set_error(VK_ERR_ARG, "fno_create: null handle pointer");
    *out = nullptr;
    if (N < 64 || N > 1024 || N % 64 || cin < 1 || cin > CIN_MAX || layers < 1 || layers > 8 || proj < 1 ||
        proj > 64 || batch < 1 || batch > 64 || 2 * modes > N)
        return vk_set_error(VK_ERR_ARG, "fno_create: N must be a multiple of 64 in [64, 1024]; cin <= 4, "
                                        "layers <= 8, proj <= 64, batch <= 64, 2*modes <= N");
    vk_fno probe;
    probe.C = width, probe.M = modes;
    fwd_fn a;
    bwd_fn b;
    int rc = dispatch(&probe, &a, &b);
    if (rc) return rc;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return vk_set_error(VK_ERR_HIP, "no ROCm device available");
    vk_fno* f = new vk_fno();
    f->N = N, f->cin = cin, f->C = width, f->M = modes, f->L = layers, f->P = proj, f->B = batch;
    if (hipStreamCreateWithFlags(&f->st, hipStreamNonBlocking) != hipSuccess) {
        delete f;
        return vk_set_error(VK_ERR_HIP, "fno: stream creation failed");
    }
    if ((rc = fno_alloc(f))) {
        vk_fno_destroy(f);
        return rc;
    }
    *out = f;
    return 0;
}

void vk_fno_destroy(vk_fno* f)
{
    if (!f) return;
    if (f->st) hipStreamSynchronize(f->st);
    void* ps[] = {f->w, f->g, f->am, f->av, f->wb, f->FT, f->FP, f->G, f->x, f->tgt, f->out, f->A, f->Yb,
                  f->Bk, f->dz, f->du, f->part, f->lpart, f->psi, f->fsrc};
    for (void* p : ps)
        if (p) hipFree(p);
    for (float* p : f->u)
        if (p) hipFree(p);
    for (c32* p : f->X)
        if (p) hipFree(p);
    if (f->st) hipStreamDestroy(f->st);
    delete f;
}

long vk_fno_nparams(const vk_fno* f) { return f ? (long)f->np : 0; }

int vk_fno_layout(const vk_fno* f, long* offsets)
{
    if (!f || !offsets) return vk_set_error(VK_ERR_ARG, "fno_layout: null");
    int k = 0;
    offsets[k++] = (long)f->oWp;
    offsets[k++] = (long)f->obp;
    for (int l = 0; l < f->L; ++l) {
        offsets[k++] = (long)f->oR[l];
        offsets[k++] = (long)f->oW[l];
        offsets[k++] = (long)f->ob[l];
    }
    offsets[k++] = (long)f->oQ1;
    offsets[k++] = (long)f->obq1;
    offsets[k++] = (long)f->oQ2;
    offsets[k++] = (long)f->obq2;
    offsets[k++] = (long)f->np;
    return k;
}

void* vk_fno_stream(const vk_fno* f) { return f ? (void*)f->st : nullptr; }

int vk_fno_set_params(vk_fno* f, const float* p)
{
    if (!f || !p) return vk_set_error(VK_ERR_ARG, "fno_set_params: null");
    FCHK(hipMemcpyAsync(f->w, p, f->np * 4, hipMemcpyDefault, f->st));
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(f->np, 256)), dim3(256), 0, f->st, f->w, f->wb, f->np);
    hipLaunchKernelGGL(k_fill0, dim3(nblk(f->np, 256)), dim3(256), 0, f->st, f->am, f->np);
    hipLaunchKernelGGL(k_fill0, dim3(nblk(f->np, 256)), dim3(256), 0, f->st, f->av, f->np);
    f->step = 0;
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    return 0;
}

int vk_fno_get_params(vk_fno* f, float* p)
{
    if (!f || !p) return vk_set_error(VK_ERR_ARG, "fno_get_params: null");
    std::vector<uint16_t> b(f->np);
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipMemcpy(b.data(), f->wb, f->np * 2, hipMemcpyDeviceToHost));
    for (size_t i = 0; i < f->np; ++i) p[i] = bf2f(b[i]);
    return 0;
}

int vk_fno_get_grad(vk_fno* f, float* gout)
{
    if (!f || !gout) return vk_set_error(VK_ERR_ARG, "fno_get_grad: null");
    // on f->st: a plain copy into device memory neither blocks the host nor is
    // ordered against this non-blocking stream, and the next step rewrites g
    FCHK(hipMemcpyAsync(gout, f->g, f->np * 4, hipMemcpyDefault, f->st));
    FCHK(hipStreamSynchronize(f->st));
    return 0;
}

int vk_fno_forward(vk_fno* f, const float* x, float* y, int nb)
{
    if (!f || !x || nb < 1 || nb > f->B) return vk_set_error(VK_ERR_ARG, "fno_forward: bad arguments");
    fwd_fn fw;
    bwd_fn bw;
    int rc = dispatch(f, &fw, &bw);
    if (rc || (rc = load_input(f, x, nb))) return rc;
    if ((rc = fw(f, nb, false))) return rc;
    if (y) FCHK(hipMemcpyAsync(y, f->out, (size_t)nb * 2 * f->NN() * 4, hipMemcpyDefault, f->st));
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    return 0;
}

int vk_fno_predict_psi(vk_fno* f, const float* x, double* psi, int flags)
{
    if (!f || !psi || (flags & ~(VK_FNO_REAL | VK_FNO_ADD_TF)) || ((flags & VK_FNO_ADD_TF) && f->cin < 3))
        return vk_set_error(VK_ERR_ARG, "fno_predict_psi: bad arguments");
    fwd_fn fw;
    bwd_fn bw;
    int rc = dispatch(f, &fw, &bw);
    if (rc || (x && (rc = load_input(f, x, 1)))) return rc;
    if ((rc = fw(f, 1, false))) return rc;
    const float* base = (flags & VK_FNO_ADD_TF) ? f->x + 2 * f->NN() : nullptr;
    hipLaunchKernelGGL(k_to_psi, dim3(nblk(f->NN(), 256)), dim3(256), 0, f->st, (const float*)f->out, base, f->psi,
                       f->NN(), flags & VK_FNO_REAL);
    FCHK(hipMemcpyAsync(psi, f->psi, f->NN() * 16, hipMemcpyDefault, f->st));
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    return 0;
}

int vk_fno_features(vk_fno* f, int nv, const double* xv, const double* yv, const int* qv, double sigma, int nobs,
                    const double* pos, double V0, double d, double vnorm, double omega, double g, float* x_out)
{
    if (!f || f->cin < 2 || nv < 0 || nv > FEAT_MAXV || nobs < 0 || nobs > FEAT_MAXO || (nv && (!xv || !yv || !qv)) ||
        (nobs && (!pos || !(d > 0.0))) || !(sigma > 0.0) || !(vnorm > 0.0) || !(g > 0.0))
        return vk_set_error(VK_ERR_ARG, "fno_features: bad arguments (nv <= 4096, nobs <= 256, cin >= 2, "
                                        "sigma, vnorm, g and d > 0)");
    std::vector<double> src(3 * (size_t)nv + 2 * (size_t)nobs);
    for (int k = 0; k < nv; ++k) {
        src[k] = xv[k];
        src[nv + k] = yv[k];
        src[2 * nv + k] = (double)qv[k];
    }
    for (int k = 0; k < 2 * nobs; ++k) src[3 * nv + k] = pos[k];
    FCHK(hipStreamSynchronize(f->st));
    if (!src.empty()) FCHK(hipMemcpy(f->fsrc, src.data(), src.size() * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_features, dim3(nblk(f->NN(), 256)), dim3(256), 0, f->st, (const double*)f->fsrc, nv, nobs,
                       f->N, sigma, V0 / vnorm, nobs ? d : 1.0, vnorm, omega, g, f->cin, f->x);
    if (x_out) FCHK(hipMemcpyAsync(x_out, f->x, (size_t)f->cin * f->NN() * 4, hipMemcpyDefault, f->st));
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    return 0;
}

int vk_fno_tf_guess(vk_fno* f, double omega, double g, double vnorm, double* psi)
{
    if (!f || !psi || f->cin < 2 || !(g > 0.0)) return vk_set_error(VK_ERR_ARG, "fno_tf_guess: bad arguments");
    hipLaunchKernelGGL(k_tf, dim3(nblk(f->NN(), 256)), dim3(256), 0, f->st, (const float*)f->x, f->NN(), omega, g,
                       vnorm, f->psi);
    FCHK(hipMemcpyAsync(psi, f->psi, f->NN() * 16, hipMemcpyDefault, f->st));
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    return 0;
}

int vk_fno_train_step(vk_fno* f, const float* x, const float* tgt, int nb, float lr, double* loss)
{
    if (!f || !x || !tgt || nb < 1 || nb > f->B || !(lr >= 0.f))
        return vk_set_error(VK_ERR_ARG, "fno_train_step: bad arguments");
    fwd_fn fw;
    bwd_fn bw;
    int rc = dispatch(f, &fw, &bw);
    if (rc || (rc = load_input(f, x, nb))) return rc;
    const size_t n = (size_t)nb * 2 * f->NN();
    FCHK(hipMemcpyAsync(f->tgt, tgt, n * 4, hipMemcpyDefault, f->st));
    double L = 0.0;
    if ((rc = fw(f, nb, true)) || (rc = bw(f, nb))) return rc;
    FCHK(hipMemcpyAsync(&L, f->lpart + row_grid(f->N, f->B * f->N, ROW_W), 8, hipMemcpyDeviceToHost, f->st));
    if (lr > 0.f) {
        f->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - powf(b1, (float)f->step), c2 = 1.f - powf(b2, (float)f->step);
        hipLaunchKernelGGL(k_adam, dim3(nblk(f->np, 256)), dim3(256), 0, f->st, f->w, f->wb, (const float*)f->g,
                           f->am, f->av, f->np, lr, b1, b2, 1e-8f, c1, c2);
    }
    FCHK(hipStreamSynchronize(f->st));
    FCHK(hipGetLastError());
    if (loss) *loss = L;
    return 0;
}

}  // extern "C"
