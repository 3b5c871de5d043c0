// SGEMM / CGEMM on FP32 MFMA for products with few tiles: a workgroup owns a 32 x 32
// tile of C and its eight waves share the depth.
//
// What bounds such products is the chain of one tile: a 64 x 64 tile walked by one
// workgroup takes 24 ns per k (51 where its operands' edges are checked), of which the
// MFMAs are 13, so 67 x 161 x 3714 took 137 us on six workgroups. Here a tile is a
// quarter of that, each wave walks an eighth of the depth in blocks of 32 (complex: 8),
// loaded straight into MFMA operand registers one block ahead (every element is used by
// one wave only, so LDS would add a copy and a barrier per slab), and the eight partial
// tiles are added in order through LDS. Rows beyond the matrix read the last row instead
// (their results are not stored) and only the depth's last block is checked, so ragged
// and unaligned operands run at the same speed: 16-byte loads need 4-byte alignment.
#include "gemm_variants.hpp"

#include <algorithm>

namespace icl {

constexpr int kWvT = 32;     // tile
constexpr int kWvWaves = 8;

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// Floats of one operand per lane and block: a block's products take 1024 cycles.
template <bool CPLX>
constexpr int kWvVals = CPLX ? 8 : 16;

// One lane's part of a block: row `x` (already at the lane's row), the k from k0 on that
// this half of the wave takes, zeros from K on. KC: k contiguous, else stride ld.
template <bool CPLX, bool KC>
struct WaveOperand {
    const float* x;
    long ld;
    static constexpr int C = CPLX ? 2 : 1;
    static constexpr int VALS = kWvVals<CPLX>, KS = VALS / C; // k per lane

    template <bool TAIL>
    __device__ __forceinline__ void load(int k0, int K, float (&v)[VALS]) const
    {
        if constexpr (KC && !TAIL) {
#pragma unroll
            for (int i = 0; i < VALS / 4; ++i) {
                const f32x4 u = *reinterpret_cast<const f32x4_any*>(x + (long)k0 * C + 4 * i);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * i + j] = u[j];
            }
        } else {
            const long step = KC ? 1 : ld;
#pragma unroll
            for (int i = 0; i < KS; ++i) {
                const int k = k0 + i;
                const float* p = x + (long)(TAIL ? min(k, K - 1) : k) * step * C;
#pragma unroll
                for (int j = 0; j < C; ++j) v[C * i + j] = !TAIL || k < K ? p[j] : 0.0f;
            }
        }
    }
};

template <bool CPLX, bool A_KC, bool B_KC, bool L3>
__global__ void __launch_bounds__(kWvWaves * 64, 4) wave_gemm_kernel(GemmArgs g, int conj_a, int conj_b)
{
    constexpr int C = CPLX ? 2 : 1;
    constexpr int LD = CPLX ? kWvT : 40; // 40: the two halves of a wave write different banks
    constexpr int VALS = kWvVals<CPLX>, HALF = VALS / C, BK = 2 * HALF;
    __shared__ float part[C][kWvWaves][kWvT][LD];
    if constexpr (L3)
        if (guarded_off(g)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    if constexpr (L3) {
        if (!tile_coords_level3<kWvT, kWvT>(g.write_tri, g.kband, (g.M + kWvT - 1) / kWvT, (g.N + kWvT - 1) / kWvT, tm, tn))
            return;
    } else
        tile_coords<8>((g.M + kWvT - 1) / kWvT, (g.N + kWvT - 1) / kWvT, tm, tn);
    const int m0 = tm * kWvT, n0 = tn * kWvT;
    int kb = 0, ke = g.K;
    if constexpr (L3)
        if (!tile_window<kWvT, kWvT>(g, m0, n0, kb, ke)) return;

    const int m = min(m0 + (lane & 31), g.M - 1), n = min(n0 + (lane & 31), g.N - 1);
    const WaveOperand<CPLX, A_KC> oa{g.A + C * (A_KC ? (long)m * g.lda : (long)m), g.lda};
    const WaveOperand<CPLX, B_KC> ob{g.B + C * (B_KC ? (long)n * g.ldb : (long)n), g.ldb};
    const int kh = HALF * (lane >> 5);
    const float sa = conj_a ? -1.0f : 1.0f, sb = conj_b ? -1.0f : 1.0f;

    f32x16 acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = f32x16{};
    auto load = [&](int k, float (&a)[VALS], float (&b)[VALS]) {
        if (k + BK <= ke) {
            oa.template load<false>(k + kh, ke, a);
            ob.template load<false>(k + kh, ke, b);
        } else {
            oa.template load<true>(k + kh, ke, a);
            ob.template load<true>(k + kh, ke, b);
        }
    };
    auto products = [&](const float (&a)[VALS], const float (&b)[VALS]) {
#pragma unroll
        for (int i = 0; i < HALF; ++i) {
            if constexpr (CPLX) {
                const float ar = a[2 * i], ai = sa * a[2 * i + 1], br = b[2 * i], bi = sb * b[2 * i + 1];
                acc[0] = mfma_32x32x2_f32(br, ar, acc[0]);
                acc[1] = mfma_32x32x2_f32(bi, ar, acc[1]);
                acc[0] = mfma_32x32x2_f32(bi, -ai, acc[0]);
                acc[1] = mfma_32x32x2_f32(br, ai, acc[1]);
            } else {
                acc[0] = mfma_32x32x2_f32(b[i], a[i], acc[0]);
            }
        }
    };
    constexpr int STEP = kWvWaves * BK;
    float a0[VALS], b0[VALS], a1[VALS], b1[VALS];
    int k = kb + wave * BK;
    if (k < ke) load(k, a0, b0);
    while (k < ke) {
        if (k + STEP < ke) load(k + STEP, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        products(a0, b0);
        k += STEP;
        if (k >= ke) break;
        if (k + STEP < ke) load(k + STEP, a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        products(a1, b1);
        k += STEP;
    }

    // Thread t stores rows t % 32 of columns t / 32 and t / 32 + 16.
    const int sm = m0 + (tid & 31), sn = n0 + (tid >> 5);
    const bool beta_zero = g.beta_re == 0.0f && (!CPLX || g.beta_im == 0.0f);
    float* const c0 = g.C + C * ((long)sn * g.ldc + sm);
    auto on = [&](int q) {
        if (sm >= g.M || sn + 16 * q >= g.N) return false;
        return !L3 || tri_writes(g.write_tri, sm, sn + 16 * q);
    };
    float old[2][C];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int c = 0; c < C; ++c) old[q][c] = !beta_zero && on(q) ? c0[C * (long)(16 * q) * g.ldc + c] : 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[c][wave][mfma32_row(lane, r)][lane & 31] = acc[c][r];
    __syncthreads();
    const TriMask tri(g.mask);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        float sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            sum[c] = part[c][0][(tid >> 5) + 16 * q][tid & 31];
#pragma unroll
            for (int w = 1; w < kWvWaves; ++w) sum[c] += part[c][w][(tid >> 5) + 16 * q][tid & 31];
        }
        if (!on(q)) continue;
        float* const c = c0 + C * (long)(16 * q) * g.ldc;
        if constexpr (CPLX) {
            const float xr = sum[0], xi = L3 && (g.cflags & ICL_CFLAG_CONJ_ACC) ? -sum[1] : sum[1];
            float vr = fmaf(g.alpha_re, xr, -g.alpha_im * xi);
            float vi = fmaf(g.alpha_re, xi, g.alpha_im * xr);
            if (!beta_zero) {
                vr += fmaf(g.beta_re, old[q][0], -g.beta_im * old[q][1]);
                vi += fmaf(g.beta_re, old[q][1], g.beta_im * old[q][0]);
            }
            if (L3 && (g.cflags & ICL_CFLAG_REAL_DIAG) && sm == sn + 16 * q) vi = 0.0f;
            *reinterpret_cast<f32x2*>(c) = f32x2{vr, vi};
        } else {
            const float v = beta_zero ? g.alpha_re * sum[0] : fmaf(g.beta_re, old[q][0], g.alpha_re * sum[0]);
            *c = tri.keep(sm, sn + 16 * q) ? v : 0.0f;
        }
    }
}

namespace {

template <bool CPLX, bool A_KC, bool B_KC>
hipError_t wave_run(const icl_gemm_args* g, int opa, int opb, hipStream_t s)
{
    const long tiles = gemm_tiles(g, kWvT, kWvT);
    if (tiles <= 0) return hipSuccess;
    if (tiles > 0x7fffffffL) return hipErrorInvalidValue;
    const auto kern = uses_level3(g) ? wave_gemm_kernel<CPLX, A_KC, B_KC, true> : wave_gemm_kernel<CPLX, A_KC, B_KC, false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(kWvWaves * 64), 0, s, *g, opa == 2, opb == 2);
    return hipGetLastError();
}

template <bool CPLX>
hipError_t wave_launch(const icl_gemm_args* g, int opa, int opb, int, void*, hipStream_t s)
{
    if (opa) return opb ? wave_run<CPLX, true, false>(g, opa, opb, s) : wave_run<CPLX, true, true>(g, opa, opb, s);
    return opb ? wave_run<CPLX, false, false>(g, opa, opb, s) : wave_run<CPLX, false, true>(g, opa, opb, s);
}

// Seconds: 3.5 us, and for each of the busiest CU's tiles 1.1 us (first loads, reduction)
// and 9 ns per k (complex 19.5); a triangle's tiles, found by a walk over the tile
// rows, 2.6 times that, and more than one round of them never pays (SSYRK 1856, k 98: 45
// us against 13). Fitted to 140 products: 512^3 7.8 us (64 x 64 tiles 17.5),
// 701 x 897 x 256 10.8 (18 to 24), 1024 x 1024 x 512 23.4 (18.8), 1991 x 3328 x 81 56 (28):
// from four rounds of tiles on the larger tile, which reads its operands half as often,
// is the faster one unless it has to check its edges.
template <bool CPLX>
double wave_estimate(const icl_gemm_args* g)
{
    constexpr long kCUs = 256;
    const long rounds = (gemm_tiles(g, kWvT, kWvT) + kCUs - 1) / kCUs;
    const double per_k = CPLX ? 19.5e-9 : 9.0e-9;
    if (g->write_tri != ICL_TRI_NONE && rounds > 1) return 1.0;
    const double each = (1.1e-6 + per_k * g->K) * (g->write_tri != ICL_TRI_NONE ? 2.6 : 1.0);
    if (g->kband != ICL_KBAND_NONE) return std::max(each, rounds * (1.1e-6 + 0.5 * per_k * g->K)) + 3.5e-6;
    return rounds * each + 3.5e-6;
}

} // namespace
} // namespace icl

#define ICL_GEMM_WAVE(name, kind, CPLX, TF)                                                                            \
    {name,                                                                                                             \
     kind,                                                                                                             \
     ICL_MATH_FP32,                                                                                                    \
     icl::kWvT,                                                                                                        \
     icl::kWvT,                                                                                                        \
     1,                                                                                                                \
     icl::kWvWaves * 64,                                                                                               \
     icl::wave_launch<CPLX>,                                                                                           \
     nullptr,                                                                                                          \
     TF,                                                                                                               \
     2,                                                                                                                \
     1,                                                                                                                \
     icl::wave_estimate<CPLX>}

static const icl_gemm_variant kTable[] = {
    ICL_GEMM_WAVE("sgemm_f32_wave_32x32", ICL_KIND_SGEMM, false, 70.0f),
    ICL_GEMM_WAVE("cgemm_f32_wave_32x32", ICL_KIND_CGEMM, true, 70.0f),
};
ICL_REGISTER_VARIANTS(kTable)
