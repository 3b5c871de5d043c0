// SGEMM / CGEMM on the BF16 matrix cores, every FP32 operand split into BF16 planes.
//
// Two planes (the split-BF16 math mode): x = hi + lo + e, hi = bf16(x), lo = bf16(x - hi),
// |e| <= 2^-16 |x|; a*b as hi hi + hi lo + lo hi, three BF16 MFMAs.
//
// Three planes (the FP32 math mode): x = x0 + x1 + x2 with x0 = bf16(x),
// x1 = bf16(x - x0), x2 = x - x0 - x1 (all round-to-nearest-even): x0 takes the leading
// 8 of the 24 significant bits, the remainder x - x0 has at most 16, x1 takes 8 of them
// and what is left (at most 7 bits) is a BF16 number itself, so nothing of the operand
// is lost. A product a*b is formed as a0 b0 + a0 b1 + a1 b0 + a0 b2 + a2 b0 + a1 b1, six
// BF16 MFMAs whose products are exact; the three terms left out are below 2^-23 |a b|
// (2^-26 root mean square), less than one FP32 rounding. The MFMA unit cuts what it adds
// off (downwards) a few bits below the largest summand, so the products must not meet a
// large sum: with the six accumulated straight into C's sums, the a1 b1 of A A^T's
// diagonal, all positive, were lost (2e-6 of the result). Each 32-deep slab's products
// therefore start from zero, the large a0 b0 last, and are added to the sums by
// ordinary additions, which round to nearest. Error against float64, root mean square
// relative to sums of same-signed products: 0.6e-7 (k = 512), 2.1e-7 (k = 8192), where
// FP32 MFMA, which rounds every fourth or second product, is at 3.1e-7 and 11.9e-7. The
// additions run beside the MFMAs and cost 3% at 8192^3.
//
// What bounds it: at 8192^3 the card's power. The three-plane kernel runs at 1570 to
// 1640 TFLOP/s of BF16 (registers alone reach 2050 on random data), its matrix pipes busy
// 83% of the cycles and the clock down to 1.75 to 1.9 GHz, where the FP32 MFMA kernel
// holds 2.3: the choices here are those that cost least energy per product,
// v_mfma_f32_16x16x32 (2048 TFLOP/s from registers against 1812 for 32x32x16), planes
// kept in registers over as many groups of products as possible (36 LDS reads per 192
// products; with the planes paired in 16-deep slabs, 56, it took 4.55 ms) and operands
// copied to LDS without passing through registers. Four waves of 128 x 128 (a third fewer
// LDS reads) do not fit the registers. SGEMM 8192^3: FP32 MFMA 7.75 ms, three planes
// 4.36 to 4.50 ms from card to card, of which 0.27 the prepass (4.9 TB/s); CGEMM 4096^3
// 3.88 -> 2.2 to 2.3 ms. Two planes 8192^3: 2.25 to 2.35 ms, 1.11 to 1.13 times the rate
// of 32x32x16 MFMA with fragments read just before use.
// The 128 x 128 tile, two workgroups per CU, serves outputs with too few large tiles;
// eight waves of 64 x 32, because a wave alone on its SIMD issues nothing beside its
// MFMAs (2048^3: 84 us, with four of 64 x 64 101).
#include "gemm_variants.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace icl {

constexpr int kSlabK = 32; // k per slab (one MFMA deep)
constexpr int kGroups = 4; // 16-byte chunks (groups of 8 k) per row, slab and plane

typedef __attribute__((address_space(3))) void sp_lds_void;

// ---------------------------------------------------------------------------
// Prepass. Packed layout P[slab][row / 64][plane][k / 8][row % 64][8]: 64 rows of one
// (slab, plane, k / 8) are 1 KB of contiguous memory, one LDS DMA instruction, and the LDS
// image keeps the rows contiguous (16 bytes apart: fragment reads are free of bank
// conflicts). What a wave copies of a slab lies at constant offsets from one 64-bit
// address, whatever the number of rows.
//
// Complex operands become real ones: op(A) (m x k) the 2m x 2k matrix with the
// 2 x 2 blocks [re -im; im re], op(B) the 2k x n matrix of its stacked parts, so
// that the real product's rows 2r and 2r + 1 are the parts of row r of the
// complex one: C's interleaved storage. Conjugation negates im.
//
// For three planes every element read is checked: outside 2^-110 <= |x| < 2^50 (or zero) the split
// is not exact or a partial product could overflow where the FP32 sum does not,
// and infinities and NaN would spread differently. Any such element stores the
// call's epoch into *guard, and the FP32 MFMA kernel computes the product instead. What
// such a call pays on top of that kernel: the blocks packed until one of them finds an
// element, and a launch that does nothing (1 in 1000 elements outside: 8192^3 7.80 ms of
// FP32 MFMA -> 7.88, 4096^3 988 -> 1012 us, 2048^3 143 -> 162, 1500^3 138 -> 144).
// ---------------------------------------------------------------------------
struct SplitSrc {
    const float* X;
    long ld;     // elements (complex ones when complex)
    int R, K;    // rows and depth (complex ones when complex)
    int Rpad;    // rows of the packed layout
    int kcontig; // element (r, k) at X[k + r * ld], else X[r + k * ld]
    int conj;
    __bf16* P;
};

__device__ __forceinline__ bool sp_outside(float x)
{
    const unsigned u = __builtin_bit_cast(unsigned, x) & 0x7fffffffu;
    return u != 0 && (u >> 23) - 17u > 159u;
}

template <int PLANES, bool CPLX>
__global__ void __launch_bounds__(256)
split_pack_kernel(SplitSrc a, SplitSrc b, int ablocks, int slabs, unsigned long long* guard, unsigned long long epoch)
{
    __shared__ float T[64][64 + 1];
    const bool is_a = (int)blockIdx.x < ablocks;
    SplitSrc o = is_a ? a : b;
    const int r0 = (is_a ? (int)blockIdx.x : (int)blockIdx.x - ablocks) * 64; // packed row
    const int by = (int)(blockIdx.y + gridDim.y * blockIdx.z), k0 = by * 64;  // packed k
    if (2 * by >= slabs) return; // the last layer of a deep grid
    // Nothing is read or packed any more once an element outside the range has been found
    // (waves may see that apart: all of them go through the barrier).
    const bool off = PLANES == 3 && __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(guard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch);
    if (off) o.R = 0;
    const int t = threadIdx.x;
    bool bad = false;
    if constexpr (!CPLX) {
        float v[16];
        const int in = t & 63, ob = t >> 6; // index along the contiguous dimension, across it (+ 4 i)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = r0 + (o.kcontig ? ob + 4 * i : in), k = k0 + (o.kcontig ? in : ob + 4 * i);
            v[i] = (r < o.R && k < o.K) ? o.X[o.kcontig ? (long)r * o.ld + k : (long)k * o.ld + r] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (PLANES == 3) bad |= sp_outside(v[i]);
            T[o.kcontig ? ob + 4 * i : in][o.kcontig ? in : ob + 4 * i] = v[i];
        }
    } else {
        // op(A): 32 complex rows x 32 complex k; op(B): 64 rows x 32 complex k.
        const int cr0 = is_a ? r0 / 2 : r0, ck0 = k0 / 2;
        const int wide = (is_a || o.kcontig) ? 32 : 64; // elements along the contiguous dimension
        const int in = t % wide, ob = t / wide, step = 256 / wide;
        f32x2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = f32x2{0.0f, 0.0f};
            if (is_a && i >= 4) continue;
            const int r = cr0 + (o.kcontig ? ob + step * i : in), k = ck0 + (o.kcontig ? in : ob + step * i);
            if (r < o.R && k < o.K)
                v[i] = *reinterpret_cast<const f32x2*>(o.X + 2 * (o.kcontig ? (long)r * o.ld + k : (long)k * o.ld + r));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (is_a && i >= 4) continue;
            const int r = o.kcontig ? ob + step * i : in, k = o.kcontig ? in : ob + step * i;
            const float re = v[i][0], im = o.conj ? -v[i][1] : v[i][1];
            if (PLANES == 3) bad |= sp_outside(re) || sp_outside(im);
            if (is_a) {
                T[2 * r][2 * k] = re;
                T[2 * r][2 * k + 1] = -im;
                T[2 * r + 1][2 * k] = im;
                T[2 * r + 1][2 * k + 1] = re;
            } else {
                T[r][2 * k] = re;
                T[r][2 * k + 1] = im;
            }
        }
    }
    if (PLANES == 3 && bad) *guard = epoch; // (an atomic store of every such lane: 2048^3 161 -> 243 us)
    __syncthreads();
    // wave w writes k = 16 w .. 16 w + 15 of slab pair by, lane = row: 1 KB per store
    const int w = t >> 6, r = t & 63, ks = 2 * by + (w >> 1);
    if (off || ks >= slabs) return;
    bf16x8 out[PLANES][2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float x = T[r][16 * w + i];
        if constexpr (PLANES == 3) {
            const __bf16 h0 = (__bf16)x;
            const float x1 = x - (float)h0;
            const __bf16 h1 = (__bf16)x1;
            out[0][i / 8][i % 8] = h0;
            out[1][i / 8][i % 8] = h1;
            out[2][i / 8][i % 8] = (__bf16)(x1 - (float)h1);
        } else {
            __bf16 hi, lo;
            split_bf16(x, hi, lo);
            out[0][i / 8][i % 8] = hi;
            out[1][i / 8][i % 8] = lo;
        }
    }
    __bf16* dst = o.P + ((size_t)ks * o.Rpad + r0) * (PLANES * kGroups * 8) + (2 * (w & 1) * 64 + r) * 8;
#pragma unroll
    for (int p = 0; p < PLANES; ++p)
#pragma unroll
        for (int c = 0; c < 2; ++c)
            *reinterpret_cast<bf16x8*>(dst + (kGroups * p + c) * (64 * 8)) = out[p][c];
}

// ---------------------------------------------------------------------------
// GEMM on the packed operands
// ---------------------------------------------------------------------------
struct SplitArgs {
    icl_gemm_args g; // A, B unused
    const __bf16* Ap;
    const __bf16* Bp;
    int Mpad, Npad; // packed rows of op(A) and of op(B)^T
    int slabs;
    const unsigned long long* guard; // three planes only
    unsigned long long epoch;
    int whole, splits; // tiles from `whole` on run in `splits` parts of their depth
    float* partial;
};

// T x T tiles of packed rows, WVM x WVN waves. LDS is a ring of RING blocks, each the
// T rows of one plane of one operand's slab.
template <int T_, int WVM_, int WVN_>
struct SplitCfg {
    static constexpr int T = T_, WVM = WVM_, WVN = WVN_;
    static constexpr int NW = WVM * WVN, NT = NW * 64;
    static constexpr int WM = T / WVM, WN = T / WVN, FM = WM / 16, FN = WN / 16;
    static constexpr int RING = 10, BLOCK = T * kSlabK * 2; // bytes
    static constexpr size_t LDS_BYTES = (size_t)RING * BLOCK;
    static constexpr int RB = T / 64; // 64-row groups
    static constexpr int COPIES = BLOCK / (NW * 1024); // per wave and block, 1 KB each
    static_assert(BLOCK == COPIES * NW * 1024 && NW % RB == 0, "whole copies");
};

// s_waitcnt immediate (expcnt not waited for): at most `vm` vector-memory
// operations outstanding and no LDS operation.
constexpr int sp_wait(int vm) { return 0x70 | (vm & 15) | (vm >> 4) << 14; }

__device__ __forceinline__ void sp_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Fragments [FROM, TO) of one plane: frag[f] = row rb + 16 f + (lane & 15), k = 8 (lane / 16) .. + 7.
template <int ROWS, int FROM, int TO, int F>
__device__ __forceinline__ void sp_frag(const unsigned char* S, int rb, int lane, bf16x8 (&frag)[F])
{
#pragma unroll
    for (int f = FROM; f < TO; ++f)
        frag[f] = *reinterpret_cast<const bf16x8*>(S + ((lane >> 4) * ROWS + rb + 16 * f + (lane & 15)) * 16);
}

template <int ROWS>
__device__ __forceinline__ bf16x8 sp_frag1(const unsigned char* S, int row, int lane)
{
    return *reinterpret_cast<const bf16x8*>(S + ((lane >> 4) * ROWS + row + (lane & 15)) * 16);
}

// f(i) for the constants i in [FROM, TO).
template <int FROM, int TO, typename F>
__device__ __forceinline__ void sp_each(const F& f)
{
    if constexpr (FROM < TO) {
        f(std::integral_constant<int, FROM>{});
        sp_each<FROM + 1, TO>(f);
    }
}

// t[j] (+)= b[j] a.
template <bool FIRST, int FN>
__device__ __forceinline__ void sp_products(const bf16x8 (&b)[FN], bf16x8 a, f32x4 (&t)[FN])
{
#pragma unroll
    for (int j = 0; j < FN; ++j)
        t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a, FIRST ? f32x4{} : t[j], 0, 0, 0);
}

// c += a b. The builtin, not an asm statement: the compiler knows its latency and the
// waits that it needs before its operands are written and its sum is read.
// Lane l supplies a = A[l % 16][8 (l / 16) .. + 7] and b = B[8 (l / 16) .. + 7][l % 16];
// register r of c is D[4 (l / 16) + r][l % 16].
__device__ __forceinline__ void sp_mfma1(bf16x8 a, bf16x8 b, f32x4& c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Waits for the last copies: LDS may be another workgroup's after this one's end.
__device__ __forceinline__ void sp_drain()
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// acc += b a over the wave's block rows [FROM, TO).
template <int FROM, int TO, int FM, int FN>
__device__ __forceinline__ void sp_mfma(const bf16x8 (&b)[FN], const bf16x8 (&a)[FM], f32x4 (&acc)[FM][FN])
{
#pragma unroll
    for (int i = FROM; i < TO; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) sp_mfma1(b[j], a[i], acc[i][j]);
}

// The same, calling after(i) behind the products of row i (i a constant): operand
// reads and copies run under the products of the next rows.
template <int FROM, int TO, int FM, int FN, typename F>
__device__ __forceinline__ void sp_rows(const bf16x8 (&b)[FN], const bf16x8 (&a)[FM], f32x4 (&acc)[FM][FN],
                                        const F& after)
{
    if constexpr (FROM < TO) {
        sp_mfma<FROM, FROM + 1>(b, a, acc);
        __builtin_amdgcn_sched_barrier(0);
        after(std::integral_constant<int, FROM>{});
        __builtin_amdgcn_sched_barrier(0);
        sp_rows<FROM + 1, TO>(b, a, acc, after);
    }
}

// The lane's value of its neighbour lane ^ 1.
__device__ __forceinline__ float sp_neighbour(float x)
{
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1 /* quad_perm 1,0,3,2 */, 0xf, 0xf, true));
}

// Columns nl + c of a lane's row that are stored (or kept by a mask): those with
// first <= nl + c < end, one subtraction and one comparison per element.
struct SpColumns {
    int from;
    unsigned count;
    __device__ __forceinline__ SpColumns(int nl, int first, int end)
        : from(nl - first), count((unsigned)max(end - first, 0))
    {
    }
    __device__ __forceinline__ bool has(int c) const { return (unsigned)(from + c) < count; }
};

// Stores G rows of FN 16 x 16 blocks, block row i at row0 + 16 i: register r of block j
// holds column ncol0 + 16 j + 4 (lane / 16) + r, the lane row `row0` (complex: the part
// lane & 1 of complex row row0 / 2). CHECK: bounds, triangle and mask are tested per
// element, as a range of columns per row. C is read for the whole group before anything
// is stored: row by row of blocks each waited for memory again (2048 x 2048 x 256 with
// beta = 1: 35 us of 128 x 128 tiles, 12 of them products). The checked stores take 0.9
// us of a call (100 x 90 x 256, two planes, 11.8 us; 128 x 128 x 256 10.9); each waiting
// for the one before, their tests kept from the reads in spilled scalar registers, they
// took 4.4.
template <bool CPLX, bool CHECK, int G, int FN>
__device__ __forceinline__ void sp_store(const GemmArgs& g, const f32x4 (&acc)[G][FN], int row0, int ncol0, int lane)
{
    const int nl = ncol0 + 4 * (lane >> 4);
    const long cstep = CPLX ? 2 * g.ldc : g.ldc;
    float* const c0 = g.C + (CPLX ? 2L : 1L) * (long)nl * g.ldc + row0;
    const bool odd = CPLX && (lane & 1);
    const bool beta_zero = g.beta_re == 0.0f && (!CPLX || g.beta_im == 0.0f);
    auto m_of = [&](int i) { return (row0 + 16 * i) >> (CPLX ? 1 : 0); };
    auto stored = [&](int i) {
        const int m = m_of(i), tri = g.write_tri & 3;
        return SpColumns(nl, tri == ICL_TRI_UPPER ? m : 0,
                         !CHECK ? INT_MAX : m >= g.M ? 0 : tri == ICL_TRI_LOWER ? min(m + 1, g.N) : g.N);
    };
    auto kept = [&](int i) {
        const int m = m_of(i), strict = g.mask == kMaskLowerStrict || g.mask == kMaskUpperStrict;
        const bool lower = g.mask == kMaskLower || g.mask == kMaskLowerStrict;
        return SpColumns(nl, g.mask == kMaskNone || lower ? 0 : m + strict, lower ? m + 1 - strict : INT_MAX);
    };
    float old[G][FN][4];
    if (!beta_zero) {
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const SpColumns on = stored(i);
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    old[i][j][r] = !CHECK || on.has(16 * j + r) ? c0[16 * i + (16 * j + r) * cstep] : 0.0f;
        }
        // Waited for here: left to their uses, the compiler waits at each of them, beta = 0
        // or not, for everything outstanding, which by then is the store before it.
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(old[i][j][r]));
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
        SpColumns on = stored(i);
        const SpColumns keep = kept(i);
        if (CHECK) asm volatile("" : "+v"(on.from)); // tested again, not kept
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v;
                if constexpr (CPLX) {
                    // even lanes: alpha_re re - alpha_im im; odd lanes: alpha_re im + alpha_im re
                    const float own = odd && (g.cflags & ICL_CFLAG_CONJ_ACC) ? -acc[i][j][r] : acc[i][j][r];
                    const float x = sp_neighbour(own), oth = odd ? x : -x;
                    v = fmaf(g.alpha_re, own, g.alpha_im * oth);
                    if (!beta_zero) {
                        const float y = sp_neighbour(old[i][j][r]), oldoth = odd ? y : -y;
                        v += fmaf(g.beta_re, old[i][j][r], g.beta_im * oldoth);
                    }
                    if (odd && (g.cflags & ICL_CFLAG_REAL_DIAG) && m_of(i) == nl + 16 * j + r) v = 0.0f;
                } else {
                    v = beta_zero ? g.alpha_re * acc[i][j][r] : fmaf(g.beta_re, old[i][j][r], g.alpha_re * acc[i][j][r]);
                }
                if (CHECK && !CPLX && !keep.has(16 * j + r)) v = 0.0f;
                if (!CHECK || on.has(16 * j + r)) c0[16 * i + (16 * j + r) * cstep] = v;
            }
    }
}

// T in rows of the packed operands: a complex tile has T / 2 rows.
//
// The copies run through the LDS ring as one sequence of blocks, block q in slot
// q % RING, and at two points of each slab a barrier frees slots for the blocks RING
// places on.
// Three planes: the blocks b2 b1 b0 a0 a1 a2. The slab's planes of op(B) are held in
// registers, those of op(A) pass through row by row of blocks, each row's products in
// the order a0 b2, a1 b1, a0 b1, a2 b0, a1 b0, a0 b0: in the last row the planes of op(B)
// fall free one after the other and the next slab's are read over them. op(B)'s slots
// are free after the first row, op(A)'s before the last.
// Two planes: a1 b0, a0 b1, a0 b0 into the sums, the blocks a1 b0 a0 b1, all in registers
// in the second group.
//
// A copy has two to six rows' products to arrive in, two workgroups' for 128 x 128 tiles
// (a ring of 20 for one of them changed nothing).
//
// The tiles from p.whole on, which would leave CUs idle in the launch's last round of
// workgroups, split their slabs over p.splits workgroups each, which leave their sums in
// p.partial for split_reduce_kernel. The parts of one depth range are neighbours (and on
// one XCD), so that they share operand panels.
template <int T, int WVM, int WVN, int PLANES, bool CPLX>
__global__ void __launch_bounds__(WVM* WVN * 64, T == 256 ? 2 : 4) split_gemm_kernel(SplitArgs p)
{
    using Cfg = SplitCfg<T, WVM, WVN>;
    constexpr int RING = Cfg::RING, COPIES = Cfg::COPIES;
    constexpr int ROW = CPLX ? 2 : 1; // packed rows (and k) per element
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_sp[];
    if (PLANES == 3 && *p.guard == p.epoch) return;
    const icl_gemm_args& g = p.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave % WVM) * Cfg::WM;
    const int wn0 = (wave / WVM) * Cfg::WN;
    const bool split = (int)blockIdx.x >= p.whole;
    const int rest = ((int)gridDim.x - p.whole) / p.splits; // tiles in parts
    int z = 0, tile;
    if (split) {
        if (g.kband) { // the longest window's parts first
            const int u = (int)blockIdx.x - p.whole;
            z = u % p.splits;
            tile = u / p.splits + p.whole;
        } else {
            const int u = xcd_id(blockIdx.x - p.whole, gridDim.x - p.whole);
            z = u / rest;
            tile = u - z * rest + p.whole;
        }
    } else {
        tile = g.kband ? (int)blockIdx.x : xcd_id(blockIdx.x, p.whole);
    }
    const int parts = split ? p.splits : 1;
    int tm, tn;
    if (!tile_level3<T / ROW, T>(tile, g.write_tri, g.kband, (ROW * g.M + T - 1) / T, (g.N + T - 1) / T, tm, tn)) return;
    int ks0 = 0, ks1 = p.slabs; // slabs [ks0, ks1) of the tile's k window, then of this part of it
    if (g.write_tri | g.kband) {
        int kb = 0, ke = 0;
        if (!tile_window<T / ROW, T>(g, tm * (T / ROW), tn * T, kb, ke)) return;
        ks0 = kb * ROW / kSlabK;
        ks1 = ke > kb ? (ke * ROW + kSlabK - 1) / kSlabK : ks0;
    }
    const int window = ks1 - ks0;
    ks1 = ks0 + window * (z + 1) / parts;
    ks0 += window * z / parts;
    const int m0 = tm * T, n0 = tn * T; // packed rows

    // This wave's copies of a block: the k groups wave / RB + (NW / RB) i of 64 rows.
    constexpr int ROW_BYTES = PLANES * kGroups * 16; // of one packed row of a slab
    const size_t a_slab = (size_t)p.Mpad * ROW_BYTES, b_slab = (size_t)p.Npad * ROW_BYTES;
    const size_t a_row = (size_t)(m0 + 64 * (wave % Cfg::RB)), b_row = (size_t)(n0 + 64 * (wave % Cfg::RB));
    const char* a_src = reinterpret_cast<const char*>(p.Ap) + ks0 * a_slab + a_row * ROW_BYTES + wave / Cfg::RB * 1024;
    const char* b_src = reinterpret_cast<const char*>(p.Bp) + ks0 * b_slab + b_row * ROW_BYTES + wave / Cfg::RB * 1024;
    const int loff = lane * 16;
    const int n = ks1 - ks0;
    // Part `i` of the copy of a slab's block c to the ring slot at `slot` (bytes), src
    // being the slab's first byte of op(A) / op(B). A buffer load: its address stays
    // scalar, and a global load would count as a FLAT access, after which the compiler
    // waits for all LDS reads at once. (A layout with all rows of a plane together reached
    // past 32-bit offsets and extents from 2^24 rows on.)
    constexpr int PER_SLAB = 2 * PLANES, KSTEP = Cfg::NW / Cfg::RB;
    auto copy = [&](const char* a, const char* b, int c, int slot, int i) {
        const bool of_a = PLANES == 3 ? c >= 3 : (c == 0 || c == 2);
        const int plane = PLANES == 3 ? (c < 3 ? 2 - c : c - 3) : (c == 0 || c == 3 ? 1 : 0);
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(of_a ? a : b), 0, 64 * ROW_BYTES, 0x20000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (sp_lds_void*)(lds_sp + slot + (wave + Cfg::NW * i) * 1024), 16,
                                                 loff, (kGroups * plane + KSTEP * i) * 1024, 0, 0);
    };

    f32x4 acc[Cfg::FM][Cfg::FN];
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::FN; ++j) acc[i][j] = f32x4{};

    if (n > 0) {
        constexpr int FM = Cfg::FM, FN = Cfg::FN, BLK = Cfg::BLOCK;
        // The copies run RING blocks ahead: into slab s's slot j goes block AHEAD + j of
        // slab s + DIST, from the pointers (a1, b1), or (a2, b2) when that is one of the
        // slab after it. Past the last slab that one is copied again, to slots nothing
        // reads any more: the number of copies in flight stays the same.
        constexpr int DIST = RING / PER_SLAB, AHEAD = RING % PER_SLAB;
        const char *a1 = a_src + min(DIST, n - 1) * a_slab, *a2 = a_src + min(DIST + 1, n - 1) * a_slab;
        const char *b1p = b_src + min(DIST, n - 1) * b_slab, *b2p = b_src + min(DIST + 1, n - 1) * b_slab;
        auto copy_to = [&](int j, int slot, int i) {
            const bool next = AHEAD + j >= PER_SLAB;
            copy(next ? a2 : a1, next ? b2p : b1p, (AHEAD + j) % PER_SLAB, slot, i);
        };
        auto advance = [&](int s) {
            const bool more = s + DIST + 2 < n;
            a1 = a2, b1p = b2p;
            a2 += more ? a_slab : 0;
            b2p += more ? b_slab : 0;
        };
        int head = 0; // ring slot (bytes) of the slab's first block
        auto slot = [&](int c) {
            const int q = head + c * BLK;
            return q < RING * BLK ? q : q - RING * BLK;
        };
#pragma unroll
        for (int q = 0; q < RING; ++q) {
            const long s = min(q / PER_SLAB, n - 1);
#pragma unroll
            for (int i = 0; i < COPIES; ++i)
                copy(a_src + s * a_slab, b_src + s * b_slab, q % PER_SLAB, q * BLK, i);
        }
        __builtin_amdgcn_s_waitcnt(sp_wait(COPIES * (RING - (PLANES == 3 ? 6 : 4)))); // the first blocks read are there
        sp_barrier();
        if constexpr (PLANES == 3) {
            bf16x8 a[2][3], b[3][FN]; // planes of two block rows of op(A), of op(B)'s slab
            f32x4 t[2][FN];           // a slab's products of one block row
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                sp_frag<T, 0, FN>(lds_sp + (2 - q) * BLK, wn0, lane, b[q]);
                a[0][q] = sp_frag1<T>(lds_sp + (3 + q) * BLK, wm0, lane);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) t[1][j] = f32x4{};
            for (int s = 0; s < n; ++s) {
                const int sa[3] = {slot(3), slot(4), slot(5)};
                sp_each<0, FM>([&](auto row) {
                    constexpr int i = row, cur = i & 1, nxt = cur ^ 1;
                    constexpr bool last = i == FM - 1;
                    int na[3] = {sa[0], sa[1], sa[2]}; // where the next row's planes are
                    if constexpr (last) {
                        // The next slab's blocks are there once only the one copied
                        // after them may be outstanding; all waves have read this slab's.
                        __builtin_amdgcn_s_waitcnt(sp_wait(COPIES * (RING - 9)));
                        sp_barrier();
                        head = slot(6);
#pragma unroll
                        for (int q = 0; q < 3; ++q) na[q] = slot(3 + q);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    constexpr int next_row = last ? 0 : 16 * (i + 1);
                    sp_products<true>(b[2], a[cur][0], t[cur]); // a0 b2
                    if constexpr (last) {
                        sp_frag<T, 0, FN>(lds_sp + slot(0), wn0, lane, b[2]);
                        copy_to(3, sa[0], 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i == 0 ? FM - 1 : i - 1][j] += t[nxt][j];
                    a[nxt][0] = sp_frag1<T>(lds_sp + na[0], wm0 + next_row, lane);
                    sp_products<false>(b[1], a[cur][1], t[cur]); // a1 b1
                    if constexpr (last && COPIES > 1) copy_to(3, sa[0], 1);
                    __builtin_amdgcn_sched_barrier(0);
                    a[nxt][1] = sp_frag1<T>(lds_sp + na[1], wm0 + next_row, lane);
                    sp_products<false>(b[1], a[cur][0], t[cur]); // a0 b1
                    if constexpr (last) {
                        sp_frag<T, 0, FN>(lds_sp + slot(1), wn0, lane, b[1]);
                        copy_to(4, sa[1], 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    a[nxt][2] = sp_frag1<T>(lds_sp + na[2], wm0 + next_row, lane);
                    sp_products<false>(b[0], a[cur][2], t[cur]); // a2 b0
                    if constexpr (last && COPIES > 1) copy_to(4, sa[1], 1);
                    __builtin_amdgcn_sched_barrier(0);
                    sp_products<false>(b[0], a[cur][1], t[cur]); // a1 b0
                    if constexpr (last) copy_to(5, sa[2], 0);
                    __builtin_amdgcn_sched_barrier(0);
                    sp_products<false>(b[0], a[cur][0], t[cur]); // a0 b0
                    if constexpr (last) {
                        sp_frag<T, 0, FN>(lds_sp + slot(2), wn0, lane, b[0]);
                        if constexpr (COPIES > 1) copy_to(5, sa[2], 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (i == 0) {
                        sp_barrier(); // all waves have the slab's planes of op(B)
                        __builtin_amdgcn_sched_barrier(0);
                    } else if constexpr (!last) {
                        constexpr int PER = (3 * COPIES + FM - 3) / (FM - 2); // three blocks over the rows between
#pragma unroll
                        for (int c = PER * (i - 1); c < PER * i; ++c)
                            if (c < 3 * COPIES) copy_to(c / COPIES, slot(c / COPIES), c % COPIES);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
                advance(s);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[FM - 1][j] += t[1][j];
        } else {
            bf16x8 a[FM], b0[FN], b1[FN];
            sp_frag<T, 0, FM>(lds_sp, wm0, lane, a);
            sp_frag<T, 0, FN>(lds_sp + BLK, wn0, lane, b0);
            for (int s = 0; s < n; ++s) {
                const int s2 = slot(2);
                sp_rows<0, FM>(b0, a, acc, [&](auto i) { // a1 b0
                    if constexpr (i == 0) sp_frag<T, 0, FN>(lds_sp + slot(3), wn0, lane, b1);
                    sp_frag<T, i, i + 1>(lds_sp + s2, wm0, lane, a);
                });
                sp_mfma<0, FM / 2>(b1, a, acc); // a0 b1
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(sp_wait(COPIES * (RING - 8)));
                sp_barrier();
                __builtin_amdgcn_sched_barrier(0);
                sp_mfma<FM / 2, FM>(b1, a, acc);
                __builtin_amdgcn_sched_barrier(0);
                sp_frag<T, 0, FN>(lds_sp + slot(5), wn0, lane, b1);
                __builtin_amdgcn_sched_barrier(0);
                const int s4 = slot(4);
                sp_rows<0, FM>(b0, a, acc, [&](auto i) { // a0 b0
                    sp_frag<T, i, i + 1>(lds_sp + s4, wm0, lane, a);
                    constexpr int PER = (4 * COPIES + FM - 1) / FM; // four blocks
#pragma unroll
                    for (int c = PER * i; c < PER * (i + 1); ++c)
                        if (c < 4 * COPIES) copy_to(c / COPIES, slot(c / COPIES), c % COPIES);
                });
                head = slot(4);
                advance(s);
#pragma unroll
                for (int j = 0; j < FN; ++j) b0[j] = b1[j];
            }
        }
        sp_drain();
    }
    if (split) {
        float* part = p.partial + ((size_t)(z * rest + tile - p.whole) * (T * T)) + (wave * Cfg::FM * Cfg::FN * 64 + lane) * 4;
#pragma unroll
        for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
            for (int j = 0; j < Cfg::FN; ++j)
                *reinterpret_cast<f32x4*>(part + (i * Cfg::FN + j) * 256) = acc[i][j];
        return;
    }
    const bool whole = m0 + T <= ROW * g.M && n0 + T <= g.N && g.write_tri == 0 && g.mask == 0;
    const int row0 = m0 + wm0 + (lane & 15), col0 = n0 + wn0;
    constexpr int G = 4;
#pragma unroll
    for (int i = 0; i < Cfg::FM; i += G) {
        const auto& part = reinterpret_cast<const f32x4(&)[G][Cfg::FN]>(acc[i]);
        if (whole)
            sp_store<CPLX, false>(g, part, row0 + 16 * i, col0, lane);
        else
            sp_store<CPLX, true>(g, part, row0 + 16 * i, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Sums the parts of a split product in their order and stores the result: a wave per
// 16 x 16 block.
template <int T, int WVM, int WVN, int PLANES, bool CPLX>
__global__ void __launch_bounds__(256) split_reduce_kernel(SplitArgs p)
{
    using Cfg = SplitCfg<T, WVM, WVN>;
    constexpr int ROW = CPLX ? 2 : 1, BLOCKS = Cfg::NW * Cfg::FM * Cfg::FN;
    if (PLANES == 3 && *p.guard == p.epoch) return;
    const icl_gemm_args& g = p.g;
    const int lane = threadIdx.x & 63;
    const int id = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rest = gridDim.x * 4 / BLOCKS, tile = id / BLOCKS, blk = id % BLOCKS;
    int tm, tn;
    if (!tile_level3<T / ROW, T>(p.whole + tile, g.write_tri, g.kband, (ROW * g.M + T - 1) / T, (g.N + T - 1) / T, tm, tn)) return;
    const float* part = p.partial + (size_t)tile * (T * T) + (blk * 64 + lane) * 4;
    const size_t step = (size_t)rest * (T * T);
    f32x4 sum[1][1] = {{f32x4{}}};
    int z = 0;
    for (; z + 8 <= p.splits; z += 8) {
        f32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const f32x4*>(part + (z + i) * step);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[0][0] += v[i];
    }
    for (; z < p.splits; ++z) sum[0][0] += *reinterpret_cast<const f32x4*>(part + z * step);
    const int w = blk / (Cfg::FM * Cfg::FN), i = blk / Cfg::FN % Cfg::FM, j = blk % Cfg::FN;
    const int row = tm * T + (w % WVM) * Cfg::WM + 16 * i + (lane & 15);
    sp_store<CPLX, true>(g, sum, row, tn * T + (w / WVM) * Cfg::WN + 16 * j, lane);
}

namespace {

inline int sp_round_up(int x, int m) { return (x + m - 1) / m * m; }

// A launch's tiles: `whole` of them as they are, in rounds that fill the CUs, and `rest`
// more in `splits` parts of their depth; and its time. Microseconds per slab of one
// workgroup, measured with every CU full at the clock that a long product settles at:
// 3.9 for a 256 x 256 tile, 2.15 for two 128 x 128 tiles on a CU and 1.25 for one (two
// planes 2.05, 1.15, 0.65); 14 or 5 more per round of workgroups, which store C together
// (4000 x 4000 x 512: 100 us with the large tile, 90 with the small); 4 and the
// partial sums at 2.7 TB/s (written, and read again) for a split. SSYRK 640 (k 20011):
// 15 tiles in 34 parts, 745 -> 122 us; 1024 x 1024 x 4096 139 -> 62 us.
// With a triangular operand (kband) the tiles start longest window first, so they fill
// the CUs evenly and the longest is the bound: STRMM 3000 x 2048, all tiles in two
// parts, 140 -> 95 us.
struct SplitPlan {
    int whole, rest, splits;
    double us;
};

SplitPlan sp_plan(const icl_gemm_args* g, long tiles, int slabs, int T, int planes)
{
    constexpr long kCUs = 256;
    constexpr size_t kMaxPartial = size_t(256) << 20;
    const long at_once = T == 256 ? kCUs : 2 * kCUs;
    const double full = T == 256 ? (planes == 3 ? 3.9 : 2.05) : (planes == 3 ? 2.15 : 1.15);
    const double alone = T == 256 ? full : (planes == 3 ? 1.25 : 0.65);
    const double per_round = T == 256 ? 14.0 : 5.0;
    auto round_us = [&](long units, int depth) {
        if (units <= 0) return 0.0;
        return (units <= kCUs ? alone : full) * depth * (0.8 + 0.2 * std::min(units, kCUs) / kCUs) + per_round;
    };
    if (g->kband != ICL_KBAND_NONE) {
        const double mean = 0.5 * (slabs + T / kSlabK);
        SplitPlan best{(int)tiles, 0, 1, 0.0};
        for (int z = 1; z <= (g->whole_depth ? 1 : 8); ++z) {
            const size_t bytes = z > 1 ? (size_t)tiles * z * T * T * sizeof(float) : 0;
            if (bytes > kMaxPartial) break;
            const double us = std::max(alone * slabs / z, full * tiles * mean / at_once) + per_round +
                              (z > 1 ? 4.0 + bytes / 2.7e6 : 0.0);
            if (z == 1)
                best.us = us;
            else if (us < 0.97 * best.us)
                best = SplitPlan{0, (int)tiles, z, us};
        }
        return best;
    }
    const long rest = tiles % at_once;
    const double whole_us = tiles / at_once * round_us(at_once, slabs);
    SplitPlan best{(int)tiles, 0, 1, whole_us + round_us(rest, slabs)};
    if (g->whole_depth || rest == 0) return best;
    for (int z = 2; z <= 64; ++z) {
        const long units = rest * z;
        const size_t bytes = (size_t)units * T * T * sizeof(float);
        const int depth = (slabs + z - 1) / z;
        if (depth < 4 || bytes > kMaxPartial || units > at_once) break;
        const double us = whole_us + round_us(units, depth) + 4.0 + bytes / 2.7e6;
        if (us < 0.97 * best.us) best = SplitPlan{(int)(tiles - rest), (int)rest, z, us};
    }
    return best;
}

// A square triangle update runs the tiles off the diagonal 256 x 256 blocks, then those
// of the blocks at a quarter of the size, on the same packed operands: half of a
// diagonal block's large tile would be thrown away, and SSYRK 8192's 528 large tiles
// end in a round of 16 on 256 CUs.
template <int T>
bool sp_in_bands(const icl_gemm_args* g)
{
    return T == 256 && (g->write_tri == ICL_TRI_LOWER || g->write_tri == ICL_TRI_UPPER) && g->M == g->N &&
           g->M >= 2 * ICL_TRI_BAND_BLOCK && g->kband == ICL_KBAND_NONE;
}

struct SplitLayout {
    int Mpad, Npad, slabs;
    size_t a_bytes, b_bytes;
    SplitPlan plan, band; // the launch (in bands: the one off the blocks) and the one on the blocks
    size_t partial_bytes;
};

template <int T, int PLANES, bool CPLX>
SplitLayout sp_layout(const icl_gemm_args* g)
{
    constexpr int R = CPLX ? 2 : 1;
    SplitLayout l;
    l.Mpad = sp_round_up(R * g->M, T);
    l.Npad = sp_round_up(g->N, T);
    l.slabs = sp_round_up(R * g->K, kSlabK) / kSlabK;
    l.a_bytes = (size_t)l.slabs * PLANES * kGroups * l.Mpad * 16;
    l.b_bytes = (size_t)l.slabs * PLANES * kGroups * l.Npad * 16;
    icl_gemm_args part = *g;
    if (sp_in_bands<T>(g)) part.write_tri |= ICL_TRI_OFF_BAND;
    const long tiles = gemm_tiles(&part, T / R, T);
    l.plan = sp_plan(&part, tiles, l.slabs, T, PLANES);
    l.band = SplitPlan{0, 0, 1, 0.0};
    size_t partial = (size_t)l.plan.rest * l.plan.splits * T * T;
    if (sp_in_bands<T>(g)) {
        part.write_tri = g->write_tri | ICL_TRI_BAND;
        const long on_blocks = gemm_tiles(&part, 128 / R, 128);
        l.band = sp_plan(&part, on_blocks, l.slabs, 128, PLANES);
        partial = std::max(partial, (size_t)l.band.rest * l.band.splits * 128 * 128);
    }
    l.partial_bytes = partial * sizeof(float);
    return l;
}

template <int T, int PLANES, bool CPLX>
size_t sp_workspace(const icl_gemm_args* g)
{
    const SplitLayout l = sp_layout<T, PLANES, CPLX>(g);
    return l.a_bytes + l.b_bytes + l.partial_bytes;
}

// Seconds: the prepass at 4.8 TB/s (4 read and 2 written bytes per plane and element,
// op(A) of a complex product written as two rows of two), the products, the launches.
template <int T, int PLANES, bool CPLX>
double sp_estimate(const icl_gemm_args* g)
{
    const SplitLayout l = sp_layout<T, PLANES, CPLX>(g);
    const double read = (CPLX ? 8.0 : 4.0) * (double(g->M) + g->N) * g->K;
    double us = (read + l.a_bytes + l.b_bytes) / 4.8e6 + l.plan.us + l.band.us + (PLANES == 3 ? 10.0 : 3.0);
    return us * 1e-6;
}

// Packs arows packed rows of `a` and brows of `b` (multiples of 64). A grid's second
// dimension ends at 65536 blocks, a depth of 2^22: deeper ones (FP32 products of few rows
// reach 2^22.4) go on in the third.
template <int PLANES, bool CPLX>
hipError_t sp_pack(const SplitSrc& a, int arows, const SplitSrc& b, int brows, const SplitArgs& p, hipStream_t s)
{
    if (p.slabs == 0) return hipSuccess; // C is only scaled
    const unsigned deep = (unsigned)((p.slabs + 1) / 2), layer = std::min(deep, 32768u);
    const dim3 grid((unsigned)((arows + brows) / 64), layer, (deep + layer - 1) / layer);
    hipLaunchKernelGGL((split_pack_kernel<PLANES, CPLX>), grid, dim3(256), 0, s, a, b, arows / 64, p.slabs,
                       const_cast<unsigned long long*>(p.guard), p.epoch);
    return hipGetLastError();
}

// The product of the rows and columns of g (a part of the packed problem p).
template <int T, int PLANES, bool CPLX>
hipError_t sp_product(SplitArgs p, const icl_gemm_args& g, const SplitPlan& plan, hipStream_t s)
{
    constexpr int WVM = 2, WVN = 4;
    using C = SplitCfg<T, WVM, WVN>;
    p.g = g;
    p.whole = plan.whole;
    p.splits = plan.splits;
    const long blocks = plan.whole + (long)plan.rest * plan.splits;
    hipError_t e = launch_blocks<C::NT, C::LDS_BYTES>(split_gemm_kernel<T, WVM, WVN, PLANES, CPLX>, blocks, s, p);
    if (e != hipSuccess || plan.rest == 0) return e;
    return launch_blocks<256, 0>(split_reduce_kernel<T, WVM, WVN, PLANES, CPLX>,
                                 (long)plan.rest * (C::NW * C::FM * C::FN / 4), s, p);
}

// The rows [r0, r0 + rows) of a real source and its packed layout (r0 a multiple of 64).
template <int PLANES>
SplitSrc sp_rows(SplitSrc src, int r0, int rows)
{
    src.X += src.kcontig ? (long)r0 * src.ld : (long)r0;
    src.R = rows;
    src.P += (size_t)r0 * (PLANES * kGroups * 8);
    return src;
}

template <int T, int PLANES, bool CPLX>
hipError_t sp_launch(const icl_gemm_args* g, int opa, int opb, int edge, void* ws, hipStream_t s)
{
    (void)edge;
    if (!ws || (PLANES == 3 && !g->guard)) return hipErrorInvalidValue;
    const SplitLayout l = sp_layout<T, PLANES, CPLX>(g);
    SplitArgs p{};
    p.Mpad = l.Mpad;
    p.Npad = l.Npad;
    p.slabs = l.slabs;
    __bf16* Ap = static_cast<__bf16*>(ws);
    __bf16* Bp = reinterpret_cast<__bf16*>(static_cast<char*>(ws) + l.a_bytes);
    p.Ap = Ap;
    p.Bp = Bp;
    p.partial = reinterpret_cast<float*>(static_cast<char*>(ws) + l.a_bytes + l.b_bytes);
    p.guard = g->guard;
    p.epoch = g->guard_epoch;
    const SplitSrc a{g->A, g->lda, g->M, g->K, l.Mpad, opa != 0, opa == 2, Ap};
    const SplitSrc b{g->B, g->ldb, g->N, g->K, l.Npad, opb == 0, opb == 2, Bp};
    hipError_t e;
    if constexpr (PLANES == 2 && T == 256 && !CPLX) {
        // Large plain products with a side stream: the operands in halves. The
        // handle's stream packs A0 and B0 and multiplies them while the side stream
        // packs A1 and B1 (after the first pack, whose bandwidth it would share);
        // then A0 B1 and A1 B follow. Each launch computes its elements exactly as a
        // single launch would (same slabs, same order).
        const icl_side_lane* side = icl_gemm_side_lane();
        const int m0 = sp_round_up(g->M / 2, T), n0 = sp_round_up(g->N / 2, T);
        if (side && !uses_level3(g) && g->M % T == 0 && g->N % T == 0 && m0 < g->M && n0 < g->N) {
            if ((e = sp_pack<2, false>(sp_rows<2>(a, 0, m0), m0, sp_rows<2>(b, 0, n0), n0, p, s)) != hipSuccess) return e;
            if ((e = hipEventRecord(side->start, s)) != hipSuccess) return e;
            if ((e = hipStreamWaitEvent(side->stream, side->start, 0)) != hipSuccess) return e;
            e = sp_pack<2, false>(sp_rows<2>(a, m0, g->M - m0), g->M - m0, sp_rows<2>(b, n0, g->N - n0), g->N - n0, p,
                                  side->stream);
            if (e != hipSuccess || (e = hipEventRecord(side->done, side->stream)) != hipSuccess) return e;
            if ((e = icl_timer_mark(s)) != hipSuccess) return e;
            // (row offset, rows, column offset, columns) of C per launch
            const int part[3][4] = {{0, m0, 0, n0}, {0, m0, n0, g->N - n0}, {m0, g->M - m0, 0, g->N}};
            for (int q = 0; q < 3; ++q) {
                if (q == 1 && (e = hipStreamWaitEvent(s, side->done, 0)) != hipSuccess) return e;
                icl_gemm_args gq = *g;
                gq.M = part[q][1];
                gq.N = part[q][3];
                gq.C = g->C + (long)part[q][2] * g->ldc + part[q][0];
                SplitArgs pq = p;
                pq.Ap = Ap + (size_t)part[q][0] * (PLANES * kGroups * 8);
                pq.Bp = Bp + (size_t)part[q][2] * (PLANES * kGroups * 8);
                if ((e = sp_product<T, PLANES, CPLX>(pq, gq, SplitPlan{gq.M / T * (gq.N / T), 0, 1, 0.0}, s)) != hipSuccess) return e;
            }
            return icl_timer_mark(s);
        }
    }
    if ((e = sp_pack<PLANES, CPLX>(a, l.Mpad, b, l.Npad, p, s)) != hipSuccess) return e;
    if (sp_in_bands<T>(g)) {
        icl_gemm_args part = *g;
        part.write_tri = g->write_tri | ICL_TRI_OFF_BAND;
        if ((e = icl_timer_mark(s)) != hipSuccess) return e;
        if ((e = sp_product<T, PLANES, CPLX>(p, part, l.plan, s)) != hipSuccess) return e;
        if ((e = icl_timer_mark(s)) != hipSuccess) return e;
        part.write_tri = g->write_tri | ICL_TRI_BAND;
        if ((e = icl_timer_mark(s)) != hipSuccess) return e;
        if ((e = sp_product<128, PLANES, CPLX>(p, part, l.band, s)) != hipSuccess) return e;
        return icl_timer_mark(s);
    }
    if ((e = icl_timer_mark(s)) != hipSuccess) return e;
    if ((e = sp_product<T, PLANES, CPLX>(p, *g, l.plan, s)) != hipSuccess) return e;
    return icl_timer_mark(s);
}

} // namespace
} // namespace icl

// TF: measured useful TFLOP/s of the main kernel (real at 8192^3, complex at 4096^3);
// OCC: workgroups per CU.
#define ICL_GEMM_SPLIT(name, kind, math, PLANES, CPLX, T, TF, OCC)                                                     \
    {name,                                                                                                             \
     kind,                                                                                                             \
     math,                                                                                                             \
     T / (CPLX ? 2 : 1),                                                                                               \
     T,                                                                                                                \
     icl::kSlabK / (CPLX ? 2 : 1),                                                                                     \
     T * 2,                                                                                                            \
     icl::sp_launch<T, PLANES, CPLX>,                                                                                  \
     icl::sp_workspace<T, PLANES, CPLX>,                                                                               \
     TF,                                                                                                               \
     OCC,                                                                                                              \
     1,                                                                                                                \
     icl::sp_estimate<T, PLANES, CPLX>}

static const icl_gemm_variant kTable[] = {
    ICL_GEMM_SPLIT("sgemm_f32_split3_256x256", ICL_KIND_SGEMM, ICL_MATH_FP32, 3, false, 256, 275.0f, 1),
    ICL_GEMM_SPLIT("sgemm_f32_split3_128x128", ICL_KIND_SGEMM, ICL_MATH_FP32, 3, false, 128, 242.0f, 2),
    ICL_GEMM_SPLIT("cgemm_f32_split3_128x256", ICL_KIND_CGEMM, ICL_MATH_FP32, 3, true, 256, 272.0f, 1),
    ICL_GEMM_SPLIT("cgemm_f32_split3_64x128", ICL_KIND_CGEMM, ICL_MATH_FP32, 3, true, 128, 240.0f, 2),
    ICL_GEMM_SPLIT("sgemm_bf16x3d_mfma_256x256", ICL_KIND_SGEMM, ICL_MATH_BF16X3, 2, false, 256, 463.0f, 1),
    ICL_GEMM_SPLIT("sgemm_bf16x3d_mfma_128x128", ICL_KIND_SGEMM, ICL_MATH_BF16X3, 2, false, 128, 366.0f, 2),
    ICL_GEMM_SPLIT("cgemm_bf16x3d_mfma_128x256", ICL_KIND_CGEMM, ICL_MATH_BF16X3, 2, true, 256, 495.0f, 1),
    ICL_GEMM_SPLIT("cgemm_bf16x3d_mfma_64x128", ICL_KIND_CGEMM, ICL_MATH_BF16X3, 2, true, 128, 387.0f, 2),
};
ICL_REGISTER_VARIANTS(kTable)
