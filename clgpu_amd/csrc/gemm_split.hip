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
// BF16 MFMAs whose products are exact and which accumulate in FP32; the three terms left
// out are below 2^-23 |a b| (2^-26 root mean square), less than one FP32 rounding. The
// error against float64 is 0.64 (k = 64) to 0.9 (k = 8192) of FP32 MFMA's on uniform
// data, since a sum is rounded less often.
//
// What bounds it: at 8192^3 the card's power. The three-plane kernel keeps the MFMA units
// 78% busy at 1.9 GHz (1650 TFLOP/s of BF16; registers alone reach 2050 on random data),
// so the choices here are those that cost least energy per product:
// v_mfma_f32_16x16x32 (2048 TFLOP/s from registers against 1812 for 32x32x16), planes
// kept in registers over as many groups of products as possible (36 LDS reads per 192
// products; with the planes paired in 16-deep slabs, 56, it took 4.55 ms) and operands
// copied to LDS without passing through registers. Four waves of 128 x 128 (a third fewer
// LDS reads) do not fit the registers. SGEMM 8192^3: FP32 MFMA 7.75 ms, three planes
// 4.29 ms, of which 0.27 the prepass (4.9 TB/s); CGEMM 4096^3 3.88 -> 2.18 ms. Two planes
// 8192^3: 2.35 ms, against 2.52 with 32x32x16 MFMA and fragments read just before use.
// The 128 x 128 tile, two workgroups per CU, serves outputs with too few large tiles
// (three planes, 2048^3: 98 us against 212).
#include "gemm_variants.hpp"

#include <type_traits>

namespace icl {

constexpr int kSlabK = 32; // k per slab (one MFMA deep)
constexpr int kGroups = 4; // 16-byte chunks (groups of 8 k) per row, slab and plane

typedef __attribute__((address_space(3))) void sp_lds_void;

// ---------------------------------------------------------------------------
// Prepass. Packed layout P[slab][plane][k / 8][row][8]: any 64 rows of one (slab,
// plane, k / 8) are 1 KB of contiguous memory, one LDS DMA instruction, and the LDS
// image keeps the rows contiguous (16 bytes apart: fragment reads are free of bank
// conflicts).
//
// Complex operands become real ones: op(A) (m x k) the 2m x 2k matrix with the
// 2 x 2 blocks [re -im; im re], op(B) the 2k x n matrix of its stacked parts, so
// that the real product's rows 2r and 2r + 1 are the parts of row r of the
// complex one: C's interleaved storage. Conjugation negates im.
//
// For three planes every element read is checked: outside 2^-110 <= |x| < 2^50 (or zero) the split
// is not exact or a partial product could overflow where the FP32 sum does not,
// and infinities and NaN would spread differently. Any such element stores the
// call's epoch into *guard, and the FP32 MFMA kernel computes the product instead.
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
    const SplitSrc o = is_a ? a : b;
    const int r0 = (is_a ? (int)blockIdx.x : (int)blockIdx.x - ablocks) * 64; // packed row
    const int k0 = blockIdx.y * 64;                                           // packed k
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
    if (PLANES == 3 && bad) *guard = epoch;
    __syncthreads();
    // wave w writes k = 16 w .. 16 w + 15 of slab pair y, lane = row: 1 KB per store
    const int w = t >> 6, r = t & 63, ks = 2 * (int)blockIdx.y + (w >> 1);
    if (ks >= slabs) return;
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
    __bf16* dst = o.P + (((size_t)ks * PLANES * kGroups + 2 * (w & 1)) * o.Rpad + r0 + r) * 8;
#pragma unroll
    for (int p = 0; p < PLANES; ++p)
#pragma unroll
        for (int c = 0; c < 2; ++c)
            *reinterpret_cast<bf16x8*>(dst + (size_t)(kGroups * p + c) * o.Rpad * 8) = out[p][c];
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
};

// T x T tiles of packed rows, WVM x WVN waves. LDS is a ring of ten chunk blocks,
// each the T rows of one plane of one operand's slab.
template <int T_, int WVM_, int WVN_>
struct SplitCfg {
    static constexpr int T = T_, WVM = WVM_, WVN = WVN_;
    static constexpr int NW = WVM * WVN, NT = NW * 64;
    static constexpr int WM = T / WVM, WN = T / WVN, FM = WM / 16, FN = WN / 16;
    static constexpr int RING = 10, BLOCK = T * kSlabK * 2; // bytes
    static constexpr size_t LDS_BYTES = (size_t)RING * BLOCK;
    static constexpr int RB = T / 64; // 64-row groups
    static_assert(BLOCK == 2 * NW * 1024 && NW % RB == 0, "two copies per wave and block");
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

// c += a b in place: v_mfma_f32_16x16x32_bf16 with the sum's registers tied. Written
// out because the compiler gives each of the builtin's results registers of its own
// and then has too few left for operands read ahead (256 per wave: 128 hold sums).
// It does not see the instruction's latency: a sum is used again only by a product
// at least FM * FN instructions later, or after sp_drain.
// Lane l supplies a = A[l % 16][8 (l / 16) .. + 7] and b = B[8 (l / 16) .. + 7][l % 16];
// register r of c is D[4 (l / 16) + r][l % 16].
__device__ __forceinline__ void sp_mfma1(bf16x8 a, bf16x8 b, f32x4& c)
{
    asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}

// Lets the last products finish before their sums are read, and the last copies.
__device__ __forceinline__ void sp_drain()
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
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

// Stores a column of FN 16 x 16 blocks: register r of block j holds column
// ncol0 + 16 j + 4 (lane / 16) + r, the lane row `row` (complex: the part lane & 1
// of complex row row / 2). CHECK: bounds, triangle and mask are tested per element.
template <bool CPLX, bool CHECK, int FN>
__device__ __forceinline__ void sp_store(const GemmArgs& g, const f32x4 (&acc)[FN], int row, int ncol0, int lane)
{
    const int nl = ncol0 + 4 * (lane >> 4);
    const int m = CPLX ? row >> 1 : row;
    float* const c0 = g.C + (CPLX ? 2L : 1L) * (long)nl * g.ldc + row;
    const long cstep = CPLX ? 2 * g.ldc : g.ldc;
    const bool odd = CPLX && (lane & 1);
    const bool beta_zero = g.beta_re == 0.0f && (!CPLX || g.beta_im == 0.0f);
    const TriMask tri(g.mask);
    auto on = [&](int n) { return !CHECK || (m < g.M && n < g.N && tri_writes(g.write_tri, m, n)); };
    float old[FN][4];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            old[j][r] = 0.0f;
            if (!beta_zero && on(nl + 16 * j + r)) old[j][r] = c0[(16 * j + r) * cstep];
        }
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = nl + 16 * j + r;
            float v;
            if constexpr (CPLX) {
                // even lanes: alpha_re re - alpha_im im; odd lanes: alpha_re im + alpha_im re
                const float own = odd && (g.cflags & ICL_CFLAG_CONJ_ACC) ? -acc[j][r] : acc[j][r];
                const float x = sp_neighbour(own), oth = odd ? x : -x;
                v = fmaf(g.alpha_re, own, g.alpha_im * oth);
                if (!beta_zero) {
                    const float y = sp_neighbour(old[j][r]), oldoth = odd ? y : -y;
                    v += fmaf(g.beta_re, old[j][r], g.beta_im * oldoth);
                }
                if (odd && (g.cflags & ICL_CFLAG_REAL_DIAG) && m == n) v = 0.0f;
            } else {
                v = beta_zero ? g.alpha_re * acc[j][r] : fmaf(g.beta_re, old[j][r], g.alpha_re * acc[j][r]);
            }
            if (CHECK && !tri.keep(m, n)) v = 0.0f;
            if (on(n)) c0[(16 * j + r) * cstep] = v;
        }
}

// T in rows of the packed operands: a complex tile has T / 2 rows.
//
// A slab's six groups of products are summed smallest first (a2 b0, a1 b1, a1 b0,
// a0 b2, a0 b1, a0 b0), so that one large product among small ones is rounded to the
// sum once, by its last group. The copies run through the LDS ring as one sequence of
// blocks, six per slab in the order their planes are used: a2 b0 b1 a1 b2 a0, block q
// in slot q % 10. A slab's first four blocks are in registers in its second group,
// the last two after its fourth, and at each of these points a barrier frees their
// slots for the blocks ten places on, which then have a whole slab's products to
// arrive. Of two planes: a1 b0, a0 b1, a0 b0, the blocks a1 b0 a0 b1, all in
// registers in the second group.
template <int T, int WVM, int WVN, int PLANES, bool CPLX>
__global__ void __launch_bounds__(WVM* WVN * 64, 2) split_gemm_kernel(SplitArgs p)
{
    using Cfg = SplitCfg<T, WVM, WVN>;
    constexpr int ROW = CPLX ? 2 : 1; // packed rows (and k) per element
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_sp[];
    if (PLANES == 3 && *p.guard == p.epoch) return;
    const icl_gemm_args& g = p.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave % WVM) * Cfg::WM;
    const int wn0 = (wave / WVM) * Cfg::WN;
    int tm, tn, ks0 = 0, ks1 = p.slabs; // slabs [ks0, ks1) of the tile's k window
    const int tiles_m = (ROW * g.M + T - 1) / T, tiles_n = (g.N + T - 1) / T;
    if (g.write_tri | g.kband) {
        if (!tile_coords_level3<T / ROW, T>(g.write_tri, g.kband, tiles_m, tiles_n, tm, tn)) return;
        int kb = 0, ke = 0;
        if (!tile_window<T / ROW, T>(g, tm * (T / ROW), tn * T, kb, ke)) return;
        ks0 = kb * ROW / kSlabK;
        ks1 = ke > kb ? (ke * ROW + kSlabK - 1) / kSlabK : ks0;
    } else {
        tile_coords<8>(tiles_m, tiles_n, tm, tn);
    }
    const int m0 = tm * T, n0 = tn * T; // packed rows

    // This wave's copies of a block: the k groups wave / RB and wave / RB + 2 of 64 rows.
    const size_t a_row = (size_t)p.Mpad * 16, b_row = (size_t)p.Npad * 16; // bytes of a chunk of all rows
    const char* a_src = reinterpret_cast<const char*>(p.Ap) + (size_t)ks0 * PLANES * kGroups * a_row +
                        (wave / Cfg::RB) * a_row + (size_t)(m0 + 64 * (wave % Cfg::RB)) * 16;
    const char* b_src = reinterpret_cast<const char*>(p.Bp) + (size_t)ks0 * PLANES * kGroups * b_row +
                        (wave / Cfg::RB) * b_row + (size_t)(n0 + 64 * (wave % Cfg::RB)) * 16;
    const int loff = lane * 16;
    const int n = ks1 - ks0;
    // Half `i` of the copy of plane `plane` of slab ks0 + ks of op(A) (else op(B)) to
    // the ring slot at `slot`. Past the last slab it copies that one again, to a slot
    // nothing reads any more: the number of copies in flight stays the same.
    auto copy = [&](bool of_a, int plane, int ks, int slot, int i) {
        const size_t row = of_a ? a_row : b_row;
        const char* src = (of_a ? a_src : b_src) + ((size_t)min(ks, n - 1) * PLANES + plane) * kGroups * row;
        // A buffer load (its address stays scalar): a global load counts as a FLAT
        // access, after which the compiler waits for all LDS reads at once.
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(src), 0, (unsigned)(2 * row + 1024), 0x20000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc, (sp_lds_void*)(lds_sp + slot + (wave + Cfg::NW * i) * 1024), 16, loff, (int)(2 * i * row), 0, 0);
    };
    auto issue = [&](bool of_a, int plane, int ks, int slot) {
        copy(of_a, plane, ks, slot, 0);
        copy(of_a, plane, ks, slot, 1);
    };

    f32x4 acc[Cfg::FM][Cfg::FN];
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::FN; ++j) acc[i][j] = f32x4{};

    if (n > 0) {
        constexpr int FM = Cfg::FM, FN = Cfg::FN, BLK = Cfg::BLOCK;
        bf16x8 a[FM], b0[FN], b1[FN];
        int head = 0; // ring position of the slab's first block
        auto slot = [&](int c) {
            const int q = head + c;
            return (q < 10 ? q : q < 20 ? q - 10 : q - 20) * BLK;
        };
        // After row i: that row's operand replaced by the block S's.
        auto next_a = [&](int S) {
            return [&, S](auto i) { sp_frag<T, i, i + 1>(lds_sp + S, wm0, lane, a); };
        };
        if constexpr (PLANES == 3) {
            issue(true, 2, 0, 0);
            issue(false, 0, 0, BLK);
            issue(false, 1, 0, 2 * BLK);
            issue(true, 1, 0, 3 * BLK);
            issue(false, 2, 0, 4 * BLK);
            issue(true, 0, 0, 5 * BLK);
            issue(true, 2, 1, 6 * BLK);
            issue(false, 0, 1, 7 * BLK);
            issue(false, 1, 1, 8 * BLK);
            issue(true, 1, 1, 9 * BLK);
            __builtin_amdgcn_s_waitcnt(sp_wait(12));
            sp_barrier();
            bf16x8 b2[FN];
            sp_frag<T, 0, FM>(lds_sp, wm0, lane, a);
            sp_frag<T, 0, FN>(lds_sp + BLK, wn0, lane, b0);
            // Each operand is read under the products before the ones that need it, and
            // the copies into the freed slots are spread over the rows (issued together
            // they hold up every wave's products).
            for (int s = 0; s < n; ++s) {
                const int s3 = slot(3);
                sp_rows<0, FM>(b0, a, acc, [&](auto i) { // a2 b0
                    if constexpr (i == 0) sp_frag<T, 0, FN>(lds_sp + slot(2), wn0, lane, b1);
                    sp_frag<T, i, i + 1>(lds_sp + s3, wm0, lane, a);
                });
                sp_mfma<0, FM / 2>(b1, a, acc); // a1 b1
                __builtin_amdgcn_sched_barrier(0);
                // The slab's b2 and a0 have arrived once at most the next slab's first
                // four blocks are outstanding.
                __builtin_amdgcn_s_waitcnt(sp_wait(8));
                sp_barrier();
                __builtin_amdgcn_sched_barrier(0);
                sp_frag<T, 0, FN>(lds_sp + slot(4), wn0, lane, b2);
                __builtin_amdgcn_sched_barrier(0);
                sp_mfma<FM / 2, FM>(b1, a, acc);
                __builtin_amdgcn_sched_barrier(0);
                const int s5 = slot(5);
                sp_rows<0, FM>(b0, a, acc, [&](auto i) { // a1 b0
                    sp_frag<T, i, i + 1>(lds_sp + s5, wm0, lane, a);
                    constexpr int PER = 8 / FM; // eight copies
#pragma unroll
                    for (int c = PER * i; c < PER * (i + 1); ++c) {
                        const int q = c / 2;
                        copy(q == 1 || q == 2, q == 0 || q == 2 ? 2 : 0, q < 2 ? s + 1 : s + 2, slot(10 + q), c & 1);
                    }
                });
                sp_mfma<0, FM>(b2, a, acc); // a0 b2
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(sp_wait(8));
                sp_barrier();
                __builtin_amdgcn_sched_barrier(0);
                sp_rows<0, FM>(b1, a, acc, [&](auto i) { // a0 b1
                    if constexpr (i == 0) sp_frag<T, 0, FN>(lds_sp + slot(7), wn0, lane, b2);
                    constexpr int PER = FM >= 8 ? 1 : 2; // four copies, after the first row
#pragma unroll
                    for (int c = PER * (i - 1); c < PER * i; ++c)
                        if (c >= 0 && c < 4) copy(c >= 2, 1, s + 2, slot(14 + c / 2), c & 1);
                });
                head = head + 6 < 10 ? head + 6 : head - 4;
                sp_rows<0, FM>(b0, a, acc, next_a(slot(0))); // a0 b0
#pragma unroll
                for (int j = 0; j < FN; ++j) b0[j] = b2[j];
            }
        } else {
            issue(true, 1, 0, 0);
            issue(false, 0, 0, BLK);
            issue(true, 0, 0, 2 * BLK);
            issue(false, 1, 0, 3 * BLK);
            issue(true, 1, 1, 4 * BLK);
            issue(false, 0, 1, 5 * BLK);
            issue(true, 0, 1, 6 * BLK);
            issue(false, 1, 1, 7 * BLK);
            issue(true, 1, 2, 8 * BLK);
            issue(false, 0, 2, 9 * BLK);
            __builtin_amdgcn_s_waitcnt(sp_wait(12));
            sp_barrier();
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
                __builtin_amdgcn_s_waitcnt(sp_wait(4));
                sp_barrier();
                __builtin_amdgcn_sched_barrier(0);
                sp_mfma<FM / 2, FM>(b1, a, acc);
                __builtin_amdgcn_sched_barrier(0);
                sp_frag<T, 0, FN>(lds_sp + slot(5), wn0, lane, b1);
                __builtin_amdgcn_sched_barrier(0);
                const int s4 = slot(4);
                sp_rows<0, FM>(b0, a, acc, [&](auto i) { // a0 b0
                    sp_frag<T, i, i + 1>(lds_sp + s4, wm0, lane, a);
                    constexpr int PER = 8 / FM; // eight copies
#pragma unroll
                    for (int c = PER * i; c < PER * (i + 1); ++c) {
                        const int q = c / 2;
                        copy(q == 0 || q == 2, q == 1 || q == 2 ? 1 : 0, q < 2 ? s + 2 : s + 3, slot(10 + q), c & 1);
                    }
                });
                head = head + 4 < 10 ? head + 4 : head - 6;
#pragma unroll
                for (int j = 0; j < FN; ++j) b0[j] = b1[j];
            }
        }
        sp_drain();
    }
    const bool whole = m0 + T <= ROW * g.M && n0 + T <= g.N && g.write_tri == 0 && g.mask == 0;
    const int row0 = m0 + wm0 + (lane & 15), col0 = n0 + wn0;
    if (whole) {
#pragma unroll
        for (int i = 0; i < Cfg::FM; ++i) {
            sp_store<CPLX, false>(g, acc[i], row0 + 16 * i, col0, lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < Cfg::FM; ++i) {
            sp_store<CPLX, true>(g, acc[i], row0 + 16 * i, col0, lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

namespace {

inline int sp_round_up(int x, int m) { return (x + m - 1) / m * m; }

struct SplitLayout {
    int Mpad, Npad, slabs;
    size_t a_bytes, b_bytes;
};

template <int T, int PLANES, bool CPLX>
SplitLayout sp_layout(const icl_gemm_args* g)
{
    SplitLayout l;
    l.Mpad = sp_round_up((CPLX ? 2 : 1) * g->M, T);
    l.Npad = sp_round_up(g->N, T);
    l.slabs = sp_round_up((CPLX ? 2 : 1) * g->K, kSlabK) / kSlabK;
    l.a_bytes = (size_t)l.slabs * PLANES * kGroups * l.Mpad * 16;
    l.b_bytes = (size_t)l.slabs * PLANES * kGroups * l.Npad * 16;
    return l;
}

template <int T, int PLANES, bool CPLX>
size_t sp_workspace(const icl_gemm_args* g)
{
    const SplitLayout l = sp_layout<T, PLANES, CPLX>(g);
    return l.a_bytes + l.b_bytes;
}

// Packs arows packed rows of `a` and brows of `b` (multiples of 64).
template <int PLANES, bool CPLX>
hipError_t sp_pack(const SplitSrc& a, int arows, const SplitSrc& b, int brows, const SplitArgs& p, hipStream_t s)
{
    const dim3 grid((unsigned)((arows + brows) / 64), (unsigned)((p.slabs + 1) / 2));
    hipLaunchKernelGGL((split_pack_kernel<PLANES, CPLX>), grid, dim3(256), 0, s, a, b, arows / 64, p.slabs,
                       const_cast<unsigned long long*>(p.guard), p.epoch);
    return hipGetLastError();
}

// The product of the rows and columns of g (a part of the packed problem p).
template <int T, int PLANES, bool CPLX>
hipError_t sp_product(SplitArgs p, const icl_gemm_args& g, hipStream_t s)
{
    constexpr int WVM = 2, WVN = T == 256 ? 4 : 2;
    using C = SplitCfg<T, WVM, WVN>;
    p.g = g;
    return launch_gemm<T / (CPLX ? 2 : 1), T, C::NT, C::LDS_BYTES>(split_gemm_kernel<T, WVM, WVN, PLANES, CPLX>, &g, s, p);
}

// The rows [r0, r0 + rows) of a real source and its packed layout.
SplitSrc sp_rows(SplitSrc src, int r0, int rows)
{
    src.X += src.kcontig ? (long)r0 * src.ld : (long)r0;
    src.R = rows;
    src.P += (size_t)r0 * 8;
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
            if ((e = sp_pack<2, false>(sp_rows(a, 0, m0), m0, sp_rows(b, 0, n0), n0, p, s)) != hipSuccess) return e;
            if ((e = hipEventRecord(side->start, s)) != hipSuccess) return e;
            if ((e = hipStreamWaitEvent(side->stream, side->start, 0)) != hipSuccess) return e;
            e = sp_pack<2, false>(sp_rows(a, m0, g->M - m0), g->M - m0, sp_rows(b, n0, g->N - n0), g->N - n0, p,
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
                pq.Ap = Ap + (size_t)part[q][0] * 8;
                pq.Bp = Bp + (size_t)part[q][2] * 8;
                if ((e = sp_product<T, PLANES, CPLX>(pq, gq, s)) != hipSuccess) return e;
            }
            return icl_timer_mark(s);
        }
    }
    if ((e = sp_pack<PLANES, CPLX>(a, l.Mpad, b, l.Npad, p, s)) != hipSuccess) return e;
    if constexpr (T == 256) {
        // A square triangle update runs the tiles off the diagonal 256 x 256 blocks,
        // then those of the blocks at a quarter of the size, on the same packed
        // operands: half of a diagonal block's large tile would be thrown away, and
        // SSYRK 8192's 528 large tiles end in a round of 16 on 256 CUs.
        if ((g->write_tri == ICL_TRI_LOWER || g->write_tri == ICL_TRI_UPPER) && g->M == g->N &&
            g->M >= 2 * ICL_TRI_BAND_BLOCK && g->kband == ICL_KBAND_NONE) {
            icl_gemm_args part = *g;
            part.write_tri = g->write_tri | ICL_TRI_OFF_BAND;
            if ((e = icl_timer_mark(s)) != hipSuccess) return e;
            if ((e = sp_product<T, PLANES, CPLX>(p, part, s)) != hipSuccess) return e;
            if ((e = icl_timer_mark(s)) != hipSuccess) return e;
            part.write_tri = g->write_tri | ICL_TRI_BAND;
            if ((e = icl_timer_mark(s)) != hipSuccess) return e;
            if ((e = sp_product<128, PLANES, CPLX>(p, part, s)) != hipSuccess) return e;
            return icl_timer_mark(s);
        }
    }
    if ((e = icl_timer_mark(s)) != hipSuccess) return e;
    if ((e = sp_product<T, PLANES, CPLX>(p, *g, s)) != hipSuccess) return e;
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
     1}

static const icl_gemm_variant kTable[] = {
    ICL_GEMM_SPLIT("sgemm_f32_split3_256x256", ICL_KIND_SGEMM, ICL_MATH_FP32, 3, false, 256, 275.0f, 1),
    ICL_GEMM_SPLIT("sgemm_f32_split3_128x128", ICL_KIND_SGEMM, ICL_MATH_FP32, 3, false, 128, 242.0f, 2),
    ICL_GEMM_SPLIT("cgemm_f32_split3_128x256", ICL_KIND_CGEMM, ICL_MATH_FP32, 3, true, 256, 272.0f, 1),
    ICL_GEMM_SPLIT("cgemm_f32_split3_64x128", ICL_KIND_CGEMM, ICL_MATH_FP32, 3, true, 128, 240.0f, 2),
    ICL_GEMM_SPLIT("sgemm_bf16x3d_mfma_256x256", ICL_KIND_SGEMM, ICL_MATH_BF16X3, 2, false, 256, 490.0f, 1),
    ICL_GEMM_SPLIT("sgemm_bf16x3d_mfma_128x128", ICL_KIND_SGEMM, ICL_MATH_BF16X3, 2, false, 128, 426.0f, 2),
    ICL_GEMM_SPLIT("cgemm_bf16x3d_mfma_128x256", ICL_KIND_CGEMM, ICL_MATH_BF16X3, 2, true, 256, 490.0f, 1),
    ICL_GEMM_SPLIT("cgemm_bf16x3d_mfma_64x128", ICL_KIND_CGEMM, ICL_MATH_BF16X3, 2, true, 128, 400.0f, 2),
};
ICL_REGISTER_VARIANTS(kTable)
