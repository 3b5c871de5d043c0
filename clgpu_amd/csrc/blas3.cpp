// Host-side level-3 algorithms: implementation selection, GEMM dispatch, the
// recursive blocked STRSM, mixed-precision refinement and the adjoints.
#include "blas3.hpp"
#include "level3_tiles.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace icl {

thread_local KernelTimer* t_active_timer = nullptr;
thread_local const icl_side_lane* t_side_lane = nullptr;

// ---------------------------------------------------------------------------
// Registry
// ---------------------------------------------------------------------------
const std::vector<const icl_gemm_variant*>& gemm_registry()
{
    static const std::vector<const icl_gemm_variant*> all = [] {
        std::vector<const icl_gemm_variant*> v;
        const int n = icl_gemm_variant_count();
        for (int i = 0; i < n; ++i) v.push_back(icl_gemm_variant_at(i));
        return v;
    }();
    return all;
}

static bool level3_problem(const icl_gemm_args& g)
{
    return g.write_tri != ICL_TRI_NONE || g.kband != ICL_KBAND_NONE || g.cflags != 0;
}

bool gemm_accept(const icl_gemm_variant& v, const GemmProblem& p)
{
    // The band flags of write_tri select tiles by whole 256 x 256 diagonal blocks.
    const bool band_ok = (p.args->write_tri & (ICL_TRI_OFF_BAND | ICL_TRI_BAND)) == 0 ||
                         (ICL_TRI_BAND_BLOCK % v.bm == 0 && ICL_TRI_BAND_BLOCK % v.bn == 0);
    const bool ws_ok = v.math != ICL_MATH_FP32 || !v.workspace || p.optional_ws;
    return v.kind == p.kind && v.math == p.math && (v.level3 || !level3_problem(*p.args)) && band_ok && ws_ok;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

bool gemm_needs_edge(const icl_gemm_variant& v, const GemmProblem& p)
{
    const icl_gemm_args& g = *p.args;
    // 16-byte loads along each operand's contiguous dimension need aligned columns.
    const long vec = p.kind == ICL_KIND_CGEMM ? 2 : 4;
    const bool even = g.M % v.bm == 0 && g.N % v.bn == 0 && g.K % v.bk == 0;
    const bool aligned = aligned16(g.A) && aligned16(g.B) && g.lda % vec == 0 && g.ldb % vec == 0;
    return !(even && aligned);
}

// Score = 1 / estimated run time (seconds). Each variant carries its measured
// full-GPU rate R (TFLOP/s at 8192^3 of its main kernel) and occupancy occ
// (workgroups per CU). With 256 CUs, 256*occ tiles run concurrently, each tile
// taking t_tile = 2*bm*bn*K*flops_per_mac_scale / (R / (256*occ)) when the CUs
// are full; the grid runs in ceil(tiles / (256*occ)) rounds, so ragged problems
// pay for padded tiles. A last round with fewer than 256*occ tiles shares the
// CUs among fewer workgroups: it is taken to last t_tile * max(tiles_last, 256)
// / (256*occ), so grids of fewer tiles than CUs favour smaller tiles. A grid
// that fills only a fraction f of the CUs from the start (a single round) runs
// its tiles faster than a full chip does (a higher clock at the lower power,
// less contention for L2 and HBM): (0.7 + 0.3 f) of that time, fitted to SSYRK
// and CHERK triangles of 72 to 156 tiles. Variants with a pack prepass add its
// HBM time ((M + N) * K elements at 4 read and 4 written bytes, complex 8 and 8, at
// 5 TB/s). The bounds-checked instantiation is taken to run 10% slower: this ranks
// implementations of one kind; whether a split-BF16 product needs a workspace, which a
// handle's cap may refuse, hangs on these figures too. FP32 products on the three-way
// split kernels are chosen in gemm_best.
// For K <= 512 a tile's fixed cost (pipeline fill, C read and write) is no
// longer small against its K loop: it is counted as kTileOverheadK * (elements
// of C per wave) extra steps of K, normalised so that the rate at K = 8192 is
// still the measured one (fitted to 64x64 and 128x128 tiles at K = 256, M up
// to 3840, N = 1024, where the larger tile took 1.5x as long as the smaller).
constexpr double kTileOverheadK = 0.12;
float gemm_score(const icl_gemm_variant& v, const GemmProblem& p)
{
    const icl_gemm_args& g = *p.args;
    constexpr double kCUs = 256.0;
    const double macs = p.kind == ICL_KIND_CGEMM ? 4.0 : 1.0; // real MACs per element MAC
    const double conc = kCUs * (v.occupancy > 0 ? v.occupancy : 1);
    // Level-3 launches: only the tiles meeting the written triangle run.
    const double tiles = g.write_tri != ICL_TRI_NONE
                             ? double(tri_tile_count(g.M, g.N, g.write_tri, v.bm, v.bn))
                             : double((g.M + v.bm - 1) / v.bm) * double((g.N + v.bn - 1) / v.bn);
    const double rate = (v.tflops_hint > 0 ? v.tflops_hint : 1.0) * 1e12;
    double t_tile = 2.0 * macs * v.bm * v.bn * double(g.K) * conc / rate;
    if (g.K > 0 && g.K <= 512) { // (a K = 0 call only scales C)
        const double k0 = kTileOverheadK * v.bm * v.bn / (v.threads / 64);
        t_tile *= (double(g.K) + k0) / double(g.K) * 8192.0 / (8192.0 + k0);
    }
    const double rounds = std::ceil(tiles / conc);
    const double last = tiles - (rounds - 1.0) * conc;
    double t = (rounds - 1.0) * t_tile + t_tile * std::max(last, kCUs) / conc;
    if (rounds == 1.0) t *= 0.7 + 0.3 * std::min(tiles, kCUs) / kCUs;
    if (gemm_needs_edge(v, p)) t *= 1.10;
    if (v.workspace) t += (double(g.M) + double(g.N)) * double(g.K) * (p.kind == ICL_KIND_CGEMM ? 16.0 : 8.0) / 5e12;
    return (float)(1.0 / t);
}

static const icl_gemm_variant* gemm_best(const GemmProblem& p);

static bool forced_is_gemm_of_kind(const std::string& name, int kind)
{
    for (const icl_gemm_variant* v : gemm_registry())
        if (name == v->name) return v->kind == kind;
    return false;
}

const icl_gemm_variant* gemm_select(iclblasContext* h, const GemmProblem& p)
{
    // Problems using the level-3 fields run only on kernels that implement them,
    // so a forced variant without them is not used there.
    const bool level3 = level3_problem(*p.args);
    if (!h->forced_impl.empty() && forced_is_gemm_of_kind(h->forced_impl, p.kind)) {
        for (const icl_gemm_variant* v : gemm_registry())
            if (h->forced_impl == v->name && (!level3 || v->level3) &&
                (v->math != ICL_MATH_FP32 || !v->workspace || p.optional_ws))
                return v;
    }
    return gemm_best(p);
}

// The three-way split kernels are candidates from a packed depth of 128 (k, or 2 k
// of a complex product) and 0.1 G real multiply-adds on: the pack, the product and the
// guarded kernel behind it take 20 us at the least. The workspace (12 bytes per padded
// element of op(A) and op(B)^T at most, and 256 MiB of partial sums) is bounded.
constexpr int kSplit3MinDepth = 128;
constexpr double kSplit3MinMacs = 0.1e9;
constexpr size_t kSplit3MaxBytes = size_t(8) << 30;
static double real_macs(int kind, const icl_gemm_args& g)
{
    return (kind == ICL_KIND_CGEMM ? 4.0 : 1.0) * g.M * double(g.N) * g.K;
}
static bool split3_candidate(int kind, const icl_gemm_args& g)
{
    return (kind == ICL_KIND_CGEMM ? 2 : 1) * g.K >= kSplit3MinDepth && real_macs(kind, g) >= kSplit3MinMacs;
}

// Seconds a product takes on a tiled kernel without a prepass: the tiles of the busiest
// CU at its full rate (alone on a CU a tile takes 1.25 times as long as its share of a
// full one: it has one wave per SIMD), FP32 bounds-checked 1.9 (complex 1.6) and with a
// triangle 1.25 times that, and 4 us. Against 120 random products this was off by 13%.
static double tiled_time(const GemmProblem& p, const icl_gemm_variant& v)
{
    const icl_gemm_args& g = *p.args;
    const bool cplx = p.kind == ICL_KIND_CGEMM;
    constexpr double kCUs = 256.0;
    const double tiles = g.write_tri != ICL_TRI_NONE
                             ? double(tri_tile_count(g.M, g.N, g.write_tri, v.bm, v.bn))
                             : double((g.M + v.bm - 1) / v.bm) * double((g.N + v.bn - 1) / v.bn);
    const double each = 2.0 * (cplx ? 4.0 : 1.0) * v.bm * v.bn * double(g.K) * kCUs / (v.tflops_hint * 1e12);
    double t = tiles <= kCUs ? 1.25 * each : std::ceil(tiles / kCUs) * each;
    if (g.kband != ICL_KBAND_NONE) t = std::max(1.25 * each, 0.5 * tiles / kCUs * each);
    if (v.math == ICL_MATH_FP32 && gemm_needs_edge(v, p)) t *= cplx ? 1.6 : 1.9;
    if (g.write_tri != ICL_TRI_NONE) t *= 1.25;
    return t + 4e-6;
}

// The accepted implementation with the highest score.
static const icl_gemm_variant* gemm_best(const GemmProblem& p)
{
    const icl_gemm_variant *best = nullptr, *split = nullptr, *wave = nullptr;
    float best_score = -1.0f;
    double split_time = 0.0;
    const bool splits = p.optional_ws && split3_candidate(p.kind, *p.args);
    for (const icl_gemm_variant* v : gemm_registry()) {
        if (!gemm_accept(*v, p) || (p.no_ws && v->workspace) || (p.tiled && (v->workspace || v->estimate))) continue;
        if (!v->workspace && v->estimate) {
            wave = v;
            continue;
        }
        if (v->workspace && splits) {
            const double t = v->estimate(p.args);
            if ((!split || t < split_time) && v->workspace(p.args) <= kSplit3MaxBytes) {
                split = v;
                split_time = t;
            }
        }
        if (v->workspace && v->math == ICL_MATH_FP32) continue;
        const float s = gemm_score(*v, p);
        if (s > best_score) {
            best = v;
            best_score = s;
        }
    }
    if (best && !best->workspace && (wave || split)) {
        // The estimates of the three families. Real FP32 products of less than 2 G
        // multiply-adds move to the packed kernels only for a gain of a third: callers
        // without a workspace (iclblasSgemmNoAlloc, capped handles, captured streams)
        // cannot, and their results should differ from iclblasSgemm's only where it pays
        // (1024 x 1536 x 1024: 49 us against 40). Chosen so, 120 random products lost 1%
        // against the fastest kernel of each (all on FP32 MFMA tiles: 50%).
        double t = tiled_time(p, *best);
        if (const double w = wave ? wave->estimate(p.args) : t; w < 0.9 * t) {
            best = wave;
            t = w;
        }
        const double margin = best->math == ICL_MATH_FP32 && p.kind == ICL_KIND_SGEMM && real_macs(p.kind, *p.args) < 2e9 ? 1.33
                              : p.args->write_tri != ICL_TRI_NONE ? 1.25 // tiled_time is high for short triangles
                                                                  : 1.0;
        if (split && t > margin * split_time) return split;
    }
    if (!best) throw status_error(ICLBLAS_STATUS_NOT_SUPPORTED, "no GEMM implementation accepts the parameters");
    if (best->math != ICL_MATH_FP32 && best->workspace) { // of the packed ones, the one that estimates the shortest time
        double best_time = best->estimate(p.args);
        for (const icl_gemm_variant* v : gemm_registry()) {
            if (v == best || !v->workspace || !gemm_accept(*v, p)) continue;
            const double t = v->estimate(p.args);
            if (t < best_time) {
                best = v;
                best_time = t;
            }
        }
    }
    return best;
}

// The workspace that a split-BF16 product may insist on, 0 for the ones that run without:
// what a handle's cap, a captured stream and the static scratch of iclblasSgemmNoAlloc
// have to have room for. A model of its own, fixed tiles at fixed rates ranked with the
// unpacked kernels by gemm_score, so that a call is not refused, or a graph does not
// need memory, because some kernel has become faster. The operands are packed once, 4
// bytes per element (complex: 8).
template <int BM, int BN, int BK, int BYTES>
static size_t packed_once(const icl_gemm_args* g)
{
    auto up = [](int x, int m) { return (size_t)((x + m - 1) / m) * m; };
    return (up(g->M, BM) + up(g->N, BN)) * up(g->K, BK) * BYTES;
}
#define ICL_PACKED_TILE(kind, BM, BN, BK, THREADS, BYTES, TF, OCC)                                                     \
    {"", kind, ICL_MATH_BF16X3, BM, BN, BK, THREADS, nullptr, packed_once<BM, BN, BK, BYTES>, TF, OCC, 1, nullptr}
static const icl_gemm_variant kPackedTiles[] = {
    ICL_PACKED_TILE(ICL_KIND_SGEMM, 256, 256, 32, 512, 4, 463.0f, 1),
    ICL_PACKED_TILE(ICL_KIND_SGEMM, 128, 128, 32, 256, 4, 366.0f, 2),
    ICL_PACKED_TILE(ICL_KIND_CGEMM, 256, 128, 16, 512, 8, 495.0f, 1),
    ICL_PACKED_TILE(ICL_KIND_CGEMM, 128, 128, 16, 256, 8, 387.0f, 1),
};
#undef ICL_PACKED_TILE

size_t gemm_required_workspace(const GemmProblem& p)
{
    const icl_gemm_variant* best = nullptr;
    float best_score = -1.0f;
    auto rank = [&](const icl_gemm_variant* v) {
        if (!gemm_accept(*v, p)) return;
        const float s = gemm_score(*v, p);
        if (s > best_score) {
            best = v;
            best_score = s;
        }
    };
    for (const icl_gemm_variant* v : gemm_registry())
        if (!v->workspace) rank(v);
    for (const icl_gemm_variant& v : kPackedTiles) rank(&v);
    return best && best->workspace ? best->workspace(p.args) : 0;
}

// A split-BF16 product without packed operands: on the unpacked kernels, or, as those
// have no level-3 options, on FP32 MFMA.
static const icl_gemm_variant* unpacked_variant(GemmProblem& p)
{
    p.optional_ws = false;
    p.no_ws = true;
    if (level3_problem(*p.args)) p.math = ICL_MATH_FP32;
    return gemm_best(p);
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------
// Smallest K for which the split-BF16 product meets the FP32 elementwise bound
// |C - C64| <= 4 k 2^-24 (|A||B|): the split leaves at most 3 * 2^-16 |a||b| per
// product (|x - hi - lo| <= 2^-16 |x| and the dropped lo*lo term), which is below
// 3 k 2^-24 |a||b| once k >= 256. Smaller K runs on FP32 MFMA instead.
constexpr int kSplitMinK = 256;

static bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hip_check(hipStreamIsCapturing(s, &capture), "hipStreamIsCapturing");
    return capture != hipStreamCaptureStatusNone;
}

// Whether a product may use memory that only makes it faster: not when it could not
// pay, when the caller has capped the handle's memory or forbidden allocation, and
// not while the stream is being captured (a later call could free a workspace that
// the graph would use).
static bool optional_workspace(iclblasContext* h, int kind, int math, const icl_gemm_args& g, hipStream_t s)
{
    if (g.K <= 0 || h->ext_ws || h->budget.limit || s != h->stream) return false;
    if (math == ICL_MATH_FP32 && h->forced_impl.empty() && !split3_candidate(kind, g)) return false;
    return !capturing(s);
}

// Whether a packed split-BF16 product fits in `room` bytes, and then how: the variant, and
// partial sums (unless whole) or the whole depth, that estimate the shortest time there.
static bool fit_packed(iclblasContext* h, const icl_gemm_variant*& v, const GemmProblem& p, icl_gemm_args& g,
                       size_t room, bool whole)
{
    const bool forced = h->forced_impl == v->name;
    const icl_gemm_variant* best = nullptr;
    int best_whole = 1;
    double best_time = 0.0;
    for (g.whole_depth = whole; g.whole_depth <= 1; ++g.whole_depth)
        for (const icl_gemm_variant* u : gemm_registry()) {
            if (forced ? u != v : !u->workspace || !gemm_accept(*u, p)) continue;
            const double t = u->estimate(&g);
            if ((best && t >= best_time) || u->workspace(&g) > room) continue;
            best = u;
            best_whole = g.whole_depth;
            best_time = t;
        }
    g.whole_depth = best_whole;
    if (best) v = best;
    return best != nullptr;
}

// The workspace of a split-BF16 product that gemm_select gave the packed variant v; may
// replace v by one that needs less, or none. Under a cap, in a captured stream and with
// the caller's scratch the product is refused when what it requires cannot be had, and
// takes no more than that, except into the optional buffer. A complex product needs more
// than its operands packed once (op(A) is packed as rows of two parts): without room for
// that it runs unpacked.
static void* packed_workspace(iclblasContext* h, const icl_gemm_variant*& v, GemmProblem& p, icl_gemm_args& g,
                              hipStream_t s)
{
    icl::DeviceScratch& own = h->scratch[iclblasContext::kSlotGemmWorkspace];
    icl::DeviceScratch& spare = h->scratch[iclblasContext::kSlotSplit3];
    const bool forced = h->forced_impl == v->name;
    icl_gemm_args once = g;
    once.whole_depth = 1;
    const size_t required = forced ? v->workspace(&once) : gemm_required_workspace(p);
    if (p.optional_ws) {
        // The lasting buffer grows, which frees the old one under any graph that holds it,
        // only for what a product requires: more goes to the optional buffer.
        const size_t bytes = v->workspace(&g);
        const bool lasting = bytes <= own.capacity() || required > own.capacity();
        if (void* ws = (lasting ? own : spare).try_get(bytes, s)) return ws;
        p.optional_ws = false;
    }
    if (required == 0) {
        v = unpacked_variant(p);
        return nullptr;
    }
    if (h->ext_ws) {
        if (required > h->ext_ws_bytes || !fit_packed(h, v, p, g, h->ext_ws_bytes, false))
            throw status_error(ICLBLAS_STATUS_INVALID_VALUE, "GEMM workspace exceeds the caller's scratch");
        return h->ext_ws;
    }
    const bool capped = h->budget.limit != 0;
    if (fit_packed(h, v, p, g, own.capacity(), capped)) return own.get(v->workspace(&g), s);
    if (p.kind == ICL_KIND_SGEMM || forced) {
        (void)fit_packed(h, v, p, g, required, true);
        return own.get(required, s);
    }
    if (!own.fits(required, true)) throw status_error(ICLBLAS_STATUS_ALLOC_FAILED, "scratch limit of the handle");
    if (capped && !capturing(s) && fit_packed(h, v, p, g, spare.room(), true))
        if (void* ws = spare.try_get(v->workspace(&g), s)) return ws;
    v = unpacked_variant(p);
    return nullptr;
}

// The product on a three-way split kernel `v`, then the FP32 MFMA kernel `native`
// guarded by its range check. False when the workspace cannot be had.
static bool run_split3(iclblasContext* h, const icl_gemm_variant* v, const icl_gemm_variant* native,
                       const GemmProblem& p, hipStream_t s)
{
    icl_gemm_args g = *p.args;
    void* ws = h->scratch[iclblasContext::kSlotSplit3].try_get(v->workspace(&g), s);
    icl::DeviceScratch& word = h->scratch[iclblasContext::kSlotGuard];
    const bool fresh = h->guard_epoch == 0;
    g.guard = ws ? static_cast<unsigned long long*>(word.try_get(256, s)) : nullptr;
    if (!g.guard) return false;
    if (fresh)
        hip_check(icl_axpby_2d(64, 1, 0.0f, nullptr, 0, 0.0f, reinterpret_cast<float*>(g.guard), 64, s), "axpby");
    g.guard_epoch = ++h->guard_epoch;
    hip_check(v->launch(&g, p.opa, p.opb, 0, ws, s), v->name);
    GemmProblem q = p;
    q.args = &g;
    hip_check(native->launch(&g, p.opa, p.opb, gemm_needs_edge(*native, q) ? 1 : 0, nullptr, s), native->name);
    return true;
}

// `stream`: the stream to run on (default the handle's; a variant with a
// workspace always runs on the handle's stream).
static void run_gemm(iclblasContext* h, int kind, int math, int opa, int opb, icl_gemm_args g, bool record,
                     hipStream_t stream = nullptr, bool tiled = false)
{
    if (math == ICL_MATH_BF16X3 && g.K < kSplitMinK) math = ICL_MATH_FP32;
    const hipStream_t s = stream ? stream : h->stream;
    GemmProblem p{kind, math, opa, opb, &g};
    p.tiled = tiled;
    p.optional_ws = !tiled && optional_workspace(h, kind, math, g, s);
    const icl_gemm_variant* v = gemm_select(h, p);
    if (level3_problem(g) && !v->level3)
        throw status_error(ICLBLAS_STATUS_INTERNAL_ERROR, "level-3 GEMM options on a kernel without them");
    if (v->math == ICL_MATH_FP32 && v->workspace) {
        p.optional_ws = false;
        const icl_gemm_variant* native = gemm_best(p);
        if (run_split3(h, v, native, p, s)) {
            if (record) h->last_impl = v->name;
            return;
        }
        v = native;
    }
    void* ws = v->workspace ? packed_workspace(h, v, p, g, s) : nullptr;
    const bool edge = gemm_needs_edge(*v, p);
    // A variant with a prepass marks its main kernel itself (icl_timer_mark),
    // and may run half of the prepass on the handle's side stream: offered for
    // products of at least 1024 tiles of that variant, never to a call that must
    // not allocate (the stream and its events are created on first use).
    if (v->workspace && s != h->stream)
        throw status_error(ICLBLAS_STATUS_INTERNAL_ERROR, "GEMM with a workspace off the handle's stream");
    if (!v->workspace) hip_check(icl_timer_mark(s), "icl_timer_mark");
    const long tiles = (long)((g.M + v->bm - 1) / v->bm) * ((g.N + v->bn - 1) / v->bn);
    struct SideGuard {
        explicit SideGuard(const icl_side_lane* l) { t_side_lane = l; }
        ~SideGuard() { t_side_lane = nullptr; }
    } side_guard(v->workspace && ws && !h->ext_ws && tiles >= 1024 && !level3_problem(g) ? h->side.ensure() : nullptr);
    hip_check(v->launch(&g, opa, opb, edge ? 1 : 0, ws, s), v->name);
    if (!v->workspace) hip_check(icl_timer_mark(s), "icl_timer_mark");
    if (record) h->last_impl = v->name;
}

void sgemm_dev(iclblasContext* h, int math, int opa, int opb, int m, int n, int k, float alpha, const float* A,
               long lda, const float* B, long ldb, float beta, float* C, long ldc, int mask, bool record)
{
    if (m <= 0 || n <= 0) return;
    if (k == 0 || alpha == 0.0f) {
        // C = beta * C; A and B are not read.
        hip_check(icl_axpby_2d(m, n, 0.0f, nullptr, 0, beta, C, ldc, h->stream), "axpby");
        if (mask != ICL_MASK_NONE)
            throw status_error(ICLBLAS_STATUS_INTERNAL_ERROR, "masked GEMM with k == 0 or alpha == 0");
        if (record) h->last_impl = "scale_c";
        return;
    }
    icl_gemm_args g{};
    g.M = m;
    g.N = n;
    g.K = k;
    g.A = A;
    g.B = B;
    g.C = C;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.alpha_re = alpha;
    g.beta_re = beta;
    g.mask = mask;
    run_gemm(h, ICL_KIND_SGEMM, math, opa, opb, g, record);
}

void cgemm_dev(iclblasContext* h, int math, int opa, int opb, int m, int n, int k, const float alpha[2],
               const float* A, long lda, const float* B, long ldb, const float beta[2], float* C, long ldc)
{
    if (m <= 0 || n <= 0) return;
    if (k == 0 || (alpha[0] == 0.0f && alpha[1] == 0.0f)) {
        hip_check(icl_caxpby_2d(m, n, 0.0f, 0.0f, nullptr, 0, beta[0], beta[1], C, ldc, h->stream), "caxpby");
        h->last_impl = "scale_c";
        return;
    }
    icl_gemm_args g{};
    g.M = m;
    g.N = n;
    g.K = k;
    g.A = A;
    g.B = B;
    g.C = C;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.alpha_re = alpha[0];
    g.alpha_im = alpha[1];
    g.beta_re = beta[0];
    g.beta_im = beta[1];
    run_gemm(h, ICL_KIND_CGEMM, math, opa, opb, g, true);
}

bool split_depth(iclblasContext* h, int k)
{
    return h->math_mode == ICLBLAS_MATH_SPLIT_BF16X3 && k >= kSplitMinK;
}

// A square triangle update (SYRK type) as two launches -- the tiles off the
// diagonal 256 x 256 blocks, which lie wholly inside the triangle and take the
// largest tile, then the diagonal band on smaller tiles -- when the scoring
// model puts the pair at least 3% below the whole triangle on one tile size
// (SSYRK 8192: 2080 tiles of 128^2 end in a 32-tile round; the 496 off-band
// tiles of 256^2 fill two rounds). FP32 path only: in the split-BF16 mode each
// launch would pack the operands again. Not with a forced implementation.
static bool band_split_pays(iclblasContext* h, int kind, int math, int opa, int opb, const icl_gemm_args& g)
{
    if (!h->forced_impl.empty() || math != ICL_MATH_FP32 || g.kband != ICL_KBAND_NONE || g.M != g.N ||
        g.M < 2 * ICL_TRI_BAND_BLOCK || (g.write_tri != ICL_TRI_LOWER && g.write_tri != ICL_TRI_UPPER))
        return false;
    auto est = [&](int tri) {
        icl_gemm_args t = g;
        t.write_tri = tri;
        GemmProblem p{kind, math, opa, opb, &t};
        p.tiled = true;
        return 1.0 / gemm_score(*gemm_best(p), p);
    };
    if (est(g.write_tri | ICL_TRI_OFF_BAND) + est(g.write_tri | ICL_TRI_BAND) >= 0.97 * est(g.write_tri)) return false;
    // The pair is two of the tiled launches that the model ranks; the packed and the wave
    // kernels run the triangle whole.
    GemmProblem whole{kind, math, opa, opb, &g};
    whole.optional_ws = optional_workspace(h, kind, math, g, h->stream);
    return !gemm_best(whole)->estimate;
}

void gemm_level3_dev(iclblasContext* h, int kind, int opa, int opb, int m, int n, int k, const float alpha[2],
                     const float* A, long lda, const float* B, long ldb, const float beta[2], float* C, long ldc,
                     int write_tri, int kband, int cflags)
{
    if (m <= 0 || n <= 0) return;
    icl_gemm_args g{};
    g.M = m;
    g.N = n;
    g.K = k;
    g.A = A;
    g.B = B;
    g.C = C;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.alpha_re = alpha[0];
    g.alpha_im = kind == ICL_KIND_CGEMM ? alpha[1] : 0.0f;
    g.beta_re = beta[0];
    g.beta_im = kind == ICL_KIND_CGEMM ? beta[1] : 0.0f;
    g.write_tri = write_tri;
    g.kband = kband;
    g.cflags = cflags;
    const int math = split_depth(h, k) ? ICL_MATH_BF16X3 : ICL_MATH_FP32;
    const bool split = band_split_pays(h, kind, math, opa, opb, g);
    if (split && opa == 0) {
        // The two launches write disjoint elements of C. With op(A) = A the band
        // runs on the handle's side stream beside the off-band launch, its small
        // workgroups sharing the CUs with the large ones (forked after the work
        // already queued, joined before the call returns): SSYRK 8192 op N 4.40 ->
        // 4.25 ms. With op(A) transposed the pair ran slower side by side (4.35 ->
        // 4.85 ms), so those launches stay one after the other.
        const icl_side_lane* side = h->side.ensure();
        hip_check(hipEventRecord(side->start, h->stream), "hipEventRecord");
        g.write_tri = write_tri | ICL_TRI_OFF_BAND;
        run_gemm(h, kind, math, opa, opb, g, true, nullptr, true);
        hip_check(hipStreamWaitEvent(side->stream, side->start, 0), "hipStreamWaitEvent");
        g.write_tri = write_tri | ICL_TRI_BAND;
        run_gemm(h, kind, math, opa, opb, g, true, side->stream, true);
        hip_check(hipEventRecord(side->done, side->stream), "hipEventRecord");
        hip_check(hipStreamWaitEvent(h->stream, side->done, 0), "hipStreamWaitEvent");
        return;
    }
    if (split) {
        g.write_tri = write_tri | ICL_TRI_OFF_BAND;
        run_gemm(h, kind, math, opa, opb, g, true, nullptr, true);
        g.write_tri = write_tri | ICL_TRI_BAND;
    }
    run_gemm(h, kind, math, opa, opb, g, true, nullptr, split);
}

// ---------------------------------------------------------------------------
// STRSM: recursive blocking. Each split solves one half, sends the coupling
// block through the FP32 GEMM (alpha = -1, beta = 1) and solves the other half;
// leaves of at most 64 unknowns go to the one-wave-per-64-RHS diagonal solver.
// ---------------------------------------------------------------------------
namespace {

constexpr int kLeaf = 64;
// Blocked STRSM above 64 unknowns: the panel solve with inverted 256 x 256
// diagonal panels (the panel's inverse applied to its right-hand sides, then a
// GEMM update of the rest) runs unless another implementation is forced; the
// panel solve with the in-workgroup panel kernel, the launch-per-64-block solve,
// the single-launch dataflow solve and the recursive solve are selectable by name.
constexpr int kPanel = 256;

// X_p = W_p B_p (left: the panel's rows of B, all columns) or B_p W_p (right:
// the panel's columns of B, all rows), as the arguments of icl_panel_apply. W_p
// is plen x plen with leading dimension kPanel; X is m x n with leading
// dimension m; p_lo is the panel's first unknown in original order; pointers
// and strides count complex elements when cplx.
icl_panel_apply_args panel_product(bool cplx, bool left, int plen, int m, int n, const float* Wp, const float* B,
                                   long ldb, float* X, int p_lo)
{
    icl_panel_apply_args a{};
    const long es = cplx ? 2 : 1;
    a.cplx = cplx ? 1 : 0;
    a.p = plen;
    a.W = Wp;
    if (left) { // X(r, l) = sum_k W(r, k) B(k, l), lines = columns
        a.nlines = n;
        a.w_rs = 1, a.w_ks = kPanel;
        a.B = B + es * p_lo, a.b_ks = 1, a.b_ls = ldb;
        a.X = X + es * p_lo, a.x_rs = 1, a.x_ls = m;
    } else { // X(l, c) = sum_k B(l, k) W(k, c), lines = rows
        a.nlines = m;
        a.w_rs = kPanel, a.w_ks = 1;
        a.B = B + es * (long)p_lo * ldb, a.b_ks = ldb, a.b_ls = 1;
        a.X = X + es * (long)p_lo * m, a.x_rs = m, a.x_ls = 1;
    }
    return a;
}

struct Trsm {
    iclblasContext* h;
    bool left, trans, unit, fwd;
    int m, n;
    const float* A;
    long lda;
    float* B;
    long ldb;
    long si, sk; // op(A)(p, q) = A[p * si + q * sk]

    // op(A)[i0.., j0..] as a GEMM operand: pointer and op flag.
    const float* sub(int i0, int j0, int* op) const
    {
        *op = trans ? 1 : 0;
        return A + (long)i0 * si + (long)j0 * sk;
    }

    void leaf(int p0, int nb, float s_post) const
    {
        icl_trsm_diag_args a{};
        a.nb = nb;
        a.unit = unit ? 1 : 0;
        a.s_pre = 1.0f;
        a.s_post = s_post;
        if (left) {
            a.nlines = n;
            a.x_sj = ldb;
            if (fwd) {
                a.L = A + (long)p0 * (si + sk);
                a.l_si = si;
                a.l_sk = sk;
                a.X = B + p0;
                a.x_si = 1;
            } else {
                const long e = p0 + nb - 1;
                a.L = A + e * (si + sk);
                a.l_si = -si;
                a.l_sk = -sk;
                a.X = B + e;
                a.x_si = -1;
            }
        } else {
            a.nlines = m;
            a.x_sj = 1;
            if (fwd) {
                a.L = A + (long)p0 * (si + sk);
                a.l_si = sk;
                a.l_sk = si;
                a.X = B + (long)p0 * ldb;
                a.x_si = ldb;
            } else {
                const long e = p0 + nb - 1;
                a.L = A + e * (si + sk);
                a.l_si = -sk;
                a.l_sk = -si;
                a.X = B + e * ldb;
                a.x_si = -ldb;
            }
        }
        hip_check(icl_trsm_diag(&a, h->stream), "trsm_diag");
    }

    // Solve unknowns [p0, p1) (rows of X for left, columns for right).
    void solve(int p0, int p1, float s_post) const
    {
        const int len = p1 - p0;
        if (len <= kLeaf) {
            leaf(p0, len, s_post);
            return;
        }
        const int half = ((len / 2 + kLeaf - 1) / kLeaf) * kLeaf;
        const int mid = p0 + half;
        int op = 0;
        if (left) {
            if (fwd) {
                solve(p0, mid, s_post);
                const float* Asub = sub(mid, p0, &op);
                sgemm_dev(h, ICL_MATH_FP32, op, 0, p1 - mid, n, mid - p0, -1.0f, Asub, lda, B + p0, ldb, 1.0f,
                          B + mid, ldb, ICL_MASK_NONE, false);
                solve(mid, p1, s_post);
            } else {
                solve(mid, p1, s_post);
                const float* Asub = sub(p0, mid, &op);
                sgemm_dev(h, ICL_MATH_FP32, op, 0, mid - p0, n, p1 - mid, -1.0f, Asub, lda, B + mid, ldb, 1.0f,
                          B + p0, ldb, ICL_MASK_NONE, false);
                solve(p0, mid, s_post);
            }
        } else {
            if (fwd) {
                solve(p0, mid, s_post);
                const float* Asub = sub(p0, mid, &op);
                sgemm_dev(h, ICL_MATH_FP32, 0, op, m, p1 - mid, mid - p0, -1.0f, B + (long)p0 * ldb, ldb, Asub, lda,
                          1.0f, B + (long)mid * ldb, ldb, ICL_MASK_NONE, false);
                solve(mid, p1, s_post);
            } else {
                solve(mid, p1, s_post);
                const float* Asub = sub(mid, p0, &op);
                sgemm_dev(h, ICL_MATH_FP32, 0, op, m, mid - p0, p1 - mid, -1.0f, B + (long)mid * ldb, ldb, Asub, lda,
                          1.0f, B + (long)p0 * ldb, ldb, ICL_MASK_NONE, false);
                solve(p0, mid, s_post);
            }
        }
    }
};

// CTRSM: recursive blocking on interleaved complex data; strides and offsets
// count complex elements. The coupling blocks go through the FP32 CGEMM with op
// N, T or C as in op(A). The splits keep every leaf on a 64-unknown block of the
// canonical (forward) order -- backward solves split from the end -- so the
// leaves are products with the diagonal blocks' inverses, all inverted up front
// in one launch, rather than substitutions.
struct CTrsm {
    iclblasContext* h;
    bool left, trans, conj, unit, fwd;
    int m, n, order;
    const float* A;
    long lda;
    float* B;
    long ldb;
    long si, sk; // op(A)(p, q) = A[p * si + q * sk] (conjugated for OP_C)
    const float* invD;

    const float* sub(int i0, int j0, int* op) const
    {
        *op = trans ? (conj ? 2 : 1) : 0;
        return A + 2 * ((long)i0 * si + (long)j0 * sk);
    }

    // The canonical forward view of the whole system (unknown 0 solved first).
    void canonical_l(const float** L, long* l_si, long* l_sk) const
    {
        const long e = fwd ? 0 : order - 1;
        *L = A + 2 * e * (si + sk);
        const long a_si = left ? si : sk, a_sk = left ? sk : si;
        *l_si = fwd ? a_si : -a_si;
        *l_sk = fwd ? a_sk : -a_sk;
    }

    void leaf(int p0, int nb, const float s_post[2]) const
    {
        icl_ctrsm_apply_args a{};
        a.nb = nb;
        const int blk = fwd ? p0 / kLeaf : (order - (p0 + nb)) / kLeaf; // canonical block of the leaf
        a.invD = invD + (long)blk * kLeaf * kLeaf * 2;
        a.s_post_re = s_post[0];
        a.s_post_im = s_post[1];
        const long e = fwd ? p0 : p0 + nb - 1; // first unknown of the canonical order
        if (left) {
            a.nlines = n;
            a.x_sj = ldb;
            a.X = B + 2 * e;
            a.x_si = fwd ? 1 : -1;
        } else {
            a.nlines = m;
            a.x_sj = 1;
            a.X = B + 2 * e * ldb;
            a.x_si = fwd ? ldb : -ldb;
        }
        hip_check(icl_ctrsm_apply(&a, h->stream), "ctrsm_apply");
    }

    // Solve unknowns [p0, p1) (rows of X for left, columns for right).
    void solve(int p0, int p1, const float s_post[2]) const
    {
        const int len = p1 - p0;
        if (len <= kLeaf) {
            leaf(p0, len, s_post);
            return;
        }
        const int half = ((len / 2 + kLeaf - 1) / kLeaf) * kLeaf;
        const int mid = fwd ? p0 + half : p1 - half; // the part solved first is a whole number of blocks
        const float minus_one[2] = {-1.0f, 0.0f}, one[2] = {1.0f, 0.0f};
        const int first0 = fwd ? p0 : mid, first1 = fwd ? mid : p1;
        const int next0 = fwd ? mid : p0, next1 = fwd ? p1 : mid;
        int op = 0;
        solve(first0, first1, s_post);
        if (left) {
            const float* Asub = sub(next0, first0, &op);
            cgemm_dev(h, ICL_MATH_FP32, op, 0, next1 - next0, n, first1 - first0, minus_one, Asub, lda,
                      B + 2 * (long)first0, ldb, one, B + 2 * (long)next0, ldb);
        } else {
            const float* Asub = sub(first0, next0, &op);
            cgemm_dev(h, ICL_MATH_FP32, 0, op, m, next1 - next0, first1 - first0, minus_one,
                      B + 2 * (long)first0 * ldb, ldb, Asub, lda, one, B + 2 * (long)next0 * ldb, ldb);
        }
        solve(next0, next1, s_post);
    }
};

} // namespace

void ctrsm_dev(iclblasContext* h, int side, int uplo, int trans, int diag, int m, int n, const float alpha[2],
               const float* A, long lda, float* B, long ldb)
{
    if (m <= 0 || n <= 0) return;
    if (alpha[0] == 0.0f && alpha[1] == 0.0f) {
        // X = 0 without reading A or B (the documented contract, reference iclBLAS.h:1713, :1924)
        hip_check(icl_caxpby_2d(m, n, 0.0f, 0.0f, nullptr, 0, 0.0f, 0.0f, B, ldb, h->stream), "caxpby");
        h->last_impl = "ctrsm_zero";
        return;
    }
    CTrsm t{};
    t.h = h;
    t.left = side == ICLBLAS_SIDE_LEFT;
    t.trans = trans != ICLBLAS_OP_N;
    t.conj = trans == ICLBLAS_OP_C;
    t.unit = diag == ICLBLAS_DIAG_UNIT;
    t.m = m;
    t.n = n;
    t.A = A;
    t.lda = lda;
    t.B = B;
    t.ldb = ldb;
    t.si = t.trans ? lda : 1;
    t.sk = t.trans ? 1 : lda;
    const bool lower_eff = (uplo == ICLBLAS_FILL_MODE_LOWER) != t.trans; // op(A) lower triangular
    t.fwd = t.left ? lower_eff : !lower_eff;
    t.order = t.left ? m : n;
    if (t.order <= kLeaf) {
        // one diagonal block: the reference's substitution in registers, alpha
        // applied to the solution as the reference kernel does (Ctrsm_naive.cl:35)
        icl_ctrsm_diag_args a{};
        a.nb = t.order;
        a.unit = t.unit ? 1 : 0;
        a.conj = t.conj ? 1 : 0;
        a.s_post_re = alpha[0];
        a.s_post_im = alpha[1];
        long l_si = 0, l_sk = 0;
        t.canonical_l(&a.L, &l_si, &l_sk);
        a.l_si = l_si;
        a.l_sk = l_sk;
        const long e = t.fwd ? 0 : t.order - 1;
        if (t.left) {
            a.nlines = n;
            a.x_sj = ldb;
            a.X = B + 2 * e;
            a.x_si = t.fwd ? 1 : -1;
        } else {
            a.nlines = m;
            a.x_sj = 1;
            a.X = B + 2 * e * ldb;
            a.x_si = t.fwd ? ldb : -ldb;
        }
        hip_check(icl_ctrsm_diag(&a, h->stream), "ctrsm_diag");
        h->last_impl = "ctrsm_diag64";
        return;
    }
    const int nblk = (t.order + kLeaf - 1) / kLeaf;
    icl_ctrsm_blocked_args ia{};
    ia.nsys = t.order;
    t.canonical_l(&ia.L, &ia.l_si, &ia.l_sk);
    ia.unit = t.unit ? 1 : 0;
    ia.conj = t.conj ? 1 : 0;
    const float one[2] = {1.0f, 0.0f}, minus_one[2] = {-1.0f, 0.0f};
    if (h->forced_impl == "ctrsm_recursive_inv64") {
        float* invD = static_cast<float*>(h->scratch[iclblasContext::kSlotTrsmWorkspace].get(
            (size_t)nblk * kLeaf * kLeaf * 2 * sizeof(float), h->stream));
        ia.invD = invD;
        hip_check(icl_ctrsm_invert_blocks(&ia, h->stream), "ctrsm_invert_blocks");
        t.invD = invD;
        t.solve(0, t.order, one);
        if (alpha[0] != 1.0f || alpha[1] != 0.0f)
            hip_check(icl_caxpby_2d(m, n, alpha[0], alpha[1], B, ldb, 0.0f, 0.0f, B, ldb, h->stream), "caxpby");
        h->last_impl = "ctrsm_recursive_inv64";
        return;
    }
    // Panels of 256 unknowns: the inverse W_p of every diagonal panel is formed
    // up front (from the inverted 64 x 64 blocks, by recursive doubling in three
    // launches over all panels; none depends on B), then panel by panel X_p = W_p B_p (left) or B_p W_p (right)
    // with the panel's right-hand sides already updated, and one CGEMM updates
    // every later unknown. W_p is stored in original coordinates: reversed in both
    // indices for a backward solve, transposed for a right-side solve
    // (X op(A) = B is op(A)^T X^T = B^T, so X = B inv(L)^T). X is kept apart from
    // B (m x n, ld m) and copied back scaled by alpha at the end.
    const int npanels = (t.order + kPanel - 1) / kPanel;
    const size_t inv_floats = (size_t)nblk * kLeaf * kLeaf * 2, x_floats = (size_t)m * n * 2;
    const size_t w_floats = (size_t)npanels * kPanel * kPanel * 2;
    const size_t t_floats = (size_t)npanels * 4 * kLeaf * kLeaf * 2;
    float* ws = static_cast<float*>(h->scratch[iclblasContext::kSlotTrsmWorkspace].get(
        (inv_floats + x_floats + w_floats + t_floats) * sizeof(float), h->stream));
    float* Xb = ws + inv_floats;
    float* W = Xb + x_floats;
    ia.invD = ws;
    hip_check(icl_ctrsm_invert_blocks(&ia, h->stream), "ctrsm_invert_blocks");
    icl_ctrsm_panel_inv_args pa{};
    pa.nsys = t.order;
    pa.L = ia.L;
    pa.l_si = ia.l_si;
    pa.l_sk = ia.l_sk;
    pa.conj = ia.conj;
    pa.invD = ws;
    pa.W = W;
    pa.w_rs = t.left ? 1 : kPanel;
    pa.w_cs = t.left ? kPanel : 1;
    pa.rev = t.fwd ? 0 : 1;
    pa.T = W + w_floats;
    hip_check(icl_ctrsm_invert_panels(&pa, h->stream), "ctrsm_invert_panels");
    for (int ps = 0; ps < t.order; ps += kPanel) {
        const int pe = std::min(t.order, ps + kPanel);
        const int plen = pe - ps, rlen = t.order - pe;
        const int p_lo = t.fwd ? ps : t.order - pe; // original index of the panel's first unknown
        const int r_lo = t.fwd ? pe : 0;            // original index of the first later unknown
        const float* Wp = W + (size_t)(ps / kPanel) * kPanel * kPanel * 2;
        const icl_panel_apply_args xa = panel_product(true, t.left, plen, m, n, Wp, B, ldb, Xb, p_lo);
        hip_check(icl_panel_apply(&xa, h->stream), "panel_apply");
        if (pe == t.order) break;
        // The later unknowns: B_r -= op(A)[r, p] X_p (left) or X_p op(A)[p, r]
        // (right), a product of depth 256 (plen), on the complex LDS-DMA panel
        // kernel when the operands allow 16-byte copies, else on a CGEMM.
        // op(A)(i, j) = A[i si + j sk] (complex elements), conjugated for op C.
        int op = 0;
        icl_panel_gemm_args g{};
        g.nprob = 1;
        icl_panel_gemm_problem& u = g.prob[0];
        u.alpha = -1.0f;
        u.beta = 1.0f;
        if (t.left) { // D(i, l) = B(r_lo + i, l), P = op(A)[r_lo + i, p_lo + k], Q = X(p_lo + k, l)
            const float* As = t.sub(r_lo, p_lo, &op);
            u.rows = rlen, u.lines = n;
            u.P = As, u.p_is = t.si, u.p_ks = t.sk, u.conj_p = op == 2;
            u.Q = Xb + 2 * (long)p_lo, u.q_ks = 1, u.q_ls = m;
            u.D = B + 2 * (long)r_lo, u.d_is = 1, u.d_ls = ldb;
            if (plen == kPanel && icl_cpanel_gemm_ok(&g)) hip_check(icl_cpanel_gemm(&g, h->stream), "cpanel_gemm");
            else
                cgemm_dev(h, ICL_MATH_FP32, op, 0, rlen, n, plen, minus_one, As, lda, Xb + 2 * (long)p_lo, m, one,
                          B + 2 * (long)r_lo, ldb);
        } else { // D(i, l) = B(i, r_lo + l), P = X(i, p_lo + k), Q = op(A)[p_lo + k, r_lo + l]
            const float* As = t.sub(p_lo, r_lo, &op);
            u.rows = m, u.lines = rlen;
            u.P = Xb + 2 * (long)p_lo * m, u.p_is = 1, u.p_ks = m;
            u.Q = As, u.q_ks = t.si, u.q_ls = t.sk, u.conj_q = op == 2;
            u.D = B + 2 * (long)r_lo * ldb, u.d_is = 1, u.d_ls = ldb;
            if (plen == kPanel && icl_cpanel_gemm_ok(&g)) hip_check(icl_cpanel_gemm(&g, h->stream), "cpanel_gemm");
            else
                cgemm_dev(h, ICL_MATH_FP32, 0, op, m, rlen, plen, minus_one, Xb + 2 * (long)p_lo * m, m, As, lda,
                          one, B + 2 * (long)r_lo * ldb, ldb);
        }
    }
    hip_check(icl_caxpby_2d(m, n, alpha[0], alpha[1], Xb, m, 0.0f, 0.0f, B, ldb, h->stream), "caxpby");
    h->last_impl = "ctrsm_panel256_inv";
}

// The panel solves of STRSM (panels of 256 unknowns in the canonical order):
//  - kPanelSubst (strsm_panel256): each panel solved by the in-workgroup panel
//    kernel, the later unknowns updated by one FP32 GEMM per panel;
//  - kPanelInv (strsm_panel256_inv): the inverses W_p of the full panels formed
//    up front, then per panel X_p = W_p B_p and the GEMM update;
//  - kPanelFused (strsm_panel256_fused, the default): W_p and M_p = L_rp W_p
//    (the later rows' coupling to the panel, times its inverse) formed up front,
//    then per panel one grouped depth-256 launch [X_p; B_r] = [W_p; -M_p] B_p
//    + [0; B_r].
enum PanelMode { kPanelSubst, kPanelInv, kPanelFused };

// Sum over the full panels p with later unknowns of 256 * rlen_p (the floats of
// the M_p stack), rlen_p = order - 256 (p + 1).
static size_t coupling_floats(int order)
{
    size_t sum = 0;
    for (int pe = kPanel; pe <= order; pe += kPanel) sum += (size_t)kPanel * (size_t)(order - pe);
    return sum;
}

// Workspace of a panel solve in floats: inverted 64 x 64 diagonal blocks, the
// solution X (m x n), the panel inverses W_p of the full panels, then one region
// holding first the identity stack W_p is formed from and afterwards (fused
// mode) the M_p stack. Zero when the solve needs none (at most 64 unknowns).
static size_t panel_ws_floats(int order, int m, int n, PanelMode mode)
{
    if (order <= kLeaf) return 0;
    const size_t nblk = (size_t)(order + kLeaf - 1) / kLeaf;
    const size_t nfull = mode == kPanelSubst ? 0 : (size_t)order / kPanel;
    const size_t ident = nfull ? (size_t)order * kPanel : 0;
    const size_t shared = mode == kPanelFused ? std::max(ident, coupling_floats(order)) : ident;
    return nblk * kLeaf * kLeaf + (size_t)m * n + nfull * kPanel * kPanel + shared;
}

// Queues the problems of `g` (any count) as launches of at most
// ICL_PANEL_GEMM_MAX problems each.
static void panel_gemm_all(iclblasContext* h, std::vector<icl_panel_gemm_problem>& probs)
{
    for (size_t i = 0; i < probs.size(); i += ICL_PANEL_GEMM_MAX) {
        icl_panel_gemm_args g{};
        g.nprob = (int)std::min<size_t>(ICL_PANEL_GEMM_MAX, probs.size() - i);
        for (int j = 0; j < g.nprob; ++j) g.prob[j] = probs[i + j];
        hip_check(icl_panel_gemm(&g, h->stream), "panel_gemm");
    }
}

// The TRSM workspace: the handle's grow-only buffer.
static void* trsm_workspace(iclblasContext* h, size_t bytes)
{
    return h->scratch[iclblasContext::kSlotTrsmWorkspace].get(bytes, h->stream);
}

void strsm_dev(iclblasContext* h, int side, int uplo, int trans, int diag, int m, int n, float alpha,
               const float* A, long lda, float* B, long ldb, bool record, bool reuse_inverses)
{
    if (m <= 0 || n <= 0) return;
    if (alpha == 0.0f) {
        // The API contract (reference iclBLAS.h:1713): with alpha == 0 neither A
        // nor B has to be initialised; X = 0.
        hip_check(icl_axpby_2d(m, n, 0.0f, nullptr, 0, 0.0f, B, ldb, h->stream), "axpby");
        if (record) h->last_impl = "strsm_zero";
        return;
    }
    Trsm t{};
    t.h = h;
    t.left = side == ICLBLAS_SIDE_LEFT;
    t.trans = trans != ICLBLAS_OP_N;
    t.unit = diag == ICLBLAS_DIAG_UNIT;
    t.m = m;
    t.n = n;
    t.A = A;
    t.lda = lda;
    t.B = B;
    t.ldb = ldb;
    t.si = t.trans ? lda : 1;
    t.sk = t.trans ? 1 : lda;
    const bool lower_eff = (uplo == ICLBLAS_FILL_MODE_LOWER) != t.trans; // op(A) lower triangular
    t.fwd = t.left ? lower_eff : !lower_eff;
    const int order = t.left ? m : n;
    const bool forced_rec = h->forced_impl == "strsm_recursive";
    if (order <= kLeaf) {
        // Single diagonal block: alpha applied to the solution, as the reference
        // kernel does (Strsm_naive.cl:35).
        t.solve(0, order, alpha);
        if (record) h->last_impl = "strsm_diag64";
    } else if (forced_rec) {
        t.solve(0, order, 1.0f);
        if (alpha != 1.0f) hip_check(icl_axpby_2d(m, n, alpha, B, ldb, 0.0f, B, ldb, h->stream), "axpby");
        if (record) h->last_impl = "strsm_recursive";
    } else {
        // Canonical forward view of the whole system (as in Trsm::leaf with p0 = 0).
        icl_trsm_blocked_args a{};
        a.nsys = order;
        a.nlines = t.left ? n : m;
        a.unit = t.unit ? 1 : 0;
        const long e = order - 1;
        if (t.left) {
            a.x_sj = ldb;
            if (t.fwd) {
                a.L = A, a.l_si = t.si, a.l_sk = t.sk, a.B = B, a.x_si = 1;
            } else {
                a.L = A + e * (t.si + t.sk), a.l_si = -t.si, a.l_sk = -t.sk, a.B = B + e, a.x_si = -1;
            }
        } else {
            a.x_sj = 1;
            if (t.fwd) {
                a.L = A, a.l_si = t.sk, a.l_sk = t.si, a.B = B, a.x_si = ldb;
            } else {
                a.L = A + e * (t.si + t.sk), a.l_si = -t.sk, a.l_sk = -t.si, a.B = B + e * ldb, a.x_si = -ldb;
            }
        }
        const int nblk = (order + kLeaf - 1) / kLeaf;
        const size_t inv_elems = (size_t)nblk * kLeaf * kLeaf;
        const std::string& f = h->forced_impl;
        const bool dataflow = f == "strsm_dataflow64";
        const bool panel = !dataflow && f != "strsm_blocked_inv64"; // the panel solves (the default among them:)
        const PanelMode mode = f == "strsm_panel256" ? kPanelSubst : f == "strsm_panel256_inv" ? kPanelInv
                                                                                              : kPanelFused;
        const bool panel_inv = mode != kPanelSubst;
        if (panel) {
            // X in original order with B's shape (m x n, ld m); the canonical X view
            // mirrors B's. Panels of 256 unknowns are solved one after the other,
            // and one FP32 GEMM per panel updates every later unknown, in original
            // coordinates (positive strides). strsm_panel256 solves each panel with
            // the in-workgroup panel kernel; strsm_panel256_inv first forms the
            // inverse of every full 256 x 256 diagonal panel at once (the panel
            // kernel on identity right-hand sides, all panels in one launch: they
            // do not depend on B) and then solves each panel with one GEMM
            // X_p = W_p B_p, which spreads over the whole GPU; the fused mode
            // (PanelMode) also forms the M_p up front and runs each panel as one
            // grouped launch.
            const int nfull = panel_inv ? order / kPanel : 0;
            const size_t w_elems = (size_t)nfull * kPanel * kPanel;
            float* ws = static_cast<float*>(trsm_workspace(h, panel_ws_floats(order, m, n, mode) * sizeof(float)));
            float* Xb = ws + inv_elems;
            float* W = Xb + (size_t)m * n;
            float* E = W + w_elems; // identity stack, then (fused) the M_p stack
            float* Mst = E;
            a.invD = ws;
            if (t.left) {
                a.X = t.fwd ? Xb : Xb + e;
                a.xv_si = t.fwd ? 1 : -1;
                a.xv_sj = m;
            } else {
                a.X = t.fwd ? Xb : Xb + e * m;
                a.xv_si = t.fwd ? (long)m : -(long)m;
                a.xv_sj = 1;
            }
            if (!reuse_inverses) hip_check(icl_trsm_invert_blocks(&a, h->stream), "trsm_invert_blocks");
            if (nfull && !reuse_inverses) {
                // W_p (256 x 256, column-major) such that the panel's unknowns in
                // original order are X_p = W_p B_p (left) or B_p W_p (right): the
                // canonical inverse inv_c, written reversed in both indices for a
                // backward solve and transposed for a right-side solve, formed by
                // recursive doubling from the inverted 64 x 64 blocks.
                icl_trsm_panel_inv_args pa{};
                pa.npanels = nfull;
                pa.L = a.L;
                pa.l_si = a.l_si;
                pa.l_sk = a.l_sk;
                pa.invD = a.invD;
                pa.W = W;
                pa.w_rs = t.left ? 1 : kPanel; // canonical (row, column) strides
                pa.w_cs = t.left ? kPanel : 1;
                pa.rev = t.fwd ? 0 : 1;
                pa.T = E; // scratch: npanels * 16384 floats of the identity / M_p region
                hip_check(icl_trsm_invert_panels(&pa, h->stream), "trsm_invert_panels");
            }
            // op(A)(i, j) = A[i * si + j * sk] in original coordinates
            auto opa = [&](int i0, int j0) { return A + (long)i0 * t.si + (long)j0 * t.sk; };
            if (mode == kPanelFused) {
                // Panel p (full, with rlen_p later unknowns) in original coordinates:
                // left  X_p = W_p B_p, B_r -= M_p B_p with M_p = op(A)[r, p] W_p
                //       (rlen_p x 256, ld rlen_p);
                // right X_p = B_p W_p, B_r -= B_p N_p with N_p = W_p op(A)[p, r]
                //       (256 x rlen_p, ld 256).
                // As panel_gemm problems D(i, l) = sum_k P(i, k) Q(k, l), i the
                // unknowns and l the lines (B's columns for left, rows for right).
                std::vector<icl_panel_gemm_problem> probs;
                size_t moff = 0;
                for (int p = 0; p < nfull; ++p) {
                    const int ps = p * kPanel, pe = ps + kPanel, rlen = order - pe;
                    if (rlen == 0) break;
                    const int p_lo = t.fwd ? ps : order - pe, r_lo = t.fwd ? pe : 0;
                    const float* Wp = W + (size_t)p * kPanel * kPanel;
                    icl_panel_gemm_problem q{};
                    q.alpha = 1.0f;
                    if (t.left) { // M(i, c) = sum_k op(A)(r_lo + i, p_lo + k) W(k, c)
                        q.rows = rlen, q.lines = kPanel;
                        q.P = opa(r_lo, p_lo), q.p_is = t.si, q.p_ks = t.sk;
                        q.Q = Wp, q.q_ks = 1, q.q_ls = kPanel;
                        q.D = Mst + moff, q.d_is = 1, q.d_ls = rlen;
                    } else { // N(j, i) = sum_k W(j, k) op(A)(p_lo + k, r_lo + i), W(j, k) = Wp[j + 256 k]
                        q.rows = kPanel, q.lines = rlen;
                        q.P = Wp, q.p_is = 1, q.p_ks = kPanel;
                        q.Q = opa(p_lo, r_lo), q.q_ks = t.si, q.q_ls = t.sk;
                        q.D = Mst + moff, q.d_is = 1, q.d_ls = kPanel;
                    }
                    if (!reuse_inverses) probs.push_back(q);
                    moff += (size_t)kPanel * rlen;
                }
                panel_gemm_all(h, probs);
                moff = 0;
                for (int ps = 0; ps < order; ps += kPanel) {
                    const int pe = std::min(order, ps + kPanel);
                    const int plen = pe - ps, rlen = order - pe;
                    const int p_lo = t.fwd ? ps : order - pe, r_lo = t.fwd ? pe : 0;
                    if (plen < kPanel) { // the last, partial panel: no later unknowns
                        hip_check(icl_trsm_panel(&a, ps, pe, h->stream), "trsm_panel");
                        break;
                    }
                    const float* Wp = W + (size_t)(ps / kPanel) * kPanel * kPanel;
                    icl_panel_gemm_args g{};
                    g.nprob = rlen > 0 ? 2 : 1;
                    icl_panel_gemm_problem& x = g.prob[0];
                    icl_panel_gemm_problem& u = g.prob[1];
                    x.rows = kPanel, x.alpha = 1.0f, x.beta = 0.0f, x.P = Wp;
                    u.rows = rlen, u.alpha = -1.0f, u.beta = 1.0f, u.P = Mst + moff;
                    if (t.left) {
                        x.lines = u.lines = n;
                        x.Q = u.Q = B + p_lo, x.q_ks = u.q_ks = 1, x.q_ls = u.q_ls = ldb;
                        x.p_is = u.p_is = 1, x.p_ks = kPanel, u.p_ks = rlen;
                        x.D = Xb + p_lo, x.d_is = 1, x.d_ls = m;
                        u.D = B + r_lo, u.d_is = 1, u.d_ls = ldb;
                    } else {
                        x.lines = u.lines = m;
                        x.Q = u.Q = B + (long)p_lo * ldb, x.q_ks = u.q_ks = ldb, x.q_ls = u.q_ls = 1;
                        x.p_is = u.p_is = kPanel, x.p_ks = u.p_ks = 1;
                        x.D = Xb + (long)p_lo * m, x.d_is = m, x.d_ls = 1;
                        u.D = B + (long)r_lo * ldb, u.d_is = ldb, u.d_ls = 1;
                    }
                    hip_check(icl_panel_gemm(&g, h->stream), "panel_gemm");
                    moff += (size_t)kPanel * rlen;
                }
                hip_check(icl_axpby_2d(m, n, alpha, Xb, m, 0.0f, B, ldb, h->stream), "axpby");
                if (record) h->last_impl = "strsm_panel256_fused";
                return;
            }
            for (int ps = 0; ps < order; ps += kPanel) {
                const int pe = std::min(order, ps + kPanel);
                const int plen = pe - ps, rlen = order - pe;
                const int p_lo = t.fwd ? ps : order - pe; // original index of the panel's first unknown
                const int r_lo = t.fwd ? pe : 0;          // original index of the first later unknown
                if (plen == kPanel && ps / kPanel < nfull) {
                    const float* Wp = W + (size_t)(ps / kPanel) * kPanel * kPanel;
                    const icl_panel_apply_args pa = panel_product(false, t.left, kPanel, m, n, Wp, B, ldb, Xb, p_lo);
                    hip_check(icl_panel_apply(&pa, h->stream), "panel_apply");
                } else {
                    hip_check(icl_trsm_panel(&a, ps, pe, h->stream), "trsm_panel");
                }
                if (pe == order) break;
                int op = 0;
                if (t.left) {
                    const float* As = t.sub(r_lo, p_lo, &op);
                    sgemm_dev(h, ICL_MATH_FP32, op, 0, rlen, n, plen, -1.0f, As, lda, Xb + p_lo, m, 1.0f, B + r_lo, ldb,
                              ICL_MASK_NONE, false);
                } else {
                    const float* As = t.sub(p_lo, r_lo, &op);
                    sgemm_dev(h, ICL_MATH_FP32, 0, op, m, rlen, plen, -1.0f, Xb + (long)p_lo * m, m, As, lda, 1.0f,
                              B + (long)r_lo * ldb, ldb, ICL_MASK_NONE, false);
                }
            }
            hip_check(icl_axpby_2d(m, n, alpha, Xb, m, 0.0f, B, ldb, h->stream), "axpby");
            if (record) h->last_impl = panel_inv ? "strsm_panel256_inv" : "strsm_panel256";
        } else if (dataflow) {
            // invD, the tile-major X (whole 64 x 64 tiles), then the flags / ticket / abort words
            const int ncb = (a.nlines + kLeaf - 1) / kLeaf;
            const size_t x_elems = (size_t)nblk * ncb * kLeaf * kLeaf;
            const size_t sync_ints = (size_t)icl_trsm_dataflow_sync_ints(order, a.nlines);
            char* ws = static_cast<char*>(h->scratch[iclblasContext::kSlotTrsmWorkspace].get(
                (inv_elems + x_elems) * sizeof(float) + sync_ints * sizeof(int), h->stream));
            a.invD = reinterpret_cast<float*>(ws);
            a.X = a.invD + inv_elems;
            a.xv_si = a.xv_sj = 0;
            a.sync = reinterpret_cast<int*>(a.X + x_elems);
            if (!h->trsm_error) {
                void* w = nullptr;
                hip_check(hipMalloc(&w, 256), "hipMalloc");
                h->trsm_error = static_cast<int*>(w);
            }
            // The word reports this solve only: cleared on the stream before it.
            hip_check(icl_axpby_2d(64, 1, 0.0f, nullptr, 0, 0.0f, reinterpret_cast<float*>(h->trsm_error), 64,
                                   h->stream),
                      "axpby");
            h->trsm_error_pending = true;
            a.error_word = h->trsm_error;
            // Diagnostics: ICLBLAS_DATAFLOW_WAIT_POLLS overrides the polls a wait
            // makes before it aborts (a negative value aborts the first wait).
            if (const char* env = std::getenv("ICLBLAS_DATAFLOW_WAIT_POLLS")) a.wait_polls = std::atoi(env);
            hip_check(icl_trsm_invert_blocks(&a, h->stream), "trsm_invert_blocks");
            hip_check(icl_trsm_dataflow(&a, alpha, h->stream), "trsm_dataflow");
            if (record) h->last_impl = "strsm_dataflow64";
        } else {
            float* ws = static_cast<float*>(h->scratch[iclblasContext::kSlotTrsmWorkspace].get(
                (inv_elems + (size_t)order * a.nlines) * sizeof(float), h->stream));
            a.invD = ws;
            a.X = ws + inv_elems;
            a.xv_si = 1;
            a.xv_sj = order;
            hip_check(icl_trsm_invert_blocks(&a, h->stream), "trsm_invert_blocks");
            for (int b = 0; b < nblk; ++b) hip_check(icl_trsm_step(&a, b, h->stream), "trsm_step");
            hip_check(icl_trsm_scatter(&a, alpha, h->stream), "trsm_scatter");
            if (record) h->last_impl = "strsm_blocked_inv64";
        }
    }
}

void trsm_check_error(iclblasContext* h)
{
    if (!h->trsm_error || !h->trsm_error_pending) return;
    h->trsm_error_pending = false;
    int e = 0;
    hip_check(hipMemcpy(&e, h->trsm_error, sizeof(int), hipMemcpyDeviceToHost), "hipMemcpy");
    if (e == 0) return;
    hip_check(icl_axpby_2d(64, 1, 0.0f, nullptr, 0, 0.0f, reinterpret_cast<float*>(h->trsm_error), 64, h->stream),
              "axpby");
    hip_check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
    throw status_error(ICLBLAS_STATUS_EXECUTION_FAILED, "STRSM dataflow solve exceeded its wait bound");
}

void strsm_refined_dev(iclblasContext* h, int side, int uplo, int trans, int diag, int m, int n, float alpha,
                       const float* A, long lda, float* B, long ldb, int sweeps, float* B0, float* R)
{
    h->last_sweeps = 0;
    if (m <= 0 || n <= 0) return;
    if (alpha == 0.0f || sweeps <= 0) {
        strsm_dev(h, side, uplo, trans, diag, m, n, alpha, A, lda, B, ldb);
        return;
    }
    // Keep the right-hand side: B0 = B (dense, ld = m).
    hip_check(hipMemcpy2DAsync(B0, (size_t)m * sizeof(float), B, (size_t)ldb * sizeof(float), (size_t)m * sizeof(float),
                               (size_t)n, hipMemcpyDeviceToDevice, h->stream),
              "hipMemcpy2DAsync");
    strsm_dev(h, side, uplo, trans, diag, m, n, alpha, A, lda, B, ldb, false);

    const bool left = side == ICLBLAS_SIDE_LEFT;
    const bool tr = trans != ICLBLAS_OP_N;
    const bool lower_eff = (uplo == ICLBLAS_FILL_MODE_LOWER) != tr;
    float* part = static_cast<float*>(
        h->scratch[iclblasContext::kSlotRefine].get(2 * ICL_ABSMAX_BLOCKS * sizeof(float), h->stream));
    float host_part[2 * ICL_ABSMAX_BLOCKS];
    h->last_sweeps = 0;
    for (int s = 0; s < sweeps; ++s) {
        icl_residual_args r{};
        r.M = m;
        r.N = n;
        r.K = left ? m : n;
        if (left) { // R = alpha*B0 - op(A) * X
            r.P = A;
            r.ldp = lda;
            r.p_trans = tr;
            r.Q = B;
            r.ldq = ldb;
            r.q_trans = 0;
            r.tri_on = 1;
        } else { // R = alpha*B0 - X * op(A)
            r.P = B;
            r.ldp = ldb;
            r.p_trans = 0;
            r.Q = A;
            r.ldq = lda;
            r.q_trans = tr;
            r.tri_on = 2;
        }
        r.tri_lower = lower_eff ? 1 : 0;
        r.tri_unit = diag == ICLBLAS_DIAG_UNIT ? 1 : 0;
        r.B0 = B0;
        r.ldb0 = m;
        r.R = R;
        r.ldr = m;
        r.alpha = (double)alpha;
        hip_check(icl_residual_f64(&r, h->stream), "residual_f64");
        // D = op(A)^-1 R (in place in R), X += D. The system is the first
        // solve's, and nothing in between uses the TRSM workspace: its inverses
        // are taken as they are.
        strsm_dev(h, side, uplo, trans, diag, m, n, 1.0f, A, lda, R, m, false, true);
        hip_check(icl_axpby_2d(m, n, 1.0f, R, m, 1.0f, B, ldb, h->stream), "axpby");
        h->last_sweeps = s + 1;
        if (s + 1 == sweeps) break;
        // Converged when the correction no longer changes X at FP32 resolution:
        // max |D| <= 2^-24 max |X|. Further sweeps would recompute the same
        // residual up to rounding, so the loop stops early.
        hip_check(icl_absmax_pair(m, n, R, m, B, ldb, part, h->stream), "absmax");
        hip_check(hipMemcpyAsync(host_part, part, sizeof(host_part), hipMemcpyDeviceToHost, h->stream),
                  "hipMemcpyAsync(D2H)");
        hip_check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
        float md = 0.0f, mx = 0.0f;
        for (int b = 0; b < ICL_ABSMAX_BLOCKS; ++b) {
            md = std::max(md, host_part[2 * b]);
            mx = std::max(mx, host_part[2 * b + 1]);
        }
        if (md <= 0x1p-24f * mx) break;
    }
    h->last_impl = "strsm_refined_f64res";
}

// ---------------------------------------------------------------------------
// Adjoints
// ---------------------------------------------------------------------------
void sgemm_backward_dev(iclblasContext* h, int transa, int transb, int m, int n, int k, float alpha, const float* A,
                        long lda, const float* B, long ldb, const float* dC, long lddc, float* dA, long ldda,
                        float* dB, long lddb)
{
    const int ta = transa != ICLBLAS_OP_N, tb = transb != ICLBLAS_OP_N;
    if (dA) {
        if (!ta) // dA (m x k) = alpha * dC * op(B)^T
            sgemm_dev(h, ICL_MATH_FP32, 0, tb ? 0 : 1, m, k, n, alpha, dC, lddc, B, ldb, 0.0f, dA, ldda);
        else // dA (k x m) = alpha * op(B) * dC^T
            sgemm_dev(h, ICL_MATH_FP32, tb, 1, k, m, n, alpha, B, ldb, dC, lddc, 0.0f, dA, ldda);
    }
    if (dB) {
        if (!tb) // dB (k x n) = alpha * op(A)^T * dC
            sgemm_dev(h, ICL_MATH_FP32, ta ? 0 : 1, 0, k, n, m, alpha, A, lda, dC, lddc, 0.0f, dB, lddb);
        else // dB (n x k) = alpha * dC^T * op(A)
            sgemm_dev(h, ICL_MATH_FP32, 1, ta, n, k, m, alpha, dC, lddc, A, lda, 0.0f, dB, lddb);
    }
    h->last_impl = "sgemm_backward";
}

void strsm_backward_dev(iclblasContext* h, int side, int uplo, int trans, int diag, int m, int n, float alpha,
                        const float* A, long lda, const float* X, long ldx, const float* dX, long lddx, float* dA,
                        long ldda, float* dB, long lddb, float* G)
{
    const bool left = side == ICLBLAS_SIDE_LEFT;
    const int ta = trans != ICLBLAS_OP_N;
    const int order = left ? m : n;
    // G = op(A)^-T dX (left) or dX op(A)^-T (right): the solve with op(A)^T.
    hip_check(hipMemcpy2DAsync(G, (size_t)m * sizeof(float), dX, (size_t)lddx * sizeof(float), (size_t)m * sizeof(float),
                               (size_t)n, hipMemcpyDeviceToDevice, h->stream),
              "hipMemcpy2DAsync");
    strsm_dev(h, side, uplo, ta ? ICLBLAS_OP_N : ICLBLAS_OP_T, diag, m, n, 1.0f, A, lda, G, m, false);
    if (dB) hip_check(icl_axpby_2d(m, n, alpha, G, m, 0.0f, dB, lddb, h->stream), "axpby");
    if (dA) {
        int mask;
        if (uplo == ICLBLAS_FILL_MODE_LOWER) mask = diag == ICLBLAS_DIAG_UNIT ? ICL_MASK_LOWER_STRICT : ICL_MASK_LOWER;
        else mask = diag == ICLBLAS_DIAG_UNIT ? ICL_MASK_UPPER_STRICT : ICL_MASK_UPPER;
        if (left) {
            if (!ta) // dA = -G * X^T  (m x m, K = n)
                sgemm_dev(h, ICL_MATH_FP32, 0, 1, order, order, n, -1.0f, G, m, X, ldx, 0.0f, dA, ldda, mask);
            else // dA = -X * G^T
                sgemm_dev(h, ICL_MATH_FP32, 0, 1, order, order, n, -1.0f, X, ldx, G, m, 0.0f, dA, ldda, mask);
        } else {
            if (!ta) // dA = -X^T * G  (n x n, K = m)
                sgemm_dev(h, ICL_MATH_FP32, 1, 0, order, order, m, -1.0f, X, ldx, G, m, 0.0f, dA, ldda, mask);
            else // dA = -G^T * X
                sgemm_dev(h, ICL_MATH_FP32, 1, 0, order, order, m, -1.0f, G, m, X, ldx, 0.0f, dA, ldda, mask);
        }
    }
    h->last_impl = "strsm_backward";
}

} // namespace icl

extern "C" const icl_side_lane* icl_gemm_side_lane(void) { return icl::t_side_lane; }

extern "C" hipError_t icl_timer_mark(hipStream_t stream)
{
    return icl::t_active_timer ? icl::t_active_timer->mark(stream) : hipSuccess;
}
