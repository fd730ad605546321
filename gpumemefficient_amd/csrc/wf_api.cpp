// wf_api.cpp -- host side of libwfdp.so: contexts, symbol encoding, strip
// planning, kernel selection and launches behind the C ABI in
// include/wfdp.h.
//
// The reference's host functions (LCS/GPU_Hyperlane_Share.cu:696-792,
// SmithWaterman/GPU_Hyperlane_Share.cu:683-781,
// EditDistance/GPU_Hyperlane_Share.cu:689-789) cudaMalloc and cudaMemset the
// whole (n1+3) x (n2+1) table, create multiProcessorCount streams and launch
// one kernel per strip on every call.  Here a context owns one stream and
// grow-only device arenas; a call encodes the two sequences to one-byte
// codes, uploads them, and runs one persistent launch whose workgroups claim
// strips in dependency order.  Device memory per pair is the codes plus one
// boundary row per strip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/wfdp.h"
#include "wf_device.h"
#include "wf_internal.h"
#include "wf_variants.h"

struct wf_plan {
    wf_ctx *ctx = nullptr;
    WfArenas own;
    WfPlanHost host;
    double kernel_ms = 0.0;
    bool ran = false;
    std::vector<WfResultDev> res;                  // of the last run
    hipGraph_t graph[2] = {nullptr, nullptr};      // per run mode, when captured
    hipGraphExec_t exec[2] = {nullptr, nullptr};
};

// ----------------------------------------------------------------------------
// Encoding
// ----------------------------------------------------------------------------

namespace {

// The encoder's two scans over the symbols, also built for AVX2 and chosen
// at run time: the baseline x86-64 target has no packed 32-bit min/max, and
// scalar scans took 40 us of a 65536-symbol pair's encoding (10 us vectorised).
__attribute__((always_inline)) inline void minmax_body(const int32_t *v, int64_t n, int32_t &lo, int32_t &hi)
{
    int32_t l = lo, h = hi;
    for (int64_t i = 0; i < n; ++i) {
        l = std::min(l, v[i]);
        h = std::max(h, v[i]);
    }
    lo = l;
    hi = h;
}
__attribute__((always_inline)) inline void scale_body(const int32_t *v, int64_t n, int scale, uint8_t *out)
{
    for (int64_t i = 0; i < n; ++i) out[i] = (uint8_t)(v[i] * scale);
}
__attribute__((target("avx2"))) void minmax_avx2(const int32_t *v, int64_t n, int32_t &lo, int32_t &hi)
{
    minmax_body(v, n, lo, hi);
}
__attribute__((target("avx2"))) void scale_avx2(const int32_t *v, int64_t n, int scale, uint8_t *out)
{
    scale_body(v, n, scale, out);
}
__attribute__((always_inline)) inline uint32_t umax_body(const int32_t *v, int64_t n)
{
    uint32_t m = 0;
    for (int64_t i = 0; i < n; ++i) m = std::max(m, (uint32_t)v[i]);
    return m;
}
__attribute__((target("avx2"))) uint32_t umax_avx2(const int32_t *v, int64_t n) { return umax_body(v, n); }
__attribute__((always_inline)) inline uint8_t bmax_body(const uint8_t *v, int64_t n)
{
    uint8_t m = 0;
    for (int64_t i = 0; i < n; ++i) m = std::max(m, v[i]);
    return m;
}
__attribute__((target("avx2"))) uint8_t bmax_avx2(const uint8_t *v, int64_t n) { return bmax_body(v, n); }
__attribute__((always_inline)) inline void shr2_body(uint8_t *v, int64_t n)
{
    for (int64_t i = 0; i < n; ++i) v[i] = (uint8_t)(v[i] >> 2);
}
__attribute__((target("avx2"))) void shr2_avx2(uint8_t *v, int64_t n) { shr2_body(v, n); }
__attribute__((always_inline)) inline void reverse_body(const uint8_t *src, int64_t n, uint8_t *dst)
{
    for (int64_t k = 0; k < n; ++k) dst[k] = src[n - 1 - k];
}
__attribute__((target("avx2"))) void reverse_avx2(const uint8_t *src, int64_t n, uint8_t *dst)
{
    reverse_body(src, n, dst);
}
bool host_avx2()
{
    static const bool yes = __builtin_cpu_supports("avx2");
    return yes;
}
void minmax(const int32_t *v, int64_t n, int32_t &lo, int32_t &hi)
{
    if (host_avx2())
        minmax_avx2(v, n, lo, hi);
    else
        minmax_body(v, n, lo, hi);
}
void scale_codes(const int32_t *v, int64_t n, int scale, uint8_t *out)
{
    if (host_avx2())
        scale_avx2(v, n, scale, out);
    else
        scale_body(v, n, scale, out);
}
// The largest symbol read as unsigned (negative symbols count as large).
uint32_t umax(const int32_t *v, int64_t n)
{
    return host_avx2() ? umax_avx2(v, n) : umax_body(v, n);
}
// The largest code, and codes divided by 4 (the byte tables' plain codes).
uint8_t bmax(const uint8_t *v, int64_t n)
{
    return host_avx2() ? bmax_avx2(v, n) : bmax_body(v, n);
}
void shr2(uint8_t *v, int64_t n)
{
    if (host_avx2())
        shr2_avx2(v, n);
    else
        shr2_body(v, n);
}
// dst[k] = src[n - 1 - k] (the reverse halves of column-split pairs).
void reverse_codes(const uint8_t *src, int64_t n, uint8_t *dst)
{
    if (host_avx2())
        reverse_avx2(src, n, dst);
    else
        reverse_body(src, n, dst);
}

}  // namespace

// Maps the symbols of one pair to one-byte codes.  Equality is all the three
// recurrences look at, so any injective renaming gives identical tables.
// Row tables need codes < 8 (SW, 4-bit fields) or < 32 (LCS, ED, 1-bit
// fields); larger alphabets fall back to comparing codes.
int wf_encode_pair(int problem, const int32_t *a, int64_t n1, const int32_t *b, int64_t n2,
                   uint8_t *out_a, uint8_t *out_b, int32_t *mode)
{
    const int table_limit = (problem == WF_SW) ? 8 : 32;
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    minmax(a, n1, lo, hi);
    minmax(b, n2, lo, hi);
    const int scale = (problem == WF_SW) ? 4 : 1;  // SW codes are bit offsets of 4-bit fields
    *mode = 0;
    if (n1 + n2 == 0) return WF_OK;
    // Unmasked steps left of column 0 (WFK_MODE_FREE_HEAD): always for LCS
    // and ED; for SW only with a code that matches no row -- the unused last
    // 4-bit field of the row tables, or any value above the codes in CMP mode.
    auto free_head = [&](int max_symbol, bool cmp) {
        if (problem != WF_SW) {
            *mode |= WFK_MODE_FREE_HEAD;
        } else if (cmp) {
            *mode |= WFK_MODE_FREE_HEAD | (0x1FF << WFK_MODE_NEVER_SHIFT);
        } else if (max_symbol < table_limit - 1) {
            *mode |= WFK_MODE_FREE_HEAD | (((table_limit - 1) * scale) << WFK_MODE_NEVER_SHIFT);
        }
    };
    if (lo >= 0 && hi < table_limit) {
        scale_codes(a, n1, scale, out_a);
        scale_codes(b, n2, scale, out_b);
        free_head(hi, false);
        return WF_OK;
    }
    // Dense renaming in order of first appearance.
    std::unordered_map<int32_t, int> ids;
    ids.reserve(64);
    auto id_of = [&](int32_t v) -> int {
        auto it = ids.find(v);
        if (it != ids.end()) return it->second;
        const int id = (int)ids.size();
        ids.emplace(v, id);
        return id;
    };
    std::vector<int> ia(n1), ib(n2);
    for (int64_t i = 0; i < n1; ++i) ia[i] = id_of(a[i]);
    for (int64_t i = 0; i < n2; ++i) ib[i] = id_of(b[i]);
    const int nsym = (int)ids.size();
    if (nsym > 256) return WF_ERR_ALPHABET;
    if (nsym <= table_limit) {
        for (int64_t i = 0; i < n1; ++i) out_a[i] = (uint8_t)(ia[i] * scale);
        for (int64_t i = 0; i < n2; ++i) out_b[i] = (uint8_t)(ib[i] * scale);
        free_head(nsym - 1, false);
    } else {
        *mode |= WFK_MODE_CMP;
        for (int64_t i = 0; i < n1; ++i) out_a[i] = (uint8_t)ia[i];
        for (int64_t i = 0; i < n2; ++i) out_b[i] = (uint8_t)ib[i];
        free_head(nsym - 1, true);
    }
    return WF_OK;
}

int wf_encode_job(const wf_job &j, int32_t tile_flags, bool perm4, uint8_t *a_out, uint8_t *b_out, int32_t *mode_out)
{
    int32_t mode = 0;
    const int st = wf_encode_pair(j.problem, j.a, j.n1, j.b, j.n2, a_out, b_out, &mode);
    if (st != WF_OK) return st;
    if (j.problem == WF_ED && ((j.flags | tile_flags) & WF_TILE_ED_TEXTBOOK)) mode |= WFK_MODE_TEXTBOOK;
    // SW with at most 4 symbols on a cell engine with two rows per lane:
    // byte row tables and plain codes (WFK_MODE_PERM4).
    if (perm4 && j.problem == WF_SW && !(mode & WFK_MODE_CMP)) {
        if (std::max(bmax(a_out, j.n1), bmax(b_out, j.n2)) <= 12) {
            shr2(a_out, j.n1);
            shr2(b_out, j.n2);
            mode = (mode & WFK_MODE_TEXTBOOK) | WFK_MODE_PERM4 | WFK_MODE_FREE_HEAD;
        }
    }
    *mode_out = mode;
    return WF_OK;
}

// Scores of degenerate pairs (an empty sequence), per the reference
// boundaries: LCS/SW 0; ED D(n2,0) = n2, D(0,n1) = n1-1 (n1 >= 1, ED.cpp
// :48-54) or n1 (textbook).
int32_t wf_empty_score(int problem, int64_t n1, int64_t n2, int flags)
{
    if (problem != WF_ED) return 0;
    if (n2 == 0) {
        if (n1 == 0) return 0;
        return (flags & WF_TILE_ED_TEXTBOOK) ? (int32_t)n1 : (int32_t)(n1 - 1);
    }
    return (int32_t)n2;
}

bool wf_perm4_enabled()
{
    const char *e = std::getenv("WFDP_PERM");
    return !(e && e[0] == '0');
}

// ----------------------------------------------------------------------------
// Variant choice
// ----------------------------------------------------------------------------

static int variant_count() { return wf_num_variants_async + wf_num_variants_lockstep + wf_num_variants_bitpar; }

static const WfVariant *variant_at(int i)
{
    if (i < 0 || i >= variant_count()) return nullptr;
    if (i < wf_num_variants_async) return &wf_variants_async[i];
    i -= wf_num_variants_async;
    if (i < wf_num_variants_lockstep) return &wf_variants_lockstep[i];
    return &wf_variants_bitpar[i - wf_num_variants_lockstep];
}

// The bit-parallel engine (wf_bitpar.hip) takes LCS and ED pairs whose
// symbols map to codes below 32 (its match-mask table has 32 rows).
bool wf_bitpar_eligible(const wf_job *jobs, int64_t njobs)
{
    for (int64_t i = 0; i < njobs; ++i) {
        const wf_job &j = jobs[i];
        if (j.problem != WF_LCS && j.problem != WF_ED) return false;
        if (std::max(umax(j.a, j.n1), umax(j.b, j.n2)) < 32u) continue;
        std::unordered_map<int32_t, int> seen;
        for (int64_t k = 0; k < j.n1 && seen.size() <= 32; ++k) seen.emplace(j.a[k], 0);
        for (int64_t k = 0; k < j.n2 && seen.size() <= 32; ++k) seen.emplace(j.b[k], 0);
        if (seen.size() > 32) return false;
    }
    return true;
}

static const WfVariant *find_variant(int E, int R, int W, int K)
{
    for (int i = 0; i < variant_count(); ++i) {
        const WfVariant *v = variant_at(i);
        if (v->engine == E && v->rows_per_lane == R && v->waves == W && v->chunk == K) return v;
    }
    return nullptr;
}

// Kernel variant for a plan, in order of precedence: explicit tile fields,
// the WFDP_VARIANT environment override ("engine,R,W,K"), the autotuned
// table (wf_tune.cpp) for this workload and device, built-in defaults.
// strip_rows = 64 * waves * rows_per_lane; tile_w maps to the chunk (the
// lock-step barrier interval, or the async progress interval).  tuned: may take
// the table's.
static const WfVariant *pick_variant(wf_ctx *ctx, const wf_tile *tile, const wf_job *jobs, int64_t njobs,
                                     int64_t max_rows, int64_t total_cells, bool tuned)
{
    int E = WF_ENGINE_LOCKSTEP, R = 0, W = 0, K = 0;
    if (const char *env = std::getenv("WFDP_VARIANT")) {
        if (std::sscanf(env, "%d,%d,%d,%d", &E, &R, &W, &K) == 4) {
            if (const WfVariant *v = find_variant(E, R, W, K)) return v;
        }
        E = WF_ENGINE_LOCKSTEP;
        R = W = K = 0;
    }
    // A hint tile (the reference's tX, tY) only keeps its flags: the
    // variant is the planner's own choice.
    wf_tile hinted{};
    if (tile && (tile->flags & WF_TILE_HINT)) {
        hinted.flags = tile->flags & ~WF_TILE_HINT;
        tile = &hinted;
    }
    const bool cache = tile && (tile->flags & WF_TILE_CACHE);
    // The tuned table applies only when the caller chose neither a size nor
    // an engine.
    const int32_t engine_flags = WF_TILE_LOCKSTEP | WF_TILE_ASYNC | WF_TILE_BITPAR | WF_TILE_BITPAR_STAGED;
    const bool explicit_tile = tile && (tile->tile_w > 0 || tile->strip_rows > 0 || tile->rows_per_lane > 0 ||
                                        (tile->flags & engine_flags));
    if (tuned && !explicit_tile && !cache && ctx) {
        int p, b, bk, te, tr, tw, tk;
        wf_tune_key(jobs, njobs, &p, &b, &bk);
        if (wf_tune_lookup(ctx->prop.gcnArchName, ctx->prop.multiProcessorCount, p, b, bk, &te, &tr, &tw, &tk)) {
            if (const WfVariant *v = find_variant(te, tr, tw, tk)) return v;
        }
    }
    // LCS and ED pairs with at most 32 symbols go to the bit-parallel engine
    // (32 rows per lane word) unless a cell engine is asked for: its chain of
    // waves down a pair is 32 times shorter and a column step costs 7 (LCS) to
    // 15 (ED) VALU operations for 32 cells.
    const bool cell_flags = tile && (tile->flags & (WF_TILE_LOCKSTEP | WF_TILE_ASYNC | WF_TILE_CACHE));
    const int32_t bp_flags = WF_TILE_BITPAR | WF_TILE_BITPAR_STAGED;
    const bool want_bitpar = (tile && ((tile->flags & bp_flags) || tile->rows_per_lane == 32)) ||
                             (!cell_flags && !(tile && tile->rows_per_lane > 0));
    if (want_bitpar && wf_bitpar_eligible(jobs, njobs)) {
        int Wb = 0, Kb = 64;
        if (tile && tile->strip_rows > 0) Wb = std::max(1, tile->strip_rows / 2048);
        if (tile && tile->tile_w > 0) Kb = tile->tile_w;
        // The staged variant (a mask-staging wave per workgroup) when every
        // 2048-row strip gets a CU of its own; the plain one, which packs
        // more compute waves per CU, for larger launches.
        bool staged;
        if (tile && (tile->flags & WF_TILE_BITPAR_STAGED))
            staged = true;
        else if (tile && (tile->flags & WF_TILE_BITPAR))
            staged = false;
        else {
            int64_t strips = 0;
            for (int64_t i = 0; i < njobs; ++i)
                if (jobs[i].n1 > 0 && jobs[i].n2 > 0) strips += (jobs[i].n2 + 2047) / 2048;
            staged = strips <= (ctx ? ctx->prop.multiProcessorCount : 256);
        }
        // Strip height, measured on ED 65536^2, unsplit: staged, one compute
        // wave (2.30 ms; W = 2 2.46); plain, two waves (3.29 ms; W = 1 3.46,
        // W = 4 3.34; K = 128 3.30).  LCS 8192^2: 0.162 (0.249); 0.297 (0.345,
        // 0.331; 0.299).
        if (Wb == 0) Wb = staged ? 1 : (max_rows > 2048 ? 2 : 1);
        const int Eb = staged ? WF_ENGINE_BITPAR_STAGED : WF_ENGINE_BITPAR;
        const WfVariant *best = nullptr;
        int best_d = 1 << 30;
        for (int i = 0; i < wf_num_variants_bitpar; ++i) {
            const WfVariant &v = wf_variants_bitpar[i];
            if (v.engine != Eb) continue;
            const int d = std::abs(v.waves - Wb) * 1000 + std::abs(v.chunk - Kb);
            if (d < best_d) {
                best_d = d;
                best = &v;
            }
        }
        return best;
    }
    if (tile && (tile->flags & bp_flags)) return nullptr;  // asked for, not possible
    // Default engine: a launch whose strips all fit on the chip at once is
    // bound by the wavefront's critical path, where the asynchronous engine's
    // shorter lag between waves and strips wins; a launch with many more
    // strips than CUs is bound by throughput, where the lock-step engine's
    // higher occupancy wins (measured on MI355X: SW 131072^2 and ED 65536^2
    // against the 4096-pair batch).
    // The async engine's counter group G trades per-step cost (a check, a
    // branch that ends the compiler's scheduling region, per group) against
    // the lag a wave adds to the chain (64 + G steps): G = 32 measured best
    // on both single pairs (SW 131072^2: G = 8 / 16 / 32 8.43 / 7.88 /
    // 7.80 ms; ED 65536^2 on this engine: 3.77 / 3.39 / 3.26 ms).
    const int async_k = 32;
    {
        int64_t strips = 0;
        for (int64_t i = 0; i < njobs; ++i)
            if (jobs[i].n1 > 0 && jobs[i].n2 > 0) strips += (jobs[i].n2 + 511) / 512;
        const int cus = ctx ? ctx->prop.multiProcessorCount : 256;
        if (strips <= 2LL * cus) E = WF_ENGINE_ASYNC;
    }
    if (tile && (tile->flags & WF_TILE_ASYNC)) E = WF_ENGINE_ASYNC;
    if (tile && (tile->flags & WF_TILE_LOCKSTEP)) E = WF_ENGINE_LOCKSTEP;
    if (cache) E = WF_ENGINE_ASYNC;
    if (tile && tile->rows_per_lane > 0) R = tile->rows_per_lane;
    if (tile && tile->tile_w > 0) K = tile->tile_w;
    if (tile && tile->strip_rows > 0) {
        const int rows = tile->strip_rows;
        if (cache) W = 1;
        if (R == 0 && W == 0) {
            // Prefer 4 waves (one per SIMD), then fewer rows per lane.
            if (rows >= 256) {
                W = 4;
                R = std::max(1, std::min(4, rows / 256));
            } else if (rows >= 128) {
                W = 2;
                R = 1;
            } else {
                W = 1;
                R = 1;
            }
        } else if (W == 0) {
            W = std::max(1, rows / (64 * R));
        } else if (R == 0) {
            R = std::max(1, rows / (64 * W));
        }
    }
    if (W == 0) W = cache ? 1 : wf_default_waves(max_rows, total_cells, (int)njobs);
    if (R == 0) R = wf_default_rows_per_lane(W, max_rows, total_cells, (int)njobs);
    if (K == 0) K = (E == WF_ENGINE_LOCKSTEP) ? 64 : async_k;
    // Snap to the nearest compiled variant of the requested engine.
    const WfVariant *best = nullptr;
    int best_d = 1 << 30;
    for (int i = 0; i < variant_count(); ++i) {
        const WfVariant &v = *variant_at(i);
        if (v.engine != E) continue;
        const int d = std::abs(v.waves - W) * 1000 + std::abs(v.rows_per_lane - R) * 10 +
                      std::abs(v.chunk - K) / 8;
        if (d < best_d) {
            best_d = d;
            best = &v;
        }
    }
    return best;
}

// Built-in defaults (measured on MI355X: SW 2^17 single pair, ED 2^16, the
// 4096-pair batch): strips of 512 rows = 4 waves x 2 rows per lane; smaller
// strips for pairs too short to fill four waves.
int wf_default_waves(int64_t max_rows, int64_t total_cells, int npairs)
{
    (void)total_cells;
    (void)npairs;
    if (max_rows >= 512) return 4;
    if (max_rows >= 256) return 2;
    return 1;
}

int wf_default_rows_per_lane(int waves, int64_t max_rows, int64_t total_cells, int npairs)
{
    (void)total_cells;
    (void)npairs;
    if (max_rows >= 64LL * waves * 2) return 2;
    return 1;
}

// ----------------------------------------------------------------------------
// Planning
// ----------------------------------------------------------------------------

// Column split of bit-parallel pairs (WfSplitDev): on unless WFDP_SPLIT=0.
static bool split_enabled()
{
    const char *e = std::getenv("WFDP_SPLIT");
    return !(e && e[0] == '0');
}
// Byte row tables for SW pairs of at most 4 symbols (WFK_MODE_PERM4): on
// unless WFDP_PERM=0 (wf_perm4_enabled).
// Bit-parallel pairs narrower than this are not split: half the steps have to
// pay for the combine launch (us a call, split / unsplit: ED 512^2 53 / 53, 640^2 55
// / 58, 800^2 60 / 65, 1000^2 62 / 71; LCS, whose steps are shorter, 640^2 47 / 46,
// 800^2 50 / 50, 1000^2 52 / 54).
constexpr int64_t kSplitMinColsEd = 576, kSplitMinColsLcs = 832;
// SW pairs narrower than this are not split (measured gains of the split:
// 13% at 1024 x 1024, 17% at 2048 x 2048, 30% at 3000 x 600).
constexpr int64_t kSwSplitMinCols = 1024;
// Narrowest pair that is split in two or three parts (without f0, WfSplitDev)
// where three or four have more strips than the chip has CUs.  With the maximum
// the line does not lie where the gain ends: three parts halve the time of narrower
// pairs too (ms in one part / three: 1024 x 65 strips 1.01 / 0.53, 10000 x 90
// 1.72 / 0.90, 16384 x 130 2.38 / 1.25), which stay in one part, as test_sw_split_*
// has it.  Without it (ms in three parts / two) two are the better ones from
// about 65536 columns on and within 4% below: 128 strips, 16384 columns 1.13 / 1.14,
// 65536 1.73 / 1.77, 98304 2.27 / 2.20, 131072 2.98 / 2.60; 170 strips, 16384
// columns 1.38 / 1.43, 49152 1.81 / 1.86, 65536 2.23 / 2.07, 98304 3.46 / 2.60.
// Narrower ones of more strips than three parts have room for stay in one part
// too (2000 x 180 strips 2.84 ms, in two 1.50).
constexpr int64_t kSwTwoPartMinCols = 16384;

// Columns where the strips of a column-split SW pair are cut (WfSplitDev):
// strip g sweeps columns 1..c[g] forward and, reversed, the rest.  A strip
// starts a lag after the strip above it (the strip below, reversed), so with
// c falling by the lag from strip to strip both sweeps' strips all end at step
// (n1 + (G - 1) lag) / 2, against n1 / 2 + (G - 1) lag with a straight cut.  The
// lag of a 512-row strip is 13.2 us, 580 steps of 22.7 ns (16384 columns, 512 to
// 32768 rows, unsplit); 640 steps gave the shortest runs at every size (lags of
// 0 / 432 / 580 / 640 / 704: 8192^2 0.323 / 0.286 / 0.252 / 0.239 / 0.239 ms,
// 32768^2 1.26 / 1.09 / 0.945 / 0.890 / 0.914 ms; with the maximum likewise).
static std::vector<int32_t> sw_cuts(int64_t n1, int64_t n2, int64_t strip, int waves)
{
    const int64_t G = (n2 + strip - 1) / strip, lag = 160 * waves;
    std::vector<int32_t> c((size_t)G);
    for (int64_t g = 0; g < G; ++g)
        c[g] = (int32_t)std::min(n1, std::max<int64_t>(0, (n1 + (G - 1) * lag) / 2 - g * lag));
    return c;
}

// The same for LCS and ED on the staged bit-parallel engine (2048-row strips),
// with a smaller lag where the pair is too narrow for it, so that every strip
// keeps columns on both sides.  Lags of 0 / 160 / 176 / 192 / 208 / 256 steps:
// ED 65536^2 1.274 / 1.198 / 1.192 / 1.194 / 1.201 / 1.219 ms, LCS 32768^2 0.360 /
// 0.342 / 0.340 / 0.338 / 0.337 / 0.341, ED 20000 x 60000 0.547 / 0.455 / 0.448 /
// 0.449 / 0.456 / 0.474.
static std::vector<int32_t> bitpar_cuts(int64_t n1, int64_t n2, int64_t strip)
{
    const int64_t G = (n2 + strip - 1) / strip;
    const int64_t lag = G > 1 ? std::min<int64_t>(192, (n1 - 64) / (G - 1)) : 0;
    std::vector<int32_t> c((size_t)G);
    for (int64_t g = 0; g < G; ++g) c[g] = (int32_t)((n1 + (G - 1) * lag) / 2 - g * lag);
    return c;
}

static int build_plan(wf_ctx *ctx, const wf_job *jobs, int64_t njobs, const wf_tile *tile, WfPlanHost *ph,
                      int64_t max_groups, bool tuned)
{
    int64_t max_rows = 0, total_cells = 0;
    for (int64_t i = 0; i < njobs; ++i) {
        const wf_job &j = jobs[i];
        if (j.problem < WF_LCS || j.problem > WF_SW) return WF_ERR_INVALID;
        if (j.n1 < 0 || j.n2 < 0 || j.n1 > (1LL << 30) || j.n2 > (1LL << 30)) return WF_ERR_INVALID;
        if ((j.n1 > 0 && !j.a) || (j.n2 > 0 && !j.b)) return WF_ERR_INVALID;
        if (j.n1 > 0 && j.n2 > 0) max_rows = std::max(max_rows, j.n2);
        total_cells += j.n1 * j.n2;
    }
    const WfVariant *v = pick_variant(ctx, tile, jobs, njobs, max_rows, total_cells, tuned);
    if (!v) return WF_ERR_NOKERNEL;
    ph->variant = v;
    const int64_t strip = 64LL * v->waves * v->rows_per_lane;
    const bool bitpar = v->engine == WF_ENGINE_BITPAR || v->engine == WF_ENGINE_BITPAR_STAGED;
    const bool perm4 = (v->engine == WF_ENGINE_ASYNC || v->engine == WF_ENGINE_LOCKSTEP) && v->rows_per_lane == 2 &&
                       wf_perm4_enabled();

    // Bit-parallel pairs are split into two column halves computed at once
    // (WfSplitDev) when the launch has room for twice its strips: a single
    // pair's time is its column count times the step time, so the halves
    // finish in about half of it.
    std::vector<int64_t> mid(njobs, 0);
    std::vector<uint8_t> swsplit(njobs, 0);
    bool two_part = false;  // SW splits without the part `f0` (WfSplitDev)
    std::vector<std::vector<uint8_t>> trial;  // SW split candidates' codes (a then b) and modes
    std::vector<int32_t> trial_mode;
    int64_t nextra = 0;
    if (bitpar && split_enabled()) {
        int64_t strips = 0;
        for (int64_t i = 0; i < njobs; ++i)
            if (jobs[i].n1 > 0 && jobs[i].n2 > 0) strips += (jobs[i].n2 + strip - 1) / strip;
        const int64_t cus = ctx ? ctx->prop.multiProcessorCount : 256;
        if (2 * strips <= std::min(cus, max_groups > 0 ? max_groups : INT64_MAX))
            for (int64_t i = 0; i < njobs; ++i)
                if (jobs[i].n1 >= (jobs[i].problem == WF_ED ? kSplitMinColsEd : kSplitMinColsLcs) && jobs[i].n2 > 0) {
                    mid[i] = jobs[i].n1 / 2;
                    ++nextra;
                }
    } else if (v->engine == WF_ENGINE_ASYNC && perm4 && split_enabled()) {
        // SW pairs split in three (bottom-right cell only) or four (with the
        // running maximum) pairs (WfSplitDev) when all of the launch's strips
        // fit on the chip at once: the parts' strip chains run side by side.
        int64_t strips = 0, extra = 0;
        std::vector<uint8_t> cand(njobs, 0);
        trial.resize(njobs);
        trial_mode.assign(njobs, 0);
        for (int64_t i = 0; i < njobs; ++i) {
            const wf_job &j = jobs[i];
            if (j.n1 <= 0 || j.n2 <= 0) continue;
            const int64_t si = (j.n2 + strip - 1) / strip;
            strips += si;
            if (j.problem != WF_SW || j.n1 < kSwSplitMinCols) continue;
            const bool nomax = ((j.flags | (tile ? tile->flags : 0)) & WF_TILE_NO_MAX) != 0;
            // The trial encoding is kept for the plan's codes below.
            std::vector<uint8_t> t((size_t)(j.n1 + j.n2));
            int32_t mode = 0;
            if (wf_encode_job(j, tile ? tile->flags : 0, perm4, t.data(), t.data() + j.n1, &mode) != WF_OK) continue;
            trial[i] = std::move(t);
            trial_mode[i] = mode;
            // Compared codes (7013 x 3001, 20 symbols: 391 us a call unsplit, 246
            // split): only on the kernels of G = 32 (the planner's own
            // choice).  Pairs of 5 to 8 symbols change over to them for the
            // four parts with the maximum; without it they stay in one part on
            // the 4-bit row tables, which have no running maximum to carry.
            // Pairs of more than 8 symbols keep the maximum whether asked to
            // or not.
            if (!(mode & WFK_MODE_PERM4) && (v->chunk != 32 || (nomax && !(mode & WFK_MODE_CMP)))) continue;
            cand[i] = nomax && !(mode & WFK_MODE_CMP) ? 2 : 3;  // extra pairs
            extra += cand[i] * si;
        }
        // Three or four parts while every strip has a CU of its own.  Beyond
        // that, a launch of one wide pair takes two or three parts, whose
        // strips share CUs only towards the end (no maximum: 131072 x 65536
        // 2.60 ms against 2.98 in three parts and 4.47 with a straight cut;
        // 131072^2 4.74 against 6.55 unsplit; with it: 65536^2 2.02 against
        // 3.62 unsplit), and a narrow one without the maximum three parts
        // (4096 x 44032, 258 strips: 0.66 ms, unsplit 1.24).  A batch, whose
        // strips all run at once, is not split beyond a strip per CU (16 pairs
        // of 4096^2, 384 strips: 0.27 ms against 0.21 unsplit).
        const bool four = std::find(cand.begin(), cand.end(), 3) != cand.end();
        const int64_t cus = ctx ? ctx->prop.multiProcessorCount : 256;
        const int64_t resident = std::min(ctx ? (int64_t)wf_max_resident_groups(ctx, v) : 256,
                                          max_groups > 0 ? max_groups : INT64_MAX);
        const bool wide = njobs == 1 && cand[0] && jobs[0].n1 >= kSwTwoPartMinCols;
        if (extra > 0 && strips + extra <= std::min(resident, (four || njobs > 1 || wide) ? cus : INT64_MAX)) {
            for (int64_t i = 0; i < njobs; ++i)
                if (cand[i]) {
                    swsplit[i] = cand[i];
                    nextra += cand[i];
                }
        } else if (wide && cand[0] * strips <= resident) {
            swsplit[0] = cand[0];
            two_part = true;
            nextra = cand[0] - 1;
        }
    }
    const int64_t np = njobs + nextra;
    ph->njobs = njobs;
    ph->npairs = np;
    ph->pairs.assign(np, WfPairDev{});
    ph->host_result.assign(np, 0);
    ph->host_only.assign(np, 0);
    ph->cells.assign(np, 0);
    ph->splits.clear();
    ph->cuts.clear();
    ph->colw_entries = 0;
    for (int64_t i = 0; i < njobs; ++i) ph->cells[i] = (uint64_t)(jobs[i].n1 * jobs[i].n2);

    // Codes: a then b per pair, 16-byte aligned; a split pair's reverse half
    // gets its own reversed copies after all jobs.
    int64_t code_bytes = 0, bnd_ints = 0;
    // Bit-parallel halves that meet along a staircase: pairs of several strips
    // (one strip has no lag to share out, and its call of 1531 x 1187 took 73 us
    // with the cut's descriptors against 70 without).
    auto stairs = [&](int64_t i) {
        return mid[i] && v->engine == WF_ENGINE_BITPAR_STAGED && v->waves == 1 && jobs[i].n2 > strip;
    };
    auto place_codes = [&](WfPairDev &p, int prob, int64_t n1, int64_t n2, int64_t a_bytes) {
        p.prob = prob;
        p.n1 = (int32_t)n1;
        p.n2 = (int32_t)n2;
        p.a_off = code_bytes;
        code_bytes += (a_bytes + 15) & ~15LL;
        p.b_off = code_bytes;
        code_bytes += (n2 + 15) & ~15LL;
        p.ngroups = (int32_t)((n2 + strip - 1) / strip);
    };
    auto place = [&](WfPairDev &p, int prob, int64_t n1, int64_t n2, int64_t a_bytes) {
        place_codes(p, prob, n1, n2, a_bytes);
        p.bnd_off = bnd_ints;
        // One word per column, or (bs_row_words in wf_bitpar.hip) 4 per 64 steps.
        bnd_ints += (int64_t)(p.ngroups - 1) * (v->engine == WF_ENGINE_BITPAR_STAGED ? 4 * ((n1 + 126) / 64) : n1);
    };
    for (int64_t i = 0; i < njobs; ++i) {
        const wf_job &j = jobs[i];
        WfPairDev &p = ph->pairs[i];
        if (j.n1 == 0 || j.n2 == 0) {
            p.prob = j.problem;
            p.n1 = (int32_t)j.n1;
            p.n2 = (int32_t)j.n2;
            p.a_off = code_bytes;
            code_bytes += (j.n1 + 15) & ~15LL;
            p.b_off = code_bytes;
            code_bytes += (j.n2 + 15) & ~15LL;
            ph->host_only[i] = 1;
            ph->host_result[i] = wf_empty_score(j.problem, j.n1, j.n2, j.flags);
            p.ngroups = 0;
            continue;
        }
        if (swsplit[i] || stairs(i))
            place_codes(p, j.problem, j.n1, j.n2, j.n1);
        else
            place(p, j.problem, mid[i] ? mid[i] : j.n1, j.n2, j.n1);
    }
    {
        int64_t r = njobs;
        for (int64_t i = 0; i < njobs; ++i) {
            if (!mid[i] && !swsplit[i]) continue;
            const wf_job &j = jobs[i];
            if (swsplit[i]) {
                // Right part from a zero boundary (pair r), reversed right
                // part (pair r + 1) and, with the running maximum, the
                // clamped reversed right part (pair r + 2); the left and the
                // reversed parts keep their last columns.
                const std::vector<int32_t> c = sw_cuts(j.n1, j.n2, strip, v->waves);
                const int64_t G = (int64_t)c.size(), pad = G * strip - j.n2;
                const int32_t base = c.back(), n1 = (int32_t)j.n1;
                const int64_t ir = r + (two_part ? 0 : 1);  // the reversed part's pair
                WfPairDev &f = ph->pairs[i], &rv = ph->pairs[ir];
                f.n1 = c[0];
                place_codes(rv, WFK_SW, n1 - base, G * strip, n1 - base);
                WfSplitDev sp{};
                sp.job = (int32_t)i;
                sp.rev = (int32_t)ir;
                sp.prob = WFK_SW;
                sp.n2 = (int32_t)j.n2;
                sp.f0 = two_part ? -1 : (int32_t)r;
                sp.r0 = n1;
                sp.strip = (int32_t)strip;
                sp.pad = (int32_t)pad;
                auto cut_pair = [&](WfPairDev &p, auto &&of) {
                    p.cut = (int32_t)ph->cuts.size();
                    for (int64_t g = 0; g < G; ++g) {
                        WfCutDev cd = of(g);
                        cd.bnd = bnd_ints;
                        if (g + 1 < G) bnd_ints += cd.n;
                        ph->cuts.push_back(cd);
                    }
                };
                auto keep_columns = [&](WfPairDev &p, int64_t rows) {
                    const int64_t at = ph->colw_entries;
                    p.col_off = at;
                    ph->colw_entries += (rows + 1) / 2;  // two words per entry, one per row
                    return at;
                };
                cut_pair(f, [&](int64_t g) { return WfCutDev{0, 0, c[g], 0, 0, 0, 0}; });
                if (!two_part) {
                    WfPairDev &p0 = ph->pairs[r];
                    p0.prob = WFK_SW;
                    p0.n1 = n1 - base;
                    p0.n2 = (int32_t)j.n2;
                    p0.a_off = f.a_off + base;
                    p0.b_off = f.b_off;
                    p0.ngroups = f.ngroups;
                    cut_pair(p0, [&](int64_t g) {
                        return WfCutDev{0, c[g] - base, n1 - c[g], g ? c[g - 1] - base : 0, 0, 0, 0};
                    });
                }
                // Strip k of the reversed parts is strip G - 1 - k; the first
                // one is filled up with rows without a symbol.
                auto reversed = [&](int64_t k) {
                    return WfCutDev{0, 0, n1 - c[G - 1 - k], 0,
                                    k == 0 ? (int32_t)(pad / (64 * v->rows_per_lane)) : 0, (int32_t)pad, 0};
                };
                cut_pair(rv, reversed);
                sp.cut = f.cut;
                sp.rcut = rv.cut;
                sp.fwd_off = keep_columns(f, j.n2);
                sp.rev_off = keep_columns(rv, G * strip);
                if (swsplit[i] == 3) {
                    WfPairDev &cv = ph->pairs[ir + 1];
                    cv = rv;
                    sp.crev = (int32_t)(ir + 1);
                    cut_pair(cv, reversed);
                    sp.ccut = cv.cut;
                    sp.crev_off = keep_columns(cv, G * strip);
                }
                ph->splits.push_back(sp);
                r += swsplit[i] - (two_part ? 1 : 0);
                continue;
            }
            WfSplitDev sp{};
            sp.job = (int32_t)i;
            sp.rev = (int32_t)r;
            sp.prob = j.problem;
            sp.n2 = (int32_t)j.n2;
            if (stairs(i)) {
                // (f0 and r0, the ends of the staircase, below.)
                const std::vector<int32_t> c = bitpar_cuts(j.n1, j.n2, strip);
                const int64_t G = (int64_t)c.size(), pad = G * strip - j.n2;
                const int32_t n1 = (int32_t)j.n1;
                WfPairDev &f = ph->pairs[i], &rv = ph->pairs[r];
                f.n1 = c[0];
                mid[i] = c.back();
                place_codes(rv, j.problem, n1 - c.back(), G * strip, n1 - c.back());
                auto cut_pair = [&](WfPairDev &p, auto &&of) {
                    p.cut = (int32_t)ph->cuts.size();
                    for (int64_t g = 0; g < G; ++g) {
                        WfCutDev cd = of(g);
                        cd.bnd = bnd_ints;
                        if (g + 1 < G) bnd_ints += 4 * ((cd.n + 126) / 64);  // bs_row_words in wf_bitpar.hip
                        ph->cuts.push_back(cd);
                    }
                    return p.cut;
                };
                sp.cut = cut_pair(f, [&](int64_t g) { return WfCutDev{0, 0, c[g], 0, 0, 0, 0}; });
                sp.rcut = cut_pair(rv, [&](int64_t k) {
                    return WfCutDev{0, 0, n1 - c[G - 1 - k], 0, 0, (int32_t)pad, 0};
                });
                sp.strip = (int32_t)strip;
                sp.pad = (int32_t)pad;
                sp.cols = n1;
            } else {
                place(ph->pairs[r], j.problem, j.n1 - mid[i], j.n2, j.n1 - mid[i]);
            }
            ph->pairs[i].col_off = ph->colw_entries;
            sp.fwd_off = ph->colw_entries;
            ph->colw_entries += (int64_t)ph->pairs[i].ngroups * v->waves * 64;
            ph->pairs[r].col_off = ph->colw_entries;
            sp.rev_off = ph->colw_entries;
            ph->colw_entries += (int64_t)ph->pairs[r].ngroups * v->waves * 64;
            ph->splits.push_back(sp);
            ++r;
        }
    }
    ph->codes.assign((size_t)std::max<int64_t>(code_bytes, 16), 0);
    for (int64_t i = 0; i < njobs; ++i) {
        const wf_job &j = jobs[i];
        WfPairDev &p = ph->pairs[i];
        int32_t mode = 0;
        if (i < (int64_t)trial.size() && !trial[i].empty()) {
            std::memcpy(ph->codes.data() + p.a_off, trial[i].data(), (size_t)j.n1);
            std::memcpy(ph->codes.data() + p.b_off, trial[i].data() + j.n1, (size_t)j.n2);
            mode = trial_mode[i];
        } else {
            const int st = wf_encode_job(j, tile ? tile->flags : 0, perm4, ph->codes.data() + p.a_off,
                                         ph->codes.data() + p.b_off, &mode);
            if (st != WF_OK) return st;
        }
        // SW pairs on the row tables may skip the running maximum (the cell
        // engines have instances without it).
        if (j.problem == WF_SW && !(mode & WFK_MODE_CMP) && ((j.flags | (tile ? tile->flags : 0)) & WF_TILE_NO_MAX))
            mode |= WFK_MODE_NOMAX;
        // The parts of a split pair take the byte tables or compare codes:
        // 5 to 8 symbols leave the 4-bit fields' bit offsets.
        if (swsplit[i] && !(mode & (WFK_MODE_PERM4 | WFK_MODE_CMP))) {
            shr2(ph->codes.data() + p.a_off, j.n1);
            shr2(ph->codes.data() + p.b_off, j.n2);
            mode = WFK_MODE_CMP | WFK_MODE_FREE_HEAD | (0x1FF << WFK_MODE_NEVER_SHIFT);
        }
        p.mode = mode;
        // The bit-parallel kernel indexes a 32-row table with the codes.
        if (bitpar && (j.problem == WF_SW || (mode & WFK_MODE_CMP))) return WF_ERR_NOKERNEL;
    }
    for (WfSplitDev &sp : ph->splits) {
        if (sp.prob == WFK_SW) {
            // Reversed parts: the right part of a and b reversed, b behind
            // its rows without a symbol; the unclamped recurrence, and the
            // clamped one for the running maximum.
            const wf_job &j = jobs[sp.job];
            const WfPairDev &f = ph->pairs[sp.job];
            WfPairDev &rv = ph->pairs[sp.rev];
            if (!(f.mode & (WFK_MODE_PERM4 | WFK_MODE_CMP)) || !(f.mode & WFK_MODE_NOMAX) != (sp.crev >= 0))
                return WF_ERR_INVALID;
            uint8_t *codes = ph->codes.data();
            reverse_codes(codes + f.a_off + (j.n1 - rv.n1), rv.n1, codes + rv.a_off);
            // (Compared codes: the engine goes by WfCutDev::pad.)
            std::memset(codes + rv.b_off, WFK_NO_SYMBOL, (size_t)sp.pad);
            reverse_codes(codes + f.b_off, j.n2, codes + rv.b_off + sp.pad);
            const int32_t mode = (f.mode & ~WFK_MODE_NOMAX) | (two_part ? 0 : WFK_MODE_NOMAX);
            if (sp.f0 >= 0) ph->pairs[sp.f0].mode = f.mode;
            rv.mode = mode | WFK_MODE_SWE;
            if (sp.crev >= 0) ph->pairs[sp.crev].mode = mode;
            continue;
        }
        // Reverse half: a[mid..n1) and b reversed, textbook ED boundary (its
        // row 0 is a plain distance from the empty prefix).
        const wf_job &j = jobs[sp.job];
        const WfPairDev &f = ph->pairs[sp.job];
        WfPairDev &r = ph->pairs[sp.rev];
        const int64_t m = mid[sp.job], nr = j.n1 - m;
        const uint8_t *fa = ph->codes.data() + f.a_off;
        const uint8_t *fb = ph->codes.data() + f.b_off;
        uint8_t *ra = ph->codes.data() + r.a_off;
        uint8_t *rb = ph->codes.data() + r.b_off;
        reverse_codes(fa + m, nr, ra);
        std::memset(rb, 0, (size_t)sp.pad);  // rows without a symbol: the engine goes by WfCutDev::pad
        reverse_codes(fb, j.n2, rb + sp.pad);
        r.mode = (f.mode & ~WFK_MODE_TEXTBOOK) | (j.problem == WF_ED ? WFK_MODE_TEXTBOOK : 0);
        if (j.problem == WF_ED) {
            // Row 0 at column mid (the staircase's first column).
            sp.f0 = (f.mode & WFK_MODE_TEXTBOOK) ? f.n1 : f.n1 - 1;
            sp.r0 = (int32_t)nr;
        }
    }

    // Tasks: pairs with the longest dependency chain first (columns plus the
    // start-up lag of every strip), then by size; the strips of a pair stay
    // contiguous and in order, which is what makes the persistent claim loop
    // deadlock-free.  The longest chains also get the highest wave issue
    // priority, so that co-resident strips of short pairs fill the issue
    // slots they leave idle instead of stretching the critical path.
    std::vector<int64_t> chain(np, 0);
    int64_t max_chain = 1;
    const int64_t strip_lag = (int64_t)v->waves * (64 + 2 * v->chunk);
    for (int64_t i = 0; i < np; ++i) {
        const WfPairDev &p = ph->pairs[i];
        if (p.ngroups == 0) continue;
        chain[i] = p.n1 + 63 + (int64_t)p.ngroups * strip_lag;
        max_chain = std::max(max_chain, chain[i]);
    }
    static const bool use_prio = [] {
        const char *e = std::getenv("WFDP_PRIORITY");
        return !(e && e[0] == '0');
    }();
    for (int64_t i = 0; i < np; ++i)
        ph->pairs[i].prio = use_prio ? (int32_t)std::min<int64_t>(3, 4 * chain[i] / (max_chain + 1)) : 0;
    std::vector<int64_t> order(np);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int64_t x, int64_t y) {
        if (chain[x] != chain[y]) return chain[x] > chain[y];
        return ph->cells[x] > ph->cells[y];
    });
    ph->tasks.clear();
    ph->task_begin.assign(np, 0);
    ph->task_end.assign(np, 0);
    // The parts of a split pair are one entry of the list, so that a launch per
    // pair (WF_RUN_PER_PAIR) runs them side by side too (SW 7013 x 3001, 20
    // symbols: 200 us, 700 in a launch per part, unsplit 333).  Those of a two-part
    // split go strip by strip:
    // the early strips of all parts, which run from the start, are then claimed
    // by the first workgroup of each CU and the late ones by the second (SW
    // 131072^2, 512 strips: 4.74 ms, part by part 5.88).  The other splits' go
    // part by part: their f0 strips all start at once (65536^2, 384 strips:
    // 1.74 ms part by part, 2.94 strip by strip).
    std::vector<int32_t> split_of(ph->splits.empty() ? 0 : np, -1);  // -2: in the list with the part that came first
    for (size_t k = 0; k < ph->splits.size(); ++k) {
        const WfSplitDev &sp = ph->splits[k];
        for (int32_t p : {sp.job, sp.prob == WFK_SW ? sp.f0 : -1, sp.rev, sp.crev})
            if (p >= 0) split_of[p] = (int32_t)k;
    }
    for (int64_t k = 0; k < np; ++k) {
        int64_t i = order[k];
        int32_t part[4] = {(int32_t)i};
        int parts = 1;
        if (!split_of.empty() && split_of[i] != -1) {
            if (split_of[i] == -2) continue;
            const WfSplitDev &sp = ph->splits[split_of[i]];
            parts = 0;
            for (int32_t p : {sp.job, sp.prob == WFK_SW ? sp.f0 : -1, sp.rev, sp.crev})
                if (p >= 0) {
                    split_of[p] = -2;
                    part[parts++] = p;
                }
            i = sp.job;
        }
        ph->task_begin[i] = (int64_t)ph->tasks.size();
        const int32_t ng = ph->pairs[i].ngroups;  // (the same in all parts)
        if (two_part) {
            for (int32_t g = 0; g < ng; ++g)
                for (int p = 0; p < parts; ++p) ph->tasks.push_back(WfTaskDev{part[p], g});
        } else {
            for (int p = 0; p < parts; ++p)
                for (int32_t g = 0; g < ng; ++g) ph->tasks.push_back(WfTaskDev{part[p], g});
        }
        ph->task_end[i] = (int64_t)ph->tasks.size();
    }
    ph->bnd_ints = bnd_ints;
    ph->order = order;
    return WF_OK;
}

// The tuned table knows a pair's size, not its symbols: LCS and ED pairs of more
// than 32, which its bit-parallel variants cannot run, take the built-in choice.
int wf_build_plan(wf_ctx *ctx, const wf_job *jobs, int64_t njobs, const wf_tile *tile, WfPlanHost *ph,
                  int64_t max_groups)
{
    const int st = build_plan(ctx, jobs, njobs, tile, ph, max_groups, true);
    if (st != WF_ERR_NOKERNEL) return st;
    *ph = WfPlanHost();
    return build_plan(ctx, jobs, njobs, tile, ph, max_groups, false);
}

int wf_upload_plan(wf_ctx *ctx, WfPlanHost *ph, WfArenas *ar)
{
    return wf_upload_plan_async(ctx, ph, ar, ctx->stream, true);
}

void wf_plan_bytes(const WfPlanHost *ph, WfPlanBytes *b)
{
    b->codes = ph->codes.size();
    b->pairs = std::max<size_t>(1, ph->pairs.size()) * sizeof(WfPairDev);
    b->tasks = std::max<size_t>(1, ph->tasks.size()) * sizeof(WfTaskDev);
    b->bnd = (size_t)std::max<int64_t>(1, ph->bnd_ints) * sizeof(uint64_t);
    b->res = (size_t)std::max<int64_t>(1, ph->npairs) * sizeof(WfResultDev);
    b->counters = (size_t)(ph->npairs + 1) * sizeof(int32_t);
    b->epoch = sizeof(uint32_t);
    b->colw = (size_t)std::max<int64_t>(1, ph->colw_entries) * 2 * sizeof(uint32_t);
    b->splits = std::max<size_t>(sizeof(WfSplitDev), wf_cuts_offset(ph) + ph->cuts.size() * sizeof(WfCutDev));
}

int wf_copy_plan(WfPlanHost *ph, WfArenas *ar, hipStream_t stream)
{
    const size_t ntasks = ph->tasks.size();
    if (hipMemcpyAsync(ar->codes.ptr, ph->codes.data(), ph->codes.size(), hipMemcpyHostToDevice,
                       stream) != hipSuccess)
        return WF_ERR_DEVICE;
    // Splits and cuts in one copy (a copy is about 8 us of a request's latency).
    if (!ph->splits.empty()) {
        const size_t at = wf_cuts_offset(ph), cuts = ph->cuts.size() * sizeof(WfCutDev);
        ph->split_block.assign(at + cuts, 0);
        std::memcpy(ph->split_block.data(), ph->splits.data(), ph->splits.size() * sizeof(WfSplitDev));
        if (cuts) std::memcpy(ph->split_block.data() + at, ph->cuts.data(), cuts);
        if (hipMemcpyAsync(ar->splits.ptr, ph->split_block.data(), at + cuts, hipMemcpyHostToDevice, stream) !=
            hipSuccess)
            return WF_ERR_DEVICE;
    }
    if (!ph->pairs.empty() &&
        hipMemcpyAsync(ar->pairs.ptr, ph->pairs.data(), ph->pairs.size() * sizeof(WfPairDev),
                       hipMemcpyHostToDevice, stream) != hipSuccess)
        return WF_ERR_DEVICE;
    if (ntasks &&
        hipMemcpyAsync(ar->tasks.ptr, ph->tasks.data(), ntasks * sizeof(WfTaskDev),
                       hipMemcpyHostToDevice, stream) != hipSuccess)
        return WF_ERR_DEVICE;
    return WF_OK;
}

// Sizes every device buffer of the plan (growing them as needed).
static int ensure_arenas(WfPlanHost *ph, WfArenas *ar, hipStream_t stream)
{
    WfPlanBytes nb;
    wf_plan_bytes(ph, &nb);
    int st;
    if ((st = ar->codes.ensure(nb.codes, false, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->pairs.ensure(nb.pairs, false, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->tasks.ensure(nb.tasks, false, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->bnd.ensure(nb.bnd, true, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->res.ensure(nb.res, false, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->counters.ensure(nb.counters, false, stream, ar->retired)) != WF_OK) return st;
    // Launch epoch: zero on allocation, so it never matches a zeroed boundary word.
    if ((st = ar->epoch.ensure(nb.epoch, true, stream, ar->retired)) != WF_OK) return st;
    if ((st = ar->colw.ensure(nb.colw, false, stream, ar->retired)) != WF_OK) return st;
    return ar->splits.ensure(nb.splits, false, stream, ar->retired);
}

int wf_upload_plan_async(wf_ctx *ctx, WfPlanHost *ph, WfArenas *ar, hipStream_t stream, bool sync)
{
    (void)ctx;
    int st;
    if ((st = ensure_arenas(ph, ar, stream)) != WF_OK) return st;
    if ((st = wf_copy_plan(ph, ar, stream)) != WF_OK) return st;
    if (sync && hipStreamSynchronize(stream) != hipSuccess) return WF_ERR_DEVICE;
    return WF_OK;
}

static size_t round256(size_t n) { return (n + 255) & ~size_t(255); }

// The context's pinned block, at least `bytes` long and idle (a call that
// failed after queueing its copies may have left them in flight).
int wf_ensure_pinned(wf_ctx *ctx, size_t bytes)
{
    if (ctx->pinned_busy) {
        if (hipStreamSynchronize(ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
        ctx->pinned_busy = false;
    }
    if (ctx->pinned_cap >= bytes) return WF_OK;
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);
    ctx->pinned = nullptr;
    ctx->pinned_cap = 0;
    const size_t cap = std::max<size_t>(round256(bytes), (size_t)1 << 20);
    if (hipHostMalloc((void **)&ctx->pinned, cap, hipHostMallocDefault) != hipSuccess) {
        ctx->pinned = nullptr;
        return WF_ERR_NOMEM;
    }
    ctx->pinned_cap = cap;
    return WF_OK;
}

namespace {

// Byte offsets of a call's buffers in the pinned block and, alike, in the
// device block it is copied to: codes, splits and cuts, pairs, tasks, the
// cleared results and claim counters, the launch epoch.
struct BlockLayout {
    size_t codes = 0, splits = 0, pairs = 0, tasks = 0, res = 0, counters = 0, epoch = 0, end = 0;
    BlockLayout() = default;
    explicit BlockLayout(const WfPlanHost *ph)
    {
        WfPlanBytes nb;
        wf_plan_bytes(ph, &nb);
        splits = round256(ph->codes.size());
        pairs = splits + round256(ph->splits.empty() ? 0 : nb.splits);
        tasks = pairs + round256(nb.pairs);
        res = tasks + round256(nb.tasks);
        counters = res + round256(nb.res);
        epoch = counters + round256(nb.counters);
        end = epoch + 256;
    }
};

// A call's plan to the device in one copy: the plan is laid out in the
// context's pinned block, results and counters cleared and the epoch set, and
// one asynchronous DMA takes the block to its twin in HBM, which `ar` then
// points into (nothing may release or grow those buffers).  Against a copy per
// buffer and a reset kernel a 256-symbol pair's call loses four launches.  The
// stream orders the copy before the launch; the block must not be rewritten
// before the stream has drained (wf_align_batch synchronises before it
// returns).
int upload_block(wf_ctx *ctx, WfPlanHost *ph, const BlockLayout &L, WfArenas *ar)
{
    WfArenas *sc = &ctx->scratch;
    WfPlanBytes nb;
    wf_plan_bytes(ph, &nb);
    int st;
    if ((st = sc->codes.ensure(L.end)) != WF_OK) return st;
    if ((st = sc->bnd.ensure(nb.bnd, true)) != WF_OK) return st;
    if ((st = sc->colw.ensure(nb.colw)) != WF_OK) return st;
    if ((st = wf_ensure_pinned(ctx, L.end)) != WF_OK) return st;
    ctx->pinned_busy = true;
    uint8_t *p = ctx->pinned;
    auto put = [&](size_t off, const void *src, size_t n) {
        if (n) std::memcpy(p + off, src, n);
    };
    put(L.codes, ph->codes.data(), ph->codes.size());
    put(L.splits, ph->splits.data(), ph->splits.size() * sizeof(WfSplitDev));
    put(L.splits + wf_cuts_offset(ph), ph->cuts.data(), ph->cuts.size() * sizeof(WfCutDev));
    put(L.pairs, ph->pairs.data(), ph->pairs.size() * sizeof(WfPairDev));
    put(L.tasks, ph->tasks.data(), ph->tasks.size() * sizeof(WfTaskDev));
    std::memset(p + L.res, 0, L.epoch - L.res);
    // Tags of calls have the top bit set, those of the sweeps and table dumps
    // that share the boundary rows, counted on the device, do not.
    ctx->calls = (ctx->calls + 1) & 0x7fffffffu;
    const uint32_t epoch = 0x80000000u | ctx->calls;
    put(L.epoch, &epoch, sizeof(epoch));
    if (hipMemcpyAsync(sc->codes.ptr, p, L.end, hipMemcpyHostToDevice, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    auto at = [&](size_t off) { return (void *)((uint8_t *)sc->codes.ptr + off); };
    ar->codes.ptr = at(L.codes);
    ar->splits.ptr = at(L.splits);
    ar->pairs.ptr = at(L.pairs);
    ar->tasks.ptr = at(L.tasks);
    ar->res.ptr = at(L.res);
    ar->counters.ptr = at(L.counters);
    ar->epoch.ptr = at(L.epoch);
    ar->bnd = sc->bnd;
    ar->colw = sc->colw;
    return WF_OK;
}

// Plans the jobs and gives the plan device memory in `ar` (`place`); where there
// is not enough for the column splits, which take up to twice the boundary rows,
// plans and places them once more without.
template <class Place>
int plan_and_place(wf_ctx *ctx, const wf_job *jobs, int64_t njobs, const wf_tile *tile, WfPlanHost *ph, WfArenas *ar,
                   Place &&place)
{
    int st = wf_build_plan(ctx, jobs, njobs, tile, ph);
    if (st != WF_OK) return st;
    st = place();
    if (st != WF_ERR_NOMEM || ph->splits.empty()) return st;
    ar->release();
    *ph = WfPlanHost();
    if ((st = wf_build_plan(ctx, jobs, njobs, tile, ph, 1)) != WF_OK) return st;
    return place();
}

}  // namespace

int wf_max_resident_groups(wf_ctx *ctx, const WfVariant *v)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, v->fn, v->block, 0) != hipSuccess ||
        per_cu < 1) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    if (const char *env = std::getenv("WFDP_WG_PER_CU")) {
        const int e = std::atoi(env);
        if (e > 0) per_cu = std::min(per_cu, e);
    }
    return per_cu * ctx->prop.multiProcessorCount;
}

// The engine launch(es) of a plan: one persistent launch, or one per pair.
static int enqueue_engine(WfPlanHost *ph, const WfVariant *v, int lim, int mode, WfKernelArgs ka, WfArenas *ar,
                          hipStream_t stream)
{
    if (mode == WF_RUN_PER_PAIR) {
        for (int64_t k = 0; k < ph->npairs; ++k) {
            const int64_t i = ph->order[k];
            const int64_t tb = ph->task_begin[i], te = ph->task_end[i];
            if (te <= tb) continue;
            ka.counter = (int32_t *)ar->counters.ptr + 1 + i;
            ka.task_begin = (int32_t)tb;
            ka.task_end = (int32_t)te;
            const int grid = (int)std::min<int64_t>(te - tb, lim);
            ph->grid = std::max(ph->grid, grid);
            if (wf_launch_engine(v, grid, &ka, stream) != hipSuccess) return WF_ERR_DEVICE;
        }
        return WF_OK;
    }
    ka.counter = (int32_t *)ar->counters.ptr;
    ka.task_begin = 0;
    ka.task_end = (int32_t)ph->tasks.size();
    ph->grid = (int)std::min<int64_t>((int64_t)ph->tasks.size(), lim);
    if (wf_launch_engine(v, ph->grid, &ka, stream) != hipSuccess) return WF_ERR_DEVICE;
    return WF_OK;
}

// Enqueue the reset kernel and the engine launch(es) of a plan on the
// context stream (also used inside hipGraph capture: no memset nodes, and
// the epoch that tags boundary values is advanced on the device).  `reset`
// false: results, counters and the epoch came with the plan's upload.
int wf_enqueue_plan(wf_ctx *ctx, WfPlanHost *ph, WfArenas *ar, int mode, int maxg, hipStream_t stream, bool reset)
{
    const int64_t ncounters = ph->npairs + 1;
    if (reset && wf_launch_reset((WfResultDev *)ar->res.ptr, ph->npairs, (int32_t *)ar->counters.ptr, ncounters,
                                 (uint32_t *)ar->epoch.ptr, 1, stream) != hipSuccess)
        return WF_ERR_DEVICE;
    WfKernelArgs ka{};
    ka.pairs = (const WfPairDev *)ar->pairs.ptr;
    ka.tasks = (const WfTaskDev *)ar->tasks.ptr;
    ka.codes = (const uint8_t *)ar->codes.ptr;
    ka.bnd = (uint64_t *)ar->bnd.ptr;
    ka.res = (WfResultDev *)ar->res.ptr;
    ka.epoch = (const uint32_t *)ar->epoch.ptr;
    ka.timeout_ticks = (int64_t)(ctx->timeout_s * 1.0e8);
    ka.colw = (uint32_t *)ar->colw.ptr;
    ka.cuts = (const WfCutDev *)((const uint8_t *)ar->splits.ptr + wf_cuts_offset(ph));
    ph->grid = 0;
    if (ph->tasks.empty()) return WF_OK;
    const WfVariant *v = ph->variant;
    const int lim = maxg > 0 ? maxg : wf_max_resident_groups(ctx, v);
    const int st = enqueue_engine(ph, v, lim, mode, ka, ar, stream);
    if (st != WF_OK) return st;
    if (!ph->cuts.empty() && v->engine == WF_ENGINE_ASYNC) {
        // About 8192 nodes of the cut a workgroup.
        int64_t nodes = 0;
        for (const WfSplitDev &sp : ph->splits) nodes = std::max<int64_t>(nodes, (int64_t)sp.r0 + sp.n2);
        const int blocks = (int)std::min<int64_t>(32, 1 + nodes / 8192);
        return wf_launch_sw_combine((const WfSplitDev *)ar->splits.ptr, (int)ph->splits.size(), blocks,
                                    (const uint32_t *)ar->colw.ptr, ka.cuts, (const uint64_t *)ar->bnd.ptr,
                                    (WfResultDev *)ar->res.ptr, stream) == hipSuccess
                   ? WF_OK
                   : WF_ERR_DEVICE;
    }
    if (!ph->splits.empty() &&
        wf_launch_bitpar_combine((const WfSplitDev *)ar->splits.ptr, (int)ph->splits.size(),
                                 (const uint32_t *)ar->colw.ptr, ka.cuts, (const uint64_t *)ar->bnd.ptr,
                                 (WfResultDev *)ar->res.ptr, stream) != hipSuccess)
        return WF_ERR_DEVICE;
    return WF_OK;
}

// Run a plan (directly, or by replaying its captured graph), time the device
// work with HIP events on the context stream and bring its pairs' results,
// which follow the launch through the context's pinned block, into `res`, if
// not null: one wait for everything.
int wf_run_plan(wf_ctx *ctx, WfPlanHost *ph, WfArenas *ar, int mode, double *kernel_ms, hipGraphExec_t exec,
                std::vector<WfResultDev> *res)
{
    const int maxg = wf_max_resident_groups(ctx, ph->variant);
    const size_t bytes = res ? (size_t)ph->npairs * sizeof(WfResultDev) : 0;
    int st;
    if (bytes && (st = wf_ensure_pinned(ctx, bytes)) != WF_OK) return st;
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (exec) {
        if (hipGraphLaunch(exec, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    } else if ((st = wf_enqueue_plan(ctx, ph, ar, mode, maxg, ctx->stream)) != WF_OK) {
        return st;
    }
    if (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (bytes) {
        ctx->pinned_busy = true;
        if (hipMemcpyAsync(ctx->pinned, ar->res.ptr, bytes, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
            return WF_ERR_DEVICE;
    }
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (bytes) {
        ctx->pinned_busy = false;
        const WfResultDev *r = reinterpret_cast<const WfResultDev *>(ctx->pinned);
        res->assign(r, r + ph->npairs);
    }
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) != hipSuccess) return WF_ERR_DEVICE;
    *kernel_ms = ms;
    return WF_OK;
}

// The caller's results from the device results r of the plan's pairs.
int wf_fill_results(const WfPlanHost *ph, const WfResultDev *r, double kernel_ms, wf_result *out, int64_t n)
{
    int worst = WF_OK;
    for (int64_t i = 0; i < std::min(n, ph->njobs); ++i) {
        wf_result &o = out[i];
        std::memset(&o, 0, sizeof(o));
        o.cells = ph->cells[i];
        o.kernel_ms = kernel_ms;
        if (ph->host_only[i]) {
            o.last = ph->host_result[i];
            o.max_score = 0;
            continue;
        }
        o.last = r[i].last;
        o.max_score = (ph->pairs[i].mode & WFK_MODE_NOMAX) ? -1 : r[i].maxs;
        o.status = r[i].status ? WF_ERR_TIMEOUT : WF_OK;
        if (o.status) worst = o.status;
    }
    return worst;
}

int wf_download_results(wf_ctx *ctx, WfPlanHost *ph, WfArenas *ar, double kernel_ms,
                            wf_result *out, int64_t n)
{
    std::vector<WfResultDev> r((size_t)std::max<int64_t>(1, ph->npairs));
    if (ph->npairs > 0 &&
        hipMemcpy(r.data(), ar->res.ptr, ph->npairs * sizeof(WfResultDev), hipMemcpyDeviceToHost) !=
            hipSuccess)
        return WF_ERR_DEVICE;
    (void)ctx;
    return wf_fill_results(ph, r.data(), kernel_ms, out, n);
}

// ----------------------------------------------------------------------------
// C ABI
// ----------------------------------------------------------------------------

extern "C" {

int wf_abi_version(void) { return WFDP_ABI_VERSION; }

int wf_variant_count(void) { return variant_count(); }

int wf_variant_info(int index, int32_t *engine, int32_t *rows_per_lane, int32_t *waves, int32_t *chunk)
{
    const WfVariant *v = variant_at(index);
    if (!v) return WF_ERR_INVALID;
    if (engine) *engine = v->engine;
    if (rows_per_lane) *rows_per_lane = v->rows_per_lane;
    if (waves) *waves = v->waves;
    if (chunk) *chunk = v->chunk;
    return WF_OK;
}

const char *wf_strerror(int status)
{
    switch (status) {
    case WF_OK: return "ok";
    case WF_ERR_INVALID: return "invalid argument";
    case WF_ERR_DEVICE: return "HIP runtime error";
    case WF_ERR_NOMEM: return "device memory exhausted";
    case WF_ERR_ALPHABET: return "more than 256 distinct symbols in one pair";
    case WF_ERR_TIMEOUT: return "device-side dependency wait timed out";
    case WF_ERR_NOKERNEL: return "no compiled kernel for the requested tile";
    case WF_ERR_AGAIN: return "queue full, retry";
    case WF_ERR_SCRATCH: return "the pair does not fit the fixed scratch area of wf_align_noalloc (64 MiB)";
    default: return "unknown error";
    }
}

int wf_ctx_create(int device, wf_ctx **out)
{
    if (!out) return WF_ERR_INVALID;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
        (void)hipGetLastError();
        return WF_ERR_DEVICE;
    }
    if (device < 0 || device >= ndev) return WF_ERR_INVALID;
    if (hipSetDevice(device) != hipSuccess) return WF_ERR_DEVICE;
    wf_ctx *c = new wf_ctx();
    c->device = device;
    if (hipGetDeviceProperties(&c->prop, device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        delete c;
        return WF_ERR_DEVICE;
    }
    // Set up this device's static scratch area of wf_align_noalloc (once per
    // device); a failure here is reported by that entry point's own call.
    (void)wf_noalloc_setup(device, c->stream, nullptr);
    wf_tune_autoload();
    *out = c;
    return WF_OK;
}

void wf_ctx_destroy(wf_ctx *ctx)
{
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    ctx->scratch.release();
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);  // after the stream's synchronisation above
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

int wf_ctx_set_timeout(wf_ctx *ctx, double seconds)
{
    if (!ctx || !(seconds > 0.0)) return WF_ERR_INVALID;
    ctx->timeout_s = seconds;
    return WF_OK;
}

int wf_device_query(wf_ctx *ctx, wf_device_info *out)
{
    if (!ctx || !out) return WF_ERR_INVALID;
    std::memset(out, 0, sizeof(*out));
    out->compute_units = ctx->prop.multiProcessorCount;
    out->max_clock_mhz = ctx->prop.clockRate / 1000;
    out->simds_per_cu = 4;
    out->wave_size = ctx->prop.warpSize;
    (void)hipSetDevice(ctx->device);
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess) {
        out->free_mem = (int64_t)fr;
        out->total_mem = (int64_t)tot;
    }
    std::snprintf(out->arch, sizeof(out->arch), "%s", ctx->prop.gcnArchName);
    return WF_OK;
}

int wf_align_batch(wf_ctx *ctx, const wf_job *jobs, int64_t njobs, const wf_tile *tile, wf_result *out)
{
    if (!ctx || (njobs > 0 && (!jobs || !out)) || njobs < 0) return WF_ERR_INVALID;
    if (njobs == 0) return WF_OK;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    WfPlanHost ph;
    BlockLayout L;
    WfArenas ar;
    int st = plan_and_place(ctx, jobs, njobs, tile, &ph, &ctx->scratch, [&] {
        L = BlockLayout(&ph);
        return upload_block(ctx, &ph, L, &ar);
    });
    if (st != WF_OK) return st;
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if ((st = wf_enqueue_plan(ctx, &ph, &ar, WF_RUN_PERSISTENT, wf_max_resident_groups(ctx, ph.variant), ctx->stream,
                              false)) != WF_OK)
        return st;
    if (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    // Results into the pinned block (its upload part is no longer read by
    // then), behind the launch: one wait for everything.
    WfResultDev *r = reinterpret_cast<WfResultDev *>(ctx->pinned + L.res);
    if (hipMemcpyAsync(r, ar.res.ptr, ph.npairs * sizeof(WfResultDev), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
        hipStreamSynchronize(ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    ctx->pinned_busy = false;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) != hipSuccess) return WF_ERR_DEVICE;
    return wf_fill_results(&ph, r, ms, out, njobs);
}

int wf_align(wf_ctx *ctx, int problem, const int32_t *a, int64_t n1, const int32_t *b, int64_t n2,
             const wf_tile *tile, wf_result *out)
{
    if (!ctx || !out) return WF_ERR_INVALID;
    wf_job j{problem, tile ? (tile->flags & WF_TILE_ED_TEXTBOOK) : 0, a, n1, b, n2};
    return wf_align_batch(ctx, &j, 1, tile, out);
}

int wf_align_table(wf_ctx *ctx, int problem, const int32_t *a, int64_t n1, const int32_t *b, int64_t n2,
                   const wf_tile *tile, int32_t *table, wf_result *out)
{
    if (!ctx || !out || !table || n1 <= 0 || n2 <= 0 || n1 * n2 > WF_TABLE_MAX_CELLS) return WF_ERR_INVALID;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    const int flags = tile ? (tile->flags & WF_TILE_ED_TEXTBOOK) : 0;
    const wf_job j{problem, flags, a, n1, b, n2};
    // The table kernel is the lock-step sweep <R=2, W=4, K=32>; the plan's
    // strips must have its geometry.
    const wf_tile lock{32, 512, 2, WF_TILE_LOCKSTEP | flags};
    WfPlanHost ph;
    int st = wf_build_plan(ctx, &j, 1, &lock, &ph);
    if (st != WF_OK) return st;
    const WfVariant *v = ph.variant;
    if (v->engine != WF_ENGINE_LOCKSTEP || v->rows_per_lane != 2 || v->waves != 4 || v->chunk != 32)
        return WF_ERR_NOKERNEL;
    if ((st = wf_upload_plan(ctx, &ph, &ctx->scratch)) != WF_OK) return st;
    DevBuf dt;
    if ((st = dt.ensure((size_t)(n1 * n2) * sizeof(int32_t))) != WF_OK) return st;
    WfArenas *ar = &ctx->scratch;
    if (wf_launch_reset((WfResultDev *)ar->res.ptr, 1, (int32_t *)ar->counters.ptr, 2, (uint32_t *)ar->epoch.ptr,
                        1, ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    WfKernelArgs ka{};
    ka.pairs = (const WfPairDev *)ar->pairs.ptr;
    ka.tasks = (const WfTaskDev *)ar->tasks.ptr;
    ka.codes = (const uint8_t *)ar->codes.ptr;
    ka.bnd = (uint64_t *)ar->bnd.ptr;
    ka.res = (WfResultDev *)ar->res.ptr;
    ka.epoch = (const uint32_t *)ar->epoch.ptr;
    ka.timeout_ticks = (int64_t)(ctx->timeout_s * 1.0e8);
    ka.counter = (int32_t *)ar->counters.ptr;
    ka.task_begin = 0;
    ka.task_end = (int32_t)ph.tasks.size();
    ka.table = (int32_t *)dt.ptr;
    const int grid = (int)std::min<int64_t>((int64_t)ph.tasks.size(), ctx->prop.multiProcessorCount);
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (grid > 0 && wf_launch_table(grid, &ka, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
    if (hipMemcpy(table, dt.ptr, (size_t)(n1 * n2) * sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess)
        return WF_ERR_DEVICE;
    dt.release();
    return wf_download_results(ctx, &ph, ar, ms, out, 1);
}

int wf_align_naive(wf_ctx *ctx, int problem, const int32_t *a, int64_t n1, const int32_t *b, int64_t n2,
                   const wf_tile *tile, int method, int32_t *table, wf_result *out)
{
    if (!ctx || !out || n1 < 0 || n2 < 0 || (n1 > 0 && !a) || (n2 > 0 && !b)) return WF_ERR_INVALID;
    if (problem != WF_LCS && problem != WF_ED && problem != WF_SW) return WF_ERR_INVALID;
    if (method != WF_NAIVE_DIAGONAL && method != WF_NAIVE_TILE) return WF_ERR_INVALID;
    if (n1 >= INT32_MAX || n2 >= INT32_MAX) return WF_ERR_INVALID;
    const bool textbook = tile && (tile->flags & WF_TILE_ED_TEXTBOOK);
    *out = wf_result{};
    out->cells = (uint64_t)n1 * (uint64_t)n2;
    if (n1 == 0 || n2 == 0) {
        // One side empty: the table is its boundary.
        out->last = (problem == WF_ED) ? (int32_t)(n2 > 0 ? n2 : (textbook ? n1 : std::max<int64_t>(0, n1 - 1))) : 0;
        return WF_OK;
    }
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    const int64_t cells = (n1 + 1) * (n2 + 1);
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) return WF_ERR_DEVICE;
    const size_t need = (size_t)cells * sizeof(int32_t) + (size_t)(n1 + n2 + 64) * sizeof(int32_t);
    if (need > fr) return WF_ERR_NOMEM;
    DevBuf dt, dab;
    int st;
    if ((st = dt.ensure((size_t)cells * sizeof(int32_t))) != WF_OK) return st;
    if ((st = dab.ensure((size_t)(n1 + n2 + 64) * sizeof(int32_t))) != WF_OK) return st;
    int32_t *da = (int32_t *)dab.ptr, *db = da + n1, *smax = db + n2;
    if (hipMemcpyAsync(da, a, (size_t)n1 * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(db, b, (size_t)n2 * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
        hipMemsetAsync(smax, 0, sizeof(int32_t), ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (wf_launch_naive(method, problem, textbook ? 1 : 0, (int *)dt.ptr, da, db, (int)n1, (int)n2,
                        problem == WF_SW ? smax : nullptr, ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    if (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
    const int32_t *dlast = (const int32_t *)dt.ptr + cells - 1;
    int32_t last = 0, mx = 0;
    if (hipMemcpy(&last, dlast, sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(&mx, smax, sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess)
        return WF_ERR_DEVICE;
    if (table && hipMemcpy2D(table, (size_t)n1 * sizeof(int32_t), (const int32_t *)dt.ptr + n1 + 2,
                             (size_t)(n1 + 1) * sizeof(int32_t), (size_t)n1 * sizeof(int32_t), (size_t)n2,
                             hipMemcpyDeviceToHost) != hipSuccess)
        return WF_ERR_DEVICE;
    out->last = last;
    out->max_score = problem == WF_SW ? mx : 0;
    out->kernel_ms = ms;
    return WF_OK;
}

int wf_plan_create(wf_ctx *ctx, const wf_job *jobs, int64_t njobs, const wf_tile *tile, wf_plan **out)
{
    if (!ctx || !out || njobs <= 0 || !jobs) return WF_ERR_INVALID;
    *out = nullptr;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    wf_plan *p = new wf_plan();
    p->ctx = ctx;
    int st = plan_and_place(ctx, jobs, njobs, tile, &p->host, &p->own,
                            [&] { return wf_upload_plan(ctx, &p->host, &p->own); });
    if (st == WF_OK) st = wf_ensure_pinned(ctx, (size_t)p->host.npairs * sizeof(WfResultDev));
    if (st != WF_OK) {
        p->own.release();
        delete p;
        return st;
    }
    *out = p;
    return WF_OK;
}

int wf_plan_run(wf_plan *plan, int mode)
{
    if (!plan || (mode != WF_RUN_PERSISTENT && mode != WF_RUN_PER_PAIR)) return WF_ERR_INVALID;
    if (hipSetDevice(plan->ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    const int st = wf_run_plan(plan->ctx, &plan->host, &plan->own, mode, &plan->kernel_ms, plan->exec[mode],
                               &plan->res);
    plan->ran = (st == WF_OK);
    return st;
}

int wf_plan_capture(wf_plan *plan, int mode)
{
    if (!plan || (mode != WF_RUN_PERSISTENT && mode != WF_RUN_PER_PAIR)) return WF_ERR_INVALID;
    wf_ctx *ctx = plan->ctx;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    if (plan->exec[mode]) return WF_OK;
    const int maxg = wf_max_resident_groups(ctx, plan->host.variant);
    if (hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return WF_ERR_DEVICE;
    const int st = wf_enqueue_plan(ctx, &plan->host, &plan->own, mode, maxg, ctx->stream);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    if (st != WF_OK || e != hipSuccess || !g) {
        if (g) (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        return st != WF_OK ? st : WF_ERR_DEVICE;
    }
    hipGraphExec_t x = nullptr;
    if (hipGraphInstantiate(&x, g, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGraphDestroy(g);
        return WF_ERR_DEVICE;
    }
    plan->graph[mode] = g;
    plan->exec[mode] = x;
    return WF_OK;
}

int wf_plan_results(wf_plan *plan, wf_result *out, int64_t n)
{
    if (!plan || !out || n < 0) return WF_ERR_INVALID;
    if (!plan->ran) return WF_ERR_INVALID;
    return wf_fill_results(&plan->host, plan->res.data(), plan->kernel_ms, out, n);
}

double wf_plan_kernel_ms(const wf_plan *plan) { return plan ? plan->kernel_ms : -1.0; }

int wf_plan_describe(const wf_plan *plan, int32_t *engine, int32_t *rows_per_lane, int32_t *waves,
                     int32_t *chunk, int64_t *ntasks, int32_t *grid)
{
    if (!plan) return WF_ERR_INVALID;
    const WfVariant *v = plan->host.variant;
    if (engine) *engine = v->engine;
    if (rows_per_lane) *rows_per_lane = v->rows_per_lane;
    if (waves) *waves = v->waves;
    if (chunk) *chunk = v->chunk;
    if (ntasks) *ntasks = (int64_t)plan->host.tasks.size();
    if (grid) *grid = plan->host.grid;
    return WF_OK;
}

void wf_plan_destroy(wf_plan *plan)
{
    if (!plan) return;
    (void)hipSetDevice(plan->ctx->device);
    (void)hipStreamSynchronize(plan->ctx->stream);
    for (int m = 0; m < 2; ++m) {
        if (plan->exec[m]) (void)hipGraphExecDestroy(plan->exec[m]);
        if (plan->graph[m]) (void)hipGraphDestroy(plan->graph[m]);
    }
    plan->own.release();
    delete plan;
}

}  // extern "C"
