// wf_bitpar.hip -- bit-parallel wavefront engine for LCS and edit distance on
// gfx950.
//
// LCS (LCS/LCS.cpp:45-82) and edit distance (EditDistance/ED.cpp:45-81) have
// unit costs, so neighbouring cells differ by -1, 0 or +1 and a column of the
// table is fully described by bit vectors of its vertical differences.  A
// lane holds 32 consecutive rows as one 32-bit word and advances its word by
// one column per step with a fixed sequence of word operations:
//
//   ED   Myers' bit-vector algorithm in Hyyro's formulation, blocked as in
//        Myers (1999) "A fast bit-vector algorithm for approximate string
//        matching based on dynamic programming", J. ACM 46(3), section 4:
//        state Pv/Mv (vertical +1/-1), horizontal deltas Ph/Mh; the word
//        above passes its last row's horizontal delta (hin) down, and a -1
//        enters the carry chain of the addition (in place of Eq | 1).
//   LCS  the bit-vector LCS of Crochemore, Iliopoulos, Pinzon and Reid (2001)
//        "A fast and practical bit-vector algorithm for the longest common
//        subsequence problem", IPL 80(6): V' = (V + (V & Eq)) | (V & ~Eq);
//        the word above passes its addition's carry down.
//
// Eq is the lane's 32-row match mask for the column's symbol, looked up in a
// per-wave LDS table (symbol code x lane) built from the row symbols at strip
// start.  The words of a wave form the same 64-lane systolic array as the
// cell engines (lane l handles column s - l at step s; the word above's
// output reaches lane l through one DPP wave_shr:1), so a wave covers 2048
// rows and a column step costs 7 (LCS, staged) to 15 (ED) VALU operations for
// 32 cells instead of 3-4 per cell.  The chain of waves down a pair is 32 times shorter than
// the cell engines' (one wave per 2048 rows instead of per 128), which is
// where a single large pair spends half its time there.
//
// Scheduling is the lock-step engine's (wf_kernels.hip): W waves per strip
// advance in chunks of K = 64 or 128 steps between barriers, D chunks apart;
// wave 0 stages the column codes and the strip's top boundary into LDS one
// chunk ahead; the last wave stores the bottom row's boundary (ED: hin bits, LCS:
// carry) to HBM as epoch-tagged words for the next strip.  The score comes
// from the last column's vertical differences: ED D(n2,n1) = D(0,n1) + sum of
// Pv - Mv over the rows, LCS = number of zero bits of V, summed over the
// lanes with atomics.
//
// Also here: the staged variant (a staging wave per workgroup looks up the
// match masks for the compute waves) and the combine kernel of pairs split
// into a forward and a reversed column half (WfSplitDev).
#include <hip/hip_runtime.h>
#include <climits>
#include <stdint.h>

#include "wf_cells.h"
#include "wf_device.h"
#include "wf_variants.h"

namespace wfb {

using wfk::kDppWaveShr1;
using wfk::now_ticks;
using wfk::pow2_at_least;

constexpr int kRowsPerWave = 64 * 32;

// Chunk geometry for K steps per chunk: D chunks between consecutive waves,
// ring slots (column c in slot (c + 64) mod RS), code window AW.  A chunk
// must outlast a global-memory round trip (wave 0 loads the next chunk's
// codes and top boundary during it): K = 64 or 128.
template <int W, int K>
struct BpCfg {
    static constexpr int D = (K + 62) / K + 1;
    static constexpr int RS = pow2_at_least((D + 2) * K + 64);
    static constexpr int AW = pow2_at_least((2 + (W - 1) * D) * K + 64 + K);
};

template <int W, int K>
struct BpShared {
    static constexpr int AW = BpCfg<W, K>::AW;
    static constexpr int RS = BpCfg<W, K>::RS;
    // Match masks: peq[wave][code * 64 + lane] = bit r set iff row r of the
    // lane's word holds symbol `code` (codes < 32).
    __attribute__((aligned(16))) int peq[W][32 * 64];
    // ring[0]: the strip's top boundary; ring[w+1]: lane 63 of wave w, read
    // by wave w+1 (w = W-1: stored to HBM).  ED: (Ph, Mh) words, whose top
    // bits are the horizontal delta (+1, -1) of the word's last row; LCS:
    // (a word whose bit 31 is the carry, 0).
    __attribute__((aligned(16))) int2 ring[W + 1][RS];
    // Lanes 0..62 store here so that the ring capture is one unmasked write.
    int2 dummy[W][64 + K];
    // Column codes, column c at slot c mod AW, the first K slots mirrored.
    uint32_t aw[AW + K];
    int task;
    int abort_at;
};

struct BpState {
    uint32_t pv, mv;   // ED: vertical +1 / -1 bits; LCS: pv = V
    int ph, mh;        // ED: this column's horizontal deltas (pre-shift); LCS: ph = carry out in bit 31
};

// A state word that the next step reads in one register.  Without it the compiler
// keeps its terms apart to fold them into the next step's three-input operations:
// a shorter chain, but an operation more a step, and issue is what bounds a wave
// (staged, one pair: LCS 32768^2 0.398 -> 0.375 ms, ED 65536^2 1.33 -> 1.30).
__device__ __forceinline__ void one_form(uint32_t &w)
{
    asm("" : "+v"(w));
}

template <int P>
__device__ __forceinline__ void bp_step(BpState &st, int2 inj, uint32_t eq)
{
    if (P == WFK_ED) {
        const int nph = __builtin_amdgcn_update_dpp(inj.x, st.ph, kDppWaveShr1, 0xf, 0xf, false);
        const int nmh = __builtin_amdgcn_update_dpp(inj.y, st.mh, kDppWaveShr1, 0xf, 0xf, false);
        // A delta of -1 from above makes row 0 a match (Eq | 1).  Added to the
        // sum instead, it does the same to xh's bit 0 and to the carry out of it
        // whatever Pv's and Eq's bits are, and needs no Eq | 1 of its own.
        const uint32_t hm = (uint32_t)nmh >> 31;  // hin == -1
        const uint32_t xv = eq | st.mv;
        const uint32_t xh = (((eq & st.pv) + st.pv + hm) ^ st.pv) | eq;
        const uint32_t ph = st.mv | ~(xh | st.pv);
        const uint32_t mh = st.pv & xh;
        // (h << 1) | the word above's last-row delta.
        const uint32_t phs = __builtin_amdgcn_alignbit(ph, (uint32_t)nph, 31);
        const uint32_t mhs = __builtin_amdgcn_alignbit(mh, (uint32_t)nmh, 31);
        st.pv = mhs | ~(xv | phs);
        st.mv = phs & xv;
        one_form(st.pv);
        one_form(st.mv);
        st.ph = (int)ph;
        st.mh = (int)mh;
    } else {
        // st.ph carries the word's carry out in bit 31 (the lane below
        // shifts it down); the sum and its carry are three-input operations.
        const int cw = __builtin_amdgcn_update_dpp(inj.x, st.ph, kDppWaveShr1, 0xf, 0xf, false);
        const uint32_t u = st.pv & eq;
        const uint32_t sum = st.pv + u + ((uint32_t)cw >> 31);
        // Carry out of bit 31: majority of the operands' top bits and the
        // carry into it, (V & U) | ((V | U) & ~sum), with U = V & Eq.
        st.ph = (int)(st.pv & (eq | ~sum));
        st.pv = sum | (st.pv & ~eq);
        one_form(st.pv);
    }
}

// One chunk of K steps from s0 for one wave.  MASKED: some lane's column is
// outside 0..n1-1; such lanes keep their state (so the lane below reads the
// delta or carry of the lane's last real column).
template <int P, int K, int AW, int RS, bool MASKED>
__device__ __forceinline__ void bp_chunk(BpState &st, int s0, int lane, int n1, const int2 *ring_prev, int2 *ring_cur,
                                         int2 *dummy, const uint32_t *aw, const int *peq)
{
    // Lane 0's column c = s0 + q lives in slot (c + 64) mod RS; a run of 64
    // slots from a multiple of 64 never wraps (K and RS are multiples of 64).
    const uint32_t *__restrict__ cp = aw + ((s0 - lane) & (AW - 1));
    int2 *cap = (lane == 63) ? ring_cur + ((s0 + 1) & (RS - 1)) : dummy + lane;
    int2 *cap_last = (lane == 63) ? ring_cur + ((s0 + K) & (RS - 1)) : dummy + lane + (K - 1);
    // Operands are read ahead of their group of 4 steps: the column codes
    // two groups ahead, the match masks they select and lane 0's upper
    // words one group ahead, so no LDS latency (nor the code -> mask
    // dependency) sits in front of a group's arithmetic.
    auto load_codes = [&](int q, uint32_t (&c)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            c[u] = cp[q + u];
            if (MASKED) c[u] &= 31u;  // window slots of columns outside the pair hold stale codes
        }
    };
    auto load_eq = [&](const uint32_t (&c)[4], uint32_t (&e)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = (uint32_t)peq[c[u] * 64 + lane];
    };
    auto load_inj = [&](int q, int2 (&v)[4]) {
        const int2 *ib = ring_prev + ((s0 + 64 + (q & ~63)) & (RS - 1)) + (q & 63);
        const int4 i01 = *reinterpret_cast<const int4 *>(ib);
        const int4 i23 = *reinterpret_cast<const int4 *>(ib + 2);
        v[0] = make_int2(i01.x, i01.y);
        v[1] = make_int2(i01.z, i01.w);
        v[2] = make_int2(i23.x, i23.y);
        v[3] = make_int2(i23.z, i23.w);
    };
    uint32_t code_n[4], eqv[4];
    int2 injv[4];
    {
        uint32_t c0[4];
        load_codes(0, c0);
        load_codes(4, code_n);
        load_eq(c0, eqv);
        load_inj(0, injv);
    }
#pragma unroll
    for (int q = 0; q < K; q += 4) {
        uint32_t eqn[4] = {0u, 0u, 0u, 0u}, code_nn[4] = {0u, 0u, 0u, 0u};
        int2 injn[4] = {};
        if (q + 4 < K) {
            load_eq(code_n, eqn);
            load_inj(q + 4, injn);
        }
        if (q + 8 < K) load_codes(q + 8, code_nn);
        int2 capv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (MASKED) {
                const bool valid = (unsigned)(s0 + q + u - lane) < (unsigned)n1;
                BpState nx = st;
                bp_step<P>(nx, injv[u], eqv[u]);
                if (valid) st = nx;
            } else {
                bp_step<P>(st, injv[u], eqv[u]);
            }
            capv[u] = make_int2(st.ph, st.mh);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = q + u;
            if (j == K - 1)
                *cap_last = capv[u];
            else
                cap[j] = capv[u];
        }
        if (q + 4 < K) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                eqv[u] = eqn[u];
                injv[u] = injn[u];
                code_n[u] = code_nn[u];
            }
        }
    }
}

// A wave's match-mask table from its rows' codes: bit r of entry (code, lane) for
// row r of the lane, where `rows` has the bit.  The codes come in two 16-byte
// loads (b's codes are 16-byte aligned and allocated to a multiple of 16) and
// every row is entered, those outside `rows` with no bit: a byte load and a branch
// a row stood at the head of every strip (LCS 256^2 43 -> 41 us a call, ED 65536^2
// 1.213 -> 1.190 ms).
__device__ __forceinline__ void build_peq(int *peq, const uint8_t *b, int64_t row0, int64_t n2, uint32_t rows,
                                          int lane)
{
    int4 *z = reinterpret_cast<int4 *>(peq);
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i * 64 + lane] = make_int4(0, 0, 0, 0);
    uint4 v[2] = {};
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (row0 + 16 * i < n2) v[i] = *reinterpret_cast<const uint4 *>(b + row0 + 16 * i);
    const uint32_t w[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
    for (int r = 0; r < 32; ++r)
        atomicOr(&peq[((w[r / 4] >> (8 * (r % 4))) & 31u) * 64 + lane], (int)((1u << r) & rows));
}

// One strip (`g`) of one pair, swept by the whole workgroup.
template <int P, int W, int K>
__device__ void bp_group(const WfKernelArgs &ka, const WfPairDev &pd, int pair, int g, BpShared<W, K> &sh, int lane,
                         int wave, uint32_t epoch)
{
    constexpr int AW = BpCfg<W, K>::AW;
    constexpr int RS = BpCfg<W, K>::RS;
    constexpr int kD = BpCfg<W, K>::D;
    constexpr int kK = K;
    const int n1 = pd.n1, n2 = pd.n2;
    const int64_t row0 = (int64_t)g * (W * kRowsPerWave) + wave * kRowsPerWave + lane * 32;
    const uint8_t *acodes = ka.codes + pd.a_off;
    const uint8_t *bcodes = ka.codes + pd.b_off;
    const int64_t rows_left = (int64_t)n2 - (int64_t)g * (W * kRowsPerWave);
    const int wa = (int)min<int64_t>(W, (rows_left + kRowsPerWave - 1) / kRowsPerWave);
    const bool active = wave < wa;
    const int nvalid = (int)max<int64_t>(0, min<int64_t>(32, (int64_t)n2 - row0));
    const uint32_t rowmask = nvalid >= 32 ? 0xffffffffu : ((1u << nvalid) - 1u);
    const bool textbook = (pd.mode & WFK_MODE_TEXTBOOK) != 0;

    // Match masks of this wave's rows.
    int *peq = sh.peq[wave];
    if (active) {
        build_peq(peq, bcodes, row0, n2, rowmask, lane);
    }

    const int nsteps = n1 + 63;
    const int nch = (nsteps + kK - 1) / kK;
    const int total = nch + (wa - 1) * kD;
    const bool has_prev = g > 0;
    const bool has_next = g + 1 < pd.ngroups;
    const uint64_t *bprev = ka.bnd + pd.bnd_off + (int64_t)(g - 1) * n1;
    uint64_t *bnext = ka.bnd + pd.bnd_off + (int64_t)g * n1;
    const uint64_t tag = (uint64_t)epoch << 32;

    // Top boundary and column codes of columns [c*K, c*K+K), staged by wave
    // 0 in K/64 batches of 64 columns (one per lane): the previous strip's
    // bottom-row words, or row 0 of the table (ED: delta 0 at column 1 and +1
    // after it, ED.cpp:48-54; +1 throughout for the textbook row; LCS: no
    // carry).
    constexpr int NB = K / 64;
    static_assert(K % 64 == 0, "K must be a multiple of 64");
    struct Pre {
        uint64_t top[NB];
        uint32_t code[NB];
    };
    auto load_pre = [&](int c, Pre &pr) {
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            const int x = c * kK + h * 64 + lane;
            pr.code[h] = x < n1 ? (uint32_t)acodes[x] : 0u;
            pr.top[h] = (!has_prev || x >= n1) ? tag
                                               : __hip_atomic_load(bprev + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    auto fill = [&](int c, Pre &pr) -> bool {
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            const int x = c * kK + h * 64 + lane;
            uint64_t top = pr.top[h];
            if (__builtin_amdgcn_ballot_w64((top >> 32) != (uint64_t)epoch) != 0) {
                const int64_t t0 = now_ticks();
                for (;;) {
                    __builtin_amdgcn_s_sleep(1);
                    if ((top >> 32) != (uint64_t)epoch)
                        top = __hip_atomic_load(bprev + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (__builtin_amdgcn_ballot_w64((top >> 32) != (uint64_t)epoch) == 0) break;
                    if (now_ticks() - t0 > ka.timeout_ticks) return false;
                }
            }
            if (x < n1) {
                uint32_t v;
                if (has_prev)
                    v = (uint32_t)top;
                else
                    v = (P == WFK_ED && (x >= 1 || textbook)) ? 1u : 0u;
                sh.ring[0][(x + 64) & (RS - 1)] = (P == WFK_ED)
                                                      ? make_int2((int)((v & 1u) << 31), (int)(((v >> 1) & 1u) << 31))
                                                      : make_int2((int)((v & 1u) << 31), 0);
                const int slot = x & (AW - 1);
                sh.aw[slot] = pr.code[h];
                if (slot < kK) sh.aw[AW + slot] = pr.code[h];
            }
        }
        return true;
    };

    if (wave == 0) {
        Pre p0;
        load_pre(0, p0);
        if (!fill(0, p0) && lane == 0) sh.abort_at = -1;
    }
    __syncthreads();

    int copied = 0;  // wave W-1: columns already stored to bnext
    auto copy_out = [&](int upto, bool from_ring) {
        while (copied < upto) {
            const int x = copied + lane;
            if (x < upto) {
                uint32_t v = 0;
                if (from_ring) {
                    const int2 w = sh.ring[W][(x + 64) & (RS - 1)];
                    v = (P == WFK_ED) ? (((uint32_t)w.x >> 31) | (((uint32_t)w.y >> 31) << 1)) : ((uint32_t)w.x >> 31);
                }
                __hip_atomic_store(bnext + x, tag | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            copied = min(upto, copied + 64);
        }
    };

    BpState st;
    st.pv = (P == WFK_ED) ? 0xffffffffu : 0xffffffffu;  // ED: column 0 rises by 1 per row; LCS: V = all ones
    st.mv = 0u;
    st.ph = 0;
    st.mh = 0;

    bool aborted = sh.abort_at <= -1;
    for (int j = 0; j < total && !aborted; ++j) {
        const int cj = j - wave * kD;
        Pre pre;
        if (wave == 0 && j + 1 < nch) load_pre(j + 1, pre);
        if (cj >= 0 && cj < nch && active) {
            const int s0 = cj * kK;
            const bool steady = (s0 >= 63) && (s0 + kK - 1 <= n1 - 1);
            if (steady)
                bp_chunk<P, K, AW, RS, false>(st, s0, lane, n1, sh.ring[wave], sh.ring[wave + 1], sh.dummy[wave], sh.aw, peq);
            else
                bp_chunk<P, K, AW, RS, true>(st, s0, lane, n1, sh.ring[wave], sh.ring[wave + 1], sh.dummy[wave], sh.aw, peq);
            // Steps < s0 + K are done: lane 63 has finished columns < s0 + K - 63.
            if (wave == W - 1 && has_next) copy_out(min(n1, s0 + kK - 63), true);
        }
        if (wave == 0 && j + 1 < nch) {
            if (!fill(j + 1, pre) && lane == 0) sh.abort_at = j;
        }
        __syncthreads();
        aborted = sh.abort_at <= j;
    }

    if (aborted) {
        if (threadIdx.x == 0) atomicOr(&ka.res[pair].status, 1);
        if (wave == W - 1 && has_next) copy_out(n1, false);
        return;
    }
    if (wave == W - 1 && has_next) copy_out(n1, true);

    // Score: the last column's vertical differences over the rows.
    if (active) {
        int v;
        if (P == WFK_ED)
            v = __builtin_popcount(st.pv & rowmask) - __builtin_popcount(st.mv & rowmask);
        else
            v = __builtin_popcount(~st.pv & rowmask);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (P == WFK_ED && g == 0 && wave == 0) v += textbook ? n1 : n1 - 1;  // D(0, n1)
        if (lane == 0) atomicAdd(&ka.res[pair].last, v);
        if (pd.col_off >= 0) {
            uint32_t *cw = ka.colw + 2 * (pd.col_off + ((int64_t)g * W + wave) * 64 + lane);
            cw[0] = st.pv;
            cw[1] = st.mv;
        }
    }
}

template <int W, int K>
__global__ __launch_bounds__(64 * W) void wf_engine_bitpar(WfKernelArgs ka)
{
    __shared__ BpShared<W, K> sh;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(*ka.epoch);
    // Codes in the window are always < 32, even in slots no strip wrote yet.
    for (int i = threadIdx.x; i < BpShared<W, K>::AW + K; i += blockDim.x) sh.aw[i] = 0;
    for (;;) {
        if (threadIdx.x == 0) {
            sh.task = ka.task_begin + atomicAdd(ka.counter, 1);
            sh.abort_at = 0x7fffffff;
        }
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sh.task);
        __syncthreads();
        if (t >= ka.task_end) break;
        const WfTaskDev td = ka.tasks[t];
        const WfPairDev pd = ka.pairs[td.pair];
        wfk::set_wave_priority(pd.prio);
        if (pd.prob == WFK_ED)
            bp_group<WFK_ED, W, K>(ka, pd, td.pair, td.group, sh, lane, wave, epoch);
        else
            bp_group<WFK_LCS, W, K>(ka, pd, td.pair, td.group, sh, lane, wave, epoch);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Staged variant: one more wave per workgroup looks up the match masks.
//
// In the engine above a compute wave spends about a sixth of its
// instructions per step on finding Eq (the column code's LDS read, the table
// address, the table read).  Here a staging wave does those lookups for the
// compute waves one chunk ahead and leaves each lane's masks in LDS in step
// order, four steps per 16-byte word, so a compute wave fetches the masks of
// four steps with one ds_read_b128 and no address arithmetic.  The staging wave
// also loads the column codes, lays out what the row above hands to lane 0, and
// publishes the bottom row, so the compute waves issue no global memory
// operation at all.  The mask buffers take 16 KB of LDS per compute wave and
// chunk parity: the planner takes this variant for launches whose strips fit on
// the chip at once (single large pairs), and the engine above, which packs more
// compute waves per CU, for throughput-bound batches.
//
// A step is bound by the issue of a lone wave (4 cycles an instruction at best,
// more where 8-byte instructions follow each other off their alignment): 13
// VALU operations for ED and 6 for LCS, one or two to collect what lane 63
// hands down, and the LDS reads.  Per step, W = 1: ED 38.4 -> 31.2 ns, LCS 25.5 ->
// 16.7 (before: every step's words stored to LDS, ED with two more operations,
// LCS with one, and the reads at their use); ED 65536^2 1.51 -> 1.25 ms, LCS
// 32768^2 0.547 -> 0.353 (and 1.19 and 0.338 along a staircase).  W = 2 overloads the one staging wave.
// ---------------------------------------------------------------------------

template <int W>
struct BsCfg {
    static constexpr int K = 64;
    // Chunks between consecutive waves: wave w's upper words of a chunk are
    // taken out of wave w-1's (two chunks of it) one iteration ahead.
    static constexpr int D = 3;
    static constexpr int AW = pow2_at_least((2 + (W - 1) * D) * K + 64 + K);
};

template <int W>
struct BsShared {
    static constexpr int K = BsCfg<W>::K;
    static constexpr int AW = BsCfg<W>::AW;
    // eqb[i & 1][w][q / 4][lane]: lane's match masks for steps q..q+3 of
    // compute wave w's chunk in iteration i (written during iteration i - 1).
    int4 eqb[2][W][K / 4][64];
    // injb[i & 1][w][q]: what the row above wave w hands to lane 0 at step q of
    // that chunk.  ED: (Ph, Mh) words whose top bits are the horizontal delta
    // (+1, -1); LCS: one word (the first K ints) whose top bit is the carry.
    __attribute__((aligned(16))) int2 injb[2][W][K];
    // cap[w][k & 7]: what lane 63 of wave w handed down in its steps 32k ..
    // 32k+31 (columns 32k-63 ..), one bit per step, the first in bit 31; ED: .x
    // +1, .y -1; LCS: .x the carry.
    int2 cap[W][8];
    int2 dummy[64];  // lanes 0..62 store here, so that the capture is one unmasked write
    __attribute__((aligned(16))) int peq[W][32 * 64];  // as in BpShared
    // Column codes as in BpShared, times 64 (a row of peq): two operations less a
    // step for the staging wave, which bounds LCS (32768^2 0.363 -> 0.353 ms).
    uint32_t aw[AW + K];
    int task;
    int abort_at;
};

// Steps of one 64-bit-word row of a strip's bottom boundary in HBM: chunk c's
// 64 steps of lane 63 are words 2c and 2c+1 (LCS), each (epoch << 32 | 32 bits
// as in BsShared::cap), or pairs of words (ED: +1 bits, -1 bits).
__device__ __forceinline__ int64_t bs_row_words(int n1) { return 4 * (int64_t)((n1 + 126) / 64); }

// One chunk of K steps of a compute wave; masks from `eqw` (= eqb[i & 1][w]),
// upper words from `inj` (= injb[i & 1][w]), lane 63's bits to cap[0] and cap[1]
// (`cap`: a dummy in the other lanes).  The bits are collected in a register
// (one v_alignbit a step and word) and stored once per 32 steps: storing
// every step's words instead took 55 cycles a step for LCS and 79 for ED where
// this took 39 and 70 (one wave, operands from LDS, no staging wave beside).
template <int P, int K, bool MASKED>
__device__ __forceinline__ void bs_chunk(BpState &st, int s0, int lane, int n1, const int2 *inj, int2 *cap,
                                         const int4 *eqw)
{
    constexpr bool ED = P == WFK_ED;
    auto load_inj = [&](int q, int2 (&v)[4]) {
        if (ED) {
            const int4 i01 = *reinterpret_cast<const int4 *>(inj + q);
            const int4 i23 = *reinterpret_cast<const int4 *>(inj + q + 2);
            v[0] = make_int2(i01.x, i01.y);
            v[1] = make_int2(i01.z, i01.w);
            v[2] = make_int2(i23.x, i23.y);
            v[3] = make_int2(i23.z, i23.w);
        } else {
            const int4 i = *reinterpret_cast<const int4 *>(reinterpret_cast<const int *>(inj) + q);
            v[0].x = i.x;
            v[1].x = i.y;
            v[2].x = i.z;
            v[3].x = i.w;
        }
    };
    const int4 *ep = eqw + lane;
    // Masks and lane 0's upper words are read A groups of 4 steps ahead, and
    // held there: the compiler moves the reads down to their use, where each
    // waits behind the staging wave's (0.375 -> 0.363 and 1.30 -> 1.26 ms; A = 1
    // or 3 within 1%).
    constexpr int A = 2;
    int4 eqv[A + 1];
    int2 injv[A + 1][4] = {};
#pragma unroll
    for (int i = 0; i < A; ++i) {
        eqv[i] = ep[4 * i * 16];
        load_inj(4 * i, injv[i]);
    }
    uint32_t accp = 0, accm = 0;
#pragma unroll
    for (int q = 0; q < K; q += 4) {
        if (q + 4 * A < K) {
            eqv[A] = ep[(q + 4 * A) * 16];
            load_inj(q + 4 * A, injv[A]);
        }
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t e[4] = {(uint32_t)eqv[0].x, (uint32_t)eqv[0].y, (uint32_t)eqv[0].z, (uint32_t)eqv[0].w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (MASKED) {
                const bool valid = (unsigned)(s0 + q + u - lane) < (unsigned)n1;
                BpState nx = st;
                bp_step<P>(nx, injv[0][u], e[u]);
                if (valid) st = nx;
            } else {
                bp_step<P>(st, injv[0][u], e[u]);
            }
            accp = __builtin_amdgcn_alignbit(accp, (uint32_t)st.ph, 31);
            if (ED) accm = __builtin_amdgcn_alignbit(accm, (uint32_t)st.mh, 31);
        }
        if (q % 32 == 28) cap[q / 32] = make_int2((int)accp, (int)accm);
#pragma unroll
        for (int i = 0; i < A; ++i) {
            eqv[i] = eqv[i + 1];
#pragma unroll
            for (int u = 0; u < 4; ++u) injv[i][u] = injv[i + 1][u];
        }
    }
}

// One strip (`g`) of one pair: waves 0..W-1 compute, wave W stages.
template <int P, int W>
__device__ void bs_group(const WfKernelArgs &ka, const WfPairDev &pd, int pair, int g, BsShared<W> &sh, int lane,
                         int wave, uint32_t epoch)
{
    constexpr int K = BsCfg<W>::K;
    constexpr int AW = BsCfg<W>::AW;
    constexpr int kD = BsCfg<W>::D;
    constexpr bool ED = P == WFK_ED;
    constexpr int NP = ED ? 2 : 1;  // bit planes of the handed-down words
    const bool stager = wave == W;
    // The strips of a split pair end at columns of their own, and the rows of a
    // reversed part start with some that hold no symbol (WfSplitDev::pad).
    const bool cut = pd.cut >= 0;
    const int n1 = cut ? ka.cuts[pd.cut + g].n : pd.n1, n2 = pd.n2;
    const int pad = cut ? ka.cuts[pd.cut + g].pad : 0;
    const int64_t row0 = (int64_t)g * (W * kRowsPerWave) + wave * kRowsPerWave + lane * 32;
    const uint8_t *acodes = ka.codes + pd.a_off;
    const uint8_t *bcodes = ka.codes + pd.b_off;
    const int64_t rows_left = (int64_t)n2 - (int64_t)g * (W * kRowsPerWave);
    const int wa = (int)min<int64_t>(W, (rows_left + kRowsPerWave - 1) / kRowsPerWave);
    const bool active = !stager && wave < wa;
    const int nvalid = active ? (int)max<int64_t>(0, min<int64_t>(32, (int64_t)n2 - row0)) : 0;
    const uint32_t rowmask = nvalid >= 32 ? 0xffffffffu : ((1u << nvalid) - 1u);
    const bool textbook = (pd.mode & WFK_MODE_TEXTBOOK) != 0;

    if (active) {
        int *peq = sh.peq[wave];
        const uint32_t symbols = pad - row0 >= 32 ? 0u : 0xffffffffu << max(0, (int)(pad - row0));
        build_peq(peq, bcodes, row0, n2, rowmask & symbols, lane);
    }

    const int nsteps = n1 + 63;
    const int nch = (nsteps + K - 1) / K;
    const int total = nch + (wa - 1) * kD;
    const bool has_prev = g > 0;
    const bool has_next = g + 1 < pd.ngroups;
    const uint64_t *bprev =
        ka.bnd + (cut ? ka.cuts[pd.cut + max(0, g - 1)].bnd : pd.bnd_off + (g - 1) * bs_row_words(n1));
    uint64_t *bnext = ka.bnd + (cut ? ka.cuts[pd.cut + g].bnd : pd.bnd_off + g * bs_row_words(n1));
    const uint64_t tag = (uint64_t)epoch << 32;

    // Staging wave: column codes of chunk c (column c*K + lane per lane) into
    // the code window, the strip's top boundary of chunk c into injb, and the
    // masks of an iteration's chunks.
    auto load_code = [&](int c) -> uint32_t {
        const int x = c * K + lane;
        return x < n1 ? (uint32_t)acodes[x] : 0u;
    };
    auto put_code = [&](int c, uint32_t code) {
        const int x = c * K + lane;
        if (x < n1) {
            const int slot = x & (AW - 1);
            sh.aw[slot] = (code & 31u) * 64;
            if (slot < K) sh.aw[AW + slot] = (code & 31u) * 64;
        }
    };
    // Column c*K + q of chunk c is step c*K + q + 63 of lane 63 of the wave
    // above, so the chunk's columns are in its words 2c + 1 .. 2c + 3.
    const int word_of = ((lane + 63) >> 5) - 1, bit_of = 31 - ((lane + 63) & 31);
    auto put_inj = [&](int it, int w, uint32_t plus, uint32_t minus) {
        if (ED)
            sh.injb[it & 1][w][lane] = make_int2((int)(plus << 31), (int)(minus << 31));
        else
            reinterpret_cast<int *>(sh.injb[it & 1][w])[lane] = (int)(plus << 31);
    };
    // The strip above's words (lane i: word 2c + 1 + i / NP, plane i % NP).
    auto has_word = [&](int c) { return has_prev && lane < 3 * NP && 2 * c + 1 + lane / NP < 2 * nch; };
    auto load_top = [&](int c) -> uint64_t {
        return has_word(c) ? __hip_atomic_load(bprev + (2 * c + 1) * NP + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                           : tag;
    };
    auto fill_top = [&](int c, uint64_t top) -> bool {
        if (__builtin_amdgcn_ballot_w64((top >> 32) != (uint64_t)epoch) != 0) {
            const int64_t t0 = now_ticks();
            for (;;) {
                __builtin_amdgcn_s_sleep(1);
                if ((top >> 32) != (uint64_t)epoch) top = load_top(c);
                if (__builtin_amdgcn_ballot_w64((top >> 32) != (uint64_t)epoch) == 0) break;
                if (now_ticks() - t0 > ka.timeout_ticks) return false;
            }
        }
        uint32_t plus, minus = 0;
        if (has_prev) {
            plus = ((uint32_t)__shfl((int)(uint32_t)top, word_of * NP) >> bit_of) & 1u;
            if (ED) minus = ((uint32_t)__shfl((int)(uint32_t)top, word_of * NP + 1) >> bit_of) & 1u;
        } else {
            plus = (ED && (c * K + lane >= 1 || textbook)) ? 1u : 0u;
        }
        put_inj(c, 0, plus, minus);  // wave 0 runs chunk c in iteration c
        return true;
    };
    // Iteration `it`: compute wave w runs chunk it - w*D; its lane l at step q
    // reads column (it - w*D)*K + q - l (codes of columns outside the pair are
    // stale, masked to a table row; those steps keep their state).
    auto produce = [&](int it) {
        for (int w = 0; w < wa; ++w) {
            const int c = it - w * kD;
            if (c < 0 || c >= nch) continue;
            if (w > 0) {
                const int2 v = sh.cap[w - 1][(2 * c + 1 + word_of) & 7];
                put_inj(it, w, ((uint32_t)v.x >> bit_of) & 1u, ((uint32_t)v.y >> bit_of) & 1u);
            }
            const uint32_t *cp = sh.aw + ((c * K - lane) & (AW - 1));
            const int *pq = sh.peq[w] + lane;
            int4 *d = &sh.eqb[it & 1][w][0][lane];
            // All codes, then all table reads, then the stores: the table
            // reads issue back to back instead of each group waiting out two
            // dependent LDS round trips.
            uint32_t code[K];
#pragma unroll
            for (int q = 0; q < K; ++q) code[q] = cp[q];
            int e[K];
#pragma unroll
            for (int q = 0; q < K; ++q) e[q] = pq[code[q]];
#pragma unroll
            for (int gq = 0; gq < K / 4; ++gq) d[gq * 64] = make_int4(e[4 * gq], e[4 * gq + 1], e[4 * gq + 2], e[4 * gq + 3]);
        }
    };
    // The last compute wave's chunk c, to HBM for the strip below.
    auto publish = [&](int c) {
        if (lane < 2 * NP) {
            const int2 v = sh.cap[W - 1][(2 * c + lane / NP) & 7];
            __hip_atomic_store(bnext + 2 * c * NP + lane, tag | (uint32_t)((lane % NP) ? v.y : v.x), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    };

    __syncthreads();  // match-mask tables built
    uint32_t code_next = 0u;  // stager: codes of chunk j + 2, loaded in iteration j
    if (stager) {
        put_code(0, load_code(0));
        if (1 < nch) code_next = load_code(1);
        produce(0);
        if (!fill_top(0, load_top(0)) && lane == 0) sh.abort_at = -1;
    }
    __syncthreads();

    BpState st;
    st.pv = 0xffffffffu;  // ED: column 0 rises by 1 per row; LCS: V = all ones
    // Rows without a symbol hand the boundary above them down: no match, and
    // for ED no vertical difference either (the boundary rises by 1 a column).
    if (ED && row0 < pad) st.pv = pad - row0 >= 32 ? 0u : 0xffffffffu << (int)(pad - row0);
    st.mv = 0u;
    st.ph = 0;
    st.mh = 0;

    bool aborted = sh.abort_at <= -1;
    for (int j = 0; j < total && !aborted; ++j) {
        if (stager) {
            // (Here rather than in the compute wave, whose next chunk would
            // otherwise wait for the stores to complete.)
            const int cl = j - 1 - (wa - 1) * kD;
            if (has_next && cl >= 0 && cl < nch) publish(cl);
            if (j + 1 < nch) put_code(j + 1, code_next);
            if (j + 2 < nch) code_next = load_code(j + 2);
            const uint64_t top = (j + 1 < nch) ? load_top(j + 1) : tag;
            if (j + 1 < total) produce(j + 1);
            if (j + 1 < nch && !fill_top(j + 1, top) && lane == 0) sh.abort_at = j;
        } else {
            const int cj = j - wave * kD;
            if (cj >= 0 && cj < nch && active) {
                const int s0 = cj * K;
                const bool steady = (s0 >= 63) && (s0 + K - 1 <= n1 - 1);
                const int4 *eqw = &sh.eqb[j & 1][wave][0][0];
                const int2 *inj = sh.injb[j & 1][wave];
                // (In the dummy, lanes 62 and 63 of different waves overlap:
                // nobody reads it.)
                int2 *cap = lane == 63 ? &sh.cap[wave][(2 * cj) & 7] : &sh.dummy[lane];
                if (steady)
                    bs_chunk<P, K, false>(st, s0, lane, n1, inj, cap, eqw);
                else
                    bs_chunk<P, K, true>(st, s0, lane, n1, inj, cap, eqw);
            }
        }
        __syncthreads();
        aborted = sh.abort_at <= j;
    }

    if (aborted) {
        if (threadIdx.x == 0) atomicOr(&ka.res[pair].status, 1);
        // Placeholders release the strip below.
        if (stager && has_next)
            for (int k = lane; k < 2 * nch * NP; k += 64)
                __hip_atomic_store(bnext + k, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    if (stager && has_next) publish(nch - 1);

    if (active) {
        int v;
        if (P == WFK_ED)
            v = __builtin_popcount(st.pv & rowmask) - __builtin_popcount(st.mv & rowmask);
        else
            v = __builtin_popcount(~st.pv & rowmask);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (P == WFK_ED && g == 0 && wave == 0) v += textbook ? n1 : n1 - 1;  // D(0, n1)
        if (lane == 0) atomicAdd(&ka.res[pair].last, v);
        if (pd.col_off >= 0) {
            uint32_t *cw = ka.colw + 2 * (pd.col_off + ((int64_t)g * W + wave) * 64 + lane);
            cw[0] = st.pv;
            cw[1] = st.mv;
        }
    }
}

// ---------------------------------------------------------------------------
// Split pairs: the score from the two halves' last-column words.
//
// The parts meet along a staircase (staged engine; otherwise a straight column):
// strip g of the forward half ends at column c_g, c falling with g by the lag of
// a strip, so that both halves' strip chains end together.  From (0, c_0) the
// staircase goes down strip 0, left along its bottom row to c_1, down strip 1 and
// so on to (n2, c_{G-1}).  The score is the smallest (ED) or largest (LCS) sum
// F + R over its nodes: an alignment leaves the forward half's region at one.
// A step down row r changes F by d_r = Pv_r - Mv_r (ED) or 1 - V_r (LCS) of the
// forward half's last column, and R by -d' of the reverse half's row for r (row
// n2 - 1 - r, behind `pad` rows without a symbol); a step left over column x
// changes F by minus the horizontal difference that the strip handed down
// there, and R by the reverse half's.  At the start F = f0 and R = r0 + the sum
// of all of R's differences.  32 steps a thread and turn, one workgroup a pair
// (10 us for 65536 rows).  Against a straight column: see bitpar_cuts.
// ---------------------------------------------------------------------------

// Column-split SW pair.  The table is cut along a staircase: strip g of 512
// rows (a row of cells from y_g + 1 to y_{g+1}) at column c_g, c falling with g,
// so that the strips of the left part and of the reversed right part, each of
// which starts a strip lag after the one before, all end together.  job holds
// H left of the cut; f0 the cells right of it from a zero boundary (its
// bottom-right cell: the best local alignment into the corner that starts
// right of the cut); rev, for a node (y, x) on or right of the cut, the best
// path weight F from it to the corner, as E = F + 2 ((n2 - y) + (n1 - x)).
//
// An alignment into the corner that starts left of the cut leaves the left
// part at a node of the staircase: (y, c_g) inside strip g, or (y_{g+1}, x)
// with c_{g+1} <= x <= c_g on the row between strips g and g+1.  So the corner
// is the largest of f0's cell and H + F over those nodes, H from job's last
// columns and bottom rows, E from rev's (rev's strips end where job's begin: its
// first one is filled up with `pad` rows without a symbol).  H on row 0 and
// column 0, E on row n2 and column n1 are 0.  The running maximum likewise: the
// parts' own maxima, or H plus the best path from a node to any cell right of
// the cut, C from the clamped reversed part.  Without f0, the alignments that
// start right of the cut are the largest F of rev, and those that lie right of
// it the largest C of crev.
//
// n1 + n2 nodes at most, over `gridDim.y` workgroups; the results by atomics
// (the reset kernel clears res, and SW cells are >= 0).
__global__ __launch_bounds__(1024) void wf_sw_combine(const WfSplitDev *splits, const uint32_t *colw,
                                                      const WfCutDev *cuts, const uint64_t *bnd, WfResultDev *res)
{
    const WfSplitDev sp = splits[blockIdx.x];
    const int n1 = sp.r0, n2 = sp.n2, S = sp.strip;
    const int G = (n2 + S - 1) / S;
    const bool mx = sp.crev >= 0;
    const int *h = reinterpret_cast<const int *>(colw) + 2 * sp.fwd_off;
    const int *e = reinterpret_cast<const int *>(colw) + 2 * sp.rev_off;
    const int *c = reinterpret_cast<const int *>(colw) + 2 * sp.crev_off;
    const WfCutDev *fc = cuts + sp.cut, *rc = cuts + sp.rcut, *cc = cuts + sp.ccut;
    int best = INT_MIN, bestm = 0;
    // (y, c_g) inside the strips, and the corner strip's end.
    for (int y = blockIdx.y * blockDim.x + threadIdx.x; y <= n2; y += gridDim.y * blockDim.x) {
        if (y > 0 && y < n2 && y % S == 0) continue;
        const int g = y > 0 ? (y - 1) / S : 0;
        const int cg = fc[g].n, dg = n1 - cg;
        const int i = n2 - y;
        const int hv = (y > 0 && cg > 0) ? h[y - 1] : 0;
        const bool right = i > 0 && dg > 0;
        const int ev = right ? e[i + sp.pad - 1] : 0;
        best = max(best, hv + ev - 2 * (i + dg));
        if (mx) bestm = max(bestm, hv + (right ? c[i + sp.pad - 1] : 0));
    }
    // (y_{g+1}, x) between the strips.
    for (int g = blockIdx.y; g + 1 < G; g += gridDim.y) {
        const int x0 = fc[g + 1].n, x1 = fc[g].n;
        const int i = n2 - (g + 1) * S;
        const uint64_t *hb = bnd + fc[g].bnd;                           // column x at word x - 1
        const uint64_t *eb = bnd + rc[G - 2 - g].bnd;                   // column x at word n1 - x - 1
        const uint64_t *cb = mx ? bnd + cc[G - 2 - g].bnd : nullptr;
        for (int x = x0 + threadIdx.x; x <= x1; x += blockDim.x) {
            const int j = n1 - x;
            const int hv = x > 0 ? (int)(uint32_t)hb[x - 1] : 0;
            const int ev = j > 0 ? (int)(uint32_t)eb[j - 1] : 0;
            best = max(best, hv + ev - 2 * (i + j));
            if (mx) bestm = max(bestm, hv + (j > 0 ? (int)(uint32_t)cb[j - 1] : 0));
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        best = max(best, __shfl_xor(best, off));
        bestm = max(bestm, __shfl_xor(bestm, off));
    }
    __shared__ int wb[16], wm[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        wb[wv] = best;
        wm[wv] = bestm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = wb[0], m = wm[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
            b = max(b, wb[k]);
            m = max(m, wm[k]);
        }
        WfResultDev &r = res[sp.job];
        atomicMax(&r.last, max(b, sp.f0 >= 0 ? res[sp.f0].last : res[sp.rev].maxs));
        int status = res[sp.rev].status | (sp.f0 >= 0 ? res[sp.f0].status : 0);
        if (mx) {
            atomicMax(&r.maxs, max(m, res[sp.f0 >= 0 ? sp.f0 : sp.crev].maxs));
            status |= res[sp.crev].status;
        }
        if (status) atomicOr(&r.status, status);
    }
}

// 32 steps of a strip's bottom row from column x (0-based) on, plane `h`: bit 31
// is column x.
__device__ __forceinline__ uint32_t bs_row_bits(const uint64_t *row, int n, int np, int x, int h)
{
    const int s = x + 63, w = s >> 5, words = 2 * ((n + 126) / 64);
    const uint32_t a = (uint32_t)row[w * np + h], b = w + 1 < words ? (uint32_t)row[(w + 1) * np + h] : 0u;
    return (uint32_t)(((((uint64_t)a << 32) | b) << (s & 31)) >> 32);
}

__global__ __launch_bounds__(1024) void wf_bitpar_combine(const WfSplitDev *splits, const uint32_t *colw,
                                                          const WfCutDev *cuts, const uint64_t *bnd, WfResultDev *res)
{
    const WfSplitDev sp = splits[blockIdx.x];
    const bool ed = sp.prob == WFK_ED;
    const int n2 = sp.n2;
    const int nw = (n2 + 31) >> 5;
    const int nwr = (n2 + sp.pad + 31) >> 5;
    const uint32_t *fw = colw + 2 * sp.fwd_off;
    const uint32_t *rw = colw + 2 * sp.rev_off;
    // Bits of reverse rows [base, base + 32) (base > -32), bit k = row
    // base + k; rows below 0 read as 0.  h: 0 Pv/V, 1 Mv.
    auto rev_bits = [&](int base, int h) -> uint32_t {
        const int lo = base >= 0 ? (base >> 5) : -1;
        const int sh = base - 32 * lo;
        const uint32_t wl = lo >= 0 ? rw[2 * lo + h] : 0u;
        const uint32_t wh = (lo + 1 < nwr) ? rw[2 * (lo + 1) + h] : 0u;
        return (uint32_t)((((uint64_t)wh << 32) | wl) >> sh);
    };
    // The staircase in words: per strip its rows, then the row below it.
    const int G = sp.strip > 0 ? (n2 + sp.strip - 1) / sp.strip : 1;
    const int ws = sp.strip > 0 ? sp.strip >> 5 : nw;
    const WfCutDev *fc = cuts + sp.cut, *rc = cuts + sp.rcut;
    const int hs = G > 1 ? (fc[0].n - fc[1].n + 31) >> 5 : 0;  // c falls by the same everywhere
    const int items = G * (ws + hs);
    const int tid = threadIdx.x;
    const int per = (items + 1023) >> 10;
    const int w0 = min(items, tid * per), w1 = min(items, w0 + per);
    int run = 0, best = 0, rtot = 0;
    for (int it = w0; it < w1; ++it) {
        const int g = it / (ws + hs), t = it - g * (ws + hs);
        // fa, fb: F rises, falls; ra, rb: R falls, rises (bit k: step k).
        uint32_t fa, fb, ra, rb;
        int nk;
        if (t < ws) {
            const int w = g * ws + t;
            nk = min(32, n2 - 32 * w);
            if (nk <= 0) continue;
            const uint32_t m = nk >= 32 ? 0xffffffffu : ((1u << nk) - 1u);
            const int base = sp.pad + n2 - 32 * w - 32;  // reverse rows of original rows 32w+31 .. 32w
            if (ed) {
                fa = fw[2 * w] & m;
                fb = fw[2 * w + 1] & m;
                ra = __builtin_bitreverse32(rev_bits(base, 0)) & m;
                rb = __builtin_bitreverse32(rev_bits(base, 1)) & m;
            } else {
                fa = ~fw[2 * w] & m;  // zeros of V: the LCS grows at that row
                fb = 0u;
                ra = __builtin_bitreverse32(~rev_bits(base, 0)) & m;
                rb = 0u;
            }
        } else {
            // Columns x .. x - nk + 1 (1-based), leftwards.
            if (g + 1 >= G) continue;
            const int x = fc[g].n - 32 * (t - ws);
            nk = min(32, x - fc[g + 1].n);
            if (nk <= 0) continue;
            const uint32_t m = nk >= 32 ? 0xffffffffu : ((1u << nk) - 1u);
            const uint64_t *f = bnd + fc[g].bnd, *r = bnd + rc[G - 2 - g].bnd;
            const int nf = fc[g].n, nr = rc[G - 2 - g].n, np = ed ? 2 : 1, xr = sp.cols - x;
            // F's columns x - nk .. x - 1 (0-based), the last of which is step 0;
            // the reverse half's from cols - x on, the first of which is.
            fb = bs_row_bits(f, nf, np, x - nk, 0) >> (32 - nk) & m;
            rb = __builtin_bitreverse32(bs_row_bits(r, nr, np, xr, 0)) & m;
            fa = ed ? bs_row_bits(f, nf, np, x - nk, 1) >> (32 - nk) & m : 0u;
            ra = ed ? __builtin_bitreverse32(bs_row_bits(r, nr, np, xr, 1)) & m : 0u;
        }
        rtot += __builtin_popcount(ra) - __builtin_popcount(rb);
        for (int k = 0; k < nk; ++k) {
            run += (int)((fa >> k) & 1u) - (int)((fb >> k) & 1u) - (int)((ra >> k) & 1u) + (int)((rb >> k) & 1u);
            best = ed ? min(best, run) : max(best, run);
        }
    }
    // Exclusive scan of the threads' sums (in word order) and the reductions.
    __shared__ int wsum[16], wbest[16], wrt[16];
    const int lane = tid & 63, wv = tid >> 6;
    int incl = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off);
        if (lane >= off) incl += t;
    }
    if (lane == 63) wsum[wv] = incl;
    int rt = rtot;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) rt += __shfl_xor(rt, off);
    if (lane == 0) wrt[wv] = rt;
    __syncthreads();
    int before = 0, rall = 0;
    for (int i = 0; i < 16; ++i) {
        if (i < wv) before += wsum[i];
        rall += wrt[i];
    }
    int cand = before + incl - run + best;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(cand, off);
        cand = ed ? min(cand, o) : max(cand, o);
    }
    if (lane == 0) wbest[wv] = cand;
    __syncthreads();
    if (tid == 0) {
        int b = wbest[0];
        for (int i = 1; i < 16; ++i) b = ed ? min(b, wbest[i]) : max(b, wbest[i]);
        res[sp.job].last = sp.f0 + sp.r0 + rall + b;
        res[sp.job].status |= res[sp.rev].status;
    }
}

template <int W>
__global__ __launch_bounds__(64 * (W + 1)) void wf_engine_bitpar_staged(WfKernelArgs ka)
{
    __shared__ BsShared<W> sh;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(*ka.epoch);
    for (int i = threadIdx.x; i < BsShared<W>::AW + BsShared<W>::K; i += blockDim.x) sh.aw[i] = 0;
    for (;;) {
        if (threadIdx.x == 0) {
            sh.task = ka.task_begin + atomicAdd(ka.counter, 1);
            sh.abort_at = 0x7fffffff;
        }
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sh.task);
        __syncthreads();
        if (t >= ka.task_end) break;
        const WfTaskDev td = ka.tasks[t];
        const WfPairDev pd = ka.pairs[td.pair];
        wfk::set_wave_priority(pd.prio);
        if (pd.prob == WFK_ED)
            bs_group<WFK_ED, W>(ka, pd, td.pair, td.group, sh, lane, wave, epoch);
        else
            bs_group<WFK_LCS, W>(ka, pd, td.pair, td.group, sh, lane, wave, epoch);
        __syncthreads();
    }
}

}  // namespace wfb

extern "C" hipError_t wf_launch_bitpar_combine(const WfSplitDev *splits, int nsplits, const uint32_t *colw,
                                               const WfCutDev *cuts, const uint64_t *bnd, WfResultDev *res,
                                               hipStream_t stream)
{
    if (nsplits <= 0) return hipSuccess;
    hipLaunchKernelGGL(wfb::wf_bitpar_combine, dim3(nsplits), dim3(1024), 0, stream, splits, colw, cuts, bnd, res);
    return hipGetLastError();
}

extern "C" hipError_t wf_launch_sw_combine(const WfSplitDev *splits, int nsplits, int blocks, const uint32_t *colw,
                                           const WfCutDev *cuts, const uint64_t *bnd, WfResultDev *res,
                                           hipStream_t stream)
{
    if (nsplits <= 0 || blocks <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wfb::wf_sw_combine, dim3(nsplits, blocks), dim3(1024), 0, stream, splits, colw, cuts, bnd, res);
    return hipGetLastError();
}

#define WF_BITPAR_STAGED(W_) \
    {WF_ENGINE_BITPAR_STAGED, 32, W_, 64, 64 * ((W_) + 1), reinterpret_cast<const void *>(&wfb::wf_engine_bitpar_staged<W_>)}

#define WF_BITPAR(W_, K_) \
    {WF_ENGINE_BITPAR, 32, W_, K_, 64 * (W_), reinterpret_cast<const void *>(&wfb::wf_engine_bitpar<W_, K_>)}

extern "C" const WfVariant wf_variants_bitpar[] = {WF_BITPAR(1, 64),        WF_BITPAR(2, 64),        WF_BITPAR(4, 64),
                                                   WF_BITPAR(1, 128),       WF_BITPAR(2, 128),       WF_BITPAR(4, 128),
                                                   WF_BITPAR_STAGED(1),     WF_BITPAR_STAGED(2)};
extern "C" const int wf_num_variants_bitpar = sizeof(wf_variants_bitpar) / sizeof(wf_variants_bitpar[0]);
