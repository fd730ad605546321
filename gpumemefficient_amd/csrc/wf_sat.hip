// wf_sat.hip -- single-pass summed-area table for gfx950.
//
//   T(y,x) = T(y,x-1) + T(y-1,x) + T(y,x) - T(y-1,x-1)   (SAT/GPU_Hyperlane_Share.cu:169)
//
// over the interior 1 <= y <= n2, 1 <= x <= n1, int32 wrapping mod 2^32.  The
// recurrence is a two-dimensional prefix sum: with p(y,x) the sum over
// 0 < x' <= x of row y's old values plus d(y) = T(y,0) - T(y-1,0),
//
//   T'(y,x) = T'(y-1,x) + p(y,x),     T'(0,x) = T(0,x),
//
// so it needs no wavefront: addition mod 2^32 is associative and every order
// gives the reference's bits.  Putting d(y) in place of the row's column-0
// value makes p a plain row prefix.
//
// Each workgroup takes one tile of 128 rows x 512 columns into registers
// (wave w rows 16w.., lane l columns 8l..8l+7), scans its rows (seven adds in
// a lane, six DPP adds across the wave) and columns, adds the rows' sums left
// of the tile and the finished row above it, and stores: every cell crosses
// HBM once each way.  The two carries travel as (launch epoch << 32 | value)
// words with relaxed device-scope atomics, as the strip boundaries do:
//
//   rows     every tile publishes its 128 row sums as soon as it has them;
//            a tile adds up those of the tiles to its left in its block of 64
//            tile columns.  No chain: a tile's sums do not wait for anybody.
//            A block's last tile publishes the sums of all columns up to its
//            own instead, which the next block's tiles add: a chain of one hop
//            per 32768 columns.  (With all tiles to the left read by each,
//            what is read grows with the square of the width and passes the
//            cells' traffic at 260 000 columns: 4M x 1024 30.3 ms against 6.8,
//            13M x 512 139 against 10.9.  Blocks of 32 or 128 tiles: 6.7, 7.9.)
//   columns  a tile's bottom row T'(y_end, x) needs the one of the tile above.
//            This chain has n2 / 128 hops of about 1.3 us, so a tile forms its own part
//            first and only adds the row above when it arrives, publishing
//            before it writes its cells.  The rows go round a ring, each turn
//            with a tag of its own (run_sat in wf_stencil_api.cpp).
//
// Tiles are claimed in row-major order from an atomic counter, so a tile only
// waits on tiles claimed before it.
//
// Bound: HBM, 8 bytes a cell (read and written once), once the table has more
// tiles than the chip has CUs; the chain of tile rows below that.  Measured
// (kernel time; before: the 64-row wavefront of wf_stencil.hip, bound by its
// chain of n2 / 64 waves): 32768 x 32768 6.4 -> 1.66 ms (5.2 TB/s; a copy of
// 4 GiB runs at 4.9), 8192 x 8192 0.124 ms, 1000 x 1000 0.025 ms.  Tiles of 64
// rows (two workgroups per CU) have twice the hops and lose at every size:
// 1.72 ms, 0.160 ms, 0.028 ms; 512 columns x 24000 rows 0.33 against 0.17 ms.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wf_cells.h"
#include "wf_device.h"

namespace wfsat {

using wfk::now_ticks;

constexpr int kRW = 16;    // rows of a wave
constexpr int kLC = 8;     // columns of a lane
constexpr int kW = 8;      // waves of a workgroup: two a SIMD, 256 VGPRs each, 128 of them the tile's cells
constexpr int kTR = WFS_SAT_TILE_ROWS, kTC = WFS_SAT_TILE_COLS, kTB = WFS_SAT_BLOCK_TILES;
static_assert(kTB % 16 == 0, "a block's tiles are read 16 at a time");
static_assert(kTR == kW * kRW && kTC == 64 * kLC, "waves stack down the tile, a wave spans its columns");

struct SatShared {
    int col[kW][kTC];   // a wave's column sums, then (col[0]) the row above the tile
    int rows[kW];       // sum of a wave's row carries
    int task;
};

template <int CTRL, int ROWMASK>
__device__ __forceinline__ int dpp_add(int v)
{
    return (int)((uint32_t)v + (uint32_t)__builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xf, false));
}

// Inclusive scan inside each row of 16 lanes (DPP row_shr), and over the wave
// (row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3).
__device__ __forceinline__ int scan16(int v)
{
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    return dpp_add<0x118, 0xf>(v);
}
__device__ __forceinline__ int scan64(int v)
{
    v = scan16(v);
    v = dpp_add<0x142, 0xa>(v);
    return dpp_add<0x143, 0xc>(v);
}

__device__ __forceinline__ uint64_t load_word(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_word(uint64_t *p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls the N loaded words w[k] = *at(k) until all carry the tag; false (and the
// words as they are) once the wait exceeds the limit.
template <int N, class At>
__device__ __forceinline__ bool wait_words(At &&at, uint32_t epoch, int64_t limit, uint64_t (&w)[N])
{
    int64_t t0 = 0;
    for (int spins = 0;; ++spins) {
        bool stale = false;
#pragma unroll
        for (int k = 0; k < N; ++k) stale = stale || (uint32_t)(w[k] >> 32) != epoch;
        if (__builtin_amdgcn_ballot_w64(stale) == 0) return true;
        const int64_t t = now_ticks();
        if (spins == 0)
            t0 = t;
        else if (t - t0 > limit)
            return false;
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int k = 0; k < N; ++k)
            if ((uint32_t)(w[k] >> 32) != epoch) w[k] = load_word(at(k));
    }
}

__device__ __forceinline__ void sat_tile(const WfSatArgs &a, int tr, int tc, SatShared &sh, int lane, int wave,
                                         uint32_t epoch)
{
    const int n1 = a.n1;
    const uint64_t tag = (uint64_t)epoch << 32;
    const int yw = 1 + tr * kTR + wave * kRW;  // the wave's first row
    const int nrows = max(0, min(kRW, a.n2 + 1 - yw));
    const int c = tc * kTC + lane * kLC;      // the lane's first column
    const bool edge = (tc + 1) * kTC - 1 > n1;
    // Rows and tags of the ring of bottom rows: the tile's, and that of the tile
    // above.  Here, and not on the way down the tile rows, which the division
    // would lengthen (500 columns x 70000 rows 0.47 -> 0.55 ms; here 0.45).
    int rout = tr;
    uint32_t tout = epoch - (uint32_t)(a.tags - 1);
    if (tr >= a.ring) {
        rout = tr % a.ring;
        tout += (uint32_t)(tr / a.ring);
    }
    int rin = rout > 0 ? rout - 1 : a.ring - 1;
    uint32_t tin = rout > 0 ? tout : tout - 1u;
    asm("" : "+s"(rout), "+s"(tout), "+s"(rin), "+s"(tin));

    // The wave's rows as a buffer resource (fields through readfirstlane, so
    // that it sits in SGPRs): loads past the last row read zeros, and a vector
    // that holds no column <= n1 gets an offset past the end, on loads and
    // stores, so neither needs a branch (kOut plus 15 pitches stays out of range
    // and does not wrap: 16 rows of the largest pitch are below 2^30 bytes).
    const uint64_t base = reinterpret_cast<uint64_t>(a.t + (int64_t)yw * a.ld);
    const uint32_t blo = __builtin_amdgcn_readfirstlane((uint32_t)base);
    const uint32_t bhi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
    const int bytes = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)nrows * (uint64_t)a.ld * 4u));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void *>(((uint64_t)bhi << 32) | blo), 0, bytes, 0x00020000);
    constexpr uint32_t kOut = 0x80000000u;
    const uint32_t pitch = (uint32_t)(a.ld * 4);
    uint32_t voff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) voff[h] = c + 4 * h <= n1 ? (uint32_t)(c + 4 * h) * 4u : kOut;

    int v[kRW][kLC];
#pragma unroll
    for (int r = 0; r < kRW; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int4 q = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[h] + r * pitch, 0, 0));
            v[r][4 * h + 0] = q.x;
            v[r][4 * h + 1] = q.y;
            v[r][4 * h + 2] = q.z;
            v[r][4 * h + 3] = q.w;
        }
    if (edge) {
#pragma unroll
        for (int r = 0; r < kRW; ++r)
#pragma unroll
            for (int k = 0; k < kLC; ++k) v[r][k] = c + k <= n1 ? v[r][k] : 0;
    }
    if (tc == 0) {
        // Column 0 becomes its difference to the row above.
        const int above = nrows > 0 ? __hip_atomic_load(a.t + (int64_t)(yw - 1) * a.ld, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP)
                                    : 0;
        if (lane == 0) {
#pragma unroll
            for (int r = kRW - 1; r > 0; --r) v[r][0] = (int)((uint32_t)v[r][0] - (uint32_t)v[r - 1][0]);
            v[0][0] = (int)((uint32_t)v[0][0] - (uint32_t)above);
        }
    }

    // Row prefixes; lane r keeps row r's sum.
    int rowsum = 0;
#pragma unroll
    for (int r = 0; r < kRW; ++r) {
#pragma unroll
        for (int k = 1; k < kLC; ++k) v[r][k] = (int)((uint32_t)v[r][k] + (uint32_t)v[r][k - 1]);
        const int incl = scan64(v[r][kLC - 1]);
        const int excl = (int)((uint32_t)incl - (uint32_t)v[r][kLC - 1]);
#pragma unroll
        for (int k = 0; k < kLC; ++k) v[r][k] = (int)((uint32_t)v[r][k] + (uint32_t)excl);
        const int sum = __builtin_amdgcn_readlane(incl, 63);
        rowsum = lane == r ? sum : rowsum;
    }
    const int blk = tc / kTB;  // the tile's block of tile columns
    const bool ends_blk = tc % kTB == kTB - 1;
    if (tc + 1 < a.ntc && !ends_blk && lane < kRW)
        store_word(a.rowsum + ((int64_t)tr * (a.ntc - 1) + tc) * kTR + wave * kRW + lane, tag | (uint32_t)rowsum);

    // Column prefixes of the wave's rows.
#pragma unroll
    for (int r = 1; r < kRW; ++r)
#pragma unroll
        for (int k = 0; k < kLC; ++k) v[r][k] = (int)((uint32_t)v[r][k] + (uint32_t)v[r - 1][k]);
    {
        int4 *d = reinterpret_cast<int4 *>(&sh.col[wave][lane * kLC]);
        d[0] = make_int4(v[kRW - 1][0], v[kRW - 1][1], v[kRW - 1][2], v[kRW - 1][3]);
        d[1] = make_int4(v[kRW - 1][4], v[kRW - 1][5], v[kRW - 1][6], v[kRW - 1][7]);
    }

    // Row carries: lane l adds up row l % 16 over the tiles l / 16 mod 4 of its
    // block left of this one, and the blocks before; carry: the inclusive prefix
    // over the wave's rows.
    uint32_t carry = 0;
    if (tc > 0) {
        const uint64_t *bp = a.blksum + ((int64_t)tr * (a.nblk - 1) + blk - 1) * kTR + wave * kRW + (lane & 15);
        uint64_t wb[1] = {blk > 0 ? load_word(bp) : tag};
        const uint64_t *rp = a.rowsum + (int64_t)tr * (a.ntc - 1) * kTR + wave * kRW + (lane & 15);
        for (int j = blk * kTB; j < tc; j += 16) {
            uint64_t w[4];
            // Tiles past the last one left of this tile: its own first
            // predecessor again, added as zero.
            const uint64_t *q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = rp + (int64_t)min(j + 4 * k + (lane >> 4), tc - 1) * kTR;
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = load_word(q[k]);
            if (!wait_words([&](int k) { return q[k]; }, epoch, a.timeout_ticks, w) && lane == 0)
                atomicOr(&a.res->status, 1);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                carry += (j + 4 * k + (lane >> 4) < tc) ? (uint32_t)w[k] : 0u;
        }
        if (!wait_words([&](int) { return bp; }, epoch, a.timeout_ticks, wb) && lane == 0) atomicOr(&a.res->status, 1);
        carry += lane < kRW ? (uint32_t)wb[0] : 0u;
        carry += (uint32_t)__shfl_xor((int)carry, 16);
        carry += (uint32_t)__shfl_xor((int)carry, 32);
    }
    if (ends_blk && tc + 1 < a.ntc && lane < kRW)
        store_word(a.blksum + ((int64_t)tr * (a.nblk - 1) + blk) * kTR + wave * kRW + lane, tag | (carry + (uint32_t)rowsum));
    carry = (uint32_t)scan16((int)carry);
    if (lane == kRW - 1) sh.rows[wave] = (int)carry;
    __syncthreads();

    // What the waves above add to each column of this wave's rows.
    uint32_t add[kLC];
    {
        uint32_t rows = 0;
#pragma unroll
        for (int k = 0; k < kLC; ++k) add[k] = 0;
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            if (w < wave) {
                const int4 *s = reinterpret_cast<const int4 *>(&sh.col[w][lane * kLC]);
                const int4 s0 = s[0], s1 = s[1];
                add[0] += (uint32_t)s0.x;
                add[1] += (uint32_t)s0.y;
                add[2] += (uint32_t)s0.z;
                add[3] += (uint32_t)s0.w;
                add[4] += (uint32_t)s1.x;
                add[5] += (uint32_t)s1.y;
                add[6] += (uint32_t)s1.z;
                add[7] += (uint32_t)s1.w;
                rows += (uint32_t)sh.rows[w];
            }
        }
#pragma unroll
        for (int k = 0; k < kLC; ++k) add[k] += rows;
    }
    __syncthreads();
    // The last wave takes the finished row above, publishes the tile's bottom
    // row and hands the row above to the other waves.
    if (wave == kW - 1) {
        uint32_t top[kLC];
        if (tr == 0) {
#pragma unroll
            for (int k = 0; k < kLC; ++k) top[k] = c + k <= n1 ? (uint32_t)a.t[c + k] : 0u;
        } else {
            const uint64_t *q = a.bottom + ((int64_t)rin * a.ntc + tc) * kTC + lane;
            uint64_t w[kLC];
#pragma unroll
            for (int k = 0; k < kLC; ++k) w[k] = load_word(q + 64 * k);
            if (!wait_words([&](int k) { return q + 64 * k; }, tin, a.timeout_ticks, w) && lane == 0)
                atomicOr(&a.res->status, 1);
#pragma unroll
            for (int k = 0; k < kLC; ++k) top[k] = (uint32_t)w[k];
        }
        if (tr + 1 < a.ntr) {
            const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)carry, kRW - 1);
            uint64_t *d = a.bottom + ((int64_t)rout * a.ntc + tc) * kTC + lane;
            const uint64_t btag = (uint64_t)tout << 32;
#pragma unroll
            for (int k = 0; k < kLC; ++k)
                store_word(d + 64 * k, btag | (uint32_t)(top[k] + add[k] + (uint32_t)v[kRW - 1][k] + all));
        }
        int4 *d = reinterpret_cast<int4 *>(&sh.col[0][lane * kLC]);
        d[0] = make_int4((int)top[0], (int)top[1], (int)top[2], (int)top[3]);
        d[1] = make_int4((int)top[4], (int)top[5], (int)top[6], (int)top[7]);
    }
    __syncthreads();
    {
        const int4 *s = reinterpret_cast<const int4 *>(&sh.col[0][lane * kLC]);
        const int4 s0 = s[0], s1 = s[1];
        add[0] += (uint32_t)s0.x;
        add[1] += (uint32_t)s0.y;
        add[2] += (uint32_t)s0.z;
        add[3] += (uint32_t)s0.w;
        add[4] += (uint32_t)s1.x;
        add[5] += (uint32_t)s1.y;
        add[6] += (uint32_t)s1.z;
        add[7] += (uint32_t)s1.w;
    }
    // Vectors that lie within the columns 1..n1 go out whole; those that reach
    // past them (the table's boundary columns, which are not written) cell by
    // cell.
    bool whole[2];
    uint32_t soff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        whole[h] = c + 4 * h >= 1 && c + 4 * h + 3 <= n1;
        soff[h] = whole[h] ? voff[h] : kOut;
    }
#pragma unroll
    for (int r = 0; r < kRW; ++r) {
        const uint32_t rc = (uint32_t)__builtin_amdgcn_readlane((int)carry, r);
        uint32_t o[kLC];
#pragma unroll
        for (int k = 0; k < kLC; ++k) o[k] = (uint32_t)v[r][k] + add[k] + rc;
        typedef __attribute__((ext_vector_type(4))) uint32_t u4;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const u4 q = {o[4 * h], o[4 * h + 1], o[4 * h + 2], o[4 * h + 3]};
            __builtin_amdgcn_raw_buffer_store_b128(q, rs, soff[h] + r * pitch, 0, 0);
        }
        if (edge || tc == 0) {
            // (Three cells: column 0's vector starts at column 1.)
            const int first = c == 0 ? 1 : 0;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int x = c + 4 * h + k + (h == 0 ? first : 0);
                    const bool cell = !whole[h] && x <= n1;
                    const uint32_t q = h == 0 && first ? o[k + 1] : o[4 * h + k];
                    __builtin_amdgcn_raw_buffer_store_b32(q, rs, (cell ? (uint32_t)x * 4u : kOut) + r * pitch, 0, 0);
                }
        }
    }
}

__global__ __launch_bounds__(64 * kW) void wf_sat_kernel(WfSatArgs a)
{
    __shared__ __attribute__((aligned(16))) SatShared sh;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(*a.epoch);
    const int ntiles = a.ntr * a.ntc;
    for (;;) {
        if (threadIdx.x == 0) sh.task = atomicAdd(a.counter, 1);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sh.task);
        if (t >= ntiles) break;
        sat_tile(a, t / a.ntc, t % a.ntc, sh, lane, wave, epoch);
        __syncthreads();
    }
}

}  // namespace wfsat

extern "C" int wf_sat_resident(int cus)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wfsat::wf_sat_kernel, 64 * wfsat::kW, 0) != hipSuccess ||
        per_cu < 1) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    return per_cu * cus;
}

extern "C" hipError_t wf_launch_sat(int grid, const WfSatArgs *a, hipStream_t stream)
{
    if (grid <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wfsat::wf_sat_kernel, dim3(grid), dim3(64 * wfsat::kW), 0, stream, *a);
    return hipGetLastError();
}
