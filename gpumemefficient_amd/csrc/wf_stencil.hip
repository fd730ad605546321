// wf_stencil.hip -- gfx950 wavefront engine for the reference's 2D-SOR
// program: an in-place sweep over a whole int32 table whose cell depends on
// its left and upper neighbours after they were updated.  (The reference's
// other user of the hyperlane schedule, the summed-area table, is a prefix
// sum and needs no wavefront: wf_sat.hip.)
//
//   SOR  one Gauss-Seidel sweep of the 5-point stencil:
//          T(y,x) = (T(y,x-1) + T(y-1,x) + T(y,x) + T(y,x+1) + T(y+1,x)) / 5
//        with left and up already updated and right and down not
//        (2D-SOR/nested_loop/GPU_Hyperlane_Share.cu:169, :197, :233); C
//        division truncating toward zero.
//
// The table has the reference's layout (SAT/GPU_Hyperlane_Share.cu:255-263):
// rows 0 .. n2+1 of pitch ld >= n1+3; row 0, row n2+1 and columns 0, n1+1,
// n1+2 are boundary values that are read, never written; the interior
// 1 <= y <= n2, 1 <= x <= n1 is updated.  Any order that visits each cell
// after its left and upper neighbours and before its right and lower ones
// gives the row-major sequential sweep's result; the reference's hyperlane
// tiles are one such order and so is this engine's.
//
// Geometry.  A strip of 64 rows is swept left to right by one workgroup of
// three waves.  Lane l of the compute wave owns one row and updates column
// x = s + 1 - l at step s (the systolic front of the alignment engines).  The
// updated left value stays in a VGPR; the updated upper value comes from lane
// l-1 through one DPP wave_shr:1; and since lane l+1 is one column behind, the
// value below, T(y+1,x), is the lane below's own right neighbour of the same
// step: one DPP wave_shl:1.
//
// The rows' old values sit in an LDS window in *step* order: column x of row
// l at slot x - 1 + l, so that the slot is the step and the same for every
// lane.  A lane reads the old values of four steps with one ds_read_b128 and
// writes the four new ones over them with one ds_write_b128, and when a chunk
// of 16 steps is done, its slots are done in all 64 rows.
//
// The mover wave carries the window: it loads the skewed 16-byte vectors of
// the rows (4-byte aligned in HBM) kAhead chunks ahead, stages them in LDS and
// stores finished chunks back.  The boundary wave stages the row above for
// lane 0 and publishes the strip's bottom row for the next strip, through HBM
// as (launch epoch << 32 | value) words written and polled at device scope, as
// the alignment engines do; the rows go round a ring, each turn with a tag of
// its own (run_device in wf_stencil_api.cpp).  The compute wave touches LDS only: about 12 issue
// slots a step, of which the division's v_mul_hi is four.  The three meet at a
// barrier per chunk.  Strips are claimed in order from an atomic counter, so a
// strip only waits on one that a running workgroup holds.
//
// Bound: the chain of n2 / 64 strips, each about 155 steps (80 of them the
// lanes' skew and a chunk, the rest the row's way through memory) behind the
// one above, and n1 steps of 26 ns; from about 16384 x 16384 on also the memory
// traffic of 64-byte row segments.  Measured (kernel time; before: 256-row strips,
// the window in column order, staging by the compute waves themselves): 9001 x
// 7043 2.01 -> 0.71 ms, 1000 x 1000 0.21 -> 0.10, 16384 x 16384 3.10 -> 1.89,
// 32768 x 32768 6.65 -> 4.5.  Two compute waves a strip (128 rows): 0.69 ms at
// 9001 x 7043 and 5.3 at 32768 x 32768.  Chunks in flight: 4 / 6 / 8 4.8 / 4.4 /
// 4.6 ms at 32768 x 32768, no difference at 9001 x 7043.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "wf_cells.h"
#include "wf_device.h"

namespace wfs {

using wfk::kDppWaveShr1;
using wfk::now_ticks;

constexpr int kDppWaveShl1 = 0x130;     // DPP_CTRL wave_shl:1 (GFX9 family)
constexpr int kRows = 64;               // rows of a strip
constexpr int kK = 16;                  // steps per chunk
constexpr int kAhead = 6;               // chunks of loads in flight (registers of the mover)
constexpr int kTW = 128;                // window slots per row (8 chunks)
constexpr int kTS = kTW + 4;            // row stride: 16 lanes' 16-byte accesses fall in distinct banks
constexpr uint32_t kOut = 0xf0000000u;  // buffer offset out of range, also 64 bytes x chunks further

struct StShared {
    __attribute__((aligned(16))) int win[kRows * kTS];
    // bot: the row below the strip, its column x at slot x + 62 (lane 63's
    // step); top: the row above, its column x at slot x + 62.
    __attribute__((aligned(16))) int bot[kTW];
    __attribute__((aligned(16))) int top[kTW];
    int task;
};

// Barrier between the waves of the workgroup that orders their LDS accesses
// only: global loads issued before it stay in flight (a __syncthreads would
// wait for them, and for the flushes' stores, at every chunk).
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// `bytes` bytes from p as a buffer resource: reads past the end give zeros,
// writes are dropped.  Offsets are 32-bit: 65 rows of the pitch must fit
// (checked by the host).  The descriptor's fields pass through readfirstlane:
// a descriptor the compiler cannot prove uniform lives in VGPRs, and every
// access then becomes a waterfall loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void *p, int64_t bytes)
{
    const uint64_t base = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
    const int size = __builtin_amdgcn_readfirstlane((int)(uint32_t)bytes);
    // Third descriptor dword of an untyped buffer on the gfx9 family.
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(((uint64_t)hi << 32) | lo), 0, size, 0x00020000);
}

// Cache policy of accesses that other workgroups of the launch see or make:
// device scope (bit 4: sc1), as a relaxed agent-scope atomic has.
constexpr int kCoherent = 16;

// One chunk of a wave's window in flight between its global loads and its LDS
// stores: slots 4k..4k+3 of row row(i) per lane, and (lanes 0..3) of the row
// below.
struct Stage {
    int4 v[4];
    int4 b;
};

// Lane's vectors: four lanes cover a row's 16 slots; the rows of 16
// consecutive lanes are 4 apart, so that their 16-byte LDS accesses fall in
// distinct banks.
__device__ __forceinline__ int vec_row(int i, int lane) { return 16 * i + 4 * ((lane >> 2) & 3) + (lane >> 4); }

// Slot q of row r holds column q + 1 - r: byte offset of a vector in the
// wave's rows.
__device__ __forceinline__ uint32_t vec_off(int r, int slot, int64_t ld)
{
    return (uint32_t)(r * (ld - 1) * 4) + (uint32_t)(slot + 1) * 4u;
}

// Four steps of a lane: old values of its row (self of steps 0..3, and the
// next one), lane 0's upper and lane 63's lower neighbours.  HEAD: x0 is the
// lane's column at step 0; columns left of 1 keep the left boundary `h`.
// Columns right of n1 and rows below n2 need no mask: nothing inside the table
// depends on them and the movers do not store them.
template <bool HEAD>
__device__ __forceinline__ int4 sor_group(int &h, int4 self, int next, int4 up4, int4 down4, int x0)
{
    const int sv[5] = {self.x, self.y, self.z, self.w, next};
    const int uv[4] = {up4.x, up4.y, up4.z, up4.w};
    const int dv[4] = {down4.x, down4.y, down4.z, down4.w};
    int out[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int down = __builtin_amdgcn_update_dpp(dv[u], sv[u + 1], kDppWaveShl1, 0xf, 0xf, false);
        const uint32_t old = (uint32_t)sv[u] + (uint32_t)sv[u + 1] + (uint32_t)down;
        const int up = __builtin_amdgcn_update_dpp(uv[u], h, kDppWaveShr1, 0xf, 0xf, false);
        const int nv = (int)((uint32_t)h + (uint32_t)up + old) / 5;
        h = (HEAD && x0 + u < 1) ? h : nv;
        out[u] = h;
    }
    return make_int4(out[0], out[1], out[2], out[3]);
}

__device__ __forceinline__ void sor_strip(const WfStencilArgs &a, int g, StShared &sh, int lane, int wave,
                                          uint32_t epoch)
{
    const int n1 = a.n1;
    const int y0 = 1 + g * kRows;  // the strip's first row
    // Lane 63 updates column n1 at step n1 + 62; whole turns of the mover's
    // loop.  Every wave passes a barrier before chunk 0 and one after each
    // chunk; none leaves early: when a dependency wait is given up the launch
    // is marked, and the strip runs on without waiting.
    const int nch = (n1 + 63 + kK * kAhead - 1) / (kK * kAhead) * kAhead;
    const bool has_prev = g > 0;
    const bool has_next = g + 1 < a.nstrips;
    // Rows and tags of the ring of bottom rows: the strip's, the strip above's.
    int rout = g;
    uint32_t tout = epoch - (uint32_t)(a.tags - 1);
    if (g >= a.ring) {
        rout = g % a.ring;
        tout += (uint32_t)(g / a.ring);
    }
    const int rin = rout > 0 ? rout - 1 : a.ring - 1;
    const uint32_t tin = rout > 0 ? tout : tout - 1u;
    const uint64_t *bprev = a.bnd + (int64_t)rin * (n1 + 1);
    uint64_t *bnext = a.bnd + (int64_t)rout * (n1 + 1);
    int *win = sh.win;

    if (wave == 0) {
        // ------------------------------------------------------ compute wave
        lds_barrier();
        int h = y0 + lane <= a.n2 ? a.t[(int64_t)(y0 + lane) * a.ld] : 0;  // column 0: the left boundary
        int *wl = win + lane * kTS;
        auto at = [](const int *p) __attribute__((always_inline)) { return *reinterpret_cast<const int4 *>(p); };
        // Old values two groups ahead (the chunk after next is staged during
        // this one), lane 63's lower neighbours one group ahead.
        int4 cur = at(wl), nxt = at(wl + 4), down = at(sh.bot);
        int up0 = sh.top[63];
        auto chunk = [&](int cj, auto head) __attribute__((always_inline)) {
            const int q0 = (cj * kK) & (kTW - 1), q1 = (q0 + kK) & (kTW - 1);
            const int *rp = sh.top + ((q0 + 64) & (kTW - 1));
            int4 up[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) up[i] = at(rp + 4 * i);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int4 nn = at(i < 2 ? wl + q0 + 4 * i + 8 : wl + q1 + 4 * i - 8);
                const int4 dn = at(i < 3 ? sh.bot + q0 + 4 * i + 4 : sh.bot + q1);
                const int4 nv = sor_group<decltype(head)::value>(
                    h, cur, nxt.x, make_int4(up0, up[i].x, up[i].y, up[i].z), down, cj * kK + 4 * i + 1 - lane);
                *reinterpret_cast<int4 *>(wl + q0 + 4 * i) = nv;
                up0 = up[i].w;
                cur = nxt;
                nxt = nn;
                down = dn;
            }
            lds_barrier();
        };
        int cj = 0;
        for (; cj < 4; ++cj) chunk(cj, std::true_type{});
        for (; cj < nch; ++cj) chunk(cj, std::false_type{});
        return;
    }

    if (wave == 2) {
        // ----------------------------------------------------- boundary wave
        // Publishes the strip's bottom row, and takes the row above the strip
        // into sh.top: row 0 of the table (4 bytes a column), or the previous
        // strip's words (8).  A wave of its own, because the words arrive late:
        // waiting for one must not wait for the mover's loads and stores, which
        // complete in one order.  One poll of the next 64 columns is issued per
        // chunk and looked at four chunks later (a round trip to memory is
        // longer than a chunk); only when the next chunk's columns are missing
        // does the wave hold up the barrier and go through its polls.
        const int tshift = has_prev ? 3 : 2;
        const __amdgpu_buffer_rsrc_t topr =
            rows_rsrc(has_prev ? (const void *)bprev : (const void *)a.t, has_prev ? (n1 + 1) * 8LL : (n1 + 3) * 4LL);
        typedef __attribute__((ext_vector_type(2))) uint32_t u2;
        struct Poll {
            u2 v;
            int x;
        };
        int have = 0;  // columns 1..have are in sh.top
        int64_t t_new = now_ticks();
        auto issue = [&](Poll &p) __attribute__((always_inline)) {
            p.x = have + 1 + lane;
            asm volatile("" ::: "memory");  // reads again what an earlier poll read
            p.v = __builtin_amdgcn_raw_buffer_load_b64(topr, p.x <= n1 ? (uint32_t)p.x << tshift : kOut, 0, kCoherent);
        };
        // Chunk c reads columns up to 16c + 17; the ring has room for six more
        // chunks.
        auto need = [&](int c) __attribute__((always_inline)) { return min(n1, c * kK + kK + 1); };
        auto examine = [&](Poll &p, int c) __attribute__((always_inline)) {
            const bool ready = p.x <= n1 && (!has_prev || p.v.y == tin);
            const uint64_t late = ~__builtin_amdgcn_ballot_w64(ready);
            const int upto = min(__builtin_amdgcn_readfirstlane(p.x) - 1 + (late ? (int)__builtin_ctzll(late) : 64),
                                 need(c + 5));
            if (upto > have) {
                if (p.x > have && p.x <= upto) sh.top[(p.x + 62) & (kTW - 1)] = (int)p.v.x;
                have = upto;
                t_new = now_ticks();
            } else if (have < need(c) && now_ticks() - t_new > a.timeout_ticks) {
                if (lane == 0) atomicOr(&a.res->status, 1);
                have = n1;
            }
            issue(p);
        };
        Poll p0, p1, p2, p3;
        issue(p0);
        issue(p1);
        issue(p2);
        issue(p3);
        // The bottom row: lane 63's columns of chunk c (16 lanes), as soon as
        // it is done.
        const __amdgpu_buffer_rsrc_t pubr =
            rows_rsrc(has_next ? (const void *)bnext : (const void *)a.t, has_next ? (n1 + 1) * 8LL : 0);
        auto publish = [&](int c) __attribute__((always_inline)) {
            const int s = c * kK + (lane & (kK - 1)), x = s - 62;
            const u2 v = {(uint32_t)win[63 * kTS + (s & (kTW - 1))], tout};
            __builtin_amdgcn_raw_buffer_store_b64(
                v, pubr, (lane < kK && c >= 0 && x >= 1 && x <= n1) ? (uint32_t)x * 8u : kOut, 0, kCoherent);
        };
        // One poll examined and reissued, one barrier passed if the next chunk's
        // columns are there, one publish (of nothing if not): always the same
        // accesses, so that waiting for a poll leaves the later ones in flight.
        int j = -1;  // the chunk before the next barrier; -1: the first barrier
        auto tick = [&](Poll &p) __attribute__((always_inline)) {
            examine(p, j + 1);
            const bool go = have >= need(j + 1) && j < nch;
            if (go) lds_barrier();
            publish(go ? j : -1);
            j += go ? 1 : 0;
        };
        do {
            tick(p0);
            tick(p1);
            tick(p2);
            tick(p3);
        } while (j < nch);
        return;
    }

    // ------------------------------------------------------------ mover wave
    // No value here is merged from a load and something else, and its loop has
    // one exit: where a path with fewer loads in flight joins, the compiler would
    // wait for nearly all of them.
    const int nrows = min(kRows, a.n2 - y0 + 1);      // interior rows of the strip
    const int trows = min(kRows + 1, a.n2 + 2 - y0);  // with the row below
    const __amdgpu_buffer_rsrc_t rs = rows_rsrc(a.t + (int64_t)y0 * a.ld, trows * a.ld * 4);
    const __amdgpu_buffer_rsrc_t outr = rows_rsrc(a.t + (int64_t)y0 * a.ld, nrows * a.ld * 4);
    int *bot = sh.bot;
    const int k4 = 4 * (lane & 3);
    const int xv0 = k4 + 1 - vec_row(0, lane);  // column of the lane's first cell in chunk 0
    uint32_t off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) off[i] = vec_off(vec_row(i, lane), k4, a.ld);
    const uint32_t boff = lane < 4 ? vec_off(64, 4 * lane + 1, a.ld) : kOut;

    // Where the pitch is n1 + 3, the vector that starts at column n1 of the
    // table's last row would reach one cell past the table: it is loaded from
    // a cell earlier (its first cell, T(n2+1, n1), is all that is needed of it).
    const uint32_t tail = y0 + trows == a.n2 + 2 ? (uint32_t)(((trows - 1) * a.ld + a.ld - 3) * 4) : kOut;
    auto load_vec = [&](uint32_t o) __attribute__((always_inline)) {
        return __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(rs, o - (o == tail ? 4u : 0u), 0, 0));
    };
    auto load = [&](Stage &st, int c) __attribute__((always_inline)) {
        const uint32_t co = (uint32_t)c * (kK * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) st.v[i] = load_vec(off[i] + co);
        st.b = load_vec(boff + co);
    };
    auto stage_vec = [&](int *d, uint32_t o, int4 v) __attribute__((always_inline)) {
        v.x = o == tail ? v.y : v.x;
        *reinterpret_cast<int4 *>(d) = v;
    };
    auto stage = [&](const Stage &st, int c) __attribute__((always_inline)) {
        const int q0 = (c * kK) & (kTW - 1);
        const uint32_t co = (uint32_t)c * (kK * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) stage_vec(win + vec_row(i, lane) * kTS + q0 + k4, off[i] + co, st.v[i]);
        if (lane < 4) stage_vec(bot + q0 + 4 * lane, boff + co, st.b);
    };
    // Chunk c, finished in all rows, back to the table: the vectors that lie in
    // columns 1..n1.  Vectors of rows past nrows lie past the descriptor's end
    // and are dropped.
    auto flush = [&](int c) __attribute__((always_inline)) {
        const int q0 = (c * kK) & (kTW - 1);
        const uint32_t co = (uint32_t)c * (kK * 4);
        typedef __attribute__((ext_vector_type(4))) uint32_t u4;
        u4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const u4 *>(win + vec_row(i, lane) * kTS + q0 + k4);
        const int xv = c * kK + xv0;  // the lane's first column is xv - 16i
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(
                v[i], outr, (uint32_t)(xv - 16 * i - 1) < (uint32_t)max(0, n1 - 3) ? off[i] + co : kOut, 0, 0);
    };
    // The cells of columns x0..x0+2 (row `lane`) whose vector is not such a one:
    // a row's first and last cells.  Once per strip and side, after the chunks
    // that hold them, and not with the chunks: a strip's first chunks are on the
    // way to the next strip's start.
    const int tail_at = (n1 + 62) / kK + 1;
    int head_at = 5;
    asm("" : "+s"(head_at));  // unknown to the compiler, which would peel the loop's first turns for it
    auto ends = [&](int x0) __attribute__((always_inline)) {
#pragma unroll
        for (int x = x0; x < x0 + 3; ++x) {
            const int s = x - 1 + lane, xs = x - (s & 3);
            const bool mine = lane < nrows && x >= 1 && x <= n1 && !(xs >= 1 && xs + 3 <= n1);
            __builtin_amdgcn_raw_buffer_store_b32(win[lane * kTS + (s & (kTW - 1))], outr,
                                                  mine ? (uint32_t)((lane * a.ld + x) * 4) : kOut, 0, 0);
        }
    };

    Stage sg[kAhead];  // chunk c travels in sg[c % kAhead]
#pragma unroll
    for (int c = 0; c < kAhead + 2; ++c) {
        if (c >= kAhead) stage(sg[c % kAhead], c - kAhead);
        load(sg[c % kAhead], c);
        // As many accesses, and in the same order, as in the loop below, which
        // otherwise would wait for more than it needs to (none is stored).
        flush(-kAhead);
        __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
    // One chunk: the compute wave runs chunk cj; `st` holds chunk cj + 2 and
    // takes chunk cj + 2 + kAhead (chunk -1 has no cell and is not stored).
    auto chunk = [&](int cj, Stage &st) __attribute__((always_inline)) {
        stage(st, cj + 2);
        load(st, cj + 2 + kAhead);
        flush(cj - 1);
        if (cj == head_at) ends(1);
        if (cj == tail_at) ends(n1 - 2);
        lds_barrier();
    };
    for (int c0 = 0; c0 < nch; c0 += kAhead) {
#pragma unroll
        for (int p = 0; p < kAhead; ++p) chunk(c0 + p, sg[(p + 2) % kAhead]);
    }
    flush(nch - 1);
    if (nch <= head_at) ends(1);
    if (nch <= tail_at) ends(n1 - 2);
}

__global__ __launch_bounds__(192) void wf_stencil_kernel(WfStencilArgs a)
{
    __shared__ StShared sh;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(*a.epoch);
    for (;;) {
        if (threadIdx.x == 0) sh.task = atomicAdd(a.counter, 1);
        __syncthreads();
        const int g = __builtin_amdgcn_readfirstlane(sh.task);
        __syncthreads();
        if (g >= a.nstrips) break;
        sor_strip(a, g, sh, lane, wave, epoch);
        __syncthreads();
    }
}

}  // namespace wfs

extern "C" int wf_stencil_resident(int cus)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wfs::wf_stencil_kernel, 192, 0) != hipSuccess ||
        per_cu < 1) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    return per_cu * cus;
}

extern "C" hipError_t wf_launch_stencil(int grid, const WfStencilArgs *a, hipStream_t stream)
{
    if (grid <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wfs::wf_stencil_kernel, dim3(grid), dim3(192), 0, stream, *a);
    return hipGetLastError();
}
