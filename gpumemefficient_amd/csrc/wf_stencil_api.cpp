// wf_stencil_api.cpp -- C ABI of the in-place table stencils: the
// reference's summed-area table (wf_sat.hip) and 2D-SOR sweep (wf_stencil.hip)
// behind
// void SOR(int n1, int n2, int *table[, int tX, int tY])
// (SAT/GPU_Hyperlane_Share.h:5, 2D-SOR/nested_loop/GPU_Hyperlane_Share.h:5 and
// the Cache headers).
#include <cstdint>
#include <cstring>

#include "wf_internal.h"

namespace {

// What a sweep may keep beside the table, in words: a row of the table for every
// 256 rows (1/32 byte a cell), or 8 MiB.  A table near the device's memory leaves
// no more.
int64_t sweep_words(int64_t n1, int64_t n2)
{
    return std::max<int64_t>(((n2 + 255) / 256 - 1) * (n1 + 1), 1 << 20);
}
// Fewest rows of the ring that the workgroups of a sweep hand their bottom rows
// down in.
constexpr int64_t kSweepRing = 4;

// A tile's strip height and rows per lane are checked and not used: both
// kernels have one shape (every shape gives the same table).
int check_tile(const wf_tile *tile)
{
    if (!tile) return WF_OK;
    const int rows = tile->strip_rows;
    if (tile->rows_per_lane > 1 || (rows > 0 && rows != 64 && rows != 128 && rows != 256)) return WF_ERR_NOKERNEL;
    return WF_OK;
}

// Reset and one launch of a sweep, timed with HIP events; the status and the
// table's last interior cell come back behind it through the context's pinned
// block, with one wait for everything.  tags: of the words that the launch's
// workgroups exchange.
template <class Launch>
int run_timed(wf_ctx *ctx, WfArenas *ar, int64_t tags, const int32_t *cell, double *ms, int32_t *last, Launch &&launch)
{
    int st;
    if ((st = wf_ensure_pinned(ctx, 256)) != WF_OK) return st;
    WfResultDev *r = reinterpret_cast<WfResultDev *>(ctx->pinned);
    int32_t *l = reinterpret_cast<int32_t *>(ctx->pinned + 128);
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    if (wf_launch_reset((WfResultDev *)ar->res.ptr, 1, (int32_t *)ar->counters.ptr, 2, (uint32_t *)ar->epoch.ptr,
                        (uint32_t)tags, ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    if (launch() != hipSuccess) return WF_ERR_DEVICE;
    if (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess) return WF_ERR_DEVICE;
    ctx->pinned_busy = true;
    if (hipMemcpyAsync(r, ar->res.ptr, sizeof(*r), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(l, cell, sizeof(*l), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
        hipStreamSynchronize(ctx->stream) != hipSuccess)
        return WF_ERR_DEVICE;
    ctx->pinned_busy = false;
    float f = 0.f;
    if (hipEventElapsedTime(&f, ctx->ev0, ctx->ev1) != hipSuccess) return WF_ERR_DEVICE;
    *ms = f;
    *last = *l;
    return r->status ? WF_ERR_TIMEOUT : WF_OK;
}

// The summed-area table: tiles instead of strips (wf_sat.hip).
int run_sat(wf_ctx *ctx, int64_t n1, int64_t n2, int32_t *dt, int64_t ld, double *ms, int32_t *last)
{
    WfArenas *ar = &ctx->scratch;
    const int cus = ctx->prop.multiProcessorCount;
    const int64_t ntc = (n1 + 1 + WFS_SAT_TILE_COLS - 1) / WFS_SAT_TILE_COLS;  // columns 0..n1
    const int64_t tr = WFS_SAT_TILE_ROWS, ntr = (n2 + tr - 1) / tr;
    const int64_t nblk = (ntc + WFS_SAT_BLOCK_TILES - 1) / WFS_SAT_BLOCK_TILES;
    // The tiles' bottom rows go round a ring: a tile's is overwritten by the one
    // `ring` tile rows below, which has had all those between, and a tag per turn
    // tells them apart.  With the rows' sums that takes no more memory than a
    // bottom row every 256 rows would (sweep_words; all tile rows: 1/13 byte a
    // cell, and 40 a row in tables of one tile column).
    const int64_t sums = ntr * tr * (ntc - 1 + nblk - 1), brow = ntc * WFS_SAT_TILE_COLS;
    const int64_t rows = std::max<int64_t>(1, ntr - 1);
    const int64_t ring = std::min(rows, std::max(kSweepRing, (sweep_words(n1, n2) - sums) / brow));
    const int64_t tags = (rows - 1) / ring + 1;
    int st;
    if ((st = ar->bnd.ensure((size_t)(sums + ring * brow) * sizeof(uint64_t), true)) != WF_OK) return st;
    if ((st = ar->res.ensure(sizeof(WfResultDev))) != WF_OK) return st;
    if ((st = ar->counters.ensure(2 * sizeof(int32_t))) != WF_OK) return st;
    if ((st = ar->epoch.ensure(sizeof(uint32_t), true)) != WF_OK) return st;
    WfSatArgs a{};
    a.t = dt;
    a.ld = ld;
    a.n1 = (int32_t)n1;
    a.n2 = (int32_t)n2;
    a.ntr = (int32_t)ntr;
    a.ntc = (int32_t)ntc;
    a.nblk = (int32_t)nblk;
    a.rowsum = (uint64_t *)ar->bnd.ptr;
    a.blksum = a.rowsum + ntr * (ntc - 1) * tr;
    a.bottom = a.rowsum + sums;
    a.ring = (int32_t)ring;
    a.tags = (int32_t)tags;
    a.counter = (int32_t *)ar->counters.ptr;
    a.res = (WfResultDev *)ar->res.ptr;
    a.epoch = (const uint32_t *)ar->epoch.ptr;
    a.timeout_ticks = (int64_t)(ctx->timeout_s * 1.0e8);
    const int grid = (int)std::min<int64_t>(ntr * ntc, std::max(1, wf_sat_resident(cus)));
    return run_timed(ctx, ar, tags, dt + n2 * ld + n1, ms, last, [&] { return wf_launch_sat(grid, &a, ctx->stream); });
}

// The sweep on a device table (pitch ld, ld % 4 == 0, 16-byte aligned); last:
// its cell (n2, n1).
int run_device(wf_ctx *ctx, int op, int64_t n1, int64_t n2, int32_t *dt, int64_t ld, double *ms, int32_t *last)
{
    *ms = 0.0;
    if (n1 == 0 || n2 == 0)  // no interior: the cell (n2, n1) is a boundary value
        return hipMemcpy(last, dt + n2 * ld + n1, sizeof(*last), hipMemcpyDeviceToHost) == hipSuccess ? WF_OK
                                                                                                      : WF_ERR_DEVICE;
    if (op == WF_SAT) return run_sat(ctx, n1, n2, dt, ld, ms, last);
    WfArenas *ar = &ctx->scratch;
    const int64_t strips = (n2 + WFS_SOR_STRIP_ROWS - 1) / WFS_SOR_STRIP_ROWS;
    // The strips' bottom rows go round a ring, as the tiles' do: a strip publishes
    // a column after the strip above has, and so on up to the one that read it.
    const int64_t rows = std::max<int64_t>(1, strips - 1);
    const int64_t ring = std::min(rows, std::max(kSweepRing, sweep_words(n1, n2) / (n1 + 1)));
    const int64_t tags = (rows - 1) / ring + 1;
    int st;
    if ((st = ar->bnd.ensure((size_t)(ring * (n1 + 1)) * sizeof(uint64_t), true)) != WF_OK) return st;
    if ((st = ar->res.ensure(sizeof(WfResultDev))) != WF_OK) return st;
    if ((st = ar->counters.ensure(2 * sizeof(int32_t))) != WF_OK) return st;
    if ((st = ar->epoch.ensure(sizeof(uint32_t), true)) != WF_OK) return st;
    WfStencilArgs a{};
    a.t = dt;
    a.ld = ld;
    a.n1 = (int32_t)n1;
    a.n2 = (int32_t)n2;
    a.nstrips = (int32_t)strips;
    a.ring = (int32_t)ring;
    a.tags = (int32_t)tags;
    a.bnd = (uint64_t *)ar->bnd.ptr;
    a.counter = (int32_t *)ar->counters.ptr;
    a.res = (WfResultDev *)ar->res.ptr;
    a.epoch = (const uint32_t *)ar->epoch.ptr;
    a.timeout_ticks = (int64_t)(ctx->timeout_s * 1.0e8);
    const int lim = wf_stencil_resident(ctx->prop.multiProcessorCount);
    const int grid = (int)std::min<int64_t>(strips, std::max(1, lim));
    return run_timed(ctx, ar, tags, dt + n2 * ld + n1, ms, last, [&] { return wf_launch_stencil(grid, &a, ctx->stream); });
}

// Host table -> device copy of pitch ldd -> sweep -> host table (or only the
// result cell with no_copyback).
int upload_run_download(wf_ctx *ctx, int op, int64_t n1, int64_t n2, int32_t *table, int64_t ld, int32_t *d,
                        int64_t ldd, bool no_copyback, wf_result *out)
{
    const int64_t rows = n2 + 2, cols = n1 + 3;
    if (hipMemcpy2D(d, (size_t)ldd * sizeof(int32_t), table, (size_t)ld * sizeof(int32_t),
                    (size_t)cols * sizeof(int32_t), (size_t)rows, hipMemcpyHostToDevice) != hipSuccess)
        return WF_ERR_DEVICE;
    double ms = 0.0;
    const int st = run_device(ctx, op, n1, n2, d, ldd, &ms, &out->last);
    out->kernel_ms = ms;
    if (st != WF_OK || no_copyback) return st;
    if (hipMemcpy2D(table, (size_t)ld * sizeof(int32_t), d, (size_t)ldd * sizeof(int32_t),
                    (size_t)cols * sizeof(int32_t), (size_t)rows, hipMemcpyDeviceToHost) != hipSuccess)
        return WF_ERR_DEVICE;
    return WF_OK;
}

bool valid_dims(int op, int64_t n1, int64_t n2, int64_t ld)
{
    // The kernel addresses a wave's 65-row window (and 8 rows of overrun)
    // with 32-bit byte offsets.
    return (op == WF_SAT || op == WF_SOR) && n1 >= 0 && n2 >= 0 && n1 + 3 <= ld && ld <= (int64_t)WF_STENCIL_MAX_PITCH &&
           n2 <= INT32_MAX - 256;
}

}  // namespace

extern "C" {

int wf_stencil_device(wf_ctx *ctx, int op, int64_t n1, int64_t n2, int32_t *dev_table, int64_t ld,
                      const wf_tile *tile, wf_result *out)
{
    if (!ctx || !out || !dev_table || !valid_dims(op, n1, n2, ld) || ld % 4 != 0 ||
        (reinterpret_cast<uintptr_t>(dev_table) & 15) != 0)
        return WF_ERR_INVALID;
    std::memset(out, 0, sizeof(*out));
    out->cells = (uint64_t)n1 * (uint64_t)n2;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    int st = check_tile(tile);
    if (st != WF_OK) return st;
    double ms = 0.0;
    st = run_device(ctx, op, n1, n2, dev_table, ld, &ms, &out->last);
    out->kernel_ms = ms;
    return st;
}

int wf_stencil(wf_ctx *ctx, int op, int64_t n1, int64_t n2, int32_t *table, int64_t ld, const wf_tile *tile,
               wf_result *out)
{
    if (!ctx || !out || !table || !valid_dims(op, n1, n2, ld)) return WF_ERR_INVALID;
    std::memset(out, 0, sizeof(*out));
    out->cells = (uint64_t)n1 * (uint64_t)n2;
    if (hipSetDevice(ctx->device) != hipSuccess) return WF_ERR_DEVICE;
    int st = check_tile(tile);
    if (st != WF_OK) return st;
    const int64_t rows = n2 + 2, cols = n1 + 3;
    const int64_t ldd = (cols + 3) & ~int64_t(3);
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) return WF_ERR_DEVICE;
    const size_t bytes = (size_t)(rows * ldd) * sizeof(int32_t);
    if (bytes + (64u << 20) > fr) return WF_ERR_NOMEM;
    DevBuf dt;
    if ((st = dt.ensure(bytes)) != WF_OK) return st;
    st = upload_run_download(ctx, op, n1, n2, table, ld, (int32_t *)dt.ptr, ldd,
                             tile && (tile->flags & WF_TILE_NO_COPYBACK), out);
    dt.release();
    return st;
}

}  // extern "C"
