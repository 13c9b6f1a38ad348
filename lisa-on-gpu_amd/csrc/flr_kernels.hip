// flr_kernels.hip -- gfx950 kernels of the LISA time-domain response.
//
// Work unit: a tile of kBlock consecutive output samples of one source, one sample per lane.
// Each tile stages its sample window (tile + delay halo) in LDS once and every lane reads all
// its stencil taps from there.
//
// projection_tile: all six links per lane. The complex h window is shared by the 3 receiver
//   and 6 emitter stencils of every lane (the reference restages it per link,
//   LISAResponse.cu:628-655). A receiver stencil depends on the receiving spacecraft only, so
//   each is computed once for its two links: 9 complex stencils per sample instead of 12,
//   with bit-identical results (6 with equal arms, where the emitter stencils are shared too).
// tdi_tile: any TDI table. The 6 y rows of the window are staged once; each lane walks every
//   unit of every channel for its sample, summing units of a channel in index order in
//   registers (no atomics), then stores X, Y, Z or A, E, T.
// tdi_stock_tile: the stock 1st/2nd-generation tables with compile-time chains
//   (flr_tdi_stock.hpp): shared delays per chain length when all light travel times are
//   equal, per-unit delays from registers otherwise.
//
// Each tile function is launched two ways: one workgroup per tile of a single source, or a
// persistent batch kernel whose workgroups walk contiguous runs of a flattened (source, tile)
// list -- many sources of uneven length in one launch.
#include "flr_paths.hpp"

namespace flr {

// ------------------------------------------------------------------ projection

template <int EXACT, int H, bool EQ>
__device__ __forceinline__ void projection_tile(const ProjConfig &cfg, const ProjSource &src,
                                                int tile, const OrbitView &orb,
                                                const LagrangeView &lg, double2 *hwin)
{
    const int tid = threadIdx.x;
    const TileRange tr = tile_range(tile, src.num_delays, src.start, cfg.zero_edges);
    const int i = tr.i0 + tid;
    const bool valid = (i >= tr.lo_valid) && (i < tr.hi_valid);
    const bool in_range = (i >= 0) && (i < src.num_delays);

    if (!valid && in_range && cfg.zero_edges) {
#pragma unroll
        for (int l = 0; l < kNLinks; ++l) src.y[(size_t)l * src.num_delays + i] = 0.0;
    }
    if (tr.first > tr.last) return;  // whole tile outside the computed range

    // The window is sized from the orbit extent, so nothing has to be known about the delays
    // before it is staged.
    const int win_lo = tr.first - cfg.halo_lo;
    const int win_len = tr.last + cfg.halo_hi - win_lo + 1;
    if (win_len > cfg.win_cap || win_lo < 0 || win_lo + win_len > src.num_inputs) {
        if (valid) {
            atomicOr(cfg.err, kErrWindow);
            for (int l = 0; l < kNLinks; ++l) src.y[(size_t)l * src.num_delays + i] = __builtin_nan("");
        }
        return;
    }
    for (int jj = tid; jj < win_len; jj += kBlock) hwin[jj] = src.h[win_lo + jj];

    const int ic = valid ? i : tr.first;
    const double t = src.t_data ? src.t_data[ic] : src.t0 + (double)ic * cfg.dt;
    const double t0_offset = src.t_data ? src.t_data[0] : src.t0 + (double)0 * cfg.dt;
    __syncthreads();
    if (!valid) return;
    const double y_deps = EXACT ? rcp_nr2(lg.deps) : 0.0;
    double *y = src.y + i;
    const size_t stride = (size_t)src.num_delays;
    if (project_links<EXACT, H, EQ>(cfg, src.k, src.u, src.v, t, t0_offset, orb, lg, hwin, win_lo,
                                win_len, y_deps, nullptr, OrbitStage{},
                                [&](int row, double val) { y[row * stride] = val; }))
        atomicOr(cfg.err, kErrWindow);
}

// ------------------------------------------------------------------ TDI (any table)

__device__ __forceinline__ void tdi_store(const TdiConfig &cfg, const TdiSource &src, int i,
                                          const double (&acc)[3])
{
    if (cfg.aet) {
        const double X = acc[0], Y = acc[1], Z = acc[2];
        src.out[i] = (Z - X) / cfg.s2;
        src.out[(size_t)src.num_delays + i] = (X - 2.0 * Y + Z) / cfg.s6;
        src.out[(size_t)2 * src.num_delays + i] = (X + Y + Z) / cfg.s3;
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) src.out[(size_t)c * src.num_delays + i] = acc[c];
    }
}

// What the y window in LDS holds: the six rows (read by tdi_units, tdi_stock_unequal or, kEqualRows,
// tdi_equal_arm_rows), the six paired rows of tdi_equal_arm_pairs or the combined series of
// tdi_linear_packed.
enum WindowLayout { kRows, kEqualRows, kPairs, kPacked };

// Zero the tile's edge samples if asked, check and stage the y window (rm: canonical links to rows, for
// kPairs and kPacked).
// Returns false when the tile has nothing (more) to do; every lane returns the same value.
template <WindowLayout LAYOUT = kRows>
__device__ __forceinline__ bool tdi_stage(const TdiConfig &cfg, const TdiSource &src,
                                          const TileRange &tr, int i, bool valid, double *ywin,
                                          int &win_lo, int &win_len,
                                          const RowMap *rm = nullptr)
{
    const bool in_range = (i >= 0) && (i < src.num_delays);
    if (!valid && in_range && cfg.zero_edges) {
#pragma unroll
        for (int c = 0; c < 3; ++c) src.out[(size_t)c * src.num_delays + i] = 0.0;
    }
    if (tr.first > tr.last) return false;
    win_lo = tr.first - cfg.halo_lo;
    win_len = tr.last + cfg.halo_hi - win_lo + 1;
    if (win_len > cfg.win_cap || win_lo < 0 || win_lo + win_len > src.num_inputs) {
        if (valid) {
            atomicOr(cfg.err, kErrWindow);
            for (int c = 0; c < 3; ++c) src.out[(size_t)c * src.num_delays + i] = __builtin_nan("");
        }
        return false;
    }
    if constexpr (LAYOUT == kPairs || LAYOUT == kPacked) {
        const double *from = src.y + win_lo;
        double2 *pairs = reinterpret_cast<double2 *>(ywin);
        double *z = ywin + 4 * cfg.win_cap;  // kPacked, after the two rows of double2
        for (int jj = threadIdx.x; jj < win_len; jj += kBlock) {
            double y[kNLinks];
#pragma unroll
            for (int l = 0; l < kNLinks; ++l) y[l] = from[(size_t)rm->row[l] * src.num_inputs + jj];
            if constexpr (LAYOUT == kPairs)
                store_link_pairs(pairs + jj, cfg.win_cap, y);
            else
                store_packed_series(pairs + jj, z + jj, cfg.win_cap, y);
        }
        return true;
    }
    for (int r = 0; r < kNLinks; ++r) {
        const double *from = src.y + (size_t)r * src.num_inputs + win_lo;
        double *to = ywin + r * cfg.win_cap;
        for (int jj = threadIdx.x; jj < win_len; jj += kBlock) to[jj] = from[jj];
    }
    return true;
}

template <int EXACT, int H>
__device__ __forceinline__ void tdi_tile(const TdiConfig &cfg, const TdiSource &src, int tile,
                                         const OrbitView &orb, const LagrangeView &lg,
                                         double *smem)
{
    double *ywin = smem;                        // [6][win_cap]
    double *Ls = smem + kNLinks * cfg.win_cap;  // [6][kBlock]
    const int tid = threadIdx.x;
    const TileRange tr = tile_range(tile, src.num_delays, src.start, cfg.zero_edges);
    const int i = tr.i0 + tid;
    const bool valid = (i >= tr.lo_valid) && (i < tr.hi_valid);
    int win_lo = 0, win_len = 0;
    if (!tdi_stage(cfg, src, tr, i, valid, ywin, win_lo, win_len)) return;

    const int ic = valid ? i : tr.first;
    const double t = src.t_arr ? src.t_arr[ic] : src.t0 + (double)ic * cfg.dt;
    const double t0_offset = src.t_arr ? src.t_arr[0] : src.t0 + (double)0 * cfg.dt;
    {
        const OrbitNode nd = orbit_node<EXACT>(orb, t);
#pragma unroll
        for (int r = 0; r < kNLinks; ++r) Ls[r * kBlock + tid] = orbit_val(nd, r);
    }
    __syncthreads();
    if (!valid) return;
    const double y_deps = EXACT ? rcp_nr2(lg.deps) : 0.0;

    double acc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
        acc[c] = cfg.overwrite ? 0.0 : src.out[(size_t)c * src.num_delays + i];

    if (tdi_units<EXACT, H>(cfg, t, t0_offset, Ls + tid, kBlock, ywin, cfg.win_cap, win_lo, win_len,
                            lg, y_deps, acc))
        atomicOr(cfg.err, kErrWindow);
    tdi_store(cfg, src, i, acc);
}

// ------------------------------------------------------------------ equal-arm stock TDI
// Stock 1st/2nd-generation tables at order 25 when all six light travel times of the orbit
// table are bitwise equal (equal-arm orbits): the distinct delays t - m*L (m = chain length
// 0..3 or 0..7) are split once each and their stencil reciprocals (exact form) or weights
// (fast form) are shared by the units of that length -- 8 groups instead of 48 units for 2nd
// generation, with bit-identical results. The fast form goes further: by linearity the two units of
// each chain length and channel become one stencil of a combined series (tdi_linear), formed while
// the window is staged -- 24 stencils instead of 48, half the LDS reads: 1,000,003 samples, 2nd
// generation, 183 -> 96 us (MI355X).
// Bound by the FP64 pipes and, beside them, LDS reads (a ds_read2_b64 returns 125 bytes per clock and
// CU, a ds_read_b128 239), so the taps that are read together lie together: the two links of a channel
// (exact forms, paired rows: each link twice, 28 KB a tile at dt = 10 s), or X and Y (fast form). The same
// bits; 1,048,577 samples, 2nd generation: exact 225.6 -> 213.9 us, fast 96.2 -> 84.4 us.

template <int NX, int EXACT, WindowLayout LAYOUT>
__device__ __forceinline__ void tdi_stock_tile(const TdiConfig &cfg, const TdiSource &src,
                                               int tile, const OrbitView &orb,
                                               const LagrangeView &lg, const RowMap &rm,
                                               double *ywin)
{
    const TileRange tr = tile_range(tile, src.num_delays, src.start, cfg.zero_edges);
    const int i = tr.i0 + (int)threadIdx.x;
    const bool valid = (i >= tr.lo_valid) && (i < tr.hi_valid);
    int win_lo = 0, win_len = 0;
    if (!tdi_stage<LAYOUT>(cfg, src, tr, i, valid, ywin, win_lo, win_len, &rm)) return;

    const int ic = valid ? i : tr.first;
    const double t = src.t_arr ? src.t_arr[ic] : src.t0 + (double)ic * cfg.dt;
    const double t0_offset = src.t_arr ? src.t_arr[0] : src.t0 + (double)0 * cfg.dt;
    const OrbitNode nd = orbit_node<EXACT>(orb, t);
    double L[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) L[k] = orbit_val(nd, rm.row[k]);
    __syncthreads();
    if (!valid) return;
    const double y_deps = EXACT ? rcp_nr2(lg.deps) : 0.0;

    double acc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
        acc[c] = cfg.overwrite ? 0.0 : src.out[(size_t)c * src.num_delays + i];
    bool ok;
    const double2 *pairs = reinterpret_cast<const double2 *>(ywin);
    if constexpr (LAYOUT == kPacked) {
        ok = tdi_linear_packed<NX>(t, L[0], t0_offset, cfg.fs, pairs, cfg.win_cap, win_lo, win_len, lg,
                                   acc);
    } else if constexpr (LAYOUT == kEqualRows) {
        ok = tdi_equal_arm_rows<NX, EXACT>(t, L[0], t0_offset, cfg.fs, ywin, cfg.win_cap, rm, win_lo,
                                           win_len, lg, y_deps, acc);
    } else if constexpr (LAYOUT == kPairs) {
        ok = tdi_equal_arm_pairs<NX, EXACT>(t, L[0], t0_offset, cfg.fs, pairs, cfg.win_cap, win_lo,
                                            win_len, lg, y_deps, acc);
    } else {
        int rowoff[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) rowoff[k] = rm.row[k] * cfg.win_cap - win_lo;
        ok = tdi_stock_unequal<NX, EXACT>(t, L, t0_offset, cfg.fs, ywin, rowoff, win_lo, win_len,
                                          lg, y_deps, acc);
    }
    if (!ok) atomicOr(cfg.err, kErrWindow);
    tdi_store(cfg, src, i, acc);
}

// ------------------------------------------------------------------ kernels

template <int EXACT, int H, bool EQ>
__global__ __launch_bounds__(kBlock) void projection_kernel(ProjConfig cfg, ProjSource src,
                                                            OrbitView orb, LagrangeView lg)
{
    extern __shared__ double2 hwin[];
    projection_tile<EXACT, H, EQ>(cfg, src, blockIdx.x, orb, lg, hwin);
}

template <int EXACT, int H, bool EQ>
__global__ __launch_bounds__(kBlock) void projection_batch_kernel(ProjConfig cfg,
                                                                  Batch<ProjSource> batch,
                                                                  OrbitView orb, LagrangeView lg)
{
    extern __shared__ double2 hwin[];
    FLR_BATCH_LOOP(batch, (projection_tile<EXACT, H, EQ>(cfg, src, tile, orb, lg, hwin)));
}

template <int EXACT, int H>
__global__ __launch_bounds__(kBlock) void tdi_kernel(TdiConfig cfg, TdiSource src, OrbitView orb,
                                                     LagrangeView lg)
{
    extern __shared__ double smem[];
    tdi_tile<EXACT, H>(cfg, src, blockIdx.x, orb, lg, smem);
}

template <int EXACT, int H>
__global__ __launch_bounds__(kBlock) void tdi_batch_kernel(TdiConfig cfg, Batch<TdiSource> batch,
                                                           OrbitView orb, LagrangeView lg)
{
    extern __shared__ double smem[];
    FLR_BATCH_LOOP(batch, (tdi_tile<EXACT, H>(cfg, src, tile, orb, lg, smem)));
}

template <int NX, int EXACT, WindowLayout LAYOUT>
__global__ __launch_bounds__(kBlock) void tdi_stock_kernel(TdiConfig cfg, TdiSource src,
                                                               OrbitView orb, LagrangeView lg,
                                                               RowMap rm)
{
    extern __shared__ __align__(16) double smem[];
    tdi_stock_tile<NX, EXACT, LAYOUT>(cfg, src, blockIdx.x, orb, lg, rm, smem);
}

template <int NX, int EXACT, WindowLayout LAYOUT>
__global__ __launch_bounds__(kBlock) void tdi_stock_batch_kernel(TdiConfig cfg,
                                                                     Batch<TdiSource> batch,
                                                                     OrbitView orb,
                                                                     LagrangeView lg, RowMap rm)
{
    extern __shared__ __align__(16) double smem[];
    FLR_BATCH_LOOP(batch, (tdi_stock_tile<NX, EXACT, LAYOUT>(cfg, src, tile, orb, lg, rm, smem)));
}

// ------------------------------------------------------------------ small kernels

__global__ void orbit_eval_kernel(OrbitView orb, const double *t, int n, int row, int sc,
                                  double *ltt_out, double *pos_out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const OrbitNode nd = orbit_node(orb, t[i]);
    if (ltt_out) ltt_out[i] = orbit_val(nd, row);
    if (pos_out) {
        for (int c = 0; c < 3; ++c) pos_out[3 * i + c] = orbit_val(nd, 6 + 3 * sc + c);
    }
}

__global__ void clear_kernel(int *word)
{
    if (threadIdx.x == 0) word[0] = 0;
}

// ------------------------------------------------------------------ launchers

int compute_units()
{
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        return n;
    }();
    return cus;
}

// Persistent grid of total_tiles: as many workgroups as take one tile count each (but the last), at most
// grid_per_cu per CU. With some of them taking one tile more than the rest, spread evenly among them, a
// launch of 1.43 tiles a workgroup took 30% longer than its share: 16 sources of 700,000 samples, 11,747
// tiles of the 1024-sample window, 975 us with 8,192 workgroups, 765 with 5,874.
int batch_grid(int total_tiles, int grid_per_cu)
{
    const int grid = compute_units() * (grid_per_cu > 0 ? grid_per_cu : 16);
    if (total_tiles <= grid) return total_tiles;
    const int each = (total_tiles + grid - 1) / grid;
    return (total_tiles + each - 1) / each;
}

static size_t proj_lds(const ProjConfig &cfg) { return (size_t)cfg.win_cap * sizeof(double2); }

// f(form, H): the kernels are compiled for order 25 (H = 13) and for any (H = 0).
template <typename F>
static hipError_t by_order(bool exact, int64_t lowest, const LagrangeView &lg, F &&f)
{
    return by_form(stencil_form(exact, lowest, lg.h), [&](auto form) {
        if (lg.h == 13) return f(form, std::integral_constant<int, 13>{});
        return f(form, std::integral_constant<int, 0>{});
    });
}

// equal_arm: all six light travel time columns of the orbit table are bitwise equal (the
// emitter stencils are then shared per emitting spacecraft; order 25 only).
hipError_t launch_projection(const ProjConfig &cfg, const ProjSource &src, const OrbitView &orb,
                             const LagrangeView &lg, bool exact, bool equal_arm,
                             hipStream_t stream)
{
    const int nb = tiles_for(src.num_delays, src.start, cfg.zero_edges);
    const size_t shm = proj_lds(cfg);
    const int64_t lowest = (int64_t)src.start - cfg.halo_lo;
    hipError_t err;
    if (launch_projection_split(cfg, src, orb, lg, stencil_form(exact, lowest, lg.h), equal_arm, stream,
                                err))
        return err;
    return by_order(exact, lowest, lg, [&](auto form, auto h) {
        constexpr int F = decltype(form)::value, H = decltype(h)::value;
        if (H == 13 && equal_arm)
            return launch(projection_kernel<F, H, H == 13>, nb, shm, stream, cfg, src, orb, lg);
        return launch(projection_kernel<F, H, false>, nb, shm, stream, cfg, src, orb, lg);
    });
}

hipError_t launch_projection_batch(const ProjConfig &cfg, const Batch<ProjSource> &b,
                                   const OrbitView &orb, const LagrangeView &lg, bool exact,
                                   bool equal_arm, int grid_per_cu, hipStream_t stream)
{
    const int nb = batch_grid(b.total_tiles, grid_per_cu);
    const size_t shm = proj_lds(cfg);
    return by_order(exact, (int64_t)b.min_start - cfg.halo_lo, lg, [&](auto form, auto h) {
        constexpr int F = decltype(form)::value, H = decltype(h)::value;
        if (H == 13 && equal_arm)
            return launch(projection_batch_kernel<F, H, H == 13>, nb, shm, stream, cfg, b, orb, lg);
        return launch(projection_batch_kernel<F, H, false>, nb, shm, stream, cfg, b, orb, lg);
    });
}

// The stock kernels keep the light travel times in registers; the generic one in LDS.
static size_t tdi_lds(const TdiConfig &cfg, bool stock)
{
    return ((size_t)kNLinks * cfg.win_cap + (stock ? 0 : (size_t)kNLinks * kBlock)) * sizeof(double);
}

// The stock tables' kernel: f(form, layout, LDS bytes). Equal arms in the exact forms read paired rows
// while the window fits (windows of up to 1706 samples; the limit of rows is 3157). Paired rows are the
// better at every window that fits, if only one workgroup does: 500,000 samples, 2nd generation,
// dt = 2 s (352 samples) 123.7 -> 115.6 us, dt = 0.2 s (616 samples) 111.2 -> 105.0 us.
template <typename F>
static hipError_t by_stock_layout(const TdiConfig &cfg, bool exact, int64_t lowest,
                                  const LagrangeView &lg, bool equal_arm, F &&f)
{
    const size_t rows = tdi_lds(cfg, true), pairs = 2 * rows;
    using std::integral_constant;
    if (equal_arm && exact && pairs > kMaxLds)
        return f(integral_constant<int, kExact>{}, integral_constant<WindowLayout, kEqualRows>{}, rows);
    return by_form(stencil_form(exact, lowest, lg.h), [&](auto form) {
        constexpr int F_ = decltype(form)::value;
        if (equal_arm)
            return f(form, integral_constant<WindowLayout, F_ == kFast ? kPacked : kPairs>{},
                     F_ == kFast ? rows : pairs);
        return f(form, integral_constant<WindowLayout, kRows>{}, rows);
    });
}

hipError_t launch_tdi(const TdiConfig &cfg, const TdiSource &src, const OrbitView &orb,
                      const LagrangeView &lg, bool exact, const StockTdi &st, hipStream_t stream)
{
    const int nb = tiles_for(src.num_delays, src.start, cfg.zero_edges);
    const RowMap &rm = st.rows;
    const int64_t lowest = (int64_t)src.start - cfg.halo_lo;
    hipError_t err;
    if (launch_tdi_split(cfg, src, orb, lg, stencil_form(exact, lowest, lg.h), st, stream, err))
        return err;
    if (use_stock(st, lg)) {
        return by_stock_layout(cfg, exact, lowest, lg, st.equal_arm, [&](auto form, auto layout, size_t shm) {
            constexpr int F = decltype(form)::value;
            constexpr WindowLayout W = decltype(layout)::value;
            return st.generation == 1
                       ? launch(tdi_stock_kernel<8, F, W>, nb, shm, stream, cfg, src, orb, lg, rm)
                       : launch(tdi_stock_kernel<16, F, W>, nb, shm, stream, cfg, src, orb, lg, rm);
        });
    }
    const size_t shm = tdi_lds(cfg, false);
    return by_order(exact, lowest, lg, [&](auto form, auto h) {
        constexpr int F = decltype(form)::value, H = decltype(h)::value;
        return launch(tdi_kernel<F, H>, nb, shm, stream, cfg, src, orb, lg);
    });
}

hipError_t launch_tdi_batch(const TdiConfig &cfg, const Batch<TdiSource> &b, const OrbitView &orb,
                            const LagrangeView &lg, bool exact, const StockTdi &st,
                            int grid_per_cu, hipStream_t stream)
{
    const int nb = batch_grid(b.total_tiles, grid_per_cu);
    const RowMap &rm = st.rows;
    const int64_t lowest = (int64_t)b.min_start - cfg.halo_lo;
    if (use_stock(st, lg)) {
        return by_stock_layout(cfg, exact, lowest, lg, st.equal_arm, [&](auto form, auto layout, size_t shm) {
            constexpr int F = decltype(form)::value;
            constexpr WindowLayout W = decltype(layout)::value;
            return st.generation == 1
                       ? launch(tdi_stock_batch_kernel<8, F, W>, nb, shm, stream, cfg, b, orb, lg, rm)
                       : launch(tdi_stock_batch_kernel<16, F, W>, nb, shm, stream, cfg, b, orb, lg, rm);
        });
    }
    const size_t shm = tdi_lds(cfg, false);
    return by_order(exact, lowest, lg, [&](auto form, auto h) {
        constexpr int F = decltype(form)::value, H = decltype(h)::value;
        return launch(tdi_batch_kernel<F, H>, nb, shm, stream, cfg, b, orb, lg);
    });
}

hipError_t launch_orbit_eval(const OrbitView &orb, const double *t, int n, int row, int sc,
                             double *ltt_out, double *pos_out, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(orbit_eval_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, orb, t, n,
                       row, sc, ltt_out, pos_out);
    return hipGetLastError();
}

hipError_t launch_clear(int *word, hipStream_t stream)
{
    hipLaunchKernelGGL(clear_kernel, dim3(1), dim3(64), 0, stream, word);
    return hipGetLastError();
}

size_t fused_lds_bytes(const ProjConfig &pc, const TdiConfig &tc, bool generic, bool lti,
                       int passes, bool utv)
{
    if (utv)  // h window or the filters, then the padded rows (fused_tile_utv)
        return ((size_t)std::max(2 * pc.win_cap, utv_filter_doubles(passes == 4 ? 2 * kBlock : kBlock)) +
                (size_t)kNLinks * blk_pitch(tc.win_cap)) *
               sizeof(double);
    const size_t doubles =
        lti ? (size_t)kNLinks * blk_pitch(tc.win_cap) + 2 * kFpad
            : (size_t)kNLinks * tc.win_cap + (generic ? (size_t)kNLinks * kBlock : 0);
    return (size_t)pc.win_cap * sizeof(double2) + doubles * sizeof(double) +
           (lti ? (size_t)passes * kBlock : 0);
}

// One workgroup per source: each thread adds the tile records g0 + t, g0 + t + kBlock, ... of
// its source, then a fixed tree over the threads -- the same order whatever ran before.
__global__ __launch_bounds__(kBlock) void inner_reduce_kernel(const double *part,
                                                              const int *tile_start,
                                                              int num_sources, double *sums)
{
    constexpr int K = 3 * kInnerSums;
    __shared__ double red[K][kBlock];
    const int s = blockIdx.x, t = threadIdx.x;
    if (s >= num_sources) return;  // whole workgroup
    const int g0 = tile_start[s], g1 = tile_start[s + 1];
    double acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0;
    for (int g = g0 + t; g < g1; g += kBlock)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] += part[(size_t)g * K + k];
#pragma unroll
    for (int k = 0; k < K; ++k) red[k][t] = acc[k];
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (t < w)
#pragma unroll
            for (int k = 0; k < K; ++k) red[k][t] += red[k][t + w];
        __syncthreads();
    }
    if (t < K) sums[(size_t)s * K + t] = red[t][0];
}

hipError_t launch_inner_reduce(const double *part, const int *tile_start, int num_sources,
                               double *sums, hipStream_t stream)
{
    return launch(inner_reduce_kernel, num_sources, 0, stream, part, tile_start, num_sources, sums);
}

hipError_t launch_fused_batch(const ProjConfig &pc, const TdiConfig &tc,
                              const Batch<FusedSource> &b, const OrbitView &orb,
                              const LagrangeView &lg, bool exact, bool mixed, int input,
                              int tile_passes, int grid_per_cu, const StockTdi &st,
                              hipStream_t stream)
{
    if (lg.h != 13) return hipErrorInvalidValue;  // fused kernels are built for order 25
    if (mixed) {
        switch (input) {
        case kInC64:
            return launch_fused_mixed(pc, tc, b, orb, lg, tile_passes, grid_per_cu, st, stream);
        case kInQ31:
            return launch_fused_q31(pc, tc, b, orb, lg, tile_passes, grid_per_cu, st, stream);
        case kInC128:
            return launch_fused_c128(pc, tc, b, orb, lg, tile_passes, grid_per_cu, st, stream);
        default:
            return hipErrorInvalidValue;
        }
    }
    if (tile_passes != 2) return hipErrorInvalidValue;
    return launch_fused_fp64(pc, tc, b, orb, lg, exact, grid_per_cu, st, stream);
}

}  // namespace flr
