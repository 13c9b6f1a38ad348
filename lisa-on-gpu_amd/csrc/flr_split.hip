// flr_split.hip -- projection and TDI of short series, a sample's work split over waves.
//
// The one-lane-per-sample kernels (flr_kernels.hip) give a wave all of 64 samples' stencils, one
// after the other: 3300 (projection) or 6500 (2nd-generation TDI, exact) issue slots in series. A
// series of a few thousand samples then runs as a handful of waves per CU, each waiting for its own
// results most of the time. Here a workgroup takes 64 samples and its waves share them: one wave
// per spacecraft stencil of the projection (then one per link), one per chain length of the
// equal-arm TDI, every eighth unit otherwise; the partial values meet in LDS and are added in
// the one-lane kernels' order, so the bits are theirs. The price is the window's halo per 64 instead of
// 256 samples and the values' way through LDS, so these kernels are used up to a length (kSplitProj
// and the following). 8,192 samples, exact, us of the launch, one-lane -> split: projection 10.9 ->
// 5.3 (equal arms), 14.4 -> 6.1 (unequal), TDI 2nd generation 28.9 -> 7.3 (equal), 45.1 -> 14.4
// (unequal), Sagnac combination at order 31 34.3 -> 8.1.
#include "flr_paths.hpp"

namespace flr {

constexpr int kSplit = 64;  // samples per workgroup: one wave's lanes

__device__ __forceinline__ int wave_index()
{
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// Sample range, window and time of a workgroup's lane, the checks and edge zeros of the one-lane
// kernels. rows: the output's rows.
struct SplitTile {
    TileRange tr;
    int i, win_lo, win_len;
    bool valid;
    double t, t0_offset;
};

// Fills the tile; false if the workgroup has nothing (more) to do (the same for every lane).
template <typename Config>
__device__ __forceinline__ bool split_tile(const Config &cfg, double *out, int rows, int num_out,
                                           int num_in, int start, const double *t_arr, double t0,
                                           SplitTile &st)
{
    const int wave = wave_index();
    st.tr = tile_range(blockIdx.x, num_out, start, cfg.zero_edges, kSplit);
    st.i = st.tr.i0 + (threadIdx.x & 63);
    st.valid = (st.i >= st.tr.lo_valid) && (st.i < st.tr.hi_valid);
    if (!st.valid && st.i >= 0 && st.i < num_out && cfg.zero_edges && wave < rows)
        out[(size_t)wave * num_out + st.i] = 0.0;
    if (st.tr.first > st.tr.last) return false;
    st.win_lo = st.tr.first - cfg.halo_lo;
    st.win_len = st.tr.last + cfg.halo_hi - st.win_lo + 1;
    if (st.win_lo < 0 || st.win_lo + st.win_len > num_in) {
        if (st.valid && wave < rows) {
            atomicOr(cfg.err, kErrWindow);
            out[(size_t)wave * num_out + st.i] = __builtin_nan("");
        }
        return false;
    }
    const int ic = st.valid ? st.i : st.tr.first;
    st.t = t_arr ? t_arr[ic] : t0 + (double)ic * cfg.dt;
    st.t0_offset = t_arr ? t_arr[0] : t0 + (double)0 * cfg.dt;
    return true;
}

// Window samples a workgroup stages (its LDS capacity).
__host__ __device__ inline int split_cap(int win_cap) { return win_cap - kBlock + kSplit; }

// ------------------------------------------------------------------ projection

// Wave w < 3: receiver stencil of spacecraft w at t. The others: emitter stencils, of spacecraft
// w - 3 (EQ: one emission time for all links) or of link w - 3. Then wave w < 6 forms link w.
constexpr int split_tasks(bool eq) { return eq ? 6 : 9; }
constexpr int kSplitVals = 5;  // per task and lane: the interpolated h+ and hx, the position

template <int FORM, int H, bool EQ>
__global__ __launch_bounds__(kSplit *split_tasks(EQ)) void projection_split_kernel(ProjConfig cfg,
                                                                                   ProjSource src,
                                                                                   OrbitView orb,
                                                                                   LagrangeView lg)
{
    constexpr int kTasks = split_tasks(EQ);
    extern __shared__ double2 hwin[];
    const int lane = threadIdx.x & 63, task = wave_index();
    SplitTile st;
    if (!split_tile(cfg, src.y, kNLinks, src.num_delays, src.num_inputs, src.start, src.t_data,
                    src.t0, st))
        return;
    for (int jj = threadIdx.x; jj < st.win_len; jj += kSplit * kTasks)
        hwin[jj] = src.h[st.win_lo + jj];
    double *vals = reinterpret_cast<double *>(hwin + split_cap(cfg.win_cap));
    const int h = H > 0 ? H : lg.h;
    const double y_deps = FORM ? rcp_nr2(lg.deps) : 0.0;
    // link q of the second phase, and of the unequal-arm emitters: receiver s, emitter e
    auto recv = [](int q) { return q >> 1; };
    auto emit = [](int q) { return ((q >> 1) + 1 + (q & 1)) % 3; };

    double tt = st.t;
    OrbitNode nd = orbit_node<FORM>(orb, st.t);
    int sc = task;
    if (task >= 3) {
        const int q = task - 3;
        const int row = EQ ? cfg.link_row[0][1] : cfg.link_row[recv(q)][emit(q)];
        sc = EQ ? q : emit(q);
        tt = st.t - orbit_val(nd, row);
        nd = orbit_node<FORM>(orb, tt);
    }
    double x[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = orbit_val(nd, 6 + 3 * sc + c);
    int d;
    double e;
    split_delay(tt - dot3(src.k, x) * kCInv, st.t0_offset, cfg.fs, d, e);
    const int l = d - st.win_lo;
    const bool bad = (l - (h - 1) < 0) || (l + h >= st.win_len);
    __syncthreads();
    double2 hv = make_double2(__builtin_nan(""), __builtin_nan(""));
    if (!bad) hv = window_stencil<FORM, H, kEArg>(hwin, l, e, lg, y_deps, nullptr);
    if (bad && st.valid) atomicOr(cfg.err, kErrWindow);
    double *mine = vals + (size_t)task * kSplitVals * kSplit + lane;
    mine[0] = hv.x;
    mine[kSplit] = hv.y;
#pragma unroll
    for (int c = 0; c < 3; ++c) mine[(2 + c) * kSplit] = x[c];
    __syncthreads();
    if (task >= kNLinks || !st.valid) return;
    const int s = recv(task), em = emit(task);
    const double *vr = vals + (size_t)s * kSplitVals * kSplit + lane;
    const double *ve = vals + (size_t)(3 + (EQ ? em : task)) * kSplitVals * kSplit + lane;
    double xr[3], xe[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        xr[c] = vr[(2 + c) * kSplit];
        xe[c] = ve[(2 + c) * kSplit];
    }
    src.y[(size_t)cfg.link_row[s][em] * src.num_delays + st.i] =
        link_value<FORM, kEArg>(src.k, src.u, src.v, xr, xe, make_double2(vr[0], vr[kSplit]),
                                make_double2(ve[0], ve[kSplit]), false);
}

// ------------------------------------------------------------------ TDI

// Channel sums (waves 0..2: channel = wave) to the outputs, through LDS for A, E, T.
__device__ __forceinline__ void split_store(const TdiConfig &cfg, const TdiSource &src,
                                            const SplitTile &st, double acc, double *sums)
{
    const int lane = threadIdx.x & 63, wave = wave_index();
    if (cfg.aet) {
        if (wave < 3) sums[wave * kSplit + lane] = acc;
        __syncthreads();
        const double X = sums[lane], Y = sums[kSplit + lane], Z = sums[2 * kSplit + lane];
        acc = wave == 0 ? (Z - X) / cfg.s2
              : wave == 1 ? (X - 2.0 * Y + Z) / cfg.s6 : (X + Y + Z) / cfg.s3;
    }
    if (wave < 3 && st.valid) src.out[(size_t)wave * src.num_delays + st.i] = acc;
}

__device__ __forceinline__ double split_start(const TdiConfig &cfg, const TdiSource &src,
                                              const SplitTile &st)
{
    const int wave = wave_index();
    if (cfg.overwrite || wave >= 3) return 0.0;
    return src.out[(size_t)wave * src.num_delays + (st.valid ? st.i : st.tr.first)];
}

namespace stock {
// The unit of chain length m on link la of X (13 or 12 for even m, 31 or 21 for odd): its index.
constexpr int unit_of(int m, int la)
{
    for (int x = 0; x < 16; ++x)
        if (kX[x].len == m && kX[x].link == la) return x;
    return -1;
}
// Per chain length: the two units' indices and signs, first link (13 / 31), then the second.
struct GroupUnits {
    int x[2];
    double sign[2];
};
constexpr GroupUnits group_units(int m)
{
    const int a = unit_of(m, m % 2 ? 31 : 13), b = unit_of(m, m % 2 ? 21 : 12);
    return GroupUnits{{a, b}, {(double)kX[a].sign, (double)kX[b].sign}};
}
static_assert(group_kind(0) == 0 && group_kind(1) == 1 && group_kind(2) == 0 && group_kind(3) == 1 &&
                  group_kind(4) == 0 && group_kind(5) == 1 && group_kind(6) == 0 && group_kind(7) == 1,
              "even chain lengths pair y13 and y12, odd ones y31 and y21");
}  // namespace stock

// Equal-arm stock TDI: wave m takes chain length m -- the six units of tdi_equal_arm's group m
// (exact) or the three outputs of tdi_linear's (fast) -- and waves 0..2 add a channel's values in
// index (exact) or chain-length (fast) order. Exact forms: the window in paired rows, for ds_read_b128, and
// the reciprocals four at a time where proven: 131,072 samples 37.0 -> 35.2 us (2nd generation), 19.7 ->
// 17.9 us (1st), 8,192 samples 7.3 -> 6.7 and 6.0 -> 5.3 us, the same bits.
template <int NX, int FORM>
__global__ __launch_bounds__(kSplit *(stock::max_len(NX) + 1)) void tdi_split_equal_kernel(
    TdiConfig cfg, TdiSource src, OrbitView orb, LagrangeView lg, RowMap rm)
{
    constexpr int H = 13;
    constexpr int NG = stock::max_len(NX) + 1;
    constexpr int kVals = FORM ? NX : NG;  // per channel
    extern __shared__ __align__(16) double smem[];
    const int lane = threadIdx.x & 63, m = wave_index();
    const int cap = split_cap(cfg.win_cap);
    double *ywin = smem;                       // [6][cap], of double2 in the exact forms
    double2 *pairs = reinterpret_cast<double2 *>(smem);
    double *vals = smem + (FORM ? 2 : 1) * kNLinks * cap;  // [3][kVals][kSplit]
    double *sums = vals + 3 * kVals * kSplit;  // [3][kSplit]
    SplitTile st;
    if (!split_tile(cfg, src.out, 3, src.num_delays, src.num_inputs, src.start, src.t_arr, src.t0,
                    st))
        return;
    for (int jj = threadIdx.x; jj < st.win_len; jj += kSplit * NG) {
        const double *from = src.y + st.win_lo + jj;
        double y[kNLinks];
#pragma unroll
        for (int l = 0; l < kNLinks; ++l) y[l] = from[(size_t)rm.row[l] * src.num_inputs];
        if constexpr (FORM) {
            store_link_pairs(pairs + jj, cap, y);
        } else {
            double k[2][3];
            combine_links(y, k);
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                ywin[(2 * o) * cap + jj] = k[0][o];
                ywin[(2 * o + 1) * cap + jj] = k[1][o];
            }
        }
    }
    const OrbitNode nd = orbit_node<FORM>(orb, st.t);
    const double L = orbit_val(nd, rm.row[0]);
    double Dm = st.t;
    for (int q = 0; q < m; ++q) Dm -= L;
    const double y_deps = FORM ? rcp_nr2(lg.deps) : 0.0;
    __syncthreads();

    bool bad;
    if constexpr (FORM) {
        static constexpr stock::GroupUnits kUnits[8] = {
            stock::group_units(0), stock::group_units(1), stock::group_units(2), stock::group_units(3),
            stock::group_units(4), stock::group_units(5), stock::group_units(6), stock::group_units(7)};
        int d;
        double e;
        split_delay(Dm, st.t0_offset, cfg.fs, d, e);
        bad = (d - st.win_lo - (H - 1) < 0) || (d - st.win_lo + H >= st.win_len);
        if (bad) d = st.win_lo + H - 1;  // in-window stand-in; the result is discarded
        const double2 *xr[3];  // paired rows as tdi_equal_arm_pairs, from the lowest tap on
        static_for<3>([&](auto c) {
            int off = (2 * c + (m & 1)) * cap + d - st.win_lo - (H - 1);
            pin(off);
            xr[c] = pairs + off;
        });
        double S[3][2] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
        for_tap_pairs<FORM, H>(e, H, [&](int j, const auto &q) {
            const double E = lg.E[j - 1];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double2 up = xr[c][H + j], dn = xr[c][H - 1 - j];
                S[c][0] += E * q.sum(up.x, dn.x);
                S[c][1] += E * q.sum(up.y, dn.y);
            }
        });
        const double A = lagrange_A_exact(lg, e, y_deps);
        const double B = 1.0 - e;
        const double C = e;
        const double D = e * (1.0 - e);
        static_for<3>([&](auto c) {
            const double2 x0 = xr[c][H - 1], x1 = xr[c][H];
            static_for<2>([&](auto k) {
                double val = A * (B * (k ? x1.y : x1.x) + C * (k ? x0.y : x0.x) + D * S[c][k]);
                val *= kUnits[m].sign[k];
                vals[(c * kVals + kUnits[m].x[k]) * kSplit + lane] = bad ? __builtin_nan("") : val;
            });
        });
    } else {
        const int kind = m & 1;
        // group_sign of chain length m
        constexpr unsigned kNegative = [] {
            unsigned w = 0;
            for (int q = 0; q < 8; ++q) w |= (stock::group_sign(q) < 0 ? 1u : 0u) << q;
            return w;
        }();
        double val[3];
        bad = !linear_group<false>(Dm, kind, (kNegative >> m) & 1 ? -1.0 : 1.0, st.t0_offset, cfg.fs,
                                   st.win_lo, st.win_len, lg,
                                   [&](int kd, int c0) { return row_taps(ywin, cap, kd, c0); }, val);
#pragma unroll
        for (int o = 0; o < 3; ++o) vals[(o * kVals + m) * kSplit + lane] = val[o];
    }
    if (bad && st.valid) atomicOr(cfg.err, kErrWindow);
    double acc = split_start(cfg, src, st);
    __syncthreads();
    if (m < 3)
        for (int x = 0; x < kVals; ++x) acc += vals[(m * kVals + x) * kSplit + lane];
    split_store(cfg, src, st, acc, sums);
}

// Any table (and the stock tables with unequal arms, whose units come to the same operations): unit
// by unit as tdi_units, wave w taking units w, w + 8, ... of a round of kSplitUnits.
constexpr int kSplitWaves = 8;
constexpr int kSplitUnits = 48;

template <int FORM, int H>
__global__ __launch_bounds__(kSplit *kSplitWaves) void tdi_split_units_kernel(TdiConfig cfg,
                                                                              TdiSource src,
                                                                              OrbitView orb,
                                                                              LagrangeView lg)
{
    extern __shared__ double smem[];
    const int h = H > 0 ? H : lg.h;
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int cap = split_cap(cfg.win_cap);
    double *ywin = smem;                           // [6][cap]
    double *Ls = smem + kNLinks * cap;             // [6][kSplit]
    double *vals = Ls + kNLinks * kSplit;          // [kSplitUnits][kSplit]
    double *sums = vals + kSplitUnits * kSplit;    // [3][kSplit]
    SplitTile st;
    if (!split_tile(cfg, src.out, 3, src.num_delays, src.num_inputs, src.start, src.t_arr, src.t0,
                    st))
        return;
    for (int jj = threadIdx.x; jj < st.win_len; jj += kSplit * kSplitWaves) {
        const double *from = src.y + st.win_lo + jj;
#pragma unroll
        for (int r = 0; r < kNLinks; ++r) ywin[r * cap + jj] = from[(size_t)r * src.num_inputs];
    }
    if (wave < kNLinks) Ls[wave * kSplit + lane] = orbit_val(orbit_node<FORM>(orb, st.t), wave);
    const double y_deps = FORM ? rcp_nr2(lg.deps) : 0.0;
    double acc = split_start(cfg, src, st);
    __syncthreads();

    bool bad = false;
    const int units = cfg.ch_begin[3];
    for (int base = 0; base < units; base += kSplitUnits) {
        const int end = min(base + kSplitUnits, units);
        for (int u = base + wave; u < end; u += kSplitWaves) {
            const TdiUnit un = cfg.units[u];
            double delay = st.t;
            for (int q = 0; q < un.chain_len; ++q) {
                const int row = cfg.chain_rows[un.chain_start + q];
                if (row >= 0) delay -= Ls[row * kSplit + lane];
            }
            int d;
            double e;
            split_delay(delay, st.t0_offset, cfg.fs, d, e);
            const int ld = d - st.win_lo;
            double val = __builtin_nan("");
            if ((ld - (h - 1) >= 0) && (ld + h < st.win_len))
                val = stencil<FORM, H>(ywin + un.base_row * cap + ld, e, lg, y_deps);
            else
                bad = true;
            val *= un.sign;
            vals[(u - base) * kSplit + lane] = val;
        }
        __syncthreads();
        if (wave < 3)
            for (int u = max(base, cfg.ch_begin[wave]); u < min(end, cfg.ch_begin[wave + 1]); ++u)
                acc += vals[(u - base) * kSplit + lane];
        __syncthreads();
    }
    if (bad && st.valid) atomicOr(cfg.err, kErrWindow);
    split_store(cfg, src, st, acc, sums);
}

// ------------------------------------------------------------------ dispatch

constexpr size_t kSplitLds = 64 * 1024;  // wider windows (fine sampling) keep the one-lane kernels

// Longest series that takes a split kernel, in samples per CU (256 CUs): where the one-lane kernel
// fills the chip well enough to win by its smaller halo. One-lane -> split, us:
//   projection: 98,304 samples 18.6 -> 16.3 (equal arms), 24.2 -> 23.8 (unequal); 131,072 19.7 -> 21.2
//   equal-arm TDI: exact 98,304 samples 32.0 -> 25.7, 163,840 46.0 -> 43.4 (131,072, where the one-lane
//     groups come to exactly two a CU, 34.8 -> 35.2), 1st generation 24.7 -> 22.0 at 163,840; fast 163,841 21.2 -> 20.0, 196,608 21.9 -> 23.1
//   unequal-arm stock TDI: exact 81,920 samples 57.2 -> 46.2, 98,304 58.4 -> 54.9, 114,689 60.1 -> 63.0,
//     131,072 64.2 -> 73.8; 1st generation 30.3 -> 29.2 and 32.5 -> 38.8 at 98,304 and 131,072; fast 98,304
//     39.6 -> 36.1, 131,072 (1st generation) 22.6 -> 24.8
//   any other table, exact, order 25: 147,456 samples 39.8 -> 32.6, 163,840 40.6 -> 37.2, 196,608
//     43.4 -> 44.3, 524,288 100 -> 112; another order: 262,144 67.5 -> 61.8 (order 31), 524,288
//     119 -> 117, 188 -> 181 (order 15; its one-lane form loops over taps, two pairs at a time)
constexpr int kSplitProj = 384;
constexpr int kSplitEqual = 640;
constexpr int kSplitStock = 384;
constexpr int kSplitTable25 = 640;
constexpr int kSplitTable = 2048;

static bool split_suits(int samples, int per_cu, size_t lds)
{
    return lds <= kSplitLds && (int64_t)samples <= (int64_t)compute_units() * per_cu;
}

bool launch_projection_split(const ProjConfig &cfg, const ProjSource &src, const OrbitView &orb,
                             const LagrangeView &lg, int form, bool equal_arm, hipStream_t stream,
                             hipError_t &err)
{
    const bool eq = lg.h == 13 && equal_arm;
    const size_t shm = (size_t)split_cap(cfg.win_cap) * sizeof(double2) +
                       (size_t)split_tasks(eq) * kSplitVals * kSplit * sizeof(double);
    if (form == kExact || !split_suits(src.num_delays, kSplitProj, shm)) return false;
    const int nb = tiles_for(src.num_delays, src.start, cfg.zero_edges, kSplit);
#define FLR_SPLIT(F)                                                                              \
    (eq ? launch_tpb(projection_split_kernel<F, 13, true>, nb, kSplit * split_tasks(true), shm,   \
                     stream, cfg, src, orb, lg)                                                   \
     : lg.h == 13 ? launch_tpb(projection_split_kernel<F, 13, false>, nb,                         \
                               kSplit * split_tasks(false), shm, stream, cfg, src, orb, lg)       \
                  : launch_tpb(projection_split_kernel<F == kFast ? kFast : kExact2, 0, false>, nb, \
                               kSplit * split_tasks(false), shm, stream, cfg, src, orb, lg))
    // any other order keeps two reciprocals at a time: with four (74 VGPRs) two of its 9-wave groups fit
    // a CU instead of three, and 65,537 samples at order 31 take 20.1 us instead of 18.1
    err = form == kFast     ? FLR_SPLIT(kFast)
          : form == kExact2 ? FLR_SPLIT(kExact2)
                            : FLR_SPLIT(kExact4);
#undef FLR_SPLIT
    return true;
}

bool launch_tdi_split(const TdiConfig &cfg, const TdiSource &src, const OrbitView &orb,
                      const LagrangeView &lg, int form, const StockTdi &stock, hipStream_t stream,
                      hipError_t &err)
{
    const bool eq = use_equal_arm(stock, lg);
    const int nx = stock.generation == 1 ? 8 : 16;
    const size_t rows = (size_t)(eq && form != kFast ? 2 : 1) * kNLinks * split_cap(cfg.win_cap);
    const size_t vals = eq ? (form == kFast ? 3 * (nx == 8 ? 4 : 8) : 3 * nx) : kSplitUnits + kNLinks;
    const size_t shm = (rows + (vals + 3) * kSplit) * sizeof(double);
    const int limit = eq ? kSplitEqual
                      : use_stock(stock, lg) ? kSplitStock
                      : form != kFast && lg.h == 13 ? kSplitTable25 : kSplitTable;
    if (form == kExact || !split_suits(src.num_delays, limit, shm)) return false;
    const int nb = tiles_for(src.num_delays, src.start, cfg.zero_edges, kSplit);
    const RowMap &rm = stock.rows;
#define FLR_SPLIT(F)                                                                             \
    (eq ? nx == 8 ? launch_tpb(tdi_split_equal_kernel<8, F>, nb,      \
                               4 * kSplit, shm, stream, cfg, src, orb, lg, rm)                   \
                  : launch_tpb(tdi_split_equal_kernel<16, F>, nb,     \
                               8 * kSplit, shm, stream, cfg, src, orb, lg, rm)                   \
     : lg.h == 13 ? launch_tpb(tdi_split_units_kernel<F, 13>, nb, kSplit * kSplitWaves, shm,     \
                               stream, cfg, src, orb, lg)                                        \
                  : launch_tpb(tdi_split_units_kernel<F, 0>, nb, kSplit * kSplitWaves, shm,      \
                               stream, cfg, src, orb, lg))
    err = form == kFast     ? FLR_SPLIT(kFast)
          : form == kExact2 ? FLR_SPLIT(kExact2)
                            : FLR_SPLIT(kExact4);
#undef FLR_SPLIT
    return true;
}

}  // namespace flr
