// extern "C" boundary of the grouped GEMM (declared in include/gg_grouped_gemm.h).
//
// Host side of the reference's ck_tile backend, redone for the hand-written gfx950 kernel:
// CkTileBackend::prepare_typed / finish / run / release (ck_kernel/ck_grouped_gemm.cpp:126-226).
// prepare validates the problem, builds the device group table (row offset, rows, first
// tile per group) and the launch shape; run enqueues one launch and never synchronizes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <numeric>
#include <string>
#include <vector>

#include "gg_few.h"
#include "gg_grouped_gemm.h"
#include "gg_kernel.h"

struct gg_plan {
    int                 mode        = 0; // 0 forward, 1 dgrad, 2 wgrad (kernel terms: KernelArgs)
    int                 dtype       = GG_DTYPE_BF16;
    int                 group_num   = 0;
    int64_t             n           = 0;
    int64_t             k           = 0;
    int64_t             total_m     = 0;
    int                 total_tiles = 0;
    int                 grid        = 0;
    const void         *x           = nullptr;
    const void         *w           = nullptr;
    void               *out         = nullptr;
    // What the launch reads on the device, filled on the host by the plan builders; bind_plan places
    // it (and ws_bytes of workspace) in device memory, `mem` if the plan owns that.
    std::vector<gg::GroupEntry> table;
    std::vector<gg::TileDesc>   desc;
    std::vector<gg::SmallTile>  small_list;
    size_t                      ws_bytes = 0;
    void                       *mem      = nullptr;
    bool                        one_call = false; // gg_call: no detail text, descriptors where one_call_desc
    gg::GroupEntry     *d_groups    = nullptr;
    gg::KernelArgs      args{};
    std::string         detail;
    // Device-resident group sizes (gg_prepare_device_lens): the table is rebuilt per run.
    bool                device_lens = false;
    const int64_t      *d_lens      = nullptr;
    const int64_t      *d_offs      = nullptr;
    gg::TableHeader    *d_header    = nullptr; // follows the table in the d_groups allocation
    bool                in_kernel_table = false; // the GEMM builds the table (no table launch)
    int64_t             in_rows     = 0;       // device-size plans: rows of the inputs
    // Small-tile plans (use_small_tiles): the launch of gg_small.hip instead of the persistent one.
    bool                small       = false;
    gg::SmallArgs       sargs{};
    int                 few         = -1;      // few-row plans: the instance of gg_few.hip, -1: none
    bool                wgrad_few   = false;   // wgrad plans: the kernel of gg_wfew.hip
};

namespace {

thread_local std::string g_last_error;

int fail(int status, const std::string &msg) {
    g_last_error = msg;
    return status;
}

int hip_fail(hipError_t e, const char *what) {
    return fail(GG_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// XCDs of the device: MI355X (gfx950) has 8, each with its own L2. Workgroups are
// dispatched round-robin over them.
int xcd_count(const hipDeviceProp_t &prop) {
    const std::string arch = prop.gcnArchName;
    if (arch.rfind("gfx950", 0) == 0 || arch.rfind("gfx942", 0) == 0)
        return 8;
    return 1;
}

// Shape and pointer rules shared by both prepare entry points; returns GG_OK or a failure.
int check_problem(int dtype, int group_num, int64_t n, int64_t k, bool has_output, const void *x,
                  const void *w, const void *out) {
    if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_FP16)
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    if (group_num < 0 || n < 0 || k < 0)
        return fail(GG_ERR_INVALID, "group_num, n and k must be >= 0");
    if (has_output && (out == nullptr || (k > 0 && (x == nullptr || w == nullptr))))
        return fail(GG_ERR_INVALID, "x, w and out must be device pointers");
    // Shapes the kernel cannot take: reported like a non-empty Backend::prepare result.
    if (n % 8 != 0)
        return fail(GG_ERR_UNSUPPORTED, "N must be a multiple of 8 (16-byte output rows)");
    if (k % 8 != 0)
        return fail(GG_ERR_UNSUPPORTED, "K must be a multiple of 8 (16-byte input rows)");
    if (has_output && (!aligned16(out) || (k > 0 && (!aligned16(x) || !aligned16(w)))))
        return fail(GG_ERR_UNSUPPORTED, "x, w and out must be 16-byte aligned");
    // 32-bit per-tile byte offsets: a 256-row slice of x, w or out must stay below 2 GiB.
    if (k > (int64_t(1) << 21) || n > (int64_t(1) << 21))
        return fail(GG_ERR_UNSUPPORTED, "N and K must be at most 2097152");
    return GG_OK;
}

// Whether a problem runs on the instances of its own formats. An fp8 one that reads nothing may come
// without scales (wgrad of groups without rows: every tile runs and stores zeros), and the fp8 instances
// load the scales whatever the rows: those zeros come from the 16-bit instance, which loads none.
bool own_format(bool f8, bool reads, const float *a_scale, const float *b_scale) {
    return !f8 || reads || (a_scale != nullptr && b_scale != nullptr);
}

// Launch facts of the current device, queried from the runtime on the device's first use.
struct Device {
    int cus   = 0;
    int n_xcd = 1;
};
constexpr int kMaxDevices = 64;

int current_device(Device *out) {
    static std::mutex mu;
    static Device     known[kMaxDevices];
    int        dev = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess)
        return hip_fail(e, "hipGetDevice");
    const bool                  keep = dev >= 0 && dev < kMaxDevices;
    std::lock_guard<std::mutex> lock(mu);
    Device                      d = keep ? known[dev] : Device{};
    if (d.cus == 0) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, dev);
        if (e != hipSuccess)
            return hip_fail(e, "hipGetDeviceProperties");
        d.cus   = prop.multiProcessorCount;
        d.n_xcd = xcd_count(prop);
        if (keep)
            known[dev] = d;
    }
    *out = d;
    return GG_OK;
}

void fill_args(gg_plan *plan, int n_xcd) {
    gg::KernelArgs &a = plan->args;
    a.x         = plan->x;
    a.w         = plan->w;
    a.out       = plan->out;
    a.groups    = plan->d_groups;
    a.group_num = plan->group_num;
    a.n         = static_cast<int>(plan->n);
    a.k         = static_cast<int>(plan->k);
    a.n_tiles   = static_cast<int>(gg::cdiv(plan->n, gg::kTileN));
    a.k_tiles   = static_cast<int>(gg::cdiv(plan->k, gg::kTileK));
    a.n_xcd     = plan->grid % n_xcd == 0 ? n_xcd : 1;
    a.band      = gg::band_for(plan->n, plan->k, plan->mode / 4 == gg::kIn16 ? 2 : 1);
    // GG_BAND=<1..64> in the environment overrides the M-tiles per band of the in-group order
    // (measurements only)
    if (const char *env = std::getenv("GG_BAND"); env != nullptr && std::atoi(env) >= 1 && std::atoi(env) <= 64)
        a.band = std::atoi(env);
    a.lda       = static_cast<int>(plan->k);
    a.ldb       = static_cast<int>(plan->k);
    a.m_out     = 0;
    a.min_steps = 0;
    a.x_scale   = nullptr;
    a.w_scale   = nullptr;
    a.splits    = 1;
    a.ws        = nullptr;
    a.tile_n    = gg::kTileN;
    a.tile_m    = gg::kTileM;
    a.tail_splits = 1;
    a.desc        = nullptr;
    a.desc_per_wg = 0;
    a.tails       = 1; // set by the plan builders that know the sizes
}

// Split-K for problems whose tiles cannot fill the GPU (fewer than half as many tiles as CUs):
// each tile's K steps are cut into S ranges computed by different workgroups, which write fp32
// partial sums (256 KB per unit) that a second kernel adds in split order (deterministic) and
// converts. S minimises a launch-time model, in microseconds, fitted to MI355X timings of
// one-round problems (24-64 tiles, 22-256 K steps):
//   S = 1: k_tiles * kStepUs (one round of tiles)
//   S > 1: ceil(k_tiles / S) * kStepUs + kSplitUs + S * tiles * kSlabUs
// within one round (S * tiles <= CUs) and at least kMinSplitSteps K steps per range, taken only
// when it predicts at least kMinSplitGain (the cost of the partial sums grows faster than
// linearly near a full round of units, so small predicted gains are often losses).
// GG_SPLIT_K=<S> in the environment forces S (clamped to [1, k_tiles]; 1 turns split-K off).
constexpr double kStepUs        = 1.2;  // one K step of a 256 x 256 tile
constexpr double kSplitUs       = 3.0;  // second launch and its latency
constexpr double kSlabUs        = 0.15; // one unit's 256 KB of partial sums, written and read back
constexpr int    kMinSplitSteps = 4;
constexpr double kMinSplitGain  = 0.15;

int choose_splits(int tiles, int k_tiles, int cus) {
    if (const char *env = std::getenv("GG_SPLIT_K")) {
        const long v = std::strtol(env, nullptr, 10);
        if (v >= 1)
            return static_cast<int>(std::min<long>(v, k_tiles));
    }
    const int max_s = std::min(cus / std::max(tiles, 1), k_tiles / kMinSplitSteps);
    const double unsplit = k_tiles * kStepUs;
    int          best    = 1;
    double       cost    = unsplit;
    for (int sp = 2; sp <= max_s; ++sp) {
        const double c = ((k_tiles + sp - 1) / sp) * kStepUs + kSplitUs + double(sp) * tiles * kSlabUs;
        if (c < cost) {
            cost = c;
            best = sp;
        }
    }
    return cost <= (1.0 - kMinSplitGain) * unsplit ? best : 1;
}

// Narrow tiles (256 x 224) for a forward plan of one round that leaves CUs idle: when the plan is
// not split and the 224-wide tiling still fits in one round, it gives more workgroups 7/8 of a
// tile each (1 x 2048 x 7168: 224 tiles of 256 x 256 on 256 CUs, 256 tiles of 256 x 224). The
// group table is rebuilt for the narrow tile count. GG_NARROW=0 in the environment turns this
// off.
void use_narrow_tiles(gg_plan *plan, const int64_t *group_m, const Device &dev) {
    gg::KernelArgs &a   = plan->args;
    const char     *env = std::getenv("GG_NARROW");
    if ((env != nullptr && *env != '\0' && std::atoi(env) == 0) || a.splits > 1 || a.tile_m != gg::kTileM ||
        plan->total_tiles >= dev.cus)
        return;
    const int64_t               n_tiles = gg::cdiv(plan->n, gg::kNarrowTileN);
    std::vector<gg::GroupEntry> table(static_cast<size_t>(plan->group_num));
    const int64_t tiles = gg::build_group_table(group_m, plan->group_num, n_tiles, table.data());
    if (tiles <= plan->total_tiles || tiles > dev.cus)
        return;
    plan->table       = std::move(table);
    plan->total_tiles = static_cast<int>(tiles);
    plan->grid        = plan->total_tiles;
    a.total_tiles     = plan->total_tiles;
    a.n_tiles         = static_cast<int>(n_tiles);
    a.tile_n          = gg::kNarrowTileN;
    const int n_xcd   = dev.n_xcd;
    a.n_xcd           = plan->grid % n_xcd == 0 ? n_xcd : 1;
}

// Modelled time, in full 256 x 256 tile steps, of the busiest workgroup when tiles of tile_m rows
// are dealt to the grid in the kernel's order (xcd_remap over the group table's banded order).
// A tile's cost by its valid rows m, fitted to MI355X timings of partial tiles (one launch
// per row count, 256 groups, cross-tile): with 256-row tiles 1 for a full tile, 0.86-1 for
// 129-255 rows, and 0.70-0.85 for at most 128 rows (thin steps); with short tiles (at most 192
// rows, six row blocks per wave) the same below 129 rows and 0.85-0.88 above.
double busiest_workgroup(const int64_t *group_m, int group_num, int64_t n_tiles, int tile_m, int tiles,
                         int grid, int n_xcd, int band) {
    std::vector<float> cost(static_cast<size_t>(tiles));
    int                L = 0;
    for (int g = 0; g < group_num; ++g) {
        const int m_tiles = static_cast<int>(gg::cdiv(group_m[g], tile_m));
        for (int local = 0; local < m_tiles * n_tiles; ++local, ++L) {
            int tm, tn;
            gg::band_coords(local, m_tiles, static_cast<int>(n_tiles), band, &tm, &tn);
            const double m = static_cast<double>(std::min<int64_t>(tile_m, group_m[g] - int64_t(tm) * tile_m));
            double       c;
            if (m <= 128)
                c = 0.70 + 0.15 * m / 128;
            else if (tile_m < gg::kTileM)
                c = 0.85 + 0.03 * (m - 128) / 64;
            else
                c = m >= gg::kTileM ? 1.0 : 0.86 + 0.14 * (m - 128) / 128;
            cost[static_cast<size_t>(L)] = static_cast<float>(c);
        }
    }
    std::vector<double> load(static_cast<size_t>(grid), 0.0);
    for (int t = 0; t < tiles; ++t)
        load[static_cast<size_t>(t % grid)] += cost[static_cast<size_t>(gg::xcd_remap(t, tiles, grid, n_xcd))];
    return *std::max_element(load.begin(), load.end());
}

// Short tiles (at most 192 x 256) for a 16-bit forward or dgrad plan whose groups keep their M-tile
// counts with fewer rows per tile (gg::short_tile_rows): the same tiles, and the same total
// loads, but no group ends in a nearly empty tile next to full ones. Taken when the modelled
// busiest workgroup is at least 3 % faster (32 groups of 520 rows, N = K = 2880: three tiles of
// 176 rows per group; 4.71 -> 4.36 tile steps). The group table is rebuilt for the tile rows.
// GG_SHORT=0 in the environment turns this off, GG_SHORT=1 takes short tiles whenever the tile
// counts allow.
int use_short_tiles(gg_plan *plan, const int64_t *group_m) {
    gg::KernelArgs &a   = plan->args;
    const char     *env = std::getenv("GG_SHORT");
    const int       opt = env != nullptr && *env != '\0' ? std::atoi(env) : -1;
    if (opt == 0 || a.splits > 1 || a.tile_n != gg::kTileN)
        return GG_OK;
    const int rows = gg::short_tile_rows(group_m, plan->group_num);
    if (rows <= 0)
        return GG_OK;
    if (opt != 1) {
        const double wide  = busiest_workgroup(group_m, plan->group_num, a.n_tiles, gg::kTileM,
                                               plan->total_tiles, plan->grid, a.n_xcd, a.band);
        const double short_ = busiest_workgroup(group_m, plan->group_num, a.n_tiles, rows,
                                                plan->total_tiles, plan->grid, a.n_xcd, a.band);
        if (short_ > 0.97 * wide)
            return GG_OK;
    }
    std::vector<gg::GroupEntry> table(static_cast<size_t>(plan->group_num));
    const int64_t tiles = gg::build_group_table(group_m, plan->group_num, a.n_tiles, table.data(), 0, rows);
    if (tiles != plan->total_tiles)
        return fail(GG_ERR_INVALID, "short tiles changed the tile count");
    plan->table = std::move(table);
    a.tile_m = rows;
    return GG_OK;
}

// Short-wide tiles (at most 192 x 288) for a cross-tile 16-bit forward plan of short tiles: nine
// column blocks per wave instead of eight, so the same loads per K step feed 9/8 of the MFMAs and
// fewer tiles make fewer rounds (32 groups of 520 rows, N = K = 2880: 1152 short tiles, 4.5
// rounds on 256 CUs; 960 short-wide tiles, 3.75 rounds, and no 64-column tail tile). A
// short-wide tile is modelled at kWideTileCost short tiles (its K step moves 7 % more bytes for
// 12.5 % more MFMAs); taken when the modelled busiest workgroup gains at least 5 % and the plan
// stays cross-tile. The group table is rebuilt for the 288-column tiles.
// GG_WIDE=0 in the environment turns this off, GG_WIDE=1 takes short-wide tiles wherever the
// plan allows them.
constexpr double kWideTileCost = 1.10;

void use_short_wide_tiles(gg_plan *plan, const int64_t *group_m, const Device &dev) {
    gg::KernelArgs &a   = plan->args;
    const char     *env = std::getenv("GG_WIDE");
    const int       opt = env != nullptr && *env != '\0' ? std::atoi(env) : -1;
    if (opt == 0 || plan->mode != gg::make_mode(gg::kFwd, gg::kIn16) || a.tile_m == gg::kTileM ||
        a.tile_n != gg::kTileN || a.splits > 1 || a.d_total != nullptr || a.d_lens != nullptr)
        return;
    const int64_t n_tiles = gg::cdiv(plan->n, gg::kShortWideTileN);
    std::vector<gg::GroupEntry> table(static_cast<size_t>(plan->group_num));
    const int64_t tiles = gg::build_group_table(group_m, plan->group_num, n_tiles, table.data(), 0, a.tile_m);
    if (tiles <= 0 || tiles > INT32_MAX)
        return;
    const int grid  = static_cast<int>(std::min<int64_t>(dev.cus, tiles));
    const int n_xcd = grid % dev.n_xcd == 0 ? dev.n_xcd : 1;
    gg::KernelArgs w = a;
    w.total_tiles    = static_cast<int>(tiles);
    w.n_tiles        = static_cast<int>(n_tiles);
    w.tile_n         = gg::kShortWideTileN;
    w.n_xcd          = n_xcd;
    if (!gg::uses_cross_tile(w, grid, plan->mode))
        return;
    if (opt != 1) {
        const double short_ = busiest_workgroup(group_m, plan->group_num, a.n_tiles, a.tile_m, plan->total_tiles,
                                                plan->grid, a.n_xcd, a.band);
        const double wide   = kWideTileCost * busiest_workgroup(group_m, plan->group_num, n_tiles, a.tile_m,
                                                                w.total_tiles, grid, n_xcd, a.band);
        if (wide > 0.95 * short_)
            return;
    }
    plan->table       = std::move(table);
    plan->total_tiles = w.total_tiles;
    plan->grid        = grid;
    a                 = w;
}

// Picks the plan's split count (plan->args filled, k_tiles set) and the size of its partial sums.
void setup_split_k(gg_plan *plan, const Device &dev) {
    gg::KernelArgs &a  = plan->args;
    const int       sp = choose_splits(plan->total_tiles, a.k_tiles, dev.cus);
    if (sp <= 1)
        return;
    plan->ws_bytes = size_t(sp) * size_t(plan->total_tiles) * 262144;
    a.splits       = sp;
    plan->grid     = static_cast<int>(std::min<int64_t>(dev.cus, int64_t(sp) * plan->total_tiles));
}

// Tail split for cross-tile 16-bit forward plans (host-size tables): when the last round holds
// rem tiles, at most half the grid, each of them is cut into two K ranges run by two workgroups,
// so the busiest workgroup does R + 1/2 tiles instead of R + 1 (R full rounds). The ranges store
// fp32 partial sums (2 * rem slabs of 256 KB) and tail_reduce_kernel, launched right after the
// GEMM on the same stream, adds and stores them. Taken when a launch-time model (microseconds,
// fitted to MI355X end-to-end timings) predicts a gain: the busiest workgroup saves T / 2 K steps
// (kStepUs each), and pays its 256 KB of partial sums through the store path (kTailStoreUs), the
// second launch (kTailLaunchUs) and the reduction's traffic, 1.5 MB per last-round tile
// (kTailTileUs). Measured: 3 x 4096 x 1536 x 2048 (32 tiles in the last round, 32 K steps) 935 ->
// 980 TFLOPS; config 5a (128 tiles, 45 steps) 1022 -> 948 and 1 x 4096 x 5376 x 2048 (80 tiles)
// 1097 -> 1030, both left unsplit by the model. At least kMinTailSteps K steps per range.
// GG_TAIL_SPLIT=0 in the environment turns it off; GG_TAIL_SPLIT=2 takes it wherever the plan
// allows a split.
constexpr int    kMinTailSteps = 8;
constexpr double kTailStoreUs  = 6.0;
constexpr double kTailLaunchUs = 5.0;
constexpr double kTailTileUs   = 0.15;

void setup_tail_split(gg_plan *plan) {
    gg::KernelArgs &a = plan->args;
    a.tail_splits     = 1;
    if (plan->mode != gg::make_mode(gg::kFwd, gg::kIn16) || a.splits > 1 || a.d_total != nullptr ||
        a.d_lens != nullptr || a.tile_n != gg::kTileN || !gg::uses_cross_tile(a, plan->grid, plan->mode))
        return;
    const int grid = plan->grid, tiles = plan->total_tiles;
    const int full = tiles / grid * grid, rem = tiles - full;
    if (full == 0 || rem == 0 || 2 * rem > grid)
        return;
    int forced = -1;
    if (const char *env = std::getenv("GG_TAIL_SPLIT"); env != nullptr && *env != '\0')
        forced = std::atoi(env);
    if (forced == 0 || forced == 1)
        return;
    constexpr int sp = 2;
    if (a.k_tiles / sp < (forced > 1 ? gg::kCrossMinStepsHost : kMinTailSteps))
        return;
    const double saved_us = (a.k_tiles - gg::cdiv(a.k_tiles, sp)) * kStepUs;
    const double cost_us  = kTailStoreUs + kTailLaunchUs + rem * kTailTileUs;
    if (forced < 0 && saved_us < 1.1 * cost_us)
        return;
    plan->ws_bytes = size_t(rem) * size_t(sp) * 262144;
    a.tail_splits  = sp;
}

// Small tiles (128 x 128, one per workgroup, gg_small.hip) for 16-bit forward plans of host-size
// groups whose 256 x 256 tiles fill at most half the CUs (one round of the per-tile variant).
// The small-tile kernel runs its K steps at about half the MFMA rate of the persistent kernel
// (twice the LDS reads per MFMA) but brings about four times the workgroups. Taken when its
// tiles (unsplit unless GG_SMALL_SPLIT says otherwise) fit two per CU and a launch-time model
// (microseconds, MI355X) predicts at most kSmallGain of the persistent plan's time:
// kSmallFixedUs + K steps * kSmallStepUs (one workgroup per CU, a 4-step ring) or
// kSmallStepTwoUs (up to two, a 2-step ring) against kSmallFixedUs + the split-K model of
// choose_splits for the plan's own splits. Against GG_SMALL=0 (gg_bench and ab runs, bf16): one
// per CU, the suite's TestIDs 109, 110, 112, 122, 157, 160, 170 and 194 1.23-1.49x, pad_test's
// 9002 and 9004 and config 1; two per CU, 1 x 2048 x 2880 x 2880 1.13x, 1 x 1024 x 5760 x 2880
// 1.05x, 2 x 1024 x 2816 x 2048 1.03x. Left out: where the persistent plan splits a long K
// (146, 266, 268, 278, 148: small tiles 0.63-0.78x) and more than two tiles per CU.
// For forced plans (GG_SMALL=1) the K ranges fill up to one workgroup per CU (128 KB of LDS
// each) with at least kMinSmallSteps K steps per range; they write fp32 partial sums (64 KB per
// tile and range) that a second launch adds in range order. GG_SMALL=0 in the environment turns
// small tiles off; GG_SMALL_SPLIT=<S> forces the ranges.
constexpr int    kMinSmallSteps = 8;
constexpr double kSmallFixedUs  = 4.0;  // launch, first DMAs, epilogue
constexpr double kSmallStepUs    = 0.62; // one K step of a 128 x 128 tile, one workgroup per CU
constexpr double kSmallStepTwoUs = 1.0;  // the same with up to two workgroups per CU
constexpr double kSmallGain      = 0.85;

// The model: `units` small tiles (times K ranges) of `per` steps each against the persistent plan's
// tiles, splits and K steps.
bool small_tiles_win(int64_t units, int per, int tiles, int splits, int k_tiles, int cus) {
    if (2 * int64_t(tiles) > cus || units > 2 * int64_t(cus))
        return false;
    const double big  = kSmallFixedUs + gg::cdiv(k_tiles, splits) * kStepUs +
                       (splits > 1 ? kSplitUs + double(splits) * tiles * kSlabUs : 0.0);
    const double step = units <= cus ? kSmallStepUs : kSmallStepTwoUs;
    return kSmallFixedUs + double(per) * step <= kSmallGain * big;
}

void use_small_tiles(gg_plan *plan, const int64_t *group_m, const Device &dev) {
    const char *env = std::getenv("GG_SMALL");
    const int   opt = env != nullptr && *env != '\0' ? std::atoi(env) : -1;
    const int   cus = dev.cus;
    const gg::KernelArgs &a = plan->args;
    if (opt == 0 || plan->group_num > 32767 || (opt != 1 && (2 * plan->total_tiles > cus || a.tail_splits > 1)))
        return;
    const int64_t              nt = gg::cdiv(plan->n, gg::kSmallTile);
    std::vector<gg::SmallTile> list;
    int64_t                    row = 0;
    for (int g = 0; g < plan->group_num; ++g) {
        const int64_t mt = gg::cdiv(group_m[g], gg::kSmallTile);
        for (int64_t tn = 0; tn < nt; ++tn)
            for (int64_t tm = 0; tm < mt; ++tm)
                list.push_back({row + tm * gg::kSmallTile,
                                static_cast<int32_t>(std::min<int64_t>(gg::kSmallTile, group_m[g] - tm * gg::kSmallTile)),
                                static_cast<int16_t>(g), static_cast<int16_t>(tn)});
        row += group_m[g];
    }
    const int64_t tiles   = static_cast<int64_t>(list.size());
    const int     k_steps = static_cast<int>(gg::cdiv(plan->k, gg::kSmallK));
    if (tiles == 0 || tiles > 65536)
        return;
    // Workgroup i runs on XCD i % n_xcd: deal the list (N-tile by N-tile, M-tiles inside) to the
    // XCDs in contiguous runs (xcd_remap), so that the workgroups of one XCD share a few x and w
    // panels in its L2 instead of every XCD reading every w panel.
    // (A grid of whole XCD rows: XCD y takes ceil((tiles - y) / n_xcd) of the list.)
    if (const int n_xcd = dev.n_xcd; n_xcd > 1) {
        const int                  rows = static_cast<int>(gg::cdiv(tiles, n_xcd)) * n_xcd;
        std::vector<gg::SmallTile> dealt(list.size());
        for (int t = 0; t < static_cast<int>(tiles); ++t)
            dealt[static_cast<size_t>(t)] = list[static_cast<size_t>(gg::xcd_remap(t, static_cast<int>(tiles), rows, n_xcd))];
        list.swap(dealt);
    }
    int sp = 1;
    if (opt == 1 && tiles < cus) // forced: fill the CUs with K ranges
        sp = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(cus / tiles, k_steps / kMinSmallSteps)));
    if (const char *e2 = std::getenv("GG_SMALL_SPLIT"); e2 != nullptr && std::atoi(e2) >= 1)
        sp = std::min(std::atoi(e2), k_steps);
    const int per = static_cast<int>(gg::cdiv(k_steps, sp));
    sp            = static_cast<int>(gg::cdiv(k_steps, per)); // no empty K range
    // a 4-step ring while every workgroup has a CU of its own, else a 2-step ring, two per CU
    const int stages = tiles * sp <= cus ? gg::kSmallStagesOne : gg::kSmallStagesTwo;
    if (opt != 1 && !small_tiles_win(tiles * sp, per, plan->total_tiles, a.splits, a.k_tiles, cus))
        return;
    // the persistent plan's table, workspace and descriptors are not used by this launch
    plan->table.clear();
    plan->desc.clear();
    plan->ws_bytes   = sp > 1 ? size_t(sp) * size_t(tiles) * gg::kSmallTile * gg::kSmallTile * sizeof(float) : 0;
    plan->small_list = std::move(list);
    gg::SmallArgs &sa    = plan->sargs;
    sa.x                 = plan->x;
    sa.w                 = plan->w;
    sa.out               = plan->out;
    sa.tiles             = static_cast<int>(tiles);
    sa.n                 = static_cast<int>(plan->n);
    sa.k                 = static_cast<int>(plan->k);
    sa.k_steps           = k_steps;
    sa.splits            = sp;
    sa.steps_per_split   = per;
    sa.stages            = stages;
    plan->small          = true;
    plan->total_tiles    = static_cast<int>(tiles);
    plan->grid           = static_cast<int>(tiles) * sp;
}

void free_plan(gg_plan *plan) {
    if (plan->mem != nullptr)
        (void)hipFree(plan->mem);
    delete plan;
}

// ---------------------------------------------------------------------------------------
// Placing a host-size plan's tables and workspace in device memory: one block, its parts at
// multiples of 256 bytes, the workspace last (nothing is uploaded into it).
// ---------------------------------------------------------------------------------------
size_t block(size_t bytes) { return (bytes + 255) / 256 * 256; }
size_t upload_bytes(const gg_plan *p) {
    return block(p->table.size() * sizeof(gg::GroupEntry)) + block(p->desc.size() * sizeof(gg::TileDesc)) +
           block(p->small_list.size() * sizeof(gg::SmallTile));
}
size_t plan_bytes(const gg_plan *p) { return upload_bytes(p) + p->ws_bytes; }

// Points the plan's arguments into `mem` (plan_bytes of device memory) and writes what belongs there
// to `image` (upload_bytes).
void bind_plan(gg_plan *p, void *mem, std::vector<char> *image) {
    image->assign(upload_bytes(p), 0);
    size_t     at    = 0;
    const auto place = [&](const auto &v) {
        char *dst = v.empty() ? nullptr : static_cast<char *>(mem) + at;
        if (!v.empty())
            std::memcpy(image->data() + at, v.data(), v.size() * sizeof(v[0]));
        at += block(v.size() * sizeof(v[0]));
        return dst;
    };
    p->d_groups        = reinterpret_cast<gg::GroupEntry *>(place(p->table));
    p->args.groups     = p->d_groups;
    p->args.desc       = reinterpret_cast<const int *>(place(p->desc));
    p->sargs.tile_list = reinterpret_cast<gg::SmallTile *>(place(p->small_list));
    p->args.ws         = p->ws_bytes > 0 ? reinterpret_cast<float *>(static_cast<char *>(mem) + at) : nullptr;
    p->sargs.ws        = p->args.ws;
}

// Device memory of a plan that owns it, uploaded on `s` and waited for.
int allocate_plan(gg_plan *p, hipStream_t s) {
    if (plan_bytes(p) == 0)
        return GG_OK;
    hipError_t e = hipMalloc(&p->mem, plan_bytes(p));
    if (e != hipSuccess) {
        p->mem = nullptr;
        return hip_fail(e, "plan memory allocation");
    }
    std::vector<char> image;
    bind_plan(p, p->mem, &image);
    e = hipMemcpyAsync(p->mem, image.data(), image.size(), hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    return e == hipSuccess ? GG_OK : hip_fail(e, "plan table upload");
}

// Few-row tiles (gg_few.hip) for forward and dgrad plans, 16-bit and fp8, host- and device-size,
// whose groups have few rows or whose whole problem is small: there the 256 x 256 tiles of the
// persistent kernel (and the 128 x 128 ones) leave CUs idle or run one long chain of K steps each.
// Chosen by a launch-time model in microseconds, the lesser instance's time against the plan
// that would run otherwise, taken at a share of it (few_gain). Both sides add the parts' squares (the memory
// traffic, the operands' way into LDS and the chain of K steps overlap, but not fully):
//   few:   kFewFixedUs + |HBM bytes / kFewHbm, staged bytes / kFewStage, rounds of workgroups x
//          (chunks per wave x chunk_us + kFewRoundUs)|
//   other: fixed + |HBM bytes / kOtherHbm, K steps of the busiest workgroup|
// Fitted to 300 random forward and dgrad problems of 1-64 groups, 1-1000 rows each, N and K
// 512-14336, bf16 and fp8 (MI355X, each instance and the other plan timed). On 1900 others, 40 % of them
// with contractions over 6000, each with its operands in cache and from HBM in turn, the choice gives
// 1.71x (HBM: 1.58x) over the other plans in the geometric mean, the best of each 1.82x (1.66x), and is
// slower in cache or from HBM on 16 of them (0.71-0.97x). Examples (us, other -> few): 4 x 256 rows,
// 512 x 1024 12.3 -> 6.4; 3 x 5 rows (device sizes), 3328 x 12256 130 -> 38; 3 x 14 rows dgrad, 1208 x 2048
// 25.3 -> 6.0; 36 x 16 rows, 2048 x 1024 35.9 -> 23.4; left: 8 x 128 rows, 4096 x 7168 100 (few 131). With rows for whole
// tiles, the staged bytes (each small tile stages its own operands) decide against it.
// Plans of more than kFewMaxSmallTiles 128 x 128 tiles whose groups average over 64 rows keep them:
// the few-row tiles ran 0.73-1.28x there (7 of the 300 problems), and the model is no better than that.
// GG_SMALL in the environment (0: no small tiles, 1: 128 x 128 tiles) turns it off; without it,
// GG_FEW=<i> takes instance i (GG_FEW=-1: none).
constexpr double kFewFixedUs = 1.6, kFewRoundUs = 1.9;
constexpr double kFewHbm = 6.2e6, kFewStageFwd = 22e6, kFewStageDgrad16 = 15e6, kFewStageDgrad8 = 10.5e6; // bytes per us
constexpr int    kFewMaxSmallTiles = 64;
constexpr double kOtherHbm16 = 6.8e6, kOtherHbm8 = 5.9e6;
constexpr double kOtherFixedUs = 7.2, kOtherStepUs = 0.88;  // persistent kernel
constexpr double kOtherSmallFixedUs = 1.8;                  // 128 x 128 tiles

// Row tiles of 16, 32, .. 256 rows: of the host's sizes, or of `rows` rows spread over the groups (device
// sizes: a group whose average fills more than half a tile is expected to end in half a tile). One pass
// of shifts: a division per group and tile height took 0.4 ms of a plan's preparation for 32768 groups.
struct RowTiles {
    double tiles[5] = {};
    RowTiles(const int64_t *group_m, int group_num, int64_t rows) {
        int64_t sum[5] = {};
        for (int g = 0; g < group_num && group_m != nullptr; ++g)
            for (int i = 0; i < 5; ++i)
                sum[i] += (group_m[g] + (16 << i) - 1) >> (4 + i);
        for (int i = 0; i < 5; ++i) {
            const double avg = double(rows) / group_num, bm = 16 << i;
            tiles[i] = group_m != nullptr ? double(sum[i])
                                          : std::max(double(std::min<int64_t>(group_num, rows)),
                                                     double(rows) / bm + (avg > bm / 2 ? 0.5 * group_num : 0.0));
        }
    }
    double of(int bm) const { return tiles[__builtin_ctz(static_cast<unsigned>(bm)) - 4]; }
};

// The share of the other plan's time that a few-row plan must promise. Where the contraction is long, most
// of the time is w's way from HBM and the model, fitted with w in the caches, promises too much: with
// 0.85 throughout, 69 of the 1900 problems were slower than the other plan, down to 0.63x, nearly all with
// less than 1.4 rounds of workgroups. dgrad with less than 3/4 of a round reads w's rows in pieces of 32-128
// bytes and has the most of them (2 x 57 rows forward, 5632 x 13008 87 -> 120 us; 3 x 26 dgrad, 1024 x 13888
// 40 -> 63).
double few_gain(bool dgrad, int64_t chunks, double rounds) {
    return chunks < 64 || rounds >= 1.4 ? 0.85 : dgrad && rounds < 0.75 ? 0.53 : 0.61;
}

// The few-row instance of a forward or dgrad plan (its problem set; group_m null: device sizes of
// `rows` rows in all), or -1.
int choose_few_rows(const gg_plan *plan, const int64_t *group_m, int64_t rows, int cus) {
    if (const char *env = std::getenv("GG_SMALL"); env != nullptr && *env != '\0')
        return -1;
    int forced = -2;
    if (const char *env = std::getenv("GG_FEW"); env != nullptr && *env != '\0')
        forced = std::atoi(env);
    if (forced == -1 || forced >= gg::kFewInstanceCount)
        return -1;
    const bool    f8 = plan->mode / 4 != gg::kIn16, dgrad = plan->mode % 4 == gg::kDgrad;
    const int     es     = f8 ? 1 : 2;
    const int64_t groups = std::min<int64_t>(plan->group_num, rows);
    const int64_t chunks = gg::cdiv(plan->k * es, 128); // 128 bytes of an operand row
    const double  bytes  = double(groups) * plan->n * plan->k * es + double(rows) * (plan->k * es + plan->n * 2);
    const RowTiles row_tiles(group_m, plan->group_num, rows);
    // the plan that would run otherwise
    const double tiles = row_tiles.of(gg::kTileM) * gg::cdiv(plan->n, gg::kTileN);
    double       steps, fixed = kOtherFixedUs;
    if (group_m == nullptr || tiles > cus) {
        steps = std::max(1.0, std::ceil(tiles / cus)) * chunks * kOtherStepUs;
    } else {
        const int s = choose_splits(static_cast<int>(tiles), static_cast<int>(chunks), cus);
        steps       = gg::cdiv(chunks, s) * kOtherStepUs + (s > 1 ? kSplitUs + s * tiles * kSlabUs : 0.0);
        const double units = row_tiles.of(gg::kSmallTile) * gg::cdiv(plan->n, gg::kSmallTile);
        if (!f8 && !dgrad && small_tiles_win(static_cast<int64_t>(units), static_cast<int>(chunks), static_cast<int>(tiles), s,
                                             static_cast<int>(chunks), cus)) {
            if (forced < 0 && units > kFewMaxSmallTiles && rows > 64 * groups)
                return -1;
            steps = chunks * (units <= cus ? kSmallStepUs : kSmallStepTwoUs);
            fixed = kOtherSmallFixedUs;
        }
    }
    const double other = fixed + std::hypot(bytes / (f8 ? kOtherHbm8 : kOtherHbm16), steps);
    const double stage = !dgrad ? kFewStageFwd : f8 ? kFewStageDgrad8 : kFewStageDgrad16;
    int          best  = -1;
    double       least = 0, rounds = 0;
    for (int i = 0; i < gg::kFewInstanceCount; ++i) {
        const gg::FewInstance &f = gg::kFewInstances[i];
        // the kernel's tile index must not pass 2^31 (device sizes may put every row in each group)
        const int64_t nt   = gg::cdiv(plan->n, f.tile_n);
        const double  most = group_m != nullptr ? row_tiles.of(f.tile_m)
                                                : double(plan->group_num) * double(gg::cdiv(rows, f.tile_m));
        if ((forced >= 0 && i != forced) || most * double(nt) > double(gg::kMaxLoopTiles))
            continue;
        const double wgs    = row_tiles.of(f.tile_m) * nt;
        const double staged = wgs * (f.tile_m + f.tile_n) * 128.0 * chunks;
        const double round  = wgs / (cus * f.per_cu);
        const double chain  = std::max(1.0, std::ceil(round)) * (gg::cdiv(chunks, f.waves) * f.chunk_us + kFewRoundUs);
        const double us     = kFewFixedUs + std::hypot(bytes / kFewHbm, staged / stage, chain);
        if (best < 0 || us < least) {
            least  = us;
            best   = i;
            rounds = round;
        }
    }
    return forced >= 0 || least < few_gain(dgrad, chunks, rounds) * other ? best : -1;
}

// The few-row kernel's operand format of a plan.
int few_format(const gg_plan *plan) {
    switch (plan->mode / 4) {
    case gg::kInE4M3: return gg::kFewE4M3;
    case gg::kInE5M2: return gg::kFewE5M2;
    case gg::kInE5M2xE4M3: return gg::kFewE5M2xE4M3;
    default: return plan->dtype == GG_DTYPE_FP16 ? gg::kFewF16 : gg::kFewBF16;
    }
}

// The tiles of a few-row plan in its arguments (after fill_args) and its launch: one workgroup per
// tile of at most `tiles`, in whole XCD rows (a workgroup goes on to further tiles if there are more).
void few_args(gg_plan *plan, int64_t tiles) {
    gg::KernelArgs &a = plan->args;
    a.tile_m          = gg::kFewInstances[plan->few].tile_m;
    a.tile_n          = gg::kFewInstances[plan->few].tile_n;
    a.n_tiles         = static_cast<int>(gg::cdiv(plan->n, a.tile_n));
    a.d_total         = nullptr;
    if (plan->mode % 4 == gg::kDgrad) {
        a.lda = static_cast<int>(plan->k);
        a.ldb = static_cast<int>(plan->n);
    }
    plan->grid = static_cast<int>(gg::cdiv(std::min<int64_t>(tiles, gg::kMaxLoopGrid), 8) * 8);
}

std::string few_detail(const gg_plan *plan, const std::string &what) {
    return "mi355x few-row " + std::to_string(plan->args.tile_m) + "x" + std::to_string(plan->args.tile_n) + " " + what +
           " grid=" + std::to_string(plan->grid) +
           (plan->device_lens ? std::string(plan->in_kernel_table ? " tiles=device (device group sizes, in-kernel table)"
                                                                  : " tiles=device (device group sizes)")
                              : " tiles=" + std::to_string(plan->total_tiles));
}

// 128 x 128 tiles (gg_wfew.hip) for wgrad plans whose groups have few rows: the persistent kernel
// runs at least four K steps per 256 x 256 tile and stores it 8 bytes per lane and row, this one
// runs the chunks there are and stores whole rows. Chosen by a launch-time model in microseconds,
// taken at a share (gain) of the persistent plan's time (|a, b| = sqrt(a^2 + b^2)):
//   few:        kWgradFewFixedUs + |bytes / kWgradFewHbm,
//                                   tiles per CU x tile + chunks x |one chunk's latency, tiles per CU x chunk||
//   persistent: kWgradFixedUs + |bytes / kWgradHbm, rounds x (tile + max(4, K steps) x step)|
// with the groups' average K steps. Fitted to 320 random problems of 1-64 groups, 1-8000 rows each,
// n and k 512-14336, bf16 and fp8 (MI355X, both kernels timed). On 900 others that the model takes at 0.9,
// half of them of 300-3500 rows per group, each with its operands in cache and from HBM in turn: up to
// 64 rows per group 1.8x (HBM 1.8x), 65-256 1.5x. Past 300 rows it pays where 256 x 256 tiles leave CUs idle,
// but inputs from HBM cost it more than the persistent kernel, and of the problems under two rounds of
// workgroups 41 were slower, down to 0.71x; at 0.73 two are (0.94x). With CUs full it loses (0.7-0.9x: a 64 x 64
// quarter per wave reads twice the LDS bytes per MFMA of the persistent kernel's 128 x 128).
// GG_SMALL in the environment turns it off; without it, GG_WFEW=1 takes it and GG_WFEW=0 does not.
constexpr double kWgradFewFixedUs = 3.7, kWgradFixedUs = 7.8; // us
constexpr double kWgradFewHbm = 6.1e6, kWgradHbm = 5.1e6;                          // bytes per us

int64_t wgrad_few_tiles(const gg_plan *plan, int64_t m_out) {
    return int64_t(plan->group_num) * gg::cdiv(m_out, gg::kWgradFewTile) * gg::cdiv(plan->n, gg::kWgradFewTile);
}

bool choose_wgrad_few(const gg_plan *plan, const int64_t *group_m, int64_t m_out, int64_t rows, int cus) {
    if (const char *env = std::getenv("GG_SMALL"); env != nullptr && *env != '\0')
        return false;
    const double tiles = static_cast<double>(wgrad_few_tiles(plan, m_out));
    if (gg::one_tile_grid(wgrad_few_tiles(plan, m_out), gg::kWgradFewThreads) == 0)
        return false;
    if (const char *env = std::getenv("GG_WFEW"); env != nullptr && *env != '\0')
        return std::atoi(env) != 0;
    const bool f8      = plan->mode / 4 != gg::kIn16;
    const int  es      = f8 ? 1 : 2;
    const auto average = [&](int rows_log2, int least) { // K steps of 2^rows_log2 rows of a group
        if (group_m == nullptr)
            return std::max<double>(least, std::ldexp(double(rows) / plan->group_num, -rows_log2) + 0.5);
        int64_t sum = 0;
        for (int g = 0; g < plan->group_num; ++g)
            sum += std::max<int64_t>(least, (group_m[g] + (1 << rows_log2) - 1) >> rows_log2);
        return double(sum) / plan->group_num;
    };
    const double bytes  = double(plan->group_num) * m_out * plan->n * 2 + double(rows) * (m_out + plan->n) * es;
    const double wide   = double(plan->group_num) * gg::cdiv(m_out, gg::kTileM) * gg::cdiv(plan->n, gg::kTileN);
    const double steps  = average(f8 ? 7 : 6, gg::kCrossMinStepsHost);
    const double chunks = average(f8 ? 7 : 5, 0);
    const double per_cu = std::max(0.25, tiles / cus);
    const double other  = kWgradFixedUs + std::hypot(bytes / kWgradHbm, std::ceil(wide / cus) *
                                                                           (f8 ? 1.75 + 1.2 * steps : 2.1 + 1.14 * steps));
    const double few    = kWgradFewFixedUs +
                       std::hypot(bytes / kWgradFewHbm, f8 ? 0.05 * per_cu + chunks * std::hypot(0.98, 0.55 * per_cu)
                                                           : 0.32 * per_cu + chunks * std::hypot(0.43, 0.24 * per_cu));
    const double gain = rows > 300 * int64_t(plan->group_num) && tiles < 8 * cus ? 0.73 : 0.9; // (4 per CU)
    return few < gain * other;
}

// The launch of such a plan, one workgroup per tile in whole XCD rows (after fill_args; m_out: the
// rows of a group's gradient).
void wgrad_few_args(gg_plan *plan, int64_t m_out, int n_xcd) {
    gg::KernelArgs &a = plan->args;
    a.total_tiles     = static_cast<int>(wgrad_few_tiles(plan, m_out));
    a.m_out           = static_cast<int>(m_out);
    a.d_total         = nullptr;
    plan->wgrad_few   = true;
    plan->grid        = static_cast<int>(gg::one_tile_grid(a.total_tiles, gg::kWgradFewThreads));
    a.n_xcd           = plan->grid % n_xcd == 0 ? n_xcd : 1;
}

// Turns a host-size forward or dgrad plan (its problem set) into a few-row plan where
// choose_few_rows takes one: the group table of the instance's tiles and the launch.
int use_few_rows(gg_plan *plan, const int64_t *group_m, const float *x_scale, const float *w_scale,
                 const std::string &what) {
    Device dev;
    if (current_device(&dev) != GG_OK)
        return GG_ERR_HIP;
    const int few = choose_few_rows(plan, group_m, plan->total_m, dev.cus);
    if (few < 0)
        return GG_OK;
    const gg::FewInstance      &f = gg::kFewInstances[few];
    std::vector<gg::GroupEntry> table(static_cast<size_t>(plan->group_num));
    const int64_t tiles = gg::build_group_table(group_m, plan->group_num, gg::cdiv(plan->n, f.tile_n), table.data(), 0, f.tile_m);
    if (tiles <= 0)
        return GG_OK;
    plan->table       = std::move(table);
    plan->few         = few;
    plan->total_tiles = static_cast<int>(tiles);
    plan->grid        = 0;
    fill_args(plan, 1);
    few_args(plan, tiles);
    const int n_xcd        = dev.n_xcd;
    plan->args.n_xcd       = plan->grid % n_xcd == 0 ? n_xcd : 1;
    plan->args.total_tiles = plan->total_tiles;
    plan->args.x_scale     = x_scale;
    plan->args.w_scale     = w_scale;
    if (!plan->one_call)
        plan->detail = few_detail(plan, what);
    return GG_OK;
}

// Whether a gg_call plan, which is used once, has tile descriptors (setup_tile_desc): where the walk
// without them is long for the tiles there are. A workgroup's scan of the table takes about 90 ns per
// group, a descriptor about 20-40 ns to build and bring to the device. Torch-level forward calls, us
// without -> with descriptors (MI355X): 2048 groups of 8 rows, N = K = 256, 2048 tiles 434 -> 238; 256
// groups, 512 x 512, 512 tiles 90 -> 77; 128 groups, 1024 x 512, 512 tiles 77 -> 71. Without it stays
// better for 1024 groups and 8192 tiles (490, with: 501), 64 groups, 2048 x 1024, 512 tiles (91, 94), 32
// of 520 rows, 2880 x 2880 (279, 296) and 8 of 4096, 14336 x 4096 (2596, 2625).
bool one_call_desc(const gg_plan *plan) {
    return plan->group_num >= 128 && plan->total_tiles <= 4 * int64_t(plan->group_num);
}

// Tile descriptors of forward, dgrad and wgrad plans of whole tiles (host-size tables): every
// workgroup's tiles in the kernel's own walk (xcd_remap, then locate_tile over the plan's group
// table with its tile rows and N-tiles), so that the kernel reads a tile's first row, group and
// N-tile from a lane of a register instead of recomputing them between its K loops. Not built
// (the kernel walks the table itself) with split-K, a tail split, more than kMaxDescPerWg tiles
// per workgroup or rows past 2^31 (output rows, and for wgrad the input tokens whose offsets its
// descriptors hold). GG_TILE_DESC=0 in the environment turns them off.
int setup_tile_desc(gg_plan *plan, const int64_t *group_m) {
    gg::KernelArgs &a   = plan->args;
    const char     *env = std::getenv("GG_TILE_DESC");
    if ((env != nullptr && env[0] == '0') || (plan->one_call && !one_call_desc(plan)) || a.splits > 1 ||
        a.tail_splits > 1 || plan->grid <= 0 || !gg::desc_rows_fit(group_m, plan->group_num, plan->total_m))
        return GG_OK;
    const int per_wg = static_cast<int>(gg::cdiv(plan->total_tiles, plan->grid));
    if (per_wg > gg::kMaxDescPerWg)
        return GG_OK;
    // wgrad: every group owns m_out / 256 x N-tiles output tiles whatever its size
    const bool    wgrad    = plan->mode % 4 == gg::kWgrad;
    const int64_t out_rows = wgrad ? a.m_out : 0;
    if (wgrad && (gg::cdiv(out_rows, a.tile_m) > 0xffff || a.n_tiles > 0x7fff))
        return GG_OK;
    std::vector<gg::GroupEntry> table(static_cast<size_t>(plan->group_num));
    const int64_t tiles = gg::build_group_table(group_m, plan->group_num, a.n_tiles, table.data(), out_rows, a.tile_m);
    if (tiles != plan->total_tiles)
        return fail(GG_ERR_INVALID, "tile descriptors: the group table's tile count differs from the plan's");
    // wgrad groups are walked by descending K steps, every other round backwards (snake_slot), so
    // that ragged groups load the workgroups evenly; equal groups keep their own order
    std::vector<int> order(static_cast<size_t>(plan->group_num));
    std::iota(order.begin(), order.end(), 0);
    if (wgrad) {
        const int rows_per = plan->mode / 4 == gg::kIn16 ? gg::kTileK : 128;
        const auto steps   = [&](int g) { return std::max<int64_t>(gg::kCrossMinStepsHost, gg::cdiv(group_m[g], rows_per)); };
        std::stable_sort(order.begin(), order.end(), [&](int l, int r) { return steps(l) > steps(r); });
    }
    // (in the order of the logical tiles, so that locate_tile's hint scans the table once for all of them:
    // scanning it again for every workgroup, 8192 groups took 1.17 ms to prepare, 0.63 now)
    std::vector<gg::TileDesc> desc(static_cast<size_t>(plan->grid) * per_wg, gg::TileDesc{0, 0, 0, 0});
    int                       g = 0;
    gg::slots_by_tile(plan->total_tiles, plan->grid, a.n_xcd, [&](int round, int i, int L) {
        const int base  = round * plan->grid; // (snake_slot is its own inverse)
        const int wg    = wgrad ? gg::snake_slot(base + i, plan->total_tiles, plan->grid) - base : i;
        gg::TileDesc &d = desc[static_cast<size_t>(wg) * per_wg + round];
        int tm, tn;
        gg::locate_tile(L, table.data(), plan->group_num, a.n_tiles, a.band, &g, &tm, &tn, static_cast<int>(out_rows),
                        a.tile_m);
        if (wgrad) { // the group's first token, (N-tile << 16) | M-tile, the group's tokens
            const int og = order[static_cast<size_t>(g)];
            d = gg::TileDesc{static_cast<int32_t>(table[og].row0), og, (tn << 16) | tm, table[og].m};
            return;
        }
        const int64_t r0 = table[g].row0 + static_cast<int64_t>(tm) * a.tile_m;
        const int     mv = static_cast<int>(std::min<int64_t>(a.tile_m, table[g].m - static_cast<int64_t>(tm) * a.tile_m));
        d = gg::TileDesc{static_cast<int32_t>(r0), g, (tn << 9) | mv, 0};
    });
    plan->desc    = std::move(desc);
    a.desc_per_wg = per_wg;
    return GG_OK;
}

} // namespace

namespace {

// ---------------------------------------------------------------------------------------
// Device-resident group sizes: the plan builder shared by gg_prepare_device_lens_op (a plan that
// owns its table, hipMalloc'd) and gg_run_device_lens_noalloc (one call that allocates nothing:
// the table and its header live in the device's `scratch` array below).
// ---------------------------------------------------------------------------------------

// Scratch of the allocation-free entry point: the group table (16 bytes per group) and its
// header. One copy per GPU, held until the process ends; every call on a GPU shares it, so
// calls that overlap on one GPU (two streams, two host threads) race on it. Host code never
// names `scratch` in a kernel argument or copy: it uses the device address that
// hipGetSymbolAddress gives for the current device (noalloc_scratch).
constexpr int    kNoAllocMaxGroups  = 8192;
constexpr size_t kNoAllocTableBytes = size_t(kNoAllocMaxGroups) * sizeof(gg::GroupEntry);
constexpr size_t kScratchBytes      = kNoAllocTableBytes + 256; // + the TableHeader, padded
static_assert(sizeof(gg::TableHeader) <= 256, "the header fits behind the largest table");
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// The current device's scratch address, looked up on its first use with that device current.
int noalloc_scratch(void **out) {
    static std::mutex mu;
    static void      *known[kMaxDevices];
    int        dev = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess)
        return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices)
        return fail(GG_ERR_UNSUPPORTED, "device index " + std::to_string(dev) + " beyond " + std::to_string(kMaxDevices));
    std::lock_guard<std::mutex> lock(mu);
    if (known[dev] == nullptr) {
        void *p = nullptr;
        e       = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (p == nullptr || (reinterpret_cast<uintptr_t>(p) & 255u) != 0)
            return fail(GG_ERR_HIP, "hipGetSymbolAddress(scratch) gave a null or misaligned address");
        known[dev] = p;
    }
    *out = known[dev];
    return GG_OK;
}

// Validates a device-size problem (the rules of gg_prepare_device_lens_op) and fills *plan.
// The group table and its header live in a hipMalloc'd block that the plan owns (kOwned: free_plan
// releases it, also on failure), in the current device's scratch array (kScratch) or in `given`
// (kGiven: device_table_bytes of device memory); only kOwned plans have a detail text. A plan without
// a launch keeps d_groups null.
enum TableMemory { kOwned, kScratch, kGiven };
size_t device_table_bytes(int group_num) { return size_t(group_num) * sizeof(gg::GroupEntry) + sizeof(gg::TableHeader); }

int plan_device_lens(gg_plan *plan, TableMemory memory, void *given, int op, int a_dtype, int b_dtype, int group_num,
                     int64_t total_m, int64_t n, int64_t k, const int64_t *group_lens, const int64_t *group_offs,
                     const void *a, const void *b, const float *a_scale, const float *b_scale, void *out) {
    if (op != GG_OP_FORWARD && op != GG_OP_DGRAD && op != GG_OP_WGRAD)
        return fail(GG_ERR_INVALID, "op must be GG_OP_FORWARD, GG_OP_DGRAD or GG_OP_WGRAD");
    if (total_m < 0 || group_num < 0 || n < 0 || k < 0)
        return fail(GG_ERR_INVALID, "group_num, total_m, n and k must be >= 0");
    if (group_num > 0 && group_lens == nullptr)
        return fail(GG_ERR_INVALID, "group_lens is null");
    // Input formats: two equal 16-bit types, or fp8 (forward: both e4m3 or both e5m2; backward
    // also an e5m2 gradient with e4m3 w / x).
    const bool f8     = a_dtype == GG_DTYPE_FP8_E4M3 || a_dtype == GG_DTYPE_FP8_E5M2;
    int        format = gg::kIn16;
    if (f8) {
        if (a_dtype == GG_DTYPE_FP8_E4M3 && b_dtype == GG_DTYPE_FP8_E4M3)
            format = gg::kInE4M3;
        else if (a_dtype == GG_DTYPE_FP8_E5M2 && b_dtype == GG_DTYPE_FP8_E5M2)
            format = gg::kInE5M2;
        else if (op != GG_OP_FORWARD && a_dtype == GG_DTYPE_FP8_E5M2 && b_dtype == GG_DTYPE_FP8_E4M3)
            format = gg::kInE5M2xE4M3;
        else
            return fail(GG_ERR_INVALID, "unsupported pair of fp8 formats");
    } else if ((a_dtype != GG_DTYPE_BF16 && a_dtype != GG_DTYPE_FP16) || b_dtype != a_dtype) {
        return fail(GG_ERR_INVALID, "dtypes must be equal bf16 / fp16 types, or fp8 formats");
    }
    const int     layout   = op == GG_OP_FORWARD ? gg::kFwd : op == GG_OP_DGRAD ? gg::kDgrad : gg::kWgrad;
    // kernel terms (KernelArgs): output columns N_out, contraction K_c, output rows
    const int64_t n_out    = op == GG_OP_FORWARD ? n : k;
    const int64_t k_c      = op == GG_OP_FORWARD ? k : op == GG_OP_DGRAD ? n : 0; // wgrad: per group
    const int64_t out_rows = op == GG_OP_WGRAD ? int64_t(group_num) * n : total_m;
    const bool    has_output = out_rows > 0 && n_out > 0;
    const bool    reads      = op == GG_OP_WGRAD ? total_m > 0 : (total_m > 0 && k_c > 0);
    if (has_output && (out == nullptr || (reads && (a == nullptr || b == nullptr))))
        return fail(GG_ERR_INVALID, "the inputs and the output must be device pointers");
    if (f8 && has_output && reads && (a_scale == nullptr || b_scale == nullptr))
        return fail(GG_ERR_INVALID, "fp8 scales must be device pointers");
    // 16-byte rows; transposed fp8 operands move 16-column blocks
    const int64_t align_n = (f8 && op != GG_OP_FORWARD) ? 16 : 8;
    const int64_t align_k = f8 ? 16 : 8;
    if (n % align_n != 0)
        return fail(GG_ERR_UNSUPPORTED, "N must be a multiple of " + std::to_string(align_n));
    if (k % align_k != 0)
        return fail(GG_ERR_UNSUPPORTED, "K must be a multiple of " + std::to_string(align_k));
    if (has_output && (!aligned16(out) || (reads && (!aligned16(a) || !aligned16(b)))))
        return fail(GG_ERR_UNSUPPORTED, "buffers must be 16-byte aligned");
    if (k > (int64_t(1) << 21) || n > (int64_t(1) << 21))
        return fail(GG_ERR_UNSUPPORTED, "N and K must be at most 2097152");
    const int64_t lim   = int64_t(1) << 31;
    const int64_t es    = f8 ? 1 : 2;
    const int64_t steps = f8 ? 128 : gg::kTileK;
    if (op == GG_OP_DGRAD && (n + steps) * k * es >= lim)
        return fail(GG_ERR_UNSUPPORTED, "one group's w must be smaller than 2 GiB");
    // wgrad: a group may hold every row
    const int64_t wg_rows = std::max<int64_t>(total_m, gg::kCrossMinStepsHost * steps) + steps;
    if (op == GG_OP_WGRAD && (wg_rows * n * es >= lim || wg_rows * k * es >= lim))
        return fail(GG_ERR_UNSUPPORTED, "grad_out and x rows must be smaller than 2 GiB");
    const int64_t n_tiles = gg::cdiv(n_out, gg::kTileN);
    // wgrad: output tiles do not depend on the sizes, m_out rows per group
    const int64_t wgrad_tiles = op == GG_OP_WGRAD ? int64_t(group_num) * gg::cdiv(n, gg::kTileM) * n_tiles : 0;
    if (wgrad_tiles > INT32_MAX)
        return fail(GG_ERR_UNSUPPORTED, "too many tiles for 32-bit tile indices");

    plan->mode        = gg::make_mode(layout, own_format(f8, reads, a_scale, b_scale) ? format : gg::kIn16);
    plan->dtype       = f8 ? GG_DTYPE_BF16 : a_dtype; // output
    plan->group_num   = group_num;
    plan->n           = n_out;
    plan->k           = k_c;
    plan->total_m     = out_rows;
    plan->in_rows     = total_m;
    plan->x           = a;
    plan->w           = b;
    plan->out         = out;
    plan->device_lens = true;
    plan->d_lens      = group_lens;
    plan->d_offs      = group_offs;
    const bool  noalloc = memory != kOwned;
    std::string what;
    if (!noalloc)
        what = std::string(op == GG_OP_FORWARD ? "" : op == GG_OP_DGRAD ? "dgrad " : "wgrad ") +
               (format == gg::kIn16     ? std::string(a_dtype == GG_DTYPE_BF16 ? "bf16" : "fp16")
                : format == gg::kInE4M3 ? std::string("fp8 e4m3")
                : format == gg::kInE5M2 ? std::string("fp8 e5m2")
                                        : std::string("fp8 e5m2 x e4m3"));
    const bool no_launch = !has_output || group_num == 0 || (op != GG_OP_WGRAD && k_c == 0);
    if (no_launch) {
        // forward / dgrad with an empty contraction: the run zero-fills the output
        if (!noalloc)
            plan->detail = "mi355x " + what + ": no launch (" +
                           (has_output && group_num > 0
                                ? (op == GG_OP_FORWARD ? "K = 0, zero fill" : "empty contraction, zero fill")
                                : "empty output") +
                           ")";
        if (!has_output || group_num == 0)
            plan->total_m = 0;
        return GG_OK;
    }
    const size_t table_bytes = static_cast<size_t>(group_num) * sizeof(gg::GroupEntry);
    Device       dev;
    if (const int st = current_device(&dev); st != GG_OK)
        return st;
    const int cus = dev.cus, n_xcd = dev.n_xcd;
    if (memory == kScratch) {
        void *mem = nullptr;
        if (const int st = noalloc_scratch(&mem); st != GG_OK)
            return st;
        plan->d_groups = static_cast<gg::GroupEntry *>(mem);
        plan->d_header = reinterpret_cast<gg::TableHeader *>(static_cast<char *>(mem) + kNoAllocTableBytes);
    } else {
        if (memory == kOwned) { // one allocation; the header is written by every run
            const hipError_t e = hipMalloc(&plan->mem, device_table_bytes(group_num));
            if (e != hipSuccess) {
                plan->mem = nullptr;
                return hip_fail(e, "group table allocation");
            }
            given = plan->mem;
        }
        plan->d_groups = static_cast<gg::GroupEntry *>(given);
        plan->d_header = reinterpret_cast<gg::TableHeader *>(static_cast<char *>(given) + table_bytes);
    }
    fill_args(plan, 1);
    gg::KernelArgs &ka = plan->args;
    ka.k_tiles         = op == GG_OP_WGRAD ? 1 : static_cast<int>(gg::cdiv(k_c, steps));
    // tails (see KernelArgs): forward has K-major operands only; dgrad's w columns are the k of
    // its output; wgrad's K steps depend on the device-resident sizes, so it keeps the masks
    ka.tails = op == GG_OP_FORWARD ? (k_c % steps != 0)
               : op == GG_OP_DGRAD ? (k_c % steps != 0 || k % gg::kTileN != 0)
                                   : 1;
    ka.x_scale         = f8 ? a_scale : nullptr;
    ka.w_scale         = f8 ? b_scale : nullptr;
    if (op != GG_OP_FORWARD) {
        ka.lda = static_cast<int>(n);
        ka.ldb = static_cast<int>(k);
    }
    if (op != GG_OP_WGRAD)
        plan->few = choose_few_rows(plan, nullptr, total_m, cus);
    if (plan->few >= 0) {
        const gg::FewInstance &f = gg::kFewInstances[plan->few];
        few_args(plan, (total_m / f.tile_m + std::min<int64_t>(group_num, total_m)) * gg::cdiv(n_out, f.tile_n));
        ka.total_tiles = 0;
        ka.d_total     = &plan->d_header->run_tiles;
    } else if (op == GG_OP_WGRAD) {
        // The K-step counts depend on the sizes; a cross-tile wgrad tile runs at least
        // kCrossMinStepsHost of them (zeros past its group's rows), so the cross-tile variant runs.
        ka.m_out          = static_cast<int>(n);
        ka.min_steps      = gg::kCrossMinStepsHost;
        plan->total_tiles = static_cast<int>(wgrad_tiles);
        plan->grid        = static_cast<int>(std::min<int64_t>(cus, wgrad_tiles));
        ka.total_tiles    = plan->total_tiles;
        ka.d_total        = nullptr;
    } else {
        // Tile count is unknown here: one workgroup per CU, or fewer if even the largest routing
        // (every group's rows tiled separately) has fewer tiles.
        const int64_t max_tiles = (gg::cdiv(total_m, gg::kTileM) + group_num) * n_tiles;
        plan->grid     = static_cast<int>(std::min<int64_t>(cus, max_tiles));
        ka.total_tiles = 0;
        ka.d_total     = &plan->d_header->total_tiles;
    }
    // At most kInKernelTableGroups groups: the GEMM builds the table itself (one group per lane of
    // every wave) and writes the header, so a run is one launch. Not for an fp8 wgrad plan that
    // would run the per-tile variant (only in builds without the cross-tile pipeline): that
    // instance has no in-kernel table.
    gg::KernelArgs probe = ka;
    probe.d_lens         = group_lens;
    const bool lane_table_ok = !(f8 && op == GG_OP_WGRAD && !gg::uses_cross_tile(probe, plan->grid, plan->mode));
    if (group_num <= gg::kInKernelTableGroups && lane_table_ok) {
        plan->in_kernel_table = true;
        ka.d_lens             = group_lens;
        ka.d_offs             = group_offs;
        ka.lens_rows          = total_m;
        ka.d_header           = plan->d_header;
        ka.d_total            = nullptr;
    }
    ka.n_xcd = plan->grid % n_xcd == 0 ? n_xcd : 1;
    if (op == GG_OP_WGRAD && choose_wgrad_few(plan, nullptr, n, total_m, cus))
        wgrad_few_args(plan, n, n_xcd);
    if (!noalloc && plan->wgrad_few)
        plan->detail = "mi355x " + what + " few-row 128x128 grid=" + std::to_string(plan->grid) + " tiles=" +
                       std::to_string(ka.total_tiles) +
                       (plan->in_kernel_table ? " (device group sizes, in-kernel table)" : " (device group sizes)");
    else if (!noalloc && plan->few >= 0)
        plan->detail = few_detail(plan, what);
    else if (!noalloc)
        plan->detail = "mi355x " + what + " persistent 256x256x" + std::to_string(f8 ? 128 : 64) + " grid=" +
                       std::to_string(plan->grid) + " tiles=" +
                       (op == GG_OP_WGRAD ? std::to_string(plan->total_tiles) : std::string("device")) +
                       " xcd=" + std::to_string(ka.n_xcd) +
                       (gg::uses_cross_tile(ka, plan->grid, plan->mode) ? " cross-tile" : " per-tile") +
                       (ka.band != gg::kBand ? " band=" + std::to_string(ka.band) : "") +
                       (plan->in_kernel_table ? " (device group sizes, in-kernel table)" : " (device group sizes)");
    return GG_OK;
}

int run_few(const gg_plan *plan, hipStream_t s) {
    const hipError_t e = plan->wgrad_few ? gg::launch_wgrad_few(plan->args, few_format(plan), plan->grid, s)
                                         : gg::launch_few_gemm(plan->args, few_format(plan), plan->mode % 4 == gg::kDgrad,
                                                               plan->few, plan->grid, s);
    return e == hipSuccess ? GG_OK : hip_fail(e, "few-row GEMM launch");
}

// Enqueue a plan's launches on `stream` (gg_run). zero_kernel: an empty contraction zero-fills
// the output with a fill kernel instead of hipMemsetAsync (which a captured graph must not
// hold).
int run_plan(const gg_plan *plan, void *stream, bool zero_kernel) {
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (plan->device_lens && plan->d_groups != nullptr) {
        hipError_t e = hipSuccess;
        if (!plan->in_kernel_table) {
            e = gg::launch_build_group_table(plan->d_lens, plan->d_offs, plan->group_num, plan->in_rows,
                                             plan->args.n_tiles, plan->d_groups, plan->d_header, s,
                                             plan->args.m_out, plan->args.tile_m,
                                             plan->few >= 0 ? static_cast<int>(gg::cdiv(plan->n, gg::kTileN)) : 0);
            if (e != hipSuccess)
                return hip_fail(e, "group table launch");
        }
        if (plan->few >= 0 || plan->wgrad_few)
            return run_few(plan, s);
        e = gg::launch_grouped_gemm(plan->args, plan->dtype == GG_DTYPE_FP16, plan->grid, s, plan->mode);
        if (e != hipSuccess)
            return hip_fail(e, "grouped GEMM launch");
        return GG_OK;
    }
    if (plan->total_tiles == 0) {
        // K == 0 with a non-empty output: out = 0.
        if (plan->total_m > 0 && plan->n > 0 && plan->k == 0) {
            const size_t     bytes = size_t(plan->total_m) * plan->n * 2;
            const hipError_t e     = zero_kernel ? gg::launch_zero_fill(plan->out, bytes, s)
                                                 : hipMemsetAsync(plan->out, 0, bytes, s);
            if (e != hipSuccess)
                return hip_fail(e, zero_kernel ? "zero fill launch" : "hipMemsetAsync");
        }
        return GG_OK;
    }
    if (plan->few >= 0 || plan->wgrad_few)
        return run_few(plan, s);
    if (plan->small) {
        const hipError_t e = gg::launch_small_gemm(plan->sargs, plan->dtype == GG_DTYPE_FP16, s);
        return e == hipSuccess ? GG_OK : hip_fail(e, "small-tile GEMM launch");
    }
    hipError_t e = gg::launch_grouped_gemm(plan->args, plan->dtype == GG_DTYPE_FP16, plan->grid, s, plan->mode);
    if (e != hipSuccess)
        return hip_fail(e, "grouped GEMM launch");
    if (plan->args.splits > 1) {
        e = gg::launch_split_reduce(plan->args, plan->dtype == GG_DTYPE_FP16, s, plan->mode);
        if (e != hipSuccess)
            return hip_fail(e, "split-K reduction launch");
    }
    if (plan->args.tail_splits > 1) {
        e = gg::launch_tail_reduce(plan->args, plan->dtype == GG_DTYPE_FP16, plan->grid, s);
        if (e != hipSuccess)
            return hip_fail(e, "tail-split reduction launch");
    }
    return GG_OK;
}

} // namespace

extern "C" {

// Validates a host-size forward problem and fills *plan (nothing on the device).
static int plan_forward(gg_plan *plan, int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
                        const void *x, const void *w, void *out) {
    if (group_num > 0 && group_m == nullptr)
        return fail(GG_ERR_INVALID, "group_m is null");
    int64_t total_m = 0;
    for (int g = 0; g < group_num; ++g) {
        if (group_m[g] < 0)
            return fail(GG_ERR_INVALID, "group_m[" + std::to_string(g) + "] < 0");
        total_m += group_m[g];
    }
    const bool has_output = total_m > 0 && n > 0;
    const int  st         = check_problem(dtype, group_num, n, k, has_output, x, w, out);
    if (st != GG_OK)
        return st;

    plan->dtype     = dtype;
    plan->group_num = group_num;
    plan->n         = n;
    plan->k         = k;
    plan->total_m   = total_m;
    plan->x         = x;
    plan->w         = w;
    plan->out       = out;

    // Group table: row offset, rows and first tile of every group (empty groups own no
    // tiles; the kernel steps over them while scanning forward).
    const int64_t n_tiles = gg::cdiv(n, gg::kTileN);
    plan->table.resize(static_cast<size_t>(group_num));
    const int64_t tiles = gg::build_group_table(group_m, group_num, n_tiles, plan->table.data());
    if (tiles < 0)
        return fail(GG_ERR_UNSUPPORTED, "too many rows or tiles for 32-bit tile indices");
    plan->total_tiles = has_output && k > 0 ? static_cast<int>(tiles) : 0;
    if (plan->total_tiles == 0) {
        plan->table.clear();
        plan->detail = "mi355x: no launch (" + std::string(has_output ? "K = 0, zero fill" : "empty output") + ")";
        return GG_OK;
    }
    if (const int st2 = use_few_rows(plan, group_m, nullptr, nullptr, dtype == GG_DTYPE_BF16 ? "bf16" : "fp16");
        st2 != GG_OK || plan->few >= 0)
        return st2;
    Device dev;
    if (current_device(&dev) != GG_OK)
        return GG_ERR_HIP;
    // Persistent grid: one workgroup per CU (160 KB of LDS each), never more than tiles.
    plan->grid = std::min(dev.cus, plan->total_tiles);
    fill_args(plan, dev.n_xcd);
    gg::KernelArgs &a = plan->args;
    a.total_tiles     = plan->total_tiles;
    a.d_total         = nullptr;
    a.tails           = k % gg::kTileK != 0; // K-major operands: only a partial K step
    setup_split_k(plan, dev);
    if (const int st2 = use_short_tiles(plan, group_m); st2 != GG_OK)
        return st2;
    use_short_wide_tiles(plan, group_m, dev);
    use_narrow_tiles(plan, group_m, dev);
    setup_tail_split(plan);
    if (const int st2 = setup_tile_desc(plan, group_m); st2 != GG_OK)
        return st2;
    use_small_tiles(plan, group_m, dev);
    if (plan->one_call)
        return GG_OK;
    const std::string dt = dtype == GG_DTYPE_BF16 ? "bf16" : "fp16";
    if (plan->small)
        plan->detail = "mi355x small 128x128x64 " + dt + " grid=" + std::to_string(plan->grid) +
                       " tiles=" + std::to_string(plan->total_tiles) +
                       (plan->sargs.stages == gg::kSmallStagesTwo ? " two-per-cu" : "") +
                       (plan->sargs.splits > 1 ? " split-k=" + std::to_string(plan->sargs.splits) : "");
    else
        plan->detail = "mi355x persistent " + std::to_string(a.tile_m) + "x" + std::to_string(a.tile_n) +
                       "x64 " + dt + " grid=" + std::to_string(plan->grid) +
                       " tiles=" + std::to_string(plan->total_tiles) + " xcd=" + std::to_string(a.n_xcd) +
                       (gg::uses_cross_tile(a, plan->grid) ? " cross-tile" : " per-tile") +
                       (a.band != gg::kBand ? " band=" + std::to_string(a.band) : "") +
                       (a.splits > 1 ? " split-k=" + std::to_string(a.splits) : "") +
                       (a.tail_splits > 1 ? " tail-split=" + std::to_string(a.tail_splits) : "");
    return GG_OK;
}

// A prepare entry point: a new plan, filled by `fill`, its device memory allocated and uploaded.
extern "C++" {
template <typename F> static int new_plan(gg_plan **plan_out, void *stream, F fill) {
    g_last_error.clear();
    if (plan_out == nullptr)
        return fail(GG_ERR_INVALID, "plan_out is null");
    *plan_out  = nullptr;
    auto *plan = new (std::nothrow) gg_plan;
    if (plan == nullptr)
        return fail(GG_ERR_INVALID, "out of host memory");
    int st = fill(plan);
    if (st == GG_OK)
        st = allocate_plan(plan, static_cast<hipStream_t>(stream));
    if (st != GG_OK) {
        free_plan(plan);
        return st;
    }
    *plan_out = plan;
    return GG_OK;
}
}

int gg_prepare(int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
               const void *x, const void *w, void *out, void *stream, gg_plan **plan_out) {
    return new_plan(plan_out, stream, [&](gg_plan *plan) { return plan_forward(plan, dtype, group_num, n, k, group_m, x, w, out); });
}

// Backward plans in kernel terms (see KernelArgs): out (rows x N) = A B^T per group with the
// contraction K. dgrad: A = grad_out (K-major, row stride n), B^T = w[g] stored n x k,
// N = k, K = n. wgrad: A^T = grad_out rows of the group (row stride n), B^T = x rows (row stride
// k), out = grad_w[g] n x k, N = k, K = the group's rows.
// dtype_a / dtype_b: formats of grad_out and of the other operand. 16-bit: both the same, no
// scales. fp8: e4m3 x e4m3, e5m2 x e5m2 or e5m2 gradient x e4m3, bf16 out scaled by a_scale[0] *
// b_scale[g].
static int plan_backward(gg_plan *plan, int layout, int dtype_a, int dtype_b, int group_num, int64_t n, int64_t k,
                         const int64_t *group_m, const void *a, const void *b, const float *a_scale,
                         const float *b_scale, void *out) {
    if (group_num > 0 && group_m == nullptr)
        return fail(GG_ERR_INVALID, "group_m is null");
    const bool f8     = dtype_a == GG_DTYPE_FP8_E4M3 || dtype_a == GG_DTYPE_FP8_E5M2;
    int        format = gg::kIn16;
    if (f8) {
        if (dtype_a == GG_DTYPE_FP8_E4M3 && dtype_b == GG_DTYPE_FP8_E4M3)
            format = gg::kInE4M3;
        else if (dtype_a == GG_DTYPE_FP8_E5M2 && dtype_b == GG_DTYPE_FP8_E5M2)
            format = gg::kInE5M2;
        else if (dtype_a == GG_DTYPE_FP8_E5M2 && dtype_b == GG_DTYPE_FP8_E4M3)
            format = gg::kInE5M2xE4M3;
        else
            return fail(GG_ERR_INVALID, "fp8 formats must be e4m3 x e4m3, e5m2 x e5m2 or e5m2 gradient x e4m3");
    } else if ((dtype_a != GG_DTYPE_BF16 && dtype_a != GG_DTYPE_FP16) || dtype_b != dtype_a) {
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    }
    int64_t total_m = 0, max_m = 0;
    for (int g = 0; g < group_num; ++g) {
        if (group_m[g] < 0)
            return fail(GG_ERR_INVALID, "group_m[" + std::to_string(g) + "] < 0");
        total_m += group_m[g];
        max_m = std::max(max_m, group_m[g]);
    }
    const bool dgrad = layout == gg::kDgrad;
    // Output rows: grad_x has total_m, grad_w has group_num * n.
    const int64_t out_rows   = dgrad ? total_m : int64_t(group_num) * n;
    const bool    has_output = out_rows > 0 && k > 0;
    // Both operands are read when the contraction (n for dgrad, the rows for wgrad) is non-zero.
    const bool reads = dgrad ? (total_m > 0 && n > 0) : (total_m > 0);
    if (group_num < 0 || n < 0 || k < 0)
        return fail(GG_ERR_INVALID, "group_num, n and k must be >= 0");
    if (has_output && (out == nullptr || (reads && (a == nullptr || b == nullptr))))
        return fail(GG_ERR_INVALID, "grad_out, the second operand and the output must be device pointers");
    if (f8 && has_output && reads && (a_scale == nullptr || b_scale == nullptr))
        return fail(GG_ERR_INVALID, "fp8 scales must be device pointers");
    // 16-byte rows; fp8 transposed operands move 16-column blocks
    const int64_t align = f8 ? 16 : 8;
    if (n % align != 0)
        return fail(GG_ERR_UNSUPPORTED, std::string("N must be a multiple of ") + std::to_string(align));
    if (k % align != 0)
        return fail(GG_ERR_UNSUPPORTED, std::string("K must be a multiple of ") + std::to_string(align));
    if (has_output && (!aligned16(out) || (reads && (!aligned16(a) || !aligned16(b)))))
        return fail(GG_ERR_UNSUPPORTED, "buffers must be 16-byte aligned");
    if (k > (int64_t(1) << 21) || n > (int64_t(1) << 21))
        return fail(GG_ERR_UNSUPPORTED, "N and K must be at most 2097152");
    // 32-bit byte offsets inside one group's transposed operand, including the rows a partial
    // last K step addresses past the end (up to one step more).
    const int64_t lim   = int64_t(1) << 31;
    const int64_t es    = f8 ? 1 : 2;
    const int64_t steps = f8 ? 128 : gg::kTileK; // contraction rows per K step
    if (dgrad && (n + steps) * k * es >= lim)
        return fail(GG_ERR_UNSUPPORTED, "one group's w must be smaller than 2 GiB");
    // (wgrad: a short group's tile addresses kCrossMinStepsHost steps)
    const int64_t rows_addr = std::max<int64_t>(max_m, gg::kCrossMinStepsHost * steps) + steps;
    if (!dgrad && (rows_addr * n * es >= lim || rows_addr * k * es >= lim))
        return fail(GG_ERR_UNSUPPORTED, "one group's rows of grad_out and x must be smaller than 2 GiB");

    plan->mode      = gg::make_mode(layout, own_format(f8, reads, a_scale, b_scale) ? format : gg::kIn16);
    plan->dtype     = f8 ? GG_DTYPE_BF16 : dtype_a; // output
    plan->group_num = group_num;
    plan->n         = k;                      // output columns
    plan->k         = dgrad ? n : 0;          // contraction (wgrad: per group)
    plan->total_m   = out_rows;               // rows zeroed when there is nothing to read
    plan->x         = a;
    plan->w         = b;
    plan->out       = out;

    const int64_t n_tiles = gg::cdiv(k, gg::kTileN);
    plan->table.resize(static_cast<size_t>(group_num));
    const int64_t tiles = gg::build_group_table(group_m, group_num, n_tiles, plan->table.data(), dgrad ? 0 : n);
    if (tiles < 0)
        return fail(GG_ERR_UNSUPPORTED, "too many rows or tiles for 32-bit tile indices");
    // dgrad with n == 0: grad_x = 0 (gg_run zero-fills). wgrad with no rows: the tiles run and
    // store zeros (each group's K steps read nothing).
    plan->total_tiles = has_output && (!dgrad || n > 0) ? static_cast<int>(tiles) : 0;
    const std::string what = std::string(dgrad ? "dgrad" : "wgrad") +
                             (format == gg::kIn16         ? ""
                              : format == gg::kInE4M3     ? " fp8 e4m3"
                              : format == gg::kInE5M2     ? " fp8 e5m2"
                                                          : " fp8 e5m2 x e4m3");
    if (plan->total_tiles > 0 && dgrad) {
        const std::string in = f8 ? "" : dtype_a == GG_DTYPE_BF16 ? " bf16" : " fp16";
        if (const int st = use_few_rows(plan, group_m, f8 ? a_scale : nullptr, f8 ? b_scale : nullptr, what + in);
            st != GG_OK || plan->few >= 0)
            return st;
    }
    if (plan->total_tiles > 0) {
        Device dev;
        if (current_device(&dev) != GG_OK)
            return GG_ERR_HIP;
        plan->grid = std::min(dev.cus, plan->total_tiles);
        fill_args(plan, dev.n_xcd);
        gg::KernelArgs &ka = plan->args;
        ka.total_tiles     = plan->total_tiles;
        ka.d_total         = nullptr;
        ka.lda             = static_cast<int>(n);
        ka.ldb             = static_cast<int>(k);
        ka.m_out           = dgrad ? 0 : static_cast<int>(n);
        ka.k_tiles         = dgrad ? static_cast<int>(gg::cdiv(n, steps)) : 1;
        if (!dgrad) // fewest K steps of a tile: a cross-tile wgrad tile runs at least
                    // kCrossMinStepsHost (zeros past a short or empty group's rows)
            ka.min_steps = gg::kCrossMinStepsHost;
        ka.x_scale         = f8 ? a_scale : nullptr;
        ka.w_scale         = f8 ? b_scale : nullptr;
        // tails (see KernelArgs). dgrad: the contraction n and w's columns k. wgrad: every group's
        // rows (its contraction) and the columns of grad_out (n) and x (k).
        if (dgrad) {
            ka.tails = n % steps != 0 || k % gg::kTileN != 0;
        } else { // and the zero steps of a group shorter than kCrossMinStepsHost steps
            bool t = n % gg::kTileN != 0 || k % gg::kTileN != 0;
            for (int g = 0; g < group_num; ++g)
                t = t || group_m[g] % steps != 0 || group_m[g] < gg::kCrossMinStepsHost * steps;
            ka.tails = t;
        }
        if (!dgrad && choose_wgrad_few(plan, group_m, n, total_m, dev.cus)) {
            wgrad_few_args(plan, n, dev.n_xcd);
            plan->total_tiles = ka.total_tiles;
            plan->detail = "mi355x " + what + " few-row 128x128 " + (f8 ? "bf16-out" : dtype_a == GG_DTYPE_BF16 ? "bf16" : "fp16") +
                           " grid=" + std::to_string(plan->grid) + " tiles=" + std::to_string(plan->total_tiles);
            return GG_OK;
        }
        // wgrad's K steps differ per group: no split
        if (dgrad)
            setup_split_k(plan, dev);
        if (dgrad && !f8) // short tiles: the output rows are the groups' tokens
            if (const int st2 = use_short_tiles(plan, group_m); st2 != GG_OK)
                return st2;
        if (const int st3 = setup_tile_desc(plan, group_m); st3 != GG_OK)
            return st3;
        if (plan->one_call)
            return GG_OK;
        plan->detail = "mi355x " + what + " persistent " + std::to_string(ka.tile_m) + "x256x" +
                       std::to_string(f8 ? 128 : 64) + " " +
                       (f8 ? "bf16-out" : dtype_a == GG_DTYPE_BF16 ? "bf16" : "fp16") +
                       " grid=" + std::to_string(plan->grid) + " tiles=" + std::to_string(plan->total_tiles) +
                       " xcd=" + std::to_string(ka.n_xcd) +
                       (gg::uses_cross_tile(ka, plan->grid, plan->mode) ? " cross-tile" : " per-tile") +
                       (ka.band != gg::kBand ? " band=" + std::to_string(ka.band) : "") +
                       (ka.splits > 1 ? " split-k=" + std::to_string(ka.splits) : "") +
                       (ka.tail_splits > 1 ? " tail-split=" + std::to_string(ka.tail_splits) : "");
    } else {
        plan->table.clear();
        plan->detail = "mi355x " + what + ": no launch (" +
                       (has_output ? "empty contraction, zero fill" : "empty output") + ")";
        if (!has_output)
            plan->total_m = 0;
    }
    return GG_OK;
}

static int plan_fp8(gg_plan *plan, int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
                    const void *x, const void *w, const float *x_scale, const float *w_scale, void *out) {
    if (dtype != GG_DTYPE_FP8_E4M3 && dtype != GG_DTYPE_FP8_E5M2)
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_FP8_E4M3 or GG_DTYPE_FP8_E5M2");
    if (group_num > 0 && group_m == nullptr)
        return fail(GG_ERR_INVALID, "group_m is null");
    int64_t total_m = 0;
    for (int g = 0; g < group_num; ++g) {
        if (group_m[g] < 0)
            return fail(GG_ERR_INVALID, "group_m[" + std::to_string(g) + "] < 0");
        total_m += group_m[g];
    }
    if (group_num < 0 || n < 0 || k < 0)
        return fail(GG_ERR_INVALID, "group_num, n and k must be >= 0");
    const bool has_output = total_m > 0 && n > 0;
    if (has_output && (out == nullptr || (k > 0 && (x == nullptr || w == nullptr || x_scale == nullptr ||
                                                    w_scale == nullptr))))
        return fail(GG_ERR_INVALID, "x, w, the scales and out must be device pointers");
    if (n % 8 != 0)
        return fail(GG_ERR_UNSUPPORTED, "N must be a multiple of 8 (16-byte output rows)");
    if (k % 16 != 0)
        return fail(GG_ERR_UNSUPPORTED, "K must be a multiple of 16 for fp8 (16-byte input rows)");
    if (has_output && (!aligned16(out) || (k > 0 && (!aligned16(x) || !aligned16(w)))))
        return fail(GG_ERR_UNSUPPORTED, "x, w and out must be 16-byte aligned");
    if (k > (int64_t(1) << 21) || n > (int64_t(1) << 21))
        return fail(GG_ERR_UNSUPPORTED, "N and K must be at most 2097152");

    plan->mode      = gg::make_mode(gg::kFwd, dtype == GG_DTYPE_FP8_E4M3 ? gg::kInE4M3 : gg::kInE5M2);
    plan->dtype     = GG_DTYPE_BF16; // output
    plan->group_num = group_num;
    plan->n         = n;
    plan->k         = k;
    plan->total_m   = total_m;
    plan->x         = x;
    plan->w         = w;
    plan->out       = out;
    const int64_t n_tiles = gg::cdiv(n, gg::kTileN);
    plan->table.resize(static_cast<size_t>(group_num));
    const int64_t tiles = gg::build_group_table(group_m, group_num, n_tiles, plan->table.data());
    if (tiles < 0)
        return fail(GG_ERR_UNSUPPORTED, "too many rows or tiles for 32-bit tile indices");
    plan->total_tiles = has_output && k > 0 ? static_cast<int>(tiles) : 0;
    if (plan->total_tiles > 0) {
        if (const int st = use_few_rows(plan, group_m, x_scale, w_scale, dtype == GG_DTYPE_FP8_E4M3 ? "fp8 e4m3" : "fp8 e5m2");
            st != GG_OK || plan->few >= 0)
            return st;
        Device dev;
        if (current_device(&dev) != GG_OK)
            return GG_ERR_HIP;
        plan->grid = std::min(dev.cus, plan->total_tiles);
        fill_args(plan, dev.n_xcd);
        gg::KernelArgs &a = plan->args;
        a.total_tiles     = plan->total_tiles;
        a.d_total         = nullptr;
        a.k_tiles         = static_cast<int>(gg::cdiv(k, 128)); // 128 fp8 values per K step
        a.tails           = k % 128 != 0;
        a.x_scale         = x_scale;
        a.w_scale         = w_scale;
        setup_split_k(plan, dev);
        if (const int st3 = setup_tile_desc(plan, group_m); st3 != GG_OK)
            return st3;
        if (plan->one_call)
            return GG_OK;
        plan->detail = std::string("mi355x fp8 ") + (dtype == GG_DTYPE_FP8_E4M3 ? "e4m3" : "e5m2") +
                       " persistent 256x256x128 bf16-out grid=" + std::to_string(plan->grid) +
                       " tiles=" + std::to_string(plan->total_tiles) + " xcd=" + std::to_string(a.n_xcd) +
                       (gg::uses_cross_tile(a, plan->grid, plan->mode) ? " cross-tile" : " per-tile") +
                       (a.band != gg::kBand ? " band=" + std::to_string(a.band) : "") +
                       (a.splits > 1 ? " split-k=" + std::to_string(a.splits) : "") +
                       (a.tail_splits > 1 ? " tail-split=" + std::to_string(a.tail_splits) : "");
    } else {
        plan->table.clear();
        plan->detail = std::string("mi355x fp8: no launch (") +
                       (has_output ? "K = 0, zero fill" : "empty output") + ")";
    }
    return GG_OK;
}

int gg_prepare_fp8(int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
                   const void *x, const void *w, const float *x_scale, const float *w_scale, void *out,
                   void *stream, gg_plan **plan_out) {
    return new_plan(plan_out, stream, [&](gg_plan *plan) {
        return plan_fp8(plan, dtype, group_num, n, k, group_m, x, w, x_scale, w_scale, out);
    });
}

int gg_prepare_dgrad(int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
                     const void *grad_out, const void *w, void *grad_x, void *stream, gg_plan **plan_out) {
    if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_FP16)
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    return new_plan(plan_out, stream, [&](gg_plan *plan) {
        return plan_backward(plan, gg::kDgrad, dtype, dtype, group_num, n, k, group_m, grad_out, w, nullptr, nullptr, grad_x);
    });
}

int gg_prepare_wgrad(int dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
                     const void *grad_out, const void *x, void *grad_w, void *stream, gg_plan **plan_out) {
    if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_FP16)
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    return new_plan(plan_out, stream, [&](gg_plan *plan) {
        return plan_backward(plan, gg::kWgrad, dtype, dtype, group_num, n, k, group_m, grad_out, x, nullptr, nullptr, grad_w);
    });
}

int gg_prepare_dgrad_fp8(int grad_dtype, int w_dtype, int group_num, int64_t n, int64_t k,
                         const int64_t *group_m, const void *grad_out, const void *w, const float *grad_scale,
                         const float *w_scale, void *grad_x, void *stream, gg_plan **plan_out) {
    if (grad_dtype != GG_DTYPE_FP8_E4M3 && grad_dtype != GG_DTYPE_FP8_E5M2)
        return fail(GG_ERR_INVALID, "grad_dtype must be GG_DTYPE_FP8_E4M3 or GG_DTYPE_FP8_E5M2");
    return new_plan(plan_out, stream, [&](gg_plan *plan) {
        return plan_backward(plan, gg::kDgrad, grad_dtype, w_dtype, group_num, n, k, group_m, grad_out, w, grad_scale, w_scale, grad_x);
    });
}

int gg_prepare_wgrad_fp8(int grad_dtype, int x_dtype, int group_num, int64_t n, int64_t k,
                         const int64_t *group_m, const void *grad_out, const void *x, const float *grad_scale,
                         const float *x_scale, void *grad_w, void *stream, gg_plan **plan_out) {
    if (grad_dtype != GG_DTYPE_FP8_E4M3 && grad_dtype != GG_DTYPE_FP8_E5M2)
        return fail(GG_ERR_INVALID, "grad_dtype must be GG_DTYPE_FP8_E4M3 or GG_DTYPE_FP8_E5M2");
    return new_plan(plan_out, stream, [&](gg_plan *plan) {
        return plan_backward(plan, gg::kWgrad, grad_dtype, x_dtype, group_num, n, k, group_m, grad_out, x, grad_scale, x_scale, grad_w);
    });
}

int gg_prepare_device_lens(int dtype, int group_num, int64_t total_m, int64_t n, int64_t k,
                           const int64_t *group_lens, const int64_t *group_offs, const void *x,
                           const void *w, void *out, void *stream, gg_plan **plan_out) {
    if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_FP16) {
        g_last_error.clear();
        if (plan_out != nullptr)
            *plan_out = nullptr;
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    }
    return gg_prepare_device_lens_op(GG_OP_FORWARD, dtype, dtype, group_num, total_m, n, k, group_lens,
                                     group_offs, x, w, nullptr, nullptr, out, stream, plan_out);
}

int gg_prepare_device_lens_op(int op, int a_dtype, int b_dtype, int group_num, int64_t total_m, int64_t n,
                              int64_t k, const int64_t *group_lens, const int64_t *group_offs, const void *a,
                              const void *b, const float *a_scale, const float *b_scale, void *out,
                              void *stream, gg_plan **plan_out) {
    (void)stream;
    g_last_error.clear();
    if (plan_out == nullptr)
        return fail(GG_ERR_INVALID, "plan_out is null");
    *plan_out = nullptr;
    auto *plan = new (std::nothrow) gg_plan;
    if (plan == nullptr)
        return fail(GG_ERR_INVALID, "out of host memory");
    const int st = plan_device_lens(plan, kOwned, nullptr, op, a_dtype, b_dtype, group_num, total_m, n, k, group_lens,
                                    group_offs, a, b, a_scale, b_scale, out);
    if (st != GG_OK) {
        free_plan(plan);
        return st;
    }
    *plan_out = plan;
    return GG_OK;
}

int gg_run_device_lens_noalloc(int op, int a_dtype, int b_dtype, int group_num, int64_t total_m, int64_t n,
                               int64_t k, const int64_t *group_lens, const int64_t *group_offs, const void *a,
                               const void *b, const float *a_scale, const float *b_scale, void *out,
                               void *stream) {
    g_last_error.clear();
    if (group_num > kNoAllocMaxGroups)
        return fail(GG_ERR_UNSUPPORTED, "gg_run_device_lens_noalloc takes at most " +
                                            std::to_string(kNoAllocMaxGroups) + " groups (got " +
                                            std::to_string(group_num) + ")");
    gg_plan plan; // on the stack: its table is the device's scratch array
    const int st = plan_device_lens(&plan, kScratch, nullptr, op, a_dtype, b_dtype, group_num, total_m, n, k, group_lens,
                                    group_offs, a, b, a_scale, b_scale, out);
    if (st != GG_OK)
        return st;
    return run_plan(&plan, stream, true);
}

// What a run's table header says about its device sizes.
static int check_header(const gg::TableHeader &h) {
    if (h.overflow != 0)
        return fail(GG_ERR_INVALID, "device group sizes: more than 2^31 tiles, nothing computed");
    if (h.first_bad >= 0)
        return fail(GG_ERR_INVALID, "device group sizes: group " + std::to_string(h.first_bad) +
                                        " has a negative length or rows outside [0, total_m); "
                                        "its rows were not written");
    return GG_OK;
}

int gg_call(int op, int a_dtype, int b_dtype, int group_num, int64_t n, int64_t k, const int64_t *group_m,
            const void *a, const void *b, const float *a_scale, const float *b_scale, void *out,
            void *workspace, size_t workspace_bytes, size_t *needed, void *stream) {
    g_last_error.clear();
    if (needed == nullptr)
        return fail(GG_ERR_INVALID, "needed is null");
    *needed = 0;
    if (op != GG_OP_FORWARD && op != GG_OP_DGRAD && op != GG_OP_WGRAD)
        return fail(GG_ERR_INVALID, "op must be GG_OP_FORWARD, GG_OP_DGRAD or GG_OP_WGRAD");
    const bool f8 = a_dtype == GG_DTYPE_FP8_E4M3 || a_dtype == GG_DTYPE_FP8_E5M2;
    if (op == GG_OP_FORWARD && a_dtype != b_dtype)
        return fail(GG_ERR_INVALID, "x and w must have one dtype");
    gg_plan plan; // on the stack: its device memory is the caller's workspace
    plan.one_call = true;
    const int st  = op != GG_OP_FORWARD ? plan_backward(&plan, op == GG_OP_DGRAD ? gg::kDgrad : gg::kWgrad, a_dtype, b_dtype,
                                                        group_num, n, k, group_m, a, b, a_scale, b_scale, out)
                    : f8 ? plan_fp8(&plan, a_dtype, group_num, n, k, group_m, a, b, a_scale, b_scale, out)
                         : plan_forward(&plan, a_dtype, group_num, n, k, group_m, a, b, out);
    if (st != GG_OK)
        return st;
    *needed = plan_bytes(&plan);
    if (*needed > workspace_bytes)
        return fail(GG_ERR_WORKSPACE, "workspace of " + std::to_string(workspace_bytes) + " bytes, " +
                                          std::to_string(*needed) + " needed");
    if (*needed > 0 && (workspace == nullptr || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0))
        return fail(GG_ERR_INVALID, "workspace must be 256-byte aligned device memory");
    if (*needed > 0) {
        std::vector<char> image;
        bind_plan(&plan, workspace, &image);
        const hipError_t e = gg::launch_upload(workspace, image.data(), image.size(), static_cast<hipStream_t>(stream));
        if (e != hipSuccess)
            return hip_fail(e, "plan table upload");
    }
    return run_plan(&plan, stream, true);
}

int gg_call_device_lens(int op, int a_dtype, int b_dtype, int group_num, int64_t total_m, int64_t n, int64_t k,
                        const int64_t *group_lens, const int64_t *group_offs, const void *a, const void *b,
                        const float *a_scale, const float *b_scale, void *out, void *workspace,
                        size_t workspace_bytes, void *status, void *stream) {
    g_last_error.clear();
    if (status == nullptr)
        return fail(GG_ERR_INVALID, "status is null");
    auto *header = static_cast<gg::TableHeader *>(status);
    *header      = gg::TableHeader{0, -1, 0, 0};
    if (group_num > 0 && (workspace == nullptr || workspace_bytes < device_table_bytes(group_num) ||
                          (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0))
        return fail(GG_ERR_INVALID, "workspace must be 16 * (group_num + 1) bytes of 256-byte aligned device memory");
    gg_plan plan;
    int     st = plan_device_lens(&plan, kGiven, workspace, op, a_dtype, b_dtype, group_num, total_m, n, k, group_lens,
                                  group_offs, a, b, a_scale, b_scale, out);
    if (st != GG_OK)
        return st;
    if (plan.in_kernel_table) // the GEMM writes the header once, straight to the host
        plan.args.d_header = header;
    st = run_plan(&plan, stream, true);
    if (st == GG_OK && plan.d_header != nullptr && !plan.in_kernel_table) {
        const hipError_t e = hipMemcpyAsync(status, plan.d_header, sizeof(gg::TableHeader), hipMemcpyDeviceToHost,
                                            static_cast<hipStream_t>(stream));
        if (e != hipSuccess)
            return hip_fail(e, "device status read");
    }
    return st;
}

int gg_check_status(const void *status) {
    g_last_error.clear();
    if (status == nullptr)
        return fail(GG_ERR_INVALID, "status is null");
    return check_header(*static_cast<const gg::TableHeader *>(status));
}

int gg_run(const gg_plan *plan, void *stream) {
    if (plan == nullptr)
        return fail(GG_ERR_INVALID, "plan is null");
    return run_plan(plan, stream, false);
}

void gg_release(gg_plan *plan) {
    if (plan == nullptr)
        return;
    free_plan(plan);
}

const char *gg_plan_detail(const gg_plan *plan) { return plan ? plan->detail.c_str() : ""; }

int gg_plan_grid(const gg_plan *plan) { return plan ? plan->grid : 0; }

int gg_plan_tiles(const gg_plan *plan) { return plan ? plan->total_tiles : 0; }

int gg_plan_device_status(const gg_plan *plan, void *stream, int *total_tiles) {
    g_last_error.clear();
    if (plan == nullptr)
        return fail(GG_ERR_INVALID, "plan is null");
    if (!plan->device_lens || plan->d_header == nullptr) {
        if (total_tiles != nullptr)
            *total_tiles = plan->total_tiles;
        return GG_OK;
    }
    gg::TableHeader h{};
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e = hipMemcpyAsync(&h, plan->d_header, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e != hipSuccess)
        return hip_fail(e, "device status read");
    if (total_tiles != nullptr)
        *total_tiles = h.total_tiles;
    return check_header(h);
}

int gg_compute_group_offs(const int64_t *group_lens, int64_t *group_offs, int group_num,
                          void *stream) {
    g_last_error.clear();
    if (group_num < 0)
        return fail(GG_ERR_INVALID, "group_num must be >= 0");
    if (group_offs == nullptr || (group_num > 0 && group_lens == nullptr))
        return fail(GG_ERR_INVALID, "group_lens and group_offs must be device pointers");
    const hipError_t e =
        gg::launch_group_offsets(group_lens, group_offs, group_num, static_cast<hipStream_t>(stream));
    if (e != hipSuccess)
        return hip_fail(e, "group offsets launch");
    return GG_OK;
}

const char *gg_last_error(void) { return g_last_error.c_str(); }

int gg_fill_randn(int dtype, void *p, size_t count, uint64_t seed, void *stream) {
    g_last_error.clear();
    if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_FP16)
        return fail(GG_ERR_INVALID, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_FP16");
    if (count > 0 && p == nullptr)
        return fail(GG_ERR_INVALID, "p is null");
    const hipError_t e = gg::launch_fill_randn(p, count, seed, dtype == GG_DTYPE_FP16,
                                               static_cast<hipStream_t>(stream));
    if (e != hipSuccess)
        return hip_fail(e, "fill launch");
    return GG_OK;
}

int gg_clock_probe(uint64_t *dev_out, double seconds, void *stream) {
    g_last_error.clear();
    if (dev_out == nullptr)
        return fail(GG_ERR_INVALID, "dev_out is null");
    if (!(seconds > 0.0 && seconds <= 10.0))
        return fail(GG_ERR_INVALID, "seconds must be in (0, 10]");
    int        dev = 0, khz = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e == hipSuccess)
        e = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev);
    if (e != hipSuccess)
        return hip_fail(e, "wall clock rate");
    if (khz <= 0)
        return fail(GG_ERR_UNSUPPORTED, "the device reports no wall clock rate");
    const unsigned long long hz    = static_cast<unsigned long long>(khz) * 1000ull;
    const unsigned long long ticks = static_cast<unsigned long long>(seconds * static_cast<double>(hz));
    e = gg::launch_clock_probe(reinterpret_cast<unsigned long long *>(dev_out), ticks, hz,
                               static_cast<hipStream_t>(stream));
    if (e != hipSuccess)
        return hip_fail(e, "clock probe launch");
    return GG_OK;
}

} // extern "C"
