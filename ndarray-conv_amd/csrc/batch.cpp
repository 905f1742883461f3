// Host side of the batched rank-1 path: per-pair validation through the
// single-problem planner, the cost model and its calibration on the device,
// work-queue construction (longest items first), graph capture, and the
// extern "C" entry points declared in ndconv.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <numeric>
#include <string>
#include <vector>

#include "batch.hpp"
#include "border1d.hpp"
#include "plan.hpp"

namespace ndc {
namespace {

struct DevMem {
    void* p = nullptr;
    size_t n = 0;
    DevMem() = default;
    DevMem(const DevMem&) = delete;
    DevMem& operator=(const DevMem&) = delete;
    ~DevMem() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    bool ensure(size_t bytes) {
        if (bytes == 0) bytes = 256;
        if (p && n >= bytes) return true;
        release();
        if (hipMalloc(&p, bytes) != hipSuccess) {
            p = nullptr;
            return false;
        }
        n = bytes;
        return true;
    }
    bool upload(const void* src, size_t bytes) {
        if (!ensure(bytes)) return false;
        return bytes == 0 || hipMemcpy(p, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
    }
};

// Throughput costs (ms per item with the device full of workgroups).
struct CostModel {
    double dir_a, dir_b;     // FP32 direct item: dir_a + dir_b * outputs * taps
    double mfma_a, mfma_b;   // BF16x3 matrix-core item: mfma_a + mfma_b * K-blocks
    double mfma6_a, mfma6_b; // BF16x6 matrix-core item, likewise
    double edge;             // a pair's first and last item more than one inside it
    // tile runs: tile_a per run (the kernel's transform), tile_b per complex tile
    double tile_a[kBatchTileClasses], tile_b[kBatchTileClasses];
    bool measured = false;
};

// Starting point before calibration, and what the calibration falls back to.
CostModel default_costs() {
    CostModel c;
    const double b[kBatchTileClasses] = {4.3e-6, 1.7e-5, 4e-5, 2.9e-4};
    for (int i = 0; i < kBatchTileClasses; ++i) {
        c.tile_a[i] = 0.3 * b[i];
        c.tile_b[i] = b[i];
    }
    c.dir_a = 2e-6;
    c.dir_b = 6e-11;
    c.mfma_a = 4e-6;
    c.mfma_b = 4e-7;
    c.mfma6_a = 4e-6;
    c.mfma6_b = 8e-7;
    c.edge = 1e-6;
    return c;
}

// Shape arithmetic of one pair (from the single-problem planner).
struct PairShape {
    int64_t n, k, p0, pds, out, kdil;
};

int direct_tile(int s) {
    const int cap = (kBatchWindow / 2 - 1) / s + 1;
    return std::min(kBatchDirectTile, std::max(cap, 1));
}

double direct_cost(const CostModel& cm, const PairShape& ps, int s) {
    const int64_t tile = direct_tile(s);
    const int64_t nt = (ps.out + tile - 1) / tile;
    return double(nt) * cm.dir_a + double(std::min<int64_t>(nt, 2)) * cm.edge + cm.dir_b * double(ps.out) * double(ps.k);
}

// Outputs per tile and phase, tiles per phase and complex tiles of a pair in
// tile class c; none when the tile does not take it.
struct TileSplit {
    int64_t V = 0, per_phase = 0, total = 0;
};
TileSplit tile_split(const PairShape& ps, int d, int c) {
    TileSplit r;
    const int64_t N = int64_t(1) << batch_tile_log2(c), reach = ps.pds + int64_t(d) * N;
    // at least an eighth of a tile is outputs; byte offsets of 30 bits, in the
    // 64-bit class positions of 31
    if (ps.k > N * 7 / 8 || reach >= (int64_t(1) << (c == kBatchTileFar ? 31 : 28))) return r;
    r.V = N - ps.k + 1;
    const int64_t U = ps.pds - ps.kdil + 1;
    r.per_phase = ((U + d - 1) / d + r.V - 1) / r.V;
    r.total = (r.per_phase * d + 1) / 2;
    return r;
}

// Workgroups resident at once per CU: 5 of 256 threads (registers), 2 of 512, 1
// of 1024.
constexpr int tile_slots(int c) { return c == 0 ? 5 : c == 1 ? 2 : 1; }

// Tiles of a run: long enough to share the kernel's transform, short enough
// that the chip gets three rounds of runs (at most eight tiles, where the
// kernel's share is small).
int64_t run_tiles(int64_t total, int64_t slots) { return std::max<int64_t>(1, std::min<int64_t>(8, total / (3 * slots))); }

// Tiles of a run that a pair's cost assumes before the batch's are known.
constexpr int kRunTiles = 4;

double tile_cost(const CostModel& cm, const PairShape& ps, int d, int c) {
    const TileSplit t = tile_split(ps, d, c);
    if (t.total <= 0) return INFINITY;
    return cm.tile_b[c] * double(t.total) + cm.tile_a[c] * double((t.total + kRunTiles - 1) / kRunTiles);
}

constexpr int kMethodTile = -4;     // tile class 0; class c is kMethodTile - c
constexpr int kMethodDirect = -1;   // FP32 direct items
constexpr int kMethodMfma = -2;     // BF16x3 matrix-core items
constexpr int kMethodMfma6 = -3;    // BF16x6 matrix-core items

int mfma_nkb(const PairShape& ps) { return int((ps.kdil + 31 + 15) / 16); }

bool mfma_eligible(const PairShape& ps, int s) { return s == 1 && ps.kdil <= kBatchMfmaMaxKdil; }

// BF16x3 meets the batch's accuracy only where every output sums enough
// products of distinct samples for their rounding errors to average (see
// kBf16x3MinTaps): the kernel needs that many taps, and no window may read one
// sample many times over, which a signal shorter than the dilated kernel (a
// circular pad wraps it) or a border repeating one value (Replicate, a
// nonzero constant) would do.  The three-term split has no such limit.
bool bf16x3_admitted(const PairShape& ps, bool repeating_border) {
    return ps.k >= kBf16x3MinTaps && ps.n >= ps.kdil && !repeating_border;
}

double mfma_item_cost(const CostModel& cm, const PairShape& ps, bool six) {
    return six ? cm.mfma6_a + cm.mfma6_b * double(mfma_nkb(ps)) : cm.mfma_a + cm.mfma_b * double(mfma_nkb(ps));
}

double mfma_cost(const CostModel& cm, const PairShape& ps, int s, bool six) {
    if (!mfma_eligible(ps, s)) return INFINITY;
    const int64_t nt = (ps.out + kBatchMfmaTile - 1) / kBatchMfmaTile;
    return double(nt) * mfma_item_cost(cm, ps, six) + double(std::min<int64_t>(nt, 2)) * cm.edge;
}

// The launch that computes a method's pairs: a tile class's, or the queue's.
int group_of(int method) { return method <= kMethodTile ? kMethodTile - method : kBatchTileClasses; }

// What every pair of a batch shares, and the chip's size.
struct BatchForm {
    int s, d;
    int32_t front, back;   // side tags of border1d.hpp
    int cus, blocks;       // CUs, resident workgroups of the queue's kernel
};

// What a pair costs in FP32 (tiles or direct items).
double fp32_cost(const CostModel& cm, const PairShape& ps, int s, int d) {
    double v = direct_cost(cm, ps, s);
    for (int c = 0; c < kBatchTileClasses; ++c) v = std::min(v, tile_cost(cm, ps, d, c));
    return v;
}

// Method of a pair in the queue: kMethodDirect, kMethodMfma or kMethodMfma6.  The
// autotuned form admits split products only to a pair for which they cost
// less than FP32 by its own costs: what launches the rest of the batch uses must
// not lower a pair's precision.  (With all pairs of a batch of 4096 moved to the
// queue together, the median error against 64 bits was 3.4e-6; FP32 tiles give 2.1e-7.)
int queue_method(const CostModel& cm, const PairShape& ps, int s, int d, int algo, bool repeating_border) {
    const bool x3 = bf16x3_admitted(ps, repeating_border);
    if (algo == NDC_BATCH_MFMA && mfma_eligible(ps, s)) return x3 ? kMethodMfma : kMethodMfma6;
    if (algo == NDC_BATCH_BF16X6 && mfma_eligible(ps, s)) return kMethodMfma6;
    if (algo == NDC_BATCH_AUTO_BF16X3 && mfma_cost(cm, ps, s, !x3) < fp32_cost(cm, ps, s, d))
        return x3 ? kMethodMfma : kMethodMfma6;
    return kMethodDirect;
}

// Methods of all pairs: a tile class or the queue's method, whichever costs
// less among the launches that the batch uses, and what that is estimated to
// take.  The costs are those of a full chip; a launch takes at least as long as
// one run on it, the queue's about one item longer than its work, and all
// choices of launches are compared with that: a few pairs of some length do not get a
// launch of their own, and a small batch is one launch (509 pairs, 6.3 M outputs: 20 us
// in one launch of 1024-point tiles, 29 us with 6 pairs in a launch of 4096-point
// tiles beside it).
std::vector<int> choose_launches(const CostModel& cm, const std::vector<PairShape>& sh, const BatchForm& f, int algo,
                                 bool repeating_border, double* estimate) {
    constexpr int Q = kBatchTileClasses, G = Q + 1;
    constexpr double kLaunchMs = 3e-3;
    const size_t P = sh.size();
    std::vector<int> m(P), queue(P);
    std::vector<std::array<double, G>> cost(P);
    std::vector<std::array<int64_t, Q>> split(P);
    const bool tiles = algo == NDC_BATCH_AUTO || algo == NDC_BATCH_AUTO_BF16X3 || algo == NDC_BATCH_FFT;
    std::vector<double> item(P);
    for (size_t i = 0; i < P; ++i) {
        const PairShape& ps = sh[i];
        queue[i] = m[i] = queue_method(cm, ps, f.s, f.d, algo, repeating_border);
        bool any = false;
        for (int c = 0; c < Q; ++c) {
            // where the queue's method is a fixed one, tiles take what it does not
            const bool ok = tiles || (algo != NDC_BATCH_DIRECT && queue[i] == kMethodDirect);
            split[i][c] = tile_split(ps, f.d, c).total;
            cost[i][c] = ok ? tile_cost(cm, ps, f.d, c) : INFINITY;
            any = any || !std::isinf(cost[i][c]);
        }
        const bool direct = queue[i] == kMethodDirect, six = queue[i] == kMethodMfma6;
        cost[i][Q] = algo == NDC_BATCH_FFT && any ? INFINITY
                     : direct                     ? direct_cost(cm, ps, f.s)
                                                  : mfma_cost(cm, ps, f.s, six);
        item[i] = direct ? cm.dir_a + cm.dir_b * double(std::min<int64_t>(direct_tile(f.s), ps.out)) * double(ps.k)
                         : mfma_item_cost(cm, ps, six);
    }
    double best = INFINITY;
    unsigned best_mask = 0;
    // the cheapest group of every set of launches (-1: none takes the pair)
    std::vector<std::array<int8_t, 1 << G>> pick(P);
    for (size_t i = 0; i < P; ++i) {
        pick[i][0] = -1;
        for (int c = 0; c < G; ++c)
            for (unsigned rest = 0; rest < (1u << c); ++rest) {
                const int g = pick[i][rest];
                const bool lower = !std::isinf(cost[i][c]) && (g < 0 || cost[i][c] < cost[i][g]);
                pick[i][rest | 1u << c] = lower ? int8_t(c) : int8_t(g);
            }
    }
    for (unsigned mask = 1; mask < (1u << G); ++mask) {
        double work = 0, longest = 0;
        int64_t total[Q] = {}, runs[Q] = {}, run[Q] = {};
        unsigned used = 0;
        bool all = true;
        for (size_t i = 0; i < P && all; ++i) {
            if (sh[i].out <= 0) continue;
            const int g = pick[i][mask];
            all = g >= 0;
            if (!all) break;
            used |= 1u << g;
            if (g == Q) {
                work += cost[i][Q];
                longest = std::max(longest, item[i]);
            } else {
                total[g] += split[i][g];
            }
        }
        if (!all || used != mask) continue;
        for (int c = 0; c < Q; ++c) run[c] = run_tiles(total[c], int64_t(f.cus) * tile_slots(c));
        for (size_t i = 0; i < P; ++i) {
            const int g = pick[i][mask];
            if (sh[i].out > 0 && g < Q) runs[g] += uint32_t(split[i][g] + run[g] - 1) / uint32_t(run[g]);
        }
        for (int c = 0; c < Q; ++c)
            if (used >> c & 1)
                work += kLaunchMs + std::max(cm.tile_a[c] * double(runs[c]) + cm.tile_b[c] * double(total[c]),
                                             (cm.tile_a[c] + cm.tile_b[c] * double(run[c])) * double(f.cus * tile_slots(c)));
        if (used >> Q & 1) work += kLaunchMs + longest * double(f.blocks);
        if (work < best) {
            best = work;
            best_mask = mask;
        }
    }
    *estimate = best;
    for (size_t i = 0; i < P; ++i) {
        const int g = sh[i].out > 0 ? pick[i][best_mask] : Q;
        m[i] = g == Q ? queue[i] : kMethodTile - g;
    }
    return m;
}

// Split products, which are less exact than FP32, have to make the batch
// faster by more than the estimates are wrong: 4096 pairs, 153 M samples, circular,
// take 370 to 380 us in FP32 tiles, 369 to 377 with every pair in the queue, and 375 to
// 384 with the 1650 in it that it serves at less cost, estimated as 0.98 of FP32.
constexpr double kSplitGain = 0.95;

std::vector<int> choose(const CostModel& cm, const std::vector<PairShape>& sh, const BatchForm& f, int algo,
                        bool repeating_border) {
    double best = 0, fp32 = 0;
    std::vector<int> m = choose_launches(cm, sh, f, algo, repeating_border, &best);
    if (algo != NDC_BATCH_AUTO_BF16X3) return m;
    std::vector<int> plain = choose_launches(cm, sh, f, NDC_BATCH_AUTO, repeating_border, &fp32);
    return best < kSplitGain * fp32 ? m : plain;
}

struct Schedule {
    std::vector<BatchItem> items;
    std::vector<BatchTile> tiles[kBatchTileClasses];   // longest runs first
    double tile_bytes[kBatchTileClasses] = {};
    int64_t ntiles = 0;            // complex tiles
    int32_t nfirst = 0;            // direct items, ahead of the matrix-core items
    double est_ms = 0;
    double main_bytes = 0, main_flops = 0;
};

// Tile runs of class c; max_run > 0 gives their length.
void build_tiles(Schedule& S, const std::vector<PairShape>& sh, const std::vector<std::array<int64_t, 3>>& offs,
                 const std::vector<int>& method, const BatchForm& f, int c, const CostModel& cm, int64_t max_run) {
    std::vector<size_t> pairs;
    std::vector<TileSplit> split;
    int64_t total = 0;
    for (size_t i = 0; i < sh.size(); ++i) {
        if (method[i] != kMethodTile - c || sh[i].out <= 0) continue;
        pairs.push_back(i);
        split.push_back(tile_split(sh[i], f.d, c));
        total += split.back().total;
    }
    if (pairs.empty()) return;
    S.ntiles += total;
    const int64_t slots = int64_t(f.cus) * tile_slots(c);
    const int64_t run = max_run > 0 ? max_run : run_tiles(total, slots);
    for (size_t j = 0; j < pairs.size(); ++j) {
        const PairShape& ps = sh[pairs[j]];
        const auto& o = offs[pairs[j]];
        S.tile_bytes[c] += 4.0 * double(ps.n + ps.k + ps.out);
        const TileSplit& t = split[j];
        const int64_t p1 = ps.pds - ps.n - ps.p0;
        auto wraps = [&](int32_t side, int64_t pad) {
            return side == kS1Reflect ? pad > ps.n - 1 : side == kS1Circular ? pad > ps.n : false;
        };
        const int64_t runs = (t.total + run - 1) / run;   // of equal length, none longer than `run`
        for (int64_t r = 0; r < runs; ++r) {
            const int64_t b = t.total * r / runs, e = t.total * (r + 1) / runs;
            BatchTile it{};
            it.x_off = o[0];
            it.k_off = o[1];
            it.y_off = o[2];
            it.n = int32_t(ps.n);
            it.k = int32_t(ps.k);
            it.p0 = int32_t(ps.p0);
            it.pds = int32_t(ps.pds);
            it.out = int32_t(ps.out);
            it.V = int32_t(t.V);
            it.tiles = int32_t(t.per_phase);
            it.first = int32_t(b);
            it.count = int32_t(e - b);
            it.wraps = wraps(f.front, ps.p0) || wraps(f.back, p1);
            S.tiles[c].push_back(it);
            S.est_ms += cm.tile_a[c] + cm.tile_b[c] * double(e - b);
        }
    }
    std::stable_sort(S.tiles[c].begin(), S.tiles[c].end(),
                     [](const BatchTile& a, const BatchTile& b) { return a.count > b.count; });
}

// Builds the tile runs and the work queue.  offs[i] = {x, k, y} element offsets
// of pair i.
Schedule build_schedule(const std::vector<PairShape>& sh, const std::vector<std::array<int64_t, 3>>& offs,
                        const std::vector<int>& method, const BatchForm& f, const CostModel& cm, int64_t max_run = 0) {
    Schedule S;
    for (int c = 0; c < kBatchTileClasses; ++c) build_tiles(S, sh, offs, method, f, c, cm, max_run);
    std::vector<std::pair<double, BatchItem>> work;
    const int tile = direct_tile(f.s);
    for (size_t i = 0; i < sh.size(); ++i) {
        const PairShape& ps = sh[i];
        if (method[i] <= kMethodTile) continue;
        S.main_bytes += 4.0 * double(ps.n + ps.out);
        if (ps.out <= 0) continue;
        S.main_bytes += 4.0 * double(ps.k);
        S.main_flops += 2.0 * double(ps.out) * double(ps.k);
        const bool direct = method[i] == kMethodDirect, six = method[i] == kMethodMfma6;
        const int64_t step = direct ? tile : kBatchMfmaTile;
        for (int64_t o = 0; o < ps.out; o += step) {
            BatchItem it{};   // the tile with its pair's metadata
            it.kind = direct ? 0 : six ? kBatchKindMfma6 : kBatchKindMfma;
            it.a = int32_t(i);
            it.b = int32_t(o);
            it.c = int32_t(std::min<int64_t>(step, ps.out - o));
            it.x_off = offs[i][0];
            it.k_off = offs[i][1];
            it.y_off = offs[i][2];
            it.n = int32_t(ps.n);
            it.k = int32_t(ps.k);
            it.p0 = int32_t(ps.p0);
            it.pds = int32_t(ps.pds);
            work.emplace_back(direct ? cm.dir_a + cm.dir_b * double(it.c) * double(ps.k) : mfma_item_cost(cm, ps, six), it);
        }
    }
    // longest items first: the queue hands them out in this order, so the
    // tail of the launch is made of the shortest items.  The direct items form
    // the first range, the matrix-core items the second.
    std::stable_sort(work.begin(), work.end(),
                     [](const std::pair<double, BatchItem>& a, const std::pair<double, BatchItem>& b) {
                         return a.first > b.first;
                     });
    const auto first_end = std::stable_partition(work.begin(), work.end(), [](const std::pair<double, BatchItem>& w) {
        return w.second.kind == 0;
    });
    S.nfirst = int32_t(first_end - work.begin());
    S.items.reserve(work.size());
    for (auto& w : work) {
        S.items.push_back(w.second);
        S.est_ms += w.first;
    }
    return S;
}

// Device-resident copy of a schedule plus the launch arguments.
struct DevSchedule {
    DevMem items, counter, consts, tiles[kBatchTileClasses];
    BatchArgs args{};
    BatchTileLaunch tl{};
    int grid = 0;
    // Border sides of every pair, and the constant cells the kernels read for
    // pad positions that hold a constant.
    bool set_borders(int32_t front, int32_t back, float cfront, float cback) {
        const float cells[4] = {0.f, cfront, cback, 0.f};
        if (!consts.upload(cells, sizeof(cells))) return false;
        args.consts = static_cast<const float*>(consts.p);
        args.front = front;
        args.back = back;
        args.cfront = cfront;
        args.cback = cback;
        return true;
    }
    bool upload(const Schedule& S, LaunchContext& ctx, int blocks) {
        if (!items.upload(S.items.data(), S.items.size() * sizeof(BatchItem)) ||
            !counter.ensure(size_t(kBatchHeads) * kBatchQueueStride * sizeof(int32_t)) || !batch_tile_tables(ctx, tl.tw))
            return false;
        args.items = static_cast<const BatchItem*>(items.p);
        args.counter = static_cast<int32_t*>(counter.p);
        args.nitems = int32_t(S.items.size());
        args.nfirst = S.nfirst;
        for (int c = 0; c < kBatchTileClasses; ++c) {
            if (!tiles[c].upload(S.tiles[c].data(), S.tiles[c].size() * sizeof(BatchTile))) return false;
            tl.items[c] = static_cast<const BatchTile*>(tiles[c].p);
            tl.n[c] = int32_t(S.tiles[c].size());
            tl.bytes[c] = S.tile_bytes[c];
        }
        grid = int(std::min<int64_t>(int64_t(S.items.size()), int64_t(blocks)));
        return true;
    }
};

// The launches of a schedule: the tile runs, which zero the queue's heads, then
// the queue.
ndc_status launch_all(const DevSchedule& D, LaunchContext& ctx, hipStream_t st, bool profile, double main_bytes,
                      double main_flops) {
    bool runs = false;
    for (const int32_t n : D.tl.n) runs = runs || n > 0;
    const ndc_status r = launch_batch_tiles(D.args, D.tl, ctx, st, profile);
    return r != NDC_OK ? r : launch_batch(D.args, D.grid, !runs, ctx, st, profile, main_bytes, main_flops);
}

int resident_blocks(LaunchContext& ctx) { return batch_blocks_per_cu() * ctx.cu_count(); }

// Times `reps` runs of a schedule on synthetic data (ms per run).
bool time_schedule(LaunchContext& ctx, const Schedule& S, const float* x, const float* k, float* y, int s, int d,
                   double* ms) {
    DevSchedule D;
    if (!D.upload(S, ctx, resident_blocks(ctx))) return false;
    D.args.x = x;
    D.args.k = k;
    D.args.y = y;
    D.args.s = s;
    D.args.d = d;
    D.args.dmul = batch_dmul(d);
    D.args.rev = 1;
    if (!D.set_borders(kS1Circular, kS1Circular, 0.f, 0.f)) return false;
    hipStream_t st = ctx.stream();
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return false;
    bool ok = launch_all(D, ctx, st, false, 0, 0) == NDC_OK;
    constexpr int reps = 3;
    ok = ok && hipEventRecord(e0, st) == hipSuccess;
    for (int r = 0; ok && r < reps; ++r) ok = launch_all(D, ctx, st, false, 0, 0) == NDC_OK;
    ok = ok && hipEventRecord(e1, st) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
    float t = 0;
    ok = ok && hipEventElapsedTime(&t, e0, e1) == hipSuccess;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = double(t) / reps;
    return ok;
}

// Measures the cost model on the device, on random samples (zeros would let
// the matrix cores run at clocks that data does not), one method at a time.
// The batches read and write 25 M samples four times over, which takes long
// enough that what a launch costs by itself is a few percent.
bool calibrate(LaunchContext& ctx, int s, int d, CostModel* cm) {
    constexpr int64_t kSamples = 96 << 18, kTaps = 1024, kTimes = 4;
    float* x = static_cast<float*>(ctx.scratch(0, size_t(kSamples) * sizeof(float)));
    float* y = static_cast<float*>(ctx.scratch(1, size_t(kSamples) * sizeof(float)));
    float* k = static_cast<float*>(ctx.scratch(2, size_t(kTaps) * sizeof(float)));
    if (!x || !y || !k) return false;
    if (fill_random(x, kSamples, ctx) != NDC_OK || fill_random(k, kTaps, ctx) != NDC_OK) return false;
    const BatchForm form{s, d, kS1Circular, kS1Circular, ctx.cu_count(), resident_blocks(ctx)};
    CostModel out = *cm;
    struct Unit {
        double ms = 0;       // per tile of a run, or per item
        double runs = 0;     // runs per tile
        double work = 0;     // outputs times taps per item
        double blocks = 0;   // K-blocks of an item
    };
    // pairs of n samples and kl taps, all by `method`
    auto measure = [&](int64_t n, int64_t kl, int method, int64_t run, Unit* u) {
        const int64_t distinct = kSamples / n;
        const size_t P = size_t(distinct * kTimes);
        std::vector<PairShape> sh(P);
        std::vector<std::array<int64_t, 3>> offs(P);
        const int64_t kdil = (kl - 1) * d + 1;
        const int64_t p0 = (kdil - 1) / 2 + ((kdil - 1) % 2), p1 = (kdil - 1) / 2;   // Same
        for (size_t i = 0; i < P; ++i) {
            sh[i] = PairShape{n, kl, p0, n + p0 + p1, (n + p0 + p1 - kdil) / s + 1, kdil};
            offs[i] = {int64_t(i) % distinct * n, 0, int64_t(i) % distinct * n};
        }
        const Schedule S = build_schedule(sh, offs, std::vector<int>(P, method), form, out, run);
        const int c = group_of(method);
        const double units = c < kBatchTileClasses ? double(S.ntiles) : double(S.items.size());
        double t = 0;
        if (units == 0 || !time_schedule(ctx, S, x, k, y, s, d, &t)) return false;
        u->ms = t / units;
        u->runs = c < kBatchTileClasses ? double(S.tiles[c].size()) / units : 0;
        u->work = double(P) * double(sh[0].out) * double(kl) / units;
        u->blocks = double(mfma_nkb(sh[0]));
        return true;
    };
    constexpr int64_t kLong = 1 << 18;
    // tile runs: a + b at pairs of one complex tile (their edges are part of a),
    // b + a / 8 inside long pairs
    for (int c = 0; c < kBatchTileClasses; ++c) {
        const int64_t N = int64_t(1) << batch_tile_log2(c), kl = 33;
        if (int64_t(d) * N >= kLong / 2) continue;
        Unit one, many;
        if (!measure(2 * (N - kl + 1) * d, kl, kMethodTile - c, 1, &one) || !measure(kLong, kl, kMethodTile - c, 8, &many))
            return false;
        if (many.runs >= 1) continue;
        out.tile_a[c] = std::max(0.0, (one.ms - many.ms) / (1 - many.runs));
        out.tile_b[c] = std::max(1e-9, many.ms - out.tile_a[c] * many.runs);
    }
    // direct items: a + b work, from two tap counts
    Unit u[2];
    if (!measure(kLong, 16, kMethodDirect, 0, &u[0]) || !measure(kLong, 256, kMethodDirect, 0, &u[1])) return false;
    if (u[1].work > u[0].work) {
        out.dir_b = std::max(1e-14, (u[1].ms - u[0].ms) / (u[1].work - u[0].work));
        out.dir_a = std::max(0.0, u[0].ms - out.dir_b * u[0].work);
    }
    // matrix-core items (stride 1 only): a + b K-blocks at two kernel lengths,
    // for each split; and what the first and last of a pair cost more
    if (s == 1) {
        const int64_t kcap = (kBatchMfmaMaxKdil - 1) / d + 1;
        for (int six = 0; six < 2; ++six) {
            const int method = six ? kMethodMfma6 : kMethodMfma;
            if (!measure(kLong, std::min<int64_t>(8, kcap), method, 0, &u[0]) ||
                !measure(kLong, std::min<int64_t>(512, kcap), method, 0, &u[1]))
                return false;
            if (u[1].blocks > u[0].blocks) {
                const double b = std::max(1e-12, (u[1].ms - u[0].ms) / (u[1].blocks - u[0].blocks));
                (six ? out.mfma6_b : out.mfma_b) = b;
                (six ? out.mfma6_a : out.mfma_a) = std::max(0.0, u[0].ms - b * u[0].blocks);
            }
        }
        if (!measure(2 * kBatchMfmaTile, std::min<int64_t>(8, kcap), kMethodMfma6, 0, &u[1])) return false;
        out.edge = std::max(0.0, u[1].ms - out.mfma6_a - out.mfma6_b * u[1].blocks);
    }
    out.measured = true;
    *cm = out;
    return true;
}

// The cost model of this handle for strides/dilation (s, d), measured once.
CostModel cost_model(LaunchContext& ctx, int s, int d, bool measure) {
    const std::string key = "batch_costs4:" + std::to_string(s) + ":" + std::to_string(d);
    std::string& m = ctx.memo(key);
    CostModel cm = default_costs();
    if (m.size() == sizeof(CostModel)) {
        std::memcpy(&cm, m.data(), sizeof(cm));
        return cm;
    }
    if (!measure) return cm;
    if (!calibrate(ctx, s, d, &cm)) cm = default_costs();
    m.assign(reinterpret_cast<const char*>(&cm), sizeof(cm));
    return cm;
}

// The rank-1 single-problem descriptor of pair i.
ndc_conv_desc pair_desc(const ndc_batch_desc* d, int64_t i) {
    ndc_conv_desc c;
    std::memset(&c, 0, sizeof(c));
    c.dtype = d->dtype;
    c.rank = 1;
    c.x_shape[0] = d->x_len[i];
    c.k_shape[0] = d->k_len[i];
    c.dilation[0] = d->dilation;
    c.reverse = d->reverse;
    c.conv_mode = d->conv_mode;
    c.padding_mode = d->padding_mode;
    return c;
}

struct Batch {
    ndc_handle h = nullptr;
    LaunchContext* ctx = nullptr;
    int algo = 0;
    bool host = false;
    int s = 1, d = 1;
    std::vector<PairShape> shapes;
    std::vector<std::array<int64_t, 3>> offs;
    std::vector<int> method;
    int64_t x_total = 0, k_total = 0, y_total = 0;
    CostModel cm;
    Schedule S;
    DevSchedule D;
    std::vector<Plan> plain;
    DevMem io[3];
    hipStream_t cap = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    const void* gx = nullptr;
    const void* gk = nullptr;
    void* gy = nullptr;

    ~Batch() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (cap) (void)hipStreamDestroy(cap);
    }

    ndc_status enqueue(const float* x, const float* k, float* y, hipStream_t st, bool profile) {
        if (algo == NDC_BATCH_PLAIN) {
            for (size_t i = 0; i < plain.size(); ++i) {
                if (shapes[i].out <= 0) continue;
                const ndc_status r = launch_fft(plain[i], x + offs[i][0], k + offs[i][1], y + offs[i][2], *ctx);
                if (r != NDC_OK) return r;
            }
            return NDC_OK;
        }
        BatchArgs a = D.args;
        a.x = x;
        a.k = k;
        a.y = y;
        D.args = a;
        return launch_all(D, *ctx, st, profile, S.main_bytes, S.main_flops);
    }
};

ndc_status fail(ndc_handle h, ndc_status s, const std::string& msg) {
    handle_set_last(h, msg);
    return s;
}

ndc_status batch_create(ndc_handle h, const ndc_batch_desc* d, Batch** out) {
    if (!h || !d || !out) return NDC_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    if (d->dtype != NDC_F32) return fail(h, NDC_ERR_UNSUPPORTED, "batches are f32");
    if (d->count < 0 || (d->count > 0 && (!d->x_len || !d->k_len)))
        return fail(h, NDC_ERR_INVALID_ARGUMENT, "bad pair count or length arrays");
    if (d->algo < NDC_BATCH_AUTO || d->algo > NDC_BATCH_BF16X6)
        return fail(h, NDC_ERR_INVALID_ARGUMENT, "unknown batch algorithm");
    if (d->flags & ~uint32_t(NDC_FLAG_HOST_MEMORY)) return fail(h, NDC_ERR_INVALID_ARGUMENT, "unknown batch flags");
    LaunchContext* ctx = handle_context(h);
    if (hipSetDevice(handle_device(h)) != hipSuccess) return fail(h, NDC_ERR_DEVICE, "hipSetDevice failed");
    auto b = std::make_unique<Batch>();
    b->h = h;
    b->ctx = ctx;
    b->algo = d->algo;
    b->host = (d->flags & NDC_FLAG_HOST_MEMORY) != 0;
    const int64_t P = d->count;
    b->shapes.resize(size_t(P));
    b->offs.resize(size_t(P));
    ndc_border front{}, back{};
    for (int64_t i = 0; i < P; ++i) {
        ndc_conv_desc cd = pair_desc(d, i);
        Plan p;
        std::string err;
        const bool maps = d->algo == NDC_BATCH_PLAIN;
        const ndc_status st = make_plan(&cd, NDC_OP_CONV_FFT, &p, &err, maps);
        if (st != NDC_OK) return fail(h, st, "pair " + std::to_string(i) + ": " + err);
        if (p.x_shape[0] >= (int64_t(1) << 30) || p.pds[0] >= (int64_t(1) << 30))
            return fail(h, NDC_ERR_UNSUPPORTED, "pair " + std::to_string(i) + ": longer than 2^30 samples");
        b->shapes[size_t(i)] = PairShape{p.x_shape[0], p.k_shape[0], p.pad[0][0], p.pds[0], p.out[0], p.kdil[0]};
        b->offs[size_t(i)] = {b->x_total, b->k_total, b->y_total};
        b->x_total += p.x_shape[0];
        b->k_total += p.k_shape[0];
        b->y_total += p.out[0];
        if (i == 0) {
            b->s = int(p.stride[0]);
            b->d = int(p.dil[0]);
            front = p.side[0][0];
            back = p.side[0][1];
        }
        if (maps) b->plain.push_back(std::move(p));
    }
    if (b->algo != NDC_BATCH_PLAIN) {
        if (int64_t(b->s) >= (int64_t(1) << 20) || int64_t(b->d) >= (int64_t(1) << 20))
            return fail(h, NDC_ERR_UNSUPPORTED, "stride or dilation too large for the batch kernels");
        b->cm = cost_model(*ctx, b->s, b->d, b->algo == NDC_BATCH_AUTO || b->algo == NDC_BATCH_AUTO_BF16X3);
        auto repeats = [](const ndc_border& side) {
            return side.tag == NDC_BORDER_REPLICATE || (side.tag == NDC_BORDER_CONST && side.value.re != 0.0);
        };
        const bool rb = repeats(front) || repeats(back);
        const BatchForm form{b->s, b->d, side1d(front.tag), side1d(back.tag), ctx->cu_count(), resident_blocks(*ctx)};
        b->method = choose(b->cm, b->shapes, form, b->algo, rb);
        b->S = build_schedule(b->shapes, b->offs, b->method, form, b->cm);
        if (!b->D.upload(b->S, *ctx, resident_blocks(*ctx)))
            return fail(h, NDC_ERR_OUT_OF_MEMORY, "batch metadata upload failed");
        BatchArgs& a = b->D.args;
        a.s = b->s;
        a.d = b->d;
        a.dmul = batch_dmul(b->d);
        a.rev = d->reverse ? 1 : 0;
        if (!b->D.set_borders(side1d(front.tag), side1d(back.tag), float(front.value.re), float(back.value.re)))
            return fail(h, NDC_ERR_OUT_OF_MEMORY, "batch metadata upload failed");
    }
    *out = b.release();
    return NDC_OK;
}

ndc_status batch_run(Batch& b, const void* x, const void* k, void* y, bool use_graph) {
    if (!x || !k || !y) {
        if (b.y_total > 0 || b.x_total > 0) return fail(b.h, NDC_ERR_INVALID_ARGUMENT, "null data pointer");
    }
    if (hipSetDevice(handle_device(b.h)) != hipSuccess) return fail(b.h, NDC_ERR_DEVICE, "hipSetDevice failed");
    LaunchContext& ctx = *b.ctx;
    ctx.err.clear();
    hipStream_t st = ctx.stream();
    const float* dx = static_cast<const float*>(x);
    const float* dk = static_cast<const float*>(k);
    float* dy = static_cast<float*>(y);
    if (b.host) {
        if (!b.io[0].ensure(size_t(b.x_total) * 4) || !b.io[1].ensure(size_t(b.k_total) * 4) ||
            !b.io[2].ensure(size_t(b.y_total) * 4))
            return fail(b.h, NDC_ERR_OUT_OF_MEMORY, "device buffer allocation failed");
        if (hipMemcpyAsync(b.io[0].p, x, size_t(b.x_total) * 4, hipMemcpyHostToDevice, st) != hipSuccess ||
            hipMemcpyAsync(b.io[1].p, k, size_t(b.k_total) * 4, hipMemcpyHostToDevice, st) != hipSuccess)
            return fail(b.h, NDC_ERR_DEVICE, "host to device copy failed");
        dx = static_cast<const float*>(b.io[0].p);
        dk = static_cast<const float*>(b.io[1].p);
        dy = static_cast<float*>(b.io[2].p);
    }
    ndc_status r = NDC_OK;
    if (use_graph && b.algo != NDC_BATCH_PLAIN) {
        if (!b.exec || b.gx != dx || b.gk != dk || b.gy != dy) {
            if (b.exec) (void)hipGraphExecDestroy(b.exec);
            if (b.graph) (void)hipGraphDestroy(b.graph);
            b.exec = nullptr;
            b.graph = nullptr;
            if (!b.cap && hipStreamCreateWithFlags(&b.cap, hipStreamNonBlocking) != hipSuccess)
                return fail(b.h, NDC_ERR_DEVICE, "capture stream creation failed");
            if (hipStreamBeginCapture(b.cap, hipStreamCaptureModeThreadLocal) != hipSuccess)
                return fail(b.h, NDC_ERR_DEVICE, "graph capture failed to start");
            r = b.enqueue(dx, dk, dy, b.cap, false);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(b.cap, &g);
            if (r != NDC_OK) {
                if (g) (void)hipGraphDestroy(g);
                return fail(b.h, r, ctx.err);
            }
            if (e != hipSuccess || !g || hipGraphInstantiate(&b.exec, g, nullptr, nullptr, 0) != hipSuccess) {
                if (g) (void)hipGraphDestroy(g);
                b.exec = nullptr;
                return fail(b.h, NDC_ERR_DEVICE, "graph capture failed");
            }
            b.graph = g;
            b.gx = dx;
            b.gk = dk;
            b.gy = dy;
        }
        if (hipGraphLaunch(b.exec, st) != hipSuccess) return fail(b.h, NDC_ERR_DEVICE, "graph launch failed");
    } else {
        r = b.enqueue(dx, dk, dy, st, true);
        if (r != NDC_OK) return fail(b.h, r, ctx.err);
    }
    if (b.host) {
        if (hipMemcpyAsync(y, dy, size_t(b.y_total) * 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return fail(b.h, NDC_ERR_DEVICE, "device to host copy failed");
    }
    return NDC_OK;
}

void append(std::string& s, const char* fmt, double v) {
    char tmp[64];
    std::snprintf(tmp, sizeof(tmp), fmt, v);
    s += tmp;
}

std::string batch_report(const Batch& b) {
    std::string r = "{\"algo\": " + std::to_string(b.algo) + ", \"pairs\": " + std::to_string(b.shapes.size());
    r += ", \"outputs\": " + std::to_string(b.y_total);
    size_t runs = 0;
    for (const auto& t : b.S.tiles) runs += t.size();
    r += ", \"items\": " + std::to_string(b.S.items.size()) + ", \"lines\": " + std::to_string(b.S.ntiles);
    r += ", \"kernel_spectra\": " + std::to_string(runs);   // one per run
    r += ", \"grid\": " + std::to_string(b.D.grid);
    r += ", \"blocks_per_cu\": " + std::to_string(batch_blocks_per_cu());
    append(r, ", \"est_ms\": %.6f", b.S.est_ms);
    append(r, ", \"main_bytes\": %.1f", b.S.main_bytes);
    append(r, ", \"main_flops\": %.1f", b.S.main_flops);
    r += ", \"costs\": {\"measured\": ";
    r += b.cm.measured ? "true" : "false";
    r += ", \"tile_run_ms\": [";
    for (int c = 0; c < kBatchTileClasses; ++c) append(r, c ? ", %.4e" : "%.4e", b.cm.tile_a[c]);
    r += "], \"tile_ms\": [";
    for (int c = 0; c < kBatchTileClasses; ++c) append(r, c ? ", %.4e" : "%.4e", b.cm.tile_b[c]);
    r += "]";
    append(r, ", \"edge_ms\": %.4e", b.cm.edge);
    append(r, ", \"direct_item_ms\": %.4e", b.cm.dir_a);
    append(r, ", \"direct_mac_ms\": %.4e", b.cm.dir_b);
    append(r, ", \"mfma_item_ms\": %.4e", b.cm.mfma_a);
    append(r, ", \"mfma_kblock_ms\": %.4e", b.cm.mfma_b);
    append(r, ", \"mfma6_item_ms\": %.4e", b.cm.mfma6_a);
    append(r, ", \"mfma6_kblock_ms\": %.4e}", b.cm.mfma6_b);
    // choice per bucket: kernel-length octave x signal-length octave
    std::map<std::pair<int, int>, std::map<std::string, int64_t>> bk;
    for (size_t i = 0; i < b.shapes.size() && i < b.method.size(); ++i) {
        const int kb = int(std::floor(std::log2(double(std::max<int64_t>(1, b.shapes[i].k)))));
        const int nb = int(std::floor(std::log2(double(std::max<int64_t>(1, b.shapes[i].n)))));
        const int m = b.method[i];
        const std::string name = m == kMethodDirect ? "direct_fp32"
                                 : m == kMethodMfma  ? "direct_bf16x3"
                                 : m == kMethodMfma6 ? "direct_bf16x6"
                                                     : "tile" + std::to_string(1 << batch_tile_log2(kMethodTile - m));
        bk[{kb, nb}][name] += 1;
    }
    r += ", \"buckets\": [";
    bool first = true;
    for (auto& e : bk) {
        r += first ? "" : ", ";
        first = false;
        r += "{\"k_log2\": " + std::to_string(e.first.first) + ", \"n_log2\": " + std::to_string(e.first.second) +
             ", \"choice\": {";
        bool f2 = true;
        for (auto& c : e.second) {
            r += (f2 ? "\"" : ", \"") + c.first + "\": " + std::to_string(c.second);
            f2 = false;
        }
        r += "}}";
    }
    r += "]}";
    return r;
}

}  // namespace
}  // namespace ndc

using ndc::Batch;

extern "C" {

ndc_status ndc_batch_create(ndc_handle h, const ndc_batch_desc* desc, ndc_batch* out) {
    if (!out) return NDC_ERR_INVALID_ARGUMENT;
    Batch* b = nullptr;
    const ndc_status s = ndc::batch_create(h, desc, &b);
    *out = reinterpret_cast<ndc_batch>(b);
    return s;
}

ndc_status ndc_batch_destroy(ndc_batch bb) {
    if (!bb) return NDC_ERR_INVALID_ARGUMENT;
    Batch* b = reinterpret_cast<Batch*>(bb);
    (void)hipStreamSynchronize(b->ctx->stream());
    delete b;
    return NDC_OK;
}

ndc_status ndc_batch_out_lens(ndc_batch bb, int64_t* y_len, int64_t* x_total, int64_t* k_total, int64_t* y_total) {
    if (!bb) return NDC_ERR_INVALID_ARGUMENT;
    const Batch* b = reinterpret_cast<const Batch*>(bb);
    if (y_len)
        for (size_t i = 0; i < b->shapes.size(); ++i) y_len[i] = b->shapes[i].out;
    if (x_total) *x_total = b->x_total;
    if (k_total) *k_total = b->k_total;
    if (y_total) *y_total = b->y_total;
    return NDC_OK;
}

ndc_status ndc_batch_run(ndc_batch bb, const void* x, const void* k, void* y) {
    if (!bb) return NDC_ERR_INVALID_ARGUMENT;
    return ndc::batch_run(*reinterpret_cast<Batch*>(bb), x, k, y, false);
}

ndc_status ndc_batch_run_graph(ndc_batch bb, const void* x, const void* k, void* y) {
    if (!bb) return NDC_ERR_INVALID_ARGUMENT;
    return ndc::batch_run(*reinterpret_cast<Batch*>(bb), x, k, y, true);
}

ndc_status ndc_batch_report(ndc_batch bb, char* buf, int64_t len) {
    if (!bb || !buf || len <= 0) return NDC_ERR_INVALID_ARGUMENT;
    const std::string r = ndc::batch_report(*reinterpret_cast<const Batch*>(bb));
    if (int64_t(r.size()) + 1 > len) return NDC_ERR_INVALID_ARGUMENT;
    std::memcpy(buf, r.c_str(), r.size() + 1);
    return NDC_OK;
}

ndc_status ndc_batch_border_map(const ndc_batch_desc* desc, int64_t pair, int32_t* codes, int64_t len) {
    if (!desc || !codes || pair < 0 || pair >= desc->count || !desc->x_len || !desc->k_len)
        return NDC_ERR_INVALID_ARGUMENT;
    ndc_conv_desc cd = ndc::pair_desc(desc, pair);
    cd.dtype = NDC_F32;
    ndc::Plan p;
    std::string err;
    const ndc_status s = ndc::make_plan(&cd, NDC_OP_CONV, &p, &err, false);
    if (s != NDC_OK) return s;
    if (len != p.pds[0]) return NDC_ERR_INVALID_ARGUMENT;
    const int32_t front = ndc::side1d(p.side[0][0].tag), back = ndc::side1d(p.side[0][1].tag);
    for (int64_t q = 0; q < len; ++q)
        codes[q] = int32_t(ndc::resolve1d<int64_t>(q, p.x_shape[0], p.pad[0][0], front, back));
    return NDC_OK;
}

}  // extern "C"
