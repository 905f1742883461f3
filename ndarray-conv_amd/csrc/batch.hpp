// Batches of independent rank-1 signal/kernel pairs of uneven lengths, run
// as one persistent launch that drains a device-side work queue.
//
// Every pair has the semantics of one rank-1 conv_fft call
// (conv_fft/mod.rs:185-292): ConvMode and PaddingMode are shared by the
// batch, lengths differ per pair.  Each pair is computed by one of
//   - direct items: a tile of outputs, FP32 multiply-adds over the taps;
//   - matrix-core items: a tile of outputs from split BF16 products;
//   - tile runs (batch_tile.hip, launches of their own): FP32 overlap-save, two
//     real tiles per complex transform, the kernel's spectrum in registers.
//     Overlap-save computes the same linear correlation as the reference's
//     single FFT of the whole padded signal, only blocked.
// The choice per pair comes from a cost model whose constants are measured
// on the device (the autotuner).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "launch.hpp"
#include "ndconv.h"
#include "tile_conv.hpp"

namespace ndc {

constexpr int kBatchThreads = 256;
constexpr int kBatchDirectTile = 2048;       // outputs per direct item (8 per thread)
constexpr int kBatchWindow = 6144;           // LDS window capacity of a direct item (floats)
constexpr int kBatchTapChunk = 1024;         // taps staged per round of a direct item
constexpr int kBatchMfmaTile = 4096;         // outputs per matrix-core item (1024 per wave)
constexpr int kBatchMfmaMaxKdil = 1024;      // longest dilated kernel of a matrix-core item (LDS)
constexpr int kBatchKindMfma = 1;            // BF16x3 matrix-core tile (two-term split)
constexpr int kBatchKindMfma6 = 2;           // BF16x6 matrix-core tile (three-term split)
// Fewest kernel taps for which the autotuned and matrix-core batch forms use
// BF16x3.  Its products carry about 16 significant bits (each within
// 3 * 2^-16 of the exact product); an output summed from a few products keeps
// that error, while with 32 or more independent products per output the
// rounding errors average to about 2^-18 of the output scale (normwise 4.7e-6
// worst in an exact-accumulation model of Uniform[-1,1) data over 1.2 M
// outputs).  Shorter kernels use the three-term split, whose products are
// within 5 * 2^-24.
constexpr int kBf16x3MinTaps = 32;

// The work queue is two ranges of the item list, each longest-first: the
// direct items [0, nfirst), then the matrix-core items [nfirst,
// nitems).  Workgroups below nfirst drain the first range, then all drain
// the second.  Each
// range is kBatchQueues sub-queues: sub-queue q of a range starting at lo
// holds items lo + q, lo + q + kBatchQueues, ...  One head per sub-queue,
// kBatchQueueStride ints (256 bytes) apart, the second range's heads after
// the first's: a single head shared by every workgroup serializes the pops
// (about 12 ns each).
constexpr int kBatchQueues = 8;
constexpr int kBatchQueueStride = 64;
constexpr int kBatchHeads = 2 * kBatchQueues;

// ceil(2^31 / d), d >= 1: for 0 <= q < 2^20 and d <= 2^11, q / d is the high
// word of 2 q * batch_dmul(d) (the error term q (2^31 mod d) / (d 2^31) stays
// below 1 / d).
constexpr uint32_t batch_dmul(int d) { return uint32_t(((uint64_t(1) << 31) + uint64_t(d) - 1) / uint64_t(d)); }

// One unit of the work queue (64 bytes).
//   kind 0: direct tile  a = pair, b = first output, c = output count
//   kind kBatchKindMfma / kBatchKindMfma6: BF16x3 / BF16x6 matrix-core tile,
//       a = pair, b = first output, c = count
// Direct and matrix-core tiles carry their pair's metadata, so a workgroup
// starts an item after one load (which it prefetches during the item before).
struct BatchItem {
    int32_t kind, a, b, c;
    int64_t x_off, k_off, y_off;   // the pair's element offsets into x, k, y
    int32_t n, k, p0, pds;         // the pair's signal and kernel lengths, front pad, padded length
    int32_t pad_[2];
};
static_assert(sizeof(BatchItem) == 64, "work-queue records are 16 dwords");

// A run of consecutive complex tiles of one pair (batch_tile.hip, 64 bytes):
// tiles 2 q and 2 q + 1 of every q in [first, first + count).
struct BatchTile {
    int64_t x_off, k_off, y_off;
    int32_t n, k, p0, pds, out;    // the pair's lengths, front pad, padded and output length
    int32_t V, tiles;              // outputs per tile and phase, tiles per phase
    int32_t first, count;
    int32_t wraps;                 // a pad repeats x or reads the other pad
};
static_assert(sizeof(BatchTile) == 64, "one record, one scalar load");

// The run of workgroup g.  Runs are sorted longest first and dispatched in the
// order of g, round-robin over the eight XCDs: of every 64 consecutive runs, an
// XCD takes eight neighbours (often of one pair, whose halos its L2 then holds),
// so that all XCDs go through the list together.  With one eighth of the whole
// list per XCD the first had up to 1.7 times its share: 4096 pairs of 153 M
// samples, FP32, 397 us against 351; 1024 pairs of 300 to 1023 taps 154 against 124;
// 300 pairs of 1000 to 6000 taps 114 against 105.  Single neighbours per XCD give the
// same, at dilation 3 41.5 against 39.9.
constexpr int batch_run_of(int g, int n) {
    return (g | 63) < n ? (g & ~63) + (g & 7) * 8 + ((g >> 3) & 7) : g;
}

// Tile classes by points.  The last addresses in 64 bits, for pairs of 2^28
// samples and more and for kernels that no other class holds.
constexpr int kBatchTileClasses = 4;
constexpr int kBatchTileFar = kBatchTileClasses - 1;
constexpr int batch_tile_log2(int c) { return c == 0 ? 10 : 11 + c; }   // 1024, 4096, 8192, 16384

struct BatchTileLaunch {
    const BatchTile* items[kBatchTileClasses] = {};
    int32_t n[kBatchTileClasses] = {};
    double bytes[kBatchTileClasses] = {};
    const void* tw[kBatchTileClasses] = {};
};

// Shared launch parameters of a batch.
struct BatchArgs {
    const float* x;
    const float* k;
    float* y;
    const BatchItem* items;
    int32_t* counter;              // kBatchHeads sub-queue heads (kBatchQueueStride apart), zero at the launch
    const float* consts;           // {0, cfront, cback, 0}: the cells constant pad positions read
    int32_t nitems;
    int32_t nfirst;                // items of the first range (direct)
    int32_t s, d, rev;
    uint32_t dmul;                 // batch_dmul(d)
    int32_t front, back;           // side tags of border1d.hpp
    float cfront, cback;           // constants of Const sides
};

// Device launchers.  With `profile` each launch is bracketed for ctx's
// per-kernel profile (not while capturing); the byte/flop counts are the
// algorithmic traffic of each launch.
//
// The queue (batch_conv.hip); `reset` zeroes its heads in a launch before it.
size_t batch_lds_bytes();
int batch_blocks_per_cu();
ndc_status launch_batch(const BatchArgs& a, int grid, bool reset, LaunchContext& ctx, hipStream_t stream, bool profile,
                        double main_bytes, double main_flops);
// The tile runs (batch_tile.hip), each launch zeroing the queue's heads, and
// their twiddle tables.
bool batch_tile_tables(LaunchContext& ctx, const void* tw[kBatchTileClasses]);
ndc_status launch_batch_tiles(const BatchArgs& a, const BatchTileLaunch& l, LaunchContext& ctx, hipStream_t stream,
                              bool profile);

// n samples of Uniform[-1, 1) (batch_conv.hip), for the cost model's measurements.
ndc_status fill_random(float* p, int64_t n, LaunchContext& ctx);

// Services of the handle behind an ndc_handle (capi.cpp).
LaunchContext* handle_context(ndc_handle h);
int handle_device(ndc_handle h);
void handle_set_last(ndc_handle h, const std::string& msg);

}  // namespace ndc
