// Batch pairs by overlap-save tiles: a workgroup takes a run of consecutive
// tiles of one pair, transforms the pair's kernel once, keeps that spectrum in
// registers and convolves its tiles with it, two real tiles in one complex
// transform (tile_kernels.hpp has the single-problem form).  FP32 throughout.
//
// A run's kernel is transformed by the workgroup that uses it: a spectrum through
// memory from a launch before costs that launch (12 us) and saves a third of a
// run.  What bounds it is the chain of a tile (two transforms of barrier-separated
// LDS exchanges) with the waves that the registers leave: 16 a CU for 4096 points
// (128 registers: spectrum, tile, next tile, twiddles), 20 for 1024.
//
// Measured (ms of a full chip): a complex tile of 1024 / 4096 / 8192 points takes
// 3.3e-6 / 1.43e-5 / 3.4e-5, a run 2.1e-6 / 1.7e-5 / 4.8e-5 more for its kernel
// and start.  Batches before (real blocks of 512 to 8192 samples from a queue
// with spectra from a launch before) and now: 509 pairs of up to 65536 samples
// and 255 taps 72 -> 20 us, 4096 pairs of 153 M samples in FP32 0.73 -> 0.35 ms, 300
// pairs with 1000 to 6000 taps 197 -> 105 us, 2000 pairs under 2000 samples 58 -> 14 us.
#include <hip/hip_runtime.h>

#include <cstring>
#include <string>
#include <vector>

#include "batch.hpp"
#include "border1d.hpp"
#include "tile_kernels.hpp"

namespace ndc {
namespace {

using tilefft::Shape;
using tilek::buffer_of;
using tilek::cell_kind;
using tilek::cell_offset;
using tilek::kNoCell;
using tilek::kNoTile;

struct BatchTileArgs {
    const float* x;
    const float* k;
    float* y;
    const void* tw;
    int32_t* heads;            // of the work queue, zeroed for the launch after
    TileDiv phases, stride;    // dilation, stride
    int32_t rev, front, back;  // side tags of border1d.hpp
    int32_t fills;             // a side writes a constant other than zero
    float cfront, cback;
};

template <typename T>
__device__ __forceinline__ T uniform(T v) {
    if constexpr (sizeof(T) == 8) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(u))));
        const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(u >> 32))));
        return __builtin_bit_cast(T, (uint64_t(hi) << 32) | lo);
    } else {
        return T(__builtin_amdgcn_readfirstlane(int(v)));
    }
}

// One run per workgroup.  FAR addresses x and y in 64 bits (a pair of 2^28
// samples and more); NEXT loads the next tile before the current one is
// transformed back, where the registers allow it.
template <class S, bool FAR, bool NEXT>
__global__ void __launch_bounds__(S::T, 4) batch_tile_kernel(BatchTileArgs a, const BatchTile* __restrict__ items, int n) {
    using C = float2;
    using F = tilefft::TileFft<float, S>;
    using Io = tilek::TileIo<float, S, false, false>;
    constexpr int PW = 1 << S::aw[0], LMW = S::LW - S::aw[0];
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x;
    if (blockIdx.x == 0 && t < kBatchHeads) a.heads[t * kBatchQueueStride] = 0;
    const BatchTile& it = items[batch_run_of(int(blockIdx.x), n)];
    TileAxis ax;
    ax.n = uniform(it.n);
    ax.p0 = uniform(it.p0);
    ax.pds = uniform(it.pds);
    ax.K = uniform(it.k);
    ax.V = uniform(it.V);
    ax.tiles.d = uint32_t(uniform(it.tiles));
    ax.d = int(a.phases.d);
    ax.phases = a.phases;
    ax.stride = a.stride;
    ax.s = int(a.stride.d);
    ax.U = ax.pds - (ax.K - 1) * ax.d;
    ax.xs = ax.ys = 4;
    ax.xlo = 0;
    ax.fa = a.front == kS1Reflect ? -1 : a.front == kS1Circular ? 1 : 0;
    ax.fb = a.front == kS1Circular ? ax.n : 0;
    ax.ba = a.back == kS1Reflect ? -1 : a.back == kS1Circular ? 1 : 0;
    ax.bb = a.back == kS1Reflect ? 2 * (ax.n - 1) : a.back == kS1Circular ? -ax.n : ax.n - 1;
    ax.fconst = a.front == kS1Const;
    ax.bconst = a.back == kS1Const;
    const bool wraps = FAR || uniform(it.wraps) != 0;
    const float* x = a.x + uniform(it.x_off);
    float* y = a.y + uniform(it.y_off);
    const __amdgpu_buffer_rsrc_t px = buffer_of(x, FAR ? 0 : ax.n * 4);
    const __amdgpu_buffer_rsrc_t pk = buffer_of(a.k + uniform(it.k_off), ax.K * 4);
    const __amdgpu_buffer_rsrc_t py = buffer_of(y, FAR ? 0 : uniform(it.out) * 4);
    const int first = uniform(it.first), last = first + uniform(it.count);
    const int mw = F::template thr_value<0, 0, LMW>(t);

    const auto tw = F::load_tw(a.tw, t);
    C w[S::PPT], nx[S::PPT];
    uint32_t co[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int j = mw + (i << LMW);
        const uint32_t o = j < ax.K ? uint32_t(a.rev ? j : ax.K - 1 - j) * 4u : kNoCell;
        w[i] = C{tilek::load_real<float>(pk, o) * (1.0f / float(S::N)), 0.0f};
    }
    auto load = [&](int q) {
#pragma unroll
        for (int im = 0; im < 2; ++im) {
            const int cell = tilek::tile_cell(ax, 2 * q + im);
            if (!wraps) {   // uniform
                Io::template cells<PW, (1 << LMW)>(co, ax, cell, S::N, mw);
#pragma unroll
                for (int i = 0; i < PW; ++i) {
                    float v = tilek::load_real<float>(px, co[i]);
                    if (a.fills && cell != kNoTile) {
                        const int kind = cell_kind(ax, cell + ax.d * (mw + (i << LMW)));
                        v = kind == 1 ? a.cfront : kind == 2 ? a.cback : v;
                    }
                    if (im) nx[i].y = v;
                    else nx[i].x = v;
                }
            } else {
#pragma unroll
                for (int i = 0; i < PW; ++i) {
                    const int P = cell + ax.d * (mw + (i << LMW));
                    const int s = cell == kNoTile || P >= ax.pds ? int(kUnwritten)
                                                                 : resolve1d<int32_t>(P, ax.n, ax.p0, a.front, a.back);
                    float v = s == int(kConstFront) ? a.cfront : s == int(kConstBack) ? a.cback : 0.0f;
                    if (s >= 0) {
                        if constexpr (FAR) v = x[s];
                        else v = tilek::load_real<float>(px, uint32_t(s) * 4u);
                    }
                    if (im) nx[i].y = v;
                    else nx[i].x = v;
                }
            }
        }
    };
    load(first);
    F::forward(w, lds, tw, t);
    __syncthreads();   // the kernel's last reads precede the first tile's writes
    for (int q = first; q < last; ++q) {
        C v[S::PPT];
        if (!NEXT && q > first) load(q);
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) v[r] = nx[r];
        F::forward(v, lds, tw, t);
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) v[r] = cmul(v[r], w[r]);
        if (NEXT && q + 1 < last) load(q + 1);   // travels while this tile is transformed back
        F::inverse(v, lds, tw, t);
#pragma unroll
        for (int im = 0; im < 2; ++im) {
            const int cell = tilek::tile_cell(ax, 2 * q + im);
            if constexpr (FAR) {
#pragma unroll
                for (int i = 0; i < PW; ++i) {
                    const int m = mw + (i << LMW), o = cell + ax.d * (m - (ax.K - 1));
                    int rem = 0;
                    const int oi = m >= ax.K - 1 && cell != kNoTile && o < ax.U ? tilek::div_by(ax.stride, o, &rem) : -1;
                    if (oi >= 0 && rem == 0) y[oi] = im ? v[i].y : v[i].x;
                }
            } else {
                Io::template outs<PW, (1 << LMW)>(co, ax, cell, mw);
#pragma unroll
                for (int i = 0; i < PW; ++i) tilek::store_real(py, co[i], im ? v[i].y : v[i].x);
            }
        }
    }
}

template <class S, bool FAR, bool NEXT>
ndc_status launch_class(const BatchTileArgs& a, const BatchTile* items, int n, const char* name, double bytes,
                        LaunchContext& ctx, hipStream_t stream, bool profile) {
    if (n <= 0) return NDC_OK;
    const auto kernel = &batch_tile_kernel<S, FAR, NEXT>;
    const size_t smem = size_t(S::N) * sizeof(float2);
    if (!lds_fits(ctx, reinterpret_cast<const void*>(kernel), smem)) return NDC_ERR_UNSUPPORTED;
    if (profile) ctx.kbegin(name, bytes, 0);
    NDC_LAUNCH(ctx, stream, kernel, dim3(unsigned(n)), dim3(S::T), smem, a, items, n);
    if (profile) ctx.kend();
    if (hipGetLastError() != hipSuccess) {
        ctx.err = std::string(name) + " launch failed";
        return NDC_ERR_DEVICE;
    }
    return NDC_OK;
}

}  // namespace

bool batch_tile_tables(LaunchContext& ctx, const void* tw[kBatchTileClasses]) {
    for (int c = 0; c < kBatchTileClasses; ++c) {
        const int lw = batch_tile_log2(c), lp = c == 0 ? 2 : c == kBatchTileFar ? 4 : 3;
        const std::vector<double>& tab = tile_twiddles(0, lw, lp);
        const std::vector<float> f(tab.begin(), tab.end());
        tw[c] = ctx.constant_table("tile:0:" + std::to_string(lw) + ":" + std::to_string(lp) + ":f", f.data(),
                                   f.size() * sizeof(float));
        if (!tw[c]) return false;
    }
    return true;
}

ndc_status launch_batch_tiles(const BatchArgs& b, const BatchTileLaunch& l, LaunchContext& ctx, hipStream_t stream,
                              bool profile) {
    BatchTileArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = b.x;
    a.k = b.k;
    a.y = b.y;
    a.heads = b.counter;
    a.phases = tile_div(b.d);
    a.stride = tile_div(b.s);
    a.rev = b.rev;
    a.front = b.front;
    a.back = b.back;
    a.cfront = b.cfront;
    a.cback = b.cback;
    a.fills = (b.front == kS1Const && b.cfront != 0.0f) || (b.back == kS1Const && b.cback != 0.0f);
    // the longer tiles first: the tail is made of the shorter
    a.tw = l.tw[3];
    ndc_status s = launch_class<Shape<0, 14, 4>, true, false>(a, l.items[3], l.n[3], "batch_tile16384", l.bytes[3], ctx,
                                                              stream, profile);
    if (s != NDC_OK) return s;
    a.tw = l.tw[2];
    s = launch_class<Shape<0, 13, 3>, false, false>(a, l.items[2], l.n[2], "batch_tile8192", l.bytes[2], ctx, stream,
                                                    profile);
    if (s != NDC_OK) return s;
    a.tw = l.tw[1];
    s = launch_class<Shape<0, 12, 3>, false, false>(a, l.items[1], l.n[1], "batch_tile4096", l.bytes[1], ctx, stream,
                                                    profile);
    if (s != NDC_OK) return s;
    a.tw = l.tw[0];
    return launch_class<Shape<0, 10, 2>, false, true>(a, l.items[0], l.n[0], "batch_tile1024", l.bytes[0], ctx, stream,
                                                      profile);
}

}  // namespace ndc
