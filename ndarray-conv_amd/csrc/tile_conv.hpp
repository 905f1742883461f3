// FFT convolution by overlap-save tiles: the plan (tile_plan.cpp) and the
// kernels' arguments.  See tile_kernels.hpp for the algorithm.
#pragma once

#include <cstdint>
#include <vector>

#include "launch.hpp"
#include "plan.hpp"

namespace ndc {

// Division of 0 <= n < 2^30 by a divisor known to the host: mulhi(n, m) with
// m = ceil(2^32 / d) is the quotient or one more.
struct TileDiv {
    uint32_t d, m;
};

// One tiled axis.  Position j of a tile at (phase f, tile t) is the padded
// cell d (t V + j) + f; rel = that - p0 indexes x, with the fills folded in as
// idx = a rel + b (front a/b for rel < 0, back for rel >= n).
struct TileAxis {
    int32_t n, p0, pds;
    int32_t fa, fb, ba, bb;
    int32_t fconst, bconst;   // the side writes a constant
    int32_t xs, xlo;          // byte stride in x, and the bytes its lowest element lies below element 0
    int32_t ks, klo;          // the same of k, in the order the spectrum's positions take the taps
    int32_t d, K, V;          // dilation (= phases), taps, outputs per tile and phase
    int32_t U, s, ys;         // outputs at stride 1, stride, byte stride in y
    TileDiv phases, tiles;    // d, and tiles per phase
    TileDiv pairs;            // positions along the axis: complex tiles, or pairs of real tiles
    TileDiv stride;
};

// One axis outside the tile: its taps are summed one by one.
struct TileOuter {
    TileAxis a;
    TileDiv out, taps;
    TileDiv cells;        // cells of x
    int32_t step;         // planes of x from one cell to the next
};

constexpr int kMaxTileOuter = kMaxRank - 2;

struct TileArgs {
    const void* x;        // the lowest element the view touches
    const void* k;
    void* y;
    void* spec;           // kernel spectra, one per outer tap: [tap][register][thread]
    void* xspec;          // spectra of x's tiles, [plane][tile][register][thread]; null when not kept
    const void* tw;
    uint32_t* flag;       // [0] set when an output is not finite, [1] counts the fix-up's blocks
    int32_t x_bytes, k_bytes, y_bytes;
    int32_t nouter, ntaps;
    int32_t xitems;       // complex tiles of all planes of x
    int32_t items;        // complex tiles of the launch
    TileDiv plane_items;  // complex tiles per outer output position
    int32_t pair_w;       // real elements: a complex tile is two neighbours along w (else along h)
    int32_t scan;         // values of x to look over for non-finite ones (one-launch plans)
    int32_t have_spec;
    TileAxis ax[2];       // h, w
    double cst[kMaxRank][2][2];   // [h, w, outer...][front, back][re, im]
    TileOuter outer[kMaxTileOuter];
};

// The form a plan takes: which tile, and how its launches are made.
struct TilePlan {
    int lh = 0, lw = 0;      // log2 of the tile
    int lp = 0;              // log2 of the points a thread holds
    bool one = false;        // one launch: every workgroup transforms the kernel itself
    bool fills = false;      // some fill writes a constant other than zero
    // what no tile of the sums over outer taps reads (a non-finite value there
    // still makes every output NaN): planes of x, and taps that only meet zero fill
    bool gaps = false, idle = false;
    int xplanes = 0;         // planes of x
    bool nan = false;        // a fill writes a non-finite constant: every output is NaN
    TileArgs a;              // shape part; pointers unset
    size_t spec_bytes = 0;
    size_t xspec_bytes = 0;  // rank 3 and up: kept spectra of x's tiles (0: transformed once per tap)
    size_t lds = 0;
    int threads = 0;
    // device tables of the handle the plan belongs to, looked up by the first launch
    mutable const void* tw = nullptr;
    mutable uint32_t* flag = nullptr;
};

// False when the plan is left to the multi-pass transforms (fft_conv.hip).
bool tile_plan(const Plan& p, size_t lds, int cus, TilePlan* t);

// The plan's tile form, decided once and kept in the plan; null when it has none.
const TilePlan* tile_of(const Plan& p, LaunchContext& ctx);

ndc_status launch_tile(const Plan& p, const TilePlan& t, const void* x, const void* k, void* y, LaunchContext& ctx,
                       KernelSpectrum* ks);

// The per-precision launchers (tile_conv.hip, tile_conv_f64.hip).
template <typename R> ndc_status launch_tile_as(const TilePlan& t, const TileArgs& a, bool cplx, int what,
                                                LaunchContext& ctx);

// For other kernels that read their input through TileAxis (cell_offset):
// whether every span of the plan is below 2^30 bytes and every pad within its
// axis, the division constants, and one axis of a plan (ystr: elements of y
// from one output to the next).
bool tile_spans_fit(const Plan& p);
TileDiv tile_div(int64_t d);
void tile_axis(const Plan& p, int i, int64_t ystr, TileAxis* a);

// Host table of a tile's twiddles (kept for the process), empty for an unknown tile.
const std::vector<double>& tile_twiddles(int lh, int lw, int lp);

// Whether the multi-pass form can transform this plan's axes at all; what it
// refuses stays refused.
bool pass_form_fits(const Plan& p, size_t lds);

}  // namespace ndc
