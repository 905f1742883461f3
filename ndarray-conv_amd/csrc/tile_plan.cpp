// Which convolutions run as overlap-save tiles (tile_kernels.hpp), on which
// tile, and the host side of their launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "border1d.hpp"
#include "tile_conv.hpp"
#include "tile_fft.hpp"

namespace ndc {

namespace {

using tilefft::Shape;

template <int LH, int LW, int LP>
std::vector<double> make_twiddles() {
    using S = Shape<LH, LW, LP>;
    static constexpr tilefft::Map<S, 5> m5{};
    static constexpr tilefft::Map<S, 4> m4{};
    // the table's layout depends on the digits only
    static_assert(m5.ntw == m4.ntw, "twiddle layout");
    std::vector<double> t(size_t(2) * m5.ntw + 2);
    auto fill = [&](int off, int digit, int low) {
        const int P = 1 << digit, M = 1 << low;
        for (int k = 1; k < P; ++k)
            for (int m = 0; m < M; ++m) {
                // an angle in 64 bits would be off by several ulp of its cosine
                const long double ang = -2.0L * 3.14159265358979323846264338327950288L * (k * m) / (P * M);
                t[size_t(2) * (off + (k - 1) * M + m)] = double(std::cos(ang));
                t[size_t(2) * (off + (k - 1) * M + m) + 1] = double(std::sin(ang));
            }
    };
    for (int p = 0; p < S::NP; ++p) {
        if (m5.wlow[p] > 0 && S::aw[p] > 0) fill(m5.tww[p], S::aw[p], m5.wlow[p]);
        if (m5.hlow[p] > 0 && S::ah[p] > 0) fill(m5.twh[p], S::ah[p], m5.hlow[p]);
    }
    return t;
}

// Made once: a plan of new shapes needs the table again (0.1 to 2 ms).
template <int LH, int LW, int LP>
const std::vector<double>& twiddles_of() {
    static const std::vector<double> t = make_twiddles<LH, LW, LP>();
    return t;
}

// The tiles, and what one costs (ns, single precision, MI355X): `lat` from
// launch to end of a single tile, `point` per complex point while a CU works
// through many.  Fitted to kernel times of 200x5000, 512x512, 2048x2048,
// 4096x32768 and 1-D inputs, which it gives within 20%.  Double precision
// takes 1.8 times as long per point.
struct Cand {
    int lh, lw, lp;
    bool f32, f64;      // built for one convolution per tile
    bool sum32, sum64;  // built for sums over outer taps
    double lat, point;
};
constexpr Cand kCands[] = {
    {0, 10, 2, true, true, false, false, 3000, 0.9},  {0, 12, 3, true, true, false, false, 6000, 1.0},
    {0, 14, 4, true, false, false, false, 22000, 1.6}, {5, 5, 2, true, true, true, true, 3000, 0.9},
    {6, 6, 3, true, true, true, true, 6000, 1.03},     {5, 7, 3, false, true, true, true, 6500, 1.05},
    {5, 7, 4, true, false, false, false, 7000, 0.97},  {6, 7, 4, true, false, false, false, 9000, 1.12},
    {7, 7, 4, true, false, false, false, 20000, 1.9},
};

// Spans stay below 2^30 bytes, so that a cell's offset is 30 bits and the
// marker of a cell that is not read (tile_kernels.hpp kNoCell) lies past it.
constexpr int64_t kSpanMax = int64_t(1) << 30;
// Inputs up to this size are looked over by every workgroup of a one-launch
// plan (64 loads per thread at most, 128 of complex elements).
constexpr int64_t kScanMax = 16384;
constexpr int64_t kMaxTaps = 16;
// Kept spectra of x's tiles, as long as they stay in cache: at 6.5 MB
// (100x100x100, 3x5x7 taps) they take 20.5 us against 21.5 transforming per tap, at
// 13.6 MB (128x128x128, 3x3x3) 59 against 33.
constexpr int64_t kKeptMax = int64_t(8) << 20;

bool side_ok(const ndc_border& b, int64_t pad, int64_t n) {
    switch (side1d(b.tag)) {
        case kS1Reflect: return pad <= n - 1;
        case kS1Circular: return pad <= n;
        default: return true;
    }
}

// What the multi-pass transforms take (ns), from the same measurements: a fixed
// part per rank (their launches) and one per point.  Tiles lose only where
// few large ones do the work: an 80x80 kernel on 512x512 (36 against 33 us), 16
// outer taps on 30x60x60 (62 against 40 us).
double pass_cost(const Plan& p) {
    double pts = 1;
    for (int i = 0; i < p.N; ++i) pts *= double(p.fft[i]);
    if (p.N == 1) return pts <= 20000 ? 8000 + 1.5 * pts : 1e30;   // one launch while a line fits LDS
    const double each = (dtype_is_complex(p.dtype) ? 2.0 : 1.0) * (p.dtype == NDC_F64 || p.dtype == NDC_C128 ? 1.4 : 1.0);
    return (p.N == 2 ? 25000 : 36000 + 9000 * (p.N - 3)) + 0.03 * each * pts;
}

bool const_nonzero(const ndc_border& b) {
    return side1d(b.tag) == kS1Const && (b.value.re != 0 || b.value.im != 0);
}

// A constant that is not finite in the element type.
bool const_nonfinite(const ndc_border& b, bool cplx, bool dbl) {
    if (side1d(b.tag) != kS1Const) return false;
    auto bad = [&](double v) { return dbl ? !std::isfinite(v) : !std::isfinite(float(v)); };
    return bad(b.value.re) || (cplx && bad(b.value.im));
}

// Whether no output reads some cell of x along axis i: cells between the taps
// of a stride, or of a dilation longer than the output, and past the last
// output.  Taken for so where looking at every cell would take the host long.
bool axis_gaps(const Plan& p, int i) {
    const int64_t s = p.stride[i], d = p.dil[i], K = p.k_shape[i], out = p.out[i], n = p.x_shape[i];
    if (s == 1) return K > 1 && out < d;
    if (n > (int64_t(1) << 20) / K) return true;
    for (int64_t c = 0; c < n; ++c) {
        bool read = false;
        for (int64_t k = 0; k < K && !read; ++k) {
            const int64_t q = c + p.pad[i][0] - k * d;
            read = q >= 0 && q % s == 0 && q / s < out;
        }
        if (!read) return true;
    }
    return false;
}

// Whether some tap of axis i meets nothing but constant fill.
bool axis_idle(const Plan& p, int i) {
    const int64_t s = p.stride[i], out = p.out[i], lo = p.pad[i][0], hi = lo + p.x_shape[i];
    const bool front = side1d(p.side[i][0].tag) != kS1Const, back = side1d(p.side[i][1].tag) != kS1Const;
    for (int64_t k = 0; k < p.k_shape[i]; ++k) {
        const int64_t P0 = k * p.dil[i], P1 = P0 + (out - 1) * s;   // its first and last cell
        const int64_t in = P0 >= lo ? P0 : P0 + (lo - P0 + s - 1) / s * s;
        if (!((in <= P1 && in < hi) || (front && P0 < lo) || (back && P1 >= hi))) return true;
    }
    return false;
}

}  // namespace

TileDiv tile_div(int64_t d) { return TileDiv{uint32_t(d), uint32_t(d == 1 ? 0 : ((int64_t(1) << 32) + d - 1) / d)}; }

void tile_axis(const Plan& p, int i, int64_t ystr, TileAxis* a) {
    const int64_t es = int64_t(dtype_size(p.dtype));
    std::memset(a, 0, sizeof(*a));
    a->n = int32_t(p.x_shape[i]);
    a->p0 = int32_t(p.pad[i][0]);
    a->pds = int32_t(p.pds[i]);
    const int32_t n = a->n;
    switch (side1d(p.side[i][0].tag)) {
        case kS1Reflect: a->fa = -1; break;
        case kS1Circular: a->fa = 1; a->fb = n; break;
        case kS1Replicate: break;
        default: a->fconst = 1; break;
    }
    switch (side1d(p.side[i][1].tag)) {
        case kS1Reflect: a->ba = -1; a->bb = 2 * (n - 1); break;
        case kS1Circular: a->ba = 1; a->bb = -n; break;
        case kS1Replicate: a->bb = n - 1; break;
        default: a->bconst = 1; break;
    }
    const int64_t st = n > 1 ? p.x_str[i] * es : 0;
    a->xs = int32_t(st);
    a->xlo = int32_t(st < 0 ? -st * (n - 1) : 0);
    // position j of the spectrum holds tap j, or K - 1 - j without the reversal
    const int64_t K = p.k_shape[i], kt = K > 1 ? p.k_str[i] * es : 0, kd = p.reverse ? kt : -kt;
    a->ks = int32_t(kd);
    a->klo = int32_t(kd < 0 ? -kd * (K - 1) : 0);
    a->d = int32_t(p.dil[i]);
    a->phases = tile_div(a->d);
    a->stride = tile_div(p.stride[i]);
    a->K = int32_t(p.k_shape[i]);
    a->s = int32_t(p.stride[i]);
    a->U = int32_t(p.pds[i] - p.kdil[i] + 1);
    a->ys = int32_t(ystr * es);
}

bool tile_spans_fit(const Plan& p) {
    const int64_t es = int64_t(dtype_size(p.dtype));
    if ((p.x_hi - p.x_lo + 1) * es >= kSpanMax || (p.k_hi - p.k_lo + 1) * es >= kSpanMax || p.y_numel * es >= kSpanMax)
        return false;
    for (int i = 0; i < p.N; ++i) {
        if (!side_ok(p.side[i][0], p.pad[i][0], p.x_shape[i]) || !side_ok(p.side[i][1], p.pad[i][1], p.x_shape[i]))
            return false;
        // room for the positions a tile reaches past the padded extent; a single
        // tap may have any dilation, and direct convolution takes dilation 0
        if (p.dil[i] < 1 || p.dil[i] >= kSpanMax >> 14 || p.pds[i] + (p.dil[i] << 14) >= kSpanMax) return false;
        if (p.stride[i] >= kSpanMax) return false;
    }
    return true;
}

const std::vector<double>& tile_twiddles(int lh, int lw, int lp) {
    static const std::vector<double> none;
    switch ((lh * 16 + lw) * 8 + lp) {
        case (0 * 16 + 10) * 8 + 2: return twiddles_of<0, 10, 2>();
        case (0 * 16 + 12) * 8 + 3: return twiddles_of<0, 12, 3>();
        case (0 * 16 + 13) * 8 + 3: return twiddles_of<0, 13, 3>();
        case (0 * 16 + 14) * 8 + 4: return twiddles_of<0, 14, 4>();
        case (5 * 16 + 5) * 8 + 2: return twiddles_of<5, 5, 2>();
        case (6 * 16 + 6) * 8 + 3: return twiddles_of<6, 6, 3>();
        case (5 * 16 + 7) * 8 + 3: return twiddles_of<5, 7, 3>();
        case (5 * 16 + 7) * 8 + 4: return twiddles_of<5, 7, 4>();
        case (6 * 16 + 7) * 8 + 4: return twiddles_of<6, 7, 4>();
        case (7 * 16 + 7) * 8 + 4: return twiddles_of<7, 7, 4>();
        default: return none;
    }
}

bool tile_plan(const Plan& p, size_t lds, int cus, TilePlan* t) {
    const bool cplx = dtype_is_complex(p.dtype);
    const bool dbl = p.dtype == NDC_F64 || p.dtype == NDC_C128;
    const int N = p.N, w = N - 1, h = N - 2;
    const int64_t es = int64_t(dtype_size(p.dtype)), cs = dbl ? 16 : 8;
    if (!tile_spans_fit(p)) return false;
    int64_t taps = 1, planes = 1, xplanes = 1;
    bool fills = false;
    t->gaps = t->idle = t->nan = false;
    for (int i = 0; i < N; ++i) {
        if (i < h) {
            taps *= p.k_shape[i];
            planes *= p.out[i];
            xplanes *= p.x_shape[i];
        }
        for (int s = 0; s < 2; ++s)
            if (p.pad[i][s] > 0) {
                fills = fills || const_nonzero(p.side[i][s]);
                t->nan = t->nan || const_nonfinite(p.side[i][s], cplx, dbl);
            }
    }
    if (taps > kMaxTaps) return false;
    for (int i = 0; i < h; ++i) {
        t->gaps = t->gaps || axis_gaps(p, i);
        t->idle = t->idle || (!fills && axis_idle(p, i));
    }
    if (t->gaps && xplanes >= kSpanMax) return false;   // a broadcast view: planes are counted in 30 bits
    t->xplanes = t->gaps ? int(xplanes) : 0;
    const bool compact = p.x_hi - p.x_lo + 1 == p.x_numel;
    const bool one = N == 1 && p.x_numel <= kScanMax;
    if (one && !compact) return false;

    auto tiles = [&](int i, int lsz, int64_t* V) -> int64_t {
        *V = (int64_t(1) << lsz) - p.k_shape[i] + 1;
        const int64_t U = p.pds[i] - p.kdil[i] + 1;
        const int64_t per = (U + p.dil[i] - 1) / p.dil[i];   // outputs of a phase
        return *V > 0 ? (per + *V - 1) / *V : 0;
    };
    double best = 0;
    for (const Cand& c : kCands) {
        if ((N == 1) != (c.lh == 0)) continue;
        if (!(N > 2 ? (dbl ? c.sum64 : c.sum32) : (dbl ? c.f64 : c.f32))) continue;
        if (one && c.lw > 12) continue;
        const int64_t pts = int64_t(1) << (c.lh + c.lw);
        if (size_t(pts * cs) + (N == 1 && dbl ? 32 : 0) > lds) continue;   // and two slots (mean_apart)
        int64_t vw, vh = 1;
        const int64_t nw = tiles(w, c.lw, &vw);
        const int64_t nh = N == 1 ? 1 : tiles(h, c.lh, &vh);
        if (nw <= 0 || nh <= 0 || vw * vh * 8 < pts) continue;
        // real elements: the axis whose number of tiles wastes the smaller
        // part of its pairs
        const int64_t cw = nw * p.dil[w], ch = N == 1 ? 1 : nh * p.dil[h];
        const bool pair_w = ((cw + 1) / 2) * ch <= cw * ((ch + 1) / 2);
        const int64_t pw = !cplx && pair_w ? (cw + 1) / 2 : cw, ph = !cplx && !pair_w ? (ch + 1) / 2 : ch;
        if (cw >= kSpanMax || ch >= kSpanMax || double(pw) * double(ph) * double(planes) >= double(kSpanMax)) continue;
        const int64_t pi = pw * ph, items = pi * planes;
        // a sum over outer taps transforms once per tap and once back, or, from
        // kept spectra of x, each tile once; the spectra stay in cache
        const double per = c.point * (dbl ? 1.8 : 1.0) * double(pts) / cus;
        const double xspec = double(xplanes) * double(pi) * double(pts * cs);
        const bool keep = N > 2 && !fills && xspec <= double(kKeptMax) && double(xplanes) < double(planes) * double(taps);
        const double trips = N > 2 ? 0.425 * (1.0 + double(taps)) : 1.0;
        const double cost = keep ? 1.1 * c.lat + 0.5 * per * double(pi) * double(xplanes + planes) +
                                       double(items) * double(taps) * double(pts * cs) / 2000.0 + 3000.0
                                 : (c.lat + per * double(items)) * trips +
                                       (one ? 0.0 : 0.6 * c.lat + 3000.0);   // the spectrum and fix-up launches
        if (best != 0 && cost >= best) continue;
        best = cost;
        t->lh = c.lh;
        t->lw = c.lw;
        t->lp = c.lp;
        t->threads = int(pts >> c.lp);
        t->lds = size_t(pts * cs);
        t->spec_bytes = size_t(pts * cs) * size_t(taps);
        t->xspec_bytes = keep ? size_t(xspec) : 0;
        std::memset(&t->a, 0, sizeof(t->a));
        t->a.xitems = int32_t(keep ? xplanes * pi : 0);
        t->a.pair_w = pair_w ? 1 : 0;
        t->a.ax[0].pairs = tile_div(ph);
        t->a.ax[1].pairs = tile_div(pw);
        t->a.plane_items = tile_div(pi);
        t->a.items = int32_t(items);
        t->a.ax[0].V = int32_t(vh);
        t->a.ax[0].tiles = tile_div(nh);
        t->a.ax[1].V = int32_t(vw);
        t->a.ax[1].tiles = tile_div(nw);
    }
    if (best == 0 || best > pass_cost(p)) return false;

    TileArgs& a = t->a;
    t->one = one;
    a.x_bytes = int32_t((p.x_hi - p.x_lo + 1) * es);
    a.y_bytes = int32_t(p.y_numel * es);
    a.ntaps = int32_t(taps);
    a.nouter = std::max(0, h);
    a.k_bytes = int32_t((p.k_hi - p.k_lo + 1) * es);
    t->fills = fills;
    // a single workgroup sees all of x anyway
    a.scan = one && a.items > 1 ? int32_t(p.x_numel * (cplx ? 2 : 1)) : 0;
    int64_t ystr[kMaxRank], ys = 1;
    for (int i = N - 1; i >= 0; --i) {
        ystr[i] = ys;
        ys *= p.out[i];
    }
    auto axis = [&](int i, TileAxis* dst, int slot) {
        const int32_t V = dst->V;
        const TileDiv nt = dst->tiles, np = dst->pairs;
        tile_axis(p, i, ystr[i], dst);
        dst->V = V;
        dst->tiles = nt;
        dst->pairs = np;
        for (int s = 0; s < 2; ++s) {
            a.cst[slot][s][0] = p.side[i][s].value.re;
            a.cst[slot][s][1] = p.side[i][s].value.im;
        }
    };
    axis(w, &a.ax[1], 1);
    if (N > 1) {
        axis(h, &a.ax[0], 0);
    } else {
        TileAxis& u = a.ax[0];   // a single row
        u.n = u.pds = u.d = u.K = u.V = u.U = u.s = 1;
        u.phases = u.tiles = u.pairs = u.stride = tile_div(1);
        u.fconst = u.bconst = 1;
    }
    int64_t step = 1;
    for (int i = h - 1; i >= 0; --i) {
        axis(i, &a.outer[i].a, 2 + i);
        a.outer[i].cells = tile_div(p.x_shape[i]);
        a.outer[i].step = int32_t(step);
        step *= p.x_shape[i];
        a.outer[i].out = tile_div(p.out[i]);
        a.outer[i].taps = tile_div(p.k_shape[i]);
    }
    return true;
}

ndc_status launch_tile(const Plan& p, const TilePlan& t, const void* x, const void* k, void* y, LaunchContext& ctx,
                       KernelSpectrum* ks) {
    const bool cplx = dtype_is_complex(p.dtype);
    const bool dbl = p.dtype == NDC_F64 || p.dtype == NDC_C128;
    TileArgs a = t.a;
    a.x = x ? static_cast<const char*>(x) + p.x_lo * int64_t(dtype_size(p.dtype)) : nullptr;
    a.k = k ? static_cast<const char*>(k) + p.k_lo * int64_t(dtype_size(p.dtype)) : nullptr;
    a.y = y;
    if (t.nan && !(ks && ks->bake))   // without a flag: y is filled in any case
        return dbl ? launch_tile_as<double>(t, a, cplx, 2, ctx) : launch_tile_as<float>(t, a, cplx, 2, ctx);
    if (!t.tw || !t.flag) {
        const std::string key = "tile:" + std::to_string(t.lh) + ":" + std::to_string(t.lw) + ":" + std::to_string(t.lp) + (dbl ? ":d" : ":f");
        const std::vector<double>& tab = tile_twiddles(t.lh, t.lw, t.lp);
        std::vector<float> f;
        if (!dbl) f.assign(tab.begin(), tab.end());
        t.tw = dbl ? ctx.constant_table(key, tab.data(), tab.size() * sizeof(double))
                   : ctx.constant_table(key, f.data(), f.size() * sizeof(float));
        const uint32_t zeros[2] = {0, 0};
        t.flag = static_cast<uint32_t*>(const_cast<void*>(ctx.constant_table("tile:flag", zeros, sizeof(zeros))));
    }
    a.tw = t.tw;
    a.flag = t.flag;
    if (!a.tw || !a.flag) {
        if (ctx.err.empty()) ctx.err = "tile table allocation failed";
        return NDC_ERR_OUT_OF_MEMORY;
    }
    auto go = [&](int what) {
        return dbl ? launch_tile_as<double>(t, a, cplx, what, ctx) : launch_tile_as<float>(t, a, cplx, what, ctx);
    };
    if (ks) {
        a.spec = ks->spec;
        a.have_spec = 1;
        if (ks->bake) return go(0);
    }
    if (!t.one && (!ks || t.xspec_bytes)) {
        const size_t own = ks ? 0 : t.spec_bytes;   // a multiple of 8 KB
        char* mem = static_cast<char*>(ctx.scratch(0, own + t.xspec_bytes));
        if (!mem) {
            if (ctx.err.empty()) ctx.err = "kernel spectrum allocation failed";
            return NDC_ERR_OUT_OF_MEMORY;
        }
        if (!ks) a.spec = mem;
        if (t.xspec_bytes) a.xspec = mem + own;
        const ndc_status s = go(t.xspec_bytes ? 3 : 0);
        if (s != NDC_OK) return s;
    }
    ndc_status s = t.gaps || t.idle ? go(4) : NDC_OK;
    if (s == NDC_OK) s = go(1);
    if (s == NDC_OK && !t.one) s = go(2);
    return s;
}

}  // namespace ndc
