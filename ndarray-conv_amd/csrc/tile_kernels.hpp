// FFT convolution by overlap-save tiles (conv_fft/mod.rs:185-292 computes one
// circular convolution of the whole padded array; the linear part it keeps is
// the same sum, so tiles of any size give it, with less rounding).
//
// A workgroup takes one complex H x W tile of the padded input, gathered
// through the border rules, transforms it (tile_fft.hpp), multiplies by the
// kernel's spectrum and transforms back: x is read and y written once, with
// no spectrum in memory.  Real data goes two tiles at a time as the real and
// imaginary part: the kernel is real, so the two never mix.  A dilated axis is
// split into its d phases, each convolved with the plain kernel, which keeps
// the halo at K - 1 cells.  Axes outside the last two are summed tap by tap
// over the spectra.
//
// Bound: vector instructions.  A 4096x32768 f32 convolution (11x31 taps,
// dilation 2) takes 457 us on 64x128 tiles, 1.1 ns per complex point and CU
// where the transforms' own arithmetic takes 0.6; its 1.07 GB would take 200 us.
// The multi-pass transforms of the same call took 9.1 ms (seven passes over
// 1.2-2.7 GB of spectra), of a 200x5000 one 38 us against 17 here, of a
// 10x100x200 complex one 65 against 26.
//
// Non-finite data: the whole-array transform makes every output NaN.  Within
// a tile the FFT spreads a non-finite value to every point, so one point per
// thread tells; it raises a flag and the fix-up launch fills y with NaN.  What
// no tile transforms is looked over apart: planes of x between the taps of a
// stride or dilation, and kept spectra of taps that only meet zero fill
// (tile_scan_kernel).  A non-finite pad constant is known to the host.
#pragma once

#include <algorithm>
#include <string>

#include "device_common.hpp"
#include "tile_conv.hpp"
#include "tile_fft.hpp"

namespace ndc {
namespace tilek {

using tilefft::Shape;
using tilefft::static_for;
using tilefft::TileFft;

// Byte offset of a cell that is not read: past every buffer, also as the sum of
// two of them and an offset below 2^30.
constexpr uint32_t kNoCell = 0x40000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* base, int bytes) {
    // word 3 of a raw 32-bit buffer
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

template <typename R> __device__ __forceinline__ R load_real(__amdgpu_buffer_rsrc_t b, uint32_t off);
template <> __device__ __forceinline__ float load_real<float>(__amdgpu_buffer_rsrc_t b, uint32_t off) {
    return __builtin_bit_cast(float, uint32_t(__builtin_amdgcn_raw_buffer_load_b32(b, int(off), 0, 0)));
}
template <> __device__ __forceinline__ double load_real<double>(__amdgpu_buffer_rsrc_t b, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, int(off), 0, 0));
}
__device__ __forceinline__ float2 load_cx(__amdgpu_buffer_rsrc_t b, uint32_t off, float) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(b, int(off), 0, 0));
}
__device__ __forceinline__ double2 load_cx(__amdgpu_buffer_rsrc_t b, uint32_t off, double) {
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(b, int(off), 0, 0));
}
using u32x2 = uint32_t __attribute__((ext_vector_type(2)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_real(__amdgpu_buffer_rsrc_t b, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), b, int(off), 0, 0);
}
__device__ __forceinline__ void store_real(__amdgpu_buffer_rsrc_t b, uint32_t off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), b, int(off), 0, 0);
}
__device__ __forceinline__ void store_cx(__amdgpu_buffer_rsrc_t b, uint32_t off, float2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), b, int(off), 0, 0);
}
__device__ __forceinline__ void store_cx(__amdgpu_buffer_rsrc_t b, uint32_t off, double2 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), b, int(off), 0, 0);
}

// Where padded cell P of an axis reads: its byte offset in x, or kNoCell.
__device__ __forceinline__ uint32_t cell_offset(const TileAxis& a, int P) {
    const int rel = P - a.p0;
    const int m = rel < 0 ? a.fa : rel >= a.n ? a.ba : 1;
    const int c = rel < 0 ? a.fb : rel >= a.n ? a.bb : 0;
    const bool none = P >= a.pds || (rel < 0 ? a.fconst : rel >= a.n ? a.bconst : 0);
    return none ? kNoCell : uint32_t(m * rel + c) * uint32_t(a.xs) + uint32_t(a.xlo);
}
// 0 reads x, 1 / 2 the front / back constant, 3 beyond the padded extent
__device__ __forceinline__ int cell_kind(const TileAxis& a, int P) {
    if (P >= a.pds) return 3;
    const int rel = P - a.p0;
    return rel < 0 ? (a.fconst ? 1 : 0) : rel >= a.n ? (a.bconst ? 2 : 0) : 0;
}
// n / d and the remainder, for a wave-uniform n.
__device__ __forceinline__ int div_by(const TileDiv& v, int n, int* rem) {
    int q = v.d == 1 ? n : int(__umulhi(uint32_t(n), v.m));
    int r = n - q * int(v.d);
    if (r < 0) {
        --q;
        r += int(v.d);
    }
    *rem = r;
    return q;
}

// Byte offset in y of output o of an axis, or kNoCell where it has none.
__device__ __forceinline__ uint32_t out_offset(const TileAxis& a, int o) {
    int r;
    const int q = div_by(a.stride, o, &r);
    return o < a.U && r == 0 ? uint32_t(q) * uint32_t(a.ys) : kNoCell;
}

// The padded cell of position 0 of tile i of an axis, tiles numbered phase
// fastest; kNoTile past the last one.
constexpr int kNoTile = -1;
__device__ __forceinline__ int tile_cell(const TileAxis& a, int i) {
    int f;
    const int t = div_by(a.phases, i, &f);
    return t < int(a.tiles.d) ? a.d * t * a.V + f : kNoTile;
}

// The two tiles (the same one twice for complex elements) of item q of a
// plane: the cells of their positions 0.
struct TilePair {
    int h[2], w[2];
};
template <bool CPLX>
__device__ __forceinline__ TilePair tile_pair(const TileArgs& a, int q) {
    int iw;
    const int ih = div_by(a.ax[1].pairs, q, &iw);
    TilePair p;
    if (CPLX) {
        p.h[0] = p.h[1] = tile_cell(a.ax[0], ih);
        p.w[0] = p.w[1] = tile_cell(a.ax[1], iw);
    } else if (a.pair_w) {
        p.h[0] = p.h[1] = tile_cell(a.ax[0], ih);
        p.w[0] = tile_cell(a.ax[1], 2 * iw);
        p.w[1] = tile_cell(a.ax[1], 2 * iw + 1);
    } else {
        p.h[0] = tile_cell(a.ax[0], 2 * ih);
        p.h[1] = tile_cell(a.ax[0], 2 * ih + 1);
        p.w[0] = p.w[1] = tile_cell(a.ax[1], iw);
    }
    return p;
}

// Consecutive tiles, which share halo cells, run on one XCD's L2: workgroups
// are dispatched round-robin over the eight XCDs, and each XCD's take one
// consecutive range of the items.
__device__ __forceinline__ int xcd_item(int g, int n) {
    const int per = n >> 3, rem = n & 7, x = g & 7;
    return x * per + (x < rem ? x : rem) + (g >> 3);
}

template <typename R, class S, bool CPLX, bool FILLS>
struct TileIo {
    using C = Cx<R>;
    using F = TileFft<R, S>;
    static constexpr int PW = 1 << S::aw[0], PH = 1 << S::ah[0];
    static constexpr int LMW = S::LW - S::aw[0], LMH = S::LH - S::ah[0];
    static constexpr int kMem = CPLX ? 1 : 2;   // tiles in a complex tile

    // Byte offsets of a thread's cells along one axis (n of them, step
    // positions apart) from the cell of its first position.  A tile inside x
    // needs no border rule: its cells are a fixed step apart.
    template <int P, int STEP>
    static __device__ __forceinline__ void cells(uint32_t* o, const TileAxis& a, int tile, int size, int m) {
        const int cell = tile + a.d * m;
        if (tile >= a.p0 && tile + a.d * (size - 1) < a.p0 + a.n) {   // uniform
            const uint32_t c0 = uint32_t(cell - a.p0) * uint32_t(a.xs) + uint32_t(a.xlo);
            const uint32_t st = uint32_t(a.d * STEP) * uint32_t(a.xs);
#pragma unroll
            for (int i = 0; i < P; ++i) o[i] = c0 + uint32_t(i) * st;
        } else {
#pragma unroll
            for (int i = 0; i < P; ++i) o[i] = tile == kNoTile ? kNoCell : cell_offset(a, cell + a.d * (i * STEP));
        }
    }
    // The same for y; positions before K - 1 and outputs past the last have none.
    template <int P, int STEP>
    static __device__ __forceinline__ void outs(uint32_t* o, const TileAxis& a, int tile, int m) {
        const int first = tile + a.d * (m - (a.K - 1));   // output of the first position
        if (a.s == 1) {   // uniform
            const uint32_t c0 = uint32_t(first) * uint32_t(a.ys), st = uint32_t(a.d * STEP) * uint32_t(a.ys);
#pragma unroll
            for (int i = 0; i < P; ++i)
                o[i] = m + i * STEP >= a.K - 1 && first + a.d * (i * STEP) < a.U && tile != kNoTile
                           ? c0 + uint32_t(i) * st : kNoCell;
        } else {
#pragma unroll
            for (int i = 0; i < P; ++i)
                o[i] = m + i * STEP >= a.K - 1 && tile != kNoTile ? out_offset(a, first + a.d * (i * STEP)) : kNoCell;
        }
    }

    // Loads the tile, or both tiles of a real pair, from plane `px`; with oc
    // the plane is the constant ocv.
    static __device__ __forceinline__ void load(C* v, const TileArgs& a, __amdgpu_buffer_rsrc_t px, const TilePair& p,
                                                int t, int oc, C ocv) {
        const int mw = F::template thr_value<0, 0, LMW>(t), mh = F::template thr_value<0, S::LW, LMH>(t);
        uint32_t co[PW], ro[PH];
        cells<PW, (1 << LMW)>(co, a.ax[1], p.w[0], 1 << S::LW, mw);
        cells<PH, (1 << LMH)>(ro, a.ax[0], p.h[0], 1 << S::LH, mh);
#pragma unroll
        for (int im = 0; im < kMem; ++im) {
            if (im && a.pair_w) cells<PW, (1 << LMW)>(co, a.ax[1], p.w[1], 1 << S::LW, mw);
            if (im && !a.pair_w) cells<PH, (1 << LMH)>(ro, a.ax[0], p.h[1], 1 << S::LH, mh);
#pragma unroll
            for (int h = 0; h < PH; ++h)
#pragma unroll
                for (int w = 0; w < PW; ++w) {
                    C& u = v[h * PW + w];
                    const uint32_t off = FILLS && oc ? kNoCell : ro[h] + co[w];
                    if constexpr (CPLX) u = load_cx(px, off, R(0));
                    else if (im) u.y = load_real<R>(px, off);
                    else u.x = load_real<R>(px, off);
                }
        }
        if constexpr (FILLS) {
#pragma unroll
            for (int im = 0; im < kMem; ++im)
                if (p.h[im] != kNoTile && p.w[im] != kNoTile)
                    fill(v, a, p.h[im] + a.ax[0].d * mh, p.w[im] + a.ax[1].d * mw, im, oc, ocv);
        }
    }
    // Constant fills: the highest axis whose fill writes a constant decides.
    static __device__ __forceinline__ void fill(C* v, const TileArgs& a, int bh, int bw, int im, int oc, C ocv) {
        const C w1 = cmake<C>(R(a.cst[1][0][0]), R(a.cst[1][0][1])), w2 = cmake<C>(R(a.cst[1][1][0]), R(a.cst[1][1][1]));
        const C h1 = cmake<C>(R(a.cst[0][0][0]), R(a.cst[0][0][1])), h2 = cmake<C>(R(a.cst[0][1][0]), R(a.cst[0][1][1]));
#pragma unroll
        for (int h = 0; h < PH; ++h) {
            const int kh = cell_kind(a.ax[0], bh + a.ax[0].d * (h << LMH));
            const C rv = kh == 1 ? h1 : kh == 2 ? h2 : ocv;
#pragma unroll
            for (int w = 0; w < PW; ++w) {
                const int kw = cell_kind(a.ax[1], bw + a.ax[1].d * (w << LMW));
                C& u = v[h * PW + w];
                if ((kw | kh | oc) != 0) {
                    C f = kw == 1 ? w1 : kw == 2 ? w2 : rv;
                    if (kw == 3 || kh == 3) f = cmake<C>(R(0), R(0));
                    if constexpr (CPLX) u = f;
                    else if (im) u.y = f.x;
                    else u.x = f.x;
                }
            }
        }
    }

    // The kernel's tile, the taps at byte offset ko of the outer axes, scaled
    // by 1/N.
    static __device__ __forceinline__ void load_kernel(C* v, const TileArgs& a, int ko, int t) {
        const int mw = F::template thr_value<0, 0, LMW>(t), mh = F::template thr_value<0, S::LW, LMH>(t);
        const R sc = R(1) / R(S::N);
        const __amdgpu_buffer_rsrc_t pk = buffer_of(static_cast<const char*>(a.k) + ko, a.k_bytes - ko);
        uint32_t co[PW], ro[PH];
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int j = mw + (i << LMW);
            co[i] = j < a.ax[1].K ? uint32_t(j) * uint32_t(a.ax[1].ks) + uint32_t(a.ax[1].klo) : kNoCell;
        }
#pragma unroll
        for (int i = 0; i < PH; ++i) {
            const int j = mh + (i << LMH);
            ro[i] = j < a.ax[0].K ? uint32_t(j) * uint32_t(a.ax[0].ks) + uint32_t(a.ax[0].klo) : kNoCell;
        }
#pragma unroll
        for (int h = 0; h < PH; ++h)
#pragma unroll
            for (int w = 0; w < PW; ++w) {
                if constexpr (CPLX) v[h * PW + w] = load_cx(pk, ro[h] + co[w], R(0));
                else v[h * PW + w] = cmake<C>(load_real<R>(pk, ro[h] + co[w]), R(0));
            }
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) v[r] = cscale(v[r], sc);
    }

    static __device__ __forceinline__ void store(const C* v, const TileArgs& a, __amdgpu_buffer_rsrc_t py,
                                                 const TilePair& p, int t) {
        const int mw = F::template thr_value<0, 0, LMW>(t), mh = F::template thr_value<0, S::LW, LMH>(t);
        uint32_t co[PW], ro[PH];
        outs<PW, (1 << LMW)>(co, a.ax[1], p.w[0], mw);
        outs<PH, (1 << LMH)>(ro, a.ax[0], p.h[0], mh);
#pragma unroll
        for (int im = 0; im < kMem; ++im) {
            if (im && a.pair_w) outs<PW, (1 << LMW)>(co, a.ax[1], p.w[1], mw);
            if (im && !a.pair_w) outs<PH, (1 << LMH)>(ro, a.ax[0], p.h[1], mh);
#pragma unroll
            for (int h = 0; h < PH; ++h)
#pragma unroll
                for (int w = 0; w < PW; ++w) {
                    if constexpr (CPLX) store_cx(py, ro[h] + co[w], v[h * PW + w]);
                    else store_real(py, ro[h] + co[w], im ? v[h * PW + w].y : v[h * PW + w].x);
                }
        }
    }
};

// One outer output position and tap: byte offsets into the kernel and into x,
// or (oc) the constant that the plane consists of.
struct OuterCell {
    int ko, xo, oc;
    int xp;         // the plane's number in x
    double re, im;
};
__device__ __forceinline__ OuterCell outer_cell(const TileArgs& a, int plane, int tap) {
    OuterCell c{0, 0, 0, 0, 0, 0};
    for (int i = a.nouter - 1; i >= 0; --i) {
        const TileOuter& o = a.outer[i];
        int pos, k;
        plane = div_by(o.out, plane, &pos);
        tap = div_by(o.taps, tap, &k);
        c.ko += k * o.a.ks + o.a.klo;
        const int P = pos * o.a.s + (o.a.K - 1 - k) * o.a.d;
        const int kind = cell_kind(o.a, P);
        if (kind) {
            if (!c.oc) {   // the highest axis's constant wins
                c.oc = 1;
                c.re = a.cst[2 + i][kind == 1 ? 0 : 1][0];
                c.im = a.cst[2 + i][kind == 1 ? 0 : 1][1];
            }
        } else {
            c.xo += int(cell_offset(o.a, P));
            const int rel = P - o.a.p0;
            const int m = rel < 0 ? o.a.fa : rel >= o.a.n ? o.a.ba : 1;
            c.xp += (m * rel + (rel < 0 ? o.a.fb : rel >= o.a.n ? o.a.bb : 0)) * o.step;
        }
    }
    if (c.oc) c.xo = 0;
    return c;
}

__device__ __forceinline__ bool nonfinite(float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7f800000u) == 0x7f800000u; }
__device__ __forceinline__ bool nonfinite(double v) {
    return (uint32_t(__builtin_bit_cast(uint64_t, v) >> 32) & 0x7ff00000u) == 0x7ff00000u;
}

// Kernel spectra: one workgroup per outer tap.  CHECK raises the flag for taps that
// no tile may use (outer axes); a kept spectrum raises none, the calls that use it do.
template <typename R, class S, bool CPLX, bool CHECK>
__global__ void __launch_bounds__(S::T) tile_spec_kernel(TileArgs a) {
    using C = Cx<R>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x;
    C v[S::PPT];
    const auto tw = TileFft<R, S>::load_tw(a.tw, t);
    TileIo<R, S, CPLX, false>::load_kernel(v, a, outer_cell(a, 0, int(blockIdx.x)).ko, t);
    TileFft<R, S>::forward(v, lds, tw, t);
    C* out = static_cast<C*>(a.spec) + size_t(blockIdx.x) * S::N + t;
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) out[r * S::T] = v[r];
    if constexpr (CHECK)
        if (nonfinite(v[0].x) || nonfinite(v[0].y)) a.flag[0] = 1;
}

// Tiles whose zero-frequency product passes the inverse transform by, in two
// more LDS slots (tile_conv_kernel).
template <typename R, class S> constexpr bool mean_apart() { return sizeof(R) == 8 && S::LH == 0; }

// One kernel spectrum, read from memory.  Long lines of 64-bit samples around a
// mean: every output is the zero-frequency product plus smaller terms, and each
// addition of the inverse transform rounds at the size of the sum.  That product
// skips all passes but the last: 1000003 samples and 1023 taps in [0, 1) come out
// with an error of 1.4e-16 of their norm, 2.2e-16 with it in every pass (whole-array
// passes: 1.8e-16), in the same 12.9 us.  Its slots follow the tile's: in front they
// would push LDS offsets past what an instruction holds (13.1 us).
template <typename R, class S, bool CPLX, bool FILLS>
__global__ void __launch_bounds__(S::T, sizeof(R) == 4 ? 4 : 1) tile_conv_kernel(TileArgs a) {
    using C = Cx<R>;
    using Io = TileIo<R, S, CPLX, FILLS>;
    using F = TileFft<R, S>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x;
    const int q = xcd_item(int(blockIdx.x), a.items);
    const auto tw = F::load_tw(a.tw, t);
    C v[S::PPT];
    const TilePair p = tile_pair<CPLX>(a, q);
    Io::load(v, a, buffer_of(a.x, a.x_bytes), p, t, 0, cmake<C>(R(0), R(0)));
    F::forward(v, lds, tw, t);
    const C* sp = static_cast<const C*>(a.spec) + t;
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) v[r] = cmul(v[r], sp[r * S::T]);
    if constexpr (mean_apart<R, S>()) {
        // bin 0, thread 0's, read behind the inverse's barriers; the others write
        // a word that nobody reads, so that no branch parts product and inverse
        const bool other = t != 0;
        lds[S::N + (other ? 1 : 0)] = v[0];
        v[0].x = other ? v[0].x : R(0);
        v[0].y = other ? v[0].y : R(0);
        F::inverse(v, lds, tw, t, [&](C* u) { u[0] = cadd(u[0], lds[S::N]); });
    } else {
        F::inverse(v, lds, tw, t);
    }
    if (nonfinite(v[0].x) || nonfinite(v[0].y)) a.flag[0] = 1;
    Io::store(v, a, buffer_of(a.y, a.y_bytes), p, t);
}

// Summed over the outer taps: the spectra of the tap's input plane and of its
// kernel slice are multiplied into one accumulator, which is transformed back
// once.
template <typename R, class S, bool CPLX, bool FILLS>
__global__ void __launch_bounds__(S::T) tile_sum_kernel(TileArgs a) {
    using C = Cx<R>;
    using Io = TileIo<R, S, CPLX, FILLS>;
    using F = TileFft<R, S>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x;
    int q;
    const int plane = div_by(a.plane_items, xcd_item(int(blockIdx.x), a.items), &q);
    const TilePair p = tile_pair<CPLX>(a, q);
    const auto tw = F::load_tw(a.tw, t);
    C acc[S::PPT], nx[S::PPT];
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) acc[r] = cmake<C>(R(0), R(0));
    // the next tap from `tap` on whose plane is not all zero
    OuterCell oc;
    auto next = [&](int tap) {
        for (; tap < a.ntaps; ++tap) {
            oc = outer_cell(a, plane, tap);
            if (FILLS || !oc.oc) break;
        }
        return tap;
    };
    auto fetch = [&]() {
        Io::load(nx, a, buffer_of(static_cast<const char*>(a.x) + oc.xo, a.x_bytes - oc.xo), p, t, oc.oc,
                 cmake<C>(R(oc.re), R(oc.im)));
    };
    int tap = next(0);
    if (tap < a.ntaps) fetch();
    bool first = true;
    while (tap < a.ntaps) {
        C v[S::PPT];
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) v[r] = nx[r];
        const C* sp = static_cast<const C*>(a.spec) + size_t(tap) * S::N + t;
        tap = next(tap + 1);
        if (tap < a.ntaps) fetch();
        if (!first) __syncthreads();   // the last transform's reads precede this one's writes
        first = false;
        F::forward(v, lds, tw, t);
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) acc[r] = cadd(acc[r], cmul(v[r], sp[r * S::T]));
    }
    F::inverse(acc, lds, tw, t);
    if (nonfinite(acc[0].x) || nonfinite(acc[0].y)) a.flag[0] = 1;
    int yo = 0, pl = plane;
    for (int i = a.nouter - 1; i >= 0; --i) {
        int pos;
        pl = div_by(a.outer[i].out, pl, &pos);
        yo += pos * a.outer[i].a.ys;
    }
    Io::store(acc, a, buffer_of(static_cast<char*>(a.y) + yo, a.y_bytes - yo), p, t);
}

// The spectra of the kernel's outer taps (unless kept ones are given) and of
// every plane of x, one workgroup each, for tile_acc_kernel.
template <typename R, class S, bool CPLX>
__global__ void __launch_bounds__(S::T) tile_fwd_kernel(TileArgs a) {
    using C = Cx<R>;
    using Io = TileIo<R, S, CPLX, false>;
    using F = TileFft<R, S>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x, nk = a.have_spec ? 0 : a.ntaps;
    uint32_t* flag = a.flag;   // loaded ahead of its use
    asm volatile("" : "+s"(flag));
    const auto tw = F::load_tw(a.tw, t);
    C v[S::PPT];
    C* out;
    if (int(blockIdx.x) < nk) {   // uniform
        Io::load_kernel(v, a, outer_cell(a, 0, int(blockIdx.x)).ko, t);
        out = static_cast<C*>(a.spec) + size_t(blockIdx.x) * S::N + t;
    } else {
        const int item = xcd_item(int(blockIdx.x) - nk, a.xitems);
        int q, xo = 0;
        int plane = div_by(a.plane_items, item, &q);
        for (int i = a.nouter - 1; i >= 0; --i) {
            int cell;
            plane = div_by(a.outer[i].cells, plane, &cell);
            xo += cell * a.outer[i].a.xs + a.outer[i].a.xlo;
        }
        Io::load(v, a, buffer_of(static_cast<const char*>(a.x) + xo, a.x_bytes - xo), tile_pair<CPLX>(a, q), t, 0,
                 cmake<C>(R(0), R(0)));
        out = static_cast<C*>(a.xspec) + size_t(item) * S::N + t;
    }
    F::forward(v, lds, tw, t);
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) out[r * S::T] = v[r];
    if (nonfinite(v[0].x) || nonfinite(v[0].y)) flag[0] = 1;
}

// tile_sum_kernel from kept spectra of x: a tile of x is transformed once and
// not once for every tap and output plane that reads it, and the chain of a
// workgroup is one transform long instead of one per tap.  For fills of zero.
// 10x100x200, 5x11x31 taps: c64 30.6 -> 24.7 us a call, f32 35.3 -> 22.8, f64 43.6 ->
// 28.2; 32x64x64, 9x9x9 taps, f32: 27.4 -> 19.5.
template <typename R, class S, bool CPLX>
__global__ void __launch_bounds__(S::T) tile_acc_kernel(TileArgs a) {
    using C = Cx<R>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x;
    int q;
    const int plane = div_by(a.plane_items, xcd_item(int(blockIdx.x), a.items), &q);
    const auto tw = TileFft<R, S>::load_tw(a.tw, t);
    C acc[S::PPT], nx[S::PPT], nk[S::PPT];
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) acc[r] = cmake<C>(R(0), R(0));
    // loads the next tap from `tap` on whose plane is not all zero
    auto fetch = [&](int tap) {
        for (; tap < a.ntaps; ++tap) {
            const OuterCell oc = outer_cell(a, plane, tap);
            if (oc.oc) continue;
            const C* sx = static_cast<const C*>(a.xspec) + (size_t(oc.xp) * a.plane_items.d + q) * S::N + t;
            const C* sk = static_cast<const C*>(a.spec) + size_t(tap) * S::N + t;
#pragma unroll
            for (int r = 0; r < S::PPT; ++r) {
                nx[r] = sx[r * S::T];
                nk[r] = sk[r * S::T];
            }
            break;
        }
        return tap;
    };
    int tap = fetch(0);
    while (tap < a.ntaps) {
        C v[S::PPT], k[S::PPT];
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) {
            v[r] = nx[r];
            k[r] = nk[r];
        }
        tap = fetch(tap + 1);
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) acc[r] = cadd(acc[r], cmul(v[r], k[r]));
    }
    TileFft<R, S>::inverse(acc, lds, tw, t);
    if (nonfinite(acc[0].x) || nonfinite(acc[0].y)) a.flag[0] = 1;
    int yo = 0, pl = plane;
    for (int i = a.nouter - 1; i >= 0; --i) {
        int pos;
        pl = div_by(a.outer[i].out, pl, &pos);
        yo += pos * a.outer[i].a.ys;
    }
    TileIo<R, S, CPLX, false>::store(acc, a, buffer_of(static_cast<char*>(a.y) + yo, a.y_bytes - yo), tile_pair<CPLX>(a, q), t);
}

// Small inputs in one launch: the workgroup transforms the kernel itself
// (unless a kept spectrum is given) and, when there is more than one, looks
// the whole input over for non-finite values, so that no fix-up launch is
// needed.
template <typename R, class S, bool CPLX, bool FILLS>
__global__ void __launch_bounds__(S::T) tile_one_kernel(TileArgs a) {
    using C = Cx<R>;
    using Io = TileIo<R, S, CPLX, FILLS>;
    using F = TileFft<R, S>;
    extern __shared__ unsigned char smem_raw[];
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int t = threadIdx.x, q = int(blockIdx.x);
    const __amdgpu_buffer_rsrc_t px = buffer_of(a.x, a.x_bytes);
    C v[S::PPT], w[S::PPT];
    if (a.have_spec) {
        const C* sp = static_cast<const C*>(a.spec) + t;
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) w[r] = sp[r * S::T];
    } else {
        Io::load_kernel(w, a, 0, t);
    }
    const TilePair p = tile_pair<CPLX>(a, q);
    Io::load(v, a, px, p, t, 0, cmake<C>(R(0), R(0)));
    const auto tw = F::load_tw(a.tw, t);
    bool bad = false;
    for (int i = t; i < a.scan; i += 8 * S::T) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            bad |= nonfinite(load_real<R>(px, uint32_t(i + u * S::T) * uint32_t(sizeof(R))));
    }
    if (!a.have_spec) {
        F::forward(w, lds, tw, t);
        __syncthreads();
    }
    F::forward(v, lds, tw, t);
#pragma unroll
    for (int r = 0; r < S::PPT; ++r) v[r] = cmul(v[r], w[r]);
    F::inverse(v, lds, tw, t);
    if (__syncthreads_or(bad)) {
        const R nan = R(__builtin_nanf(""));
#pragma unroll
        for (int r = 0; r < S::PPT; ++r) v[r] = cmake<C>(nan, nan);
    }
    Io::store(v, a, buffer_of(a.y, a.y_bytes), p, t);
}

// Whether some output reads cell c of an outer axis inside x.
__device__ __forceinline__ bool cell_read(const TileOuter& o, int c) {
    for (int k = 0; k < o.a.K; ++k) {
        const int q = c + o.a.p0 - k * o.a.d;
        if (q < 0) break;
        if (q % o.a.s == 0 && q / o.a.s < int(o.out.d)) return true;
    }
    return false;
}

// How a wave goes over a plane of x: parts of eight steps of 64 cells, cw columns (a
// power of two) of 64 / cw rows to a step, `steps` steps side by side.
struct ScanParts {
    int planes;              // planes to look at
    int cw, steps;
    TileDiv across;          // parts along a row
    int parts;               // of a plane
    int nspec;               // values of kept spectra
};

// Raises the flag for non-finite values that no tile transforms: in planes of
// x that no outer tap reads, and in kept spectra.  Bound by memory, a read of
// those planes: a call on 17x1612x287 f64 at outer stride 3 (42 MB of unread planes)
// takes 25 us without and 41 with it, small ones 4 to 5 more (in whole-array passes, which
// transform every plane, 639 and 35 to 50).
template <typename R, bool CPLX>
__global__ void __launch_bounds__(256) tile_scan_kernel(TileArgs a, ScanParts p) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    // the waves of a workgroup share a plane, or take one each where it is small
    const bool share = p.parts >= 4;
    const int q0 = share ? int(blockIdx.x) : int(blockIdx.x) * 4 + wave, dq = int(gridDim.x) * (share ? 1 : 4);
    const int i0 = share ? int(blockIdx.y) * 4 + wave : int(blockIdx.y), di = int(gridDim.y) * (share ? 4 : 1);
    const int lr = lane / p.cw, lc = lane & (p.cw - 1), rs = 64 / p.cw;
    bool bad = false;
    for (int q = q0; q < p.planes; q += dq) {
        int plane = q, xo = 0;
        bool read = true;
        for (int e = a.nouter - 1; e >= 0; --e) {
            int cell;
            plane = div_by(a.outer[e].cells, plane, &cell);
            read = read && cell_read(a.outer[e], cell);
            xo += cell * a.outer[e].a.xs + a.outer[e].a.xlo;
        }
        if (read) continue;
        const __amdgpu_buffer_rsrc_t px = buffer_of(static_cast<const char*>(a.x) + xo, a.x_bytes - xo);
        for (int i = i0; i < p.parts; i += di) {
            int pw;
            const int r0 = div_by(p.across, i, &pw) * (8 / p.steps) * rs + lr, c0 = pw * p.steps * 64 + lc;
            Cx<R> v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int r = r0 + u / p.steps * rs, c = c0 + (u & (p.steps - 1)) * 64;
                const uint32_t off = uint32_t(r) * uint32_t(a.ax[0].xs) + uint32_t(a.ax[0].xlo) +
                                     uint32_t(c) * uint32_t(a.ax[1].xs) + uint32_t(a.ax[1].xlo);
                const uint32_t at = r < a.ax[0].n && c < a.ax[1].n ? off : kNoCell;
                if constexpr (CPLX) v[u] = load_cx(px, at, R(0));
                else v[u] = cmake<Cx<R>>(load_real<R>(px, at), R(0));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) bad |= nonfinite(v[u].x) || nonfinite(v[u].y);
        }
    }
    const int block = int(blockIdx.y * gridDim.x + blockIdx.x), blocks = int(gridDim.x * gridDim.y);
    for (int i = block * 256 + int(threadIdx.x); i < p.nspec; i += blocks * 256)
        bad |= nonfinite(static_cast<const R*>(a.spec)[i]);
    if (bad) a.flag[0] = 1;
}

// Fills y with NaN when a tile met a non-finite value, and clears the flag;
// without a flag it fills y in any case.
template <typename R>
__global__ void __launch_bounds__(256) tile_nan_kernel(R* y, int64_t n, uint32_t* flag) {
    if (flag && __builtin_amdgcn_readfirstlane(int(flag[0])) == 0) return;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
        y[i] = R(__builtin_nanf(""));
    if (!flag) return;
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&flag[1], 1u) == gridDim.x - 1) {
        flag[1] = 0;   // every block has read the flag
        flag[0] = 0;
    }
}

template <typename R, class S, bool CPLX, bool FILLS>
ndc_status launch_conv(const TilePlan& p, const TileArgs& a, LaunchContext& ctx) {
    const size_t smem = size_t(S::N) * sizeof(Cx<R>);
    auto go = [&](auto kernel, const char* name, int64_t grid, double bytes, double flops, size_t more = 0) -> ndc_status {
        ctx.kbegin(name, bytes, flops);
        if (!lds_fits(ctx, reinterpret_cast<const void*>(kernel), smem + more)) return NDC_ERR_UNSUPPORTED;
        NDC_LAUNCH(ctx, ctx.stream(), kernel, dim3(unsigned(grid)), dim3(S::T), smem + more, a);
        ctx.kend();
        return NDC_OK;
    };
    const double fft = 5.0 * S::N * S::LN;
    const double io = double(a.x_bytes) + double(a.y_bytes);
    if (p.one) {
        if constexpr (S::LH == 0 && S::LW <= 12)
            return go(tile_one_kernel<R, S, CPLX, FILLS>, "tile_conv_one", a.items, io + double(a.k_bytes),
                      3 * fft * a.items);
        return NDC_ERR_UNSUPPORTED;
    }
    if (a.nouter) {
        if constexpr (S::LH != 0 && S::LP < 4) {
            if constexpr (!FILLS)
                if (a.xspec)
                    return go(tile_acc_kernel<R, S, CPLX>, "tile_conv_sum", a.items,
                              double(p.xspec_bytes) + double(a.y_bytes) + double(p.spec_bytes), fft * a.items);
            return go(tile_sum_kernel<R, S, CPLX, FILLS>, "tile_conv_sum", a.items, io + double(p.spec_bytes),
                      (1.0 + a.ntaps) * fft * a.items);
        }
        return NDC_ERR_UNSUPPORTED;
    }
    if constexpr (sizeof(R) == 8 || !(S::LH == 5 && S::LP == 3))
        return go(tile_conv_kernel<R, S, CPLX, FILLS>, "tile_conv", a.items, io + double(p.spec_bytes),
                  2 * fft * a.items, mean_apart<R, S>() ? 2 * sizeof(Cx<R>) : 0);
    return NDC_ERR_UNSUPPORTED;
}

template <typename R, class S, bool CPLX>
ndc_status launch_shape(const TilePlan& p, const TileArgs& a, int what, LaunchContext& ctx) {
    if (what == 1)
        return p.fills ? launch_conv<R, S, CPLX, true>(p, a, ctx) : launch_conv<R, S, CPLX, false>(p, a, ctx);
    const size_t smem = size_t(S::N) * sizeof(Cx<R>);
    if (what == 3) {
        if constexpr (S::LH != 0 && S::LP < 4) {
            const int blocks = a.xitems + (a.have_spec ? 0 : a.ntaps);
            ctx.kbegin("tile_forward", double(a.x_bytes) + double(p.xspec_bytes), 5.0 * S::N * S::LN * blocks);
            if (!lds_fits(ctx, reinterpret_cast<const void*>(&tile_fwd_kernel<R, S, CPLX>), smem)) return NDC_ERR_UNSUPPORTED;
            NDC_LAUNCH(ctx, ctx.stream(), (tile_fwd_kernel<R, S, CPLX>), dim3(unsigned(blocks)), dim3(S::T), smem, a);
            ctx.kend();
            return NDC_OK;
        }
        return NDC_ERR_UNSUPPORTED;
    }
    ctx.kbegin("tile_spec", double(a.k_bytes) + double(p.spec_bytes), 5.0 * S::N * S::LN * a.ntaps);
    auto go = [&](auto kernel) -> ndc_status {
        if (!lds_fits(ctx, reinterpret_cast<const void*>(kernel), smem)) return NDC_ERR_UNSUPPORTED;
        NDC_LAUNCH(ctx, ctx.stream(), kernel, dim3(unsigned(a.ntaps)), dim3(S::T), smem, a);
        ctx.kend();
        return NDC_OK;
    };
    if constexpr (S::LH != 0 && S::LP < 4)
        if (a.nouter && !a.have_spec) return go(&tile_spec_kernel<R, S, CPLX, true>);
    return go(&tile_spec_kernel<R, S, CPLX, false>);
}

template <typename R, bool CPLX>
ndc_status launch_any(const TilePlan& p, const TileArgs& a, int what, LaunchContext& ctx) {
    switch ((p.lh * 16 + p.lw) * 8 + p.lp) {
        case (0 * 16 + 10) * 8 + 2: return launch_shape<R, Shape<0, 10, 2>, CPLX>(p, a, what, ctx);
        case (0 * 16 + 12) * 8 + 3: return launch_shape<R, Shape<0, 12, 3>, CPLX>(p, a, what, ctx);
        case (5 * 16 + 5) * 8 + 2: return launch_shape<R, Shape<5, 5, 2>, CPLX>(p, a, what, ctx);
        case (6 * 16 + 6) * 8 + 3: return launch_shape<R, Shape<6, 6, 3>, CPLX>(p, a, what, ctx);
        case (5 * 16 + 7) * 8 + 3: return launch_shape<R, Shape<5, 7, 3>, CPLX>(p, a, what, ctx);
        default: break;
    }
    if constexpr (sizeof(R) == 4) {
        switch ((p.lh * 16 + p.lw) * 8 + p.lp) {
            case (0 * 16 + 14) * 8 + 4: return launch_shape<R, Shape<0, 14, 4>, CPLX>(p, a, what, ctx);
            case (5 * 16 + 7) * 8 + 4: return launch_shape<R, Shape<5, 7, 4>, CPLX>(p, a, what, ctx);
            case (6 * 16 + 7) * 8 + 4: return launch_shape<R, Shape<6, 7, 4>, CPLX>(p, a, what, ctx);
            case (7 * 16 + 7) * 8 + 4: return launch_shape<R, Shape<7, 7, 4>, CPLX>(p, a, what, ctx);
            default: break;
        }
    }
    ctx.err = "unknown tile";
    return NDC_ERR_UNSUPPORTED;
}

// Looks over what the plan's tiles leave out: planes of x (not where every
// plane is transformed), kept spectra of taps that no tile uses.
template <typename R, bool CPLX>
ndc_status launch_scan(const TilePlan& p, const TileArgs& a, LaunchContext& ctx) {
    ScanParts s;
    s.planes = p.gaps && !a.xspec ? p.xplanes : 0;
    s.nspec = p.idle && a.have_spec ? int(p.spec_bytes / sizeof(R)) : 0;
    if (!s.planes && !s.nspec) return NDC_OK;
    const int h = a.ax[0].n, w = a.ax[1].n;
    s.cw = 64;
    while (s.cw / 2 >= w) s.cw /= 2;
    s.steps = 1;
    while (s.steps < 8 && s.steps * 64 < w) s.steps *= 2;
    const int rows = 8 / s.steps * (64 / s.cw), cols = s.steps * 64, across = (w + cols - 1) / cols;
    s.across = tile_div(across);
    s.parts = across * ((h + rows - 1) / rows);
    // about 32 workgroups for each of 256 CUs, of which those on planes that are read leave at once
    const bool share = s.parts >= 4;
    const unsigned gx = unsigned(std::max(1, std::min(share ? s.planes : (s.planes + 3) / 4, 16384)));
    const int ny = !s.planes ? std::min(256, (s.nspec + 255) / 256)
                   : std::min(share ? (s.parts + 3) / 4 : s.parts, std::max(1, 8192 / int(gx)));
    ctx.kbegin("tile_scan", 0, 0);
    NDC_LAUNCH(ctx, ctx.stream(), (tile_scan_kernel<R, CPLX>), dim3(gx, unsigned(ny)), dim3(256), 0, a, s);
    ctx.kend();
    return NDC_OK;
}

// what: 0 the kernel spectra, 1 the convolution, 2 the fix-up, 3 the spectra of
// kernel and x, 4 the look over what these leave out
template <typename R>
ndc_status launch_tile_r(const TilePlan& p, const TileArgs& a, bool cplx, int what, LaunchContext& ctx) {
    ndc_status s = NDC_OK;
    if (what == 2) {
        const int64_t n = int64_t(a.y_bytes) / int64_t(sizeof(R));
        const unsigned grid = unsigned(n < 256 * 256 ? (n + 255) / 256 : 256);
        ctx.kbegin("tile_nan", 0, 0);
        NDC_LAUNCH(ctx, ctx.stream(), (tile_nan_kernel<R>), dim3(grid), dim3(256), 0, static_cast<R*>(a.y), n, a.flag);
        ctx.kend();
    } else if (what == 4) {
        s = cplx ? launch_scan<R, true>(p, a, ctx) : launch_scan<R, false>(p, a, ctx);
    } else {
        s = cplx ? launch_any<R, true>(p, a, what, ctx) : launch_any<R, false>(p, a, what, ctx);
    }
    if (s != NDC_OK || ctx.dry_run()) return s;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        ctx.err = std::string("tile launch: ") + hipGetErrorString(e);
        return NDC_ERR_DEVICE;
    }
    return NDC_OK;
}

}  // namespace tilek
}  // namespace ndc
