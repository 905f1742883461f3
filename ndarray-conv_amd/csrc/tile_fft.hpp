// A two-dimensional FFT of one H x W tile held by one workgroup: the points
// sit in registers and meet in LDS only between passes.
//
// The forward transform is decimation in frequency and the inverse
// decimation in time, both in place: every pass reads, transforms and writes
// the same positions, so one LDS buffer serves and a pass needs one barrier.
// The spectrum comes out in a permuted order that both operands of a
// convolution's product share and the inverse undoes, so nothing is ever
// reordered.  A pass transforms 2^ah x 2^aw points per thread (16 or 32 in
// registers); between the forward's last pass and the inverse's first one
// the spectrum never leaves the registers.
//
// Index bits: w bits 0 .. LW-1, h bits LW .. LW+LH-1.  A pass holds the
// index bits it transforms (w digit, then h digit) and, in a pass that
// transforms fewer bits than a thread holds, already transformed high bits as
// its register bits; the remaining bits number the threads.  A pass works on
// one axis where the sizes allow: 64 = 8 x 8 takes one twiddle per point and
// axis, 4 x 4 x 4 two.
//
// Few points per thread, many threads: with 4 to 16 points a workgroup has 4
// to 16 waves to hide its LDS and memory latencies, and the smaller register
// count lets two to four workgroups share a CU.  A 4096x32768 f32 convolution
// (11x31 taps, dilation 2) took 790 us with 32 points a thread (64x256 tiles)
// and 460 us with 16 (64x128); a 5000-sample one 12.0 us with 16 points and
// 6.9 us with 4.
//
// LDS slot of index i: the low kLow bits are XORed with a fixed vector per
// set high bit (swz), the rest is unchanged.  The vectors are chosen so that
// in every pass the first kLow thread bits reach independent bank bits: no
// pass has a bank conflict, with no padding, which leaves 128 KB for 16384
// single-precision points.
#pragma once

#include <type_traits>
#include <utility>

#include "device_common.hpp"
#include "fft_bfly.hpp"

namespace ndc {
namespace tilefft {

constexpr int kMaxPass = 6;

// Compile-time description of a tile: LP = log2 points per thread, the digit
// sizes of each pass (top bits first), and the bank vectors of the index bits
// from kLow up for 8-byte (swz5: 32 slots of 8 bytes) and 16-byte elements
// (swz4: 16 slots).
template <int LH, int LW, int LP> struct Shape;
#define NDC_TILE_SHAPE(LH_, LW_, LP_, NP_, AH, AW, S5, S4)                     \
    template <> struct Shape<LH_, LW_, LP_> {                                      \
        static constexpr int LH = LH_, LW = LW_, LP = LP_, NP = NP_;           \
        static constexpr int ah[kMaxPass] = AH;                               \
        static constexpr int aw[kMaxPass] = AW;                               \
        static constexpr int swz5[16] = S5;                                   \
        static constexpr int swz4[16] = S4;                                   \
        static constexpr int LN = LH_ + LW_, N = 1 << LN, T = 1 << (LN - LP_); \
        static constexpr int PPT = 1 << LP_, LT = LN - LP_;                    \
    };
#define NDC_B(...) {__VA_ARGS__}
NDC_TILE_SHAPE(0, 10, 2, 5, NDC_B(0, 0, 0, 0, 0), NDC_B(2, 2, 2, 2, 2), NDC_B(16, 0, 29, 27, 0),
               NDC_B(7, 0, 14, 14, 0, 0))
NDC_TILE_SHAPE(0, 12, 3, 4, NDC_B(0, 0, 0, 0), NDC_B(3, 3, 3, 3), NDC_B(8, 17, 17, 3, 0, 0, 30),
               NDC_B(9, 1, 0, 0, 15, 0, 2, 0))
NDC_TILE_SHAPE(0, 13, 3, 5, NDC_B(0, 0, 0, 0, 0), NDC_B(3, 3, 2, 2, 3), NDC_B(9, 29, 0, 0, 5, 0, 11, 0),
               NDC_B(2, 0, 8, 0, 0, 4, 0, 1, 0))
NDC_TILE_SHAPE(0, 14, 4, 4, NDC_B(0, 0, 0, 0), NDC_B(4, 4, 4, 2), NDC_B(0, 0, 16, 1, 8, 4, 2, 0, 0),
               NDC_B(0, 0, 0, 8, 1, 8, 2, 4, 0, 2))
NDC_TILE_SHAPE(6, 6, 3, 4, NDC_B(3, 0, 3, 0), NDC_B(0, 3, 0, 3), NDC_B(8, 17, 17, 3, 0, 0, 30),
               NDC_B(9, 1, 0, 0, 15, 0, 2, 0))
NDC_TILE_SHAPE(5, 7, 4, 3, NDC_B(3, 0, 2), NDC_B(1, 4, 2), NDC_B(0, 0, 0, 24, 5, 10, 0),
               NDC_B(0, 0, 11, 1, 0, 11, 11, 6))
NDC_TILE_SHAPE(5, 7, 3, 4, NDC_B(3, 0, 0, 2), NDC_B(0, 3, 3, 1), NDC_B(0, 0, 0, 24, 5, 10, 0),
               NDC_B(0, 11, 0, 0, 0, 12, 9, 0))
NDC_TILE_SHAPE(5, 5, 2, 5, NDC_B(2, 0, 2, 0, 1), NDC_B(0, 2, 0, 2, 1), NDC_B(0, 0, 23, 0, 11),
               NDC_B(8, 0, 0, 15, 0, 4))
NDC_TILE_SHAPE(7, 7, 4, 4, NDC_B(4, 0, 3, 0), NDC_B(0, 4, 0, 3), NDC_B(0, 0, 2, 8, 16, 0, 4, 1, 0),
               NDC_B(0, 0, 0, 0, 2, 8, 0, 4, 1, 0))
NDC_TILE_SHAPE(6, 7, 4, 4, NDC_B(3, 0, 3, 0), NDC_B(1, 4, 0, 2), NDC_B(28, 12, 0, 6, 15, 18, 0, 0),
               NDC_B(0, 0, 1, 0, 2, 8, 4, 0, 0))
#undef NDC_B
#undef NDC_TILE_SHAPE

// Register and thread bits of every pass, and where the passes' twiddles sit
// in the tile's table.  The thread bits' first kLow are chosen to be
// independent in the bank vectors, taking the lowest index bits first (pass 0
// keeps ascending order, so its global accesses run along w).
template <class S, int kLow>
struct Map {
    int reg[kMaxPass][5] = {};
    int thr[kMaxPass][12] = {};
    int wlow[kMaxPass] = {};    // w bits below the digit: their count
    int hlow[kMaxPass] = {};
    int tww[kMaxPass] = {};     // table offset of the w twiddles W_(2^aw M)^(k m) at (k - 1) M + m, M = 2^wlow
    int twh[kMaxPass] = {};
    int ntw = 0;
    int regw[kMaxPass] = {};    // where a thread keeps its own w and h twiddles (k = 1 ..) of the pass
    int regh[kMaxPass] = {};
    int nreg = 0;

    static constexpr int vec(int bit) {
        return bit < kLow ? 1 << bit : (kLow == 5 ? S::swz5[bit - kLow] : S::swz4[bit - kLow]);
    }
    constexpr Map() {
        int wt = S::LW, ht = S::LW + S::LH;
        for (int p = 0; p < S::NP; ++p) {
            int n = 0;
            bool used[20] = {};
            for (int b = wt - S::aw[p]; b < wt; ++b) { reg[p][n++] = b; used[b] = true; }
            for (int b = ht - S::ah[p]; b < ht; ++b) { reg[p][n++] = b; used[b] = true; }
            for (int b = S::LN - 1; b >= 0 && n < S::LP; --b)
                if (!used[b] && (b >= ht || (b < S::LW && b >= wt))) { reg[p][n++] = b; used[b] = true; }
            // greedy independent set over the bank vectors, then the rest
            int basis[5] = {}, nt = 0;
            bool taken[20] = {};
            for (int pass = 0; pass < 2; ++pass)
                for (int b = 0; b < S::LN; ++b) {
                    if (used[b] || taken[b]) continue;
                    if (pass == 0) {
                        int v = vec(b);
                        for (int i = 0; i < kLow; ++i)
                            if ((v >> i & 1) && basis[i]) v ^= basis[i];
                        if (!v) continue;
                        int i = 0;
                        while (!(v >> i & 1)) ++i;
                        basis[i] = v;
                        // keep the basis reduced from the low end
                        for (int j = 0; j < kLow; ++j)
                            if (j != i && basis[j] && (basis[j] >> i & 1)) basis[j] ^= v;
                    }
                    taken[b] = true;
                    thr[p][nt++] = b;
                }
            wlow[p] = wt - S::aw[p];
            hlow[p] = ht - S::ah[p] - S::LW;
            tww[p] = ntw;
            regw[p] = nreg;
            if (wlow[p] > 0) { ntw += ((1 << S::aw[p]) - 1) << wlow[p]; nreg += (1 << S::aw[p]) - 1; }
            twh[p] = ntw;
            regh[p] = nreg;
            if (hlow[p] > 0) { ntw += ((1 << S::ah[p]) - 1) << hlow[p]; nreg += (1 << S::ah[p]) - 1; }
            wt -= S::aw[p];
            ht -= S::ah[p];
        }
    }
    // the bank-swizzled slot of an index made of one set bit
    constexpr int slot(int bit) const { return bit < kLow ? 1 << bit : (1 << bit) | vec(bit); }
    // XOR part (low bits) and plain part (high bits) of register r's offset in pass p
    constexpr int reg_off(int p, int r) const {
        int v = 0;
        for (int j = 0; j < S::LP; ++j)
            if (r >> j & 1) v ^= slot(reg[p][j]);
        return v;
    }
    // all thread bits independent in the banks: kLow of them in every pass
    constexpr bool conflict_free() const {
        for (int p = 0; p < S::NP; ++p) {
            int basis[5] = {}, rank = 0;
            for (int j = 0; j < kLow && j < S::LT; ++j) {
                int v = vec(thr[p][j]);
                for (int i = 0; i < kLow; ++i)
                    if (v >> i & 1) {
                        if (basis[i]) v ^= basis[i];
                        else { basis[i] = v; ++rank; break; }
                    }
            }
            if (rank < kLow) return false;
        }
        return true;
    }
};

template <typename R> struct LowOf;
template <> struct LowOf<float> { static constexpr int v = 5; };
template <> struct LowOf<double> { static constexpr int v = 4; };

#ifdef __HIPCC__

// f(integral_constant<int, 0>), .. f(integral_constant<int, N - 1>)
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

template <typename R, class S>
struct TileFft {
    using C = Cx<R>;
    static constexpr int kLow = LowOf<R>::v;
    static constexpr Map<S, kLow> M{};
    static_assert(M.conflict_free(), "bank vectors of the tile shape");
    static constexpr int kLowMask = (1 << kLow) - 1;

    // The bits of `t` that pass P's thread bits of index [B0, B0 + NB) take,
    // moved to their index positions less B0: one shift and mask per run of
    // consecutive bits.
    template <int P, int B0, int NB, int J = 0>
    static __device__ __forceinline__ int thr_value(int t) {
        if constexpr (J >= S::LT) {
            return 0;
        } else {
            constexpr int b = M.thr[P][J];
            if constexpr (b < B0 || b >= B0 + NB) {
                return thr_value<P, B0, NB, J + 1>(t);
            } else {
                constexpr int n = run_of(P, J, B0 + NB);
                constexpr int mask = ((1 << n) - 1) << J, sh = b - B0 - J;
                const int v = J + n == S::LT && J == 0 ? t : (t & mask);
                return (sh >= 0 ? v << (sh & 31) : v >> (-sh & 31)) | thr_value<P, B0, NB, J + n>(t);
            }
        }
    }
    // consecutive index bits, below `end`, from thread bit j on
    static constexpr int run_of(int p, int j, int end) {
        int n = 1;
        while (j + n < S::LT && M.thr[p][j + n] == M.thr[p][j] + n && M.thr[p][j + n] < end) ++n;
        return n;
    }
    // LDS slot part of thread t in pass P
    template <int P>
    static __device__ __forceinline__ int thr_slot(int t) {
        int a = thr_value<P, 0, S::LN>(t);
        static_for<S::LT>([&](auto j) {
            constexpr int b = M.thr[P][j()];
            if constexpr (b >= kLow && M.vec(b) != 0) a ^= -((t >> j()) & 1) & M.vec(b);
        });
        return a;
    }

    template <int P>
    static __device__ __forceinline__ void lds_read(C* v, const C* lds, int base) {
        static_for<S::PPT>([&](auto r) {
            constexpr int o = M.reg_off(P, r());
            v[r()] = lds[(base ^ (o & kLowMask)) + (o & ~kLowMask)];
        });
    }
    template <int P>
    static __device__ __forceinline__ void lds_write(const C* v, C* lds, int base) {
        static_for<S::PPT>([&](auto r) {
            constexpr int o = M.reg_off(P, r());
            lds[(base ^ (o & kLowMask)) + (o & ~kLowMask)] = v[r()];
        });
    }

    // The pass's in-register transforms: 2^aw points along w, 2^ah along h.
    template <int P>
    static __device__ __forceinline__ void bfly_pass(C* v, bool inv) {
        constexpr int PW = 1 << S::aw[P], PH = 1 << S::ah[P], B = S::PPT / (PW * PH);
#pragma unroll
        for (int e = 0; e < B; ++e) {
            C* b = v + e * PW * PH;
            if constexpr (PW > 1) {
#pragma unroll
                for (int h = 0; h < PH; ++h) fftb::bfly<PW>(b + h * PW, inv);
            }
            if constexpr (PH > 1) {
#pragma unroll
                for (int w = 0; w < PW; ++w) {
                    C t[PH];
#pragma unroll
                    for (int h = 0; h < PH; ++h) t[h] = b[h * PW + w];
                    fftb::bfly<PH>(t, inv);
#pragma unroll
                    for (int h = 0; h < PH; ++h) b[h * PW + w] = t[h];
                }
            }
        }
    }

    // A thread's twiddles.  Up to 64 registers of them are loaded once at the
    // kernel's start, where their latency hides behind the data's; longer
    // sets (radix-16 passes in double precision) are read where they are used.
    static constexpr bool kKeep = M.nreg * int(sizeof(C)) <= 64 * 4;
    struct Tw {
        C r[kKeep ? (M.nreg > 0 ? M.nreg : 1) : 1];
        const C* tab;
        int t;
    };
    template <int P, bool H, int K>
    static __device__ __forceinline__ C tw_entry(const C* __restrict__ tab, int t) {
        constexpr int low = H ? M.hlow[P] : M.wlow[P];
        constexpr int off = (H ? M.twh[P] : M.tww[P]) + ((K - 1) << low);
        return tab[off + thr_value<P, H ? S::LW : 0, low>(t)];
    }
    template <int P, bool H, int K>
    static __device__ __forceinline__ C tw_of(const Tw& w) {
        if constexpr (kKeep) {
            return w.r[(H ? M.regh[P] : M.regw[P]) + K - 1];
        } else {
            int t = w.t;
            asm volatile("" : "+v"(t));   // read here, not kept across a loop over tiles
            return tw_entry<P, H, K>(w.tab, t);
        }
    }
    static __device__ __forceinline__ Tw load_tw(const void* tab, int t) {
        Tw w;
        w.tab = static_cast<const C*>(tab);
        w.t = t;
        if constexpr (kKeep) {
            static_for<S::NP>([&](auto p) {
                constexpr int P = p();
                if constexpr (M.wlow[P] > 0)
                    static_for<(1 << S::aw[P]) - 1>([&](auto k) {
                        w.r[M.regw[P] + k()] = tw_entry<P, false, k() + 1>(w.tab, t);
                    });
                if constexpr (M.hlow[P] > 0)
                    static_for<(1 << S::ah[P]) - 1>([&](auto k) {
                        w.r[M.regh[P] + k()] = tw_entry<P, true, k() + 1>(w.tab, t);
                    });
            });
        }
        return w;
    }

    // Multiplies by the pass's twiddles (or their conjugates).
    template <int P>
    static __device__ __forceinline__ void twiddle(C* v, const Tw& w, bool conj) {
        constexpr int PW = 1 << S::aw[P], PH = 1 << S::ah[P], B = S::PPT / (PW * PH);
        if constexpr (M.wlow[P] > 0)
            static_for<PW - 1>([&](auto kk) {
                constexpr int k = kk() + 1;
                const C f = tw_of<P, false, k>(w);
#pragma unroll
                for (int i = 0; i < B * PH; ++i) v[i * PW + k] = cmulc(v[i * PW + k], f, conj);
            });
        if constexpr (M.hlow[P] > 0)
            static_for<PH - 1>([&](auto kk) {
                constexpr int k = kk() + 1;
                const C f = tw_of<P, true, k>(w);
#pragma unroll
                for (int e = 0; e < B; ++e)
#pragma unroll
                    for (int i = 0; i < PW; ++i) {
                        C& u = v[(e * PH + k) * PW + i];
                        u = cmulc(u, f, conj);
                    }
            });
    }

    // Forward transform: v holds pass 0's points, and the last pass's on return.
    template <int P = 0>
    static __device__ __forceinline__ void forward(C* v, C* lds, const Tw& tw, int t) {
        bfly_pass<P>(v, false);
        if constexpr (P + 1 < S::NP) {
            twiddle<P>(v, tw, false);
            lds_write<P>(v, lds, thr_slot<P>(t));
            __syncthreads();
            lds_read<P + 1>(v, lds, thr_slot<P + 1>(t));
            forward<P + 1>(v, lds, tw, t);
        }
    }
    // Unnormalised inverse: v holds the last pass's points, and pass 0's on
    // return.  The last pass's points are written where they were read, so no
    // barrier precedes the first write.  before_first(v) sees pass 0's points
    // ahead of its transforms: point 0 of each thread is the group of bin 0.
    struct None {
        __device__ __forceinline__ void operator()(C*) const {}
    };
    template <int P = S::NP - 1, class First = None>
    static __device__ __forceinline__ void inverse(C* v, C* lds, const Tw& tw, int t, First before_first = First{}) {
        if constexpr (P == 0) before_first(v);
        bfly_pass<P>(v, true);
        if constexpr (P > 0) {
            lds_write<P>(v, lds, thr_slot<P>(t));
            __syncthreads();
            lds_read<P - 1>(v, lds, thr_slot<P - 1>(t));
            twiddle<P - 1>(v, tw, true);
            inverse<P - 1>(v, lds, tw, t, before_first);
        }
    }
};

#endif  // __HIPCC__

}  // namespace tilefft
}  // namespace ndc
