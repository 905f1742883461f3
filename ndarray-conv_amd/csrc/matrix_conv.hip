// Direct 2-D convolution on the matrix cores with accumulators that stay in
// place: exact FP32 (v_mfma_f32_4x4x1, one rounding per product and sum), BF16
// and split BF16x3 (v_mfma_f32_16x16x32_bf16), and wrapping integers of 8 to 32
// bits (v_mfma_i32_16x16x64_i8 on the bytes).  Same sum as conv/mod.rs:177-197.
//
// One output row segment of 256 values is a matrix product over one kernel
// row: y[N m + n] = sum_j X[N m + j] T[j][n], T[j][n] = k[j - n].  The data
// operand is read from the staged row as it lies (m rows of N columns apart);
// the tap operand is the Toeplitz band.  N = 16 for the 16x16 instructions; N =
// 4 for FP32, whose 4x4 instruction multiplies 64 rows by 4 columns at full
// rate, so that only 3 of K + 3 products of the band are zeros (15 of K + 15
// with N = 16).
//
// A workgroup of NW waves makes NW R output rows of 256 columns: it stages
// their whole input region once, split into planes (hi / lo, or bytes), and
// takes the kernel rows in groups of G whose tap operands sit in registers;
// each staged row read from LDS then meets all G kernel rows.
//
// A stride equal to the dilation reads a decimated input with the plain
// kernel; stride 1 and dilation d make d such problems, one per phase.
//
// Measured (before: the vector kernel of direct_conv.hip, the systolic one of
// mfma_conv.hip): 4096x4096 f32, 31x31 taps, stride and dilation 2: FP32 180 ->
// 87 us, BF16x3 69 -> 43, BF16 63 -> 25; 200x5000 i32, 11x31 taps 36.8 -> 14;
// 512x512, 7x7 taps: f32 22 -> 8, i32 21 -> 10.6, i16 17 -> 7.7.
// Bound: FP32 by the matrix pipe (34 x 32 products for 31 x 31, 4.1 ns an
// instruction and SIMD, 70 of the 87 us); BF16 and integers by staging (17 us
// of the 43), which one workgroup per CU does not overlap with its products.
// Two accumulators in turn left the 4x4 instruction waiting (G = 2: 110 us);
// reading a row's operands a row ahead took BF16x3 from 61 to 48 us, four
// staged rows in flight instead of eight from 48 to 46 (twelve: 61).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>

#include "bf16_split.hpp"
#include "device_common.hpp"
#include "matrix_conv.hpp"
#include "tile_kernels.hpp"

namespace ndc {
namespace {

using tilek::buffer_of;
using tilek::cell_kind;
using tilek::cell_offset;
using tilek::div_by;
using tilek::kNoCell;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileX = 256;
// LDS for the staged region, the taps and two groups of tap operands.
constexpr size_t kLdsMax = 156 * 1024;

struct MatArgs {
    const void* x;       // the lowest element the view touches
    const void* k;
    void* y;
    int32_t x_bytes, k_bytes, y_bytes;
    TileAxis ax[2];      // rows, columns; V outputs per tile and phase, U outputs, s = 1: step d per output
    int32_t os[2];       // output step of neighbouring tile positions: the dilation, or 1 when strided
    int32_t KWp;         // tap row pitch in LDS
    int32_t NR;          // staged rows
    int32_t fills;       // some fill writes a constant other than zero
    float cst[2][2];
    int32_t icst[2][2];
};

enum Kind { kF32 = 0, kBf16 = 1, kBf16x3 = 2, kI32 = 3, kI16 = 4, kI8 = 5 };

template <int KIND> struct KindOf;
template <> struct KindOf<kF32> { using E = float; static constexpr int PL = 1, ESZ = 4, ACC = 1, G = 4, N = 4, STEP = 2; };
template <> struct KindOf<kBf16> { using E = float; static constexpr int PL = 1, ESZ = 2, ACC = 1, G = 4, N = 16, STEP = 32; };
template <> struct KindOf<kBf16x3> { using E = float; static constexpr int PL = 2, ESZ = 2, ACC = 1, G = 4, N = 16, STEP = 32; };
template <> struct KindOf<kI32> { using E = int32_t; static constexpr int PL = 4, ESZ = 1, ACC = 4, G = 4, N = 16, STEP = 64; };
template <> struct KindOf<kI16> { using E = int16_t; static constexpr int PL = 2, ESZ = 1, ACC = 2, G = 4, N = 16, STEP = 64; };
template <> struct KindOf<kI8> { using E = int8_t; static constexpr int PL = 1, ESZ = 1, ACC = 1, G = 4, N = 16, STEP = 64; };

// Staged columns: the last row's window of KB operand blocks ends here (rows
// start 16 bytes aligned).
constexpr int staged_width(int n, int step, int kb) { return kTileX - n + (step * kb + 3) / 4 * 4; }

template <typename E> __device__ __forceinline__ uint32_t load_bits(__amdgpu_buffer_rsrc_t b, uint32_t off) {
    if constexpr (sizeof(E) == 4) return uint32_t(__builtin_amdgcn_raw_buffer_load_b32(b, int(off), 0, 0));
    else if constexpr (sizeof(E) == 2) return uint32_t(uint16_t(__builtin_amdgcn_raw_buffer_load_b16(b, int(off), 0, 0)));
    else return uint32_t(uint8_t(__builtin_amdgcn_raw_buffer_load_b8(b, int(off), 0, 0)));
}
template <typename E> __device__ __forceinline__ void store_bits(__amdgpu_buffer_rsrc_t b, uint32_t off, uint32_t v) {
    if constexpr (sizeof(E) == 4) __builtin_amdgcn_raw_buffer_store_b32(v, b, int(off), 0, 0);
    else if constexpr (sizeof(E) == 2) __builtin_amdgcn_raw_buffer_store_b16(uint16_t(v), b, int(off), 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b8(uint8_t(v), b, int(off), 0, 0);
}

// The planes of a value: bf16 terms, or balanced base-256 digits (v = sum d_a
// 256^a with -128 <= d_a < 128, modulo the type's range): adding 128 to every
// byte and flipping its top bit carries what a digit above 127 owes the next.
template <int KIND>
__device__ __forceinline__ uint32_t split_value(uint32_t bits) {
    if constexpr (KIND == kBf16) return bf16_bits(__builtin_bit_cast(float, bits));
    else if constexpr (KIND == kBf16x3) return split_pack(__builtin_bit_cast(float, bits));
    else if constexpr (KIND == kI32) return (bits + 0x80808080u) ^ 0x80808080u;
    else if constexpr (KIND == kI16) return (bits + 0x8080u) ^ 0x8080u;
    else return bits;
}

template <int KIND>
__device__ __forceinline__ bool not_finite(uint32_t bits) {
    const float v = __builtin_fabsf(__builtin_bit_cast(float, bits));
    if constexpr (KIND == kF32) return !(v < __builtin_inff());
    else return !(v <= 3.38e38f);   // its bf16 rounding would overflow
}

// NW waves of R output rows each.  KB: operand blocks along a kernel row (N - 1
// + K columns in blocks of STEP).
template <int KIND, int NW, int R, int KB>
__global__ void __launch_bounds__(64 * NW) matrix_conv_kernel(MatArgs a) {
    constexpr int kWaves = NW, kThreads = 64 * NW;
    using T = KindOf<KIND>;
    using E = typename T::E;
    constexpr int G = KIND == kF32 && KB > 17 ? 2 : T::G, PL = T::PL, W = staged_width(T::N, T::STEP, KB);
    constexpr bool kFloat = KIND <= kBf16x3;
    constexpr int NC = (W + 63) / 64;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int32_t s_bad[NW];   // by wave: it staged a non-finite value
    unsigned char* region = smem;                              // [plane][row][W]
    const int plane = a.NR * W * T::ESZ;
    uint32_t* taps = reinterpret_cast<uint32_t*>(smem + PL * plane);   // [KH][KWp], element bits
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int KH = a.ax[0].K, KW = a.ax[1].K;
    // tap operands, 16 bytes a lane: [2][G][KB][PL][64] (matrix kinds);
    // FP32: [KH][4 shifts][4 KB] copies of the taps, all at once
    unsigned char* frags = reinterpret_cast<unsigned char*>(taps + ((KH * a.KWp + 3) & ~3));

    int bid = int(blockIdx.x), tx, fx, fy;
    bid = div_by(a.ax[1].tiles, bid, &tx);
    bid = div_by(a.ax[1].phases, bid, &fx);
    const int ty = div_by(a.ax[0].phases, bid, &fy);
    const int y0 = ty * NW * R, x0 = tx * kTileX;               // first output of the phase
    const int py0 = a.ax[0].d * y0 + fy, px0 = a.ax[1].d * x0 + fx;

    const __amdgpu_buffer_rsrc_t px = buffer_of(a.x, a.x_bytes);
    // ---- the region: a wave stages every fourth row, a lane every 64th column
    uint32_t co[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int c = lane + 64 * i;
        co[i] = c < W ? cell_offset(a.ax[1], px0 + a.ax[1].d * c) : kNoCell;
    }
    bool bad = false;
    constexpr int kRows = 4;   // rows in flight
    for (int r0 = wave; r0 < a.NR; r0 += kWaves * kRows) {
        uint32_t v[kRows][NC];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const int r = r0 + kWaves * u;
            const uint32_t ro = r < a.NR ? cell_offset(a.ax[0], py0 + a.ax[0].d * r) : kNoCell;
#pragma unroll
            for (int i = 0; i < NC; ++i) v[u][i] = load_bits<E>(px, ro + co[i]);
        }
        if (a.fills) {
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                const int kr = cell_kind(a.ax[0], py0 + a.ax[0].d * (r0 + kWaves * u));
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    const int kc = cell_kind(a.ax[1], px0 + a.ax[1].d * (lane + 64 * i));
                    if ((kr | kc) == 0 || kr == 3 || kc == 3) continue;
                    // the higher axis's constant wins
                    const float f = kc == 1 ? a.cst[1][0] : kc == 2 ? a.cst[1][1] : kr == 1 ? a.cst[0][0] : a.cst[0][1];
                    const int32_t n = kc == 1 ? a.icst[1][0] : kc == 2 ? a.icst[1][1] : kr == 1 ? a.icst[0][0] : a.icst[0][1];
                    v[u][i] = kFloat ? __builtin_bit_cast(uint32_t, f) : uint32_t(n);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const int r = r0 + kWaves * u;
            if (r >= a.NR) break;
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int c = lane + 64 * i;
                if (64 * i + 63 >= W && c >= W) continue;
                if (kFloat) bad |= not_finite<KIND>(v[u][i]);
                const uint32_t s = split_value<KIND>(v[u][i]);
                if constexpr (T::ESZ == 4) reinterpret_cast<uint32_t*>(region)[r * W + c] = s;
                else if constexpr (T::ESZ == 2) {
                    uint16_t* h = reinterpret_cast<uint16_t*>(region);
                    h[r * W + c] = uint16_t(s);
                    if constexpr (PL == 2) h[a.NR * W + r * W + c] = uint16_t(s >> 16);
                } else {
#pragma unroll
                    for (int q = 0; q < PL; ++q) region[q * plane + r * W + c] = uint8_t(s >> (8 * q));
                }
            }
        }
    }
    // ---- the taps, in the order the outputs meet them
    const __amdgpu_buffer_rsrc_t pk = buffer_of(a.k, a.k_bytes);
    for (int i = t; i < KH * a.KWp; i += kThreads) {
        const int r = i / a.KWp, c = i - r * a.KWp;
        uint32_t v = 0;
        if (c < KW)
            v = load_bits<E>(pk, uint32_t((KH - 1 - r) * a.ax[0].ks + a.ax[0].klo + (KW - 1 - c) * a.ax[1].ks + a.ax[1].klo));
        if (kFloat) bad |= not_finite<KIND>(v);
        taps[i] = v;
    }
    // every wave writes its own word, so the words need no clearing before
    if constexpr (kFloat) {
        const bool any = __ballot(bad) != 0;
        if (lane == 0) s_bad[wave] = any;
    }
    __syncthreads();

    // A non-finite value makes a matrix product non-finite even where the
    // reference's sum skips it (zero taps, the band's zeros).  Such workgroups
    // compute their outputs as the reference does, and only so: FP32, the view's
    // taps in row-major order, zero taps skipped, separate multiply and add
    // (conv/mod.rs:177-197, dilation/mod.rs:34-60).
    if constexpr (kFloat) {
        int exact = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) exact |= s_bad[w];
        if (__builtin_amdgcn_readfirstlane(exact)) {
            const __amdgpu_buffer_rsrc_t py = buffer_of(a.y, a.y_bytes);
            for (int e = t; e < NW * R * kTileX; e += kThreads) {
                const int yo = a.os[0] * (y0 + e / kTileX) + fy, xo = a.os[1] * (x0 + e % kTileX) + fx;
                if (yo >= a.ax[0].U || xo >= a.ax[1].U) continue;
                const int py_ = py0 + a.ax[0].d * (e / kTileX), px_ = px0 + a.ax[1].d * (e % kTileX);
                float sum = 0.0f;
                for (int r = 0; r < KH; ++r) {
                    const int pr = py_ + a.ax[0].d * r;
                    for (int c = 0; c < KW; ++c) {
                        const float kv = __builtin_bit_cast(float, taps[r * a.KWp + c]);
                        if (kv == 0.0f) continue;
                        const int pc = px_ + a.ax[1].d * c;
                        float v = __builtin_bit_cast(float, load_bits<float>(px, cell_offset(a.ax[0], pr) + cell_offset(a.ax[1], pc)));
                        const int kr = cell_kind(a.ax[0], pr), kc = cell_kind(a.ax[1], pc);
                        if (kc) v = a.cst[1][kc - 1];
                        else if (kr) v = a.cst[0][kr - 1];
                        sum = __fadd_rn(sum, __fmul_rn(v, kv));
                    }
                }
                store_bits<float>(py, uint32_t(yo) * uint32_t(a.ax[0].ys) + uint32_t(xo) * uint32_t(a.ax[1].ys),
                                  __builtin_bit_cast(uint32_t, sum));
            }
            return;
        }
    }

    if constexpr (KIND == kF32) {
        // copy j of a kernel row holds k[c - j] at c, so a lane of column j
        // reads four consecutive band entries as one aligned word of 16 bytes
        constexpr int TQ = (KB + 1) / 2, TW = 4 * TQ;
        float* cp = reinterpret_cast<float*>(frags);
        for (int i = t; i < KH * 4 * TW; i += kThreads) {
            const int r = i / (4 * TW), j = (i / TW) & 3, c = i % TW - j;
            cp[i] = c >= 0 && c < KW ? __builtin_bit_cast(float, taps[r * a.KWp + c]) : 0.0f;
        }
        __syncthreads();
        f32x4 acc[R];
#pragma unroll
        for (int y = 0; y < R; ++y) acc[y] = f32x4{0, 0, 0, 0};
        const float* reg = reinterpret_cast<const float*>(region) + wave * R * W + 4 * lane;
        const float* cpl = cp + (lane & 3) * TW;
        for (int g = 0; g < KH; g += G) {
            f32x4 b[G][TQ];
#pragma unroll
            for (int r = 0; r < G; ++r)
#pragma unroll
                for (int q = 0; q < TQ; ++q)
                    b[r][q] = g + r < KH ? reinterpret_cast<const f32x4*>(cpl + (g + r) * 4 * TW)[q] : f32x4{0, 0, 0, 0};
            // the row past the region's last (a group beyond KH) meets zero taps only
            auto fetch = [&](f32x4* w, int p) {
                const f32x4* row = reinterpret_cast<const f32x4*>(reg + min(g + p, a.NR - 1 - wave * R) * W);
#pragma unroll
                for (int q = 0; q < TQ; ++q) w[q] = row[q];
            };
            f32x4 ww[2][TQ];
            fetch(ww[0], 0);
#pragma unroll
            for (int p = 0; p < R + G - 1; ++p) {
                // the next row's reads run during this row's products
                f32x4* w = ww[p & 1];
                if (p + 1 < R + G - 1) fetch(ww[(p + 1) & 1], p + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < TQ; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int r = 0; r < G; ++r)
                            if (4 * q + e < 2 * KB && p - r >= 0 && p - r < R)
                                acc[p - r] = __builtin_amdgcn_mfma_f32_4x4x1f32(w[q][e], b[r][q][e], acc[p - r], 0, 0, 0);
            }
        }
        const __amdgpu_buffer_rsrc_t py = buffer_of(a.y, a.y_bytes);
        uint32_t yc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int x = x0 + 16 * (lane >> 2) + 4 * i + (lane & 3), o = a.os[1] * x + fx;
            yc[i] = o < a.ax[1].U ? uint32_t(o) * uint32_t(a.ax[1].ys) : kNoCell;
        }
#pragma unroll
        for (int y = 0; y < R; ++y) {
            const int o = a.os[0] * (y0 + wave * R + y) + fy;
            const uint32_t yr = o < a.ax[0].U ? uint32_t(o) * uint32_t(a.ax[0].ys) : kNoCell;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float f = acc[y][i];
                store_bits<E>(py, yr + yc[i], __builtin_bit_cast(uint32_t, f));
            }
        }
    } else {
        constexpr int kFrag = G * KB * PL * 1024;   // bytes of one group's operands
        const int n = lane & 15, kg = lane >> 4;
        constexpr int kEl = 16 / T::ESZ;            // elements of an operand a lane holds
        auto build = [&](int g, int buf) {
            for (int i = wave; i < G * KB; i += kWaves) {
                const int r = g + i / KB, kb = i % KB;
                uint32_t w[PL][4] = {};
                const int c0 = T::STEP * kb + kEl * kg - n;
#pragma unroll
                for (int e = 0; e < kEl; ++e) {
                    const int c = c0 + e;
                    const uint32_t s = r < KH && c >= 0 && c < KW ? split_value<KIND>(taps[r * a.KWp + c]) : 0u;
#pragma unroll
                    for (int q = 0; q < PL; ++q) {
                        if constexpr (T::ESZ == 2) w[q][e / 2] |= ((s >> (16 * q)) & 0xffffu) << (16 * (e & 1));
                        else w[q][e / 4] |= ((s >> (8 * q)) & 0xffu) << (8 * (e & 3));
                    }
                }
#pragma unroll
                for (int q = 0; q < PL; ++q)
                    reinterpret_cast<u32x4*>(frags + buf * kFrag)[(i * PL + q) * 64 + lane] =
                        u32x4{w[q][0], w[q][1], w[q][2], w[q][3]};
            }
        };
        i32x4 acc[R][T::ACC];
#pragma unroll
        for (int y = 0; y < R; ++y)
#pragma unroll
            for (int q = 0; q < T::ACC; ++q) acc[y][q] = i32x4{0, 0, 0, 0};
        // operand m of a row: 16 columns apart, kEl elements from 16 kg... on
        const unsigned char* reg = region + (wave * R * W + 16 * n + kEl * kg) * T::ESZ;
        build(0, 0);
        for (int g = 0, buf = 0; g < KH; g += G, buf ^= 1) {
            __syncthreads();
            u32x4 b[G][KB][PL];
#pragma unroll
            for (int r = 0; r < G; ++r)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int q = 0; q < PL; ++q)
                        b[r][kb][q] = reinterpret_cast<const u32x4*>(frags + buf * kFrag)[((r * KB + kb) * PL + q) * 64 + lane];
            if (g + G < KH) build(g + G, buf ^ 1);
            auto fetch = [&](u32x4 (*w)[PL], int p) {
                const unsigned char* row = reg + min(g + p, a.NR - 1 - wave * R) * W * T::ESZ;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int q = 0; q < PL; ++q)
                        w[kb][q] = *reinterpret_cast<const u32x4*>(row + q * plane + T::STEP * kb * T::ESZ);
            };
            u32x4 ww[2][KB][PL];
            fetch(ww[0], 0);
#pragma unroll
            for (int p = 0; p < R + G - 1; ++p) {
                u32x4 (*w)[PL] = ww[p & 1];
                if (p + 1 < R + G - 1) fetch(ww[(p + 1) & 1], p + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int qa = 0; qa < PL; ++qa)
#pragma unroll
                        for (int qb = 0; qb < (KIND == kBf16x3 ? PL - qa : KIND == kBf16 ? 1 : T::ACC - qa); ++qb)
#pragma unroll
                            for (int r = 0; r < G; ++r) {
                                if (p - r < 0 || p - r >= R) continue;
                                i32x4& c = acc[p - r][kFloat ? 0 : qa + qb];
                                if constexpr (kFloat)
                                    c = __builtin_bit_cast(i32x4, __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                            __builtin_bit_cast(bf16x8, w[kb][qa]), __builtin_bit_cast(bf16x8, b[r][kb][qb]),
                                            __builtin_bit_cast(f32x4, c), 0, 0, 0));
                                else
                                    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, w[kb][qa]),
                                                                              __builtin_bit_cast(i32x4, b[r][kb][qb]), c, 0, 0, 0);
                            }
            }
        }
        const __amdgpu_buffer_rsrc_t py = buffer_of(a.y, a.y_bytes);
        uint32_t yc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int x = x0 + 16 * (4 * kg + i) + n, o = a.os[1] * x + fx;
            yc[i] = o < a.ax[1].U ? uint32_t(o) * uint32_t(a.ax[1].ys) : kNoCell;
        }
#pragma unroll
        for (int y = 0; y < R; ++y) {
            const int o = a.os[0] * (y0 + wave * R + y) + fy;
            const uint32_t yr = o < a.ax[0].U ? uint32_t(o) * uint32_t(a.ax[0].ys) : kNoCell;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t v = 0;
#pragma unroll
                for (int q = 0; q < T::ACC; ++q) v += uint32_t(acc[y][q][i]) << (8 * q);
                store_bits<E>(py, yr + yc[i], v);
            }
        }
    }
}

template <int KIND, int NW, int R, int KB>
ndc_status launch_one(const MatArgs& a, int64_t blocks, size_t smem, LaunchContext& ctx) {
    if (!lds_fits(ctx, reinterpret_cast<const void*>(&matrix_conv_kernel<KIND, NW, R, KB>), smem))
        return NDC_ERR_UNSUPPORTED;
    NDC_LAUNCH(ctx, ctx.stream(), (matrix_conv_kernel<KIND, NW, R, KB>), dim3(unsigned(blocks)), dim3(64 * NW), smem, a);
    return NDC_OK;
}

template <int KIND, int KB>
ndc_status launch_kb(int rows, const MatArgs& a, int64_t blocks, size_t smem, LaunchContext& ctx) {
    if (rows == 16) return launch_one<KIND, 4, 4, KB>(a, blocks, smem, ctx);
    if (rows == 32) return launch_one<KIND, 8, 4, KB>(a, blocks, smem, ctx);
    if constexpr (KIND <= kBf16x3)
        if (rows == 64) return launch_one<KIND, 8, 8, KB>(a, blocks, smem, ctx);
    return NDC_ERR_UNSUPPORTED;
}

template <int KIND>
ndc_status launch_kind(int rows, int KB, const MatArgs& a, int64_t blocks, size_t smem, LaunchContext& ctx) {
    if constexpr (KIND == kF32) {
        if (KB == 3) return launch_kb<KIND, 3>(rows, a, blocks, smem, ctx);
        if (KB == 5) return launch_kb<KIND, 5>(rows, a, blocks, smem, ctx);
        if (KB == 7) return launch_kb<KIND, 7>(rows, a, blocks, smem, ctx);
        if (KB == 9) return launch_kb<KIND, 9>(rows, a, blocks, smem, ctx);
        if (KB == 11) return launch_kb<KIND, 11>(rows, a, blocks, smem, ctx);
        if (KB == 13) return launch_kb<KIND, 13>(rows, a, blocks, smem, ctx);
        if (KB == 15) return launch_kb<KIND, 15>(rows, a, blocks, smem, ctx);
        if (KB == 17) return launch_kb<KIND, 17>(rows, a, blocks, smem, ctx);
        if (KB == 21) return launch_kb<KIND, 21>(rows, a, blocks, smem, ctx);
        if (KB == 25) return launch_kb<KIND, 25>(rows, a, blocks, smem, ctx);
    } else if constexpr (KIND <= kBf16x3) {
        if (KB == 1) return launch_kb<KIND, 1>(rows, a, blocks, smem, ctx);
        if (KB == 2) return launch_kb<KIND, 2>(rows, a, blocks, smem, ctx);
    } else {
        if (KB == 1) return launch_kb<KIND, 1>(rows, a, blocks, smem, ctx);
    }
    return NDC_ERR_UNSUPPORTED;
}

struct KindShape { int PL, ESZ, G, N, STEP, maxKB, max_rows; };
KindShape shape_of(int kind) {
    switch (kind) {
        case kF32: return {1, 4, 4, 4, 2, 25, 64};
        case kBf16: return {1, 2, 4, 16, 32, 2, 64};
        case kBf16x3: return {2, 2, 4, 16, 32, 2, 64};
        case kI32: return {4, 1, 4, 16, 64, 1, 32};
        case kI16: return {2, 1, 4, 16, 64, 1, 32};
        default: return {1, 1, 4, 16, 64, 1, 32};
    }
}

int kind_of(const Plan& p, bool exact) {
    switch (p.dtype) {
        case NDC_F32:
            return exact ? kF32 : p.algo == NDC_ALGO_MFMA_BF16 ? kBf16 : kBf16x3;
        case NDC_I32: case NDC_U32: return kI32;
        case NDC_I16: case NDC_U16: return kI16;
        case NDC_I8: case NDC_U8: return kI8;
        default: return -1;
    }
}

// Whether the matrix form is the faster one, by the part of its tiles that is
// output.  A workgroup stages and multiplies 256 columns whatever the output
// has; the vector kernel's tiles are 64 wide, and it reads and writes a dilated
// axis in one piece, where the phases here touch every line d times over.  So a
// tile must be filled the more, the fewer taps (products, which the matrix cores do
// faster) an output has.  Where every workgroup has a CU of its own, its latency
// is all that counts.
//
// The lines are fitted to both forms on 2228 problems a type: images 24 to 2048
// wide of 60 K to 16 M elements, 1x1 to 31x31 taps, strides and dilations 1 to 3.
// Time lost against the better form: FP32 2.9%, i32 1.7%, i16 1.4%, i8 1.8% (with
// the matrix form throughout 48, 153, 54 and 27%, in single cases 8, 28, 9 and 5
// times).  16 M elements, us, matrix and vector: i32 62500x256, 9x1 taps, dilation 3:
// 323, 56; FP32 the same, 1x1: 84, 37; i32 250000x64, 3x3: 246, 111; 7812x2048: 68, 117.
bool matrix_pays(int kind, double fill, int64_t phases, double taps, int64_t blocks, int64_t cus) {
    struct Line { double phased, plain, plain_taps; int64_t few; double few_taps; };
    static constexpr Line f32 = {30, 0.15, 1e9, 1, 9}, i32 = {40, 0.7, 60, 1, 9}, i16 = {12, 0.25, 10, 2, 1},
                          i8 = {4, 0.15, 5, 2, 1};
    const Line& l = kind == kF32 ? f32 : kind == kI32 ? i32 : kind == kI16 ? i16 : i8;
    if (blocks <= l.few * cus && taps >= l.few_taps) return true;
    return fill >= (phases > 1 ? l.phased / taps : std::min(l.plain, l.plain_taps / taps));
}

// The same for BF16x3 against the systolic kernel of mfma_conv.hip, whose tiles are
// narrower too: that one serves tall kernels on narrow outputs (31x31 taps, dilation
// 2, 62500x64: 137 us against 286 here; 15x15, dilation 3, 125000x128: 171 against 315).
// 58 of 1876 such problems were slower here; single BF16 never was.
bool split_pays(double fill, int64_t phases, int64_t kh, int64_t kw, int64_t blocks, int64_t cus) {
    if (std::min(kh, kw) < 12 || fill >= 0.2) return true;
    return kh * kw >= 900 ? blocks <= 3 * cus : phases == 1 || blocks <= 6 * cus;
}

}  // namespace

bool launch_matrix(const Plan& p, bool exact, const void* x, const void* k, void* y, LaunchContext& ctx,
                   ndc_status* status) {
    const int kind = kind_of(p, exact);
    if (p.N != 2 || kind < 0 || !tile_spans_fit(p)) return false;
    const KindShape ks = shape_of(kind);
    const int64_t KH = p.k_shape[0], KW = p.k_shape[1], es = int64_t(dtype_size(p.dtype));
    MatArgs a;
    std::memset(&a, 0, sizeof(a));
    int64_t phases[2];
    for (int i = 0; i < 2; ++i) {
        if (p.stride[i] != 1 && p.stride[i] != p.dil[i]) return false;
        tile_axis(p, i, i == 0 ? p.out[1] : 1, &a.ax[i]);
        phases[i] = p.stride[i] == 1 ? p.dil[i] : 1;
        a.os[i] = int32_t(phases[i]);
        a.ax[i].U = int32_t(p.out[i]);
        a.ax[i].phases = tile_div(phases[i]);
        for (int s = 0; s < 2; ++s) {
            const ndc_value& v = p.side[i][s].value;
            a.cst[i][s] = float(v.re);
            a.icst[i][s] = int32_t(v.i);
            const bool fills = s == 0 ? a.ax[i].fconst : a.ax[i].bconst;
            if (p.pad[i][s] > 0 && fills && (kind <= kBf16x3 ? v.re != 0 : v.i != 0)) a.fills = 1;
        }
    }
    int KB = int((KW + ks.N - 1 + ks.STEP - 1) / ks.STEP);
    // pairs of band entries: odd counts are built, above 17 every fourth
    if (kind == kF32) KB = KB <= 17 ? std::max(3, KB | 1) : KB <= 21 ? 21 : std::max(25, KB);
    if (KB > ks.maxKB) return false;
    const int W = staged_width(ks.N, ks.STEP, KB);
    a.KWp = int32_t(KW);
    // rows per workgroup: the most whose region fits and whose workgroups still
    // fill the chip (each row step halves what is staged twice: 94 rows for 64
    // outputs, 62 for 32)
    const int64_t per = (p.out[0] + phases[0] - 1) / phases[0], pex = (p.out[1] + phases[1] - 1) / phases[1];
    const int64_t ntx = (pex + kTileX - 1) / kTileX * phases[1];
    int rows = 0;
    size_t smem = 0;
    int64_t blocks = 0;
    for (int r = ks.max_rows; r >= 16; r /= 2) {
        const int64_t nr = r + KH - 1;
        const size_t frag = kind == kF32 ? size_t(KH) * 64 * ((KB + 1) / 2) : size_t(2) * ks.G * KB * ks.PL * 1024;
        const size_t bytes = size_t(ks.PL) * nr * W * ks.ESZ + size_t((KH * KW + 3) & ~int64_t(3)) * 4 + frag;
        if (bytes > std::min(kLdsMax, ctx.max_lds())) continue;
        rows = r;
        smem = bytes;
        blocks = ntx * ((per + r - 1) / r) * phases[0];
        a.NR = int32_t(nr);
        a.ax[0].V = r;
        if (blocks * 10 >= int64_t(ctx.cu_count()) * 9) break;
    }
    if (!rows || blocks >= (int64_t(1) << 30)) return false;
    const double fill = double(p.out[0]) * double(p.out[1]) / (double(blocks) * rows * kTileX);
    if (exact && !matrix_pays(kind, fill, phases[1], double(KH) * double(KW), blocks, ctx.cu_count())) return false;
    if (kind == kBf16x3 && !split_pays(fill, phases[1], KH, KW, blocks, ctx.cu_count())) return false;
    a.ax[1].V = kTileX;
    a.ax[1].tiles = tile_div((pex + kTileX - 1) / kTileX);
    a.x = static_cast<const char*>(x) + p.x_lo * es;
    a.k = static_cast<const char*>(k) + p.k_lo * es;
    a.y = y;
    a.x_bytes = int32_t((p.x_hi - p.x_lo + 1) * es);
    a.k_bytes = int32_t((p.k_hi - p.k_lo + 1) * es);
    a.y_bytes = int32_t(p.y_numel * es);
    static const char* names[6] = {"matrix_conv_f32", "mfma_conv_bf16", "mfma_conv_bf16x3", "matrix_conv_i32",
                                   "matrix_conv_i16", "matrix_conv_i8"};
    ctx.kbegin(names[kind], double(es) * double(p.x_numel + p.k_numel + p.y_numel),
               2.0 * double(p.y_numel) * double(p.k_numel));
    ndc_status s = NDC_ERR_UNSUPPORTED;
    switch (kind) {
        case kF32: s = launch_kind<kF32>(rows, KB, a, blocks, smem, ctx); break;
        case kBf16: s = launch_kind<kBf16>(rows, KB, a, blocks, smem, ctx); break;
        case kBf16x3: s = launch_kind<kBf16x3>(rows, KB, a, blocks, smem, ctx); break;
        case kI32: s = launch_kind<kI32>(rows, KB, a, blocks, smem, ctx); break;
        case kI16: s = launch_kind<kI16>(rows, KB, a, blocks, smem, ctx); break;
        default: s = launch_kind<kI8>(rows, KB, a, blocks, smem, ctx); break;
    }
    ctx.kend();
    if (s == NDC_OK && !ctx.dry_run()) {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            ctx.err = std::string("matrix convolution launch: ") + hipGetErrorString(e);
            s = NDC_ERR_DEVICE;
        }
    }
    *status = s;
    return true;
}

}  // namespace ndc
