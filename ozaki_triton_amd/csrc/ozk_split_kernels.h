#pragma once
// ozk_split_kernels.h -- the split of ozaki_triton.py:137-211 as gfx950 kernels.
//
// Included by one translation unit per slice dtype (ozk_split_i8.hip, _f16,
// _bf16, _f32), which instantiate their kernels in parallel; the planner and
// the kernels without a slice type live in ozk_split.hip.
//
// For every operand row (a row of A, or a column of B seen through B^T) and
// every level l < L:
//   mu  = max(1e-38f, fl32(max_k |src_k|))
//   E   = ceil(log2_f32(mu)),  s = 2^(E - alpha)          (scales[b, l, row])
//   q   = src / s (in RES = fp64 for fp64 input, else fp32)
//   slice = int8: trunc(clamp(fl(q +/- 0.5), -128, 127));  fp16: RN(q)
//   src <- fl32(src - slice * s)   (the reference's fp32 residual buffer)
//
// Arithmetic per element (bit-identical to the above, fewer instructions):
//   level 0, fp64 input   q = x * 2^(alpha-E) and t = fl64(q +/- 0.5) in fp64;
//                         residual fma(-slice, s, x) rounded to fp64 then fp32
//                         (the product is exact, so this is fl32(fl64(x - slice*s))).
//   level >= 1, fp64 input: src is an fp32 residual r.  q = r * 2^(alpha-E)
//                         is exact in fp32 (or below 2^-126, where the slice
//                         is 0 either way), so q is computed with ldexp in
//                         fp32; fl64(q +/- 0.5) is exact, and trunc of it
//                         equals trunc(fl32(q +/- c)) with c = 0.5 - 2^-25
//                         for every fp32 q (c keeps q = 0.5 - 2^-25 from
//                         rounding up to 1; for |q| >= 0.5 subtracting 2^-25
//                         moves no sum across an integer).  The residual
//                         r - slice*s is exact in fp32 (for |q| >= 0.5 it is a
//                         multiple of ulp(r) not above |r|; else it is r), so
//                         one fp32 fma gives it.
//   fp32 input (RES = fp32): q = ldexp(x, alpha-E) is the correctly rounded
//                         quotient; t = fl32(q +/- 0.5) as in the reference;
//                         residual fma(-slice, s, x) = fl32(x - fl32(slice*s))
//                         because slice*s is exact.
//   fp16 slices: RN(q) from fp64 at level 0 of fp64 input (f64_to_f16);
//                elsewhere q is an fp32 value and the hardware RNE conversion
//                rounds it once; slice*s is exact in fp32 in every case.
//
// Any K, any column count and any element-aligned row: 16-byte loads and 4- /
// 8-byte stores need only element alignment (gfx950 takes unaligned global
// accesses), the last K % 4 elements of a row and the last columns of a group
// go element by element.  A slice row is written up to Kp >= K elements, zeros
// beyond K: ozk_matmul pads its slice rows to 16 bytes, so that the
// cross-GEMM reads them in place.
//
// Kernels:
//   split_fused_kernel  one or both operands of a matmul in one launch, K <=
//                       8192, each either K-contiguous rows or row-contiguous
//                       columns (the B^T view), in the input's own dtype.
//                       Rows: a group of 64*GW lanes owns one row.  Columns: a
//                       workgroup owns SEG * VEC adjacent columns for all of
//                       K.  Either way the operand stays in VGPRs across the
//                       levels: X is read from HBM once, each slice written
//                       once.
//   split_rows_kernel   the same body for rows alone, of up to 65536 elements.
//   split_cols_kernel   ... for columns alone, of 8192 < K <= 16384.
//   split_rows_coop_kernel  rows longer than 16384: K chunks of a row in
//                       separate workgroups that exchange the level maxima
//                       through the workspace.
//   split_coop_kernel   column groups, 128-byte row segments wide, cut along K
//                       over several workgroups that exchange the level maxima
//                       through the workspace (the default for columns of 64
//                       KB and more, up to 32 K chunks).
//   transpose_kernel    + a row kernel: columns longer than the cooperative
//                       kernel takes, transposed into the workspace first.
//   convert_kernel      narrow inputs of K > 8192: an exact fp32 copy in the
//                       workspace, split as fp32.
//   split_generic_kernel any strides: one workgroup per row, multi-pass over
//                       K, each level's residual recomputed from the input (no
//                       workspace).
#include "ozk_common.h"
#include "ozk_internal.h"
#include "ozk_split_launch.h"

#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <type_traits>

namespace ozk {

// ---------------------------------------------------------------------------
// Per-level constants from the row maximum m (wave-uniform).
// ---------------------------------------------------------------------------
struct LevelScale {
    float s;       // 2^(E - alpha), the stored scale
    int up;        // alpha - E
    double s64;    // s as double
    double inv64;  // 2^(alpha - E) as double (always a normal double)
};
OZK_DEV LevelScale level_scale(float m, int alpha) {
    const float mu = fmaxf(1e-38f, m);
    const int ema = ceil_log2_f32(mu) - alpha;
    LevelScale c;
    c.s = pow2f(ema);
    c.up = -ema;
    c.s64 = (double)c.s;
    c.inv64 = pow2d(-ema);
    // a row with an infinite entry has m = inf, for which the reference's
    // exp2(ceil(log2(m)) - alpha) is inf: that scale is stored as it is, so
    // the row's terms in C come out non-finite (its slices carry no meaning)
    if (!(m <= 3.402823466e38f)) c.s = m;
    return c;
}

// Truncation to int32 as the instruction does it: saturating, NaN to 0 (a C++
// cast leaves both undefined).  NaN entries quantise to 0 this way, with no
// compare and select per value.
OZK_DEV int cvt_i32(float x) {
    int k;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(k) : "v"(x));
    return k;
}
OZK_DEV int cvt_i32(double x) {
    int k;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(x));
    return k;
}

// Quantisation of one value at one level.  MODE: kQF64 = level 0 of fp64
// input; kQExact = level >= 1 of fp64 input (fp32 residuals, exact fp32
// arithmetic); kQF32 = every level of fp32 input.  Returns the slice bits
// (int8 value in the low byte, or fp16 bits) and writes the fp32 residual.
enum { kQF64 = 0, kQExact = 1, kQF32 = 2 };
template <typename ST, int MODE> struct Quant;

template <> struct Quant<int8_t, kQF64> {
    OZK_DEV static uint32_t run(double x, const LevelScale &c, float *res) {
        const double q = x * c.inv64;
        const int k = max(min(cvt_i32(q + __builtin_copysign(0.5, q)), 127), -128);
        *res = (float)__builtin_fma(-(double)k, c.s64, x);
        return (uint32_t)k;
    }
};
template <> struct Quant<int8_t, kQExact> {
    OZK_DEV static uint32_t run(float r, const LevelScale &c, float *res) {
        const float q = __builtin_ldexpf(r, c.up);
        const int k = max(min(cvt_i32(q + __builtin_copysignf(0x1.fffffep-2f, q)), 127), -128);
        *res = __builtin_fmaf(-(float)k, c.s, r);
        return (uint32_t)k;
    }
};
template <> struct Quant<int8_t, kQF32> {
    OZK_DEV static uint32_t run(float x, const LevelScale &c, float *res) {
        const float q = __builtin_ldexpf(x, c.up);
        const int k = max(min(cvt_i32(q + __builtin_copysignf(0.5f, q)), 127), -128);
        *res = __builtin_fmaf(-(float)k, c.s, x);
        return (uint32_t)k;
    }
};
template <> struct Quant<_Float16, kQF64> {
    OZK_DEV static uint32_t run(double x, const LevelScale &c, float *res) {
        const double q = x * c.inv64;
        const _Float16 h = f64_to_f16(q);
        *res = (float)__builtin_fma(-(double)(float)h, c.s64, x);
        return (uint32_t)__builtin_bit_cast(uint16_t, h);
    }
};
template <int MODE> struct QuantF16F32 {
    OZK_DEV static uint32_t run(float x, const LevelScale &c, float *res) {
        const float q = __builtin_ldexpf(x, c.up);
        const _Float16 h = (_Float16)q;
        *res = __builtin_fmaf(-(float)h, c.s, x);
        return (uint32_t)__builtin_bit_cast(uint16_t, h);
    }
};
template <> struct Quant<_Float16, kQExact> : QuantF16F32<kQExact> {};
template <> struct Quant<_Float16, kQF32> : QuantF16F32<kQF32> {};

// bfloat16 slices: one RNE rounding of q to 8 significant bits (integer code
// from fp64 at level 0 of fp64 input; from the exact fp32 q elsewhere)
template <> struct Quant<__bf16, kQF64> {
    OZK_DEV static uint32_t run(double x, const LevelScale &c, float *res) {
        const double q = x * c.inv64;
        const uint32_t h = f64_to_bf16_bits(q);
        const double d = (double)bf16_bits_to_f32(h);
        *res = (float)__builtin_fma(-d, c.s64, x);
        return h;
    }
};
template <int MODE> struct QuantBF16F32 {
    OZK_DEV static uint32_t run(float x, const LevelScale &c, float *res) {
        const float q = __builtin_ldexpf(x, c.up);
        const uint32_t h = f32_to_bf16_bits(q);
        *res = __builtin_fmaf(-bf16_bits_to_f32(h), c.s, x);
        return h;
    }
};
template <> struct Quant<__bf16, kQExact> : QuantBF16F32<kQExact> {};
template <> struct Quant<__bf16, kQF32> : QuantBF16F32<kQF32> {};

// fp32 slices: the slice is q rounded once to fp32 (exact when RES is fp32 or
// at levels >= 1, where q is an fp32 value or below 2^-126 either way)
template <> struct Quant<float, kQF64> {
    OZK_DEV static uint32_t run(double x, const LevelScale &c, float *res) {
        const float q = (float)(x * c.inv64);
        *res = (float)__builtin_fma(-(double)q, c.s64, x);
        return __float_as_uint(q);
    }
};
template <int MODE> struct QuantF32F32 {
    OZK_DEV static uint32_t run(float x, const LevelScale &c, float *res) {
        const float q = __builtin_ldexpf(x, c.up);
        *res = __builtin_fmaf(-q, c.s, x);
        return __float_as_uint(q);
    }
};
template <> struct Quant<float, kQExact> : QuantF32F32<kQExact> {};
template <> struct Quant<float, kQF32> : QuantF32F32<kQF32> {};

template <typename XT> struct Modes;
template <> struct Modes<double> { static constexpr int first = kQF64, rest = kQExact; };
template <> struct Modes<float> { static constexpr int first = kQF32, rest = kQF32; };

// ---------------------------------------------------------------------------
// Element classes.  The kernels are instantiated for fp64 and fp32 inputs and
// for the narrow ones together: those are converted to fp32 as they are
// loaded (exact, as the reference loads them into its fp32 RES,
// ozaki_triton.py:188) by their dtype code, which is uniform over a launch.
// Every load and store here needs element alignment only.
// ---------------------------------------------------------------------------
struct NarrowIn {};   // fp16 / bf16 / int8, SplitParams::x_code
template <typename XC> struct In {
    using V = XC;
    static constexpr int VEC = 16 / (int)sizeof(XC);   // columns one lane covers
};
template <> struct In<NarrowIn> {
    using V = float;
    static constexpr int VEC = 4;
};
typedef double dbl2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float flt4u __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 half4u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint16_t u16x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef int8_t i8x4u __attribute__((ext_vector_type(4), aligned(1)));

template <typename XC> struct Load;   // one(), and vec<N>(): N consecutive elements at index i
template <> struct Load<double> {
    OZK_DEV static double one(const void *x, int64_t i, int) { return ((const double *)x)[i]; }
    template <int N> OZK_DEV static void vec(const void *x, int64_t i, int, double *v) {
#pragma unroll
        for (int u = 0; u < N; u += 2) {
            const dbl2u a = *(const dbl2u *)((const double *)x + i + u);
            v[u] = a.x; v[u + 1] = a.y;
        }
    }
};
template <> struct Load<float> {
    OZK_DEV static float one(const void *x, int64_t i, int) { return ((const float *)x)[i]; }
    template <int N> OZK_DEV static void vec(const void *x, int64_t i, int, float *v) {
        static_assert(N == 4, "one 16-byte load");
        const flt4u a = *(const flt4u *)((const float *)x + i);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    }
};
template <> struct Load<NarrowIn> {
    OZK_DEV static float one(const void *x, int64_t i, int code) {
        if (code == 2) return (float)((const _Float16 *)x)[i];
        if (code == 3) return bf16_bits_to_f32(((const uint16_t *)x)[i]);
        return (float)((const int8_t *)x)[i];
    }
    template <int N> OZK_DEV static void vec(const void *x, int64_t i, int code, float *v) {
        static_assert(N == 4, "four elements");
        if (code == 2) {
            const half4u a = *(const half4u *)((const _Float16 *)x + i);
            v[0] = (float)a.x; v[1] = (float)a.y; v[2] = (float)a.z; v[3] = (float)a.w;
        } else if (code == 3) {
            const u16x4u a = *(const u16x4u *)((const uint16_t *)x + i);
            v[0] = bf16_bits_to_f32(a.x); v[1] = bf16_bits_to_f32(a.y);
            v[2] = bf16_bits_to_f32(a.z); v[3] = bf16_bits_to_f32(a.w);
        } else {
            const i8x4u a = *(const i8x4u *)((const int8_t *)x + i);
            v[0] = (float)a.x; v[1] = (float)a.y; v[2] = (float)a.z; v[3] = (float)a.w;
        }
    }
};
// N consecutive elements at index i, of which `left` exist (0 in the others)
template <typename XC, int N>
OZK_DEV void load_some(const void *x, int64_t i, int left, int code, typename In<XC>::V *v) {
    if (left >= N) {
        Load<XC>::template vec<N>(x, i, code, v);
    } else {
#pragma unroll
        for (int u = 0; u < N; ++u)
            v[u] = u < left ? Load<XC>::one(x, i + u, code) : (typename In<XC>::V)0;
    }
}

// ... all of them, or none (zeros)
template <typename XC, int N>
OZK_DEV void load_quad(const void *x, int64_t i, bool there, int code, typename In<XC>::V *v) {
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = (typename In<XC>::V)0;
    if (there) Load<XC>::template vec<N>(x, i, code, v);
}

// Store 4 consecutive slice values (k .. k+3) of one row.
typedef uint32_t u32a1 __attribute__((aligned(1)));
typedef uint64_t u64a2 __attribute__((aligned(2)));
typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
template <typename ST> struct Store4;
template <> struct Store4<int8_t> {
    OZK_DEV static void run(void *base, int64_t off, const uint32_t v[4]) {
        const uint32_t w = __builtin_amdgcn_perm(v[1], v[0], 0x0c0c0400u) |
                           __builtin_amdgcn_perm(v[3], v[2], 0x04000c0cu);
        *(u32a1 *)((int8_t *)base + off) = w;
    }
};
struct Store4Half {
    OZK_DEV static void run(void *base, int64_t off, const uint32_t v[4]) {
        const uint32_t lo = v[0] | (v[1] << 16), hi = v[2] | (v[3] << 16);
        *(u64a2 *)((uint16_t *)base + off) = (uint64_t)lo | ((uint64_t)hi << 32);
    }
};
template <> struct Store4<_Float16> : Store4Half {};
template <> struct Store4<__bf16> : Store4Half {};
template <> struct Store4<float> {
    OZK_DEV static void run(void *base, int64_t off, const uint32_t v[4]) {
        *(u32x4a4 *)((uint32_t *)base + off) = u32x4a4{v[0], v[1], v[2], v[3]};
    }
};
template <typename ST> OZK_DEV void store1(void *base, int64_t off, uint32_t v) {
    if constexpr (sizeof(ST) == 1) ((uint8_t *)base)[off] = (uint8_t)v;
    else if constexpr (sizeof(ST) == 2) ((uint16_t *)base)[off] = (uint16_t)v;
    else ((uint32_t *)base)[off] = v;
}
// ... of a row of which `left` elements remain, and `pleft` with its padding:
// the padding is zero whatever the quantisation of an absent element gave (NaN
// in a float slice of a row with an infinite entry)
template <typename ST>
OZK_DEV void store_some(void *base, int64_t off, int left, int pleft, uint32_t v[4]) {
    if (left >= 4) {
        Store4<ST>::run(base, off, v);
    } else if (pleft > 0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = u < left ? v[u] : 0u;
        if (pleft >= 4) {
            Store4<ST>::run(base, off, v);
        } else {
#pragma unroll
            for (int u = 0; u < 3; ++u)
                if (u < pleft) store1<ST>(base, off + u, v[u]);
        }
    }
}

// ... of elements that all exist, or are all padding
template <typename ST>
OZK_DEV void store_quad(void *base, int64_t off, bool there, uint32_t v[4]) {
    // (an absent element's int8 quantisation is zero whatever the scale)
    if constexpr (sizeof(ST) > 1) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = there ? v[u] : 0u;
    }
    Store4<ST>::run(base, off, v);
}

// The forms of the row and column bodies, chosen on the host (split_form), one
// to a kernel: as branches of one body they cost every column kernel 15 to 58
// spilled scalar registers, the small ones up to 16 vector registers as well.
// ozaki_matmul, us, branches / one to a kernel: 192^3 f64 -> 4 int8 15.1 / 13.8,
// 448^3 18.0 / 16.7, 16 x 512 x 128 x 512 f32 -> 3 fp16 30.8 / 30.1, 2688 x 448 x
// 128 f32 -> 2 int8 15.8 / 14.1, 613 x 1492 x 1664 f32 -> 5 bf16 (triangle) 87.4 /
// 83.9, 14 x 256 x 3724 x 158 f32 -> 3 int8 101.6 / 86.0.  Whole rows beside columns
// of any pitch keep their form (the split of 4 x 2240 rows and 111 columns of 1344,
// f32 -> 3 bf16, 48.4 / 31.2; both any before).
enum { kExact = 0, kWhole = 1, kAny = 2 };

// The same value afresh: the row's limits, taken at each level through this,
// are compared there, and not held as one lane mask per store across the levels
// (which spilled the scalar registers).
OZK_DEV int per_level(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
OZK_DEV int per_level_uniform(int x) {
    asm volatile("" : "+s"(x));
    return x;
}

OZK_DEV float absf(double x) { return (float)fabs(x); }   // fl32(|x|)
OZK_DEV float absf(float x) { return fabsf(x); }

// Maximum of non-negative values (no NaN among them: the callers' maxima start
// from 0 and ignore NaN) over the 64 lanes of a wave, returned wave-uniform.
// Such floats order like their bit patterns, and the integer maximum needs no
// canonicalised operands.  DPP row reductions, then the row broadcasts of
// GFX9; lanes a step does not write see 0, the maximum's identity.
template <int CTRL, int ROWS> OZK_DEV uint32_t dpp_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false));
}
OZK_DEV float wave_max(float f) {
    uint32_t v = __float_as_uint(f);
    v = dpp_max<0xB1, 0xF>(v);    // quad_perm [1,0,3,2]
    v = dpp_max<0x4E, 0xF>(v);    // quad_perm [2,3,0,1]
    v = dpp_max<0x141, 0xF>(v);   // row_half_mirror
    v = dpp_max<0x140, 0xF>(v);   // row_mirror: every lane holds its row's max
    v = dpp_max<0x142, 0xA>(v);   // row_bcast15 into rows 1 and 3
    v = dpp_max<0x143, 0xC>(v);   // row_bcast31 into rows 2 and 3
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 63));
}
// Maximum over the lanes of a wave that are congruent modulo SEG (2, 4 or 8):
// rotations within 16-lane rows, then across the four rows.
template <int SEG> OZK_DEV float seg_max(float f) {
    uint32_t v = __float_as_uint(f);
    v = dpp_max<0x128, 0xF>(v);                            // row_ror:8
    if constexpr (SEG <= 4) v = dpp_max<0x124, 0xF>(v);    // row_ror:4
    if constexpr (SEG <= 2) v = dpp_max<0x122, 0xF>(v);    // row_ror:2
    v = max(v, (uint32_t)__shfl_xor((int)v, 16));
    v = max(v, (uint32_t)__shfl_xor((int)v, 32));
    return __uint_as_float(v);
}

// Workgroup barrier for LDS exchanges: completes this wave's LDS accesses,
// then s_barrier.  Unlike __syncthreads() it does not wait for outstanding
// global stores (the previous level's slices).
OZK_DEV void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
}

// a / b and its remainder (a >= 0, b > 0, uniform over the workgroup): in 32 bits
// where they fit.  Every workgroup's first load waits for its row's batch and
// row.
struct Quot {
    int64_t q, r;
};
OZK_DEV Quot quot(int64_t a, int64_t b) {
    if (((uint64_t)(a | b) >> 32) == 0) {
        const uint32_t q = (uint32_t)a / (uint32_t)b;
        return {(int64_t)q, (int64_t)((uint32_t)a - q * (uint32_t)b)};
    }
    return {a / b, a % b};
}

// Where row `row` (of all batches) starts in X, the slices and the scales.  Short
// rows are bound by the scalar instructions before their first load (a wave of 4
// to 8 elements a lane issues more of them than vector ones): one batch goes
// without the division and half of the 64-bit products, several with a
// multiplication for it.  With the operand's parameters no longer selected
// from both operands' and the waves past a row's end idle, rows alone, f32 -> 2
// fp16, us, before / now: 12000 of 192 8.8 / 6.8, 9000 of 704 13.4 / 9.1, 8960 of
// 1280 22.6 / 16.6, 4 x 2240 of 1344 22.5 / 18.1; f64 -> 4 int8 11.6 / 9.6, 20.0 /
// 16.6, 33.2 / 27.6, 34.4 / 29.3.
struct RowAt {
    int64_t x, slice, scale;
};
OZK_DEV RowAt row_at(const SplitParams &p, int64_t row) {
    if (p.batch == 1) return {row * p.xs_r, row * p.ss_r, row * p.cs_r};
    Quot at;
    if (p.row_mul) {   // row < 2^31
        at.q = __umulhi((uint32_t)row, p.row_mul) >> p.row_shift;
        at.r = (uint32_t)row - (uint32_t)at.q * (uint32_t)p.rows;
    } else {
        at = quot(row, p.rows);
    }
    return {at.q * p.xs_b + at.r * p.xs_r, at.q * p.ss_b + at.r * p.ss_r,
            at.q * p.cs_b + at.r * p.cs_r};
}

// ---------------------------------------------------------------------------
// Row-resident split.  Block = RPB groups of G = 64*GW lanes; group g owns
// global row block*RPB + g.  Lane t of a group holds elements
// (c*G + t)*4 + {0..3} for c < NC, so each wave load covers 1 KB (fp64: 2 KB)
// of contiguous row and each wave store 256 B (int8) of contiguous slice.
// Level 0 quantises the input values; levels >= 1 the fp32 residuals.
// Requirements (checked on the host): xs_k == 1, ss_k == 1, Kp <= 4 * NC * G.
// ---------------------------------------------------------------------------
template <int GW, int RPB>
OZK_DEV float row_max(float m, float (*red)[RPB][GW], int buf, int grp, int t) {
    m = wave_max(m);
    if constexpr (GW > 1) {
        if ((t & 63) == 0) red[buf][grp][t / 64] = m;
        lds_barrier();
        float r = red[buf][grp][0];
#pragma unroll
        for (int w = 1; w < GW; ++w) r = fmaxf(r, red[buf][grp][w]);
        m = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(r)));
    }
    return m;
}

// One row per group of 64 * GW lanes.  xrow / srow: the row's first element in X
// and in the slices; K, Kp: its elements in X and in the slices; off: row of
// this lane's group unused (its lanes only take part in the barriers).  FORM:
// kExact tests nothing; kWhole takes K and Kp of whole quads; kAny: whole
// chunks inside K go without tests.  smax(m, l): maximum of the row at
// level l from a lane's; put(l, c): stores the scale.
template <typename XC, typename ST, int G, int NC, int FORM, typename SMax, typename Put>
OZK_DEV void split_row(const SplitParams &p, int64_t xrow, int64_t srow, int K, int Kp, bool off,
                       int t, SMax &&smax, Put &&put) {
    using V = typename In<XC>::V;
    constexpr int NE = 4 * NC;
    V v[NE];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int e0 = (c * G + t) * 4;
        if (FORM == kExact || (FORM == kAny && (c + 1) * G * 4 <= K))
            Load<XC>::template vec<4>(p.X, xrow + e0, p.x_code, v + 4 * c);
        else if (FORM == kWhole)
            load_quad<XC, 4>(p.X, xrow + e0, e0 < K && !off, p.x_code, v + 4 * c);
        else
            load_some<XC, 4>(p.X, xrow + e0, off ? 0 : K - e0, p.x_code, v + 4 * c);
    }
    float w[NE];
    auto level = [&](int l, auto first, auto &src) {
        constexpr int MODE = decltype(first)::value ? Modes<V>::first : Modes<V>::rest;
        float m = 0.0f;
#pragma unroll
        for (int e = 0; e < NE; ++e) m = fmaxf(m, absf(src[e]));
        const LevelScale c = level_scale(smax(m, l), p.alpha);
        put(l, c);
        const int64_t sl = srow + l * p.ss_l;
        const int Ks = per_level_uniform(K), Kps = per_level_uniform(Kp);
        const int lt = per_level(t);
        const int wt = __builtin_amdgcn_readfirstlane(lt);
#pragma unroll
        for (int ch = 0; ch < NC; ++ch) {
            const int e0 = (ch * G + lt) * 4;
            if (FORM != kExact && (ch * G + wt) * 4 >= Kps) {   // the wave is past the row's end
                if (decltype(first)::value)
#pragma unroll
                    for (int u = 0; u < 4; ++u) w[ch * 4 + u] = 0.0f;
                continue;
            }
            uint32_t qv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) qv[u] = Quant<ST, MODE>::run(src[ch * 4 + u], c, &w[ch * 4 + u]);
            if (FORM == kExact || (FORM == kAny && (ch + 1) * G * 4 <= Ks && !off))
                Store4<ST>::run(p.slices, sl + e0, qv);
            else if (FORM == kWhole) {
                if (e0 < Kps && !off) store_quad<ST>(p.slices, sl + e0, e0 < Ks, qv);
            } else if (!off) store_some<ST>(p.slices, sl + e0, Ks - e0, Kps - e0, qv);
            // the residuals here, not at their first use (the next level's
            // maximum): sunk there, every input and every slice value are live
            // at once
#pragma unroll
            for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(w[ch * 4 + u]));
        }
    };
    if constexpr (std::is_same<V, float>::value) {
        // one body for every level: less code to fetch
#pragma unroll
        for (int e = 0; e < NE; ++e) w[e] = v[e];
        for (int l = 0; l < p.L; ++l) level(l, std::false_type{}, w);
    } else {
        level(0, std::true_type{}, v);
        for (int l = 1; l < p.L; ++l) level(l, std::false_type{}, w);
    }
}

// The body of the row kernel for row block `block`; red: LDS for the row maxima.
template <typename XC, typename ST, int GW, int RPB, int NC, int FORM>
OZK_DEV void split_rows_body(const SplitParams &p, int64_t block, float (*red)[RPB][GW]) {
    constexpr int G = 64 * GW;
    const int tid = threadIdx.x;
    // the lanes' group and row are uniform over a wave
    const int grp = __builtin_amdgcn_readfirstlane(tid / G);
    const int t = tid % G;
    const int64_t nrows = p.batch * p.rows;
    const int64_t grow = block * RPB + grp;
    const bool off = grow >= nrows;
    const RowAt at = row_at(p, off ? 0 : grow);
    float *srow_scale = p.scales + at.scale;
    auto smax = [&](float m, int l) { return row_max<GW, RPB>(m, red, l & 1, grp, t); };
    auto put = [&](int l, const LevelScale &c) {
        if (!off && t == 0) srow_scale[l * p.cs_l] = c.s;
    };
    split_row<XC, ST, G, NC, FORM>(p, at.x, at.slice, (int)p.K, (int)p.Kp, off, t, smax, put);
}

template <typename XC, typename ST, int GW, int RPB, int NC, int FORM>
__global__ __launch_bounds__(64 * GW * RPB) void split_rows_kernel(SplitParams p) {
    __shared__ float red[2][RPB][GW];
    split_rows_body<XC, ST, GW, RPB, NC, FORM>(p, blockIdx.x, red);
}

// ---------------------------------------------------------------------------
// Column-resident split for operands whose rows are contiguous (xs_r == 1):
// the B^T view, where a "row" is a column of B.  A workgroup of NT lanes owns
// SW = SEG * VEC adjacent columns for all K: lane t covers the VEC columns
// col0 + VEC * (t % SEG) + {0..VEC-1} and the rows 4 * (t / SEG + RPP * g) +
// {0..3}, g < NQ, RPP = NT / SEG, so that a wave load covers 64 / SEG row
// pieces of SEG * 16 bytes and a lane holds 4 consecutive k of each column (4-
// / 8-byte slice stores along K).  Workgroups that share a 128-byte line of X
// are consecutive on one XCD.
// Requirements (host-checked): xs_r == 1, ss_k == 1, Kp <= 4 * NQ * RPP.
// ---------------------------------------------------------------------------
OZK_DEV int64_t xcd_remap(int64_t g, int64_t n) {
    // hardware dispatches workgroup g to XCD g % 8; give each XCD a contiguous
    // range of logical ids (the tail beyond a multiple of 8 keeps its id)
    const int64_t q = n / 8;
    if (g >= q * 8) return g;
    return (g % 8) * q + g / 8;
}

// LDS of one column workgroup: each wave's maxima, and (SEG > 1) the columns'
// scale and shift.
template <int NT, int SEG, int VEC> struct ColsShared {
    float red[2][NT / 64][SEG][VEC];
    float2 scale[2][SEG * VEC];
};

// The level's constants of a lane's VEC columns from the lane maxima m.  With
// one piece per row (SEG = 1) they are uniform over the workgroup and every
// wave computes them in scalar registers; else one lane per column does, and
// the others read them from the LDS (computed by every lane they cost 100
// VALU instructions a level beside the 8 per value).
template <int NT, int SEG, int VEC>
OZK_DEV void cols_scale(float m[VEC], ColsShared<NT, SEG, VEC> &sh, int buf, int tid, int alpha,
                        LevelScale c[VEC]) {
    constexpr int NW = NT / 64, SW = SEG * VEC;
    const int lane = tid & 63;
#pragma unroll
    for (int u = 0; u < VEC; ++u) {
        if constexpr (SEG == 1) m[u] = wave_max(m[u]);
        else m[u] = seg_max<SEG>(m[u]);
    }
    if (lane < SEG) {
#pragma unroll
        for (int u = 0; u < VEC; ++u) sh.red[buf][tid / 64][lane][u] = m[u];
    }
    lds_barrier();
    if constexpr (SEG == 1) {
#pragma unroll
        for (int u = 0; u < VEC; ++u) {
            uint32_t r = __float_as_uint(sh.red[buf][0][0][u]);
#pragma unroll
            for (int w = 1; w < NW; ++w) r = max(r, __float_as_uint(sh.red[buf][w][0][u]));
            r = (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
            c[u] = level_scale(__uint_as_float(r), alpha);
        }
    } else {
        if (tid < SW) {
            uint32_t r = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w)
                r = max(r, __float_as_uint(sh.red[buf][w][tid / VEC][tid % VEC]));
            const LevelScale d = level_scale(__uint_as_float(r), alpha);
            sh.scale[buf][tid] = make_float2(d.s, __int_as_float(d.up));
        }
        lds_barrier();
#pragma unroll
        for (int u = 0; u < VEC; ++u) {
            const float2 d = sh.scale[buf][(tid % SEG) * VEC + u];
            c[u].s = d.x;
            c[u].up = __float_as_int(d.y);
            c[u].s64 = pow2d(-c[u].up);
            c[u].inv64 = pow2d(c[u].up);
        }
    }
}

// The columns of one lane.  xb / sbase: its first element (row 4 * ro, its first
// column) in X and in the slices; K, Kp: rows from there on, with the padding;
// ncol: of its VEC columns, those that exist; col_ok, kin: uniform over the
// workgroup, every lane has VEC columns / rows below kin exist for every lane.
// FORM: kExact tests nothing; kWhole: every lane has all of its columns or none,
// K and Kp are whole quads; SKIP: rows past the last one are left out; BYCOL: a
// column's four slice values are stored before the next column's are made.  With
// all at once the kernels of K up to 8192 spilled scalar registers, and f32 into
// bf16 took 139 vector ones; the cooperative ones take it, which by columns
// grow past the 168 that leave three waves a SIMD.
// scale(m, l, c): the level's constants of the lane's columns from its maxima;
// put(l, c): stores their scales.
template <typename XC, typename ST, int RPP, int NQ, int FORM, bool SKIP, bool BYCOL,
          typename Scale, typename Put>
OZK_DEV void split_cols(const SplitParams &p, int64_t xb, int64_t sbase, int K, int Kp, int ncol,
                        bool col_ok, int kin, Scale &&scale, Put &&put) {
    using V = typename In<XC>::V;
    constexpr int VEC = In<XC>::VEC;
    V v[NQ][4][VEC];
#pragma unroll
    for (int g = 0; g < NQ; ++g) {
#pragma unroll
        for (int dk = 0; dk < 4; ++dk) {
            const int k = 4 * g * RPP + dk;
            if (FORM == kExact || (FORM == kAny && col_ok && 4 * (g + 1) * RPP <= kin))
                Load<XC>::template vec<VEC>(p.X, xb + k * p.xs_k, p.x_code, v[g][dk]);
            else if (FORM == kWhole)
                load_quad<XC, VEC>(p.X, xb + k * p.xs_k, 4 * g * RPP < K && ncol > 0, p.x_code,
                                   v[g][dk]);
            else
                load_some<XC, VEC>(p.X, xb + k * p.xs_k, k < K ? ncol : 0, p.x_code, v[g][dk]);
        }
    }
    float w[NQ][4][VEC];
    auto level = [&](int l, auto first, auto &src) {
        constexpr int MODE = decltype(first)::value ? Modes<V>::first : Modes<V>::rest;
        float m[VEC];
#pragma unroll
        for (int u = 0; u < VEC; ++u) m[u] = 0.0f;
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
            for (int dk = 0; dk < 4; ++dk)
#pragma unroll
                for (int u = 0; u < VEC; ++u) m[u] = fmaxf(m[u], absf(src[g][dk][u]));
        LevelScale c[VEC];
        scale(m, l, c);
        put(l, c);
        const int64_t sl = sbase + l * p.ss_l;
        const int Ks = per_level(K), Kps = per_level(Kp), nc = per_level(ncol);
        // of the wave's first row
        const int kpw = SKIP ? __builtin_amdgcn_readfirstlane(Kps) : 0;
#pragma unroll
        for (int g = 0; g < NQ; ++g) {
            const int k0 = 4 * g * RPP;
            if (SKIP && k0 >= kpw) {   // the wave is past the last row
                if (decltype(first)::value)
#pragma unroll
                    for (int dk = 0; dk < 4; ++dk)
#pragma unroll
                        for (int u = 0; u < VEC; ++u) w[g][dk][u] = 0.0f;
                continue;
            }
            if constexpr (BYCOL) {
#pragma unroll
                for (int u = 0; u < VEC; ++u) {
                    uint32_t qv[4];
#pragma unroll
                    for (int dk = 0; dk < 4; ++dk)
                        qv[dk] = Quant<ST, MODE>::run(src[g][dk][u], c[u], &w[g][dk][u]);
                    const int64_t at = sl + u * p.ss_r + k0;
                    if (FORM == kExact || (FORM == kAny && col_ok && 4 * (g + 1) * RPP <= kin))
                        Store4<ST>::run(p.slices, at, qv);
                    else if (FORM == kWhole) {
                        if (k0 < Kps && nc > 0) store_quad<ST>(p.slices, at, k0 < Ks, qv);
                    } else if (u < nc)
                        store_some<ST>(p.slices, at, Ks - k0, Kps - k0, qv);
                }
            } else {
                static_assert(BYCOL || FORM != kWhole, "the cooperative kernels' forms");
                uint32_t qv[VEC][4];
#pragma unroll
                for (int dk = 0; dk < 4; ++dk)
#pragma unroll
                    for (int u = 0; u < VEC; ++u)
                        qv[u][dk] = Quant<ST, MODE>::run(src[g][dk][u], c[u], &w[g][dk][u]);
                if (FORM == kExact || (FORM == kAny && col_ok && 4 * (g + 1) * RPP <= kin)) {
#pragma unroll
                    for (int u = 0; u < VEC; ++u)
                        Store4<ST>::run(p.slices, sl + u * p.ss_r + k0, qv[u]);
                } else {
#pragma unroll
                    for (int u = 0; u < VEC; ++u)
                        if (u < nc)
                            store_some<ST>(p.slices, sl + u * p.ss_r + k0, Ks - k0, Kps - k0, qv[u]);
                }
            }
            // the residuals here, not at their first use (see split_row)
#pragma unroll
            for (int dk = 0; dk < 4; ++dk)
#pragma unroll
                for (int u = 0; u < VEC; ++u) asm volatile("" : "+v"(w[g][dk][u]));
        }
    };
    if constexpr (std::is_same<V, float>::value) {
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
            for (int dk = 0; dk < 4; ++dk)
#pragma unroll
                for (int u = 0; u < VEC; ++u) w[g][dk][u] = v[g][dk][u];
        for (int l = 0; l < p.L; ++l) level(l, std::false_type{}, w);
    } else {
        level(0, std::true_type{}, v);
        for (int l = 1; l < p.L; ++l) level(l, std::false_type{}, w);
    }
}

template <typename XC, typename ST, int NT, int SEG, int NQ, int FORM>
OZK_DEV void split_cols_body(const SplitParams &p, int64_t sidx,
                             ColsShared<NT, SEG, In<XC>::VEC> &sh) {
    constexpr int VEC = In<XC>::VEC;
    constexpr int SW = SEG * VEC;
    constexpr int RPP = NT / SEG;

    const int tid = threadIdx.x;
    const int seg = tid % SEG, ro = tid / SEG;
    const int64_t nstr = (p.rows + SW - 1) / SW;
    const Quot at = quot(sidx, nstr);
    const int64_t b = at.q, col0 = at.r * SW, col = col0 + seg * VEC;
    const int ncol = (int)(p.rows - col < VEC ? p.rows - col : VEC);
    const bool col_ok = col0 + SW <= p.rows;
    const int64_t xb = b * p.xs_b + col + 4 * ro * p.xs_k;
    const int64_t sbase = b * p.ss_b + col * p.ss_r + 4 * ro;
    float *sc_base = p.scales + b * p.cs_b + col * p.cs_r;
    auto scale = [&](float m[VEC], int l, LevelScale c[VEC]) {
        cols_scale<NT, SEG, VEC>(m, sh, l & 1, tid, p.alpha, c);
    };
    auto put = [&](int l, const LevelScale c[VEC]) {
        if (ro == 0) {
#pragma unroll
            for (int u = 0; u < VEC; ++u)
                if (FORM == kExact || u < ncol) sc_base[l * p.cs_l + u * p.cs_r] = c[u].s;
        }
    };
    split_cols<XC, ST, RPP, NQ, FORM, FORM != kExact, true>(
        p, xb, sbase, (int)p.K - 4 * ro, (int)p.Kp - 4 * ro, ncol, col_ok, (int)p.K, scale, put);
}

template <typename XC, typename ST, int NT, int SEG, int NQ, int FORM>
__global__ __launch_bounds__(NT) void split_cols_kernel(SplitParams p) {
    __shared__ ColsShared<NT, SEG, In<XC>::VEC> sh;
    split_cols_body<XC, ST, NT, SEG, NQ, FORM>(p, xcd_remap(blockIdx.x, (int64_t)gridDim.x), sh);
}

// ---------------------------------------------------------------------------
// One or both operands of a matmul in one launch (K <= 8192).  The first n0
// workgroups split operand 0, the others operand 1; each operand is rows or
// columns (SplitParams::cols), rows beside columns operand 1.  Neither waits on
// another workgroup.  FORM: the rows' form, CFORM: the columns'.
// ---------------------------------------------------------------------------
struct FusedSplit {
    SplitParams op[2];
};
template <typename XC, typename ST, int NT, int GW, int NC, int SEG, int NQ, int FORM, int CFORM>
__global__ __launch_bounds__(NT) void split_fused_kernel(FusedSplit f, uint32_t n0) {
    const bool which = blockIdx.x >= n0;
    const uint32_t g = blockIdx.x - (which ? n0 : 0);
    constexpr int RPB = NT / (64 * GW);
    if constexpr (SEG > 0) {
        __shared__ union {
            ColsShared<NT, SEG, In<XC>::VEC> cols;
            float rows[2][RPB][GW];
        } sh;
        if (!which || f.op[1].cols)
            split_cols_body<XC, ST, NT, SEG, NQ, CFORM>(
                f.op[which], xcd_remap(g, which ? gridDim.x - n0 : n0), sh.cols);
        else   // (not f.op[which]: every wave would load both and select)
            split_rows_body<XC, ST, GW, RPB, NC, FORM>(f.op[1], g, sh.rows);
    } else {
        __shared__ float red[2][RPB][GW];
        split_rows_body<XC, ST, GW, RPB, NC, FORM>(f.op[which], g, red);
    }
}

// ---------------------------------------------------------------------------
// Column split shared by a group of workgroups (row-contiguous operands, the
// B^T view).  A 16-byte load per lane covers only 16 bytes of a row, so a
// strip one load wide (split_cols_kernel, SEG = 1) touches one cache line per 16
// bytes read; reads of 128-byte row segments run at copy speed.  A strip of
// SW = 128 / sizeof(XT) columns over all of K does not fit one CU, so it is
// cut along K into P chunks of CH rows, one workgroup each, and the level
// maxima are combined through global memory.  A column group is SEG 16-byte
// pieces of each row: 128 bytes (SEG = 8), or 32 bytes (SEG = 2, when forced)
// for columns too long for 32 chunks of those, whose chunks then hold 4x the
// rows with the same registers (65536-long fp32 columns: 32 chunks of 2048):
//   * workgroup g = blockIdx.x is member g % P of column group g / P (batch
//     b, columns col0 .. col0 + SW, SW = SEG * VEC); lane t covers the VEC
//     columns col0 + VEC * (t % SEG) + {0..VEC-1} and the rows
//     member * CH + 4 * (t / SEG + RPP * j) + {0..3}, j < RPL / 4, RPP = 256 /
//     SEG, so a wave load covers 64 / SEG whole row segments and a lane holds
//     4 consecutive k of each column (4- / 8-byte slice stores along K);
//   * per level, wave 0 stores the workgroup's column maxima into
//     slot[group][level][member][SW], one 64-bit word each (the tag 1 in the
//     high half, the fp32 maximum in the low half), with agent-scope stores,
//     and polls the P * SW words of its group and level with agent-scope
//     loads until all carry the tag.  Every word validates itself, so no
//     fence (no L2 write-back or invalidation) is needed;
//   * the members of a group are consecutive workgroup ids, and the planner
//     keeps P at most 8 below the workgroups one XCD holds (the residency
//     limit before plan_split_raw), so every group becomes resident and its
//     waits end.  A wait is still bounded (2 s of the 100 MHz real-time
//     counter): a member that gives up sets the launch's status word and
//     member 0 stores NaN scales.  After ozk_split the poison kernel then
//     makes every scale of the split NaN and records the failure in the
//     sticky device status (ozk_device_status); in a matmul the cross-GEMM
//     reads the status word instead, writes NaN for C and records it.
// slot and the status word after it must be zero at launch (the launcher
// clears them first).
// ---------------------------------------------------------------------------
// LDS of one cooperative column workgroup
template <typename XT, int SEG> struct CoopShared {
    static constexpr int VEC = 16 / (int)sizeof(XT);
    float red[kCoopNT / 64][SEG][VEC];
    float fin[SEG * VEC];
    int bad;
};

// The body of the cooperative column kernel for logical workgroup g (member
// g % P of column group g / P): its own workgroup, or one of split_pair_kernel.
template <typename XT, typename ST, int RPL, int SEG>
OZK_DEV void split_coop_body(const SplitParams &p, uint64_t *slot, int P, uint32_t want_tag,
                             uint64_t tick_limit, uint32_t *status, int64_t g,
                             CoopShared<XT, SEG> &sh) {
    constexpr int NT = kCoopNT, NG = RPL / 4;
    constexpr int VEC = 16 / (int)sizeof(XT);
    constexpr int SW = SEG * VEC;        // columns per group
    constexpr int RPP = NT / SEG;        // row quads per pass
    constexpr int NW = NT / 64;
    static_assert(SEG == 8 || SEG == 2, "128- or 32-byte row segments");
    auto &red = sh.red;
    auto &fin = sh.fin;
    int &bad = sh.bad;

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int seg = t % SEG, ro = t / SEG;
    const int member = (int)(g % P);
    const int64_t grp = g / P;
    const int64_t nstr = (p.rows + SW - 1) / SW;
    const Quot at = quot(grp, nstr);
    const int64_t b = at.q, col0 = at.r * SW;
    const int64_t mycol = col0 + seg * VEC;
    const int64_t kbase = (int64_t)member * (RPP * RPL) + 4 * ro;   // this lane's first row
    // of this lane's columns, those that exist; and its rows' limits
    const int ncol = (int)(p.rows - mycol < VEC ? p.rows - mycol : VEC);
    const int K = (int)(p.K - kbase), Kp = (int)(p.Kp - kbase);
    const bool col_ok = col0 + SW <= p.rows;
    const int64_t mleft = p.K - (int64_t)member * (RPP * RPL);   // the chunk's rows
    const int kin = (int)(mleft < RPP * RPL ? mleft : RPP * RPL);

    if (t == 0) bad = 0;

    // maximum over the group of the lane maxima m (fl32 values >= 0), per column
    auto group_max = [&](float m[VEC], int l) {
#pragma unroll
        for (int u = 0; u < VEC; ++u)
#pragma unroll
            for (int x = SEG; x < 64; x *= 2) m[u] = fmaxf(m[u], __shfl_xor(m[u], x));
        if (lane < SEG) {
#pragma unroll
            for (int u = 0; u < VEC; ++u) red[wave][lane][u] = m[u];
        }
        lds_barrier();
        float r = 0.0f;
        if (t < SW) {
            r = red[0][t / VEC][t % VEC];
#pragma unroll
            for (int w = 1; w < NW; ++w) r = fmaxf(r, red[w][t / VEC][t % VEC]);
        }
        if (P > 1 && wave == 0) {
            // publish this member's maxima, then poll until every member's
            // word of this level carries the tag (words already seen are not
            // read again)
            uint64_t *sl = slot + (grp * p.L + l) * (int64_t)P * SW;
            if (t < SW)
                __hip_atomic_store(sl + (int64_t)member * SW + t, kCoopTag | __float_as_uint(r),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int nw = P * SW;
            uint64_t seen = 0;
            const uint64_t want = (lane < nw) ? (((nw - 1 - lane) / 64 >= 63)
                                                     ? ~0ull
                                                     : (2ull << ((nw - 1 - lane) / 64)) - 1)
                                              : 0;
            float q = 0.0f;
            const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
            for (;;) {
                for (int n = 0; n < (nw + 63) / 64; ++n) {
                    const int i = lane + 64 * n;
                    if (i < nw && !((seen >> n) & 1)) {
                        const uint64_t w64 =
                            __hip_atomic_load(sl + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if ((uint32_t)(w64 >> 32) == want_tag) {
                            seen |= 1ull << n;
                            q = fmaxf(q, __uint_as_float((uint32_t)w64));
                        }
                    }
                }
                if (__all(seen == want)) break;
                if (__builtin_amdgcn_s_memrealtime() - t0 >= tick_limit) {
                    if (lane == 0) {
                        bad = 1;
                        __hip_atomic_fetch_or(status, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
                    }
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            // lane i holds the maximum of column i % SW over members i / SW + 64 / SW * n
            r = q;
#pragma unroll
            for (int x = SW; x < 64; x *= 2) r = fmaxf(r, __shfl_xor(r, x));
        }
        if (t < SW) fin[t] = r;
        lds_barrier();
#pragma unroll
        for (int u = 0; u < VEC; ++u) m[u] = fin[seg * VEC + u];
    };
    // scales of level l (member 0 stores them; NaN after a wait that ran out)
    auto store_scales = [&](int l) {
        if (member == 0 && t < SW && col0 + t < p.rows) {
            const LevelScale c = level_scale(fin[t], p.alpha);
            p.scales[b * p.cs_b + l * p.cs_l + (col0 + t) * p.cs_r] =
                bad ? __int_as_float(0x7fc00000) : c.s;
        }
    };
    const int64_t xb = b * p.xs_b + mycol + kbase * p.xs_k;
    const int64_t sbase = b * p.ss_b + mycol * p.ss_r + kbase;
    auto scale = [&](float m[VEC], int l, LevelScale c[VEC]) {
        group_max(m, l);
        store_scales(l);
#pragma unroll
        for (int u = 0; u < VEC; ++u) c[u] = level_scale(m[u], p.alpha);
    };
    auto put = [](int, const LevelScale *) {};
    if (col_ok && kin == 4 * NG * RPP)
        split_cols<XT, ST, RPP, NG, kExact, false, false>(p, xb, sbase, 0, 0, 0, true, 0, scale, put);
    else
        split_cols<XT, ST, RPP, NG, kAny, false, false>(p, xb, sbase, K, Kp, ncol, col_ok, kin, scale,
                                                        put);
}

// fp64 into int8, fp16 and fp32 slices takes 167 or 168 registers, three waves a
// SIMD.  With one or two more, two waves, us: f64 2 x 8192^2 -> 4 int8
// (split_pair_kernel) 338 -> 372, 4096 columns of 16384 -> 2 int8 176 -> 203, of
// 8192 -> 3 fp16 121 -> 128.
template <typename XT, typename ST, int RPL, int SEG>
__global__ __launch_bounds__(kCoopNT) void split_coop_kernel(SplitParams p, uint64_t *slot, int P,
                                                             uint32_t want_tag,
                                                             uint64_t tick_limit,
                                                             uint32_t *status) {
    __shared__ CoopShared<XT, SEG> sh;
    split_coop_body<XT, ST, RPL, SEG>(p, slot, P, want_tag, tick_limit, status, blockIdx.x, sh);
}

// ---------------------------------------------------------------------------
// Both splits of a matmul in one launch, where A's rows take a 256-lane row
// configuration (4 waves per row) and B's columns the cooperative column
// kernel with 128-byte groups (fp64 operands, 4096 <= K <= 8192: config 3).
// The grid runs in periods of P + KA workgroups: the P members of one
// column group of B, then KA row blocks of A.  The row blocks never wait, so
// they keep CUs busy while column groups wait on their exchanges, and the
// two splits cost one launch.  The members of a group stay consecutive
// workgroup ids, which the cooperative kernel's residency argument needs
// (row blocks between groups retire without waiting).
// ---------------------------------------------------------------------------
template <typename XT, typename ST, int RPL, int NC>
__global__ __launch_bounds__(kCoopNT) void split_pair_kernel(SplitParams pb, uint64_t *slot, int P,
                                                             uint32_t want_tag,
                                                             uint64_t tick_limit,
                                                             uint32_t *status, SplitParams pa,
                                                             int ka) {
    __shared__ CoopShared<XT, 8> sh;
    __shared__ float red[2][1][4];
    const int64_t period = (int64_t)P + ka;
    const int64_t q = blockIdx.x / period;
    const int pos = (int)(blockIdx.x % period);
    if (pos < P) {
        split_coop_body<XT, ST, RPL, 8>(pb, slot, P, want_tag, tick_limit, status, q * P + pos, sh);
    } else {
        const int64_t ab = q * ka + (pos - P);
        if (ab >= pa.batch * pa.rows) return;
        if (pa.K == 4 * NC * 256) split_rows_body<XT, ST, 4, 1, NC, kExact>(pa, ab, red);
        else split_rows_body<XT, ST, 4, 1, NC, kAny>(pa, ab, red);
    }
}

// ---------------------------------------------------------------------------
// Row split shared by workgroups, for K-contiguous rows too long for one
// workgroup per row to keep a CU busy (rows over 16384 elements: one
// 1024-lane workgroup per CU, whose loads then never overlap another's
// arithmetic).  Workgroup g takes K chunk g % P of row g / P: CHR = 4 * NC *
// 64 * GW elements, laid out per lane as in split_rows_kernel.  Per level the
// workgroup's row maximum is combined over the P chunks through tagged words as
// in split_coop_kernel: slot[row][level][P], one word per chunk (lane i of
// wave 0 polls chunk i's word; P <= 64).
// ---------------------------------------------------------------------------
template <typename XT, typename ST, int GW, int NC>
__global__ __launch_bounds__(64 * GW) void split_rows_coop_kernel(SplitParams p, uint64_t *slot,
                                                                  int P, uint32_t want_tag,
                                                                  uint64_t tick_limit,
                                                                  uint32_t *status) {
    constexpr int G = 64 * GW;
    constexpr int NE = 4 * NC;
    constexpr int CHR = NE * G;
    __shared__ float red[2][1][GW];
    __shared__ float fin[2];
    __shared__ int bad;

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t g = blockIdx.x;
    const int member = (int)(g % P);
    const int64_t grow = g / P;
    const Quot at = quot(grow, p.rows);
    const int64_t b = at.q, r = at.r;
    const int64_t kbase = (int64_t)member * CHR;
    const int kleft = (int)(p.K - kbase);    // this chunk's elements inside the row
    const int sleft = (int)(p.Kp - kbase);   // and inside the slice row
    const int64_t xrow = b * p.xs_b + r * p.xs_r + kbase;
    const int64_t srow = b * p.ss_b + r * p.ss_r + kbase;
    float *srow_scale = p.scales + b * p.cs_b + r * p.cs_r;

    if (t == 0) bad = 0;

    // the row's maximum at level l (wave-uniform)
    auto rmax = [&](float m, int l) {
        m = row_max<GW, 1>(m, red, l & 1, 0, t);
        if (P > 1) {
            if (wave == 0) {
                uint64_t *sl = slot + (grow * p.L + l) * (int64_t)P;
                if (lane == 0)
                    __hip_atomic_store(sl + member, kCoopTag | __float_as_uint(m), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                bool seen = lane >= P;
                float q = 0.0f;
                const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
                for (;;) {
                    if (!seen) {
                        const uint64_t w64 =
                            __hip_atomic_load(sl + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if ((uint32_t)(w64 >> 32) == want_tag) {
                            seen = true;
                            q = __uint_as_float((uint32_t)w64);
                        }
                    }
                    if (__all(seen)) break;
                    if (__builtin_amdgcn_s_memrealtime() - t0 >= tick_limit) {
                        if (lane == 0) {
                            bad = 1;
                            __hip_atomic_fetch_or(status, 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
                        }
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                q = wave_max(q);
                if (lane == 0) fin[l & 1] = q;
            }
            lds_barrier();
            m = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fin[l & 1])));
        }
        return m;
    };
    auto store_scale = [&](int l, const LevelScale &c) {
        if (member == 0 && t == 0) srow_scale[l * p.cs_l] = bad ? __int_as_float(0x7fc00000) : c.s;
    };

    if (kleft >= CHR)
        split_row<XT, ST, G, NC, kExact>(p, xrow, srow, 0, 0, false, t, rmax, store_scale);
    else
        split_row<XT, ST, G, NC, kAny>(p, xrow, srow, kleft, sleft, false, t, rmax, store_scale);
}

// ---------------------------------------------------------------------------
// Generic split: one workgroup of 256 lanes per row, any strides, any K, no
// workspace.  Level l sweeps the row twice (maximum, then quantise).  The
// level-l source of an element is recomputed from the input with the scales
// of levels < l, kept in LDS: the same chain of quantisations as the
// reference's residual buffer (ozaki_triton.py:208-211), so the same bits,
// with L(L+1) reads of the input instead of a residual written and re-read.
// ---------------------------------------------------------------------------
template <typename XT, typename ST>
__global__ __launch_bounds__(256) void split_generic_kernel(SplitParams p) {
    __shared__ float red[2][1][4];
    __shared__ LevelScale cs[kMaxLevels];
    const int t = threadIdx.x;
    const int64_t grow = blockIdx.x;
    const int64_t b = grow / p.rows;
    const int64_t r = grow % p.rows;
    const XT *xrow = (const XT *)p.X + b * p.xs_b + r * p.xs_r;
    const int64_t srow = b * p.ss_b + r * p.ss_r;

    // the fp32 residual entering level l >= 1 of input value x
    auto resid = [&](XT x, int l) {
        float rr;
        (void)Quant<ST, Modes<XT>::first>::run(x, cs[0], &rr);
        for (int j = 1; j < l; ++j) (void)Quant<ST, Modes<XT>::rest>::run(rr, cs[j], &rr);
        return rr;
    };
    for (int l = 0; l < p.L; ++l) {
        float m = 0.0f;
        for (int64_t k = t; k < p.K; k += 256) {
            const XT x = xrow[k * p.xs_k];
            m = fmaxf(m, l == 0 ? absf(x) : fabsf(resid(x, l)));
        }
        const LevelScale c = level_scale(row_max<4, 1>(m, red, l & 1, 0, t), p.alpha);
        if (t == 0) {
            cs[l] = c;
            p.scales[b * p.cs_b + l * p.cs_l + r * p.cs_r] = c.s;
        }
        __syncthreads();
        for (int64_t k = t; k < p.Kp; k += 256) {
            const XT x = k < p.K ? xrow[k * p.xs_k] : (XT)0;
            float rr;
            const uint32_t qv = (l == 0) ? Quant<ST, Modes<XT>::first>::run(x, c, &rr)
                                         : Quant<ST, Modes<XT>::rest>::run(resid(x, l), c, &rr);
            store1<ST>(p.slices, srow + l * p.ss_l + k * p.ss_k, k < p.K ? qv : 0u);
        }
    }
}

// ---------------------------------------------------------------------------
// Launches with slices of type ST (declared in ozk_split_launch.h).
// ---------------------------------------------------------------------------
template <typename Kern> static void min_occupancy(Kern kernel, int &occ, bool &ok) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kCoopNT, 0) != hipSuccess ||
        n <= 0) {
        ok = false;
        return;
    }
    occ = n < occ ? n : occ;
}

template <typename ST> void SplitLaunch<ST>::coop_occupancy(int &occ, bool &ok) {
    min_occupancy(split_rows_coop_kernel<double, ST, 4, 8>, occ, ok);
    min_occupancy(split_rows_coop_kernel<float, ST, 4, 16>, occ, ok);
    min_occupancy(split_coop_kernel<double, ST, 32, 8>, occ, ok);
    min_occupancy(split_coop_kernel<double, ST, 32, 2>, occ, ok);
    min_occupancy(split_coop_kernel<float, ST, 16, 8>, occ, ok);
    min_occupancy(split_coop_kernel<float, ST, 16, 2>, occ, ok);
    min_occupancy(split_pair_kernel<double, ST, 32, 4>, occ, ok);
    min_occupancy(split_pair_kernel<double, ST, 32, 8>, occ, ok);
}

template <typename XT, typename ST>
static hipError_t launch_rows_coop(const SplitParams &p, hipStream_t st) {
    const int xsz = (int)sizeof(XT);
    uint64_t *slot = (uint64_t *)p.resid;
    const int64_t P = rows_coop_members(p.K, xsz);
    const int64_t n = rows_coop_slots(p, xsz);
    uint32_t *status = nullptr;
    if (P > 1) {
        if (hipError_t e = clear_slots(slot, n, st)) return e;
        status = (uint32_t *)(slot + n);
    }
    const WaitRule w = wait_rule();
    const dim3 grid((unsigned)(p.batch * p.rows * P)), block(256);
    if constexpr (sizeof(XT) == 8)
        hipLaunchKernelGGL((split_rows_coop_kernel<XT, ST, 4, 8>), grid, block, 0, st, p, slot,
                           (int)P, w.tag, w.ticks, status);
    else
        hipLaunchKernelGGL((split_rows_coop_kernel<XT, ST, 4, 16>), grid, block, 0, st, p, slot,
                           (int)P, w.tag, w.ticks, status);
    if (hipError_t e = hipGetLastError()) return e;
    return P > 1 ? launch_poison(p, slot + n, st) : hipSuccess;
}

template <typename XT, typename ST>
static hipError_t launch_cols_coop(const SplitParams &p, int seg, hipStream_t st) {
    // seg: 16-byte pieces per row of a column group
    const int64_t sw = seg * (16 / (int)sizeof(XT));
    const int64_t groups = p.batch * ((p.rows + sw - 1) / sw);
    const int64_t P = coop_members(p.K, (int)sizeof(XT), seg);
    uint64_t *slot = nullptr;
    uint32_t *status = nullptr;
    const int64_t n = coop_slots(p, (int)sizeof(XT), seg);
    if (P > 1) {
        slot = (uint64_t *)p.resid;
        if (hipError_t e = clear_slots(slot, n, st)) return e;
        status = (uint32_t *)(slot + n);
    }
    const dim3 grid((unsigned)(groups * P)), block(kCoopNT);
    constexpr int RPL = 64 / (16 / (int)sizeof(XT));
    const WaitRule w = wait_rule();
    if (seg == 8)
        hipLaunchKernelGGL((split_coop_kernel<XT, ST, RPL, 8>), grid, block, 0, st, p, slot,
                           (int)P, w.tag, w.ticks, status);
    else if (seg == 2)
        hipLaunchKernelGGL((split_coop_kernel<XT, ST, RPL, 2>), grid, block, 0, st, p, slot,
                           (int)P, w.tag, w.ticks, status);
    else
        return hipErrorInvalidValue;
    if (hipError_t e = hipGetLastError()) return e;
    return P > 1 ? launch_poison(p, slot + n, st) : hipSuccess;
}

// The form an operand allows: cap, the K a workgroup's lanes hold exactly; n, the
// rows or columns of a workgroup; vec, the columns of a lane.
static int split_form(const SplitParams &p, bool cols, int64_t cap, int64_t n, int64_t vec) {
    const int64_t total = cols ? p.rows : p.batch * p.rows;
    if (p.K == cap && total % n == 0) return kExact;
    return p.K % 4 == 0 && p.Kp % 4 == 0 && (!cols || p.rows % vec == 0) ? kWhole : kAny;
}
// f(integral constant) for a form
template <typename F> static void with_form(int form, F &&f) {
    if (form == kExact) f(std::integral_constant<int, kExact>{});
    else if (form == kWhole) f(std::integral_constant<int, kWhole>{});
    else f(std::integral_constant<int, kAny>{});
}

// rows and columns longer than the fused kernel takes (variants 6 on)
template <typename XT, typename ST, int GW, int NC>
static void launch_long_rows(const SplitParams &p, hipStream_t st) {
    with_form(split_form(p, false, 4 * NC * 64 * GW, 1, 1), [&](auto form) {
        hipLaunchKernelGGL((split_rows_kernel<XT, ST, GW, 1, NC, decltype(form)::value>),
                           dim3((unsigned)(p.batch * p.rows)), dim3(64 * GW), 0, st, p);
    });
}
template <typename XT, typename ST, int NT, int NQ>
static void launch_long_cols(const SplitParams &p, hipStream_t st) {
    constexpr int VEC = In<XT>::VEC;
    with_form(split_form(p, true, 4 * NQ * NT, VEC, VEC), [&](auto form) {
        hipLaunchKernelGGL((split_cols_kernel<XT, ST, NT, 1, NQ, decltype(form)::value>),
                           dim3((unsigned)(p.batch * ((p.rows + VEC - 1) / VEC))), dim3(NT), 0, st, p);
    });
}
template <typename XT, typename ST>
static hipError_t launch_long(const SplitParams &p, const SplitPlan &plan, hipStream_t st) {
    constexpr bool F32 = sizeof(XT) == 4;
    if (plan.path == kSplitRows && plan.variant == 6) launch_long_rows<XT, ST, 8, 8>(p, st);
    else if (plan.path == kSplitRows && plan.variant == 7) launch_long_rows<XT, ST, 16, 8>(p, st);
    else if (plan.path == kSplitRows && plan.variant == 8) {
        if constexpr (F32) launch_long_rows<XT, ST, 16, 16>(p, st);
        else return hipErrorInvalidValue;
    } else if (plan.path == kSplitStrip && plan.variant == 6) {
        launch_long_cols<XT, ST, F32 ? 1024 : 512, F32 ? 4 : 8>(p, st);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// split_fused_kernel's configurations <NT, GW, NC, SEG, NQ> by class of K
// (<= 256 << cls) and kind: rows only, narrow column groups or wide ones.  A
// 16-byte piece of a row costs a whole 128-byte line between L2 and the CU, so
// wider pieces win wherever their fewer, larger groups still fill the chip;
// groups that hold more rows a lane would leave the rows' workgroups of the
// same launch two waves a SIMD (<512,4,4,4,8> at K = 4096: 34 us against 39
// where B is 16 times A, 60 against 50 where they are alike).  Columns alone,
// us, N columns, f64 into 4 int8 / f32 into 2 fp16 slices (in brackets the
// 256- or 512-lane 16-byte strips of before this kernel):
//   K =  256 <256,4,1>  N = 1024  4.8 / 4.3   8192  9.4 / 5.9 [13.2 / 7.8]
//   K =  512 <256,2,1>  N = 1024  5.9 / 4.3   8192 14.5 / 10.1 [20.2 / 12.9]
//   K = 1024 <256,2,2>  N = 1024  6.7 / 5.3   8192 33.1 / 15.5 [39.5 / 19.1]
//     wide   <256,4,4>  (f64)                 8192 29.8
//   K = 2048 <256,2,4>  N = 1024 10.4 / 7.3   8192 57.9 / 39.9 [71.6 / 46.5]
//     wide   <512,4,4>  (f64)  4096 30.7 (narrow 36.2)
//   K = 4096 <256,1,4>  N =  512 12.1 / 8.9 [14.6 / 10.0]
//     wide   <512,2,4>  N = 2048 35.5 / 15.9   8192 118.8 / 79.5 [152.9 / 96.5]
//   K = 8192 <512,1,4>  N = 2048 73.0 / 51.1 [97.5 / 58.4]
// (<NT, SEG, NQ> here.)  Rows of up to 1024 take a wave each: two waves and their
// exchange a level were 10.9 us against 9.1 for 9000 f32 rows of 704 alone.
// Rows and columns in one launch, narrow / wide: 4096^2 f64 -> 5 int8 115 / 108,
// 4096^2 f32 -> 2 fp16 68 / 66, f64 -> 4 int8 2048 rows and 4096 columns of
// 2048 41.9 / 39.9, 4096 and 4096 of 1024 27.9 / 24.5 (two launches: 120,
// 67, 47, 28).
template <typename XC, typename ST, int NT, int GW, int NC, int SEG, int NQ>
static hipError_t launch_fused_cfg(const FusedSplit &f, int n, hipStream_t st) {
    constexpr int VEC = In<XC>::VEC, SW = SEG > 0 ? SEG * VEC : 1, RPB = NT / (64 * GW);
    constexpr int64_t CAP = 4 * NC * 64 * GW;
    static_assert(SEG == 0 || CAP == 4 * NQ * (NT / (SEG > 0 ? SEG : 1)),
                  "rows and columns of one class");
    auto blocks = [](const SplitParams &p) -> int64_t {
        return p.cols ? p.batch * ((p.rows + SW - 1) / SW) : (p.batch * p.rows + RPB - 1) / RPB;
    };
    int form[2] = {kExact, kExact};   // rows, columns
    bool has_rows = false;
    for (int i = 0; i < n; ++i) {
        const int c = f.op[i].cols != 0;
        const int fi = split_form(f.op[i], c, CAP, c ? SW : RPB, VEC);
        form[c] = fi > form[c] ? fi : form[c];
        has_rows |= !c;
    }
    const int64_t n0 = blocks(f.op[0]);
    const int64_t total = n0 + (n > 1 ? blocks(f.op[1]) : 0);
    // one form for both, but whole rows beside any columns (a ragged pitch of
    // theirs) keep their own
    const int all = form[0] > form[1] ? form[0] : form[1];
    auto launch = [&](auto fm, auto cf) {
        hipLaunchKernelGGL((split_fused_kernel<XC, ST, NT, GW, NC, SEG, NQ, decltype(fm)::value,
                                               decltype(cf)::value>),
                           dim3((unsigned)total), dim3(NT), 0, st, f, (uint32_t)n0);
    };
    if constexpr (SEG > 0) {
        if (has_rows && form[0] != kAny && form[1] == kAny) {
            launch(std::integral_constant<int, kWhole>{}, std::integral_constant<int, kAny>{});
            return hipGetLastError();
        }
    } else if (n == 1) {
        with_form(all, [&](auto fm) {
            hipLaunchKernelGGL((split_rows_kernel<XC, ST, GW, RPB, NC, decltype(fm)::value>),
                               dim3((unsigned)total), dim3(NT), 0, st, f.op[0]);
        });
        return hipGetLastError();
    }
    with_form(all, [&](auto fm) { launch(fm, fm); });
    return hipGetLastError();
}
template <typename XC, typename ST>
static hipError_t launch_fused_x(const FusedSplit &f, int n, int cls, int width, hipStream_t st) {
    constexpr bool F64 = std::is_same<XC, double>::value;
#define OZK_FUSED(NT, GW, NC, SEG, NQ) return launch_fused_cfg<XC, ST, NT, GW, NC, SEG, NQ>(f, n, st)
    switch (3 * cls + width) {
    case 0: OZK_FUSED(256, 1, 1, 0, 0);
    case 1: OZK_FUSED(256, 1, 1, 4, 1);
    case 3: OZK_FUSED(256, 1, 2, 0, 0);
    case 4: OZK_FUSED(256, 1, 2, 2, 1);
    case 6: OZK_FUSED(256, 1, 4, 0, 0);
    case 7: OZK_FUSED(256, 1, 4, 2, 2);
    case 9: OZK_FUSED(256, 4, 2, 0, 0);
    case 10: OZK_FUSED(256, 4, 2, 2, 4);
    case 12: OZK_FUSED(256, 4, 4, 0, 0);
    case 13: OZK_FUSED(256, 4, 4, 1, 4);
    case 14: OZK_FUSED(512, 4, 4, 2, 4);
    case 15: OZK_FUSED(256, 4, 8, 0, 0);
    case 16: OZK_FUSED(512, 4, 8, 1, 4);
    }
    if constexpr (F64) {
        switch (3 * cls + width) {
        case 8: OZK_FUSED(256, 1, 4, 4, 4);
        case 11: OZK_FUSED(512, 4, 2, 4, 4);
        }
    }
#undef OZK_FUSED
    return hipErrorInvalidValue;
}

template <typename ST>
hipError_t SplitLaunch<ST>::fused(const SplitParams *p0, const SplitParams *p1, int cls, int width,
                                  int x_dtype, hipStream_t st) {
    FusedSplit f;
    const bool swap = p1 && !p0->cols && p1->cols;   // columns first
    f.op[0] = swap ? *p1 : *p0;
    f.op[1] = p1 && !swap ? *p1 : *p0;
    const int n = p1 ? 2 : 1;
    if (x_dtype == 0) return launch_fused_x<double, ST>(f, n, cls, width, st);
    if (x_dtype == 1) return launch_fused_x<float, ST>(f, n, cls, width, st);
    return launch_fused_x<NarrowIn, ST>(f, n, cls, width, st);
}

template <typename XT, typename ST>
static hipError_t launch_one(const SplitParams &p, const SplitPlan &plan, hipStream_t st) {
    if (plan.path == kSplitRows && plan.variant == kRowsCoopVariant)
        return launch_rows_coop<XT, ST>(p, st);
    if (plan.path == kSplitCoop) return launch_cols_coop<XT, ST>(p, plan.variant, st);
    if (plan.path == kSplitRows || plan.path == kSplitStrip) return launch_long<XT, ST>(p, plan, st);
    hipLaunchKernelGGL((split_generic_kernel<XT, ST>), dim3((unsigned)(p.batch * p.rows)),
                       dim3(256), 0, st, p);
    return hipGetLastError();
}
template <typename ST>
hipError_t SplitLaunch<ST>::one(const SplitParams &p, const SplitPlan &plan, int x_dtype,
                                hipStream_t st) {
    return x_dtype == 0 ? launch_one<double, ST>(p, plan, st) : launch_one<float, ST>(p, plan, st);
}

template <typename ST>
hipError_t SplitLaunch<ST>::pair(const SplitParams &pa, const SplitPlan &plan_a,
                                 const SplitParams &pb, hipStream_t st) {
    using XT = double;
    constexpr int RPL = 64 / (16 / (int)sizeof(XT));
    const int64_t sw = 8 * (16 / (int)sizeof(XT));
    const int64_t groups = pb.batch * ((pb.rows + sw - 1) / sw);
    const int64_t P = coop_members(pb.K, (int)sizeof(XT), 8);
    const int64_t n = coop_slots(pb, (int)sizeof(XT), 8);
    uint64_t *slot = nullptr;
    uint32_t *status = nullptr;
    if (P > 1) {
        slot = (uint64_t *)pb.resid;
        if (hipError_t e = clear_slots(slot, n, st)) return e;
        status = (uint32_t *)(slot + n);
    }
    const int64_t na = pa.batch * pa.rows;
    const int64_t ka = groups > 0 ? (na + groups - 1) / groups : 0;
    const dim3 grid((unsigned)(groups * (P + ka))), block(kCoopNT);
    const WaitRule w = wait_rule();
    if (pair_nc(plan_a) == 4)
        hipLaunchKernelGGL((split_pair_kernel<XT, ST, RPL, 4>), grid, block, 0, st, pb, slot,
                           (int)P, w.tag, w.ticks, status, pa, (int)ka);
    else
        hipLaunchKernelGGL((split_pair_kernel<XT, ST, RPL, 8>), grid, block, 0, st, pb, slot,
                           (int)P, w.tag, w.ticks, status, pa, (int)ka);
    if (hipError_t e = hipGetLastError()) return e;
    return P > 1 ? launch_poison(pb, slot + n, st) : hipSuccess;
}

}  // namespace ozk
