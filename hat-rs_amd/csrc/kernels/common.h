// Shared device helpers for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "../kargs.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define HAT_LOG2E 1.4426950408889634f

// v_mfma_f32_16x16x4_f32: A 16x4 (lane l: row l%16, k l/16), B 4x16 (lane l:
// k l/16, col l%16), D 16x16 (lane l, reg r: row 4*(l/16)+r, col l%16).
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// v_mfma_f32_32x32x2_f32: A 32x2 (lane l: row l%32, k l/32), B 2x32 (lane l:
// k l/32, col l%32), D 32x32 (lane l, reg r: row 8*(r/4)+4*(l/32)+r%4, col l%32).
__device__ __forceinline__ f32x16 mfma32(float a, float b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// ---- split-bf16 arithmetic (the BF16 MFMA path at fp32 accuracy, conv_last's): an
// fp32 operand as three bf16 parts, a product as the six terms of order <= 2; what
// is dropped is below 2^-24 of the product.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// (a, b) rounded to nearest bf16, packed: a in the low half (element 0).
__device__ __forceinline__ unsigned pk_bf16(float a, float b)
{
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// The three-way split of a pair: (a, b) = p0 + p1 + p2 (+ below 2^-27 of
// each), every part a packed pair of bf16, each the round-to-nearest of what
// the earlier parts leave (x - its rounding is exact in fp32).
__device__ __forceinline__ void split3_pk(float a, float b, unsigned& p0, unsigned& p1, unsigned& p2)
{
    p0 = pk_bf16(a, b);
    a -= __uint_as_float(p0 << 16);
    b -= __uint_as_float(p0 & 0xffff0000u);
    p1 = pk_bf16(a, b);
    a -= __uint_as_float(p1 << 16);
    b -= __uint_as_float(p1 & 0xffff0000u);
    p2 = pk_bf16(a, b);
}

// Eight consecutive fp32 values as three 8-wide bf16 parts.
__device__ __forceinline__ void split3_x8(const float (&v)[8], u32x4 (&out)[3])
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        unsigned p0, p1, p2;
        split3_pk(v[2 * j], v[2 * j + 1], p0, p1, p2);
        out[0][j] = p0;
        out[1][j] = p1;
        out[2][j] = p2;
    }
}

// v_mfma_f32_16x16x32_bf16: A 16x32 (lane l: row l%16, k 8*(l/16) .. +7), B
// 32x16 (lane l: k 8*(l/16) .. +7, col l%16), D as mfma16's.
__device__ __forceinline__ f32x4 mfma16_bf16(u32x4 a, u32x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16x6(const u32x4 (&a)[3], const u32x4 (&b)[3], f32x4 c)
{
    c = mfma16_bf16(a[2], b[0], c);
    c = mfma16_bf16(a[1], b[1], c);
    c = mfma16_bf16(a[0], b[2], c);
    c = mfma16_bf16(a[1], b[0], c);
    c = mfma16_bf16(a[0], b[1], c);
    return mfma16_bf16(a[0], b[0], c);
}

// ---- split-f16 arithmetic (the F16 MFMA path at fp32 accuracy): an fp32
// operand x as two f16 parts, x = x0 + x1 + e, x0 the round-to-nearest f16 of x
// and x1 of what x0 leaves (exact in fp32), so |e| <= 2^-22 |x| while x1 is a
// normal number and 2^-25 absolute below that (F16 MFMA takes subnormals as they
// are); a product as a0 b0 + a0 b1 + a1 b0 (the term dropped is below 2^-22
// |ab|), three MFMAs where the three-part bf16 split takes six. The operands
// must lie inside f16's range, so the host scales every weight matrix, and the
// activations it can bound, by powers of two (exact) and takes the scale out
// after the accumulation. Measured against a double reference (N(0,1)
// activations, N(0,0.02) weights scaled to 2^14, rms of the error over the rms
// of the result): K = 144 1.45e-7 (six-product bf16: 1.64e-7, FP32 MFMA
// 2.14e-7), K = 180 1.61e-7 (1.91e-7, 2.40e-7), K = 288 1.95e-7 (2.46e-7,
// 3.01e-7): half the accumulator roundings outweigh the wider split. Only very
// short products are less exact (K = 24: 9.0e-8 against 3.5e-8, FP32 MFMA
// 9.0e-8).
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// (a, b) = p0 + p1 (+ e), each part a packed pair of f16 (a in the low half):
// two v_cvt_pk_f16_f32 and two v_fma_mix_f32, 2 instructions a value.
__device__ __forceinline__ void split2_pk(float a, float b, unsigned& p0, unsigned& p1)
{
    const f16x2 h = __builtin_convertvector((f32x2){a, b}, f16x2);
    const float ra = __builtin_fmaf((float)h[0], -1.0f, a), rb = __builtin_fmaf((float)h[1], -1.0f, b);
    p0 = __builtin_bit_cast(unsigned, h);
    p1 = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){ra, rb}, f16x2));
}

// Eight consecutive fp32 values as two 8-wide f16 parts.
__device__ __forceinline__ void split2_x8(const float (&v)[8], u32x4 (&out)[2])
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        unsigned p0, p1;
        split2_pk(v[2 * j], v[2 * j + 1], p0, p1);
        out[0][j] = p0;
        out[1][j] = p1;
    }
}

// v_mfma_f32_16x16x32_f16 (the layout of mfma16_bf16).
__device__ __forceinline__ f32x4 mfma16_f16(u32x4 a, u32x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

__device__ __forceinline__ f32x4 mfma16x3h(const u32x4 (&a)[2], const u32x4 (&b)[2], f32x4 c)
{
    c = mfma16_f16(a[1], b[0], c);
    c = mfma16_f16(a[0], b[1], c);
    return mfma16_f16(a[0], b[0], c);
}

// The packed last k-step of a K = 144 linear (the host's split2_half_step): lane
// group lg's slots j < 4 and 4 + j both hold channel 128 + 4 lg + j, the weight
// planes (a0 | a0) and (a1 | a1), the activation operand (b0 | b1): two MFMAs
// give the three products (and a1 b1) that three give for a whole step.
__device__ __forceinline__ u32x4 half_operand(const f32x4& v)
{
    unsigned p0a, p1a, p0b, p1b;
    split2_pk(v[0], v[1], p0a, p1a);
    split2_pk(v[2], v[3], p0b, p1b);
    return (u32x4){p0a, p0b, p1a, p1b};
}

__device__ __forceinline__ f32x4 mfma16x2h(const u32x4 (&a)[2], const u32x4& b, f32x4 c)
{
    c = mfma16_f16(a[1], b, c);
    return mfma16_f16(a[0], b, c);
}

// v_mfma_f32_32x32x16_f16 (the layout of mfma_bf16).
__device__ __forceinline__ f32x16 mfma_f16(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

__device__ __forceinline__ f32x16 mfma3(const u32x4 (&a)[2], const u32x4 (&b)[2], f32x16 c)
{
    c = mfma_f16(a[1], b[0], c);
    c = mfma_f16(a[0], b[1], c);
    return mfma_f16(a[0], b[0], c);
}

// ---- weight steps for the split-f16 linears: one 32-k step of up to 192 rows
// as two f16 planes [rows][32] with swizzled k-groups (ws_mma2), packed on the
// host.

// The NL loads (1 KB each) of one stage into an LDS buffer, NL / WAVES from
// every wave: wave w issues loads w, w + WAVES, ...; lane l of a load writes
// 16 bytes at the load's LDS base + 16 l. Straight-line code: as a loop, the
// per-load scalar bookkeeping (M0, the address, the counter and the branch)
// cost the tails 1-4% (same-box timings). The compiler's waits stay where
// they were: the callers wait for the copies explicitly before reading a
// buffer.
template <int NL, int WAVES>
__device__ __forceinline__ void wc_issue(unsigned short* dst, const unsigned short* src, int wave, int lane)
{
    static_assert(NL % WAVES == 0, "whole loads per wave");
    const unsigned loff = (unsigned)lane * 16;  // the lane's bytes within a load: one VGPR for every load
#pragma unroll
    for (int j = 0; j < NL / WAVES; ++j) {
        const int i = wave + j * WAVES;  // wave-uniform: the load's base goes in scalar registers
        const char* base = (const char*)src + (size_t)i * 1024;
        __builtin_amdgcn_global_load_lds((const void*)(base + loff),
                                         (__attribute__((address_space(3))) void*)(dst + i * 512), 16, 0, 0);
    }
}

// acc[mt][nt] += W[rows 16 nt .. +15] . xb[mt] for one step in the swizzled
// layout of the weight-stationary kernels: two planes [ROWS][32] (plane stride
// ROWS * 32), row r's four 16-byte k-groups g stored at slot ws_slot(r, g), so
// that the fragment reads down the rows at one k-group are free of bank
// conflicts without padding. HALF: the packed last step of a K = 144 linear
// (xb[mt][0] from half_operand, two MFMAs a tile).
template <int NT, int ROWS, bool HALF = false, int MT = 2>
__device__ __forceinline__ void ws_mma2(const unsigned short* Ws, int lr, int lg, const u32x4 (&xb)[MT][2],
                                        f32x4 (&acc)[MT][NT])
{
    const unsigned short* wr = Ws + lr * 32 + (hatk::ws_slot(lr, lg) * 8);
    // one tile ahead; with one token tile a wave (half the MFMAs a fragment) two
    constexpr int A = MT == 1 ? 2 : 1;
    u32x4 wa[A + 1][2];
#pragma unroll
    for (int t = 0; t < A && t < NT; ++t)
#pragma unroll
        for (int pl = 0; pl < 2; ++pl) wa[t][pl] = *(const u32x4*)(wr + t * 16 * 32 + pl * ROWS * 32);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        __builtin_amdgcn_sched_barrier(0);
        if (nt + A < NT) {
#pragma unroll
            for (int pl = 0; pl < 2; ++pl)
                wa[(nt + A) % (A + 1)][pl] = *(const u32x4*)(wr + (nt + A) * 16 * 32 + pl * ROWS * 32);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            acc[mt][nt] = HALF ? mfma16x2h(wa[nt % (A + 1)], xb[mt][0], acc[mt][nt])
                               : mfma16x3h(wa[nt % (A + 1)], xb[mt], acc[mt][nt]);
    }
}

// A compile-time int carried by a value, for generic lambdas: decltype(x)::value.
template <int V> struct CInt {
    static constexpr int value = V;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// GELU(v) = v Phi(v) = max(v, 0) - |v|/2 erfc(a), a = |v|/sqrt2, with erfc(a) =
// t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-a^2), t = 1/(1 + p a): the same
// published method (Abramowitz & Stegun 7.1.26, |erf error| <= 1.5e-7) as the
// reference CPU path's erf, arranged for few instructions: the 1/2 folded into
// the coefficients, p/sqrt2 into the reciprocal's argument, exp(-a^2) taken as
// exp2(v^2 * (-log2(e)/2)), the reciprocal by v_rcp_f32 (1 ulp). 11 VALU + 2
// transcendental ops; within 3.4e-7 of the exact GELU over [-12, 12] in fp32.
__device__ __forceinline__ float gelu(float v)
{
    const float av = fabsf(v);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f * 0.70710678f, av, 1.0f));
    float q = __builtin_fmaf(0.5f * 1.061405429f, t, 0.5f * -1.453152027f);
    q = __builtin_fmaf(q, t, 0.5f * 1.421413741f);
    q = __builtin_fmaf(q, t, 0.5f * -0.284496736f);
    q = __builtin_fmaf(q, t, 0.5f * 0.254829592f);
    const float e = fast_exp2((v * v) * (-0.5f * HAT_LOG2E));
    return __builtin_fmaf(-av, (q * t) * e, fmaxf(v, 0.0f));
}

// s GELU(v) from V = s v for a power of two s > 0: gelu's form with s in its
// constants, g0 = 0.3275911 / (sqrt2 s), g1 = -log2(e) / (2 s^2).
__device__ __forceinline__ float gelu_scaled(float V, float g0, float g1)
{
    const float av = fabsf(V);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(g0, av, 1.0f));
    float q = __builtin_fmaf(0.5f * 1.061405429f, t, 0.5f * -1.453152027f);
    q = __builtin_fmaf(q, t, 0.5f * 1.421413741f);
    q = __builtin_fmaf(q, t, 0.5f * -0.284496736f);
    q = __builtin_fmaf(q, t, 0.5f * 0.254829592f);
    const float e = fast_exp2((V * V) * g1);
    return __builtin_fmaf(-av, (q * t) * e, fmaxf(V, 0.0f));
}

// 1 KB of zeros in global memory, never written (and not const, so the
// compiler cannot fold loads from it). Loads that fall outside an operand -
// rows past M, padding channels, taps outside the plane, padding slots of the
// weight chunks - read here. The alternatives cost more: a branch around the
// load makes the number of loads in flight path-dependent, so the compiler's
// later waits drain every load; zeroing the value after the load makes it wait
// for that load at once.
__device__ __attribute__((aligned(16))) float hat_zero_row[256] = {};

// Where stores of rows past the end of an output go, so that a wave issues
// the same number of stores whatever the row count (never read).
__device__ __attribute__((aligned(16))) float hat_sink_row[64];

// s_waitcnt for "at most n vector memory operations of this wave still
// outstanding, and every LDS operation done" (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14, expcnt 6:4 left at its maximum, lgkmcnt 11:8 = 0). Vector
// memory operations complete in issue order for this count (the compiler's
// own waits rely on it), so waiting for an operation means waiting until no
// more than the number issued after it are outstanding.
constexpr int wc_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | 0x70; }

// A workgroup barrier for LDS data only: this wave's LDS accesses complete,
// then the barrier. __syncthreads() adds a release fence, which on gfx950 waits
// for every outstanding vector memory operation as well - global loads issued
// ahead for later use included. The memory clobber keeps the compiler from
// moving memory accesses across it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A float4 from p, or zeros (from hat_zero_row) where ok is false.
__device__ __forceinline__ f32x4 load_or_zero(const float* p, bool ok)
{
    return *(const f32x4*)(ok ? p : hat_zero_row);
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// max(m, |v|), infinities and NaN left out.
__device__ __forceinline__ float finite_max(float m, float v)
{
    const float a = fabsf(v);
    return a <= 3.402823466e38f ? fmaxf(m, a) : m;
}

// A plane's largest magnitude (kargs.h AMAX_LANES): the block's, by an LDS maximum
// over its waves and one atomic into the lane of its XCD, blockIdx.x & 7. (An atomic a
// wave into one word took 70 us of the 64-channel conv at 512 x 512.) The bits of
// non-negative floats order as unsigned integers do, and a maximum does not depend
// on the order. lds: zeroed before an earlier barrier; every thread of the block
// calls this.
__device__ __forceinline__ void block_amax(unsigned* out, unsigned* lds, float m)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(lds, __float_as_uint(m));
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(out + (blockIdx.x % AMAX_LANES) * AMAX_STRIDE, *lds);
}

// The magnitude (its bits) that block_amax left.
__device__ __forceinline__ unsigned read_amax(const unsigned* p)
{
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < AMAX_LANES; ++i) m = max(m, p[i * AMAX_STRIDE]);
    return m;
}

// The wave's sum in registers alone (DPP, no LDS round trips), wave-uniform:
// pairs, quads, 8 (half-row mirror), 16 (row mirror), then row 0 into row 1
// and row 2 into row 3 (row_bcast:15), rows 0-1 into row 3 (row_bcast:31);
// lane 63 ends with the total. A fixed order, so the result does not depend on
// timing.
__device__ __forceinline__ float wave_sum_dpp(float v)
{
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xb1, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4e, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
