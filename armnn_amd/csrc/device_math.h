// Device-side arithmetic shared by every kernel: the requantization epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "common.h"

namespace mi355x
{

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// float value -> output code, exactly armnn::Quantize (src/armnn/TypesUtils.cpp:29-45):
//   clamp(float(offset) + round(value / scale), lowest, max), round = half away from zero, fp32 division,
// followed by the fused activation's integer clamp.
__device__ __forceinline__ int QuantizeDev(float f, const Requant& rq)
{
    float q = roundf(__fdiv_rn(f, rq.out_scale));
    float v = __fadd_rn(rq.out_offset_f, q);
    v = fmaxf(v, rq.type_min_f);
    v = fminf(v, rq.type_max_f);
    int r = static_cast<int>(v);
    r = max(r, rq.act_lo);
    r = min(r, rq.act_hi);
    return r;
}

// int32 accumulator of sum (x - zx)(w - zw) -> output code, the reference's way:
//   f = float(acc) * (s_in * s_w[c]) + float(bias[c]) * s_b[c]      (separate multiply and add, no FMA)
// `mult` and `biasf` are prepared on the host in fp32 exactly as the reference's decoders would produce them.
__device__ __forceinline__ int RequantExactDev(int acc, float mult, float biasf, const Requant& rq)
{
    return QuantizeDev(__fadd_rn(__fmul_rn(static_cast<float>(acc), mult), biasf), rq);
}

// Per-channel constants, four rows of `stride` floats, built on the host (bracket.h):
//   row 0 mult   s_in * s_w[c]                      row 1 biasf  float(bias[c]) * s_b[c]
//   row 2 m, row 3 b   the fast path (below)
// A kernel's accumulators start from the plan's `corr` array (or get it added before the requantization): the zero-point
// correction of a sum of raw products, raised by Requant::acc_base.
struct ChanTab
{
    const float* p;
    int stride;
};

// The first BYTES of the kernel's arguments come to the scalar cache in one round trip.  The compiler loads an argument where it is first
// used, and a launch finds that cache empty: one line of 64 bytes after the other, each waited for ahead of the loads of tensors behind
// it.  Passes, three networks in turn: ResNet-50 at one image 115.5 -> 112.8 us (alone 310 -> 297), at 32 images 412 -> 403.6, MobileNetV1 at one
// image 35.7 -> 34.8 (alone 113 -> 107), at 64 the same; launches, three sets of tensors in turn: FullyConnected 4096 -> 4096 of one row 4.48 -> 4.30,
// 3 x 3 over 64 x 56 x 56 x 64 14.09 -> 13.86, 1 x 1 over 32 x 28 x 28 x 128 -> 512 7.69 -> 7.59.  Not in IgemmKernel, whose launches took 0.05 us longer with it.
template <int BYTES>
__device__ __forceinline__ void FetchArgs()
{
    typedef const __attribute__((address_space(4))) int* ArgPtr;
    const ArgPtr args = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int N = (BYTES + 63) / 64;
    static_assert(N >= 1 && N <= 12, "up to 12 lines");
    int v[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) v[i] = args[(i < N ? i : 0) * 16];
    asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]), "s"(v[6]), "s"(v[7]), "s"(v[8]), "s"(v[9]), "s"(v[10]), "s"(v[11]));
}

// four accumulators of a 32 x 32 result: channels 8 q + 4 (lane / 32) + 0 .. 3
__device__ __forceinline__ v4i Quad(const v16i& v, int q)
{
    return v4i{v[4 * q + 0], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
}

// Fast path with an exact fallback.
//   t = float(acc) * mult / s_out + biasf / s_out + offset' is the reference's value before rounding, with its roundings (offset': 128
//   higher for signed outputs, codes as unsigned bytes).  The fast path works on a scale on which v_cvt_pknorm_u16_f32 (two values
//   per instruction: rint(65535 x), saturated to 0 .. 65535 -- exactly, for every float: peaks.hip has the check) leaves the code in
//   the high byte of its 16 bits,
//       65535 x = 256 (t + 0.5) - 0.5,
//   so that x crosses from one high byte to the next where t is a half-integer.  The host chooses c above every rounding on both
//   sides (the reference's four; those of m, b, the conversion, the fma and the subtraction: bracket.h has the sum), so that
//       p = fma(float(acc), m, b)  and  q = p - 2c     enclose the reference's x:   q < x(t) < p.
//   When both give the same high byte, t -- strictly between them -- rounds to that code under any tie rule, the reference's
//   half-away-from-zero included.  Values whose two bytes differ (about two in 10^4) are recomputed with the reference's own
//   sequence.  A channel without a fast path has m = 0 and a b on a byte's edge, so that its bytes always differ.
//   Where Requant::acc_base is not zero, accumulators run that much higher than the sums, and their bits are the float 1.5 * 2^23 +
//   sum: one subtraction instead of a conversion.  That is exact up to 2^22; beyond, the steps are larger or smaller than one,
//   but still in order, and the host has checked that no sum gets there or that all codes are saturated.  (Not so in a
//   4096-wide FullyConnected with small scales.)
//   What instructions cost here was measured pair by pair: conversions, permutes and packed integers take a SIMD four cycles a wave,
//   float additions two, and fma and additions issue beside the conversions of another wave.  Four values: 4 subtract, 4 fma, 4
//   subtract, 4 conversions, 2 permutes, xor, compare -- where the form before (v_cvt_f32_i32, one fma and one
//   v_cvt_pk_u8_f32 per side) had 12 conversions.  A loop of little else: 10.8 against 7.9 T values/s on the whole device, 9.3
//   with the accumulators converted.
//   Passes (RequantCore's batches included): MobileNetV1 at 64 images 177.3 -> 170.2 us, at 256 647.8 -> 615.1, ResNet-50 at 32 459.6 ->
//   454.0, FullyConnected 8192 x 4096 x 4096 130.3 -> 125.1, depthwise 64 x 112 x 112 x 32 15.3 -> 14.4.
//   The activation's clamp, where it is narrower than 0..255, is applied to the codes.

// Stores of layer outputs.  An ordinary store leaves its line dirty in the XCD's L2 until the end-of-kernel write-back,
// which then moves the whole output tensor (up to the 32 MB the eight L2s hold) after the last wave has finished, with
// nothing to overlap it.  With the sc1 bit (agent scope) the L2 writes the line through as the store is issued, so the
// write-back runs beside the rest of the kernel and the data is where the next kernel -- whose blocks run on any XCD --
// reads it from.  (The nt bit instead also helps a kernel timed alone but makes the next layer slower.)  Only for stores
// of 16 bytes per lane that cover whole lines per instruction: the depthwise blocks' and the pooling kernel's dwords,
// written through one by one, are slower than ordinary stores that L2 merges.
//   The bit is set through the buffer-store builtins (their cache-policy argument), which the compiler knows as vector
// memory instructions; a hand-written store instruction in inline assembly is invisible to its hazard and wait-count
// bookkeeping and produced wrong bytes now and then.  A buffer store takes a wave-uniform base and an unsigned 32-bit
// byte offset, so tensors of 4 GiB and more fall back to ordinary stores.
#ifndef MI355X_STORE_THROUGH
#define MI355X_STORE_THROUGH 1
#endif
typedef int StoreVec4 __attribute__((ext_vector_type(4)));

struct OutPtr
{
    __amdgpu_buffer_rsrc_t rsrc;
    uint8_t* base;
    bool through;
};

// `base` must be the same in every lane of the wave (a kernel argument, or derived from block-uniform values)
__device__ __forceinline__ OutPtr MakeOutPtr(uint8_t* base, long long bytes)
{
    OutPtr o;
    o.base = base;
    o.through = MI355X_STORE_THROUGH != 0 && bytes > 0 && bytes <= 0xffffffffll;
    o.rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, -1, 0x00020000);
    return o;
}

constexpr int kStoreAuxSc1 = 16;     // cache-policy operand of the buffer-store builtins: bit 4 = sc1

__device__ __forceinline__ void StoreOut16(const OutPtr& o, long long offset, const StoreVec4& v)
{
    typedef unsigned int U4 __attribute__((ext_vector_type(4)));
    if (o.through) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), o.rsrc, static_cast<int>(offset), 0, kStoreAuxSc1);
    else *reinterpret_cast<StoreVec4*>(o.base + offset) = v;
}

__device__ __forceinline__ uint32_t Pack4(int q0, int q1, int q2, int q3)
{
    // four codes -> one dword (byte 0 = q0), three v_perm_b32
    const uint32_t t0 = __builtin_amdgcn_perm(static_cast<uint32_t>(q1), static_cast<uint32_t>(q0), 0x0c0c0400u);
    const uint32_t t1 = __builtin_amdgcn_perm(static_cast<uint32_t>(q3), static_cast<uint32_t>(q2), 0x0c0c0400u);
    return __builtin_amdgcn_perm(t1, t0, 0x05040100u);
}

struct Fast4
{
    float4 m, b;   // rows 2 and 3 (the rare exact path fetches rows 0 and 1 when it is entered)
};

__device__ __forceinline__ Fast4 LoadFast4(const ChanTab& ct, int c)
{
    Fast4 f;
    f.m = *reinterpret_cast<const float4*>(ct.p + 2 * ct.stride + c);
    f.b = *reinterpret_cast<const float4*>(ct.p + 3 * ct.stride + c);
    return f;
}

// The sum in an accumulator as a float; BITS: Requant::acc_base is not zero.
template <bool BITS>
__device__ __forceinline__ float AccValue(int acc)
{
    if constexpr (BITS) return __fsub_rn(__builtin_bit_cast(float, acc), kAccBaseValue);
    else return static_cast<float>(acc);
}

// Which of codes k - 1 and k (unsigned bytes, before the activation's clamp) a value has that the bracket puts into one of them; k
// when `open` is 0.
//   f is the reference's fp32 value, h = k - 0.5 - offset' the half-integer in question.  fl(f / s_out) >= h exactly if f / s_out >= h -
//   d with d half the distance from |h| to the float below it (h - d is a tie that rounds to h, whose mantissa is even), and
//   fl(f / s_out) > h for negative h exactly if f / s_out > h + d; rounding half away from zero asks for the first where h is
//   positive, for the second where it is negative.  f - h s_out has few bits and is exact in the fma, d s_out is a shift: the
//   division's result is known without the division.
//   Against the division in its place, MobileNetV1 at one image 35.4 against 35.8 us, at 64 155.5 against 156.3, at 256 544 against 542; the 3x3
//   layer 64 x 56 x 56 x 64 14.1 against 13.9.  (A bracket whose width bounds the constants' roundings instead of taking them as
//   they are, 35.7, 156.8, 547 and 14.2.)
__device__ __forceinline__ int SettleDev(float sum, float mult, float biasf, int k, uint32_t open, const Requant& rq)
{
    const float f = __fadd_rn(__fmul_rn(sum, mult), biasf);
    const float h = static_cast<float>(k) - rq.half_offset_f;
    const float r = __fmaf_rn(-h, rq.out_scale, f);
    const uint32_t below = (__builtin_bit_cast(uint32_t, fabsf(h)) - 1u) & 0x7f800000u;         // 2^exponent of the float below |h|
    const float ds = __fmul_rn(__fmul_rn(__builtin_bit_cast(float, below), 0x1p-24f), rq.out_scale);
    const bool up = h > 0.0f ? r >= -ds : r > ds;
    return k - (open != 0u && !up ? 1 : 0);
}

typedef unsigned short U16x2 __attribute__((ext_vector_type(2)));

// the high bytes of four 16-bit values -> one dword
__device__ __forceinline__ uint32_t HighBytes4(U16x2 v01, U16x2 v23)
{
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, v23), __builtin_bit_cast(uint32_t, v01), 0x07050301u);
}

// the activation's clamp, two codes at a time, where it is narrower than 0..255; then signed codes are signed
template <int N>
__device__ __forceinline__ void ClampCodes(uint32_t (&out)[N], const Requant& rq)
{
    if (!rq.pk_full)
    {
        const U16x2 least = __builtin_bit_cast(U16x2, rq.pk_lo2), most = __builtin_bit_cast(U16x2, rq.pk_hi2);
#pragma unroll
        for (int n = 0; n < N; ++n)
        {
            const U16x2 even = __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(U16x2, out[n] & 0x00ff00ffu), least), most);
            const U16x2 odd = __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(U16x2, (out[n] >> 8) & 0x00ff00ffu), least), most);
            out[n] = __builtin_bit_cast(uint32_t, even) | (__builtin_bit_cast(uint32_t, odd) << 8);
        }
    }
#pragma unroll
    for (int n = 0; n < N; ++n) out[n] ^= rq.pk_xor;
}

// N times four values -> N packed dwords; their constants: f[n], or f[0] for all.
// The N are independent chains of arithmetic with one test at their end, so that a wave has all of them to issue from: a test
// per four values is a branch, which the compiler moves nothing across.  Where some lane of the wave has a byte that differs between
// the two sides, values are redone with the reference's sequence; load_exact(n, mult, biasf) supplies rows 0 and 1 of the table for
// that.  It happens to one batch of four in six, and the waves of a block wait for one another soon after: kernels of many
// values have those rows in LDS (from L2, 1.5 k cycles, a pass of MobileNetV1 at 64 images took 5 % longer).  One copy of that code
// serves the batch, each lane choosing among the N (a copy for each of the N: 161.0 against 158.7 us at 64 images, 584 against 572
// at 256; the instructions are cold when they are wanted).  The constants are finite (the host checks them and the accumulator
// range), so no NaN reaches a conversion.
template <bool BITS, int N, int NF, typename LoadExact>
__device__ __forceinline__ void RequantCore(const v4i (&acc)[N], uint32_t (&out)[N], const Fast4 (&f)[NF], const Requant& rq, LoadExact load_exact)
{
    static_assert(NF == 1 || NF == N, "one set of constants, or one each");
    uint32_t differ[N], any = 0u;
#pragma unroll
    for (int n = 0; n < N; ++n)
    {
        const Fast4& c = f[NF == 1 ? 0 : n];
        const float p0 = __fmaf_rn(AccValue<BITS>(acc[n][0]), c.m.x, c.b.x), p1 = __fmaf_rn(AccValue<BITS>(acc[n][1]), c.m.y, c.b.y);
        const float p2 = __fmaf_rn(AccValue<BITS>(acc[n][2]), c.m.z, c.b.z), p3 = __fmaf_rn(AccValue<BITS>(acc[n][3]), c.m.w, c.b.w);
        const U16x2 hi01 = __builtin_amdgcn_cvt_pknorm_u16(p0, p1), hi23 = __builtin_amdgcn_cvt_pknorm_u16(p2, p3);
        const U16x2 lo01 = __builtin_amdgcn_cvt_pknorm_u16(__fsub_rn(p0, rq.two_c), __fsub_rn(p1, rq.two_c));
        const U16x2 lo23 = __builtin_amdgcn_cvt_pknorm_u16(__fsub_rn(p2, rq.two_c), __fsub_rn(p3, rq.two_c));
        out[n] = HighBytes4(hi01, hi23);
        differ[n] = out[n] ^ HighBytes4(lo01, lo23);
        any |= differ[n];
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(any != 0u) != 0, 0))
    {
        constexpr int base = BITS ? kAccBaseBits : 0;
        // every lane redoes its first flagged value (some value where none is: the result is always the right one)
        do
        {
            int s0 = acc[N - 1][0], s1 = acc[N - 1][1], s2 = acc[N - 1][2], s3 = acc[N - 1][3], which = N - 1;
            uint32_t d = differ[N - 1], o = out[N - 1];
#pragma unroll
            for (int n = N - 2; n >= 0; --n)
            {
                const int a0 = acc[n][0], a1 = acc[n][1], a2 = acc[n][2], a3 = acc[n][3];
                const uint32_t dn = differ[n], on = out[n];
                const bool take = dn != 0u;
                s0 = take ? a0 : s0; s1 = take ? a1 : s1; s2 = take ? a2 : s2; s3 = take ? a3 : s3;
                d = take ? dn : d; o = take ? on : o; which = take ? n : which;
            }
            float4 m, b;
            load_exact(which, m, b);
            const bool upper = (d & 0xffffu) == 0u, odd = ((upper ? d >> 16 : d) & 0xffu) == 0u;
            const int sum = upper ? (odd ? s3 : s2) : (odd ? s1 : s0);
            const float mult = upper ? (odd ? m.w : m.z) : (odd ? m.y : m.x), biasf = upper ? (odd ? b.w : b.z) : (odd ? b.y : b.x);
            const int shift = (upper ? 16 : 0) + (odd ? 8 : 0);
            const uint32_t mask = 0xffu << shift;
            // (AccValue, and not the conversion of sum - base, 0.8 us of 120 in FullyConnected 8192 x 4096 x 4096: beyond 2^22, where the bits are
            // not the sum, a value is open only if its channel's slope is so small that neither moves its bias)
            int code = SettleDev(AccValue<BITS>(sum), mult, biasf, static_cast<int>((o >> shift) & 0xffu), d & mask, rq);
            // bytes 128 and 127: a channel without a fast path (or a value between these two codes, which either way settles)
            if (!rq.all_fast && (d & mask) == mask) code = RequantExactDev(sum - base, mult, biasf, rq) + rq.pk_bias;
            o = (o & ~mask) | (static_cast<uint32_t>(code) << shift);
            any = 0u;
#pragma unroll
            for (int n = 0; n < N; ++n)
            {
                out[n] = which == n ? o : out[n];
                differ[n] = which == n ? d & ~mask : differ[n];
                any |= differ[n];
            }
        } while (__builtin_amdgcn_ballot_w64(any != 0u) != 0);
    }
    ClampCodes(out, rq);
}

// N pixels, channels c .. c + 3 of each.  `ct`: the table, or rows 0 and 1 of it (a copy in LDS).
template <bool BITS, int N>
__device__ __forceinline__ void RequantPixels(const v4i (&acc)[N], uint32_t (&out)[N], const Fast4& f, const ChanTab& ct, int c, const Requant& rq)
{
    const Fast4 fs[1] = {f};
    RequantCore<BITS, N, 1>(acc, out, fs, rq, [&](int, float4& m, float4& b) {
        m = *reinterpret_cast<const float4*>(ct.p + c);
        b = *reinterpret_cast<const float4*>(ct.p + ct.stride + c);
    });
}

// one pixel, channels c + STEP n .. c + STEP n + 3
template <bool BITS, int N, int STEP>
__device__ __forceinline__ void RequantChannels(const v4i (&acc)[N], uint32_t (&out)[N], const Fast4 (&f)[N], const ChanTab& ct, int c, const Requant& rq)
{
    RequantCore<BITS, N, N>(acc, out, f, rq, [&](int n, float4& m, float4& b) {
        m = *reinterpret_cast<const float4*>(ct.p + c + STEP * n);
        b = *reinterpret_cast<const float4*>(ct.p + ct.stride + c + STEP * n);
    });
}

// channels c .. c + 3 of one pixel; BITS must say whether Requant::acc_base is not zero (in a 3x3 depthwise plan it never is zero)
template <bool BITS>
__device__ __forceinline__ uint32_t Requant4Dev(int a0, int a1, int a2, int a3, const Fast4& f, const ChanTab& ct, int c, const Requant& rq)
{
    const v4i acc[1] = {{a0, a1, a2, a3}};
    uint32_t out[1];
    RequantPixels<BITS, 1>(acc, out, f, ct, c, rq);
    return out[0];
}

// ... where the kernel is not worth two copies of its write-out
__device__ __forceinline__ uint32_t Requant4Any(int a0, int a1, int a2, int a3, const Fast4& f, const ChanTab& ct, int c, const Requant& rq)
{
    return rq.acc_base != 0 ? Requant4Dev<true>(a0, a1, a2, a3, f, ct, c, rq) : Requant4Dev<false>(a0, a1, a2, a3, f, ct, c, rq);
}

// ... and where it is: `write_out` is called with std::true_type or std::false_type for BITS
template <typename F>
__device__ __forceinline__ void WithBits(const Requant& rq, F write_out)
{
    if (rq.acc_base != 0) write_out(std::true_type{});
    else write_out(std::false_type{});
}

// one channel (scalar kernels): the same bracket.  m, b: rows 2 and 3 of the table at channel c
__device__ __forceinline__ int Requant1Dev(int acc, float m, float b, const ChanTab& ct, int c, const Requant& rq)
{
    const float p = __fmaf_rn(rq.acc_base != 0 ? AccValue<true>(acc) : AccValue<false>(acc), m, b);
    const U16x2 v = __builtin_amdgcn_cvt_pknorm_u16(p, __fsub_rn(p, rq.two_c));
    const int hi = v.x >> 8, lo = v.y >> 8;
    if (__builtin_expect(hi != lo, 0)) return RequantExactDev(acc - rq.acc_base, ct.p[c], ct.p[ct.stride + c], rq);
    return min(max(hi - rq.pk_bias, rq.act_lo), rq.act_hi);
}

__device__ __forceinline__ int Requant1Dev(int acc, const ChanTab& ct, int c, const Requant& rq)
{
    return Requant1Dev(acc, ct.p[2 * ct.stride + c], ct.p[3 * ct.stride + c], ct, c, rq);
}

// value already in float (pooling, add, ...): reciprocal fast path with the exact fallback near ties.
//   r' = fma(f, fl(1/scale), offset) is within 2^-24 * (|f/scale| + |r'|) of f/scale + offset and the correctly rounded
//   quotient within 2^-24 * |f/scale|; |offset| <= 255 is checked on the host (else fast_ok = 0).
__device__ __forceinline__ int QuantizeFastDev(float f, const Requant& rq)
{
    if (!rq.fast_ok) return QuantizeDev(f, rq);
    const float r = __fmaf_rn(f, rq.inv_scale, rq.out_offset_f);
    const float k = __builtin_rintf(r);
    const float e = __fsub_rn(r, k);
    // 3 |r'| + 2 |offset| <= 3 |r'| + 510, with the same 1.5x margin as above
    if (__builtin_expect(!(fabsf(e) <= __fmaf_rn(fabsf(r), -4.5f / 16777216.0f, 0.5f - 1024.0f / 16777216.0f)), 0))
        return QuantizeDev(f, rq);
    return static_cast<int>(__builtin_amdgcn_fmed3f(k, rq.act_lo_f, rq.act_hi_f));
}

// Four float values -> packed dword of output codes: QuantizeFastDev's test per value, then v_cvt_pk_u8_f32 (convert,
// saturate, pack) in the biased domain of Requant::pk_bias.  |offset + pk_bias| <= 383 here, hence the wider constant.
__device__ __forceinline__ uint32_t QuantizePack4Dev(float f0, float f1, float f2, float f3, const Requant& rq)
{
    if (!rq.fast_ok) return Pack4(QuantizeDev(f0, rq), QuantizeDev(f1, rq), QuantizeDev(f2, rq), QuantizeDev(f3, rq));
    const float off = rq.out_offset_f + static_cast<float>(rq.pk_bias);
    const float f[4] = {f0, f1, f2, f3};
    uint32_t out = 0u;
    unsigned slow = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const float r = __fmaf_rn(f[i], rq.inv_scale, off);
        float k = __builtin_rintf(r);
        const float e = __fsub_rn(r, k);
        if (!(fabsf(e) <= __fmaf_rn(fabsf(r), -4.5f / 16777216.0f, 0.5f - 1536.0f / 16777216.0f))) slow |= 1u << i;
        if (!rq.pk_full) k = __builtin_amdgcn_fmed3f(k, rq.pk_lo_f, rq.pk_hi_f);
        out = __builtin_amdgcn_cvt_pk_u8_f32(k, i, out);
    }
    if (__builtin_expect(slow != 0u, 0))
    {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (slow & (1u << i))
                out = (out & ~(0xffu << (8 * i))) | ((static_cast<uint32_t>(QuantizeDev(f[i], rq) + rq.pk_bias) & 0xffu) << (8 * i));
    }
    return out ^ rq.pk_xor;
}

struct QIn
{
    float scale;
    int   offset;
    int   is_u8;
};

__device__ __forceinline__ float DequantDev(uint8_t code, const QIn& q)
{
    const int v = q.is_u8 ? static_cast<int>(code) : static_cast<int>(static_cast<int8_t>(code));
    return __fmul_rn(static_cast<float>(v - q.offset), q.scale);   // armnn::Dequantize, TypesUtils.cpp:47-56
}

// The four codes of a dword -> float values: signed codes are made unsigned with one xor for the dword (offset moves by
// 128 with them), then v_cvt_f32_ubyteN converts byte N directly; value - offset is an exact small integer either way,
// so the single multiplication rounds exactly as in armnn::Dequantize.
__device__ __forceinline__ void Dequant4Dev(uint32_t w, const QIn& q, float (&v)[4])
{
    const uint32_t u = q.is_u8 ? w : (w ^ 0x80808080u);
    const float off = static_cast<float>(q.is_u8 ? q.offset : q.offset + 128);
    v[0] = __fmul_rn(__fsub_rn(static_cast<float>(u & 0xffu), off), q.scale);
    v[1] = __fmul_rn(__fsub_rn(static_cast<float>((u >> 8) & 0xffu), off), q.scale);
    v[2] = __fmul_rn(__fsub_rn(static_cast<float>((u >> 16) & 0xffu), off), q.scale);
    v[3] = __fmul_rn(__fsub_rn(static_cast<float>(u >> 24), off), q.scale);
}

inline QIn MakeQIn(const mi355x_quant& q)
{
    QIn r;
    r.scale = q.scale;
    r.offset = q.offset;
    r.is_u8 = q.dtype == MI355X_QASYMM_U8;
    return r;
}

// An Addition of two quantized tensors: dequantize both, one fp32 add, quantize with the Addition's output quantization and
// its fused activation (RefElementwiseBinaryWorkload.cpp:27-107 over Decoder / Encoder).  Used by the Addition layer's
// kernel and, inside a convolution's write-out, for the Addition that follows the convolution (`own`: the convolution's
// finished output codes with quantization qa, `other`: the Addition's other input with qr) -- so the bytes are those of
// the two layers run apart.
//   The reference's sequence costs 14 vector instructions per value (two dequantizations of three, the add, a quantization
//   with its own tie test).  The value before rounding is, in exact arithmetic, a linear function of the two codes,
//     T = ua ka + ub kb + k0,   ka = sa / so, kb = sr / so, k0 = offset_out + pk_bias - oa ka - or kb   (ua, ub: codes as 0..255),
//   and the reference's own fp32 value P' (its four roundings: two products, the sum, the division) lies within
//   3.01 * 2^-24 * 255 (ka + kb) of T.  As in the requantization above, 65535 x = 256 (T + 0.5) - 0.5 puts the code in the high
//   byte of v_cvt_pknorm_u16_f32's result, and the three constants are scaled to give x: with p = fma(ua, ka', fma(ub, kb', k0' + c'))
//   and q = p - 2c', c above that distance plus the roundings of the constants, of the two FMAs and of the subtraction (for
//   |T| <= 512: 2^-24 (1533 ka + 1278 kb + 2048) in all, relative errors that the scaling leaves alone; c = 1.5 x that), p and q
//   enclose x(P'); beyond |T| = 512 all three saturate alike.  Where both have the same high byte, P' -- strictly between them --
//   rounds to that code under any tie rule.  Otherwise (a few values in 10^4) that value is redone with the reference's sequence.
//   Per value: two byte conversions, two fma, one subtraction, one conversion (two before, which packed one value each and came behind
//   a clamp each), and one test for 16 values instead of four.  ResNet-50 at 32 images, whose Additions are in convolutions'
//   write-outs: 419 -> 411.5 us a pass; the Addition layer over 2 x 12.8 MB with exact ties in 0.5 % of the values: 8.7 -> 7.8 us, with
//   none 6.1 either way (memory).
struct AddFuse
{
    QIn qa, qr;
    Requant rq;
    float ka, kb, k0p, two_c;     // scaled by 256 / 65535
    int bracket_ok;
};

inline AddFuse MakeAddFuse(const mi355x_quant& a, const mi355x_quant& r, const mi355x_quant& out, int32_t activation, float act_a, float act_b)
{
    AddFuse f;
    f.qa = MakeQIn(a);
    f.qr = MakeQIn(r);
    f.rq = MakeRequant(out, activation, act_a, act_b);
    const double so = static_cast<double>(out.scale);
    const double ka = static_cast<double>(a.scale) / so, kb = static_cast<double>(r.scale) / so;
    const double oa = f.qa.is_u8 ? a.offset : a.offset + 128, ob = f.qr.is_u8 ? r.offset : r.offset + 128;
    const double k0 = static_cast<double>(out.offset) + f.rq.pk_bias - oa * ka - ob * kb;
    const double c = 1.5 * (1533.0 * ka + 1278.0 * kb + 2048.0) / 16777216.0;
    constexpr double unit = 256.0 / 65535.0;
    f.ka = static_cast<float>(unit * ka);
    f.kb = static_cast<float>(unit * kb);
    f.k0p = static_cast<float>(unit * (k0 + c) + 127.5 / 65535.0);
    f.two_c = nextafterf(static_cast<float>(2.0 * unit * c), 1.0e30f);
    f.bracket_ok = f.rq.fast_ok && std::isnormal(f.ka) && std::isnormal(f.kb) && ka < 1024.0 && kb < 1024.0 && std::fabs(k0) < 1048576.0 &&
                   oa >= 0.0 && oa <= 255.0 && ob >= 0.0 && ob <= 255.0;     // offsets inside the type's range: |code - offset| <= 255
    return f;
}

// 16 codes of each input -> the 16 sums' codes.  One test for all of them, and one copy of the reference's sequence behind it.
__device__ __forceinline__ StoreVec4 AddQuantize16Dev(const StoreVec4& own, const StoreVec4& other, const AddFuse& f)
{
    uint32_t out[4];
    if (!f.bracket_ok)
    {
#pragma unroll
        for (int n = 0; n < 4; ++n)
        {
            float va[4], vb[4];
            Dequant4Dev(static_cast<uint32_t>(own[n]), f.qa, va);
            Dequant4Dev(static_cast<uint32_t>(other[n]), f.qr, vb);
            out[n] = QuantizePack4Dev(__fadd_rn(va[0], vb[0]), __fadd_rn(va[1], vb[1]), __fadd_rn(va[2], vb[2]), __fadd_rn(va[3], vb[3]), f.rq);
        }
        return StoreVec4{static_cast<int>(out[0]), static_cast<int>(out[1]), static_cast<int>(out[2]), static_cast<int>(out[3])};
    }
    const uint32_t xa = f.qa.is_u8 ? 0u : 0x80808080u, xb = f.qr.is_u8 ? 0u : 0x80808080u;
    uint32_t differ[4], any = 0u;
#pragma unroll
    for (int n = 0; n < 4; ++n)
    {
        const uint32_t ua = static_cast<uint32_t>(own[n]) ^ xa, ub = static_cast<uint32_t>(other[n]) ^ xb;
        const float af[4] = {static_cast<float>(ua & 0xffu), static_cast<float>((ua >> 8) & 0xffu), static_cast<float>((ua >> 16) & 0xffu), static_cast<float>(ua >> 24)};
        const float bf[4] = {static_cast<float>(ub & 0xffu), static_cast<float>((ub >> 8) & 0xffu), static_cast<float>((ub >> 16) & 0xffu), static_cast<float>(ub >> 24)};
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = __fmaf_rn(af[i], f.ka, __fmaf_rn(bf[i], f.kb, f.k0p));
        out[n] = HighBytes4(__builtin_amdgcn_cvt_pknorm_u16(p[0], p[1]), __builtin_amdgcn_cvt_pknorm_u16(p[2], p[3]));
        differ[n] = out[n] ^ HighBytes4(__builtin_amdgcn_cvt_pknorm_u16(__fsub_rn(p[0], f.two_c), __fsub_rn(p[1], f.two_c)),
                                        __builtin_amdgcn_cvt_pknorm_u16(__fsub_rn(p[2], f.two_c), __fsub_rn(p[3], f.two_c)));
        any |= differ[n];
    }
    while (__builtin_expect(__builtin_amdgcn_ballot_w64(any != 0u) != 0, 0))
    {
        // every lane redoes its first flagged value (some value where none is)
        int wa = own[3], wb = other[3], which = 3;
        uint32_t d = differ[3], o = out[3];
#pragma unroll
        for (int n = 2; n >= 0; --n)
        {
            const bool take = differ[n] != 0u;
            wa = take ? own[n] : wa; wb = take ? other[n] : wb; d = take ? differ[n] : d; o = take ? out[n] : o; which = take ? n : which;
        }
        const int shift = (d & 0xffu) != 0u ? 0 : (d & 0xff00u) != 0u ? 8 : (d & 0xff0000u) != 0u ? 16 : 24;
        const uint32_t mask = 0xffu << shift;
        const float sum = __fadd_rn(DequantDev(static_cast<uint8_t>(static_cast<uint32_t>(wa) >> shift), f.qa),
                                    DequantDev(static_cast<uint8_t>(static_cast<uint32_t>(wb) >> shift), f.qr));
        o = (o & ~mask) | ((static_cast<uint32_t>(QuantizeDev(sum, f.rq) + f.rq.pk_bias) & 0xffu) << shift);
        any = 0u;
#pragma unroll
        for (int n = 0; n < 4; ++n)
        {
            out[n] = which == n ? o : out[n];
            differ[n] = which == n ? d & ~mask : differ[n];
            any |= differ[n];
        }
    }
    ClampCodes(out, f.rq);
    return StoreVec4{static_cast<int>(out[0]), static_cast<int>(out[1]), static_cast<int>(out[2]), static_cast<int>(out[3])};
}

} // namespace mi355x
