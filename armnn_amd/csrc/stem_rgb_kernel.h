// Stems over three-channel images at stride 2 (3x3 and 7x7 filters, up to 64 output channels) on the matrix cores.
//
// SmallCiMfmaKernel gathers each pixel's filter rows from packed bytes: at 7x7 49 LDS reads, 42 byte alignments and 48 selects per 32
// pixels and wave, several times the work of the products and the requantization, and both layers' constants again for each row.
// Here a block unpacks its halo once, to four bytes a pixel, so that a filter row of eight (3x3: four) pixels is 32 (16) bytes in a row at
// an 8-byte aligned address -- a matrix operand as it lies:
//   * v_mfma_i32_16x16x64_i8, pixels as rows, channels as columns; lane (j, g) of a k-step reads 16 bytes, pixel j of 16, half of filter
//     row 2 step + g / 2 (3x3: row g; one step).  The fourth byte of a pixel, the pixels past the filter's width and the row past its
//     last one meet zero weights.
//   * column j of result t is channel 4 j + t (32 channels: 2 j + t), so that a lane has the same channels in all results; weights and
//     constants stay in registers.  With 32 channels a lane has two channels of four pixels, and neighbours trade two for two.
//   * the outputs of 32 pixels pass a wave-private LDS area and leave as 16 bytes per lane.
// The halo comes as unaligned 12-byte loads of four pixels (packed bytes staged as aligned dwords and assembled at the edges, as the other
// kernel has them, were more than the rest of the kernel together at left padding: 28.2 us where it now takes 18.8).
// Before -> here: 7x7 to 64 channels over 224 x 224, 32 images 30.1 -> 18.8 us, one 8.9 -> 6.5; 3x3 to 32 channels, 64 images 13.5 -> 12.1.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"
#include "dw_stem_kernels.h"

namespace mi355x
{

// bytes of K of a channel: filter rows of 32 (7x7) or 16 bytes, pixels of four, the rows rounded up to whole k-steps
constexpr int StemRgbK(int kh) { return kh == 7 ? 256 : 64; }
constexpr int StemRgbRow(int kh) { return kh == 7 ? 32 : 16; }

struct __attribute__((packed, aligned(1))) Bytes12
{
    uint32_t d[3];
};

// The input tensor must have twelve bytes.  NT: output channels / 32, rounded up; TH: rows of the block's tile (32 pixels wide); W2: weights in two halves
template <int KH, int NT, int TH, bool W2 = false>
__global__ __launch_bounds__(256) void StemRgbKernel(SmallCiArgs a)
{
    static_assert(KH == 3 || KH == 7, "three or seven filter rows");
    constexpr int S = 2, TW = 32, RPW = TH / 4;
    constexpr int KST = StemRgbK(KH) / 64;
    constexpr int RP = KH == 7 ? 8 : 4;                              // pixels of a filter row, as operands have them
    constexpr int GROUPS = ((TW - 1) * S + RP + 3) / 4, PITCH = GROUPS * 16;     // four pixels unpacked at a time; bytes of a row
    constexpr int HR = (TH - 1) * S + KH;
    constexpr int NQ = 2 * NT;                                       // results (of 16 channels) per 16 pixels
    constexpr int CH = 32 * NT, LDO = CH + 16;
    __shared__ __attribute__((aligned(16))) uint8_t px4[(HR + 1) * PITCH];       // rows of GROUPS groups of 16 bytes (the row behind the last one meets zero weights)
    __shared__ __attribute__((aligned(16))) uint8_t stage[4][TW * LDO];
    __shared__ __attribute__((aligned(16))) float exact[2][CH];      // mult, biasf

    int b = blockIdx.x;
    const int tx = b % a.tiles_x; b /= a.tiles_x;
    const int ty = b % a.tiles_y;
    const int n = b / a.tiles_y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, g = lane >> 4;

    // ---- the halo, four pixels at a time: twelve bytes wherever they lie, all of a thread's requests in flight together ---------------
    const int iy_org = ty * TH * S - a.pad_top, ix_org = tx * TW * S - a.pad_left;
    const long long image = static_cast<long long>(n) * a.H * a.W * 3, all = static_cast<long long>(a.N) * a.H * a.W * 3;
    constexpr int NG = HR * GROUPS, NIT = (NG + 255) / 256;
    Bytes12 raw[NIT];
#pragma unroll
    for (int k = 0; k < NIT; ++k)
    {
        const int i = min(tid + k * 256, NG - 1), row = i / GROUPS;
        const int iy = iy_org + row, ix = ix_org + 4 * (i - row * GROUPS);
        const long long at = image + (static_cast<long long>(iy) * a.W + ix) * 3;
        // (what is not wholly inside the tensor reads its first bytes and is not used)
        const bool inside = static_cast<unsigned>(iy) < static_cast<unsigned>(a.H) && at >= 0 && at + 12 <= all;
        raw[k] = *reinterpret_cast<const Bytes12*>(a.x + (inside ? at : 0));
    }

    // ---- weights and constants of the lane's channels --------------------------------------------------------------------------
    v4i w[KST][NQ], w2[W2 ? KST : 1][W2 ? NQ : 1], init[NQ];
#pragma unroll
    for (int t = 0; t < NQ; ++t)
    {
        const int c = NT == 2 ? 4 * j + t : 2 * j + t;
#pragma unroll
        for (int s = 0; s < KST; ++s)
        {
            w[s][t] = *reinterpret_cast<const v4i*>(a.w_rgb + c * StemRgbK(KH) + s * 64 + g * 16);
            if constexpr (W2) w2[s][t] = *reinterpret_cast<const v4i*>(a.w_rgb2 + c * StemRgbK(KH) + s * 64 + g * 16);
        }
        const int v = a.corr[c];
        init[t] = v4i{v, v, v, v};
    }
    Fast4 f;
    if constexpr (NT == 2) f = LoadFast4(a.ct, 4 * j);
    else
    {
        // the lane's quads are two channels of two pixels
        const float2 m = *reinterpret_cast<const float2*>(a.ct.p + 2 * a.ct.stride + 2 * j), bb = *reinterpret_cast<const float2*>(a.ct.p + 3 * a.ct.stride + 2 * j);
        f = {float4{m.x, m.y, m.x, m.y}, float4{bb.x, bb.y, bb.x, bb.y}};
    }
    for (int i = tid; i < 2 * CH; i += 256) exact[i / CH][i % CH] = a.ct.p[i / CH * a.ct.stride + i % CH];

    // ---- three bytes a pixel -> four; pixels outside the image hold the padding value ---------------------------------------------
    const uint32_t xm = (a.xor_mask & 0xffu) * 0x01010101u, pad = (a.pad_byte & 0xffu) * 0x01010101u;
#pragma unroll
    for (int k = 0; k < NIT; ++k)
    {
        const int i = tid + k * 256, row = i / GROUPS;
        const int iy = iy_org + row, ix = ix_org + 4 * (i - row * GROUPS);
        const uint32_t e0 = raw[k].d[0] ^ xm, e1 = raw[k].d[1] ^ xm, e2 = raw[k].d[2] ^ xm;
        uint32_t px[4] = {e0, __builtin_amdgcn_alignbyte(e1, e0, 3), __builtin_amdgcn_alignbyte(e2, e1, 2), e2 >> 8};
        const bool row_ok = static_cast<unsigned>(iy) < static_cast<unsigned>(a.H);
        const long long at = image + (static_cast<long long>(iy) * a.W + ix) * 3;
        // the tensor's first or last pixels, where twelve bytes would begin before it or end behind it
        const bool corner = row_ok && (at < 0 || at + 12 > all);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(corner) != 0, 0))
        {
            if (corner)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (static_cast<unsigned>(ix + q) < static_cast<unsigned>(a.W))
                    {
                        const uint8_t* const p = a.x + at + 3 * q;
                        px[q] = (static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8) | (static_cast<uint32_t>(p[2]) << 16)) ^ xm;
                    }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) px[q] = row_ok && static_cast<unsigned>(ix + q) < static_cast<unsigned>(a.W) ? px[q] : pad;
        if (i < NG) *reinterpret_cast<uint4*>(px4 + i * 16) = uint4{px[0], px[1], px[2], px[3]};
    }
    __syncthreads();

    // ---- 32 pixels of a row at a time ----------------------------------------------------------------------------------------------
    typedef long Pair8 __attribute__((ext_vector_type(2), aligned(8)));
    const uint8_t* const operand = px4 + (KH == 7 ? (g >> 1) * PITCH + 16 * (g & 1) : g * PITCH) + j * (S * 4);
    uint8_t* const area = stage[wave];
    const OutPtr outp = MakeOutPtr(a.y, static_cast<long long>(a.N) * a.Ho * a.Wo * a.Co);
#pragma unroll 1
    for (int rr = 0; rr < RPW; ++rr)
    {
        const int ly = wave * RPW + rr;
        const int oy = ty * TH + ly;
        if (oy >= a.Ho) break;                    // wave-uniform
        WithBits(a.rq, [&](auto bits) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
            {
                v4i acc[NQ];
#pragma unroll
                for (int s = 0; s < KST; ++s)
                {
                    const v4i x = __builtin_bit_cast(v4i, *reinterpret_cast<const Pair8*>(operand + ly * (S * PITCH) + s * (2 * PITCH) + mt * (16 * S * 4)));
#pragma unroll
                    for (int t = 0; t < NQ; ++t)
                    {
                        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, w[s][t], s == 0 ? init[t] : acc[t], 0, 0, 0);
                        if constexpr (W2) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, w2[s][t], acc[t], 0, 0, 0);
                    }
                }
                // rows of a result are pixels 4 g + r
                if constexpr (NT == 2)
                {
                    v4i v[4];
                    uint32_t out[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
                    RequantPixels<decltype(bits)::value, 4>(v, out, f, ChanTab{exact[0], CH}, 4 * j, a.rq);
#pragma unroll
                    for (int r = 0; r < 4; ++r) *reinterpret_cast<uint32_t*>(area + (mt * 16 + 4 * g + r) * LDO + 4 * j) = out[r];
                }
                else
                {
                    v4i v[2];
                    uint32_t out[2];
#pragma unroll
                    for (int r = 0; r < 2; ++r) v[r] = v4i{acc[0][2 * r], acc[1][2 * r], acc[0][2 * r + 1], acc[1][2 * r + 1]};
                    const Fast4 fs[1] = {f};
                    RequantCore<decltype(bits)::value, 2, 1>(v, out, fs, a.rq, [&](int, float4& m, float4& bb) {
                        const float2 m2 = *reinterpret_cast<const float2*>(&exact[0][2 * j]), b2 = *reinterpret_cast<const float2*>(&exact[1][2 * j]);
                        m = float4{m2.x, m2.y, m2.x, m2.y};
                        bb = float4{b2.x, b2.y, b2.x, b2.y};
                    });
                    // channels 2 j, 2 j + 1 of pixels 0, 1 | 2, 3 here, the next two channels in lane j ^ 1: the even lane takes pixels 0 and 1
                    const bool odd = (j & 1) != 0;
                    const uint32_t keep = odd ? out[1] : out[0];
                    const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(odd ? out[0] : out[1]), 0xb1, 0xf, 0xf, true));
                    const uint32_t lo = odd ? got : keep, hi = odd ? keep : got;
                    uint8_t* const at = area + (mt * 16 + 4 * g + (odd ? 2 : 0)) * LDO + (j >> 1) * 4;
                    *reinterpret_cast<uint32_t*>(at) = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                    *reinterpret_cast<uint32_t*>(at + LDO) = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
                }
            }
        });
        // the wave reads back what its own lanes wrote: LDS operations of one wave complete in order; the fences keep the compiler
        // from moving the reads above the writes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const long long row_at = ((static_cast<long long>(n) * a.Ho + oy) * a.Wo + tx * TW) * a.Co;
#pragma unroll
        for (int k = 0; k < NT; ++k)
        {
            const int id = k * 64 + lane, px = id / (CH / 16), c0 = id % (CH / 16) * 16;
            const v4i v = *reinterpret_cast<const v4i*>(area + px * LDO + c0);
            if (tx * TW + px < a.Wo && c0 < a.Co)
            {
                const long long at = row_at + static_cast<long long>(px) * a.Co + c0;
                if (a.vec16) StoreOut16(outp, at, v);
                else
                {
                    // (channels come in fours; those past the layer's last one do not exist)
                    uint32_t* const dst = reinterpret_cast<uint32_t*>(a.y + at);
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        if (c0 + 4 * d < a.Co) dst[d] = static_cast<uint32_t>(v[d]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

} // namespace mi355x
