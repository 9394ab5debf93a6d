// Convolutions and FullyConnected layers with few output rows: a block owns 32 rows x 32 channels and its waves split K.  (Filters of nine taps and more over many
// whole k-steps take TapPanelKernel, tap_panel_kernel.h.)
//
// A layer of one or a few small images gives the 64 x 64 tiles of IgemmLdsKernel too few blocks, each of which then walks
// its whole K one k-tile and one barrier at a time: at one image a 3 x 3 layer of ResNet-50 over 14 x 14 x 256 is 16 blocks
// of 18 k-tiles.  What such a launch costs is the length of that chain, not bytes or operations.  Here
//   * four times the blocks (32 x 32 outputs), and the four waves of a block each take a contiguous quarter of the k-steps;
//   * a wave reads its MFMA operands straight from global memory into registers, four k-steps at once, so all of K is on
//     its way after a quarter as many round trips and no LDS staging or barrier lies in between;
//   * the partial tiles meet in LDS, where the waves add them up in a fixed order, requantize four channels per lane, and
//     one wave writes the tile in 16-byte pieces (with a following Addition on the way, if there is one).
// What is left is latency: waves wait 59 % of their cycles (3 x 3 over 14 x 14 x 256, one image), and of the 13 k cycles of a block the
// CU's address unit, which takes an instruction's cache lines one after the other, is busy for 4.3 k.  Hence v_mfma_i32_16x16x64_i8,
// whose activation operand is 16 pixels x 64 contiguous bytes (32x32x32: 32 pixels x 32), and weights stored in operand order
// (PackFragKernel), so that a wave's weight load is one run of 1 KB instead of 32 rows.
// The other part of a launch is instructions that are fetched to be executed once or twice: pixels are decoded with reciprocals and a
// wave's start in K comes from the host.  With the divisions -> here, us: launched one by one 28 x 28 x 128 4.78 -> 4.53, 14 x 14 x 256 5.78
// -> 5.50, 7 x 7 x 512 7.70 -> 7.48, 56 x 56 x 64 3.87 -> 3.68; from a graph of 120, three sets of tensors in turn, 4.21 -> 4.18, 5.25 -> 5.19, 7.18 ->
// 7.20, 3.33 -> 3.29, FullyConnected of 64 rows 4096 -> 4096 9.20 -> 8.80.  From such a graph layers whose channels are no multiple of 64, with
// the divisions -> walking taps by selects -> here: 3 x 3 over 14 x 14 x 144, two images 3.80 -> 3.90 -> 3.71, 5 x 5 to 128 channels at stride 2
// over 16 x 16, four images, from 272 7.83 -> 8.28 -> 7.46, from 496 15.7 -> 16.3 -> 15.2; no multiple of 16, 3 x 3 over 14 x 14 x 72 3.50 -> 3.62 ->
// 3.40, 12 x 12 x 300 5.78 -> 6.14 -> 5.69.
// Launches back to back, against the larger tiles (one image unless said): 3 x 3 over 28 x 28 x 128 7.2 -> 4.5 us, 14 x 14 x 256 9.1 ->
// 5.5, 7 x 7 x 512 13.3 -> 7.4, 56 x 56 x 64 5.9 -> 3.7, 28 x 28 x 96 7.2 -> 3.8; 1 x 1 over 14 x 14 x 1024 -> 256 5.7 -> 4.0, 28 x 28 x
// 128 -> 256 5.6 -> 3.1; FullyConnected 4096 -> 4096 of 64 rows 12.9 -> 9.6.  An empty kernel takes 2.75 us in such a row.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"

namespace mi355x
{

// Weights in the order the kernel below loads them: [Co / 16][steps][64 lanes][16 bytes], lane l of a step = bytes
// 64 step + 16 (l / 16) .. + 15 of row l % 16.  `steps` = K / 64 rounded up; bytes beyond K_pad are zero.
// interleave: byte 4 i + e of those 16 is byte 64 step + 16 e + 4 (l / 16) + i of the row instead (dwpw_panel_kernel.h).
static __global__ __launch_bounds__(256) void PackFragKernel(const int8_t* __restrict__ w, int8_t* __restrict__ out, int K_pad, int steps, long long pieces, int interleave)
{
    const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int l = static_cast<int>(i & 63);
    const long long gs = i >> 6;
    const int s = static_cast<int>(gs % steps);
    const long long row = gs / steps * 16 + (l & 15);
    const int k = s * 64 + (l >> 4) * 16;
    v4i v = {0, 0, 0, 0};
    if (interleave != 0)
    {
        for (int e = 0; e < 4; ++e)
            for (int b = 0; b < 4; ++b)
            {
                const int kb = s * 64 + 16 * e + 4 * (l >> 4) + b;
                if (kb < K_pad) v[b] |= static_cast<int>(static_cast<uint32_t>(static_cast<uint8_t>(w[row * K_pad + kb])) << (8 * e));
            }
    }
    else if (k < K_pad) v = *reinterpret_cast<const v4i*>(w + row * K_pad + k);
    *reinterpret_cast<v4i*>(out + i * 16) = v;
}

// a.w in PackFragKernel's order.  AW: the weights have a zero point (row sums beside the products); RG: Ci is no multiple of
// 16; both as in IgemmKernel.  WHOLE: Ci is a multiple of 64, a filter tap whole k-steps (LaunchSmallConv has the rule).  a.tiles_n = ceil(Co / 32), a.tiles_m = ceil(M / 32); one tile per block.
template <bool AW, bool RG, bool WHOLE>
__global__ __launch_bounds__(256) void SmallConvKernel(IgemmArgs a)
{
    FetchArgs<sizeof(IgemmArgs)>();
    static_assert(!(RG && WHOLE), "channels that are no multiple of 16 make no whole k-steps");
    constexpr int NW = 4;                                // (8 and 16 waves were slower: more instructions for the same lines)
    __shared__ __attribute__((aligned(16))) v4i part[NW][4][64];
    __shared__ int rowpart[NW][2][64];
    __shared__ __attribute__((aligned(16))) uint32_t stage[32][12];      // 32 rows x 32 bytes, 48 bytes apart
    // each XCD gets a contiguous run of tiles: column tiles of a row tile share the pixels
    const int nblocks = a.tiles_m * a.tiles_n;
    const int per_xcd = (nblocks + 7) >> 3;
    const int tile = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || tile >= nblocks) return;
    const int tn = tile % a.tiles_n, tm = tile / a.tiles_n;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, g = lane >> 4;              // operand: pixel or channel j, bytes 16 g of a k-step; result: pixel j, channels 4 g ..
    const int xm = static_cast<int>(a.xor_mask);

    int iy0[2], ix0[2];
    const uint8_t* xrow[2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
    {
        const int m = min(tm * 32 + p * 16 + j, a.M - 1);        // rows past the end re-read the last row (never stored)
        int n, oy, ox;
        if (a.unit) { n = 0; oy = 0; ox = m; }
        else
        {
            // (a divisor of 1 has no reciprocal in 32 bits)
            const int t = a.Wo == 1 ? m : a.wo_magic != 0 ? static_cast<int>(__umulhi(static_cast<uint32_t>(m), a.wo_magic)) : m / a.Wo;
            ox = m - t * a.Wo;
            n = a.Ho == 1 ? t : a.ho_magic != 0 ? static_cast<int>(__umulhi(static_cast<uint32_t>(t), a.ho_magic)) : t / a.Ho;
            oy = t - n * a.Ho;
        }
        iy0[p] = oy * a.stride_y - a.pad_top;
        ix0[p] = ox * a.stride_x - a.pad_left;
        xrow[p] = a.x + static_cast<long long>(n) * a.H * a.W * a.Ci + (static_cast<long long>(iy0[p]) * a.W + ix0[p]) * a.Ci;
    }
    // this wave's k-steps of 64 bytes
    const int tap_bytes = RG ? a.Ck : a.Ci;
    const int steps = (a.Kh * a.Kw * tap_bytes + 63) >> 6;
    const int uw = __builtin_amdgcn_readfirstlane(wave);
    const int s0 = RG ? steps * uw / NW : a.wave_k[uw].step, s1 = RG ? steps * (uw + 1) / NW : a.wave_k[uw + 1].step;
    const int8_t* wp = a.w + static_cast<long long>(2 * tn) * steps * 1024 + lane * 16;
    const long long w_next = static_cast<long long>(steps) * 1024;       // the tile's second group of 16 channels
    // the lane's chunk: filter tap and channel, advanced by 64 bytes per step.  Where the wave starts comes from the host, 0.05 to 0.1 us less
    // than dividing for it -- but 0.02 to 0.2 more in most of the RG layers, whose lanes then have to walk to their own start
    int ci, ky, kx;
    if constexpr (RG)
    {
        ci = s0 * 64 + g * 16;
        const int tap = ci / tap_bytes;
        ci -= tap * tap_bytes;
        ky = tap / a.Kw;
        kx = tap - ky * a.Kw;
    }
    else
    {
        ci = a.wave_k[uw].ci + g * 16;
        ky = a.wave_k[uw].ky;
        kx = a.wave_k[uw].kx;
    }
    // WHOLE walks by selects.  (`wide` always holds there: a branch between the steps, without which the compiler mixes their loads and a
    // launch takes 2 % longer.)  By itself such a launch would be faster with the loop, 3 x 3 over 14 x 14 x 256 5.07 against 5.20 us, but not beside
    // others: ResNet-50, 192 x 192, two images, three networks in turn, 118.9 with selects, 119.7 with the loop.  In the other layers the
    // selects, which need a tap's offset anew for every step, cost up to a tenth (below).
    const bool wide = tap_bytes >= 64;
    auto wrap = [&] {
        if (WHOLE && wide)
        {
            const bool over = ci >= tap_bytes;
            ci -= over ? tap_bytes : 0;
            kx += over ? 1 : 0;
            const bool row = kx == a.Kw;
            kx = row ? 0 : kx;
            ky += row ? 1 : 0;
            return;
        }
        while (ci >= tap_bytes)
        {
            ci -= tap_bytes;
            if (++kx == a.Kw) { kx = 0; ++ky; }
        }
    };
    if constexpr (!RG) wrap();
    // what this wave will requantize with (wave 2 c + p finishes channel group c of pixel group p), requested ahead of the operands (RG: rows 0
    // and 1 of the table when a value asks for them, 0.02 to 0.1 us less)
    const int cg = wave >> 1, pg = wave & 1;
    const int cq = tn * 32 + cg * 16 + 4 * g;
    const v4i corr4 = *reinterpret_cast<const v4i*>(a.corr + cq);
    const Fast4 f4[1] = {LoadFast4(a.ct, cq)};
    const auto exact_row = [&](int r) { return *reinterpret_cast<const float4*>(a.ct.p + r * a.ct.stride + cq); };
    float4 mult = {}, biasf = {};
    if constexpr (!RG) { mult = exact_row(0); biasf = exact_row(1); }
    v4i acc[2][2];                                       // [channel group][pixel group]
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 2; ++p) acc[c][p] = v4i{0, 0, 0, 0};
    int xs[2] = {0, 0};
    // U k-steps: all their loads, then their products
    auto batch = [&](int s, auto un) {
        constexpr int U = decltype(un)::value;
        v4i xv[U][2], wv[U][2];
        int back[RG ? U : 1][2], real[RG && AW ? U : 1];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            // a chunk outside the image or beyond K reads 16 prepared padding bytes (the weights beyond K are zero): no load sits
            // in a divergent branch
            const int dy = ky * a.dil_y, dx = kx * a.dil_x;
            const long long off = (static_cast<long long>(dy) * a.W + dx) * a.Ci + ci;
#pragma unroll
            for (int p = 0; p < 2; ++p)
            {
                const bool ok = ky < a.Kh && static_cast<unsigned>(iy0[p] + dy) < static_cast<unsigned>(a.H) && static_cast<unsigned>(ix0[p] + dx) < static_cast<unsigned>(a.W);
                const uint8_t* src = ok ? xrow[p] + off : a.pad16;
                if constexpr (RG)
                {
                    back[u][p] = ok && src > a.x_last16 ? static_cast<int>(src - a.x_last16) : 0;
                    xv[u][p] = LoadUnaligned16(src - back[u][p]);
                }
                else xv[u][p] = *reinterpret_cast<const v4i*>(src);
            }
            if constexpr (RG && AW) real[u] = min(16, a.Ci - ci);
            const int8_t* ws = wp + static_cast<long long>(s + u) * 1024;
            wv[u][0] = *reinterpret_cast<const v4i*>(ws);
            wv[u][1] = *reinterpret_cast<const v4i*>(ws + w_next);
            ci += 64;
            wrap();
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < 2; ++p)
            {
                v4i xb = xv[u][p];
                if constexpr (RG)
                {
                    if (__builtin_expect(__builtin_amdgcn_ballot_w64(back[u][p] != 0) != 0, 0)) xb = ShiftDown16(xb, back[u][p]);
                }
                xb ^= xm;
                if constexpr (RG && AW) xb = KeepBytes16(xb, real[u], a.pad_word);
                acc[0][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[u][0], xb, acc[0][p], 0, 0, 0);
                acc[1][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[u][1], xb, acc[1][p], 0, 0, 0);
                if constexpr (AW)
                {
#pragma unroll
                    for (int d = 0; d < 4; ++d) xs[p] = __builtin_amdgcn_sdot4(xb[d], 0x01010101, xs[p], false);
                }
            }
    };
    using std::integral_constant;
    int s = s0;
    for (; s1 - s >= 4; s += 4) batch(s, integral_constant<int, 4>{});
    if (s1 - s == 3) batch(s, integral_constant<int, 3>{});
    else if (s1 - s == 2) batch(s, integral_constant<int, 2>{});
    else if (s1 - s == 1) batch(s, integral_constant<int, 1>{});
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 2; ++p) part[wave][2 * c + p][lane] = acc[c][p];
    if constexpr (AW) { rowpart[wave][0][lane] = xs[0]; rowpart[wave][1][lane] = xs[1]; }
    // the write-out's pieces: lane = (row, 16-byte half) of the tile, wave 0; an Addition's other input is requested here
    const int orow = lane >> 1, oc = (lane & 1) * 16;
    const int om = tm * 32 + orow, c0 = tn * 32 + oc;
    v4i other = {0, 0, 0, 0};
    const bool fuse = a.res != nullptr;
    if (fuse && wave == 0) other = *reinterpret_cast<const v4i*>(a.res + static_cast<long long>(min(om, a.M - 1)) * a.Co + min(c0, a.Co - 16));
    __syncthreads();
    {
        v4i v = corr4;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += part[w][wave][lane];
        if constexpr (AW)
        {
            int total = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) total += rowpart[w][pg][j] + rowpart[w][pg][j + 16] + rowpart[w][pg][j + 32] + rowpart[w][pg][j + 48];
            // what the bytes beyond K added are padding values
            v += (total - (steps * 64 - a.Kh * a.Kw * a.Ci) * static_cast<int>(static_cast<int8_t>(a.pad_word & 0xffu))) * a.zw_neg;
        }
        const v4i sums[1] = {v};
        uint32_t out[1];
        WithBits(a.rq, [&](auto bits) {
            RequantCore<decltype(bits)::value, 1, 1>(sums, out, f4, a.rq, [&](int, float4& m, float4& b) { m = RG ? exact_row(0) : mult; b = RG ? exact_row(1) : biasf; });
        });
        stage[pg * 16 + j][cg * 4 + g] = out[0];
    }
    __syncthreads();
    if (wave == 0 && om < a.M && c0 < a.Co)
    {
        v4i v = *reinterpret_cast<const v4i*>(&stage[orow][(lane & 1) * 4]);
        const long long at = static_cast<long long>(om) * a.Co + c0;
        if (fuse) v = AddQuantize16Dev(v, other, a.add);
        if (a.vec_out) StoreOut16(MakeOutPtr(a.y, static_cast<long long>(a.M) * a.Co), at, v);
        else StoreRagged16(a.y + at, v, a.Co - c0);
    }
}

} // namespace mi355x
