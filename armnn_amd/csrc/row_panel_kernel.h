// 1x1 convolutions (stride 1, no padding) of many rows: a block of four waves owns 64 rows x 64 CG output channels.
//
//   * The block's rows, all of K up to 512 bytes of it, are requested at once as whole lines and lie in LDS as [K / 16][row][16
//     bytes]: one round trip and one barrier where the tiled kernels have one per k-tile.
//   * A wave owns 16 CG of the channels for all rows and reads its weights in operand order straight from L2, RD k-steps ahead.
//   * The outputs meet in LDS and leave as 16 bytes per lane, with an Addition behind the layer on the way, whose other input was
//     requested at the start.
// Four waves per SIMD (128 registers) are what hides the round trips: the same kernel at 144 registers took 7.0 us where it takes
// 5.3.  What takes the time is waiting (54 % of a wave's life) and the CU's L1, at two clocks a line: 64 rows and 128 rows of weights per 128 bytes
// of K, at 28 x 28 x 128 -> 512 4.1 k accesses per CU, 8 k of the launch's 18 k clocks; over 56 x 56 x 256 -> 64 the rows' way from memory is
// (3.9 TB/s, 840 clocks a request).  With the Addition the write-out's VALU work comes on top.  Before -> here, 32 images unless said: 28 x 28 x 128 -> 512 14.8 -> 8.3 us, 14 x 14 x 256 -> 1024
// 9.4 -> 6.7, 56 x 56 x 256 -> 64 18.1 -> 9.7, 56 x 56 x 256 -> 512 52.7 -> 33.1, 56 x 56 x 48 -> 96 (16 images) 7.4 -> 5.1.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"
#include "dw_mfma_kernel.h"

namespace mi355x
{

constexpr int kRowPanelK = 512;                          // bytes of K in LDS at a time
constexpr int kRowPanelGp = 65 * 16;                     // bytes per 16 channels: 64 rows of 16 bytes, an odd number of pieces

template <int CG>
constexpr int RowPanelSmem(int K)
{
    const int in = ((K < kRowPanelK ? K : kRowPanelK) + 63) / 64 * 4 * kRowPanelGp, out = 64 * (64 * CG + 16);
    return (in > out ? in : out) + 16 * 64 * CG;         // + the block's slice of the channel table
}

// a.w in operand order (PackFragKernel); a.tiles_n = ceil(Co / (64 CG)), a.tiles_m = ceil(M / 64).  a.res: an Addition behind.
// KB: bytes of K in LDS at a time at most (a.Ci <= KB where KB < kRowPanelK).
template <int CG, int KB, bool AW>
__global__ __launch_bounds__(256, KB <= 256 ? 4 : 3) void RowPanelKernel(IgemmArgs a, int co_groups, uint32_t rcp_tiles_n)
{
    constexpr int NT = 256, NW = 4, PG = 4, GP = kRowPanelGp, HS = KB / 16 * 64 / NT;
    constexpr int RD = CG == 1 ? 8 : 4;                  // k-steps of weights in flight
    constexpr int NCOL = 16 * NW * CG, OP = NCOL + 16, CHUNKS = NCOL / 16, NP = 64 * CHUNKS / NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t row_lds[];
    const int nblocks = a.tiles_m * a.tiles_n, per_xcd = (nblocks + 7) >> 3;
    const int tile = XcdContiguousWorkItem(blockIdx.x, per_xcd);
    if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || tile >= nblocks) return;
    const int tm = DivByInvariant(tile, a.tiles_n, rcp_tiles_n), bn = tile - tm * a.tiles_n;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int steps = (a.Ci + 63) >> 6;
    const int xm = static_cast<int>(a.xor_mask);

    // ---- rows: thread (row, 16-byte piece); a run of lanes takes whole lines of a row -----------------------------------------
    v4i h[HS];
    auto load_rows = [&](int k0) {                       // K bytes k0 .. k0 + 511
        const int pr = min(a.Ci - k0, KB) >> 4;  // pieces per row: a power of two or any multiple of 1
        const int sh = 31 - __clz(pr);
        const bool pow2 = (pr & (pr - 1)) == 0;
        const int pieces = 64 * pr;
#pragma unroll
        for (int k = 0; k < HS; ++k)
        {
            if (k * NT >= pieces) continue;
            const int i = min(tid + k * NT, pieces - 1);
            const int row = pow2 ? i >> sh : i / pr;
            const int part = i - row * pr;
            h[k] = *reinterpret_cast<const v4i*>(a.x + static_cast<long long>(min(tm * 64 + row, a.M - 1)) * a.Ci + k0 + part * 16);
        }
    };
    auto store_rows = [&](int k0) {
        const int pr = min(a.Ci - k0, KB) >> 4;
        const int sh = 31 - __clz(pr);
        const bool pow2 = (pr & (pr - 1)) == 0;
        const int pieces = 64 * pr;
#pragma unroll
        for (int k = 0; k < HS; ++k)
        {
            if (k * NT >= pieces) continue;
            const int i = min(tid + k * NT, pieces - 1);
            const int row = pow2 ? i >> sh : i / pr;
            const int part = i - row * pr;
            *reinterpret_cast<v4i*>(row_lds + part * GP + row * 16) = h[k] ^ xm;
        }
        // pieces that complete the last k-step: their weights are zero, and with AW they must not count either
        for (int i = tid + pr * 64; i < (pr + 3) / 4 * 4 * 64; i += NT) *reinterpret_cast<v4i*>(row_lds + (i >> 6) * GP + (i & 63) * 16) = v4i{0, 0, 0, 0};
    };
    // the block's slice of the channel table (channels past the last one: some other channel's, nothing is stored)
    float* const tab_lds = reinterpret_cast<float*>(row_lds + RowPanelSmem<CG>(a.Ci) - 16 * NCOL);
    v4i tab_piece = {0, 0, 0, 0};
    if (tid < NCOL) tab_piece = *reinterpret_cast<const v4i*>(a.ct.p + tid / (NCOL / 4) * a.ct.stride + min(bn * NCOL + tid % (NCOL / 4) * 4, co_groups * 16 - 4));
    load_rows(0);
    // ---- weights of the wave's CG groups of output channels -----------------------------------------------------------------------
    int cgrp[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) cgrp[c] = min((bn * NW + wave) * CG + c, co_groups - 1);
    v4i wv[RD][CG];
    auto load_weights = [&](int ks, int r) {
#pragma unroll
        for (int c = 0; c < CG; ++c) wv[r][c] = *reinterpret_cast<const v4i*>(a.w + static_cast<long long>(cgrp[c] * steps + ks) * 1024 + lane * 16);
    };
#pragma unroll
    for (int r = 0; r < RD; ++r)
        if (r < steps) load_weights(r, r);
    // (what the accumulators start from)
    v4i corr[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) corr[c] = *reinterpret_cast<const v4i*>(a.corr + cgrp[c] * 16 + 4 * g);
    // ---- the Addition's other input ---------------------------------------------------------------------------------------------
    v4i other[NP];
    const bool fuse = a.res != nullptr;
    if (fuse)
    {
#pragma unroll
        for (int i = 0; i < NP; ++i)
        {
            const int idx = tid + i * NT, r = idx / CHUNKS, chunk = idx - r * CHUNKS;
            other[i] = *reinterpret_cast<const v4i*>(a.res + static_cast<long long>(min(tm * 64 + r, a.M - 1)) * a.Co + min(bn * NCOL + chunk * 16, a.Co - 16));
        }
    }
    v4i acc[CG][PG];
    int xs[PG];
#pragma unroll
    for (int p = 0; p < PG; ++p)
    {
        xs[p] = 0;
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c][p] = corr[c];
    }
    const uint8_t* const pb = row_lds + g * GP + j * 16;
    for (int k0 = 0; k0 < a.Ci; k0 += KB)
    {
        if (k0 != 0) __syncthreads();                    // the rows before have been read
        store_rows(k0);
        if (k0 == 0 && tid < NCOL) *reinterpret_cast<v4i*>(tab_lds + tid * 4) = tab_piece;
        __syncthreads();
        const bool more = k0 + KB < a.Ci;
        if (more) load_rows(k0 + KB);
        const int s0 = k0 >> 6, s1 = min(steps, s0 + KB / 64);
        for (int k1 = s0; k1 < s1; k1 += RD)
        {
#pragma unroll
            for (int r = 0; r < RD; ++r)
            {
                const int ks = k1 + r;
                if (ks >= s1) break;
                v4i xb[PG];
#pragma unroll
                for (int p = 0; p < PG; ++p) xb[p] = *reinterpret_cast<const v4i*>(pb + (ks - s0) * 4 * GP + p * 256);
#pragma unroll
                for (int c = 0; c < CG; ++c)
#pragma unroll
                    for (int p = 0; p < PG; ++p) acc[c][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[r][c], xb[p], acc[c][p], 0, 0, 0);
                if constexpr (AW)
                {
#pragma unroll
                    for (int p = 0; p < PG; ++p)
#pragma unroll
                        for (int d = 0; d < 4; ++d) xs[p] = __builtin_amdgcn_sdot4(xb[p][d], 0x01010101, xs[p], false);
                }
                if (ks + RD < steps) load_weights(ks + RD, r);
            }
        }
    }
    // ---- write-out ----------------------------------------------------------------------------------------------------------------
    if constexpr (AW)
    {
#pragma unroll
        for (int p = 0; p < PG; ++p)
        {
            xs[p] += __shfl_xor(xs[p], 16);
            xs[p] += __shfl_xor(xs[p], 32);
            xs[p] *= a.zw_neg;
        }
    }
    __syncthreads();                                     // the rows have been read; the outputs take their place
    WithBits(a.rq, [&](auto bits) {
#pragma unroll
    for (int c = 0; c < CG; ++c)
    {
        const int cl = (wave * CG + c) * 16 + 4 * g;
        const Fast4 f = {*reinterpret_cast<const float4*>(tab_lds + 2 * NCOL + cl), *reinterpret_cast<const float4*>(tab_lds + 3 * NCOL + cl)};
        uint32_t out[PG];
        if constexpr (AW)
        {
#pragma unroll
            for (int p = 0; p < PG; ++p) acc[c][p] += xs[p];
        }
        RequantPixels<decltype(bits)::value, PG>(acc[c], out, f, ChanTab{tab_lds, NCOL}, cl, a.rq);
#pragma unroll
        for (int p = 0; p < PG; ++p) *reinterpret_cast<uint32_t*>(row_lds + (16 * p + j) * OP + (wave * CG + c) * 16 + 4 * g) = out[p];
    }
    });
    __syncthreads();
    const OutPtr outp = MakeOutPtr(a.y, static_cast<long long>(a.M) * a.Co);
#pragma unroll
    for (int i = 0; i < NP; ++i)
    {
        const int idx = tid + i * NT, r = idx / CHUNKS, chunk = idx - r * CHUNKS;
        const int m = tm * 64 + r, c0 = bn * NCOL + chunk * 16;
        if (m < a.M && c0 < a.Co)
        {
            v4i v = *reinterpret_cast<const v4i*>(row_lds + r * OP + chunk * 16);
            if (fuse) v = AddQuantize16Dev(v, other[i], a.add);
            StoreOut16(outp, static_cast<long long>(m) * a.Co + c0, v);
        }
    }
}

} // namespace mi355x
