// Which block tile a launch of the LDS-tiled implicit GEMM takes.
#pragma once

namespace mi355x
{

// 64 (64 x 64 pixels x channels), 96 (128 x 64), 128 (128 x 128), 256 (256 x 128) or 512 (256 x 256); what is forced otherwise names
// other kernels and passes through.  `narrow`: the caller knows that 128 x 64 is right.
//   64 x 64 while the 128-wide tiling would leave CUs idle.  256 x 256 (16 waves) halves the operand traffic per output once such tiles
// alone fill three quarters of the CUs.
//   A block reads weights and constants for all channels of its tile, those past the layer's last one as well: the width has to divide
// what the plan pads the channels to, a multiple of 128.  (257 to 384 channels under a filter of 49 taps: the second column of 256 wide
// tiles would read 128 rows behind the weights.)
inline int IgemmTile(int forced, bool narrow, long long pixels, int channels, int padded_channels)
{
    const long long big = (pixels + 127) / 128 * ((channels + 127) / 128);
    const long long huge = (pixels + 255) / 256 * ((channels + 255) / 256);
    const int tile = forced != 0 ? forced : narrow ? 96 : big < 400 ? 64 : huge >= 192 && channels >= 256 ? 512 : 128;
    return tile == 512 && padded_channels % 256 != 0 ? 128 : tile;
}

} // namespace mi355x
