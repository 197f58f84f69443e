// Tokens per thread of the causal convolution of prompts: plain host arithmetic, checked on the CPU.
#pragma once
#include <stdint.h>

namespace mi355 {

constexpr int kMaxTaps = 16, kMostConvTile = 16;
static_assert(kMostConvTile >= kMaxTaps - 1, "tiles behind the first stay inside their portion");

// A tile reads the taps - 1 tokens in front of it, and the one at the start of a portion overwrites the ring that holds what came before the portion.  Tiles run in
// any order, so those behind the first must not reach back to that ring: a tile is never shorter than taps - 1.
// As short as that allows where a call is small.  us with 4 / 8 / 16 tokens per thread, 4 taps: 64 tokens of 4352 channels 5.1, 5.0, 6.7; 577 of 4352 7.4, 7.4, 9.0;
// 1024 9.1, 10.1, 10.1; 4000 of 1280 10.3, 10.7, 10.9; 8000 16.5, 14.1, 15.2; 8192 of 1280 (10.5 M inputs) -, 15.3, 15.9; 2800 of 4352 (12.2 M) -, 15.2, 14.4; 8192 of
// 4352 40.9, 34.2, 26.3
inline int conv_tile(int64_t n_rows, int channels, int taps) {
    const int64_t inputs = n_rows * channels;
    int tile = inputs <= 6 << 20 ? 4 : inputs <= 11 << 20 ? 8 : kMostConvTile;
    while (tile < taps - 1) tile *= 2;
    return tile;
}

}  // namespace mi355
