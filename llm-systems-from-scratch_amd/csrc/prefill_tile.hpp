// LDS tile layout shared by the prefill forward and backward kernels: row-major tiles of D bf16
// per row, unpadded (direct-to-LDS loads write 1 KiB of consecutive LDS per wavefront), with an
// XOR swizzle of the 16-byte chunk index instead of padding.
#pragma once
#include "common.hpp"

namespace mi355 {

// XOR pattern applied to the 16-byte chunk index of LDS row `row` (rows hold D bf16).
// Chosen so that (a) 16 lanes reading one logical chunk of 16 consecutive rows and
// (b) a transposed read touching 4 consecutive rows x 32 bytes both spread over
// distinct banks (LDS banks repeat every 256 bytes).
template <int D>
__device__ __forceinline__ int swz(int row) {
    if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
    else if constexpr (D == 64) return (((row >> 1) & 3) << 1) | ((row >> 3) & 1);
    else return (row >> 2) & 3;
}

// Heads that the kernels of short sequences keep on one XCD.  Rows of 32 elements are half a line: where a tensor's heads stand side by side (V, the output and its gradient are views of
// (batch, seq, heads, d)), two heads share each line, and on two XCDs both fetch it.  us, heads dealt one by one / two together / eight: forward of 64 x 16 heads, 256 tokens 20.6 /
// 18.2 / 18.2, with gradients (forward, backward) 21.1, 44.3 / 18.9, 40.4 / 19.0, 40.0; 200 x 16 heads, 100 tokens 28.1, 46.2 / 25.6, 42.1 / 23.2, 39.5.  Heads of 64
// (64 x 16, 256 tokens 41.1, 81.8 / 40.3, 82.4 / 40.3, 80.6; 64 x 8, 128 tokens 9.55 / 9.57 / 9.92) have lines of their own.
constexpr int short_heads(int D) { return D == 32 ? 8 : 1; }

// Per-lane LDS offsets of the two read patterns of a swizzled 64 x D tile.
template <int D>
struct TileReads {
    static constexpr int NS = D / 16, NDT = D / 32, kRow = D * 2;
    int row_off[NS];        // A fragment "row n of the tile, k = 16s + 8kg ..": add 32*t*kRow
    int tr_off[2][NDT];     // transposed fragment of d-tile dt for a 16-row slice: add 16*u*kRow
    __device__ __forceinline__ void init(int lane) {
        const int n = lane & 31, kg = lane >> 5;
#pragma unroll
        for (int s = 0; s < NS; ++s) row_off[s] = n * kRow + (((2 * s + kg) ^ swz<D>(n)) << 4);
        const int g16 = lane >> 4, s16 = lane & 15;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int row = 4 * (g16 >> 1) + (s16 >> 2) + 8 * e;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const int d = 32 * dt + 16 * (g16 & 1) + 4 * (s16 & 3);
                tr_off[e][dt] = row * kRow + (((d >> 3) ^ swz<D>(row)) << 4) + (d & 7) * 2;
            }
        }
    }
};

}  // namespace mi355
