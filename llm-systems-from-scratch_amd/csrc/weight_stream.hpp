// 32 rows of a weight matrix against 16 or 32 rows of activations, as a wavefront's share of a product with few rows.
//
// Such a product reads every weight once, so what counts is how the weights come in.  16-byte loads straight into the
// MFMA's operand layout touch 64 bytes of each of 16 rows per instruction, and the address unit takes four times as long for
// one as for a load of whole lines; here a direct load to LDS brings 8 rows of 128 bytes.  Each wavefront has a ring of its own
// (no barrier inside the stream) and takes every fourth (of eight wavefronts every eighth) 64-wide step of k; the caller adds them up.
#pragma once
#include "common.hpp"

namespace mi355 {

// The ring of a wavefront where three workgroups of four share a compute unit (two where a norm's 16 KB come on top): two steps of 32 + 16 rows, or one of 32 + 32.
// Others: kWideStreamBytes of eight wavefronts (rows_linear.hip), kDirectRing of experts with many pairs (moe_ops.hip).
constexpr int kStreamBytes = 12 * 1024;

// Workgroups that stream rows of whole 4096 bytes side by side, all from step 0 on, want the same few of an L2's sixteen channels (256 bytes each in turn) at any
// time: 16 experts of 2048 x 1024, 32 tokens 44.0 us, 4.6 TB/s; 39.5, 5.1 TB/s, with the steps begun somewhere else by every one of an XCD's workgroups (every eighth of a launch).  The same
// beginning within an XCD and another on each other one gives nothing (45.0); nor does any with rows of 2048 bytes (24.3 / 25.1), which have two sets of channels.
inline bool turn_pays(int k) { return k % 2048 == 0; }
// (at: the workgroup among those that read other weights, so that a row's sums do not depend on what else the launch has)
__device__ __forceinline__ int turn_of(int k, int waves, int at) { return at / 8 * waves % (k / 64); }

// The weights of a wavefront's first step, requested while the rows are still being looked for (slot 0 begins with them, whatever MT);
// k a multiple of 64.
__device__ __forceinline__ void first_weights(const void* w, const uint32_t (&w_off)[4], int k, int wave, unsigned char* ring, int turn) {
    if (64 * wave >= k) return;
    const int t = wave + turn >= k / 64 ? wave + turn - k / 64 : wave + turn;
#pragma unroll
    for (int j = 0; j < 4; ++j) dma_to_lds_16((const char*)w + 128 * (int64_t)t, w_off[j], lds_address(ring) + j * 1024);
}

// w_off, a_off: byte offsets of this lane's 16 bytes in step 0: rows 8 j + lane / 8 of the weights (32) and of the activations
// (16 * MT), piece (lane % 8) ^ (lane / 8) of the row's eight, so that the LDS row holds piece q at q ^ (row % 8).
// k: row length in elements, a multiple of 8; meanwhile() runs when the first steps have been requested; on_rows(t, s, m, fragment) may
// change a fragment of activations: lane holds row 16 m + lane % 16, elements 64 t + 32 s + 8 (lane / 16) .. + 7 (zeros from k on).
// sent: first_weights has been called (its requests are older than all of these, so the waits count the same).
// acc[m][i]: lane holds row 16 m + lane % 16 of the activations, rows 16 i + 4 (lane / 16) .. + 3 of the weights.
// turn: the step that the wavefronts begin with, 0 <= turn < steps of k (TURN, with k a multiple of 64; else 0).  WAVES wavefronts share the steps; RING: bytes at `ring`, which
// hold one to three steps.
template <int MT, int WAVES, int RING, bool TURN, typename G, typename F>
__device__ __forceinline__ void weight_stream(const void* w, const uint32_t (&w_off)[4], const void* a, const uint32_t (&a_off)[2 * MT],
                                              int k, int turn, int wave, unsigned char* ring, f32x4 (&acc)[MT][2], G&& meanwhile, F&& on_rows, bool sent = false) {
    constexpr int kStep = (32 + 16 * MT) * 128, kDeep = RING / kStep, kLoads = 4 + 2 * MT;
    static_assert(kDeep >= 1 && kDeep <= 3, "ring");
    const int lane = threadIdx.x & 63, r = lane & 15, kg = lane >> 4;
    const uint32_t ring0 = lds_address(ring);
    const int n_steps = (k + 63) / 64;
    const auto turned = [&](int i) { return TURN && i + turn >= n_steps ? i + turn - n_steps : i + turn; };
    const auto request = [&](int i, int slot, bool weights = true) {
        const int t = turned(i);
        const char* wt = (const char*)w + 128 * (int64_t)t;
        const char* at = (const char*)a + 128 * (int64_t)t;
        // (pieces behind the end of a row: its first piece of this step once more)
        const uint32_t piece = (lane & 7) ^ (lane >> 3), back = 8 * (int)piece >= k - 64 * t ? 16 * piece : 0;
        if (weights)
#pragma unroll
            for (int j = 0; j < 4; ++j) dma_to_lds_16(wt, w_off[j] - back, ring0 + slot * kStep + j * 1024);
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) dma_to_lds_16(at, a_off[j] - back, ring0 + slot * kStep + (4 + j) * 1024);
    };
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < kDeep; ++d)
        if (wave + WAVES * d < n_steps) request(wave + WAVES * d, d, d > 0 || !sent);
    meanwhile();
    int slot = 0;
    for (int i0 = wave; i0 < n_steps; i0 += WAVES) {
        const int t = turned(i0);
        if (kDeep > 2 && i0 + 2 * WAVES < n_steps) wait_vmcnt<2 * kLoads>();
        else if (kDeep > 1 && i0 + WAVES < n_steps) wait_vmcnt<kLoads>();
        else wait_vmcnt<0>();
        const unsigned char* at = ring + slot * kStep;
        bf16x8 wf[2][2], af[MT][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int piece = ((4 * s + kg) ^ (r & 7)) * 16;
#pragma unroll
            for (int i = 0; i < 2; ++i) wf[i][s] = as_bf16x8(*reinterpret_cast<const u32x4*>(at + (16 * i + r) * 128 + piece));
#pragma unroll
            for (int m = 0; m < MT; ++m) af[m][s] = as_bf16x8(*reinterpret_cast<const u32x4*>(at + (32 + 16 * m + r) * 128 + piece));
        }
        if (k - 64 * t < 64) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (32 * s + 8 * kg >= k - 64 * t) {          // (the weights too: zero times an infinity is no zero)
#pragma unroll
                    for (int m = 0; m < MT; ++m) af[m][s] = as_bf16x8(u32x4{0u, 0u, 0u, 0u});
#pragma unroll
                    for (int i = 0; i < 2; ++i) wf[i][s] = as_bf16x8(u32x4{0u, 0u, 0u, 0u});
                }
        }
        if (i0 + WAVES * kDeep < n_steps) {
            wait_lgkmcnt0();                      // the slot's bytes are in registers
            request(i0 + WAVES * kDeep, slot);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int m = 0; m < MT; ++m) on_rows(t, s, m, af[m][s]);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[m][i] = mfma16(wf[i][s], af[m][s], acc[m][i]);
        slot = slot + 1 == kDeep ? 0 : slot + 1;
    }
}

}  // namespace mi355
