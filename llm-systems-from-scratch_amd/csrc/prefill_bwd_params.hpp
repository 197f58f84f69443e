// Arguments of the prefill backward kernels, and how they store gradients (shared by the two kernel files).
#pragma once
#include "common.hpp"

namespace mi355 {

// Units of a head in a launch's grid: pairs of tiles, or single ones; then also heads that an XCD takes at a time, and its compute units if all
// workgroups are resident at once (else 0)
struct BwdDeal {
    int units, chunk_heads, round;
    bool singles;
};

struct BwdParams {
    const __bf16* q;
    const __bf16* k;
    const __bf16* v;
    const __bf16* out;
    const __bf16* dout;
    const float* lse;
    float* delta;
    void* dq;                     // bf16 or fp32
    void* dk;
    void* dv;
    bool dq_f32, dk_f32, dv_f32;
    int64_t qs[3], ks[3], vs[3], os[3], dos[3], dqs[3], dks[3], dvs[3];   // batch, head, row strides (elements)
    int64_t ls[2];                                                          // lse / delta: batch, head strides
    const int32_t* cu_q;
    const int32_t* cu_k;
    const uint8_t* mask;          // MI355_MASK_BOOL: (B, Hq, Sq, Sk) bytes, non-zero = keep; rows 4-byte aligned
    int64_t ms[3];                // batch, head, row strides of the mask in bytes (0 = broadcast), multiples of 4
    int B, Hq, Hkv, Sq, Sk;
    float scale, scale_log2;
    int n_qtiles, n_ktiles;
    BwdDeal deal;                         // of bwd_dq_kernel and bwd_dkv_one_kernel
    // with dS in memory (see DsLayout): units of one pass over it, and for packed sequences the lists that the plan wrote
    unsigned char* ds;
    int unit0, n_units;           // dense: (sequence, kv head) pairs; packed: kv heads
    const int32_t* n_jobs;        // packed: entries of k_jobs and q_jobs
    const int32_t* ds_base;       // packed: blocks of one head in front of a sequence
    const int2* k_jobs;           // packed: (sequence, key tile), the dearest first
    const int2* q_jobs;           // packed: (sequence, set of kDqWaves (row tile, query head) pairs), the dearest first
    // row tiles of a key tile dealt to `shares` workgroups, whose sums meet in fp32: dk, then dv, each (shares, rows, Hkv, D)
    int shares;
    float* part;
    int64_t part_rows;
    bool wide;                    // dK, dV and dS by bwd_dkv_wide_kernel
};

// Gradients leave in bf16, or in fp32 for an fp32 input: the sums as they are, where a conversion behind the kernel would
// read and write them once more (64 x 16 heads x 256 x 32: 8.8 us each for dq and dk).
// Four adjacent elements at element offset `at`.
__device__ __forceinline__ void store_grad4(void* grad, bool f32, int64_t at, float a, float b, float c, float d) {
    if (f32) {
        *reinterpret_cast<f32x4*>((float*)grad + at) = f32x4{a, b, c, d};
    } else {
        u32x2 w;
        w[0] = pack_bf16(a, b);
        w[1] = pack_bf16(c, d);
        *reinterpret_cast<u32x2*>((__bf16*)grad + at) = w;
    }
}

// Up to 256 queries and keys at head sizes 32 and 64, dense layout, as many key heads as query heads: prefill_bwd_short.hip.
bool prefill_bwd_short_takes(int Hq, int Hkv, int Sq, int Sk, int D, int mask_mode);
int launch_prefill_bwd_short(const BwdParams& p, int D, int mask_mode, hipStream_t stream);

}  // namespace mi355
