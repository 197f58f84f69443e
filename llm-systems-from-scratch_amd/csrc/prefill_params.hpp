// Arguments of the prefill forward kernels (shared by the two kernel files).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "common.hpp"

namespace mi355 {

struct PrefillParams {
    const __bf16* q;
    const __bf16* k;
    const __bf16* v;
    __bf16* out;
    int64_t qs[3], ks[3], vs[3], os[3];   // batch, head, row strides (elements)
    const int32_t* cu_q;
    const int32_t* cu_k;
    const uint8_t* mask;
    int64_t ms[3];
    float* lse;                           // optional: natural-log sum of exp of the scaled scores, per query row
    int64_t ls[2];                        // its batch and head strides (elements); rows are contiguous
    int B, Hq, Hkv, Sq, Sk;
    float scale_log2;
    // optional per-query-head terms (forward only): a factor on the scores, and a sink -- a score without key or value
    // (natural-log units, not scaled) that only enters the softmax denominator, once per query row
    const float* head_scale;
    const float* sink;
    int mask_mode;
    int window, keep_first;               // causal only: query i sees key j when i - j < window or j < keep_first (window 0: every key j <= i)
    int n_qtiles;
    int n_pairs;                          // units per (batch, head) of prefill_fwd_kernel's grid: pairs of query tiles, or ...
    int single_tiles;                     // ... single query tiles when this is not 0; 1: by their number, and then also ...
    int chunk_heads, round;               // ... query heads that an XCD takes at a time, and its compute units if all workgroups are resident at once (else 0)
    // paged keys and values (prefill of a chunk on top of cached context): k, v are cache pools
    // (num_blocks, Hkv, 16, D); sequence b owns blocks block_table[b * table_stride + j] and ctx_lens[b] keys
    const int32_t* block_table;
    const int32_t* ctx_lens;
    int64_t table_stride;
    int num_blocks;
    int max_blocks;                       // entries of a table row that may be read: a longer context is cut to 16 * max_blocks keys
    // split keys (n_split > 1): workgroup (.., split c) serves the c-th share of every query tile's K/V tiles and
    // writes, instead of `out`, a normalised fp32 partial result and its log-sum-exp per query row:
    //   part_o  (n_split, Hq, part_rows, D)    part_lse (n_split, Hq, part_rows)
    // row = packed row, or b * Sq + i in the dense layout; a second kernel merges the partials into `out`
    int n_split;
    float* part_o;
    float* part_lse;
    int64_t part_rows;
};

// The 64-queries-per-wavefront kernel (head_dim 128, no mask or causal): prefill_fwd_w64.hip.
// prefill_w64_takes: whether its 32-bit address arithmetic covers the strides of p.
bool prefill_w64_takes(const PrefillParams& p);
int launch_prefill_w64(const PrefillParams& p, hipStream_t stream);

// Up to 256 keys at head sizes 32 and 64, dense layout: prefill_short.hip.
bool prefill_short_takes(const PrefillParams& p, int D);
int launch_prefill_short(const PrefillParams& p, int D, hipStream_t stream);
// The same with fp32 among q, k and v: what is given here (else null) is read in place of p's and leaves rounded in bf16 where there is an out.
struct RoundedInputs {
    const float* in[3];                   // with p's strides
    __bf16* out[3];
    int64_t strides[3][3];                // of out: batch, head, row
};
// Operands whose elements fill their memory
struct RoundedOperands {
    const float* in[3];
    __bf16* out[3];
    int64_t n[3], room[3];                // elements; rounded up to eight
};
int launch_round_operands(const float* const in[3], __bf16* const out[3], const int64_t n[3], hipStream_t stream);
int launch_prefill_short_rounded(const PrefillParams& p, const RoundedInputs& r, int D, hipStream_t stream);

// Small query tiles whose keys are dealt to a workgroup's wavefronts: prefill_keys.hip.  The plan: how many wavefronts, and about how long it takes.
struct PrefillKeysPlan {
    int wavefronts;
    double us;
};
// Two times of which the longer one counts, and more where they are alike (the larger the power, the less)
inline double together(double a, double b, double power) { return std::pow(std::pow(a, power) + std::pow(b, power), 1.0 / power); }
bool prefill_keys_takes(const PrefillParams& p, int D);
PrefillKeysPlan prefill_keys_plan(int B, int Hq, int D, int Sq, int Sk, bool causal, int n_cu);
int launch_prefill_keys(const PrefillParams& p, int D, int wavefronts, hipStream_t stream);

}  // namespace mi355
