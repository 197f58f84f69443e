// FlashAttention-style prefill backward for gfx950 (bf16, MFMA 32x32x16): dQ, dK, dV from
// q, k, v, out, dout and the forward's log-sum-exp.  No atomics; results are deterministic.
//
//   delta_i = sum_d dO[i,d] * O[i,d]                       (computed, and stored, by the dQ kernel)
//   P_ij    = exp(scale * q_i.k_j - lse_i)                 (recomputed, never stored)
//   dV_j    = sum_i P_ij dO_i                              (bwd_dkv_kernel: one workgroup per key tile,
//   dP_ij   = dO_i . v_j                                    summing over the query heads of a GQA group;
//   dS_ij   = P_ij (dP_ij - delta_i)                        dV on half of its wavefronts, dK on the other half;
//   dK_j    = scale * sum_i dS_ij q_i                       head sizes 32 and 64: bwd_dkv_one_kernel)
//   dQ_i    = scale * sum_j dS_ij k_j                      (bwd_dq_kernel: one workgroup per query tile)
//
// With a workspace (mi355_prefill_bwd_ds): bwd_delta_kernel computes delta, the dK/dV kernel also writes dS (bf16, as
// it enters the MFMAs), and bwd_dq_ds_kernel is one product over it: 5 GEMM-sized products where the form above executes 7.
//
// Both kernels work on transposed problems, like the forward: the wavefront owns 32 columns
// (queries in the dQ kernel, keys in the dK/dV kernel) whose operand fragments stay in
// registers; the other side streams through LDS tiles of 64 rows.  The accumulator of the first
// MFMA (S or dP, column = lane) is, converted to bf16, directly the B operand of the second
// (dQ^T += K^T dS^T; dV^T += dO^T P, dK^T += Q^T dS), and the matching A operand is a transposed
// LDS read (ds_read_b64_tr_b16) of the streamed tile with the same row permutation.
// Without dS in memory 7 GEMM-sized products are executed (S and dP in both kernels) where 5 are needed.
//
// Masks: none, causal (bottom-right aligned, as in the forward), or an explicit boolean keep-mask (the mask argument
// of llm-core/llm_core/model.py:308-325, which its non-flash branch passes at model.py:384-385).  The explicit mask is
// the general, slower path: every tile takes the per-element select and reads its mask bytes from global memory.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "prefill_bwd_params.hpp"
#include "xcd_order.hpp"
#include "prefill_tile.hpp"

namespace mi355 {

constexpr int kBwWaves = 8;
constexpr int kBwCols = 32 * kBwWaves;   // query columns per workgroup of the dQ kernel (one workgroup of 8 wavefronts per CU)
constexpr int kBwRows = 64;              // rows of a streamed LDS tile

// dS in memory: blocks of 64 query rows x 32 keys, 4 KiB, as the dK/dV kernel's lanes hold them.  A head's blocks go by row tile,
// inside it by keys, and are only those that some row of the tile sees.
constexpr int kDsBlock = 4096, kDsKeys = 32, kDqWaves = 4;
constexpr int kFuPairs = 4;               // pairs of wavefronts of the dK/dV kernel, 32 keys each
constexpr int kFuCols = 32 * kFuPairs;

// (T: int64_t where the number of blocks is asked for, int where it is known to fit)
template <typename T>
struct DsLayoutOf {
    T n_kb, first, lo, hi;        // key blocks; row tile r has clamp(first + 2 r, 0, n_kb) of them, none up to lo, all from hi on
    __host__ __device__ __forceinline__ DsLayoutOf(T sq, T sk, bool causal) {
        n_kb = (sk + kDsKeys - 1) / kDsKeys;
        first = causal ? ((sk - sq + kBwRows - 1) >> 5) + 1 : n_kb;
        lo = first > 0 ? 0 : (-first >> 1) + 1;
        hi = n_kb > first ? (n_kb - first + 1) >> 1 : 0;
        hi = hi > lo ? hi : lo;
    }
    __host__ __device__ __forceinline__ T count(T r) const { return r < lo ? 0 : r < hi ? first + 2 * r : n_kb; }
    __host__ __device__ __forceinline__ T before(T r) const {                      // blocks of the row tiles in front of r
        const T m = r < lo ? lo : r < hi ? r : hi;
        return (m - lo) * first + m * (m - 1) - lo * (lo - 1) + (r > hi ? (r - hi) * n_kb : 0);
    }
};
using DsLayout = DsLayoutOf<int>;

// Loader of a 64-row tile (rows of D bf16, row stride `stride` elements) into swizzled LDS:
// wavefront w, instruction j covers LDS chunks (w*NI + j)*64 .. +63; rows past `last` re-read row `last`.
template <int D, int NW>
struct TileLoader {
    static constexpr int CPR = D / 8;
    static constexpr int TOTAL = kBwRows * CPR / 64;            // 1 KiB instructions per tile
    static constexpr int NI = (TOTAL + NW - 1) / NW;            // per wavefront (the last wavefronts may have none)
    int row[NI], col[NI];
    bool active;
    __device__ __forceinline__ void init(int wave, int lane) {
        active = wave * NI < TOTAL;
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int idx = (wave * NI + j) * 64 + lane;
            row[j] = idx / CPR;
            col[j] = ((idx % CPR) ^ swz<D>(idx / CPR)) * 16;
        }
    }
    __device__ __forceinline__ void issue(const __bf16* first_row, int stride, int last, uint32_t lds_wave_base) const {
        if (!active) return;
#pragma unroll
        for (int j = 0; j < NI; ++j)
            dma_to_lds_16(first_row, (uint32_t)(min(row[j], last) * stride * 2 + col[j]), lds_wave_base + j * 1024);
    }
};

// ---------------------------------------------------------------------------------------------
// dQ: one workgroup of NWV wavefronts per 32 NWV queries of one (batch, query head); K/V stream through LDS.
// Per wavefront: Q and dO fragments of its 32 query columns in registers (64), dQ^T accumulators (64).
// NWV 4 at head sizes 64 and 32: three and four workgroups per compute unit (165 and 120 registers), where of eight wavefronts one is all that 161
// registers leave at 64.  They wait less for the wavefront with the most keys and a launch is dealt finer (as in prefill_fwd_kernel).
// us, eight wavefronts and pairs of tiles / four and single tiles, causal: heads of 64: 136 of 700 tokens 57 / 27, 136 of 1456 100 / 72, 64 of 3000 168 /
// 119, 64 of 8192 869 / 774; 35 packed of 269 to 2871, 32 heads, 1136 / 805; heads of 32: 136 of 700 31 / 18, 64 of 3000 98 / 76, 256 of 1456 86 / 78.
constexpr int dq_resident(int D) { return D == 32 ? 4 : 3; }                        // workgroups of four wavefronts per compute unit
template <int D, int MODE, int NWV>
__global__ __launch_bounds__(NWV * 64, NWV == 4 ? dq_resident(D) : 1) void bwd_dq_kernel(BwdParams p) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL, BOOLM = MODE == MI355_MASK_BOOL;
    constexpr int BM = 32 * NWV;                  // queries per workgroup
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, kTile = kBwRows * kRow;
    // [K buffer 0][K buffer 1][V buffer 0][V buffer 1]
    __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kTile];

    // Workgroup ids are dealt round-robin to the 8 XCDs (private L2s) and, in order, to their shader
    // engines: a periodic heavy/light pattern starves the engines that always draw the light ones, and the workgroups that stream
    // the same K/V should share an XCD.  So a workgroup takes the query-tile PAIR (nq-1-i, i), and the pairs and query heads of
    // one kv head -- a chunk of the logical order (pair, query head, batch) -- run on one XCD; or one tile, the dearest of the
    // launch first.
    const bool singles = p.deal.singles;
    int pair, head;
    if (singles) {
        const HeadUnit at = xcd_unit(blockIdx.x, p.deal.units, p.Hq / p.Hkv, p.Hkv * p.B, p.deal.chunk_heads, p.deal.round);
        if (at.unit < 0) return;
        pair = p.deal.units - 1 - at.unit;
        head = at.head;
    } else {
        const int lid = xcd_chunked_id(blockIdx.x, gridDim.x, p.deal.units * (p.Hq / p.Hkv));
        pair = lid % p.deal.units;
        head = lid / p.deal.units;
    }
    pair = __builtin_amdgcn_readfirstlane(pair);
    const int b = __builtin_amdgcn_readfirstlane(head / p.Hq), h = __builtin_amdgcn_readfirstlane(head - b * p.Hq);
    const int hk = h / (p.Hq / p.Hkv);
    int sq, sk;
    int64_t q_base, k_base, v_base, do_base, dq_base, l_base, o_base;
    if (p.cu_q) {
        const int q_start = p.cu_q[b], k_start = p.cu_k[b];
        sq = p.cu_q[b + 1] - q_start;
        sk = p.cu_k[b + 1] - k_start;
        o_base = (int64_t)q_start * p.os[2] + (int64_t)h * p.os[1];
        q_base = (int64_t)q_start * p.qs[2] + (int64_t)h * p.qs[1];
        do_base = (int64_t)q_start * p.dos[2] + (int64_t)h * p.dos[1];
        dq_base = (int64_t)q_start * p.dqs[2] + (int64_t)h * p.dqs[1];
        k_base = (int64_t)k_start * p.ks[2] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)k_start * p.vs[2] + (int64_t)hk * p.vs[1];
        l_base = q_start + (int64_t)h * p.ls[1];
    } else {
        sq = p.Sq;
        sk = p.Sk;
        o_base = (int64_t)b * p.os[0] + (int64_t)h * p.os[1];
        q_base = (int64_t)b * p.qs[0] + (int64_t)h * p.qs[1];
        do_base = (int64_t)b * p.dos[0] + (int64_t)h * p.dos[1];
        dq_base = (int64_t)b * p.dqs[0] + (int64_t)h * p.dqs[1];
        k_base = (int64_t)b * p.ks[0] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)b * p.vs[0] + (int64_t)hk * p.vs[1];
        l_base = (int64_t)b * p.ls[0] + (int64_t)h * p.ls[1];
    }
    const int nq = (sq + BM - 1) / BM;
    if ((singles ? pair : 2 * pair) >= nq) return;                                         // (a sequence without keys still gets dq = 0 written)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int coff = sk - sq;

    TileLoader<D, NWV> ld;
    ld.init(wave, lane);
    R rd;
    rd.init(lane);
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_address(lds) + wave * TileLoader<D, NWV>::NI * 1024);

    // single tiles: one, unless a packed sequence is longer than the caller said
    for (int half = 0, qtile = singles ? pair : nq - 1 - pair; singles ? qtile < nq : half < 2; ++half, qtile = singles ? qtile + p.deal.units : pair) {
        if (!singles && half == 1 && pair == nq - 1 - pair) break;                 // odd tile count: the middle tile has no partner
        const int q0 = qtile * BM;
        const int qw0 = q0 + 32 * wave;
        const int qi = qw0 + n;
        const bool q_ok = qi < sq;
        __syncthreads();                                                // the previous half's readers are done with the LDS buffers

        // fragments of this lane's query column: step s covers d = 16s + 8kg + j
        bf16x8 qf[NS], dof[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            u32x4 a = {0u, 0u, 0u, 0u}, g = {0u, 0u, 0u, 0u};
            if (q_ok) {
                a = *reinterpret_cast<const u32x4*>(p.q + q_base + (int64_t)qi * p.qs[2] + 16 * s + 8 * kg);
                g = *reinterpret_cast<const u32x4*>(p.dout + do_base + (int64_t)qi * p.dos[2] + 16 * s + 8 * kg);
            }
            qf[s] = as_bf16x8(a);
            dof[s] = as_bf16x8(g);
        }
        // a padded query column gets lse = +inf, i.e. P = 0 everywhere
        const float lse2 = q_ok ? p.lse[l_base + qi] * kLog2e : INFINITY;
        // delta = rowsum(dO * O) of this lane's query: each lane of the pair (kg = 0, 1) covers half of d.
        // It is also written out: the dK kernel, launched after this one, reads it per row.
        float delta = 0.f;
        if (q_ok) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const bf16x8 o8 = as_bf16x8(*reinterpret_cast<const u32x4*>(p.out + o_base + (int64_t)qi * p.os[2] + 16 * s + 8 * kg));
#pragma unroll
                for (int e = 0; e < 8; ++e) delta += (float)o8[e] * (float)dof[s][e];
            }
        }
        delta = xor32_sum(delta);
        if (q_ok && kg == 0) p.delta[l_base + qi] = delta;

        f32x16 dq[NDT];
#pragma unroll
        for (int i = 0; i < NDT; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) dq[i][j] = 0.f;
        const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        // dP - delta comes straight out of the MFMAs: -delta (one value per lane: its query) is their C operand
        f32x16 neg_delta16;
#pragma unroll
        for (int j = 0; j < 16; ++j) neg_delta16[j] = -delta;

        int kv_end = sk;
        if (CAUSAL) kv_end = max(0, min(sk, min(sq, q0 + BM) + coff));
        const int n_tiles = (kv_end + kBwRows - 1) / kBwRows;
        const int last_key = CAUSAL ? min(sk - 1, qi + coff) : sk - 1;      // last key this lane's query sees
        const int wave_last_key = CAUSAL ? min(sk - 1, qw0 + coff) : sk - 1;   // ... and the last one ALL queries of the wavefront see
        // explicit mask: the row of this lane's query (a padded lane re-reads the last row; its lse keeps P at 0);
        // four keys at a time as one 32-bit word (rows are 4-byte aligned; a word past the last key is the last word)
        const uint8_t* mrow = nullptr;
        if constexpr (BOOLM) mrow = p.mask + (int64_t)b * p.ms[0] + (int64_t)h * p.ms[1] + (int64_t)min(qi, sq - 1) * p.ms[2];
        const int last_word = (sk - 1) & ~3;
        const auto issue = [&](int tile) {
            const int r0 = tile * kBwRows, buf = (tile & 1) * kTile;
            ld.issue(p.k + k_base + (int64_t)r0 * p.ks[2], (int)p.ks[2], sk - 1 - r0, dst + buf);
            ld.issue(p.v + v_base + (int64_t)r0 * p.vs[2], (int)p.vs[2], sk - 1 - r0, dst + 2 * kTile + buf);
        };
        // The LDS fragments of every MFMA are read kDepth MFMAs ahead, in program order, fenced by scheduling
        // barriers: left alone the compiler puts each read, and a full wait, directly in front of its MFMA,
        // and the wavefront then sits through the LDS latency once per MFMA.
        constexpr int kDepth = 2;
        // (32 rows of the tile at a_lds) x (this lane's query column, fragments b)
        const auto scores = [&](const unsigned char* a_lds, const bf16x8 (&bfr)[NS], const f32x16& c0) {
            u32x4 a[NS];
#pragma unroll
            for (int s = 0; s < kDepth && s < NS; ++s) a[s] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s]);
            f32x16 r = c0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + kDepth < NS) a[s + kDepth] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s + kDepth]);
                r = mfma32(as_bf16x8(a[s]), bfr[s], r);
                __builtin_amdgcn_sched_barrier(0);
            }
            return r;
        };
        const auto step = [&](auto masked_c, int tile) {
            constexpr bool MASKED = decltype(masked_c)::value;
            const int k0 = tile * kBwRows;
            const unsigned char* k_lds = lds + (tile & 1) * kTile;
            const unsigned char* v_lds = k_lds + 2 * kTile;
            const int key_lim = last_key - k0 - 4 * kg;      // element (t,i) is kept iff its tile-relative key index <= key_lim
            u32x4 ds[4];
            uint32_t mw[8] = {};
            if constexpr (BOOLM && MASKED) {
#pragma unroll
                for (int g = 0; g < 8; ++g)      // keys k0 + 32(g/4) + 8(g%4) + 4kg .. + 3
                    mw[g] = *reinterpret_cast<const uint32_t*>(mrow + min(k0 + 32 * (g >> 2) + 8 * (g & 3) + 4 * kg, last_word));
            }
            // one 32-key half at a time: element i of this lane is key k0 + 32t + 8(i/4) + 4kg + i%4, query qi
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const f32x16 s_acc = scores(k_lds + t * 32 * kRow, qf, zero16);
                const f32x16 dp_acc = scores(v_lds + t * 32 * kRow, dof, neg_delta16);             // dP - delta
                float x[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float pr = fast_exp2(fmaf(s_acc[i], p.scale_log2, -lse2));
                    x[i] = pr * dp_acc[i];                                             // dS (without the scale factor)
                    if constexpr (MASKED) {
                        // key index relative to the tile (compile-time part) against this lane's last visible key
                        bool keep = 32 * t + 8 * (i >> 2) + (i & 3) <= key_lim;
                        if constexpr (BOOLM) keep = keep & (((mw[4 * t + (i >> 2)] >> (8 * (i & 3))) & 0xffu) != 0u);
                        x[i] = keep ? x[i] : 0.f;
                    }
                }
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    ds[2 * t][w] = pack_bf16(x[2 * w], x[2 * w + 1]);
                    ds[2 * t + 1][w] = pack_bf16(x[8 + 2 * w], x[8 + 2 * w + 1]);
                }
            }
            // dQ^T (D x 32 queries) += K^T . dS^T, 16 keys at a time
            constexpr int NC = 4 * NDT;
            i16x4 lo[NC], hi[NC];
            const auto read = [&](int c) {
                const int u = c / NDT, dt = c % NDT;
                lo[c] = lds_read_tr16(k_lds + 16 * u * kRow + rd.tr_off[0][dt]);
                hi[c] = lds_read_tr16(k_lds + 16 * u * kRow + rd.tr_off[1][dt]);
            };
#pragma unroll
            for (int c = 0; c < kDepth && c < NC; ++c) read(c);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (c + kDepth < NC) read(c + kDepth);
                dq[c % NDT] = mfma32(join_bf16x8(lo[c], hi[c]), as_bf16x8(ds[c / NDT]), dq[c % NDT]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        // Two loops over the tile stream: first the tiles that every query of the wavefront sees in full, then
        // those that reach past wave_last_key (the diagonal, a ragged end), which run the instantiation with the
        // per-element compare/select.  (Two loops, not a branch in one: each loop body is scheduled on its own.)
        const int n_full = BOOLM ? 0 : min(n_tiles, max(0, wave_last_key + 1) / kBwRows);
        if (n_tiles > 0) issue(0);
        for (int tile = 0; tile < n_full; ++tile) {
            wait_vmcnt<0>();                                   // this wavefront's share of tile `tile` has landed
            __syncthreads();                                   // ... and everybody's; all are done reading the other buffer
            if (tile + 1 < n_tiles) issue(tile + 1);
            step(std::false_type{}, tile);
        }
        for (int tile = n_full; tile < n_tiles; ++tile) {
            wait_vmcnt<0>();
            __syncthreads();
            if (tile + 1 < n_tiles) issue(tile + 1);
            if (CAUSAL && tile * kBwRows > qw0 + 31 + coff) continue;      // wholly above this wavefront's diagonal (uniform)
            step(std::true_type{}, tile);
        }

        // store: lane owns query qi, d = 32dt + 8(i/4) + 4kg + i%4
        if (q_ok) {
            const int64_t row = dq_base + (int64_t)qi * p.dqs[2];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    store_grad4(p.dq, p.dq_f32, row + 32 * dt + 8 * g + 4 * kg, dq[dt][4 * g + 0] * p.scale, dq[dt][4 * g + 1] * p.scale,
                                dq[dt][4 * g + 2] * p.scale, dq[dt][4 * g + 3] * p.scale);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// dK and dV in one kernel, the two roles on different wavefronts: a workgroup owns 128 keys of one
// (batch, kv head); wavefronts 0-3 (role A) hold the K fragments of 32 keys each and the dV
// accumulators, wavefronts 4-7 (role B) hold the V fragments of the same keys and the dK accumulators
// (each role fits 256 registers, so two wavefronts share a SIMD - an A and a B wavefront).  Per step
// (64 query rows of one query head):
//   A:  S = Q K^T,  P = exp2(S c - lse)  -> LDS (fp32, for B) and registers (bf16),  dV^T += dO^T P
//   B:  dP = dO V^T,  dS = P (dP - delta)  with A's P from LDS,                        dK^T += Q^T dS
// so S is computed once for both gradients (4 GEMM-sized products per step instead of 2 + 3 in two
// kernels).  A runs one step ahead of B with its P: at iteration i, A produces P(i+1) while B consumes
// P(i), and the only synchronisation is the one workgroup barrier per iteration that the tile stream
// needs anyway.  Q tiles therefore live for three iterations (landing, read by A, read by B): a ring
// of three; dO tiles, read by both roles in the same iteration, alternate between two buffers.
//
// DS: dS also goes to memory, and a workgroup takes one key tile instead of a pair, the dearest of the launch first: with
// unequal lengths the last workgroups are then short ones.  Writing dS costs 14 % of the kernel (8 x 4096 tokens, 32 / 8 heads: 2340
// us against 2740 at 1.9 GHz, where the board holds it), and takes two of the three products of bwd_dq_kernel away: all kernels of
// the backward 3640 -> 3480 us there, 16 packed sequences of 256 to 4096 tokens 1850 -> 1460, 40 of 50 to 800 192 -> 100.
template <int D, int MODE, bool DS>
__global__ __launch_bounds__(2 * kFuPairs * 64, 1) void bwd_dkv_kernel(BwdParams p) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL, BOOLM = MODE == MI355_MASK_BOOL;
    static_assert(!DS || !BOOLM, "dS goes to memory without an explicit mask");
    constexpr int NWV = 2 * kFuPairs;
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, kTile = kBwRows * kRow;
    constexpr int kPSlab = 64 * 32 * 4;                              // one wavefront's P of one step, fp32
    // [Q ring 0..2][dO buffer 0..1][P: 2 x kFuPairs slabs]
    __shared__ __attribute__((aligned(1024))) unsigned char lds[5 * kTile + 2 * kFuPairs * kPSlab];
    __shared__ __attribute__((aligned(16))) float lse_lds2[2 * kBwRows];
    __shared__ __attribute__((aligned(16))) float delta_lds2[2 * kBwRows];

    int pair, hk, b, share = 0;                                         // (DS: the key tile in place of a pair)
    if constexpr (DS) {
        const int places = p.n_units * p.shares, id = (int)blockIdx.x / places, place = (int)blockIdx.x % places;
        const int unit = p.unit0 + place / p.shares;
        share = place % p.shares;
        if (p.cu_q) {
            if (id >= p.n_jobs[0]) return;
            const int2 job = p.k_jobs[id];
            b = job.x;
            pair = job.y;
            hk = unit;
        } else {
            pair = id;
            b = unit / p.Hkv;
            hk = unit % p.Hkv;
        }
    } else {
        // (the key-tile pairs of one (batch, kv head), which stream the same Q and dO tiles, run on one XCD)
        const int n_pairs = (p.n_ktiles + 1) / 2;
        const int lid = xcd_chunked_id(blockIdx.x, gridDim.x, n_pairs);
        pair = lid % n_pairs;
        hk = (lid / n_pairs) % p.Hkv;
        b = lid / (n_pairs * p.Hkv);
    }
    const int G = p.Hq / p.Hkv;
    int sq, sk, q_start = 0;
    int ds_base = 0;                                                    // (DS, packed: negative: no room for the sequence, its gradients are zero)
    int64_t k_base, v_base, dk_base, dv_base;
    if (p.cu_q) {
        q_start = p.cu_q[b];
        const int k_start = p.cu_k[b];
        sq = p.cu_q[b + 1] - q_start;
        sk = p.cu_k[b + 1] - k_start;
        if constexpr (DS) {                                             // (as the plan counts them)
            sq = max(sq, 0);
            sk = max(sk, 0);
            ds_base = p.ds_base[b];
        }
        k_base = (int64_t)k_start * p.ks[2] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)k_start * p.vs[2] + (int64_t)hk * p.vs[1];
        dk_base = (int64_t)k_start * p.dks[2] + (int64_t)hk * p.dks[1];
        dv_base = (int64_t)k_start * p.dvs[2] + (int64_t)hk * p.dvs[1];
    } else {
        sq = p.Sq;
        sk = p.Sk;
        k_base = (int64_t)b * p.ks[0] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)b * p.vs[0] + (int64_t)hk * p.vs[1];
        dk_base = (int64_t)b * p.dks[0] + (int64_t)hk * p.dks[1];
        dv_base = (int64_t)b * p.dvs[0] + (int64_t)hk * p.dvs[1];
    }
    const int nk = (sk + kFuCols - 1) / kFuCols;
    if (!DS && 2 * pair >= nk) return;                                  // (a sequence without queries still gets dk = dv = 0 written)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool role_b = wave >= kFuPairs;
    const int pw = wave & (kFuPairs - 1);
    const int n = lane & 31, kg = lane >> 5;
    const int coff = sk - sq;

    TileLoader<D, NWV> ld;
    ld.init(wave, lane);
    R rd;
    rd.init(lane);
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_address(lds) + wave * TileLoader<D, NWV>::NI * 1024);
    unsigned char* const p_lds = lds + 5 * kTile + pw * kPSlab + lane * 16;       // + parity * kFuPairs * kPSlab + 1024 * vector
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    for (int half = 0; half < (DS ? 1 : 2); ++half) {
        const int ktile = half == 0 ? pair : nk - 1 - pair;
        if (half == 1 && ktile == pair) break;                          // odd tile count: the middle tile has no partner
        const int k0 = ktile * kFuCols;
        const int kw0 = k0 + 32 * pw;
        const int kj = kw0 + n;
        const bool k_ok = kj < sk;
        __syncthreads();                                                // the previous half's readers are done with the LDS buffers

        // fragments of this lane's key column (K for role A, V for role B): step s covers d = 16s + 8kg + j
        bf16x8 frag[NS];
        {
            const __bf16* src = role_b ? p.v + v_base + (int64_t)kj * p.vs[2] : p.k + k_base + (int64_t)kj * p.ks[2];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                u32x4 a = {0u, 0u, 0u, 0u};
                if (k_ok) a = *reinterpret_cast<const u32x4*>(src + 16 * s + 8 * kg);
                frag[s] = as_bf16x8(a);
            }
        }
        f32x16 acc[NDT];
#pragma unroll
        for (int i = 0; i < NDT; ++i) acc[i] = zero16;

        int first_tile = 0;
        if (CAUSAL) first_tile = max(0, k0 - coff) / kBwRows;
        const int n_tiles = (sq + kBwRows - 1) / kBwRows;
        // Steps: (query head of the group, row tile), heads innermost; the first key tile of the pair walks
        // its row tiles from the last one down, the second from its first one up, which keeps all workgroups
        // of a (batch, kv head) on the same Q/dO tiles at the same time (they share them through the L2).
        const int n_steps = DS && ds_base < 0 ? 0 : G * (DS ? max(0, n_tiles - first_tile - share + p.shares - 1) / p.shares : max(0, n_tiles - first_tile));
        // position of a step: first row of its tile and query head within the group; advanced incrementally
        // (steps i, i+1 and i+2 are in flight at any time; no division per step)
        struct Pos {
            int r0, hq;
        };
        const int r_step = DS ? -kBwRows * p.shares : half == 0 ? -kBwRows : kBwRows;
        const auto advance = [&](Pos ps) {
            ++ps.hq;
            if (ps.hq == G) {
                ps.hq = 0;
                ps.r0 += r_step;
            }
            return ps;
        };
        // a step whose rows all lie above this wavefront's first key column has nothing for it (uniform)
        const auto idle = [&](Pos ps) { return CAUSAL && kw0 > ps.r0 + kBwRows - 1 + coff; };

        float pend_lse = 0.f, pend_delta = 0.f;      // (delta_lds2 holds -delta)
        const auto bases = [&](Pos ps, int64_t& q_base, int64_t& do_base, int64_t& l_base) {
            const int h = hk * G + ps.hq;
            if (p.cu_q) {
                q_base = (int64_t)q_start * p.qs[2] + (int64_t)h * p.qs[1];
                do_base = (int64_t)q_start * p.dos[2] + (int64_t)h * p.dos[1];
                l_base = q_start + (int64_t)h * p.ls[1];
            } else {
                q_base = (int64_t)b * p.qs[0] + (int64_t)h * p.qs[1];
                do_base = (int64_t)b * p.dos[0] + (int64_t)h * p.dos[1];
                l_base = (int64_t)b * p.ls[0] + (int64_t)h * p.ls[1];
            }
        };
        // Q tile of step st (at ps) into ring slot `slot`; its lse into a register
        const auto issue_q = [&](Pos ps, int slot) {
            int64_t q_base, do_base, l_base;
            bases(ps, q_base, do_base, l_base);
            const int r0 = ps.r0;
            ld.issue(p.q + q_base + (int64_t)r0 * p.qs[2], (int)p.qs[2], sq - 1 - r0, dst + slot * kTile);
            const float* rows = p.lse + l_base + r0;                                   // uniform base, 32-bit lane offset
            if (tid < kBwRows) pend_lse = rows[(unsigned)min(tid, sq - 1 - r0)];       // consumed only by publish_lse
        };
        const auto issue_do = [&](int st, Pos ps) {
            int64_t q_base, do_base, l_base;
            bases(ps, q_base, do_base, l_base);
            const int r0 = ps.r0;
            ld.issue(p.dout + do_base + (int64_t)r0 * p.dos[2], (int)p.dos[2], sq - 1 - r0, dst + (3 + (st & 1)) * kTile);
            const float* rows = p.delta + l_base + r0;
            if (tid < kBwRows) pend_delta = rows[(unsigned)min(tid, sq - 1 - r0)];
        };
        // (the values are scaled and masked here, not where they are loaded: consuming them there would put a
        // wait for all outstanding loads - the tiles just issued - in front of the step's arithmetic)
        const auto publish_lse = [&](int st, Pos ps) {
            if (tid < kBwRows) lse_lds2[(st & 1) * kBwRows + tid] = ps.r0 + tid < sq ? pend_lse * kLog2e : INFINITY;
        };
        const auto publish_delta = [&](int st, Pos ps) {
            // a causal row that sees no key has out = NaN, hence delta = NaN, and P = 0 everywhere: any finite
            // delta gives the dS = 0 it must have
            if (tid < kBwRows)
                delta_lds2[(st & 1) * kBwRows + tid] = (ps.r0 + tid < sq && pend_delta == pend_delta) ? -pend_delta : 0.f;
        };

        // second GEMM of either role: acc^T (D x 32 keys) += tile^T . W, 16 query rows at a time.
        // The transposed fragments are read kDepth MFMAs ahead, in this order, fenced by scheduling barriers:
        // left alone the compiler puts each pair of reads, and a full wait, directly in front of its MFMA.
        constexpr int kDepth = 2;
        const auto update = [&](const unsigned char* a_lds, const u32x4 (&w)[4]) {
            constexpr int NC = 4 * NDT;
            i16x4 lo[NC], hi[NC];
            const auto read = [&](int c) {
                const int u = c / NDT, dt = c % NDT;
                lo[c] = lds_read_tr16(a_lds + 16 * u * kRow + rd.tr_off[0][dt]);
                hi[c] = lds_read_tr16(a_lds + 16 * u * kRow + rd.tr_off[1][dt]);
            };
#pragma unroll
            for (int c = 0; c < kDepth && c < NC; ++c) read(c);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (c + kDepth < NC) read(c + kDepth);
                acc[c % NDT] = mfma32(join_bf16x8(lo[c], hi[c]), as_bf16x8(w[c / NDT]), acc[c % NDT]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // first GEMM of either role: (32 rows of the tile at a_lds) x (this lane's key column), fragments read ahead likewise
        const auto scores = [&](const unsigned char* a_lds, const f32x16& c0) {
            u32x4 a[NS];
#pragma unroll
            for (int s = 0; s < kDepth && s < NS; ++s) a[s] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s]);
            f32x16 r = c0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + kDepth < NS) a[s + kDepth] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s + kDepth]);
                r = mfma32(as_bf16x8(a[s]), frag[s], r);
                __builtin_amdgcn_sched_barrier(0);
            }
            return r;
        };
        // role A: P of step st from the Q tile in ring slot `slot`: fp32 to LDS for role B, bf16 into p_cur
        u32x4 p_cur[4];
        const auto make_p = [&](auto masked_c, int st, Pos ps, int slot) {
            constexpr bool MASKED = decltype(masked_c)::value;
            const unsigned char* q_lds = lds + slot * kTile;
            const float* lse_lds = lse_lds2 + (st & 1) * kBwRows;
            unsigned char* out = p_lds + (st & 1) * (kFuPairs * kPSlab);
            const int row_lim = CAUSAL ? kj - coff - ps.r0 - 4 * kg : -1;
            // explicit mask: the bytes (row, this lane's key) of the step's 64 rows (a row or key past the end re-reads
            // the last one: its P is 0 through lse = inf, or its column is never stored)
            uint8_t mb[32] = {};
            if constexpr (BOOLM && MASKED) {
                const uint8_t* mcol = p.mask + (int64_t)b * p.ms[0] + (int64_t)(hk * G + ps.hq) * p.ms[1] + min(kj, sk - 1);
#pragma unroll
                for (int e = 0; e < 32; ++e)     // row r0 + 32(e/16) + 8((e/4)%4) + 4kg + e%4
                    mb[e] = mcol[(int64_t)min(ps.r0 + 32 * (e >> 4) + 8 * ((e >> 2) & 3) + 4 * kg + (e & 3), sq - 1) * p.ms[2]];
            }
            // one 32-row half at a time: element i of this lane is query row r0 + 32t + 8(i/4) + 4kg + i%4, key kj
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const f32x16 s_acc = scores(q_lds + t * 32 * kRow, zero16);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 l4 = *reinterpret_cast<const f32x4*>(lse_lds + 32 * t + 8 * j + 4 * kg);
                    f32x4 x4;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float x = fast_exp2(fmaf(s_acc[4 * j + r], p.scale_log2, -l4[r]));
                        // kept iff kj <= row + coff, i.e. the tile-relative row (compile-time part) >= row_lim
                        if constexpr (MASKED) {
                            bool keep = 32 * t + 8 * j + r >= row_lim;
                            if constexpr (BOOLM) keep = keep & (mb[16 * t + 4 * j + r] != 0);
                            x = keep ? x : 0.f;
                        }
                        x4[r] = x;
                    }
                    *reinterpret_cast<f32x4*>(out + (4 * t + j) * 1024) = x4;
                    p_cur[2 * t + (j >> 1)][2 * (j & 1)] = pack_bf16(x4[0], x4[1]);
                    p_cur[2 * t + (j >> 1)][2 * (j & 1) + 1] = pack_bf16(x4[2], x4[3]);
                }
            }
        };
        // where this wavefront's dS blocks of its kv head begin
        const DsLayout dsl(sq, sk, CAUSAL);
        unsigned char* ds_head = nullptr;
        int ds_blocks = 0;                                             // of one query head
        if constexpr (DS) {
            ds_blocks = dsl.before((sq + kBwRows - 1) / kBwRows);
            const int64_t first = p.cu_q ? (int64_t)ds_base * p.n_units * G + (int64_t)(hk - p.unit0) * G * ds_blocks
                                         : (int64_t)(b * p.Hkv + hk - p.unit0) * G * ds_blocks;
            ds_head = p.ds + first * kDsBlock;
        }
        // role B: dS of step st (Q tile in ring slot `slot`), dK^T += Q^T dS
        const auto step_b = [&](int st, Pos ps, int slot) {
            const unsigned char* q_lds = lds + slot * kTile;
            const unsigned char* do_lds = lds + (3 + (st & 1)) * kTile;
            const float* delta_lds = delta_lds2 + (st & 1) * kBwRows;
            const unsigned char* in = p_lds + (st & 1) * (kFuPairs * kPSlab);
            u32x4 ds[4];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                // dP - delta comes straight out of the MFMAs: the -delta of the rows (as published) is their C operand
                f32x16 c0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(delta_lds + 32 * t + 8 * j + 4 * kg);
#pragma unroll
                    for (int r = 0; r < 4; ++r) c0[4 * j + r] = d4[r];
                }
                const f32x16 dp_acc = scores(do_lds + t * 32 * kRow, c0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 p4 = *reinterpret_cast<const f32x4*>(in + (4 * t + j) * 1024);
                    float x[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[r] = p4[r] * dp_acc[4 * j + r];                 // dS without the scale factor
                    ds[2 * t + (j >> 1)][2 * (j & 1)] = pack_bf16(x[0], x[1]);
                    ds[2 * t + (j >> 1)][2 * (j & 1) + 1] = pack_bf16(x[2], x[3]);
                }
            }
            if constexpr (DS) {
                // Block: 16 rows at a time (u), in it by key, 32 bytes a key: the 16 bytes of this lane.  (Keys of odd u change places
                // in fours, which takes the reader's two halves of a transposed read to different banks.)
                if (kw0 < sk) {
                    if (!CAUSAL && !k_ok) {                            // a padded key has P != 0 (under the causal mask no row sees it)
#pragma unroll
                        for (int u = 0; u < 4; ++u) ds[u] = u32x4{0u, 0u, 0u, 0u};
                    }
                    unsigned char* block = ds_head + ((int64_t)ps.hq * ds_blocks + dsl.before(ps.r0 >> 6) + (kw0 >> 5)) * kDsBlock;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        __builtin_nontemporal_store(ds[u], reinterpret_cast<u32x4*>(block + (unsigned)(u * 1024 + (n ^ (4 * (u & 1))) * 32 + kg * 16)));
                }
            }
            update(q_lds, ds);
        };

        // iteration i = -1 .. n_steps-1; ring slots: Q(i) in s_b, Q(i+1) in s_a, Q(i+2) lands in s_l;
        // positions: ps0 of step i, ps1 of step i+1, ps2 of step i+2
        Pos ps1 = {(half == 0 ? n_tiles - 1 - share : first_tile) * kBwRows, 0};
        Pos ps0 = ps1, ps2 = advance(ps1);
        if (n_steps > 0) {
            issue_q(ps1, 0);
            publish_lse(0, ps1);
        }
        int s_b = 2, s_a = 0, s_l = 1;
        // what every wavefront does around its role's work in an iteration (the same number of barriers in both loops)
        const auto open_iteration = [&](int i) {
            wait_vmcnt<0>();                                   // this wavefront's share of the tiles issued one iteration ago has landed
            __syncthreads();                                   // ... and everybody's; P(i), lse(i+1), delta(i) are visible; older buffers are free
            if (i + 2 < n_steps) issue_q(ps2, s_l);
            if (i + 1 < n_steps) issue_do(i + 1, ps1);
        };
        const auto close_iteration = [&](int i) {
            if (i + 2 < n_steps) publish_lse(i + 2, ps2);
            if (i + 1 < n_steps) publish_delta(i + 1, ps1);
            const int t3 = s_b;
            s_b = s_a;
            s_a = s_l;
            s_l = t3;
            ps0 = ps1;
            ps1 = ps2;
            ps2 = advance(ps2);
        };
        // One loop per role: in a shared loop the accumulators of the two branches meet again after every
        // iteration, and the compiler then copies all 64 of them, and more, each time round.
        if (!role_b) {
            for (int i = -1; i < n_steps; ++i) {
                open_iteration(i);
                if (i >= 0 && !idle(ps0)) update(lds + (3 + (i & 1)) * kTile, p_cur);      // dV^T += dO(i)^T P(i)
                if (i + 1 < n_steps && !idle(ps1)) make_p(std::integral_constant<bool, CAUSAL || BOOLM>{}, i + 1, ps1, s_a);
                close_iteration(i);
            }
        } else {
            for (int i = -1; i < n_steps; ++i) {
                open_iteration(i);
                if (i >= 0 && !idle(ps0)) step_b(i, ps0, s_b);
                close_iteration(i);
            }
        }

        // store: lane owns key kj, d = 32dt + 8(i/4) + 4kg + i%4
        if (k_ok) {
            const float f = role_b ? p.scale : 1.0f;
            int64_t row = role_b ? dk_base + (int64_t)kj * p.dks[2] : dv_base + (int64_t)kj * p.dvs[2];
            void* grad = role_b ? p.dk : p.dv;
            bool f32 = role_b ? p.dk_f32 : p.dv_f32;
            if (DS && p.shares > 1) {
                const int64_t at = (p.cu_q ? (int64_t)p.cu_k[b] : (int64_t)b * p.Sk) + kj;
                row = ((((role_b ? 0 : p.shares) + share) * p.part_rows + at) * p.Hkv + hk) * D;
                grad = p.part;
                f32 = true;
            }
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    store_grad4(grad, f32, row + 32 * dt + 8 * g + 4 * kg, acc[dt][4 * g + 0] * f, acc[dt][4 * g + 1] * f, acc[dt][4 * g + 2] * f,
                                acc[dt][4 * g + 3] * f);
        }
    }
}

}  // namespace mi355
#include "prefill_bwd_wide.hpp"
namespace mi355 {

// ---------------------------------------------------------------------------------------------
// delta, and for packed sequences the plan of the launches behind it.
//
// delta: D / 8 lanes a row, eight heads of the workgroup's rows; reads dO and O once (HBM-bound).
// Plan (workgroups 0 and 1 of a packed launch): the key tiles and the sets of row tiles of all sequences in falling order of what
// they cost (counting sort), and where each sequence's dS blocks begin.
constexpr int kPlanThreads = 256, kPlanSeqs = 4096, kPlanBins = 2048;

struct PlanParams {
    int32_t* n_jobs;              // [0] key tiles, [1] sets of row tiles
    int32_t* ds_base;
    int2* k_jobs;
    int2* q_jobs;
    int k_room, q_room, ds_room;  // entries and blocks (of one head) there is room for
    int most_q, most_k;           // lengths up to which every sequence has its blocks
    int shift, n_bins;            // costs in steps are binned by cost >> shift
    int k_width, q_width;         // of plan_list
    int total_q;
};

// What the plan holds in LDS.  Every workgroup of the launch has that much, so it is what this batch takes, not what the largest would (41 KB, three workgroups per compute
// unit): 46 sequences of 298 tokens 13.0 -> 12.3 us.
inline size_t plan_lds_bytes(const PlanParams& plan, int B) { return 4 * ((size_t)plan.n_bins + kPlanThreads / 64 + 2 * (size_t)B); }

// One list: entries (b, i), i < n(b), of cost(b, i) < n_bins << shift.  `width` lanes (a power of two up to 64) per sequence, over its entries: as many as the longest
// promised sequence has, so that a batch of short ones is a few rounds of the workgroup (46 sequences of
// 298 tokens, a wavefront each 12.3 us of the launch, like this 8.4).
template <class N, class Cost>
__device__ __forceinline__ int plan_list(int* bins, int* sums, int n_bins, int B, int shift, int width, int2* out, int room, N n_of, Cost cost) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, b0 = tid / width, i0 = tid % width, step = kPlanThreads / width;
    for (int i = tid; i < n_bins; i += kPlanThreads) bins[i] = 0;
    __syncthreads();
    for (int b = b0; b < B; b += step)
        for (int i = i0, n = n_of(b); i < n; i += width) atomicAdd(&bins[min(cost(b, i) >> shift, n_bins - 1)], 1);
    __syncthreads();
    // where a bin's entries begin: the sum of the dearer bins
    int total = 0;
    for (int first = n_bins - kPlanThreads; first > -kPlanThreads; first -= kPlanThreads) {
        const int bin = first + kPlanThreads - 1 - tid, n = bin >= 0 ? bins[bin] : 0;
        const int upto = running_sum(n);
        if (lane == 63) sums[wave] = upto;
        __syncthreads();
        int at = total + upto - n;
        for (int w = 0; w < kPlanThreads / 64; ++w) {
            if (w < wave) at += sums[w];
            total += sums[w];
        }
        if (bin >= 0) bins[bin] = at;
        __syncthreads();
    }
    for (int b = b0; b < B; b += step)
        for (int i = i0, n = n_of(b); i < n; i += width) {
            const int pos = atomicAdd(&bins[min(cost(b, i) >> shift, n_bins - 1)], 1);
            if (pos < room) out[pos] = int2{b, i};
        }
    return min(total, room);
}

template <int D, int MODE>
__global__ __launch_bounds__(kPlanThreads) void bwd_delta_kernel(BwdParams p, PlanParams plan) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL;
    constexpr int kHeads = 8, kLanes = D / 8;
    const int tid = threadIdx.x;
    int bid = blockIdx.x;
    if (p.cu_q) {
        if (bid < 2) {
            extern __shared__ int plan_lds[];     // plan_lds_bytes
            int *bins = plan_lds, *sums = bins + plan.n_bins, *lens_q = sums + kPlanThreads / 64, *lens_k = lens_q + p.B;
            const int G = p.Hq / p.Hkv;
            for (int b = tid; b < p.B; b += kPlanThreads) {
                lens_q[b] = max(p.cu_q[b + 1] - p.cu_q[b], 0);
                lens_k[b] = max(p.cu_k[b + 1] - p.cu_k[b], 0);
            }
            __syncthreads();
            const auto row_tiles = [&](int b) { return (lens_q[b] + kBwRows - 1) / kBwRows; };
            if (bid == 0) {
                const int n = plan_list(bins, sums, plan.n_bins, p.B, plan.shift, plan.k_width, plan.k_jobs, plan.k_room,
                                        [&](int b) { return (lens_k[b] + kFuCols - 1) / kFuCols; },
                                        [&](int b, int i) {
                                            const int skip = CAUSAL ? max(0, i * kFuCols - (lens_k[b] - lens_q[b])) / kBwRows : 0;
                                            return max(0, row_tiles(b) - skip);
                                        });
                if (tid == 0) plan.n_jobs[0] = n;
                return;
            }
            // dS blocks in front of every sequence: first of those of the promised lengths, then, one by one, of longer ones that still fit
            // (the room counts with the longest everywhere).  What does not fit (and, with bounds that do not rise, anything) has none: -1.
            if (tid < 64) {
                int before = 0;
                const auto promised = [&](int b) { return lens_q[b] <= plan.most_q && lens_k[b] <= plan.most_k; };
                for (int b0 = 0; b0 < p.B; b0 += 64) {
                    const int b = b0 + tid;
                    const int n = b < p.B && promised(b) ? DsLayout(lens_q[b], lens_k[b], CAUSAL).before(row_tiles(b)) : 0;
                    const int upto = running_sum(n), first = before + upto - n;
                    if (b < p.B) plan.ds_base[b] = promised(b) && first >= 0 && n <= plan.ds_room - first ? first : -1;
                    before += __shfl(upto, 63, 64);
                }
                if (before < 0) before = plan.ds_room;
                for (int b0 = 0; b0 < p.B; b0 += 64) {
                    uint64_t more = __builtin_amdgcn_ballot_w64(b0 + tid < p.B && !promised(min(b0 + tid, p.B - 1)));
                    for (; more != 0; more &= more - 1) {
                        const int b = b0 + __builtin_ctzll(more);
                        const int64_t n = DsLayoutOf<int64_t>(lens_q[b], lens_k[b], CAUSAL).before((int64_t)row_tiles(b));
                        if (n > plan.ds_room - before) continue;
                        if (tid == 0) plan.ds_base[b] = before;
                        before += (int)n;
                    }
                }
            }
            const int n = plan_list(bins, sums, plan.n_bins, p.B, plan.shift, plan.q_width, plan.q_jobs, plan.q_room,
                                    [&](int b) { return (row_tiles(b) * G + kDqWaves - 1) / kDqWaves; },
                                    [&](int b, int i) {
                                        return DsLayout(lens_q[b], lens_k[b], CAUSAL).count(min(row_tiles(b) * G - 1, kDqWaves * (i + 1) - 1) / G) >> 1;
                                    });
            if (tid == 0) plan.n_jobs[1] = n;
            return;
        }
        bid -= 2;
    }
    const int head_sets = (p.Hq + kHeads - 1) / kHeads;
    const int row = bid / head_sets * (kPlanThreads / kLanes) + tid / kLanes, h0 = bid % head_sets * kHeads, part = tid % kLanes;
    const int n_rows = p.cu_q ? plan.total_q : p.B * p.Sq;
    if (row >= n_rows) return;
    const int b = p.cu_q ? 0 : row / p.Sq, r = p.cu_q ? row : row % p.Sq;
    const __bf16* o = p.out + (p.cu_q ? 0 : (int64_t)b * p.os[0]) + (int64_t)r * p.os[2] + 8 * part;
    const __bf16* g = p.dout + (p.cu_q ? 0 : (int64_t)b * p.dos[0]) + (int64_t)r * p.dos[2] + 8 * part;
    float* out = p.delta + (p.cu_q ? 0 : (int64_t)b * p.ls[0]) + r;
    u32x4 x[kHeads], y[kHeads];
#pragma unroll
    for (int i = 0; i < kHeads; ++i) {
        const int h = min(h0 + i, p.Hq - 1);
        x[i] = *reinterpret_cast<const u32x4*>(o + (int64_t)h * p.os[1]);
        y[i] = *reinterpret_cast<const u32x4*>(g + (int64_t)h * p.dos[1]);
    }
#pragma unroll
    for (int i = 0; i < kHeads; ++i) {
        const bf16x8 o8 = as_bf16x8(x[i]), g8 = as_bf16x8(y[i]);
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += (float)o8[e] * (float)g8[e];
#pragma unroll
        for (int m = kLanes / 2; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
        if (part == 0 && h0 + i < p.Hq) out[(int64_t)(h0 + i) * p.ls[1]] = sum;
    }
}

// ---------------------------------------------------------------------------------------------
// dQ from dS in memory: dQ^T (D x 64 queries) += K^T dS^T, 32 keys at a time.  A wavefront owns one row tile of one query head
// (128 accumulators at head size 128) and streams its dS blocks, which nobody else reads, through LDS of its own; the K rows are shared by the
// four wavefronts, which take neighbours of the kv head's list (row tile, query head).  What bounds it is reading dS, so three
// steps are kept in LDS, two of them in flight: 72 KB, two workgroups per compute unit.  8 x 4096 tokens, 32 / 8 heads: two passes of
// 463 us, 5.3 TB/s (bwd_dq_kernel, three products: 1480); without the MFMAs it takes as long.  dS is written and read once, so both
// sides say so (non-temporal): 528 -> 463 us.  Eight wavefronts, one workgroup: 436, but half as many workgroups where they are few.
template <int D, int MODE>
__global__ __launch_bounds__(kDqWaves * 64, 2) void bwd_dq_ds_kernel(BwdParams p) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL;
    constexpr int kStages = 3;
    using R = TileReads<D>;
    constexpr int NDT = R::NDT, kRow = R::kRow, kKTile = kDsKeys * kRow, kStage = kKTile + kDqWaves * kDsBlock;
    constexpr int kKReq = (kKTile + kDqWaves * 1024 - 1) / (kDqWaves * 1024), kReq = kKReq + kDsBlock / 1024;      // requests of a wavefront a step
    static_assert(kStage % 1024 == 0, "stages begin at whole requests");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kStages * kStage];       // per stage: [K rows][dS of each wavefront]

    const int G = p.Hq / p.Hkv;
    const int id = (int)blockIdx.x / p.n_units, unit = p.unit0 + (int)blockIdx.x % p.n_units;
    int b, set, hk;
    int sq, sk;
    int ds_base = 0;
    int64_t k_base, dq_base, first;
    if (p.cu_q) {
        if (id >= p.n_jobs[1]) return;
        const int2 job = p.q_jobs[id];
        b = job.x;
        set = job.y;
        hk = unit;
        const int q_start = p.cu_q[b], k_start = p.cu_k[b];
        sq = max(p.cu_q[b + 1] - q_start, 0);
        sk = max(p.cu_k[b + 1] - k_start, 0);
        ds_base = p.ds_base[b];
        k_base = (int64_t)k_start * p.ks[2] + (int64_t)hk * p.ks[1];
        dq_base = (int64_t)q_start * p.dqs[2];
    } else {
        b = unit / p.Hkv;
        hk = unit % p.Hkv;
        sq = p.Sq;
        sk = p.Sk;
        set = (((sq + kBwRows - 1) / kBwRows) * G + kDqWaves - 1) / kDqWaves - 1 - id;                  // the dearest first
        k_base = (int64_t)b * p.ks[0] + (int64_t)hk * p.ks[1];
        dq_base = (int64_t)b * p.dqs[0];
    }
    const DsLayout dsl(sq, sk, CAUSAL);
    const int n_rt = (sq + kBwRows - 1) / kBwRows, ds_blocks = dsl.before(n_rt);
    first = p.cu_q ? (int64_t)ds_base * p.n_units * G + (int64_t)(hk - p.unit0) * G * ds_blocks
                   : (int64_t)(b * p.Hkv + hk - p.unit0) * G * ds_blocks;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int last_of_set = min(kDqWaves * set + kDqWaves, n_rt * G) - 1;
    const int mine = min(kDqWaves * set + wave, last_of_set);
    const bool busy = kDqWaves * set + wave <= last_of_set;
    const int rt = mine / G, h = hk * G + mine % G;
    const int n_steps = ds_base < 0 ? 0 : dsl.count(last_of_set / G), my_steps = dsl.count(rt);
    const unsigned char* ds = p.ds + (first + (int64_t)(mine % G) * ds_blocks + dsl.before(rt)) * kDsBlock;

    R rd;
    rd.init(lane);
    // K rows: request j of wavefront w covers 16-byte pieces (kKReq w + j) * 64 .. + 63 of the 32 rows (head size 32 has two wavefronts' worth
    // of them, and the other two bring the same bytes to the same places)
    int k_row[kKReq], k_col[kKReq];
    const int k_first = kKReq * wave * 1024 % kKTile;
#pragma unroll
    for (int j = 0; j < kKReq; ++j) {
        const int idx = k_first / 16 + j * 64 + lane;
        k_row[j] = idx / (D / 8);
        k_col[j] = ((idx % (D / 8)) ^ swz<D>(k_row[j])) * 16;
    }
    // transposed reads of dS: rows 16 (g16 & 1) .. of 32, keys 4 (g16 >> 1) + 8 e ..
    const int g16 = lane >> 4, s16 = lane & 15;
    int ds_off[2][2];                                                  // [keys + 16][e]: even and odd sets of 16 rows sit in the lanes
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int key = 16 * c + 4 * (g16 >> 1) + 8 * e + (s16 >> 2);
            ds_off[c][e] = (g16 & 1) * 1024 + (key ^ (4 * (g16 & 1))) * 32 + (s16 & 3) * 8;
        }
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_address(lds));
    // (every step issues the same requests, so that their number in flight is known: past the end they re-read the last block and row)
    const auto issue = [&](int step, int stage) {
        const uint32_t at = base + stage * kStage;
        const int r0 = min(step, n_steps - 1) * kDsKeys;
        const __bf16* rows = p.k + k_base + (int64_t)r0 * p.ks[2];
#pragma unroll
        for (int j = 0; j < kKReq; ++j)
            dma_to_lds_16(rows, (uint32_t)(min(k_row[j], sk - 1 - r0) * (int)p.ks[2] * 2 + k_col[j]), at + k_first + j * 1024);
        const unsigned char* block = ds + (int64_t)max(0, min(step, my_steps - 1)) * kDsBlock;
#pragma unroll
        for (int j = 0; j < 4; ++j) dma_to_lds_16_once(block, (uint32_t)(j * 1024 + lane * 16), at + kKTile + wave * kDsBlock + j * 1024);
    };

    f32x16 dq[2][NDT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < NDT; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) dq[t][i][j] = 0.f;
    // Column n of half t is row 32 t + my_row of the sequence.  From step `diagonal` on some row does not see all keys of the step: dS is zero there
    // unless its dP overflowed (0 * inf), so it is set to zero here, where there is time (the dK/dV kernel takes 5 % longer with it).  It may also never have been
    // written: bwd_dkv_wide_kernel stores nothing of a half of a row tile of which no row sees any of a wavefront's 64 keys.
    const int my_row = kBwRows * rt + 16 * (n >> 4) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + (n & 3);
    const int diagonal = (kBwRows * rt + sk - sq + 1) >> 5;
    if (n_steps > 0) {
        issue(0, 0);
        issue(1, 1);
        int stage = 0;
        for (int step = 0; step < n_steps; ++step) {
            wait_vmcnt<kReq>();                                           // this wavefront's share of the step has landed
            __syncthreads();                                           // ... and everybody's K rows; all are done with the step before
            issue(step + 2, stage >= 1 ? stage - 1 : 2);
            if (busy && step < my_steps) {
                const unsigned char* k_lds = lds + stage * kStage;
                const unsigned char* d_lds = k_lds + kKTile + wave * kDsBlock;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    bf16x8 w[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        w[t] = join_bf16x8(lds_read_tr16(d_lds + 2048 * t + ds_off[c][0]), lds_read_tr16(d_lds + 2048 * t + ds_off[c][1]));
                    if (CAUSAL && step >= diagonal) {
                        const int lim = my_row + sk - sq - 32 * step - 16 * c - 4 * kg;         // the last of these 16 keys (less 4 kg) that this lane's row of half 0 sees
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            u32x4 x = __builtin_bit_cast(u32x4, w[t]);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {                // elements 2 i and 2 i + 1: keys 8 (i / 2) + 2 (i % 2) and the next one
                                const int key = 8 * (i >> 1) + 2 * (i & 1) - 32 * t;
                                x[i] &= (key <= lim ? 0xffffu : 0u) | (key + 1 <= lim ? 0xffff0000u : 0u);
                            }
                            w[t] = as_bf16x8(x);
                        }
                    }
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) {
                        const bf16x8 a = join_bf16x8(lds_read_tr16(k_lds + 16 * c * kRow + rd.tr_off[0][dt]), lds_read_tr16(k_lds + 16 * c * kRow + rd.tr_off[1][dt]));
#pragma unroll
                        for (int t = 0; t < 2; ++t) dq[t][dt] = mfma32(a, w[t], dq[t][dt]);
                    }
                }
            }
            stage = stage == 2 ? 0 : stage + 1;
        }
        wait_vmcnt<0>();
    }
    if (!busy) return;
    // store: d = 32 dt + 8 (i / 4) + 4 kg + i % 4
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int qi = my_row + 32 * t;
        if (qi >= sq) continue;
        const int64_t row = dq_base + (int64_t)qi * p.dqs[2] + (int64_t)h * p.dqs[1];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                store_grad4(p.dq, p.dq_f32, row + 32 * dt + 8 * g + 4 * kg, dq[t][dt][4 * g + 0] * p.scale, dq[t][dt][4 * g + 1] * p.scale,
                            dq[t][dt][4 * g + 2] * p.scale, dq[t][dt][4 * g + 3] * p.scale);
    }
}

// dK and dV of key tiles whose row tiles were dealt out: the sum of the shares (in their order), 4 elements a thread.
template <int D>
__global__ __launch_bounds__(256) void bwd_sum_shares_kernel(BwdParams p) {
    const bool is_dv = blockIdx.y == 1;
    const int64_t quad = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = quad / (D / 4) / p.Hkv;
    const int hk = (int)(quad / (D / 4) % p.Hkv), d = (int)(quad % (D / 4)) * 4;
    if (row >= p.part_rows) return;
    const float* src = p.part + (((is_dv ? p.shares : 0) * p.part_rows + row) * p.Hkv + hk) * D + d;
    const int64_t step = p.part_rows * p.Hkv * D;
    f32x4 sum = *reinterpret_cast<const f32x4*>(src);
    for (int i = 1; i < p.shares; ++i) sum += *reinterpret_cast<const f32x4*>(src + i * step);
    const int64_t* st = is_dv ? p.dvs : p.dks;
    const int64_t at = (p.cu_q ? row * st[2] : row / p.Sk * st[0] + row % p.Sk * st[2]) + hk * st[1] + d;
    store_grad4(is_dv ? p.dv : p.dk, is_dv ? p.dv_f32 : p.dk_f32, at, sum[0], sum[1], sum[2], sum[3]);
}

// ---------------------------------------------------------------------------------------------
// dK and dV at head sizes 32 and 64, where one wavefront has the registers for both: it holds the K and V fragments of 32
// keys and both accumulators, so that P need not travel.  Workgroups of four wavefronts (128 keys) with 16 or 32 KB of LDS:
// two to four of them on a compute unit fill each other's barriers and load latencies, which is what the kernel with two
// roles (87 / 107 KB: one workgroup) spends most of its time in at these sizes.
template <int D, int MODE>
__global__ __launch_bounds__(256, D == 32 ? 4 : 2) void bwd_dkv_one_kernel(BwdParams p) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL, BOOLM = MODE == MI355_MASK_BOOL;
    constexpr int NWV = kFuPairs;
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, kTile = kBwRows * kRow;
    // [Q buffer 0][Q buffer 1][dO buffer 0][dO buffer 1]
    __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kTile];
    __shared__ __attribute__((aligned(16))) float lse_lds2[2 * kBwRows];
    __shared__ __attribute__((aligned(16))) float delta_lds2[2 * kBwRows];       // -delta

    // (key-tile pairs as in the kernel with two roles: equal work, and one (batch, kv head) on one XCD; or single tiles, the first and
    // dearest ones first, all walking their rows downwards)
    const bool singles = p.deal.singles;
    int pair, head;
    if (singles) {
        const HeadUnit at = xcd_unit(blockIdx.x, p.deal.units, 1, p.Hkv * p.B, p.deal.chunk_heads, p.deal.round);
        if (at.unit < 0) return;
        pair = at.unit;
        head = at.head;
    } else {
        const int lid = xcd_chunked_id(blockIdx.x, gridDim.x, p.deal.units);
        pair = lid % p.deal.units;
        head = lid / p.deal.units;
    }
    pair = __builtin_amdgcn_readfirstlane(pair);
    const int b = __builtin_amdgcn_readfirstlane(head / p.Hkv), hk = __builtin_amdgcn_readfirstlane(head - b * p.Hkv);
    const int G = p.Hq / p.Hkv;
    int sq, sk;
    int64_t q_base, do_base, l_base, k_base, v_base, dk_base, dv_base;           // (q, dO, lse, delta: of the batch; heads are added)
    if (p.cu_q) {
        const int q_start = p.cu_q[b], k_start = p.cu_k[b];
        sq = p.cu_q[b + 1] - q_start;
        sk = p.cu_k[b + 1] - k_start;
        q_base = (int64_t)q_start * p.qs[2];
        do_base = (int64_t)q_start * p.dos[2];
        l_base = q_start;
        k_base = (int64_t)k_start * p.ks[2] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)k_start * p.vs[2] + (int64_t)hk * p.vs[1];
        dk_base = (int64_t)k_start * p.dks[2] + (int64_t)hk * p.dks[1];
        dv_base = (int64_t)k_start * p.dvs[2] + (int64_t)hk * p.dvs[1];
    } else {
        sq = p.Sq;
        sk = p.Sk;
        q_base = (int64_t)b * p.qs[0];
        do_base = (int64_t)b * p.dos[0];
        l_base = (int64_t)b * p.ls[0];
        k_base = (int64_t)b * p.ks[0] + (int64_t)hk * p.ks[1];
        v_base = (int64_t)b * p.vs[0] + (int64_t)hk * p.vs[1];
        dk_base = (int64_t)b * p.dks[0] + (int64_t)hk * p.dks[1];
        dv_base = (int64_t)b * p.dvs[0] + (int64_t)hk * p.dvs[1];
    }
    const int nk = (sk + kFuCols - 1) / kFuCols;
    if ((singles ? pair : 2 * pair) >= nk) return;                                         // (a sequence without queries still gets dk = dv = 0 written)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int coff = sk - sq;

    TileLoader<D, NWV> ld;
    ld.init(wave, lane);
    R rd;
    rd.init(lane);
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_address(lds) + wave * TileLoader<D, NWV>::NI * 1024);
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // single tiles: one, unless a packed sequence is longer than the caller said
    for (int half = 0, ktile = pair; singles ? ktile < nk : half < 2; ++half, ktile = singles ? ktile + p.deal.units : nk - 1 - pair) {
        if (!singles && half == 1 && ktile == pair) break;              // odd tile count: the middle tile has no partner
        const int k0 = ktile * kFuCols;
        const int kw0 = k0 + 32 * wave;
        const int kj = kw0 + n;
        const bool k_ok = kj < sk;
        __syncthreads();                                                // the previous half's readers are done with the LDS buffers

        // fragments of this lane's key column: step s covers d = 16s + 8kg + j
        bf16x8 kf[NS], vf[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            u32x4 a = {0u, 0u, 0u, 0u}, c = {0u, 0u, 0u, 0u};
            if (k_ok) {
                a = *reinterpret_cast<const u32x4*>(p.k + k_base + (int64_t)kj * p.ks[2] + 16 * s + 8 * kg);
                c = *reinterpret_cast<const u32x4*>(p.v + v_base + (int64_t)kj * p.vs[2] + 16 * s + 8 * kg);
            }
            kf[s] = as_bf16x8(a);
            vf[s] = as_bf16x8(c);
        }
        f32x16 dk[NDT], dv[NDT];
#pragma unroll
        for (int i = 0; i < NDT; ++i) dk[i] = dv[i] = zero16;

        int first_tile = 0;
        if (CAUSAL) first_tile = max(0, k0 - coff) / kBwRows;
        const int n_tiles = (sq + kBwRows - 1) / kBwRows;
        const int n_steps = G * max(0, n_tiles - first_tile);           // (row tile, query head of the group), heads innermost
        struct Pos {
            int r0, hq;
        };
        const int r_step = singles || half == 0 ? -kBwRows : kBwRows;
        const auto advance = [&](Pos ps) {
            ++ps.hq;
            if (ps.hq == G) {
                ps.hq = 0;
                ps.r0 += r_step;
            }
            return ps;
        };
        float pend_lse = 0.f, pend_delta = 0.f;
        const auto issue = [&](int st, Pos ps) {
            const int h = hk * G + ps.hq, r0 = ps.r0, buf = (st & 1) * kTile;
            ld.issue(p.q + q_base + (int64_t)h * p.qs[1] + (int64_t)r0 * p.qs[2], (int)p.qs[2], sq - 1 - r0, dst + buf);
            ld.issue(p.dout + do_base + (int64_t)h * p.dos[1] + (int64_t)r0 * p.dos[2], (int)p.dos[2], sq - 1 - r0, dst + 2 * kTile + buf);
            if (tid < kBwRows) {
                const int64_t at = l_base + (int64_t)h * p.ls[1] + r0 + min(tid, sq - 1 - r0);
                pend_lse = p.lse[at];
                pend_delta = p.delta[at];
            }
        };
        // (a causal row that sees no key has out = NaN, hence delta = NaN, and P = 0 everywhere: any finite delta gives the
        // dS = 0 it must have)
        const auto publish = [&](int st, Pos ps) {
            if (tid < kBwRows) {
                const bool in = ps.r0 + tid < sq;
                lse_lds2[(st & 1) * kBwRows + tid] = in ? pend_lse * kLog2e : INFINITY;
                delta_lds2[(st & 1) * kBwRows + tid] = in && pend_delta == pend_delta ? -pend_delta : 0.f;
            }
        };
        // fragments read kDepth MFMAs ahead, in order, as in the other kernels
        constexpr int kDepth = 2;
        const auto scores = [&](const unsigned char* a_lds, const bf16x8 (&bfr)[NS], const f32x16& c0) {
            u32x4 a[NS];
#pragma unroll
            for (int s = 0; s < kDepth && s < NS; ++s) a[s] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s]);
            f32x16 r = c0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + kDepth < NS) a[s + kDepth] = *reinterpret_cast<const u32x4*>(a_lds + rd.row_off[s + kDepth]);
                r = mfma32(as_bf16x8(a[s]), bfr[s], r);
                __builtin_amdgcn_sched_barrier(0);
            }
            return r;
        };
        // acc^T (D x 32 keys) += tile^T . w over 32 rows of the tile
        const auto update = [&](f32x16 (&acc)[NDT], const unsigned char* a_lds, const u32x4 (&w)[2]) {
            constexpr int NC = 2 * NDT;
            i16x4 lo[NC], hi[NC];
            const auto read = [&](int c) {
                const int u = c / NDT, dt = c % NDT;
                lo[c] = lds_read_tr16(a_lds + 16 * u * kRow + rd.tr_off[0][dt]);
                hi[c] = lds_read_tr16(a_lds + 16 * u * kRow + rd.tr_off[1][dt]);
            };
#pragma unroll
            for (int c = 0; c < kDepth && c < NC; ++c) read(c);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (c + kDepth < NC) read(c + kDepth);
                acc[c % NDT] = mfma32(join_bf16x8(lo[c], hi[c]), as_bf16x8(w[c / NDT]), acc[c % NDT]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        const auto step = [&](int st, Pos ps) {
            const unsigned char* q_lds = lds + (st & 1) * kTile;
            const unsigned char* do_lds = q_lds + 2 * kTile;
            const float* lse_lds = lse_lds2 + (st & 1) * kBwRows;
            const float* delta_lds = delta_lds2 + (st & 1) * kBwRows;
            const int row_lim = CAUSAL ? kj - coff - ps.r0 - 4 * kg : -1;
            // one 32-row half at a time: element i of this lane is query row r0 + 32t + 8(i/4) + 4kg + i%4, key kj
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                uint8_t mb[16] = {};
                if constexpr (BOOLM) {           // (a row or key past the end re-reads the last one, see bwd_dkv_kernel)
                    const uint8_t* mcol = p.mask + (int64_t)b * p.ms[0] + (int64_t)(hk * G + ps.hq) * p.ms[1] + min(kj, sk - 1);
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        mb[e] = mcol[(int64_t)min(ps.r0 + 32 * t + 8 * (e >> 2) + 4 * kg + (e & 3), sq - 1) * p.ms[2]];
                }
                f32x16 c0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(delta_lds + 32 * t + 8 * j + 4 * kg);
#pragma unroll
                    for (int r = 0; r < 4; ++r) c0[4 * j + r] = d4[r];
                }
                const f32x16 s_acc = scores(q_lds + t * 32 * kRow, kf, zero16);
                const f32x16 dp_acc = scores(do_lds + t * 32 * kRow, vf, c0);              // dP - delta
                u32x4 pw[2], dsw[2];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 l4 = *reinterpret_cast<const f32x4*>(lse_lds + 32 * t + 8 * j + 4 * kg);
                    float x[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        x[r] = fast_exp2(fmaf(s_acc[4 * j + r], p.scale_log2, -l4[r]));
                        // kept iff kj <= row + coff, i.e. the tile-relative row (compile-time part) >= row_lim
                        if constexpr (CAUSAL || BOOLM) {
                            bool keep = 32 * t + 8 * j + r >= row_lim;
                            if constexpr (BOOLM) keep = keep & (mb[4 * j + r] != 0);
                            x[r] = keep ? x[r] : 0.f;
                        }
                    }
                    pw[j >> 1][2 * (j & 1)] = pack_bf16(x[0], x[1]);
                    pw[j >> 1][2 * (j & 1) + 1] = pack_bf16(x[2], x[3]);
                    dsw[j >> 1][2 * (j & 1)] = pack_bf16(x[0] * dp_acc[4 * j], x[1] * dp_acc[4 * j + 1]);          // dS without the scale factor
                    dsw[j >> 1][2 * (j & 1) + 1] = pack_bf16(x[2] * dp_acc[4 * j + 2], x[3] * dp_acc[4 * j + 3]);
                }
                update(dv, do_lds + 32 * t * kRow, pw);
                update(dk, q_lds + 32 * t * kRow, dsw);
            }
        };

        Pos ps = {(singles || half == 0 ? n_tiles - 1 : first_tile) * kBwRows, 0};
        if (n_steps > 0) {
            issue(0, ps);
            publish(0, ps);
        }
        for (int i = 0; i < n_steps; ++i) {
            const Pos next = advance(ps);
            wait_vmcnt<0>();                                   // this wavefront's share of the step's tiles has landed
            __syncthreads();                                   // ... and everybody's; lse and delta are visible; the other buffers are free
            if (i + 1 < n_steps) issue(i + 1, next);
            // (a step whose rows all lie above this wavefront's first key column has nothing for it)
            if (!CAUSAL || kw0 <= ps.r0 + kBwRows - 1 + coff) step(i, ps);
            if (i + 1 < n_steps) publish(i + 1, next);
            ps = next;
        }

        // store: lane owns key kj, d = 32dt + 8(i/4) + 4kg + i%4
        if (k_ok) {
            const int64_t k_row = dk_base + (int64_t)kj * p.dks[2], v_row = dv_base + (int64_t)kj * p.dvs[2];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int d = 32 * dt + 8 * g + 4 * kg;
                    store_grad4(p.dk, p.dk_f32, k_row + d, dk[dt][4 * g] * p.scale, dk[dt][4 * g + 1] * p.scale, dk[dt][4 * g + 2] * p.scale,
                                dk[dt][4 * g + 3] * p.scale);
                    store_grad4(p.dv, p.dv_f32, v_row + d, dv[dt][4 * g], dv[dt][4 * g + 1], dv[dt][4 * g + 2], dv[dt][4 * g + 3]);
                }
        }
    }
}

// How the units of a launch are dealt (see xcd_unit): tiles of equal and of falling cost in pairs or one by one.  An XCD takes as many heads at a time as
// have 8 MB of streamed rows.  (With 4 MB and less launches of one and two rounds lose up to a quarter: 136 heads of 32, 2048 tokens, dK and dV
// 106 us with 8, 135 with 4.)
constexpr int64_t kCus = 256;
static void deal_units(BwdDeal& d, bool pairs, int64_t n_tiles, int64_t n_heads, int64_t resident, int64_t head_bytes, int64_t kv_heads) {
    // (an even number of tiles: lengths beyond the promised one are covered as far as pairs cover them)
    const int64_t n_pairs = (n_tiles + 1) / 2;
    d.singles = !pairs && xcd_units_fit(2 * n_pairs, n_heads / kv_heads, kv_heads, 256);
    d.units = (int)(n_pairs * (d.singles ? 2 : 1));
    d.chunk_heads = (int)(n_heads / kv_heads * std::max<int64_t>(1, std::min<int64_t>(kv_heads / 8, (8 << 20) / head_bytes)));
    d.round = n_tiles * n_heads <= resident ? (int)(kCus / 8) : 0;
}
static unsigned deal_grid(const BwdDeal& d, int64_t n_heads, int64_t kv_heads) {
    return d.singles ? (unsigned)xcd_units_grid(d.units, (int)(n_heads / kv_heads), (int)kv_heads) : (unsigned)(d.units * n_heads);
}

template <int D, int MODE>
static void launch_dq(BwdParams p, hipStream_t stream) {
    constexpr bool kSmall = D <= 64 && MODE != MI355_MASK_BOOL;             // (explicit masks: their words and bounds leave no registers for more)
    constexpr int NW = kSmall ? 4 : kBwWaves;
    const int64_t heads = (int64_t)p.Hq * p.B, kv_heads = (int64_t)p.Hkv * p.B, tiles = p.n_qtiles * (kBwWaves / NW), resident = kCus * dq_resident(D);
    // one length and the causal triangle: pairs where the launch goes over the chip more than four times (256 heads of 64, 2048 tokens: 231 us either way)
    const bool equal = MODE == MI355_MASK_CAUSAL && (!p.cu_q || p.B == 1);
    deal_units(p.deal, !kSmall || (equal && tiles * heads > 4 * resident), tiles, heads, resident, (int64_t)p.Sk * D * 4, kv_heads);
    hipLaunchKernelGGL((bwd_dq_kernel<D, MODE, NW>), dim3(deal_grid(p.deal, heads, kv_heads)), dim3(NW * 64), 0, stream, p);
}
template <int D, int MODE>
static void launch_dkv_one(BwdParams p, hipStream_t stream) {
    const int64_t heads = (int64_t)p.Hkv * p.B, tiles = p.n_ktiles, resident = kCus * (D == 32 ? 4 : 2), pairs = (tiles + 1) / 2 * heads;
    // One length and the causal triangle: pairs at head size 32 beyond four rounds of the chip; at 64, where two workgroups per compute unit wait longer
    // for rows that another head has pushed out of the L2, wherever pairs fill their rounds.  us, pairs / singles, heads of 64: 256 of 512 tokens
    // (512 pairs, 1.0 rounds) 35 / 38, of 1024 (2.0) 102 / 107, 136 of 1456 (1.6) 124 / 104, 136 of 1024 (1.1) 81 / 58; of 32: 256 of 1024 59 / 56,
    // 136 of 2048 131 / 106, 64 of 8192 (4 rounds) 791 / 740; 14 packed of 111 to 1172, 32 / 16 heads, 85 / 72.
    const bool equal = MODE == MI355_MASK_CAUSAL && (!p.cu_q || p.B == 1);
    const bool filled = D == 32 ? tiles * heads > 4 * resident : (pairs + resident - 1) / resident * resident * 10 <= 11 * pairs;
    deal_units(p.deal, equal && filled, tiles, heads, resident, (int64_t)p.Sq * (p.Hq / p.Hkv) * D * 4, heads);
    hipLaunchKernelGGL((bwd_dkv_one_kernel<D, MODE>), dim3(deal_grid(p.deal, heads, heads)), dim3(kFuPairs * 64), 0, stream, p);
}

template <int D, int MODE>
static void launch_bwd_mode(const BwdParams& p, hipStream_t stream) {
    launch_dq<D, MODE>(p, stream);                                           // dQ, writes delta
    // dK and dV, reads delta.  Head sizes 32 and 64: both roles in each wavefront, but for few pairs of key tiles with many steps, where a workgroup's own
    // chain is what counts.  us with dQ, roles apart / together: one of 8160 tokens, 64 / 8 heads of 32 2067 / 2100 (with the forward); 16 heads of 32,
    // 3000 tokens 105 / 103; 64 of 32, 300 tokens 20 / 19, 64 of 64, 2048 tokens 192 / 157.
    const dim3 grid((unsigned)((p.n_ktiles + 1) / 2 * p.Hkv * p.B));
    if constexpr (D <= 64) {
        if (grid.x > kCus || (int64_t)(p.Sq + kBwRows - 1) / kBwRows * (p.Hq / p.Hkv) < 64) {
            launch_dkv_one<D, MODE>(p, stream);
            return;
        }
    }
    hipLaunchKernelGGL((bwd_dkv_kernel<D, MODE, false>), grid, dim3(2 * kFuPairs * 64), 0, stream, p);
}

// ---- with dS in memory ----
// The passes of a call over dS of at most kDsMost bytes: unit ranges of one size (give or take one), a unit being a kv head of all
// packed sequences or of one sequence of a dense batch.
constexpr int64_t kDsMost = (int64_t)4 << 30;

struct DsPasses {
    int64_t unit_bytes = 0;       // dS of a unit (packed: a bound)
    int64_t plan_bytes = 0;       // lists, in front of dS
    int n_units = 0, units_per_pass = 0;
    int shares = 1;
    bool wide = false;            // dK, dV and dS by bwd_dkv_wide_kernel
    int64_t part_rows = 0, part_bytes = 0;       // fp32 shares of dk and dv, behind the lists
    int64_t ds_room = 0, k_room = 0, q_room = 0, most_q = 0, most_k = 0;
    int64_t bytes() const { return plan_bytes + part_bytes + unit_bytes * units_per_pass; }
};

static int64_t round_up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

static bool ds_passes(int B, int Hq, int Hkv, int Sq, int Sk, int D, int mask_mode, bool packed, bool same_bounds, int64_t total_q, int64_t total_k,
                      DsPasses& out) {
    if (mask_mode != MI355_MASK_NONE && mask_mode != MI355_MASK_CAUSAL) return false;
    // Heads that the short kernel takes are one launch there, whatever their number.  256 tokens, head size 32, 8 / 64 / 128 heads: 9, 9, 10 us, here
    // 20, 21, 22; head size 64, 8 / 64 / 192 heads: 13, 14, 19 / 24, 25, 37 (the form without a workspace, before: 28, 29, 33).
    if (!packed && prefill_bwd_short_takes(Hq, Hkv, Sq, Sk, D, mask_mode)) return false;
    const bool causal = mask_mode == MI355_MASK_CAUSAL;
    const int64_t G = Hq / Hkv, n_rt = (Sq + kBwRows - 1) / kBwRows;
    if (packed) {
        if (B > kPlanSeqs || total_q <= 0 || total_k <= 0 || total_q > 0x7fffffffLL || total_k > 0x7fffffffLL) return false;
        // row tiles of all sequences, times the most blocks a row tile can have; causal over the same bounds, row tile r has 2 r + 2.
        // (Lengths up to the next multiple of 256: as far as the form without a workspace reaches behind a promise that is too small.)
        out.most_q = round_up(Sq, kBwCols);
        out.most_k = round_up(Sk, kBwCols);
        const int64_t tiles = std::max(total_q, out.most_q) / kBwRows + B;
        out.ds_room = tiles * (causal && same_bounds ? out.most_q / kBwRows + 1 : out.most_k / kDsKeys);
        out.k_room = std::max<int64_t>(total_k, Sk) / kFuCols + B;
        out.q_room = (tiles * G + kDqWaves - 1) / kDqWaves + B;
        out.plan_bytes = round_up(16 + 4 * (int64_t)B, 16) + 8 * (out.k_room + out.q_room);
        out.n_units = Hkv;
    } else {
        out.ds_room = DsLayoutOf<int64_t>(Sq, Sk, causal).before(n_rt);
        out.n_units = B * Hkv;
    }
    if (out.ds_room * G > 0x7fffffffLL || out.k_room > 0x7fffffffLL || out.q_room > 0x7fffffffLL) return false;
    out.plan_bytes = round_up(out.plan_bytes, kDsBlock);
    // Key tiles are what fills the chip in the dK/dV kernel, and the first one of a sequence walks through all its row tiles.  With fewer
    // than one per compute unit, or two where the walk is long, their row tiles are dealt out, down to about eight steps each: one
    // sequence of 8192 tokens, 8 / 1 heads, dK/dV 1743 -> 361 us (and 12 for the sums); 4 x 1024, 32 / 8 heads 134 -> 101 (15); 16 x 512,
    // 16 / 4 heads, 32 steps, would be 73 -> 68 (15).
    const int64_t rows_k = packed ? total_k : (int64_t)B * Sk, tiles_k = (rows_k + kFuCols - 1) / kFuCols * Hkv;
    while (tiles_k * out.shares < (n_rt * G >= 48 * out.shares ? 512 : 256) && out.shares < 16 && n_rt * G >= 16 * out.shares &&
           n_rt >= 2 * out.shares)
        out.shares *= 2;
    // Up to 128 tokens that do not fill the chip either way: one launch more costs what dS saves (4 x 128, 8 / 2 heads 33 us against
    // 37; 64 x 128, 16 / 4 heads 83 against 73), and up to 64 it is most of what runs (16 x 64, 8 heads 17 against 20).
    if (std::max(Sq, Sk) <= (tiles_k < 256 ? 128 : 64)) return false;
    // At head sizes 64 and 32 the products that dS saves are worth less than its bytes.  What this form has over the other is that the row tiles of a key tile can be dealt
    // out (shares) and that workgroups come in order of cost.  So it is for launches whose longest chain -- the steps of the first key tile of the longest
    // sequence -- is many steps and many times what a workgroup's place on the chip has to do on average (`over`, for the causal triangle; longest: of the
    // lengths, over their mean).  us with dS / without (steps, over):
    //   heads of 32, causal: 16 of 2048 tokens (32, 8) 80 / 68, 8 of 4096 (64, 8) 122 / 128, 4 x 1024, 32 / 8 heads, (64, 8) 96 / 113, 2 x 3494, 32 / 4, (440, 9.3) 435 / 623,
    //     16 / 4 heads, 512 (32, 128) 34 / 51, 6 x 326, 32 / 8, (24, 16) 42 / 45, 4 x 3900, 16 / 4, (244, 4.2) 562 / 450; not dealt out: 24 of 1456 (23, 7.1) 61 / 53;
    //     packed, 32 of up to 339 tokens, 64 / 8, (48, 14, longest 2.2) 127 / 107, 12 of 490 to 5500, 8 / 1, (688, 13, 2) 630 / 1041
    //   heads of 64, causal: 8 of 1456 (23, 11) 59 / 63, 16 of 1456 (23, 5.3) 64 / 64, 24 of 1024 (16, 5.3) 58 / 50, 32 / 16, 3 x 738 (24, 3.6) 70 / 64, 8 x 1589,
    //     16 / 4, (100, 2.56) 268 / 260, 6315, 32 / 8, (396, 2.56) 933 / 840, 6 x 6166, 8 / 2, packed, (388, 2.9) 814 / 933, 8 of up to 764, 16 / 8, (24, 7.4, longest 1.7) 72 / 64; not dealt out: 16 of 3000 (47, 2.7) 126 / 133, 24 of 2048 (32, 2.7) 95 / 96
    //   without a mask, of 32: 4223, 16 / 4, (264, 16) 349 / 622, 24 x 1234, 4 / 1, (80, 8.8) 160 / 209; of 64: 3796, 64 / 16, (240, 2.1) 1231 / 995; not dealt out: packed,
    //     12 of up to 2001, 4 heads, (32, 8.4) 95 / 116
    // Of 2619 drawn calls of 130 to 7000 tokens none is more than 8 % slower than by the number of key tiles alone, and 6 by more than 3 %.  (Short sequences with few key
    // tiles, and at 64 lengths far apart, keep dS: up to 10 us of the GPU more, in calls that the host's side of a gradient, some 70 us, outlasts either way.)
    if (D < 128) {
        const int64_t steps = n_rt * G, places = kCus * (D == 32 ? 4 : 2);
        const double longest = packed ? (double)B * Sk / total_k : 1.0, over = 2.0 * places / tiles_k * longest;
        const bool short_ones = std::max(Sq, Sk) <= 160, few = !short_ones && tiles_k <= (D == 64 ? 384 : 256) && steps < 24;
        const double line = D == 32 ? (causal ? 490.0 : 600.0) : causal ? 164.0 : 270.0;
        const bool dealt = out.shares > 1 && (D == 64 || !short_ones) && over >= (D == 32 ? 8.0 : causal ? 2.69 : 3.5) && steps >= 24 &&
                           steps * over >= line * std::sqrt(longest);
        const bool ordered = D == 64 && ((packed && 2 * total_k < (int64_t)B * Sk) ||
                                         (out.shares == 1 && !short_ones && (causal ? steps >= 36 && over >= 2.69 : steps >= 20 && over >= 5.0)));
        if (!dealt && !ordered && !few) return false;
    }
    if (out.shares > 1) {
        out.part_rows = rows_k;
        out.part_bytes = round_up(2 * out.shares * rows_k * Hkv * D * 4, kDsBlock);
    }
    // Wavefronts of 64 keys: key tiles with many steps on average (packed: of the mean length).  us of dK/dV, roles apart / wide (steps): 40 packed of 50 to 800 tokens, 8 heads, (2)
    // 56 / 70; 4 x 602, 16 heads (5) 32 / 37; 16 x 920 (7) 231 / 243; 4 packed of 324 to 5199, 4 / 2 heads, 4 shares (11) 116 / 120; 51 packed of 1701, one head (13) all kernels
    // 258 / 262; 21 packed of 995, 16 / 8 (15.5) all kernels 548 / 554; 2 x 2048, 32 heads (16) 186 / 175; 3000
    // tokens, 16 heads (23) 103 / 93; 6 packed of 100 to 1500, 64 / 8 (50) 235 / 232; 8192, 8 / 1 (64) 307 / 278; 16 of 256 to 4096, 32 / 8 (43) 905 / 832; 8 x 4096 (128) 2553 / 2250
    // From sixteen on where no rows are dealt out, and not few of them under the diagonal, else from 24 on.  us of the whole backward, packed sequences of one length, roles apart / wide
    // (steps): one share, 5 x 2113, 12 heads (16.5) 305 / 298, 4 x 2200, 4 heads (17) 126 / 122, 2 x 1250 without a mask, 16 heads (19.5) 134 / 131, but 100 x 257, 16 / 2 (16) 277 / 298, 32 x 600,
    // 32 / 8 (18.8) 563 / 572, 16 x 700, 32 / 8 (22) 329 / 333; two shares, 90 x 556, 8 / 1 (17.4) 387 / 408, 4500, 8 heads (17.6) 218 / 223, 16 x 1280, 8 / 2 (20) 259 / 262, 16 x 1536, 8 / 2
    // (24) 346 / 331; four, 4 x 1100, 32 / 4 (17) 224 / 231; eight, 3000, 16 / 2 (23) 178 / 186, 4500, 16 / 2 (35) 359 / 355; sixteen, 4096, 8 / 1 (16) 185 / 190, without a mask (32) 256 / 250
    const double row_tiles = (double)(packed ? total_q : (int64_t)B * Sq) / kBwRows / B;
    out.wide = D == 128 && row_tiles * G * (causal ? 0.5 : 1.0) >= (out.shares == 1 && (!causal || row_tiles >= 24.0) ? 16.0 : 24.0) * out.shares;
    out.unit_bytes = out.ds_room * G * kDsBlock;
    const int64_t fit = out.unit_bytes > 0 ? kDsMost / out.unit_bytes : out.n_units;
    if (fit < 1) return false;
    const int64_t passes = (out.n_units + fit - 1) / fit;
    out.units_per_pass = (int)((out.n_units + passes - 1) / passes);
    return true;
}

template <int D, int MODE>
static int launch_bwd_ds(BwdParams p, const DsPasses& d, int64_t total_q, unsigned char* ws, hipStream_t stream) {
    constexpr int kRowsPerWg = kPlanThreads / (D / 8), kHeadsPerWg = 8;
    PlanParams plan = {};
    if (p.cu_q) {
        plan.n_jobs = (int32_t*)ws;
        plan.ds_base = plan.n_jobs + 4;
        plan.k_jobs = (int2*)(ws + round_up(16 + 4 * (int64_t)p.B, 16));
        plan.q_jobs = plan.k_jobs + d.k_room;
        plan.k_room = (int)d.k_room;
        plan.q_room = (int)d.q_room;
        plan.ds_room = (int)d.ds_room;
        plan.most_q = (int)std::min<int64_t>(d.most_q, 0x7fffffff);
        plan.most_k = (int)std::min<int64_t>(d.most_k, 0x7fffffff);
        const int most = std::max(p.Sq, p.Sk) / kBwRows + 1;                      // (costs count row tiles, or pairs of dS blocks)
        while (most >> plan.shift >= kPlanBins) ++plan.shift;
        plan.n_bins = (most >> plan.shift) + 1;
        const auto width = [](int64_t entries) {
            int w = 1;
            while (w < 64 && w < entries) w *= 2;
            return w;
        };
        plan.k_width = width((p.Sk + kFuCols - 1) / kFuCols);
        plan.q_width = width(((p.Sq + kBwRows - 1) / kBwRows * (int64_t)(p.Hq / p.Hkv) + kDqWaves - 1) / kDqWaves);
        plan.total_q = (int)total_q;
        p.n_jobs = plan.n_jobs;
        p.ds_base = plan.ds_base;
        p.k_jobs = plan.k_jobs;
        p.q_jobs = plan.q_jobs;
    }
    p.shares = d.shares;
    p.part = (float*)(ws + d.plan_bytes);
    p.part_rows = d.part_rows;
    p.ds = ws + d.plan_bytes + d.part_bytes;
    const int64_t rows = p.cu_q ? total_q : (int64_t)p.B * p.Sq;
    const int64_t delta_wgs = (rows + kRowsPerWg - 1) / kRowsPerWg * ((p.Hq + kHeadsPerWg - 1) / kHeadsPerWg) + (p.cu_q ? 2 : 0);
    const int64_t G = p.Hq / p.Hkv, k_jobs = p.cu_q ? d.k_room : p.n_ktiles;
    const int64_t q_jobs = p.cu_q ? d.q_room : ((int64_t)(p.Sq + kBwRows - 1) / kBwRows * G + kDqWaves - 1) / kDqWaves;
    if (delta_wgs > 0x7fffffffLL || k_jobs * d.units_per_pass * d.shares > 0x7fffffffLL || q_jobs * d.units_per_pass > 0x7fffffffLL)
        return (int)hipErrorInvalidValue;
    p.wide = d.wide;
    hipLaunchKernelGGL((bwd_delta_kernel<D, MODE>), dim3((unsigned)delta_wgs), dim3(kPlanThreads), p.cu_q ? plan_lds_bytes(plan, p.B) : 0, stream, p, plan);
    for (p.unit0 = 0; p.unit0 < d.n_units; p.unit0 += p.n_units) {
        p.n_units = std::min(d.units_per_pass, d.n_units - p.unit0);
        const dim3 grid((unsigned)(k_jobs * p.n_units * p.shares));
        if constexpr (D == 128) {
            if (p.wide) hipLaunchKernelGGL((bwd_dkv_wide_kernel<MODE>), grid, dim3(kWdWaves * 64), 0, stream, p);
        }
        if (!p.wide) hipLaunchKernelGGL((bwd_dkv_kernel<D, MODE, true>), grid, dim3(2 * kFuPairs * 64), 0, stream, p);
        hipLaunchKernelGGL((bwd_dq_ds_kernel<D, MODE>), dim3((unsigned)(q_jobs * p.n_units)), dim3(kDqWaves * 64), 0, stream, p);
    }
    if (p.shares > 1)
        hipLaunchKernelGGL((bwd_sum_shares_kernel<D>), dim3((unsigned)((p.part_rows * p.Hkv * (D / 4) + 255) / 256), 2), dim3(256), 0, stream, p);
    return (int)hipGetLastError();
}

template <int D>
static int launch_bwd_ds_mode(const BwdParams& p, const DsPasses& d, int mask_mode, int64_t total_q, unsigned char* ws, hipStream_t stream) {
    return mask_mode == MI355_MASK_CAUSAL ? launch_bwd_ds<D, MI355_MASK_CAUSAL>(p, d, total_q, ws, stream)
                                          : launch_bwd_ds<D, MI355_MASK_NONE>(p, d, total_q, ws, stream);
}

template <int D>
static int launch_bwd(const BwdParams& p, int mask_mode, hipStream_t stream) {
    if (mask_mode == MI355_MASK_CAUSAL) launch_bwd_mode<D, MI355_MASK_CAUSAL>(p, stream);
    else if (mask_mode == MI355_MASK_BOOL) launch_bwd_mode<D, MI355_MASK_BOOL>(p, stream);
    else launch_bwd_mode<D, MI355_MASK_NONE>(p, stream);
    return (int)hipGetLastError();
}

}  // namespace mi355

using namespace mi355;

static int prefill_bwd_common(const void* q, const void* k, const void* v, const void* out, const void* dout,
                              const float* lse, float* delta, void* dq, void* dk, void* dv,
                              const int64_t q_strides[3], const int64_t k_strides[3], const int64_t v_strides[3],
                              const int64_t o_strides[3], const int64_t do_strides[3], const int64_t dq_strides[3],
                              const int64_t dk_strides[3], const int64_t dv_strides[3], const int64_t lse_strides[2],
                              const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, const uint8_t* mask,
                              const int64_t* mask_strides, int B, int Hq, int Hkv, int Sq_max, int Sk_max, int D,
                              float softmax_scale, int mask_mode, int dtype, void* stream, int f32_grads = 0, int64_t total_q = 0,
                              int64_t total_k = 0, void* workspace = nullptr, int64_t workspace_bytes = 0) {
    if (!q || !k || !v || !out || !dout || !lse || !delta || !dq || !dk || !dv)
        return set_error(MI355_EINVAL, "prefill_bwd: null pointer argument");
    if (!q_strides || !k_strides || !v_strides || !o_strides || !do_strides || !dq_strides || !dk_strides || !dv_strides ||
        !lse_strides)
        return set_error(MI355_EINVAL, "prefill_bwd: null stride argument");
    if (dtype != MI355_BF16) return set_error(MI355_EDTYPE, "prefill_bwd: dtype must be MI355_BF16");
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || Sq_max <= 0 || Sk_max <= 0)
        return set_error(MI355_EINVAL, "prefill_bwd: B, Hq, Hkv, Sq_max and Sk_max must be positive");
    if (Hq % Hkv != 0) return set_error(MI355_EINVAL, "prefill_bwd: Hq must be a multiple of Hkv");
    if (!(D == 128 || D == 64 || D == 32)) return set_error(MI355_EINVAL, "prefill_bwd: head_dim must be 32, 64 or 128");
    if ((cu_seqlens_q == nullptr) != (cu_seqlens_k == nullptr))
        return set_error(MI355_EINVAL, "prefill_bwd: cu_seqlens_q and cu_seqlens_k must be given together");
    if (mask_mode < MI355_MASK_NONE || mask_mode > MI355_MASK_BOOL) return set_error(MI355_EINVAL, "prefill_bwd: unknown mask_mode");
    if (mask_mode == MI355_MASK_BOOL) {
        if (!mask || !mask_strides || cu_seqlens_q)
            return set_error(MI355_EINVAL, "prefill_bwd: MI355_MASK_BOOL needs mask + mask_strides and the dense layout");
        if (((uintptr_t)mask | (uintptr_t)mask_strides[0] | (uintptr_t)mask_strides[1] | (uintptr_t)mask_strides[2]) & 3)
            return set_error(MI355_EINVAL, "prefill_bwd: the mask and its strides must be multiples of 4 bytes");
        if (mask_strides[0] < 0 || mask_strides[1] < 0 || mask_strides[2] < 0)
            return set_error(MI355_EINVAL, "prefill_bwd: mask strides must not be negative");
    }
    const int64_t* all[8] = {q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides, dk_strides, dv_strides};
    for (const int64_t* st : all)
        for (int i = 0; i < 3; ++i)
            if (st[i] & 7) return set_error(MI355_EINVAL, "prefill_bwd: strides must be multiples of 8 elements (16-byte rows)");
    const int64_t* rows[4] = {q_strides, k_strides, v_strides, do_strides};
    for (const int64_t* st : rows)
        if (st[2] <= 0 || st[2] >= (1 << 24))
            return set_error(MI355_EINVAL, "prefill_bwd: row strides must be positive and below 2^24 elements");
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk |
         (uintptr_t)dv) & 15)
        return set_error(MI355_EINVAL, "prefill_bwd: tensors must be 16-byte aligned");

    BwdParams p;
    p.q = (const __bf16*)q;
    p.k = (const __bf16*)k;
    p.v = (const __bf16*)v;
    p.out = (const __bf16*)out;
    p.dout = (const __bf16*)dout;
    p.lse = lse;
    p.delta = delta;
    p.dq = dq;
    p.dk = dk;
    p.dv = dv;
    p.dq_f32 = f32_grads & 1;
    p.dk_f32 = f32_grads & 2;
    p.dv_f32 = f32_grads & 4;
    for (int i = 0; i < 3; ++i) {
        p.qs[i] = q_strides[i];
        p.ks[i] = k_strides[i];
        p.vs[i] = v_strides[i];
        p.os[i] = o_strides[i];
        p.dos[i] = do_strides[i];
        p.dqs[i] = dq_strides[i];
        p.dks[i] = dk_strides[i];
        p.dvs[i] = dv_strides[i];
    }
    p.ls[0] = lse_strides[0];
    p.ls[1] = lse_strides[1];
    p.cu_q = cu_seqlens_q;
    p.cu_k = cu_seqlens_k;
    p.mask = mask_mode == MI355_MASK_BOOL ? mask : nullptr;
    for (int i = 0; i < 3; ++i) p.ms[i] = mask_mode == MI355_MASK_BOOL ? mask_strides[i] : 0;
    p.B = B;
    p.Hq = Hq;
    p.Hkv = Hkv;
    p.Sq = Sq_max;
    p.Sk = Sk_max;
    p.scale = softmax_scale;
    p.scale_log2 = softmax_scale * kLog2e;
    p.n_qtiles = (Sq_max + kBwCols - 1) / kBwCols;
    p.n_ktiles = (Sk_max + kFuCols - 1) / kFuCols;
    if ((int64_t)p.n_qtiles * Hq * B > 0x7fffffffLL || (int64_t)p.n_ktiles * Hkv * B > 0x7fffffffLL)
        return set_error(MI355_EINVAL, "prefill_bwd: too many workgroups");

    hipStream_t s = (hipStream_t)stream;
    p.ds = nullptr;
    p.unit0 = p.n_units = 0;
    p.n_jobs = p.ds_base = nullptr;
    p.k_jobs = p.q_jobs = nullptr;
    p.shares = 1;
    p.part = nullptr;
    p.part_rows = 0;
    p.wide = false;
    if (workspace) {
        DsPasses d;
        if (!ds_passes(B, Hq, Hkv, Sq_max, Sk_max, D, mask_mode, cu_seqlens_q != nullptr, cu_seqlens_q == cu_seqlens_k, total_q, total_k, d))
            return set_error(MI355_EINVAL, "prefill_bwd: no form with a workspace for this call (packed: total_q and total_k are the tensors' rows)");
        // (a smaller workspace takes more passes)
        if (d.unit_bytes > 0) d.units_per_pass = (int)std::min<int64_t>(d.units_per_pass, (workspace_bytes - d.plan_bytes - d.part_bytes) / d.unit_bytes);
        if (((uintptr_t)workspace & 255) || workspace_bytes < d.bytes() || d.units_per_pass < 1)
            return set_error(MI355_EINVAL, "prefill_bwd: the workspace is too small or not 256-byte aligned");
        unsigned char* ws = (unsigned char*)workspace;
        const int rc = D == 128 ? launch_bwd_ds_mode<128>(p, d, mask_mode, total_q, ws, s)
                                : (D == 64 ? launch_bwd_ds_mode<64>(p, d, mask_mode, total_q, ws, s) : launch_bwd_ds_mode<32>(p, d, mask_mode, total_q, ws, s));
        return rc == 0 ? MI355_OK : set_error(rc, hipGetErrorString((hipError_t)rc));
    }
    if (!p.cu_q && prefill_bwd_short_takes(Hq, Hkv, Sq_max, Sk_max, D, mask_mode)) {
        const int rc = launch_prefill_bwd_short(p, D, mask_mode, s);
        return rc == 0 ? MI355_OK : set_error(rc, hipGetErrorString((hipError_t)rc));
    }
    int rc = D == 128 ? launch_bwd<128>(p, mask_mode, s)
                      : (D == 64 ? launch_bwd<64>(p, mask_mode, s) : launch_bwd<32>(p, mask_mode, s));
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

extern "C" int mi355_prefill_bwd(const void* q, const void* k, const void* v, const void* out, const void* dout,
                                 const float* lse, float* delta, void* dq, void* dk, void* dv,
                                 const int64_t q_strides[3], const int64_t k_strides[3], const int64_t v_strides[3],
                                 const int64_t o_strides[3], const int64_t do_strides[3], const int64_t dq_strides[3],
                                 const int64_t dk_strides[3], const int64_t dv_strides[3], const int64_t lse_strides[2],
                                 const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int B, int Hq,
                                 int Hkv, int Sq_max, int Sk_max, int D, float softmax_scale, int mask_mode, int dtype,
                                 void* stream) {
    if (mask_mode == MI355_MASK_BOOL)
        return set_error(MI355_EINVAL, "prefill_bwd: mask_mode must be MI355_MASK_NONE or MI355_MASK_CAUSAL (an explicit mask goes through mi355_prefill_bwd_mask)");
    return prefill_bwd_common(q, k, v, out, dout, lse, delta, dq, dk, dv, q_strides, k_strides, v_strides, o_strides,
                              do_strides, dq_strides, dk_strides, dv_strides, lse_strides, cu_seqlens_q, cu_seqlens_k,
                              nullptr, nullptr, B, Hq, Hkv, Sq_max, Sk_max, D, softmax_scale, mask_mode, dtype, stream);
}

extern "C" int mi355_prefill_bwd_mask(const void* q, const void* k, const void* v, const void* out, const void* dout,
                                      const float* lse, float* delta, void* dq, void* dk, void* dv,
                                      const int64_t q_strides[3], const int64_t k_strides[3], const int64_t v_strides[3],
                                      const int64_t o_strides[3], const int64_t do_strides[3], const int64_t dq_strides[3],
                                      const int64_t dk_strides[3], const int64_t dv_strides[3],
                                      const int64_t lse_strides[2], const uint8_t* mask, const int64_t mask_strides[3],
                                      int B, int Hq, int Hkv, int Sq, int Sk, int D, float softmax_scale, int dtype,
                                      void* stream) {
    return prefill_bwd_common(q, k, v, out, dout, lse, delta, dq, dk, dv, q_strides, k_strides, v_strides, o_strides,
                              do_strides, dq_strides, dk_strides, dv_strides, lse_strides, nullptr, nullptr, mask,
                              mask_strides, B, Hq, Hkv, Sq, Sk, D, softmax_scale, MI355_MASK_BOOL, dtype, stream);
}

extern "C" int mi355_prefill_bwd_typed(const void* q, const void* k, const void* v, const void* out, const void* dout,
                                       const float* lse, float* delta, void* dq, void* dk, void* dv,
                                       const int64_t q_strides[3], const int64_t k_strides[3], const int64_t v_strides[3],
                                       const int64_t o_strides[3], const int64_t do_strides[3], const int64_t dq_strides[3],
                                       const int64_t dk_strides[3], const int64_t dv_strides[3],
                                       const int64_t lse_strides[2], const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                       const uint8_t* mask, const int64_t mask_strides[3], int f32_grads, int B, int Hq, int Hkv,
                                       int Sq_max, int Sk_max, int D, float softmax_scale, int mask_mode, int dtype, void* stream) {
    if (f32_grads < 0 || f32_grads > 7) return set_error(MI355_EINVAL, "prefill_bwd: f32_grads has three bits");
    return prefill_bwd_common(q, k, v, out, dout, lse, delta, dq, dk, dv, q_strides, k_strides, v_strides, o_strides,
                              do_strides, dq_strides, dk_strides, dv_strides, lse_strides, cu_seqlens_q, cu_seqlens_k, mask,
                              mask_strides, B, Hq, Hkv, Sq_max, Sk_max, D, softmax_scale, mask_mode, dtype, stream, f32_grads);
}

extern "C" int64_t mi355_prefill_bwd_ds_workspace(int B, int Hq, int Hkv, int Sq_max, int Sk_max, int D, int mask_mode, int packed, int same_bounds,
                                                  int64_t total_q, int64_t total_k) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Sq_max <= 0 || Sk_max <= 0) return 0;
    DsPasses d;
    return ds_passes(B, Hq, Hkv, Sq_max, Sk_max, D, mask_mode, packed != 0, same_bounds != 0, total_q, total_k, d) ? d.bytes() : 0;
}

extern "C" int mi355_prefill_bwd_ds_kernel(int B, int Hq, int Hkv, int Sq_max, int Sk_max, int D, int mask_mode, int packed, int same_bounds, int64_t total_q,
                                           int64_t total_k, int* shares) {
    DsPasses d;
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Sq_max <= 0 || Sk_max <= 0 ||
        !ds_passes(B, Hq, Hkv, Sq_max, Sk_max, D, mask_mode, packed != 0, same_bounds != 0, total_q, total_k, d))
        return 0;
    if (shares) *shares = d.shares;
    return d.wide ? MI355_BWD_DS_WIDE : MI355_BWD_DS_ROLES;
}

extern "C" int mi355_prefill_bwd_ds(const void* q, const void* k, const void* v, const void* out, const void* dout, const float* lse,
                                    float* delta, void* dq, void* dk, void* dv, const int64_t q_strides[3], const int64_t k_strides[3],
                                    const int64_t v_strides[3], const int64_t o_strides[3], const int64_t do_strides[3],
                                    const int64_t dq_strides[3], const int64_t dk_strides[3], const int64_t dv_strides[3],
                                    const int64_t lse_strides[2], const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int f32_grads, int B,
                                    int Hq, int Hkv, int Sq_max, int Sk_max, int D, float softmax_scale, int mask_mode, int dtype, int64_t total_q,
                                    int64_t total_k, void* workspace, int64_t workspace_bytes, void* stream) {
    if (f32_grads < 0 || f32_grads > 7) return set_error(MI355_EINVAL, "prefill_bwd: f32_grads has three bits");
    if (!workspace) return set_error(MI355_EINVAL, "prefill_bwd: null workspace");
    return prefill_bwd_common(q, k, v, out, dout, lse, delta, dq, dk, dv, q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides,
                              dk_strides, dv_strides, lse_strides, cu_seqlens_q, cu_seqlens_k, nullptr, nullptr, B, Hq, Hkv, Sq_max, Sk_max, D,
                              softmax_scale, mask_mode, dtype, stream, f32_grads, total_q, total_k, workspace, workspace_bytes);
}
