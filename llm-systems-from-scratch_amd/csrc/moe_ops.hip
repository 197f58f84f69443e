// Mixture-of-experts feed-forward on gfx950: router, grouping of tokens by expert, grouped matrix products.
//
// Every token of a step chooses `top` of E experts; a (token, choice) is a pair, numbered token * top + choice.
//   route   logits in fp32 (bf16 operands on MFMA, or fp32 throughout), the largest `top` of them, softmax over those
//   group   pairs sorted by expert: order[], and offsets[e] = first place of expert e's pairs in it
//   gate_up act[i] = silu(Wg h_i) * (Wu h_i) for place i of the order, h_i the pair's token
//   down    out[pair] = weight[pair] * (Wd act[i])
// The products are tiled per expert.  Tiles of expert e start at number offsets[e] / BM + e (the large tiles: where those of
// e - 1 end), so the tile -> expert search needs the offsets alone, and a launch of n_pairs / BM + E row tiles covers every
// distribution of the tokens.  A row of a product depends on its own token only, so neither the order inside an expert nor the tiling shows in a result.
//   moe_wide_kernel    256 x 256 tiles through LDS: long prompts
//   moe_gemm_kernel    128 x 128 tiles through LDS: prompts
//   moe_direct_kernel  32 weight rows, streamed through LDS, against an expert's rows, no grouping needed: decoding
//   moe_skinny_kernel  16 rows x 16 (+ 16) weight rows, weights straight to registers: few pairs per expert, many experts
//   moe_f32_kernel     fp32 on the vector unit
#include "common.hpp"
#include "launch.hpp"
#include "weight_stream.hpp"
#include "xcd_order.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mi355 {

constexpr int kMaxExperts = 1024;
constexpr int kMaxTop = 64;

__device__ __forceinline__ float moe_wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// ---- router -------------------------------------------------------------------------------------
struct RouteParams {
    const void* h;
    const void* w;               // (E + extra, k) rows of h's type, stride w_stride
    const float* bias;           // (E + extra)
    int32_t* ids;                // (T, top)
    float* weights;              // (T, top)
    float* extra_logit;          // (T): the logit of row E, or null
    int64_t T, h_stride, w_stride;
    int k, E, n_logits, top;
};

// One wavefront: the `top` largest of the E logits at z (LDS; overwritten), their softmax.  Ties go to the lower index.
__device__ __forceinline__ void choose_experts(const RouteParams& p, float* z, int64_t token, int lane) {
    float mine = -INFINITY;                       // logit of choice `lane`
    int mine_id = 0;
    for (int c = 0; c < p.top; ++c) {
        float best = -INFINITY;
        int id = 0x7fffffff;
        for (int e = lane; e < p.E; e += 64) {
            const float v = z[e];
            if (v > best || (v == best && e < id && v > -INFINITY)) {
                best = v;
                id = e;
            }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float v = __shfl_xor(best, off, 64);
            const int i = __shfl_xor(id, off, 64);
            if (v > best || (v == best && i < id)) {
                best = v;
                id = i;
            }
        }
        id = min(id, p.E - 1);                    // (logits that are not numbers: some valid expert)
        if (lane == id % 64) z[id] = -INFINITY;
        if (lane == c) {
            mine = best;
            mine_id = id;
        }
    }
    const float top1 = __shfl(mine, 0, 64);
    const float e = lane < p.top ? expf(mine - top1) : 0.f;
    const float sum = moe_wave_sum(e);
    if (lane < p.top) {
        p.ids[token * p.top + lane] = mine_id;
        p.weights[token * p.top + lane] = e / sum;
    }
}

// Up to 64 logits: GROUP lanes per token, a lane owns one logit and counts those in front of it (larger, or as large with a
// lower index), which is its place; 64 / GROUP tokens at a time.  The general form above walks the maxima one after the other,
// six exchanges each: 16 of 23 us for 8192 tokens of 16 logits, four chosen, were spent there.  What is no number counts as
// -inf, and a choice without a logit above -inf is expert E - 1, as there.  (Router of 32 logits with 64 / 32 lanes per token: 81 tokens 7.7 / 6.1 us,
// 3588 8.4 / 6.5.)
template <int GROUP>
__device__ __forceinline__ void choose_by_rank(const RouteParams& p, const float* z, int64_t t0, int lane, int wave, int n_waves) {
    const int e = lane % GROUP;
    for (int t = wave * (64 / GROUP) + lane / GROUP; t < 16; t += n_waves * (64 / GROUP)) {
        const float* zt = z + t * p.n_logits;
        float mine = e < p.E ? zt[e] : -INFINITY;
        mine = mine > -INFINITY ? mine : -INFINITY;
        float top1 = mine;
#pragma unroll
        for (int off = GROUP / 2; off >= 1; off >>= 1) top1 = fmaxf(top1, __shfl_xor(top1, off, 64));
        int rank = 0;
        for (int j = 0; j < p.E; ++j) {
            float v = zt[j];
            v = v > -INFINITY ? v : -INFINITY;
            rank += v > mine || (v == mine && j < e);
        }
        const bool chosen = e < p.E && rank < p.top;
        const float w = chosen ? expf(mine - top1) : 0.f;
        float sum = w;
#pragma unroll
        for (int off = GROUP / 2; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (chosen && t0 + t < p.T) {
            p.ids[(t0 + t) * p.top + rank] = mine > -INFINITY ? e : p.E - 1;
            p.weights[(t0 + t) * p.top + rank] = w / sum;
        }
    }
}

// 16 tokens per workgroup; the wavefronts take the 32-wide steps of k in turn and meet in LDS.  TILES: 16-logit tiles per pass.
// The loads of BATCH steps are in flight together: with one or two tiles, eight (k = 2048 in one go), which is what a launch
// of few tokens is made of (32 tokens, 16 logits, k = 2048: 13.9 us with four tiles and four steps, 7.6 us like this).
constexpr int kRouteWaves = 8;
template <int TILES, int BATCH>
__global__ __launch_bounds__(64 * kRouteWaves) void moe_route_kernel(RouteParams p) {
    extern __shared__ __attribute__((aligned(16))) float route_lds[];
    f32x4* part = reinterpret_cast<f32x4*>(route_lds);                         // [wave][tile][lane]
    float* z = route_lds + kRouteWaves * TILES * 64 * 4;                              // [16][n_logits]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int64_t t0 = (int64_t)blockIdx.x * 16;
    const __bf16* h = (const __bf16*)p.h + min(t0 + r, p.T - 1) * p.h_stride;
    for (int l0 = 0; l0 < p.n_logits; l0 += 16 * TILES) {
        f32x4 acc[TILES];
        const __bf16* w[TILES];
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
            acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            w[j] = (const __bf16*)p.w + (int64_t)min(l0 + 16 * j + r, p.n_logits - 1) * p.w_stride;
        }
        for (int k0 = 32 * wave; k0 < p.k; k0 += 32 * kRouteWaves * BATCH) {       // BATCH steps' loads, then their products
            u32x4 hv[BATCH], wv[TILES][BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const int col = k0 + 32 * kRouteWaves * i + 8 * kg;
                const bool in = col < p.k;
                hv[i] = u32x4{0u, 0u, 0u, 0u};
                if (in) hv[i] = *reinterpret_cast<const u32x4*>(h + col);
#pragma unroll
                for (int j = 0; j < TILES; ++j) {
                    wv[j][i] = u32x4{0u, 0u, 0u, 0u};
                    if (in && l0 + 16 * j < p.n_logits) wv[j][i] = *reinterpret_cast<const u32x4*>(w[j] + col);
                }
            }
#pragma unroll
            for (int j = 0; j < TILES; ++j)
                if (l0 + 16 * j < p.n_logits)
#pragma unroll
                    for (int i = 0; i < BATCH; ++i) acc[j] = mfma16(as_bf16x8(wv[j][i]), as_bf16x8(hv[i]), acc[j]);      // column r: token, rows 4 kg + i: logits
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TILES; ++j) part[(wave * TILES + j) * 64 + lane] = acc[j];
        __syncthreads();
        // wavefront j sums tile j
        if (wave < TILES) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w8 = 0; w8 < kRouteWaves; ++w8) s += part[(w8 * TILES + wave) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int l = l0 + 16 * wave + 4 * kg + i;
                if (l < p.n_logits) z[r * p.n_logits + l] = s[i] + p.bias[l];
            }
        }
    }
    __syncthreads();
    if (p.extra_logit && tid < 16 && t0 + tid < p.T) p.extra_logit[t0 + tid] = z[tid * p.n_logits + p.E];
    if (p.E <= 16) return choose_by_rank<16>(p, z, t0, lane, wave, kRouteWaves);
    if (p.E <= 32) return choose_by_rank<32>(p, z, t0, lane, wave, kRouteWaves);
    if (p.E <= 64) return choose_by_rank<64>(p, z, t0, lane, wave, kRouteWaves);
    for (int t = wave; t < 16; t += kRouteWaves) {
        if (t0 + t >= p.T) break;
        choose_experts(p, z + t * p.n_logits, t0 + t, lane);
    }
}

// fp32: one wavefront per token
__global__ __launch_bounds__(256) void moe_route_f32_kernel(RouteParams p) {
    extern __shared__ __attribute__((aligned(16))) float route_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t = (int64_t)blockIdx.x * 4 + wave;
    if (t >= p.T) return;
    float* z = route_lds + wave * p.n_logits;
    const float* h = (const float*)p.h + t * p.h_stride;
    for (int l = 0; l < p.n_logits; ++l) {
        const float* w = (const float*)p.w + (int64_t)l * p.w_stride;
        float s = 0.f;
        for (int c = lane; c < p.k; c += 64) s = fmaf(w[c], h[c], s);
        s = moe_wave_sum(s) + p.bias[l];
        if (lane == l % 64) z[l] = s;             // (the lane that reads it below)
    }
    if (p.extra_logit && lane == p.E % 64) p.extra_logit[t] = z[p.E];
    choose_experts(p, z, t, lane);
}

static void launch_route(const RouteParams& p, hipStream_t s) {
    const dim3 grid((unsigned)((p.T + 15) / 16)), block(64 * kRouteWaves);
    const auto lds = [&](int tiles) { return (kRouteWaves * tiles * 64 * 4 + 16 * p.n_logits) * sizeof(float); };
    if (p.n_logits <= 16) hipLaunchKernelGGL((moe_route_kernel<1, 8>), grid, block, lds(1), s, p);
    else if (p.n_logits <= 32) hipLaunchKernelGGL((moe_route_kernel<2, 8>), grid, block, lds(2), s, p);
    else hipLaunchKernelGGL((moe_route_kernel<4, 4>), grid, block, lds(4), s, p);
}

// ---- pairs sorted by expert -----------------------------------------------------------------------
// Workgroup e lists expert e's pairs: each of its 16 wavefronts counts the pairs of lower experts and of its own expert in
// its share of the ids, the shares are summed, and a second pass writes.
__global__ __launch_bounds__(1024) void moe_group_kernel(const int32_t* ids, int n_pairs, int E, int32_t* offsets, int32_t* order) {
    __shared__ int below[16], equal[16];
    const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int share = ((n_pairs + 15) / 16 + 63) / 64 * 64;
    const int i0 = min(n_pairs, wave * share), i1 = min(n_pairs, i0 + share);
    constexpr int kAhead = 8;                     // loads in flight: one at a time, 32768 pairs took 23 us
    int n_below = 0, n_equal = 0;
    for (int i = i0; i < i1; i += 64 * kAhead) {
        int id[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) id[j] = i + 64 * j + lane < i1 ? ids[i + 64 * j + lane] : E;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            n_below += __popcll(__builtin_amdgcn_ballot_w64(id[j] < e));
            n_equal += __popcll(__builtin_amdgcn_ballot_w64(id[j] == e));
        }
    }
    if (lane == 0) {
        below[wave] = n_below;
        equal[wave] = n_equal;
    }
    __syncthreads();
    int at = 0;
    for (int w = 0; w < 16; ++w) at += below[w] + (w < wave ? equal[w] : 0);
    if (threadIdx.x == 0) {
        offsets[e] = at;
        if (e == E - 1) offsets[E] = n_pairs;
    }
    if (n_equal == 0) return;
    for (int i = i0; i < i1; i += 64 * kAhead) {
        int id[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) id[j] = i + 64 * j + lane < i1 ? ids[i + 64 * j + lane] : E;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const uint64_t m = __builtin_amdgcn_ballot_w64(id[j] == e);
            if (id[j] == e) order[at + __popcll(m & ((1ull << lane) - 1))] = i + 64 * j + lane;
            at += __popcll(m);
        }
    }
}

// ---- grouped products -------------------------------------------------------------------------------
struct MoeParams {
    const void* a;               // rows of the left operand: tokens (gather) or places of the order
    const void* w;               // (E, rows of w, k)
    void* out;
    const int32_t *offsets, *order;
    const float* weights;        // down: per pair
    int64_t a_stride, a_rows, out_stride, out_rows;
    int n_pairs, E, k, n;        // n: output columns (gate_up: w has 2 n rows, gates first)
    int top;
};

// expert and first place of row tile `tile`; false: the tile has no rows.  A lane looks at one expert (64 at a time): one load
// in front of a tile's first operand where a binary search has a chain of them.
template <int BM>
__device__ __forceinline__ bool find_tile(const MoeParams& p, int tile, int& e, int& first, int& end) {
    const int lane = threadIdx.x & 63;
    int start = 0, stop = 0;
    e = 0;
    for (int e0 = 0; e0 < p.E; e0 += 64) {
        const int mine = min(e0 + lane, p.E - 1), o0 = p.offsets[mine], o1 = p.offsets[mine + 1];
        const uint64_t m = __builtin_amdgcn_ballot_w64(e0 + lane < p.E && o0 / BM + mine <= tile);
        if (m == 0) break;                        // (the first tile numbers rise with the expert)
        const int last = 63 - __builtin_clzll(m);
        e = e0 + last;
        start = __builtin_amdgcn_readlane(o0, last);
        stop = __builtin_amdgcn_readlane(o1, last);
    }
    end = min(stop, p.n_pairs);
    first = start + (tile - (start / BM + e)) * BM;
    return first >= start && first < end;
}

// The same for workgroup `bid` of a launch with n_tiles columns of tiles, for the large tiles, where a round of the chip counts more
// than a scan over the experts: the tiles are numbered without gaps and dealt to the XCDs by how many of them have rows, not by the
// launch's bound, so that no XCD gets more workgroups than the others (16 experts of 2048 x 1024, top 4, 128 x 128 tiles, 1800
// tokens: both products 138 -> 115 us; 32 of 2048 x 2048, 512 pairs: 240 -> 200.  Numbered without gaps but dealt by the bound, what
// came behind the last whole round fell on some of the XCDs: 16 experts, 512 tokens, uniform ids 61 us and 55 like this, skewed ones
// 68 and 57; 32 experts of 1024 x 512, top 2, 1500 tokens 36 and 31).
template <int BM>
__device__ __forceinline__ bool find_dense_tile(const MoeParams& p, int bid, int n_tiles, int chunk, int& n_tile, int& e, int& first, int& end) {
    const int lane = threadIdx.x & 63;
    int o0, o1, n, sum, total = 0;
    const auto scan = [&](int e0) {               // tiles of the 64 experts from e0 on; sum: with those in front of each
        const int mine = min(e0 + lane, p.E - 1);
        o0 = p.offsets[mine];
        o1 = p.offsets[mine + 1];
        n = e0 + lane < p.E ? (max(o1 - o0, 0) + BM - 1) / BM : 0;
        sum = running_sum(n);
    };
    for (int e0 = 0; e0 < p.E; e0 += 64) {
        scan(e0);
        total += __builtin_amdgcn_readlane(sum, 63);
    }
    total = min(total, p.n_pairs / BM + p.E);     // (the launch's bound, whatever the offsets are)
    if (bid >= total * n_tiles) return false;
    const int id = __builtin_amdgcn_readfirstlane(xcd_even_id(bid, total * n_tiles, chunk)), tile = id / n_tiles;
    n_tile = id - tile * n_tiles;
    for (int e0 = 0, before = 0; e0 < p.E; e0 += 64) {
        if (p.E > 64) scan(e0);
        const uint64_t m = __builtin_amdgcn_ballot_w64(tile < before + sum);
        if (m != 0) {
            const int at = __builtin_ctzll(m), start = __builtin_amdgcn_readlane(o0, at);
            e = e0 + at;
            first = start + (tile - before - __builtin_amdgcn_readlane(sum - n, at)) * BM;
            end = min(__builtin_amdgcn_readlane(o1, at), p.n_pairs);
            return first >= start && first < end;
        }
        before += __builtin_amdgcn_readlane(sum, 63);
    }
    return false;
}

// row of the left operand for place i of the order
template <bool GATE_UP>
__device__ __forceinline__ int64_t left_row(const MoeParams& p, int i) {
    const int64_t row = GATE_UP ? p.order[i] / p.top : i;
    return min(max(row, (int64_t)0), p.a_rows - 1);
}

__device__ __forceinline__ float silu_fast(float x) { return x * __builtin_amdgcn_rcpf(1.0f + fast_exp2(-kLog2e * x)); }

// Four adjacent columns of one row into the output; out_row: place (gate_up) or pair (down)
__device__ __forceinline__ void store4(const MoeParams& p, int64_t out_row, int col, const float (&v)[4]) {
    __bf16* o = (__bf16*)p.out + out_row * p.out_stride + col;
    if (col + 4 <= p.n) {
        *reinterpret_cast<u32x2*>(o) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (col + i < p.n) o[i] = (__bf16)v[i];
    }
}

// 128 rows x 128 rows of w per workgroup (gate_up: 64 gates and the 64 ups of the same columns), k in steps of 64 through LDS,
// filled by direct loads.  A 128-byte LDS row holds its eight 16-byte pieces in the order piece ^ (row % 8).
// Wavefront (wm, wn) computes 64 x 64; weights are the MFMA's first operand, so that a lane ends with adjacent columns.
// Bound by the latency of its weights where there are few rows: they come from HBM, the rows from an L2.  So weights have three buffers
// and are requested two steps ahead, rows two and one: all that two workgroups per compute unit leave of its 160 KB.  us of router and both
// products, two buffers of each / this / rows two and weights five steps ahead with one workgroup per compute unit:
//   tokens x hidden, experts of width, top k    334 x 2048, 8 of 2048, 1    320 x 2048, 16 of 1024, 4    550 x 2048, 32 of 2048, 4
//                                               86 / 75 / 78                78 / 72 / 73                 222 / 215 / 222
//                                               2640 x 1024, 32 of 512, 4   4108 x 1024, 16 of 1024, 4   2609 x 2048, 8 of 1024, 1
//                                               97 / 90 / 88                173 / 167 / 188              84 / 82 / 104
// TURN: the workgroups of an XCD begin 0, 8, 16 or 24 steps of k in, by their columns and expert, so that a row's sums do not depend on the tile it falls into.  Rows of whole 4096 bytes from step 0 on all want the same channels of its L2 (turn_of), and
// weights that come from HBM wait for these: 32 experts of 2048 x 2048, 64 pairs an expert 200 -> 154 us, 16 of 2048 x 1024 32 pairs 54.5 -> 45.7, 128 pairs 78.1 -> 77.1,
// 8 of 2048 x 2048 75 pairs 66 -> 56, 250 pairs 103.9 / 104.2.  Where an expert's row tiles share its weights in the L2 their steps had better go together, so
// not behind 256 pairs an expert (longer rows: 96; pairs an expert, without / with: 16 of 4096 x 1024 64 11 % less, 128 4 % more, 4 of 4096 x 4096 64 10 % less, 128 7 % more), and not in the
// 256 x 256 tiles (396 -> 399 to 409).
template <bool GATE_UP, bool TURN>
__global__ __launch_bounds__(256, 2) void moe_gemm_kernel(MoeParams p, int n_tiles, int chunk) {
    constexpr int BM = 128, BK = 64, kTile = 128 * BK * 2, NA = 2, NW = 3;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[(NA + NW) * kTile];          // rows, then w
    int n_tile, e, first, end;
    if (!find_dense_tile<BM>(p, blockIdx.x, n_tiles, chunk, n_tile, e, first, end)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, r = lane & 15, kg = lane >> 4;
    const int n0 = n_tile * (GATE_UP ? 64 : 128);
    const __bf16* a_base = (const __bf16*)p.a;
    const __bf16* w_base = (const __bf16*)p.w + (int64_t)e * (GATE_UP ? 2 : 1) * p.n * p.k;
    // wavefront w fills rows 32 w .. 32 w + 31 of both tiles, 8 rows per load
    uint32_t a_off[4], w_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 32 * wave + 8 * j + (lane >> 3), piece = (lane & 7) ^ (row & 7);
        a_off[j] = (uint32_t)((left_row<GATE_UP>(p, min(first + row, end - 1)) * p.a_stride + piece * 8) * 2);
        int64_t wr = GATE_UP ? (row < 64 ? min(n0 + row, p.n - 1) : p.n + min(n0 + row - 64, p.n - 1)) : min(n0 + row, p.n - 1);
        w_off[j] = (uint32_t)((wr * p.k + piece * 8) * 2);
    }
    const uint32_t lds0 = lds_address(lds);
    const int n_steps = p.k / BK, turn = TURN ? (e * n_tiles + n_tile) % 4 * 8 : 0;
    const auto turned = [&](int step) { return (TURN && step + turn >= n_steps ? step + turn - n_steps : step + turn) * BK; };
    const auto issue_a = [&](int step, int slot) {
#pragma unroll
        for (int j = 0; j < 4; ++j) dma_to_lds_16(a_base + turned(step), a_off[j], lds0 + slot * kTile + (32 * wave + 8 * j) * 128);
    };
    const auto issue_w = [&](int step, int slot) {
#pragma unroll
        for (int j = 0; j < 4; ++j) dma_to_lds_16(w_base + turned(step), w_off[j], lds0 + (NA + slot) * kTile + (32 * wave + 8 * j) * 128);
    };
    f32x4 acc[4][4];                              // [16 rows of w][16 rows]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // 16-row groups of w of this wavefront: gate_up: gates 32 wn, 32 wn + 16, then the ups of these columns
    const auto w_group = [&](int i) { return GATE_UP ? (i >> 1) * 64 + 32 * wn + (i & 1) * 16 : 64 * wn + 16 * i; };
    // in the order of the loop: w of a step, its rows, w of the next
    issue_w(0, 0);
    issue_a(0, 0);
    if (n_steps > 1) issue_w(1, 1);
    for (int t = 0, sa = 0, sw = 0; t < n_steps; ++t) {
        if (t + 1 < n_steps) wait_vmcnt<4>();     // all but w of step t + 1 has landed
        else wait_vmcnt<0>();
        __syncthreads();                          // ... everybody's, and everybody has read the step before
        if (t + 1 < n_steps) issue_a(t + 1, sa ^ 1);
        if (t + 2 < n_steps) issue_w(t + 2, sw == 0 ? 2 : sw - 1);
        const unsigned char* at = lds + sa * kTile;
        const unsigned char* wt = lds + (NA + sw) * kTile;
        sa ^= 1;
        sw = sw == 2 ? 0 : sw + 1;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int piece = ((4 * s + kg) ^ (r & 7)) * 16;
            bf16x8 wf[4], af[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wf[i] = as_bf16x8(*reinterpret_cast<const u32x4*>(wt + (w_group(i) + r) * 128 + piece));
                af[i] = as_bf16x8(*reinterpret_cast<const u32x4*>(at + (64 * wm + 16 * i + r) * 128 + piece));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma16(wf[i], af[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int place = first + 64 * wm + 16 * j + r;
        if (place >= end) continue;
        if constexpr (GATE_UP) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = silu_fast(acc[i][j][q]) * acc[i + 2][j][q];
                store4(p, place, n0 + 32 * wn + 16 * i + 4 * kg, v);
            }
        } else {
            const int pair = min(max(p.order[place], 0), p.n_pairs - 1);
            const float wgt = p.weights[pair];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = wgt * acc[i][j][q];
                store4(p, pair, n0 + 64 * wn + 16 * i + 4 * kg, v);
            }
        }
    }
}

// ---- 256 x 256 tiles ----
// The row tiles of a launch in the order in which they are worked on: an expert's full ones, then what remains of the experts with more
// than half a tile left, then of those with less.  n tiles of the widest kind in columns make up a row tile.
struct WideTiles {
    int o0, o1;                                   // this lane's expert of the first 64: where its places begin and end
    int full, large, small;                       // row tiles of each kind
};
__device__ __forceinline__ void wide_kinds(int o0, int o1, bool any, int (&n)[3]) {
    const int rows = any ? max(o1 - o0, 0) : 0;
    n[0] = rows >> 8;
    n[1] = (rows & 255) > 128;
    n[2] = (rows & 255) > 0 && (rows & 255) <= 128;
}
__device__ __forceinline__ WideTiles wide_tiles(const MoeParams& p) {
    const int lane = threadIdx.x & 63;
    WideTiles t{};
    for (int e0 = 0; e0 < p.E; e0 += 64) {
        const int mine = min(e0 + lane, p.E - 1), o0 = p.offsets[mine], o1 = p.offsets[mine + 1];
        if (e0 == 0) {
            t.o0 = o0;
            t.o1 = o1;
        }
        int n[3];
        wide_kinds(o0, o1, e0 + lane < p.E, n);
        t.full += __builtin_amdgcn_readlane(running_sum(n[0]), 63);
        t.large += __popcll(__builtin_amdgcn_ballot_w64(n[1] != 0));
        t.small += __popcll(__builtin_amdgcn_ballot_w64(n[2] != 0));
    }
    // (the launch's bound, whatever the offsets are)
    const int most = p.n_pairs / 256 + p.E;
    t.full = min(t.full, most);
    t.large = min(t.large, most - t.full);
    t.small = min(t.small, most - t.full - t.large);
    return t;
}
// expert, first place and end of row tile `tile`
__device__ __forceinline__ bool find_wide_tile(const MoeParams& p, const WideTiles& t, int tile, int& e, int& first, int& end) {
    const int lane = threadIdx.x & 63;
    const int kind = tile < t.full ? 0 : (tile < t.full + t.large ? 1 : 2);
    int before = kind == 0 ? 0 : (kind == 1 ? t.full : t.full + t.large);
    for (int e0 = 0; e0 < p.E; e0 += 64) {
        int o0 = t.o0, o1 = t.o1;
        if (e0 > 0) {
            const int mine = min(e0 + lane, p.E - 1);
            o0 = p.offsets[mine];
            o1 = p.offsets[mine + 1];
        }
        int n[3];
        wide_kinds(o0, o1, e0 + lane < p.E, n);
        const int mine = kind == 0 ? n[0] : (kind == 1 ? n[1] : n[2]), sum = running_sum(mine);
        const uint64_t m = __builtin_amdgcn_ballot_w64(tile < before + sum);
        if (m != 0) {
            const int at = __builtin_ctzll(m), start = __builtin_amdgcn_readlane(o0, at);
            e = e0 + at;
            first = start + 256 * (kind == 0 ? tile - before - __builtin_amdgcn_readlane(sum - mine, at) : __builtin_amdgcn_readlane(n[0], at));
            end = min(__builtin_amdgcn_readlane(o1, at), p.n_pairs);
            return first >= 0 && first < end;
        }
        before += __builtin_amdgcn_readlane(sum, 63);
    }
    return false;
}

// NF 4: 256 rows x 256 rows of w per tile (gate_up: 128 gates and the 128 ups of the same columns), four wavefronts of 128 x 128 on
// 32x32x16 MFMAs, k in steps of 64.  A byte that is brought into LDS feeds twice, a byte read from it 1.5 times the MFMAs it
// feeds in the 128 x 128 kernel, which is bound by the requests (a compute unit takes in about 40 bytes per cycle, that kernel
// wants 62 at the full MFMA rate).  One wavefront per SIMD hides nothing of another, so what comes next has to be on its way:
//   In the loop: LDS is a ring of five halves of a step (rows 0, w 0, rows 1, w 1, rows 2, ..), all 160 KB.  The fragments of a
//   step are in registers at three quarters of it; its two halves then make room for the next step but one's w and the one behind
//   its rows.  Their 16 requests per wavefront go out one behind every third MFMA, w first, and only w's have to land within
//   the next step.  The fragments of a quarter are read one in front of each of the first MFMAs of the quarter before.
// Results leave through the ring, each wavefront's through a part of its own: whole lines, and no barrier.
// NF 2: a quarter of such a tile, 128 x 128, in the same way.
// 32768 pairs, 16 equal experts, us for k 1024 / 2048 / 4096, two buffers that change hands at three quarters of a step before, the ring now:
// gate and up (1024 columns) 133 / 209 / 438 -> 135 / 210 / 403, down (2048 columns) 136 / 256 / 484 -> 128 / 232 / 418 (1.3 PFLOP/s).  With no
// request in the loop k 4096 takes 346 of them: that is the MFMAs at the clock they are held at.  (So the ring gives something to gate and up only for a
// long k; with unequal experts, k 2048, what they gain is the order of the tiles and the last round's quarters: 1.04 PFLOP/s, down with k 1024 0.83.)
// (One workgroup per compute unit that goes on to its next tile, its first steps requested in front of this one's results: all
// workgroups end their tiles at the same time then, and nobody's MFMAs run beside the stores; gate and up 254, down 236.)
__device__ __forceinline__ int wide_swz(int row) { return (((row >> 1) & 3) << 1) | ((row >> 3) & 1); }       // (banks repeat every 256 bytes)
constexpr int kWideHalf = 256 * 64 * 2, kWideRing = 5;
template <bool GATE_UP, int NF>
__device__ __forceinline__ void moe_wide_tile(const MoeParams& p, unsigned char* lds, int n0, int e, int first, int end) {
    constexpr int BM = 64 * NF, BK = 64, kLoads = 2 * NF;                          // requests of a wavefront per half
    constexpr int kCols = GATE_UP ? 16 * NF : 32 * NF;                             // output columns of a wavefront
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, r = lane & 31, kg = lane >> 5;
    const __bf16* a_base = (const __bf16*)p.a;
    const __bf16* w_base = (const __bf16*)p.w + (int64_t)e * (GATE_UP ? 2 : 1) * p.n * p.k;
    // a wavefront brings in a quarter of the rows of both operands, 8 rows per load
    uint32_t a_off[kLoads], w_off[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int row = 16 * NF * wave + 8 * j + (lane >> 3), piece = (lane & 7) ^ wide_swz(row);
        a_off[j] = (uint32_t)((left_row<GATE_UP>(p, min(first + row, end - 1)) * p.a_stride + piece * 8) * 2);
        const int64_t wr = GATE_UP ? (row < BM / 2 ? min(n0 + row, p.n - 1) : p.n + min(n0 + row - BM / 2, p.n - 1)) : min(n0 + row, p.n - 1);
        w_off[j] = (uint32_t)((wr * p.k + piece * 8) * 2);
    }
    const uint32_t lds0 = lds_address(lds) + 16 * NF * wave * 128;
    const auto issue_w = [&](int step, int slot, int j) { dma_to_lds_16(w_base + step * BK, w_off[j], lds0 + slot * kWideHalf + 8 * j * 128); };
    const auto issue_a = [&](int step, int slot, int j) { dma_to_lds_16(a_base + step * BK, a_off[j], lds0 + slot * kWideHalf + 8 * j * 128); };
    const int n_steps = p.k / BK;
    // down: the pairs whose results this wavefront writes (row 32 j + r of its 32 NF) and their weights, asked for in front of the loop
    int pair[GATE_UP ? 1 : NF];
    float wgt[GATE_UP ? 1 : NF];
    if constexpr (!GATE_UP)
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            pair[j] = min(max(p.order[min(first + 32 * (NF * wm + j) + r, end - 1)], 0), p.n_pairs - 1);
            wgt[j] = p.weights[pair[j]];
        }
    // rows 0, w 0, rows 1, w 1, rows 2, what there is of them
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue_a(0, 0, j);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue_w(0, 1, j);
    if (n_steps > 1) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue_a(1, 2, j);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue_w(1, 3, j);
        if (n_steps > 2) {
#pragma unroll
            for (int j = 0; j < kLoads; ++j) issue_a(2, 4, j);
            wait_vmcnt<3 * kLoads>();
        } else {
            wait_vmcnt<2 * kLoads>();
        }
    } else {
        wait_vmcnt<0>();
    }
    __syncthreads();

    f32x16 acc[NF][NF];                           // [32 rows of w][32 rows]
    // 32-row groups of w of this wavefront: gate_up: half of them gates, then the ups of these columns
    const auto w_group = [&](int i) { return GATE_UP ? i / (NF / 2) * (BM / 2) + 16 * NF * wn + i % (NF / 2) * 32 : 32 * NF * wn + 32 * i; };
    bf16x8 wf[2][NF], af[2][NF];
    // One fragment of quarter s of a step in slots sa, sw: first the weights', then the rows'
    const auto fetch1 = [&](int sa, int sw, int s, int f) {
        const int piece = ((2 * s + kg) ^ wide_swz(r)) * 16;
        if (f < NF) wf[s & 1][f] = as_bf16x8(*reinterpret_cast<const u32x4*>(lds + sw * kWideHalf + (w_group(f) + r) * 128 + piece));
        else af[s & 1][f - NF] = as_bf16x8(*reinterpret_cast<const u32x4*>(lds + sa * kWideHalf + (32 * NF * wm + 32 * (f - NF) + r) * 128 + piece));
    };
    const auto ring = [](int slot, int by) { return slot + by >= kWideRing ? slot + by - kWideRing : slot + by; };
    // The MFMAs of quarter s, the fragments of quarter fs (of the step in slots fa, fw; -1: none) in front of the first of them.  turn: which
    // quarter behind the change of slots this is; the requests of w of step t_w and rows of step t_w + 1 are dealt out over the four.
    const auto quarter = [&](int s, int fs, int fa, int fw, int turn, int t_w, int to_w, int to_a, bool w_ahead, bool a_ahead) {
        constexpr int kEvery = NF == 4 ? 3 : 1;
#pragma unroll
        for (int m = 0; m < NF * NF; ++m) {
            if (fs >= 0)
#pragma unroll
                for (int f = m * 8 / (2 * NF); f < 2 * NF && f < (m + 1) * 8 / (2 * NF); ++f) fetch1(fa, fw, fs, f);
            acc[m % NF][m / NF] = mfma32(wf[s & 1][m % NF], af[s & 1][m / NF], acc[m % NF][m / NF]);
            const int at = turn * NF * NF + m;
            if (at % kEvery == kEvery - 1) {
                const int j = at / kEvery;
                if (j < kLoads) {
                    if (w_ahead) issue_w(t_w, to_w, j);
                } else if (j < 2 * kLoads) {
                    if (a_ahead) issue_a(t_w + 1, to_a, j - kLoads);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int sa = 0;                                   // step t is in slots sa and sa + 1
#pragma unroll
    for (int f = 0; f < 2 * NF; ++f) fetch1(0, 1, 0, f);
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < NF; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    // three quarters of step t, with the rest of the requests that the change of slots in front of it began: w of step t + 1 and rows of
    // step t + 2 into the slots of step t - 1
    const auto head = [&](int t, bool w_ahead, bool a_ahead) {
        const int sw = ring(sa, 1), to_w = ring(sa, 3), to_a = ring(sa, 4);
        quarter(0, 1, sa, sw, 1, t + 1, to_w, to_a, w_ahead, a_ahead);
        quarter(1, 2, sa, sw, 2, t + 1, to_w, to_a, w_ahead, a_ahead);
        quarter(2, 3, sa, sw, 3, t + 1, to_w, to_a, w_ahead, a_ahead);
    };
    // the change of slots and the last quarter of step t: w of t + 2 and rows of t + 3 follow if there are such
    const auto tail = [&](int t, auto rows_fly, bool w_ahead, bool a_ahead) {
        wait_lgkmcnt0();                          // the last fragments of this step are in registers,
        wait_vmcnt<decltype(rows_fly)::value ? kLoads : 0>();          // the next step has landed (the rows of the one behind it need not)
        __syncthreads();
        quarter(3, 0, ring(sa, 2), ring(sa, 3), 0, t + 2, sa, ring(sa, 1), w_ahead, a_ahead);
        sa = ring(sa, 2);
    };
    constexpr std::integral_constant<bool, true> yes{};
    constexpr std::integral_constant<bool, false> no{};
    int t = 0;
    if (n_steps > 1) {
        head(t, false, false);                    // (its requests are out)
        for (; t + 3 < n_steps; ++t) {
            tail(t, yes, true, true);
            head(t + 1, true, true);
        }
        if (t + 2 < n_steps) {
            tail(t, yes, true, false);
            head(t + 1, true, false);
            ++t;
        }
        tail(t, no, false, false);
    }
    head(t, false, false);
    quarter(3, -1, 0, 0, 0, 0, 0, 0, false, false);
    __syncthreads();                              // everybody has read the ring
    // lane: row 32 j + r of the wavefront's, columns 8 g + 4 kg + q of a 32-column group
    constexpr int kPieces = kCols / 8, kAtOnce = 64 / kPieces;
    static_assert(32 * kCols * 2 <= 16 * NF * 128, "32 rows of results");
    unsigned char* stage = lds + 16 * NF * wave * 128;
    const int piece = lane % kPieces, c0 = n0 + kCols * wn, row0 = first + 32 * NF * wm;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
#pragma unroll
        for (int i = 0; i < (GATE_UP ? NF / 2 : NF); ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (GATE_UP) v[q] = silu_fast(acc[i][j][4 * g + q]) * acc[i + NF / 2][j][4 * g + q];
                    else v[q] = wgt[j] * acc[i][j][4 * g + q];
                }
                *reinterpret_cast<u32x2*>(stage + (r * kPieces + ((4 * i + g) ^ (r & (kPieces - 1)))) * 16 + 8 * kg) =
                    u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            }
#pragma unroll
        for (int i = 0; i < 32 / kAtOnce; ++i) {
            const int row = i * kAtOnce + lane / kPieces, col = c0 + 8 * piece;
            const u32x4 v = *reinterpret_cast<const u32x4*>(stage + (row * kPieces + (piece ^ (row & (kPieces - 1)))) * 16);
            int64_t to = row0 + 32 * j + row;
            const bool there = to < end && col < p.n;
            if constexpr (!GATE_UP) to = __shfl(pair[j], row, 64);
            if (!there) continue;
            __bf16* o = (__bf16*)p.out + to * p.out_stride + col;
            if (col + 8 <= p.n) {
                *reinterpret_cast<u32x4*>(o) = v;
            } else {
                const bf16x8 b = as_bf16x8(v);
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (col + q < p.n) o[q] = b[q];
            }
        }
    }
}
// Whole rounds of the chip's 256 compute units go tile by tile; what is left goes in quarters where these are one round, half as long as a
// round of tiles.  Experts' last tiles come last, those with less than half their rows at the very end, so what is left mostly has two quarters.
template <bool GATE_UP>
__global__ __launch_bounds__(256, 1) void moe_wide_kernel(MoeParams p, int n_tiles, int chunk) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kWideRing * kWideHalf];
    constexpr int kCols = GATE_UP ? 128 : 256;
    const WideTiles kinds = wide_tiles(p);
    const int total = (kinds.full + kinds.large + kinds.small) * n_tiles;
    const int left = total % 256, whole = 4 * left - 2 * min(left, kinds.small * n_tiles) <= 256 ? total - left : total;
    int job = blockIdx.x, e, first, end;
    const auto tile = [&](int id, int& n_tile) {
        const int row_tile = id / n_tiles;
        n_tile = id - row_tile * n_tiles;
        return find_wide_tile(p, kinds, row_tile, e, first, end);
    };
    int n_tile;
    if (job < whole) {
        if (!tile(__builtin_amdgcn_readfirstlane(xcd_even_id(job, whole, chunk)), n_tile)) return;
        moe_wide_tile<GATE_UP, 4>(p, lds, n_tile * kCols, e, first, min(end, first + 256));
        return;
    }
    job -= whole;
    if (whole == total || job >= 4 * left) return;
    const int lower = job >= 2 * left, id = __builtin_amdgcn_readfirstlane(xcd_even_id(job - 2 * left * lower, 2 * left, 2 * chunk));
    if (!tile(whole + id / 2, n_tile)) return;
    const int n0 = n_tile * kCols + id % 2 * (kCols / 2);
    first += 128 * lower;
    end = min(end, first + 128);
    if (first < end && n0 < p.n) moe_wide_tile<GATE_UP, 2>(p, lds, n0, e, first, end);
}

// 16 rows x 16 rows of w (gate_up: 16 gates and their 16 ups).  The four wavefronts take the 64-wide steps of k in turn, read
// their operands straight from memory and meet in LDS.
template <bool GATE_UP>
__global__ __launch_bounds__(256) void moe_skinny_kernel(MoeParams p, int n_tiles, int m_tiles) {
    constexpr int BM = 16, NW = GATE_UP ? 2 : 1, kBatch = 4;        // steps of k whose loads are in flight together
    __shared__ f32x4 part[4][NW][64];
    const int id = xcd_chunked_id(blockIdx.x, n_tiles * m_tiles, n_tiles);
    const int n0 = id % n_tiles * 16;
    int e, first, end;
    if (!find_tile<BM>(p, id / n_tiles, e, first, end)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const __bf16* a = (const __bf16*)p.a + left_row<GATE_UP>(p, min(first + r, end - 1)) * p.a_stride + 8 * kg;
    const __bf16* w = (const __bf16*)p.w + ((int64_t)e * NW * p.n + min(n0 + r, p.n - 1)) * p.k + 8 * kg;
    const int64_t up = (int64_t)p.n * p.k;
    f32x4 acc[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 64 * wave; k0 < p.k; k0 += 256 * kBatch) {
        u32x4 av[kBatch][2], wv[NW][kBatch][2];
#pragma unroll
        for (int t = 0; t < kBatch; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int col = k0 + 256 * t + 32 * s;
                av[t][s] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < NW; ++i) wv[i][t][s] = av[t][s];
                if (k0 + 256 * t < p.k) {
#pragma unroll
                    for (int i = 0; i < NW; ++i) wv[i][t][s] = *reinterpret_cast<const u32x4*>(w + i * up + col);
                    av[t][s] = *reinterpret_cast<const u32x4*>(a + col);
                }
            }
#pragma unroll
        for (int t = 0; t < kBatch; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < NW; ++i) acc[i] = mfma16(as_bf16x8(wv[i][t][s]), as_bf16x8(av[t][s]), acc[i]);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) part[wave][i][lane] = acc[i];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int w4 = 1; w4 < 4; ++w4) acc[i] += part[w4][i][lane];
    const int place = first + r;
    if (place >= end) return;
    float v[4];
    if constexpr (GATE_UP) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = silu_fast(acc[0][q]) * acc[1][q];
        store4(p, place, n0 + 4 * kg, v);
    } else {
        const int pair = min(max(p.order[place], 0), p.n_pairs - 1);
        const float wgt = p.weights[pair];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = wgt * acc[0][q];
        store4(p, pair, n0 + 4 * kg, v);
    }
}

// The same product for the few pairs of a decode step, without an order: a workgroup per expert and 32 rows of w (gate_up: 16
// gates and their ups) looks through the ids for its expert's pairs itself, and row `pair` of the left and the output matrix
// belongs to the pair.  The weights are read once for every 32 rows.  What it saves against group + skinny: a launch, and the
// chain of dependent loads offsets -> order -> rows in front of the first weight.  Bound by the weights' stream (16 experts of
// 2048 x 1024, 32 tokens: 134 + 67 MB in 39.5 us, 5.1 TB/s, 44 where all workgroups began with the same step of k, see turn_of; group + skinny took 58).
// FEW (fewer pairs than experts, up to a wavefront's lanes): workgroups per pair instead, of which those of an expert's first one go on.  Experts without pairs, most of
// them then, have no workgroups that hold LDS while they find out, and one load tells a wavefront all it has to know.  Us of both products, workgroups per expert /
// like this: 32 experts of 2048 x 1024, top 2, one token 13.9 / 10.1, 6 tokens 25.4 / 23.2, 15 tokens 45.2 / 42.8; 32 of 1024 x 512, top 2, 1 token 9.6 / 7.6; 8 of
// 2048 x 1024, 7 tokens 19.5 / 19.1; 16 of 512 x 256, top 2, 4 tokens 7.8 / 7.0.  (Eight wavefronts with 18 KB each, one workgroup per compute unit: 10.2, 30.0, 51.6.)
constexpr int kDirectPairs = 2048, kFewPairs = 64;
constexpr int kDirectRing = 18 * 1024;            // three steps of 32 + 16 rows, two of 32 + 32; two workgroups per compute unit
template <bool GATE_UP, int RING, bool TURN, bool FEW>
__global__ __launch_bounds__(256) void moe_direct_kernel(MoeParams p, const int32_t* ids, int n_tiles) {
    constexpr int NW = GATE_UP ? 2 : 1;
    __shared__ __attribute__((aligned(1024))) unsigned char ring[4 * RING];
    __shared__ uint16_t mine[FEW ? kFewPairs : kDirectPairs];
    __shared__ int counts[4];
    // (an expert's tiles go round the XCDs: a step of one token uses few experts)
    const int n0 = blockIdx.x % n_tiles * (GATE_UP ? 16 : 32);
    int e = blockIdx.x / n_tiles;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    uint64_t of_expert = 0;
    if constexpr (FEW) {                          // workgroups of pair e: for its expert, if no pair in front has the same
        const int id = lane < p.n_pairs ? ids[lane] : -1, pair = e;
        e = __builtin_amdgcn_readlane(id, pair);
        of_expert = __builtin_amdgcn_ballot_w64(id == e);
        if ((unsigned)e >= (unsigned)p.E || (of_expert & ((1ull << pair) - 1)) != 0) return;
    }
    const __bf16* w_base = (const __bf16*)p.w + (int64_t)e * (GATE_UP ? 2 : 1) * p.n * p.k;
    const int piece = (lane & 7) ^ (lane >> 3);   // what a lane requests of its row's 128 bytes: see weight_stream
    uint32_t w_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 8 * j + (lane >> 3);
        const int64_t wr = GATE_UP ? (row < 16 ? min(n0 + row, p.n - 1) : p.n + min(n0 + row - 16, p.n - 1)) : min(n0 + row, p.n - 1);
        w_off[j] = (uint32_t)((wr * p.k + piece * 8) * 2);
    }
    // The first weights are requested in front of the look through the ids, from two pairs an expert on: with fewer, workgroups whose expert has
    // none would read weights for nothing (one in seven at two).  Us of router, experts and norm, without / with: 16 experts of 2048 x 1024, top
    // 4, 8 tokens 51.2 / 49.9, 16 57.4 / 55.7, 32 59.8 / 58.0; at 16 pairs an expert, where most take two row tiles and one step
    // at a time, 73.9 / 74.1.
    const int turn = TURN ? turn_of(p.k, 4, e * n_tiles + (int)(blockIdx.x % n_tiles)) : 0;     // (an expert's columns: whichever pairs it has)
    const bool ahead = !FEW && p.n_pairs >= 2 * p.E && p.n_pairs < 16 * p.E;
    int n_rows = 0;
    if constexpr (FEW) {
        n_rows = __popcll(of_expert);
        if (wave == 0 && (of_expert >> lane & 1)) mine[__popcll(of_expert & ((1ull << lane) - 1))] = (uint16_t)lane;
    } else {
        if (ahead) first_weights(w_base, w_off, p.k, wave, ring + wave * RING, turn);
        // wavefront w looks through pairs 64 (w + 4 i) + lane, kLook of them at a time
        constexpr int kLook = kDirectPairs / 256;
        uint64_t hit[kLook];
        int found = 0;
#pragma unroll
        for (int i = 0; i < kLook; ++i) {
            const int pair = 64 * (wave + 4 * i) + lane;
            hit[i] = 0;
            if (64 * (wave + 4 * i) < p.n_pairs) hit[i] = __builtin_amdgcn_ballot_w64(pair < p.n_pairs && ids[min(pair, p.n_pairs - 1)] == e);
            found += __popcll(hit[i]);
        }
        if (lane == 0) counts[wave] = found;
        __syncthreads();
        int at = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            at += w < wave ? counts[w] : 0;
            n_rows += counts[w];
        }
        if (n_rows == 0) {
            wait_vmcnt<0>();                          // (nothing lands in LDS that is somebody else's by then)
            return;
        }
#pragma unroll
        for (int i = 0; i < kLook; ++i) {
            if (hit[i] >> lane & 1) mine[at + __popcll(hit[i] & ((1ull << lane) - 1))] = (uint16_t)(64 * (wave + 4 * i) + lane);
            at += __popcll(hit[i]);
        }
    }
    __syncthreads();
    const auto rows = [&](int r0, auto tiles) {
        constexpr int MT = decltype(tiles)::value;
        uint32_t a_off[2 * MT];
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) {
            const int pair = mine[min(r0 + 8 * j + (lane >> 3), n_rows - 1)];
            a_off[j] = (uint32_t)(((int64_t)(GATE_UP ? pair / p.top : pair) * p.a_stride + piece * 8) * 2);
        }
        f32x4 acc[MT][2];
        weight_stream<MT, 4, RING, TURN>(w_base, w_off, p.a, a_off, p.k, turn, wave, ring + wave * RING, acc, [] {}, [](int, int, int, bf16x8&) {}, ahead && r0 == 0);
        __syncthreads();                          // (the sums travel through the ring)
        f32x4* part = reinterpret_cast<f32x4*>(ring);                           // [wave][row tile][16 rows of w][lane]
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 2; ++i) part[((wave * MT + m) * 2 + i) * 64 + lane] = acc[m][i];
        __syncthreads();
        // a wavefront sums one row tile (gate_up), or one row tile and 16 columns (down)
        if (wave < (GATE_UP ? MT : 2 * MT)) {
            const int m = GATE_UP ? wave : wave >> 1, half = GATE_UP ? 0 : wave & 1;
            f32x4 sum[NW];
#pragma unroll
            for (int i = 0; i < NW; ++i) {
                sum[i] = part[(m * 2 + half + i) * 64 + lane];
#pragma unroll
                for (int w4 = 1; w4 < 4; ++w4) sum[i] += part[((w4 * MT + m) * 2 + half + i) * 64 + lane];
            }
            if (r0 + 16 * m + r < n_rows) {
                const int pair = mine[r0 + 16 * m + r];
                const float wgt = GATE_UP ? 1.f : p.weights[pair];
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (GATE_UP) v[q] = silu_fast(sum[0][q]) * sum[NW - 1][q];
                    else v[q] = wgt * sum[0][q];
                }
                store4(p, pair, n0 + 16 * half + 4 * kg, v);
            }
        }
        __syncthreads();
    };
    for (int r0 = 0; r0 < n_rows; r0 += 32) {
        if (n_rows - r0 <= 16) rows(r0, std::integral_constant<int, 1>{});
        else rows(r0, std::integral_constant<int, 2>{});
    }
}

// From twelve pairs an expert on most experts take two row tiles, of which the small ring holds one step: with the large one 8 experts of 2048 x 2048, top 2, 64 tokens
// 46.5 -> 41.1 us, 16 of 2048 x 1024, top 4, 100 tokens 49.5 -> 45.8; below, three workgroups per compute unit are worth more (32 tokens 39.5 / 40.7), and so they are where a
// wavefront has four steps (16 of 1024 x 1024, top 4, 64 tokens 25.3 / 25.8).  (24 of 1536 x 768, top 4, 96 tokens 42, in tiles of 128 rows 50.)  With more workgroups than the
// two per compute unit that it leaves, from sixteen: up to fifteen pairs the third one is worth as much or more.  Pairs an expert, small / large ring: 10 of 1792 x 1792 12 39.9 / 43.4, 15 42.0 / 43.2, 16
// 46.0 / 44.9; 16 of 1792 x 896 15 35.0 / 36.3, 16 39.0 / 38.6; 16 of 2560 x 1280 12 60.4 / 62.1, 16 68.9 / 64.9; 4 of 2048 x 1024, 256 workgroups, 13 19.4 / 17.5.
template <bool GATE_UP>
static void launch_direct(const MoeParams& p, const int32_t* ids, hipStream_t s) {
    const int tiles = (p.n + (GATE_UP ? 15 : 31)) / (GATE_UP ? 16 : 32);
    const dim3 grid((unsigned)(tiles * p.E)), block(256);
    const bool large = p.k >= 1536 && p.n_pairs >= (grid.x <= 512 ? 12 : 16) * p.E, turn = turn_pays(p.k);
    if (p.n_pairs < p.E && p.n_pairs <= kFewPairs) {
        const dim3 few((unsigned)(tiles * p.n_pairs));
        if (turn) hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kStreamBytes, true, true>), few, block, 0, s, p, ids, tiles);
        else hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kStreamBytes, false, true>), few, block, 0, s, p, ids, tiles);
    } else if (large && turn) {
        hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kDirectRing, true, false>), grid, block, 0, s, p, ids, tiles);
    } else if (large) {
        hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kDirectRing, false, false>), grid, block, 0, s, p, ids, tiles);
    } else if (turn) {
        hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kStreamBytes, true, false>), grid, block, 0, s, p, ids, tiles);
    } else {
        hipLaunchKernelGGL((moe_direct_kernel<GATE_UP, kStreamBytes, false, false>), grid, block, 0, s, p, ids, tiles);
    }
}

// fp32: 16 rows x 64 columns per workgroup, a thread owns four rows of one column
template <bool GATE_UP>
__global__ __launch_bounds__(256) void moe_f32_kernel(MoeParams p, int n_tiles, int m_tiles) {
    constexpr int BM = 16, BK = 16, NW = GATE_UP ? 2 : 1;
    __shared__ float a_lds[BM][BK + 1], w_lds[NW][64][BK + 1];
    const int n0 = blockIdx.x % n_tiles * 64;
    int e, first, end;
    if (!find_tile<BM>(p, blockIdx.x / n_tiles, e, first, end)) return;
    const int tid = threadIdx.x, col = tid & 63, rows = (tid >> 6) * 4;
    const float* w = (const float*)p.w + (int64_t)e * NW * p.n * p.k;
    const int ar = tid / BK, ac = tid % BK;
    const float* a = (const float*)p.a + left_row<GATE_UP>(p, min(first + ar, end - 1)) * p.a_stride;
    float acc[NW][4];
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int k0 = 0; k0 < p.k; k0 += BK) {
        __syncthreads();
        a_lds[ar][ac] = k0 + ac < p.k ? a[k0 + ac] : 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t row = (int64_t)i * p.n + min(n0 + 16 * j + ar, p.n - 1);
                w_lds[i][16 * j + ar][ac] = k0 + ac < p.k ? w[row * p.k + k0 + ac] : 0.f;
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; ++k)
#pragma unroll
            for (int i = 0; i < NW; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(w_lds[i][col][k], a_lds[rows + j][k], acc[i][j]);
    }
    if (n0 + col >= p.n) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int place = first + rows + j;
        if (place >= end) continue;
        float v;
        int64_t row = place;
        if constexpr (GATE_UP) {
            v = acc[0][j] / (1.0f + expf(-acc[0][j])) * acc[1][j];
        } else {
            row = min(max(p.order[place], 0), p.n_pairs - 1);
            v = p.weights[row] * acc[0][j];
        }
        ((float*)p.out)[row * p.out_stride + n0 + col] = v;
    }
}

// The 256 x 256 tiles are faster where they fill the chip's rounds: a round of them counts 1, their last one a half where it goes in
// quarters, and a round of 128 x 128 tiles, two per compute unit, 0.69.  Us of both products, with these tiles and with 128 x 128 ones:
// 16 experts of 2048 x 1024, top 4, 700 tokens 70 / 56, 1356 96 / 95, 2048 119 / 136, 2600 157 / 161, 4096 207 / 260, 8192 386 / 499; 8 of
// 1024 x 512, top 2, 2263 tokens 50 / 37, 7536 (top 1) 53 / 42; 16 of 1024 x 512, top 4, 6313 102 / 112; 32 of 2048 x 1024, top 4, 5059
// 297 / 355; 8 of 512 x 256, top 2, 4096 36 / 26.  Below 256 pairs an expert most of a tile is padding.
static bool wide_pays(const MoeParams& p, bool gate_up) {
    const double n_tiles = (p.n + (gate_up ? 127 : 255)) / (gate_up ? 128 : 256);
    const double tiles = (p.n_pairs / 256.0 + 0.5 * p.E) * n_tiles, whole = std::floor(tiles / 256.0), left = tiles - 256.0 * whole;
    const double quarters = 4.0 * left - 2.0 * std::min(left, 0.5 * p.E * n_tiles);
    const double wide = whole + (quarters <= 256.0 ? 0.5 : 1.0), large = 0.69 * std::max(1.0, (p.n_pairs / 128.0 + 0.5 * p.E) * 2.0 * n_tiles / 512.0);
    return p.k >= 512 && p.n_pairs >= 256LL * p.E && wide <= large;
}

template <bool GATE_UP>
static int launch_moe(const MoeParams& p, int dtype, int tiling, hipStream_t s) {
    // From 8 pairs per expert on the large tiles, mostly padding then, still read the weights faster (2048 x 1024, 16 experts, both
    // products: 8 pairs 44 us against 55, 32 pairs 49 against 109)
    const bool large = tiling >= MI355_TILING_LARGE || (tiling == MI355_TILING_AUTO && p.n_pairs > 8 * (int64_t)p.E);
    const bool fits = p.out_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    const bool wide = dtype == MI355_BF16 && fits && (tiling == MI355_TILING_WIDE || (tiling == MI355_TILING_AUTO && large && wide_pays(p, GATE_UP)));
    const int bm = dtype == MI355_BF16 && large ? (wide ? 256 : 128) : 16;
    const int bn = dtype == MI355_FP32 ? 64 : (!large ? 16 : (GATE_UP ? 64 : 128) * (wide ? 2 : 1));
    const int n_tiles = (p.n + bn - 1) / bn, m_tiles = p.n_pairs / bm + p.E;
    if ((int64_t)n_tiles * m_tiles > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)(n_tiles * m_tiles)), block(256);
    // An XCD takes as many neighbouring row tiles in turn as fill its 32 compute units twice: they mostly belong to one expert
    // and share its weights in that L2.  (One row tile per turn, so that eight XCDs read eight tiles of one expert: 2048
    // tokens, 16 experts of 2048 x 1024, top 4 176 us for both products, 146 us like this; 8192 tokens 518 against 511.)
    const int chunk = n_tiles * std::max(1, (wide ? 32 : 64) / n_tiles);
    if (dtype == MI355_FP32) hipLaunchKernelGGL(moe_f32_kernel<GATE_UP>, grid, block, 0, s, p, n_tiles, m_tiles);
    else if (wide) hipLaunchKernelGGL(moe_wide_kernel<GATE_UP>, dim3((unsigned)(n_tiles * m_tiles + 384)), block, 0, s, p, n_tiles, chunk);
    else if (large && turn_pays(p.k) && p.n_pairs <= (p.k == 2048 ? 256LL : 96LL) * p.E) hipLaunchKernelGGL((moe_gemm_kernel<GATE_UP, true>), grid, block, 0, s, p, n_tiles, chunk);
    else if (large) hipLaunchKernelGGL((moe_gemm_kernel<GATE_UP, false>), grid, block, 0, s, p, n_tiles, chunk);
    else hipLaunchKernelGGL(moe_skinny_kernel<GATE_UP>, grid, block, 0, s, p, n_tiles, m_tiles);
    return (int)hipGetLastError();
}

static int moe_check(MoeParams& p, bool gate_up, const void* a, const void* w, void* out, const int32_t* offsets, const int32_t* order,
                     const float* weights, int64_t a_stride, int64_t a_rows, int64_t out_stride, int64_t out_rows, int64_t n_pairs,
                     int E, int top, int k, int n, int dtype, int tiling) {
    if (!a || !w || !out || !offsets || !order || (!gate_up && !weights)) return set_error(MI355_EINVAL, "moe: null pointer argument");
    if (dtype != MI355_BF16 && dtype != MI355_FP32) return set_error(MI355_EDTYPE, "moe: dtype must be MI355_BF16 or MI355_FP32");
    if (E <= 0 || E > kMaxExperts || top <= 0 || k <= 0 || n <= 0 || n_pairs < 0 || n_pairs > 0x3fffffffLL)
        return set_error(MI355_EINVAL, "moe: experts, top, k, n, n_pairs out of range");
    if (tiling < MI355_TILING_AUTO || tiling > MI355_TILING_WIDE) return set_error(MI355_EINVAL, "moe: unknown tiling");
    if (a_stride < k || out_stride < n) return set_error(MI355_EINVAL, "moe: row strides shorter than a row");
    if (a_rows < (gate_up ? (n_pairs + top - 1) / top : n_pairs) || out_rows < n_pairs) return set_error(MI355_EINVAL, "moe: too few rows");
    if (dtype == MI355_BF16) {
        if (k % 64 || a_stride % 8 || out_stride % 4 || (reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(w) & 15) ||
            (reinterpret_cast<uintptr_t>(out) & 7))
            return set_error(MI355_EINVAL, "moe: bf16 operands need k in multiples of 64 and 16-byte aligned rows");
        if (a_rows * a_stride > 0x7fffffffLL || 2LL * n * k > 0x7fffffffLL)
            return set_error(MI355_EINVAL, "moe: an operand is too large for 32-bit byte offsets");
    }
    p.a = a;
    p.w = w;
    p.out = out;
    p.offsets = offsets;
    p.order = order;
    p.weights = weights;
    p.a_stride = a_stride;
    p.a_rows = a_rows;
    p.out_stride = out_stride;
    p.out_rows = out_rows;
    p.n_pairs = (int)n_pairs;
    p.E = E;
    p.k = k;
    p.n = n;
    p.top = top;
    return MI355_OK;
}

static int moe_product(bool gate_up, const void* a, const void* w, void* out, const int32_t* offsets, const int32_t* order,
                       const float* weights, int64_t a_stride, int64_t a_rows, int64_t out_stride, int64_t out_rows, int64_t n_pairs,
                       int E, int top, int k, int n, int dtype, int tiling, void* stream) {
    MoeParams p;
    if (int e = moe_check(p, gate_up, a, w, out, offsets, order, weights, a_stride, a_rows, out_stride, out_rows, n_pairs, E, top, k, n, dtype, tiling))
        return e;
    if (n_pairs == 0) return MI355_OK;
    const int rc = gate_up ? launch_moe<true>(p, dtype, tiling, (hipStream_t)stream) : launch_moe<false>(p, dtype, tiling, (hipStream_t)stream);
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_moe_route(const void* h, const void* w, const float* bias, int32_t* ids, float* weights, float* extra_logit,
                               int64_t n_tokens, int64_t h_row_stride, int64_t w_row_stride, int k, int n_experts, int top, int dtype,
                               void* stream) {
    if (!h || !w || !bias || !ids || !weights) return set_error(MI355_EINVAL, "moe_route: null pointer argument");
    if (dtype != MI355_BF16 && dtype != MI355_FP32) return set_error(MI355_EDTYPE, "moe_route: dtype must be MI355_BF16 or MI355_FP32");
    if (n_tokens < 0 || k <= 0 || n_experts <= 0 || n_experts > kMaxExperts || top <= 0 || top > n_experts || top > kMaxTop)
        return set_error(MI355_EINVAL, "moe_route: n_tokens, k, n_experts (up to 1024), top (up to 64) out of range");
    if (h_row_stride < k || w_row_stride < k) return set_error(MI355_EINVAL, "moe_route: row strides shorter than a row");
    if (dtype == MI355_BF16 && (k % 8 || h_row_stride % 8 || w_row_stride % 8 || (reinterpret_cast<uintptr_t>(h) & 15) ||
                                (reinterpret_cast<uintptr_t>(w) & 15)))
        return set_error(MI355_EINVAL, "moe_route: bf16 rows must be 16-byte aligned and k a multiple of 8");
    if (n_tokens > 0x7fffff00LL) return set_error(MI355_EINVAL, "moe_route: too many tokens");
    if (n_tokens == 0) return MI355_OK;
    RouteParams p;
    p.h = h;
    p.w = w;
    p.bias = bias;
    p.ids = ids;
    p.weights = weights;
    p.extra_logit = extra_logit;
    p.T = n_tokens;
    p.h_stride = h_row_stride;
    p.w_stride = w_row_stride;
    p.k = k;
    p.E = n_experts;
    p.n_logits = n_experts + (extra_logit ? 1 : 0);
    p.top = top;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == MI355_BF16)
        launch_route(p, s);
    else
        hipLaunchKernelGGL(moe_route_f32_kernel, dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 4 * p.n_logits * sizeof(float), s, p);
    const int rc = (int)hipGetLastError();
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

extern "C" int mi355_moe_group(const int32_t* ids, int64_t n_pairs, int n_experts, int32_t* offsets, int32_t* order, void* stream) {
    if (!ids || !offsets || !order) return set_error(MI355_EINVAL, "moe_group: null pointer argument");
    if (n_pairs < 0 || n_pairs > 0x3fffffffLL || n_experts <= 0 || n_experts > kMaxExperts)
        return set_error(MI355_EINVAL, "moe_group: n_pairs, n_experts (up to 1024) out of range");
    hipLaunchKernelGGL(moe_group_kernel, dim3((unsigned)n_experts), dim3(1024), 0, (hipStream_t)stream, ids, (int)n_pairs, n_experts, offsets, order);
    const int rc = (int)hipGetLastError();
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

extern "C" int mi355_moe_gate_up(const void* h, const void* w, void* act, const int32_t* offsets, const int32_t* order, int64_t n_tokens,
                                 int64_t h_row_stride, int64_t act_row_stride, int n_experts, int top, int k, int ff, int dtype,
                                 int tiling, void* stream) {
    return moe_product(true, h, w, act, offsets, order, nullptr, h_row_stride, n_tokens, act_row_stride, n_tokens * top,
                       n_tokens * top, n_experts, top, k, ff, dtype, tiling, stream);
}

extern "C" int mi355_moe_down(const void* act, const void* w, const float* weights, void* out, const int32_t* offsets, const int32_t* order,
                              int64_t n_tokens, int64_t act_row_stride, int64_t out_row_stride, int n_experts, int top, int ff, int n,
                              int dtype, int tiling, void* stream) {
    return moe_product(false, act, w, out, offsets, order, weights, act_row_stride, n_tokens * top, out_row_stride, n_tokens * top,
                       n_tokens * top, n_experts, top, ff, n, dtype, tiling, stream);
}

extern "C" int mi355_moe_direct(const void* h, const void* w_gate_up, const void* w_down, const int32_t* ids, const float* weights, void* act,
                                void* out, int64_t n_tokens, int64_t h_row_stride, int64_t out_row_stride, int n_experts, int top, int k,
                                int ff, int n, void* stream) {
    if (!ids) return set_error(MI355_EINVAL, "moe_direct: null pointer argument");
    if (n_tokens < 0 || top <= 0 || n_tokens > kDirectPairs || n_tokens * top > kDirectPairs) return set_error(MI355_EINVAL, "moe_direct: up to 2048 pairs");
    // (ids stands in for the order, which these kernels do not read; nothing is launched before both products' arguments are checked)
    MoeParams up, down;
    int rc = moe_check(up, true, h, w_gate_up, act, ids, ids, nullptr, h_row_stride, n_tokens, ff, n_tokens * top, n_tokens * top, n_experts, top,
                       k, ff, MI355_BF16, MI355_TILING_AUTO);
    if (rc == MI355_OK)
        rc = moe_check(down, false, act, w_down, out, ids, ids, weights, ff, n_tokens * top, out_row_stride, n_tokens * top, n_tokens * top,
                       n_experts, top, ff, n, MI355_BF16, MI355_TILING_AUTO);
    if (rc != MI355_OK || n_tokens == 0) return rc;
    hipStream_t s = (hipStream_t)stream;
    launch_direct<true>(up, ids, s);
    if ((rc = (int)hipGetLastError()) != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    launch_direct<false>(down, ids, s);
    if ((rc = (int)hipGetLastError()) != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}
