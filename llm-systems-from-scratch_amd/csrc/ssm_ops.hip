// Mamba-2 mixers (state-space duality) on gfx950: short causal convolution, selective state recurrence, decode step.
//
// Per head, with log decay a_t = neg_a dt_t (dt after softplus) and channels x | B | C behind a causal convolution and silu:
//     S_t = exp(a_t) S_(t-1) + dt_t B_t x_t^T        y_t = S_t^T C_t + D x_t             S: state x vdim, fp32
//
// What a sequence carries from one call to the next lives in slots of two pools:
//   conv_state (slots, taps, channels)            the convolution's inputs as a ring: position p sits in row p % taps.  A
//                                                 convolution reads the taps - 1 rows in front of a token and writes the
//                                                 token's own row, so a step's reads and writes never meet.
//   ssm_state  (slots, heads, state, vdim_pad)    S in fp32 (vdim_pad: vdim rounded up to 4)
// A sequence's first token is at position 0: its history is zero whatever the slot holds, so slots are never cleared.
//
// Kernels besides the convolution:
//   ssd_chunk_kernel   bf16 prompts: chunks of 64 tokens on MFMA, the state in accumulators from chunk to chunk; where
//                      that walk leaves the chip idle, segments of a sequence side by side (ssd_carry_kernel between them)
//   ssd_walk_kernel    the same in chunks of 128, outputs and state on different wavefronts: states of 64 or 128 rows
//   ssm_scan_kernel    any sizes and fp32: token by token, the state in registers
//   ... the same kernel with the convolution inside: one decode step of every sequence
#include "common.hpp"
#include "launch.hpp"
#include "prefill_tile.hpp"
#include "ssm_conv.hpp"

#include <type_traits>

namespace mi355 {

constexpr int kScanVecs = 16;        // most 4-wide state pieces per thread of the scan

template <typename T>
struct SsmParams {
    const T* proj;                   // rows of the input projection
    int64_t proj_stride, xbc_at, dt_at;
    const float *conv_w, *conv_b;    // (taps, channels), (channels)
    const float *dt_bias, *neg_a, *d_skip;
    T* conv_state;
    float* ssm_state;
    const int32_t *slots, *positions, *cu;      // cu null: sequence b owns row b
    T* xbc;                          // (rows, channels): the convolution's output
    T* y;
    int64_t y_stride, n_rows;
    int B, H, P, Pp, N, G, taps, channels, n_slots;
    int np4, slices;                 // scan: 4-wide pieces of vdim per workgroup, and workgroups per head
    float *seg_state, *seg_decay;    // segments: (segment, head) states (N x Pp), log2 of the decay across a segment
    int seg_len, n_segs, whole_len;  // whole_len: sequences of up to so many tokens are one segment
};

template <typename T>
__device__ __forceinline__ int state_slot(const SsmParams<T>& p, int b) {
    return min(max(p.slots[b], 0), p.n_slots - 1);
}
// the sequence that unit `unit` of `size` tokens lies in: units of sequence b start at number first_row / size + b
template <typename T>
__device__ __forceinline__ int seq_of_unit(const SsmParams<T>& p, int unit, int size) {
    int lo = 0, hi = p.B - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if ((p.cu ? p.cu[mid] : mid) / size + mid <= unit) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
// rows of sequence b
template <typename T>
__device__ __forceinline__ void seq_rows(const SsmParams<T>& p, int b, int& first, int& len) {
    first = p.cu ? p.cu[b] : b;
    len = (p.cu ? p.cu[b + 1] : b + 1) - first;
    len = max(0, min(len, (int)p.n_rows - first));
}
__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
template <bool FAST>
__device__ __forceinline__ float silu_of(float x) {
    if constexpr (FAST) return x * __builtin_amdgcn_rcpf(1.0f + fast_exp2(-kLog2e * x));
    else return x / (1.0f + expf(-x));
}

// V adjacent channels (8: 16-byte pieces of bf16, 32-byte pieces of fp32; or 1)
template <typename T, int V>
__device__ __forceinline__ void load_ch(const T* p, float (&v)[V]) {
    if constexpr (V == 1) {
        v[0] = (float)p[0];
    } else if constexpr (sizeof(T) == 2) {
        const bf16x8 a = as_bf16x8(*reinterpret_cast<const u32x4*>(p));
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)a[e];
    } else {
        const f32x4 a = reinterpret_cast<const f32x4*>(p)[0], b = reinterpret_cast<const f32x4*>(p)[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    }
}
template <typename T, int V>
__device__ __forceinline__ void store_ch(T* p, const float (&v)[V]) {
    if constexpr (V == 1) {
        p[0] = (T)v[0];
    } else if constexpr (sizeof(T) == 2) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = pack_bf16(v[2 * e], v[2 * e + 1]);
        *reinterpret_cast<u32x4*>(p) = o;
    } else {
        reinterpret_cast<f32x4*>(p)[0] = f32x4{v[0], v[1], v[2], v[3]};
        reinterpret_cast<f32x4*>(p)[1] = f32x4{v[4], v[5], v[6], v[7]};
    }
}

// Causal convolution + silu of packed prompts.  A thread owns V adjacent channels of TILE tokens of one sequence; the inputs it has read
// slide through registers when the number of taps is known at compile time (TAPS > 0).  The thread of a sequence's first tile is the only
// one that touches the sequence's ring for its channels: it reads the history first and writes the last taps - 1 inputs of the portion at its end.
// (So a tile has at least taps - 1 tokens: conv_tile.)
//
// Bound by its bytes where a call is large (8192 tokens, 4352 channels: 142 MB in 26 us) and by one load's latency where it is small, so all rows of a tile of 4 or 8
// tokens, and those that go to the ring, are requested before the first is used: a load in front of every token's sum took 11 to 13 us for 600 to 1700 tokens,
// 4 tokens per thread take 7.  Tiles of 4 read 7 rows for 4, tiles of 16 19 for 16.  In those, whose calls have wavefronts enough, loads stand where
// they are used: eight rows ahead hold registers that wavefronts would have.  us like this / eight ahead: 4000 tokens of 4352 channels 15.7 / 18.0, 64 x 100 26.4 / 29.6,
// 2 x 7000 49.2 / 52.1, 4 x 8000 of 1792 47.7 / 51.0.
template <typename T>
struct ChannelRow {                                      // eight adjacent channels as they are in memory
    static constexpr int kPieces = 8 * sizeof(T) / 16;
    u32x4 w[kPieces];
    __device__ __forceinline__ void load(const T* p) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) w[i] = reinterpret_cast<const u32x4*>(p)[i];
    }
    __device__ __forceinline__ void store(T* p) const {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) reinterpret_cast<u32x4*>(p)[i] = w[i];
    }
    __device__ __forceinline__ void get(float (&v)[8]) const {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t x = sizeof(T) == 2 ? w[e / 8][e / 2] : w[e / 4][e % 4];
            v[e] = __builtin_bit_cast(float, sizeof(T) == 2 ? (e % 2 ? x & 0xffff0000u : x << 16) : x);
        }
    }
};

template <typename T, int V, int TAPS, int TILE>
__global__ __launch_bounds__(256) void causal_conv_silu_kernel(SsmParams<T> p) {
    static_assert(TILE >= TAPS - 1, "only the first tile reads the ring");
    constexpr bool FAST = sizeof(T) == 2;
    const int taps = TAPS > 0 ? TAPS : p.taps;
    const int ch_groups = p.channels / V;
    const int g_blocks = (ch_groups + (int)blockDim.x - 1) / (int)blockDim.x;
    const int tile = blockIdx.x / g_blocks;
    const int cg = (blockIdx.x % g_blocks) * blockDim.x + threadIdx.x;
    const int b = seq_of_unit(p, tile, TILE);
    int first, len;
    seq_rows(p, b, first, len);
    const int t0 = (tile - (first / TILE + b)) * TILE;
    if (t0 < 0 || t0 >= len || cg >= ch_groups) return;
    const int c = cg * V;
    const int pos0 = p.positions[first];
    T* ring = p.conv_state + (int64_t)state_slot(p, b) * taps * p.channels + c;
    const T* in = p.proj + (int64_t)first * p.proj_stride + p.xbc_at + c;
    const auto input = [&](int t, float (&v)[V]) {              // token t of the portion, or (t < 0) one before it
        if (t >= 0) {
            load_ch<T, V>(in + (int64_t)t * p.proj_stride, v);
        } else if (pos0 + t >= 0) {
            load_ch<T, V>(ring + (int64_t)((pos0 + t) % taps) * p.channels, v);
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) v[e] = 0.f;
        }
    };
    float bias[V];
    const int n = min(TILE, len - t0);
    T* out = p.xbc + (int64_t)(first + t0) * p.channels + c;
    if constexpr (TAPS > 0) {
        static_assert(V == 8 && TAPS > 1, "rows in whole pieces");
        float w[TAPS][V], x[TAPS][V];
        const auto load_weights = [&]() {
            load_ch<float, V>(p.conv_b + c, bias);
#pragma unroll
            for (int j = 0; j < TAPS; ++j) load_ch<float, V>(p.conv_w + (int64_t)j * p.channels + c, w[j]);
        };
        const auto load_history = [&]() {
#pragma unroll
            for (int j = 0; j + 1 < TAPS; ++j) input(t0 - (TAPS - 1) + j, x[j]);
        };
        const auto emit = [&](int t) {                           // token t of the tile, whose own input is in x[TAPS - 1]
            float a[V];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                a[e] = bias[e];
#pragma unroll
                for (int j = 0; j < TAPS; ++j) a[e] = fmaf(w[j][e], x[j][e], a[e]);
                a[e] = silu_of<FAST>(a[e]);
            }
            if (t < n) store_ch<T, V>(out + (int64_t)t * p.channels, a);
#pragma unroll
            for (int j = 0; j + 1 < TAPS; ++j)
#pragma unroll
                for (int e = 0; e < V; ++e) x[j][e] = x[j + 1][e];
        };
        if constexpr (TILE < kMostConvTile) {
            ChannelRow<T> row[TILE], keep[TAPS - 1];
#pragma unroll
            for (int i = 0; i < TILE; ++i) row[i].load(in + (int64_t)(t0 + min(i, n - 1)) * p.proj_stride);       // (rows past the end: the last one again)
            load_history();
            if (t0 == 0)
#pragma unroll
                for (int j = 0; j + 1 < TAPS; ++j) keep[j].load(in + (int64_t)max(0, len - (TAPS - 1) + j) * p.proj_stride);
            load_weights();
#pragma unroll
            for (int i = 0; i < TILE; ++i) {
                row[i].get(x[TAPS - 1]);
                emit(i);
            }
            if (t0 == 0) {
#pragma unroll
                for (int j = 0; j + 1 < TAPS; ++j) {
                    const int t = len - (TAPS - 1) + j;
                    if (t >= 0) keep[j].store(ring + (int64_t)((pos0 + t) % TAPS) * p.channels);
                }
            }
            return;
        } else {
            load_weights();
            load_history();
#pragma unroll
            for (int t = 0; t < TILE; ++t) {
                if (t < n) {
                    load_ch<T, V>(in + (int64_t)(t0 + t) * p.proj_stride, x[TAPS - 1]);
                    emit(t);
                }
            }
        }
    } else {
        load_ch<float, V>(p.conv_b + c, bias);
        for (int t = 0; t < n; ++t) {
            float a[V];
#pragma unroll
            for (int e = 0; e < V; ++e) a[e] = bias[e];
            for (int j = 0; j < taps; ++j) {
                float w[V], x[V];
                load_ch<float, V>(p.conv_w + (int64_t)j * p.channels + c, w);
                input(t0 + t - (taps - 1) + j, x);
#pragma unroll
                for (int e = 0; e < V; ++e) a[e] = fmaf(w[e], x[e], a[e]);
            }
#pragma unroll
            for (int e = 0; e < V; ++e) a[e] = silu_of<FAST>(a[e]);
            store_ch<T, V>(out + (int64_t)t * p.channels, a);
        }
    }
    if (t0 == 0) {
        for (int t = max(0, len - (taps - 1)); t < len; ++t) {
            float x[V];
            load_ch<T, V>(in + (int64_t)t * p.proj_stride, x);
            store_ch<T, V>(ring + (int64_t)((pos0 + t) % taps) * p.channels, x);
        }
    }
}

// Token-by-token recurrence.  One workgroup per (sequence, head, slice of vdim); a thread owns a fixed 4-wide piece of vdim
// and every (256 / np4)-th row of the state, in registers.  DECODE: one token per sequence, the convolution of the head's
// channels inside (B and C channels, shared by the heads of a group, are convolved by each of them and entered into the ring by
// the group's first).
template <typename T, int NV, bool DECODE>
__global__ __launch_bounds__(256) void ssm_scan_kernel(SsmParams<T> p) {
    constexpr bool FAST = sizeof(T) == 2;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int np = 4 * p.np4;                                  // columns of the slice
    float* x_l = smem;                                         // np
    float* b_l = x_l + np;                                     // N
    float* c_l = b_l + p.N;                                    // N
    f32x4* red = reinterpret_cast<f32x4*>(smem + (np + 2 * p.N + 3) / 4 * 4);       // rows x np4
    const int slice = blockIdx.x % p.slices;
    const int h = (blockIdx.x / p.slices) % p.H;
    const int b = blockIdx.x / (p.slices * p.H);
    int first, len;
    seq_rows(p, b, first, len);
    if (len <= 0) return;
    const int per_group = p.H / p.G, g = h / per_group;
    const int col0 = slice * np;                               // first column of the slice
    const int tid = threadIdx.x, rows = 256 / p.np4;
    const int p4 = tid % p.np4, r = tid / p.np4;
    const bool mine = r < rows && col0 + 4 * p4 < p.Pp;
    const int slot = state_slot(p, b);
    float* st = p.ssm_state + ((int64_t)slot * p.H + h) * p.N * p.Pp + col0 + 4 * p4;
    const int pos0 = p.positions[first];
    f32x4 S[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int n = r + i * rows;
        if (mine && n < p.N && pos0 > 0) S[i] = *reinterpret_cast<const f32x4*>(st + (int64_t)n * p.Pp);
    }
    const float bias = p.dt_bias[h], na = p.neg_a[h], skip = p.d_skip[h];
    const int inner = p.H * p.P;
    // channel of staged value i: x columns of the slice, then B, then C
    const auto channel = [&](int i) {
        if (i < np) return col0 + i < p.P ? h * p.P + col0 + i : -1;
        return i < np + p.N ? inner + g * p.N + (i - np) : inner + (p.G + g) * p.N + (i - np - p.N);
    };
    for (int t = 0; t < len; ++t) {
        const int64_t row = first + t;
        if (t) __syncthreads();                                // the staged values of the token before have been read
        for (int i = tid; i < np + 2 * p.N; i += 256) {
            const int c = channel(i);
            float v = 0.f;
            if (c >= 0) {
                if constexpr (DECODE) {
                    T* ring = p.conv_state + (int64_t)slot * p.taps * p.channels + c;
                    const T now = p.proj[row * p.proj_stride + p.xbc_at + c];
                    v = p.conv_b[c];
                    for (int j = 0; j + 1 < p.taps; ++j) {
                        const int q = pos0 - (p.taps - 1) + j;
                        if (q >= 0) v = fmaf(p.conv_w[(int64_t)j * p.channels + c], (float)ring[(int64_t)(q % p.taps) * p.channels], v);
                    }
                    v = silu_of<FAST>(fmaf(p.conv_w[(int64_t)(p.taps - 1) * p.channels + c], (float)now, v));
                    if (i < np || (h % per_group == 0 && slice == 0)) ring[(int64_t)(pos0 % p.taps) * p.channels] = now;
                } else {
                    v = (float)p.xbc[row * p.channels + c];
                }
            }
            smem[i] = v;
        }
        const float dt = softplus((float)p.proj[row * p.proj_stride + p.dt_at + h] + bias);
        const float decay = FAST ? fast_exp2(kLog2e * (na * dt)) : expf(na * dt);
        __syncthreads();
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (mine) {
            f32x4 xd = *reinterpret_cast<const f32x4*>(x_l + 4 * p4);
            xd *= dt;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int n = r + i * rows;
                if (n < p.N) {
                    const float bn = b_l[n], cn = c_l[n];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        S[i][e] = fmaf(decay, S[i][e], bn * xd[e]);
                        acc[e] = fmaf(S[i][e], cn, acc[e]);
                    }
                }
            }
        }
        if (r < rows) red[r * p.np4 + p4] = acc;
        __syncthreads();
        for (int i = tid; i < np; i += 256) {
            if (col0 + i < p.P) {
                const float* rf = reinterpret_cast<const float*>(red);
                float s = skip * x_l[i];
                for (int k = 0; k < rows; ++k) s += rf[k * np + i];
                p.y[row * p.y_stride + h * p.P + col0 + i] = (T)s;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int n = r + i * rows;
        if (mine && n < p.N) *reinterpret_cast<f32x4*>(st + (int64_t)n * p.Pp) = S[i];
    }
}

// ---- segments of the chunked scan ----
// Segments are numbered without gaps, sequence by sequence, so that the workgroups that have one are a launch's first: one that has
// none still holds 66 KB of LDS while it finds out (32 sequences of 1000 tokens, 16 heads, two of three numbers without a segment
// 199 us, like this 133; 125 where the caller says that nothing need be cut).
// Walks the sequences 64 at a time, a lane each: at(e0, rows, sum) with this lane's sequence and the segments of all up to it (of this
// walk's 64) says whether to go on.
struct SeqSegments {
    int first, len, n;           // rows; segments
};
template <typename F>
__device__ __forceinline__ void walk_segments(const SsmParams<__bf16>& p, F&& at) {
    const int lane = threadIdx.x & 63;
    for (int e0 = 0; e0 < p.B; e0 += 64) {
        SeqSegments q = {0, 0, 0};
        if (e0 + lane < p.B) {
            seq_rows(p, e0 + lane, q.first, q.len);
            q.n = q.len <= max(p.seg_len, p.whole_len) ? q.len > 0 : (q.len + p.seg_len - 1) / p.seg_len;
        }
        if (!at(e0, q, running_sum(q.n))) return;
    }
}
// The sequence of segment `unit` of the segments that have `skip` behind them in their sequence, its rows, the segment's place
// there and its number among all; false: there are not so many
template <int SKIP>
__device__ __forceinline__ bool find_segment(const SsmParams<__bf16>& p, int unit, int& b, int& first, int& len, int& place, int& seg) {
    bool found = false;
    int before = 0, before_all = 0;
    walk_segments(p, [&](int e0, const SeqSegments& q, int sum) {
        const int mine = max(q.n - SKIP, 0), mine_sum = SKIP == 0 ? sum : running_sum(mine);
        const uint64_t m = __builtin_amdgcn_ballot_w64(unit < before + mine_sum);
        if (m != 0) {
            const int at = __builtin_ctzll(m);
            b = e0 + at;
            first = __builtin_amdgcn_readlane(q.first, at);
            len = __builtin_amdgcn_readlane(q.len, at);
            place = unit - before - __builtin_amdgcn_readlane(mine_sum - mine, at);
            seg = before_all + __builtin_amdgcn_readlane(sum - q.n, at) + place;
            found = true;
            return false;
        }
        before += __builtin_amdgcn_readlane(mine_sum, 63);
        before_all += __builtin_amdgcn_readlane(sum, 63);
        return true;
    });
    return found;
}

// two values -> their bf16 parts and the bf16 parts of what those leave: v = hi + lo to 16 bits
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = pack_bf16(a, b);
    lo = pack_bf16(a - __builtin_bit_cast(float, hi << 16), b - __builtin_bit_cast(float, hi & 0xffff0000u));
}

// Chunked form for bf16 prompts.  With c_t = a_1 + .. + a_t inside a chunk of 64 tokens and S the state in front of it:
//     y_t = exp(c_t) S^T C_t + sum_{s <= t} [exp(c_t - c_s) dt_s (C_t . B_s)] x_s + D x_t
//     S  <- exp(c_last) S + sum_s B_s (exp(c_last - c_s) dt_s x_s)^T
// One workgroup of four wavefronts per (sequence, head, 64 columns of vdim) walks the chunks; wavefront w owns 16 columns
// and keeps its part of S, all 32 * NT rows of it, in MFMA accumulators.  v_mfma_f32_16x16x32_bf16 throughout:
//   G^T (s x t)   = B C^T         rows from LDS, the ten 16 x 16 tiles that hold an s <= t shared out over the wavefronts;
//                                 weighted in fp32, they go to LDS as the rows t of bracketed factors
//   Y^T (p x t)   = S^T C^T       S^T is the accumulator itself: the MFMA's k order is that of the accumulator's rows, which
//                                 the reads of C mirror; scaled by exp(c_t), then
//                 + X^T F^T       X^T fragments through the transposed LDS read
//   S   (n x p)  += B^T (w x)     B^T through the transposed read; w x: the X^T fragments again, weighted in registers
// x, B and C are bf16 (the convolution's output); what is computed in fp32 -- S, the bracketed factors, the weighted x -- enters
// the MFMAs as a bf16 pair of leading part and remainder, so nothing of the recurrence is rounded to 8 bits.
//
// kWhole: a workgroup walks its whole sequence.  Few sequences and heads leave most of the chip idle then, so their segments
// of seg_len tokens go side by side: kSegState leaves what each segment but the last adds to the state, ssd_carry_kernel turns
// these into the states in front of the segments, and kSegOut computes every segment's outputs from there.  A sequence of up to
// seg_len or whole_len tokens is one segment, which only kSegOut sees.
//
// Bound by the chain through a chunk -- three barriers, products that wait for LDS -- with two wavefronts per SIMD (NT 4: 220 registers,
// 66 KB of LDS per workgroup).  What keeps it short: no branch inside a phase (one around each factor took half the VALU cycles),
// four accumulators side by side in each product, one wavefront that prepares the next chunk's decays while the others take its
// share of G, exponentials once per token instead of once per use.  4 sequences of 2048 tokens, 64 heads, state 128: states 50 -> 33
// us, outputs 136 -> 105.  (Four heads per workgroup with shared B C^T: 108 to 124 before that, but one workgroup per compute unit: a
// fifth slower where its rounds do not come out even.)
enum { kWhole, kSegState, kSegOut };
template <int NT, int MODE>
__global__ __launch_bounds__(256, NT == 8 ? 1 : 2) void ssd_chunk_kernel(SsmParams<__bf16> p) {
    constexpr int Q = 64, NP = 32 * NT;
    constexpr int kBRow = NP * 2 + 32, kCRow = NP * 2 + 16, kXRow = 64 * 2 + 32, kFRow = Q * 2 + 16;
    __shared__ __attribute__((aligned(16))) unsigned char b_lds[Q * kBRow];
    __shared__ __attribute__((aligned(16))) unsigned char c_lds[Q * kCRow];
    __shared__ __attribute__((aligned(16))) unsigned char x_lds[Q * kXRow];
    __shared__ __attribute__((aligned(16))) unsigned char f_lds[2][Q * kFRow];        // leading parts, remainders
    // per token, of this chunk and the next one: c_t, dt_t, exp(c_t), exp(c_last - c_t) dt_t
    __shared__ __attribute__((aligned(16))) float cum_lds[2][Q], dt_lds[2][Q], grow_lds[2][Q], left_lds[2][Q];

    const int h = blockIdx.x / p.slices % p.H;
    const int col0 = (blockIdx.x % p.slices) * 64;
    const int unit = blockIdx.x / (p.slices * p.H);
    int b = unit, first, len, place = 0, seg = 0;
    if constexpr (MODE == kWhole) {
        seq_rows(p, b, first, len);
        if (len <= 0) return;
    } else {
        if (!find_segment<MODE == kSegState ? 1 : 0>(p, unit, b, first, len, place, seg)) return;       // (nobody comes after a last one)
        if (seg >= p.n_segs) return;                     // (sequences that overlap: no scratch beyond the caller's)
    }
    bool last = true, alone = true;                      // the sequence's last segment, its only one
    if constexpr (MODE != kWhole) {
        alone = len <= max(p.seg_len, p.whole_len);
        last = alone || (place + 1) * p.seg_len >= len;
        first += place * p.seg_len;
        len = last ? len - place * p.seg_len : p.seg_len;
    }
    const int g = h / (p.H / p.G), inner = p.H * p.P;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int pc = col0 + 16 * wave;                    // first column of this wavefront
    const bool has_cols = pc < p.P;
    const int slot = state_slot(p, b);
    float* st = p.ssm_state + ((int64_t)slot * p.H + h) * p.N * p.Pp + pc + r;
    float* seg_st = MODE == kWhole ? nullptr : p.seg_state + ((int64_t)seg * p.H + h) * p.N * p.Pp + pc + r;
    const float bias = p.dt_bias[h], na2 = p.neg_a[h] * kLog2e, skip = p.d_skip[h];
    const __bf16* xsrc = p.xbc + h * p.P + col0;
    const __bf16* bsrc = p.xbc + inner + g * p.N;
    const __bf16* csrc = p.xbc + inner + (p.G + g) * p.N;

    // S: lane holds column pc + r, rows 16 j + 4 kg + i
    f32x4 S[2 * NT];
    const float* from = alone ? st : seg_st;
    const bool resumed = MODE != kSegState && (!alone || p.positions[first] > 0);
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = 16 * j + 4 * kg + i;
            S[j][i] = resumed && n < p.N && pc + r < p.P ? from[(int64_t)n * p.Pp] : 0.f;
        }

    // one chunk's loads: NT 16-byte pieces of B and C and two of x per thread
    u32x4 rb[NT], rc[NT], rx[2];
    float total = 0.f;                                   // log2 of the decay so far
    const auto fetch = [&](int t0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int idx = j * 256 + tid, row = idx / (4 * NT), col = idx % (4 * NT) * 8;
            rb[j] = rc[j] = u32x4{0u, 0u, 0u, 0u};
            if (t0 + row < len && col < p.N) {
                const int64_t at = (int64_t)(first + t0 + row) * p.channels + col;
                rb[j] = *reinterpret_cast<const u32x4*>(bsrc + at);
                if constexpr (MODE != kSegState) rc[j] = *reinterpret_cast<const u32x4*>(csrc + at);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int idx = j * 256 + tid, row = idx / 8, col = idx % 8 * 8;
            rx[j] = u32x4{0u, 0u, 0u, 0u};
            if (t0 + row < len && col0 + col < p.P)
                rx[j] = *reinterpret_cast<const u32x4*>(xsrc + (int64_t)(first + t0 + row) * p.channels + col);
        }
    };
    // dt of token t0 + lane, and what follows from it, by one wavefront
    const auto fetch_dt = [&](int t0) {
        return p.proj[(int64_t)(first + min(t0 + lane, len - 1)) * p.proj_stride + p.dt_at + h];
    };
    const auto decays = [&](__bf16 raw, int t0, int buf) {
        const float dt = t0 + lane < len ? softplus((float)raw + bias) : 0.f;
        float cum = na2 * dt;                            // running sum of the log2 decays, per lane = token
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float up = __shfl_up(cum, off, 64);
            cum += lane >= off ? up : 0.f;
        }
        cum_lds[buf][lane] = cum;
        dt_lds[buf][lane] = dt;
        grow_lds[buf][lane] = fast_exp2(cum);
        left_lds[buf][lane] = fast_exp2(__shfl(cum, 63, 64) - cum) * dt;
    };
    __bf16 rdt = (__bf16)0.f;
    fetch(0);
    if (wave == 0) {
        const __bf16 dt0 = fetch_dt(0);
        rdt = fetch_dt(Q);
        decays(dt0, 0, 0);
    }
    if constexpr (MODE != kSegState) {                   // the tiles of the factors that are read but have no s <= t
        if (wave % 2 == 0)
#pragma unroll
            for (int part = 0; part < 2; ++part)
                *reinterpret_cast<u32x2*>(f_lds[part] + (16 * wave + r) * kFRow + (16 * wave + 16 + 4 * kg) * 2) = u32x2{0u, 0u};
    }
    int buf = 0;
    for (int t0 = 0; t0 < len; t0 += Q, buf ^= 1) {
        __syncthreads();                                 // everybody has read the chunk before
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int idx = j * 256 + tid, row = idx / (4 * NT), col = idx % (4 * NT) * 8;
            *reinterpret_cast<u32x4*>(b_lds + row * kBRow + col * 2) = rb[j];
            if constexpr (MODE != kSegState) *reinterpret_cast<u32x4*>(c_lds + row * kCRow + col * 2) = rc[j];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int idx = j * 256 + tid;
            *reinterpret_cast<u32x4*>(x_lds + (idx / 8) * kXRow + (idx % 8) * 16) = rx[j];
        }
        if (t0 + Q < len) fetch(t0 + Q);
        __syncthreads();
        const float cum_last = cum_lds[buf][Q - 1];
        total += cum_last;
        if (wave == 0 && t0 + Q < len) {                 // (it has the least to do below)
            decays(rdt, t0 + Q, buf ^ 1);
            rdt = fetch_dt(t0 + 2 * Q);
        }

        // ---- bracketed factors: n tiles of 16 s from 16 s0 on of the tokens t = 16 tt + r ----------
        if constexpr (MODE != kSegState) {
            const auto factors = [&](int tt, int s0, auto n_c) {
                constexpr int n = decltype(n_c)::value;
                const int t = 16 * tt + r;
                const float ct = cum_lds[buf][t];
                f32x4 acc[n];
#pragma unroll
                for (int m = 0; m < n; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const bf16x8 cf = as_bf16x8(*reinterpret_cast<const u32x4*>(c_lds + t * kCRow + (32 * u + 8 * kg) * 2));
#pragma unroll
                    for (int m = 0; m < n; ++m)
                        acc[m] = mfma16(as_bf16x8(*reinterpret_cast<const u32x4*>(b_lds + (16 * (s0 + m) + r) * kBRow + (32 * u + 8 * kg) * 2)),
                                        cf, acc[m]);
                }
#pragma unroll
                for (int m = 0; m < n; ++m) {
                    const int s = 16 * (s0 + m) + 4 * kg;
                    const f32x4 cs = *reinterpret_cast<const f32x4*>(cum_lds[buf] + s);
                    const f32x4 ds = *reinterpret_cast<const f32x4*>(dt_lds[buf] + s);
                    float f[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = acc[m][i] * (fast_exp2(ct - cs[i]) * ds[i]);
                        f[i] = s + i <= t ? v : 0.f;
                    }
                    uint32_t h0, h1, l0, l1;
                    split_bf16(f[0], f[1], h0, l0);
                    split_bf16(f[2], f[3], h1, l1);
                    *reinterpret_cast<u32x2*>(f_lds[0] + t * kFRow + s * 2) = u32x2{h0, h1};
                    *reinterpret_cast<u32x2*>(f_lds[1] + t * kFRow + s * 2) = u32x2{l0, l1};
                }
            };
            if (wave == 0) {
                factors(0, 0, std::integral_constant<int, 1>{});
            } else if (wave == 1) {
                factors(1, 0, std::integral_constant<int, 2>{});
                factors(3, 3, std::integral_constant<int, 1>{});
            } else {
                factors(wave, 0, std::integral_constant<int, 3>{});
            }
            __syncthreads();
        }
        if (!has_cols) continue;

        // X^T fragments: row p = r, k = token 32 u + 8 kg + j
        bf16x8 xf[2];
        const int tr_row = 8 * kg + (r >> 2), tr_col = (r & 3) * 8;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const unsigned char* src = x_lds + (32 * u + tr_row) * kXRow + 32 * wave + tr_col;
            xf[u] = join_bf16x8(lds_read_tr16(src), lds_read_tr16(src + 4 * kXRow));
        }
        // ---- Y^T -------------------------------------------------------------------------------
        if constexpr (MODE != kSegState) {
            f32x4 acc[4];                                // tokens 16 tt + r: four chains side by side
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                u32x4 hi, lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t a, c;
                    split_bf16(S[2 * u + e / 2][2 * (e % 2)], S[2 * u + e / 2][2 * (e % 2) + 1], a, c);
                    hi[e] = a;
                    lo[e] = c;
                }
                bf16x8 cf[4];
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    const unsigned char* src = c_lds + (16 * tt + r) * kCRow + (32 * u + 4 * kg) * 2;
                    const u32x2 c0 = *reinterpret_cast<const u32x2*>(src), c1 = *reinterpret_cast<const u32x2*>(src + 32);
                    cf[tt] = as_bf16x8(u32x4{c0[0], c0[1], c1[0], c1[1]});
                }
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(as_bf16x8(hi), cf[tt], acc[tt]);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) acc[tt] = mfma16(as_bf16x8(lo), cf[tt], acc[tt]);
            }
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) acc[tt] *= grow_lds[buf][16 * tt + r];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int tt = 2 * u; tt < 4; ++tt)
                        acc[tt] = mfma16(xf[u], as_bf16x8(*reinterpret_cast<const u32x4*>(f_lds[part] + (16 * tt + r) * kFRow + (32 * u + 8 * kg) * 2)), acc[tt]);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const int t = 16 * tt + r;
                const u32x2 xw = *reinterpret_cast<const u32x2*>(x_lds + t * kXRow + (16 * wave + 4 * kg) * 2);
                const uint32_t x01 = xw[0], x23 = xw[1];
                const bf16x2 xa = __builtin_bit_cast(bf16x2, x01), xb = __builtin_bit_cast(bf16x2, x23);
                u32x2 o;
                o[0] = pack_bf16(fmaf(skip, (float)xa[0], acc[tt][0]), fmaf(skip, (float)xa[1], acc[tt][1]));
                o[1] = pack_bf16(fmaf(skip, (float)xb[0], acc[tt][2]), fmaf(skip, (float)xb[1], acc[tt][3]));
                if (t0 + t < len && pc + 4 * kg < p.P)
                    *reinterpret_cast<u32x2*>(p.y + (int64_t)(first + t0 + t) * p.y_stride + h * p.P + pc + 4 * kg) = o;
            }
        }
        // ---- S --------------------------------------------------------------------------------
        if (MODE != kSegOut || last || t0 + Q < len) {   // (nobody reads what a segment's last chunk would leave)
            const float decay = fast_exp2(cum_last);
            bf16x8 wh[2], wl[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                u32x4 hi, lo;
                const f32x4* left = reinterpret_cast<const f32x4*>(left_lds[buf] + 32 * u + 8 * kg);
                const f32x4 w0 = left[0], w1 = left[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t a, c;
                    split_bf16((float)xf[u][2 * e] * (e < 2 ? w0 : w1)[2 * e % 4], (float)xf[u][2 * e + 1] * (e < 2 ? w0 : w1)[2 * e % 4 + 1], a, c);
                    hi[e] = a;
                    lo[e] = c;
                }
                wh[u] = as_bf16x8(hi);
                wl[u] = as_bf16x8(lo);
            }
#pragma unroll
            for (int j = 0; j < 2 * NT; ++j) {
                S[j] *= decay;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const unsigned char* src = b_lds + (32 * u + tr_row) * kBRow + 32 * j + tr_col;
                    const bf16x8 bt = join_bf16x8(lds_read_tr16(src), lds_read_tr16(src + 4 * kBRow));
                    S[j] = mfma16(bt, wh[u], S[j]);
                    S[j] = mfma16(bt, wl[u], S[j]);
                }
            }
        }
    }
    if constexpr (MODE == kSegState) {
        if (tid == 0 && col0 == 0) p.seg_decay[(int64_t)seg * p.H + h] = total;
    }
    if (MODE == kSegOut && !last) return;
    float* to = MODE == kSegState ? seg_st : st;
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = 16 * j + 4 * kg + i;
            if (n < p.N && pc + r < p.P) to[(int64_t)n * p.Pp] = S[j][i];
        }
}

// The same recurrence in chunks of 128 tokens, outputs and state on different wavefronts: a workgroup of eight walks the chunks of a sequence or segment for
// one head and 64 columns of vdim.  v_mfma_f32_32x32x16_bf16 throughout; what is computed in fp32 enters as a bf16 pair, as above.
//   wavefronts 0-3, 32 tokens t each (column = lane = t; c: running sums from the chunk's start):
//     G^T (s x t)  = B C^T           B's rows from LDS, C's in registers, tile by tile of 32 tokens s
//     Y^T (p x t)  = S^T C^T + X^T F^T     F^T is G^T weighted in its registers: the accumulator is the operand
//     A tile in front of the wavefront's own 32 tokens, which start behind c_r, is weighted by exp(c_r - c_s) dt_s, 32 factors for 1024 weights, and the sum
//     over these and the state by exp(c_t - c_r): no exponent is above zero.  The tile on the diagonal has its exponentials one by one.
//   wavefronts 4-7, half of the state's rows and 32 columns each: S <- exp(c_last) S + B^T (w x), w_s = exp(c_last - c_s) dt_s, in registers; S in front of the
//     next chunk goes to LDS, column by column, so that the others read it as rows.  They also request the next chunk's B and x; wavefront 0 works out its decays.
// Two barriers a chunk: everything that a chunk reads is there; S has been read and may change.
//
// Bound by the instructions of the fourth block of tokens, with its four tiles, and of the state wavefront on the same SIMD: some 8000 cycles a chunk, 5200 of
// them vector instructions issued, 3300 MFMAs.  What keeps it there: fragments read one step ahead behind scheduling barriers (left alone, the compiler
// holds all at once and spills), a body per block of tokens without branches, addresses it cannot hoist, rows that leave behind the next chunk's first product (a
// wait for C in front of which stores stand waits for these too: 9 us of 82), decays on the wavefront with the least to do.  4 sequences of 2048
// tokens, 64 heads, state 128: segments of 512, three launches of the kernels around this one 148 us; whole sequences on ssd_chunk_kernel 138; like this 78.
constexpr int kWalkChunk = 128, kWalkAhead = 3;      // (steps of 16 tokens that the state takes while the outputs read it)
template <int N, int MODE>
__global__ __launch_bounds__(512, 2) void ssd_walk_kernel(SsmParams<__bf16> p) {
    using RX = TileReads<64>;
    constexpr int Q = kWalkChunk, NS = N / 16, kB = Q * N * 2, kX = Q * 128, kS = 64 * N * 2, NT = N / 64;      // NT: 32-row tiles of the state per wavefront
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kB + 2 * kX + 2 * kS];
    __shared__ __attribute__((aligned(16))) float cum_lds[2][Q], dt_lds[2][Q], left_lds[2][Q], col_lds[4][Q];
    unsigned char *const x_lds = lds + 2 * kB, *const s_lds = lds + 2 * kB + 2 * kX;
    const int h = blockIdx.x / p.slices % p.H, col0 = blockIdx.x % p.slices * 64, unit = blockIdx.x / (p.slices * p.H);
    int b = unit, first, len, place = 0, seg = 0;
    bool last = true, alone = true;                      // the sequence's last segment, its only one
    if constexpr (MODE == kWhole) {
        seq_rows(p, b, first, len);
        if (len <= 0) return;
    } else {
        if (!find_segment<0>(p, unit, b, first, len, place, seg) || seg >= p.n_segs) return;
        alone = len <= max(p.seg_len, p.whole_len);
        last = alone || (place + 1) * p.seg_len >= len;
        first += place * p.seg_len;
        len = last ? len - place * p.seg_len : p.seg_len;
    }
    const bool resumed = !alone || p.positions[first] > 0;
    const int g = h / (p.H / p.G), inner = p.H * p.P;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const bool state_wave = wave >= 4;
    const __bf16* xsrc = p.xbc + (int64_t)first * p.channels + h * p.P + col0;
    const __bf16* bsrc = p.xbc + (int64_t)first * p.channels + inner + g * N;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
    const int row_bytes = p.channels * 2;

    // ---- wavefronts 4-7 ----
    const int sw = wave & 3, pt = sw & 1, nt0 = (sw >> 1) * NT;
    f32x16 S[NT];                                        // lane: column 32 pt + n, rows 32 (nt0 + i) + 8 (j / 4) + 4 kg + j % 4
    float* const slot = p.ssm_state + ((int64_t)state_slot(p, b) * p.H + h) * N * p.Pp + col0 + 32 * pt + n;
    // B and x of chunk c (rows past the end: the last one again, weighted by zero); offsets from a chunk's first row
    const auto b_place = [&](int j, int last_row) {
        const int at = 64 * (sw * (kB / 4096) + j) + lane, row = at / (N / 8);
        return (uint32_t)(min(row, last_row) * row_bytes + (((at % (N / 8)) ^ swz<N>(row)) << 4));
    };
    const auto x_place = [&](int j, int last_row) {
        const int row = 8 * (sw * (kX / 4096) + j) + lane / 8;
        return (uint32_t)(min(row, last_row) * row_bytes + (((lane % 8) ^ swz<64>(row)) << 4));
    };
    uint32_t b_voff[kB / 4096], x_voff[kX / 4096];
    const auto issue = [&](int c) {
        const int last_row = len - 1 - c * Q;
        const unsigned char* bs = reinterpret_cast<const unsigned char*>(bsrc) + (int64_t)(c * Q) * row_bytes;
        const unsigned char* xs = reinterpret_cast<const unsigned char*>(xsrc) + (int64_t)(c * Q) * row_bytes;
        const uint32_t b_dst = lds0 + (c & 1) * kB + sw * (kB / 4), x_dst = lds0 + 2 * kB + (c & 1) * kX + sw * (kX / 4);
        if (last_row >= Q - 1) {
#pragma unroll
            for (int j = 0; j < kB / 4096; ++j) dma_to_lds_16(bs, b_voff[j], b_dst + j * 1024);
#pragma unroll
            for (int j = 0; j < kX / 4096; ++j) dma_to_lds_16(xs, x_voff[j], x_dst + j * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < kB / 4096; ++j) dma_to_lds_16(bs, b_place(j, last_row), b_dst + j * 1024);
#pragma unroll
            for (int j = 0; j < kX / 4096; ++j) dma_to_lds_16(xs, x_place(j, last_row), x_dst + j * 1024);
        }
    };
    const auto publish = [&]() {                         // S as rows of columns, leading parts and remainders
        const int col = 32 * pt + n;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                u32x2 hi, lo;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    uint32_t a, c;
                    split_bf16(S[i][4 * q + 2 * e], S[i][4 * q + 2 * e + 1], a, c);
                    hi[e] = a;
                    lo[e] = c;
                }
                unsigned char* to = s_lds + col * (N * 2) + (((4 * (nt0 + i) + q) ^ swz<N>(col)) << 4) + 8 * kg;
                *reinterpret_cast<u32x2*>(to) = hi;
                *reinterpret_cast<u32x2*>(to + kS) = lo;
            }
    };
    const float bias = p.dt_bias[h], na2 = p.neg_a[h] * kLog2e;
    const __bf16* dtsrc = p.proj + (int64_t)first * p.proj_stride + p.dt_at + h;
    __bf16 raw[2] = {(__bf16)0.f, (__bf16)0.f};          // wavefront 0: dt of tokens 2 lane, 2 lane + 1 of the chunk whose decays come next
    const auto fetch_dt = [&](int c) {
#pragma unroll
        for (int i = 0; i < 2; ++i) raw[i] = dtsrc[(int64_t)min(c * Q + 2 * lane + i, len - 1) * p.proj_stride];
    };
    const auto decays = [&](int c) {
        float dt[2], sum = 0.f, cum[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            dt[i] = c * Q + 2 * lane + i < len ? softplus((float)raw[i] + bias) : 0.f;
            sum += na2 * dt[i];
            cum[i] = sum;
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float up = __shfl_up(sum, off, 64);
            sum += lane >= off ? up : 0.f;
        }
        const float all = __shfl(sum, 63, 64);
        float before = __shfl_up(sum, 1, 64);
        before = lane > 0 ? before : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = 2 * lane + i;
            cum_lds[c & 1][t] = before + cum[i];
            dt_lds[c & 1][t] = dt[i];
            left_lds[c & 1][t] = fast_exp2(all - (before + cum[i])) * dt[i];
        }
    };
    int sb_off[2][NT], sx_off[2];                        // transposed fragments: tokens 8 kg + .. of a step of 16
    {
        const int g16 = lane >> 4, s16 = lane & 15;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int row = 8 * (g16 >> 1) + (s16 >> 2) + 4 * e, d = 16 * (g16 & 1) + 4 * (s16 & 3);
            sx_off[e] = row * 128 + (((4 * pt + (d >> 3)) ^ swz<64>(row)) << 4) + (d & 7) * 2;
#pragma unroll
            for (int i = 0; i < NT; ++i) sb_off[e][i] = row * (N * 2) + (((4 * (nt0 + i) + (d >> 3)) ^ swz<N>(row)) << 4) + (d & 7) * 2;
        }
    }
    const int n_chunks = (len + Q - 1) / Q;
    if (state_wave) {
#pragma unroll
        for (int j = 0; j < kB / 4096; ++j) b_voff[j] = b_place(j, Q);
#pragma unroll
        for (int j = 0; j < kX / 4096; ++j) x_voff[j] = x_place(j, Q);
        issue(0);
        const float* from = alone ? slot : p.seg_state + ((int64_t)seg * p.H + h) * N * p.Pp + col0 + 32 * pt + n;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) S[i][j] = 0.f;
        if (resumed) {
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) S[i][j] = from[(int64_t)(32 * (nt0 + i) + 8 * (j >> 2) + 4 * kg + (j & 3)) * p.Pp];
            publish();
        }
        for (int c = 0; c < n_chunks; ++c) {
            const int buf = c & 1;
            wait_vmcnt<0>();
            __syncthreads();                             // B, x, decays and S of this chunk are there
            if (c + 1 < n_chunks) issue(c + 1);
            const bool wanted = MODE == kWhole || last || c + 1 < n_chunks;
            const float decay = fast_exp2(cum_lds[buf][Q - 1]);
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) S[i][j] *= decay;
            // (addresses that the compiler cannot trace: it then adds constants in the reads instead of holding every sum in a register of its own)
            uint32_t x_at[2], b_at[2][NT];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                x_at[e] = lds0 + 2 * kB + buf * kX + sx_off[e];
                asm volatile("" : "+v"(x_at[e]));
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    b_at[e][i] = lds0 + buf * kB + sb_off[e][i];
                    asm volatile("" : "+v"(b_at[e][i]));
                }
            }
            // steps of 16 tokens, their fragments read one step ahead
            bf16x8 xf[2], bf[2][NT];
            f32x4 w[2][2];
            const auto fragments = [&](int u) {
                xf[u & 1] = join_bf16x8(lds_read_tr16_at(x_at[0] + 16 * u * 128), lds_read_tr16_at(x_at[1] + 16 * u * 128));
#pragma unroll
                for (int e = 0; e < 2; ++e) w[u & 1][e] = *reinterpret_cast<const f32x4*>(left_lds[buf] + 16 * u + 8 * kg + 4 * e);
#pragma unroll
                for (int i = 0; i < NT; ++i) bf[u & 1][i] = join_bf16x8(lds_read_tr16_at(b_at[0][i] + 16 * u * N * 2), lds_read_tr16_at(b_at[1][i] + 16 * u * N * 2));
            };
            const auto gather = [&](auto from_c, auto to_c) {
                constexpr int from = decltype(from_c)::value, to = decltype(to_c)::value;
                if constexpr (from == 0) fragments(0);
#pragma unroll
                for (int u = from; u < to; ++u) {
                    if (u + 1 < Q / 16) fragments(u + 1);
                    u32x4 hi, lo;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t a, v;
                        split_bf16((float)xf[u & 1][2 * e] * w[u & 1][e / 2][2 * e % 4], (float)xf[u & 1][2 * e + 1] * w[u & 1][e / 2][2 * e % 4 + 1], a, v);
                        hi[e] = a;
                        lo[e] = v;
                    }
#pragma unroll
                    for (int i = 0; i < NT; ++i) S[i] = mfma32(bf[u & 1][i], as_bf16x8(hi), S[i]);
#pragma unroll
                    for (int i = 0; i < NT; ++i) S[i] = mfma32(bf[u & 1][i], as_bf16x8(lo), S[i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if (wanted) gather(std::integral_constant<int, 0>{}, std::integral_constant<int, kWalkAhead>{});
            __syncthreads();                             // S has been read
            if (wanted) gather(std::integral_constant<int, kWalkAhead>{}, std::integral_constant<int, Q / 16>{});
            if (c + 1 < n_chunks) publish();
        }
        if (last)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) slot[(int64_t)(32 * (nt0 + i) + 8 * (j >> 2) + 4 * kg + (j & 3)) * p.Pp] = S[i][j];
        return;
    }

    // ---- wavefronts 0-3 ----
    const int tb = wave, tq = 32 * tb + n;               // 32-token block, this lane's token of a chunk
    RX rx;
    rx.init(lane);
    // rows of B and of S (column n): rows 16 s + 8 kg .. at this ^ s << 5
    const uint32_t row0 = n * (N * 2) + ((kg ^ swz<N>(n)) << 4);
    bf16x8 cf[NS];
    const __bf16* csrc = p.xbc + (int64_t)first * p.channels + inner + (p.G + g) * N + 8 * kg;
    const auto fetch_c = [&](int c) {
        const __bf16* row = csrc + (int64_t)min(c * Q + tq, len - 1) * p.channels;
#pragma unroll
        for (int s = 0; s < NS; ++s) cf[s] = as_bf16x8(*reinterpret_cast<const u32x4*>(row + 16 * s));
    };
    const float skip = p.d_skip[h];
    // A chunk's rows leave behind the next one's first product: in front of it, the wait for C would be one for the stores too
    u32x2 out[2][4];
    const auto store = [&](int c) {
        if (c * Q + tq >= len) return;
        __bf16* row = p.y + (int64_t)(first + c * Q + tq) * p.y_stride + h * p.P + col0 + 4 * kg;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int q = 0; q < 4; ++q) *reinterpret_cast<u32x2*>(row + 32 * dt + 8 * q) = out[dt][q];
    };
    if (tb == 0) {
        fetch_dt(0);
        decays(0);
        fetch_dt(1);
    }
    fetch_c(0);
    // a loop for every block, without branches inside a chunk: the products of one tile stand among the weights of another
    const auto walk = [&](auto tb_c) {
        constexpr int TB = decltype(tb_c)::value;
        for (int c = 0; c < n_chunks; ++c) {
            const int t0 = c * Q, buf = c & 1;
            const bool busy = t0 + 32 * TB < len;
            __syncthreads();
#pragma unroll
            for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(cf[s]));       // (the wait for C: further down it would be one for the stores as well)
            const float* cum = cum_lds[buf];
            const float* dts = dt_lds[buf];
            f32x16 acc[2];
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
            if (busy && (resumed || c > 0)) {
                uint32_t s_at = lds0 + 2 * kB + 2 * kX + row0;
                asm volatile("" : "+v"(s_at));
                u32x4 sf[2][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) sf[0][i] = lds_load_at<u32x4>(s_at + (i >> 1) * kS + 32 * (i & 1) * N * 2);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (s + 1 < NS) sf[(s + 1) & 1][i] = lds_load_at<u32x4>((s_at ^ ((s + 1) << 5)) + (i >> 1) * kS + 32 * (i & 1) * N * 2);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i & 1] = mfma32(as_bf16x8(sf[s & 1][i]), cf[s], acc[i & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();
            if (c > 0) store(c - 1);
            if (!busy) continue;
            const float ct = cum[tq], cref = TB > 0 ? cum[32 * TB - 1] : 0.f;
            uint32_t b_at = lds0 + buf * kB + row0, x_at[2][2];
            asm volatile("" : "+v"(b_at));
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    x_at[e][dt] = lds0 + 2 * kB + buf * kX + rx.tr_off[e][dt];
                    asm volatile("" : "+v"(x_at[e][dt]));
                }
            for (int s = lane; s < 32 * TB; s += 64) col_lds[TB][s] = fast_exp2(cref - cum[s]) * dts[s];
            // X^T F^T of the tile of tokens 32 st .. , F^T in accumulator order
            const auto add = [&](int st, const float (&f)[16]) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    u32x4 hi, lo;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        uint32_t a, v;
                        split_bf16(f[8 * u + 2 * w], f[8 * u + 2 * w + 1], a, v);
                        hi[w] = a;
                        lo[w] = v;
                    }
                    bf16x8 xf[2];
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
                        xf[dt] = join_bf16x8(lds_read_tr16_at(x_at[0][dt] + (32 * st + 16 * u) * 128), lds_read_tr16_at(x_at[1][dt] + (32 * st + 16 * u) * 128));
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) acc[dt] = mfma32(xf[dt], as_bf16x8(hi), acc[dt]);
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) acc[dt] = mfma32(xf[dt], as_bf16x8(lo), acc[dt]);
                }
            };
            {
                f32x16 G[TB + 1];
#pragma unroll
                for (int st = 0; st <= TB; ++st)
#pragma unroll
                    for (int j = 0; j < 16; ++j) G[st][j] = 0.f;
                // (fragments one step ahead, in program order: left alone, the compiler holds all of them at once, and spills)
                u32x4 bfr[2][TB + 1];
#pragma unroll
                for (int st = 0; st <= TB; ++st) bfr[0][st] = lds_load_at<u32x4>(b_at + 32 * st * N * 2);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
#pragma unroll
                    for (int st = 0; st <= TB; ++st)
                        if (s + 1 < NS) bfr[(s + 1) & 1][st] = lds_load_at<u32x4>((b_at ^ ((s + 1) << 5)) + 32 * st * N * 2);
#pragma unroll
                    for (int st = 0; st <= TB; ++st) G[st] = mfma32(as_bf16x8(bfr[s & 1][st]), cf[s], G[st]);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const float head = fast_exp2(cref), rowf = fast_exp2(ct - cref);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc[dt][j] *= head;
                float f[2][16];
                const auto weigh = [&](int st, float (&to)[16]) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f32x4 w = *reinterpret_cast<const f32x4*>(col_lds[TB] + 32 * st + 8 * q + 4 * kg);
#pragma unroll
                        for (int e = 0; e < 4; ++e) to[4 * q + e] = G[st][4 * q + e] * w[e];
                    }
                };
                const auto weigh_diagonal = [&](float (&to)[16]) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int s = 8 * q + 4 * kg;
                        const f32x4 cs = *reinterpret_cast<const f32x4*>(cum + 32 * TB + s), ds = *reinterpret_cast<const f32x4*>(dts + 32 * TB + s);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = G[TB][4 * q + e] * (fast_exp2(ct - cs[e]) * ds[e]);
                            to[4 * q + e] = s + e <= n ? v : 0.f;
                        }
                    }
                };
                if constexpr (TB > 0) weigh(0, f[0]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int st = 0; st < TB; ++st) {
                    if (st + 1 < TB) weigh(st + 1, f[(st + 1) & 1]);
                    else weigh_diagonal(f[TB & 1]);
                    add(st, f[st & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (TB == 0) weigh_diagonal(f[0]);
                if (c + 1 < n_chunks) fetch_c(c + 1);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc[dt][j] *= rowf;
                add(TB, f[TB & 1]);
            }
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const u32x2 xw = *reinterpret_cast<const u32x2*>(x_lds + buf * kX + tq * 128 + (((4 * dt + q) ^ swz<64>(tq)) << 4) + 8 * kg);
                    const uint32_t x01 = xw[0], x23 = xw[1];
                    const bf16x2 xa = __builtin_bit_cast(bf16x2, x01), xb = __builtin_bit_cast(bf16x2, x23);
                    out[dt][q][0] = pack_bf16(fmaf(skip, (float)xa[0], acc[dt][4 * q]), fmaf(skip, (float)xa[1], acc[dt][4 * q + 1]));
                    out[dt][q][1] = pack_bf16(fmaf(skip, (float)xb[0], acc[dt][4 * q + 2]), fmaf(skip, (float)xb[1], acc[dt][4 * q + 3]));
                }
            if constexpr (TB == 0) {                         // (the block with the least to do)
                if (c + 1 < n_chunks) {
                    decays(c + 1);
                    fetch_dt(c + 2);
                }
            }
        }
    };
    if (tb == 0) walk(std::integral_constant<int, 0>{});
    else if (tb == 1) walk(std::integral_constant<int, 1>{});
    else if (tb == 2) walk(std::integral_constant<int, 2>{});
    else walk(std::integral_constant<int, 3>{});
    store(n_chunks - 1);
}

// What the segments of a sequence add -> the states in front of them, in place: a thread owns four columns of one row.
__global__ __launch_bounds__(256) void ssd_carry_kernel(SsmParams<__bf16> p) {
    constexpr int kAhead = 4;
    const int h = blockIdx.x % p.H, b = blockIdx.x / p.H;
    const int64_t size = (int64_t)p.N * p.Pp, at = 4 * (blockIdx.y * 256LL + threadIdx.x);
    int first = 0, n = 0;
    int64_t seg0 = 0;
    walk_segments(p, [&](int e0, const SeqSegments& q, int sum) {
        if (b - e0 > 63) {
            seg0 += __builtin_amdgcn_readlane(sum, 63);
            return true;
        }
        first = __builtin_amdgcn_readlane(q.first, b - e0);
        n = __builtin_amdgcn_readlane(q.n, b - e0);
        seg0 += __builtin_amdgcn_readlane(sum, b - e0) - n;
        return false;
    });
    if (n <= 1) return;
    if (at >= size || seg0 + n > p.n_segs) return;
    f32x4 S = {0.f, 0.f, 0.f, 0.f};
    if (p.positions[first] > 0) S = *reinterpret_cast<const f32x4*>(p.ssm_state + ((int64_t)state_slot(p, b) * p.H + h) * size + at);
    float* seg = p.seg_state + (seg0 * p.H + h) * size + at;
    const float* decay = p.seg_decay + seg0 * p.H + h;
    for (int i = 0; i < n; i += kAhead) {
        f32x4 add[kAhead];
        float d[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (i + j < n - 1) {                         // (the last segment's state is nobody's start)
                add[j] = *reinterpret_cast<const f32x4*>(seg + (i + j) * p.H * size);
                d[j] = decay[(i + j) * p.H];
            }
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (i + j < n) {
                *reinterpret_cast<f32x4*>(seg + (i + j) * p.H * size) = S;
                if (i + j < n - 1) {
                    const float f = fast_exp2(d[j]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[e] = fmaf(f, S[e], add[j][e]);
                }
            }
    }
}

template <typename T, int TILE>
static int launch_conv_tiles(const SsmParams<T>& p, bool vec, hipStream_t s) {
    const int64_t groups = vec ? p.channels / 8 : p.channels;
    const int threads = (groups + 255) / 256 * 256 <= (groups + 191) / 192 * 192 ? 256 : 192;      // (fewer without channels)
    const int64_t wgs = (p.n_rows / TILE + p.B) * ((groups + threads - 1) / threads);
    if (wgs > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs), block(threads);
    if (!vec) hipLaunchKernelGGL((causal_conv_silu_kernel<T, 1, 0, TILE>), grid, block, 0, s, p);
    else if (p.taps == 2) hipLaunchKernelGGL((causal_conv_silu_kernel<T, 8, 2, TILE>), grid, block, 0, s, p);
    else if (p.taps == 3) hipLaunchKernelGGL((causal_conv_silu_kernel<T, 8, 3, TILE>), grid, block, 0, s, p);
    else if (p.taps == 4) hipLaunchKernelGGL((causal_conv_silu_kernel<T, 8, 4, TILE>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((causal_conv_silu_kernel<T, 8, 0, TILE>), grid, block, 0, s, p);
    return (int)hipGetLastError();
}

template <typename T>
static int launch_conv(const SsmParams<T>& p, hipStream_t s) {
    bool vec = p.channels % 8 == 0 && p.xbc_at % 8 == 0 && p.proj_stride % 8 == 0;
    for (const void* ptr : {(const void*)p.proj, (const void*)p.conv_w, (const void*)p.conv_b, (const void*)p.conv_state, (const void*)p.xbc})
        vec = vec && (reinterpret_cast<uintptr_t>(ptr) & 15) == 0;
    const int tile = conv_tile(p.n_rows, p.channels, p.taps);
    return tile == 4 ? launch_conv_tiles<T, 4>(p, vec, s) : tile == 8 ? launch_conv_tiles<T, 8>(p, vec, s) : launch_conv_tiles<T, 16>(p, vec, s);
}

template <typename T, bool DECODE>
static int launch_scan(SsmParams<T> p, hipStream_t s) {
    // the widest slice of vdim whose state fits the registers of a workgroup
    int np4 = p.Pp / 4 < 64 ? p.Pp / 4 : 64;
    while (np4 > 1 && (p.N + 256 / np4 - 1) / (256 / np4) > kScanVecs) --np4;
    const int rows = 256 / np4, nv = (p.N + rows - 1) / rows;
    if (nv > kScanVecs) return (int)hipErrorInvalidValue;
    p.np4 = np4;
    p.slices = (p.Pp / 4 + np4 - 1) / np4;
    const int64_t wgs = (int64_t)p.B * p.H * p.slices;
    if (wgs > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const size_t lds = (size_t)((4 * np4 + 2 * p.N + 3) / 4 * 4) * 4 + (size_t)rows * np4 * 16;
    const dim3 grid((unsigned)wgs), block(256);
    if (nv <= 1) hipLaunchKernelGGL((ssm_scan_kernel<T, 1, DECODE>), grid, block, lds, s, p);
    else if (nv <= 2) hipLaunchKernelGGL((ssm_scan_kernel<T, 2, DECODE>), grid, block, lds, s, p);
    else if (nv <= 4) hipLaunchKernelGGL((ssm_scan_kernel<T, 4, DECODE>), grid, block, lds, s, p);
    else if (nv <= 8) hipLaunchKernelGGL((ssm_scan_kernel<T, 8, DECODE>), grid, block, lds, s, p);
    else hipLaunchKernelGGL((ssm_scan_kernel<T, 16, DECODE>), grid, block, lds, s, p);
    return (int)hipGetLastError();
}

static bool chunked_takes(const SsmParams<__bf16>& p) {
    return p.N % 8 == 0 && p.N <= 256 && p.P % 8 == 0 && p.y_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(p.xbc) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(p.y) & 7) == 0;
}

// Sizes that ssd_walk_kernel takes: a state of 64 or 128 rows, whole slices of vdim, rows in 16-byte pieces
static bool walk_takes(const SsmParams<__bf16>& p) { return (p.N == 64 || p.N == 128) && p.P % 64 == 0 && p.channels % 8 == 0 && p.channels < (1 << 23); }

// ... and where it is the faster one.  Its workgroup has a compute unit to itself and needs some 4.6 us per 128 tokens, the other kernel's needs half of one and
// 3.3 us per 64 when it has company (less with a state of 64 rows): launches that give no compute unit a second workgroup, and whole sequences unless they
// are short.  Us, this / the other, 64 heads, state 128: 4 x 2048 tokens whole 143 / 186, 9 x 961 172 / 200, 1 x 64 18 / 21, 16 x 64 45 / 42; 8000 tokens in
// segments of 512 198 / 190; 16 heads, 4000 in segments of 256 57 / 64; state 64, 64 heads: 5 of 122 to 1965 75 / 97, 5 x 111 31 / 30, 14 of 56 to 911 88 / 86.
// (A call that cuts only long sequences has most of them whole.)
static bool walk_pays(const SsmParams<__bf16>& p, int64_t wgs, bool whole) {
    const int n_cu = device_compute_units();
    if (n_cu <= 0) return false;
    const bool longer = whole && p.n_rows >= 192LL * p.B;
    return wgs <= (p.N == 128 || longer ? n_cu + n_cu / 4 : n_cu) || (longer && p.N == 128);
}

template <int MODE>
static int launch_chunks(const SsmParams<__bf16>& p, int64_t units, hipStream_t s) {
    const int64_t wgs = units * p.H * p.slices;
    if (wgs > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs), block(256);
    if constexpr (MODE != kSegState) {
        if (walk_takes(p) && grid_fits(wgs, 512) && walk_pays(p, wgs, MODE == kWhole || p.whole_len > 0)) {
            if (p.N == 64) hipLaunchKernelGGL((ssd_walk_kernel<64, MODE>), grid, dim3(512), 0, s, p);
            else hipLaunchKernelGGL((ssd_walk_kernel<128, MODE>), grid, dim3(512), 0, s, p);
            return (int)hipGetLastError();
        }
    }
    if (p.N <= 32) hipLaunchKernelGGL((ssd_chunk_kernel<1, MODE>), grid, block, 0, s, p);
    else if (p.N <= 64) hipLaunchKernelGGL((ssd_chunk_kernel<2, MODE>), grid, block, 0, s, p);
    else if (p.N <= 128) hipLaunchKernelGGL((ssd_chunk_kernel<4, MODE>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((ssd_chunk_kernel<8, MODE>), grid, block, 0, s, p);
    return (int)hipGetLastError();
}

static int launch_chunked(SsmParams<__bf16> p, hipStream_t s) {
    p.slices = (p.P + 63) / 64;
    if (p.seg_len == 0) return launch_chunks<kWhole>(p, p.B, s);
    // (of a sequence's segments all but the last are full ones)
    const int64_t full = p.n_rows / p.seg_len, pieces = ((int64_t)p.N * p.Pp / 4 + 255) / 256, heads = (int64_t)p.B * p.H;
    p.n_segs = (int)full + p.B;
    if (full > 0) {
        if (int e = launch_chunks<kSegState>(p, full, s)) return e;
        if (pieces > 65535 || heads > 0x7fffffffLL) return (int)hipErrorInvalidValue;
        hipLaunchKernelGGL(ssd_carry_kernel, dim3((unsigned)heads, (unsigned)pieces), dim3(256), 0, s, p);
        if (int e = (int)hipGetLastError()) return e;
    }
    return launch_chunks<kSegOut>(p, p.n_segs, s);
}

template <typename T>
static SsmParams<T> ssm_params(const mi355_ssm_args& a) {
    SsmParams<T> p{};
    p.proj = (const T*)a.proj;
    p.proj_stride = a.proj_row_stride;
    p.xbc_at = a.xbc_col;
    p.dt_at = a.dt_col;
    p.conv_w = a.conv_weight;
    p.conv_b = a.conv_bias;
    p.dt_bias = a.dt_bias;
    p.neg_a = a.neg_a;
    p.d_skip = a.d_skip;
    p.conv_state = (T*)a.conv_state;
    p.ssm_state = a.ssm_state;
    p.slots = a.slots;
    p.positions = a.positions;
    p.cu = a.cu_seqlens;
    p.xbc = (T*)a.xbc;
    p.y = (T*)a.y;
    p.y_stride = a.y_row_stride;
    p.n_rows = a.n_rows;
    p.B = a.batch;
    p.H = a.heads;
    p.P = a.vdim;
    p.Pp = (a.vdim + 3) / 4 * 4;
    p.N = a.state;
    p.G = a.groups;
    p.taps = a.taps;
    p.channels = a.heads * a.vdim + 2 * a.groups * a.state;
    p.n_slots = a.n_slots;
    p.seg_state = a.seg_state;
    p.seg_decay = a.seg_decay;
    p.seg_len = a.seg_len;
    p.whole_len = a.whole_len;
    return p;
}

static int ssm_check(const mi355_ssm_args* a) {
    if (!a || !a->proj || !a->conv_weight || !a->conv_bias || !a->dt_bias || !a->neg_a || !a->d_skip || !a->conv_state || !a->ssm_state ||
        !a->slots || !a->positions || !a->y)
        return set_error(MI355_EINVAL, "ssm: null pointer argument");
    if (a->dtype != MI355_BF16 && a->dtype != MI355_FP32) return set_error(MI355_EDTYPE, "ssm: dtype must be MI355_BF16 or MI355_FP32");
    if (a->batch <= 0 || a->heads <= 0 || a->vdim <= 0 || a->state <= 0 || a->groups <= 0 || a->heads % a->groups || a->n_slots <= 0 || a->n_rows < 0)
        return set_error(MI355_EINVAL, "ssm: batch, heads, vdim, state, groups, n_slots, n_rows out of range (heads a multiple of groups)");
    if (a->taps < 1 || a->taps > kMaxTaps) return set_error(MI355_EINVAL, "ssm: taps must be in 1..16");
    if (a->state > 256 * kScanVecs || a->vdim > (1 << 20)) return set_error(MI355_EINVAL, "ssm: state must be at most 4096");
    if ((reinterpret_cast<uintptr_t>(a->ssm_state) & 15) != 0) return set_error(MI355_EINVAL, "ssm: ssm_state must be 16-byte aligned");
    const int64_t channels = (int64_t)a->heads * a->vdim + 2LL * a->groups * a->state;
    if (a->xbc_col < 0 || a->dt_col < 0 || a->xbc_col + channels > a->proj_row_stride || a->dt_col + a->heads > a->proj_row_stride ||
        a->y_row_stride < (int64_t)a->heads * a->vdim)
        return set_error(MI355_EINVAL, "ssm: columns outside the rows of proj or y");
    if (a->n_rows > 0x7fffff00LL || channels > 0x7fffff00LL) return set_error(MI355_EINVAL, "ssm: too many rows or channels");
    return MI355_OK;
}

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_ssm_prefill(const mi355_ssm_args* args, int scan, void* stream) {
    if (int e = ssm_check(args)) return e;
    if (!args->xbc) return set_error(MI355_EINVAL, "ssm_prefill: null xbc buffer");
    if (!args->cu_seqlens && args->n_rows != args->batch) return set_error(MI355_EINVAL, "ssm_prefill: one row per sequence without cu_seqlens");
    if (scan < MI355_SCAN_AUTO || scan > MI355_SCAN_CHUNKED) return set_error(MI355_EINVAL, "ssm_prefill: unknown scan");
    if (args->seg_len < 0 || args->seg_len % 64 ||
        (args->seg_len > 0 && (!args->seg_state || !args->seg_decay || (reinterpret_cast<uintptr_t>(args->seg_state) & 15))))
        return set_error(MI355_EINVAL, "ssm_prefill: segments are multiples of 64 tokens and need their buffers");
    if (args->n_rows == 0) return MI355_OK;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (args->dtype == MI355_BF16) {
        const SsmParams<__bf16> p = ssm_params<__bf16>(*args);
        const bool chunked = scan != MI355_SCAN_SERIAL && chunked_takes(p);
        if (scan == MI355_SCAN_CHUNKED && !chunked) return set_error(MI355_EINVAL, "ssm_prefill: the chunked scan needs state and vdim in multiples of 8 and state <= 256");
        rc = launch_conv(p, s);
        if (rc == 0) rc = chunked ? launch_chunked(p, s) : launch_scan<__bf16, false>(p, s);
    } else {
        if (scan == MI355_SCAN_CHUNKED) return set_error(MI355_EDTYPE, "ssm_prefill: the chunked scan is bf16");
        const SsmParams<float> p = ssm_params<float>(*args);
        rc = launch_conv(p, s);
        if (rc == 0) rc = launch_scan<float, false>(p, s);
    }
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

extern "C" int mi355_ssm_decode(const mi355_ssm_args* args, void* stream) {
    if (int e = ssm_check(args)) return e;
    if (args->cu_seqlens || args->n_rows != args->batch) return set_error(MI355_EINVAL, "ssm_decode: one row per sequence");
    hipStream_t s = (hipStream_t)stream;
    const int rc = args->dtype == MI355_BF16 ? launch_scan<__bf16, true>(ssm_params<__bf16>(*args), s)
                                             : launch_scan<float, true>(ssm_params<float>(*args), s);
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}
