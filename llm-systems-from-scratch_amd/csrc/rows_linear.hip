// Linear layers of a decode step on gfx950: up to 32 rows of activations against a weight matrix, with what stands in front of
// and behind the product in a decoder layer.
//
//   in front   the rows may be looked up (token embedding), and normed: y = W (x / rms(x) * g) is computed as (W (x * g)) / rms(x),
//              the squares being summed while the rows pass by
//   behind     STORE bf16, F32 logits, ADD to a residual row, GATE_UP silu(gate) * up of two halves of W, QKV rotation of
//              queries and keys and the write of keys and values into the paged cache
//
// A layer of the decoder is four of these and the attention, where it was four library products, two norms, an activation, a
// rotation and the attention.  All of them are a few microseconds of latency in a small model (8 rows, width 512: products 6.1,
// norms 3.9, rotation 4.1, activation 3.0 us), so fewer launches is what counts there; in a large one the weights' stream is,
// see weight_stream.hpp.  GPU time of a whole step, this against library products and separate operators: 4 layers of width 512,
// 8 rows 84 / 180 us, 32 rows 104 / 225; 4 layers of 2048, 8 rows 212 / 349, 32 rows 284 / 392; 2 layers of 4096, 16 rows
// 265 / 375, 32 rows 335 / 340.  The line at 32 rows is not where it breaks even but what the ring and the accumulators are laid out
// for, two tiles of 16 rows: a small model's step doubles behind it (width 512, 33 rows 227 us), a wide one's does not (4096: 350).  A workgroup takes 32 weight rows; its four or eight wavefronts share k and meet in LDS.
//
// The rows of short prompts go the same way in tiles of 32 (blockIdx.y), each of which reads the weights again: out of the L2s, and what that
// costs is less than the launches that it saves up to a few hundred rows.  GPU us of a layer's four products and what stands between them,
// this / library products and separate operators: width 512, feed-forward 1344, 40 rows 17 / 33, 200 21 / 37, 1024 44 / 54; width
// 1024, 2688, 100 rows 29 / 50, 400 54 / 60, 800 94 / 69.  Of host time a product of the library takes 19, one of these 4.
#include "common.hpp"
#include "launch.hpp"
#include "weight_stream.hpp"

namespace mi355 {

constexpr int kMaxRows = 32, kMaxPromptRows = 1024, kMaxNormCols = 4096;
constexpr int kWideStreamBytes = 16 * 1024;       // of eight wavefronts: two steps each, with a norm's columns one workgroup per compute unit

struct RowsParams {
    const __bf16* x;
    const int64_t* x_rows;           // row ids, or null: row i
    const float* norm;
    const __bf16* w;                 // (n, k), GATE_UP: (2 n, k)
    void* out;
    const __bf16* resid;
    const int64_t* resid_rows;
    int64_t x_count, x_stride, out_stride, resid_count, resid_stride;
    float eps;
    int T, n, k;
    // QKV
    __bf16 *k_cache, *v_cache;
    const int64_t* slots;
    const int32_t* positions;
    const float* freq;               // (2, ctx_len, D/2)
    int64_t n_slots;
    int ctx_len, Hq, Hkv, D;
};

__device__ __forceinline__ int64_t row_id(const int64_t* ids, int64_t count, int i) {
    return ids ? min(max(ids[i], (int64_t)0), count - 1) : i;
}

__device__ __forceinline__ void store_row4(__bf16* to, const float (&v)[4]) {
    *reinterpret_cast<u32x2*>(to) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
}

template <int MODE, int MT, bool NORM, int WAVES, bool TURN>
__global__ __launch_bounds__(64 * WAVES) void rows_linear_kernel(RowsParams p) {
    constexpr int kRing = WAVES == 4 ? kStreamBytes : kWideStreamBytes;
    __shared__ __attribute__((aligned(1024))) unsigned char ring[WAVES * kRing];
    __shared__ __attribute__((aligned(16))) float norm_l[NORM ? kMaxNormCols : 4];
    __shared__ float squares[WAVES][16 * MT];
    constexpr bool kGateUp = MODE == MI355_ROWS_GATE_UP;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4, piece = (lane & 7) ^ (lane >> 3);
    const int n0 = blockIdx.x * (kGateUp ? 16 : 32), row0 = blockIdx.y * 16 * MT;
    uint32_t w_off[4], x_off[2 * MT];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 8 * j + (lane >> 3);
        const int64_t wr = kGateUp ? (row < 16 ? min(n0 + row, p.n - 1) : p.n + min(n0 + row - 16, p.n - 1)) : min(n0 + row, p.n - 1);
        w_off[j] = (uint32_t)((wr * p.k + piece * 8) * 2);
    }
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j)
        x_off[j] = (uint32_t)((row_id(p.x_rows, p.x_count, min(row0 + 8 * j + (lane >> 3), p.T - 1)) * p.x_stride + piece * 8) * 2);
    // What the end of the kernel wants from memory is asked for in front of the stream.  A wavefront sums one row tile and 16
    // columns (GATE_UP: 16 gates and their ups); a lane has four adjacent columns of a row.
    const bool sums = wave < (kGateUp ? MT : 2 * MT);
    const int m_sum = kGateUp ? wave : wave >> 1, half = kGateUp ? 0 : wave & 1;
    const int row = 16 * m_sum + r, t_out = row0 + row, col = n0 + 16 * half + 4 * kg;
    const bool writes = sums && t_out < p.T && col < p.n;
    const bool whole = p.n % 4 == 0;              // (then columns and row strides are too)
    u32x2 res = {0u, 0u};
    f32x2 cs = {0.f, 0.f}, sn = {0.f, 0.f};
    int64_t slot = -1;
    const __bf16* res_at = nullptr;
    if (writes) {
        if constexpr (MODE == MI355_ROWS_ADD) {
            res_at = p.resid + row_id(p.resid_rows, p.resid_count, t_out) * p.resid_stride + col;
            if (whole) res = *reinterpret_cast<const u32x2*>(res_at);
        }
        if constexpr (MODE == MI355_ROWS_QKV) {
            const int pos = min(max(p.positions[t_out], 0), p.ctx_len - 1), pair = col % p.D / 2;
            cs = *reinterpret_cast<const f32x2*>(p.freq + (int64_t)pos * (p.D / 2) + pair);
            sn = *reinterpret_cast<const f32x2*>(p.freq + ((int64_t)p.ctx_len + pos) * (p.D / 2) + pair);
            slot = p.slots[t_out];
        }
    }
    f32x4 acc[MT][2];
    float sq[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) sq[m] = 0.f;
    weight_stream<MT, WAVES, kRing, TURN>(p.w, w_off, p.x, x_off, p.k, TURN ? turn_of(p.k, WAVES, (int)blockIdx.x) : 0, wave, ring + wave * kRing, acc, [&] {
        if constexpr (NORM) {
            for (int c = tid; c < (p.k + 63) / 64 * 64; c += 64 * WAVES) norm_l[c] = c < p.k ? p.norm[c] : 0.f;
            __syncthreads();
        }
    }, [&](int t, int s, int m, bf16x8& x) {
        if constexpr (NORM) {
            const f32x4* g = reinterpret_cast<const f32x4*>(norm_l + 64 * t + 32 * s + 8 * kg);
            const f32x4 g0 = g[0], g1 = g[1];
            u32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = (float)x[2 * e], b = (float)x[2 * e + 1];
                sq[m] = fmaf(a, a, fmaf(b, b, sq[m]));
                y[e] = pack_bf16(a * (e < 2 ? g0[2 * e] : g1[2 * e - 4]), b * (e < 2 ? g0[2 * e + 1] : g1[2 * e - 3]));
            }
            x = as_bf16x8(y);
        }
    });
    __syncthreads();                              // (the sums travel through the ring)
    f32x4* part = reinterpret_cast<f32x4*>(ring);                               // [wave][row tile][16 rows of w][lane]
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int i = 0; i < 2; ++i) part[((wave * MT + m) * 2 + i) * 64 + lane] = acc[m][i];
        if constexpr (NORM) {
            const float s = xor_sum_16_32(sq[m]);
            if (kg == 0) squares[wave][16 * m + r] = s;
        }
    }
    __syncthreads();
    if (!sums) return;
    constexpr int NW = kGateUp ? 2 : 1;
    f32x4 sum[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        sum[i] = part[(m_sum * 2 + half + i) * 64 + lane];
#pragma unroll
        for (int w4 = 1; w4 < WAVES; ++w4) sum[i] += part[((w4 * MT + m_sum) * 2 + half + i) * 64 + lane];
    }
    if (!writes) return;
    if constexpr (NORM) {
        float ssq = 0.f;
#pragma unroll
        for (int w4 = 0; w4 < WAVES; ++w4) ssq += squares[w4][row];
        const float rstd = 1.0f / sqrtf(ssq / (float)p.k + p.eps);
#pragma unroll
        for (int i = 0; i < NW; ++i) sum[i] *= rstd;
    }
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if constexpr (kGateUp) v[q] = sum[0][q] * __builtin_amdgcn_rcpf(1.0f + fast_exp2(-kLog2e * sum[0][q])) * sum[1][q];
        else v[q] = sum[0][q];
    }
    if constexpr (MODE == MI355_ROWS_QKV) {
        const int n_q = p.Hq * p.D, n_k = p.Hkv * p.D;
        const int sect = col < n_q ? 0 : (col < n_q + n_k ? 1 : 2), c = col - (sect == 0 ? 0 : (sect == 1 ? n_q : n_q + n_k));
        if (sect < 2) {
            const float a0 = v[0], a1 = v[2];
            v[0] = cs[0] * a0 - sn[0] * v[1];
            v[1] = sn[0] * a0 + cs[0] * v[1];
            v[2] = cs[1] * a1 - sn[1] * v[3];
            v[3] = sn[1] * a1 + cs[1] * v[3];
        }
        if (sect == 0) return store_row4((__bf16*)p.out + (int64_t)t_out * p.out_stride + c, v);
        if (slot < 0 || slot >= p.n_slots) return;
        store_row4((sect == 1 ? p.k_cache : p.v_cache) + ((slot / 16 * p.Hkv + c / p.D) * 16 + slot % 16) * p.D + c % p.D, v);
        return;
    }
    if constexpr (MODE == MI355_ROWS_ADD) {
        if (whole) {
            const uint32_t r01 = res[0], r23 = res[1];
            const bf16x2 a = __builtin_bit_cast(bf16x2, r01), b = __builtin_bit_cast(bf16x2, r23);
            v[0] += (float)a[0];
            v[1] += (float)a[1];
            v[2] += (float)b[0];
            v[3] += (float)b[1];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (col + q < p.n) v[q] += (float)res_at[q];
        }
    }
    if constexpr (MODE == MI355_ROWS_F32) {
        float* o = (float*)p.out + (int64_t)t_out * p.out_stride + col;
        if (whole) {
            *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (col + q < p.n) o[q] = v[q];
        }
    } else {
        __bf16* o = (__bf16*)p.out + (int64_t)t_out * p.out_stride + col;
        if (whole) {
            store_row4(o, v);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (col + q < p.n) o[q] = (__bf16)v[q];
        }
    }
}

// Eight wavefronts with two steps each, one workgroup per compute unit, where every workgroup has one to itself and k is long: four have their steps one or
// two at a time, a wait on memory each.  Us, four / eight (k x n): 17 rows and more, whose ring of four has one step: 1024 x 2048 4.8 / 4.2, 2048 x 512 4.75 / 4.39, 100 rows 4.85 / 4.52,
// 4096 x 1024, 32 rows 7.4 / 6.4, 14336 x 4096 50 / 34 to 38; norm and 2048 x 6144, 8 rows 10.2 / 9.4, and 1280 x 2048 5.3 / 5.0.  At k = 512 both are the launch (2.41 / 2.48,
// with a norm 3.24 / 3.14 and 17 rows 3.73 / 3.76), at 256 eight lose 0.1 to 0.25; with more workgroups than units a second one hides the waits (300 rows,
// 2688 x 1024 7.0 / 7.1).  Up to 16 rows without a norm have two steps of four wavefronts as well, and less to gain: one row of 2048 x 512 8 % and of 4096 x 512 11 %, 12 and 16 rows of
// 1024 to 1536 lose 1 to 2 %, and 256 workgroups, which fill the chip by themselves, lose up to 5 (8192 rows of w, 8 rows of 1024 5.2 / 5.4, of 1536 6.7 / 6.9, of 3072 10.6 / 10.8) but for rows of whole 4096 bytes (2048 and 4096 gain 3).
template <int MODE, int MT, bool NORM>
static bool eight_pay(const RowsParams& p, int64_t workgroups) {
    if (p.k < 1024 || workgroups > 256) return false;
    if (MT > 1 || NORM) return true;
    return p.k >= 1280 && (workgroups <= 128 ? p.T <= 8 || p.k >= 2048 : p.k % 2048 == 0);
}
// More workgroups than units over rows of whole 4096 bytes begin with steps of their own (turn_of): norm and 4096 x 12288, 8 rows 27.5 -> 23.6, 8192 x 8448 20 % less, 2048 x 16384 12;
// with fewer it costs 1 to 2 %.  Gate and up, two runs of rows a workgroup, only at k = 2048 (5632 11.5 -> 11.0, 8192 10 % less): at 4096 they are -5 to +11 % (5120 +1, 6144 +7, 7168 -3, 8192 +8, 9216
// -3, 11008 0, 14336 +10).
template <int MODE>
static bool rows_turn(const RowsParams& p, int64_t workgroups) {
    return workgroups > 256 && (MODE == MI355_ROWS_GATE_UP ? p.k == 2048 : turn_pays(p.k));
}
template <int MODE, int MT, bool NORM>
static void launch_rows_as(const RowsParams& p, const dim3& grid, hipStream_t s) {
    const int64_t workgroups = (int64_t)grid.x * grid.y;
    if (eight_pay<MODE, MT, NORM>(p, workgroups)) hipLaunchKernelGGL((rows_linear_kernel<MODE, MT, NORM, 8, false>), grid, dim3(512), 0, s, p);
    else if (rows_turn<MODE>(p, workgroups)) hipLaunchKernelGGL((rows_linear_kernel<MODE, MT, NORM, 4, true>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((rows_linear_kernel<MODE, MT, NORM, 4, false>), grid, dim3(256), 0, s, p);
}

template <int MODE>
static int launch_rows(const RowsParams& p, hipStream_t s) {
    const int bn = MODE == MI355_ROWS_GATE_UP ? 16 : 32;
    const int bm = p.T <= 16 ? 16 : 32;
    const dim3 grid((unsigned)((p.n + bn - 1) / bn), (unsigned)((p.T + bm - 1) / bm));
    if (p.norm && p.T <= 16) launch_rows_as<MODE, 1, true>(p, grid, s);
    else if (p.norm) launch_rows_as<MODE, 2, true>(p, grid, s);
    else if (p.T <= 16) launch_rows_as<MODE, 1, false>(p, grid, s);
    else launch_rows_as<MODE, 2, false>(p, grid, s);
    return (int)hipGetLastError();
}

}  // namespace mi355

using namespace mi355;

static int rows_linear_of(const mi355_rows_args* a, int mode, int most_rows, void* stream) {
    if (!a || !a->x || !a->w || !a->out) return set_error(MI355_EINVAL, "rows_linear: null pointer argument");
    if (mode < MI355_ROWS_STORE || mode > MI355_ROWS_QKV) return set_error(MI355_EINVAL, "rows_linear: unknown mode");
    if (a->n_rows < 0 || a->n_rows > most_rows || a->n <= 0 || a->k <= 0 || a->k % 8 || (a->norm && a->k > kMaxNormCols))
        return set_error(MI355_EINVAL, "rows_linear: up to 32 rows (a prompt: 1024); k a multiple of 8, up to 4096 with a norm");
    if (a->n_rows == 0) return MI355_OK;
    const int64_t w_rows = (int64_t)a->n * (mode == MI355_ROWS_GATE_UP ? 2 : 1), x_count = a->x_rows ? a->x_count : a->n_rows;
    if (a->x_row_stride < a->k || a->x_row_stride % 8 || (reinterpret_cast<uintptr_t>(a->x) & 15) || (reinterpret_cast<uintptr_t>(a->w) & 15) ||
        (reinterpret_cast<uintptr_t>(a->out) & 15) || x_count <= 0)
        return set_error(MI355_EINVAL, "rows_linear: rows must be 16-byte aligned");
    if (w_rows * a->k > 0x7fffffffLL || x_count * a->x_row_stride > 0x7fffffffLL)
        return set_error(MI355_EINVAL, "rows_linear: an operand is too large for 32-bit byte offsets");
    const int64_t out_cols = mode == MI355_ROWS_QKV ? (int64_t)a->n_q_heads * a->head_dim : a->n;
    if (a->out_row_stride < out_cols || (a->n % 4 == 0 && a->out_row_stride % 4)) return set_error(MI355_EINVAL, "rows_linear: stride of the output rows");
    if (mode == MI355_ROWS_ADD && a->resid && a->n % 4 == 0 && (a->resid_row_stride % 4 || (reinterpret_cast<uintptr_t>(a->resid) & 7)))
        return set_error(MI355_EINVAL, "rows_linear: residual rows must be 8-byte aligned");
    if (mode == MI355_ROWS_ADD && (!a->resid || a->resid_row_stride < a->n || (a->resid_rows && a->resid_count <= 0)))
        return set_error(MI355_EINVAL, "rows_linear: residual rows");
    if (mode == MI355_ROWS_QKV) {
        if (!a->k_cache || !a->v_cache || !a->slots || !a->positions || !a->freq_cache) return set_error(MI355_EINVAL, "rows_linear: null pointer argument");
        if (a->n_q_heads <= 0 || a->n_kv_heads <= 0 || (a->head_dim != 32 && a->head_dim != 64 && a->head_dim != 128) || a->context_length <= 0 ||
            a->n != (int64_t)(a->n_q_heads + 2 * a->n_kv_heads) * a->head_dim || a->num_blocks <= 0)
            return set_error(MI355_EINVAL, "rows_linear: heads, head_dim (32, 64, 128), context_length, num_blocks");
        if ((reinterpret_cast<uintptr_t>(a->k_cache) | reinterpret_cast<uintptr_t>(a->v_cache) | reinterpret_cast<uintptr_t>(a->freq_cache)) & 7)
            return set_error(MI355_EINVAL, "rows_linear: caches and table must be 8-byte aligned");
    }
    RowsParams p{};
    p.x = (const __bf16*)a->x;
    p.x_rows = a->x_rows;
    p.norm = a->norm;
    p.w = (const __bf16*)a->w;
    p.out = a->out;
    p.resid = (const __bf16*)a->resid;
    p.resid_rows = a->resid_rows;
    p.x_count = x_count;
    p.x_stride = a->x_row_stride;
    p.out_stride = a->out_row_stride;
    p.resid_count = a->resid_count;
    p.resid_stride = a->resid_row_stride;
    p.eps = a->eps;
    p.T = a->n_rows;
    p.n = a->n;
    p.k = a->k;
    p.k_cache = (__bf16*)a->k_cache;
    p.v_cache = (__bf16*)a->v_cache;
    p.slots = a->slots;
    p.positions = a->positions;
    p.freq = a->freq_cache;
    p.n_slots = a->num_blocks * 16;
    p.ctx_len = a->context_length;
    p.Hq = a->n_q_heads;
    p.Hkv = a->n_kv_heads;
    p.D = a->head_dim;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    switch (mode) {
        case MI355_ROWS_STORE: rc = launch_rows<MI355_ROWS_STORE>(p, s); break;
        case MI355_ROWS_F32: rc = launch_rows<MI355_ROWS_F32>(p, s); break;
        case MI355_ROWS_ADD: rc = launch_rows<MI355_ROWS_ADD>(p, s); break;
        case MI355_ROWS_GATE_UP: rc = launch_rows<MI355_ROWS_GATE_UP>(p, s); break;
        default: rc = launch_rows<MI355_ROWS_QKV>(p, s);
    }
    if (rc != 0) return set_error(rc, hipGetErrorString((hipError_t)rc));
    return MI355_OK;
}

extern "C" int mi355_rows_linear(const mi355_rows_args* a, int mode, void* stream) { return rows_linear_of(a, mode, kMaxRows, stream); }

extern "C" int mi355_prompt_linear(const mi355_rows_args* a, int mode, void* stream) { return rows_linear_of(a, mode, kMaxPromptRows, stream); }
