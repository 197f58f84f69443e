// Prefill forward of short heads for gfx950: head sizes 32 and 64, dense layout, up to 256 keys, no mask or causal.
//
// A sequence of the reference's sample model (16 heads of 32, 256 tokens) is four key tiles: what the 8-wavefront kernel does
// around a tile -- a barrier and a wait for tiles that are requested one ahead, query and output rows through LDS, the vote on
// a second attempt -- outweighs the tile.  Here all keys and values of a head are requested at once, there is one wait and one
// barrier, and from there every wavefront is on its own: four wavefronts take the blocks of 32 query rows from both ends, so that
// under a causal mask each has the same number of tiles.  The row maxima are tracked tile by tile; the second block's query rows
// arrive under the first.  (Tiles that come in one after the other under the first one's work, with a barrier each: 22.5 us.)
#include <type_traits>

#include "launch.hpp"
#include "prefill_params.hpp"
#include "prefill_tile.hpp"

namespace mi355 {

constexpr int kShKeys = 256, kShRows = 256;      // keys of a sequence, query rows of a workgroup

// Eight fp32 values as bf16
__device__ __forceinline__ u32x4 rounded8(const float* x) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(x), b = *reinterpret_cast<const f32x4*>(x + 4);
    return u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])};
}

// ROUND (one query tile, a key head per query head): fp32 operands are rounded on their way in, and what a backward will read in bf16 leaves from here.  64 x 16 heads of 32, 256 tokens, fp32 Q and K, without a backward: two conversions and this kernel without it 38.7 us, like
// this 24.9; 8 x 32 heads, 128 tokens 15.3 / 5.7; 64 x 16 heads of 64, 256 tokens 69.7 / 49.2.
template <int D, bool CAUSAL, bool ROUND>
__global__ __launch_bounds__(256, D == 32 ? 4 : 2) void prefill_short_kernel(PrefillParams p, int n_qtiles, int group, int chunk, RoundedInputs r) {
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, kTile = 64 * kRow, CPR = D / 8;
    __shared__ __attribute__((aligned(1024))) unsigned char k_lds[kShKeys / 64 * kTile];
    __shared__ __attribute__((aligned(1024))) unsigned char v_lds[kShKeys / 64 * kTile];
    // (the query tiles and query heads that read one key head's rows, and heads that share lines, run on one XCD)
    const int id = xcd_chunked_id(blockIdx.x, gridDim.x, chunk);
    const int q0 = id % n_qtiles * kShRows, h = id / n_qtiles % p.Hq, b = id / (n_qtiles * p.Hq), hk = h / group;
    const int rows = min(kShRows, p.Sq - q0), coff = p.Sk - p.Sq;
    const __bf16* qb = p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[1];
    const __bf16* kb = p.k + (int64_t)b * p.ks[0] + (int64_t)hk * p.ks[1];
    const __bf16* vb = p.v + (int64_t)b * p.vs[0] + (int64_t)hk * p.vs[1];
    __bf16* ob = p.out + (int64_t)b * p.os[0] + (int64_t)h * p.os[1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int kv_end = CAUSAL ? max(0, min(p.Sk, q0 + rows + coff)) : p.Sk;
    const int n_tiles = (kv_end + 63) / 64;

    // wavefront w brings tile w in (rows past the end: the last one again, their scores are masked)
    if (wave < n_tiles) {
        const int last = p.Sk - 1 - 64 * wave;
        const __bf16* kt = kb + (int64_t)(64 * wave) * p.ks[2];
        const __bf16* vt = vb + (int64_t)(64 * wave) * p.vs[2];
        const uint32_t k_dst = lds_address(k_lds) + wave * kTile, v_dst = lds_address(v_lds) + wave * kTile;
        const auto bring = [&](const __bf16* tile, int64_t stride, uint32_t dst) {
#pragma unroll
            for (int j = 0; j < CPR; ++j) {
                const int idx = 64 * j + lane, row = idx / CPR, col = ((idx % CPR) ^ swz<D>(row)) * 16, at = min(row, last);
                dma_to_lds_16(tile, (uint32_t)(at * (int)stride * 2 + col), dst + 1024 * j);
            }
        };
        const auto bring_rounded = [&](int which, const int64_t (&st)[3], unsigned char* tile) {
            const float* in = r.in[which] + b * st[0] + hk * st[1] + (int64_t)(64 * wave) * st[2];
            __bf16* out = r.out[which] ? r.out[which] + b * r.strides[which][0] + hk * r.strides[which][1] + (int64_t)(64 * wave) * r.strides[which][2] : nullptr;
            u32x4 x[CPR];
#pragma unroll
            for (int j = 0; j < CPR; ++j) {
                const int idx = 64 * j + lane;
                x[j] = rounded8(in + (int64_t)min(idx / CPR, last) * st[2] + idx % CPR * 8);
            }
#pragma unroll
            for (int j = 0; j < CPR; ++j) {
                const int idx = 64 * j + lane, row = idx / CPR, c = idx % CPR;
                *reinterpret_cast<u32x4*>(tile + row * kRow + ((c ^ swz<D>(row)) << 4)) = x[j];
                if (out && row <= last) *reinterpret_cast<u32x4*>(out + row * r.strides[which][2] + c * 8) = x[j];
            }
        };
        if (!ROUND || !r.in[2]) bring(vt, p.vs[2], v_dst);
        if (!ROUND || !r.in[1]) bring(kt, p.ks[2], k_dst);
        if constexpr (ROUND) {
            if (r.in[1]) bring_rounded(1, p.ks, k_lds + wave * kTile);
            if (r.in[2]) bring_rounded(2, p.vs, v_lds + wave * kTile);
        }
    }
    // blocks of 32 rows: the last ones first, then those that are left from the front
    const int n_blocks = (rows + 31) / 32;
    const int block[2] = {n_blocks - 1 - wave, wave < n_blocks - 4 ? wave : -1};
    bf16x8 qf[2][NS];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            u32x4 a = {0u, 0u, 0u, 0u};
            const int qi = q0 + 32 * block[i] + n;
            if (block[i] >= 0 && qi < p.Sq) {
                const int64_t at = (int64_t)qi * p.qs[2] + 16 * s + 8 * kg;
                if (ROUND && r.in[0]) {
                    a = rounded8(r.in[0] + b * p.qs[0] + h * p.qs[1] + at);
                    if (r.out[0]) *reinterpret_cast<u32x4*>(r.out[0] + b * r.strides[0][0] + h * r.strides[0][1] + qi * r.strides[0][2] + 16 * s + 8 * kg) = a;
                } else {
                    a = *reinterpret_cast<const u32x4*>(qb + at);
                }
            }
            qf[i][s] = as_bf16x8(a);
        }
    R rd;
    rd.init(lane);
    const bf16x2 ones2 = {(__bf16)1.0f, (__bf16)1.0f};
    wait_vmcnt<0>();
    __syncthreads();

#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (block[i] < 0) continue;
        const int qw0 = q0 + 32 * block[i], qi = qw0 + n;
        f32x16 o[NDT];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 16; ++j) o[dt][j] = 0.f;
        float m_ref = -INFINITY, neg_ref = 0.f, l = 0.f;        // m_ref in raw scores (the scale is positive)
        // HALVES of 32 keys from key `first` on
        const auto step = [&](auto masked_c, auto halves_c, int first) {
            constexpr int HALVES = decltype(halves_c)::value;
            const unsigned char* kt = k_lds + first * kRow;
            const unsigned char* vt = v_lds + first * kRow;
            f32x16 s_acc[HALVES];
#pragma unroll
            for (int t = 0; t < HALVES; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) s_acc[t][j] = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    s_acc[t] = mfma32(as_bf16x8(*reinterpret_cast<const u32x4*>(kt + t * 32 * kRow + rd.row_off[s])), qf[i][s], s_acc[t]);
            }
            // element (t, j) of this lane: key first + 32 t + 8 (j / 4) + 4 kg + j % 4, query qi
            if constexpr (decltype(masked_c)::value) {
                const int lim = (CAUSAL ? min(p.Sk - 1, qi + coff) : p.Sk - 1) - first - 4 * kg;
#pragma unroll
                for (int t = 0; t < HALVES; ++t)
#pragma unroll
                    for (int j = 0; j < 16; ++j) s_acc[t][j] = 32 * t + 8 * (j >> 2) + (j & 3) <= lim ? s_acc[t][j] : -INFINITY;
            }
            float mx = s_acc[0][0];
#pragma unroll
            for (int t = 0; t < HALVES; ++t)
#pragma unroll
                for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s_acc[t][j]);
            mx = xor32_max(mx);
            if (__builtin_amdgcn_ballot_w64(mx > m_ref) != 0) {
                const float m_new = fmaxf(m_ref, mx), m_use = m_new == -INFINITY ? 0.f : m_new;     // no key yet: weights 0, not NaN
                const float alpha = fast_exp2((m_ref - m_use) * p.scale_log2);
                m_ref = m_new;
                neg_ref = -m_use * p.scale_log2;
                l *= alpha;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) o[dt][j] *= alpha;
            }
#pragma unroll
            for (int u = 0; u < 2 * HALVES; ++u) {
                const int t = u >> 1, e0 = 8 * (u & 1);
                u32x4 pw;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float a0 = fast_exp2(fmaf(s_acc[t][e0 + 2 * w], p.scale_log2, neg_ref));
                    const float a1 = fast_exp2(fmaf(s_acc[t][e0 + 2 * w + 1], p.scale_log2, neg_ref));
                    pw[w] = pack_bf16(a0, a1);
                    const uint32_t both = pw[w];
                    l = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, both), ones2, l, false);       // what multiplies V
                }
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    const i16x4 lo = lds_read_tr16(vt + 16 * u * kRow + rd.tr_off[0][dt]);
                    const i16x4 hi = lds_read_tr16(vt + 16 * u * kRow + rd.tr_off[1][dt]);
                    o[dt] = mfma32(join_bf16x8(lo, hi), as_bf16x8(pw), o[dt]);
                }
            }
        };
        constexpr std::integral_constant<int, 1> one{};
        constexpr std::integral_constant<int, 2> two{};
        // halves that some query of the block sees, the first n_plain of them in full: on the diagonal that is one, not a tile
        const int last_key = CAUSAL ? min(p.Sk - 1, min(qw0 + 31, p.Sq - 1) + coff) : p.Sk - 1;
        const int halves = last_key < 0 ? 0 : last_key / 32 + 1;
        const int n_plain = min(halves, (CAUSAL ? min(p.Sk, max(0, qw0 + coff + 1)) : p.Sk) / 32);
        int at = 0;
        for (; at + 2 <= n_plain; at += 2) step(std::false_type{}, two, 32 * at);
        if (at < n_plain) step(std::false_type{}, one, 32 * at++);
        for (; at < halves; ++at) step(std::true_type{}, one, 32 * at);

        l = xor32_sum(l);
        const float inv = 1.0f / l;              // no key: NaN row, like the reference softmax
        if (qi < p.Sq) {
            if (p.lse && kg == 0)
                p.lse[(int64_t)b * p.ls[0] + (int64_t)h * p.ls[1] + qi] = l > 0.f ? 0.69314718056f * (__log2f(l) - neg_ref) : -INFINITY;
            __bf16* row = ob + (int64_t)qi * p.os[2];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    u32x2 w;
                    w[0] = pack_bf16(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv);
                    w[1] = pack_bf16(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
                    *reinterpret_cast<u32x2*>(row + 32 * dt + 8 * g + 4 * kg) = w;
                }
        }
    }
}

// fp32 operands of a prefill as bf16, up to three in one launch, in their order in memory; 8 elements a thread.  Bound by bytes, and by the launch where they are few.  Whole call with
// fp32 Q and K, us, a library conversion each / this: 2 x 4 heads of 128, 177 tokens 14.9 / 10.1, 22 x 8 heads, 221 tokens 28.7 / 26.5, 4 x 16 heads of 64, 600 tokens 25.1 / 22.3,
// 8 x 16 heads of 128, 2000 tokens 203 / 201.
__global__ __launch_bounds__(256) void round_operands_kernel(RoundedOperands r) {
    int64_t at = 8 * (blockIdx.x * 256LL + threadIdx.x);
    int i = 0;
    while (i < 2 && at >= r.room[i]) at -= r.room[i++];
    if (at + 8 <= r.n[i]) {
        *reinterpret_cast<u32x4*>(r.out[i] + at) = rounded8(r.in[i] + at);
    } else {
        for (; at < r.n[i]; ++at) r.out[i][at] = (__bf16)r.in[i][at];
    }
}

int launch_round_operands(const float* const in[3], __bf16* const out[3], const int64_t n[3], hipStream_t s) {
    RoundedOperands r{};
    int64_t total = 0;
    for (int i = 0; i < 3; ++i) {
        r.in[i] = in[i];
        r.out[i] = out[i];
        r.n[i] = in[i] ? n[i] : 0;
        r.room[i] = (r.n[i] + 7) / 8 * 8;
        total += r.room[i];
    }
    hipLaunchKernelGGL(round_operands_kernel, dim3((unsigned)((total / 8 + 255) / 256)), dim3(256), 0, s, r);
    return (int)hipGetLastError();
}

// Without a mask every block sees every key, and what is saved around the tiles no longer pays for the row maxima at 256 keys (64 x
// 16 heads of 32: 200 keys 23.6 -> 18.8 us, 256 keys 24.5 -> 24.8; 8 x 16 heads of 64, 256 keys 10.8 -> 11.5).
bool prefill_short_takes(const PrefillParams& p, int D) {
    return (D == 32 || D == 64) && p.Sk <= (p.mask_mode == MI355_MASK_CAUSAL ? kShKeys : 224) && !p.cu_q && !p.block_table && p.mask_mode != MI355_MASK_BOOL && p.window == 0 &&
           p.n_split <= 1 && !p.head_scale && !p.sink && p.scale_log2 > 0.f;
}

template <int D, bool ROUND>
static void launch_short(const PrefillParams& p, const RoundedInputs& r, hipStream_t s) {
    const int n_qtiles = (p.Sq + kShRows - 1) / kShRows;
    const dim3 grid((unsigned)(n_qtiles * p.Hq * p.B));
    // Heads that are neighbours run on one XCD, see short_heads
    const int group = p.Hq / p.Hkv, chunk = n_qtiles * ((short_heads(D) + group - 1) / group * group);
    if (p.mask_mode == MI355_MASK_CAUSAL) hipLaunchKernelGGL((prefill_short_kernel<D, true, ROUND>), grid, dim3(256), 0, s, p, n_qtiles, group, chunk, r);
    else hipLaunchKernelGGL((prefill_short_kernel<D, false, ROUND>), grid, dim3(256), 0, s, p, n_qtiles, group, chunk, r);
}

int launch_prefill_short(const PrefillParams& p, int D, hipStream_t s) {
    if (D == 32) launch_short<32, false>(p, RoundedInputs{}, s);
    else launch_short<64, false>(p, RoundedInputs{}, s);
    return (int)hipGetLastError();
}

int launch_prefill_short_rounded(const PrefillParams& p, const RoundedInputs& r, int D, hipStream_t s) {
    if (p.Sq > kShRows || p.Hq != p.Hkv || !prefill_short_takes(p, D)) return (int)hipErrorInvalidValue;
    if (D == 32) launch_short<32, true>(p, r, s);
    else launch_short<64, true>(p, r, s);
    return (int)hipGetLastError();
}

}  // namespace mi355
