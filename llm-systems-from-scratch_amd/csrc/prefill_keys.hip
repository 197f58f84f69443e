// Prefill forward for gfx950 with small query tiles whose keys are dealt to the wavefronts: no mask or causal; keys and values
// dense, packed or in a paged cache.
//
// A workgroup owns 32 query rows of one (sequence, head); each of its NW wavefronts takes every NW-th tile of 32 keys, with K and V in
// LDS of its own, and keeps its own row maxima, row sums and accumulators.  There is no barrier until the end, where the partial rows meet
// in LDS, so a query tile's chain of dependent key tiles is an NW-th as long, and a launch has a workgroup for every 32 rows.  The maxima are
// exact: the largest weight of a share of a row is a power of two and not rounded, and errors are a tenth smaller than with a reference set beforehand.
//
// Bound by that chain where a launch is small -- the ends of a workgroup some 4 us, then about 1 us per four tiles at head size 128, for loads
// that go out when their place is free, LDS, eight products one behind the other, weights, eight products -- and by instructions issued where it
// is large: 2200 cycles a tile and SIMD for 512 of MFMAs, so the kernels with more rows per workgroup keep the large calls.  (64 rows per workgroup, every
// fragment for two products: 1.3 to 2 times slower at head size 128, where the registers leave one wavefront per SIMD, 5 to 30 % at 64 and 32.)
// Causal, one sequence, us before / like this: 16 heads of 128, 183 tokens 26.4 / 7.6, 1000 41.9 / 18.7; of 64, 1000 21.9 / 12.1; of 32, 1000 17.5 / 9.7;
// 11 packed sequences of 114 tokens, two heads of 128: 37.9 / 6.2.
#include <algorithm>
#include <cmath>

#include "launch.hpp"
#include "prefill_params.hpp"
#include "prefill_tile.hpp"

namespace mi355 {

constexpr int kKyRows = 32, kKyKeys = 32;
// A row's largest weight is 2^-kKyDown: sums over a million of the largest bf16 values stay finite, and products with values down to 2^-106 normal.
constexpr float kKyDown = 20.0f;

// Workgroups by number, worked out on the host: query tiles of a sequence and head, those of all query heads of a key head, of all heads;
// query heads of a key head; workgroups in whole rounds of eight chunks (as in xcd_chunked_id)
struct KeysGrid {
    uint32_t n_qtiles, chunk, per_seq, group, whole;
};

// PAGED: keys and values are read from a paged cache through a block table; a tile of 32 keys is two blocks, whose ids a wavefront holds for its next 32
// tiles, one per lane.
template <int D, bool CAUSAL, int NW, bool PAGED>
__global__ __launch_bounds__(NW * 64, 2) void prefill_keys_kernel(PrefillParams p, KeysGrid g) {
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, kTile = kKyKeys * kRow, CPR = D / 8, NI = kTile / 1024;
    constexpr int kPart = D * 4 + 16, kSlab = kKyRows * kPart;                        // a wavefront's partial rows, fp32
    // per wavefront K, V; at the end the partial rows
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NW * (2 * kTile > kSlab ? 2 * kTile : kSlab)];
    __shared__ float m_lds[NW][kKyRows], l_lds[NW][kKyRows];
    // (the query tiles and query heads that read one key head's rows run on one XCD, the dearest tiles first)
    const uint32_t bid = blockIdx.x, k8 = bid >> 3, turn = k8 / g.chunk;
    const uint32_t id = bid >= g.whole ? bid : (turn * 8 + (bid & 7)) * g.chunk + (k8 - turn * g.chunk);
    const int b = __builtin_amdgcn_readfirstlane(id / g.per_seq);
    const uint32_t in_seq = id - b * g.per_seq;
    const int h = __builtin_amdgcn_readfirstlane(in_seq / g.n_qtiles), hk = __builtin_amdgcn_readfirstlane((uint32_t)h / g.group);
    const int q0 = __builtin_amdgcn_readfirstlane((g.n_qtiles - 1 - (in_seq - h * g.n_qtiles)) * kKyRows);
    int sq = p.Sq, sk = p.Sk;
    int64_t q_at = b * p.qs[0], k_at = b * p.ks[0], v_at = b * p.vs[0], o_at = b * p.os[0], l_at = b * p.ls[0];
    if constexpr (PAGED) {
        const int q_start = p.cu_q[b];
        sq = p.cu_q[b + 1] - q_start;
        sk = max(0, min(p.ctx_lens[b], 16 * p.max_blocks));              // a length beyond what the table row addresses is cut, never chased
        q_at = q_start * p.qs[2];
        o_at = q_start * p.os[2];
        k_at = v_at = 0;
    } else if (p.cu_q) {
        const int q_start = p.cu_q[b], k_start = p.cu_k[b];
        sq = p.cu_q[b + 1] - q_start;
        sk = p.cu_k[b + 1] - k_start;
        q_at = q_start * p.qs[2];
        k_at = k_start * p.ks[2];
        v_at = k_start * p.vs[2];
        o_at = q_start * p.os[2];
        l_at = q_start;
    }
    const __bf16* qb = p.q + q_at + h * p.qs[1];
    const __bf16* kb = p.k + k_at + hk * p.ks[1];
    const __bf16* vb = p.v + v_at + hk * p.vs[1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int coff = sk - sq;
    const int ks2 = (int)p.ks[2], vs2 = (int)p.vs[2];
    unsigned char* const k_lds = lds + wave * 2 * kTile;
    unsigned char* const v_lds = k_lds + kTile;
    const uint32_t k_dst = __builtin_amdgcn_readfirstlane(lds_address(k_lds)), v_dst = k_dst + kTile;
    // byte offset of this lane's 16 bytes of request j of a tile, from the tile's first row; rows past `last`: that one again
    const auto place = [&](int j, int last, int stride) {
        const int idx = 64 * j + lane, row = idx / CPR, col = ((idx % CPR) ^ swz<D>(row)) * 16;
        return (uint32_t)(min(row, last) * stride * 2 + col);
    };
    uint32_t k_voff[NI], v_voff[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        k_voff[j] = place(j, kKyKeys, ks2);
        v_voff[j] = place(j, kKyKeys, vs2);
    }
    R rd;
    rd.init(lane);
    const bf16x2 ones2 = {(__bf16)1.0f, (__bf16)1.0f};

    for (int qw0 = q0; qw0 < sq; qw0 += g.n_qtiles * kKyRows) {           // (once, unless a packed sequence is longer than the caller said)
        const int qi = qw0 + n;
        const int kv_end = CAUSAL ? max(0, min(sk, min(sq, qw0 + kKyRows) + coff)) : sk;
        const int n_tiles = (kv_end + kKyKeys - 1) / kKyKeys;
        const int n_plain = (CAUSAL ? min(sk, max(0, qw0 + coff + 1)) : sk) / kKyKeys;         // tiles that every row sees in full
        bf16x8 qf[NS];
        const __bf16* qrow = qb + (int64_t)min(qi, sq - 1) * p.qs[2];      // (rows past the end are not stored)
#pragma unroll
        for (int s = 0; s < NS; ++s) qf[s] = as_bf16x8(*reinterpret_cast<const u32x4*>(qrow + 16 * s + 8 * kg));
        int ids = 0;
        const auto look_up = [&](int i) {                                 // block ids of this wavefront's tiles number i to i + 31; none past the last block, none outside the pool
            const int block = min(2 * (wave + NW * (i + (lane >> 1))) + (lane & 1), (sk - 1) >> 4);
            const int32_t* at = p.block_table + (int64_t)b * p.table_stride + block;
            asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=&v"(ids) : "v"(at) : "memory");
            ids = min(max(ids, 0), p.num_blocks - 1);
        };
        // K (V) rows of tile number i of this wavefront
        const auto issue = [&](const __bf16* rows, int stride, const uint32_t (&voff)[NI], int i, uint32_t dst) {
            const int tile = wave + NW * i, last = sk - 1 - tile * kKyKeys;
            const __bf16 *at = rows + (int64_t)(tile * kKyKeys) * stride, *at1 = at;
            if constexpr (PAGED) {
                const int64_t elems = (int64_t)p.Hkv * 16 * D;           // from one block of the pool to the next
                at = rows + __builtin_amdgcn_readlane(ids, 2 * i & 63) * elems;
                at1 = last < 16 ? at : rows + __builtin_amdgcn_readlane(ids, (2 * i & 63) + 1) * elems - 16 * D;
            }
            if (last >= kKyKeys - 1) {
#pragma unroll
                for (int j = 0; j < NI; ++j) dma_to_lds_16(j < NI / 2 ? at : at1, voff[j], dst + 1024 * j);
            } else {                                                       // (finite; their scores are masked)
#pragma unroll
                for (int j = 0; j < NI; ++j) dma_to_lds_16(j < NI / 2 ? at : at1, place(j, last, stride), dst + 1024 * j);
            }
        };
        if (wave < n_tiles) {
            if constexpr (PAGED) look_up(0);
            issue(kb, ks2, k_voff, 0, k_dst);
            issue(vb, vs2, v_voff, 0, v_dst);
        }
        // (the one wait on loads that the compiler knows of: inside the loop it would wait for the tiles in flight too)
#pragma unroll
        for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(qf[s]));
        f32x16 o[NDT];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 16; ++j) o[dt][j] = 0.f;
        float m_ref = -INFINITY, neg_ref = 0.f, l = 0.f;                   // m_ref in raw scores (the scale is positive)
        for (int tile = wave, i = 0; tile < n_tiles; tile += NW, ++i) {
            const bool more = tile + NW < n_tiles;
            wait_vmcnt<NI>();                                              // K is in
            f32x16 s_acc;
            {
                u32x4 kf[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) kf[s] = *reinterpret_cast<const u32x4*>(k_lds + rd.row_off[s]);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // ... and read: its place is free
                if constexpr (PAGED) {
                    if (more && (i + 1) % 32 == 0) look_up(i + 1);
                }
                if (more) issue(kb, ks2, k_voff, i + 1, k_dst);
#pragma unroll
                for (int j = 0; j < 16; ++j) s_acc[j] = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s) s_acc = mfma32(as_bf16x8(kf[s]), qf[s], s_acc);
            }
            // element j of this lane: key 32 tile + 8 (j / 4) + 4 kg + j % 4, query qi
            if (tile >= n_plain) {
                const int lim = (CAUSAL ? min(sk - 1, qi + coff) : sk - 1) - tile * kKyKeys - 4 * kg;
#pragma unroll
                for (int j = 0; j < 16; ++j) s_acc[j] = 8 * (j >> 2) + (j & 3) <= lim ? s_acc[j] : -INFINITY;
            }
            float m4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) m4[j] = fmaxf(fmaxf(s_acc[j], s_acc[4 + j]), fmaxf(s_acc[8 + j], s_acc[12 + j]));
            const float mx = xor32_max(fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3])));
            if (__builtin_amdgcn_ballot_w64(mx > m_ref) != 0) {
                const float m_new = fmaxf(m_ref, mx), m_use = m_new == -INFINITY ? 0.f : m_new;     // no key yet: weights 0, not NaN
                const float alpha = fast_exp2((m_ref - m_use) * p.scale_log2);
                m_ref = m_new;
                neg_ref = -m_use * p.scale_log2 - kKyDown;
                l *= alpha;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) o[dt][j] *= alpha;
            }
            u32x4 pw[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float a0 = fast_exp2(fmaf(s_acc[8 * u + 2 * w], p.scale_log2, neg_ref));
                    const float a1 = fast_exp2(fmaf(s_acc[8 * u + 2 * w + 1], p.scale_log2, neg_ref));
                    pw[u][w] = pack_bf16(a0, a1);
                    const uint32_t both = pw[u][w];
                    l = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, both), ones2, l, false);       // what multiplies V
                }
            if (more) wait_vmcnt<NI>();                                    // V is in
            else wait_vmcnt<0>();
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    const i16x4 lo = lds_read_tr16(v_lds + 16 * u * kRow + rd.tr_off[0][dt]);
                    const i16x4 hi = lds_read_tr16(v_lds + 16 * u * kRow + rd.tr_off[1][dt]);
                    o[dt] = mfma32(join_bf16x8(lo, hi), as_bf16x8(pw[u]), o[dt]);
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (more) issue(vb, vs2, v_voff, i + 1, v_dst);
        }

        // ---- the partial rows meet: weights by the common maximum, sums over the wavefronts that had keys ----
        const int n_parts = min(n_tiles, NW);
        l = xor32_sum(l);
        if (kg == 0) {
            m_lds[wave][n] = m_ref;
            l_lds[wave][n] = l;
        }
        __syncthreads();                                                   // (and everybody is done with the keys)
        float m = m_lds[0][n];
#pragma unroll
        for (int w = 1; w < NW; ++w) m = fmaxf(m, m_lds[w][n]);
        const float mine = m == -INFINITY ? 0.f : fast_exp2((m_ref - m) * p.scale_log2);
        if (wave < n_parts) {
            unsigned char* const row = lds + wave * kSlab + n * kPart + 16 * kg;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    *reinterpret_cast<f32x4*>(row + (32 * dt + 8 * e) * 4) =
                        f32x4{o[dt][4 * e] * mine, o[dt][4 * e + 1] * mine, o[dt][4 * e + 2] * mine, o[dt][4 * e + 3] * mine};
        }
        __syncthreads();
        constexpr int kRowsPerPass = NW * 64 / CPR;
        const int ch = tid % CPR;
        for (int r = tid / CPR; r < min(kKyRows, sq - qw0); r += kRowsPerPass) {
            float mr = m_lds[0][r];
#pragma unroll
            for (int w = 1; w < NW; ++w) mr = fmaxf(mr, m_lds[w][r]);
            float sum = 0.f, x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            for (int w = 0; w < n_parts; ++w) {
                sum += mr == -INFINITY ? 0.f : l_lds[w][r] * fast_exp2((m_lds[w][r] - mr) * p.scale_log2);
                const unsigned char* part = lds + w * kSlab + r * kPart + 32 * ch;
                const f32x4 a = *reinterpret_cast<const f32x4*>(part), d = *reinterpret_cast<const f32x4*>(part + 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] += a[e];
                    x[4 + e] += d[e];
                }
            }
            const float inv = 1.0f / sum;                                  // no key: NaN row, like the reference softmax
            u32x4 w8;
#pragma unroll
            for (int e = 0; e < 4; ++e) w8[e] = pack_bf16(x[2 * e] * inv, x[2 * e + 1] * inv);
            *reinterpret_cast<u32x4*>(p.out + o_at + h * p.os[1] + (int64_t)(qw0 + r) * p.os[2] + 8 * ch) = w8;
            if (p.lse && ch == 0) p.lse[l_at + h * p.ls[1] + qw0 + r] = sum > 0.f ? 0.69314718056f * (__log2f(sum) + (mr * p.scale_log2 + kKyDown)) : -INFINITY;
        }
        __syncthreads();                                                   // (the next rows' keys land in the partial rows' place)
    }
}

bool prefill_keys_takes(const PrefillParams& p, int D) {
    return (D == 128 || D == 64 || D == 32) && p.mask_mode != MI355_MASK_BOOL && p.window == 0 && p.n_split <= 1 && !p.head_scale && !p.sink &&
           p.scale_log2 > 0.f;
}

// Microseconds of this kernel, from timings on an MI355X (256 compute units): a launch and the ends of a workgroup, then a chain -- of the query tile with the most
// key tiles, an NW-th of them one behind the other -- and what all workgroups need when they share the compute units: so much each, and so much per tile of
// 32 keys.  D 128: the longer of the two (1 to 32 heads, 1 to 64 sequences of 16 to 4096 tokens); D 32 and 64: of which the longer one counts, and more where they are alike
// (1500 calls of 1 to 4096 heads, 16 to 8000 queries and 16 to 12000 keys: rms 6 to 8 % with four wavefronts, 9 to 12 with eight.  By the longer alone 512 heads of 73 tokens
// at D 64 were 7.4 us, 9.8 as measured, and 256 of 312 17.0, 22.4).
// With eight wavefronts instead of four a compute unit holds half as many workgroups (D 128) and each costs more to end, but the chain is half
// as long: for launches that give no compute unit a second workgroup, from 16 tiles on (one head, 512 / 2000 / 4000 tokens, D 128: 9.2 / 20.1 / 33.8 us
// with four, 9.4 / 16.9 / 26.0 with eight; D 64: 6.5 / 14.0 / 23.5, 6.8 / 11.4 / 17.7).
PrefillKeysPlan prefill_keys_plan(int B, int Hq, int D, int Sq, int Sk, bool causal, int n_cu) {
    const double over = causal && Sk > Sq ? Sk - Sq : 0, most = causal ? std::min<double>(Sk, over + Sq) : Sk, seeing = std::min(Sq, Sk);
    const double tiles = std::ceil(most / kKyKeys), mean = causal ? seeing / Sq * std::min(tiles, (over + 0.5 * seeing) / kKyKeys + 0.5) : tiles;
    const double n = (double)((Sq + kKyRows - 1) / kKyRows) * Hq * B;
    PrefillKeysPlan r{4, 0.0};
    if (D == 128) r.us = 5.0 + std::max(tiles / 4, n / n_cu * (2.0 + 0.24 * mean));
    else if (D == 64) r.us = 4.197 + together(0.6195 * tiles / 4, n / n_cu * (0.9588 + 0.09975 * mean), 1.504);
    else r.us = 3.738 + together(0.4722 * tiles / 4, n / n_cu * (0.5321 + 0.05937 * mean), 1.223);
    if (n <= n_cu && tiles >= 16) {
        double us = 5.0 + 1.45 * tiles / 8;
        if (D == 64) us = 4.221 + together(0.8226 * tiles / 8, n / n_cu * (2.805 + 0.1274 * mean), 1.649);
        else if (D == 32) us = 3.903 + together(0.6298 * tiles / 8, n / n_cu * (1.18 + 0.06362 * mean), 1.254);
        if (D == 128 || us < r.us) r = {8, us};
    }
    if (n >= 1LL << 31 || !grid_fits((int64_t)n, r.wavefronts * 64)) r.us = INFINITY;
    return r;
}

template <int D, int NW>
static void launch_keys(const PrefillParams& p, hipStream_t s) {
    KeysGrid g;
    g.n_qtiles = (p.Sq + kKyRows - 1) / kKyRows;
    g.group = p.Hq / p.Hkv;
    g.chunk = g.n_qtiles * g.group;
    g.per_seq = g.n_qtiles * p.Hq;
    const uint32_t n = g.per_seq * p.B;
    g.whole = n / (8 * g.chunk) * (8 * g.chunk);
    if (p.block_table) hipLaunchKernelGGL((prefill_keys_kernel<D, true, NW, true>), dim3(n), dim3(NW * 64), 0, s, p, g);
    else if (p.mask_mode == MI355_MASK_CAUSAL) hipLaunchKernelGGL((prefill_keys_kernel<D, true, NW, false>), dim3(n), dim3(NW * 64), 0, s, p, g);
    else hipLaunchKernelGGL((prefill_keys_kernel<D, false, NW, false>), dim3(n), dim3(NW * 64), 0, s, p, g);
}

int launch_prefill_keys(const PrefillParams& p, int D, int wavefronts, hipStream_t s) {
    if (wavefronts == 8) {
        if (D == 128) launch_keys<128, 8>(p, s);
        else if (D == 64) launch_keys<64, 8>(p, s);
        else launch_keys<32, 8>(p, s);
    } else {
        if (D == 128) launch_keys<128, 4>(p, s);
        else if (D == 64) launch_keys<64, 4>(p, s);
        else launch_keys<32, 4>(p, s);
    }
    return (int)hipGetLastError();
}

}  // namespace mi355
