// Prefill backward of short heads for gfx950: head sizes 32 and 64, dense layout, up to 256 queries and keys, no mask or causal, every
// query head with a key head of its own.
//
// A workgroup holds Q, K, V and dO of a whole head in LDS (64 or 128 KB for 256 rows) and computes all three gradients from there, so each is
// read once, delta never leaves the workgroup, and there is one launch with one wait and one barrier.  Wavefront w owns query rows
// 32 w .. 32 w + 31, for delta and dQ, and then the same keys, for dK and dV: under a causal mask it has w + 1 blocks of keys in
// front and 8 - w blocks of rows behind, nine in all whichever it is.  S and dP are computed in both orientations (seven products where
// five are needed): exchanging dS between the wavefronts would cost more than the MFMAs, which are not what bounds this.
//
// What does is memory and the latency of one load, nine blocks and one store per workgroup.  64 x 16 heads of 32, 256 tokens, fp32 Q and K
// (168 MB, 35 us at copy rate): 60 -> 43 us for the whole backward against bwd_dq_kernel and bwd_dkv_one_kernel, bf16 55 -> 39; heads of 64 110 ->
// 87; 128 tokens of 32 32 -> 23, 100 of 64 54 -> 29; 32 x 32 heads of 64, 160 tokens 74 -> 53; without a mask, 256 of 32 63 -> 46.
#include "launch.hpp"
#include "prefill_bwd_params.hpp"
#include "prefill_tile.hpp"

#include <type_traits>

namespace mi355 {

template <int D, bool CAUSAL, int NWV>
__global__ __launch_bounds__(NWV * 64, D == 32 ? 4 : 2) void bwd_short_kernel(BwdParams p) {
    using R = TileReads<D>;
    constexpr int NS = R::NS, NDT = R::NDT, kRow = R::kRow, CPR = D / 8, kBytes = 32 * NWV * kRow;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kBytes];     // Q, dO, K, V
    __shared__ __attribute__((aligned(16))) float lse_l[32 * NWV], nd_l[32 * NWV];        // log2 units; -delta
    const int id = xcd_chunked_id(blockIdx.x, gridDim.x, short_heads(D)), h = id % p.Hq, b = id / p.Hq;     // (a constant: divisions by it are 0.2 us of a small call)
    const int sq = p.Sq, sk = p.Sk, coff = sk - sq;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5, row0 = 32 * wave, me = row0 + n;
    unsigned char *q_l = lds, *do_l = lds + kBytes, *k_l = lds + 2 * kBytes, *v_l = lds + 3 * kBytes;

    // this wavefront's rows of all four (rows past the end: the last one again)
    const auto bring = [&](const __bf16* head, int64_t stride, int rows, unsigned char* to) {
        const uint32_t dst = lds_address(to) + row0 * kRow;
#pragma unroll
        for (int j = 0; j < CPR / 2; ++j) {
            const int idx = 64 * j + lane, row = idx / CPR, col = ((idx % CPR) ^ swz<D>(row)) * 16;
            dma_to_lds_16(head + row0 * stride, (uint32_t)(min(row, rows - 1 - row0) * (int)stride * 2 + col), dst + 1024 * j);
        }
    };
    if (row0 < sq) {
        bring(p.q + b * p.qs[0] + h * p.qs[1], p.qs[2], sq, q_l);
        bring(p.dout + b * p.dos[0] + h * p.dos[1], p.dos[2], sq, do_l);
    }
    if (row0 < sk) {
        bring(p.k + b * p.ks[0] + h * p.ks[1], p.ks[2], sk, k_l);
        bring(p.v + b * p.vs[0] + h * p.vs[1], p.vs[2], sk, v_l);
    }
    bf16x8 of[NS];
    const __bf16* o_row = p.out + b * p.os[0] + h * p.os[1] + (int64_t)min(me, sq - 1) * p.os[2] + 8 * kg;
#pragma unroll
    for (int s = 0; s < NS; ++s) of[s] = as_bf16x8(*reinterpret_cast<const u32x4*>(o_row + 16 * s));
    const int64_t l_at = b * p.ls[0] + h * p.ls[1];
    const float lse = p.lse[l_at + min(me, sq - 1)];
    R rd;
    rd.init(lane);
    wait_vmcnt<0>();

    // operand fragments of this lane's own row: elements 16 s + 8 kg ..
    const auto own = [&](const unsigned char* tile, bf16x8 (&f)[NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s) f[s] = as_bf16x8(*reinterpret_cast<const u32x4*>(tile + row0 * kRow + rd.row_off[s]));
    };
    float my_lse = INFINITY, my_nd = 0.f;
    bf16x8 dof[NS];
    if (row0 < sq) {
        own(do_l, dof);
        float delta = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) delta = fmaf((float)dof[s][e], (float)of[s][e], delta);
        delta = xor32_sum(delta);
        if (me < sq) {
            my_lse = lse * kLog2e;
            my_nd = delta == delta ? -delta : 0.f;       // (a row without keys has out = NaN, and P = 0 everywhere: any finite delta will do)
            if (kg == 0) p.delta[l_at + me] = delta;
        }
    }
    if (kg == 0) {
        lse_l[me] = my_lse;
        nd_l[me] = my_nd;
    }
    __syncthreads();

    const auto scores = [&](const unsigned char* tile, const bf16x8 (&f)[NS], f32x16 r) {
#pragma unroll
        for (int s = 0; s < NS; ++s) r = mfma32(as_bf16x8(*reinterpret_cast<const u32x4*>(tile + rd.row_off[s])), f[s], r);
        return r;
    };
    // acc^T (D x 32 columns) += tile^T . w over 32 rows of the tile
    const auto update = [&](f32x16 (&acc)[NDT], const unsigned char* tile, const u32x4 (&w)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
                acc[dt] = mfma32(join_bf16x8(lds_read_tr16(tile + 16 * u * kRow + rd.tr_off[0][dt]), lds_read_tr16(tile + 16 * u * kRow + rd.tr_off[1][dt])),
                                 as_bf16x8(w[u]), acc[dt]);
    };
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // a lane's column, elements 32 dt + 8 g + 4 kg ..
    const auto store = [&](void* grad, bool f32, const int64_t (&st)[3], const f32x16 (&acc)[NDT], float scale) {
        const int64_t at = b * st[0] + h * st[1] + (int64_t)me * st[2];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                store_grad4(grad, f32, at + 32 * dt + 8 * g + 4 * kg, acc[dt][4 * g] * scale, acc[dt][4 * g + 1] * scale, acc[dt][4 * g + 2] * scale,
                            acc[dt][4 * g + 3] * scale);
    };

    // ---- dQ of this wavefront's rows: column = query, 32 keys at a time ----
    if (row0 < sq) {
        bf16x8 qf[NS];
        own(q_l, qf);
        f32x16 dq[NDT], c0;
#pragma unroll
        for (int i = 0; i < NDT; ++i) dq[i] = zero16;
#pragma unroll
        for (int j = 0; j < 16; ++j) c0[j] = my_nd;
        const auto step = [&](auto masked_c, int t) {
            const f32x16 s_acc = scores(k_l + 32 * t * kRow, qf, zero16), dp = scores(v_l + 32 * t * kRow, dof, c0);
            // element i: key 32 t + 8 (i / 4) + 4 kg + i % 4
            const int lim = (CAUSAL ? min(sk - 1, me + coff) : sk - 1) - 32 * t - 4 * kg;
            u32x4 dsw[2];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float ds[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int i = 2 * j + e;
                    ds[e] = fast_exp2(fmaf(s_acc[i], p.scale_log2, -my_lse)) * dp[i];
                    // (behind the product: dP of a key that the row does not see may have overflowed)
                    if constexpr (decltype(masked_c)::value) ds[e] = 8 * (i >> 2) + (i & 3) <= lim ? ds[e] : 0.f;
                }
                dsw[j >> 2][j & 3] = pack_bf16(ds[0], ds[1]);
            }
            update(dq, k_l + 32 * t * kRow, dsw);
        };
        const int last = CAUSAL ? min(sk - 1, min(row0 + 31, sq - 1) + coff) : sk - 1;
        const int blocks = last < 0 ? 0 : last / 32 + 1, plain = min(blocks, (CAUSAL ? min(sk, max(0, row0 + coff + 1)) : sk) / 32);
        for (int t = 0; t < plain; ++t) step(std::false_type{}, t);
        for (int t = plain; t < blocks; ++t) step(std::true_type{}, t);
        if (me < sq) store(p.dq, p.dq_f32, p.dqs, dq, p.scale);
    }
    // ---- dK and dV of the same keys: column = key, 32 rows at a time ----
    if (row0 < sk) {
        bf16x8 kf[NS], vf[NS];
        own(k_l, kf);
        own(v_l, vf);
        f32x16 dk[NDT], dv[NDT];
#pragma unroll
        for (int i = 0; i < NDT; ++i) dk[i] = dv[i] = zero16;
        const auto step = [&](auto masked_c, int t) {
            f32x16 c0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 d4 = *reinterpret_cast<const f32x4*>(nd_l + 32 * t + 8 * j + 4 * kg);
#pragma unroll
                for (int e = 0; e < 4; ++e) c0[4 * j + e] = d4[e];
            }
            const f32x16 s_acc = scores(q_l + 32 * t * kRow, kf, zero16), dp = scores(do_l + 32 * t * kRow, vf, c0);
            // element 4 j + e: row 32 t + 8 j + 4 kg + e; it sees this key from row me - coff on
            const int lim = CAUSAL ? me - coff - 32 * t - 4 * kg : 0;
            u32x4 pw[2], dsw[2];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 l4 = *reinterpret_cast<const f32x4*>(lse_l + 32 * t + 8 * j + 4 * kg);
                float x[4], ds[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] = fast_exp2(fmaf(s_acc[4 * j + e], p.scale_log2, -l4[e]));
                    ds[e] = x[e] * dp[4 * j + e];
                    if constexpr (decltype(masked_c)::value) {
                        const bool keep = 8 * j + e >= lim;
                        x[e] = keep ? x[e] : 0.f;
                        ds[e] = keep ? ds[e] : 0.f;
                    }
                }
                pw[j >> 1][2 * (j & 1)] = pack_bf16(x[0], x[1]);
                pw[j >> 1][2 * (j & 1) + 1] = pack_bf16(x[2], x[3]);
                dsw[j >> 1][2 * (j & 1)] = pack_bf16(ds[0], ds[1]);
                dsw[j >> 1][2 * (j & 1) + 1] = pack_bf16(ds[2], ds[3]);
            }
            update(dv, do_l + 32 * t * kRow, pw);
            update(dk, q_l + 32 * t * kRow, dsw);
        };
        const int blocks = (sq + 31) / 32, first = CAUSAL ? max(0, row0 - coff) / 32 : 0;
        // (every row from 32 t on sees this wavefront's last key)
        const int plain = CAUSAL ? max(first, (max(0, row0 + 31 - coff) + 31) / 32) : 0;
        for (int t = first; t < min(plain, blocks); ++t) step(std::true_type{}, t);
        for (int t = plain; t < blocks; ++t) step(std::false_type{}, t);
        if (me < sk) {
            store(p.dk, p.dk_f32, p.dks, dk, p.scale);
            store(p.dv, p.dv_f32, p.dvs, dv, 1.f);
        }
    }
}

bool prefill_bwd_short_takes(int Hq, int Hkv, int Sq, int Sk, int D, int mask_mode) {
    return (D == 32 || D == 64) && Hq == Hkv && Sq <= 256 && Sk <= 256 && (mask_mode == MI355_MASK_NONE || mask_mode == MI355_MASK_CAUSAL);
}

template <int D, bool CAUSAL>
static void launch_short(const BwdParams& p, hipStream_t s) {
    const dim3 grid((unsigned)(p.Hq * p.B));
    const int rows = p.Sq > p.Sk ? p.Sq : p.Sk;
    if (rows <= 64) hipLaunchKernelGGL((bwd_short_kernel<D, CAUSAL, 2>), grid, dim3(128), 0, s, p);
    else if (rows <= 128) hipLaunchKernelGGL((bwd_short_kernel<D, CAUSAL, 4>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((bwd_short_kernel<D, CAUSAL, 8>), grid, dim3(512), 0, s, p);
}

int launch_prefill_bwd_short(const BwdParams& p, int D, int mask_mode, hipStream_t s) {
    const bool causal = mask_mode == MI355_MASK_CAUSAL;
    if (D == 32) causal ? launch_short<32, true>(p, s) : launch_short<32, false>(p, s);
    else causal ? launch_short<64, true>(p, s) : launch_short<64, false>(p, s);
    return (int)hipGetLastError();
}

}  // namespace mi355
