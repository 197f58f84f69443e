// dK, dV and dS at head size 128 on wavefronts of 64 keys.  Included by prefill_bwd.hip, whose layouts it shares.
#pragma once

namespace mi355 {

// acc += a b with the accumulator in AGPRs: the 256 of a wavefront are its dK and dV, and the compiler keeps its hands off them.
// (NEW: an operand may come out of the vector instruction right in front -- a result just rounded, an accumulator just moved -- which an MFMA may read two
// wait states later.)
template <bool NEW>
__device__ __forceinline__ void mfma32_into(f32x16& acc, bf16x8 a, bf16x8 b) {
    if constexpr (NEW) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// This lane's number, worked out where it is used: what depends on it would be held in registers that this kernel does not have
__device__ __forceinline__ int lane_here() {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}

// pack_bf16 where it stands (the compiler gathers the words of a vector in one place)
__device__ __forceinline__ uint32_t pack_bf16_here(float a, float b) {
    uint32_t w;
    asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(w) : "v"(a), "v"(b));
    return w;
}

constexpr int kWdWaves = 4, kWdRows = 32, kWdRing = 4, kWdSteps = 64;
// Tiles in LDS: groups of four rows of 256 bytes, as one request brings them, 16 bytes apart.  16-byte piece c of row r is at c ^ 4 (r % 4), so that pieces of one
// column and 16 rows, and 32 bytes of four rows, fall on different banks.
constexpr int kWdGroup = 1040, kWdTile = kBwRows / 4 * kWdGroup;

// dK, dV and dS (layout of bwd_dkv_kernel with DS) of 128 keys of one (batch, kv head).  A wavefront holds K and V of 64 keys, 128 registers, and both accumulators of
// them, all 256 AGPRs: every fragment read from LDS feeds two MFMAs where bwd_dkv_kernel's feed one, and P stays in registers.  Wavefronts 0 and 1 take the
// first 32 rows of a tile of 64, 2 and 3 the others, each 64 of the keys; the halves' sums meet in LDS at the end.
//   bwd_dkv_kernel reads 320 KB of LDS for 64 rows x 128 keys, 2560 cycles against the 2048 of its MFMAs, and takes some 4900; here 144 KB.
// Bound by what stands between its MFMAs: 64 rows take 3300 to 3500 cycles for 2048 of MFMAs, 2575 without memory instructions, 2885 without the stores of dS.
// What brought it there, cycles a step: a table of steps in LDS in place of scalar arithmetic and branches, 4350 -> 3600 (a branch that is taken stands in the
// only wavefront's way); lane offsets of stores worked out, not read, in front of them 300; tiles in groups of four rows 16 bytes apart, so that
// constants in the reads take the place of exclusive ors; rare blocks out of line.
// A workgroup costs 25 K cycles around its steps (first rows 10 K, sums and rows out 12 K), so this is for key tiles with many of them: see ds_passes.
template <int MODE>
__global__ __launch_bounds__(kWdWaves * 64, 1) void bwd_dkv_wide_kernel(BwdParams p) {
    constexpr bool CAUSAL = MODE == MI355_MASK_CAUSAL;
    constexpr int D = 128, NS = D / 16, NDT = D / 32, kRow = D * 2, kTile = kWdTile, kReq = 2 * kBwRows / 4 / kWdWaves + 1, kAhead = 3;
    static_assert(kWdWaves / 2 * 64 == kFuCols && 2 * kWdRows == kBwRows, "a workgroup owns a key tile of the plan");
    static_assert(2 * kWdRing * kTile >= kWdWaves * 64 * 512, "half of the sums pass through the rings");
    // [Q ring][dO ring][lse and delta ring][offsets of each lane's requests][steps of each wavefront]
    constexpr int kRows = 2 * kWdRing * kTile, kOffsets = kRows + kWdRing * 512, kSteps = kOffsets + kReq * kWdWaves * 256;
    constexpr int kStepBytes = 40;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kSteps + kWdWaves * kWdSteps * kStepBytes];

    const int places = p.n_units * p.shares, id = (int)blockIdx.x / places, place = (int)blockIdx.x % places;
    const int unit = p.unit0 + place / p.shares, share = place % p.shares;
    int b, ktile, hk, sq, sk, q_start = 0, k_start = 0, ds_base = 0;
    if (p.cu_q) {
        if (id >= p.n_jobs[0]) return;
        const int2 job = p.k_jobs[id];
        b = __builtin_amdgcn_readfirstlane(job.x);
        ktile = __builtin_amdgcn_readfirstlane(job.y);
        hk = unit;
        q_start = __builtin_amdgcn_readfirstlane(p.cu_q[b]);
        k_start = __builtin_amdgcn_readfirstlane(p.cu_k[b]);
        sq = max(__builtin_amdgcn_readfirstlane(p.cu_q[b + 1]) - q_start, 0);
        sk = max(__builtin_amdgcn_readfirstlane(p.cu_k[b + 1]) - k_start, 0);
        ds_base = __builtin_amdgcn_readfirstlane(p.ds_base[b]);
    } else {
        b = unit / p.Hkv;
        hk = unit % p.Hkv;
        ktile = id;
        sq = p.Sq;
        sk = p.Sk;
    }
    const int G = p.Hq / p.Hkv, coff = sk - sq, k0 = ktile * kFuCols;
    const auto base_of = [&](const int64_t (&st)[3], int start, int head) { return (p.cu_q ? start * st[2] : b * st[0]) + head * st[1]; };

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int keys = wave & 1, rows = wave >> 1;           // which 64 keys, which half of a tile of 64 rows
    const int kw0 = k0 + 64 * keys;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));

    // K and -V of this lane's keys kw0 + 32 c + n: step s covers d = 16 s + 8 kg + j.  (With -V the C operand of dP is delta as it is: the products give delta - dP, and the
    // sign that dS needs is a modifier of its multiplication.)
    bf16x8 kf[2][NS], vf[2][NS];
    f32x16 dk[2][NDT], dv[2][NDT];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < NDT; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) dk[c][i][j] = dv[c][i][j] = 0.f;

    // Steps: 64 rows of one query head, heads innermost, rows from the last ones up; a share takes every shares-th tile of rows.
    const int n_tiles = (sq + kBwRows - 1) / kBwRows, r_top = (n_tiles - 1 - share) * kBwRows, apart = p.shares * kBwRows;
    const auto steps_from = [&](int key, int row) {      // steps whose row `row` of the tile sees `key`: the first ones
        if (ds_base < 0 || r_top < 0 || key >= sk) return 0;
        const int lowest = CAUSAL ? max(key - coff - row, 0) : 0;
        return lowest > r_top ? 0 : ((r_top - lowest) / apart + 1) * G;
    };
    const int n_steps = __builtin_amdgcn_readfirstlane(steps_from(k0, kBwRows - 1));
    // (Behind these no row of this half sees a key of this wavefront, and its dS is not written: bwd_dq_ds_kernel takes what a row does not see as zero.)
    const int my_steps = __builtin_amdgcn_readfirstlane(steps_from(kw0, kWdRows * rows + kWdRows - 1));

    // ---- what a step is: worked out 32 steps at a time, a lane each, and kept in LDS ----
    // (addresses of the tiles of Q and dO | of lse (keys 0) or delta, and of this wavefront's dS blocks | its first row, whether rows or keys are masked, how
    // many of its two blocks some row sees | the lanes that request it: none for steps past the end, so that a step is always as many instructions)
    const bool ragged = r_top + kBwRows > sq;
    const DsLayout dsl(sq, sk, CAUSAL);
    const auto describe = [&](int from) __attribute__((always_inline)) {
        int G = p.Hq / p.Hkv;
        asm volatile("" : "+s"(G));                  // (a reciprocal worked out here, not held in a register over the steps)
        const int lane = lane_here() & 31, t = min(from + lane, n_steps - 1), tile = t / G, head = t - tile * G, r = r_top - tile * apart, first = r + kWdRows * rows;
        const int ds_blocks = dsl.before(n_tiles), most = CAUSAL ? min(sk - 1, r + kBwRows - 1 + coff) : sk - 1;
        const __bf16* q = p.q + base_of(p.qs, q_start, hk * G) + head * p.qs[1] + r * p.qs[2];
        const __bf16* g = p.dout + base_of(p.dos, q_start, hk * G) + head * p.dos[1] + r * p.dos[2];
        const float* row = (keys == 0 ? p.lse : p.delta) + (p.cu_q ? q_start : b * p.ls[0]) + (hk * G + head) * p.ls[1] + r;
        const int64_t ds_first = p.cu_q ? (int64_t)ds_base * p.n_units * G + (int64_t)(hk - p.unit0) * G * ds_blocks : (int64_t)(b * p.Hkv + hk - p.unit0) * G * ds_blocks;
        unsigned char* block = p.ds + (ds_first + (int64_t)head * ds_blocks + dsl.before(r >> 6) + (kw0 >> 5)) * kDsBlock + rows * (kDsBlock / 2);
        const int seen = (kw0 <= most) + (kw0 + 32 <= most), masked = (CAUSAL && kw0 + 63 > first + coff) || first + kWdRows > sq;
        const auto words = [](const void* x) { return u32x2{(uint32_t)(uintptr_t)x, (uint32_t)((uintptr_t)x >> 32)}; };
        unsigned char* const to = lds + kSteps + wave * (kWdSteps * kStepBytes);
        const int at = (from + lane) & (kWdSteps - 1);
        reinterpret_cast<u32x2*>(to)[2 * at] = words(q);
        reinterpret_cast<u32x2*>(to)[2 * at + 1] = words(g);
        reinterpret_cast<u32x2*>(to + kWdSteps * 16)[2 * at] = words(row);
        reinterpret_cast<u32x2*>(to + kWdSteps * 16)[2 * at + 1] = words(block);
        reinterpret_cast<int*>(to + kWdSteps * 32)[at] = first / kWdRows * 8 + masked * 4 + seen;
        reinterpret_cast<int*>(to + kWdSteps * 36)[at] = from + lane < n_steps ? -1 : 0;
    };
    const uint32_t steps_at = lds0 + kSteps + wave * (kWdSteps * kStepBytes);
    const auto scalar64 = [](uint32_t lo, uint32_t hi) {
        return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(hi) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(lo);
    };

    // ---- requests ----
    // Requests 2 i and 2 i + 1 of this wavefront bring rows 16 wave + 4 i + lane / 16 of the tiles of Q and dO, the last one 64 of lse or delta
    uint64_t q_from = 0, do_from = 0, row_from = 0;      // of the step that is requested
    const auto aim = [&](const u32x4& tiles, const u32x2& row) {
        q_from = scalar64(tiles[0], tiles[1]);
        do_from = scalar64(tiles[2], tiles[3]);
        row_from = scalar64(row[0], row[1]);
    };
    const auto read_tiles = [&](int step) { return lds_load_at<u32x4>(steps_at + (step & (kWdSteps - 1)) * 16); };
    const auto read_lanes = [&](int step) { return lds_load_at<int>(steps_at + kWdSteps * 36 + (step & (kWdSteps - 1)) * 4); };
    const auto read_row_src = [&](int step) { return lds_load_at<u32x2>(steps_at + kWdSteps * 16 + (step & (kWdSteps - 1)) * 16); };
    const auto write_offsets = [&](int last) __attribute__((always_inline)) {           // (rows past the last one: that one again)
        const int lane = lane_here(), col = 8 * ((lane & 15) ^ ((lane >> 4) << 2));
        uint32_t* const to = reinterpret_cast<uint32_t*>(lds + kOffsets) + 64 * wave + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = min(16 * wave + 4 * i + (lane >> 4), last);
            to[256 * (2 * i)] = 2u * (uint32_t)(row * (int)p.qs[2] + col);
            to[256 * (2 * i + 1)] = 2u * (uint32_t)(row * (int)p.dos[2] + col);
        }
        to[256 * 8] = 4 * min(lane, last);
    };
    uint32_t offsets_at = 0;                             // (worked out again for each stretch)
    const auto find_offsets = [&]() { offsets_at = lds0 + kOffsets + wave * 256 + lane_here() * 4; };
    const auto offset = [&](int j) { return lds_load_at<uint32_t>(offsets_at + j * 1024); };
    // The step behind the present one has landed; where nothing was requested after it, everything has
    const auto landed = [&](int lanes) __attribute__((always_inline)) {
        if (__builtin_expect(lanes == 0, 0)) wait_vmcnt<0>();
        wait_vmcnt<kReq>();
    };
    const auto request = [&](int lanes, int step, int j, uint32_t off) {      // j-th of kReq
        const uint32_t slot = step & (kWdRing - 1), at = lds0 + slot * kTile + 4 * kWdGroup * wave;
        if (j == 8) dma_to_lds_4_of(lanes, (const void*)row_from, off, lds0 + kRows + slot * 512 + keys * 256);
        else if (j & 1) dma_to_lds_16_of(lanes, (const void*)do_from, off, at + kWdRing * kTile + (j >> 1) * kWdGroup);
        else dma_to_lds_16_of(lanes, (const void*)q_from, off, at + (j >> 1) * kWdGroup);
    };

    // ---- LDS reads ----
    // (addresses of this wavefront's half of a tile)  rows: pieces 2 s + kg of row n; down the columns: d tile i of 16 rows u, the second four of them 8 rows further
    const uint32_t row_at = (n >> 2) * kWdGroup + (n & 3) * kRow + kg * 16, row_swz = (n & 3) << 6;
    const int g16 = lane >> 4, s16 = lane & 15;
    const uint32_t tr_at = (g16 >> 1) * kWdGroup + (s16 >> 2) * kRow + (g16 & 1) * 32 + (s16 & 3) * 8, tr_swz = (s16 >> 2) << 6;
    const auto read_row = [&](uint32_t tile_at, int s) { return lds_load_at<u32x4>((row_swz ^ ((s >> 1) << 6)) + (tile_at + row_at) + (s & 1) * 32); };
    const auto read_tr = [&](uint32_t tile_at, int c) {       // c: 4 u + i
        const uint32_t a = (tr_swz ^ ((c & 3) << 6)) + (tile_at + tr_at) + (c >> 2) * 4 * kWdGroup;
        return join_bf16x8(lds_read_tr16_at(a), lds_read_tr16_at(a + 2 * kWdGroup));
    };

    f32x16 s[2], dp[2];
    u32x4 pw[2][2], dsw[2][2];                           // P and dS of 16 rows (second index), bf16

    uint64_t block = 0;                                  // of the step whose dS is in registers, then of the next one
    int seen = 0, first_row = 0;
    bool masked = false;
    const auto go_on = [&](const u32x2& at, int flags) {
        block = scalar64(at[0], at[1]);
        flags = __builtin_amdgcn_readfirstlane(flags);
        seen = flags & 3;
        masked = flags & 4;
        first_row = flags / 8 * kWdRows;
    };
    const auto read_block = [&](int step) { return lds_load_at<u32x2>(steps_at + kWdSteps * 16 + 8 + (step & (kWdSteps - 1)) * 16); };
    const auto read_flags = [&](int step) { return lds_load_at<int>(steps_at + kWdSteps * 32 + (step & (kWdSteps - 1)) * 4); };
    u32x4 next_rows[2];                                  // the first fragments of the next step's S
    // One step: S, P, dP and dS of step `step` and its dV; dK of the step in front.  Four stretches of sixteen MFMAs.  What goes between two of them is fixed
    // here, since one wavefront a SIMD has nothing else to fill the matrix unit: an MFMA takes 32 cycles, some twelve of them of the wavefront's, so that five
    // vector instructions (an exponential counts for two) fit and a sixth costs eight cycles.  LDS reads stand kAhead fragments in front; memory instructions
    // are spread, as the four wavefronts' would queue up.
    const auto body = [&](auto first_c, auto last_c, int step) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value, LAST = decltype(last_c)::value;
        const uint32_t slot = step & (kWdRing - 1), prev = (step - 1) & (kWdRing - 1), next = (step + 1) & (kWdRing - 1);
        const uint32_t half = lds0 + rows * (kTile / 2), q_at = half + slot * kTile, do_at = q_at + kWdRing * kTile, pq_at = half + prev * kTile;
        const uint32_t rows_at = lds0 + kRows + slot * 512 + 128 * rows + (lane_here() >> 5) * 16;
        u32x4 a[NS], ar[NS];
        bf16x8 tr[8], td[8];
        f32x4 l4[4];
        f32x16 c0;
        uint32_t off = 0;
        int lanes = 0;
        u32x4 tiles;
        u32x2 row_src, block_at;
        int flags = 0;
        const auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        uint32_t ds_at = 0;
        const auto find_ds = [&]() {
            const uint32_t ln = lane_here();
            ds_at = (ln & 31) * 32 + (ln & 32) / 2;
        };
        const auto store_ds = [&](int i) {
            const int c = i >> 1, u = i & 1;
            if (__builtin_expect(seen <= c, 0)) return;
            const bool real = CAUSAL || kw0 + 32 * c + (lane_here() & 31) < sk;       // (a padded key has P != 0; under the causal mask no row sees it)
            uint64_t to = block + c * kDsBlock;
            asm volatile("" : "+s"(to));                 // (an address of scalars and one lane offset)
            __builtin_nontemporal_store(real ? dsw[c][u] : u32x4{0u, 0u, 0u, 0u},
                                        reinterpret_cast<__attribute__((address_space(1))) u32x4*>(to + (uint64_t)((ds_at ^ (128 * u)) + 1024 * u)));
        };
        const auto scale_s = [&](int e) { s[e >> 4][e & 15] = fmaf(s[e >> 4][e & 15], p.scale_log2, l4[(e & 15) >> 2][e & 3]); };
        const auto exp_s = [&](int e) { s[e >> 4][e & 15] = fast_exp2(s[e >> 4][e & 15]); };
        // word w & 3 of rows u = w / 4 & 1 of keys c = w / 8
        const auto pack_p = [&](int w) { pw[w >> 3][(w >> 2) & 1][w & 3] = pack_bf16_here(s[w >> 3][2 * (w & 7)], s[w >> 3][2 * (w & 7) + 1]); };
        const auto make_ds = [&](int w) {
            dsw[w >> 3][(w >> 2) & 1][w & 3] = pack_bf16_here(s[w >> 3][2 * (w & 7)] * -dp[w >> 3][2 * (w & 7)], s[w >> 3][2 * (w & 7) + 1] * -dp[w >> 3][2 * (w & 7) + 1]);
        };
        const auto read_delta = [&](int g) {
            const f32x4 d4 = lds_load_at<f32x4>(rows_at + 256 + 32 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r) c0[4 * g + r] = d4[r];
        };
        const auto mask = [&]() {
            if (__builtin_expect(!masked, 1)) return;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int ln = lane_here(), lim = CAUSAL ? kw0 + 32 * c + (ln & 31) - coff - first_row - 4 * (ln >> 5) : -1, end = sq - first_row - 4 * (ln >> 5);
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = 8 * (e >> 2) + (e & 3);
                    s[c][e] = ((row >= lim) & (row < end)) ? s[c][e] : -INFINITY;
                }
            }
            // (a row that sees no key has delta NaN: any finite one gives the dS = 0 it must have)
#pragma unroll
            for (int e = 0; e < 16; ++e) c0[e] = c0[e] == c0[e] ? c0[e] : 0.f;
        };

        if constexpr (LAST) {
            find_ds();
#pragma unroll
            for (int i = 0; i < 4; ++i) store_ds(i);
#pragma unroll
            for (int i = 0; i < kAhead; ++i) tr[i] = read_tr(pq_at, i);
        } else {
            // ---- S; the dS in front leaves ----
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < 16; ++j) s[c][j] = 0.f;
#pragma unroll
            for (int i = 0; i < kAhead; ++i) a[i] = FIRST || i >= 2 ? read_row(q_at, i) : next_rows[i];
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const int i = m >> 1, c = m & 1;
                s[c] = mfma32(as_bf16x8(a[i]), kf[c][i], s[c]);
                fence();
                if (c == 0) {
                    if (i + kAhead < NS) a[i + kAhead] = read_row(q_at, i + kAhead);
                    else if (!FIRST) tr[i + kAhead - NS] = read_tr(pq_at, i + kAhead - NS);
                }
                if (m < 4) l4[m] = lds_load_at<f32x4>(rows_at + 32 * m);
                if (m == 0) {
                    find_offsets();
                    off = offset(0);
                    tiles = read_tiles(step + 2);
                    row_src = read_row_src(step + 2);
                    lanes = read_lanes(step + 2);
                }
                if (m == 1 && !FIRST) find_ds();
                if (m % 8 == 2 && !FIRST) store_ds(m / 8);
                if (m == 5) {
                    aim(tiles, row_src);
                    lanes = __builtin_amdgcn_readfirstlane(lanes);
                }
                if (m % 8 == 6) {
                    request(lanes, step + 2, m / 8, off);
                    off = offset(m / 8 + 1);             // (of the next one)
                }
                if (m >= 7 && m < 15) {
                    l4[(m - 7) >> 1][2 * ((m - 7) & 1)] *= -kLog2e;
                    l4[(m - 7) >> 1][2 * ((m - 7) & 1) + 1] *= -kLog2e;
                }
                fence();
            }
        }
        // ---- dK of the step in front; S c - lse ----
        if constexpr (FIRST) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) ar[i] = read_row(do_at, i);
#pragma unroll
            for (int j = 2; j < 4; ++j) request(lanes, step + 2, j, offset(j));
            off = offset(4);
            go_on(read_block(step), read_flags(step));
#pragma unroll
            for (int e = 0; e < 32; ++e) scale_s(e);
#pragma unroll
            for (int g = 0; g < 4; ++g) read_delta(g);
        } else {
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const int i = m >> 1, c = m & 1;
                mfma32_into<LAST>(dk[c][i & 3], tr[i], as_bf16x8(dsw[c][i >> 2]));
                fence();
                if (c == 0) {
                    if (i + kAhead < 8) tr[i + kAhead] = read_tr(pq_at, i + kAhead);
                    else if (!LAST) ar[i + kAhead - 8] = read_row(do_at, i + kAhead - 8);
                }
                if constexpr (!LAST) {
                    if (m >= 2) {
#pragma unroll
                        for (int e = (m - 2) * 32 / 14; e < (m - 1) * 32 / 14; ++e) scale_s(e);
                    }
                    if (m == 1) find_ds();
                    if (m % 8 == 2) store_ds(2 + m / 8);
                    if (m == 5) find_offsets();
                    if (m % 8 == 6) {
                        request(lanes, step + 2, 2 + m / 8, off);
                        off = offset(3 + m / 8);
                    }
                    if (m == 8) {
                        block_at = read_block(step);
                        flags = read_flags(step);
                    }
                    if (m == 12) go_on(block_at, flags);
                    if (m >= 8 && m < 12) read_delta(m - 8);
                }
                fence();
            }
        }
        if constexpr (!LAST) {
            mask();
            fence();
            // ---- delta - dP; P ----
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const int i = m >> 1, c = m & 1;
                dp[c] = mfma32(as_bf16x8(ar[i]), vf[c][i], i == 0 ? c0 : dp[c]);
                fence();
                if (c == 0) {
                    if (i + kAhead < NS) ar[i + kAhead] = read_row(do_at, i + kAhead);
                    else td[i + kAhead - NS] = read_tr(do_at, i + kAhead - NS);
                }
                exp_s(2 * m);
                exp_s(2 * m + 1);
                if (m > 0) pack_p(m - 1);
                if (m == 1) find_offsets();
                if (m % 4 == 2) {
                    request(lanes, step + 2, 4 + m / 4, off);
                    off = offset(5 + m / 4);
                }
                fence();
            }
            // ---- dV; dS ----
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const int i = m >> 1, c = m & 1;
                mfma32_into<FIRST>(dv[c][i & 3], td[i], as_bf16x8(pw[c][i >> 2]));
                fence();
                if (c == 0 && i + kAhead < 8) td[i + kAhead] = read_tr(do_at, i + kAhead);
                if (m == 0) pack_p(15);
                if (m == 2) request(lanes, step + 2, 8, off);
                if (m >= 2) make_ds(m - 2);
                if (m >= 14) make_ds(m);
                if (m == 9) {                            // the next step's rows are there, and all are done with the rows two steps in front
                    landed(lanes);
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                if (m >= 10 && m < 14 && m % 2 == 0) next_rows[(m - 10) / 2] = read_row(half + next * kTile, (m - 10) / 2);
                fence();
            }
        }
    };

    if (n_steps > 0) {
        // behind step `step`, whose requests were those of step + 2
        const auto between = [&](int step) __attribute__((always_inline)) {
            if (__builtin_expect(ragged && step + 3 == G && n_steps > G, 0)) write_offsets(kBwRows - 1);        // (where it is the only one, its rows come again)
            if (__builtin_expect((step & 31) == 31, 0)) describe(step + 33);
        };
        // The first two steps; K and V through the places of the third and fourth (keys past the end: the last one again)
        {
            const int row0 = 16 * wave + (lane >> 4), col = 8 * ((lane & 15) ^ ((lane >> 4) << 2));
            const auto bring = [&](const __bf16* from, int64_t stride, int last, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) dma_to_lds_16(from, 2 * (uint32_t)(min(row0 + 4 * i, last) * (int)stride + col), to + (4 * wave + i) * kWdGroup);
            };
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int head = t < G ? t : 0, r = t < G ? r_top : r_top - apart, h = hk * G + head;
                if (t < n_steps) {
                    bring(p.q + base_of(p.qs, q_start, h) + r * p.qs[2], p.qs[2], sq - 1 - r, lds0 + t * kTile);
                    bring(p.dout + base_of(p.dos, q_start, h) + r * p.dos[2], p.dos[2], sq - 1 - r, lds0 + (kWdRing + t) * kTile);
                    const float* row = (keys == 0 ? p.lse : p.delta) + (p.cu_q ? q_start : b * p.ls[0]) + h * p.ls[1] + r;
                    dma_to_lds_4(row, (uint32_t)(4 * min(lane, sq - 1 - r)), lds0 + kRows + t * 512 + keys * 256);
                }
                const int key = k0 + kBwRows * t, last = sk - 1 - key;        // (no key there: the last one)
                const int64_t from = last < 0 ? key + last : key;
                bring(p.k + base_of(p.ks, k_start, hk) + from * p.ks[2], p.ks[2], max(last, 0), lds0 + (2 + t) * kTile);
                bring(p.v + base_of(p.vs, k_start, hk) + from * p.vs[2], p.vs[2], max(last, 0), lds0 + (kWdRing + 2 + t) * kTile);
            }
        }
        write_offsets(sq - 1 - r_top);
        describe(0);
        between(-2);
        between(-1);
        wait_vmcnt<0>();
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint32_t at = lds0 + (2 + keys) * kTile + c * (kTile / 2);
                kf[c][s] = as_bf16x8(read_row(at, s));
                vf[c][s] = as_bf16x8(read_row(at + kWdRing * kTile, s) ^ 0x80008000u);
            }
        __syncthreads();
        if (my_steps > 0) {
            body(std::true_type{}, std::false_type{}, 0);
            between(0);
            for (int step = 1; step < my_steps; ++step) {
                body(std::false_type{}, std::false_type{}, step);
                between(step);
            }
            body(std::false_type{}, std::true_type{}, my_steps);
        }
        for (int step = my_steps; step < n_steps; ++step) {                 // steps that only other wavefronts have something to do in
            aim(read_tiles(step + 2), read_row_src(step + 2));
            const int lanes = __builtin_amdgcn_readfirstlane(read_lanes(step + 2));
            find_offsets();
            asm volatile("s_nop 4" : "+s"(q_from), "+s"(do_from), "+s"(row_from));       // (vector instructions wrote these)
#pragma unroll
            for (int j = 0; j < kReq; ++j) request(lanes, step + 2, j, offset(j));
            between(step);
            landed(lanes);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < NDT; ++i) asm volatile("s_nop 15" : "+a"(dk[c][i]), "+a"(dv[c][i]));       // (the last products are written)

    // The two halves of the rows meet: wavefronts of the first half take dK of their keys, the others dV
    __syncthreads();
    const int lane_out = lane_here(), n_out = lane_out & 31, kg_out = lane_out >> 5;
    unsigned char *const mine = lds + wave * 32768, *const theirs = lds + (wave ^ 2) * 32768;
    const auto give = [&](const f32x16 (&x)[2][NDT]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const int c = t >> 4, i = (t >> 2) & 3, g = 4 * (t & 3);
            *reinterpret_cast<f32x4*>(mine + t * 1024 + lane_out * 16) = f32x4{x[c][i][g], x[c][i][g + 1], x[c][i][g + 2], x[c][i][g + 3]};
            if ((t & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
    };
    const auto finish = [&](f32x16 (&x)[2][NDT], const int64_t (&st)[3], void* grad, bool f32, float f, int part) __attribute__((always_inline)) {
        const int64_t first = base_of(st, k_start, hk);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            unsigned char* const from = theirs + c * 16384;           // (read by this wavefront only, which then has the place to itself)
            f32x4 y[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const f32x4 o = *reinterpret_cast<const f32x4*>(from + t * 1024 + lane_out * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) y[t][r] = (x[c][t >> 2][4 * (t & 3) + r] + o[r]) * f;
            }
            __builtin_amdgcn_sched_barrier(0);
            const int key = kw0 + 32 * c;
            if (p.shares > 1 || f32) {                   // lane owns key n, d = 8 t + 4 kg + ..
                if (key + n_out >= sk) continue;
                const int64_t row = (p.cu_q ? (int64_t)k_start : (int64_t)b * p.Sk) + key + n_out;
                float* const to = p.shares > 1 ? p.part + (((part * p.shares + share) * p.part_rows + row) * p.Hkv + hk) * D : (float*)grad + first + (key + n_out) * st[2];
#pragma unroll
                for (int t = 0; t < 16; ++t) *reinterpret_cast<f32x4*>(to + 8 * t + 4 * kg_out) = y[t];
            } else {                                     // bf16: through rows of 272 bytes in LDS, so that a store writes four whole rows
#pragma unroll
                for (int t = 0; t < 16; ++t)
                    *reinterpret_cast<u32x2*>(from + n_out * 272 + t * 16 + kg_out * 8) = u32x2{pack_bf16(y[t][0], y[t][1]), pack_bf16(y[t][2], y[t][3])};
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int row = 4 * t + (lane_out >> 4), piece = lane_out & 15;
                    const u32x4 w = *reinterpret_cast<const u32x4*>(from + row * 272 + piece * 16);
                    if (key + row < sk) *reinterpret_cast<u32x4*>((__bf16*)grad + first + (key + row) * st[2] + piece * 8) = w;
                }
            }
        }
    };
    if (rows == 0) give(dv);
    else give(dk);
    __syncthreads();
    if (rows == 0) finish(dk, p.dks, p.dk, p.dk_f32, p.scale, 0);
    else finish(dv, p.dvs, p.dv, p.dv_f32, 1.f, 1);
}

}  // namespace mi355
