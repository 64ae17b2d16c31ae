// attn_decode_q256.hpp: the decode kernel's form for quantized rows (q8_0, q4_0) of 256 values. Included by attn_decode.hip
// inside its anonymous namespace, behind DecodeParams.
//
// Bound: vector instructions beside HBM. A q4_0 key and value row are 288 bytes and 512 numbers to widen, so a tile's
// arithmetic weighs as much as its bytes, and what a wave waits for - its tile, LDS, the matrix unit's results - passes only
// under other waves' work. Two row tiles of 256 features are 128 registers of sums: with the queries' 64 beside them a wave
// has a SIMD to itself. Here the queries are LDS's (one copy, in operand layout, for the work-group's 8 waves), so two waves fit a
// SIMD, each with tiles of its own: wave w takes the 32-key tiles with (tile index % 8 == w) and meets the others only where
// the queries are staged and the sums merged. (Two waves sharing a tile, half the features or half the keys each, need a
// barrier a tile, and the slowest of eight transfers then sets the pace: 28.5 us where this form took 24 to 25.)
//
// A tile's step: raw keys out of LDS into registers, the next transfer requested into their place, widened two 16-key
// halves at a time, scored; softmax; raw values out of LDS, the next transfer requested, widened 64 features at a time into a
// stage of [key][64] halfs, read back transposed, weighed. q4_0: keys and values have a buffer each, a tile ahead; q8_0, twice
// the bytes: one buffer in turn - the values travel under the scores, the next keys under the values' product - which keeps
// as many bytes in flight.
// A lane's raw key words are whole blocks of its key row (lane group g4: blocks g4 and 4 + g4), so a lane has two scales a key;
// the queries are staged in the order that gives. A row's softmax reference is its running maximum; lanes
// look for a larger score among their own first, so a tile without one takes no reduction over a row's lanes. (A reference that
// moves only past 2^8 saves another 0.9 us of 27.8, but then the largest weights are no longer 1, which a half holds
// exactly: 4 rows behind 43003 keys lay 2.7 % further from float64, 2 rows behind 100000 4.3 %.)
//
// Kernel and merge, before (a wave a SIMD) -> now, 24 / 4 heads behind 43003 q4_0 keys: one row 25.5 -> 20.6 us, 4 rows 35.4 ->
// 26.8, 8 rows 66.8 -> 48.4; 4 rows behind 20000 q8_0 keys 27.2 -> 22.8. Error against float64 as before (4 rows: relative
// 3.44e-4 against 3.46e-4).
template <int RT, int KT>
__global__ __launch_bounds__(512, 2) void attn_decode_q256_kernel(const DecodeParams p) {
    static_assert(KT == 1 || KT == 2, "quantized rows");
    constexpr int D = 256, KB = D / 32, DT = D / 16, W = 8;
    constexpr int QRB = KT == 1 ? D + D / 16 : D / 2 + D / 16;    // bytes a cache row
    constexpr int QVB = QRB - D / 16;                             // of them values
    // 16-byte chunks a row, as they lie (an odd number: 16 lanes a row each meet no bank conflict), a tile, its transfers
    constexpr int CH = QRB / 16, CN = TILE * CH, QRAW = CN * 16, NI = (CN + 63) / 64;
    static_assert(CH % 2 == 1 && CN % 64 == 32, "rows of 256 values; the last transfer instruction is half");
    constexpr bool TWO = KT == 2;                                 // raw keys and raw values have a buffer each
    constexpr int PARTS = 4, PDT = DT / PARTS, RS = PDT * 32 + 32, VTILE = TILE * RS;
    constexpr int CPP = QVB / 16 / PARTS, NL = TILE * CPP / 64;   // a part's chunks a row, and a lane
    constexpr int MERGE = DT * 1024;                              // (the merge takes a row tile at a time)
    constexpr int ATV = TWO ? QRAW : 0, ATW = ATV + QRAW, USED = ATW + VTILE;
    constexpr int WREG = ((USED > MERGE ? USED : MERGE) + 255) / 256 * 256;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[W * WREG];
    __shared__ s8v qs[RT * KB * 64];
    __shared__ __attribute__((aligned(16))) float ml[RT * 16][2][W];

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (split, key head, row chunk): as in attn_decode_kernel - of rows a gap apart (position-major) the key heads of one split take
    // consecutive places of ONE XCD instead (abreast): a row of 272 or 144 bytes ends within a line that the next head's row begins, and
    // that L2 then holds it for both. In the plain order they lie there only where the split count is a multiple of 8: behind
    // 90000 keys (59 splits) one row x 24 / 4 heads over q8_0 49.1 -> 42.1 us, over q4_0 36.8 -> 29.8, 4 rows 53.3 -> 46.7 and
    // 41.7 -> 39.3; behind 86000 (56 splits) unchanged
    const int xj = blockIdx.x / 8, u = (xj / p.nz) * 8 + (int) (blockIdx.x % 8), z = xj % p.nz;
    const int Hkv = p.Hq / p.G;
    const int split = p.abreast ? u / (8 * Hkv) * 8 + u % 8 : u % p.ns, hk = p.abreast ? u / 8 % Hkv : u / p.ns;
    if (split >= p.ns || hk >= Hkv) return;
    const int rows = p.T * p.G;
    const int64_t pass_end = p.p0 + p.T;
    const int64_t fmin = p.kfirst >= 0 ? p.kfirst : p.win > 0 ? std::max<int64_t>(0, p.p0 + 1 - p.win) : 0;
    const int64_t jb = std::max((p.sp0 + split) * p.kbs, fmin), je = std::min((p.sp0 + split + 1) * p.kbs, pass_end);
    const uint8_t* kbase = p.kc + (int64_t) hk * p.head_stride;
    const uint8_t* vbase = p.vc + (int64_t) hk * p.head_stride;
    uint8_t* const stage = lds + w * WREG;                        // [raw keys | raw values | 64 features' widened values]

    // a tile's raw rows on their way: a tile wholly inside the split whose slots follow each other is read at a wave-uniform
    // address - as one run of bytes where its rows are (head-major), else each row a gap further on (position-major) -; of any
    // other tile keys outside are clamped into the split (masked, or met by P = 0) and every lane works out its row's slot, a
    // wrapped ring's too. With two row tiles a lane's chunks are worked out anew each time, from a lane index whose origin the
    // compiler does not see: kept over the loop they are registers that form does not have, and a spilled address's way back
    // waits for every transfer under way. Kernel and merge where they were kept, and where only rows without a gap were read
    // at a uniform address -> now, 4 rows x 24 / 4 heads: behind 43003 q8_0 keys 36.9 -> 28.4 us, position-major 44.2 -> 29.8; q4_0
    // 27.2 -> 26.5 and 29.8 -> 27.2; 131000 q8_0 keys 70.4 -> 56.6 and 100.9 -> 61.6
    const int64_t jb_slot = p.wrap && jb < je ? jb % p.cap : jb;
    const int span = (int) (je - jb) - 1;
    // (a gap of 24 bits: what a lane's one multiplication takes. One row tile over q8_0 rows, which HBM bounds, keeps the lanes'
    // own addresses: its transfers then leave further apart in time, and one row x 24 / 4 heads behind 98000 keys takes 42.4 us
    // where a uniform address takes 43.9, behind 131000 53.7 and 55.6; over q4_0 rows 31.7 and 30.3 behind 98000)
    const int64_t gap64 = p.row_stride - QRB;
    const bool near = RT == 1 && KT == 1 ? gap64 == 0 : gap64 >= 0 && gap64 < 1 << 24;
    const uint32_t gap = (uint32_t) gap64;
    constexpr uint32_t RECIP = 65536 / CH + 1;                    // un / CH = un RECIP / 65536 over a tile's chunks
    static_assert(65536 % CH != 0 && (RECIP * CH - 65536) * NI * 64 < 65536, "the division by multiplication is exact");
    auto request = [&](int64_t ti, const uint8_t* cache, uint8_t* dst) __attribute__((always_inline)) {
        const int j0 = (int) (ti * TILE - jb);
        int64_t slot0 = jb_slot + j0;
        if (p.wrap) {
            slot0 = slot0 >= p.cap ? slot0 - p.cap : slot0;
            slot0 = slot0 >= p.cap ? slot0 - p.cap : slot0;
        }
        const bool whole = near && j0 >= 0 && j0 + TILE - 1 <= span && !(p.wrap && slot0 + TILE > p.cap);
        // (each half of the address through uint32_t: the builtin returns a signed int)
        const uint64_t base_v = (uint64_t) (uintptr_t) (cache + (whole ? slot0 * p.row_stride : 0));
        const uint8_t* const base = (const uint8_t*) (uintptr_t) ((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) base_v) |
                                                                  (uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (base_v >> 32)) << 32);
        const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t) (uintptr_t) dst);
        uint32_t l = lane;
        if constexpr (RT == 2) asm volatile("" : "+v"(l));
        if (whole) {
            uint32_t off[NI];                                     // (of `base` and the transfer's own KiB)
#pragma unroll
            for (int i = 0; i < NI; ++i) off[i] = l * 16;
            if (gap) {
#pragma unroll
                for (int i = 0; i < NI; ++i) off[i] += __umul24(__umul24(i * 64 + l, RECIP) >> 16, gap);
            }
            lds_fetch_run<true, NI - 1>(base, off, at);
            if (lane < 32) lds_fetch<true>(base + (NI - 1) * 1024, off[NI - 1], at + (NI - 1) * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const uint32_t un = i * 64 + l, row = __umul24(un, RECIP) >> 16;
                int64_t slot = jb_slot + std::min(std::max(j0 + (int) row, 0), span);
                if (p.wrap) {
                    slot = slot >= p.cap ? slot - p.cap : slot;
                    slot = slot >= p.cap ? slot - p.cap : slot;
                }
                if (i < NI - 1 || lane < 32) lds_fetch_any<true>(cache + slot * p.row_stride + (un - row * CH) * 16, at + i * 1024);
            }
        }
    };

    // the wave's tiles: absolute tile index % 8 == w, over [jb, je); the first is requested before anything else
    const int64_t tb = jb / TILE, te = jb < je ? (je + TILE - 1) / TILE : tb;
    const int64_t t0 = tb + ((w - (int) (tb % W) + W) % W);
    if (t0 < te) {
        request(t0, kbase, stage);
        if constexpr (TWO) request(t0, vbase, stage + ATV);
    }

    // ---- the queries as operands: k-block kb, lane l' = 16 g + n: 8 features of row n's block b = 4 (kb / 4) + g, with
    // j = kb % 4 - q8_0: 8 j .. 8 j + 7; q4_0: the nibbles of the block's bytes 4 j .. 4 j + 3 in the order dq4_word leaves
    // them: 4 j + {0, 2, 1, 3}, then 16 further on
    for (int e = tid; e < RT * KB * 64; e += W * 64) {
        const int rt = e / (KB * 64), kb = e / 64 % KB, ri = (z * RT + rt) * 16 + (e & 15);
        const bool live = ri < rows;
        const int t = live ? ri / p.G : 0, gq = live ? ri % p.G : 0;
        const int64_t at = (int64_t) t * p.qs + ((int64_t) hk * p.G + gq) * D + kb / 4 * 128 + (e >> 4 & 3) * 32 + kb % 4 * (KT == 1 ? 8 : 4);
        constexpr int second = KT == 1 ? 4 : 16;
        float f[8];
        if (p.qt == 0) {
            const float4 a = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.q) + at);
            const float4 b = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.q) + at + second);
            f[0] = a.x, f[1] = a.y, f[2] = a.z, f[3] = a.w, f[4] = b.x, f[5] = b.y, f[6] = b.z, f[7] = b.w;
        } else {
            const uint2 a = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p.q) + at);
            const uint2 b = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p.q) + at + second);
            const uint32_t ww[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint16_t b16 = (uint16_t) (ww[i >> 1] >> (16 * (i & 1)));
                f[i] = p.qt == 1 ? f16_to_f32(b16) : bf16_to_f32(b16);    // (a half is itself again below)
            }
        }
        s8v v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = live ? to16<false>(f[KT == 1 ? i : (i & 4) | ((i & 1) << 1) | ((i >> 1) & 1)]) : (short) 0;
        qs[e] = v;
    }
    // ---- this lane's rows (one per row tile): their key ranges
    int lo_r[RT], hi_r[RT];
    bool live_r[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int ri = (z * RT + rt) * 16 + n;
        const bool live = ri < rows;
        const int64_t pos = p.p0 + (live ? ri / p.G : 0), first = p.kfirst >= 0 ? p.kfirst : p.win > 0 ? std::max<int64_t>(0, pos + 1 - p.win) : 0;
        live_r[rt] = live;
        const int64_t hi64 = std::min(p.causal ? pos : pass_end - 1, je - 1);
        lo_r[rt] = live && hi64 >= jb ? (int) (std::max(first, jb) - jb) : 1;
        hi_r[rt] = live && hi64 >= jb ? (int) (hi64 - jb) : 0;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    float m_r[RT], l_r[RT];                                       // (l: this lane's share of the row's sum)
    f4v o[RT][DT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m_r[rt] = -INFINITY;
        l_r[rt] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[rt][dt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    }

    // the stage's pieces: a lane widens chunk lane % CPP (of the part's) of key lane / CPP, and - q8_0 - the same 16 keys on.
    // Pieces 0 and 2 go to w_even, 1 and 3 to w_odd: the two 16-byte pieces of every 32 bytes change places - q4_0: in the part's second chunk; q8_0: in keys 2, 3, 6, 7, .. -
    // so that the writes of 16 lanes meet nearly every bank once
    const int vkey = lane / CPP, vc = lane % CPP, vswap = (KT == 2 ? vc & 1 : (vkey >> 1) & 1) * 16;
    const uint32_t w_even = (uint32_t) (uintptr_t) (stage + ATW) + (uint32_t) (vkey * RS + vc * (KT == 1 ? 32 : 64) + vswap), w_odd = w_even + 16 - 2 * (uint32_t) vswap;
    const int kk = g4 * 4 + (n >> 2);
    const uint32_t tr_at = (uint32_t) (uintptr_t) (stage + ATW) + (uint32_t) (kk * RS);
    const uint32_t tr_lo = tr_at + (uint32_t) ((8 * (n & 3)) ^ (KT == 2 ? 0 : ((kk >> 1) & 1) * 16)), tr_hi = tr_at + (uint32_t) ((8 * (n & 3)) ^ 16);
    const uint32_t q_at = (uint32_t) (uintptr_t) qs + (uint32_t) lane * 16;
    for (int64_t ti = t0; ti < te; ti += W) {
        const bool next = ti + W < te;
        // ---- S^T = K Q^T (the values' transfers - q4_0 - may still be out)
        if constexpr (TWO) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        f4v s[RT][2];
        {
            constexpr int NW = KT == 1 ? 2 : 1;                   // 16-byte pieces of a block
            u4v raw[2][2][NW];
            uint32_t sc[2][2];
#pragma unroll
            for (int kt2 = 0; kt2 < 2; ++kt2) {
                const uint8_t* kr = stage + (kt2 * 16 + n) * QRB;
#pragma unroll
                for (int j2 = 0; j2 < 2; ++j2) {
#pragma unroll
                    for (int j = 0; j < NW; ++j) raw[kt2][j2][j] = *reinterpret_cast<const u4v*>(kr + ((4 * j2 + g4) * NW + j) * 16);
                    sc[kt2][j2] = *reinterpret_cast<const uint16_t*>(kr + QVB + 2 * (4 * j2 + g4));
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if constexpr (!TWO) request(ti, vbase, stage);
            else if (next) request(ti + W, kbase, stage);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s[rt][0] = s[rt][1] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
            // two k-blocks at a time: their queries requested, their keys widened meanwhile (written out: the compiler would read a
            // query operand, wait for it and use it, one after the other)
#pragma unroll
            for (int kb = 0; kb < KB; kb += 2) {
                s8v q[2][RT], ka[2][2];
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(q[j][rt]) : "v"(q_at), "n"((rt * KB + kb + j) * 1024));
#pragma unroll
                for (int kt2 = 0; kt2 < 2; ++kt2) {
                    const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t) sc[kt2][kb / 4]);
                    const u4v x = raw[kt2][kb / 4][NW == 2 ? kb / 2 % 2 : 0];
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        if constexpr (KT == 1) {
                            ka[kt2][j] = dq8x8(x[2 * j], x[2 * j + 1], d);
                        } else {
                            uint32_t y[4];
                            dq4_word(x[kb % 4 + j], d, y);
                            ka[kt2][j] = __builtin_bit_cast(s8v, u4v{y[0], y[1], y[2], y[3]});
                        }
                    }
                }
                if constexpr (RT == 2) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(q[0][0]), "+v"(q[0][RT - 1]), "+v"(q[1][0]), "+v"(q[1][RT - 1]));
                else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(q[0][0]), "+v"(q[1][0]));
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                        for (int kt2 = 0; kt2 < 2; ++kt2) s[rt][kt2] = mfma16<false>(ka[kt2][j], q[j][rt], s[rt][kt2]);
            }
        }
        // ---- online softmax a row (this lane: row n of each row tile, keys 16 kt2 + 4 g4 + i of the tile)
        const int j0r = (int) (ti * TILE - jb);
        int lo_t[RT];
        unsigned span_t[RT];
        bool edge = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int lo_ = std::min(std::max(lo_r[rt] - j0r, 0), 32);
            const int hi = std::min(std::max(hi_r[rt] - j0r, -1), 31);
            lo_t[rt] = hi < lo_ ? 64 : lo_;
            span_t[rt] = hi < lo_ ? 0u : (unsigned) (hi - lo_);
            edge |= live_r[rt] && (lo_ > 0 || hi < 31);
        }
        if (__any(edge)) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    s[rt][e >> 2][e & 3] = (unsigned) ((e >> 2) * 16 + g4 * 4 + (e & 3) - lo_t[rt]) <= span_t[rt] ? s[rt][e >> 2][e & 3] : -INFINITY;
        }
        float mx[RT];
        bool grow = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            mx[rt] = fmaxf(fmaxf(fmaxf(s[rt][0][0], s[rt][0][1]), fmaxf(s[rt][0][2], s[rt][0][3])), fmaxf(fmaxf(s[rt][1][0], s[rt][1][1]), fmaxf(s[rt][1][2], s[rt][1][3]))) * p.sl2;
            grow |= mx[rt] > m_r[rt];
        }
        if (__any(grow)) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float rmx = rows_max(mx[rt]);
                const float mn = rmx > m_r[rt] ? rmx : m_r[rt];
                const float c = mn == m_r[rt] ? 1.0f : fast_exp2(m_r[rt] - mn);
                m_r[rt] = mn;
                l_r[rt] *= c;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[rt][dt] *= c;
            }
        }
        s8v pb[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float ms = m_r[rt] == -INFINITY ? 0.0f : m_r[rt];      // (a row that has seen no key: weights 2^(-inf) = 0)
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pv = fast_exp2(fmaf(s[rt][e >> 2][e & 3], p.sl2, -ms));
                sum += pv;
                pb[rt][e] = to16<false>(pv);
            }
            l_r[rt] += sum;
        }
        // ---- O^T += V^T P^T (q4_0: the next tile's keys may still be out)
        if (TWO && next) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u4v raw[PARTS][NL];
        uint32_t sc[PARTS][NL];
#pragma unroll
        for (int part = 0; part < PARTS; ++part)
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const uint8_t* vr = stage + ATV + (vkey + 16 * i) * QRB;
                raw[part][i] = *reinterpret_cast<const u4v*>(vr + (part * CPP + vc) * 16);
                sc[part][i] = *reinterpret_cast<const uint16_t*>(vr + QVB + 2 * (KT == 1 ? part * 2 + vc / 2 : part * 2 + vc));
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (next) request(ti + W, TWO ? vbase : kbase, stage + ATV);
        // a part's writes, in assembly like the reads behind them: 4 of them, counted by the waits below (a wave's LDS operations
        // complete in order: a part may be written as soon as the reads of the one before have been requested)
        auto widen = [&](int part) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t) sc[part][i]);
                const u4v x = raw[part][i];
                if constexpr (KT == 1) {
                    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(w_even), "v"(dq8x8(x[0], x[1], d)), "n"(16 * i * RS) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(w_odd), "v"(dq8x8(x[2], x[3], d)), "n"(16 * i * RS) : "memory");
                } else {
                    uint32_t y[4][4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) dq4_word(x[j], d, y[j]);
                    // (positions 0 .. 3 of every 4 features hold features 0, 2, 1, 3: put right where the sums leave)
                    asm volatile("ds_write_b128 %0, %1" ::"v"(w_even), "v"(u4v{y[0][0], y[0][1], y[1][0], y[1][1]}) : "memory");
                    asm volatile("ds_write_b128 %0, %1" ::"v"(w_odd), "v"(u4v{y[2][0], y[2][1], y[3][0], y[3][1]}) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:32" ::"v"(w_even), "v"(u4v{y[0][2], y[0][3], y[1][2], y[1][3]}) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:32" ::"v"(w_odd), "v"(u4v{y[2][2], y[2][3], y[3][2], y[3][3]}) : "memory");
                }
            }
        };
        widen(0);
#pragma unroll
        for (int part = 0; part < PARTS; ++part) {
            s4v lo[PDT], hi[PDT];
#pragma unroll
            for (int d2 = 0; d2 < PDT; ++d2)
                asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
                             : "=&v"(lo[d2]), "=&v"(hi[d2]) : "v"(KT == 2 && d2 >= 2 ? tr_hi : tr_lo), "n"(d2 * 32), "n"(d2 * 32 + 16 * RS));
            if (part + 1 < PARTS) widen(part + 1);
#pragma unroll
            for (int d2 = 0; d2 < PDT; ++d2) {
                // reads return in order: the pairs behind this one and the next part's 4 writes may still be out
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo[d2]), "+v"(hi[d2]) : "n"(2 * (PDT - 1 - d2) + (part + 1 < PARTS ? 4 : 0)));
                const s8v va = {lo[d2][0], lo[d2][1], lo[d2][2], lo[d2][3], hi[d2][0], hi[d2][1], hi[d2][2], hi[d2][3]};
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) o[rt][part * PDT + d2] = mfma16<false>(va, pb[rt], o[rt][part * PDT + d2]);
            }
        }
        asm volatile("" ::: "memory");
    }

    // ---- the waves' (O, m, l) merged in wave order and written as the split's partial, a row tile at a time: a wave parks its
    // sums as they lie in its registers, then works out two of the 16 column tiles over all the waves, a lane the 4 features of
    // its own row again, whose place and weights it works out once (a thread a (row, 4 features) in row order: 27.2 us a pass of
    // 4 rows where this took 26.9, one row 20.9 and 20.2)
    const int live_rows = std::min(RT * 16, rows - z * RT * 16);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float lsum = rows_sum(l_r[rt]);
        if (g4 == 0) {
            ml[rt * 16 + n][0][w] = m_r[rt];
            ml[rt * 16 + n][1][w] = lsum;
        }
    }
    f4v* const park = reinterpret_cast<f4v*>(stage);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt) __syncthreads();
        const bool live = rt * 16 + n < live_rows;
        if (live) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) park[dt * 64 + lane] = o[rt][dt];
        }
        __syncthreads();
        if (live) {
            const int ri = (z * RT + rt) * 16 + n, t = ri / p.G, gq = ri % p.G;
            float* const part = p.part + (((int64_t) t * p.Hq + hk * p.G + gq) * p.ns + split) * (D + 2);
            float m[W], f[W], M = -INFINITY, L = 0.0f;
#pragma unroll
            for (int k = 0; k < W; ++k) m[k] = ml[rt * 16 + n][0][k];
#pragma unroll
            for (int k = 0; k < W; ++k) M = fmaxf(M, m[k]);
#pragma unroll
            for (int k = 0; k < W; ++k) {
                f[k] = m[k] == -INFINITY ? 0.0f : fast_exp2(m[k] - M);
                L += ml[rt * 16 + n][1][k] * f[k];
            }
#pragma unroll
            for (int i = 0; i < DT / W; ++i) {
                const int dt = (DT / W) * w + i;
                f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < W; ++k) acc += reinterpret_cast<const f4v*>(lds + k * WREG)[dt * 64 + lane] * f[k];
                // (q4_0: features 0, 2, 1, 3 of every 4; partial rows are D + 2 floats: 8-byte aligned)
                const int at = dt * 16 + g4 * 4;
                *reinterpret_cast<float2*>(part + at) = float2{acc[0], KT == 1 ? acc[1] : acc[2]};
                *reinterpret_cast<float2*>(part + at + 2) = float2{KT == 1 ? acc[2] : acc[1], acc[3]};
            }
            if (w == 0 && g4 == 0) *reinterpret_cast<float2*>(part + D) = float2{M, L};
        }
    }
}
