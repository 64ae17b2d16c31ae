// attn_prefill_wave.hpp: the body of the prompt kernel (attn_prefill.hip), included where D, BF, KT, PW, QS, NTS, FLAT, RT (a wave's row
// tiles of 16) and p are known: in the kernel itself, and in the function that a FLAT kernel's waves call for one tile or two. (All of it
// as a function, the kernels that hold whole waves of one head's rows came out with another schedule: q4_0 rows of 128, 19 rows x 64
// / 4 heads behind 3316 keys 22.9 -> 23.4 us, 25 x 32 / 8 behind 30842 36.2 -> 37.4.)
    static_assert(D == 128 || D == 256, "head size 128 or 256");
    static_assert(KT == 0 || !BF, "quantized rows are widened to half");
    static_assert(!QS || BF, "query rows in two parts: bfloat16 operands only");
    constexpr int WROWS = RT * 16;
    constexpr int KB = D / 32, DT = D / 16;
    // Half operands: the query enters the first product scaled by the softmax scale x log2 e and rounded once to half - what
    // the reference's kernels do (qwen35/silo/attn.cpp:112,147: qh = half(q x qscale)) - and the product starts from minus
    // the softmax reference (ntile), so a score leaves the matrix unit as the argument of its exponential: no vector
    // instruction a score between the two. bfloat16 operands (8 bits: a second rounding would show) keep the scale in a
    // fused multiply-add a score.
    constexpr bool PRESCALE = !BF;
    constexpr int KS = padded_row(D), VS = padded_row(D);
    constexpr int KBUF = KT_TILE * KS, VBUF = KT_TILE * VS;
    // DMA: 8 waves over 16-bit rows of 128 stage their tiles global -> LDS directly (global_load_lds_dwordx4: no register in
    // between, no LDS write instruction, a tile requested two tiles ahead). The tiles are unpadded 256-byte rows, a row's
    // 16-byte chunks exclusive-ored into place by its key (keys: chunk c of key r at position c ^ (r % 16); values:
    // c ^ 2 (r % 8)) so that neither the operand reads of 16 keys' same chunk nor the transposing reads meet a bank
    // conflict; three buffers a stream, each an array of its own so that the compiler can tell a transfer's target from
    // the arrays being read (it waits for every transfer in flight before a read it cannot tell apart)
    // The 4-wave form (two work-groups a CU) has LDS for two buffers a stream: a tile is then requested one tile ahead,
    // right behind the barrier that frees its buffer, and the next barrier waits for every transfer of the wave.
    constexpr bool DMA = by_dma(D, KT, PW);
    constexpr int NBUF = tile_bufs(PW);
    constexpr int NJ = 16 / PW;                                   // transfer instructions a wave, tile and stream
    constexpr int TB = KT_TILE * 256;

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // ---- which (row block, head) this work-group owns. Consecutive work-group ids go round the 8 XCDs (each with its
    // own L2). The G query heads of one key head on one row block stream the same K / V tiles: they are one unit, and a
    // unit's work-groups are consecutive on one XCD. Units are dealt to the XCDs round-robin in order of weight (the last
    // row block sees the most keys), so every XCD gets the same mix of heavy and light units, heaviest first. The grid is
    // padded to a multiple of 8 units; the work-groups of the padding leave at once.
    const int pid = blockIdx.x, xcd = pid % 8, xi = pid / 8;
    const int pk = p.pack, wh = w % pk, wr = w / pk;              // (scalars: this wave's head of the work-group's, its rows' place)
    const int wslots = PW / pk;                                   // waves a head (a wave past pk x wslots has no rows: 5 heads to 8 waves)
    const int RB = wslots * WROWS;                                // rows of a head a work-group holds
    // (FLAT: pair r of a key head is row r / G, head r % G of its group)
    const int pairs = p.T * p.G;
    auto row_of = [&](int pair) { return p.G == 1 ? pair : (int) __umulhi((uint32_t) pair, p.ginv); };
    const int nblk = FLAT ? ((pairs + 15) / 16 + p.tb - 1) / p.tb : (p.T + RB - 1) / RB;
    const int Hkv = p.Hq / p.G;
    // (with key splits a split is one more factor of the units, the slowest: a pass of fewer than 8 units still puts work on
    // every XCD, and a unit's splits - different keys - go to different ones)
    // (FLAT: a unit is a group of a key head's row blocks over a split of its keys; the first nfull units are blocks over all of them)
    const int nfull = FLAT ? p.nbf * Hkv : 0;
    const int u2 = (xi / (FLAT ? p.gb : p.gw)) * 8 + xcd - nfull;
    const int nun = FLAT ? p.ngb * Hkv - nfull : nblk * Hkv;
    if (u2 >= nun * p.ns) return;
    const bool whole = FLAT && u2 < 0;
    const int unit = whole ? u2 + nfull : u2 % nun + nfull;
    const int hk = unit % Hkv;
    const int hq = hk * p.G + (xi % p.gw) * pk + wh;
    const int blk = nblk - 1 - (FLAT ? unit / Hkv * p.gb + xi % p.gb : unit / Hkv);
    if (FLAT && blk < 0) return;
    const int tile0 = FLAT ? blk * p.tb : 0;                      // (FLAT: the block's first row tile)
    const int r0 = FLAT ? row_of(tile0 * 16) : blk * RB;
    const int rl = FLAT ? row_of(std::min((tile0 + p.tb) * 16, pairs) - 1) : std::min(r0 + RB, p.T) - 1;   // the block's last row
    // this wave's first row, or pair (none: past the pass's last), and the end of what there is
    const bool idle = FLAT && RT == 1 && wave_tiles(w, flat_tiles(p, tile0), PW) == 0;
    const int wbase = idle ? pairs : FLAT ? (tile0 + wave_tile0(w, flat_tiles(p, tile0), PW)) * 16 : wr < wslots ? r0 + wr * WROWS : p.T;
    const int wend = FLAT ? pairs : p.T;
    // keys [kbeg, kend) cover every row of the block; with key splits, the part of them in this work-group's split
    const int split = whole ? 0 : u2 / nun;
    int64_t kend = p.causal ? p.p0 + rl + 1 : p.p0 + p.T;
    int64_t kbeg = p.kfirst >= 0 ? p.kfirst : p.win > 0 ? std::max<int64_t>(0, p.p0 + r0 + 1 - p.win) : 0;
    if (p.ns > 1 && !whole) {
        kbeg = std::max(kbeg, p.k0 + split * p.kbs);
        kend = std::max(kbeg, std::min(kend, p.k0 + (split + 1) * p.kbs));      // (none: an empty range at kbeg)
    }

    // ---- this lane's two rows: positions, key ranges, Q^T operands
    int64_t lo_r[RT], hi_r[RT];
    s8v qreg[RT][KB], qlo[QS ? RT : 1][KB];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int place = wbase + rt * 16 + n;
        const bool live = place < wend;
        const int rr = !live ? p.T - 1 : FLAT ? row_of(place) : place;
        const int64_t pos = p.p0 + rr;
        lo_r[rt] = live ? std::max(kbeg, p.kfirst >= 0 ? p.kfirst : p.win > 0 ? std::max<int64_t>(0, pos + 1 - p.win) : 0) : 1;
        hi_r[rt] = live ? std::min(p.causal ? pos : p.p0 + p.T - 1, kend - 1) : 0;
        const int64_t qoff = (int64_t) rr * p.qs + (int64_t) (FLAT ? hk * p.G + (live ? place - rr * p.G : 0) : hq) * D + g4 * 8;
        if (p.qt == 0) {
            float4 raw[KB][2];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                raw[kb][0] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.q) + qoff + kb * 32);
                raw[kb][1] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.q) + qoff + kb * 32 + 4);
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const float f[8] = {raw[kb][0].x, raw[kb][0].y, raw[kb][0].z, raw[kb][0].w, raw[kb][1].x, raw[kb][1].y, raw[kb][1].z, raw[kb][1].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    qreg[rt][kb][i] = to16<BF>(PRESCALE ? f[i] * p.sl2 : f[i]);
                    if constexpr (QS) qlo[rt][kb][i] = to16<true>(f[i] - bf16_to_f32((uint16_t) qreg[rt][kb][i]));
                }
            }
        } else {
            uint4 raw[KB];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) raw[kb] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.q) + qoff + kb * 32);
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const uint32_t ww[4] = {raw[kb].x, raw[kb].y, raw[kb].z, raw[kb].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint16_t b16 = (uint16_t) (ww[i >> 1] >> (16 * (i & 1)));
                    // bfloat16 operands: rows of that type pass through bit for bit, others are rounded once; half operands:
                    // the row x the scale, rounded once
                    if constexpr (PRESCALE) qreg[rt][kb][i] = to16<BF>((p.qt == 1 ? f16_to_f32(b16) : bf16_to_f32(b16)) * p.sl2);
                    else qreg[rt][kb][i] = (p.qt == 2) == BF ? (short) b16 : to16<BF>(p.qt == 1 ? f16_to_f32(b16) : bf16_to_f32(b16));
                    if constexpr (QS) qlo[rt][kb][i] = p.qt == 1 ? to16<true>(f16_to_f32(b16) - bf16_to_f32((uint16_t) qreg[rt][kb][i])) : (short) 0;
                }
            }
        }
    }
    const uint8_t* kbase = p.kc + (int64_t) hk * p.head_stride;
    const uint8_t* vbase = p.vc + (int64_t) hk * p.head_stride;
    const int64_t t0 = kbeg / KT_TILE, t1 = (kend + KT_TILE - 1) / KT_TILE;
    const int nt = kend > kbeg ? (int) (t1 - t0) : 0;             // (a split past the block's last key: nothing to do)
    // From here on keys are counted from the first tile's first key (32-bit): tile k holds keys 64 k .. 64 k + 63, step
    // s = 2 k + h its 32-key half h
    const int64_t base = t0 * KT_TILE;
    int lo32[RT], hi32[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const bool live = wbase + rt * 16 + n < wend;
        lo32[rt] = live ? (int) (lo_r[rt] - base) : 1;
        hi32[rt] = live ? (int) (hi_r[rt] - base) : 0;
    }
    // the wave's own steps: from its first row's first key to its last row's last; steps in between that no row's edge
    // crosses need no mask
    const int wrow0 = FLAT ? row_of(std::min(wbase, pairs - 1)) : wbase;
    const int wrow1 = FLAT ? row_of(std::min(wbase + WROWS, pairs) - 1) : std::min(wrow0 + WROWS - 1, p.T - 1);
    const int w_full_end = (int) ((p.causal ? p.p0 + wrow0 + 1 : p.p0 + p.T) - base);
    const int w_full_beg = p.kfirst >= 0 ? (int) (p.kfirst - base) : p.win > 0 ? (int) (std::max<int64_t>(0, p.p0 + wrow1 + 1 - p.win) - base) : 0;

    // Online softmax state, in base-2 exponent units (scores x scale x log2 e): nbr = minus the reference the weights
    // are taken against, thr = how far a score may exceed it before the reference moves (-inf while the row has seen no
    // key: the first one sets it). The row's sum of weights l4 comes out of the matrix unit: a product of the rounded weights
    // with an operand of ones beside each step's V^T P^T (every slot of l4 then holds the whole row's sum - no vector
    // additions, no cross-lane step, and numerator and denominator carry the very same rounded weights)
    float nbr[RT], thr[RT];
    f4v l4[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        nbr[rt] = 0.0f;
        thr[rt] = -INFINITY;
        l4[rt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    f4v o[RT][DT], ntile[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        ntile[rt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[rt][dt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    }

    // ---- global -> registers -> LDS. A cache row is fetched in 16-byte raw chunks: 16-bit rows D / 8 of them, each one
    // LDS piece; q8_0 rows D / 16 (16 int8 -> 2 pieces of 8 halfs, the block's half scale fetched beside it); q4_0 rows
    // D / 32 (one block: 32 nibbles -> 4 pieces). A thread's chunks of a tile: chunk c = tid + 256 i -> key c / CPR, raw
    // chunk c % CPR. A tile wholly inside [kbeg, kend) of an unwrapped cache is read at a wave-uniform address plus a
    // 32-bit lane offset; otherwise keys outside are clamped into the range (a valid row, masked; a tile past the last
    // is fetched as the last row over and over and never used) and a wrapped ring's slot is position % cap: the first
    // key's once, then offsets from it with at most two wraps (a pass's keys span less than two rings)
    // (8 waves over q4_0 rows of 128 have two threads a block: chunks of 8 bytes, 8 low nibbles and 8 high ones)
    constexpr bool HALF = KT == 2 && D == 128 && PW == 8;
    constexpr int CPR = KT == 0 ? D / 8 : KT == 1 || HALF ? D / 16 : D / 32;      // raw chunks a row
    constexpr int NST = KT_TILE * CPR / (PW * 64);                                // raw chunks a thread per tile
    constexpr int KPI = PW * 64 / CPR;                                            // keys between a thread's chunks
    constexpr int PPC = KT == 0 ? 1 : KT == 1 ? 2 : 4;                            // LDS pieces a raw chunk
    static_assert(NST >= 1 && NST * PW * 64 == KT_TILE * CPR, "whole chunks a thread");
    struct Stage {
        u4v raw[NST];
        uint16_t sc[KT == 0 ? 1 : NST];
    };
    const int64_t kbeg_slot = p.wrap ? kbeg % p.cap : kbeg;
    const int kspan = (int) (kend - kbeg) - 1;
    const int kbeg32 = (int) (kbeg - base);
    const int key0 = tid / CPR, rc = tid % CPR;                   // chunk i of this thread: key key0 + KPI i, raw chunk rc
    constexpr int CB = HALF ? 8 : 16;                             // bytes a chunk
    const uint32_t lane_off = (uint32_t) (key0 * p.row_stride) + (uint32_t) rc * CB;
    // where a chunk's scale sits in its row: q8_0 a half a block of 32 behind D values, q4_0 behind D / 2 bytes
    // (as a distance from the chunk itself)
    const uint32_t sc_rel = (KT == 1 ? (uint32_t) (D + 2 * (rc / 2)) : (uint32_t) (D / 2 + 2 * (HALF ? rc / 2 : rc))) - (uint32_t) rc * CB;
    // tiles seg0 .. seg1 hold keys in range only, in slots seg_base + 64 krel and on: the whole tiles of an unwrapped cache; of a
    // ring those of one lap, and the next lap's once a tile of it has been fetched a lane at a time (seam), so that only the
    // tiles about a ring's end are: 2001 rows x 32 / 2 heads, window 1024, behind 10007 keys 53.1 -> 50.3 us, 129 x 16 / 2,
    // window 4096, 37.8 -> 33.3. (Direct transfers only: the fetch through registers keeps lane addresses for a wrapped ring -
    // it gained 1 - 4 % there and lost 1 - 2 % on unwrapped caches)
    const int plain1 = p.wrap && !DMA ? -1 : (int) ((kend - base) / KT_TILE) - 1;
    int64_t seg_base = DMA ? kbeg_slot - kbeg32 : base;
    int seg0 = kbeg32 > 0 ? 1 : 0, seg1 = DMA && p.wrap ? (int) std::min<int64_t>(plain1, (p.cap - seg_base) / KT_TILE - 1) : plain1;
    auto seam = [&](int krel) __attribute__((always_inline)) {
        if (p.wrap && krel > seg1 && krel <= plain1 && seg_base - p.cap + (int64_t) krel * KT_TILE >= 0) {
            seg_base -= p.cap;
            seg0 = krel;
            seg1 = (int) std::min<int64_t>(plain1, (p.cap - seg_base) / KT_TILE - 1);
        }
    };
    auto fetch = [&](Stage& st, const uint8_t* cache, int krel) {
        const int64_t rs = p.row_stride;
        const bool wrap = p.wrap;
        const uint8_t* sp = cache;
        uint32_t off[NST];                                        // of the raw chunk
        if (krel >= seg0 && krel <= seg1) {
            sp += (base + (int64_t) krel * KT_TILE) * rs;
#pragma unroll
            for (int i = 0; i < NST; ++i) off[i] = lane_off + (uint32_t) (i * KPI * rs);
        } else {
            const int rel0 = krel * KT_TILE - kbeg32 + key0;
#pragma unroll
            for (int i = 0; i < NST; ++i) {
                const int rel = std::min(std::max(rel0 + KPI * i, 0), kspan);
                int64_t slot = kbeg_slot + rel;
                if (wrap) {
                    slot = slot >= p.cap ? slot - p.cap : slot;
                    slot = slot >= p.cap ? slot - p.cap : slot;
                }
                off[i] = (uint32_t) (slot * rs) + (uint32_t) rc * CB;   // a head's cache spans less than 4 GiB
            }
        }
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            if constexpr (HALF) {
                const uint2 x = *reinterpret_cast<const uint2*>(sp + off[i]);
                st.raw[i][0] = x.x;
                st.raw[i][1] = x.y;
            } else if constexpr (KT != 0 && D == 128) st.raw[i] = *reinterpret_cast<const u4a8*>(sp + off[i]);
            else st.raw[i] = *reinterpret_cast<const u4v*>(sp + off[i]);
            if constexpr (KT != 0) st.sc[i] = *reinterpret_cast<const uint16_t*>(sp + off[i] + sc_rel);
        }
    };
    lds_u8* const L = tile_lds<D, KT, PW, 0>();
    // LDS map: K tiles at 0 and KBUF, V tiles at 2 KBUF and 2 KBUF + VBUF; rows of D halfs (+ padding) whatever the cache
    constexpr uint32_t V0 = 2 * KBUF;
    // a raw chunk's pieces written at row stride RS from byte offset at (quantized rows widened: one rounding to half of
    // (float) q x (float) scale, what the reference stages - qwen35/silo/attn.cpp:56-76)
    const uint32_t row_wr = HALF ? rc / 2 * 64 + rc % 2 * 16 : rc * 16 * PPC;
    const uint32_t k_wr = (uint32_t) (key0 * KS) + row_wr, v_wr = (uint32_t) (key0 * VS) + row_wr;
    auto put = [&](const Stage& st, uint32_t at0, int RS) {
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const uint32_t at = at0 + (uint32_t) (i * KPI * RS);
            if constexpr (KT == 0) {
                *reinterpret_cast<__attribute__((address_space(3))) u4v*>(L + at) = st.raw[i];
            } else {
                const _Float16 d = __builtin_bit_cast(_Float16, st.sc[i]);
                if constexpr (KT == 1) {
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at) = dq8x8(st.raw[i][0], st.raw[i][1], d);
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at + 16) = dq8x8(st.raw[i][2], st.raw[i][3], d);
                } else if constexpr (HALF) {
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at) = dq4x8(st.raw[i][0], st.raw[i][1], 0, d);
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at + 32) = dq4x8(st.raw[i][0], st.raw[i][1], 4, d);
                } else {
                    // values 0 .. 15: the low nibbles of the 16 bytes, 16 .. 31: the high ones
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at) = dq4x8(st.raw[i][0], st.raw[i][1], 0, d);
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at + 16) = dq4x8(st.raw[i][2], st.raw[i][3], 0, d);
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at + 32) = dq4x8(st.raw[i][0], st.raw[i][1], 4, d);
                    *reinterpret_cast<__attribute__((address_space(3))) s8v*>(L + at + 48) = dq4x8(st.raw[i][2], st.raw[i][3], 4, d);
                }
            }
        }
    };
    auto stash_k = [&](const Stage& st, int buf) { put(st, (uint32_t) (buf * KBUF) + k_wr, KS); };
    auto stash_v = [&](const Stage& st, int buf) { put(st, V0 + (uint32_t) (buf * VBUF) + v_wr, VS); };

    // DMA: a wave's two 1 KiB instructions a tile and stream: instruction j fills rows 4 (2 w + j) .. + 3 of the tile (16
    // lanes a row: lane l position l % 16 of row 4 (2 w + j) + l / 16), so it fetches the chunk that belongs there. Whole
    // tiles of an unwrapped cache: a wave-uniform tile address plus lane offsets worked out once (less the KiB by which the
    // instructions of a group move the address themselves, from a base as much lower); else the row is clamped
    // into the pass's keys (masked anyway) and a ring's slot worked out, as the register path does
    uint32_t koff[DMA ? NJ : 1], voff[DMA ? NJ : 1];
    if constexpr (DMA) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int r = (w * NJ + j) * 4 + (lane >> 4), cp = lane & 15;
            koff[j] = (uint32_t) (r * p.row_stride) + (uint32_t) ((cp ^ (r & 15)) << 4) + (NJ - 1 - j) * 1024;
            voff[j] = (uint32_t) (r * p.row_stride) + (uint32_t) ((cp ^ (2 * (r & 7))) << 4) + (NJ - 1 - j) * 1024;
        }
    }
    auto dma = [&](lds_u8* dst, const uint8_t* cache, int krel, auto which_c) __attribute__((always_inline)) {
        constexpr bool VAL = decltype(which_c)::value;
        const int64_t rs = p.row_stride;
        const bool wrap = p.wrap;
        const uint32_t lds_at = __builtin_amdgcn_readfirstlane((uint32_t) (uintptr_t) dst);
        if (krel >= seg0 && krel <= seg1) {
            const uint8_t* sp = cache + (seg_base + (int64_t) krel * KT_TILE) * rs - (NJ - 1) * 1024;
            lds_fetch_run<NTS, NJ>(sp, VAL ? voff : koff, lds_at + (uint32_t) (w * NJ) * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int r = (w * NJ + j) * 4 + (lane >> 4), cp = lane & 15;
                const int rel = std::min(std::max(krel * KT_TILE - kbeg32 + r, 0), kspan);
                int64_t slot = kbeg_slot + rel;
                if (wrap) {
                    slot = slot >= p.cap ? slot - p.cap : slot;
                    slot = slot >= p.cap ? slot - p.cap : slot;
                }
                const uint32_t off = (uint32_t) (slot * rs) + (uint32_t) ((VAL ? cp ^ (2 * (r & 7)) : cp ^ (r & 15)) << 4);
                lds_fetch<NTS>(cache, off, lds_at + (uint32_t) (w * NJ + j) * 1024);
            }
            seam(krel);
        }
    };
    // a tile's barrier. DMA: this wave's transfers of the tile about to be read are done when at most the two younger
    // requests (2 instructions each) are still in flight, and every LDS read it has issued has returned (a wave past the
    // barrier may request a transfer into a buffer this wave read from); a bare barrier then - no fence over the
    // transfers still in flight
    auto tile_barrier = [&]() __attribute__((always_inline)) {
        if constexpr (DMA) {
            if constexpr (NBUF == 3) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else {
            __syncthreads();
        }
    };
    const uint32_t k_rd = (uint32_t) (n * KS + g4 * 16);                          // + kt2 * 16 * KS + kb * 64
    const uint32_t v_rd = (uint32_t) ((g4 * 4 + (n >> 2)) * VS + (n & 3) * 8);    // + dt * 32 (+ 16 * VS)
    // (DMA tiles: where the lane's key-operand chunk kb and value-operand column tile dt sit in their swizzled rows)
    uint32_t k_rd4[DMA ? KB : 1], v_rd8[DMA ? DT : 1];
    if constexpr (DMA) {
        const int kkv = g4 * 4 + (n >> 2);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) k_rd4[kb] = (uint32_t) (n * 256 + (((kb * 4 + g4) ^ n) << 4));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) v_rd8[dt] = (uint32_t) (kkv * 256 + ((dt ^ (kkv & 7)) << 5) + (((n & 3) >> 1) << 4) + (n & 1) * 8);
    }
    // (bfloat16 operands: a weight enters the second product as two bfloat16 numbers, the rounded weight pb and the rounded
    // rest pl - 16 significant bits between them, where one alone would carry 8 and cost the output ~1.6e-3 of relative L2)
    s8v pb[RT], pl[BF ? RT : 1];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) pb[rt] = s8v{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int rt = 0; rt < (BF ? RT : 1); ++rt) pl[rt] = s8v{0, 0, 0, 0, 0, 0, 0, 0};
    // S^T of one 32-key half (LDS byte offset kl) against the wave's 32 rows: the raw dot products
    // (the operands of a block's first matrix instructions are read a block earlier - kread / vread - so that their LDS
    // latency passes under the other block's work instead of at the head of this one)
    // (rows in two parts: the registers of half the value operands read ahead go to the rows' second part - no spills)
    constexpr int VPRE = D == 128 && !QS ? DT : 4;                // value operands read ahead
    constexpr int KPRE = D == 128 ? 2 : 1;                        // 16-key halves whose key operands are read ahead
    auto kread = [&](s8v (&ka)[KPRE][KB], const lds_u8* kl) __attribute__((always_inline)) {
#pragma unroll
        for (int kt2 = 0; kt2 < KPRE; ++kt2)
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                if constexpr (DMA) ka[kt2][kb] = *reinterpret_cast<const __attribute__((address_space(3))) s8v*>(kl + k_rd4[kb] + kt2 * 16 * 256);
                else ka[kt2][kb] = *reinterpret_cast<const __attribute__((address_space(3))) s8v*>(kl + k_rd + kt2 * 16 * KS + kb * 64);
            }
    };
    auto vread1 = [&](const lds_u8* vl, int dt) __attribute__((always_inline)) {
        if constexpr (DMA) {
            const s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*) (vl + v_rd8[dt]));
            const s4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*) (vl + v_rd8[dt] + 16 * 256));
            return s8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            const s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*) (vl + v_rd + dt * 32));
            const s4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*) (vl + v_rd + dt * 32 + 16 * VS));
            return s8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
    };
    auto vread = [&](s8v (&va)[VPRE], const lds_u8* vl) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < VPRE; ++dt) va[dt] = vread1(vl, dt);
    };
    auto scores = [&](f4v (&s)[RT][2], const lds_u8* kl, const s8v (&kpre)[KPRE][KB]) __attribute__((always_inline)) {
        if constexpr (KPRE == 2) {
            // every operand is in registers: the 2 RT chains of dependent products advance side by side
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int kt2 = 0; kt2 < 2; ++kt2)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                    {
                        s[rt][kt2] = mfma16<BF>(kpre[kt2][kb], qreg[rt][kb], kb == 0 ? ntile[rt] : s[rt][kt2]);
                        if constexpr (QS) s[rt][kt2] = mfma16<BF>(kpre[kt2][kb], qlo[rt][kb], s[rt][kt2]);
                    }
        } else {
#pragma unroll
            for (int kt2 = 0; kt2 < 2; ++kt2) {
                s8v ka[KB];
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
                    ka[kb] = kt2 == 0 ? kpre[0][kb] : *reinterpret_cast<const __attribute__((address_space(3))) s8v*>(kl + k_rd + kt2 * 16 * KS + kb * 64);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    f4v acc = mfma16<BF>(ka[0], qreg[rt][0], ntile[rt]);
#pragma unroll
                    for (int kb = 1; kb < KB; ++kb) acc = mfma16<BF>(ka[kb], qreg[rt][kb], acc);
                    if constexpr (QS) {
#pragma unroll
                        for (int kb = 0; kb < KB; ++kb) acc = mfma16<BF>(ka[kb], qlo[rt][kb], acc);
                    }
                    s[rt][kt2] = acc;
                }
            }
        }
    };
    // O^T += V^T P^T of one 32-key half (LDS byte offset vl) with the weights in pb
    constexpr short ONE16 = BF ? (short) 0x3F80 : (short) 0x3C00;
    const s8v ones = {ONE16, ONE16, ONE16, ONE16, ONE16, ONE16, ONE16, ONE16};
    auto weigh = [&](const lds_u8* vl, const s8v (&vpre)[VPRE]) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            l4[rt] = mfma16<BF>(ones, pb[rt], l4[rt]);
            if constexpr (BF) l4[rt] = mfma16<BF>(ones, pl[rt], l4[rt]);
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const s8v va = dt < VPRE ? vpre[dt] : vread1(vl, dt);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                o[rt][dt] = mfma16<BF>(va, pb[rt], o[rt][dt]);
                if constexpr (BF) o[rt][dt] = mfma16<BF>(va, pl[rt], o[rt][dt]);
            }
        }
    };
    // One step of the wave's software pipeline. Step s holds the scores of its own half in sc (computed a step earlier)
    // and runs, as two straight-line blocks in which matrix and vector work are independent and overlap:
    //   A: O^T += V^T P^T of step s - 1   ||   exponent arguments of step s against the reference as it stands, and
    //      this lane's largest
    //   (only if some row's score outgrew its reference by more than 2^8: move the references, rescale; the weights may
    //    otherwise exceed 1, by at most 2^8: harmless in float32 sums and 16-bit operands, and the final division by
    //    the row's sum makes the result the same function of the inputs)
    //   B: S^T of step s + 1              ||   weights of step s = exp2(arguments), rounded to 16 bit
    // Every LDS operand of a block is requested a block ahead (vread at the step's start, kread at the head of A), and
    // sched_group_barrier deals the vector instructions out between the matrix instructions.
    // The mask is applied under a wave-uniform branch: steps no row's causal or window edge crosses pay no comparison.
    auto step = [&](f4v (&sc)[RT][2], f4v (&sn)[RT][2], const lds_u8* kl_next, const lds_u8* vl_prev, int j0, bool masked, bool bar_mid = false) __attribute__((always_inline)) {
        if (FLAT && RT == 1 && idle) {                            // (a wave without rows only stages its share of the tiles)
            if (bar_mid) tile_barrier();
            return;
        }
        float a[RT][8], amax[RT];
        s8v vpre[VPRE], kpre[KPRE][KB];
        vread(vpre, vl_prev);
        // (the mask goes onto the raw scores: minus infinity stays minus infinity under the positive scale)
        if (masked) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                // keys lo .. hi of this half (relative, clamped into 0 .. 32 / -1 .. 31) are the row's: one unsigned
                // compare a key (no key at all: lo = 64 puts every key below it)
                const int lo_ = std::min(std::max(lo32[rt] - j0, 0), 32);
                const int hi = std::min(std::max(hi32[rt] - j0, -1), 31);
                const int lo = hi < lo_ ? 64 : lo_;
                const unsigned span = hi < lo_ ? 0u : (unsigned) (hi - lo_);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int j = (e >> 2) * 16 + g4 * 4 + (e & 3);
                    sc[rt][e >> 2][e & 3] = (unsigned) (j - lo) <= span ? sc[rt][e >> 2][e & 3] : -INFINITY;
                }
            }
        }
        __builtin_amdgcn_s_setprio(1);
        kread(kpre, kl_next);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 8; ++e) a[rt][e] = PRESCALE ? sc[rt][e >> 2][e & 3] : __builtin_fmaf(sc[rt][e >> 2][e & 3], p.sl2, nbr[rt]);
        weigh(vl_prev, vpre);
        bool grow = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            // (the first maximum as the compiler's own instruction where its schedule is none the worse for it: one instruction less,
            // 512 float32 rows x 32 / 8 heads behind 20000 bfloat16 keys in their own form 253.8 -> 248.1 us)
            if constexpr (PRESCALE) amax[rt] = max3f(max3f(max3f(max3f(a[rt][0], a[rt][1], a[rt][2]), a[rt][3], a[rt][4]), a[rt][5], a[rt][6]), a[rt][7], a[rt][7]);
            else amax[rt] = max3f(max3f(max3f(fmaxf(a[rt][0], a[rt][1]), a[rt][2], a[rt][3]), a[rt][4], a[rt][5]), a[rt][6], a[rt][7]);
            grow |= amax[rt] > thr[rt];
        }
        if constexpr (D == 128) {
            // the matrix instructions of this block with two vector instructions between each
#pragma unroll
            for (int i = 0; i < (BF ? 2 : 1) * (RT * DT + RT); ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, PRESCALE ? 1 : 2, 0);
            }
        }
        if (bar_mid) tile_barrier();
        if (__any(grow)) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float mx = rows_max(amax[rt]);
                const bool fresh = thr[rt] < 0.0f;
                const bool nokey = mx == -INFINITY;
                const float delta = fresh ? (nokey ? 0.0f : mx) : fmaxf(mx, 0.0f);
                const float c = fresh ? 1.0f : fast_exp2(-delta);
                l4[rt] *= c;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[rt][dt] *= c;
                nbr[rt] -= delta;
                if constexpr (PRESCALE) ntile[rt] = f4v{nbr[rt], nbr[rt], nbr[rt], nbr[rt]};
#pragma unroll
                for (int e = 0; e < 8; ++e) a[rt][e] -= delta;
                // (end to end under a window a wave's few rows begin at one key half, whose maximum would stay their reference; 32 rows of one head
                // begin at two. With the second half's too, the largest weights are 1 - a half as it is - as often as there: 2001 x 32 / 2, window
                // 1024, 2.969e-4 of relative L2 from float64 in whole waves of a head, 2.971e-4 end to end, 2.961e-4 so, for 0.1 of 43.2 us)
                thr[rt] = fresh && nokey ? -INFINITY : FLAT && PRESCALE && fresh && p.win > 0 ? 0.0f : 8.0f;
            }
        }
        scores(sn, kl_next, kpre);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pv = fast_exp2(a[rt][e]);                                   // -inf -> 0
                pb[rt][e] = to16<BF>(pv);
                if constexpr (BF) pl[rt][e] = to16<BF>(pv - __builtin_bit_cast(float, (uint32_t) (uint16_t) pb[rt][e] << 16));
            }
        }
        if constexpr (D == 128) {
            // a matrix instruction, an exponential, and a conversion after every other
#pragma unroll
            for (int i = 0; i < RT * 2 * KB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
                if (i & 1) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
            }
        }
        // the step's results are complete here, in program order: nothing of it drifts past the next barrier or branch
        if constexpr (RT == 2) asm volatile("" : "+v"(pb[0]), "+v"(pb[1]));
        else asm volatile("" : "+v"(pb[0]));
        if constexpr (BF && RT == 2) asm volatile("" : "+v"(pl[0]), "+v"(pl[1]));
        else if constexpr (BF) asm volatile("" : "+v"(pl[0]));
        __builtin_amdgcn_s_setprio(0);
    };

    // ---- the pipeline over tiles. K and V tiles have two LDS buffers each (tile k in buffer k & 1) and one register
    // set each; one barrier a tile, between its two steps:
    //   step 2k   : K(k+1) registers -> LDS, fetch K(k+2); A reads V(k-1) half 1, B reads K(k) half 1
    //   barrier
    //   step 2k+1 : V(k+1) registers -> LDS, fetch V(k+2); A reads V(k) half 0,   B reads K(k+1) half 0
    // A wave runs steps sb - 1 .. se of its own (the one before its first computes nothing it keeps except the scores of
    // the first; the one after its last adds the last step's product); all waves take part in the staging of every tile.
    // 8 waves of 128-wide heads: the upper four meet a tile's barrier a block earlier in their own stream - inside the
    // tile's first step, between its product with the values and its scores, whose key operands (and the values') are all
    // in registers by then, so nothing they read later can be overwritten by a wave that is already past the barrier. The
    // two waves of a SIMD then run half a step apart: one asks LDS for its value operands while the other is between
    // reads (config 2: -1 % of the kernel's time)
    const bool upper = D == 128 && PW == 8 && KPRE == 2 && VPRE == DT && w >= PW / 2;
    if (nt > 0) {
        f4v sA[RT][2], sB[RT][2];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int kt2 = 0; kt2 < 2; ++kt2) sA[rt][kt2] = sB[rt][kt2] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
      if constexpr (DMA) {
        // ---- three buffers a stream, tile k in buffer k % 3:
        //   step 2k   : request K(k+2);  A reads V(k-1) half 1, B's operands K(k) half 1
        //   barrier (the upper waves: inside step 2k, see above)
        //   step 2k+1 : request V(k+2);  A reads V(k) half 0,   B's operands K(k+1) half 0
        const std::false_type KEYS;
        const std::true_type VALUES;
        lds_u8* const K0 = tile_lds<D, KT, PW, 1>(); lds_u8* const K1 = tile_lds<D, KT, PW, 2>(); lds_u8* const K2 = tile_lds<D, KT, PW, 3>();
        lds_u8* const W0 = tile_lds<D, KT, PW, 4>(); lds_u8* const W1 = tile_lds<D, KT, PW, 5>(); lds_u8* const W2 = tile_lds<D, KT, PW, 6>();
       if constexpr (NBUF == 2) {
        // ---- two buffers a stream, tile k in buffer k % 2; behind tile k's barrier K(k) and V(k - 1) have been read, so
        // K(k + 2) and V(k + 1) are requested into their buffers there and have a tile's time to land:
        //   step 2k   : A reads V(k-1) half 1, B's operands K(k) half 1
        //   barrier (every transfer of this wave has landed: K(k+1), V(k));  request K(k+2), V(k+1)
        //   step 2k+1 : A reads V(k) half 0,   B's operands K(k+1) half 0
        dma(K0, kbase, 0, KEYS);
        dma(W0, vbase, 0, VALUES);
        dma(K1, kbase, 1, KEYS);
        {   // the V buffer step 0 "adds" with zero weights must hold numbers
            const u4v z = {0u, 0u, 0u, 0u};
            for (uint32_t at = (uint32_t) tid * 16; at < (uint32_t) TB; at += PW * 64 * 16)
                *reinterpret_cast<__attribute__((address_space(3))) u4v*>(W1 + at) = z;
        }
        tile_barrier();
        {
            s8v kpre[KPRE][KB];
            kread(kpre, K0);
            scores(sA, K0, kpre);
        }
        // kb / vb: the tile's own buffers; kn: the next tile's keys, vp: the tile before's values (the other buffers)
        auto tile2 = [&](int k, lds_u8* kb, lds_u8* vb, lds_u8* kn, lds_u8* vp) __attribute__((always_inline)) {
            step(sA, sB, kb + 32 * 256, vp + 32 * 256, 64 * k, !(64 * k >= w_full_beg && 64 * k + 32 <= w_full_end));
            tile_barrier();
            dma(kb, kbase, k + 2, KEYS);
            dma(vp, vbase, k + 1, VALUES);
            step(sB, sA, kn, vb, 64 * k + 32, !(64 * k + 32 >= w_full_beg && 64 * k + 64 <= w_full_end));
        };
        for (int k = 0; k < nt; k += 2) {
            tile2(k, K0, W0, K1, W1);
            if (k + 1 >= nt) break;
            tile2(k + 1, K1, W1, K0, W0);
        }
        {
            s8v vpre[VPRE];
            lds_u8* const vl = (((nt - 1) & 1) ? W1 : W0) + 32 * 256;
            vread(vpre, vl);
            weigh(vl, vpre);
        }
       } else {
        dma(K0, kbase, 0, KEYS);
        dma(W0, vbase, 0, VALUES);
        dma(K1, kbase, 1, KEYS);
        dma(W1, vbase, 1, VALUES);
        {   // the V buffer step 0 "adds" with zero weights must hold numbers
            const u4v z = {0u, 0u, 0u, 0u};
            for (uint32_t at = (uint32_t) tid * 16; at < (uint32_t) TB; at += PW * 64 * 16)
                *reinterpret_cast<__attribute__((address_space(3))) u4v*>(W2 + at) = z;
        }
        tile_barrier();
        {
            s8v kpre[KPRE][KB];
            kread(kpre, K0);
            scores(sA, K0, kpre);
        }
        // one tile: its two steps; kb / vb: the tile's own buffers, kn: the next tile's keys, vp: the tile before's values,
        // k2 / v2: where the tile after the next goes
        auto tile = [&](int k, lds_u8* kb, lds_u8* vb, lds_u8* kn, lds_u8* vp, lds_u8* k2, lds_u8* v2) __attribute__((always_inline)) {
            dma(k2, kbase, k + 2, KEYS);
            step(sA, sB, kb + 32 * 256, vp + 32 * 256, 64 * k, !(64 * k >= w_full_beg && 64 * k + 32 <= w_full_end), upper);
            if (!upper) tile_barrier();
            dma(v2, vbase, k + 2, VALUES);
            step(sB, sA, kn, vb, 64 * k + 32, !(64 * k + 32 >= w_full_beg && 64 * k + 64 <= w_full_end));
        };
        for (int k = 0; k < nt; k += 3) {
            tile(k, K0, W0, K1, W2, K2, W2);
            if (k + 1 >= nt) break;
            tile(k + 1, K1, W1, K2, W0, K0, W0);
            if (k + 2 >= nt) break;
            tile(k + 2, K2, W2, K0, W1, K1, W1);
        }
        // the last step's product
        {
            s8v vpre[VPRE];
            lds_u8* const vl = ((nt - 1) % 3 == 0 ? W0 : (nt - 1) % 3 == 1 ? W1 : W2) + 32 * 256;
            vread(vpre, vl);
            weigh(vl, vpre);
        }
       }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // (transfers past the last tile land in buffers the output goes through)
      } else {
        Stage stk, stv;
        fetch(stk, kbase, 0);
        fetch(stv, vbase, 0);
        {   // the V buffer step 0 "adds" with zero weights must hold numbers
            const u4v z = {0u, 0u, 0u, 0u};
            for (uint32_t at = (uint32_t) tid * 16; at < (uint32_t) VBUF; at += PW * 64 * 16)
                *reinterpret_cast<__attribute__((address_space(3))) u4v*>(L + V0 + VBUF + at) = z;
        }
        stash_k(stk, 0);
        stash_v(stv, 0);
        fetch(stk, kbase, 1);
        fetch(stv, vbase, 1);
        __syncthreads();
        {
            s8v kpre[KPRE][KB];
            kread(kpre, L);
            scores(sA, L, kpre);
        }
        for (int k = 0; k < nt; k += 2) {
            // tile k: buffers 0
            stash_k(stk, 1);
            fetch(stk, kbase, k + 2);
            step(sA, sB, L + 32 * KS, L + V0 + VBUF + 32 * VS, 64 * k, !(64 * k >= w_full_beg && 64 * k + 32 <= w_full_end), upper);
            if (!upper) __syncthreads();
            stash_v(stv, 1);
            fetch(stv, vbase, k + 2);
            step(sB, sA, L + KBUF, L + V0, 64 * k + 32, !(64 * k + 32 >= w_full_beg && 64 * k + 64 <= w_full_end));
            if (k + 1 >= nt) break;
            // tile k + 1: buffers 1
            stash_k(stk, 0);
            fetch(stk, kbase, k + 3);
            step(sA, sB, L + KBUF + 32 * KS, L + V0 + 32 * VS, 64 * k + 64, !(64 * k + 64 >= w_full_beg && 64 * k + 96 <= w_full_end), upper);
            if (!upper) __syncthreads();
            stash_v(stv, 0);
            fetch(stv, vbase, k + 3);
            step(sB, sA, L, L + V0 + VBUF, 64 * k + 96, !(64 * k + 96 >= w_full_beg && 64 * k + 128 <= w_full_end));
        }
        // the last step's product
        {
            s8v vpre[VPRE];
            lds_u8* const vl = L + V0 + (uint32_t) ((nt - 1) & 1) * VBUF + 32 * VS;
            vread(vpre, vl);
            weigh(vl, vpre);
        }
      }
    }

    // ---- out = O / l. A lane holds dims 16 dt + 4 g4 .. + 3 of its rows: the wave's 32 x D block goes through LDS (the
    // tile buffers, free now) so that it leaves as whole rows, 16 bytes a lane and 4 (float32: 2) rows an instruction
    __syncthreads();                                              // every wave is done with the tiles
    // (DMA: the tile buffers are arrays of their own; two waves' staging regions go through each of the first four)
    lds_u8* const OB = DMA && NBUF == 2 ? (w == 0 ? tile_lds<D, KT, PW, 1>() : w == 1 ? tile_lds<D, KT, PW, 2>() : w == 2 ? tile_lds<D, KT, PW, 4>() : tile_lds<D, KT, PW, 5>())
                       : DMA ? ((w & 3) == 0 ? tile_lds<D, KT, PW, 1>() : (w & 3) == 1 ? tile_lds<D, KT, PW, 2>() : (w & 3) == 2 ? tile_lds<D, KT, PW, 3>() : tile_lds<D, KT, PW, 4>()) + (w >> 2) * 16 * (D * 4 + 16)
                           : L + w * 16 * (D * 4 + 16);
    // a place's (row, head) among the pass's
    auto out_row = [&](int place) __attribute__((always_inline)) -> int64_t {
        if constexpr (FLAT) return (int64_t) row_of(place) * (p.Hq - p.G) + hk * p.G + place;
        else return (int64_t) place * p.Hq + hq;
    };
    if (p.ns > 1 && !whole) {
        // ---- a key split's partial: the rows' unnormalized sums as float32, then (m, l) - D + 2 floats a (row, head, split),
        // rows 8 bytes aligned: 8-byte pieces, 8 rows an instruction
        const uint32_t rowp = D * 4 + 16;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float lsum = l4[rt][0];
            const uint32_t at = (uint32_t) n * rowp + (uint32_t) (g4 * 16);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<__attribute__((address_space(3))) f4v*>(OB + at + dt * 64) = o[rt][dt];
            const int place = wbase + rt * 16 + n;
            if (g4 == 0 && place < wend) {
                float* pr = p.part + (out_row(place) * p.ns + split) * (D + 2);
                *reinterpret_cast<float2*>(pr + D) = float2{thr[rt] < 0.0f ? -INFINITY : -nbr[rt], lsum};
            }
            for (int c = lane; c < 16 * (D / 2); c += 64) {
                const int rl_ = c / (D / 2), piece = c % (D / 2), prow = wbase + rt * 16 + rl_;
                if (prow < wend) {
                    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
                    const u2v x = *reinterpret_cast<const __attribute__((address_space(3))) u2v*>(OB + (uint32_t) rl_ * rowp + (uint32_t) piece * 8);
                    *reinterpret_cast<u2v*>(p.part + (out_row(prow) * p.ns + split) * (D + 2) + piece * 2) = x;
                }
            }
        }
        return;
    }
    {
        const int esz = p.qt == 0 ? 4 : 2;
        const uint32_t rowb = (uint32_t) (D * esz), rowp = rowb + 16;    // bytes a row, padded in LDS
        const int ppr = (int) rowb / 16;                          // 16-byte pieces a row
        uint8_t* const orow = reinterpret_cast<uint8_t*>(p.out) + (FLAT ? 0 : (int64_t) hq * rowb);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float lsum = l4[rt][0];
            const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
            const uint32_t at = (uint32_t) n * rowp + (uint32_t) (g4 * 4 * esz);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const f4v v = o[rt][dt] * inv;
                if (p.qt == 0) {
                    *reinterpret_cast<__attribute__((address_space(3))) f4v*>(OB + at + dt * 64) = v;
                } else {
                    typedef uint16_t us4v __attribute__((ext_vector_type(4)));
                    us4v h;
                    if (p.qt == 1) h = us4v{f32_to_f16(v[0]), f32_to_f16(v[1]), f32_to_f16(v[2]), f32_to_f16(v[3])};
                    else h = us4v{f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3])};
                    *reinterpret_cast<__attribute__((address_space(3))) us4v*>(OB + at + dt * 32) = h;
                }
            }
            // the wave reads back its own block only: no barrier, the LDS queue keeps a wave's accesses in order
            for (int c = lane; c < 16 * ppr; c += 64) {
                const int rl_ = c / ppr, piece = c % ppr, row = wbase + rt * 16 + rl_;
                if (row < wend) {
                    const u4v x = *reinterpret_cast<const __attribute__((address_space(3))) u4v*>(OB + (uint32_t) rl_ * rowp + (uint32_t) piece * 16);
                    *reinterpret_cast<u4v*>(orow + (FLAT ? out_row(row) : (int64_t) row * p.Hq) * rowb + piece * 16) = x;
                }
            }
        }
    }
