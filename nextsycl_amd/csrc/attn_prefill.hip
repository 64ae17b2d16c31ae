// attn_prefill.hip: causal GQA flash attention of a prompt pass's rows against the KV cache (half, bfloat16, q8_0 or q4_0
// rows; D = 128 or 256) for gfx950.
//
// Bound: MFMA. 4 D flops a visible (row, key) pair against 2 x 2 D bytes a key shared by every row that sees it:
// thousands of flops a byte at prompt lengths.
//
// Work split: one work-group per (row block, query head). A work-group of 8 waves owns ROWS = 256 consecutive query rows
// of one query head (a wave 32 of them: two 16-row MFMA tiles) and streams the keys its rows see in 64-key tiles,
// heaviest row blocks first (the last block sees the most keys). The G query heads of a key head on one row block are
// neighbours in the logical order and, through the XCD-aware mapping of work-group ids, share one L2. A tile's K and V
// rows are fetched by all the work-group's threads (16-byte chunks). Over 16-bit rows at D = 128 they go global -> LDS
// directly (global_load_lds_dwordx4, unpadded buffers, the bank swizzle applied to the global addresses, one barrier a
// tile that waits on the wave's transfers): the 8-wave form two tiles ahead into three buffers a stream, the barrier
// leaving the newest tile's transfers in flight; the 4-wave form (two work-groups a CU) one tile ahead into two buffers a
// stream, requested right behind the barrier that frees them. The other forms (quantized rows, D = 256) go global ->
// registers two tiles ahead -> LDS one tile ahead: two register sets, two padded LDS buffers.
// A pass of few rows packs several query heads of one key head into a work-group (a wave slot a head: the tile staged
// once serves them all) or, behind a context worth it, lays its (row, head) pairs end to end (attn_prefill_flat_kernel), and a pass of few rows over a long context is cut into key splits whose partials a merge
// kernel puts together. bfloat16, q8_0 and q4_0 rows read many times are first widened to half rows in the library's
// scratch (bit for bit the halfs the kernel would stage); the kernel's own forms of them serve short passes and caches
// the scratch does not hold.
//
// A wave's tile step, in the transposed orientation (a lane owns one query row of each row tile, so the row maximum,
// the rescale and the normalisation never leave the lane):
//   S^T[key][row] = K Q^T        K from LDS as the A operand (ds_read_b128; rows padded to 288 bytes, or swizzled), Q^T in registers.
//                                Half operands: Q carries the softmax scale x log2 e and the product starts from minus the
//                                softmax reference, so a score leaves the matrix unit as the argument of its exponential
//   base-2 online softmax in float32 (the accumulators rescaled only when a row's maximum moved); only 32-key halves
//   crossing a row's causal or window edge are masked
//   P^T -> 16 bit = the B operand of the second product as it stands
//   O^T[d][row]  += V^T P^T      V^T from LDS through ds_read_b64_tr_b16 (rows padded to 288 bytes, or swizzled)
//
// Reference behaviour kept: kernels/llm/museglimmer/silo/attn.cpp:56-267 and kernels/llm/qwen35/silo/attn.cpp:105-313
// (prompt form: causal from p0, window, ring slots, 16-bit operands with float32 softmax and accumulation, rows past T
// not written, no scratch).
#include "ns_internal.hpp"
#include "ns_attn.h"
#include "attn_common.hpp"
#include "attn_host.hpp"
#include "kv_formats.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace {

constexpr int KT_TILE = 64;
// waves a work-group (PW): at D = 128 a wave owns 32 rows and a work-group 8 waves = 256 rows when that still leaves two
// work-groups for every CU - a tile staged for 256 rows costs half the fetches and LDS writes a row, and two work-groups
// of 4 waves on a CU were measured to run no faster than one of 8 - else 4 waves = 128 rows; at D = 256 4 waves of 16 rows
constexpr int rows_of(int D, int PW) { return PW * (D == 128 ? 32 : 16); }   // query rows a work-group

struct PrefillParams {
    const void* q;
    int qt;
    int64_t qs;
    const uint8_t* kc;
    const uint8_t* vc;
    int64_t head_stride, row_stride, cap;
    int wrap;
    int T, Hq, G;
    int64_t p0, win;
    int causal;                 // 0: every row sees to the pass's last key (a draft block)
    int64_t kfirst;             // >= 0: every row's first key, instead of its own window's
    float sl2;
    void* out;
    // key splits (passes of few row blocks over many keys): work-group (x, y) takes the keys [k0 + y kbs, k0 + (y + 1) kbs)
    // of its rows' own ranges and leaves a partial {O, m, l} a (row, head, split) for the decode path's merge kernel
    int ns;
    int64_t kbs, k0;
    float* part;                // [T][Hq][ns][D + 2]
    // a pass of few rows: a work-group holds `pack` query heads of its key head - wave w rows (w / pack) x (a wave's rows)
    // .. of head w % pack - so the heads share every key and value tile the work-group stages. 1: one head, every wave rows
    // of its own. gw = G / pack: work-groups a (row block, key head)
    int pack, gw;
    // rows end to end (attn_prefill_flat_kernel): row tiles of 16 (row, head) pairs a work-group, row blocks that share an XCD's keys,
    // groups of them a key head, the blocks in front that are not cut into splits (the last rows'; gb 1 then), and ceil(2^32 / G) (a pair's
    // row is a multiplication away)
    int tb, gb, ngb, nbf;
    uint32_t ginv;
};

// a 16-byte chunk of a K or V row on its way from global memory to LDS (a plain vector type: arrays of it stay in registers)
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
// the same at an address that is only 8-byte aligned (q8_0 / q4_0 rows of 128 values are 136 / 72 bytes long)
typedef uint32_t u4a8 __attribute__((ext_vector_type(4), aligned(8)));

typedef __attribute__((address_space(3))) uint8_t lds_u8;
// bytes a staged key row / value row: rows 32 bytes apart modulo 256, so that the 16-byte operand reads of 16 keys (and
// the transposing reads of the values) meet no bank conflict - 16 bytes apart the key reads would, two ways
constexpr int padded_row(int D) { return D * 2 + 32; }
constexpr bool by_dma(int D, int KT, int PW) { return D == 128 && KT == 0 && (PW == 8 || PW == 4); }
constexpr int tile_bufs(int PW) { return PW == 8 ? 3 : 2; }       // tile buffers a stream (DMA)
// a work-group's LDS, one array a name for all waves' functions: padded tiles (WHICH 0), or - DMA - three (two) buffers each of key
// (1 - 3) and value tiles (4 - 6)
template <int D, int KT, int PW, int WHICH>
__device__ __forceinline__ lds_u8* tile_lds() {
    constexpr bool DMA = by_dma(D, KT, PW), there = WHICH == 0 ? !DMA : DMA && (WHICH % 3 != 0 || tile_bufs(PW) == 3);
    // (two waves' output staging, 8448 B each, go through one array)
    constexpr int BYTES = !there ? 16 : WHICH == 0 ? 4 * KT_TILE * padded_row(D) : KT_TILE * 256 + 512;
    static __shared__ __attribute__((aligned(WHICH == 0 ? 16 : 1024))) uint8_t mem[BYTES];
    return (lds_u8*) mem;
}

// FLAT: the row tiles of a block that begins with tile tile0, and those of wave w among a block's tn: the first waves take
// two where there are more than waves
__device__ __forceinline__ int flat_tiles(const PrefillParams& p, int tile0) { return std::min(p.tb, (p.T * p.G + 15) / 16 - tile0); }
__device__ __forceinline__ int wave_tile0(int w, int tn, int waves) { return w + std::min(w, std::max(0, tn - waves)); }
__device__ __forceinline__ int wave_tiles(int w, int tn, int waves) { return w < tn - waves ? 2 : w < tn ? 1 : 0; }

// BF: bfloat16 operands (a bfloat16 cache too long to be widened to half first), else half. QS (bfloat16 operands only):
// query rows of another type enter the first product as two bfloat16 numbers - the rounded row and the rounded rest, 16
// significant bits between them - a second matrix instruction a key block.
// NTS (16-bit rows of 128 only): the tiles' transfers carry the streaming cache policy - a pass whose keys are each read
// by one work-group, once.
template <int D, bool BF, int KT, int PW, bool QS = false, bool NTS = false>
__global__ __launch_bounds__(PW * 64, PW == 4 && D == 128 ? 2 : 1) void attn_prefill_kernel(const PrefillParams p) {
    constexpr bool FLAT = false;
    // a wave owns RT row tiles of 16: 32 rows at D = 128; 16 at D = 256, whose accumulators are twice as wide
    constexpr int RT = D == 128 ? 2 : 1;
#include "attn_prefill_wave.hpp"
}

template <int D, bool BF, int KT, int PW, bool QS, bool NTS, int RT>
__device__ __forceinline__ void flat_wave(const PrefillParams& p) {
    constexpr bool FLAT = true;
#include "attn_prefill_wave.hpp"
}

// (row, head) pairs of a key head end to end - pair r is row r / G, head r % G of the group - 16 a row tile: a work-group's tiles
// over its 8 waves, one each and, at D = 128, the first waves two where there are more (a SIMD's two waves then hold 2 or 3, not 2 and
// 4); waves without one stage their share of the keys and meet the barriers. For passes whose rows leave places of whole
// 32-row waves empty (flat_plan). Bound: at few pairs HBM, else as the kernel above, LDS the more where waves hold one tile. New turn of 37 rows x
// 32 / 8 bfloat16 heads behind 20011 keys, this kernel 34 us, the one above 41.7.
template <int D, bool BF, int KT, bool QS = false, bool NTS = false, int PW = 8>
__global__ __launch_bounds__(PW * 64, PW == 4 ? 2 : 1) void attn_prefill_flat_kernel(const PrefillParams p) {
    const int w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const int Hkv = p.Hq / p.G, xi = (int) blockIdx.x / 8, nfull = p.nbf * Hkv, u2 = xi / p.gb * 8 + (int) blockIdx.x % 8 - nfull;
    const int unit = u2 < 0 ? u2 + nfull : u2 % std::max(1, p.ngb * Hkv - nfull) + nfull;
    const int nblk = ((p.T * p.G + 15) / 16 + p.tb - 1) / p.tb, blk = nblk - 1 - (unit / Hkv * p.gb + xi % p.gb);
    if (D == 128 && wave_tiles(w, flat_tiles(p, blk * p.tb), PW) == 2) flat_wave<D, BF, KT, PW, QS, NTS, D == 128 ? 2 : 1>(p);
    else flat_wave<D, BF, KT, PW, QS, NTS, 1>(p);
}

// A bfloat16 cache's rows on their way to half rows in position order: positions [kf, kf + n) of every key head, out of a
// cache of any geometry (head-major, position-major, a ring) into [which][head][n][D]. Every bfloat16 value whose
// magnitude lies in half's normal range is a half exactly; larger ones saturate at 65504 (the reference's caches are
// half: kernels/llm/qwen35/q35.cpp:573-588 rounds float32 rows into them), smaller ones round to half's subnormals.
struct WidenParams {
    const uint8_t* src[2];
    uint8_t* dst[2];
    int64_t head_stride, row_stride, cap, kf, n;
    int wrap;
};
template <int CPR>   // 16-byte chunks a row: D / 8
__global__ __launch_bounds__(256) void kv_bf16_to_half_kernel(const WidenParams p) {
    const int64_t j = (int64_t) blockIdx.x * (256 / CPR) + threadIdx.x / CPR;
    const int c = threadIdx.x % CPR, h = blockIdx.y, z = blockIdx.z;
    if (j >= p.n) return;
    const int64_t pos = p.kf + j, slot = p.wrap ? pos % p.cap : pos;
    const u4v x = __builtin_nontemporal_load(reinterpret_cast<const u4v*>(p.src[z] + h * p.head_stride + slot * p.row_stride + c * 16));
    u4v y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = fminf(fmaxf(__builtin_bit_cast(float, x[i] << 16), -65504.0f), 65504.0f);
        const float hi = fminf(fmaxf(__builtin_bit_cast(float, x[i] & 0xFFFF0000u), -65504.0f), 65504.0f);
        y[i] = (uint32_t) __builtin_bit_cast(uint16_t, (_Float16) lo) | ((uint32_t) __builtin_bit_cast(uint16_t, (_Float16) hi) << 16);
    }
    *reinterpret_cast<u4v*>(p.dst[z] + (((int64_t) h * p.n + j) * CPR + c) * 16) = y;
}

// The same for q8_0 (KT = 1) and q4_0 (KT = 2) rows: a thread takes 8 values of a 32-value block - 8 bytes, or one nibble
// of each of 8 bytes - and writes the 8 halfs the kernels' own staging makes of them (half(q x d), one rounding: dq8x8 /
// dq4x8), so the pass over the widened rows sees the operands the pass over the raw rows would have built.
template <int KT, int CPR>   // 8-value chunks a row: D / 8
__global__ __launch_bounds__(256) void kv_quant_to_half_kernel(const WidenParams p) {
    constexpr int D = CPR * 8;
    const int64_t j = (int64_t) blockIdx.x * (256 / CPR) + threadIdx.x / CPR;
    const int c = threadIdx.x % CPR, h = blockIdx.y, z = blockIdx.z;
    if (j >= p.n) return;
    const int64_t pos = p.kf + j, slot = p.wrap ? pos % p.cap : pos;
    const uint8_t* const row = p.src[z] + h * p.head_stride + slot * p.row_stride;
    const int b = c / 4, cc = c % 4;
    dq_s8v y;
    if constexpr (KT == 1) {
        const uint2 x = *reinterpret_cast<const uint2*>(row + c * 8);
        y = dq8x8(x.x, x.y, __builtin_bit_cast(_Float16, *reinterpret_cast<const uint16_t*>(row + D + 2 * b)));
    } else {
        const uint2 x = *reinterpret_cast<const uint2*>(row + b * 16 + (cc & 1) * 8);
        y = dq4x8(x.x, x.y, cc >= 2 ? 4 : 0, __builtin_bit_cast(_Float16, *reinterpret_cast<const uint16_t*>(row + D / 2 + 2 * b)));
    }
    *reinterpret_cast<dq_s8v*>(p.dst[z] + (((int64_t) h * p.n + j) * CPR + c) * 16) = y;
}

// Query heads a work-group holds (PrefillParams::pack): a pass of so few rows that they fill only some of a work-group's
// waves gives the other waves further heads of the same key head - 32 rows and fewer: 4 heads to 4 waves - and every
// staged tile then serves them all (17 rows x 32 / 8 heads behind 32768 keys: each head's work-group re-staged the keys
// for one live wave). A divisor of the group: 5 heads take 5 of 8 waves.
int64_t pack_of(int64_t T, int64_t G, int64_t D, int64_t PW) {
    const int64_t need = (T + (D == 128 ? 32 : 16) - 1) / (D == 128 ? 32 : 16);       // waves the rows of one head fill
    int64_t pack = 1;
    for (int64_t c = 2; c * need <= PW; ++c)
        if (G % c == 0) pack = c;
    return pack;
}

// A short pass's (row, head) pairs laid end to end (FLAT): row blocks a key head, row tiles of 16 a block, key splits, blocks
// that share an XCD's keys and groups of them a key head
struct FlatPlan {
    int64_t waves = 0;                                            // a work-group's: 8, or 4 (half the places, two a CU), or the pass stays as it is: 0
    int64_t blocks = 1, tb = 1, ns = 1, gb = 1, ngb = 1, nbf = 0;  // (nbf: of the blocks, the last ones that are not split)
    void cut(int64_t T, int64_t G, int64_t D, int64_t w) {
        const int64_t row_tiles = (T * G + 15) / 16, per = w * (D == 128 ? 2 : 1);
        waves = w;
        blocks = (row_tiles + per - 1) / per;
        tb = (row_tiles + blocks - 1) / blocks;
        ns = gb = 1;
        ngb = blocks;
        nbf = 0;
    }
};
// How such a pass is cut, and whether it is the shorter way (pays = false: only the cut is asked for).
// Rows of one head to a wave, 37 rows fill 64 of its work-group's places; end to end their 148 pairs over 4 heads fill 160, and a key
// is staged once for 256 of them instead of 128. What is lost is the start: one work-group of 8 waves a CU and a kernel of two forms of
// the step. Both sides in us, this way last: 37 rows x 32 / 8 heads behind 20011 keys, half 38.4 / 32.8, bfloat16 49.2 / 40.4, behind
// 1000 19.5 / 20.0; 37 x 24 / 4 heads of 256 behind 20011 82.0 / 42.7, behind 1000 22.6 / 24.2; 128 x 32 / 8 behind 20011 58.8 / 58.7.
// The cut: the splits, and the grouping of blocks, that cost least by a model fitted to 183 passes' times under a sweep of split counts
// (it picks within 1 % of the best on average): rounds of the 256 CUs, counted an XCD, each 20 + a split's key tiles times a tile's cost,
// which grows with the row tiles that share it, and 5.4 a million floats of partials. A unit of the unit: some 0.45 us.
// The choice: what the passes' full places would take at 1 PFLOP/s or 5.5 TB/s (us), on the other way's places (old), against this
// way's (us / how full its rounds are); fitted to 795 passes of 17 - 600 rows x 13 head layouts behind 700 - 120000 keys in every cache form:
// of the time between the two ways' shorter one and the other way, it finds nine tenths, and loses 2.5 % and more on 9. q8_0 rows of
// 128, kept as they are this way (own_form_pays), gain where a model of widened rows does not see it: from 700 keys on in one block and where heads
// share no keys, from 1500 in up to seven blocks, from 2000 in more; one or two key heads in more than one block from 8000 or 2800 - the other way's
// heads fill the CUs, this way's blocks are few and its splits short: 36 x 16 / 8 heads behind 2041 keys 23.6 / 16.4, 17 x 64 / 64 behind 1649
// 42.7 / 21.0, 58 x 64 / 8 behind 1201 28.1 / 30.3, 88 x 24 / 2 behind 1849 27.4 / 30.8, 364 x 24 / 2 behind 7055 73.1 / 54.2. Over 1800 passes of 17 - 600
// q8_0 rows x 20 layouts behind 250 - 60000 keys 1.215 on the geometric mean (the shorter way each time: 1.228), 17 lose more than 4 %.
// Rows that see unequal parts of the keys - a prompt's start, a window little longer than the pass - stay with the other way, and so does
// what the fit's 700 keys and more do not reach: under 448 keys (44 x 96 / 8 behind 391 16.7 / 19.5), under 1024 behind less than four times
// the rows (158 x 64 / 64 behind 487 22.0 / 25.3), under 1400 where eight blocks a key head fill the other way's rounds (278 x 64 / 8 behind 865 31.2 / 37.3).
// Over 1200 passes of up to 600 rows x 18 layouts these lines take the gain from 1.038 to 1.053 on the geometric mean.
bool flat_plan(FlatPlan& f, bool pays, int kt, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t p0, int64_t keys, int64_t most_splits) {
    const int64_t G = Hq / Hkv;
    f.cut(T, G, D, 8);
    double us = 0.0, old = 0.0;
    const int64_t from = std::max<int64_t>(Hkv == 1 ? 8000 : Hkv == 2 ? 2800 : 0, G == 1 || f.blocks == 1 ? 700 : f.blocks <= 7 ? 1500 : 2000);
    const bool always = kt == 1 && D == 128 && keys >= from;
    // (q4_0 rows of 128, one block: widening them in 8 waves' step bounds it - 27 x 32 / 8 heads behind 94406 keys 66.7 / 75.1, 105 x 32 / 32 behind 84857
    // 206 / 232, 49 x 64 / 32 behind 60339 153 / 172; 31 passes of such rows in up to half a block behind 24000 keys and more 0.975, 32 behind 4000 - 24000 1.08)
    const double share = D == 256 ? 2.0 : kt != 2 ? 1.1 : f.blocks == 1 ? 0.95 : 1.15, margin = D == 256 ? 6.0 : kt == 2 ? 4.0 : 1.0;
    if (pays) {
        if (T > 600 || p0 < 3 * T || keys < 4 * T || most_splits < 1) return false;
        if (keys < (p0 < 4 * T ? 1024 : 448) || (D == 128 && f.blocks >= 8 && keys < 1400)) return false;
        const int64_t PW = D == 128 || T <= 64 ? 4 : 8, pack = pack_of(T, G, D, PW), rb = PW / pack * (D == 128 ? 32 : 16);
        // (q4_0 rows of 128 in half a block, each read once this way and the other: 8 waves' step is the slower then, and from here on it shows)
        if (kt == 2 && D == 128 && f.blocks == 1 && f.tb <= 8 && pack == G && T <= rb && keys >= 24000) return false;
        const double places = (double) (f.blocks * f.tb * 16);
        us = std::max(4.0e-9 * places * (double) (Hkv * keys * D), (double) (Hkv * keys * D) / 1.375e6);
        old = us * (double) ((T + rb - 1) / rb * rb * G) / places * share;
        if (!always && old - us <= margin) return false;
    }
    const int64_t tiles = (keys + KT_TILE - 1) / KT_TILE + 1;
    const double step = D == 128 ? 1.2 + 0.25 * (double) f.tb : 5.9 + 0.19 * (double) f.tb, part = 5.4e-6 * (double) (T * Hq * (D + 2));
    double least = 1e30, full = 0.0;
    for (int64_t m = 1; m <= std::min<int64_t>(f.blocks, 8); ++m) {
        const int64_t gb = (f.blocks + m - 1) / m, r0 = ((Hkv * m + 7) / 8 * gb + 31) / 32;
        for (int64_t r = r0; r <= r0 + 2; ++r) {
            // (the most splits that r rounds hold, or as many as their partials pay for)
            const int64_t hold = std::min({8 * (32 * r / gb) / (Hkv * m), most_splits, tiles}), best = (int64_t) std::sqrt((double) (r * tiles) * step / part);
            for (int64_t ns : {std::min(best, hold), std::min(best + 1, hold)}) {
                if (ns < 1) continue;
                const int64_t a_split = (tiles + ns - 1) / ns;
                const double c = (double) r * (20.0 + step * (double) a_split) + part * (double) ns;
                if (c >= 0.995 * least) continue;
                least = c, f.ns = ns, f.ngb = m, f.gb = gb;
                full = (double) (Hkv * ns * f.blocks * tiles) / (double) (r * 256 * ns * a_split);
            }
        }
    }
    return !pays || always || old - us / std::max(full, D == 128 ? 0.5 : 0.7) > margin;
}

// A pass's form: its (row, head) pairs end to end, in splits or whole, or whole waves of one head's rows (f.waves 0). Beside the short
// passes of flat_plan, rows end to end pay wherever a block of few rows x all the group's heads sees less of what it masks than one of
// 128 - 256 rows x one head - a prompt's diagonal, a window's two edges - and where its work-groups make fuller rounds of the CUs. By
// measurement, over 430 passes of 129 - 8192 rows x 13 head layouts, this way (geometric mean): n8 = work-groups of 8 waves
//   window, p0 + T past 2 1/4 of it: 4 waves at heads of 128 (n8 of 100 and more, 20 with a short window) 1.15, 3000 rows x 32 / 8,
//     window 512, 94.5 -> 49 us; 8 waves for one round of the CUs nearly or quite full, 2001 x 32 / 2, window 1024, 52.2 -> 45.2, 2043 rows, window 2048, 76.4 -> 71.8 in
//     4 waves, 68.3 in 8 (63 passes of n8 200 - 249 1.03, 21 of 256 1.02, 42 of 257 - 330 0.92); 8 at heads of 256 1.2
//   behind little or nothing, no splits: n8 of 512 (256 behind nearly its own length) and more at heads of 128, 250 of 256: 1.03 and
//     1.1; 8192 x 40 / 8 595 -> 587, 3596 x 64 / 4 256 -> 217, 2048 x 24 / 4 of 256 109 -> 74 (the other way cuts it in two); fewer leave
//     CUs idle that blocks half as long fill: 1024 x 32 / 8 25.9 / 31.4
//   behind its own length and more: cut as the short ones while a round holds the blocks, 1.09 (645 x 48 / 8 behind 2663 85 -> 64, 1319 x 24 / 4
//     of 256 behind 4598 252 -> 203); more blocks run whole in whole rounds, and what is left over in splits - a share of the rows leaves
//     partials, and a count between rounds costs what it should: 1403 x 48 / 8 behind 9568 376 -> 333, 2439 x 32 / 2 behind 3321 211 -> 186, 3072
//     x 24 / 4 of 256 behind 8192 854 -> 791. Where the other way's rounds are full as they are it stays: 2048 x 24 / 4 of 256 behind 8192 519 /
//     577, 4000 x 16 / 4 behind 5000 230 / 243
void rows_form(FlatPlan& f, int kt, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t p0, int64_t win, int64_t kfirst, int64_t keys, int64_t most_splits) {
    const int64_t G = Hq / Hkv;
    if (flat_plan(f, true, kt, T, Hq, Hkv, D, p0, keys, most_splits)) return;
    f.cut(T, G, D, 8);
    const int64_t n8 = f.blocks * Hkv;
    f.waves = 0;
    if (G == 1 || kfirst >= 0) return;
    // (how full the other way's rounds are: blocks of 128 rows a head, two work-groups a CU, or heads of 256 in two splits, one)
    const int64_t wgs = (T + 127) / 128 * Hq * (D == 256 ? 2 : 1), round = D == 256 ? 256 : 512;
    const double other = (double) wgs / (double) ((wgs + round - 1) / round * round);
    if (win > 0 && p0 + T > win) {
        if (4 * (p0 + T) < 9 * win) return;
        if (D == 256 ? win <= 1024 && n8 >= 100 && n8 <= 900 : n8 >= 100 || (win <= 640 && n8 >= 20)) f.cut(T, G, D, D == 256 || (n8 >= 200 && n8 <= 256) ? 8 : 4);
    } else if (n8 <= 256 && ((T > 600 && p0 >= 2 * T) || (p0 >= T && p0 < 2 * T && n8 >= 176 && other < 0.93))) {
        flat_plan(f, false, kt, T, Hq, Hkv, D, p0, keys, most_splits);
    } else if (n8 >= (D == 256 ? 250 : 5 * p0 >= 4 * T ? 257 : 512)) {
        if (D == 256 && p0 >= T && other > 0.95) return;
        f.cut(T, G, D, 8);
        if (5 * p0 < 4 * T) return;
        // whole rounds of blocks over all their keys, and what is left over - as many blocks as end with a row - in splits, which first take
        // the places that the whole blocks leave: the shortest way in the units of flat_plan, counted on the XCD that has most
        const int64_t rounds = n8 / 256, tiles = (keys + KT_TILE - 1) / KT_TILE + 1, first = f.blocks - rounds * 256 / Hkv;
        const double rows = 20.0 + (D == 128 ? 1.2 + 0.25 * (double) f.tb : 5.9 + 0.19 * (double) f.tb) * (double) tiles, part = 5.4e-6 * (double) (f.tb * 16 * Hkv * (D + 2));
        double least = n8 % 256 ? 0.97 * rows : 0.0;
        for (int64_t left = std::max<int64_t>(first, 1); left <= std::min(f.blocks, first + 16); ++left) {
            if (left < f.blocks && left * f.tb * 16 % G) continue;
            const int64_t spare = rounds * 32 - ((f.blocks - left) * Hkv + 7) / 8;
            for (int64_t ns = 2; ns <= std::min<int64_t>({16, most_splits, tiles / 8}); ++ns) {
                const int64_t over = std::max<int64_t>(0, (left * Hkv * ns + 7) / 8 - spare * ns);
                const double c = (double) ((over + 31) / 32) * (20.0 + (rows - 20.0) / (double) ns) + part * (double) (left * ns);
                if (c < least) least = c, f.ns = ns, f.nbf = f.blocks - left;
            }
        }
    }
}

// Whether a pass over rows that are not half keeps their form in the kernel instead of widening them to half rows first
// (knob 5 = 0: the measured rule). What widening costs is read and written once a key; a pass of few rows reads a key
// only once a row block and query head of its group, and the kernel's own staging of it is then the shorter way. T rows x
// G heads a key head behind `keys` keys, float32 query rows, widened / own form in us:
//   bfloat16 (bfloat16 query rows up to 128 rows x D / 32 heads; rows of another type, which enter the first product in
//     two parts - twice its matrix instructions - up to 2 D rows a key head; behind fewer than 4096 keys the widening
//     costs next to nothing and its pass is the shorter): 64 x 4 of 128 behind 32768 keys 107 / 84, 17 x 4 behind 131072
//     333 / 164, 128 x 4 behind 32768 120 / 122; 17 bfloat16 rows x 1 behind 2048 35 / 38
//   q8_0 rows of 128 behind 32768 keys and more, up to 8 reads a key: 17 x 4 behind 131072 294 / 158, 128 x 4 behind
//     32768 111 / 86, 64 x 4 behind 8192 42 / 54; 17 x 16 behind 131072 217 / 215. Rows of 256 behind 65536 keys and
//     more, up to 256 rows a key head: 17 x 4 behind 131072 130 / 86, 32 x 8 154 / 139, 64 x 8 220 / 240; 17 x 8 behind
//     32768 54 / 62
//   q4_0 rows of 128 up to 1400 rows a key head, whatever the heads share them: 64 x 4 behind 32768 92 / 67, 17 x 16 behind
//     131072 214 / 157, 1100 x 1 alone 43 / 36, 300 x 4 behind 2000 33 / 29, behind 30000 120 / 111, 257 x 5 behind 2000 44 / 40,
//     behind 32768 266 / 256; many reads of a key: 87 x 16 (64 / 4 heads) behind 2000 30 / 28, behind 8000 56 / 54, behind 32768
//     147 / 142, 129 x 8 (32 / 4) 32 / 28, 57 / 53, 146 / 141; the least gained: 175 x 8 (64 / 8) behind 8000 80.8 / 81.6, 700 x 2 (32
//     / 16) behind 2000 54 / 56, behind 32768 437 / 426; beyond, some shapes gain and others lose: 400 x 5 behind 8000 104 / 101, 500 x
//     4 there 83 / 86, 2000 x 1 91 / 94, 128 x 16 behind 32768 143 / 148. Rows of 256 behind 32768 keys and more, up to 8 reads a
//     key: 64 x 8 behind 131072 217 / 176, 17 x 8 there 147 / 95, 17 x 8 behind 8192 36 / 43
bool own_form_pays(int kt, int qt, int64_t D, int64_t T, int64_t G, int64_t keys, const FlatPlan* flat) {
    // (rows end to end: a key is read once a row block. Widened / own form: q8_0 rows of 128, one block behind 20000 keys 1.3 - 2.2 times,
    // seven blocks 1.03; q4_0 rows of 128 1.05 at six and seven, of 256 1.1 at two to four, 1.02 at six; bfloat16 rows behind 20000
    // keys 1.3 - 1.9 at one block, 1.1 at 400 pairs, behind 2000 1.0; q8_0 rows of 256 0.6 - 0.9 but at few pairs behind 65536 keys)
    const int64_t key_reads = ((T + 127) / 128) * G, pairs = T * G;
    if (flat) {
        const int64_t n = flat->blocks;
        if (kt == 1) return D == 128 ? n <= 7 : keys >= 65536 && pairs <= 256;
        if (kt == 2) return n <= (D == 128 ? 10 : 6);
        if (kt == 3 && (D == 256 ? n <= 5 && keys >= (qt == 2 ? 4096 : 2048) : pairs <= 256 ? keys >= (qt == 2 ? 2500 : 3072) : qt == 2 && pairs <= 580 && keys >= 9000)) return true;
        // (bfloat16 rows besides wherever the other form keeps them: their own form carries 16 bits a weight and every bfloat16 value, and a
        // pass does not lose them for the way its rows lie. Widened / own: 338 x 32 / 32 behind 7747 101 / 78, 76 x 64 / 16 behind 7373 60 / 49,
        // 178 x 16 / 4 of 256 behind 23635 127 / 120, 238 x 16 / 8 behind 6845 48.5 / 47.6; over 140 such passes 1.06)
    }
    switch (kt) {
        case 3: return keys >= 4096 && key_reads <= D / 32 && (qt == 2 || pairs <= 2 * D);
        case 1: return D == 128 ? keys >= 32768 && key_reads <= 8 : keys >= 65536 && pairs <= 256;
        case 2: return D == 128 ? pairs <= 1400 : keys >= 32768 && key_reads <= 8;
        default: return false;
    }
}

// the passes whose rows lie end to end: work-groups of 8 waves, or of 4 (small: half rows of 128)
template <int D>
void launch_flat(ns_gpu* g, int kt, const PrefillParams& p, dim3 grid, bool stream, bool small) {
    constexpr int TH = 512;
    if constexpr (D == 128) {
        if (small && kt == 0) {
            attn_prefill_flat_kernel<D, false, 0, false, false, 4><<<grid, 256, 0, g->q>>>(p);
            return;
        }
    }
    if (kt == 0) {
        if (D == 128 && stream) attn_prefill_flat_kernel<D, false, 0, false, D == 128><<<grid, TH, 0, g->q>>>(p);
        else attn_prefill_flat_kernel<D, false, 0><<<grid, TH, 0, g->q>>>(p);
    } else if (kt == 3) {
        if (p.qt != 2) attn_prefill_flat_kernel<D, true, 0, true><<<grid, TH, 0, g->q>>>(p);
        else attn_prefill_flat_kernel<D, true, 0><<<grid, TH, 0, g->q>>>(p);
    } else if (kt == 1) {
        attn_prefill_flat_kernel<D, false, 1><<<grid, TH, 0, g->q>>>(p);
    } else {
        attn_prefill_flat_kernel<D, false, 2><<<grid, TH, 0, g->q>>>(p);
    }
}

template <int D, int PW>
int launch_prefill(ns_gpu* g, int kt, const PrefillParams& p, dim3 grid, bool stream) {
    constexpr int TH = PW * 64;
    if constexpr (D == 128) {
        // (the streaming forms: half rows with either work-group size, bfloat16 rows - short passes keep them - with 4 waves)
        if (stream && kt == 0) {
            attn_prefill_kernel<D, false, 0, PW, false, true><<<grid, TH, 0, g->q>>>(p);
            return 0;
        }
        if constexpr (PW == 4) {
            if (stream && kt == 3) {
                if (p.qt != 2) attn_prefill_kernel<D, true, 0, PW, true, true><<<grid, TH, 0, g->q>>>(p);
                else attn_prefill_kernel<D, true, 0, PW, false, true><<<grid, TH, 0, g->q>>>(p);
                return 0;
            }
        }
    }
    if (kt == 0) {
        attn_prefill_kernel<D, false, 0, PW><<<grid, TH, 0, g->q>>>(p);
    } else if (kt == 3) {
        if (p.qt != 2) attn_prefill_kernel<D, true, 0, PW, true><<<grid, TH, 0, g->q>>>(p);
        else attn_prefill_kernel<D, true, 0, PW><<<grid, TH, 0, g->q>>>(p);
    } else if (kt == 1) {
        attn_prefill_kernel<D, false, 1, PW><<<grid, TH, 0, g->q>>>(p);
    } else if constexpr (D == 256 || PW == 4) {
        attn_prefill_kernel<D, false, 2, PW><<<grid, TH, 0, g->q>>>(p);
    } else {
        // (a q4_0 tile of 128-value rows is 256 chunks: fewer than 8 waves have threads - the caller takes 4 waves)
        return ns_fail("ns_attn_prompt: internal: q4_0 rows of 128 values take 4 waves");
    }
    return 0;
}


// How a pass runs: its form (fl.waves 0: whole waves of one head's rows), key splits, whether its rows are widened first, waves a work-group
struct PromptPlan {
    FlatPlan fl;
    int64_t ns = 1, kbs = 0, k0 = 0;                              // key splits: [k0 + y kbs, k0 + (y + 1) kbs), y < ns
    int64_t kf = 0, keys = 0;                                     // the pass's first key and how many there are from it
    size_t part_bytes = 0, wide_bytes = 0;                        // of the scratch: partials; widened keys, or values
    bool widen = false;
    bool stream = false;                                          // one work-group reads a key, once: the streaming cache policy
    int waves = 4, pack = 1;                                      // of a work-group; query heads it holds (rows end to end: fl's)
};
// The plan of a pass whose arguments have been checked, with `own` floats of scratch: arithmetic on the sizes alone
PromptPlan prompt_plan(size_t own, int qt, int kt, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t p0, int64_t win, int causal, int64_t kfirst) {
    // (512 work-groups of 256 rows: two for each of the chip's 256 CUs; NS_PREFILL_WAVES = 4 or 8 overrides, 16 - 12 with
    // work-groups of 4 waves, unsplit - lays rows end to end: tuning, tests)
    PromptPlan pl;
    int64_t& sns = pl.ns;
    // heads a work-group of a short pass holds (pack_of): with 4 waves, or - where only 8 waves let a group share at all,
    // 5 or 7 heads - with 8
    const int64_t pk4 = pack_of(T, Hq / Hkv, D, 4), pk8 = pack_of(T, Hq / Hkv, D, 8);
    const bool wide_pack = pk8 > 2 * pk4 && (pk4 == 1 || p0 + T >= 8192);     // (a group that shares with 4 waves too: only behind a long context)
    // (heads of 256, up to 64 rows behind a long context: 8 waves - twice the heads a work-group, and one work-group a CU
    // is all its LDS admits - 17 rows x 16 / 2 heads behind 131072 keys 130 -> 92 us)
    const bool long256 = D == 256 && T <= 64 && p0 + T >= 16384;
    const int64_t pkp = wide_pack || long256 ? pk8 : pk4;
    const int64_t wkf = pl.kf = kfirst >= 0 ? kfirst : win > 0 ? std::max<int64_t>(0, p0 + 1 - win) : 0, wn = pl.keys = p0 + T - wkf;
    const int64_t waves = ns_tune_get(NS_TUNE_PREFILL_WAVES), fit_splits = (int64_t) (own / (size_t) (T * Hq * (D + 2)));
    FlatPlan& fl = pl.fl;
    if (T * (Hq / Hkv) < ((int64_t) 1 << 31) / (Hq / Hkv)) {
        // (no more splits than leave room to widen the rows behind the partials: 8224 rows x 64 / 8 bfloat16 heads behind 60000 keys, three splits
        // that left none against two: 21.4 -> 14.5 ms, q8_0 16.3 -> 14.9, q4_0 16.0 -> 14.6)
        const size_t wide = kt != 0 ? (size_t) (Hkv * wn * D) + 64 : 0;
        const int64_t most = std::min<int64_t>(128, wide < own ? (int64_t) ((own - wide) / (size_t) (T * Hq * (D + 2))) : fit_splits);
        if (waves == 0) rows_form(fl, kt, T, Hq, Hkv, D, p0, causal ? win : 0, kfirst, wn, most);
        else if (waves == 16) flat_plan(fl, false, kt, T, Hq, Hkv, D, p0, wn, most);
        else if (waves == 12 && D == 128) fl.cut(T, Hq / Hkv, D, 4);
    }
    const bool flat = fl.waves > 0;
    // Key splits. A pass of few rows over a long context - a chunk of a prompt behind 32K tokens, a long draft block - has
    // too few (row block, head) pairs to fill the chip, each walking every key: its keys are cut into ns splits of whole
    // tiles, a work-group a (row block, head, split), the partials merged by the decode path's merge kernel. ns is
    // decided from the pass alone (128-row blocks x heads against ~512 work-groups; splits no shorter than the context's length warrants), not
    // from the work-group size, so both sizes sum a row in the same order. The partials live in the library's own
    // scratch (the prompt entry points have no scratch argument): what fits bounds ns.
    {
        const int64_t kf = wkf, keys = wn;
        const int64_t pairs = ((T + 127) / 128) * Hq / pkp;
        // (how far a context is worth cutting grows with its root where the (row block, head) pairs are few - under 32:
        // splits of about 256 keys at 2048, 512 at 8192, 1024 at 32768, 2048 at 131072; shorter ones cost more in partials
        // and their merge than they save, longer ones leave a work-group a long chain of tiles; under 512 keys none. Up to
        // 64 pairs: twice that; more: 1024 keys and more. 17 rows x 32 / 8 heads behind 1024 keys 25.3 -> 17.5 us, behind 2048
        // 28.1 -> 20.2, behind 8192 32.8 -> 29.7; 128 rows behind 2048 keys 30.8 -> 26.1.
        // A pass about as long as its context is mostly diagonal - its row blocks see different key counts, and equal cuts
        // of the keys leave them unequal work - and is cut as a long pass is, by 1024 keys; so is a pass whose work-groups
        // hold one head's few rows, three waves of four idle: 17 rows x 40 / 8 heads behind 8192 keys 42 us in 8 splits, 49 in 13)
        const bool filled = pkp > 1 || T > (D == 128 ? 64 : 32);      // (rows for three of 4 waves of 32 rows, or of 16)
        const int64_t root = keys < 512 ? 1 : (int64_t) (0.177 * std::sqrt((double) keys));
        // (few pairs: at least the splits that give every CU a work-group, down to a tile or 2 T keys a split - the partials
        // grow with the rows - 17 rows x 8 / 1 heads behind 32768 keys in 32 splits 30.0 us, in 128 20.3; 32 / 8 heads behind
        // 8192 keys in 16 24.7, in 32 21.3; 17 rows x 4 / 4 heads, a head's few rows a work-group, behind 8192 keys in 8
        // 32.4, in 64 15.4. Heads of 256 - one work-group a CU - take exactly those: 40 rows x 16 / 2 heads behind 131072
        // keys in 32 splits 163 us, in 64 175)
        const int64_t fill = keys < 512 ? 1 : std::min<int64_t>((256 + pairs - 1) / pairs, keys / std::max<int64_t>(KT_TILE, 2 * T));
        const int64_t by_keys = p0 < 2 * T || pairs > 64 ? keys / 1024
                                : pairs < 32         ? (D == 256 ? std::max<int64_t>(fill, 1) : std::max(root, fill))
                                : !filled            ? keys / 1024
                                                     : std::max(keys / 1024, root / 2);
        const int64_t aim = 512;
        int64_t ns = std::min<int64_t>({(aim + pairs - 1) / pairs, by_keys, 128,
                                        (int64_t) (own / (size_t) (T * Hq * (D + 2)))});
        // (a pass the context dominates - equal work-groups - whose count would fill the chip's 512 places unevenly, say 640:
        // cut further, to about two and a half rounds. 1024 rows x 40 heads behind 32768 keys: 740 -> 652 us; 2048 rows: 1467 -> 1280)
        // (a pass of few pairs whose splits overfill a round of the chip's places - heads of 256: one work-group a CU; 24
        // heads x 16 splits = a round and a half - is cut into fewer, to whole rounds: 33 rows x 24 / 4 heads of 256 behind
        // 8192 keys 59 -> 45 us)
        {
            const int64_t slots = D == 128 ? 512 : 256, wg = pairs * std::max<int64_t>(ns, 1);
            if (ns > 1 && wg > slots && wg <= 2 * slots && 100 * wg < 85 * ((wg + slots - 1) / slots * slots)) ns = std::max<int64_t>(1, slots / pairs);
        }
        if (p0 >= T && keys / 1024 >= 2) {
            const int64_t slots = D == 128 ? 512 : 256;
            const int64_t cap_ns = std::min<int64_t>({keys / 1024, 64, (int64_t) (own / (size_t) (T * Hq * (D + 2)))});
            auto fill_of = [&](int64_t n) { const int64_t w = pairs * n; return (double) w / (double) ((w + slots - 1) / slots * slots); };
            if (fill_of(std::max<int64_t>(ns, 1)) < 0.85) ns = std::max(ns, std::min<int64_t>((5 * slots / 2 + pairs - 1) / pairs, cap_ns));
            // (and from there the count - up to three more - whose rounds are fullest, a split more charged what its
            // partials cost against the pass, 620 / keys: 5000 rows x 32 heads behind 32768 keys are 1280 work-groups, two
            // rounds and a half; in two splits five whole ones: 2657 -> 2505 us, x 40 heads 3613 -> 3178)
            const int64_t from = std::max<int64_t>(ns, 1);
            if (p0 >= 2 * T && fill_of(from) < 0.92) {      // (behind less than two passes' keys the diagonal makes the work-groups unequal)
                double best = 0.0;
                for (int64_t n = from; n <= std::min(from + 3, std::max(cap_ns, from)); ++n) {
                    const double fill = fill_of(n) - 620.0 / (double) keys * (double) (n - from);
                    if (n == from || fill > best + 0.02) best = fill, ns = n;
                }
            }
        }
        // (few pairs of rows of 128, two work-groups a CU: a count between one and two a CU leaves some CUs two to work off while
        // others have one. The places to fill are an XCD's 64, since a split's units - a key head and row block each - go to the
        // XCDs whole: 20 / 4 heads in 25 splits are 500 work-groups, but 13 units of 5 on four of the XCDs, and a 65th waits for
        // a place to fall free: 64 rows behind 9500 keys in 17 splits 32 us, in 25 39, in 24 30. So a count whose fullest XCD holds
        // 40 - 59 work-groups, or more than 64, takes as many splits as its places hold; one of 34 - 39 too, but behind fewer
        // than 9216 keys, where the partials of two rounds cost what they save, and at 33 takes one work-group a CU; 60 - 64 stay. Over 1388
        // passes of 17 - 128 rows x 6 - 28 pairs behind 3000 - 41000 keys 5 % less time than uncut counts, none more than 7 % over; 37 rows x
        // 32 / 8 bfloat16 heads behind 13000 keys in 20 splits 45.3 us, in 32 38.4; behind 20011 in 25 50.4, in 32 46.3)
        if (const int64_t wg = pairs * ns; D == 128 && !wide_pack && pairs < 32 && p0 >= 2 * T && ns > 1 && wg > 256 && wg <= 512) {
            const int64_t heads = (T + 127) / 128 * Hkv, gw = pairs / heads, most = (heads * ns + 7) / 8 * gw;
            if (most > 32 && (most < 60 || most > 64)) {
                const int64_t places = most == 33 || (most < 40 && keys < 9216) ? 32 : 64, whole = std::max<int64_t>(1, 8 * (places / gw) / heads);
                if ((size_t) (T * Hq * (D + 2) * whole) <= own) ns = whole;
            }
        }
        if (flat) ns = fl.ns;
        // (a forced count - tests - stays within what the scratch and the merge kernel hold)
        if (const int64_t forced = ns_tune_get(NS_TUNE_PREFILL_SPLITS)) ns = std::min<int64_t>({forced, 2048, (int64_t) (own / (size_t) (T * Hq * (D + 2)))});
        if (ns >= 2) {
            pl.k0 = kf / KT_TILE * KT_TILE;
            pl.kbs = ((p0 + T - pl.k0 + ns - 1) / ns + KT_TILE - 1) / KT_TILE * KT_TILE;
            sns = (p0 + T - pl.k0 + pl.kbs - 1) / pl.kbs;
        }
    }
    // head size 256, 16-bit rows: a wave owns one 16-row tile, so 8 waves (two a SIMD, 128-row blocks) run the job 1.5 x
    // as fast as 4 (one a SIMD) whenever there are blocks enough for half the CUs
    // (heads of 128: 256-row blocks pay only where whole ones fill the chip twice over; a pass cut into key splits has few rows -
    // 64 rows x 64 heads behind 32768 keys: 476 us in 256-row blocks that are three quarters empty, 267 us in 128-row ones;
    // 256 rows: 518 against 308)
    // A cache that is not half is widened first when its rows fit the library's scratch behind the partials (below)
    pl.part_bytes = sns > 1 ? ((size_t) (T * Hq * sns * (D + 2)) * 4 + 255) / 256 * 256 : 0;
    pl.wide_bytes = (size_t) (Hkv * wn * D * 2);
    const bool own_form = ns_tune_get(NS_TUNE_PREFILL_BF16) == 1 || (ns_tune_get(NS_TUNE_PREFILL_BF16) == 0 && own_form_pays(kt, qt, D, T, Hq / Hkv, wn, flat ? &fl : nullptr));
    pl.widen = kt != 0 && !own_form && pl.part_bytes + 2 * pl.wide_bytes <= own * 4 && wn * D * 2 < (int64_t) 1 << 32;
    int& PWs = pl.waves;
    PWs = D == 128 ? (sns == 1 && ((T + 255) / 256) * Hq >= 512 ? 8 : 4) : (T > 64 && ((T + 127) / 128) * Hq * sns >= 128 ? 8 : 4);
    // (a pass cut into key splits takes 8 waves after all where its rows - some heads of them to a work-group - fill
    // every 256-row block to 70 % and the blocks the chip, one a CU: a staged tile then serves twice the rows. 128 rows x 64 / 4
    // heads behind 32768 keys 142 -> 131 us, 256 rows 260 -> 240; x 32 / 8 heads 192 rows 141 -> 130)
    // (heads of 256: 33 - 64 rows behind a long context - 128 rows of two heads to an 8-wave work-group, one staging of the
    // keys for both - 16 / 2 heads behind 32768 keys 92 -> 70 us, 32 / 8 heads 131 -> 94; behind 8192 keys the 4-wave form)
    if (long256 && sns > 1) PWs = 8;
    if (D == 128 && sns > 1 && T >= 96) {
        const int64_t rb8 = (8 / pk8) * 32, blocks8 = (T + rb8 - 1) / rb8;
        const int64_t last8 = T - (blocks8 - 1) * rb8, wg8 = blocks8 * (Hq / pk8) * sns;
        // (the last block filled like the others - 384 rows = a block and a half: 233 -> 286 us - and whole rounds of the
        // 256 CUs - 520 work-groups, 40 heads x 13 splits, are three rounds: 74 -> 80 us)
        if (10 * last8 >= 7 * rb8 && wg8 >= 256 && 100 * wg8 >= 85 * ((wg8 + 255) / 256 * 256)) PWs = 8;
    }
    if (wide_pack) PWs = 8;
    if (const int64_t forced = ns_tune_get(NS_TUNE_PREFILL_WAVES); forced == 4 || forced == 8) PWs = (int) forced;
    if (kt == 2 && D == 128 && !pl.widen) PWs = 4;                              // (a q4_0 tile of 128-value rows has chunks for 256 threads)
    // (rows end to end: half the waves over half rows only)
    const int64_t G = Hq / Hkv;
    if (fl.waves == 4 && kt != 0 && !pl.widen) fl.cut(T, G, D, 8);
    pl.pack = flat ? 1 : (int) pack_of(T, G, D, PWs);
    // (a pass whose keys are each read by one work-group - all the group's heads in it, one row block - behind a long
    // context streams them: 17 rows x 32 / 8 heads behind 131072 keys 110 -> 97 us; where several work-groups read a key
    // the streaming policy loses what they share in L2: x 64 / 4 heads 142 -> 156)
    pl.stream = D == 128 && p0 + T >= 32768 && (flat ? fl.blocks == 1 : pl.pack == G && T <= PWs / pl.pack * (rows_of((int) D, PWs) / PWs));
    return pl;
}

}  // namespace

int ns_attn_prompt_any(ns_gpu* g, const char* who, int qt, int kt, int pm, const void* q, int64_t qs, const void* kc, const void* vc, int64_t T,
                       int64_t Hq, int64_t Hkv, int64_t D, int64_t cap, int64_t p0, int64_t win, int causal, int64_t kfirst, float scale,
                       void* out) {
    NS_TRY
    const std::string w(who);
    if (T <= 0) return 0;
    if (D != 128 && D != 256) return ns_fail(w + ": heads of 128 or 256");
    if (Hkv <= 0 || Hq <= 0 || Hq % Hkv) return ns_fail(w + ": query heads a multiple of the key heads");
    if (kt < 0 || kt > 3) return ns_fail(w + ": a cache form 0 (half), 1 (q8_0), 2 (q4_0) or 3 (bfloat16)");
    if (qt < 0 || qt > 2) return ns_fail(w + ": rows of type 0 (float32), 1 (half) or 2 (bfloat16)");
    if (p0 < 0 || cap <= 0 || win < 0) return ns_fail(w + ": a position, a capacity and a window of 0 or more");
    if (kfirst > p0) return ns_fail(w + ": a block's first key lies at or before its first row");
    const int64_t need = pm ? p0 + T : (win > 0 ? std::min(p0 + T, win + T - 1) : p0 + T);
    if (need > cap) return ns_fail(w + (win > 0 ? ": the cache's ring is shorter than the window and the pass" : ": past the cache's capacity"));
    if (!q || !kc || !vc || !out) return ns_fail(w + ": a null buffer");
    if ((uintptr_t) q % 16 || qs % (qt == 0 ? 4 : 8) || (uintptr_t) out % 16) return ns_fail(w + ": query and output rows 16-byte aligned");
    const int64_t rb = kv_row_bytes(kt, D);
    // rows are fetched in 16-byte chunks: every 16-bit row keeps that alignment, q8_0 / q4_0 rows do at D = 256 (272 / 144
    // bytes; the reference's quantized prompt form is D = 256 only); at D = 128 (136 / 72 bytes) the chunks are 8-byte aligned
    if (((uintptr_t) kc | (uintptr_t) vc) % (rb % 16 ? 8 : 16)) return ns_fail(w + (rb % 16 ? ": caches 8-byte aligned" : ": caches 16-byte aligned"));
    const PromptPlan pl = prompt_plan(ns_own_floats(g), qt, kt, T, Hq, Hkv, D, p0, win, causal, kfirst);
    const int PWs = pl.waves;
    const int64_t ROWS = rows_of((int) D, PWs);
    if (T > (int64_t) 1 << 30 || ((T + ROWS - 1) / ROWS + 1) * Hq > (int64_t) 1 << 30) return ns_fail(w + ": too many rows or heads");
    if ((pm ? cap * Hkv : cap) * rb >= (int64_t) 1 << 32) return ns_fail(w + ": a key head's cache spans 4 GiB or more");
    NS_HIP(hipSetDevice(g->dev));
    PrefillParams p{};
    p.q = q;
    p.qt = qt;
    p.qs = qs;
    p.kc = (const uint8_t*) kc;
    p.vc = (const uint8_t*) vc;
    p.head_stride = pm ? rb : cap * rb;
    p.row_stride = pm ? Hkv * rb : rb;
    p.cap = cap;
    p.wrap = !pm && p0 + T > cap;
    p.T = (int) T;
    p.Hq = (int) Hq;
    p.G = (int) (Hq / Hkv);
    p.p0 = p0;
    p.win = win;
    p.causal = causal;
    p.kfirst = kfirst;
    p.sl2 = (scale > 0.0f ? scale : 1.0f / sqrtf((float) D)) * 1.4426950408889634f;
    p.out = out;
    p.ns = (int) pl.ns;
    p.kbs = pl.kbs;
    p.k0 = pl.k0;
    p.part = g->own_scratch;
    // A cache that is not half. As bfloat16 operands the softmax weights carry 8 significant bits each - the kernel then
    // enters them as two numbers, twice the second product's matrix instructions - query rows of another type are rounded
    // to 8 bits, and the query cannot take the scale (a second rounding at 8 bits shows); q8_0 / q4_0 rows are staged as
    // halfs by every work-group that reads them, once a row block and query head. So the pass's key and value rows are
    // first widened to half (bfloat16 exactly, quantized rows to the halfs the kernel's own staging builds) into the
    // library's scratch, behind the key splits' partials, and the pass runs as one over a half cache: half weights and a
    // scaled half query, as in the reference's kernels (8192 rows behind 32768 keys, rows of 256: q8_0 7062 -> 4827 us,
    // q4_0 5288 -> 4742, bfloat16 5963 -> 4666). A pass whose rows do not fit the scratch keeps the rows' own form.
    int kt_run = kt;
    if (pl.widen) {
        {
            const int64_t kf = pl.kf, n = pl.keys;
            const size_t one = pl.wide_bytes;
            uint8_t* const buf = (uint8_t*) g->own_scratch + pl.part_bytes;
            WidenParams wp{};
            wp.src[0] = (const uint8_t*) kc;
            wp.dst[0] = buf;
            wp.src[1] = (const uint8_t*) vc;
            wp.dst[1] = buf + one;
            wp.head_stride = p.head_stride;
            wp.row_stride = p.row_stride;
            wp.cap = cap;
            wp.kf = kf;
            wp.n = n;
            wp.wrap = p.wrap;
            const dim3 wgrid((unsigned) ((n * (D / 8) + 255) / 256), (unsigned) Hkv, 2u);
            if (kt == 3) {
                if (D == 128) kv_bf16_to_half_kernel<16><<<wgrid, 256, 0, g->q>>>(wp);
                else kv_bf16_to_half_kernel<32><<<wgrid, 256, 0, g->q>>>(wp);
            } else if (kt == 1) {
                if (D == 128) kv_quant_to_half_kernel<1, 16><<<wgrid, 256, 0, g->q>>>(wp);
                else kv_quant_to_half_kernel<1, 32><<<wgrid, 256, 0, g->q>>>(wp);
            } else {
                if (D == 128) kv_quant_to_half_kernel<2, 16><<<wgrid, 256, 0, g->q>>>(wp);
                else kv_quant_to_half_kernel<2, 32><<<wgrid, 256, 0, g->q>>>(wp);
            }
            NS_LAUNCHED("kv_to_half");
            // (position j of head h at buf + (h n + j - kf) 2 D: the kernel is given the address position 0 would have)
            p.kc = buf - kf * D * 2;
            p.vc = buf + one - kf * D * 2;
            p.head_stride = n * D * 2;
            p.row_stride = D * 2;
            p.wrap = 0;
            kt_run = 0;
        }
    }
    if (const FlatPlan& fl = pl.fl; fl.waves > 0) {
        const int64_t G = Hq / Hkv;
        p.tb = (int) fl.tb;
        p.gb = (int) fl.gb;
        p.ngb = (int) fl.ngb;
        p.nbf = p.ns > 1 ? (int) fl.nbf : 0;
        p.ginv = (uint32_t) (((int64_t) 1 << 32) / G + (((int64_t) 1 << 32) % G != 0));
        p.pack = p.gw = 1;
        dim3 grid((unsigned) ((Hkv * (p.nbf + (p.ngb - p.nbf) * p.ns) + 7) / 8 * 8 * p.gb));
        if (ns_profile_mark(g, 0)) return -1;
        if (D == 256) launch_flat<256>(g, kt_run, p, grid, false, false);
        else launch_flat<128>(g, kt_run, p, grid, pl.stream, fl.waves == 4);
        NS_LAUNCHED("attn_prefill");
        if (ns_profile_mark(g, 1)) return -1;
        if (p.ns > 1) {
            if (ns_attn_merge_partials(g, D, p.part, p.ns, qt, (p.nbf ? (fl.blocks - p.nbf) * fl.tb * 16 / G : T) * Hq, out)) return -1;
            return ns_profile_mark(g, 2);
        }
        return 0;
    }
    p.pack = pl.pack;
    p.gw = (int) (Hq / Hkv) / p.pack;
    const int64_t RB = (PWs / p.pack) * (ROWS / PWs);
    const int64_t units = ((T + RB - 1) / RB) * Hkv * p.ns;            // (split, row block, key head); padded to the 8 XCDs
    if ((units + 7) / 8 * 8 * p.gw >= (int64_t) 1 << 31) return ns_fail(w + ": too many work-groups");
    dim3 grid((unsigned) ((units + 7) / 8 * 8 * p.gw));
    if (ns_profile_mark(g, 0)) return -1;
    if ((D == 256 ? (PWs == 8 ? launch_prefill<256, 8>(g, kt_run, p, grid, false) : launch_prefill<256, 4>(g, kt_run, p, grid, false))
                  : PWs == 8 ? launch_prefill<128, 8>(g, kt_run, p, grid, pl.stream) : launch_prefill<128, 4>(g, kt_run, p, grid, pl.stream)) != 0)
        return -1;
    NS_LAUNCHED("attn_prefill");
    if (ns_profile_mark(g, 1)) return -1;
    if (p.ns > 1) {
        if (ns_attn_merge_partials(g, D, p.part, p.ns, qt, T * Hq, out)) return -1;
        return ns_profile_mark(g, 2);
    }
    return 0;
    NS_CATCH
}

extern "C" {

int ns_attn_prompt_t(ns_gpu* g, int qt, int kt, int pm, const void* q, int64_t qs, const void* kc, const void* vc, int64_t T, int64_t Hq,
                     int64_t Hkv, int64_t D, int64_t cap, int64_t p0, int64_t win, float scale, void* out) {
    return ns_attn_prompt_any(g, "ns_attn_prompt_t", qt, kt, pm, q, qs, kc, vc, T, Hq, Hkv, D, cap, p0, win, 1, -1, scale, out);
}

int ns_attn_prompt_plan(int qt, int kt, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t p0, int64_t win, int causal, int64_t kfirst, int64_t* plan) {
    NS_TRY
    if (T <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv || (D != 128 && D != 256) || qt < 0 || qt > 2 || kt < 0 || kt > 3 || p0 < 0 || win < 0 || kfirst > p0 || !plan ||
        p0 > (int64_t) 1 << 40 || T > (int64_t) 1 << 30 || Hq > (int64_t) 1 << 20)
        return ns_fail("ns_attn_prompt_plan: a prompt pass's rows, heads, forms and positions");
    const int64_t mib = ns_tune_get(NS_TUNE_SCRATCH_MIB);
    const PromptPlan pl = prompt_plan(mib > 0 ? std::min<size_t>(OWN_SCRATCH_FLOATS, (size_t) mib << 18) : OWN_SCRATCH_FLOATS, qt, kt, T, Hq, Hkv, D, p0, win, causal, kfirst);
    const bool flat = pl.fl.waves > 0;
    const int64_t out[8] = {flat, flat ? pl.fl.waves : pl.waves, pl.ns, pl.widen, flat ? pl.fl.blocks : 0, flat && pl.ns > 1 ? pl.fl.nbf : 0, pl.pack, pl.stream};
    std::copy(out, out + 8, plan);
    return 0;
    NS_CATCH
}

}  // extern "C"
