// indexer.hip: MiniMax-M3's block indexer, which feeds the block-sparse attention its lists: a score a block of 128 keys
// (the best key's), then the K best blocks a (row, key head). Bound: a token's pass by HBM over the indexer's half key
// rows (256 bytes a key), a prompt's by the matrix unit; selection is comparisons only and bit-exact.
//
// Reference behaviour kept: kernels/llm/minimaxm3/mm3.cpp:59-116 (scores: max over the block's keys j <= pos of iq . ik_j,
// -inf for a block wholly past the row, + 1e30 for the `local` most recent blocks; top-k: best first, the lowest index of
// equal scores, -1 once nothing finite is left, picked scores overwritten with -inf).
#include "ns_internal.hpp"
#include "ns_attn.h"
#include "ns_mla.h"
#include "kv_formats.hpp"
#include "attn_common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

constexpr int BLK = 128;

// A wave a block of 128 keys, the scores a matrix product: S[key][query] = ik . iq on v_mfma_f32_16x16x32_f16. The keys are
// halfs as they are; a float32 query enters as three halfs of the row scaled by a power of two that puts its largest feature
// below 2^15: the rounded value, the rounded rest, and 2^24 times the rest of that, whose products have a sum of their own.
// Halfs end at 2^-24, so together they hold every feature down to 2^-27 of the row's largest exactly, all 24 bits, and a
// smaller one if it has few. A row with a feature they do not hold is taken as a float32 product: a score holds no less of
// a query than that. (With the third part at the others' scale a feature under 2^-15 of the largest lost bits, one under
// 2^-39 all of them: behind keys that are zero in a large feature of 2^20 / 2^24 / 2^30 times the others, scores were off by
// 6e-7 / 1e-5 / 7e-4 of the sum of their products' sizes, the float32 product by 3e-7; 1024 rows x 4 heads behind 16384 keys
// took 53.5 us.) Of standard normal rows one in 500000 has so small a feature.
// 18 GF of a prompt's products are 55 GF of matrix work, and still far less than the
// vector unit's: 1024 rows x 4 heads behind 16384 keys 52.8 us = 1.04 PFLOP/s of matrix work, 376 us as a dot product a
// (key, query) in lanes; a token of 4 heads behind 131072 keys 8.9 us against 9.4, 4 rows of it 10.7 against 19.7.
// The block's keys stay in the wave's registers (128) while a slice of the queries, 16 at a time, passes through LDS,
// split there once for the work-group's NW blocks. The block's best key a query is a maximum over registers and 4 lanes.
constexpr int QT = 16, KT8 = BLK / 16, KB4 = BLK / 32;         // queries a tile; key tiles, feature steps

template <int NW>
__global__ __launch_bounds__(NW * 64, 8 / NW) void idx_scores_kernel(const float* __restrict__ iq, const uint16_t* __restrict__ ik, float* __restrict__ bs, int64_t TG,
                                                                int64_t G, int64_t nblk, int64_t pos0, int64_t local, int64_t tiles_a_slice) {
    constexpr int QBUF = 3 * QT * BLK * 2;                     // a query tile: 3 parts [16][128] halfs
    constexpr int HS = NW == 1 ? 1 : 2;                        // a key block is staged whole, or by halves where LDS is shared by four
    constexpr int HALF = BLK / HS * BLK * 2;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NW * HALF > 2 * QBUF ? NW * HALF : 2 * QBUF];
    __shared__ float unscale[2][QT];                           // a NaN: the parts do not hold the query
    constexpr float THIRD = 16777216.0f;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t b = (int64_t) blockIdx.x * NW + w;
    const int64_t last = pos0 + (TG - 1) / G;                  // the pass's last row sees the most keys
    const int64_t t0 = (int64_t) blockIdx.y * tiles_a_slice, t1 = std::min((TG + QT - 1) / QT, t0 + tiles_a_slice);
    // a thread's share of a query tile: 8 features of NW * 64 / 16 queries at a time
    constexpr int SH = QT * 16 / (NW * 64);
    typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));
    f4a qn[SH][2];
    auto load_q = [&](int64_t ti) {
#pragma unroll
        for (int i = 0; i < SH; ++i) {
            const int64_t q = std::min(TG - 1, ti * QT + (tid >> 4) + i * (NW * 4));
            const f4a* src = reinterpret_cast<const f4a*>(iq + q * BLK + (tid & 15) * 8);
            qn[i][0] = src[0];
            qn[i][1] = src[1];
        }
    };
    load_q(t0);

    // the block's keys: half a block at a time global -> LDS (1 KiB an instruction, key 4 i + g4, position n of its row taking
    // the 16-byte chunk n ^ (key % 16)), then as matrix operands into registers. Keys past the pass's last repeat it
    h8v kreg[KT8][KB4];
    {
        uint8_t* stage = lds + w * HALF;
#pragma unroll
        for (int h = 0; h < HS; ++h) {
#pragma unroll
            for (int i = 0; i < 32 / HS; ++i) {
                const int kk = 4 * i + g4;
                const int64_t key = std::min(last, b * BLK + h * (BLK / HS) + kk);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) (reinterpret_cast<const uint8_t*>(ik) + key * (BLK * 2) + (n ^ (kk & 15)) * 16),
                                                 (__attribute__((address_space(3))) void*) (stage + i * 1024), 16, 0, 0);
            }
            // (vmcnt(0) as the builtin: the compiler then knows that nothing is on its way into LDS any more, and puts no wait of
            // its own - for the next tile's queries - in front of the loop's first LDS read)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0F70);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int kt = 0; kt < KT8 / HS; ++kt)
#pragma unroll
                for (int kb = 0; kb < KB4; ++kb) kreg[h * (KT8 / HS) + kt][kb] = *reinterpret_cast<const h8v*>(stage + (kt * 16 + n) * (BLK * 2) + (((kb * 4 + g4) ^ n) * 16));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    }
    __syncthreads();

    auto put_q = [&](int buf) {
        auto put = [&](int i, auto any_c) __attribute__((always_inline)) {
            const int q = (tid >> 4) + i * (NW * 4), c = tid & 15;
            s8v part[3] = {};
            float down = 1.0f;
            bool odd = false;
            if constexpr (decltype(any_c)::value) {
                float f[8] = {qn[i][0][0], qn[i][0][1], qn[i][0][2], qn[i][0][3], qn[i][1][0], qn[i][1][1], qn[i][1][2], qn[i][1][3]};
                float mx = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(f[e]));
                mx = row16_max(mx);
                const int up = mx > 0.0f ? std::min(126, 15 - (int) __builtin_amdgcn_frexp_expf(mx)) : 0;
                down = __builtin_amdgcn_ldexpf(1.0f, -up);
                uint32_t left = 0;                               // bits of a feature that are in no part (an infinity or a NaN leaves some)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float r = __builtin_amdgcn_ldexpf(f[e], up);
                    left |= __builtin_bit_cast(uint32_t, fmaf(-r, down, f[e]));
#pragma unroll
                    for (int x = 0; x < 3; ++x) {
                        if (x == 2) r *= THIRD;
                        const _Float16 h = (_Float16) r;
                        part[x][e] = __builtin_bit_cast(short, h);
                        r -= (float) h;
                    }
                    left |= __builtin_bit_cast(uint32_t, r);
                }
                odd = (__ballot(left != 0) >> (lane & 48) & 0xFFFF) != 0;      // (a row's 16 lanes are neighbours in a wave)
            }
#pragma unroll
            for (int x = 0; x < 3; ++x) *reinterpret_cast<s8v*>(lds + buf * QBUF + (x * QT + q) * (BLK * 2) + ((c ^ q) * 16)) = part[x];
            if (c == 0) unscale[buf][q] = odd ? __builtin_nanf("") : down;
        };
        // (a pass of up to four queries, a token's: the tile's other rows are zeros)
        const bool few = SH > 1 && TG <= NW * 4;
        put(0, std::true_type());
        if (few) {
#pragma unroll
            for (int i = 1; i < SH; ++i) put(i, std::false_type());
        } else {
#pragma unroll
            for (int i = 1; i < SH; ++i) put(i, std::true_type());
        }
    };
    put_q(0);
    __syncthreads();
    // A tile, and whether the slice has another behind it (one wave: one tile). Its only wait on memory is for the next tile's
    // queries, at their split: the compiler counts outstanding loads along every path, so none may come round with one of its
    // own (the float32 branch ends with a wait, the last tile is a copy of its own), and the bests are stored behind the split,
    // whose wait would be for the store too. With a wait in front of the first products - for queries asked for just before -
    // and one on the last tile's store, and each part's operands read as they were needed, the same passes took 57.0 us behind
    // 16384 keys (now 52.8), 403 behind 131072 (376), 12.5 behind none (11.2)
    auto tile = [&](int64_t ti, auto more_c) __attribute__((always_inline)) {
        const int buf = (int) (ti - t0) & 1;
        if constexpr (decltype(more_c)::value) load_q(ti + 1);
        // (32-bit divisions: the host keeps rows x heads below 2^31)
        const uint32_t q0 = (uint32_t) (ti * QT), q = q0 + n, qe = (uint32_t) TG - 1, G32 = (uint32_t) G;
        const int64_t pos = pos0 + std::min(q, qe) / G32;
        const int64_t first = pos0 + q0 / G32, seen = pos0 + std::min(q0 + QT - 1, qe) / G32;    // the tile's first and last rows' positions
        float m = -INFINITY;
        if (b * BLK <= seen) {
            const int lim = (int) std::min<int64_t>(pos - b * BLK, BLK - 1);                // the row's last key in the block
            const bool cut = b * BLK + BLK - 1 > first;        // (the tile's first row does not see the whole block)
            uint32_t again = 0;                                // key tiles with a sum that is no number
            // half the block's keys at a time, a part's products while the next part's operands are read
            h8v bq[2][KB4];
            auto read = [&](int x, h8v (&to)[KB4]) __attribute__((always_inline)) {
#pragma unroll
                for (int kb = 0; kb < KB4; ++kb) to[kb] = *reinterpret_cast<const h8v*>(lds + buf * QBUF + (x * QT + n) * (BLK * 2) + (((kb * 4 + g4) ^ n) * 16));
            };
            read(2, bq[0]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f4v acc[KT8 / 2], third[KT8 / 2];
#pragma unroll
                for (int kt = 0; kt < KT8 / 2; ++kt) acc[kt] = third[kt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int x = 2; x >= 0; --x) {
                    const int now = (h * 3 + 2 - x) & 1;
                    __builtin_amdgcn_sched_barrier(0);
                    if (h == 0 || x > 0) read(x > 0 ? x - 1 : 2, bq[now ^ 1]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int kb = 0; kb < KB4; ++kb)
#pragma unroll
                        for (int kt = 0; kt < KT8 / 2; ++kt) {
                            f4v& a = x == 2 ? third[kt] : acc[kt];
                            a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kreg[h * (KT8 / 2) + kt][kb], bq[now][kb], a, 0, 0, 0);
                        }
                }
#pragma unroll
                for (int kt = 0; kt < KT8 / 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[kt][i] = fmaf(third[kt][i], 1.0f / THIRD, acc[kt][i]);
#pragma unroll
                for (int kt = 0; kt < KT8 / 2; ++kt) {
                    const float sum = (acc[kt][0] + acc[kt][1]) + (acc[kt][2] + acc[kt][3]);
                    again |= (uint32_t) __any(!(fabsf(sum) < INFINITY)) << (h * (KT8 / 2) + kt);
                }
                if (cut) {
#pragma unroll
                    for (int kt = 0; kt < KT8 / 2; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[kt][i] = (h * (KT8 / 2) + kt) * 16 + g4 * 4 + i <= lim ? acc[kt][i] : -INFINITY;
                }
#pragma unroll
                for (int kt = 0; kt < KT8 / 2; ++kt) m = fmaxf(fmaxf(fmaxf(acc[kt][0], acc[kt][1]), fmaxf(acc[kt][2], acc[kt][3])), m);
            }
            // A query whose parts do not hold it, or an infinity or a NaN among a key tile's operands - a part of a query may be 0
            // where the query is not, and the three products then say NaN where the float32 product says infinity. Those key
            // tiles - all of them for such a query - are taken again as float32 products, features 32 kb + 8 g4 + e of both
            // operands at a time. 1024 rows x 4 heads behind 16384 keys, 53 us: with a NaN in one key 67, an infinity in every
            // block 88, every query in float32 243; a token's four queries 5.8 -> 11.5 (a dot product a (key, query) in lanes
            // took 375 and 6.9 whatever the values, feature by feature in this branch 6500 - 16900 and 310)
            const float us = unscale[buf][n];
            m = us == us ? m * us : -INFINITY;
            if (__any(us != us)) again = (1u << KT8) - 1;
            if (again) {
                const f4a* src = reinterpret_cast<const f4a*>(iq + (int64_t) std::min(q, qe) * BLK + g4 * 8);
                f4a x[KB4][2];
#pragma unroll
                for (int kb = 0; kb < KB4; ++kb) {
                    x[kb][0] = src[kb * 8];
                    x[kb][1] = src[kb * 8 + 1];
                }
#pragma unroll
                for (int kt = 0; kt < KT8; ++kt) {
                    if (!(again >> kt & 1)) continue;
                    f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int kb = 0; kb < KB4; ++kb) {
                        h8v k = kreg[kt][kb];
                        asm volatile("" : "+v"(k));              // (widened here: ahead of the loop over the tiles the widened keys would spill)
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32((float) k[e], x[kb][e >> 2][e & 3], acc, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) m = fmaxf(m, kt * 16 + g4 * 4 + i <= lim ? acc[i] : -INFINITY);
                }
                __builtin_amdgcn_s_waitcnt(0x0F70);
            }
            m = rows_max(m);
        }
        if constexpr (decltype(more_c)::value) put_q(buf ^ 1);
        if (g4 == 0 && q <= qe && b < nblk) {
            if (b * BLK > pos) m = -INFINITY;
            else if (b + local > pos / BLK) m = m + 1e30f;
            bs[(int64_t) q * nblk + b] = m;
        }
    };
    if constexpr (NW > 1) {
        for (int64_t ti = t0; ti + 1 < t1; ++ti) {
            tile(ti, std::true_type());
            __syncthreads();
        }
    }
    tile(t1 - 1, std::false_type());
}

// The same for a pass of one or two queries: a work-group of 128 threads a block, a thread its key's row in registers and the dot
// products in feature order. Nothing is staged or split, and that is what the matrix form spends its time on there: 1 query
// behind 1000 / 16384 / 131072 keys 3.3 / 3.4 / 6.7 us against 4.9 / 5.0 / 8.9, 2 queries 3.9 / 4.0 / 7.6 against 4.9 / 5.0 / 9.0;
// 4 queries 6.1 / 6.3 / 9.4 against 4.9 / 5.0 / 8.9 (replays of a graph)
constexpr int FEW_QUERIES = 2;
__global__ __launch_bounds__(BLK) void idx_scores_few_kernel(const float* __restrict__ iq, const uint16_t* __restrict__ ik, float* __restrict__ bs, int TG, int64_t G,
                                                             int64_t nblk, int64_t pos0, int64_t local) {
    __shared__ float qs[FEW_QUERIES][BLK];
    __shared__ float red[FEW_QUERIES][2];
    const int64_t b = blockIdx.x;
    const int lid = threadIdx.x;
    const int64_t j = b * BLK + lid, last = pos0 + (TG - 1) / G;      // the pass's last row sees the most keys
    h8v row[BLK / 8];
    const h8v* kr = reinterpret_cast<const h8v*>(ik + std::min(j, last) * BLK);
#pragma unroll
    for (int c = 0; c < BLK / 8; ++c) row[c] = kr[c];
    for (int i = 0; i < TG; ++i) qs[i][lid] = iq[i * BLK + lid];
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < TG; ++i) {
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < BLK / 8; ++c) {
            asm volatile("" : "+v"(row[c]));                       // (widened here: ahead of the loop the widened row would cost half the waves)
#pragma unroll
            for (int e = 0; e < 8; ++e) s = fmaf(qs[i][c * 8 + e], (float) row[c][e], s);
            if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);     // (nor all of the query's reads at once)
        }
        const float v = wave_max(j <= pos0 + i / G ? s : -INFINITY);
        if ((lid & 63) == 0) red[i][lid >> 6] = v;
    }
    __syncthreads();
    if (lid < TG) {
        const int64_t pos = pos0 + lid / G;
        float m = fmaxf(red[lid][0], red[lid][1]);
        if (b * BLK > pos) m = -INFINITY;
        else if (b + local > pos / BLK) m = m + 1e30f;
        bs[lid * nblk + b] = m;
    }
}

// one wave a (row, head): K rounds of (largest score, its lowest index)
__global__ __launch_bounds__(64) void idx_topk_kernel(float* __restrict__ bs, int32_t* __restrict__ sel, int64_t nblk, int64_t K) {
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x;
    float* s = bs + row * nblk;
    for (int64_t k = 0; k < K; ++k) {
        float best = -INFINITY;
        for (int64_t b = lane; b < nblk; b += 64) best = fmaxf(best, s[b]);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) best = fmaxf(best, __shfl_xor(best, o));
        int at = 0x7fffffff;
        if (best > -INFINITY)
            for (int64_t b = lane; b < nblk; b += 64)
                if (s[b] == best) { at = (int) b; break; }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) at = min(at, __shfl_xor(at, o));
        if (lane == 0) {
            sel[row * K + k] = best > -INFINITY ? at : -1;
            if (best > -INFINITY) s[at] = -INFINITY;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the write above before the next round's reads (one wave)
        __builtin_amdgcn_s_barrier();
    }
}

__device__ __forceinline__ uint32_t order_key(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);             // a larger float, a larger key
}
// The same selection with the row's scores held in registers (VPL a lane: rows of up to 64 VPL blocks), over the few that can be
// among the K best: the K-th largest of the lanes' own largest scores, its first 16 bits, is a bound that at least K scores
// reach, and some 20 of a row do for K = 16. Those move to a lane each, and a candidate's place in the list is the number of
// candidates in front of it - no rounds, each waiting for two reductions over the wave. Rows whose candidates outgrow the
// lanes (many equal scores) and lists of more than 64 go round by round: a few compares and two wave reductions a round.
// Bound: one memory latency and a chain of some hundred instructions. 4096 rows of 136 blocks, K 16: 13.2 -> 5.8 us, 4 rows of
// 1024 blocks 18.9 -> 5.7. The chosen blocks' scores are overwritten with -inf in memory too, as the kernel above leaves them.
template <int VPL>
__global__ __launch_bounds__(64) void idx_topk_reg_kernel(float* __restrict__ bs, int32_t* __restrict__ sel, int nblk, int K) {
    __shared__ uint32_t ckey[64];
    __shared__ int cpos[64];
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x;
    float* s = bs + row * nblk;
    int32_t* out = sel + row * K;
    float v[VPL];
    // (unconditional loads at clamped places: all in flight at once)
    if (nblk > 0) {
#pragma unroll
        for (int j = 0; j < VPL; ++j) v[j] = s[std::min(lane + 64 * j, nblk - 1)];
    }
#pragma unroll
    for (int j = 0; j < VPL; ++j) v[j] = lane + 64 * j < nblk ? v[j] : -INFINITY;
    if (K <= 64) {
        // (0: nothing to choose - -inf, a NaN, past the row; the two zeros are equal scores)
        auto key = [](float f) { return f > -INFINITY ? order_key(f + 0.0f) : 0u; };
        uint32_t most = 0;
#pragma unroll
        for (int j = 0; j < VPL; ++j) most = std::max(most, key(v[j]));
        uint32_t bound = 0;
#pragma unroll
        for (int bit = 31; bit >= 16; --bit) {
            const uint32_t c = bound | 1u << bit;
            if (__popcll(__ballot(most >= c)) >= K) bound = c;
        }
        bound = std::max(bound, 1u);
        int count = 0;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const uint32_t kj = key(v[j]);
            const uint64_t in = __ballot(kj >= bound);
            const int at = count + __popcll(in & (((uint64_t) 1 << lane) - 1));
            if (kj >= bound && at < 64) {
                ckey[at] = kj;
                cpos[at] = lane + 64 * j;
            }
            count += __popcll(in);
        }
        if (count <= 64) {
            __syncthreads();                                       // (one wave: its LDS writes before its reads)
            const uint32_t ck = lane < count ? ckey[lane] : 0u;
            const int cp = lane < count ? cpos[lane] : -1;
            int rank = 0;                                          // candidates are in block order: of equal scores the earlier first
            for (int i = 0; i < count; ++i) rank += (uint32_t) __builtin_amdgcn_readlane((int) ck, i) >= ck + (i < lane ? 0u : 1u);
            if (lane < count && rank < K) {
                out[rank] = cp;
                s[cp] = -INFINITY;
            }
            if (lane >= count && lane < K) out[lane] = -1;
            return;
        }
    }
    for (int k = 0; k < K; ++k) {
        float best = -INFINITY;
#pragma unroll
        for (int j = 0; j < VPL; ++j) best = fmaxf(best, v[j]);
        best = wave_max(best);
        int at = 0x7fffffff;
        if (best > -INFINITY) {
#pragma unroll
            for (int j = VPL - 1; j >= 0; --j) at = v[j] == best ? lane + 64 * j : at;     // this lane's lowest index of it
        }
        at = wave_min(at);
        if (best > -INFINITY) {
#pragma unroll
            for (int j = 0; j < VPL; ++j)
                if (lane + 64 * j == at) {
                    v[j] = -INFINITY;
                    s[at] = -INFINITY;
                }
        }
        if (lane == 0) out[k] = best > -INFINITY ? at : -1;
    }
}

// ---- GLM's DSA indexer (kernels/llm/glm5next/glm.cpp:876-1019): pools of 4 consecutive tokens --------------------------

// the pools completed by this pass: pooled[j][c] = sum_m softmax_m(ig_m[c] + ape[m][c]) ik_m[c] over pool j's 4 members
// (positions 4 j + m; a member before pos0 comes from the ring: ik | ig at slot position % 8). A thread a (pool, feature)
__global__ __launch_bounds__(256) void glm_idx_pool_kernel(const float* __restrict__ ring, const float* __restrict__ ik, const float* __restrict__ ig,
                                                           const float* __restrict__ ape, float* __restrict__ pooled, int64_t pos0, int64_t j_lo, int64_t npool,
                                                           int64_t D) {
    const int64_t gi = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (gi >= npool * D) return;
    const int64_t j = j_lo + gi / D, c = gi % D;
    float lg[4], kv[4], mx = -INFINITY;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int64_t pp = 4 * j + m;
        const float* k = pp >= pos0 ? ik + (pp - pos0) * D : ring + (pp % 8) * 2 * D;
        const float* gg = pp >= pos0 ? ig + (pp - pos0) * D : ring + (pp % 8) * 2 * D + D;
        kv[m] = k[c];
        lg[m] = gg[c] + ape[m * D + c];
        mx = fmaxf(mx, lg[m]);
    }
    float sum = 0.0f, acc = 0.0f;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const float e = expf(lg[m] - mx);
        sum += e;
        acc += e * kv[m];
    }
    pooled[j * D + c] = acc / sum;
}

// the ring takes the pass's last (up to 8) tokens: ik | ig at slot position % 8
__global__ __launch_bounds__(256) void glm_idx_ring_kernel(float* __restrict__ ring, const float* __restrict__ ik, const float* __restrict__ ig, int64_t pos0,
                                                           int64_t first, int64_t rows, int64_t D) {
    const int64_t gi = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (gi >= rows * D) return;
    const int64_t pp = first + gi / D, c = gi % D;
    ring[(pp % 8) * 2 * D + c] = ik[(pp - pos0) * D + c];
    ring[(pp % 8) * 2 * D + D + c] = ig[(pp - pos0) * D + c];
}

// score[r][j0 + jj] = sum_h relu(S[r H + h][jj]) w[r][h] in head order for the pools row r sees, -inf for the others. A thread
// a (row, pool), 16 heads' products on their way at a time: a step of two rows is one memory latency or two and little
// else (2 rows x 32 heads x 25000 pools: 11.7 us with a load a head in turn, 3.4 so; 128 rows 121 -> 73)
__global__ __launch_bounds__(256) void glm_idx_score_kernel(const float* __restrict__ S, const float* __restrict__ w, float* __restrict__ score, int64_t H,
                                                            int64_t j0, int64_t n, int64_t ld, int64_t pos0) {
    constexpr int HB = 16;
    const int64_t r = blockIdx.y, jj = (int64_t) blockIdx.x * 256 + threadIdx.x, j = j0 + jj;
    if (jj >= n) return;
    float s = -INFINITY;
    if (j < (pos0 + r + 1) / 4) {
        s = 0.0f;
        const float* col = S + r * H * n + jj;
        const float* wr = w + r * H;
        int64_t h = 0;
        for (; h + HB <= H; h += HB) {
            float x[HB];
#pragma unroll
            for (int i = 0; i < HB; ++i) x[i] = col[(h + i) * n];
#pragma unroll
            for (int i = 0; i < HB; ++i) s += fmaxf(x[i], 0.0f) * wr[h + i];
        }
        for (; h < H; ++h) s += fmaxf(col[h * n], 0.0f) * wr[h];
    }
    score[r * ld + j] = s;
}

// the K highest of a row's n scores as positions in ascending order, ties at the K-th value to the lowest positions: a
// radix select over the floats' order-preserving keys (4 digits of 8 bits, a histogram a digit in LDS), then one ordered
// compaction - every thread its own run of positions, two scans over the work-group, no atomics in what is written, so
// the list (and the sums of the attention that reads it) is the same every run. A work-group of 1024 a row.
constexpr int TOPK_WG = 1024, TOPK_NH = 16;
// exclusive prefix sum of one value a thread over the work-group (the total to every thread through `total`)
__device__ uint32_t wg_exclusive_scan(uint32_t v, uint32_t* wsum, uint32_t& total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int i = 0; i < TOPK_WG / 64; ++i) {
        const uint32_t t = wsum[i];
        if (i < wv) before += t;
        all += t;
    }
    __syncthreads();
    total = all;
    return before + x - v;
}
__global__ __launch_bounds__(TOPK_WG) void glm_topk_kernel(const float* __restrict__ score, int32_t* __restrict__ sel, int64_t n, int64_t ld, int64_t K) {
    __shared__ uint32_t hist[TOPK_NH * 256];
    __shared__ uint32_t st[3];                                     // prefix, mask, still needed
    __shared__ uint32_t wsum[TOPK_WG / 64];
    const int64_t r = blockIdx.x;
    const int lid = threadIdx.x;
    const float* row = score + r * ld;
    if (lid == 0) {
        st[0] = 0;
        st[1] = 0;
        st[2] = (uint32_t) K;
    }
    uint32_t* mine = hist + (lid % TOPK_NH) * 256;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (int b = lid; b < TOPK_NH * 256; b += TOPK_WG) hist[b] = 0;
        __syncthreads();
        const uint32_t prefix = st[0], mask = st[1];
        for (int64_t j = lid; j < n; j += TOPK_WG) {
            const uint32_t k = order_key(row[j]);
            if ((k & mask) == prefix) atomicAdd(&mine[(k >> shift) & 255], 1u);
        }
        __syncthreads();
        if (lid < 256) {
            uint32_t c = 0;
            for (int m = 0; m < TOPK_NH; ++m) c += hist[m * 256 + lid];
            hist[lid] = c;
        }
        __syncthreads();
        if (lid == 0) {
            // the digit, from the top, at which the count of keys at or above it reaches what is still needed
            const uint32_t need = st[2];
            uint32_t above = 0;
            int d = 255;
            for (; d > 0; --d) {
                if (above + hist[d] >= need) break;
                above += hist[d];
            }
            st[0] = prefix | ((uint32_t) d << shift);
            st[1] = mask | (255u << shift);
            st[2] = need - above;
        }
        __syncthreads();
    }
    const uint32_t kth = st[0], ties = st[2];
    const int64_t seg = (n + TOPK_WG - 1) / TOPK_WG, j0 = std::min<int64_t>(n, lid * seg), j1 = std::min<int64_t>(n, j0 + seg);
    uint32_t gt = 0, eq = 0;
    for (int64_t j = j0; j < j1; ++j) {
        const uint32_t k = order_key(row[j]);
        gt += k > kth;
        eq += k == kth;
    }
    uint32_t total;
    const uint32_t eq_before = wg_exclusive_scan(eq, wsum, total);
    const uint32_t eq_take = eq_before >= ties ? 0u : std::min(eq, ties - eq_before);
    uint32_t at = wg_exclusive_scan(gt + eq_take, wsum, total);
    uint32_t eq_left = eq_take;
    for (int64_t j = j0; j < j1; ++j) {
        const uint32_t k = order_key(row[j]);
        if (k > kth || (k == kth && eq_left > 0)) {
            if (k == kth) --eq_left;
            if (at < (uint32_t) K) sel[r * K + at] = (int32_t) j;
            ++at;
        }
    }
}

// an inclusive running sum over a wave's lanes: within rows of 16 by row shifts, then the rows' last lanes broadcast on
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    auto dpp = [](uint32_t x, auto ctrl, auto rows) { return (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, decltype(ctrl)::value, decltype(rows)::value, 0xF, false); };
    v += dpp(v, std::integral_constant<int, 0x111>(), std::integral_constant<int, 0xF>());
    v += dpp(v, std::integral_constant<int, 0x112>(), std::integral_constant<int, 0xF>());
    v += dpp(v, std::integral_constant<int, 0x114>(), std::integral_constant<int, 0xF>());
    v += dpp(v, std::integral_constant<int, 0x118>(), std::integral_constant<int, 0xF>());
    v += dpp(v, std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xA>());     // rows 1 and 3 add row 0's, row 2's last
    return v + dpp(v, std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xC>()); // rows 2 and 3 add lane 31's
}
// the sum of the words of the waves before this one (one LDS read and a wave sum; a walk over them is 16 LDS latencies)
__device__ __forceinline__ uint32_t sum_before(const uint32_t* words, int wv) {
    const int lane = threadIdx.x & 63;
    return wave_reduce_u32(lane < wv ? words[lane] : 0u, [](uint32_t a, uint32_t b) { return a + b; });
}

// The K-th largest of the work-group's keys (fewer than K: the smallest) and how many keys of that value the K largest hold,
// by PASSES digits of 11, 11 and 10 bits (with 2: the first 22 bits, the last 10 zero): the first is sign, exponent and two
// bits of the mantissa, so the later ones are counted over few keys. each(f) calls f(key) for every key of the calling
// thread. The histogram - zero on entry and on return - has NC copies (lane % NC, 2049 words apart: lanes that meet in a
// digit meet in no bank); a thread adds up two digits and a suffix scan finds the one the K-th key has.
template <int NC, int PASSES, typename F>
__device__ __forceinline__ void kth_key(uint32_t K, uint32_t* hist, uint32_t* st, uint32_t* wsum, F each, uint32_t& kth, uint32_t& ties) {
    constexpr int BINS = 2048, CS = BINS + 1;
    const int lid = threadIdx.x, lane = lid & 63, wv = lid >> 6;
    uint32_t* const mine = hist + (lane % NC) * CS;
    uint32_t prefix = 0, mask = 0, need = K;
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
        const uint32_t field = pass == 2 ? 1023u : 2047u;
        each([&](uint32_t key) {
            if ((key & mask) == prefix) atomicAdd(&mine[(key >> shift) & field], 1u);
        });
        __syncthreads();
        // thread lid takes the digits d and d - 1, d = 2047 - 2 lid: their counts, then the count of every digit at or above
        const int d = BINS - 1 - 2 * lid;
        uint32_t hi = 0, lo = 0;
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            hi += hist[m * CS + d];
            lo += hist[m * CS + d - 1];
            hist[m * CS + d] = 0;
            hist[m * CS + d - 1] = 0;
        }
        uint32_t incl = wave_scan(hi + lo);
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        incl += sum_before(wsum, wv);
        const uint32_t above = incl - hi - lo;                     // keys in digits above d
        if (above < need && (incl >= need || d == 1)) {            // (digit 0 takes what is left)
            const bool first = above + hi >= need;
            st[0] = (uint32_t) (first ? d : d - 1);
            st[1] = need - above - (first ? 0u : hi);
        }
        __syncthreads();
        prefix |= st[0] << shift;
        mask |= field << shift;
        need = st[1];
    }
    kth = prefix;
    ties = need;
}

// The same selection for rows of up to PER x 1024 scores, their keys held in registers (slice i: position 1024 i + lid:
// loaded once, coalesced, all in flight). A work-group is one CU, and what a row costs is the instructions spent on each of
// its scores, so the exact selection runs over few of them: the K-th largest of the threads' own largest scores (its first
// 22 bits) is a bound that at least K scores reach - of 25000 scores and K = 512 some 700 do, wherever in the row the
// large ones sit - and those, compacted into LDS in position order, are selected from. A row whose candidates outgrow the
// LDS list (many equal scores), or a K past the threads, is selected from in full. Measured where it also took the
// longer rows that the next kernel takes now, 2 rows of 25000 scores, K 512: 28.6 us -> 12.4, of which the loads - one in turn after the other, each under its own test - were 7 and passes over all scores
// the rest.
template <int PER>
__global__ __launch_bounds__(TOPK_WG) void glm_topk_reg_kernel(const float* __restrict__ score, int32_t* __restrict__ sel, int n, int64_t ld, int K) {
    constexpr int NC = 8, CAND = 2 * TOPK_WG, NW = TOPK_WG / 64;
    static_assert(PER * NW <= TOPK_WG && PER * TOPK_WG <= 65536, "a count a thread, running sums of 16 bits");
    __shared__ uint32_t hist[NC * 2049];                           // (one copy serves the few keys of the bound and the candidates)
    __shared__ uint32_t ckey[CAND];
    __shared__ int cpos[CAND];
    __shared__ uint32_t st[2], wsum[NW], cnt[TOPK_WG];
    const int64_t r = blockIdx.x;
    const int lid = threadIdx.x, lane = lid & 63, wv = __builtin_amdgcn_readfirstlane(lid >> 6);
    const float* row = score + r * ld;
    const int per = (n + TOPK_WG - 1) / TOPK_WG;                   // slices
    for (int b = lid; b < NC * 2049; b += TOPK_WG) hist[b] = 0;
    // (every load is unconditional, its index clamped: a load under a test is waited for before the next is issued. A key of
    // 0 stands for no score: order_key gives it to no number)
    uint32_t key[PER], most = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) key[i] = __builtin_bit_cast(uint32_t, row[std::min(TOPK_WG * i + lid, n - 1)]);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        key[i] = i < per && TOPK_WG * i + lid < n ? order_key(__builtin_bit_cast(float, key[i])) : 0u;
        most = max(most, key[i]);
    }
    const uint64_t below = ((uint64_t) 1 << lane) - 1;
    __syncthreads();
    // cnt [slices][waves] -> what lies before each entry; the whole sum returned
    auto running = [&](int entries) -> uint32_t {
        __syncthreads();
        const uint32_t v = lid < entries ? cnt[lid] : 0u, incl = wave_scan(v);
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        cnt[lid] = incl - v + sum_before(wsum, wv);
        const uint32_t all = sum_before(wsum, NW);
        __syncthreads();
        return all;
    };
    // the list in position order: of the slices' keys the greater ones, and of those equal to the K-th the first `ties`. Counts
    // of both share a word (greater ones below bit 16). pos_of: -1 where a slice has no key
    uint32_t kth, ties, bound = 0;
    auto emit = [&](auto most_slices, int slices, auto key_of, auto pos_of) __attribute__((always_inline)) {
        constexpr int N = decltype(most_slices)::value;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i >= slices) continue;
            const uint32_t c = (uint32_t) __popcll(__ballot(key_of(i) > kth)) | (uint32_t) __popcll(__ballot(key_of(i) == kth && pos_of(i) >= 0)) << 16;
            if (lane == 0) cnt[i * NW + wv] = c;
        }
        running(slices * NW);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i >= slices) continue;
            const bool gt = key_of(i) > kth, eq = key_of(i) == kth && pos_of(i) >= 0;
            const uint64_t bg = __ballot(gt), be = __ballot(eq);
            if (!(bg | be)) continue;
            const uint32_t c = cnt[i * NW + wv], eq_before = (c >> 16) + (uint32_t) __popcll(be & below);
            const uint32_t at = (c & 0xFFFFu) + (uint32_t) __popcll(bg & below) + std::min(eq_before, ties);
            if ((gt || (eq && eq_before < ties)) && at < (uint32_t) K) sel[r * K + at] = pos_of(i);
        }
    };
    int count = n;
    if (K <= TOPK_WG && n > TOPK_WG) {
        kth_key<1, 2>((uint32_t) K, hist, st, wsum, [&](auto f) { f(most); }, bound, ties);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (i >= per) continue;
            const uint32_t c = (uint32_t) __popcll(__ballot(key[i] >= bound));
            if (lane == 0) cnt[i * NW + wv] = c;
        }
        count = (int) running(per * NW);
    }
    if (bound && count <= CAND) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (i >= per) continue;
            const bool in = key[i] >= bound;
            const uint64_t b = __ballot(in);
            if (in) {
                const uint32_t c = cnt[i * NW + wv] + (uint32_t) __popcll(b & below);
                ckey[c] = key[i];
                cpos[c] = TOPK_WG * i + lid;
            }
        }
        __syncthreads();
        uint32_t ck[2];
        int cp[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool in = TOPK_WG * i + lid < count;
            ck[i] = in ? ckey[TOPK_WG * i + lid] : 0u;
            cp[i] = in ? cpos[TOPK_WG * i + lid] : -1;
        }
        kth_key<1, 3>((uint32_t) K, hist, st, wsum, [&](auto f) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (cp[i] >= 0) f(ck[i]);
        }, kth, ties);
        emit(std::integral_constant<int, 2>(), 2, [&](int i) { return ck[i]; }, [&](int i) { return cp[i]; });
    } else {
        kth_key<NC, 3>((uint32_t) K, hist, st, wsum, [&](auto f) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
                if (i < per && TOPK_WG * i + lid < n) f(key[i]);
        }, kth, ties);
        emit(std::integral_constant<int, PER>(), per, [&](int i) { return key[i]; }, [&](int i) { return TOPK_WG * i + lid < n ? TOPK_WG * i + lid : -1; });
    }
}

// Keys in [base, hi] of the work-group's, the need-th largest of them among the count that are left
struct KeyRange {
    uint32_t base, hi, need, count;
};
// One digit of the way to that key: [base, hi] cut into up to 2048 parts of a power of two, the keys in each counted (a histogram in NC
// copies, as kth_key's), the range narrowed to the part that holds it. The parts are cut out of the keys' own range, so few keys share the
// last one after a single pass: the key itself is seldom needed
template <int NC, typename F>
__device__ __forceinline__ void narrow(KeyRange& r, uint32_t* hist, uint32_t* st, uint32_t* wsum, F each) {
    constexpr int BINS = 2048, CS = BINS + 1;
    const int lid = threadIdx.x, lane = lid & 63, wv = lid >> 6;
    uint32_t* const mine = hist + (lane % NC) * CS;
    const int shift = std::max(0, 21 - (int) __clz((int) (r.hi - r.base)));
    each([&](uint32_t key) {
        if (key - r.base <= r.hi - r.base) atomicAdd(&mine[(key - r.base) >> shift], 1u);
    });
    __syncthreads();
    const int d = BINS - 1 - 2 * lid;
    uint32_t hi = 0, lo = 0;
#pragma unroll
    for (int m = 0; m < NC; ++m) {
        hi += hist[m * CS + d];
        lo += hist[m * CS + d - 1];
        hist[m * CS + d] = 0;
        hist[m * CS + d - 1] = 0;
    }
    uint32_t incl = wave_scan(hi + lo);
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    incl += sum_before(wsum, wv);
    const uint32_t above = incl - hi - lo;                         // keys in parts above d
    if (above < r.need && (incl >= r.need || d == 1)) {            // (part 0 takes what is left)
        const bool first = above + hi >= r.need;
        st[0] = (uint32_t) (first ? d : d - 1);
        st[1] = r.need - above - (first ? 0u : hi);
        st[2] = first ? hi : lo;
    }
    __syncthreads();
    r.base += st[0] << shift;
    r.hi = r.base + std::min(r.hi - r.base, (1u << shift) - 1);
    r.need = st[1];
    r.count = st[2];
}

// The same selection for longer rows, of up to 4096 NV scores: a thread holds 4 neighbouring scores of each of NV slices. What a row
// costs here is the instructions a score takes on the one CU that selects from it, so a score is compared as the integer its bits are -
// the order of floats from 0 up, and the bound nearly always lies there -, its test shifted into a mask; and barriers, of which each
// digit of a selection has three, so both selections cut their digits out of the keys' own range (narrow) and take one or two. The
// candidates are collected in any order, their keys read again, and the chosen ones brought into position order by a bit a score. 2 rows
// of 25000 scores, K 512: 13.8 us as in glm_topk_reg_kernel (slices of a score a thread, order keys, two and three digits), 8.8 so.
template <int NV>
__global__ __launch_bounds__(TOPK_WG) void glm_topk_long_kernel(const float* __restrict__ score, int32_t* __restrict__ sel, int n, int64_t ld, int K, bool bounded) {
    constexpr int NC = 8, CAND = 2 * TOPK_WG, NW = TOPK_WG / 64, MAPW = NV * 4096 / 32, WPT = (MAPW + TOPK_WG - 1) / TOPK_WG;
    typedef int i4a __attribute__((ext_vector_type(4), aligned(4)));
    __shared__ uint32_t hist[NC * 2049], map_gt[MAPW], map_eq[MAPW];
    __shared__ int cpos[CAND];
    __shared__ uint32_t st[3], wsum[NW], wlo[NW], whi[NW], ncand, nabove;
    const int64_t r = blockIdx.x;
    const int lid = threadIdx.x, lane = lid & 63, wv = __builtin_amdgcn_readfirstlane(lid >> 6);
    const float* row = score + r * ld;
    // (slice i: scores 4096 i + 4 lid and on. A thread at the row's end takes its last four, and leaves the ones that are others': every
    // load unconditional)
    i4a x[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) x[i] = *reinterpret_cast<const i4a*>(row + std::min(4096 * i + 4 * lid, n - 4));
    for (int b = lid; b < 2049; b += TOPK_WG) hist[b] = 0;
    for (int b = lid; b < MAPW; b += TOPK_WG) map_gt[b] = map_eq[b] = 0;
    if (lid == 0) ncand = nabove = 0;
    // the thread's scores again, as f(order key, position, bit 4 i + c): what is done without the integers is seldom done, and out of
    // the registers all the same (the row read again a digit at a time: 64 rows of 65536 negative scores, K 512, 23.5 us for 15.4). The
    // values pass the compiler opaque: hoisted out of a digit's loop the keys would take twice the registers, and spill
    auto each = [&](auto f) __attribute__((always_inline)) {
        int first = 4 * lid;
        asm volatile("" : "+v"(first));
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                int v = x[i][c];
                asm volatile("" : "+v"(v));
                const int from = 4096 * i + first, pos = std::min(from, n - 4) + c;
                if (pos >= from) f(order_key(__builtin_bit_cast(float, v)), pos, 4 * i + c);
            }
    };
    // (no score: the lowest integer, which no bound from 0 up lets through)
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (4096 * (i + 1) > n) {
#pragma unroll
            for (int c = 0; c < 4; ++c) x[i][c] = std::min(4096 * i + 4 * lid, n - 4) + c >= 4096 * i + 4 * lid ? x[i][c] : INT32_MIN;
        }
    int top = INT32_MIN;
#pragma unroll
    for (int i = 0; i < NV; ++i) top = std::max(std::max(std::max(top, x[i][0]), std::max(x[i][1], x[i][2])), x[i][3]);
    uint32_t most = (uint32_t) top | 0x80000000u;
    if (top < 0) {                                                 // no score from 0 up: the largest of the rest
        most = 0;
        each([&](uint32_t key, int, int) { most = std::max(most, key); });
    }
    const uint32_t lo = wave_reduce_u32(most, [](uint32_t a, uint32_t b) { return std::min(a, b); });
    const uint32_t hi = wave_reduce_u32(most, [](uint32_t a, uint32_t b) { return std::max(a, b); });
    if (lane == 0) {
        wlo[wv] = lo;
        whi[wv] = hi;
    }
    __syncthreads();
    KeyRange of{wave_reduce_u32(wlo[lane % NW], [](uint32_t a, uint32_t b) { return std::min(a, b); }),
                wave_reduce_u32(whi[lane % NW], [](uint32_t a, uint32_t b) { return std::max(a, b); }), (uint32_t) K, (uint32_t) TOPK_WG};
    const uint32_t largest = of.hi;
    uint32_t count = CAND + 1;
    // the bound: the K-th largest of the threads' own largest, or a little less
    if (bounded) {
        int digits = 0;
        do narrow<1>(of, hist, st, wsum, [&](auto f) { f(most); });
        while (of.count > (K > TOPK_WG / 2 ? 4u : 32u) && of.base < of.hi && ++digits < 2);
        const uint32_t bound = of.base;
        uint64_t in = 0;                                           // bit 4 i + c: score c of slice i reaches it
        if (bound & 0x80000000u) {
            const int b = (int) (bound & 0x7FFFFFFFu);
            uint32_t m[2] = {0, 0};
#pragma unroll
            for (int i = NV - 1; i >= 0; --i)
#pragma unroll
                for (int c = 3; c >= 0; --c) m[i / 8] = m[i / 8] + m[i / 8] + (x[i][c] >= b);
            in = (uint64_t) m[1] << 32 | m[0];
        } else {
            each([&](uint32_t key, int, int bit) { in |= (uint64_t) (key >= bound) << bit; });
        }
        const uint32_t own = (uint32_t) __popcll(in), incl = wave_scan(own);
        uint32_t at = 0;
        if (lane == 63) at = atomicAdd(&ncand, incl);
        at = (uint32_t) __builtin_amdgcn_readlane((int) at, 63) + incl - own;
        for (; in && at < CAND; in &= in - 1) {
            const int bit = __ffsll((unsigned long long) in) - 1;
            cpos[at++] = std::min(4096 * (bit >> 2) + 4 * lid, n - 4) + (bit & 3);
        }
        __syncthreads();
        count = ncand;
    }
    auto choose = [&](uint32_t key, int pos) {
        if (key > of.hi) atomicOr(&map_gt[pos >> 5], 1u << (pos & 31));
        else if (key >= of.base) atomicOr(&map_eq[pos >> 5], 1u << (pos & 31));
    };
    if (count <= CAND) {
        uint32_t ck[2];
        int cp[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) cp[i] = TOPK_WG * i + lid < (int) count ? cpos[TOPK_WG * i + lid] : -1;
#pragma unroll
        for (int i = 0; i < 2; ++i) ck[i] = order_key(row[std::max(cp[i], 0)]);
        of = {of.base, largest, (uint32_t) K, count};
        do {
            narrow<1>(of, hist, st, wsum, [&](auto f) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    if (cp[i] >= 0) f(ck[i]);
            });
        } while (of.count > of.need && of.base < of.hi);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (cp[i] >= 0) choose(ck[i], cp[i]);
    } else {
        // many equal scores, or a list longer than the threads: every score. Of many equal ones the bound is the likeliest, and the K-th
        // itself where fewer than K lie above it: rows of 12000 scores, K 512, 98 of 100 zero, 21.9 -> 13.5 us, all equal 19.4 -> 12.4
        for (int b = 2049 + lid; b < NC * 2049; b += TOPK_WG) hist[b] = 0;
        if (bounded) {
            uint32_t above = 0;
            each([&](uint32_t key, int, int) { above += key > of.base; });
            above = wave_reduce_u32(above, [](uint32_t a, uint32_t b) { return a + b; });
            if (lane == 0) atomicAdd(&nabove, above);
        }
        __syncthreads();
        if (!bounded) of = {0u, largest, (uint32_t) std::min(K, n), (uint32_t) n};
        else if (nabove < (uint32_t) K) of = {of.base, of.base, (uint32_t) K - nabove, count - nabove};
        else of = {of.base + 1, largest, (uint32_t) K, nabove};
        while (of.count > of.need && of.base < of.hi) narrow<NC>(of, hist, st, wsum, [&](auto f) { each([&](uint32_t key, int, int) { f(key); }); });
        each([&](uint32_t key, int pos, int) { choose(key, pos); });
    }
    __syncthreads();
    // the chosen positions in ascending order, of the scores equal to the last the first `need`: a thread's words of the maps, counts of
    // both (greater ones below bit 16) summed over the threads before it
    uint32_t g[WPT], e[WPT], c = 0;
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
        const int w = lid * WPT + k;
        g[k] = w < MAPW ? map_gt[w] : 0u;
        e[k] = w < MAPW ? map_eq[w] : 0u;
        c += (uint32_t) __popc(g[k]) | (uint32_t) __popc(e[k]) << 16;
    }
    const uint32_t incl = wave_scan(c);
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    const uint32_t before = incl - c + sum_before(wsum, wv);
    uint32_t eq = before >> 16, at = (before & 0xFFFFu) + std::min(eq, of.need);
#pragma unroll
    for (int k = 0; k < WPT; ++k)
        for (uint32_t b = g[k] | e[k]; b; b &= b - 1) {
            const int bit = __ffs((int) b) - 1;
            const bool tie = e[k] >> bit & 1;
            if (tie && eq++ >= of.need) continue;
            if (at < (uint32_t) K) sel[r * K + at] = (lid * WPT + k) * 32 + bit;
            ++at;
        }
}

// A row's latent cells as a list (the prompt path that gathers them): row t of the pass sees, with a selection, the 4
// tokens of each of its sel_cnt[t] listed pools and then its incomplete pool's tokens 4 ((p + 1) / 4) .. p; without one
// (no counts, or a negative count) the cells 0 .. p. idx [T][NC] takes the first NC of them (0 past their end), n [T]
// their count, at most NC (kernels/llm/glm5next/glm.cpp:1023-1039)
__global__ __launch_bounds__(256) void glm_cells_kernel(const int32_t* __restrict__ sel, const int32_t* __restrict__ sel_cnt, int64_t T, int64_t K,
                                                        int64_t pos0, int32_t* __restrict__ idx, int32_t* __restrict__ n, int64_t NC) {
    const int64_t t = blockIdx.y;
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i >= NC) return;
    const int64_t pos = pos0 + t;
    const int64_t ns = sel_cnt ? sel_cnt[t] : -1;
    const int64_t tail0 = 4 * ((pos + 1) / 4);
    const int64_t cnt = ns < 0 ? pos + 1 : 4 * ns + (pos + 1 - tail0);
    int64_t c = 0;
    if (i < cnt) c = ns < 0 ? i : i < 4 * ns ? 4 * (int64_t) sel[t * K + i / 4] + i % 4 : tail0 + (i - 4 * ns);
    idx[t * NC + i] = (int32_t) c;
    if (i == 0) n[t] = (int32_t) std::min(cnt, NC);
}

// Row softmax of scores S [R H rows of NC]: row r's heads over its first n[r] cells, scaled; the rest of the row 0
// (kernels/llm/glm5next/glm.cpp:1041-1060). A work-group a row. VEC: 16-byte accesses (rows of a multiple of 4 cells at
// 16-byte aligned addresses), else one cell an access. Rows of up to 256 PER accesses stay in registers between the
// maximum, the sum and the division - one read and one write of the row, up to 32768 cells: the long rows of a prompt's
// chain are this kernel's everyday case - longer ones are read three times (PER = 0)
template <int PER, bool VEC>
__global__ __launch_bounds__(256) void glm_softmax_masked_kernel(float* __restrict__ S, int64_t H, int64_t NC, const int32_t* __restrict__ n, float scale) {
    constexpr int W = VEC ? 4 : 1;
    typedef float fw __attribute__((ext_vector_type(W)));
    __shared__ float red[8];
    const int64_t rh = blockIdx.x, r = rh / H;
    float* row = S + rh * NC;
    const int64_t m = std::min<int64_t>(std::max<int32_t>(n[r], 0), NC);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // access j of this thread: cells i0 .. i0 + W - 1, i0 = (tid + 256 j) W
    auto load = [&](int64_t i0) {
        fw v;
        if constexpr (VEC) {
            v = i0 < m ? *reinterpret_cast<const fw*>(row + i0) : fw{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < W; ++e) v[e] = i0 + e < m ? v[e] * scale : -INFINITY;
        } else {
            v[0] = i0 < m ? row[i0] * scale : -INFINITY;
        }
        return v;
    };
    fw x[PER > 0 ? PER : 1];
    float mx = -INFINITY;
    if constexpr (PER > 0) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            x[j] = load((int64_t) (tid + 256 * j) * W);
#pragma unroll
            for (int e = 0; e < W; ++e) mx = fmaxf(mx, x[j][e]);
        }
    } else {
        for (int64_t i0 = (int64_t) tid * W; i0 < m; i0 += 256 * W) {
            const fw v = load(i0);
#pragma unroll
            for (int e = 0; e < W; ++e) mx = fmaxf(mx, v[e]);
        }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wv] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.0f;
    if constexpr (PER > 0) {
#pragma unroll
        for (int j = 0; j < PER; ++j)
#pragma unroll
            for (int e = 0; e < W; ++e) {
                x[j][e] = x[j][e] == -INFINITY ? 0.0f : expf(x[j][e] - mx);
                sum += x[j][e];
            }
    } else {
        for (int64_t i0 = (int64_t) tid * W; i0 < m; i0 += 256 * W) {
            const fw v = load(i0);
#pragma unroll
            for (int e = 0; e < W; ++e) sum += v[e] == -INFINITY ? 0.0f : expf(v[e] - mx);
        }
    }
    sum = wave_sum(sum);
    if (lane == 0) red[4 + wv] = sum;
    __syncthreads();
    sum = (red[4] + red[5]) + (red[6] + red[7]);
    auto store = [&](int64_t i0, fw v) {
        if (i0 >= NC) return;
#pragma unroll
        for (int e = 0; e < W; ++e) v[e] = i0 + e < m ? v[e] / sum : 0.0f;
        if constexpr (VEC) *reinterpret_cast<fw*>(row + i0) = v;
        else row[i0] = v[0];
    };
    if constexpr (PER > 0) {
#pragma unroll
        for (int j = 0; j < PER; ++j) store((int64_t) (tid + 256 * j) * W, x[j]);
    } else {
        for (int64_t i0 = (int64_t) tid * W; i0 < NC; i0 += 256 * W) {
            fw v = load(i0);
#pragma unroll
            for (int e = 0; e < W; ++e) v[e] = v[e] == -INFINITY ? 0.0f : expf(v[e] - mx);
            store(i0, v);
        }
    }
}

}  // namespace

extern "C" {

int ns_idx_pool(ns_gpu* g, float* ring, const float* ik, const float* ig, const float* ape, float* pooled, int64_t pos0, int64_t T, int64_t D) {
    NS_TRY
    if (T <= 0 || D <= 0) return 0;
    if (pos0 < 0) return ns_fail("ns_idx_pool: a position");
    if (!g || !ring || !ik || !ig || !ape || !pooled) return ns_fail("ns_idx_pool: a null buffer");
    NS_HIP(hipSetDevice(g->dev));
    const int64_t j_lo = pos0 / 4, j_hi = (pos0 + T) / 4;
    if (j_hi > j_lo) {
        glm_idx_pool_kernel<<<(unsigned) (((j_hi - j_lo) * D + 255) / 256), 256, 0, g->q>>>(ring, ik, ig, ape, pooled, pos0, j_lo, j_hi - j_lo, D);
        NS_LAUNCHED("idx_pool");
    }
    const int64_t first = std::max<int64_t>(pos0, pos0 + T - 8);
    glm_idx_ring_kernel<<<(unsigned) (((pos0 + T - first) * D + 255) / 256), 256, 0, g->q>>>(ring, ik, ig, pos0, first, pos0 + T - first, D);
    NS_LAUNCHED("idx_pool ring");
    return 0;
    NS_CATCH
}

int ns_idx_score(ns_gpu* g, const float* S, const float* w, float* score, int64_t T, int64_t H, int64_t j0, int64_t n, int64_t ld, int64_t pos0) {
    NS_TRY
    if (T <= 0 || n <= 0) return 0;
    if (H < 0 || j0 < 0 || ld < j0 + n || pos0 < 0) return ns_fail("ns_idx_score: heads, a pool range inside a score row, a position");
    if (!g || !S || !w || !score) return ns_fail("ns_idx_score: a null buffer");
    NS_HIP(hipSetDevice(g->dev));
    for (int64_t t0 = 0; t0 < T; t0 += 65535) {
        const int64_t nr = std::min<int64_t>(65535, T - t0);
        glm_idx_score_kernel<<<dim3((unsigned) ((n + 255) / 256), (unsigned) nr), 256, 0, g->q>>>(S + t0 * H * n, w + t0 * H, score + t0 * ld, H, j0, n, ld,
                                                                                               pos0 + t0);
    }
    NS_LAUNCHED("idx_score");
    return 0;
    NS_CATCH
}

int ns_topk(ns_gpu* g, const float* score, int32_t* sel, int64_t T, int64_t n, int64_t ld, int64_t K) {
    NS_TRY
    if (T <= 0 || K <= 0) return 0;
    // (fewer scores than K: the reference's select then takes all n, in position order, and leaves the list's rest as it was)
    if (n < 0 || ld < n || n > (int64_t) 1 << 30 || K > (int64_t) 1 << 30) return ns_fail("ns_topk: score rows at least n apart");
    if (!g || !score || !sel) return ns_fail("ns_topk: a null buffer");
    if (n == 0) return 0;
    NS_HIP(hipSetDevice(g->dev));
    if (n <= 8 * TOPK_WG) glm_topk_reg_kernel<8><<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, (int) n, ld, (int) K);
    // (lists longer than the threads, of fewer rows than CUs: with no bound to find, the kernel above is the shorter up to here and the other
    // from there. 64 rows of 8200 scores, K 2048: 10.9 / 12.9 us, of 12001 12.0 / 13.1, of 14001 13.7 / 13.2, of 16384 14.7 / 13.5; 600 rows of 8200 33.8 / 24.9)
    else if (K > TOPK_WG && T <= 256 && n <= 12 * TOPK_WG) glm_topk_reg_kernel<12><<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, (int) n, ld, (int) K);
    else if (n <= 64 * TOPK_WG) {
        // (of scores in any order so many reach the K-th largest of the threads' largest: worth looking for where the candidates' list - 2048,
        // less what rows differ by - holds them. Two rows of 8200, K 1024, with it and without: 13.9 / 10.2 us, K 870 8.1 / 10.1)
        const bool bounded = K < TOPK_WG && (double) n * (1.0 - std::pow(1.0 - (double) K / TOPK_WG, TOPK_WG / (double) n)) < 1960.0;
        if (n <= 16 * TOPK_WG) glm_topk_long_kernel<4><<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, (int) n, ld, (int) K, bounded);
        else if (n <= 32 * TOPK_WG) glm_topk_long_kernel<8><<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, (int) n, ld, (int) K, bounded);
        else glm_topk_long_kernel<16><<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, (int) n, ld, (int) K, bounded);
    }
    else glm_topk_kernel<<<(unsigned) T, TOPK_WG, 0, g->q>>>(score, sel, n, ld, K);
    NS_LAUNCHED("topk");
    return 0;
    NS_CATCH
}

int ns_mla_cells(ns_gpu* g, const int32_t* sel, const int32_t* sel_cnt, int64_t T, int64_t K, int64_t pos0, int32_t* idx, int32_t* n, int64_t NC) {
    NS_TRY
    if (T <= 0 || NC <= 0) return 0;
    if (sel_cnt && !sel) return ns_fail("ns_mla_cells: counts, but no lists");
    if (!g || !idx || !n) return ns_fail("ns_mla_cells: a null buffer");
    if (pos0 < 0 || K < 0 || pos0 + T > (int64_t) 1 << 31 || T > 65535) return ns_fail("ns_mla_cells: positions below 2^31, at most 65535 rows");
    NS_HIP(hipSetDevice(g->dev));
    glm_cells_kernel<<<dim3((unsigned) ((NC + 255) / 256), (unsigned) T), 256, 0, g->q>>>(sel, sel_cnt, T, K, pos0, idx, n, NC);
    NS_LAUNCHED("mla_cells");
    return 0;
    NS_CATCH
}

int ns_softmax_masked(ns_gpu* g, float* S, int64_t R, int64_t H, int64_t NC, const int32_t* n, float scale) {
    NS_TRY
    if (R <= 0 || H <= 0 || NC <= 0) return 0;
    if (!g || !S || !n) return ns_fail("ns_softmax_masked: a null buffer");
    if (R * H >= (int64_t) 1 << 31) return ns_fail("ns_softmax_masked: too many rows");
    NS_HIP(hipSetDevice(g->dev));
    const unsigned rows = (unsigned) (R * H);
    if (NC % 4 == 0 && (uintptr_t) S % 16 == 0) {
        if (NC <= 1024) glm_softmax_masked_kernel<1, true><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else if (NC <= 4096) glm_softmax_masked_kernel<4, true><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else if (NC <= 16384) glm_softmax_masked_kernel<16, true><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else if (NC <= 32768) glm_softmax_masked_kernel<32, true><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else glm_softmax_masked_kernel<0, true><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
    } else {
        if (NC <= 256 * 4) glm_softmax_masked_kernel<4, false><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else if (NC <= 256 * 16) glm_softmax_masked_kernel<16, false><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
        else glm_softmax_masked_kernel<0, false><<<rows, 256, 0, g->q>>>(S, H, NC, n, scale);
    }
    NS_LAUNCHED("softmax_masked");
    return 0;
    NS_CATCH
}

int ns_llm_minimaxm3_idx_scores(ns_gpu* g, const float* iq, const uint16_t* ik, float* bs, int64_t T, int64_t G, int64_t nblk, int64_t pos0, int64_t local) {
    NS_TRY
    if (T <= 0 || G <= 0 || nblk <= 0) return 0;
    if (!iq || !ik || !bs) return ns_fail("ns_llm_minimaxm3_idx_scores: a null buffer");
    if ((uintptr_t) ik % 16) return ns_fail("ns_llm_minimaxm3_idx_scores: key rows 16-byte aligned");
    if (T * G * nblk > (int64_t) 1 << 31) return ns_fail("ns_llm_minimaxm3_idx_scores: too many blocks");
    NS_HIP(hipSetDevice(g->dev));
    const int64_t TG = T * G, tiles = (TG + QT - 1) / QT, nw = tiles > 1 ? 4 : 1, gx = (nblk + nw - 1) / nw;
    if (TG <= FEW_QUERIES) {
        idx_scores_few_kernel<<<(unsigned) nblk, BLK, 0, g->q>>>(iq, ik, bs, (int) TG, G, nblk, pos0, local);
        NS_LAUNCHED("idx_scores");
        return 0;
    }
    // slices of the queries: the count whose rounds of the chip's 512 places (two work-groups a CU) times a work-group's
    // length - its query tiles, and the block's keys read once a slice, as long as 4 tiles - is least (1024 rows x 4 heads:
    // behind 16384 keys 57.7 us in 15 slices, 62.8 in 33; behind 131072 keys 417 us in 15, 619 in one)
    int64_t per = tiles, best = INT64_MAX;
    for (int64_t s = 1; s <= std::min<int64_t>(tiles, 64); ++s) {
        const int64_t len = (tiles + s - 1) / s, cost = (gx * ((tiles + len - 1) / len) + 511) / 512 * (len + 4);
        if (cost < best) best = cost, per = len;
    }
    const dim3 grid((unsigned) gx, (unsigned) ((tiles + per - 1) / per));
    if (nw == 4) idx_scores_kernel<4><<<grid, 4 * 64, 0, g->q>>>(iq, ik, bs, TG, G, nblk, pos0, local, per);
    else idx_scores_kernel<1><<<grid, 64, 0, g->q>>>(iq, ik, bs, TG, G, nblk, pos0, local, per);
    NS_LAUNCHED("idx_scores");
    return 0;
    NS_CATCH
}

int ns_llm_minimaxm3_idx_topk(ns_gpu* g, float* bs, int32_t* sel, int64_t T, int64_t G, int64_t nblk, int64_t K) {
    NS_TRY
    if (T <= 0 || G <= 0 || K <= 0) return 0;
    if (nblk < 0) return ns_fail("ns_llm_minimaxm3_idx_topk: a block count");
    if (!bs || !sel) return ns_fail("ns_llm_minimaxm3_idx_topk: a null buffer");
    NS_HIP(hipSetDevice(g->dev));
    const unsigned rows = (unsigned) (T * G);
    if (K > (int64_t) 1 << 30) return ns_fail("ns_llm_minimaxm3_idx_topk: a list length");
    if (nblk <= 64 * 8) idx_topk_reg_kernel<8><<<rows, 64, 0, g->q>>>(bs, sel, (int) nblk, (int) K);
    else if (nblk <= 64 * 32) idx_topk_reg_kernel<32><<<rows, 64, 0, g->q>>>(bs, sel, (int) nblk, (int) K);
    else if (nblk <= 64 * 128) idx_topk_reg_kernel<128><<<rows, 64, 0, g->q>>>(bs, sel, (int) nblk, (int) K);
    else idx_topk_kernel<<<rows, 64, 0, g->q>>>(bs, sel, nblk, K);
    NS_LAUNCHED("idx_topk");
    return 0;
    NS_CATCH
}

}  // extern "C"
