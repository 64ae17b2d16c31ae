// attn_sel.hip: attention of a prompt's rows over listed blocks of 128 keys (MiniMax-M3's block-sparse layers), float32
// rows, position-major half cache [position][Hkv][128], up to 16 query heads a key head.
//
// Bound: the tile steps and their waits, beside the caches' way from L2: matrix pipe 27 % busy, a wave issuing vector instructions for 27 % of its
// life and ready but not issued for 33 %; a form with 2.2 times fewer bytes from L2 took 270 us for 205. Every (row, key head) reads the keys and values of its own list - 16 blocks are 1 MB -
// so a pass of 1024 rows x 4 key heads moves 4.3 GB out of a 36 MB cache; its flops are 69 GF.
// One wave a (row, key head): the key head's query heads are one 16-row matrix tile, the wave walks its list alone and
// writes its rows itself - no partials, no merge, no barrier. What decides its speed is how often a block is found in the
// XCD's L2 (4 MB): a wave takes its blocks in ascending order, so the 256 waves of an XCD, which start together, sweep the
// cache together; neighbouring waves of an XCD serve neighbouring rows, and an XCD serves one key head where the head count
// allows. 1024 rows x 64 / 4 heads of 16 blocks: behind 16384 keys 207 us (21 TB/s), behind 4096 keys, whose heads fit L2,
// 168 us (26 TB/s), behind 65536 keys 407 us. The decode kernel, which such passes took before (a work-group a (row,
// head), blocks in list order, its loads streaming past L2, a merge behind it), spent 1323, 1219 and 1358 us; with its
// loads kept in L2, 870.
// The softmax weights enter the second product as two halfs, the rounded one and the rounded rest. A weight of 1 - a key
// at its chain's running maximum - is a half as it is, and one chain a row has fewer such keys than the decode kernel's
// chain a wave and split: with one half a weight the rows lay further from float64 than that kernel's (relative 2.82e-4
// against 2.74e-4; with two 2.10e-4, what is left being the queries' rounding to half). The second half costs 2 % behind
// 16384 keys (202 us without), 9 % where the keys fit L2 (154).
// Passes of few (row, head) pairs give each a work-group, its waves every fourth block, merged through LDS.
// A wave has one 32-key tile on its way, keys and values global -> LDS (8 KiB buffers), the next tile's keys requested as
// soon as this one's are in operand registers, its values likewise: 16 KiB in flight a wave, 8 waves a CU.
#include "ns_internal.hpp"
#include "attn_common.hpp"
#include "attn_host.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));   // (a caller's rows: any float's alignment)
constexpr int D = 128, KB = D / 32, DT = D / 16, TILE = 32, BLK = 128;
constexpr int ROW = 2 * D, STILE = TILE * ROW;                     // a cached row, a stage of 32 of them

struct SelParams {
    const float* q;
    const uint8_t* kc;
    const uint8_t* vc;
    const int32_t* sel;             // [T][Hkv][K]
    float* out;
    int64_t pos0;
    int T, Hq, Hkv, G, K;
    float sl2;                      // scale x log2(e)
};

// UW waves a (row, key head), WAVES a work-group
template <int UW, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void attn_sel_kernel(const SelParams p) {
    constexpr int UNITS = WAVES / UW;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[WAVES * 2 * STILE];
    static_assert(UW == 1 || UW == WAVES, "a unit is a wave or the work-group");
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the work-group's key head and rows: an XCD (work-group id % 8) keeps to one key head where 8 is a multiple of them
    const int x = blockIdx.x % 8, j8 = blockIdx.x / 8;
    const bool spread = 8 % p.Hkv == 0;
    const int hk = spread ? x % p.Hkv : (int) (blockIdx.x % p.Hkv);
    const int rg = spread ? j8 * (8 / p.Hkv) + x / p.Hkv : (int) (blockIdx.x / p.Hkv);
    const int t = rg * UNITS + (UW == 1 ? w : 0), uw = UW == 1 ? 0 : w;
    if (t >= p.T) return;                                          // (of a unit that is a work-group: all its waves)
    const int pos = (int) (p.pos0 + t);
    const int64_t rs = (int64_t) p.Hkv * ROW;                     // bytes between positions
    const uint8_t* kbase = p.kc + hk * ROW;
    const uint8_t* vbase = p.vc + hk * ROW;
    uint8_t* stage = lds + w * 2 * STILE;

    // the query heads as the first product's B operand: lane (n, g4) holds row n's features 32 kb + 8 g4 .. + 7
    s8v qreg[KB];
    {
        const bool live = n < p.G;
        const float* qr = p.q + ((int64_t) t * p.Hq + (int64_t) hk * p.G + (live ? n : 0)) * D + 8 * g4;
        float4 raw[KB][2];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            raw[kb][0] = *reinterpret_cast<const float4*>(qr + 32 * kb);
            raw[kb][1] = *reinterpret_cast<const float4*>(qr + 32 * kb + 4);
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const float f[8] = {raw[kb][0].x, raw[kb][0].y, raw[kb][0].z, raw[kb][0].w, raw[kb][1].x, raw[kb][1].y, raw[kb][1].z, raw[kb][1].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) qreg[kb][i] = live ? to16<false>(f[i]) : (short) 0;
        }
    }
    // A tile travels as 1 KiB an instruction, key g4 + 4 i: position n of its row takes the row's 16-byte chunk
    // n ^ (key % 16) (keys: the operand reads of 16 keys' same chunk meet no bank conflict) or n ^ 2 (key % 8) (values: the
    // transposing reads). (The key operands straight from memory - lane = key - were three times slower than the rest
    // together: neighbouring lanes then ask for 16 bytes of different rows. 1024 rows 293 us.)
    const uint32_t rs32 = (uint32_t) rs, row0 = g4 * rs32, ck = (n ^ g4) * 16, cv = (n ^ (2 * g4)) * 16;
    const uint32_t k_rd = (uint32_t) (uintptr_t) stage + n * ROW;
    const uint32_t v_rd = (uint32_t) (uintptr_t) stage + STILE + (g4 * 4 + (n >> 2)) * ROW + (n & 1) * 8;
    const int v_sw = 2 * ((g4 * 4 + (n >> 2)) & 7);

    float m_r, l_r;                                               // (l: this lane's own keys; summed over the row's lanes at the end)
    f4v o[DT];

    // a tile's keys (which 0) or values (1) on their way into their buffer: 8 requests. Keys past the row's position repeat
    // its own (the cache may end there; they are masked)
    auto request = [&](int key0, int which) __attribute__((always_inline)) {
        const int at = std::min(key0, pos), lim = pos - at;        // (the row's own block may hold tiles wholly past it)
        const uint8_t* base = (which ? vbase : kbase) + (int64_t) at * rs;
        uint8_t* dst = stage + which * STILE;
        auto to_lds = [&](const uint8_t* src, int i) __attribute__((always_inline)) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) src, (__attribute__((address_space(3))) void*) (dst + i * 1024), 16, 0, 0);
        };
        auto chunk = [&](int i) { return which ? cv ^ (128u * (i & 1)) : ck ^ (64u * (i & 3)); };
        if (lim >= TILE - 1) {
#pragma unroll
            for (int i = 0; i < 8; ++i) to_lds(base + 4 * i * rs + (row0 + chunk(i)), i);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) to_lds(base + (__umul24(std::min(g4 + 4 * i, lim), rs32) + chunk(i)), i);
        }
        asm volatile("" ::: "memory");
    };
    // a tile's step; MORE: the next tile's keys (at next0) are requested as soon as this tile's are in registers, its values
    // likewise. Requests complete in the order they were issued - K(i), V(i), K(i + 1), V(i + 1) - so a wait that leaves 8
    // outstanding has seen all but the newest stream. The LDS reads and the waits are assembly: of its own the compiler would
    // wait for every request in front of each read
    auto step = [&](int key0, int next0, auto more_c, auto two_c) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_c)::value, TWO = decltype(two_c)::value;
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        s8v k[2][KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3" : "=&v"(k[0][kb]), "=&v"(k[1][kb]) : "v"(k_rd + (((kb * 4 + g4) ^ n) * 16)), "n"(16 * ROW));
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(k[0][0]), "+v"(k[0][1]), "+v"(k[0][2]), "+v"(k[0][3]), "+v"(k[1][0]), "+v"(k[1][1]), "+v"(k[1][2]), "+v"(k[1][3])::"memory");
        if constexpr (MORE) request(next0, 0);
        f4v s[2];
#pragma unroll
        for (int kt2 = 0; kt2 < 2; ++kt2) {
            s[kt2] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) s[kt2] = mfma16<false>(k[kt2][kb], qreg[kb], s[kt2]);
        }
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = s[e >> 2][e & 3];
        if (key0 + TILE - 1 > pos) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = key0 + (e >> 2) * 16 + g4 * 4 + (e & 3) <= pos ? v[e] : -INFINITY;
        }
        const float mx = rows_max(fmaxf(max3f(v[0], v[1], v[2]), max3f(fmaxf(v[3], v[4]), v[5], fmaxf(v[6], v[7]))));
        const float mn = fmaxf(m_r, mx * p.sl2), ms = mn == -INFINITY ? 0.0f : mn;
        const bool shrink = m_r != mn;
        // the weights as two halfs, the rounded one and the rounded rest (see the head of the file)
        s8v pb, pl;
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float pv = fast_exp2(fmaf(v[e], p.sl2, -ms));
            sum += pv;
            const _Float16 h = (_Float16) pv;
            pb[e] = __builtin_bit_cast(short, h);
            pl[e] = to16<false>(pv - (float) h);
        }
        if (__any(shrink)) {
            const float c = fast_exp2(m_r - ms);
            l_r *= c;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= c;
            m_r = mn;
        }
        l_r += sum;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MORE ? 8 : 0) : "memory");
        s4v lo[DT], hi[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const uint32_t src = v_rd + (((dt * 2 + ((n & 3) >> 1)) ^ v_sw) * 16);
            asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:%3" : "=&v"(lo[dt]), "=&v"(hi[dt]) : "v"(src), "n"(16 * ROW));
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            // reads return in order: 2 (DT - 1 - dt) may still be out when this pair is needed; after the last the buffer is free
            asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo[dt]), "+v"(hi[dt]) : "n"(2 * (DT - 1 - dt)) : "memory");
            if constexpr (MORE) {
                if (dt == DT - 1) request(next0, 1);
            }
            const s8v va = {lo[dt][0], lo[dt][1], lo[dt][2], lo[dt][3], hi[dt][0], hi[dt][1], hi[dt][2], hi[dt][3]};
            if constexpr (TWO) o[dt] = mfma16<false>(va, pl, o[dt]);
            o[dt] = mfma16<false>(va, pb, o[dt]);
        }
    };

    // the list, 64 entries at a time, each lot in ascending order (holes and blocks wholly past the row behind the others
    // and left out): a lane an entry, its place = the entries before it, pushed there across the wave
    const int32_t* selp = p.sel + ((int64_t) t * p.Hkv + hk) * p.K;
    auto walk = [&](auto two_c) __attribute__((always_inline)) {
        m_r = -INFINITY, l_r = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        for (int k0 = 0; k0 < p.K; k0 += 64) {
            const int m = std::min(64, p.K - k0);
            int b = lane < m ? selp[k0 + lane] : -1;
            const bool there = b >= 0 && b <= pos / BLK;
            const int key = there ? b : INT32_MAX;
            int rank = 0;
            for (int i = 0; i < m; ++i) {
                const int o_ = __builtin_amdgcn_readlane(key, i);
                rank += o_ < key || (o_ == key && i < lane);
            }
            const int count = (int) __popcll(__ballot(there));
            if (lane >= m) rank = lane;
            const int sorted = __builtin_amdgcn_ds_permute(rank * 4, key);
            // this wave's blocks: every UW-th of the lot
            const int tiles = (count - uw + UW - 1) / UW * (BLK / TILE);
            if (tiles <= 0) continue;
            auto first_key = [&](int i) { return __builtin_amdgcn_readlane(sorted, i / (BLK / TILE) * UW + uw) * BLK + i % (BLK / TILE) * TILE; };
            int at = first_key(0);
            request(at, 0);
            request(at, 1);
            for (int i = 1; i < tiles; ++i) {
                const int next = first_key(i);
                step(at, next, std::true_type(), two_c);
                at = next;
            }
            step(at, 0, std::false_type(), two_c);
        }
    };
    walk(std::true_type());
    // An infinite value makes the second half's product a NaN - that half is 0 or of either sign - where the weight's own is the
    // infinity: features that end in no number are taken from a second walk, with the first half alone
    const float l = rows_sum(l_r);
    float odd = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) odd += (o[dt][0] + o[dt][1]) + (o[dt][2] + o[dt][3]);
    if (__any(l > 0.0f && !(fabsf(odd) < INFINITY))) {
        f4v two[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) two[dt] = o[dt];
        walk(std::false_type());
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[dt][e] = fabsf(two[dt][e]) < INFINITY ? two[dt][e] : o[dt][e];
    }
    // (a row without a weight - nothing listed, or an infinite or NaN score among them - is zeros, as the reference leaves it)
    float* const out = p.out + ((int64_t) t * p.Hq + (int64_t) hk * p.G) * D;
    if constexpr (UW == 1) {
        const float inv = 1.0f / l;
        if (n < p.G) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f4a*>(out + n * D + 16 * dt + 4 * g4) = l > 0.0f ? o[dt] * inv : f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
    } else {
        // the waves' (O, m, l) added in wave order: each parks its rows in its own value buffers (every read of them has
        // returned), then a thread a (row, 4 features)
        __shared__ float ml[UW][16][2];
        constexpr int OROW = D + 4;
        static_assert(16 * OROW * 4 <= 2 * STILE, "a wave's rows fit its buffers");
        float* ow = reinterpret_cast<float*>(stage);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f4v*>(ow + n * OROW + 16 * dt + 4 * g4) = o[dt];
        if (g4 == 0) {
            ml[w][n][0] = m_r;
            ml[w][n][1] = l;
        }
        __syncthreads();
        for (int idx = tid; idx < p.G * (D / 4); idx += WAVES * 64) {
            const int row = idx / (D / 4), c = idx % (D / 4);
            float M = -INFINITY, L = 0.0f;
#pragma unroll
            for (int k = 0; k < UW; ++k) M = fmaxf(M, ml[k][row][0]);
            f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < UW; ++k) {
                const float f = ml[k][row][0] == -INFINITY ? 0.0f : fast_exp2(ml[k][row][0] - M);
                L += ml[k][row][1] * f;
                acc += *reinterpret_cast<const f4v*>(reinterpret_cast<const float*>(lds + k * 2 * STILE) + row * OROW + c * 4) * f;
            }
            *reinterpret_cast<f4a*>(out + row * D + c * 4) = L > 0.0f ? acc * (1.0f / L) : f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
}

template <int UW, int WAVES>
int launch(ns_gpu* g, const SelParams& p) {
    constexpr int UNITS = WAVES / UW;
    const int64_t groups = (p.T + UNITS - 1) / UNITS, nx = 8 % p.Hkv == 0 ? 8 / p.Hkv : 1;
    const int64_t wgs = 8 % p.Hkv == 0 ? (groups + nx - 1) / nx * 8 : groups * p.Hkv;
    if (wgs >= (int64_t) 1 << 31) return ns_fail("ns_attn_sel_rows: too many work-groups");
    attn_sel_kernel<UW, WAVES><<<(unsigned) wgs, WAVES * 64, 0, g->q>>>(p);
    NS_LAUNCHED("attn_sel");
    return 0;
}

}  // namespace

int ns_attn_sel_rows(ns_gpu* g, const float* q, const uint16_t* kc, const uint16_t* vc, const int32_t* sel, int64_t K, float* out, int64_t T,
                     int64_t Hq, int64_t Hkv, int64_t pos0, float scale) {
    SelParams p{};
    p.q = q;
    p.kc = (const uint8_t*) kc;
    p.vc = (const uint8_t*) vc;
    p.sel = sel;
    p.out = out;
    p.pos0 = pos0;
    p.T = (int) T;
    p.Hq = (int) Hq;
    p.Hkv = (int) Hkv;
    p.G = (int) (Hq / Hkv);
    p.K = (int) K;
    p.sl2 = scale * 1.4426950408889634f;
    // (row, key head) pairs short of the chip's 2048 wave places are a work-group each: 17 rows x 4 key heads behind 16384 keys
    // 17 us against 50 with a wave each, 128 rows 31 against 51, 200 rows 55 against 53, 256 rows 58 against 54
    // Otherwise a wave a pair. A work-group of one wave spreads pairs that are no multiple of the chip's places evenly, and its place is the
    // next pair's as soon as it ends: four waves a work-group / one, 300 rows x 4 key heads behind 40000 keys - 1200 pairs - 181 / 156 us with
    // the indexer, 800 rows behind 12000 207 / 196 (two waves 169, 205). Rounds that are full anyway keep four, whose rows sweep the cache
    // together: 1024 rows behind 16384 keys 258.9 / 262.9
    const int64_t pairs = T * Hkv, places = (pairs + 2047) / 2048 * 2048;
    if (pairs < 768) return launch<4, 4>(g, p);
    return 20 * pairs >= 19 * places ? launch<1, 4>(g, p) : launch<1, 1>(g, p);
}
