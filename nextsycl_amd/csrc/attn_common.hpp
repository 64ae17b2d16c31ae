// attn_common.hpp: MFMA operand types and small device helpers shared by the attention kernels (gfx950, wave64).
//
// v_mfma_f32_16x16x32_{f16,bf16}: D[16x16] += A[16x32] B[32x16]. Per lane l (n = l % 16, g = l / 16):
//   A operand: row m = n, the 8 values k = 8 g .. 8 g + 7        B operand: column n, the same 8 k
//   D / C:     column n, rows m = 4 g .. 4 g + 3 (4 floats)
// v_mfma_f32_32x32x16_{f16,bf16}: D[32x32] += A[32x16] B[16x32]. Per lane l (n = l % 32, g = l / 32):
//   A operand: row m = n, k = 8 g .. 8 g + 7                     B operand: column n, the same 8 k
//   D / C:     column n, rows m = 8 (i / 4) + 4 g + i % 4 for register i = 0..15
// ds_read_b64_tr_b16 (the transposing LDS read): in each group of 16 lanes, lane s supplies the address of 4
// consecutive 16-bit values; lane i receives element i % 4 of the rows of lanes i / 4, 4 + i / 4, 8 + i / 4, 12 + i / 4.
// With lane s pointing at &M[k0 + s / 4][m0 + 4 (s % 4)] of a row-major M[k][m], lane i receives M[k0 .. k0 + 3][m0 + i]:
// the four k of one m - an MFMA operand's packing read out of the other-major matrix.
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>
#include <cstdint>

typedef short s8v __attribute__((ext_vector_type(8)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

template <bool BF>
__device__ __forceinline__ f4v mfma16(s8v a, s8v b, f4v c) {
    if constexpr (BF) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, a), __builtin_bit_cast(b8v, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}
template <bool BF>
__device__ __forceinline__ f16v mfma32(s8v a, s8v b, f16v c) {
    if constexpr (BF) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, a), __builtin_bit_cast(b8v, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}

// float -> the kernel's 16-bit operand type, round to nearest even
template <bool BF>
__device__ __forceinline__ short to16(float f) {
    if constexpr (BF) {
        const __bf16 b = (__bf16) f;
        return __builtin_bit_cast(short, b);
    } else {
        const _Float16 h = (_Float16) f;
        return __builtin_bit_cast(short, h);
    }
}

// the transposing LDS read of 4 x 16 bits
__device__ __forceinline__ s4v lds_read_tr16(void* lds_addr) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*) lds_addr);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// The largest of three numbers (never NaN) as one instruction, in the first one's register: the compiler's copy of it there
// waits for the matrix instructions that still read or write that register, which it does not do for a register that only
// written-out code writes. (fmaxf(fmaxf(a, b), c) is the same instruction, but one the compiler schedules: the prompt kernel's
// matrix instructions then lie another way, and 8192 rows x 40 / 8 heads take 624 us where this takes 601)
__device__ __forceinline__ float max3f(float a, float b, float c) {
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
    return a;
}

// Transfers from memory straight into LDS, 1 KiB an instruction: 64 lanes x 16 bytes from base + the lane's offset to dst, both wave-
// uniform. Written out so that the compiler's wait-count pass does not see a memory instruction that writes LDS - it would make
// every later LDS read wait for all of them; the caller writes the waits. M0 holds the LDS address and takes a wait state to
// reach a transfer after the scalar unit has written it: the s_nop, which the compiler does not add in here. Transfers to
// consecutive KiB share one such write, as an instruction's immediate offset moves both its addresses: transfer i of `lds_fetch_run` reads
// base + off[i] + 1024 i. (M0 is reserved: nothing of the compiler's lives in it across these.) NT: each line read once.
#define NS_TO_LDS(OFF, BASE, AT) "\n\tglobal_load_lds_dwordx4 " OFF ", " BASE AT
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT>
__device__ __forceinline__ void lds_fetch(const uint8_t* base, uint32_t off, uint32_t dst) {
    if constexpr (NT) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%2", " nt")::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%2", "")::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
// (every lane an address of its own)
template <bool NT>
__device__ __forceinline__ void lds_fetch_any(const uint8_t* src, uint32_t dst) {
    if constexpr (NT) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "off", " nt")::"s"(dst), "v"(src) : "memory", "m0");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "off", "")::"s"(dst), "v"(src) : "memory", "m0");
}
template <bool NT, int N>
__device__ __forceinline__ void lds_fetch_run(const uint8_t* base, const uint32_t* off, uint32_t dst) {
    static_assert(N == 2 || N % 4 == 0, "two transfers, or groups of four");
    if constexpr (N == 2) {
        if constexpr (NT)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%3", " nt") NS_TO_LDS("%2", "%3", " offset:1024 nt")::"s"(dst), "v"(off[0]), "v"(off[1]), "s"(base) : "memory", "m0");
        else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%3", "") NS_TO_LDS("%2", "%3", " offset:1024")::"s"(dst), "v"(off[0]), "v"(off[1]), "s"(base) : "memory", "m0");
    } else {
        if constexpr (NT)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%5", " nt") NS_TO_LDS("%2", "%5", " offset:1024 nt") NS_TO_LDS("%3", "%5", " offset:2048 nt")
                         NS_TO_LDS("%4", "%5", " offset:3072 nt")::"s"(dst), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory", "m0");
        else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" NS_TO_LDS("%1", "%5", "") NS_TO_LDS("%2", "%5", " offset:1024") NS_TO_LDS("%3", "%5", " offset:2048")
                          NS_TO_LDS("%4", "%5", " offset:3072")::"s"(dst), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory", "m0");
        if constexpr (N > 4) lds_fetch_run<NT, N - 4>(base + 4096, off + 4, dst + 4096);
    }
}
#pragma clang diagnostic pop
#undef NS_TO_LDS

// Reductions over the 4 lanes {n, n + 16, n + 32, n + 48} that hold one query row's scores. The partner's value comes
// by v_permlane16_swap / v_permlane32_swap (vector instructions: given two copies of v they return, in every lane, the
// values of the even and the odd 16-lane row of its pair / of the lower and the upper half of the wave), not through LDS
// as a general shuffle does: no LDS round trip to wait for in the softmax's dependency chain. Same operands, same sums.
__device__ __forceinline__ void pair16(float v, float& a, float& b) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    a = __builtin_bit_cast(float, (uint32_t) r[0]);
    b = __builtin_bit_cast(float, (uint32_t) r[1]);
}
__device__ __forceinline__ void pair32(float v, float& a, float& b) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    a = __builtin_bit_cast(float, (uint32_t) r[0]);
    b = __builtin_bit_cast(float, (uint32_t) r[1]);
}
__device__ __forceinline__ float rows_max(float v) {
    float a, b;
    pair16(v, a, b);
    pair32(fmaxf(a, b), a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float rows_sum(float v) {
    float a, b;
    pair16(v, a, b);
    pair32(a + b, a, b);
    return a + b;
}

// Reductions over all 64 lanes without LDS: lane pairs inside a row of 16 through DPP (quad permutes, then the mirror
// of 8 and of 16 lanes, which pair the two halves as well as an exclusive-or would), rows through the permlane swaps.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, CTRL, 0xF, 0xF, true);
}
template <typename F>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v, F f) {
    v = f(v, dpp_u32<0xB1>(v));        // quad_perm [1, 0, 3, 2]
    v = f(v, dpp_u32<0x4E>(v));        // quad_perm [2, 3, 0, 1]
    v = f(v, dpp_u32<0x141>(v));       // row_half_mirror
    v = f(v, dpp_u32<0x140>(v));       // row_mirror
    auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = f((uint32_t) r[0], (uint32_t) r[1]);
    r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return f((uint32_t) r[0], (uint32_t) r[1]);
}
__device__ __forceinline__ float wave_max(float v) {
    return __builtin_bit_cast(float, wave_reduce_u32(__builtin_bit_cast(uint32_t, v), [](uint32_t a, uint32_t b) {
        return __builtin_bit_cast(uint32_t, fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)));
    }));
}
__device__ __forceinline__ float wave_sum(float v) {
    return __builtin_bit_cast(float, wave_reduce_u32(__builtin_bit_cast(uint32_t, v), [](uint32_t a, uint32_t b) {
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b));
    }));
}
__device__ __forceinline__ double wave_sum(double v) {
    auto halfs = [](double x) { return __builtin_bit_cast(uint64_t, x); };
    auto join = [](uint32_t lo, uint32_t hi) { return __builtin_bit_cast(double, (uint64_t) hi << 32 | lo); };
    auto add = [&](auto ctrl) { v += join(dpp_u32<decltype(ctrl)::value>((uint32_t) halfs(v)), dpp_u32<decltype(ctrl)::value>((uint32_t) (halfs(v) >> 32))); };
    add(std::integral_constant<int, 0xB1>());
    add(std::integral_constant<int, 0x4E>());
    add(std::integral_constant<int, 0x141>());
    add(std::integral_constant<int, 0x140>());
    auto lo = __builtin_amdgcn_permlane16_swap((uint32_t) halfs(v), (uint32_t) halfs(v), false, false);
    auto hi = __builtin_amdgcn_permlane16_swap((uint32_t) (halfs(v) >> 32), (uint32_t) (halfs(v) >> 32), false, false);
    v = join(lo[0], hi[0]) + join(lo[1], hi[1]);
    lo = __builtin_amdgcn_permlane32_swap((uint32_t) halfs(v), (uint32_t) halfs(v), false, false);
    hi = __builtin_amdgcn_permlane32_swap((uint32_t) (halfs(v) >> 32), (uint32_t) (halfs(v) >> 32), false, false);
    return join(lo[0], hi[0]) + join(lo[1], hi[1]);
}
// the sum over each row of 16 lanes, in every lane of the row
__device__ __forceinline__ float row16_sum(float v) {
    auto f = [](float x) { return __builtin_bit_cast(uint32_t, x); };
    auto g = [](uint32_t x) { return __builtin_bit_cast(float, x); };
    v += g(dpp_u32<0xB1>(f(v)));
    v += g(dpp_u32<0x4E>(f(v)));
    v += g(dpp_u32<0x141>(f(v)));
    return v + g(dpp_u32<0x140>(f(v)));
}
__device__ __forceinline__ float row16_max(float v) {
    auto f = [](float x) { return __builtin_bit_cast(uint32_t, x); };
    auto g = [](uint32_t x) { return __builtin_bit_cast(float, x); };
    v = fmaxf(v, g(dpp_u32<0xB1>(f(v))));
    v = fmaxf(v, g(dpp_u32<0x4E>(f(v))));
    v = fmaxf(v, g(dpp_u32<0x141>(f(v))));
    return fmaxf(v, g(dpp_u32<0x140>(f(v))));
}
__device__ __forceinline__ int wave_min(int v) {
    return (int) wave_reduce_u32((uint32_t) v, [](uint32_t a, uint32_t b) { return (uint32_t) min((int) a, (int) b); });
}

// element i of a row of query / output type QT (0 float32, 1 half, 2 bfloat16)
template <int QT>
__device__ __forceinline__ float load_q(const void* p, int64_t i) {
    if constexpr (QT == 0) return reinterpret_cast<const float*>(p)[i];
    else if constexpr (QT == 1) return (float) reinterpret_cast<const _Float16*>(p)[i];
    else return (float) reinterpret_cast<const __bf16*>(p)[i];
}
template <int QT>
__device__ __forceinline__ void store_o(void* p, int64_t i, float v) {
    if constexpr (QT == 0) reinterpret_cast<float*>(p)[i] = v;
    else if constexpr (QT == 1) reinterpret_cast<_Float16*>(p)[i] = (_Float16) v;
    else reinterpret_cast<__bf16*>(p)[i] = (__bf16) v;
}
