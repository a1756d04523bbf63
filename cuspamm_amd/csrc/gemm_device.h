// Device code shared by the multiply kernels, the gate and the selection of tau (kernels_gemm.hip, kernels_small.hip, kernels_gate.hip, kernels_tau.hip).
#pragma once
#include <type_traits>
#include <utility>

#include "spamm_internal.h"

namespace spamm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// f(integral_constant 0), ..., f(integral_constant N - 1)
template <typename F, int... I>
__device__ __forceinline__ void static_for_(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_(f, std::make_integer_sequence<int, N>{});
}

// s_waitcnt immediates (gfx9 encoding: vmcnt [3:0]+[15:14], expcnt [6:4], lgkmcnt [11:8])
constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | 0x70 | ((lgkm & 15) << 8); }

// One 1 KiB wave-load straight from global memory into LDS: lane l's 16 bytes
// land at lds_addr + IMM + 16*l, read from sbase + IMM + voff (the instruction
// offset applies to the global and to the LDS address alike).  Written as
// inline assembly so that the compiler's wait-count insertion does not see an
// LDS write it cannot disambiguate (it would put a full vmcnt(0) wait before
// every LDS read and serialise the staging ring); completion is awaited
// explicitly with s_waitcnt vmcnt before the workgroup barrier.  M0 carries
// the LDS address and is declared clobbered, so the compiler keeps nothing
// live in it across a load.  Both scalar operands must come from scalar
// instructions (as all callers' do): a VALU-written SGPR (v_readfirstlane)
// read by a vector-memory instruction within five instructions is a hazard
// the compiler does not see inside inline assembly.
template <int IMM>
__device__ __forceinline__ void dma_load(const unsigned char *sbase, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(sbase), "n"(IMM)
                 : "memory", "m0");
}

// Sum over the 64 lanes in every lane, added as shuffles down by 32, 16, .. 1 add in lane 0, without LDS operations: behind the first
// two steps a lane's partner is anywhere in its row, which repeats every 8, 4, 2 lanes.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    struct Words {
        uint32_t w[sizeof(T) / 4];
    };
    auto both = [&](auto swap) {
        Words x = __builtin_bit_cast(Words, v), lo, hi;
#pragma unroll
        for (unsigned i = 0; i < sizeof(T) / 4; i++) {
            const auto r = swap(x.w[i]);
            lo.w[i] = r[0];
            hi.w[i] = r[1];
        }
        v = __builtin_bit_cast(T, lo) + __builtin_bit_cast(T, hi);
    };
    both([](uint32_t x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
    both([](uint32_t x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    auto turned = [&](auto ctrl) {
        Words x = __builtin_bit_cast(Words, v);
#pragma unroll
        for (unsigned i = 0; i < sizeof(T) / 4; i++)
            x.w[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)x.w[i], (int)x.w[i], decltype(ctrl)::value, 0xF, 0xF, false);
        v = v + __builtin_bit_cast(T, x);
    };
    turned(std::integral_constant<int, 0x128>{});                // row rotated by 8, 4, 2, 1
    turned(std::integral_constant<int, 0x124>{});
    turned(std::integral_constant<int, 0x122>{});
    turned(std::integral_constant<int, 0x121>{});
    return v;
}

// Inclusive sum over the lanes up to each, without LDS operations
template <typename T>
__device__ __forceinline__ T wave_scan(T v) {
    auto step = [&](auto ctrl, auto rows) {
        struct Words {
            uint32_t w[sizeof(T) / 4];
        } x = __builtin_bit_cast(Words, v);
#pragma unroll
        for (unsigned i = 0; i < sizeof(T) / 4; i++)
            x.w[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x.w[i], decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
        v += __builtin_bit_cast(T, x);
    };
    constexpr std::integral_constant<int, 0xF> all{};
    step(std::integral_constant<int, 0x111>{}, all);             // from 1, 2, 4, 8 lanes below in the row
    step(std::integral_constant<int, 0x112>{}, all);
    step(std::integral_constant<int, 0x114>{}, all);
    step(std::integral_constant<int, 0x118>{}, all);
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});      // the last lane of rows 0 and 2 to the row above,
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});      // of row 1 to the two above it
    return v;
}

// Where the k lists of the macro tiles of one super tile start: the k where its diagonal would sit.
// Macro tile (mi, mj) of MT x MT output tiles.
__device__ __forceinline__ int list_anchor(int mi, int mj, int MT, int nbM, int nbK, int nbN) {
    const int sm = mi / SUPER_M, sn = mj / SUPER_N;
    const float ic = ((sm * SUPER_M + 0.5f * SUPER_M) * MT) / (float)nbM;
    const float jc = ((sn * SUPER_N + 0.5f * SUPER_N) * MT) / (float)nbN;
    const float fa = 0.5f * (ic + jc) * (float)nbK - 0.5f * SUPER_N * MT;
    const int anchor = (int)fa;
    return anchor < 0 ? 0 : (anchor > nbK - 1 ? nbK - 1 : anchor);
}

}  // namespace spamm
