// Launch plumbing and small device helpers shared by the kernel files.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"

namespace hs {

// The caller of an op may hand it a pair of events (set_op_events): the first kernel the op
// launches then records `start` as it begins and every one records `stop` as it ends (the
// events ride on the dispatches, hipExtLaunchKernelGGL), so stop - start is the op's GPU time
// with no event packets between its kernels.
struct OpEvents {
    hipEvent_t start = nullptr, stop = nullptr;
    int launches = 0;
};
OpEvents &op_events();  // this host thread's

template <typename K, typename... Args>
static inline void launch_k(K kernel, dim3 grid, dim3 block, size_t lds, hipStream_t stream, Args... args) {
    OpEvents &ev = op_events();
    if (ev.stop) {
        hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)lds, stream, ev.launches == 0 ? ev.start : nullptr,
                              ev.stop, 0u, args...);
        ev.launches++;
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, args...);
    }
}

// Raises the dynamic-LDS limit of `fn` on the current device to at least `bytes`.
hipError_t allow_dynamic_lds(const void *fn, size_t bytes);

// The products of few rows (gemm_rows.hip): whether a product takes them, and the launch. `g` as
// launch_gemm has checked it.
bool gemm_rows_fits(Epi epi, const GemmArgs &g);
hipError_t launch_gemm_rows(Epi epi, const GemmArgs &g, hipStream_t stream);

// The LM head of few rows with compact logits (gemm_rows.hip).
bool head_rows_fits(const GemmArgs &g);
hipError_t launch_head_rows(const GemmArgs &g, hipStream_t stream);

// LayerNorm with 8-bit outputs in single precision (layernorm.hip).
bool layernorm_f32_fits(const LnArgs &a);
hipError_t launch_layernorm_f32(const LnArgs &a, int n_rows, hipStream_t stream);

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int32_t RES = (1 << 30) - 1;  // gpt2/mod.rs:116

typedef __attribute__((address_space(3))) void lds_void;
typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i lds_v2i;

// s_waitcnt vmcnt(N) with the other counters left at their maximum (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// A workgroup barrier for LDS data only: this wave's LDS operations complete (lgkmcnt 0), then
// s_barrier, without the wait for every outstanding global load that the release fence of
// __syncthreads brings. Global data read after it must not depend on other waves' stores.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt 63 and expcnt 7 leave those alone
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Attention: the output of row r at column col: row-major (ldo) for the op entries, or the operand panels
// of the next product (out_rows > 0). Groups of up to 16 columns from a multiple of 16 (of 4
// for 4-byte groups) lie in one panel.
__device__ __forceinline__ int8_t *attn_out(const AttnArgs &a, int r, int col) {
    return a.out + (a.out_rows ? panel_off(r, col, a.out_rows) : (size_t)r * a.ldo + col);
}

// 4 x 4 byte transpose: out[k] holds byte k of w0, w1, w2, w3 (in that order).
__device__ __forceinline__ void byte_transpose(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3,
                                               uint32_t out[4]) {
    const uint32_t t0 = __builtin_amdgcn_perm(w1, w0, 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(w3, w2, 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
    out[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
}

// x, hidden from the optimizer (a value it cannot prove invariant in a loop)
__device__ __forceinline__ int opaque_vgpr(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// v_med3_i32(x, 0, hi) for a wave-uniform hi (the compiler forms med3 only for constant bounds)
__device__ __forceinline__ int32_t clamp0_uniform(int32_t x, int32_t hi) {
    int32_t r;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(x), "s"(hi));
    return r;
}

// Butterfly moves inside a row of 16 lanes: xor 1, xor 2, then mirrors (equal inside the quads and
// octets by then), 64-bit values as two words; xor 16 and 32 across.
template <int CTRL>
__device__ __forceinline__ int32_t dpp_mov(int32_t v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int STEP>
__device__ __forceinline__ int32_t lane_move(int32_t v) {
    if constexpr (STEP == 0) return dpp_mov<0xB1>(v);        // quad_perm [1,0,3,2]
    else if constexpr (STEP == 1) return dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
    else if constexpr (STEP == 2) return dpp_mov<0x141>(v);  // row_half_mirror
    else if constexpr (STEP == 3) return dpp_mov<0x140>(v);  // row_mirror
    else return __shfl_xor(v, STEP == 4 ? 16 : 32, 64);  // across the rows
}
template <int STEP>
__device__ __forceinline__ int64_t lane_move64(int64_t v) {
    const uint32_t lo = (uint32_t)lane_move<STEP>((int32_t)v), hi = (uint32_t)lane_move<STEP>((int32_t)(v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Runs f(step) for the butterfly steps over LPR lanes.
template <int LPR, typename F>
__device__ __forceinline__ void butterfly(F f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{});
    if constexpr (LPR >= 32) f(std::integral_constant<int, 4>{});
    if constexpr (LPR >= 64) f(std::integral_constant<int, 5>{});
}

}  // namespace hs
