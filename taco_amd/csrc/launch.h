// Launch plumbing and small device helpers shared by the kernel files.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

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

// LayerNorm with 8-bit outputs in single precision (layernorm.hip).
bool layernorm_f32_fits(const LnArgs &a);
hipError_t launch_layernorm_f32(const LnArgs &a, int n_rows, hipStream_t stream);

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int32_t RES = (1 << 30) - 1;  // gpt2/mod.rs:116

}  // namespace hs
