// gfx950 (CDNA4, MI355X) kernels of the HardShell forward pass. Every result is the exact integer
// value of the reference CPU rule it cites (crates/hardshell/src/...); where a kernel takes a
// floating-point shortcut, it proves or checks exactness and otherwise takes the integer rule.
// Reductions are fixed-order wave/LDS trees, and the only atomics are the coder op's integer
// histogram counts in LDS, whose sums do not depend on order: results do not depend on
// scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

#include "intmath.h"
#include "kernels.h"
#include "launch.h"

namespace hs {

// ---- kernel launches and their profiling events (launch.h) --------------------------------------
OpEvents &op_events() {
    static thread_local OpEvents ev;
    return ev;
}

void set_op_events(hipEvent_t start, hipEvent_t stop) { op_events() = OpEvents{start, stop, 0}; }

int op_launches() { return op_events().launches; }

// ---- launch attributes, per kernel and device ---------------------------------------------------
// A kernel's dynamic-LDS limit is raised on the current device before its first launch that needs
// more than the default, and the resident-workgroup count of the persistent kernels is taken
// from the occupancy query once per (kernel, device, LDS size). Launchers may run on several
// host threads at once (one batch per thread), so both caches sit behind one mutex.
static std::mutex g_attr_mutex;

hipError_t allow_dynamic_lds(const void *fn, size_t bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    static std::map<std::pair<const void *, int>, size_t> raised;
    std::lock_guard<std::mutex> lock(g_attr_mutex);
    size_t &have = raised[{fn, dev}];
    if (bytes <= have) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return e;
    have = bytes;
    return hipSuccess;
}

// CUs x workgroups per CU of `fn` at `threads` threads and `lds` bytes of dynamic LDS.
static hipError_t resident_workgroups(const void *fn, int threads, size_t lds, int *out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    static std::map<std::tuple<const void *, int, size_t>, int> known;
    std::lock_guard<std::mutex> lock(g_attr_mutex);
    const auto key = std::make_tuple(fn, dev, lds);
    const auto it = known.find(key);
    if (it != known.end()) {
        *out = it->second;
        return hipSuccess;
    }
    int cus = 0, per_cu = 0;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, lds);
    if (e != hipSuccess) return e;
    const int p = (cus > 0 ? cus : 1) * (per_cu > 0 ? per_cu : 1);
    known.emplace(key, p);
    *out = p;
    return hipSuccess;
}

constexpr int64_t SCORE_LIMIT = (int64_t)1 << 40;  // gpt2/mod.rs:119

__device__ __forceinline__ int32_t med3_i32(int32_t x, int32_t lo, int32_t hi) {
    return x < lo ? lo : (x > hi ? hi : x);
}

// ---- wave reductions (wave64) -------------------------------------------------------------

__device__ __forceinline__ int64_t wave_max64(int64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        int64_t u = __shfl_xor(v, o, 64);
        v = u > v ? u : v;
    }
    return v;
}

__device__ __forceinline__ int64_t wave_sum64(int64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// =============================================================================================
// Int8 GEMM on MFMA: C[m][n] = sum_k A[m][k] * W[n][k] (both operands in panels of 64 bytes of
// K, panel_off; "NT"), exact int32 (|C| <= 2^30 for K <= 2^16, crates/hardshell/src/kernels.rs:24-29), with the
// requantize epilogue of the op fused (crates/hardshell/src/gpt2/ops.rs:107-176).
//
// Block tile 256 x 128 x 64, 256 threads = 4 waves in 2 x 2; each wave owns 128 x 64 = 8 x 4
// tiles of v_mfma_i32_16x16x64_i8. Operands go straight from global memory to LDS
// (global_load_lds_dwordx4: lane l's 16 bytes land at base + 16 l) in MFMA fragment order: a
// fragment is 16 rows x 64 k, lane l holding row l % 16, k 16 (l / 16) .. +16, so the LDS image
// of a fragment is exactly what one ds_read_b128 per lane reads back, without bank conflicts.
// A stage is the 16 A and 8 W fragments of one k-step (24 KiB); GEMM_STAGES stages form a ring,
// loads run GEMM_STAGES - 1 k-steps ahead, and each k-step has one barrier after each wave's
// own loads of that stage have landed (vmcnt).
// =============================================================================================

constexpr int GEMM_STAGES = 3;
static_assert(GEMM_BM == 256 && GEMM_BK == 64 && GEMM_NPAD % 256 == 0, "tile shape of k_gemm");

// A compile-time flag for the steps of an unrolled loop (the first k-step differs).
template <bool B>
struct Flag {
    static constexpr bool value = B;
};

// NARROW: g.fast32 holds and the shift is at least 31, so every rescaled value fits i32: with
// |a + bias| <= 2^31 - 1 and -2^31 <= mult < 2^31, |(a + bias) mult| <= (2^31 - 1) 2^31, so
// ((a + bias) mult + 2^30) >> 31 lies in [-2^31 + 1, 2^31 - 1] (larger shifts shrink it).
// BN = 128 (4 waves, 2 x 2) or 256 (8 waves, 2 x 4); every wave computes 128 x 64.
// VEC: the output rows are 16-byte aligned (checked by the launcher); the four-columns epilogues
// then stage and store 16-byte pieces, else they store each output on its own.
// BM x BN tiles: 256 x 128 (2 x 2 waves), 256 x 256 (2 x 4, the full-line
// loop), 128 x 192 (2 x 2 waves of 64 x 96) and 64 x 64 (2 x 1 waves of 32 x 64, small
// products). Each wave computes a (BM / 2) x (BN / WN) sub-tile: TI x TJ tiles of 16 x 16.
constexpr int gemm_wn(int bn) { return bn == 192 ? 2 : bn / 64; }  // waves along N
// The ring's stages: 3, or 6 for the 64 x 64 tiles with K >= 1,024 (DEEP: their
// k-steps hold little MFMA work, so more k-steps of loads stay in flight; one workgroup per CU at
// most there). Measured, GPT-2-medium unfold passes: c_attn and c_fc (K 1,024) 7-10% and
// mlp.c_proj (K 4,096) 18% faster; the GPT-2-small c_attn (K 768) 6.0 -> 6.4 us, so it keeps 3.
constexpr int gemm_stages(int bm, bool deep) { return bm == 64 && deep ? 6 : GEMM_STAGES; }
constexpr int gemm_waves(int bn) { return 2 * gemm_wn(bn); }

template <int EPI, bool NARROW, int BN, bool VEC, int BM = GEMM_BM, bool DEEP = false>
__global__ __launch_bounds__(64 * gemm_waves(BN)) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm(GemmArgs g) {
    constexpr int WN = gemm_wn(BN), WAVES = 2 * WN, TI = BM / 32, TJ = BN / WN / 16;
    constexpr int FRAGS = BM / 16 + BN / 16, LOADS = FRAGS / WAVES, NST = gemm_stages(BM, DEEP);
    static_assert(FRAGS % WAVES == 0, "whole fragments per wave");
    static_assert(NST <= 6 && (NST - 1) * LOADS < 64, "ring depth");
    static_assert(TI * TJ <= 32 && (BM == GEMM_BM || (BM == 128 && BN == 192) || (BM == 64 && BN == 64)),
                  "tile shapes");
    // The wide epilogues: tiles 2 i and 2 i + 1 of a wave hold the hi and lo planes of the same 16
    // rows (plane_row), so a wave's TI tiles are TR = TI / 2 tiles of outputs, staged and stored as
    // those of the i8 products. (With planes in adjacent rows a lane held single columns, and
    // stored 2 or 4 bytes at a time after i128 rescales: mlp.c_proj of 3,370 rows 49.7 us, 30.8
    // now; the head's 2,048-row chunk 398 -> 209 us.)
    constexpr bool WIDE = EPI == (int)Epi::ResidualWide || EPI == (int)Epi::LogitsWide ||
                          EPI == (int)Epi::LogitsCompactWide;
    constexpr int TR = WIDE ? TI / 2 : TI;
    extern __shared__ __attribute__((aligned(1024))) int8_t gemm_lds[];  // [stages][FRAGS][1024]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    // XCD-aware tile order: workgroup L runs on XCD L % 8, and XCD x takes the x-th contiguous
    // chunk of a grouped order (groups of `group` M-tiles, N outermost inside a group), so an
    // A row-tile stays in one XCD's L2 while the W tiles stream past it.
    int mt, nt;
    {
        const int gm = (g.m + BM - 1) / BM, gn = (g.n + BN - 1) / BN;
        const int T = gm * gn, L = blockIdx.x, x = L & 7, k = L >> 3;
        const int q = T >> 3, r = T & 7;
        const int p = x * q + (x < r ? x : r) + k;
        const int G = g.group, grp = p / (G * gn), in = p - grp * G * gn;
        const int gs = gm - grp * G < G ? gm - grp * G : G;
        nt = in / gs;
        mt = grp * G + in % gs;
    }
    const int m0 = mt * BM, n0 = nt * BN;
    const int K = g.k_pad;

    // The first k-step's MFMAs take the accumulators' start values as their C operand (no
    // zeroing moves): 0, or, for the NARROW epilogues with a bias, the bias of the lane's columns
    // (columns cw + 16 j + 4 (lane / 16) + e). fast32 bounds every partial sum plus the
    // bias by k 2^14 + max|b| < 2^31, so the i32 accumulation stays exact and the epilogue adds
    // no bias.
    constexpr bool FOLD_BIAS = NARROW && (EPI == (int)Epi::Act || EPI == (int)Epi::Residual ||
                                                  EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide);
    v4i acc[TI][TJ];
    v4i init[TJ];
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        init[j] = v4i{0, 0, 0, 0};
        if constexpr (FOLD_BIAS) {
            const int n4 = n0 + wn * 16 * TJ + 16 * j + 4 * (lane >> 4);
            if (g.params_padded) {
                init[j] = *(const v4i *)(g.bias + n4);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) init[j][e] = n4 + e < g.n ? g.bias[n4 + e] : 0;
            }
        }
    }
    auto mfma_ij = [&](const v4i &a, const v4i &b, const v4i &c) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, c, 0, 0, 0);
    };
    auto mfma_step = [&](const v4i *af, const v4i *bf) {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = mfma_ij(af[i], bf[j], acc[i][j]);
    };
    auto mfma_first = [&](const v4i *af, const v4i *bf) {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = mfma_ij(af[i], bf[j], init[j]);
    };

    if constexpr (BN == 256) {
        // 256 x 256 tiles (8 waves, one workgroup per CU) stream stages of 128 k (two panels),
        // eight lanes to a row (8 rows per instruction, 512 contiguous bytes of each panel).
        // Row r's 16-byte chunk c sits at r * 128 + 16 (c ^ ((r >> 1) & 7)) of the stage, so the
        // MFMA reads of 16 consecutive rows (one chunk) hit 16 distinct bank groups. Two stages
        // of 64 KiB: the next stage loads while this one is multiplied. A k_pad that is an odd
        // multiple of 64 ends with a half stage (chunks 0-3 only; the lanes of chunks 4-7 reload
        // a chunk of the last panel that nothing reads).
        constexpr int ROWS = BM + BN, LD = ROWS / 8 / WAVES, SB = ROWS * 128;
        const int nk2 = (K + 127) / 128;
        const bool half = (K & 127) != 0;
        // A wave's LD instructions all read one operand (waves 0-3 the A rows, 4-7 the W rows),
        // rows 8 i + lane / 8 of its block; the chunk swizzle alternates with i, so two lane bases
        // (even and odd i) and a uniform stride of 16 rows give every address.
        static_assert(BM / 8 % LD == 0, "a wave loads rows of one operand");
        const int ld_r = lane >> 3, ld_s = lane & 7;
        const int row0 = wave * LD * 8 + ld_r;  // the row of instruction 0 (row of i = row0 + 8 i)
        const int c_even = ld_s ^ ((row0 >> 1) & 7), c_odd = c_even ^ 4;
        const bool is_a = wave * LD * 8 < BM;  // uniform per wave
        const size_t pb = (size_t)(is_a ? g.a_rows : g.w_rows) * 64;  // bytes per panel
        const int8_t *base_row = is_a ? g.a + (size_t)(m0 + row0) * 64 : g.w + (size_t)(n0 + row0 - BM) * 64;
        const int8_t *p_even = base_row + (c_even >> 2) * pb + (c_even & 3) * 16;
        const int8_t *p_odd = base_row + 8 * 64 + (c_odd >> 2) * pb + (c_odd & 3) * 16;
        // a half stage: the lanes whose chunk is 4-7 step back one panel
        const long long h_even = c_even >= 4 ? -(long long)pb : 0, h_odd = c_odd >= 4 ? -(long long)pb : 0;
        auto issue = [&](int kt, int stage) {
            int8_t *base = gemm_lds + stage * SB + wave * LD * 1024;
            const bool last_half = half && kt == nk2 - 1;
            const long long ok = (long long)kt * 2 * (long long)pb;
            const long long oe = ok + (last_half ? h_even : 0), oo = ok + (last_half ? h_odd : 0);
#pragma unroll
            for (int i = 0; i < LD; i++) {
                const int8_t *p = (i & 1 ? p_odd + oo : p_even + oe) + (i >> 1) * 1024;
                __builtin_amdgcn_global_load_lds((const void *)p, (lds_void *)(base + i * 1024), 16, 0, 0);
            }
        };
        // lane l reads row l % 16 of each 16-row block (rows differ by multiples of 16, so the
        // swizzle is the lane's) at chunk 4 h + l / 16 of the stage's k half h
        const int rl = lane & 15, swz = (rl >> 1) & 7;
        auto frag_ptr = [&](int stage, int h) {
            return gemm_lds + stage * SB + rl * 128 + 16 * ((4 * h + (lane >> 4)) ^ swz);
        };
        auto read_a = [&](const int8_t *st, int i) { return *(const v4i *)(st + (wm * 16 * TI + 16 * i) * 128); };
        auto read_b = [&](const int8_t *st, int j) {
            return *(const v4i *)(st + (BM + wn * 16 * TJ + 16 * j) * 128);
        };
        issue(0, 0);
        auto body = [&](int kt, auto first_tag) {
            constexpr bool FIRST = decltype(first_tag)::value;
            const int stage = kt & 1;
            if (kt + 1 < nk2) {
                // stage kt + 1 goes to the buffer read in step kt - 1 (free after its barrier)
                issue(kt + 1, stage ^ 1);
                wait_vmcnt<LD>();
            } else {
                wait_vmcnt<0>();
            }
            asm volatile("s_barrier" ::: "memory");  // every wave's part of stage kt landed
            const int8_t *s0 = frag_ptr(stage, 0), *s1 = frag_ptr(stage, 1);
            v4i af[TI], bf[TJ];
#pragma unroll
            for (int i = 0; i < TI; i++) af[i] = read_a(s0, i);
#pragma unroll
            for (int j = 0; j < TJ; j++) bf[j] = read_b(s0, j);
            // The second half's fragments load while the first half's MFMAs run: its W fragments
            // first, then each A fragment into the registers of the one just used. A half stage
            // multiplies its second half by zero W fragments (no branch around the MFMAs).
            const bool zero_second = half && kt == nk2 - 1;
            v4i bn[TJ];
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const v4i b = read_b(s1, j);
                bn[j] = zero_second ? v4i{0, 0, 0, 0} : b;
            }
#pragma unroll
            for (int i = 0; i < TI; i++) {
#pragma unroll
                for (int j = 0; j < TJ; j++) acc[i][j] = mfma_ij(af[i], bf[j], FIRST ? init[j] : acc[i][j]);
                af[i] = read_a(s1, i);
            }
            mfma_step(af, bn);
            // every wave finished reading this stage before step kt + 1 reloads it
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        };
        body(0, Flag<true>{});
        for (int kt = 1; kt < nk2; kt++) body(kt, Flag<false>{});
    } else {
    // Split-K: workgroup row blockIdx.y takes K bytes [kb0, kb0 + kslice) of a product whose
    // partials go to out + blockIdx.y * m * ldo (Raw only).
    const int kb0 = (int)blockIdx.y * g.kslice;
    const int nk = (g.kslice ? min(g.kslice, K - kb0) : K) / GEMM_BK;

    // This wave loads fragments LOADS * wave .. +LOADS of each stage (0..15: A row blocks, then
    // the W row blocks, of 16 rows x 64 bytes). Each lane quad reads one row's 64 bytes of the
    // panel (lane l: row l / 4, 16-byte chunk (l % 4) ^ sw(row)); the 16 rows of a fragment are
    // adjacent in the panel, so a load reads 1 KiB of contiguous memory, 8 whole 128-byte lines.
    // The fragment lands in LDS in lane order, so chunk c of row r sits at 16-byte slot
    // 4 r + (c ^ sw(r)); sw(r) = ((r >> 1) ^ (r >> 3)) % 4 makes the MFMA operand reads (lane l:
    // row l % 16, chunk l / 16) of any 8 (and any 16) consecutive lanes hit distinct 16-byte
    // bank groups.
    auto sw = [](int r) { return ((r >> 1) ^ (r >> 3)) & 3; };
    const size_t pa = (size_t)g.a_rows * 64, pw = (size_t)g.w_rows * 64;  // bytes per panel
    // A load's address is a wave-uniform fragment base (scalar registers, recomputed by scalar
    // instructions each k-step) plus the lane's 32-bit offset inside the fragment, the same for
    // every load (one vector add per load). The 64 x 64 tiles, whose k-steps hold
    // 8 MFMAs per wave, keep a per-lane pointer per load instead: their loop is too short to hide
    // the scalar work (GPT-2-medium unfold GEMMs 2-4% slower with the shared form).
    const uint32_t lane_off = (uint32_t)((lane >> 2) * 64 + (((lane & 3) ^ sw(lane >> 2)) * 16));
    auto frag_base = [&](int i) -> const int8_t * {
        const int f = wave * LOADS + i;
        return f < BM / 16 ? g.a + (size_t)(kb0 / GEMM_BK) * pa + (size_t)(m0 + 16 * f) * 64
                           : g.w + (size_t)(kb0 / GEMM_BK) * pw + (size_t)(n0 + 16 * (f - BM / 16)) * 64;
    };
    constexpr bool LANE_PTRS = BM == 64;
    const int8_t *src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        src[i] = nullptr;
        if constexpr (LANE_PTRS) {
            const int f = wave * LOADS + i;
            const int r = lane >> 2, c = (lane & 3) ^ sw(r);
            const int row = (f < BM / 16 ? f : f - BM / 16) * 16 + r;
            src[i] = (f < BM / 16 ? g.a + (size_t)(kb0 / GEMM_BK) * pa + (size_t)(m0 + row) * 64
                                  : g.w + (size_t)(kb0 / GEMM_BK) * pw + (size_t)(n0 + row) * 64) + c * 16;
        }
    }
    const int rd_slot = 4 * (lane & 15) + ((lane >> 4) ^ sw(lane & 15));
    auto issue = [&](int kt, int stage) {
        int8_t *base = gemm_lds + stage * (FRAGS * 1024) + wave * LOADS * 1024;
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const size_t step = wave * LOADS + i < BM / 16 ? pa : pw;
            const int8_t *p = LANE_PTRS ? src[i] + (size_t)kt * step : frag_base(i) + (size_t)kt * step + lane_off;
            __builtin_amdgcn_global_load_lds((const void *)p, (lds_void *)(base + i * 1024), 16, 0, 0);
        }
    };

    // The operand fragments of k-step kt + 1 are read from LDS while the MFMAs of k-step kt
    // run on registers read the step before. Of the NST stages (3, or 6 for the 64 x 64 tiles)
    // one is being read and the others are in flight.
    auto read_frags = [&](int kt, v4i *af, v4i *bf) {
        const int8_t *st = gemm_lds + (kt % NST) * (FRAGS * 1024) + rd_slot * 16;
#pragma unroll
        for (int i = 0; i < TI; i++) af[i] = *(const v4i *)(st + (wm * TI + i) * 1024);
#pragma unroll
        for (int j = 0; j < TJ; j++) bf[j] = *(const v4i *)(st + (BM / 16 + wn * TJ + j) * 1024);
    };
    // wait until at most n stages' loads are in flight (n <= NST - 1)
    auto wait_stages = [&](int n) {
        if (NST > 5 && n >= 5) wait_vmcnt<(NST > 5 ? 5 * LOADS : 0)>();
        else if (NST > 4 && n == 4) wait_vmcnt<(NST > 4 ? 4 * LOADS : 0)>();
        else if (NST > 3 && n == 3) wait_vmcnt<(NST > 3 ? 3 * LOADS : 0)>();
        else if (n == 2) wait_vmcnt<2 * LOADS>();
        else if (n == 1) wait_vmcnt<LOADS>();
        else wait_vmcnt<0>();
    };
#pragma unroll
    for (int s = 0; s < NST; s++)
        if (s < nk) issue(s, s);
    // stage 0 landed (the later stages' loads may be outstanding); a bare s_barrier (a compiler
    // memory barrier, no fence: a fence would also wait for the stages in flight)
    if constexpr (NST == 3) {
        if (nk >= 3) wait_vmcnt<2 * LOADS>();
        else if (nk == 2) wait_vmcnt<LOADS>();
        else wait_vmcnt<0>();
    } else {
        wait_stages((nk < NST ? nk : NST) - 1);
    }
    asm volatile("s_barrier" ::: "memory");
    // One k-step: the MFMAs of step kt on (ca, cb) while step kt + 1's fragments are read into
    // (na, nb). Two register sets alternate (the loop is unrolled by two), so no fragment moves
    // between registers.
    auto step = [&](int kt, const v4i *ca, const v4i *cb, v4i *na, v4i *nb, auto first_tag) {
        const bool more = kt + 1 < nk;
        if (more) {
            // stage kt + 1 landed (stage kt + 2's loads may be outstanding); this wave's reads of
            // stage kt % 3 (issued the step before) completed, so after the barrier no wave
            // reads it and it takes k-step kt + 3
            if constexpr (NST == 3) {
                if (kt + 2 < nk) wait_vmcnt<LOADS>();
                else wait_vmcnt<0>();
            } else {  // the stages after kt + 1 that were issued: kt + 2 .. min(kt + NST - 1, nk - 1)
                const int ahead = nk - kt - 2;
                wait_stages(ahead < NST - 2 ? ahead : NST - 2);
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (kt + NST < nk) issue(kt + NST, kt % NST);
        }
        // unconditional (the last step re-reads its own stage), so the reads share the MFMAs'
        // basic block and no wait for them lands before the MFMAs; the empty asm keeps the
        // compiler from sinking them into the next step (where they would wait at its barrier)
        read_frags(more ? kt + 1 : kt, na, nb);
        if constexpr (decltype(first_tag)::value) mfma_first(ca, cb);
        else mfma_step(ca, cb);
        // The step's order: two MFMAs, then one fragment read of the next step, repeated, then
        // the remaining MFMAs (one MFMA per read for the 64 x 64 tiles, 8 MFMAs and 6 reads).
        // Opening with MFMAs keeps the wait that precedes the first of them from landing after a
        // read; spreading the reads keeps the LDS busy under the MFMAs (the compiler left them
        // after 24 of 32 MFMAs, or all before with a wait on the first).
        constexpr int NR = TI + TJ;
        if constexpr (2 * NR <= TI * TJ) {
#pragma unroll
            for (int z = 0; z < NR; z++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            }
            __builtin_amdgcn_sched_group_barrier(0x008, TI * TJ - 2 * NR, 0);
        } else if constexpr (NR <= TI * TJ) {
#pragma unroll
            for (int z = 0; z < NR; z++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, TI * TJ - NR, 0);
        } else {
            asm volatile("" ::: "memory");
        }
    };
    v4i fa0[TI], fb0[TJ], fa1[TI], fb1[TJ];
    read_frags(0, fa0, fb0);
    step(0, fa0, fb0, fa1, fb1, Flag<true>{});
    int kt = 1;
    for (; kt + 1 < nk; kt += 2) {
        step(kt, fa1, fb1, fa0, fb0, Flag<false>{});
        step(kt + 1, fa0, fb0, fa1, fb1, Flag<false>{});
    }
    if (kt < nk) step(kt, fa1, fb1, fa0, fb0, Flag<false>{});
    }

    // Epilogue. The W fragment is the MFMA's first operand, so of each 16 x 16 tile (i, j) of the wave
    // the lane holds C[16 i + lane % 16][16 j + 4 (lane / 16) + e]: four consecutive columns of a row.
    // rescale(a + bias, mult, shift) (int.rs:63-67). With the host's bound |a + bias| < 2^31
    // (fast32; the logits have no bias and |a| <= 2^30), |(a + bias) mult| < 2^62: one i64
    // multiply-add and an arithmetic shift are exact, and a shift of 63 or more gives 0 as
    // the rule does.
    const bool fast = EPI == (int)Epi::Logits || EPI == (int)Epi::LogitsCompact || g.fast32;
    const int s_eff = g.shift < 63 ? g.shift : 63;
    const int64_t half = s_eff ? (int64_t)1 << (s_eff - 1) : 0;
    auto rq = [&](int32_t a, int32_t bias, int32_t mult) -> int64_t {
        if (NARROW || fast) return ((int64_t)(a + bias) * mult + half) >> s_eff;
        return rescale_small((int64_t)a + bias, mult, g.shift);
    };
    // rescale of 256 hi + lo + add (add = 128 wsum + bias): |dot + bias| <= K 2^22 + 2^31 < 2^39
    auto rqw = [&](int32_t hi, int32_t lo, int64_t add, int32_t mult) -> int64_t {
        const int64_t v = (int64_t)hi * 256 + add + lo;
        if (NARROW || (g.shift >= 16 && g.shift <= 62)) return rescale_wide47(v, mult, (uint32_t)g.shift);
        return clamp128(rescale_full(v, mult, g.shift), -((int64_t)1 << 62), (int64_t)1 << 62);
    };
    // the same without a bias: 256 hi + 128 ws = 128 (2 hi + ws), an i32 for the NARROW forms (K < 2^15)
    auto rqw2 = [&](int32_t hi, int32_t lo, int32_t ws, int32_t mult) -> int64_t {
        if (NARROW) return rescale_wide47((int64_t)(2 * hi + ws) * 128 + lo, mult, (uint32_t)g.shift);
        return rqw(hi, lo, 128 * (int64_t)ws, mult);
    };
    const int cw = n0 + wn * 16 * TJ;                     // the wave's first column
    const int rw = (m0 + wm * 16 * TI) / (WIDE ? 2 : 1);  // and output row
    const int M = WIDE ? g.rows : g.m;
    {
        const int rl = lane & 15, cg = lane >> 4;
        constexpr bool RESIDUAL = EPI == (int)Epi::Residual || EPI == (int)Epi::ResidualWide;
        constexpr bool COMPACT = EPI == (int)Epi::LogitsCompact || EPI == (int)Epi::LogitsCompactWide;
        constexpr bool HAS_BIAS = EPI == (int)Epi::Act || RESIDUAL || EPI == (int)Epi::Gelu ||
                                  EPI == (int)Epi::GeluWide;
        constexpr bool vec = VEC;
        // The rescale parameters of column group j of the lane (columns cw + 16 j + 4 cg + e).
        auto params = [&](int j, int32_t *bj, int32_t *mj) {
            const int n4 = cw + 16 * j + 4 * cg;
            if (g.params_padded) {  // every column of a tile is below n_pad: 16-byte loads
                const v4i b4 = HAS_BIAS && !FOLD_BIAS ? *(const v4i *)(g.bias + n4) : v4i{0, 0, 0, 0};
                const v4i m4 = EPI != (int)Epi::Raw ? *(const v4i *)(g.mult + n4) : v4i{0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    bj[e] = b4[e];
                    mj[e] = m4[e];
                }
                return;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int n = n4 + e;
                const bool ok = n < g.n;
                bj[e] = (HAS_BIAS && !FOLD_BIAS && ok) ? g.bias[n] : 0;
                mj[e] = (EPI != (int)Epi::Raw && ok) ? g.mult[n] : 0;
            }
        };
        // The wide epilogues: 128 wsum + bias of column group j.
        auto addends = [&](int j, const int32_t *bj, int64_t *aj) {
            const int n4 = cw + 16 * j + 4 * cg;
#pragma unroll
            for (int e = 0; e < 4; e++) aj[e] = n4 + e < g.n ? 128 * (int64_t)g.wsum[n4 + e] + bj[e] : 0;
        };
        if constexpr (EPI == (int)Epi::ResidualWide) {  // ops.rs:178-206: the i32 (saturated) updates, in place
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                int32_t bj[4], mj[4];
                int64_t aj[4];
                params(j, bj, mj);
                addends(j, bj, aj);
#pragma unroll
                for (int i = 0; i < TR; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int64_t r = rqw(acc[2 * i][j][e], acc[2 * i + 1][j][e], aj[e], mj[e]);
                        acc[i][j][e] = NARROW ? (int32_t)r : (int32_t)clamp64(r, INT32_MIN, INT32_MAX);
                    }
                asm volatile("" ::: "memory");  // the next group's parameter loads stay below
            }
        }
        // Act, Gelu, GeluWide, Residual: the op's rule in place, one column group at a time.
        if (EPI == (int)Epi::Act || EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide || EPI == (int)Epi::Residual) {
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                int32_t bj[4], mj[4];
                params(j, bj, mj);
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int64_t r = rq(acc[i][j][e], bj[e], mj[e]);
                        int32_t v;
                        if (EPI == (int)Epi::Act) {  // ops.rs:123-130
                            v = NARROW ? med3_i32((int32_t)r, -127, 127) : (int32_t)clamp64(r, -127, 127);
                        } else if (EPI == (int)Epi::Residual) {
                            v = NARROW ? (int32_t)r : (int32_t)clamp64(r, INT32_MIN, INT32_MAX);
                        } else if (EPI == (int)Epi::Gelu) {  // ops.rs:146-154, gelu.rs:58-62: table[clamp(r) + off]
                            // clamped to the table's span (the same entry), as an index from gelu_lo
                            v = (NARROW ? med3_i32((int32_t)r, g.gelu_clo, g.gelu_chi)
                                        : (int32_t)clamp64(r, g.gelu_clo, g.gelu_chi)) +
                                g.gelu_shift;
                        } else {
                            // GeluWide: the index from gelu_lo, as Gelu
                            v = (NARROW ? med3_i32((int32_t)r, g.gelu_clo, g.gelu_chi)
                                        : (int32_t)clamp64(r, g.gelu_clo, g.gelu_chi)) +
                                g.gelu_shift;
                            if (BN != 256) v = g.gelu16[g.gelu_lo + v];  // the i16 table through the caches
                        }
                        acc[i][j][e] = v;
                    }
                asm volatile("" ::: "memory");  // the next group's parameter loads stay below
            }
        }
        if (RESIDUAL) {  // ops.rs:131-145
            // clamp(x + clamp(r, +-2^40), +-R) == clamp(x + sat32(r), +-R) for |x| <= R, and
            // == med3(sat32(x + sat32(r)), -R, R): a sum beyond i32 saturates to a value beyond R
            // on the same side, so the i32 saturating add and one med3 give it exactly.
            auto res = [](int32_t x, int32_t r) { return med3_i32(__builtin_elementwise_add_sat(x, r), -RES, RES); };
            if (!vec) {
#pragma unroll
                for (int i = 0; i < TR; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++) {
                        const int m = rw + 16 * i + rl, n4 = cw + 16 * j + 4 * cg;
                        if (m >= M) continue;
                        int32_t *x = (int32_t *)g.out + (size_t)m * g.ldo + n4;
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (n4 + e < g.n) x[e] = res(x[e], acc[i][j][e]);
                    }
                return;
            }
            // Staged in parts of 32 of the wave's rows through this wave's region (row stride RS):
            // the lane's four outputs of a row are one 16-byte LDS write; the read-modify-write of
            // x then covers whole 16-byte pieces of rows (CPR per row), all Q loads of a part in
            // flight together (parts of 64 rows of 64 columns held 32 vectors per lane and spilled).
            constexpr int HR = TR >= 2 ? 32 : 16, NH = 16 * TR / HR, RS = 64 * TJ + 16;
            constexpr int CPR = 4 * TJ, Q = HR * CPR / 64;
            static_assert(NH * HR == 16 * TR && HR * RS <= 18432 && Q * 64 == HR * CPR, "residual staging");
            __syncthreads();  // every wave finished reading the stages
            int8_t *wr = gemm_lds + wave * 18432;
#pragma unroll
            for (int h = 0; h < NH; h++) {
#pragma unroll
                for (int ii = 0; ii < HR / 16; ii++)
#pragma unroll
                    for (int j = 0; j < TJ; j++)
                        *(v4i *)(wr + (16 * ii + rl) * RS + (16 * j + 4 * cg) * 4) = acc[(HR / 16) * h + ii][j];
                v4i xv[Q], rv[Q];
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int pc = q * 64 + lane, rl2 = pc / CPR, cl = (pc % CPR) * 4;
                    const int m = rw + HR * h + rl2, n = cw + cl;
                    rv[q] = *(const v4i *)(wr + rl2 * RS + cl * 4);
                    xv[q] = (m < M && n + 4 <= g.n) ? *(const v4i *)((const int32_t *)g.out + (size_t)m * g.ldo + n)
                                                       : v4i{0, 0, 0, 0};
                }
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int pc = q * 64 + lane, rl2 = pc / CPR, cl = (pc % CPR) * 4;
                    const int m = rw + HR * h + rl2, n = cw + cl;
                    if (m >= M) continue;
                    int32_t *x = (int32_t *)g.out + (size_t)m * g.ldo + n;
                    if (n + 4 <= g.n) {
                        v4i o;
#pragma unroll
                        for (int t = 0; t < 4; t++) o[t] = res(xv[q][t], rv[q][t]);
                        *(v4i *)x = o;
                    } else {
#pragma unroll
                        for (int t = 0; t < 4; t++)
                            if (n + t < g.n) x[t] = res(x[t], rv[q][t]);
                    }
                }
            }
            return;
        }
        if (EPI == (int)Epi::Raw || EPI == (int)Epi::Logits || EPI == (int)Epi::LogitsWide) {  // i32 products; ops.rs:229-234 (i64)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                int32_t bj[4], mj[4];
                int64_t aj[4] = {0, 0, 0, 0};
                params(j, bj, mj);
                if constexpr (WIDE) addends(j, bj, aj);
#pragma unroll
                for (int i = 0; i < TR; i++) {
                    const int m = rw + 16 * i + rl, n4 = cw + 16 * j + 4 * cg;
                    if (m >= M || n4 >= g.n) continue;
                    if (EPI == (int)Epi::Raw) {
                        int32_t *o = (int32_t *)g.out + ((size_t)blockIdx.y * M + m) * g.ldo + n4;
                        if (vec && n4 + 4 <= g.n) *(v4i *)o = acc[i][j];
                        else
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                if (n4 + e < g.n) o[e] = acc[i][j][e];
                    } else {
                        int64_t *o = (int64_t *)g.out + (size_t)m * g.ldo + n4;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int64_t r = WIDE ? rqw(acc[WIDE ? 2 * i : 0][j][e], acc[WIDE ? 2 * i + 1 : 0][j][e], aj[e], mj[e])
                                               : rq(acc[i][j][e], 0, mj[e]);
                            if (n4 + e < g.n) o[e] = NARROW ? r : clamp64(r, -SCORE_LIMIT, SCORE_LIMIT);
                        }
                    }
                }
            }
            return;
        }
        if constexpr (COMPACT) {
            static_assert(TI == 8 && TJ == 4, "the compact logits keep 64-column tiles");
            // logit = clamp(rescale(acc, m[n], s), +-2^40) (ops.rs:229-234), stored as the
            // largest logit of this wave's 64 columns (per row) and per logit the distance
            // tilemax - logit capped at c: c = 65535 (NARROW: a saturating pack) or cap16; the
            // table index min(max - l, len - 1) follows exactly from them, because
            // max - l = (max - tilemax) + (tilemax - l) and c >= cap16 >= len - 1. Each row's 64
            // columns are 16 in each of the 4 lanes lane % 16 + 16 c.
            int32_t mult[4][4];
            int32_t ws[4][4];  // the wide form (no bias): wsum, 16 registers where the i64 addends take 32
#pragma unroll
            for (int j = 0; j < 4; j++) {
                int32_t bj[4];
                params(j, bj, mult[j]);
                if constexpr (WIDE) {
                    const int n4 = cw + 16 * j + 4 * cg;
#pragma unroll
                    for (int e = 0; e < 4; e++) ws[j][e] = n4 + e < g.n ? g.wsum[n4 + e] : 0;
                }
            }
            int8_t *wr = gemm_lds + wave * 18432;  // this wave's staging region: 128 rows x 144 B
            if (vec) __syncthreads();              // every wave finished reading the stages
            // NARROW: every logit lies in [-2^31 + 1, 2^31 - 1] (no clamp), so the row max is an
            // i32 max (INT32_MIN marks the columns past n) and tilemax - l < 2^32 a u32 difference.
            using L = typename std::conditional<NARROW, int32_t, int64_t>::type;
            using U = typename std::conditional<NARROW, uint32_t, int64_t>::type;
            constexpr L LMIN = NARROW ? (L)INT32_MIN : (L)INT64_MIN;
            // Only the wave tile holding column N (the last) has columns past it: the others take
            // a form without the per-logit column test (a wave-uniform choice).
            const bool full = cw + 64 <= g.n;
            auto rows = [&](auto FULL) {
#pragma unroll
            for (int i = 0; i < TR; i++) {
                L l[4][4], mx = LMIN;
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int64_t r = WIDE ? rqw2(acc[WIDE ? 2 * i : 0][j][e], acc[WIDE ? 2 * i + 1 : 0][j][e], ws[j][e], mult[j][e])
                                               : rq(acc[i][j][e], 0, mult[j][e]);
                        const bool ok = FULL || cw + 16 * j + 4 * cg + e < g.n;
                        l[j][e] = ok ? (NARROW ? (L)r : (L)clamp64(r, -SCORE_LIMIT, SCORE_LIMIT)) : LMIN;
                        mx = l[j][e] > mx ? l[j][e] : mx;
                    }
#pragma unroll
                for (int o = 16; o < 64; o <<= 1) {
                    const L u = __shfl_xor(mx, o, 64);
                    mx = u > mx ? u : mx;
                }
                const int m = rw + 16 * i + rl;
                if (m < M && cg == 0 && cw < g.n) g.tmax[(size_t)m * g.tmax_ld + cw / 64] = (int64_t)mx;
                const U cap = (U)g.cap16;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint32_t w2[2];
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        const U d0 = (U)mx - (U)l[j][2 * p], d1 = (U)mx - (U)l[j][2 * p + 1];
                        if constexpr (NARROW) {
                            // two u32 distances to a u16 pair, each min(d, 65535), in one
                            // instruction: every distance of cap16 or more stays at least cap16
                            const us2 pk = __builtin_amdgcn_cvt_pk_u16((uint32_t)d0, (uint32_t)d1);
                            __builtin_memcpy(&w2[p], &pk, 4);
                        } else {
                            const uint32_t u0 = (uint32_t)(d0 < cap ? d0 : cap);
                            const uint32_t u1 = (uint32_t)(d1 < cap ? d1 : cap);
                            w2[p] = (u0 & 0xFFFF) | (u1 << 16);
                        }
                    }
                    if (vec) {
                        *(uint2 *)(wr + (16 * i + rl) * 144 + (16 * j + 4 * cg) * 2) = make_uint2(w2[0], w2[1]);
                    } else if (m < M) {
                        uint16_t *o = (uint16_t *)g.out + (size_t)m * g.ldo + cw + 16 * j + 4 * cg;
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (cw + 16 * j + 4 * cg + e < g.n) o[e] = (uint16_t)(w2[e >> 1] >> (16 * (e & 1)));
                    }
                }
            }
            };
            if (full) rows(std::true_type{});
            else rows(std::false_type{});
            if (!vec) return;
#pragma unroll
            for (int q = 0; q < 2 * TR; q++) {
                const int rl2 = q * 8 + (lane >> 3), cl = (lane & 7) * 8;
                const v4i v = *(const v4i *)(wr + rl2 * 144 + cl * 2);
                const int m = rw + rl2, n = cw + cl;
                if (m >= M) continue;
                uint16_t *o = (uint16_t *)g.out + (size_t)m * g.ldo + n;
                if (n + 8 <= g.n) {
                    *(v4i *)o = v;
                } else {
#pragma unroll
                    for (int t = 0; t < 8; t++)
                        if (n + t < g.n) o[t] = (uint16_t)((uint32_t)v[t >> 1] >> (16 * (t & 1)));
                }
            }
            return;
        }
        // Act, Gelu, GeluWide: i8 outputs (GeluWide: the two planes of each i16 output), staged
        // per wave in LDS (the wave's rows x RS8 bytes) and stored as 16-byte row pieces. Gelu copies its
        // table's span (gelu_copy bytes from entry gelu_lo) into LDS first; the staging regions
        // follow it. The 64 x 64 tiles read the table through the caches instead
        // (a copy per workgroup would outweigh the 4,096 lookups of its tile).
        constexpr bool GELU_LDS = BM != 64;
        const int8_t *gspan = EPI == (int)Epi::GeluWide ? (const int8_t *)(g.gelu16 + g.gelu_lo) : g.gelu + g.gelu_lo;
        constexpr bool TABLE16 = EPI == (int)Epi::GeluWide && BN == 256;  // the i16 span, 2 bytes an entry
        int toff = 0;
        if (vec) {
            __syncthreads();  // every wave finished reading the stages
            if ((EPI == (int)Epi::Gelu && GELU_LDS) || TABLE16) {
                const int T = (TABLE16 ? 2 : 1) * g.gelu_copy;
                for (int c = threadIdx.x; c < T / 16; c += 64 * WAVES)
                    *(v4i *)(gemm_lds + 16 * c) = *(const v4i *)(gspan + 16 * c);
                __syncthreads();
                toff = (T + 1023) & ~1023;
            }
        }
        if constexpr (TABLE16) {
#pragma unroll
            for (int j = 0; j < TJ; j++) {
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] = ((const int16_t *)gemm_lds)[acc[i][j][e]];
                asm volatile("" ::: "memory");  // 4 TI lookups in flight at most
            }
        }
        constexpr int RS8 = 16 * TJ + 16, Q8 = TI * TJ / 4;
        static_assert(16 * TI * RS8 <= 10240 && Q8 * 64 == 16 * TI * TJ, "i8 staging");
        int8_t *wr = gemm_lds + toff + wave * 10240;
        // Act with the caches: when TJ divides 64, the lane's 16-column piece of every row it
        // stores, cw + 16 (lane % TJ), is the same for each of its Q8 rows, so whether it goes to
        // K or V, its head and the offset in the head are found once; the rows' slots and
        // positions load before the staging (their latency under the packing). Other TJ (the
        // 128 x 192 tiles) find them per row.
        constexpr bool KV_LANE = 64 % TJ == 0;
        const int n_l = cw + 16 * (lane % TJ);
        const bool to_kv = KV_LANE && EPI == (int)Epi::Act && vec && g.kv_rows && n_l >= g.kv_d;
        int8_t *kv_base = nullptr;
        int kv_slot[Q8], kv_pos[Q8];
        if (to_kv) {
            const int part = n_l >= 2 * g.kv_d, c = n_l - (part + 1) * g.kv_d;
            const int hh = c / g.kv_hd, cc = c - hh * g.kv_hd;
            kv_base = (part ? g.vc : g.kc) + (size_t)hh * g.kv_ctx * g.kv_hd + cc;
#pragma unroll
            for (int q = 0; q < Q8; q++) {
                const int m = rw + (q * 64 + lane) / TJ;
                const RowInfo ri = g.kv_rows[m < M ? m : M - 1];
                kv_slot[q] = ri.slot;
                kv_pos[q] = ri.pos;
            }
        }
        const size_t kv_slot_stride = (size_t)g.kv_h * g.kv_ctx * g.kv_hd;
        // GeluWide: the hi plane of every row, then the lo plane (this wave's region is rewritten
        // only after its own reads: LDS operations of a wave stay in order)
        constexpr int PLANES = EPI == (int)Epi::GeluWide ? 2 : 1;
#pragma unroll
        for (int pl = 0; pl < PLANES; pl++) {
            auto byte_of = [&](int32_t v) -> uint32_t {
                if (EPI == (int)Epi::GeluWide) return (uint32_t)(pl == 0 ? v >> 8 : (v & 255) - 128) & 255;
                return (uint32_t)v;  // the low byte is packed
            };
            // Unaligned output rows: bytes, or in the 64 x 64 tiles a group of Act in one unaligned store
            // (256 x 4099 x 6400 32.7 -> 27.9 us). (In 256 x 128 tiles it took 6 to 15% off most products
            // but made those of just over 256 tiles 5 to 13% slower: 2048 x 4099 x 3000 53 -> 60 us.)
            if (!vec) {
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++) {
                        const int n4 = cw + 16 * j + 4 * cg;
                        if (BM == 64 && EPI == (int)Epi::Act && !g.kv_rows && n4 + 4 <= g.n) {
                            const int m = rw + 16 * i + rl;
                            if (m >= M) continue;
                            uint32_t b = 0;
#pragma unroll
                            for (int e = 0; e < 4; e++) b |= (byte_of(acc[i][j][e]) & 255) << (8 * e);
                            __builtin_memcpy((int8_t *)g.out + (size_t)m * g.ldo + n4, &b, 4);
                            continue;
                        }
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int m = rw + 16 * i + rl, n = cw + 16 * j + 4 * cg + e;
                            if (m >= M || n >= g.n) continue;
                            const int32_t a = EPI == (int)Epi::Gelu ? (int32_t)gspan[acc[i][j][e]] : acc[i][j][e];
                            const int8_t v = (int8_t)byte_of(a);
                            if (EPI == (int)Epi::Act && g.kv_rows && n >= g.kv_d) {
                                const RowInfo ri = g.kv_rows[m];
                                const int part = n >= 2 * g.kv_d, c = n - (part + 1) * g.kv_d;
                                const int hh = c / g.kv_hd, cc = c - hh * g.kv_hd;
                                (part ? g.vc : g.kc)[(((size_t)ri.slot * g.kv_h + hh) * g.kv_ctx + ri.pos) * g.kv_hd + cc] = v;
                                continue;
                            }
                            if (EPI == (int)Epi::Act) {
                                ((int8_t *)g.out)[(size_t)m * g.ldo + n] = v;
                            } else {  // the operand of the next product, in panels
                                const size_t orow = EPI == (int)Epi::GeluWide ? plane_row(m, pl) : (size_t)m;
                                ((int8_t *)g.out)[panel_off(orow, n, g.out_rows)] = v;
                            }
                        }
                    }
                continue;
            }
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++) {
                    uint32_t b[4];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        b[e] = EPI == (int)Epi::Gelu ? (uint32_t)(uint8_t)(GELU_LDS ? gemm_lds[acc[i][j][e]] : gspan[acc[i][j][e]])
                                                     : byte_of(acc[i][j][e]);
                    // the low bytes of b[0..3] packed by three byte permutes: [b0 b1 0 0],
                    // [b2 b3 0 0], then their low halves side by side
                    const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
                    const uint32_t hi = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
                    *(uint32_t *)(wr + (16 * i + rl) * RS8 + 16 * j + 4 * cg) = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                    if (EPI == (int)Epi::Gelu && j == TJ - 1) asm volatile("" ::: "memory");  // 4 TJ lookups in flight at most
                }
#pragma unroll
            for (int q = 0; q < Q8; q++) {
                const int pc = q * 64 + lane, rl2 = pc / TJ, cl = (pc % TJ) * 16;
                const v4i v = *(const v4i *)(wr + rl2 * RS8 + cl);
                const int m = rw + rl2, n = cw + cl;
                if (m >= M) continue;
                if (to_kv) {
                    // K or V of the row straight into the cache (kv_d, kv_hd multiples of 16);
                    // the columns past N = 3 kv_d are padding and go nowhere
                    if (n + 16 > g.n) continue;
                    *(v4i *)(kv_base + (size_t)kv_slot[q] * kv_slot_stride + (size_t)kv_pos[q] * g.kv_hd) = v;
                    continue;
                }
                if (!KV_LANE && EPI == (int)Epi::Act && g.kv_rows && n >= g.kv_d) {
                    if (n + 16 > g.n) continue;
                    const RowInfo ri = g.kv_rows[m];
                    const int part = n >= 2 * g.kv_d, c = n - (part + 1) * g.kv_d;
                    const int hh = c / g.kv_hd, cc = c - hh * g.kv_hd;
                    *(v4i *)((part ? g.vc : g.kc) +
                             (((size_t)ri.slot * g.kv_h + hh) * g.kv_ctx + ri.pos) * g.kv_hd + cc) = v;
                    continue;
                }
                const size_t orow = EPI == (int)Epi::GeluWide ? plane_row(m, pl) : (size_t)m;
                // Gelu and GeluWide write the operand of the next product, in panels (16 columns
                // from a multiple of 16 lie in one panel)
                int8_t *o = (int8_t *)g.out + (EPI == (int)Epi::Act ? orow * g.ldo + n : panel_off(orow, n, g.out_rows));
                if (n + 16 <= g.n) {
                    *(v4i *)o = v;
                } else {
#pragma unroll
                    for (int t = 0; t < 16; t++)
                        if (n + t < g.n) o[t] = (int8_t)(v[t >> 2] >> (8 * (t & 3)));
                }
            }
        }
        return;
    }
}

// The largest span of an i16 GELU table that 256 x 256 tiles copy into LDS, in entries (beside 80 KiB of
// staging regions).
constexpr int GELU16_LDS = 40960;

template <int EPI, bool NARROW, int BN, bool VEC, int BM = GEMM_BM, bool DEEP = false>
static hipError_t launch_gemm_t(const GemmArgs &ga, hipStream_t stream) {
    constexpr int WAVES = gemm_waves(BN), FRAGS = BM / 16 + BN / 16;
    GemmArgs g = ga;
    if ((EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide) && g.gelu_copy <= 0) {  // the whole table
        g.gelu_lo = 0;
        g.gelu_clo = -g.gelu_off;
        g.gelu_chi = g.gelu_off - 1;
        g.gelu_shift = g.gelu_off;
        g.gelu_copy = 2 * g.gelu_off;
    }
    const int gm = (g.m + BM - 1) / BM, gn = (g.n + BN - 1) / BN;
    // the group of the tile order counts 256-row tiles: the same band of rows in BM-row tiles
    if (BM != GEMM_BM) g.group = (GEMM_BM / BM) * g.group < gm ? (GEMM_BM / BM) * g.group : gm;
    // the stages, and the epilogue's LDS: per-wave staging regions (18 KiB for the u16 logits
    // and the i16-plane epilogues, 10 KiB for i8 outputs), after the GELU table for Gelu
    constexpr size_t stages = BN == 256 ? (size_t)2 * (BM + BN) * 128 : (size_t)gemm_stages(BM, DEEP) * FRAGS * 1024;
    constexpr bool I8OUT = EPI == (int)Epi::Act || EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide;
    constexpr size_t regions = (size_t)WAVES * (I8OUT ? 10240 : 18432);
    // the largest request: the stages, or the GELU table (64 KiB of i8 entries, or the i16 span of
    // 256 x 256 tiles) and the staging regions after it
    constexpr bool TABLE16 = EPI == (int)Epi::GeluWide && BN == 256;
    constexpr bool GELU_LDS = (EPI == (int)Epi::Gelu && BM != 64) || TABLE16;  // the 64 x 64 tiles read it from memory
    constexpr size_t after_table = (TABLE16 ? (size_t)2 * GELU16_LDS : GELU_LDS ? 65536 : 0) + regions;
    constexpr size_t lds_max = stages > after_table ? stages : after_table;
    static_assert(lds_max <= 160 * 1024, "LDS of one workgroup");
    {
        const hipError_t e = allow_dynamic_lds((const void *)k_gemm<EPI, NARROW, BN, VEC, BM, DEEP>, lds_max);
        if (e != hipSuccess) return e;
    }
    size_t lds = stages > regions ? stages : regions;
    if (GELU_LDS && VEC) {
        const size_t t = ((size_t)(TABLE16 ? 2 : 1) * g.gelu_copy + 1023) & ~(size_t)1023;
        lds = stages > t + regions ? stages : t + regions;
    }
    launch_k((k_gemm<EPI, NARROW, BN, VEC, BM, DEEP>), dim3(gm * gn), dim3(64 * WAVES), lds, stream, g);
    return hipGetLastError();
}

// The products that take 64 x 64 tiles over the whole of K: all of at most 512 rows, and larger ones
// while their 64 x 64 tiles are few enough that the larger tiles would leave CUs idle (the narrow
// layers of a few thousand rows). Measured against the larger tiles, us a launch: 1024 x 2304 x
// 768 (576 tiles) 8.6 -> 6.9, 1536 x 2304 x 768 (864) 8.8 -> 7.5, 2048 x 2304 x 768 (1,152) 9.0
// -> 9.5; residual 3400 x 768 x 768 (648) 13.9 -> 9.3, 2048 x 768 x 3072 (384) 24.6 -> 17.8,
// 1536 x 1600 x 6400 (600) 42.3 -> 32.1, 2048 x 1600 x 6400 (800) 42.8 -> 51.7: the line lies
// lower for long K, where the larger tiles' fewer loads per output count for more. Rows that are not
// 16-byte aligned change the stores alone, so the same lines hold for them (256 x 4099 x 6400: 67 us in
// 256 x 128 tiles, 28 here; 512 x 5000 x 3000 47 -> 18;
// 1024 x 3001 x 1024 34 -> 10).
static bool gemm_small_tiles(int m, int n, int k_pad) {
    const long long tiles = ((m + 63) / 64) * (long long)((n + 63) / 64);
    return m <= 2 * GEMM_BM || tiles <= (k_pad <= 1024 ? 900 : 640);
}

// 256 x 128 tiles (two workgroups per CU, so one's epilogue overlaps the other's main loop),
// or 256 x 256 (below). Outputs whose rows are not 16-byte aligned take the store path without staging,
// in 64 x 64 or 256 x 128 tiles.
template <int EPI, bool NARROW>
static hipError_t launch_gemm_w(const GemmArgs &g, hipStream_t stream) {
    {
        constexpr bool RESIDUAL = EPI == (int)Epi::Residual || EPI == (int)Epi::ResidualWide;
        constexpr size_t ES = RESIDUAL || EPI == (int)Epi::Raw ? 4
                              : EPI == (int)Epi::LogitsCompact || EPI == (int)Epi::LogitsCompactWide ? 2
                              : EPI == (int)Epi::Logits || EPI == (int)Epi::LogitsWide ? 8 : 1;
        // (the GELU outputs are panels of 64-byte rows: aligned when the base is)
        constexpr bool PANEL_OUT = EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide;
        const bool vec = ((uintptr_t)g.out & 15) == 0 && (PANEL_OUT || ((size_t)g.ldo * ES) % 16 == 0);
        if constexpr (EPI == (int)Epi::Act || RESIDUAL || EPI == (int)Epi::Gelu || EPI == (int)Epi::GeluWide ||
                      EPI == (int)Epi::Raw) {
            if (gemm_small_tiles(g.m, g.n, g.k_pad)) {
                if constexpr (!PANEL_OUT)
                    if (!vec)
                        return g.k_pad >= 1024 ? launch_gemm_t<EPI, NARROW, 64, false, 64, true>(g, stream)
                                               : launch_gemm_t<EPI, NARROW, 64, false, 64>(g, stream);
                if (vec)
                    return g.k_pad >= 1024 ? launch_gemm_t<EPI, NARROW, 64, true, 64, true>(g, stream)
                                           : launch_gemm_t<EPI, NARROW, 64, true, 64>(g, stream);
            }
        }
        if (!vec) return launch_gemm_t<EPI, NARROW, 128, false>(g, stream);
        // 256 x 256 tiles (one workgroup per CU, full-line 128-k stages) for long K, where their
        // faster main loop outweighs the lost overlap of a second workgroup per CU and the
        // coarser rounds (measured: GPT-2 small mlp.c_proj, K 3,072, 12% faster; c_attn and the
        // LM head, K 768, 10% and 7% slower), and for the i8 GELU epilogue of a wide product
        // whose table span exceeds 32 KiB (each workgroup copies it into LDS, and beside the
        // staging regions of 256 x 128 tiles it would leave room for one workgroup per CU; the
        // full 64 KiB table measured 4% faster in 256 x 256 tiles) or whose K is 1,536 or more.
        // A span of at most 32 KiB fits in the 256 x 128 tiles' stages: two workgroups per CU
        // (measured, c_fc with a 23 KiB span: GPT-2 small, K 768, 66 -> 58 us; GPT-2 medium,
        // K 1,024, 10.4 -> 9.3 ms per step; GPT-2 XL, K 1,600, 190 -> 214 ms per step, so it
        // keeps 256 x 256).
        const int gcopy = g.gelu_copy > 0 ? g.gelu_copy : 2 * g.gelu_off;
        const bool wide = g.n > 512 && (g.k_pad >= 2048 ||
                                        (EPI == (int)Epi::Gelu && g.n > 1024 && (gcopy > 32768 || g.k_pad >= 1536)));
        // The i16 GELU table, 2 bytes an entry, is gathered from LDS only in 256 x 256 tiles (its span takes
        // most of what the staging leaves); through the caches the gathers took longer than the product
        // (3,370 x 3,072 x 768: 37 us, 25 from LDS).
        if constexpr (EPI == (int)Epi::GeluWide) {
            if (gcopy <= GELU16_LDS) return launch_gemm_t<EPI, NARROW, 256, true>(g, stream);
            return launch_gemm_t<EPI, NARROW, 128, true>(g, stream);
        }
        if constexpr (EPI == (int)Epi::Act || RESIDUAL) {
            // 128 x 192 tiles for a product that is one partial round of resident workgroups
            // (at most 512 of 256 x 128, or 256 of 256 x 256) and one round of 128 x 192: the
            // round then holds three quarters of the work per CU, spread over every CU
            // (measured, GPT-2 small fold: c_proj 32.8 -> 29.6 us, mlp.c_proj 60.9 -> 52.8 us).
            // Over several rounds the smaller tile's lower efficiency per output (its loads per
            // output are 11% more) outweighs the fuller last round (c_attn, 1,152 tiles of
            // 256 x 128: 47.0 us, 1,536 of 128 x 192: 47.8 us).
            const long long gm2 = (g.m + 255) / 256, gm1 = (g.m + 127) / 128, gn3 = (g.n + 191) / 192;
            const long long base_tiles = wide ? gm2 * ((g.n + 255) / 256) : gm2 * ((g.n + 127) / 128);
            const bool one_round = base_tiles <= (wide ? 256 : 512) && gm1 * gn3 <= 512;
            if (one_round && gn3 * 192 <= g.w_rows) return launch_gemm_t<EPI, NARROW, 192, true, 128>(g, stream);
        }
        if (wide) return launch_gemm_t<EPI, NARROW, 256, true>(g, stream);
        return launch_gemm_t<EPI, NARROW, 128, true>(g, stream);
    }
}

template <int EPI>
static hipError_t launch_gemm_e(const GemmArgs &g, hipStream_t stream) {
    constexpr bool WIDE = EPI == (int)Epi::ResidualWide || EPI == (int)Epi::LogitsWide ||
                          EPI == (int)Epi::LogitsCompactWide;
    const bool fast = EPI == (int)Epi::Logits || EPI == (int)Epi::LogitsCompact || g.fast32;
    if (fast && (WIDE || g.shift >= 31)) return launch_gemm_w<EPI, true>(g, stream);
    return launch_gemm_w<EPI, false>(g, stream);
}

// ---- Split-K of a Raw product, on the caller's wish (matmul_i8_split, ops.rs:163-184) -------------
// Slices of K in 64 x 64 tiles write exact i32 partials (|each| <= 2^30, and i32 sums of them are
// exact in any order), and k_split_sum_raw adds a tile's slices. (The layers' products of few rows
// split K inside a workgroup instead: gemm_rows.hip.)

size_t gemm_split_elems(int m, int n, int splits) {
    return (size_t)splits * (size_t)m * (size_t)((n + 3) & ~3);
}

int gemm_split_plan(int k_pad, int wanted) {
    const int nks = k_pad / GEMM_BK;
    return wanted > nks ? nks : (wanted > 1 ? wanted : 1);
}

// Sums the `splits` partials of one output row x 4 columns. A whole group of 4 columns whose
// destination is 16-byte aligned is stored with one access.
__global__ __launch_bounds__(256) void k_split_sum_raw(GemmArgs g, int splits, int ldp) {
    const int groups = ldp / 4;
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const int m = (int)(idx / groups), n4 = (int)(idx % groups) * 4;
    if (m >= g.m || n4 >= g.n) return;
    // four slices' loads in flight at a time (i32 sums of the partials are exact in any order)
    const int32_t *src = g.partials + (size_t)m * ldp + n4;
    const size_t slice = (size_t)g.m * ldp;
    v4i acc = {0, 0, 0, 0};
    int sl = 0;
    for (; sl + 4 <= splits; sl += 4) {
        const v4i p0 = *(const v4i *)(src + sl * slice), p1 = *(const v4i *)(src + (sl + 1) * slice);
        const v4i p2 = *(const v4i *)(src + (sl + 2) * slice), p3 = *(const v4i *)(src + (sl + 3) * slice);
        acc += (p0 + p1) + (p2 + p3);
    }
    for (; sl < splits; sl++) acc += *(const v4i *)(src + sl * slice);
    const int cnt = g.n - n4 < 4 ? g.n - n4 : 4;
    int32_t *o = (int32_t *)g.out + (size_t)m * g.ldo + n4;
    if (cnt == 4 && ((uintptr_t)o & 15) == 0) *(v4i *)o = acc;
    else
        for (int e = 0; e < cnt; e++) o[e] = acc[e];
}

static hipError_t launch_gemm_split(const GemmArgs &ga, int splits, hipStream_t stream) {
    if (ga.group < 1 || ga.group > (ga.m + GEMM_BM - 1) / GEMM_BM || splits < 2 || splits > 16)
        return hipErrorInvalidValue;
    GemmArgs p = ga;  // the partial products: Raw into the scratch, [splits][m][ldp]
    const int ldp = (ga.n + 3) & ~3;
    const int nks = ga.k_pad / GEMM_BK;
    p.kslice = ((nks + splits - 1) / splits) * GEMM_BK;
    splits = (ga.k_pad + p.kslice - 1) / p.kslice;  // every slice holds at least one k-step
    p.out = ga.partials;
    p.ldo = ldp;
    const int gm = (ga.m + 63) / 64, gn = (ga.n + 63) / 64;
    p.group = 4 * ga.group < gm ? 4 * ga.group : gm;
    constexpr size_t lds = (size_t)gemm_stages(64, false) * 8 * 1024;
    hipError_t e = allow_dynamic_lds((const void *)k_gemm<(int)Epi::Raw, false, 64, true, 64>, lds);
    if (e != hipSuccess) return e;
    launch_k((k_gemm<(int)Epi::Raw, false, 64, true, 64>), dim3(gm * gn, splits), dim3(64 * gemm_waves(64)), lds,
             stream, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const long long threads = (long long)ga.m * (ldp / 4);
    launch_k(k_split_sum_raw, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, ga, splits, ldp);
    return hipGetLastError();
}

// The i16-activation product from its plane rows (matvec_i8_i16, ADR 0004 addendum B):
// out[i][r] = 256 p[2i][r] + p[2i + 1][r] + 128 wsum[r], exact in i64.
__global__ void k_wide_combine(const int32_t *p, const int32_t *wsum, int m, int n, int64_t *out) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)m * n) return;
    const int i = (int)(idx / n), r = (int)(idx % n);
    out[idx] = 256 * (int64_t)p[(size_t)(2 * i) * n + r] + p[(size_t)(2 * i + 1) * n + r] + 128 * (int64_t)wsum[r];
}

hipError_t launch_wide_combine(const int32_t *planes, const int32_t *wsum, int m, int n, int64_t *out,
                               hipStream_t stream) {
    const long long t = (long long)m * n;
    if (t == 0) return hipSuccess;
    launch_k(k_wide_combine, dim3((unsigned)((t + 255) / 256)), dim3(256), 0, stream, planes, wsum, m, n, out);
    return hipGetLastError();
}

hipError_t launch_gemm(Epi epi, const GemmArgs &ga, hipStream_t stream) {
    GemmArgs g = ga;
    if (g.m <= 0 || g.n <= 0) return hipSuccess;
    // at least one k-step: the loop's first step runs unconditionally
    if (g.k_pad < GEMM_BK || g.k_pad % GEMM_BK != 0) return hipErrorInvalidValue;
    // the tile order's M-tile group (the kernel divides by it): set and checked before any launch
    const int gm = (g.m + GEMM_BM - 1) / GEMM_BM;
    if (g.group == 0) g.group = gemm_group(g.m);
    if (g.group < 1 || g.group > gm) return hipErrorInvalidValue;
    // the panel row counts cover every row a tile reads (whole 256-row tiles of A and of W)
    const int n_pad = (g.n + GEMM_NPAD - 1) / GEMM_NPAD * GEMM_NPAD;
    if (g.a_rows == 0) g.a_rows = gm * GEMM_BM;
    if (g.w_rows == 0) g.w_rows = n_pad;
    if (g.a_rows < gm * GEMM_BM || g.w_rows < n_pad) return hipErrorInvalidValue;
    if ((epi == Epi::Gelu && g.out_rows < g.m) || (epi == Epi::GeluWide && g.out_rows < plane_rows(g.m)))
        return hipErrorInvalidValue;
    // the wide epilogues: whole blocks of planes, their row sums, and a shift inside the bound of fast32
    if (epi == Epi::ResidualWide || epi == Epi::LogitsWide || epi == Epi::LogitsCompactWide) {
        if (!g.wsum || g.rows <= 0 || g.m != plane_rows(g.rows)) return hipErrorInvalidValue;
        if (g.fast32 && (g.shift < 16 || g.shift > 62)) return hipErrorInvalidValue;
    }
    g.kslice = 0;
    if (g.splits > 1) {
        const int sp = gemm_split_plan(g.k_pad, g.splits);
        if (sp > 1) {
            if (epi != Epi::Raw || !g.partials || gemm_split_elems(g.m, g.n, sp) > g.partials_cap)
                return hipErrorInvalidValue;
            return launch_gemm_split(g, sp, stream);
        }
    }
    if (gemm_rows_fits(epi, g)) return launch_gemm_rows(epi, g, stream);
    switch (epi) {
        case Epi::Raw: return launch_gemm_w<0, false>(g, stream);
        case Epi::Act: return launch_gemm_e<1>(g, stream);
        case Epi::Residual: return launch_gemm_e<2>(g, stream);
        case Epi::Gelu: return launch_gemm_e<3>(g, stream);
        case Epi::Logits: return launch_gemm_e<4>(g, stream);
        case Epi::LogitsCompact:
            if (head_rows_fits(g)) return launch_head_rows(g, stream);
            return launch_gemm_e<5>(g, stream);
        case Epi::GeluWide: return launch_gemm_e<6>(g, stream);
        case Epi::ResidualWide:
        case Epi::LogitsWide:
        case Epi::LogitsCompactWide:
            if (epi == Epi::ResidualWide) return launch_gemm_e<7>(g, stream);
            if (epi == Epi::LogitsWide) return launch_gemm_e<8>(g, stream);
            return launch_gemm_e<9>(g, stream);
    }
    return hipErrorInvalidValue;
}

// =============================================================================================
// Stream read (the probe of crates/hardshell-cuda/src/ops.rs:328-335, read_gpu_ns): each thread
// keeps 8 16-byte loads in flight per round and folds them with xor.
// =============================================================================================

__global__ __launch_bounds__(256) void k_read_bw(const v4i *p, size_t n16, int *sink) {
    const size_t stride = (size_t)gridDim.x * 256;
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    v4i acc = {0, 0, 0, 0};
    for (; i + 7 * stride < n16; i += 8 * stride) {
        v4i v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = __builtin_nontemporal_load(p + i + u * stride);
#pragma unroll
        for (int u = 0; u < 8; u++) acc ^= v[u];
    }
    for (; i < n16; i += stride) acc ^= p[i];
    sink[(size_t)blockIdx.x * 256 + threadIdx.x] = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
}

hipError_t launch_read_bw(const void *buf, size_t n16, int *sink, int grid, hipStream_t stream) {
    launch_k(k_read_bw, dim3(grid), dim3(256), 0, stream, (const v4i *)buf, n16, sink);
    return hipGetLastError();
}

// =============================================================================================
// Issue-rate probe: `iters` rounds of independent instructions of one kind per wave (8 chains of
// a VALU form, or 8 accumulators of 16 x 16 x 64 / 4 of 32 x 32 x 32 MFMAs), workgroups of 4
// waves (one per SIMD of a CU), 256 x `waves_per_simd` workgroups; the time over the instruction count gives the
// clocks per instruction per SIMD (hs_probe_issue). The results go to `sink` only when a lane
// sees an impossible value, so nothing is folded away.
// =============================================================================================

typedef int v16i __attribute__((ext_vector_type(16)));

// OP 5 v_ashrrev_i64 and 6 v_mul_hi_i32 (8 chains each); OP 7 and 8: workgroups of 8 waves
// (two per SIMD), waves 0-3 the 16 x 16 x 64 MFMA chains and waves 4-7 three times as many
// rounds of v_add_u32 (7) or v_mad_i64_i32 (8), so the time shows whether a SIMD issues one
// wave's VALU work while another wave's MFMAs run.
template <int OP>
__global__ __launch_bounds__(512) void k_issue_probe(int *sink, int iters, int seed) {
    const int t = threadIdx.x;
    constexpr bool MIX = OP == 7 || OP == 8;
    const bool mfma_wave = MIX && __builtin_amdgcn_readfirstlane(t >> 6) < 4;
    int32_t a[8];
    int64_t b[8];
    double c[8];
    v4i x[8];
    v16i y[4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        a[i] = seed + i + t;
        b[i] = (int64_t)a[i] * 3;
        c[i] = a[i];
        x[i] = v4i{a[i], i, t, seed};
    }
#pragma unroll
    for (int i = 0; i < 4; i++) y[i] = v16i{};
    const v4i fa = {seed, t, 7, 9}, fb = {t, seed, 3, 5};
    const int m = seed | 1;
    const double md = 1.000001;
    if (MIX && mfma_wave) {
        for (int it = 0; it < iters; it++) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(x[i]) : "v"(fa), "v"(fb));
        }
    } else if (MIX) {
        for (int it = 0; it < 3 * iters; it++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (OP == 7) asm volatile("v_add_u32 %0, %0, %1" : "+v"(a[i]) : "s"(m));
                if (OP == 8) asm volatile("v_mad_i64_i32 %0, vcc, %1, %2, %0" : "+v"(b[i]) : "v"(a[i]), "s"(m) : "vcc");
            }
        }
    } else {
        for (int it = 0; it < iters; it++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (OP == 0) asm volatile("v_add_u32 %0, %0, %1" : "+v"(a[i]) : "s"(m));
                if (OP == 1) asm volatile("v_mad_i64_i32 %0, vcc, %1, %2, %0" : "+v"(b[i]) : "v"(a[i]), "s"(m) : "vcc");
                if (OP == 2) asm volatile("v_fma_f64 %0, %0, %1, %1" : "+v"(c[i]) : "s"(md));
                if (OP == 3) asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(x[i]) : "v"(fa), "v"(fb));
                if (OP == 4 && i < 4) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+v"(y[i]) : "v"(fa), "v"(fb));
                if (OP == 5) asm volatile("v_ashrrev_i64 %0, %1, %0" : "+v"(b[i]) : "s"(m & 31));
                if (OP == 6) asm volatile("v_mul_hi_i32 %0, %0, %1" : "+v"(a[i]) : "s"(m));
            }
        }
    }
    int64_t acc = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) acc += a[i] + b[i] + (int64_t)c[i] + x[i][0] + x[i][3];
#pragma unroll
    for (int i = 0; i < 4; i++) acc += y[i][0] + y[i][15];
    if (acc == 0x7fffffffffffll) sink[t] = (int)acc;
}

hipError_t launch_issue_probe(int op, int waves_per_simd, int iters, int *sink, hipStream_t stream) {
    if (op == 7 || op == 8) {  // 8 waves per workgroup: waves_per_simd counts both kinds
        if (waves_per_simd % 2) return hipErrorInvalidValue;
        const dim3 grid(256 * waves_per_simd / 2), block(512);
        if (op == 7) launch_k(k_issue_probe<7>, grid, block, 0, stream, sink, iters, 7);
        else launch_k(k_issue_probe<8>, grid, block, 0, stream, sink, iters, 7);
        return hipGetLastError();
    }
    const dim3 grid(256 * waves_per_simd), block(256);
    switch (op) {
        case 0: launch_k(k_issue_probe<0>, grid, block, 0, stream, sink, iters, 7); break;
        case 1: launch_k(k_issue_probe<1>, grid, block, 0, stream, sink, iters, 7); break;
        case 2: launch_k(k_issue_probe<2>, grid, block, 0, stream, sink, iters, 7); break;
        case 3: launch_k(k_issue_probe<3>, grid, block, 0, stream, sink, iters, 7); break;
        case 4: launch_k(k_issue_probe<4>, grid, block, 0, stream, sink, iters, 7); break;
        case 5: launch_k(k_issue_probe<5>, grid, block, 0, stream, sink, iters, 7); break;
        case 6: launch_k(k_issue_probe<6>, grid, block, 0, stream, sink, iters, 7); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// =============================================================================================
// Embedding (reference.rs:208-221): x = clamp(rescale(wte[tok]) + rescale(wpe[pos]), -R, R).
// =============================================================================================

// wte is the LM head's operand: panels of wte_rows rows (panel_off).
__global__ void k_embed(const RowInfo *rows, const int8_t *wte, int wte_rows, const int8_t *wpe,
                        const int32_t *embed_m, int embed_s, const int32_t *pos_m, int pos_s,
                        int d, int32_t *x) {
    const int r = blockIdx.x, j = blockIdx.y * blockDim.x + threadIdx.x;
    if (j >= d) return;
    const RowInfo ri = rows[r];
    const int64_t v = rescale_small(wte[panel_off(ri.token, j, wte_rows)], embed_m[ri.token], embed_s) +
                      rescale_small(wpe[(size_t)ri.pos * d + j], pos_m[ri.pos], pos_s);
    x[(size_t)r * d + j] = (int32_t)clamp64(v, -RES, RES);
}

// d % 4 == 0: one wave per row, each lane four consecutive columns at a time (one 4-byte load
// of each table: the four lie in one panel of wte; one 16-byte store). |w m| < 2^38, so the
// rescale is one i64 multiply-add and shift, exactly shift_round64's result.
__global__ __launch_bounds__(256) void k_embed4(const RowInfo *rows, int n_rows, const int8_t *wte, int wte_rows,
                                                const int8_t *wpe, const int32_t *embed_m, int embed_s,
                                                const int32_t *pos_m, int pos_s, int d, int32_t *x) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= n_rows) return;
    const RowInfo ri = rows[r];
    const int64_t em = embed_m[ri.token], pm = pos_m[ri.pos];
    auto rs = [](int64_t p, int s) -> int64_t {  // shift_round64 for |p| < 2^62
        if (s == 0) return p;
        if (s >= 64) return 0;
        return (p + ((int64_t)1 << (s - 1))) >> s;
    };
    for (int j = 4 * lane; j < d; j += 256) {
        const uint32_t tw = *(const uint32_t *)(wte + panel_off(ri.token, j, wte_rows));
        const uint32_t pw = *(const uint32_t *)(wpe + (size_t)ri.pos * d + j);
        v4i o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t v = rs((int64_t)(int8_t)(tw >> (8 * e)) * em, embed_s) +
                              rs((int64_t)(int8_t)(pw >> (8 * e)) * pm, pos_s);
            o[e] = (int32_t)clamp64(v, -RES, RES);
        }
        *(v4i *)(x + (size_t)r * d + j) = o;
    }
}

hipError_t launch_embed(const RowInfo *rows, int n_rows, const int8_t *wte, int wte_rows,
                        const int8_t *wpe, const int32_t *embed_m, int embed_s,
                        const int32_t *pos_m, int pos_s, int d, int32_t *x, hipStream_t stream) {
    if (n_rows <= 0) return hipSuccess;
    if (d % 4 == 0) {
        launch_k(k_embed4, dim3((n_rows + 3) / 4), dim3(256), 0, stream, rows, n_rows, wte, wte_rows, wpe,
                 embed_m, embed_s, pos_m, pos_s, d, x);
        return hipGetLastError();
    }
    dim3 grid(n_rows, (d + 255) / 256);
    launch_k(k_embed, grid, dim3(256), 0, stream, rows, wte, wte_rows, wpe, embed_m,
                       embed_s, pos_m, pos_s, d, x);
    return hipGetLastError();
}

// =============================================================================================
// Integer LayerNorm (crates/hardshell/src/layernorm.rs:201-256), one workgroup per row:
// mean = floor(sum / n); var = floor(sum (x - mean)^2 / n) in u128; inv = 2^K / isqrt(var *
// 2^2J + eps); y = rescale_wide((x - mean) * inv * gamma, m, s) + beta (or the one-rounding form
// with beta_frac); out = clamp(y, -127, 127), or clamp(y, -32767, 32767) as two i8 planes for
// the 16-bit final LayerNorm of a version-2 model (layernorm.rs:197, ops.rs:246-277).
// =============================================================================================

__device__ __forceinline__ u128 wave_sum128(u128 v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t lo = __shfl_xor((uint64_t)v, o, 64);
        const uint64_t hi = __shfl_xor((uint64_t)(v >> 64), o, 64);
        v += ((u128)hi << 64) | lo;
    }
    return v;
}

// One wave per row, four rows per workgroup, no LDS and no barriers: the row sum, then the sum
// of squares of c = x - mean (|c| < 2^32, so a square fits u64 and each lane carries into a
// high word), and the per-row inv of ln_inv (no 128-bit division). The product c * inv * gamma
// * m is formed as (c * inv) * (gamma * m): the reference's bounds (|t| < 2^95, |m| < 2^31,
// layernorm.rs:31-39) keep it below 2^126, so its wrapping product never wraps and the two
// forms are the same integer. When max|c| * inv < 2^63 (exact test), c * inv is an i64.
__global__ __launch_bounds__(256) void k_layernorm(LnArgs a, int n_rows) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n_rows) return;
    const int d = a.d;
    const int src = a.src ? a.src[row] : row;
    const int32_t *x = a.x + (size_t)src * d;
    int64_t sum = 0;
    for (int j = lane; j < d; j += 64) sum += x[j];
    sum = wave_sum64(sum);
    const double inv_d = 1.0 / (double)d;  // |sum| <= d RES < 2^52, sq < d 2^62: the estimate forms
    const int64_t mean = floor_div_est(sum, d, inv_d);
    uint64_t lo = 0, hi = 0, cmax = 0;
    for (int j = lane; j < d; j += 64) {
        const int64_t c = (int64_t)x[j] - mean;
        const uint64_t u = c < 0 ? (uint64_t)(-c) : (uint64_t)c;
        const uint64_t v = u * u;
        lo += v;
        hi += lo < v;
        cmax = u > cmax ? u : cmax;
    }
    const u128 sq = wave_sum128(((u128)hi << 64) | lo);
    cmax = (uint64_t)wave_max64((int64_t)cmax);
    const uint64_t inv = ln_inv_est(sq, (uint32_t)d, (uint32_t)a.k, (uint32_t)a.j, a.eps, inv_d);
    const bool small = (u128)cmax * inv < ((u128)1 << 63);
    const bool wide = a.bits == 16;
    // the operand rows of this row (two planes when wide), in panels (panel_off)
    auto at = [&](int pl, int j) { return a.out + panel_off(wide ? plane_row(row, pl) : (size_t)row, j, a.out_rows); };
    // clamp_act_i8, or clamp_act_i16 stored as the planes hi = v >> 8, lo = (v & 255) - 128
    auto put = [&](int j, int64_t y) {
        if (!wide) {
            *at(0, j) = (int8_t)clamp64(y, -127, 127);
        } else {
            const int32_t v = (int32_t)clamp64(y, -32767, 32767);
            *at(0, j) = (int8_t)(v >> 8);
            *at(1, j) = (int8_t)((v & 255) - 128);
        }
    };
    if (small && a.beta_frac == 0 && a.s >= 64 && a.s <= 126) {
        // the rounding shift from the high word of (c inv) (gamma m) alone (shift_round_hi)
        for (int j = lane; j < d; j += 64) {
            const int64_t c = (int64_t)x[j] - mean;
            put(j, shift_round_hi(c * (int64_t)inv, a.gm[j], (uint32_t)a.s) + a.beta[j]);
        }
        return;
    }
    for (int j = lane; j < d; j += 64) {
        const int64_t c = (int64_t)x[j] - mean;
        const i128 cinv = small ? (i128)(c * (int64_t)inv) : (i128)c * (i128)(u128)inv;
        const i128 p = cinv * (i128)a.gm[j];
        i128 y;
        if (a.beta_frac == 0) {
            y = shift_round128(p, a.s, 126) + (i128)a.beta[j];
        } else {
            const i128 cb = (i128)a.beta[j] << (a.s - a.beta_frac);
            y = shift_round128(p + cb, a.s, 126);
        }
        put(j, clamp128(y, -32767, 32767));
    }
}

// One wave per row, the row in registers as NG groups of 4 consecutive columns per lane
// (d % 4 == 0, d <= 256 NG): 16-byte loads of x and beta, 32-byte loads of gamma m, one 4-byte
// store per 4 outputs. One pass gives sum x, sum x^2 (u64 squares, |x| <= 2^30, with a carry
// word), min and max; then sum (x - mean)^2 = sum x^2 - 2 mean sum x + d mean^2 (the same
// integer) and max|x - mean| = max(max - mean, mean - min).
template <int NG>
__global__ __launch_bounds__(256) void k_layernorm_rows(LnArgs a, int n_rows) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);  // no LDS, no barrier
    if (row >= n_rows) return;
    const int d = a.d;
    const int32_t *x = a.x + (size_t)(a.src ? a.src[row] : row) * d;
    v4i xv[NG];
    int64_t sum = 0;
    uint64_t lo = 0, hi = 0;
    int32_t mx = INT32_MIN, mn = INT32_MAX;
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = 4 * (lane + 64 * t);
        xv[t] = j < d ? *(const v4i *)(x + j) : v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = 4 * (lane + 64 * t);
        if (j >= d) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int32_t v = xv[t][e];
            sum += v;
            const uint32_t u = (uint32_t)(v < 0 ? -v : v);
            const uint64_t p = (uint64_t)u * u;
            lo += p;
            hi += lo < p;
            mx = v > mx ? v : mx;
            mn = v < mn ? v : mn;
        }
    }
    sum = wave_sum64(sum);
    const u128 Q = wave_sum128(((u128)hi << 64) | lo);
    mx = (int32_t)wave_max64(mx);
    mn = (int32_t)-wave_max64(-(int64_t)mn);
    const double inv_d = 1.0 / (double)d;  // |sum| <= d RES < 2^52, sq < d 2^62: the estimate forms
    const int64_t mean = floor_div_est(sum, d, inv_d);
    const u128 sq = (u128)((i128)Q - 2 * (i128)mean * sum + (i128)d * mean * mean);
    const uint64_t inv = ln_inv_est(sq, (uint32_t)d, (uint32_t)a.k, (uint32_t)a.j, a.eps, inv_d);
    const int64_t c1 = (int64_t)mx - mean, c2 = mean - (int64_t)mn;
    const uint64_t cmax = (uint64_t)(c1 > c2 ? c1 : c2);
    const bool small = (u128)cmax * inv < ((u128)1 << 63);
    const bool fast = small && a.beta_frac == 0 && a.s >= 64 && a.s <= 126;
    const bool wide = a.bits == 16;
    // the operand rows of this row (two planes when wide), in panels (panel_off)
    auto at = [&](int pl, int j) { return a.out + panel_off(wide ? plane_row(row, pl) : (size_t)row, j, a.out_rows); };
    // Each element first takes the double-precision form of the rule (ln_elem_f64), which gives
    // the exact integer or declines; a declined element takes the integer rule below.
    const bool fpath = a.beta_frac == 0 && a.s <= 126;
    const double kr = ldexp((double)inv * (double)a.m, -a.s);
    const int32_t mean32 = (int32_t)mean;  // |x|, |mean| < 2^30, so x - mean fits i32
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = 4 * (lane + 64 * t);
        if (j >= d) continue;
        const v4i bv = *(const v4i *)(a.beta + j);
        const int64_t *gp = a.gm + j;
        const uint2 graw = *(const uint2 *)(a.gamma + j);  // four i16 gammas (j % 4 == 0)
        uint32_t packed = 0, packed_lo = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t c = (int64_t)xv[t][e] - mean;
            int64_t y = 0;
            bool done = false;
            if (fpath) {
                const int32_t ge = (int32_t)(int16_t)((e < 2 ? graw.x : graw.y) >> (16 * (e & 1)));
                int32_t f = 0;
                done = ln_elem_f64(xv[t][e] - mean32, kr, (double)ge, &f);
                y = (int64_t)f + bv[e];
            }
            if (done) {
            } else if (fast) {  // the rounding shift from the high word of (c inv) (gamma m)
                y = shift_round_hi(c * (int64_t)inv, gp[e], (uint32_t)a.s) + bv[e];
            } else {
                const i128 cinv = small ? (i128)(c * (int64_t)inv) : (i128)c * (i128)(u128)inv;
                const i128 p = cinv * (i128)gp[e];
                i128 yy;
                if (a.beta_frac == 0) {
                    yy = shift_round128(p, a.s, 126) + (i128)bv[e];
                } else {
                    const i128 cb = (i128)bv[e] << (a.s - a.beta_frac);
                    yy = shift_round128(p + cb, a.s, 126);
                }
                y = clamp128(yy, -32767, 32767);
            }
            if (!wide) {
                packed |= (uint32_t)(uint8_t)(int8_t)clamp64(y, -127, 127) << (8 * e);
            } else {
                const int32_t v = (int32_t)clamp64(y, -32767, 32767);
                packed |= (uint32_t)(uint8_t)(v >> 8) << (8 * e);
                packed_lo |= (uint32_t)(uint8_t)((v & 255) - 128) << (8 * e);
            }
        }
        *(uint32_t *)at(0, j) = packed;  // 4 bytes from j % 4 == 0: one panel
        if (wide) *(uint32_t *)at(1, j) = packed_lo;
    }
}

// Four rows per wave, 16 lanes per row (d % 4 == 0, d <= 64 NG <= 1024), 64 rows per workgroup
// of 16 waves. Lane q of a row holds columns 4 (q + 16 t) .. +4 for t < NG. Each row's sums
// (the 16 lanes' partials over 4 butterfly steps) go to LDS; then wave 0 forms mean, ln_inv and
// the rule's per-row terms for all 64 rows, one row per lane (not once per four rows in every
// wave: that per-row work is about 700 instructions of 128-bit integer and double arithmetic), and
// every wave reads its rows' terms back for the element rule. beta and gamma (the same columns
// for every row) are copied into LDS once per workgroup.
// Every load is unconditional, from a clamped address (a row past n_rows reads the last row, a
// column past d the last group; neither value is used): no branch around the loads.
// The input is the residual stream (|x| <= RES = 2^30 - 1): every square is below 2^60, so the
// four of a group sum in i64 without a carry.
// (8-bit outputs with |beta| <= 256 take k_layernorm_f32 instead: layernorm.hip.)
constexpr int LN_WAVES = 16;

template <int NG>
__global__ __launch_bounds__(64 * LN_WAVES) void k_layernorm_rows4(LnArgs a, int n_rows) {
    constexpr int NT = 64 * LN_WAVES, CI = (64 * NG + NT - 1) / NT, RW = 4 * LN_WAVES;
    __shared__ __attribute__((aligned(16))) int32_t s_beta[64 * NG];
    __shared__ __attribute__((aligned(16))) double s_gamma[64 * NG];
    // per row of the workgroup: the sums, then the rule's terms
    __shared__ int64_t s_sum[RW];
    __shared__ uint64_t s_lo[RW], s_hi[RW];
    __shared__ int32_t s_mx[RW], s_mn[RW];
    __shared__ int64_t s_mean[RW];
    __shared__ uint64_t s_inv[RW];
    __shared__ double s_kr[RW];
    __shared__ uint32_t s_flags[RW];  // bit 0 small, bit 1 fast
    const int lane = threadIdx.x & 63, q = lane & 15;
    const int rw = (threadIdx.x >> 6) * 4 + (lane >> 4);  // the lane's row in the workgroup
    const int row = blockIdx.x * RW + rw;
    const bool live = row < n_rows;
    const int d = a.d;
    const int rc = live ? row : n_rows - 1;
    const int32_t *x = a.x + (size_t)(a.src ? a.src[rc] : rc) * d;
    v4i xv[NG];
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = 4 * (q + 16 * t);
        xv[t] = *(const v4i *)(x + (j < d ? j : d - 4));
    }
#pragma unroll
    for (int i = 0; i < CI; i++) {  // gamma as doubles (exact)
        const int c = threadIdx.x + NT * i;
        if (c >= d) continue;
        s_beta[c] = a.beta[c];
        s_gamma[c] = (double)a.gamma[c];
    }
    // squares: the four of a group to an i64 partial (each < 2^60), the partials into a 128-bit
    // lo/hi with carries
    {
        int64_t sum = 0;
        uint64_t lo = 0, hi = 0;
        int32_t mx = INT32_MIN, mn = INT32_MAX;
#pragma unroll
        for (int t = 0; t < NG; t++) {
            const int j = 4 * (q + 16 * t);
            if (j >= d) continue;
            int64_t part = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int32_t v = xv[t][e];
                sum += v;
                part += (int64_t)v * v;
                mx = v > mx ? v : mx;
                mn = v < mn ? v : mn;
            }
            lo += (uint64_t)part;
            hi += lo < (uint64_t)part;
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {  // the 16 lanes of this row
            sum += __shfl_xor(sum, o, 64);
            const uint64_t lo2 = __shfl_xor(lo, o, 64), hi2 = __shfl_xor(hi, o, 64);
            lo += lo2;
            hi += hi2 + (lo < lo2);
            const int32_t mx2 = __shfl_xor(mx, o, 64), mn2 = __shfl_xor(mn, o, 64);
            mx = mx2 > mx ? mx2 : mx;
            mn = mn2 < mn ? mn2 : mn;
        }
        if (q == 0) {
            s_sum[rw] = sum;
            s_lo[rw] = lo;
            s_hi[rw] = hi;
            s_mx[rw] = mx;
            s_mn[rw] = mn;
        }
    }
    lds_barrier();  // the rows' sums, beta and gamma are in LDS
    const double inv_d = 1.0 / (double)d;  // |sum| <= d RES < 2^52, sq < d 2^62: the estimate forms
    if (threadIdx.x < RW) {  // wave 0: row threadIdx.x of the workgroup
        const int r = threadIdx.x;
        const int64_t sum = s_sum[r];
        const u128 Q = ((u128)s_hi[r] << 64) | s_lo[r];
        const int64_t mean = floor_div_est(sum, d, inv_d);
        const u128 sq = (u128)((i128)Q - 2 * (i128)mean * sum + (i128)d * mean * mean);
        const uint64_t inv = ln_inv_est(sq, (uint32_t)d, (uint32_t)a.k, (uint32_t)a.j, a.eps, inv_d);
        const int64_t c1 = (int64_t)s_mx[r] - mean, c2 = mean - (int64_t)s_mn[r];
        const uint64_t cmax = (uint64_t)(c1 > c2 ? c1 : c2);
        const bool small = (u128)cmax * inv < ((u128)1 << 63);
        const bool fast = small && a.beta_frac == 0 && a.s >= 64 && a.s <= 126;
        s_mean[r] = mean;
        s_inv[r] = inv;
        s_kr[r] = ldexp((double)inv * (double)a.m, -a.s);
        s_flags[r] = (small ? 1u : 0u) | (fast ? 2u : 0u);
    }
    lds_barrier();  // the rows' terms are in LDS
    if (!live) return;
    const bool wide = a.bits == 16;
    const int64_t mean = s_mean[rw];
    const uint64_t inv = s_inv[rw];
    const uint32_t flags = s_flags[rw];
    const bool small = flags & 1, fast = (flags >> 1) & 1;
    // the operand rows of this row (two planes when wide), in panels (panel_off); a wave's four
    // rows are adjacent in every panel, so each store instruction writes 256 contiguous bytes
    auto at = [&](int pl, int j) {
        return (uint32_t *)(a.out + panel_off(wide ? plane_row(row, pl) : (size_t)row, j, a.out_rows));
    };
    // Each element first takes the double-precision form of the rule (ln_elem_f64), which gives
    // the exact integer or declines. Every group is stored from it; the groups with a declined
    // element are then recomputed by the integer rule and stored again (the same lane rewrites
    // its own bytes, in order).
    const bool fpath = a.beta_frac == 0 && a.s <= 126;
    const double kr = s_kr[rw];
    const int32_t lim = wide ? 32767 : 127;
    const int32_t mean32 = (int32_t)mean;  // |x|, |mean| < 2^30, so x - mean fits i32
    auto put = [&](int j, const int32_t *y) {
        uint32_t packed = 0, packed_lo = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (!wide) {
                packed |= (uint32_t)(uint8_t)(int8_t)y[e] << (8 * e);
            } else {
                packed |= (uint32_t)(uint8_t)(y[e] >> 8) << (8 * e);
                packed_lo |= (uint32_t)(uint8_t)((y[e] & 255) - 128) << (8 * e);
            }
        }
        *at(0, j) = packed;  // 4 bytes from j % 4 == 0: one panel
        if (wide) *at(1, j) = packed_lo;
    };
    uint32_t redo = fpath ? 0u : ~0u;  // bit t: group t takes the integer rule
    if (fpath) {
#pragma unroll
        for (int t = 0; t < NG; t++) {
            const int j = 4 * (q + 16 * t);
            if (j >= d) continue;
            int32_t y[4];
            bool all = true;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int32_t f = 0;
                all &= ln_elem_f64(xv[t][e] - mean32, kr, s_gamma[j + e], &f);
                // a saturated f + beta lies beyond the clamp exactly when the sum does
                y[e] = med3_i32(__builtin_elementwise_add_sat(f, s_beta[j + e]), -lim, lim);
            }
            put(j, y);
            redo |= all ? 0u : 1u << t;
        }
    }
    if (redo == 0) return;
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = 4 * (q + 16 * t);
        if (j >= d || !((redo >> t) & 1)) continue;
        const int64_t *gp = a.gm + j;
        const int32_t *bp = a.beta + j;
        int32_t y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t c = (int64_t)xv[t][e] - mean;
            int64_t yy64;
            if (fast) {  // the rounding shift from the high word of (c inv) (gamma m)
                yy64 = shift_round_hi(c * (int64_t)inv, gp[e], (uint32_t)a.s) + bp[e];
            } else {
                const i128 cinv = small ? (i128)(c * (int64_t)inv) : (i128)c * (i128)(u128)inv;
                const i128 p = cinv * (i128)gp[e];
                i128 yy;
                if (a.beta_frac == 0) {
                    yy = shift_round128(p, a.s, 126) + (i128)bp[e];
                } else {
                    const i128 cb = (i128)bp[e] << (a.s - a.beta_frac);
                    yy = shift_round128(p + cb, a.s, 126);
                }
                yy64 = clamp128(yy, -32767, 32767);
            }
            y[e] = (int32_t)clamp64(yy64, -lim, lim);
        }
        put(j, y);
    }
}

hipError_t launch_layernorm(const LnArgs &a, int n_rows, hipStream_t stream) {
    if (n_rows <= 0) return hipSuccess;
    const dim3 grid((n_rows + 3) / 4);
    if (layernorm_f32_fits(a)) return launch_layernorm_f32(a, n_rows, stream);
    // the vector forms need d a multiple of 4 (4-byte groups of a row lie in one panel)
    // Fewer than 4,096 rows: a one-wave workgroup per row, spread over the CUs; the 16-lane form
    // would leave most of them idle (256 rows: 16 workgroups)
    if (n_rows < 4096 && a.d % 4 == 0 && a.d <= 2048) {
        if (a.d <= 1024) launch_k(k_layernorm_rows<4>, dim3(n_rows), dim3(64), 0, stream, a, n_rows);
        else launch_k(k_layernorm_rows<8>, dim3(n_rows), dim3(64), 0, stream, a, n_rows);
    } else if (a.d % 4 == 0 && a.d <= 1024) {
        const dim3 g4((n_rows + 4 * LN_WAVES - 1) / (4 * LN_WAVES)), b4(64 * LN_WAVES);
        if (a.d <= 768) launch_k(k_layernorm_rows4<12>, g4, b4, 0, stream, a, n_rows);
        else launch_k(k_layernorm_rows4<16>, g4, b4, 0, stream, a, n_rows);
    } else if (a.d % 4 == 0 && a.d <= 2048) {
        launch_k(k_layernorm_rows<8>, grid, dim3(256), 0, stream, a, n_rows);
    } else {
        launch_k(k_layernorm, dim3((n_rows + 3) / 4), dim3(256), 0, stream, a, n_rows);
    }
    return hipGetLastError();
}

// =============================================================================================
// K and V of each row into the cache at the row's position (reference.rs:246-252).
// Cache layout of one layer: [slot][head][position][hd].
// =============================================================================================

__global__ void k_kv_store(const RowInfo *rows, const int8_t *qkv, int d, int n_head, int hd,
                           int n_ctx, int8_t *kc, int8_t *vc) {
    const int r = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= d) return;
    const RowInfo ri = rows[r];
    const int h = c / hd, cc = c - h * hd;
    const size_t o = (((size_t)ri.slot * n_head + h) * n_ctx + ri.pos) * hd + cc;
    kc[o] = qkv[(size_t)r * 3 * d + d + c];
    vc[o] = qkv[(size_t)r * 3 * d + 2 * d + c];
}

hipError_t launch_kv_store(const RowInfo *rows, int n_rows, const int8_t *qkv, int d, int n_head,
                           int hd, int n_ctx, int8_t *kc, int8_t *vc, hipStream_t stream) {
    dim3 grid(n_rows, (d + 255) / 256);
    launch_k(k_kv_store, grid, dim3(256), 0, stream, rows, qkv, d, n_head, hd, n_ctx,
                       kc, vc);
    return hipGetLastError();
}

// =============================================================================================
// Causal integer attention (reference.rs:254-283, softmax.rs:78-104): one wave per (row, head)
// over the keys 0..pos of the row's slot. Three passes over the keys: the max score, the sum of
// the table entries, then p = floor(e * 2^P / S) and sum p * v in i64. Dots with v_dot4_i32_i8.
// =============================================================================================

__device__ __forceinline__ int32_t dot_key(const int *q4, const int8_t *k, int hd) {
    int32_t s = 0;
    const int *k4 = (const int *)k;
    for (int c = 0; c < hd / 4; c++) s = __builtin_amdgcn_sdot4(q4[c], k4[c], s, false);
    return s;
}

__global__ __launch_bounds__(256) void k_attend(AttnArgs a, int n_tasks) {
    __shared__ __attribute__((aligned(16))) int s_q[4][64];  // hd <= 256 bytes per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int task = blockIdx.x * 4 + wave;
    const bool valid = task < n_tasks;
    const int r = valid ? task / a.n_head : 0, h = valid ? task % a.n_head : 0;
    const int hd = a.hd;
    int slot, keys;
    if (a.rows) {
        slot = a.rows[r].slot;
        keys = a.keys ? (int)a.keys[r] : a.rows[r].pos + 1;
    } else {
        slot = r;
        keys = (int)a.keys[r];
    }
    keys = keys < 1 ? 1 : (keys > a.ctx_cap ? a.ctx_cap : keys);  // never read past the cache
    if (valid && lane < hd / 4) s_q[wave][lane] = ((const int *)(a.q + (size_t)r * a.ldq + h * hd))[lane];
    __syncthreads();
    if (!valid) return;
    const int *q4 = s_q[wave];
    const size_t base = ((size_t)slot * a.n_head + h) * a.ctx_cap * hd;
    const int8_t *K = a.kc + base, *V = a.vc + base;
    const int last = a.exp_len - 1;

    // pass 1: M = max score
    int64_t mx = INT64_MIN;
    for (int j = lane; j < keys; j += 64) {
        const int64_t s = clamp64(rescale_small(dot_key(q4, K + (size_t)j * hd, hd), a.score_m,
                                                a.score_s), -SCORE_LIMIT, SCORE_LIMIT);
        mx = s > mx ? s : mx;
    }
    mx = wave_max64(mx);
    // pass 2: S = sum e_j
    int64_t sum = 0;
    for (int j = lane; j < keys; j += 64) {
        const int64_t s = clamp64(rescale_small(dot_key(q4, K + (size_t)j * hd, hd), a.score_m,
                                                a.score_s), -SCORE_LIMIT, SCORE_LIMIT);
        const int64_t dd = mx - s;
        sum += a.exp_table[dd < last ? dd : last];
    }
    sum = wave_sum64(sum);
    // pass 3: p_j and the weighted sum of the values (c = lane + 64 t)
    int64_t acc[4] = {0, 0, 0, 0};
    for (int j0 = 0; j0 < keys; j0 += 64) {
        const int j = j0 + lane;
        uint64_t p = 0;
        if (j < keys) {
            const int64_t s = clamp64(rescale_small(dot_key(q4, K + (size_t)j * hd, hd), a.score_m,
                                                    a.score_s), -SCORE_LIMIT, SCORE_LIMIT);
            const int64_t dd = mx - s;
            const uint64_t e = (uint64_t)a.exp_table[dd < last ? dd : last];
            p = (e << a.softmax_p) / (uint64_t)sum;
        }
        const int cnt = keys - j0 < 64 ? keys - j0 : 64;
        for (int jj = 0; jj < cnt; jj++) {
            const int64_t pj = (int64_t)__shfl(p, jj, 64);
            const int8_t *v = V + (size_t)(j0 + jj) * hd;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int c = lane + 64 * t;
                if (c < hd) acc[t] += pj * (int64_t)v[c];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int c = lane + 64 * t;
        if (c < hd)
            *attn_out(a, r, h * hd + c) =
                (int8_t)clamp128(rescale_full(acc[t], a.out_m, a.out_s), -127, 127);
    }
}

hipError_t launch_attend(const AttnArgs &a, int n_rows, hipStream_t stream) {
    const int tasks = n_rows * a.n_head;
    if (tasks <= 0) return hipSuccess;
    launch_k(k_attend, dim3((tasks + 3) / 4), dim3(256), 0, stream, a, tasks);
    return hipGetLastError();
}

// =============================================================================================
// Decode attention split over key chunks, for few rows over long contexts (the row kernel above
// has only rows x heads waves). The same integer steps as reference.rs:254-283, over
// (row, head, chunk) waves in four launches:
//   1. the dots q . k of the chunk's keys (kept) and the chunk's smallest and largest dot;
//   2. the row max M (the score is monotone in the dot: the largest score is the score of the
//      largest or of the smallest dot over all chunks) and the chunk's sum of the table entries
//      e = table[min(M - s, last)];
//   3. S = the sum over chunks, p = floor(e 2^P / S) from the kept dots again and the chunk's sum
//      of p v per channel in i64 (hd / 16 lanes x 16 channels per key, 16-byte loads of V);
//   4. the sum of the chunk partials and the output rescale.
// Integer sums are exact in any order, so the result is the reference's.
// =============================================================================================

// score = clamp(rescale(dot, m, s), +-2^40): |dot| <= hd 2^14 <= 2^22, so |dot m| < 2^53 and one
// multiply-add and an arithmetic shift are exact (a shift of 63 or more gives 0). With s >= 13
// the score stays within +-2^40 and the clamp is a no-op.
__host__ __device__ inline bool attn_noclamp(const AttnArgs &a) { return a.score_s >= 13; }

// The attention output byte clamp(rescale(v, m, s), +-127) for an exact |v| < 2^53 (the sum of
// p v): y = v m 2^-s + 1/2 in double (mo = m 2^-s, exact; v exact; one rounding in the fused
// multiply-add, relative 2^-53). When |y| >= 256 the clamp decides; when y lies at least 2^-30
// from an integer floor(y) is exact (|y| < 256: the error is below 2^-45); else the i128 rule.
__device__ __forceinline__ int32_t attn_out_byte(int64_t v, double mo, int32_t m, int s) {
    const double y = fma((double)v, mo, 0.5);
    const double f = __builtin_amdgcn_fract(y);
    if (fabs(y) >= 256.0 || fabs(f - 0.5) <= 0.5 - 0x1p-30) return (int32_t)fmin(fmax(y - f, -127.0), 127.0);
    return (int32_t)clamp128(rescale_full(v, m, s), -127, 127);
}

template <bool NOCLAMP>
__device__ __forceinline__ int64_t attn_score(const AttnArgs &a, int32_t dot) {
    const int s_eff = a.score_s < 63 ? a.score_s : 63;
    const int64_t s_half = s_eff ? (int64_t)1 << (s_eff - 1) : 0;
    const int64_t r = ((int64_t)dot * a.score_m + s_half) >> s_eff;
    return NOCLAMP ? r : clamp64(r, -SCORE_LIMIT, SCORE_LIMIT);
}

struct SplitScratch {
    int32_t *dots, *mm;
    uint64_t *ps;
    int64_t *part;
};

__device__ __forceinline__ SplitScratch split_scratch(void *base, int n_rows, int H, int cap, int chunks, int hd) {
    SplitScratch s;
    auto al = [](size_t x) { return (x + 255) / 256 * 256; };
    char *p = (char *)base;
    const size_t rh = (size_t)n_rows * H;
    s.dots = (int32_t *)p;
    p += al(rh * cap * 4);
    s.mm = (int32_t *)p;
    p += al(rh * chunks * 8);
    s.ps = (uint64_t *)p;
    p += al(rh * chunks * 8);
    s.part = (int64_t *)p;
    return s;
}

__device__ __forceinline__ int split_keys(const AttnArgs &a, int r) {
    int keys = a.keys ? (int)a.keys[r] : a.rows[r].pos + 1;
    return keys < 1 ? 1 : (keys > a.ctx_cap ? a.ctx_cap : keys);
}

__device__ __forceinline__ int split_slot(const AttnArgs &a, int r) { return a.rows ? a.rows[r].slot : r; }

// The row maximum of the scores, from every chunk's extreme dots (the score is monotone in the dot).
template <bool NOCLAMP>
__device__ __forceinline__ int64_t split_max(const AttnArgs &a, const SplitScratch &S, const SplitPlan &pl,
                                             int rh, int nch) {
    int64_t M = INT64_MIN;
    for (int cc = 0; cc < nch; cc++) {
        const int32_t mn = S.mm[((size_t)rh * pl.chunks + cc) * 2], mx = S.mm[((size_t)rh * pl.chunks + cc) * 2 + 1];
        const int64_t s0 = attn_score<NOCLAMP>(a, mn), s1 = attn_score<NOCLAMP>(a, mx);
        M = s0 > M ? s0 : M;
        M = s1 > M ? s1 : M;
    }
    return M;
}

// HD = the head dimension (16 .. 256, a power of two). A lane takes J keys per round and issues
// the loads of all J (HD bytes each) before the first dot, so a wave keeps up to 1 KB per lane
// of K in flight instead of one key's.
template <int HD>
__global__ __launch_bounds__(64) void k_split_dots(AttnArgs a, int n_rows, SplitPlan pl, void *scratch) {
    constexpr int NT = HD / 16, J = NT >= 16 ? 1 : (16 / NT > 4 ? 4 : 16 / NT);
    __shared__ __attribute__((aligned(16))) int s_q[64];  // hd <= 256 bytes
    const int rh = blockIdx.x, c = blockIdx.y, lane = threadIdx.x;
    const int r = rh / a.n_head, h = rh - r * a.n_head;
    const SplitScratch S = split_scratch(scratch, n_rows, a.n_head, a.ctx_cap, pl.chunks, HD);
    const int keys = split_keys(a, r), k0 = c * pl.chunk_keys;
    const int k1 = k0 + pl.chunk_keys < keys ? k0 + pl.chunk_keys : keys;
    if (lane < HD / 4) s_q[lane] = ((const int *)(a.q + (size_t)r * a.ldq + h * HD))[lane];
    __syncthreads();
    const int8_t *K = a.kc + ((size_t)split_slot(a, r) * a.n_head + h) * a.ctx_cap * HD;
    int32_t dmin = INT32_MAX, dmax = INT32_MIN;
    for (int kb = k0 + lane; kb < k1; kb += J * 64) {
        v4i kk[J][NT];
#pragma unroll
        for (int j = 0; j < J; j++) {  // a key past the chunk reloads the lane's first key
            const int k = kb + 64 * j;
            const v4i *k16 = (const v4i *)(K + (size_t)(k < k1 ? k : kb) * HD);
#pragma unroll
            for (int t = 0; t < NT; t++) kk[j][t] = k16[t];
        }
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int k = kb + 64 * j;
            if (k >= k1) break;
            int32_t d = 0;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                d = __builtin_amdgcn_sdot4(s_q[4 * t], kk[j][t][0], d, false);
                d = __builtin_amdgcn_sdot4(s_q[4 * t + 1], kk[j][t][1], d, false);
                d = __builtin_amdgcn_sdot4(s_q[4 * t + 2], kk[j][t][2], d, false);
                d = __builtin_amdgcn_sdot4(s_q[4 * t + 3], kk[j][t][3], d, false);
            }
            S.dots[(size_t)rh * a.ctx_cap + k] = d;
            dmin = d < dmin ? d : dmin;
            dmax = d > dmax ? d : dmax;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int32_t u = __shfl_xor(dmin, o, 64), v = __shfl_xor(dmax, o, 64);
        dmin = u < dmin ? u : dmin;
        dmax = v > dmax ? v : dmax;
    }
    if (lane == 0) {  // an empty chunk keeps (min, max) = (INT32_MAX, INT32_MIN)
        S.mm[((size_t)rh * pl.chunks + c) * 2] = dmin;
        S.mm[((size_t)rh * pl.chunks + c) * 2 + 1] = dmax;
    }
}

template <bool NOCLAMP>
__global__ __launch_bounds__(64) void k_split_sum(AttnArgs a, int n_rows, SplitPlan pl, void *scratch) {
    const int rh = blockIdx.x, c = blockIdx.y, lane = threadIdx.x;
    const int r = rh / a.n_head;
    const SplitScratch S = split_scratch(scratch, n_rows, a.n_head, a.ctx_cap, pl.chunks, a.hd);
    const int keys = split_keys(a, r), k0 = c * pl.chunk_keys;
    const int k1 = k0 + pl.chunk_keys < keys ? k0 + pl.chunk_keys : keys;
    const int64_t M = split_max<NOCLAMP>(a, S, pl, rh, (keys + pl.chunk_keys - 1) / pl.chunk_keys);
    const int64_t last = a.exp_len - 1;
    uint64_t sum = 0;
    for (int k = k0 + lane; k < k1; k += 64) {
        const int64_t dd = M - attn_score<NOCLAMP>(a, S.dots[(size_t)rh * a.ctx_cap + k]);
        sum += (uint64_t)a.exp_table[dd < last ? dd : last];
    }
    sum = (uint64_t)wave_sum64((int64_t)sum);
    if (lane == 0) S.ps[(size_t)rh * pl.chunks + c] = sum;
}

__global__ void k_split_out(AttnArgs a, int n_rows, SplitPlan pl, void *scratch) {
    const int rh = blockIdx.x, t = threadIdx.x;
    const int r = rh / a.n_head, h = rh - r * a.n_head, hd = a.hd;
    if (t >= hd) return;
    const SplitScratch S = split_scratch(scratch, n_rows, a.n_head, a.ctx_cap, pl.chunks, hd);
    const int keys = split_keys(a, r), nch = (keys + pl.chunk_keys - 1) / pl.chunk_keys;
    int64_t o = 0;
    for (int cc = 0; cc < nch; cc++) o += S.part[((size_t)rh * pl.chunks + cc) * hd + t];
    *attn_out(a, r, h * hd + t) = (int8_t)clamp128(rescale_full(o, a.out_m, a.out_s), -127, 127);
}

// ---- The pieces of the one-launch decode kernels ---------------------------------------------------
// Sum p v of one query row is a product of a 64-channel x 64-key matrix with p, and p is four
// balanced i8 digits (the bytes of p + 0x80808080, xor 0x80): one v_mfma_i32_16x16x64_i8 takes 16
// channels x 64 keys against the four digit planes as four of its columns (the other twelve
// repeat them), so a block of 64 keys is 4 MFMAs where 24-bit multiplies took 192 VALU
// instructions a wave, and the sums need no butterfly over the lanes.
// A block's V rows lie in LDS as dense rows of 16 NC bytes (NC = 4: head dims from 64 on, in groups
// of 64 channels; below that one group of hd), 16-byte chunk c of row r at slot NC r + (c ^ vsw(r));
// the V^T operand comes by transposing reads (as in k_attend_short), whose operand byte 4 t + e of
// lane group g holds key 16 t + 4 g + e. `mem` is 1 KiB of the wave.
template <int NC>
__device__ __forceinline__ int vsw(int r) {
    return NC == 4 ? ((r >> 1) ^ (r >> 3)) & 3 : NC == 2 ? (r >> 2) & 1 : 0;
}

// Lane l's p of key l to the digit operand of the block.
__device__ __forceinline__ v4i decode_pv_digits(int8_t *mem, uint32_t p, int lane) {
    const uint32_t q = (p + 0x80808080u) ^ 0x80808080u;
    int8_t *w = mem + 16 * ((lane >> 2) & 3) + 4 * (lane >> 4) + (lane & 3);
#pragma unroll
    for (int k = 0; k < 4; k++) w[64 * k] = (int8_t)(q >> (8 * k));
    return *(const v4i *)(mem + 64 * (lane & 3) + 16 * (lane >> 4));
}
template <int NC>
__device__ __forceinline__ void decode_pv_block(const int8_t *sv, const v4i &pf, int lane, v4i *acc) {
    const int ql = lane & 15, qg = lane >> 4;
    const int tr_k = ql >> 1, tr_h = ql & 1;
    const int key0 = 16 * (tr_k >> 2) + 4 * qg + (tr_k & 3);
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int8_t *p0 = sv + (NC * key0 + (c ^ vsw<NC>(key0 & 15))) * 16 + 8 * tr_h;
        const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)p0);
        const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)(p0 + 32 * 16 * NC));
        acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{r0[0], r0[1], r1[0], r1[1]}, pf, acc[c], 0, 0, 0);
    }
}

// acc[c][e] of lane l holds channel 16 c + 4 (l / 16) + e of plane l % 16 (< 4): to [plane][64] in mem.
template <int NC>
__device__ __forceinline__ void decode_pv_store(int8_t *mem, int lane, const v4i *acc) {
    if ((lane & 15) < 4) {
#pragma unroll
        for (int c = 0; c < NC; c++) *(v4i *)(mem + 256 * (lane & 15) + 64 * c + 16 * (lane >> 4)) = acc[c];
    }
}
// The planes' sum of channel ch: below 2^24 per plane, |sum| <= 1,024 2^30 2^7 < 2^53.
__device__ __forceinline__ int64_t decode_pv_sum(const int8_t *mem, int ch) {
    const int32_t *m = (const int32_t *)mem + ch;
    return (int64_t)m[0] + (int64_t)m[64] * 256 + (int64_t)m[128] * 65536 + (int64_t)m[192] * 16777216;
}

// The split form's sums p v of a chunk: one wave, 64 keys at a time on the digit planes (above), the
// next block's V rows in flight. (One i64 multiply-add a channel and key and a butterfly at the end
// took 29.1 us at head_dim 64, 2,000 keys, 512 row-heads; this 13.0.) At most 4,096 keys: below 2^26
// a plane.
template <bool NOCLAMP, int HD>
__global__ __launch_bounds__(64) void k_split_pv(AttnArgs a, int n_rows, SplitPlan pl, void *scratch) {
    constexpr int QT = HD / 16, NC = HD < 64 ? QT : 4, NG = QT / NC, RB = 16 * NC, RL = 64 / NC, SH = NC / 2;
    __shared__ __attribute__((aligned(16))) int8_t s_v[64 * HD], s_mem[1024];
    const int rh = blockIdx.x, c = blockIdx.y, lane = threadIdx.x;
    const int r = rh / a.n_head, h = rh - r * a.n_head;
    const SplitScratch S = split_scratch(scratch, n_rows, a.n_head, a.ctx_cap, pl.chunks, HD);
    int64_t *part = S.part + ((size_t)rh * pl.chunks + c) * HD;
    const int keys = split_keys(a, r), k0 = c * pl.chunk_keys;
    const int k1 = k0 + pl.chunk_keys < keys ? k0 + pl.chunk_keys : keys;
    if (k0 >= k1) {  // an empty chunk contributes nothing
        for (int i = lane; i < HD; i += 64) part[i] = 0;
        return;
    }
    // lane l: chunk (l % NC) ^ vsw of rows l / NC + RL u (keys past the chunk reload its last key;
    // their weight is 0)
    const int8_t *V = a.vc + ((size_t)split_slot(a, r) * a.n_head + h) * a.ctx_cap * HD;
    v4i vr[NG][NC];
    auto load = [&](int kb) {
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int row = RL * u + (lane >> SH), k = kb + row;
            const int8_t *v = V + (size_t)(k < k1 ? k : k1 - 1) * HD + 16 * ((lane & (NC - 1)) ^ vsw<NC>(row & 15));
#pragma unroll
            for (int g = 0; g < NG; g++) vr[g][u] = *(const v4i *)(v + 64 * g);
        }
    };
    load(k0);
    const int nch = (keys + pl.chunk_keys - 1) / pl.chunk_keys;
    const int64_t M = split_max<NOCLAMP>(a, S, pl, rh, nch);
    uint64_t sum = 0;
    for (int cc = 0; cc < nch; cc++) sum += S.ps[(size_t)rh * pl.chunks + cc];
    const uint64_t frac = sum >= 2 ? div_2p64(sum) : 0;
    const int64_t last = a.exp_len - 1;
    v4i acc[NG][NC];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int i = 0; i < NC; i++) acc[g][i] = v4i{0, 0, 0, 0};
    for (int kb = k0; kb < k1; kb += 64) {
        uint64_t q = 0;
        if (kb + lane < k1) {
            const int64_t dd = M - attn_score<NOCLAMP>(a, S.dots[(size_t)rh * a.ctx_cap + kb + lane]);
            const uint64_t num = (uint64_t)a.exp_table[dd < last ? dd : last] << a.softmax_p;
            q = num;
            if (sum >= 2) {
                q = __umul64hi(num, frac);  // q <= floor(num / S) <= q + 1
                if (num - q * sum >= sum) q++;
            }
        }
#pragma unroll
        for (int g = 0; g < NG; g++)
#pragma unroll
            for (int u = 0; u < NC; u++) *(v4i *)(s_v + 64 * RB * g + 1024 * u + 16 * lane) = vr[g][u];
        load(kb + 64);
        const v4i pf = decode_pv_digits(s_mem, (uint32_t)q, lane);  // q <= 2^P <= 2^30
#pragma unroll
        for (int g = 0; g < NG; g++) decode_pv_block<NC>(s_v + 64 * RB * g, pf, lane, acc[g]);
    }
#pragma unroll
    for (int g = 0; g < NG; g++) {
        decode_pv_store<NC>(s_mem, lane, acc[g]);
        asm volatile("" ::: "memory");  // (the wave's LDS operations stay in order)
        if (lane < RB) part[64 * g + lane] = decode_pv_sum(s_mem, lane);
        asm volatile("" ::: "memory");
    }
}

// The extreme values over the wave.
__device__ __forceinline__ void wave_min_max(int32_t &mn, int32_t &mx) {
    butterfly<64>([&](auto st) {
        constexpr int S = decltype(st)::value;
        const int32_t u = lane_move<S>(mn), v = lane_move<S>(mx);
        mn = u < mn ? u : mn;
        mx = v > mx ? v : mx;
    });
}
__device__ __forceinline__ uint64_t wave_sum_dpp(uint64_t v) {
    butterfly<64>([&](auto st) { v += (uint64_t)lane_move64<decltype(st)::value>((int64_t)v); });
    return v;
}

// Decode attention for head_dim 64 and at most 1,024 keys in one launch: one workgroup (4 waves)
// per (row, head). The row's K rows (thread t: keys t + 256 j) and the V rows of the
// wave's key blocks go to registers in one round of
// loads with no branch around them, K first, so the dots wait for K alone (the compiler counts the
// in-order loads exactly; with part of V going to LDS by global_load_lds it waited for every
// load); the dots, the row max, the table sum, the weights p and the sums p v then follow the rules
// of the split kernels above. 140 VGPRs: three workgroups per CU (768 row-heads in one round). Measured
// at 768 row-heads over cold caches: 1,024 keys 20.2 us (100.8 MB: 5.0 TB/s), 512 keys 12.4. What the layout
// rests on, at 1,024 keys with the sums p v still on 24-bit multiplies: 34.2 us with all of V in LDS
// (two workgroups per CU), 31.0 with half, 29.8 with none.
template <bool NOCLAMP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attend_decode64(AttnArgs a,
                                                                                                  int kmax) {
    __shared__ __attribute__((aligned(16))) int8_t s_v[4][4096];    // a wave's block of V rows
    __shared__ __attribute__((aligned(16))) int8_t s_mem[4][1024];  // a wave's digits, then its plane sums
    __shared__ int32_t s_mm[2][4];
    __shared__ uint64_t s_sum[4];
    const int rh = blockIdx.x, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int r = rh / a.n_head, h = rh - r * a.n_head;
    int keys = split_keys(a, r);
    keys = keys < kmax ? keys : kmax;  // the launch's bound holds every row's count
    const size_t base = ((size_t)split_slot(a, r) * a.n_head + h) * a.ctx_cap * 64;
    // q straight into every thread's registers (one 64-byte row, the same for all)
    int qv[16];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const v4i q4 = ((const v4i *)(a.q + (size_t)r * a.ldq + h * 64))[t];
#pragma unroll
        for (int e = 0; e < 4; e++) qv[4 * t + e] = q4[e];
    }
    // K: four keys per thread, with no branch around the loads (keys past the row reload the
    // row's last key and are left out of every sum)
    v4i kk[4][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = tid + 256 * j;
        const v4i *k16 = (const v4i *)(a.kc + base + (size_t)(k < keys ? k : keys - 1) * 64);
#pragma unroll
        for (int t = 0; t < 4; t++) kk[j][t] = k16[t];
    }
    // V after K: the rows of this wave's four blocks of 64 keys, 64 (4 j + w) .. (the keys whose p its
    // lanes form), lane l the chunk (l % 4) ^ vsw of row 16 u + l / 4 (keys past the row reload the
    // row's last key; their weight is 0)
    v4i vr[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int row = 16 * (i & 3) + (lane >> 2), k = 64 * (4 * (i >> 2) + w) + row;
        vr[i] = *(const v4i *)(a.vc + base + (size_t)(k < keys ? k : keys - 1) * 64 + 16 * ((lane & 3) ^ vsw<4>(row & 15)));
    }
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first wait
    // the dots wait for K alone (the compiler's waits on the K registers)
    int32_t d[4];
    int32_t dmin = INT32_MAX, dmax = INT32_MIN;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int32_t x = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            x = __builtin_amdgcn_sdot4(qv[4 * t], kk[j][t][0], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 1], kk[j][t][1], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 2], kk[j][t][2], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 3], kk[j][t][3], x, false);
        }
        d[j] = x;
        if (tid + 256 * j < keys) {
            dmin = x < dmin ? x : dmin;
            dmax = x > dmax ? x : dmax;
        }
    }
    wave_min_max(dmin, dmax);
    if (lane == 0) {
        s_mm[0][w] = dmin;
        s_mm[1][w] = dmax;
    }
    lds_barrier();  // not the fence of __syncthreads, which would wait for the V loads too
    // the row max of the scores: the score is monotone in the dot, so it is the score of the
    // smallest or of the largest dot
    int64_t M = INT64_MIN;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int32_t mn = s_mm[0][i], mx = s_mm[1][i];
        if (mn > mx) continue;  // a wave with no key
        const int64_t s0 = attn_score<NOCLAMP>(a, mn), s1 = attn_score<NOCLAMP>(a, mx);
        M = s0 > M ? s0 : M;
        M = s1 > M ? s1 : M;
    }
    const int64_t last = a.exp_len - 1;
    uint32_t e[4];
    uint64_t sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        e[j] = 0;
        if (tid + 256 * j < keys) {
            const int64_t dd = M - attn_score<NOCLAMP>(a, d[j]);
            e[j] = (uint32_t)a.exp_table[dd < last ? dd : last];
            sum += e[j];
        }
    }
    sum = wave_sum_dpp(sum);
    if (lane == 0) s_sum[w] = sum;
    __syncthreads();
    sum = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    const double R = ldexp(1.0 / (double)sum, a.softmax_p);
    const double sp = softmax_sp(sum, a.softmax_p);
    v4i acc[4];
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (64 * (4 * j + w) >= keys) break;  // uniform
#pragma unroll
        for (int u = 0; u < 4; u++) *(v4i *)(s_v[w] + 1024 * u + 16 * lane) = vr[4 * j + u];
        // p <= 2^P <= 2^30; 0 for keys past the row (e = 0)
        decode_pv_block<4>(s_v[w], decode_pv_digits(s_mem[w], softmax_p_of(e[j], R, sp), lane), lane, acc);
    }
    decode_pv_store<4>(s_mem[w], lane, acc);
    __syncthreads();
    if (tid < 64) {
        const int64_t o = decode_pv_sum(s_mem[0], tid) + decode_pv_sum(s_mem[1], tid) +
                          decode_pv_sum(s_mem[2], tid) + decode_pv_sum(s_mem[3], tid);
        const double mo = a.out_s > 95 ? 0.0 : ldexp((double)a.out_m, -a.out_s);
        *attn_out(a, r, h * 64 + tid) = (int8_t)attn_out_byte(o, mo, a.out_m, a.out_s);
    }
}

// The same for head dims 16, 32 and 128: 4 waves of 4 keys a lane, at head_dim 128 8 of 2. (At head_dim
// 64 this form, with the same loads in the same order, took 14.3 us where k_attend_decode64 takes
// 14.0, 768 row-heads at 640 keys.) Kernel time against
// the four split launches: head_dim 128, 600 row-heads at 388 keys 35.3 -> 16.9 us; head_dim 32, 1,200
// row-heads at 1,000 keys 41.7 -> 12.1 us.
template <bool NOCLAMP, int HD>
__global__ __launch_bounds__(HD > 64 ? 512 : 256) __attribute__((amdgpu_waves_per_eu(2))) void k_attend_decode_wg(
    AttnArgs a, int kmax) {
    constexpr int NW = HD > 64 ? 8 : 4, NTH = 64 * NW, KT = 1024 / NTH, QT = HD / 16;
    constexpr int NC = HD < 64 ? QT : 4, NG = QT / NC, RB = 16 * NC;  // 64-channel groups of NC chunks
    __shared__ __attribute__((aligned(16))) int8_t s_v[NW][64 * RB];  // a wave's block of V rows, one group
    __shared__ __attribute__((aligned(16))) int8_t s_mem[NW][NG * 1024];  // a wave's digits, then its plane sums
    __shared__ int32_t s_mm[2][NW];
    __shared__ uint64_t s_sum[NW];
    const int rh = blockIdx.x, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int r = rh / a.n_head, h = rh - r * a.n_head;
    int keys = split_keys(a, r);
    keys = keys < kmax ? keys : kmax;  // the launch's bound holds every row's count
    const size_t base = ((size_t)split_slot(a, r) * a.n_head + h) * a.ctx_cap * HD;
    // q straight into every thread's registers (one row, the same for all)
    int qv[4 * QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        const v4i q4 = ((const v4i *)(a.q + (size_t)r * a.ldq + h * HD))[t];
#pragma unroll
        for (int e = 0; e < 4; e++) qv[4 * t + e] = q4[e];
    }
    // K: KT keys per thread, with no branch around the loads (keys past the row reload the
    // row's last key and are left out of every sum)
    v4i kk[KT][QT];
#pragma unroll
    for (int j = 0; j < KT; j++) {
        const int k = tid + NTH * j;
        const v4i *k16 = (const v4i *)(a.kc + base + (size_t)(k < keys ? k : keys - 1) * HD);
#pragma unroll
        for (int t = 0; t < QT; t++) kk[j][t] = k16[t];
    }
    // V after K: the rows of this wave's KT blocks of 64 keys, 64 (NW j + w) .. (the keys whose p its
    // lanes form), by group of channels; a load takes 64 / NC rows, lane l the chunk (l % NC) ^ vsw of
    // row l / NC of them (keys past the row reload the row's last key; their weight is 0)
    constexpr int RL = 64 / NC, SH = NC / 2;  // (log2 of NC)
    v4i vr[KT][NG][NC];
#pragma unroll
    for (int j = 0; j < KT; j++) {
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int row = RL * u + (lane >> SH), k = 64 * (NW * j + w) + row;
            const int8_t *v = a.vc + base + (size_t)(k < keys ? k : keys - 1) * HD + 16 * ((lane & (NC - 1)) ^ vsw<NC>(row & 15));
#pragma unroll
            for (int g = 0; g < NG; g++) vr[j][g][u] = *(const v4i *)(v + 64 * g);
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first wait
    // the dots wait for K alone (the compiler's waits on the K registers)
    int32_t d[KT];
    int32_t dmin = INT32_MAX, dmax = INT32_MIN;
#pragma unroll
    for (int j = 0; j < KT; j++) {
        int32_t x = 0;
#pragma unroll
        for (int t = 0; t < QT; t++) {
            x = __builtin_amdgcn_sdot4(qv[4 * t], kk[j][t][0], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 1], kk[j][t][1], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 2], kk[j][t][2], x, false);
            x = __builtin_amdgcn_sdot4(qv[4 * t + 3], kk[j][t][3], x, false);
        }
        d[j] = x;
        if (tid + NTH * j < keys) {
            dmin = x < dmin ? x : dmin;
            dmax = x > dmax ? x : dmax;
        }
    }
    wave_min_max(dmin, dmax);
    if (lane == 0) {
        s_mm[0][w] = dmin;
        s_mm[1][w] = dmax;
    }
    lds_barrier();  // not the fence of __syncthreads, which would wait for the V loads too
    // the row max of the scores: the score is monotone in the dot, so it is the score of the
    // smallest or of the largest dot
    int64_t M = INT64_MIN;
#pragma unroll
    for (int i = 0; i < NW; i++) {
        const int32_t mn = s_mm[0][i], mx = s_mm[1][i];
        if (mn > mx) continue;  // a wave with no key
        const int64_t s0 = attn_score<NOCLAMP>(a, mn), s1 = attn_score<NOCLAMP>(a, mx);
        M = s0 > M ? s0 : M;
        M = s1 > M ? s1 : M;
    }
    const int64_t last = a.exp_len - 1;
    uint32_t e[KT];
    uint64_t sum = 0;
#pragma unroll
    for (int j = 0; j < KT; j++) {
        e[j] = 0;
        if (tid + NTH * j < keys) {
            const int64_t dd = M - attn_score<NOCLAMP>(a, d[j]);
            e[j] = (uint32_t)a.exp_table[dd < last ? dd : last];
            sum += e[j];
        }
    }
    sum = wave_sum_dpp(sum);
    if (lane == 0) s_sum[w] = sum;
    __syncthreads();
    sum = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) sum += s_sum[i];
    const double R = ldexp(1.0 / (double)sum, a.softmax_p);
    const double sp = softmax_sp(sum, a.softmax_p);
    v4i acc[NG][NC];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[g][c] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < KT; j++) {
        if (64 * (NW * j + w) >= keys) break;  // uniform
        v4i pf;
#pragma unroll
        for (int g = 0; g < NG; g++) {
#pragma unroll
            for (int u = 0; u < NC; u++) *(v4i *)(s_v[w] + 1024 * u + 16 * lane) = vr[j][g][u];
            if (g == 0) {  // p <= 2^P <= 2^30; 0 for keys past the row (e = 0)
                __builtin_amdgcn_sched_barrier(0);  // the weights' arithmetic covers the stores of V
                pf = decode_pv_digits(s_mem[w], softmax_p_of(e[j], R, sp), lane);
            }
            decode_pv_block<NC>(s_v[w], pf, lane, acc[g]);
        }
    }
#pragma unroll
    for (int g = 0; g < NG; g++) decode_pv_store<NC>(s_mem[w] + 1024 * g, lane, acc[g]);
    __syncthreads();
    if (tid < HD) {
        int64_t o = 0;
#pragma unroll
        for (int i = 0; i < NW; i++) o += decode_pv_sum(s_mem[i] + 1024 * (tid >> 6), tid & 63);
        const double mo = a.out_s > 95 ? 0.0 : ldexp((double)a.out_m, -a.out_s);
        *attn_out(a, r, h * HD + tid) = (int8_t)attn_out_byte(o, mo, a.out_m, a.out_s);
    }
}

// Decode attention for at most 64 KB keys (head_dim 64: KB <= 4): one wave per (row, head), four
// independent waves per workgroup, no barrier. Lane l holds the K rows of keys l + 64 j, and the
// wave's V rows go to its own LDS region ([channel group][key][16 NC B], 64 / NC keys per
// global_load_lds), all loads issued at once. The dots, the row max (from the extreme dots), the table
// sum and p = floor(e 2^P / S) follow the rules of the kernels above, the sums p v come from the digit
// planes block by block. Against the four split launches, a prefill pass of 120,792 row-heads at
// head_dim 32 and up to 400 keys: 665 -> 196 us a layer.
template <bool NOCLAMP, int KB, int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attend_decode_wave(AttnArgs a, int n_rh,
                                                                                                     int kmax) {
    constexpr int QT = HD / 16, NC = HD < 64 ? QT : 4, NG = QT / NC, RB = 16 * NC, RL = 64 / NC, SH = NC / 2;
    const int lane = threadIdx.x & 63;
    const int rh = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (rh >= n_rh) return;
    const int r = rh / a.n_head, h = rh - r * a.n_head;
    int keys = split_keys(a, r);
    keys = keys < kmax ? keys : kmax;
    const size_t base = ((size_t)split_slot(a, r) * a.n_head + h) * a.ctx_cap * HD;
    int qv[4 * QT];
#pragma unroll
    for (int t = 0; t < 4 * QT; t++) qv[t] = ((const int *)(a.q + (size_t)r * a.ldq + h * HD))[t];
    extern __shared__ __attribute__((aligned(16))) int8_t s_v[];  // 4 waves x (KB blocks of V rows, 1 KiB)
    int8_t *sv = s_v + (threadIdx.x >> 6) * (KB * 64 * HD + 1024), *mem = sv + KB * 64 * HD;
    v4i kk[KB][QT];
#pragma unroll
    for (int j = 0; j < KB; j++) {
        if (64 * j >= keys) break;  // uniform: the rounds past the row issue nothing
        const int k = lane + 64 * j;
        const v4i *k16 = (const v4i *)(a.kc + base + (size_t)(k < keys ? k : keys - 1) * HD);
#pragma unroll
        for (int t = 0; t < QT; t++) kk[j][t] = k16[t];
    }
#pragma unroll
    for (int i = 0; i < NC * KB; i++) {
        if (RL * i >= keys) break;
        const int k = (lane >> SH) + RL * i, c = (lane & (NC - 1)) ^ vsw<NC>((lane >> SH) & 15);
        const int8_t *v = a.vc + base + (size_t)(k < keys ? k : keys - 1) * HD + 16 * c;
#pragma unroll
        for (int g = 0; g < NG; g++)
            __builtin_amdgcn_global_load_lds((const void *)(v + 64 * g), (lds_void *)(sv + (g * NC * KB + i) * 1024), 16, 0, 0);
    }
    int32_t d[KB];
    int32_t dmin = INT32_MAX, dmax = INT32_MIN;
#pragma unroll
    for (int j = 0; j < KB; j++) {
        int32_t x = 0;
        if (64 * j < keys) {
#pragma unroll
            for (int t = 0; t < QT; t++) {
                x = __builtin_amdgcn_sdot4(qv[4 * t], kk[j][t][0], x, false);
                x = __builtin_amdgcn_sdot4(qv[4 * t + 1], kk[j][t][1], x, false);
                x = __builtin_amdgcn_sdot4(qv[4 * t + 2], kk[j][t][2], x, false);
                x = __builtin_amdgcn_sdot4(qv[4 * t + 3], kk[j][t][3], x, false);
            }
        }
        d[j] = x;
        if (lane + 64 * j < keys) {
            dmin = x < dmin ? x : dmin;
            dmax = x > dmax ? x : dmax;
        }
    }
    wave_min_max(dmin, dmax);
    // the row max of the scores: the score is monotone in the dot (keys >= 1)
    const int64_t s0 = attn_score<NOCLAMP>(a, dmin), s1 = attn_score<NOCLAMP>(a, dmax);
    const int64_t M = s0 > s1 ? s0 : s1;
    const int64_t last = a.exp_len - 1;
    uint32_t e[KB];
    uint64_t sum = 0;
#pragma unroll
    for (int j = 0; j < KB; j++) {
        e[j] = 0;
        if (lane + 64 * j < keys) {
            const int64_t dd = M - attn_score<NOCLAMP>(a, d[j]);
            e[j] = (uint32_t)a.exp_table[dd < last ? dd : last];
            sum += e[j];
        }
    }
    sum = wave_sum_dpp(sum);
    const double R = ldexp(1.0 / (double)sum, a.softmax_p);
    const double sp = softmax_sp(sum, a.softmax_p);
    wait_vmcnt<0>();  // this wave's V rows landed in its LDS region
    v4i acc[NG][NC];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[g][c] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < KB; j++) {
        if (64 * j >= keys) break;
        // p <= 2^P <= 2^30; 0 for keys past the row (e = 0)
        const v4i pf = decode_pv_digits(mem, softmax_p_of(e[j], R, sp), lane);
#pragma unroll
        for (int g = 0; g < NG; g++) decode_pv_block<NC>(sv + (g * KB + j) * 64 * RB, pf, lane, acc[g]);
    }
    const double mo = a.out_s > 95 ? 0.0 : ldexp((double)a.out_m, -a.out_s);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        decode_pv_store<NC>(mem, lane, acc[g]);
        asm volatile("" ::: "memory");  // (the wave's LDS operations stay in order)
        if (lane < RB)
            *attn_out(a, r, h * HD + 64 * g + lane) =
                (int8_t)attn_out_byte(decode_pv_sum(mem, lane), mo, a.out_m, a.out_s);
        asm volatile("" ::: "memory");
    }
}

// The most keys k_attend_decode_wave takes: eight blocks of 64 or 64 VGPRs of K, whichever is less. Past
// it a workgroup per row-head, up to 1,024 keys.
static int decode_wave_keys(int hd) { return hd == 128 ? 128 : hd == 64 ? 256 : 512; }

template <bool NOCLAMP, int HD>
static hipError_t launch_decode(const AttnArgs &a, int n_rows, int kmax, hipStream_t stream) {
    const int n_rh = n_rows * a.n_head;
    if (kmax > decode_wave_keys(HD)) {
        if constexpr (HD == 64) launch_k(k_attend_decode64<NOCLAMP>, dim3(n_rh), dim3(256), 0, stream, a, kmax);
        else launch_k((k_attend_decode_wg<NOCLAMP, HD>), dim3(n_rh), dim3(HD > 64 ? 512 : 256), 0, stream, a, kmax);
        return hipGetLastError();
    }
    auto run = [&](auto kernel, int kb) {
        const size_t lds = (size_t)4 * (kb * 64 * HD + 1024);
        const hipError_t e = lds > 65536 ? allow_dynamic_lds((const void *)kernel, lds) : hipSuccess;
        if (e != hipSuccess) return e;
        launch_k(kernel, dim3((n_rh + 3) / 4), dim3(256), lds, stream, a, n_rh, kmax);
        return hipGetLastError();
    };
    const int kb = (kmax + 63) / 64;
    if (kb <= 1) return run(k_attend_decode_wave<NOCLAMP, 1, HD>, 1);
    if (kb == 2) return run(k_attend_decode_wave<NOCLAMP, 2, HD>, 2);
    if constexpr (HD <= 64) {
        if (kb == 3) return run(k_attend_decode_wave<NOCLAMP, 3, HD>, 3);
        if (kb == 4) return run(k_attend_decode_wave<NOCLAMP, 4, HD>, 4);
        if constexpr (HD < 64) return run(k_attend_decode_wave<NOCLAMP, 8, HD>, 8);
    }
    return hipErrorInvalidValue;
}

template <bool NOCLAMP>
static hipError_t launch_decode_hd(const AttnArgs &a, int n_rows, int kmax, hipStream_t stream) {
    switch (a.hd) {
    case 16: return launch_decode<NOCLAMP, 16>(a, n_rows, kmax, stream);
    case 32: return launch_decode<NOCLAMP, 32>(a, n_rows, kmax, stream);
    case 64: return launch_decode<NOCLAMP, 64>(a, n_rows, kmax, stream);
    case 128: return launch_decode<NOCLAMP, 128>(a, n_rows, kmax, stream);
    default: return hipErrorInvalidValue;
    }
}

SplitPlan attend_split_plan(int n_rows, int n_head, int max_keys, int mean_keys) {
    // about 4096 waves over (row, head, chunk), chunks of a multiple of 64 keys
    SplitPlan p;
    const long long rh = (long long)n_rows * n_head;
    const int blocks64 = (max_keys + 63) / 64;
    int want = (int)((4096 + rh - 1) / (rh > 0 ? rh : 1));
    want = want < 1 ? 1 : (want > blocks64 ? blocks64 : want);
    p.chunk_keys = 64 * ((blocks64 + want - 1) / want);
    // One wave walks a chunk from end to end, so a chunk holds at most 64 blocks of keys, however many
    // row-heads there are (the i32 sums of k_split_pv's digit planes would hold 32 times as many).
    p.chunk_keys = p.chunk_keys > 4096 ? 4096 : p.chunk_keys;
    p.chunks = (max_keys + p.chunk_keys - 1) / p.chunk_keys;
    p.max_keys = max_keys;
    p.row_heads = rh;
    p.mean_keys = mean_keys;
    return p;
}

// The one-launch kernels. Past 128 keys a row-head of head_dim 128 takes a workgroup of 512 threads that
// fills a CU for 4 us and more, however few of those keys it has: 3,072 row-heads of 16 to 32 keys in
// caches of 256 took 48.7 us, 16,384 of them 259 (the four split launches 19.8 and 55.6), and the passes
// of a prefill, whose rows hold half of the longest one's keys in the mean, 577 us for 32,768
// row-heads of up to 256 (176 split). So it is for few row-heads (768 at 300 keys 20.2 us, split 29.3;
// 800 at 500 keys 29.5 and 32.2), and for more of them where the caller knows that most hold many
// keys (4,096 at 900: 188 and 208; 16,384 at 512 keys: 475 and 456).
constexpr long long DECODE_WG128_MOST = 1024;
constexpr int DECODE_WG128_KEYS = 640;

bool attend_split_one_launch(int hd, int ctx_cap, const SplitPlan &p) {
    const int kmax = p.max_keys < ctx_cap ? p.max_keys : ctx_cap;
    if (kmax < 1 || kmax > 1024) return false;
    if (hd == 128)
        return kmax <= decode_wave_keys(hd) || p.row_heads <= DECODE_WG128_MOST || p.mean_keys >= DECODE_WG128_KEYS;
    return hd == 16 || hd == 32 || hd == 64;
}

size_t attend_split_partials(const AttnArgs &a, int n_rows, const SplitPlan &p) {
    auto al = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t rh = (size_t)n_rows * a.n_head;
    return al(rh * a.ctx_cap * 4) + 2 * al(rh * p.chunks * 8) + al(rh * p.chunks * a.hd * 8);
}

size_t attend_split_bytes(const AttnArgs &a, int n_rows, const SplitPlan &p) {
    return attend_split_one_launch(a.hd, a.ctx_cap, p) ? 0 : attend_split_partials(a, n_rows, p);
}

template <int HD>
static void launch_split(const AttnArgs &a, int n_rows, const SplitPlan &p, void *scratch, hipStream_t stream) {
    const dim3 grid(n_rows * a.n_head, p.chunks);
    launch_k(k_split_dots<HD>, grid, dim3(64), 0, stream, a, n_rows, p, scratch);
    if (attn_noclamp(a)) {
        launch_k(k_split_sum<true>, grid, dim3(64), 0, stream, a, n_rows, p, scratch);
        launch_k((k_split_pv<true, HD>), grid, dim3(64), 0, stream, a, n_rows, p, scratch);
    } else {
        launch_k(k_split_sum<false>, grid, dim3(64), 0, stream, a, n_rows, p, scratch);
        launch_k((k_split_pv<false, HD>), grid, dim3(64), 0, stream, a, n_rows, p, scratch);
    }
}

hipError_t launch_attend_split(const AttnArgs &a, int n_rows, const SplitPlan &p, void *scratch,
                               hipStream_t stream) {
    if (n_rows <= 0) return hipSuccess;
    if (!attend_split_ok(a.hd) || p.chunk_keys % 64 != 0 || p.chunk_keys > 4096) return hipErrorInvalidValue;
    const int kmax = p.max_keys < a.ctx_cap ? p.max_keys : a.ctx_cap;
    // one launch and no scratch up to 1,024 keys; of it a wave per (row, head) up to 256 keys at
    // head_dim 64 (768 row-heads at 128 keys 9.6 us a launch where a workgroup per row-head took 10.7, 4,096
    // row-heads of a GPT-2-medium decode pass 37 against 42, both with the sums p v on 24-bit multiplies;
    // the wave form now takes 5.8 us for the first)
    if (attend_split_one_launch(a.hd, a.ctx_cap, p))
        return attn_noclamp(a) ? launch_decode_hd<true>(a, n_rows, kmax, stream)
                               : launch_decode_hd<false>(a, n_rows, kmax, stream);
    switch (a.hd) {
    case 16: launch_split<16>(a, n_rows, p, scratch, stream); break;
    case 32: launch_split<32>(a, n_rows, p, scratch, stream); break;
    case 64: launch_split<64>(a, n_rows, p, scratch, stream); break;
    case 128: launch_split<128>(a, n_rows, p, scratch, stream); break;
    default: launch_split<256>(a, n_rows, p, scratch, stream); break;
    }
    launch_k(k_split_out, dim3(n_rows * a.n_head), dim3(a.hd), 0, stream, a, n_rows, p, scratch);
    return hipGetLastError();
}

// =============================================================================================
// Prefill attention on MFMA (head_dim 64). One workgroup = one group of <= 64 rows x one head;
// wave w owns rows 16w .. 16w + 15, lane l the row 16w + l % 16. QK^T comes from
// v_mfma_i32_16x16x64_i8 with K as the first operand (exact i32), for a super-block of up to
// AT_SB key blocks of 64 held in registers: lane l holds the dots of its row with the keys
// 16t + 4(l / 16) + e (t, e < 4) of each block. With <= 256 keys the product runs once, else
// once per pass. Pass 1 takes the row max (from the extreme dots: the score is monotone in the
// dot), pass 2 turns the dots into the table entries attn_exp[min(M - s, last)] in place and
// sums them, pass 3 forms p = floor(e 2^P / S) and sum_j p_j v_j. The PV product splits p into
// four balanced signed base-256 digits (crates/hardshell/src/gpt2/attention.rs:36-46): for
// p < 2^31 the bytes of (p + 0x80808080) ^ 0x80808080 are those digits. Each plane is an exact
// i8 product (|sum_j d_j v_j| <= 2^16 128 127 < 2^31) with V^T first: the key order inside a
// block is permuted (key 16t + 4g + e at byte 16g + 4t + e) so that the digits a lane needs as
// the second operand are the ones it already holds (4 x 4 byte transposes, no LDS round trip),
// and V^T enters LDS in the same order.
// =============================================================================================

constexpr int AT_ST = 80;               // LDS row stride in bytes (64 + 16)
constexpr int AT_SB = 4;                // key blocks of 64 held in registers
constexpr int ATTN_LDS_TABLE = 16384;   // attn_exp entries kept in LDS (64 KiB)


// NOCLAMP: score_s >= 13, so |dot m| < 2^53 keeps every score within +-2^40 (the clamp is a no-op).
// LDS_TABLE: attn_exp (<= ATTN_LDS_TABLE entries) is read from a copy in LDS.
// MULTI: some group has more than AT_SB 64 keys (Q K^T is recomputed per pass); without it the
// kernel holds one super-block and has no recompute path.
template <bool NOCLAMP, bool LDS_TABLE, bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attend_mfma(AttnArgs a, const AttnGroup *groups) {
    __shared__ __attribute__((aligned(16))) int8_t sQ[64 * AT_ST];
    // the K rows of a super-block (AT_SB x 64 keys), later the V^T of its blocks (64 channels each)
    __shared__ __attribute__((aligned(1024))) int8_t sKV[AT_SB * 64 * AT_ST];
    // without MULTI: the V rows of the (single) super-block, as loaded
    __shared__ __attribute__((aligned(1024))) int8_t sV[MULTI ? 16 : AT_SB * 64 * 64];
    extern __shared__ __attribute__((aligned(1024))) int32_t s_exp[];  // attn_exp when LDS_TABLE
    const AttnGroup G = groups[blockIdx.x];
    const int h = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int ql = lane & 15, qg = lane >> 4;
    int nk = G.pos0 + G.count;  // keys 0 .. nk - 1, never past the cache
    nk = nk > a.ctx_cap ? a.ctx_cap : nk;
    const size_t base = ((size_t)G.slot * a.n_head + h) * a.ctx_cap * 64;
    const int last = a.exp_len - 1;
    // Dense LDS rows of 64 bytes with 16-byte chunk c of row r at slot 4 r + (c ^ sw(r % 16)), so
    // the fragment reads of 16 consecutive rows hit distinct bank groups.
    auto sw = [](int r) { return ((r >> 1) ^ (r >> 3)) & 3; };
    if (!MULTI) {
        // every K and V row of the group's blocks, and the table, straight into LDS before any
        // other work (global_load_lds: lane l's 16 bytes land at the wave's base + 16 l). Rows
        // past the cache read its last row (their keys are masked).
        const int r = 16 * w + (lane >> 2), c = (lane & 3) ^ sw(r & 15);
        const int nkb0 = (nk + 63) / 64;
#pragma unroll
        for (int b = 0; b < AT_SB; b++) {
            if (b >= nkb0) break;
            int key = b * 64 + r;
            key = key < a.ctx_cap ? key : a.ctx_cap - 1;
            const size_t off = base + (size_t)key * 64 + 16 * c;
            __builtin_amdgcn_global_load_lds((const void *)(a.kc + off), (lds_void *)(sKV + (b * 64 + 16 * w) * 64), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const void *)(a.vc + off), (lds_void *)(sV + (b * 64 + 16 * w) * 64), 16, 0, 0);
        }
        if (LDS_TABLE)  // whole 1 KiB chunks (the table is readable to a multiple of 256 entries)
            for (int ch = w; ch < (a.exp_len + 255) / 256; ch += 4)
                __builtin_amdgcn_global_load_lds((const void *)(a.exp_table + ch * 256 + 4 * lane),
                                                 (lds_void *)(s_exp + ch * 256), 16, 0, 0);
    } else if (LDS_TABLE) {  // 16-byte copies when the table is 16-byte aligned (a device allocation)
        const bool vec = ((uintptr_t)a.exp_table & 15) == 0;
        const int n4 = vec ? a.exp_len / 4 : 0;
        for (int i = tid; i < n4; i += 256) ((v4i *)s_exp)[i] = ((const v4i *)a.exp_table)[i];
        for (int i = 4 * n4 + tid; i < a.exp_len; i += 256) s_exp[i] = a.exp_table[i];
    }
    const int32_t *etab = LDS_TABLE ? (const int32_t *)s_exp : a.exp_table;
    {
        const int r = tid >> 2, c = (tid & 3) * 16;
        v4i v = {0, 0, 0, 0};
        if (r < G.count) v = *(const v4i *)(a.q + (size_t)(G.first + r) * a.ldq + h * 64 + c);
        *(v4i *)&sQ[r * AT_ST + c] = v;
    }
    if (!MULTI) wait_vmcnt<0>();  // this wave's direct loads landed (the barrier shows them to all)
    __syncthreads();
    const v4i qf = *(const v4i *)&sQ[(16 * w + ql) * AT_ST + qg * 16];
    const int myrow = 16 * w + ql, mypos = G.pos0 + myrow;  // this lane's row and its position
    const int nkb = (nk + 63) / 64, nsb = MULTI ? (nkb + AT_SB - 1) / AT_SB : 1;
    // score = clamp(rescale(dot, m, s), +-2^40): |dot| <= hd 2^14 <= 2^22, so |dot m| < 2^53 and
    // one multiply-add and an arithmetic shift are exact (a shift of 63 or more gives 0).
    const int s_eff = a.score_s < 63 ? a.score_s : 63;
    const int64_t s_half = s_eff ? (int64_t)1 << (s_eff - 1) : 0;
    auto score = [&](int32_t dot) -> int64_t {
        const int64_t r = ((int64_t)dot * a.score_m + s_half) >> s_eff;
        return NOCLAMP ? r : clamp64(r, -SCORE_LIMIT, SCORE_LIMIT);
    };
    auto key_of = [&](int sb, int b, int t, int e) { return (sb * AT_SB + b) * 64 + 16 * t + 4 * qg + e; };
    v4i S[AT_SB][4];  // S[b][t][e]: the dot (then the table entry) of the row with key_of(sb, b, t, e)
    // this thread's 16 bytes of key block kb: key kb * 64 + tid / 4, bytes 16 (tid % 4)
    auto k_load = [&](int kb) {
        const int key = kb * 64 + (tid >> 2), c = (tid & 3) * 16;
        v4i v = {0, 0, 0, 0};
        if (key < nk) v = *(const v4i *)(a.kc + base + (size_t)key * 64 + c);
        return v;
    };
    // this thread's 4 keys x 4 channels of value block kb (one word per key): keys kb * 64 +
    // 4 (tid / 16) .. +4, channels 4 (tid % 16) .. +4
    auto vt_load = [&](int kb) {
        const int k0 = kb * 64 + 4 * (tid >> 4), c = 4 * (tid & 15);
        v4i v = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (k0 + i < nk) v[i] = *(const int32_t *)(a.vc + base + (size_t)(k0 + i) * 64 + c);
        return v;
    };
    auto qk_super = [&](int sb) {
        const int nb = nkb - sb * AT_SB < AT_SB ? nkb - sb * AT_SB : AT_SB;
        if (!MULTI) {  // the K rows are in LDS (dense, swizzled)
#pragma unroll
            for (int b = 0; b < AT_SB; b++)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    if (b < nb) {
                        const int r = t * 16 + ql;
                        const v4i kf = *(const v4i *)&sKV[(4 * (b * 64 + r) + (qg ^ sw(r & 15))) * 16];
                        S[b][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qf, v4i{0, 0, 0, 0}, 0, 0, 0);
                    } else {
                        S[b][t] = v4i{0, 0, 0, 0};
                    }
                }
            __syncthreads();  // the K rows are read: sKV may take V^T
            return;
        }
        v4i kreg[AT_SB];  // every key block of the super-block in flight at once
#pragma unroll
        for (int b = 0; b < AT_SB; b++)
            if (b < nb) kreg[b] = k_load(sb * AT_SB + b);
#pragma unroll
        for (int b = 0; b < AT_SB; b++)
            if (b < nb) *(v4i *)&sKV[(b * 64 + (tid >> 2)) * AT_ST + (tid & 3) * 16] = kreg[b];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < AT_SB; b++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (b < nb) {
                    const v4i kf = *(const v4i *)&sKV[(b * 64 + t * 16 + ql) * AT_ST + qg * 16];
                    S[b][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qf, v4i{0, 0, 0, 0}, 0, 0, 0);
                } else {
                    S[b][t] = v4i{0, 0, 0, 0};
                }
            }
        __syncthreads();  // the K rows are read: sKV may take the next super-block or V^T
    };

    // pass 1: the row max, from the largest and the smallest dot
    int32_t dmax = INT32_MIN, dmin = INT32_MAX;
    for (int sb = 0; sb < nsb; sb++) {
        qk_super(sb);
#pragma unroll
        for (int b = 0; b < AT_SB; b++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int key = key_of(sb, b, t, e);
                    const bool ok = key <= mypos && key < nk;
                    const int32_t hiv = ok ? S[b][t][e] : INT32_MIN, lov = ok ? S[b][t][e] : INT32_MAX;
                    dmax = hiv > dmax ? hiv : dmax;
                    dmin = lov < dmin ? lov : dmin;
                }
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {  // the 4 lanes of this row
        const int32_t u = __shfl_xor(dmax, o, 64), v = __shfl_xor(dmin, o, 64);
        dmax = u > dmax ? u : dmax;
        dmin = v < dmin ? v : dmin;
    }
    const int64_t mx = score(dmax) > score(dmin) ? score(dmax) : score(dmin);
    // the dots of super-block sb -> the table entries attn_exp[min(M - s, last)] (>= 0), 0 for a
    // masked key (it adds nothing to S and gets p = 0). Every index is in range and every lookup
    // is issued (the empty asm keeps each one out of a per-key branch), all before the masking.
    auto to_weight = [&](int sb) {
#pragma unroll
        for (int b = 0; b < AT_SB; b++) {  // one block of 64 keys (16 lookups) at a time
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int64_t dd = mx - score(S[b][t][e]);
                    S[b][t][e] = dd < 0 ? 0 : (dd < last ? (int)dd : last);
                }
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    S[b][t][e] = etab[S[b][t][e]];
                }
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int key = key_of(sb, b, t, e);
                    S[b][t][e] = (key <= mypos && key < nk) ? S[b][t][e] : 0;
                }
        }
    };
    // pass 2: the sum of the table entries
    uint64_t sum = 0;
    for (int sb = 0; sb < nsb; sb++) {
        if (MULTI && nsb > 1) qk_super(sb);
        to_weight(sb);
#pragma unroll
        for (int b = 0; b < AT_SB; b++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum += (uint32_t)S[b][t][e];
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    // p = floor(e 2^P / S) (softmax_p_of)
    const double R = ldexp(1.0 / (double)sum, a.softmax_p);
    const double sp = softmax_sp(sum, a.softmax_p);
    // pass 3: p, its packed digits, and the digit-plane PV products
    v4i acc[4][4];  // [digit plane][channel tile]: channel 16 c + 4 (l / 16) + e of row l % 16
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[k][c] = v4i{0, 0, 0, 0};
    for (int sb = 0; sb < nsb; sb++) {
        if (MULTI && nsb > 1) {
            qk_super(sb);
            to_weight(sb);
        }
        const int nb = nkb - sb * AT_SB < AT_SB ? nkb - sb * AT_SB : AT_SB;
        {  // V^T of the super-block's blocks into sKV, keys in the operand order
            v4i vreg[AT_SB];
            const int kg = tid >> 4, cg = tid & 15;  // keys 4 kg .. +4, channels 4 cg .. +4
#pragma unroll
            for (int b = 0; b < AT_SB; b++) {
                if (b >= nb) continue;
                if (MULTI) {
                    vreg[b] = vt_load(sb * AT_SB + b);
                } else {  // from the dense V rows (a key past nk has p = 0)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int kk = 4 * kg + i;
                        vreg[b][i] = *(const int32_t *)&sV[(4 * (b * 64 + kk) + ((cg >> 2) ^ sw(kk & 15))) * 16 + 4 * (cg & 3)];
                    }
                }
            }
            const int pos0 = 16 * (kg & 3) + 4 * (kg >> 2);
#pragma unroll
            for (int b = 0; b < AT_SB; b++) {
                if (b >= nb) continue;
                uint32_t tw[4];
                byte_transpose((uint32_t)vreg[b][0], (uint32_t)vreg[b][1], (uint32_t)vreg[b][2], (uint32_t)vreg[b][3], tw);
#pragma unroll
                for (int j = 0; j < 4; j++) *(uint32_t *)&sKV[(b * 64 + 4 * cg + j) * AT_ST + pos0] = tw[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < AT_SB; b++) {
            if (b >= nb) break;
            uint32_t dg[4][4];
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) dg[t][e] = softmax_p_of((uint32_t)S[b][t][e], R, sp);
            v4i pf[4];  // [digit plane]: word t holds the digits of keys 16 t + 4 (l / 16) + e
#pragma unroll
            for (int t = 0; t < 4; t++) {
                uint32_t o[4];
                byte_transpose((dg[t][0] + 0x80808080u) ^ 0x80808080u, (dg[t][1] + 0x80808080u) ^ 0x80808080u,
                               (dg[t][2] + 0x80808080u) ^ 0x80808080u, (dg[t][3] + 0x80808080u) ^ 0x80808080u, o);
#pragma unroll
                for (int k = 0; k < 4; k++) pf[k][t] = (int32_t)o[k];
            }
            v4i vf[4];
#pragma unroll
            for (int c = 0; c < 4; c++) vf[c] = *(const v4i *)&sKV[(b * 64 + 16 * c + ql) * AT_ST + 16 * qg];
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    acc[k][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf[c], pf[k], acc[k][c], 0, 0, 0);
        }
        __syncthreads();  // V^T is read: sKV may take the next super-block
    }
    if (myrow < G.count) {
        int8_t *o = attn_out(a, G.first + myrow, h * 64);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            uint32_t packed = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int64_t v = (int64_t)acc[0][c][e] + ((int64_t)acc[1][c][e] << 8) +
                                  ((int64_t)acc[2][c][e] << 16) + ((int64_t)acc[3][c][e] << 24);
                packed |= (uint32_t)(uint8_t)(int8_t)clamp128(rescale_full(v, a.out_m, a.out_s), -127, 127) << (8 * e);
            }
            *(uint32_t *)(o + 16 * c + 4 * qg) = packed;
        }
    }
}

// =============================================================================================
// Prefill attention of short windows: head_dim 64, at most 8 key blocks of 64 per group, attn_exp
// in LDS, score shift 22 .. 63 and P <= 30. The algorithm and the layouts are k_attend_mfma's;
// the per-score work is smaller:
//  - |dot| <= 64 2^14 and |m| <= 2^31, so |score| <= 2^29 + 1 for s >= 22: the distance M - s is
//    an i32 and its clamp to [0, last] one med3;
//  - blocks past the group's keys are skipped, and the causal mask is applied only to the
//    blocks that some row of the wave does not fully see (a wave-uniform test per block);
//  - p = floor(e 2^P / S) is the nearest integer of e R (one fused multiply-add) less one where
//    e 2^P < n S (softmax_p_of: exact, no branch), and tiles of 16 keys that no row of the wave
//    sees get p = 0 without it;
//  - the output rescale floor(v m 2^-s + 1/2), clamped to +-127, is one fused multiply-add in
//    double precision: v = sum of the four digit-plane products is an exact double (|v| <= 2^30
//    128 < 2^38 and every partial sum stays below 2^47), so y = v m 2^-s + 1/2 carries one
//    rounding (relative 2^-53); when |y| >= 256 the clamp decides, when y lies at least 2^-30
//    from an integer floor(y) is exact, else the element takes the i128 rule.
//  - the Q fragment is read straight from global memory (each lane's 16 bytes of its row).
// =============================================================================================
// NB: key blocks of 64 (4: three workgroups per CU with a 32 KiB table; 8: two).
// Persistent: the grid holds the resident workgroups (at most n_tasks), and workgroup i takes
// the tasks (group, head), task = group n_head + head, of rounds r = 0, 1, .. in snake order:
// task r P + i for even r and r P + P - 1 - i for odd r (P workgroups). The host orders the
// groups by key count, largest first, so the rounds pair long tasks with short ones. The table
// is copied once per workgroup; the next task's group loads under the current task's softmax,
// its K rows as soon as every wave has read the current V rows (under the output rescale).
template <int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB <= 4 ? 3 : 2))) void k_attend_short(AttnArgs a, const AttnGroup *groups, int n_tasks) {
    // the K rows, then the V rows (as loaded)
    __shared__ __attribute__((aligned(1024))) int8_t sKV[NB * 64 * 64];
    extern __shared__ __attribute__((aligned(1024))) int32_t s_exp[];  // attn_exp
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the entries up to the zero tail (exp_last) or the whole table
    const int last = a.exp_last > 0 ? a.exp_last : a.exp_len - 1;
    const int P = gridDim.x, wg = blockIdx.x;
    auto task_at = [&](int r) { return r * P + ((r & 1) ? P - 1 - wg : wg); };
    auto sw = [](int r) { return ((r >> 1) ^ (r >> 3)) & 3; };
    auto key_blocks = [&](const AttnGroup &g) {
        const int nk = g.pos0 + g.count < a.ctx_cap ? g.pos0 + g.count : a.ctx_cap;
        return (nk + 63) / 64;  // 1 .. NB (checked by the launcher)
    };
    // the K (then V) rows of the group's blocks straight into LDS (dense rows, 16-byte chunk c of
    // row r at slot 4 r + (c ^ sw(r % 16))); rows past the cache read its last row (their keys
    // are masked)
    auto rows_to_lds = [&](const int8_t *cache, size_t base_, int nkb_) {
        const int ln = opaque_vgpr(lane);
        const int r = 16 * w + (ln >> 2), c = (ln & 3) ^ sw(r & 15);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b >= nkb_) break;
            int key = b * 64 + r;
            key = key < a.ctx_cap ? key : a.ctx_cap - 1;
            const size_t off = base_ + (size_t)key * 64 + 16 * c;
            __builtin_amdgcn_global_load_lds((const void *)(cache + off), (lds_void *)(sKV + (b * 64 + 16 * w) * 64), 16, 0, 0);
        }
    };
    auto q_frag = [&](const AttnGroup &g, int hh) -> v4i {  // this lane's row is 16 w + ql
        const int ln = opaque_vgpr(lane), row = 16 * w + (ln & 15);
        if (row < g.count) return *(const v4i *)(a.q + (size_t)(g.first + row) * a.ldq + hh * 64 + 16 * (ln >> 4));
        return v4i{0, 0, 0, 0};
    };
    int t = task_at(0);  // below n_tasks: the launcher takes P <= n_tasks
    AttnGroup G = groups[t / a.n_head];
    int h = t % a.n_head;
    rows_to_lds(a.kc, ((size_t)G.slot * a.n_head + h) * a.ctx_cap * 64, key_blocks(G));
    for (int ch = w; ch < (last + 256) / 256; ch += 4)  // whole 1 KiB chunks of entries 0 .. last
        __builtin_amdgcn_global_load_lds((const void *)(a.exp_table + ch * 256 + 4 * lane),
                                         (lds_void *)(s_exp + ch * 256), 16, 0, 0);
    v4i qf = q_frag(G, h);
    for (int round = 0;; round++) {
    // the lane's indexes, recomputed each round from an opaque copy of the lane: the compiler
    // then derives the LDS addresses at their use instead of keeping them in registers across
    // the loop
    const int lane_r = opaque_vgpr(lane);
    const int ql = lane_r & 15, qg = lane_r >> 4;
    const int myrow = 16 * w + ql;
    const int nk = G.pos0 + G.count < a.ctx_cap ? G.pos0 + G.count : a.ctx_cap;
    const int nkb = key_blocks(G);
    const size_t base = ((size_t)G.slot * a.n_head + h) * a.ctx_cap * 64;
    const int mypos = G.pos0 + myrow;  // this lane's position
    wait_vmcnt<0>();  // this wave's direct loads landed (the barrier shows them to all)
    __syncthreads();
    // S[b][t][e]: the dot (then the table entry) of this lane's row with key 64 b + 16 t + 4 qg + e
    v4i S[NB][4];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (b < nkb) {
                const int r = t * 16 + ql;
                const v4i kf = *(const v4i *)&sKV[(4 * (b * 64 + r) + (qg ^ sw(r & 15))) * 16];
                S[b][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qf, v4i{0, 0, 0, 0}, 0, 0, 0);
            } else {
                S[b][t] = v4i{0, 0, 0, 0};
            }
        }
    __syncthreads();  // every K row is read: the V rows load in their place during passes 1 and 2
    rows_to_lds(a.vc, base, nkb);
    // the next task's group, loading under passes 1 .. 3
    const int tn = task_at(round + 1);
    const bool more = tn < n_tasks;  // uniform
    AttnGroup Gn = G;
    if (more) Gn = groups[tn / a.n_head];
    // key 64 b + 16 t + 4 qg + e is visible to this lane's row iff 16 t + e <= lim - 64 b - 4 qg;
    // block b is visible to every row of the wave iff 64 b + 63 <= wlim, and its keys
    // 64 b + 16 t .. +15 to none iff 64 b + 16 t > wmax (both uniform): such a tile has e = 0
    // and p = 0 for every row, and the passes skip it
    const int lim = mypos < nk - 1 ? mypos : nk - 1;
    const int wlim = G.pos0 + 16 * w < nk - 1 ? G.pos0 + 16 * w : nk - 1;
    const int wmax = G.pos0 + 16 * w + 15 < nk - 1 ? G.pos0 + 16 * w + 15 : nk - 1;
    // pass 1: the row max, from the largest and the smallest visible dot
    int32_t dmax = INT32_MIN, dmin = INT32_MAX;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        if (b >= nkb) break;
        if (64 * b + 63 <= wlim) {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    dmax = S[b][t][e] > dmax ? S[b][t][e] : dmax;
                    dmin = S[b][t][e] < dmin ? S[b][t][e] : dmin;
                }
        } else {
            const int L = lim - 64 * b - 4 * qg;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (64 * b + 16 * t > wmax) continue;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const bool ok = 16 * t + e <= L;
                    const int32_t hiv = ok ? S[b][t][e] : INT32_MIN, lov = ok ? S[b][t][e] : INT32_MAX;
                    dmax = hiv > dmax ? hiv : dmax;
                    dmin = lov < dmin ? lov : dmin;
                }
            }
        }
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {  // the 4 lanes of this row
        const int32_t u = __shfl_xor(dmax, o, 64), v = __shfl_xor(dmin, o, 64);
        dmax = u > dmax ? u : dmax;
        dmin = v < dmin ? v : dmin;
    }
    // score = (dot m + 2^(s-1)) >> s (exact in i64: |dot m| <= 2^51), an i32 for s >= 22
    const int s_eff = a.score_s < 63 ? a.score_s : 63;
    const int64_t s_half = (int64_t)1 << (s_eff - 1);
    auto score = [&](int32_t dot) -> int32_t { return (int32_t)(((int64_t)dot * a.score_m + s_half) >> s_eff); };
    const int32_t mx = score(dmax) > score(dmin) ? score(dmax) : score(dmin);
    // pass 2: the table entries attn_exp[min(M - s, last)] (0 for a masked key) and their sum
    uint64_t sum = 0;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        if (b >= nkb) break;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) S[b][t][e] = clamp0_uniform(mx - score(S[b][t][e]), last);
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) S[b][t][e] = s_exp[S[b][t][e]];
        if (64 * b + 63 > wlim) {
            const int L = lim - 64 * b - 4 * qg;
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) S[b][t][e] = 16 * t + e <= L ? S[b][t][e] : 0;
        }
#pragma unroll
        for (int t = 0; t < 4; t++)  // entries are < 2^31: a pair sums in u32
#pragma unroll
            for (int e = 0; e < 4; e += 2) sum += (uint32_t)S[b][t][e] + (uint32_t)S[b][t][e + 1];
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    const double R = ldexp(1.0 / (double)sum, a.softmax_p);
    const double sp = softmax_sp(sum, a.softmax_p);
    // The V^T operand comes straight from the V rows: ds_read_b64_tr_b8 gives lane 8 h + j of each
    // 16-lane group byte j of the 8-byte pieces that lanes h, h + 2, .., h + 14 address. Lane i of
    // group qg addresses key 16 t + 4 qg + e (t = 2 r + i / 8, e = (i / 2) % 4 for read r) at
    // channels 16 c + 8 (i % 2) .. +8, so lane l receives channel 16 c + l % 16 of the keys of
    // operand bytes 8 r .. 8 r + 7 (byte 4 t + e holds key 16 t + 4 qg + e, as in the digits).
    const int tr_k = ql >> 1, tr_h = ql & 1;
    const int tr_key0 = 16 * (tr_k >> 2) + 4 * qg + (tr_k & 3);  // read 0; read 1 is 32 keys on
    auto vt_frag = [&](int b, int c) -> v4i {
        const int8_t *p0 = sKV + (4 * (b * 64 + tr_key0) + (c ^ sw(tr_key0 & 15))) * 16 + 8 * tr_h;
        const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)p0);
        const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)(p0 + 32 * 64));
        return v4i{r0[0], r0[1], r1[0], r1[1]};
    };
    wait_vmcnt<0>();  // this wave's V rows landed (the barrier shows them to all)
    __syncthreads();
    // pass 3: p + 0x80808080 (the packed digits), and the digit-plane PV products
    v4i acc[4][4];  // [digit plane][channel tile]: channel 16 c + 4 (l / 16) + e of row l % 16
#pragma unroll
    for (int b = 0; b < NB; b++) {
        if (b >= nkb) break;
        uint32_t dg[4][4];
        const bool part = 64 * b + 63 > wlim;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (part && 64 * b + 16 * t > wmax) {
#pragma unroll
                for (int e = 0; e < 4; e++) dg[t][e] = 0x80808080u;  // p = 0
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                dg[t][e] = softmax_p_of((uint32_t)S[b][t][e], R, sp) + 0x80808080u;
        }
        v4i pf[4];  // [digit plane]: word t holds the digits of keys 16 t + 4 (l / 16) + e
#pragma unroll
        for (int t = 0; t < 4; t++) {
            uint32_t o[4];
            byte_transpose(dg[t][0], dg[t][1], dg[t][2], dg[t][3], o);
#pragma unroll
            for (int k = 0; k < 4; k++) pf[k][t] = (int32_t)(o[k] ^ 0x80808080u);
        }
        v4i vf[4];
#pragma unroll
        for (int c = 0; c < 4; c++) vf[c] = vt_frag(b, c);
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int k = 0; k < 4; k++)  // block 0 (every task has it) starts the sums
                acc[k][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf[c], pf[k], b == 0 ? v4i{0, 0, 0, 0} : acc[k][c],
                                                                  0, 0, 0);
    }
    // Every wave has issued its reads of the V rows: after the barrier sKV takes the next task's
    // K rows, which load while this task's outputs are formed.
    const int out_count = G.count, out_first = G.first, out_h = h;
    if (more) {
        __syncthreads();
        G = Gn;
        h = tn % a.n_head;
        rows_to_lds(a.kc, ((size_t)G.slot * a.n_head + h) * a.ctx_cap * 64, key_blocks(G));
    }
    // Shifts 48..63 with at most 4 blocks (|plane| <= 2^22): the exact rescale in i64 from the two
    // pairwise plane sums (attn_out_planes: two multiply-adds and two shifts per output)
    if (NB <= 4 && a.out_s >= 48 && a.out_s <= 63 && myrow < out_count) {
        uint32_t packed[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            packed[c] = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int32_t hi = (int32_t)((uint32_t)acc[3][c][e] << 8) + acc[2][c][e];
                const int32_t lo = (int32_t)((uint32_t)acc[1][c][e] << 8) + acc[0][c][e];
                const int32_t r = attn_out_planes(hi, lo, a.out_m, (uint32_t)a.out_s);
                packed[c] |= (uint32_t)(uint8_t)(int8_t)r << (8 * e);
            }
        }
        int8_t *o = attn_out(a, out_first + myrow, out_h * 64);
#pragma unroll
        for (int c = 0; c < 4; c++) *(uint32_t *)(o + 16 * c + 4 * qg) = packed[c];
    } else if (myrow < out_count) {
        // rescale: s = 0 keeps v m, a shift above 95 gives 0
        const double mo = a.out_s > 95 ? 0.0 : ldexp((double)a.out_m, -a.out_s);
        uint32_t packed[4];
        bool ok = true;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            packed[c] = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                double v;
                if (NB <= 4) {  // |acc| <= 256 2^7 2^7 = 2^22 per plane: each pair of planes sums in i32
                    const int32_t hi = (int32_t)((uint32_t)acc[3][c][e] << 8) + acc[2][c][e];
                    const int32_t lo = (int32_t)((uint32_t)acc[1][c][e] << 8) + acc[0][c][e];
                    v = fma((double)hi, 65536.0, (double)lo);
                } else {  // |acc| <= 2^23: the planes in double precision (every partial sum exact)
                    v = (((double)acc[3][c][e] * 16777216.0 + (double)acc[2][c][e] * 65536.0) +
                         (double)acc[1][c][e] * 256.0) + (double)acc[0][c][e];
                }
                const double y = fma(v, mo, 0.5);
                const double f = __builtin_amdgcn_fract(y);
                ok &= fabs(y) >= 256.0 || fabs(f - 0.5) <= 0.5 - 0x1p-30;
                const int32_t r = (int32_t)fmin(fmax(y - f, -127.0), 127.0);
                packed[c] |= (uint32_t)(uint8_t)(int8_t)r << (8 * e);
            }
        }
        if (!ok) {  // some element lies too close to a rounding boundary: the i128 rule for all
#pragma unroll
            for (int c = 0; c < 4; c++) {
                packed[c] = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int64_t vi = (int64_t)acc[0][c][e] + ((int64_t)acc[1][c][e] << 8) +
                                       ((int64_t)acc[2][c][e] << 16) + ((int64_t)acc[3][c][e] << 24);
                    const int32_t r = (int32_t)clamp128(rescale_full(vi, a.out_m, a.out_s), -127, 127);
                    packed[c] |= (uint32_t)(uint8_t)(int8_t)r << (8 * e);
                }
            }
        }
        int8_t *o = attn_out(a, out_first + myrow, out_h * 64);
#pragma unroll
        for (int c = 0; c < 4; c++) *(uint32_t *)(o + 16 * c + 4 * qg) = packed[c];
    }
    if (!more) break;
    qf = q_frag(G, h);
    }
}

// =============================================================================================
// Prefill attention over any number of keys (head_dim 64, attn_exp in LDS, score shift 22 .. 63,
// P <= 30, at most 2^15 keys): windows of a whole context. The exact integer softmax needs the row
// max before the table entries and their sum before p, so the keys are walked three times, 128
// at a time: the extreme dots; the sum of the entries; p, its digits and the PV products. Each
// walk forms Q K^T again (4 MFMAs per 64 keys, less than keeping 1,024 scores a row would cost in
// registers: a wave stays within 168, three workgroups per CU). What bounds it is the VALU work
// of the scores, as in k_attend_short (per score: 2 instructions, then about 6 and a lookup,
// then about 13 and a lookup), so the loads must not add waits: the K and V rows of 128 keys are
// 8 KiB stages of one stream over a ring of three, two stages ahead of their use and across the
// end of a task into the next one's.
// Persistent, tasks in snake order, as k_attend_short.
// =============================================================================================
constexpr int AL_SB = 2;                  // key blocks of 64 per stage
constexpr int AL_STAGE = AL_SB * 64 * 64;  // bytes

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_attend_long(AttnArgs a, const AttnGroup *groups, int n_tasks) {
    __shared__ __attribute__((aligned(1024))) int8_t ring[3 * AL_STAGE];
    extern __shared__ __attribute__((aligned(1024))) int32_t s_exp[];  // attn_exp
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int last = a.exp_last > 0 ? a.exp_last : a.exp_len - 1;
    const int P = gridDim.x, wg = blockIdx.x;
    auto task_at = [&](int r) { return r * P + ((r & 1) ? P - 1 - wg : wg); };
    auto sw = [](int r) { return ((r >> 1) ^ (r >> 3)) & 3; };
    auto keys_of = [&](const AttnGroup &g) { return g.pos0 + g.count < a.ctx_cap ? g.pos0 + g.count : a.ctx_cap; };
    auto stages_of = [&](const AttnGroup &g) { return (keys_of(g) + 64 * AL_SB - 1) / (64 * AL_SB); };
    // Stage sb of K or V of a (group, head) into ring slot `slot`: dense rows, 16-byte chunk c of row r at
    // slot 4 r + (c ^ sw(r % 16)); rows past the cache read its last row (their keys are masked).
    // Each wave issues AL_SB loads of 1 KiB.
    auto stage = [&](const int8_t *cache, const AttnGroup &g, int hh, int sb, int slot) {
        const int r = 16 * w + (lane >> 2), c = (lane & 3) ^ sw(r & 15);
        const size_t base = ((size_t)g.slot * a.n_head + hh) * a.ctx_cap * 64;
#pragma unroll
        for (int b = 0; b < AL_SB; b++) {
            int key = (sb * AL_SB + b) * 64 + r;
            key = key < a.ctx_cap ? key : a.ctx_cap - 1;
            __builtin_amdgcn_global_load_lds((const void *)(cache + base + (size_t)key * 64 + 16 * c),
                                             (lds_void *)(ring + slot * AL_STAGE + (b * 64 + 16 * w) * 64), 16, 0, 0);
        }
    };
    // Load j of a task of n stages: K 0 .. n - 1 (walk 1), K n - 2 .. 0 (walk 2 starts on the stage that
    // walk 1 ends on), then V 0, K 1, V 1, K 2, .. V n - 1 (walk 3 starts on K 0): 4 n - 2 loads.
    auto issue_load = [&](const AttnGroup &g, int hh, int n, int j, int slot) {
        const int t = j - (2 * n - 1);
        if (t < 0) stage(a.kc, g, hh, j < n ? j : 2 * n - 2 - j, slot);
        else if (t & 1) stage(a.kc, g, hh, (t + 1) >> 1, slot);
        else stage(a.vc, g, hh, t >> 1, slot);
    };
    auto q_frag = [&](const AttnGroup &g, int hh) -> v4i {  // this lane's row is 16 w + lane % 16
        const int row = 16 * w + (lane & 15);
        if (row < g.count) return *(const v4i *)(a.q + (size_t)(g.first + row) * a.ldq + hh * 64 + 16 * (lane >> 4));
        return v4i{0, 0, 0, 0};
    };
    // score = (dot m + 2^(s-1)) >> s (exact in i64: |dot m| <= 2^51), an i32 for s >= 22
    const int s_eff = a.score_s < 63 ? a.score_s : 63;
    const int64_t s_half = (int64_t)1 << (s_eff - 1);
    auto score = [&](int32_t dot) -> int32_t { return (int32_t)(((int64_t)dot * a.score_m + s_half) >> s_eff); };

    int t = task_at(0);  // below n_tasks: the launcher takes P <= n_tasks
    AttnGroup G = groups[t / a.n_head], Gn = G;
    int h = t % a.n_head, hn = h, n = stages_of(G);
    bool more = false;
    int issued = 0, used = 0;  // loads of this task (issued: and of the next) issued and waited for
    int slot_in = 0, slot = 0;
    auto issue_next = [&]() {
        const int T = 4 * n - 2;
        if (issued < T) issue_load(G, h, n, issued, slot_in);
        else if (more) issue_load(Gn, hn, stages_of(Gn), issued - T, slot_in);
        else return;
        issued++;
        slot_in = slot_in == 2 ? 0 : slot_in + 1;
    };
    // The next load's stage: its loads landed (this wave's by the count, the others' by the barrier), and
    // every wave is done with the stage before it, whose slot takes the load after next.
    auto next_stage = [&]() -> const int8_t * {
        if (issued > used + 1) wait_vmcnt<AL_SB>();
        else wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int8_t *p = ring + slot * AL_STAGE;
        slot = slot == 2 ? 0 : slot + 1;
        used++;
        issue_next();
        return p;
    };
    for (int ch = w; ch < (last + 256) / 256; ch += 4)  // whole 1 KiB chunks of entries 0 .. last
        __builtin_amdgcn_global_load_lds((const void *)(a.exp_table + ch * 256 + 4 * lane),
                                         (lds_void *)(s_exp + ch * 256), 16, 0, 0);
    issue_next();
    issue_next();
    for (int round = 0;; round++) {
        const int ql = lane & 15, qg = lane >> 4;
        const int tn = task_at(round + 1);
        more = tn < n_tasks;  // uniform
        if (more) {
            Gn = groups[tn / a.n_head];
            hn = tn % a.n_head;
        }
        const v4i qf = q_frag(G, h);
        wait_vmcnt<0>();  // (stores of the task before may leave the count out of order: start from zero)
        const int nk = keys_of(G), nkb = (nk + 63) / 64;
        const int myrow = 16 * w + ql, mypos = G.pos0 + myrow;
        // key 64 b + 16 t + 4 qg + e is visible to this lane's row iff 16 t + e <= lim - 64 b - 4 qg;
        // block b is visible to every row of the wave iff 64 b + 63 <= wlim (uniform), and to none
        // iff 64 b > wmax
        const int lim = mypos < nk - 1 ? mypos : nk - 1;
        const int wlim = G.pos0 + 16 * w < nk - 1 ? G.pos0 + 16 * w : nk - 1;
        const int wmax = G.pos0 + 16 * w + 15 < nk - 1 ? G.pos0 + 16 * w + 15 : nk - 1;
        // D[t][e]: the dot of this lane's row with key 64 kb + 16 t + 4 qg + e (block b of the stage at st)
        auto dots = [&](const int8_t *st, int b, v4i (&D)[4]) {
#pragma unroll
            for (int tt = 0; tt < 4; tt++) {
                const int r = tt * 16 + ql;
                const v4i kf = *(const v4i *)&st[(4 * (b * 64 + r) + (qg ^ sw(r & 15))) * 16];
                D[tt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qf, v4i{0, 0, 0, 0}, 0, 0, 0);
            }
        };
        // walk 1: the extreme visible dots
        int32_t dmax = INT32_MIN, dmin = INT32_MAX;
        const int8_t *st = nullptr;
        for (int sb = 0; sb < n; sb++) {
            st = next_stage();
#pragma unroll
            for (int b = 0; b < AL_SB; b++) {
                const int kb = sb * AL_SB + b;
                if (kb >= nkb || 64 * kb > wmax) continue;
                v4i D[4];
                dots(st, b, D);
                if (64 * kb + 63 <= wlim) {
#pragma unroll
                    for (int tt = 0; tt < 4; tt++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            dmax = D[tt][e] > dmax ? D[tt][e] : dmax;
                            dmin = D[tt][e] < dmin ? D[tt][e] : dmin;
                        }
                } else {
                    const int L = lim - 64 * kb - 4 * qg;
#pragma unroll
                    for (int tt = 0; tt < 4; tt++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const bool ok = 16 * tt + e <= L;
                            const int32_t hiv = ok ? D[tt][e] : INT32_MIN, lov = ok ? D[tt][e] : INT32_MAX;
                            dmax = hiv > dmax ? hiv : dmax;
                            dmin = lov < dmin ? lov : dmin;
                        }
                }
            }
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) {  // the 4 lanes of this row
            const int32_t u = __shfl_xor(dmax, o, 64), v = __shfl_xor(dmin, o, 64);
            dmax = u > dmax ? u : dmax;
            dmin = v < dmin ? v : dmin;
        }
        const int32_t mx = score(dmax) > score(dmin) ? score(dmax) : score(dmin);
        // the table entries attn_exp[min(M - s, last)] of a block's keys, 0 for a masked key
        auto entries = [&](const int8_t *stg, int b, int kb, v4i (&E)[4]) {
            dots(stg, b, E);
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int e = 0; e < 4; e++) E[tt][e] = clamp0_uniform(mx - score(E[tt][e]), last);
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int e = 0; e < 4; e++) E[tt][e] = s_exp[E[tt][e]];
            if (64 * kb + 63 > wlim) {
                const int L = lim - 64 * kb - 4 * qg;
#pragma unroll
                for (int tt = 0; tt < 4; tt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) E[tt][e] = 16 * tt + e <= L ? E[tt][e] : 0;
            }
        };
        // walk 2: their sum (entries are < 2^31: a pair sums in u32)
        uint64_t sum = 0;
        for (int sb = n - 1; sb >= 0; sb--) {
            if (sb < n - 1) st = next_stage();
#pragma unroll
            for (int b = 0; b < AL_SB; b++) {
                const int kb = sb * AL_SB + b;
                if (kb >= nkb || 64 * kb > wmax) continue;
                v4i E[4];
                entries(st, b, kb, E);
#pragma unroll
                for (int tt = 0; tt < 4; tt++)
#pragma unroll
                    for (int e = 0; e < 4; e += 2) sum += (uint32_t)E[tt][e] + (uint32_t)E[tt][e + 1];
            }
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
        const double R = ldexp(1.0 / (double)sum, a.softmax_p);
        const double sp = softmax_sp(sum, a.softmax_p);
        // walk 3: p + 0x80808080 (the packed digits), and the digit-plane PV products, the V^T operand
        // by transposing LDS reads (the layouts of k_attend_short)
        const int tr_k = ql >> 1, tr_h = ql & 1;
        const int tr_key0 = 16 * (tr_k >> 2) + 4 * qg + (tr_k & 3);
        v4i acc[4][4];  // [digit plane][channel tile]: channel 16 c + 4 (l / 16) + e of row l % 16
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int c = 0; c < 4; c++) acc[k][c] = v4i{0, 0, 0, 0};
        for (int sb = 0; sb < n; sb++) {
            if (sb > 0) st = next_stage();
            v4i pf[AL_SB][4];  // [block][digit plane]: word t holds the digits of keys 16 t + 4 (l / 16) + e
#pragma unroll
            for (int b = 0; b < AL_SB; b++) {
                const int kb = sb * AL_SB + b;
                if (kb >= nkb || 64 * kb > wmax) continue;
                v4i E[4];
                entries(st, b, kb, E);
#pragma unroll
                for (int tt = 0; tt < 4; tt++) {
                    uint32_t dg[4], o[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) dg[e] = softmax_p_of((uint32_t)E[tt][e], R, sp) + 0x80808080u;
                    byte_transpose(dg[0], dg[1], dg[2], dg[3], o);
#pragma unroll
                    for (int k = 0; k < 4; k++) pf[b][k][tt] = (int32_t)(o[k] ^ 0x80808080u);
                }
            }
            const int8_t *sv = next_stage();
#pragma unroll
            for (int b = 0; b < AL_SB; b++) {
                const int kb = sb * AL_SB + b;
                if (kb >= nkb || 64 * kb > wmax) continue;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int8_t *p0 = sv + (4 * (b * 64 + tr_key0) + (c ^ sw(tr_key0 & 15))) * 16 + 8 * tr_h;
                    const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)p0);
                    const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)(p0 + 32 * 64));
                    const v4i vf = v4i{r0[0], r0[1], r1[0], r1[1]};
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        acc[k][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf, pf[b][k], acc[k][c], 0, 0, 0);
                }
            }
        }
        // The sum of the planes is |v| <= 2^P 128 <= 2^37 and each plane an i32 (|acc| <= keys 2^14): for
        // shifts 48 .. 63 attn_out_planes on v = hi 2^16 + lo, 0 <= lo < 2^16, else the i128 rule.
        if (myrow < G.count) {
            int8_t *o = attn_out(a, G.first + myrow, h * 64);
            const bool planes = a.out_s >= 48 && a.out_s <= 63;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                uint32_t packed = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int64_t v = (int64_t)acc[0][c][e] + (int64_t)acc[1][c][e] * 256 +
                                      (int64_t)acc[2][c][e] * 65536 + (int64_t)acc[3][c][e] * 16777216;
                    const int32_t r = planes ? attn_out_planes((int32_t)(v >> 16), (int32_t)(v & 0xffff), a.out_m,
                                                               (uint32_t)a.out_s)
                                             : (int32_t)clamp128(rescale_full(v, a.out_m, a.out_s), -127, 127);
                    packed |= (uint32_t)(uint8_t)(int8_t)r << (8 * e);
                }
                *(uint32_t *)(o + 16 * c + 4 * qg) = packed;
            }
        }
        if (!more) break;
        issued -= 4 * n - 2;
        used = 0;
        G = Gn;
        h = hn;
        n = stages_of(G);
    }
}

template <bool NOCLAMP, bool LDS_TABLE, bool MULTI>
static hipError_t launch_attend_groups_t(const AttnArgs &a, const AttnGroup *groups, int n_groups,
                                         hipStream_t stream) {
    // without MULTI the table lands in whole 1 KiB chunks
    const size_t lds = LDS_TABLE ? (MULTI ? sizeof(int32_t) * (size_t)a.exp_len : ((size_t)a.exp_len + 255) / 256 * 1024) : 0;
    {
        const hipError_t e = allow_dynamic_lds((const void *)k_attend_mfma<NOCLAMP, LDS_TABLE, MULTI>, lds);
        if (e != hipSuccess) return e;
    }
    launch_k((k_attend_mfma<NOCLAMP, LDS_TABLE, MULTI>), dim3(n_groups, a.n_head), dim3(256), lds, stream, a, groups);
    return hipGetLastError();
}

template <bool NOCLAMP, bool LDS_TABLE>
static hipError_t launch_attend_groups_m(const AttnArgs &a, const AttnGroup *groups, int n_groups, int max_keys,
                                         hipStream_t stream) {
    if (max_keys <= AT_SB * 64) return launch_attend_groups_t<NOCLAMP, LDS_TABLE, false>(a, groups, n_groups, stream);
    return launch_attend_groups_t<NOCLAMP, LDS_TABLE, true>(a, groups, n_groups, stream);
}

hipError_t launch_attend_groups(const AttnArgs &a, const AttnGroup *groups, int n_groups, int max_keys,
                                hipStream_t stream) {
    if (n_groups <= 0) return hipSuccess;
    // the output of a row is four 4-byte stores per head
    if (a.hd != 64 || (a.out_rows == 0 && a.ldo % 4 != 0) || ((uintptr_t)a.out & 3) != 0 || max_keys < 1)
        return hipErrorInvalidValue;
    const bool noclamp = a.score_s >= 13, lds_table = a.exp_len <= ATTN_LDS_TABLE;
    if (lds_table && max_keys <= 1 << 15 && a.score_s >= 22 && a.softmax_p <= 30 && a.out_s >= 0) {
        // whole 1 KiB chunks of the entries up to the zero tail (or the whole table)
        const int last = a.exp_last > 0 && a.exp_last < a.exp_len ? a.exp_last : a.exp_len - 1;
        const size_t lds = ((size_t)last + 256) / 256 * 1024;
        // the scores of up to 256 or 512 keys stay in registers (48 windows of 512, 16 heads: 141 us
        // against 172 walked); more keys are walked again (13 windows of 1,024, 12 heads: 235 ->
        // 120 us against k_attend_mfma, which held four blocks' scores in i64 forms and loaded K
        // and V between barriers)
        auto run = [&](auto kernel) -> hipError_t {
            const void *fn = (const void *)kernel;
            hipError_t e = allow_dynamic_lds(fn, lds);
            if (e != hipSuccess) return e;
            // the resident workgroups (CUs x workgroups per CU at this LDS size), at most one per task
            int resident = 0;
            e = resident_workgroups(fn, 256, lds, &resident);
            if (e != hipSuccess) return e;
            const int n_tasks = n_groups * a.n_head;
            const int P = resident < n_tasks ? resident : n_tasks;
            launch_k(kernel, dim3(P), dim3(256), lds, stream, a, groups, n_tasks);
            return hipGetLastError();
        };
        if (max_keys <= 256) return run(k_attend_short<4>);
        if (max_keys <= 512) return run(k_attend_short<8>);
        return run(k_attend_long);
    }
    if (noclamp && lds_table) return launch_attend_groups_m<true, true>(a, groups, n_groups, max_keys, stream);
    if (noclamp) return launch_attend_groups_m<true, false>(a, groups, n_groups, max_keys, stream);
    if (lds_table) return launch_attend_groups_m<false, true>(a, groups, n_groups, max_keys, stream);
    return launch_attend_groups_m<false, false>(a, groups, n_groups, max_keys, stream);
}

// =============================================================================================
// The coder op: logits -> weights (logits.rs:62-72) -> the interval of FreqTable::from_weights
// (crates/taco-coder/src/freq.rs:103-149) for an Encode(token) or Decode(target) query.
// One workgroup per row; thread t owns the symbols [t * chunk, (t + 1) * chunk).
// f_i = 1 + floor(w_i * spare / W) with an exact quotient: a 64-bit reciprocal of W and one
// correction step (W >= 2^32), or a plain u64 division (W < 2^32).
// =============================================================================================


// The weight of symbol j of a row: the table entry of its logit (SRC 0) or given weights
// (SRC 1); MODE 2 maps it by the row's mix record (mixer.rs:491-516): max(1, w) without a
// prediction, w'[p] for the prediction, max(1, (w m) >> k) for the others (an exact u128
// product: given weights may reach 2^64 - 1).
template <int SRC, int MODE>
struct RowWeights {
    const int64_t *l;
    const uint64_t *w;
    const uint64_t *table;
    int64_t M;
    int last;
    MixRec rec;
    __device__ __forceinline__ uint64_t base(int j) const {
        if (SRC == 1) return w[j];
        const int64_t dd = M - l[j];
        return table[dd < last ? dd : last];
    }
    __device__ __forceinline__ uint64_t at(int j) const {
        const uint64_t v = base(j);
        if (MODE != 2 || rec.p == MIX_PLAIN) return v;
        if (rec.p == MIX_NONE) return v > 1 ? v : 1;
        if ((uint32_t)j == rec.p) return rec.wp;
        const u128 x = ((u128)v * rec.m) >> rec.k;
        return x > 1 ? (uint64_t)x : 1;
    }
};

// MODE 0: the coder op; 1: the mixer statistics (sum w, w[p], top) of each row; 2: the coder op
// on the mixed weights of each row's record.
template <int SRC, int MODE>
__global__ __launch_bounds__(256) void k_coder(CoderArgs a) {
    __shared__ int64_t s_i64[256];
    __shared__ uint64_t s_u64[256];
    __shared__ uint32_t s_idx[256];
    __shared__ uint64_t s_W, s_frac;
    __shared__ uint32_t s_largest;
    const int row = blockIdx.x, tid = threadIdx.x;
    const int V = a.vocab;
    const int chunk = (V + 255) / 256;
    const int j0 = tid * chunk, j1 = min(V, j0 + chunk);
    RowWeights<SRC, MODE> rw;
    rw.l = SRC == 0 ? a.logits + (size_t)row * a.ld : nullptr;
    rw.w = SRC == 1 ? a.wsrc + (size_t)row * V : nullptr;
    rw.table = a.table;
    rw.last = a.table_len - 1;
    rw.M = 0;
    if (MODE != 0) rw.rec = a.mix[row];

    if (SRC == 0) {  // pass 1: the largest logit
        int64_t mx = INT64_MIN;
        for (int j = j0; j < j1; j++) mx = rw.l[j] > mx ? rw.l[j] : mx;
        s_i64[tid] = mx;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o) s_i64[tid] = s_i64[tid + o] > s_i64[tid] ? s_i64[tid + o] : s_i64[tid];
            __syncthreads();
        }
        rw.M = s_i64[0];
        __syncthreads();
    }
    // pass 2: W = sum w and the largest weight (the lowest id on a tie)
    uint64_t W = 0, best = 0;
    uint32_t bidx = 0xFFFFFFFFu;
    for (int j = j0; j < j1; j++) {
        const uint64_t w = MODE == 1 ? rw.base(j) : rw.at(j);
        if (MODE == 0 && a.weights) a.weights[(size_t)row * V + j] = w;
        W += w;
        if (bidx == 0xFFFFFFFFu || w > best) {
            best = w;
            bidx = j;
        }
    }
    s_u64[tid] = W;
    s_i64[tid] = (int64_t)best;
    s_idx[tid] = bidx;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            s_u64[tid] += s_u64[tid + o];
            const uint64_t b0 = (uint64_t)s_i64[tid], b1 = (uint64_t)s_i64[tid + o];
            const uint32_t i0 = s_idx[tid], i1 = s_idx[tid + o];
            // the larger weight wins; on a tie the lower index (a strided tree does not keep
            // the lower slot on the lower indices, so compare them)
            if (i0 == 0xFFFFFFFFu || (i1 != 0xFFFFFFFFu && (b1 > b0 || (b1 == b0 && i1 < i0)))) {
                s_i64[tid] = (int64_t)b1;
                s_idx[tid] = i1;
            }
        }
        __syncthreads();
    }
    if (MODE == 1) {  // mixer.rs:278-288: top is token 0 when every weight is 0
        if (tid == 0) {
            const uint32_t p = rw.rec.p;
            uint64_t *st = a.stats + 3 * (size_t)row;
            st[0] = s_u64[0];
            st[1] = p < (uint32_t)V ? rw.base((int)p) : 0;
            st[2] = s_u64[0] == 0 ? 0 : s_idx[0];
        }
        return;
    }
    if (tid == 0) {
        uint64_t Wt = s_u64[0];
        uint32_t largest = s_idx[0];
        if (Wt == 0) {  // every weight 0: every weight is 1 (freq.rs:119-123)
            Wt = (uint64_t)V;
            largest = 0;
        }
        const uint64_t total = (uint64_t)1 << a.bits;
        const uint64_t spare = total - (uint64_t)V;
        s_W = Wt;
        s_largest = largest;
        s_frac = Wt >= ((uint64_t)1 << 32) ? coder_frac(spare, Wt) : 0;
    }
    __syncthreads();
    const uint64_t Wt = s_W, frac = s_frac;
    const bool all_zero = s_u64[0] == 0;
    const uint32_t largest = s_largest;
    const uint64_t total = (uint64_t)1 << a.bits, spare = total - (uint64_t)V;
    const uint32_t kind = a.queries ? a.queries[2 * row] : 0;
    const uint32_t value = a.queries ? a.queries[2 * row + 1] : 0;
    // pass 3: the sum of f over the chunk, and over the symbols below the encode token
    uint64_t F = 0, Fbelow = 0, ftok = 0;
    for (int j = j0; j < j1; j++) {
        const uint64_t w = all_zero ? 1 : rw.at(j);
        const uint64_t f = 1 + quotient(w, spare, Wt, frac);
        F += f;
        if (kind == 0 && (uint32_t)j < value) Fbelow += f;
        if (kind == 0 && (uint32_t)j == value) ftok = f;
    }
    __syncthreads();
    s_u64[tid] = F;
    __syncthreads();
    if (tid == 0) {  // exclusive scan of the chunk sums, in order
        uint64_t run = 0;
        for (int t = 0; t < 256; t++) {
            const uint64_t v = s_u64[t];
            s_u64[t] = run;
            run += v;
        }
        s_W = run;  // sum of all f
    }
    __syncthreads();
    const uint64_t base = s_u64[tid];
    const uint64_t Q = s_W;
    const uint64_t rem = total - Q;
    uint64_t *out = a.intervals ? a.intervals + 3 * (size_t)row : nullptr;
    if (!out) return;
    if (kind == 0) {
        // start = sum_{j < tok} f_j (+ rem if the largest is below tok); the owner writes it
        const uint32_t tok = value;
        if ((int)tok >= j0 && (int)tok < j1) {
            const uint64_t start = base + Fbelow + (largest < tok ? rem : 0);
            const uint64_t freq = ftok + (largest == tok ? rem : 0);
            out[0] = tok;
            out[1] = start;
            out[2] = freq;
        }
        return;
    }
    // Decode: the largest i with start_i <= target; starts increase with i.
    const uint64_t target = value;
    uint64_t run = base;
    int cand = -1;
    uint64_t cstart = 0, cfreq = 0;
    for (int j = j0; j < j1; j++) {
        const uint64_t w = all_zero ? 1 : rw.at(j);
        const uint64_t f = 1 + quotient(w, spare, Wt, frac);
        const uint64_t start = run + ((uint32_t)j > largest ? rem : 0);
        run += f;
        if (start <= target) {
            cand = j;
            cstart = start;
            cfreq = f + ((uint32_t)j == largest ? rem : 0);
        } else {
            break;
        }
    }
    __syncthreads();
    s_i64[tid] = cand;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) s_i64[tid] = s_i64[tid + o] > s_i64[tid] ? s_i64[tid + o] : s_i64[tid];
        __syncthreads();
    }
    if (cand >= 0 && cand == s_i64[0]) {
        out[0] = (uint64_t)cand;
        out[1] = cstart;
        out[2] = cfreq;
    }
}

template <int MODE>
static hipError_t launch_coder_mode(const CoderArgs &a, int n_rows, hipStream_t stream) {
    if (n_rows <= 0) return hipSuccess;
    if (MODE != 0 && !a.mix) return hipErrorInvalidValue;
    if (a.wsrc)
        launch_k((k_coder<1, MODE>), dim3(n_rows), dim3(256), 0, stream, a);
    else
        launch_k((k_coder<0, MODE>), dim3(n_rows), dim3(256), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_coder(const CoderArgs &a, int n_rows, hipStream_t stream) {
    return launch_coder_mode<0>(a, n_rows, stream);
}
hipError_t launch_mix_stats(const CoderArgs &a, int n_rows, hipStream_t stream) {
    return a.stats ? launch_coder_mode<1>(a, n_rows, stream) : hipErrorInvalidValue;
}
hipError_t launch_coder_mixed(const CoderArgs &a, int n_rows, hipStream_t stream) {
    return launch_coder_mode<2>(a, n_rows, stream);
}


// =============================================================================================
// The coder op over compact logits. One workgroup per row, one coalesced pass over the row: the
// table index d_j = min(M - l_j, len - 1) of every symbol goes into a histogram in LDS (and a
// second one for the symbols below an Encode token), so the quotients floor(table[d] * spare /
// W) are computed once per table entry, not once per symbol:
//   W = sum_d cnt[d] table[d];  sum f = V + sum_d cnt[d] q[d];  sum_{j<tok} f = tok + sum_d
//   cnt_lo[d] q[d].  largest = the first symbol whose weight is table[0] (d <= d0).
// A Decode query needs the starts in symbol order: an ordered block scan over the row.
// =============================================================================================

__device__ __forceinline__ int64_t block_max64(int64_t v, int64_t *s, int tid) {
    s[tid] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) s[tid] = s[tid + o] > s[tid] ? s[tid + o] : s[tid];
        __syncthreads();
    }
    v = s[0];
    __syncthreads();
    return v;
}

__device__ __forceinline__ uint64_t block_sum64(uint64_t v, uint64_t *s, int tid) {
    s[tid] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) s[tid] += s[tid + o];
        __syncthreads();
    }
    v = s[0];
    __syncthreads();
    return v;
}

// Reductions over a block of NW waves through wave shuffles and one LDS slot per wave.
template <int NW = 4>
__device__ __forceinline__ int64_t block_max64w(int64_t v, int64_t *slots, int tid) {
    v = wave_max64(v);
    if ((tid & 63) == 0) slots[tid >> 6] = v;
    __syncthreads();
    int64_t r = slots[0];
#pragma unroll
    for (int w = 1; w < NW; w++) r = slots[w] > r ? slots[w] : r;
    __syncthreads();
    return r;
}

template <int NW = 4>
__device__ __forceinline__ uint64_t block_sum64w(uint64_t v, uint64_t *slots, int tid) {
    v = (uint64_t)wave_sum64((int64_t)v);
    if ((tid & 63) == 0) slots[tid >> 6] = v;
    __syncthreads();
    uint64_t r = slots[0];
#pragma unroll
    for (int w = 1; w < NW; w++) r += slots[w];
    __syncthreads();
    return r;
}

// Exclusive prefix sum over a block of NW waves in thread order, and the block total: wave scans
// through shuffles, then the wave totals through one LDS slot per wave.
template <int NW = 4>
__device__ __forceinline__ uint64_t block_scan64w(uint64_t v, uint64_t *slots, int tid, uint64_t &total) {
    const int lane = tid & 63, w = tid >> 6;
    int64_t x = (int64_t)v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t u = __shfl_up(x, o, 64);
        if (lane >= o) x += u;
    }
    if (lane == 63) slots[w] = (uint64_t)x;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const uint64_t t = slots[k];
        before += k < w ? t : 0;
        all += t;
    }
    __syncthreads();
    total = all;
    return before + (uint64_t)x - v;
}

// The weights of rows of compact logits (run_weights): 2,048 symbols per workgroup, so that the
// 402 KB a row of GPT-2's vocabulary writes come from 25 CUs (one workgroup per row took 100 us
// for a row; the row max is redone per workgroup, 6 KB of tile maxes from the caches).
__global__ __launch_bounds__(256) void k_weights_compact(CompactCoderArgs a) {
    __shared__ int64_t slots[4];
    const int row = blockIdx.y, tid = threadIdx.x, V = a.vocab, last = a.table_len - 1;
    const uint16_t *d16 = a.d16 + (size_t)row * a.ld16;
    const int64_t *tm = a.tmax + (size_t)row * a.ntiles;
    const int j0 = blockIdx.x * 2048 + tid;
    int64_t t8[8];
    uint16_t d8[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {  // no branch around the loads: a symbol past the row reads the last one
        const int j = j0 + 256 * u < V ? j0 + 256 * u : V - 1;
        t8[u] = tm[j >> 6];
        d8[u] = d16[j];
    }
    int64_t mx = INT64_MIN;
    for (int t = tid; t < a.ntiles; t += 1024) {
        int64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = tm[min(t + 256 * u, a.ntiles - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) mx = v[u] > mx ? v[u] : mx;
    }
    const int64_t M = block_max64w(mx, slots, tid);
    uint64_t w8[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int64_t d = M - t8[u] + d8[u];
        w8[u] = a.table[d < last ? d : last];
    }
    uint64_t *out = a.weights + (size_t)row * V;
#pragma unroll
    for (int u = 0; u < 8; u++)
        if (j0 + 256 * u < V) out[j0 + 256 * u] = w8[u];
}

// One row per workgroup. The histogram counts the symbols of each table index d < zcut (the
// bins with a nonzero weight; a symbol's index is min(d, len - 1)); with V < 2^16 the count and
// the count below the Encode token share one u32 (low and high half), else they are two arrays.
// When the table ends in zeros (zcut < len), symbols with d >= zcut have weight 0, f = 1 and no
// share of the spare, and need no count; else (zcut = len) every symbol has a bin.
// STATS: the mixer statistics of the row (sum w, w[p] for the record's p, the top token = the
// largest) instead of the coder interval.
// PACKED: V < 2^16 (the launch picks the form). The histogram is the only sizeable LDS of the
// workgroup (4 (zcut + 64) bytes); with at most 128 registers four rows share a CU, so a chunk
// of 2,048 rows runs in two full rounds of 1,024.
// FIND: queries may be Decode ones (a template parameter, so that the fold's Encode launches keep
// the registers and the S pass they had: 58.6 against 55.2 us per 2,048 rows otherwise). A Decode
// query finds its symbol from the sums of f over segments of 64 symbols (more for
// vocabularies above 65,536): f = 1 + q of a symbol's bin by one LDS lookup (the S pass leaves q in
// the histogram's place), a scan over the segment sums, and one wave's scan of the segment that
// holds the target. (A scan of the whole row in symbol order, with the quotients formed again,
// took 65 us of an 88 us launch.)
constexpr int CODER_SEGS = 1024;  // at most this many segments

template <bool STATS, bool PACKED, bool FIND, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_coder_compact(CompactCoderArgs a) {
    constexpr int NW = NT / 64;
    // LDS: the histogram from address 0 (a bin's byte address is 4 d), then the reduction slots and
    // the segment sums of a Decode query
    extern __shared__ uint4 lds4[];
    uint32_t *hist = (uint32_t *)lds4;
    const int V = a.vocab, len = a.table_len, last = len - 1;
    const int zc = a.zcut;
    constexpr bool packed = PACKED;
    const int n4 = ((packed ? zc + 64 : 2 * zc) + 3) >> 2;  // histogram words in uint4
    int64_t *s_i = (int64_t *)(lds4 + n4);
    uint64_t *s_u = (uint64_t *)s_i + NW;
    uint32_t *seg = (uint32_t *)(s_u + 2 * NW);
    const int row = blockIdx.x, tid = threadIdx.x;
    const uint16_t *d16 = a.d16 + (size_t)row * a.ld16;
    const int64_t *tm = a.tmax + (size_t)row * a.ntiles;
    const uint32_t kind = a.queries ? a.queries[2 * row] : 0;
    const uint32_t value = a.queries ? a.queries[2 * row + 1] : 0;
    const uint32_t tok = kind == 0 && !STATS ? value : 0;  // Encode token (0: no symbol below)
    // thread 0 of an Encode row needs the token's weight last: its tile max and offset are
    // loaded first, its table entry as soon as the row max is known
    const bool tok_lead = !STATS && tid == 0 && kind == 0 && a.intervals;
    int64_t tok_tm = 0;
    uint32_t tok_off = 0;
    if (tok_lead) {
        tok_tm = tm[tok >> 6];
        tok_off = d16[tok];
    }

    // The symbol pass reads 8 consecutive symbols per thread and group (one 16-byte load of d16;
    // the 8 share a 64-column tile), four groups per step, and the tile maxes of those groups:
    // d16 rows are padded to whole tiles, so every load is in range. Two register sets take the
    // steps in turn, each step's loads issued one step ahead (the first before the row max). A
    // group past the row loads the row's last group instead (no branch around the loads, so a
    // step waits only for its own loads).
    constexpr int STEP = 4 * NT * 8;
    const int last_group = (V - 1) & ~7;
    auto fetch = [&](uint4 (&raw)[4], int64_t (&tmv)[4], int g0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int gq = g0 + u * NT * 8;
            const int gc = gq < V ? gq : last_group;
            raw[u] = *(const uint4 *)(d16 + gc);
            tmv[u] = tm[gc >> 6];
        }
    };
    uint4 ra[4], rb[4];
    int64_t ta[4], tb[4];
    // The row max: the tile maxes are loaded first (four per thread at a time, clamped indexes,
    // no branch), so the max waits for them alone while the first step's groups arrive; the
    // histogram is cleared meanwhile (the barriers of the max order it before the symbol pass).
    int64_t mx = INT64_MIN;
    for (int t = tid; t < a.ntiles; t += 4 * NT) {
        int64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = tm[min(t + NT * u, a.ntiles - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) mx = v[u] > mx ? v[u] : mx;
    }
    fetch(ra, ta, tid * 8);
    for (int k = tid; k < n4; k += NT) lds4[k] = make_uint4(0, 0, 0, 0);
    const int64_t M = block_max64w<NW>(mx, s_i, tid);
    uint64_t tok_w = 0;
    if (tok_lead) {
        const int64_t dt = M - tok_tm + tok_off;
        tok_w = a.table[dt < last ? dt : last];
    }
    int64_t first = INT64_MAX;  // the first symbol with weight table[0] (d <= d0)
    // A symbol's index is min(d, last) (logits.rs:62-72). tail0: the table ends in zeros, so
    // every d >= zcut weighs 0 (no count needed); else (zcut = len) every d >= last weighs
    // table[last] and counts in the last bin, and no group can be skipped.
    const bool tail0 = zc < len;
    const unsigned short zl = (unsigned short)(tail0 ? zc + (tid & 63) : last);
    // the packed path forms bin byte addresses in 16 bits: 4 zl < 2^16 (other tables take the
    // per-symbol path)
    const bool addr16 = tail0 ? zc <= 16320 : last <= 16383;
    auto process = [&](const uint4 (&cur)[4], const int64_t (&tmv)[4], int g0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int gq = g0 + u * NT * 8;
            // with tail0, a group whose tile max is zcut or more below M has only weight-0
            // symbols; else its symbols' indexes start at min(M - tile max, last)
            if (gq >= V) continue;
            const int64_t b64 = M - tmv[u];
            if (tail0 && b64 >= zc) continue;
            const int base = (int)(b64 < last ? b64 : last);
            const uint16_t *dv = (const uint16_t *)&cur[u];
            if (packed && addr16 && gq + 8 <= V) {
                // two symbols per packed u16 add and min: d = min(base + d16, zl), the add
                // saturating at 65535 (> zl; a d16 may be up to 65535, base <= last < 2^14):
                // with tail0 the symbols of weight 0 (d >= zc) land in the 64 spare bins
                // past the weighted ones (never read), each lane in its own, else d >= last lands
                // in the last bin, and no symbol needs a test; the count below the Encode token
                // rides in the high half
                const us2 bb = {(unsigned short)base, (unsigned short)base};
                const us2 zz = {zl, zl};
                const uint32_t *wv = (const uint32_t *)&cur[u];
                // then both bins' byte addresses in one packed shift (4 d <= 4 (zc + 63) < 2^16)
                us2 v[4];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    __builtin_memcpy(&v[p], &wv[p], 4);
                    v[p] = __builtin_elementwise_min(__builtin_elementwise_add_sat(v[p], bb), zz) << (unsigned short)2;
                }
                uint8_t *hb = (uint8_t *)hist;
                auto bin = [&](unsigned short byte) { return (uint32_t *)(hb + byte); };
                if (!(gq < (int)tok && (int)tok < gq + 8)) {
                    const uint32_t inc = gq < (int)tok ? 0x10001u : 1u;
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        atomicAdd(bin(v[p].x), inc);
                        atomicAdd(bin(v[p].y), inc);
                    }
                } else {  // the group of the Encode token
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        atomicAdd(bin(v[p].x), gq + 2 * p < (int)tok ? 0x10001u : 1u);
                        atomicAdd(bin(v[p].y), gq + 2 * p + 1 < (int)tok ? 0x10001u : 1u);
                    }
                }
                if (base <= a.d0) {  // the top weight needs min(d, last) <= d0, so base <= d0
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        const int dq = base + (int)dv[q];
                        if ((dq < last ? dq : last) <= a.d0 && gq + q < first) first = gq + q;
                    }
                }
                continue;
            }
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int j = gq + q;
                const int dd = base + (int)dv[q] < last ? base + (int)dv[q] : last;
                if (j < V && dd < zc) {
                    if (packed) {
                        atomicAdd(&hist[dd], (uint32_t)j < tok ? 0x10001u : 1u);
                    } else {
                        atomicAdd(&hist[dd], 1u);
                        if ((uint32_t)j < tok) atomicAdd(&hist[zc + dd], 1u);
                    }
                    if (dd <= a.d0 && j < first) first = j;
                }
            }
        }
    };
    for (int s0 = 0; s0 < V; s0 += 2 * STEP) {  // uniform trip count; groups past V are skipped
        const int g0 = s0 + tid * 8;
        fetch(rb, tb, g0 + STEP);
        process(ra, ta, g0);
        if (s0 + STEP >= V) break;
        fetch(ra, ta, g0 + 2 * STEP);
        process(rb, tb, g0 + STEP);
    }
    __syncthreads();

    // The weighted bins of this thread: d = tid + NT k. The first KB (zcut up to 8,192) take
    // their table entries in one batch of loads (the table holds CODER_TABLE_READ entries; a bin
    // past zcut has count 0), kept in registers for the S pass; bins from 8,192 on go 8 at a
    // time, loaded in each pass.
    // c t = c t_lo + 2^32 c t_hi with t <= 2^40: the low parts accumulate in 64 bits (one
    // multiply-add each), the high parts (c t_hi <= V 2^8 summed over a thread's bins) in 32.
    constexpr int KB = 8192 / NT, BU = 8;
    static_assert(NT * KB <= CODER_TABLE_READ, "the first bins' entries are read without bounds tests");
    const int kept = zc < NT * KB ? zc : NT * KB;
    uint64_t tk[KB];
#pragma unroll
    for (int k = 0; k < KB; k++) {
        const int d = tid + NT * k;
        tk[k] = a.table[d];
    }
    uint64_t W = 0;
    uint32_t w_hi = 0;
#pragma unroll
    for (int k = 0; k < KB; k++) {
        const int d = tid + NT * k;
        const uint32_t h = d < kept ? hist[d] : 0;
        const uint32_t c = packed ? (h & 0xffffu) : h;
        W += (uint64_t)c * (uint32_t)tk[k];
        w_hi += c * (uint32_t)(tk[k] >> 32);
    }
    for (int d0 = tid + NT * KB; d0 < zc; d0 += NT * BU) {
        uint32_t c[BU];
        uint64_t t[BU];
#pragma unroll
        for (int u = 0; u < BU; u++) {
            const int d = d0 + NT * u;
            c[u] = d < zc ? (packed ? (hist[d] & 0xffffu) : hist[d]) : 0;
        }
#pragma unroll
        for (int u = 0; u < BU; u++) t[u] = c[u] ? a.table[d0 + NT * u] : 0;
#pragma unroll
        for (int u = 0; u < BU; u++) {
            W += (uint64_t)c[u] * (uint32_t)t[u];
            w_hi += c[u] * (uint32_t)(t[u] >> 32);
        }
    }
    W += (uint64_t)w_hi << 32;
    // W and the largest (the first symbol of weight table[0]) in one round
    W = (uint64_t)wave_sum64((int64_t)W);
    first = -wave_max64(-first);
    if ((tid & 63) == 0) {
        s_u[tid >> 6] = W;
        s_i[tid >> 6] = first;
    }
    __syncthreads();
    W = s_u[0];
    int64_t largest = s_i[0];
#pragma unroll
    for (int w = 1; w < NW; w++) {
        W += s_u[w];
        largest = s_i[w] < largest ? s_i[w] : largest;
    }
    __syncthreads();
    if (STATS) {  // mixer.rs:278-288 (W >= table[0] >= 1, so top is the largest)
        if (tid == 0) {
            const uint32_t p = a.mix[row].p;
            uint64_t wp = 0;
            if (p < (uint32_t)V) {
                const int64_t dp = M - tm[p >> 6] + d16[p];
                wp = a.table[dp < last ? dp : last];
            }
            uint64_t *st = a.stats + 3 * (size_t)row;
            st[0] = W;
            st[1] = wp;
            st[2] = (uint64_t)largest;
        }
        return;
    }
    const uint64_t total = (uint64_t)1 << a.bits, spare = total - (uint64_t)V;
    // q(td) = floor(td spare / W) for a weight td <= W, so q < 2^32: v = td R with R = spare / W
    // in double takes three roundings (W to double, the quotient, the product),
    // |v - q| < 2^32 4 2^-53 = 2^-19; when v lies at least 2^-18 from an integer, floor(v) is q
    // (1.5 2^52 added rounds v to the nearest integer, the low word of the sum), else the exact
    // quotient, whose 64-bit reciprocal floor(spare 2^64 / W) only the thread that needs it forms.
    const double Rq = (double)spare / (double)W;
    auto q_of = [&](uint64_t td) -> uint64_t {
        if (!td) return 0;
        const double v = (double)td * Rq;
        const double t = v + 6755399441055744.0;
        const double dl = v - (t - 6755399441055744.0);
        if (fabs(dl) >= 0x1p-18) {
            uint64_t bits;
            __builtin_memcpy(&bits, &t, sizeof bits);
            return (uint64_t)(uint32_t)bits - (dl < 0.0 ? 1 : 0);
        }
        return quotient(td, spare, W, W >= ((uint64_t)1 << 32) ? coder_frac(spare, W) : 0);
    };
    // q for a bin from the double estimate; a live bin (count nonzero) whose estimate lies too
    // close to an integer is marked instead and takes the exact quotient after the pass (its
    // entry loaded again), which keeps the unrolled pass small. t <= 2^40 goes to double as
    // 2^32 t_hi + t_lo (exact).
    auto q_est = [&](uint64_t td, bool &close) -> uint32_t {
        const double x = (double)(uint32_t)(td >> 32) * 4294967296.0 + (double)(uint32_t)td;
        const double v = x * Rq;
        const double t = v + 6755399441055744.0;
        const double dl = v - (t - 6755399441055744.0);
        uint64_t bits;
        __builtin_memcpy(&bits, &t, sizeof bits);
        close = !(fabs(dl) >= 0x1p-18);
        return (uint32_t)bits - (dl < 0.0 ? 1u : 0u);
    };
    const bool find = FIND && kind != 0;  // a Decode query: each counted bin keeps its q in the histogram's place
    uint64_t S = 0, Slo = 0;
    uint32_t exact = 0;  // bit k: bin tid + NT k needs the exact quotient
#pragma unroll
    for (int k = 0; k < KB; k++) {
        const int d = tid + NT * k;
        const uint32_t h = d < kept ? hist[d] : 0;
        const uint32_t c = packed ? (h & 0xffffu) : h;
        const uint32_t clo = packed ? (h >> 16) : (c ? hist[zc + d] : 0);
        bool close;
        const uint32_t q = q_est(tk[k], close);
        if (close && c) {
            exact |= 1u << k;
        } else {
            S += (uint64_t)c * q;
            Slo += (uint64_t)clo * q;
            if (find && c) hist[d] = q;
        }
    }
    auto add_exact = [&](int d) {
        const uint32_t h = hist[d];
        const uint32_t c = packed ? (h & 0xffffu) : h;
        const uint32_t clo = packed ? (h >> 16) : hist[zc + d];
        const uint64_t q = quotient(a.table[d], spare, W, W >= ((uint64_t)1 << 32) ? coder_frac(spare, W) : 0);
        S += (uint64_t)c * q;
        Slo += (uint64_t)clo * q;
        if (find) hist[d] = (uint32_t)q;  // q < 2^32: the weight is at most W
    };
    while (exact) {
        const int k = __builtin_ctz(exact);
        exact &= exact - 1;
        add_exact(tid + NT * k);
    }
    for (int d0 = tid + NT * KB; d0 < zc; d0 += NT * BU) {
        uint32_t c[BU], clo[BU];
        uint64_t td[BU];
#pragma unroll
        for (int u = 0; u < BU; u++) {
            const int d = d0 + NT * u;
            const uint32_t h = d < zc ? hist[d] : 0;
            c[u] = packed ? (h & 0xffffu) : h;
            clo[u] = packed ? (h >> 16) : (c[u] ? hist[zc + d] : 0);
        }
#pragma unroll
        for (int u = 0; u < BU; u++) td[u] = c[u] ? a.table[d0 + NT * u] : 0;
        uint32_t ex = 0;
#pragma unroll
        for (int u = 0; u < BU; u++) {
            bool close;
            const uint32_t q = q_est(td[u], close);
            if (close && c[u]) {
                ex |= 1u << u;
            } else {
                S += (uint64_t)c[u] * q;
                Slo += (uint64_t)clo[u] * q;
                if (find && c[u]) hist[d0 + NT * u] = q;
            }
        }
        while (ex) {
            const int u = __builtin_ctz(ex);
            ex &= ex - 1;
            add_exact(d0 + NT * u);
        }
    }
    // S and Slo in one round
    S = (uint64_t)wave_sum64((int64_t)S);
    Slo = (uint64_t)wave_sum64((int64_t)Slo);
    if ((tid & 63) == 0) {
        s_u[tid >> 6] = S;
        s_u[NW + (tid >> 6)] = Slo;
    }
    __syncthreads();
    S = s_u[0];
    Slo = s_u[NW];
#pragma unroll
    for (int w = 1; w < NW; w++) {
        S += s_u[w];
        Slo += s_u[NW + w];
    }
    __syncthreads();
    const uint64_t rem = total - ((uint64_t)V + S);
    uint64_t *out = a.intervals ? a.intervals + 3 * (size_t)row : nullptr;
    if (!out) return;
    if (kind == 0) {
        if (tok_lead) {
            const uint64_t f = 1 + q_of(tok_w);
            out[0] = tok;
            out[1] = (uint64_t)tok + Slo + ((int64_t)tok > largest ? rem : 0);
            out[2] = f + ((int64_t)tok == largest ? rem : 0);
        }
        return;
    }
    if constexpr (!FIND) return;
    // Decode: the symbol whose interval [start, start + f) holds the target (every f is at least 1
    // and their sum is the total, so there is one).
    const uint64_t target = value;
    int shift = 6;  // a segment is 2^shift symbols
    while (((V - 1) >> shift) >= CODER_SEGS) shift++;
    const int nseg = ((V - 1) >> shift) + 1;
    for (int k = tid; k < CODER_SEGS; k += NT) seg[k] = 0;
    if (packed && tid < 64) hist[zc + tid] = 0;  // the spare bins: weight 0
    __syncthreads();
    auto q_at = [&](int64_t d) -> uint32_t {  // q of a symbol at distance d (d >= zc: weight 0)
        const int dd = (int)(d < last ? d : last);
        return dd < zc ? hist[dd] : 0;
    };
    // The sums of q over the 8 symbols of a thread's group, then over the eight threads of a tile of
    // 64, in 32 bits: all the q of a row add up to at most spare < 2^32.
    auto tiles = [&](const uint4 (&cur)[4], const int64_t (&tmv)[4], int g0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int gq = g0 + u * NT * 8;
            uint32_t sum = 0;
            const int64_t b64 = M - tmv[u];
            if (gq < V && !(tail0 && b64 >= zc)) {
                if (packed && addr16 && gq + 8 <= V) {  // bin addresses as in the symbol pass
                    const unsigned short base = (unsigned short)(b64 < last ? b64 : last);
                    const us2 bb = {base, base}, zz = {zl, zl};
                    const uint32_t *wv = (const uint32_t *)&cur[u];
                    const uint8_t *hb = (const uint8_t *)hist;
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        us2 v;
                        __builtin_memcpy(&v, &wv[p], 4);
                        v = __builtin_elementwise_min(__builtin_elementwise_add_sat(v, bb), zz) << (unsigned short)2;
                        sum += *(const uint32_t *)(hb + v.x) + *(const uint32_t *)(hb + v.y);
                    }
                } else {
                    const uint16_t *dv = (const uint16_t *)&cur[u];
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        if (gq + q < V) sum += q_at(b64 + dv[q]);
                }
            }
#pragma unroll
            for (int o = 1; o < 8; o <<= 1) sum += __shfl_xor(sum, o, 64);
            if ((tid & 7) == 0 && sum) atomicAdd(&seg[gq >> shift], sum);
        }
    };
    for (int s0 = 0; s0 < V; s0 += STEP) {  // uniform trip count; groups past V add nothing
        fetch(ra, ta, s0 + tid * 8);
        tiles(ra, ta, s0 + tid * 8);
    }
    __syncthreads();
    // the segment that holds the target: each thread scans SP consecutive segments
    constexpr int SP = CODER_SEGS / NT;
    const int lseg = (int)(largest >> shift);
    uint64_t mine[SP], local = 0, all;
#pragma unroll
    for (int u = 0; u < SP; u++) {
        const int k = tid * SP + u;
        const int count = min(V - (k << shift), 1 << shift);  // the segment's symbols (k < nseg)
        mine[u] = k < nseg ? (uint64_t)seg[k] + (uint64_t)count + (k == lseg ? rem : 0) : 0;
        local += mine[u];
    }
    uint64_t at = block_scan64w<NW>(local, s_u, tid, all);
#pragma unroll
    for (int u = 0; u < SP; u++) {
        if (at <= target && target - at < mine[u]) {
            s_u[0] = (uint64_t)(tid * SP + u);
            s_u[1] = at;
        }
        at += mine[u];
    }
    __syncthreads();
    if (tid >= 64) return;
    const int j_end = min(V, (int)(s_u[0] + 1) << shift);
    uint64_t start = s_u[1];
    for (int j0 = (int)s_u[0] << shift; j0 < j_end; j0 += 64) {  // one tile at a time
        const int j = j0 + tid;
        uint64_t f = 0;
        if (j < V) f = 1 + (uint64_t)q_at(M - tm[j >> 6] + d16[j]) + (j == largest ? rem : 0);
        uint64_t end = f;  // inclusive scan
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint64_t v = __shfl_up(end, o, 64);
            if (tid >= o) end += v;
        }
        const uint64_t mystart = start + end - f;
        const bool here = mystart <= target && target - mystart < f;
        if (here) {
            out[0] = (uint64_t)j;
            out[1] = mystart;
            out[2] = f;
        }
        if (__any(here)) return;
        start += __shfl(end, 63, 64);
    }
}

// The mixed coder op over compact logits: k_coder_compact with the weights of each row's mix
// record (mixer.rs:256-292, 491-516). The histogram leaves out the predicted token p; the
// weight of bin d is g(d) = max(1, (table[d] m) >> k) (max(1, table[d]) without a prediction,
// table[d] for a plain row), non-increasing in d, and every symbol with d >= zcut (table 0; a
// symbol's index is min(d, len - 1), so with zcut = len there are none) weighs g_rest = 1 (0
// for a plain row), counted as V - (p) - the binned symbols. Then
//   W' = sum_d cnt[d] g(d) + n_rest g_rest + w'[p],
//   sum_{j<tok} f = tok + sum_d cnt_lo[d] q(g(d)) + rest_lo q(g_rest) + [p < tok] q(w'[p]).
// The largest weight of the others is g of their smallest bin; the first symbol other than p
// whose weight reaches it (d <= dthr) comes from a pass that skips tiles by their max, and
// competes with w'[p] (the lower id on a tie).
__global__ __launch_bounds__(256) void k_coder_compact_mixed(CompactCoderArgs a) {
    extern __shared__ uint32_t hist[];
    __shared__ int64_t s_i[256];
    __shared__ uint64_t s_u[256];
    __shared__ uint64_t s_frac;
    const int row = blockIdx.x, tid = threadIdx.x;
    const int V = a.vocab, len = a.table_len, last = len - 1;
    const int zc = a.zcut;
    const bool packed = V < 65536;
    const uint16_t *d16 = a.d16 + (size_t)row * a.ld16;
    const int64_t *tm = a.tmax + (size_t)row * a.ntiles;
    const uint32_t kind = a.queries ? a.queries[2 * row] : 0;
    const uint32_t value = a.queries ? a.queries[2 * row + 1] : 0;
    const uint32_t tok = kind == 0 ? value : 0;
    const MixRec rec = a.mix[row];
    const bool plain = rec.p == MIX_PLAIN, none = rec.p == MIX_NONE, has_p = !plain && !none;
    const uint32_t p = has_p ? rec.p : 0xFFFFFFFFu;  // the host checked p < V
    const uint32_t mk = rec.k;
    const uint64_t mm = rec.m, wpm = rec.wp;
    auto g = [&](int d) -> uint64_t {  // table[d] <= 2^40 and m <= 2^16: the product fits u64
        const uint64_t w = a.table[d];
        if (plain) return w;
        if (none) return w > 1 ? w : 1;
        const uint64_t v = mk < 64 ? (w * mm) >> mk : 0;
        return v > 1 ? v : 1;
    };
    const uint64_t g_rest = plain ? 0 : 1;

    int64_t mx = INT64_MIN;
    for (int t = tid; t < a.ntiles; t += 256) mx = tm[t] > mx ? tm[t] : mx;
    const int64_t M = block_max64w(mx, s_i, tid);
    for (int d = tid; d < (packed ? zc : 2 * zc); d += 256) hist[d] = 0;
    __syncthreads();
    int64_t first = INT64_MAX;  // plain rows: the first symbol with weight table[0]
    // A symbol's index is min(d, last) (logits.rs:62-72): with a zero tail (zcut < len) every
    // d >= zcut is in the rest; else every d >= last counts in the last bin and no group skips.
    const bool tail0 = zc < len;
    for (int g0 = tid * 8; g0 < V; g0 += 4 * 256 * 8) {
        uint4 raw[4];
        int64_t b64[4];
        bool live[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int gq = g0 + u * 256 * 8;
            b64[u] = gq < V ? M - tm[gq >> 6] : (int64_t)zc;
            live[u] = gq < V && !(tail0 && b64[u] >= zc);
            if (live[u]) raw[u] = *(const uint4 *)(d16 + gq);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (!live[u]) continue;
            const int gq = g0 + u * 256 * 8, base = (int)(b64[u] < last ? b64[u] : last);
            const uint16_t *dv = (const uint16_t *)&raw[u];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int j = gq + q;
                const int dd = base + (int)dv[q] < last ? base + (int)dv[q] : last;
                if (j < V && dd < zc && (uint32_t)j != p) {
                    if (packed) {
                        atomicAdd(&hist[dd], (uint32_t)j < tok ? 0x10001u : 1u);
                    } else {
                        atomicAdd(&hist[dd], 1u);
                        if ((uint32_t)j < tok) atomicAdd(&hist[zc + dd], 1u);
                    }
                    if (dd <= a.d0 && j < first) first = j;
                }
            }
        }
    }
    __syncthreads();
    // the binned sums, the smallest bin in use
    uint64_t W = 0, n_in = 0, n_lo = 0;
    int64_t dmin = INT64_MAX;
    for (int d = tid; d < zc; d += 256) {
        const uint32_t h = hist[d];
        const uint32_t c = packed ? (h & 0xffffu) : h, clo = packed ? (h >> 16) : hist[zc + d];
        W += (uint64_t)c * g(d);
        n_in += c;
        n_lo += clo;
        if (c && d < dmin) dmin = d;
    }
    W = block_sum64w(W, s_u, tid);
    n_in = block_sum64w(n_in, s_u, tid);
    n_lo = block_sum64w(n_lo, s_u, tid);
    dmin = -block_max64w(-dmin, s_i, tid);
    const uint64_t n_rest = (uint64_t)V - (has_p ? 1 : 0) - n_in;
    const uint64_t rest_lo = (uint64_t)tok - (has_p && p < tok ? 1 : 0) - n_lo;
    W += n_rest * g_rest + (has_p ? wpm : 0);
    const uint64_t total = (uint64_t)1 << a.bits, spare = total - (uint64_t)V;
    if (tid == 0) s_frac = W >= ((uint64_t)1 << 32) ? coder_frac(spare, W) : 0;
    __syncthreads();
    const uint64_t frac = s_frac;

    // the largest weight (mixer weights are >= 1, so W' >= V and plain rows have W >= table[0])
    int64_t largest;
    if (plain) {
        largest = -block_max64w(-first, s_i, tid);
    } else {
        // gmax: the largest weight among the symbols other than p; dthr: the largest d with g(d)
        // >= gmax (a prefix, g is non-increasing); INT64_MAX when every index reaches it
        const uint64_t gmax = dmin != INT64_MAX ? g((int)dmin) : (n_rest ? g_rest : 0);
        int64_t dthr = -1;
        for (int d = tid; d < len; d += 256)
            if (g(d) >= gmax && d > dthr) dthr = d;
        dthr = block_max64w(dthr, s_i, tid);
        if (dthr == last) dthr = INT64_MAX;
        int64_t fo = INT64_MAX;  // the first symbol other than p with d <= dthr
        if (gmax) {
            for (int g0 = tid * 8; g0 < V; g0 += 256 * 8) {
                const int64_t base = M - tm[g0 >> 6];
                if (base > dthr) continue;  // every symbol of the tile has d >= base
                const uint4 raw = *(const uint4 *)(d16 + g0);
                const uint16_t *dv = (const uint16_t *)&raw;
                bool hit = false;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int j = g0 + q;
                    const int64_t dd = base + dv[q];
                    if (!hit && j < V && (uint32_t)j != p && (dd < last ? dd : last) <= dthr) {
                        fo = j;
                        hit = true;
                    }
                }
                if (hit) break;  // this thread's later symbols are larger
            }
        }
        fo = -block_max64w(-fo, s_i, tid);
        if (!has_p) largest = fo;
        else if (fo == INT64_MAX || wpm > gmax) largest = (int64_t)p;
        else if (wpm == gmax) largest = (int64_t)p < fo ? (int64_t)p : fo;
        else largest = fo;
    }

    uint64_t S = 0, Slo = 0;
    for (int d = tid; d < zc; d += 256) {
        const uint32_t h = hist[d];
        const uint32_t c = packed ? (h & 0xffffu) : h, clo = packed ? (h >> 16) : hist[zc + d];
        if (!c) continue;
        const uint64_t q = quotient(g(d), spare, W, frac);
        S += (uint64_t)c * q;
        Slo += (uint64_t)clo * q;
    }
    S = block_sum64w(S, s_u, tid);
    Slo = block_sum64w(Slo, s_u + 8, tid);
    const uint64_t q_rest = g_rest ? quotient(g_rest, spare, W, frac) : 0;
    S += n_rest * q_rest;
    Slo += rest_lo * q_rest;
    if (has_p) {
        const uint64_t qp = quotient(wpm, spare, W, frac);
        S += qp;
        if (p < tok) Slo += qp;
    }
    const uint64_t rem = total - ((uint64_t)V + S);
    uint64_t *out = a.intervals ? a.intervals + 3 * (size_t)row : nullptr;
    if (!out) return;
    auto weight = [&](int j, int64_t base_j, uint16_t dj) -> uint64_t {
        if ((uint32_t)j == p) return wpm;
        const int64_t dd = base_j + dj;
        return g((int)(dd < last ? dd : last));
    };
    if (kind == 0) {
        if (tid == 0) {
            const uint64_t f = 1 + quotient(weight((int)tok, M - tm[tok >> 6], d16[tok]), spare, W, frac);
            out[0] = tok;
            out[1] = (uint64_t)tok + Slo + ((int64_t)tok > largest ? rem : 0);
            out[2] = f + ((int64_t)tok == largest ? rem : 0);
        }
        return;
    }
    // Decode: the largest i with start_i <= target, in symbol order, 2048 symbols per step.
    const uint64_t target = value;
    uint64_t run = 0;
    int64_t cand = -1;
    uint64_t cstart = 0, cfreq = 0;
    for (int b = 0; b < V; b += 2048) {
        uint64_t f[8];
        uint64_t local = 0;
        const int j0 = b + tid * 8;
        if (j0 < V) {
            const uint4 raw = *(const uint4 *)(d16 + j0);
            const uint16_t *dv = (const uint16_t *)&raw;
            const int64_t base = M - tm[j0 >> 6];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int j = j0 + q;
                f[q] = 0;
                if (j < V) {
                    f[q] = 1 + quotient(weight(j, base, dv[q]), spare, W, frac) + (j == largest ? rem : 0);
                    local += f[q];
                }
            }
        }
        s_u[tid] = local;
        __syncthreads();
        if (tid == 0) {  // exclusive scan of the 256 partial sums, in order
            uint64_t acc = run;
            for (int t = 0; t < 256; t++) {
                const uint64_t v = s_u[t];
                s_u[t] = acc;
                acc += v;
            }
            s_i[0] = (int64_t)acc;
        }
        __syncthreads();
        uint64_t start = s_u[tid];
        const uint64_t next_run = (uint64_t)s_i[0];
        __syncthreads();
        if (j0 < V) {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int j = j0 + q;
                if (j >= V) break;
                if (start <= target) {
                    cand = j;
                    cstart = start;
                    cfreq = f[q];
                }
                start += f[q];
            }
        }
        run = next_run;
    }
    const int64_t best = block_max64(cand, s_i, tid);
    if (cand >= 0 && cand == best) {
        out[0] = (uint64_t)cand;
        out[1] = cstart;
        out[2] = cfreq;
    }
}

template <typename K>
static hipError_t launch_compact(K kernel, int threads, size_t extra, const CompactCoderArgs &a, int n_rows,
                                 hipStream_t stream) {
    if (n_rows <= 0) return hipSuccess;
    // packed counts: zcut bins and 64 spare bins of the weight-0 symbols; else two arrays;
    // rounded up to whole 16-byte words (the kernels clear them so), and `extra` bytes after them
    const size_t words = a.vocab < 65536 ? (size_t)a.zcut + 64 : 2 * (size_t)a.zcut;
    const size_t lds = sizeof(uint32_t) * ((words + 3) & ~(size_t)3) + extra;
    {
        const hipError_t e = allow_dynamic_lds((const void *)kernel, lds);
        if (e != hipSuccess) return e;
    }
    launch_k(kernel, dim3(n_rows), dim3(threads), lds, stream, a);
    return hipGetLastError();
}

// The reduction slots (three per wave) and the segment sums after the histogram.
constexpr size_t coder_extra(int nt, bool find) { return (size_t)(3 * nt / 64) * 8 + (find ? CODER_SEGS * 4 : 0); }
static_assert(2 * 4 * CODER_MAX_TABLE + coder_extra(1024, true) <= 160 * 1024, "LDS of one workgroup");

template <bool STATS, bool FIND, int NT>
static hipError_t launch_coder_compact_t(const CompactCoderArgs &a, int n_rows, hipStream_t stream) {
    const size_t extra = coder_extra(NT, FIND);
    return a.vocab < 65536 ? launch_compact(k_coder_compact<STATS, true, FIND, NT>, NT, extra, a, n_rows, stream)
                           : launch_compact(k_coder_compact<STATS, false, FIND, NT>, NT, extra, a, n_rows, stream);
}

hipError_t launch_coder_compact(const CompactCoderArgs &a, int n_rows, hipStream_t stream) {
    if (a.weights && n_rows > 0) {
        for (int r0 = 0; r0 < n_rows; r0 += 32768) {  // the grid's y dimension
            CompactCoderArgs c = a;
            c.d16 += (size_t)r0 * a.ld16;
            c.tmax += (size_t)r0 * a.ntiles;
            c.weights += (size_t)r0 * a.vocab;
            launch_k(k_weights_compact, dim3((a.vocab + 2047) / 2048, std::min(n_rows - r0, 32768)), dim3(256), 0,
                     stream, c);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    if (!a.intervals) return hipSuccess;
    // up to one row per CU: 1,024 threads a row (64 rows 18.0 -> 13.9 us, 42 -> 20 us with Decode
    // queries); past that four rows of 256 threads share a CU (383 rows 20.5 us against 26.5)
    if (n_rows <= 256) {
        return a.decode ? launch_coder_compact_t<false, true, 1024>(a, n_rows, stream)
                        : launch_coder_compact_t<false, false, 1024>(a, n_rows, stream);
    }
    return a.decode ? launch_coder_compact_t<false, true, 256>(a, n_rows, stream)
                    : launch_coder_compact_t<false, false, 256>(a, n_rows, stream);
}

hipError_t launch_mix_stats_compact(const CompactCoderArgs &a, int n_rows, hipStream_t stream) {
    if (!a.mix || !a.stats) return hipErrorInvalidValue;
    return launch_coder_compact_t<true, false, 256>(a, n_rows, stream);
}

hipError_t launch_coder_compact_mixed(const CompactCoderArgs &a, int n_rows, hipStream_t stream) {
    if (!a.mix) return hipErrorInvalidValue;
    return launch_compact(k_coder_compact_mixed, 256, 128, a, n_rows, stream);
}

// ---- kernel resources (CudaDevice::kernel_resources, crates/hardshell-cuda/src/device.rs:65-74) --
// The main kernels of the path with the registers, spill (private) bytes and static LDS bytes
// the compiler gave each.

int kernel_resources(KernelResource *out, int cap) {
    struct Entry {
        const char *name;
        const void *fn;
    };
    static const Entry table[] = {
        {"k_gemm<Act, narrow, 256x128>", (const void *)k_gemm<1, true, 128, true>},
        {"k_gemm<Residual, narrow, 256x128>", (const void *)k_gemm<2, true, 128, true>},
        {"k_gemm<Residual, narrow, 256x256>", (const void *)k_gemm<2, true, 256, true>},
        {"k_gemm<Gelu, narrow, 256x256>", (const void *)k_gemm<3, true, 256, true>},
        {"k_gemm<LogitsCompact, narrow, 256x128>", (const void *)k_gemm<5, true, 128, true>},
        {"k_gemm<Act, 256x128>", (const void *)k_gemm<1, false, 128, true>},
        {"k_gemm<Residual, 256x128>", (const void *)k_gemm<2, false, 128, true>},
        {"k_gemm<GeluWide, 256x128>", (const void *)k_gemm<6, false, 128, true>},
        {"k_gemm<GeluWide, narrow, 256x256>", (const void *)k_gemm<6, true, 256, true>},
        {"k_gemm<ResidualWide, narrow, 256x256>", (const void *)k_gemm<7, true, 256, true>},
        {"k_gemm<LogitsCompactWide, narrow, 256x128>", (const void *)k_gemm<9, true, 128, true>},
        {"k_gemm<Raw, split-K partials, 64x64>", (const void *)k_gemm<0, false, 64, true, 64>},
        {"k_gemm<Act, narrow, 128x192>", (const void *)k_gemm<1, true, 192, true, 128>},
        {"k_gemm<Residual, narrow, 128x192>", (const void *)k_gemm<2, true, 192, true, 128>},
        {"k_gemm<Act, narrow, 64x64>", (const void *)k_gemm<1, true, 64, true, 64>},
        {"k_gemm<Residual, narrow, 64x64>", (const void *)k_gemm<2, true, 64, true, 64>},
        {"k_gemm<Gelu, narrow, 64x64>", (const void *)k_gemm<3, true, 64, true, 64>},
        {"k_split_sum_raw", (const void *)k_split_sum_raw},
        {"k_embed", (const void *)k_embed},
        {"k_embed4", (const void *)k_embed4},
        {"k_layernorm", (const void *)k_layernorm},
        {"k_layernorm_rows<4>", (const void *)k_layernorm_rows<4>},
        {"k_layernorm_rows<8>", (const void *)k_layernorm_rows<8>},
        {"k_layernorm_rows4<12>", (const void *)k_layernorm_rows4<12>},
        {"k_layernorm_rows4<16>", (const void *)k_layernorm_rows4<16>},
        {"k_kv_store", (const void *)k_kv_store},
        {"k_attend", (const void *)k_attend},
        {"k_attend_short<4>", (const void *)k_attend_short<4>},
        {"k_attend_short<8>", (const void *)k_attend_short<8>},
        {"k_attend_long", (const void *)k_attend_long},
        {"k_attend_mfma<noclamp, lds table>", (const void *)k_attend_mfma<true, true, false>},
        {"k_attend_decode64<noclamp>", (const void *)k_attend_decode64<true>},
        {"k_attend_decode_wg<noclamp, 128>", (const void *)k_attend_decode_wg<true, 128>},
        {"k_attend_decode_wave<noclamp, 4, 64>", (const void *)k_attend_decode_wave<true, 4, 64>},
        {"k_split_dots<64>", (const void *)k_split_dots<64>},
        {"k_split_pv<noclamp, 64>", (const void *)k_split_pv<true, 64>},
        {"k_coder_compact", (const void *)k_coder_compact<false, true, false, 256>},
        {"k_coder_compact, few rows with Decode", (const void *)k_coder_compact<false, true, true, 1024>},
        {"k_weights_compact", (const void *)k_weights_compact},
        {"k_coder_compact_mixed", (const void *)k_coder_compact_mixed},
        {"k_read_bw", (const void *)k_read_bw},
    };
    const int n = (int)(sizeof(table) / sizeof(table[0]));
    for (int i = 0; i < n && i < cap; i++) {
        hipFuncAttributes at;
        const hipError_t e = hipFuncGetAttributes(&at, table[i].fn);
        if (e != hipSuccess) return -(int)e;
        out[i].name = table[i].name;
        out[i].regs = at.numRegs;
        out[i].private_bytes = (int)at.localSizeBytes;
        out[i].static_lds_bytes = (int)at.sharedSizeBytes;
    }
    return n;
}

}  // namespace hs
