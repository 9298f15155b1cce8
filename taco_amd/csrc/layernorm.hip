// LayerNorm with 8-bit outputs (layernorm.rs:66-108,188-256): the row's mean and scale in 64-bit
// arithmetic, the elements in single precision, each proved exact or declined (intmath.h), and the
// integer rule for what is declined.
//
// Two costs bound it: for decode passes the chain of one row (loads, reductions, the row terms,
// the elements: nothing else runs), for folds the VALU work of about 50 elements a lane on top
// of reading x once. So each wave works alone (no LDS, no barrier: its compute overlaps other
// waves' loads), LPR lanes share a row (64, or 32 for many narrow rows), the reductions run on DPP
// moves, and a row whose values are all within 2^24 (the residual stream
// of a model stays far below) takes ln_terms_small, about 90 instructions where the 128-bit
// form of the larger rows takes 700.
#include "intmath.h"
#include "launch.h"

namespace hs {

// NG groups of 4 columns per lane (d % 4 == 0, d <= 4 NG LPR). Every load of x is unconditional,
// from a clamped address (a row past n_rows reads the last row, a column past d the last group;
// neither value is used).
template <int NG, int LPR>
__global__ __launch_bounds__(64) void k_layernorm_f32(LnArgs a, int n_rows) {
    constexpr int RPW = 64 / LPR;  // rows per wave (a workgroup is one wave)
    const int lane = threadIdx.x, q = lane & (LPR - 1);
    const int row = blockIdx.x * RPW + lane / LPR;
    const bool live = row < n_rows;
    const int d = a.d;
    const int rc = live ? row : n_rows - 1;
    const int32_t *x = a.x + (size_t)(a.src ? a.src[rc] : rc) * d;
    auto col = [&](int t) { return 4 * (q + LPR * t); };
    v4i xv[NG];
#pragma unroll
    for (int t = 0; t < NG; t++) xv[t] = *(const v4i *)(x + (col(t) < d ? col(t) : d - 4));
    typedef float v4f __attribute__((ext_vector_type(4)));
    v4f gv[NG], bv[NG];  // gamma and 128 + beta as floats, loaded under x
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = col(t) < d ? col(t) : d - 4;
        gv[t] = *(const v4f *)(a.gf + j);
        bv[t] = *(const v4f *)(a.bf + j);
    }
    int64_t sum = 0;
    uint64_t Q = 0;
    int32_t mx = INT32_MIN, mn = INT32_MAX;
#pragma unroll
    for (int t = 0; t < NG; t++) {
        if (col(t) >= d) continue;
        const v4i v = xv[t];
        // (sums of four and of squares wrap only for rows that the test below refuses)
        sum += (int32_t)((uint32_t)v[0] + (uint32_t)v[1] + (uint32_t)v[2] + (uint32_t)v[3]);
#pragma unroll
        for (int e = 0; e < 4; e++) Q += (uint64_t)((int64_t)v[e] * v[e]);
        mx = max(max(max(v[0], v[1]), max(v[2], v[3])), mx);
        mn = min(min(min(v[0], v[1]), min(v[2], v[3])), mn);
    }
    butterfly<LPR>([&](auto st) {
        constexpr int S = decltype(st)::value;
        sum += lane_move64<S>(sum);
        Q += (uint64_t)lane_move64<S>((int64_t)Q);
        mx = max(mx, lane_move<S>(mx));
        mn = min(mn, lane_move<S>(mn));
    });
    const double inv_d = a.inv_d;
    int64_t mean;
    uint64_t inv;
    uint32_t redo = 0;  // bit t: group t takes the integer rule
    {
        const LnTerms t = ln_terms_small(sum, Q, d, inv_d, (uint32_t)a.k, (uint32_t)a.j, a.eps);
        mean = t.mean;
        inv = t.inv;
        if (__any(live && !(t.ok && mx <= (1 << 24) && mn >= -(1 << 24)))) {
            // a row outside the 64-bit terms: all rows of the wave by the 128-bit form (x again
            // from memory, so that the registers above stay what the usual case needs)
            uint64_t lo = 0, hi = 0;
            sum = 0;
#pragma unroll 1
            for (int j = 4 * q; j < d; j += 4 * LPR) {
                const v4i v = *(const v4i *)(x + j);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    sum += v[e];
                    const uint64_t p = (uint64_t)((int64_t)v[e] * v[e]);
                    lo += p;
                    hi += lo < p;
                }
            }
            butterfly<LPR>([&](auto st) {
                constexpr int S = decltype(st)::value;
                sum += lane_move64<S>(sum);
                const uint64_t lo2 = (uint64_t)lane_move64<S>((int64_t)lo);
                const uint64_t hi2 = (uint64_t)lane_move64<S>((int64_t)hi);
                lo += lo2;
                hi += hi2 + (lo < lo2);
            });
            mean = floor_div_est(sum, d, inv_d);
            const u128 sq = (u128)((i128)(((u128)hi << 64) | lo) - 2 * (i128)mean * sum + (i128)d * mean * mean);
            inv = ln_inv_est(sq, (uint32_t)d, (uint32_t)a.k, (uint32_t)a.j, a.eps, inv_d);
        }
    }
    if (!live) return;
    const double kr = (double)inv * a.mk;  // inv m 2^-s
    const float krf = (float)kr;
    const int32_t mean32 = (int32_t)mean;  // |x|, |mean| < 2^30, so x - mean fits i32
    auto at = [&](int j) { return (uint32_t *)(a.out + panel_off(row, j, a.out_rows)); };
#pragma unroll
    for (int t = 0; t < NG; t++) {
        const int j = col(t);
        if (j >= d) continue;
        const v4f g4 = gv[t], b4 = bv[t];
        uint32_t packed = 0;
        float near = 1.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float z = ln_elem_z(xv[t][e] - mean32, krf * g4[e], b4[e]);
            near = fminf(near, fabsf(ln_half_dist(z)));
            packed = __builtin_amdgcn_cvt_pk_u8_f32(z, e, packed);  // to nearest
        }
        if (near < a.margin) {
            // an element too near a half: the group in double precision, whose error is below
            // 2^-20 for |v| <= 2^30 (ln_elem_f64; b4 - 127.5 = 1/2 + beta is exact)
            packed = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const double v = fma((double)(xv[t][e] - mean32) * kr, (double)g4[e], (double)b4[e] - 127.5);
                const double f = __builtin_floor(v), r = v - f;
                if (!(fabs(v) <= 0x1p30 && r >= 0x1p-20 && r <= 1.0 - 0x1p-20)) redo |= 1u << t;
                const double c = fmin(fmax(f, -127.0), 127.0);
                packed |= ((uint32_t)(int32_t)c + 128u) << (8 * e);
            }
        }
        *at(j) = packed ^ 0x80808080u;  // 4 bytes from j % 4 == 0: one panel
    }
    // the integer rule, group by group (x again from memory)
    if (redo) {
        const int64_t c1 = (int64_t)mx - mean, c2 = mean - (int64_t)mn;
        const uint64_t cmax = (uint64_t)(c1 > c2 ? c1 : c2);
        const bool small = (u128)cmax * inv < ((u128)1 << 63);
#pragma unroll 1
        while (redo) {
            const int t = __builtin_ctz(redo);
            redo &= redo - 1;
            const int j = col(t);
            const v4i v = *(const v4i *)(x + j);
            uint32_t packed = 0;
#pragma unroll 1
            for (int e = 0; e < 4; e++) {
                const int64_t c = (int64_t)v[e] - mean;
                const i128 cinv = small ? (i128)(c * (int64_t)inv) : (i128)c * (i128)(u128)inv;
                const i128 p = cinv * (i128)a.gm[j + e];
                const i128 y = a.beta_frac == 0
                                   ? shift_round128(p, a.s, 126) + (i128)a.beta[j + e]
                                   : shift_round128(p + ((i128)a.beta[j + e] << (a.s - a.beta_frac)), a.s, 126);
                packed |= (uint32_t)(uint8_t)(int8_t)clamp128(y, -127, 127) << (8 * e);
            }
            *at(j) = packed;
        }
    }
}

bool layernorm_f32_fits(const LnArgs &a) { return a.gf && a.bits == 8 && a.d % 4 == 0 && a.d <= 2048; }

// One-wave workgroups, a row each (nothing is shared, and workgroups of four waves measured the same
// or slower). Against the kernels that served these rows before, us a launch of the op alone, its
// operands still in the caches: 768 columns, 1 row 5.6 -> 2.7, 256 rows 6.0 -> 4.4, 3,400 10.6 -> 7.0,
// 16,384 21.2 -> 15.7; 1,024 columns, 24,576 rows 48.6 -> 24.6; 1,600 columns, 6,600 rows 27.1 -> 14.9.
// Inside a fold, 16,384 rows of 768 take 16 to 18 us (63 MB: 3.5 to 3.9 TB/s). Two rows a wave
// are better only where a row leaves lanes idle and there are many (384 columns, 24,576 rows:
// 14.1 against 17.9); four rows a wave, the earlier split, nowhere (768 columns, 16,384 rows 18.2).
hipError_t launch_layernorm_f32(const LnArgs &a, int n_rows, hipStream_t stream) {
    auto run = [&](auto kernel, int rows_per_wave) {
        launch_k(kernel, dim3((n_rows + rows_per_wave - 1) / rows_per_wave), dim3(64), 0, stream, a, n_rows);
        return hipGetLastError();
    };
    if (a.d <= 512) return n_rows <= 4096 ? run(k_layernorm_f32<2, 64>, 1) : run(k_layernorm_f32<4, 32>, 2);
    if (a.d <= 768) return run(k_layernorm_f32<3, 64>, 1);
    if (a.d <= 1024) return run(k_layernorm_f32<4, 64>, 1);
    return run(k_layernorm_f32<8, 64>, 1);
}

}  // namespace hs
