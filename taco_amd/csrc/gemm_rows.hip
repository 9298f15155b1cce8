// The linear layers of passes with few rows (decode passes, small folds): int8 MFMA products
// whose operands go from memory straight into registers.
//
// What bounds these products is latency, not bytes or MFMAs: a 256-row c_attn of GPT-2 small holds
// 2.6 MB of operands and 0.9 GOP, well under 1 us of either, while a tile that streams K through
// LDS pays a load round trip, a barrier and an LDS read for every k-step. Here the waves of a
// workgroup take the k-steps of its tile in turn (wave w: steps w, w + WAVES, ..), so a wave has
// all of its few loads in flight at once, the partial tiles meet once in LDS (i32 sums, exact in
// any order), and the epilogue's rule runs on the total. The panels of 64 bytes of K hold an MFMA
// fragment (16 rows x 64 bytes) as 1 KiB of contiguous memory in exactly the order the lanes need
// it, so nothing is gained by staging operands in LDS; the row tiles that share columns of W
// re-read them through the caches.
#include "intmath.h"
#include "launch.h"

namespace hs {

// One output row x 4 columns from the exact product `acc`, with the epilogue rule of the fused
// kernels. A whole group of 4 columns whose destination is 4-byte aligned (16-byte for the i32
// outputs) is stored with one access. `bias`, `mult`, `x` (the residual row's 4 values) and `ri`
// (the row's slot and position) were loaded before the product.
struct RowsEpi {
    v4i bias, mult, x, wsum;
    RowInfo ri;
};

template <int EPI>
__device__ __forceinline__ RowsEpi rows_epi_load(const GemmArgs &g, int m, int n4) {
    RowsEpi p{};
    if constexpr (EPI == (int)Epi::Raw) return p;
    if (g.params_padded) {
        p.bias = *(const v4i *)(g.bias + n4);
        p.mult = *(const v4i *)(g.mult + n4);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int n = n4 + e < g.n ? n4 + e : g.n - 1;
            p.bias[e] = g.bias[n];
            p.mult[e] = g.mult[n];
        }
    }
    constexpr bool WIDE = EPI == (int)Epi::ResidualWide;
    const int rows = WIDE ? g.rows : g.m, mc = m < rows ? m : rows - 1;
    if constexpr (WIDE) {
#pragma unroll
        for (int e = 0; e < 4; e++) p.wsum[e] = g.wsum[n4 + e < g.n ? n4 + e : g.n - 1];
    }
    if constexpr (EPI == (int)Epi::Residual || WIDE) {
        const int32_t *x = (const int32_t *)g.out + (size_t)mc * g.ldo + n4;
        if (n4 + 4 <= g.n && ((uintptr_t)x & 15) == 0) {
            p.x = *(const v4i *)x;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n4 + e < g.n) p.x[e] = x[e];
        }
    }
    if constexpr (EPI == (int)Epi::Act) {
        if (g.kv_rows) p.ri = g.kv_rows[mc];
    }
    return p;
}

template <int EPI>
__device__ __forceinline__ void rows_epi(const GemmArgs &g, int m, int n4, const v4i &acc, const v4i &lo,
                                         const RowsEpi &p) {
    constexpr bool WIDE = EPI == (int)Epi::ResidualWide;  // acc and lo: the planes' products
    if (m >= (WIDE ? g.rows : g.m) || n4 >= g.n) return;
    const int cnt = g.n - n4 < 4 ? g.n - n4 : 4;
    if (EPI == (int)Epi::Raw) {
        int32_t *o = (int32_t *)g.out + (size_t)m * g.ldo + n4;
        if (cnt == 4 && ((uintptr_t)o & 15) == 0) *(v4i *)o = acc;
        else
            for (int e = 0; e < cnt; e++) o[e] = acc[e];
        return;
    }
    // rescale(a + bias, mult, shift) (int.rs:63-67): |a + bias| < 2^32, exact in i64
    int64_t r[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if constexpr (WIDE) {  // dot = 256 hi + lo + 128 wsum (below 2^39)
            const int64_t v = (int64_t)acc[e] * 256 + lo[e] + 128 * (int64_t)p.wsum[e] + p.bias[e];
            r[e] = g.shift >= 16 && g.shift <= 62
                       ? rescale_wide47(v, p.mult[e], (uint32_t)g.shift)
                       : clamp128(rescale_full(v, p.mult[e], (uint32_t)g.shift), INT32_MIN, INT32_MAX);
        } else {
            r[e] = rescale_small((int64_t)acc[e] + p.bias[e], p.mult[e], (uint32_t)g.shift);
        }
    }
    if (EPI == (int)Epi::Residual || WIDE) {  // ops.rs:131-145: x = clamp(x + sat32(r), +-R)
        int32_t *x = (int32_t *)g.out + (size_t)m * g.ldo + n4;
        v4i v;
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] = (int32_t)clamp64((int64_t)p.x[e] + clamp64(r[e], INT32_MIN, INT32_MAX), -RES, RES);
        if (cnt == 4 && ((uintptr_t)x & 15) == 0) *(v4i *)x = v;
        else
            for (int e = 0; e < cnt; e++) x[e] = v[e];
        return;
    }
    uint32_t b[4];  // the i8 outputs (GeluWide: the i16 values)
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (EPI == (int)Epi::Act) {  // ops.rs:123-130
            b[e] = (uint32_t)clamp64(r[e], -127, 127);
        } else {  // table[clamp(r, -off, off - 1) + off] (ops.rs:146-154, gelu.rs:58-62)
            const int t = (int)clamp64(r[e], -g.gelu_off, g.gelu_off - 1) + g.gelu_off;
            b[e] = EPI == (int)Epi::Gelu ? (uint32_t)g.gelu[t] : (uint32_t)g.gelu16[t];
        }
    }
    auto store4 = [&](int8_t *o, auto byte) {
        if (cnt == 4 && ((uintptr_t)o & 3) == 0) {
            *(uint32_t *)o = (byte(0) & 255) | ((byte(1) & 255) << 8) | ((byte(2) & 255) << 16) | ((byte(3) & 255) << 24);
        } else {
            for (int e = 0; e < cnt; e++) o[e] = (int8_t)byte(e);
        }
    };
    if (EPI == (int)Epi::Act) {
        if (g.kv_rows && n4 >= g.kv_d) {
            // K or V of the row into the cache: kv_d and kv_hd are multiples of 4, so the group
            // lies in one head of one part; the columns past 3 kv_d are padding
            if (n4 >= 3 * g.kv_d) return;
            const int part = n4 >= 2 * g.kv_d, c = n4 - (part + 1) * g.kv_d;
            const int hh = c / g.kv_hd, cc = c - hh * g.kv_hd;
            store4((part ? g.vc : g.kc) + (((size_t)p.ri.slot * g.kv_h + hh) * g.kv_ctx + p.ri.pos) * g.kv_hd + cc,
                   [&](int e) { return b[e]; });
        } else {
            store4((int8_t *)g.out + (size_t)m * g.ldo + n4, [&](int e) { return b[e]; });
        }
    } else if (EPI == (int)Epi::Gelu) {  // the operand of the next product, in panels
        store4((int8_t *)g.out + panel_off(m, n4, g.out_rows), [&](int e) { return b[e]; });
    } else {  // GeluWide: the two planes of each i16 output, hi = v >> 8, lo = (v & 255) - 128
        store4((int8_t *)g.out + panel_off(plane_row(m, 0), n4, g.out_rows),
               [&](int e) { return (uint32_t)((int32_t)(int16_t)b[e] >> 8); });
        store4((int8_t *)g.out + panel_off(plane_row(m, 1), n4, g.out_rows),
               [&](int e) { return (uint32_t)(((int32_t)(int16_t)b[e] & 255) - 128); });
    }
}

// A workgroup computes 16 MT rows x 16 NT columns; its WAVES waves split the k-steps of 64. A wave
// keeps U k-steps of fragments in flight: (MT + NT) U 16-byte registers per lane.
template <int EPI, int MT, int NT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_rows(GemmArgs g) {
    constexpr int U = MT + NT <= 3 ? 6 : 4, TILES = MT * NT;
    // the wide product: row tiles 2 i and 2 i + 1 hold the planes of the same 16 rows (plane_row)
    constexpr int PL = EPI == (int)Epi::ResidualWide ? 2 : 1, OUTS = TILES / PL, TPW = (OUTS + WAVES - 1) / WAVES;
    static_assert(MT % PL == 0, "whole plane pairs");
    __shared__ __attribute__((aligned(16))) v4i red[WAVES][TILES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup L runs on XCD L % 8: XCD x takes the x-th contiguous chunk of the tiles, row tiles
    // innermost, so the row tiles of a column block read its W from one L2.
    int mt, nt;
    {
        const int gm = (g.m + 16 * MT - 1) / (16 * MT);
        const int T = gridDim.x, L = blockIdx.x, x = L & 7, k = L >> 3;
        const int q = T >> 3, r = T & 7;
        const int p = x * q + (x < r ? x : r) + k;
        nt = p / gm;
        mt = p - nt * gm;
    }
    const int m0 = mt * 16 * MT, n0 = nt * 16 * NT;
    const int nk = g.k_pad / GEMM_BK;
    const int steps = wave < nk ? (nk - wave + WAVES - 1) / WAVES : 0;  // this wave's k-steps

    // The epilogue's operands of the tiles this wave finishes (tile wave + t WAVES of the
    // workgroup): lane l holds row 16 i + l % 16, columns 16 j + 4 (l / 16) ..
    RowsEpi ep[TPW];
    auto tile_m = [&](int t) { return m0 / PL + 16 * (t / NT) + (lane & 15); };
    auto tile_n = [&](int t) { return n0 + 16 * (t % NT) + 4 * (lane >> 4); };
    // fragment loads: lane l reads row l % 16, bytes 16 (l / 16) .. of a 16 x 64 block
    const size_t pa = (size_t)g.a_rows * 64, pw = (size_t)g.w_rows * 64;  // bytes per panel
    const uint32_t lane_off = (uint32_t)((lane & 15) * 64 + (lane >> 4) * 16);
    const int8_t *ab = g.a + (size_t)m0 * 64 + lane_off, *wb = g.w + (size_t)n0 * 64 + lane_off;
    v4i fa[U][MT], fw[U][NT], acc[MT][NT];
    auto load = [&](int u, int s) {  // step s of this wave (clamped by the caller) into slot u
        const size_t ks = (size_t)(wave + s * WAVES);
#pragma unroll
        for (int j = 0; j < NT; j++) fw[u][j] = *(const v4i *)(wb + ks * pw + j * 1024);
#pragma unroll
        for (int i = 0; i < MT; i++) fa[u][i] = *(const v4i *)(ab + ks * pa + i * 1024);
    };
    auto mul = [&](int u) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[u][j], fa[u][i], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = v4i{0, 0, 0, 0};
    if (steps > 0) {
        // every load is unconditional, from a clamped step: a wait then counts exactly its own loads
#pragma unroll
        for (int u = 0; u < U; u++) load(u, u < steps ? u : steps - 1);
#pragma unroll
        for (int t = 0; t < TPW; t++) {
            const int tile = wave + t * WAVES;
            if (tile < OUTS) ep[t] = rows_epi_load<EPI>(g, tile_m(tile), tile_n(tile));
        }
        int s = 0;
        for (; s + U < steps; s += U) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                mul(u);
                load(u, s + u + U < steps ? s + u + U : steps - 1);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < steps) mul(u);
    } else {
#pragma unroll
        for (int t = 0; t < TPW; t++) {
            const int tile = wave + t * WAVES;
            if (tile < OUTS) ep[t] = rows_epi_load<EPI>(g, tile_m(tile), tile_n(tile));
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) red[wave][i * NT + j][lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        const int tile = wave + t * WAVES;
        if (tile >= OUTS) break;
        const int src = PL == 2 ? (tile / NT) * 2 * NT + tile % NT : tile;
        v4i sum = red[0][src][lane], lo = v4i{0, 0, 0, 0};
#pragma unroll
        for (int w = 1; w < WAVES; w++) sum += red[w][src][lane];
        if constexpr (PL == 2) {
#pragma unroll
            for (int w = 0; w < WAVES; w++) lo += red[w][src + NT][lane];
        }
        rows_epi<EPI>(g, tile_m(tile), tile_n(tile), sum, lo, ep[t]);
    }
}

template <int EPI, int MT, int NT, int WAVES>
static hipError_t launch_rows_t(const GemmArgs &g, hipStream_t stream) {
    const int gm = (g.m + 16 * MT - 1) / (16 * MT), gn = (g.n + 16 * NT - 1) / (16 * NT);
    launch_k((k_gemm_rows<EPI, MT, NT, WAVES>), dim3(gm * gn), dim3(64 * WAVES), 0, stream, g);
    return hipGetLastError();
}

// The tile of a product, or no tile (mt 0) where the LDS-tiled k_gemm is the better one. A tile is
// as good as the CUs it keeps busy: up to one workgroup per CU (256) the time hardly grows with
// the tiles (a product of one row or of 64 x 768 x 768 takes 3.1-3.2 us, the launch itself),
// so the smallest tile that needs at most 256 workgroups wins, and larger tiles (fewer bytes per
// output) where it needs more. Measured against what served these products before (us a launch,
// weights from the Infinity Cache; m x n x k):
//   Act       1 x 2304 x 768    5.1 -> 3.4      Residual   1 x 768 x 3072    8.5 -> 3.9
//            64 x 2304 x 768    5.2 -> 4.0               64 x 768 x 3072     9.4 -> 4.0
//           128 x 4096 x 1024   6.4 -> 4.9              256 x 1024 x 1024    7.6 -> 3.8
//           256 x 2304 x 768    5.4 (5.9 here: stays)   256 x 1024 x 4096   10.9 -> 6.7
//            64 x 6400 x 1600   8.2 -> 6.5              512 x 1600 x 6400   25   -> 17
// Two rounds of 32 x 32 tiles still beat 64 x 64 LDS tiles for K up to 2,048 (128 x 2304 x 768
// 5.3 -> 4.8), three only where k_gemm's epilogue is a slow one (the residual one: 1024 x 768 x 768
// 7.2 -> 6.3; the one for products without the i32 bound: 256 x 2304 x 768 8.2 -> 5.9); past that
// the loads per output decide and k_gemm is faster. With longer K the 64-row tiles take over at one
// round (512 x 768 x 3072: 12.8 -> 8.2). What needs more than one round of those takes the 64 x 64 LDS
// tiles (512 x 4096 x 6400, two slices of K and a summing pass before: 35 -> 29).
struct RowsTile {
    int mt = 0, nt = 0;
};

static RowsTile rows_tile(Epi epi, const GemmArgs &g) {
    const int m = g.m, n = g.n, k_pad = g.k_pad;
    auto tiles = [&](int mt, int nt) {
        return ((m + 16 * mt - 1) / (16 * mt)) * (long long)((n + 16 * nt - 1) / (16 * nt));
    };
    if (epi != Epi::ResidualWide) {  // (its row tiles come in pairs)
        if (tiles(1, 1) <= 256) return {1, 1};
        if (m <= 16) return {1, 2};
    }
    if (tiles(2, 1) <= 256) return {2, 1};
    const bool narrow = epi != Epi::Residual && epi != Epi::ResidualWide && g.fast32 && g.shift >= 31;
    const long long most = k_pad > 2048 ? 256 : narrow ? 512 : 768;
    if (tiles(2, 2) <= most) return {2, 2};
    if (k_pad > 2048 && tiles(4, 2) <= 256) return {4, 2};
    if (k_pad > 2048 && tiles(4, 4) <= 256) return {4, 4};
    return {};
}

template <int EPI>
static hipError_t launch_rows_e(const GemmArgs &g, const RowsTile &t, hipStream_t stream) {
    // four waves share a tile's k-steps; eight for the 64 x 64 tiles, whose waves hold the most
    if constexpr (EPI != (int)Epi::ResidualWide)
        if (t.mt == 1) return t.nt == 1 ? launch_rows_t<EPI, 1, 1, 4>(g, stream) : launch_rows_t<EPI, 1, 2, 4>(g, stream);
    if (t.mt == 2) return t.nt == 1 ? launch_rows_t<EPI, 2, 1, 4>(g, stream) : launch_rows_t<EPI, 2, 2, 4>(g, stream);
    return t.nt == 2 ? launch_rows_t<EPI, 4, 2, 4>(g, stream) : launch_rows_t<EPI, 4, 4, 8>(g, stream);
}

bool gemm_rows_fits(Epi epi, const GemmArgs &g) {
    const bool ok = epi == Epi::Raw || epi == Epi::Act || epi == Epi::Residual || epi == Epi::Gelu ||
                    epi == Epi::GeluWide || epi == Epi::ResidualWide;
    return ok && rows_tile(epi, g).mt > 0;
}

hipError_t launch_gemm_rows(Epi epi, const GemmArgs &g, hipStream_t stream) {
    const RowsTile t = rows_tile(epi, g);
    if (!t.mt) return hipErrorInvalidValue;
    switch (epi) {
        case Epi::Raw: return launch_rows_e<0>(g, t, stream);
        case Epi::Act: return launch_rows_e<1>(g, t, stream);
        case Epi::Residual: return launch_rows_e<2>(g, t, stream);
        case Epi::Gelu: return launch_rows_e<3>(g, t, stream);
        case Epi::GeluWide: return launch_rows_e<6>(g, t, stream);
        case Epi::ResidualWide: return launch_rows_e<7>(g, t, stream);
        default: return hipErrorInvalidValue;
    }
}

// ---- The LM head of few rows, compact logits (LogitsCompact) -------------------------------------
// What bounds it is wte (39 MB at width 768: 8 us at 5 TB/s), once every column block is read once
// and ahead of its use: the 256 x 128 tiles of k_gemm compute 256 rows for one and wait at every
// k-step. Here the rows' A goes to LDS once, in fragment order (lane l's 16 bytes at 16 l: no bank
// conflicts), and each wave takes 16 columns over all of K with U k-steps of W in flight in
// registers. Every wave holding A from the caches instead read 4 bytes of it for each byte of W:
// 18.6 us at 64 rows. A row's tile max meets over the 4 waves of a 64-column tile in LDS.
// Measured against the tiles of k_gemm, us a launch of the head alone, wte in the Infinity Cache (inside a
// token step 16.1 -> 9.6 us, inside a 64-row decode pass 20.3 -> 14.6): width 768 1 row 15.8 -> 8.2, 16 rows 15.9 -> 8.5,
// 32 rows 16.5 -> 9.6, 64 rows 17.6 -> 12.2; width 1024 1 row 19.0 -> 11.2, 64 rows 20.5 -> 15.6;
// width 1600 1 row 29.3 -> 17.3, 64 rows 31.3 -> 22.2. 128 rows (128 accumulated rows a wave): 20.3 ->
// 19.5 at width 768 but 32.9 -> 41 at 1600, so more than 64 rows stay with the tiles.
template <int MT, bool NARROW, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_head_rows(GemmArgs g) {
    constexpr int U = 12;
    extern __shared__ __align__(16) char s_a[];  // the rows' A: [k-step][16-row tile][lane][16 B]
    using L = typename std::conditional<NARROW, int32_t, int64_t>::type;
    constexpr L LMIN = NARROW ? (L)INT32_MIN : (L)INT64_MIN;
    __shared__ L s_max[WAVES][16 * MT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * 16 * WAVES;
    const int steps = g.k_pad / GEMM_BK;
    const size_t pa = (size_t)g.a_rows * 64, pw = (size_t)g.w_rows * 64;  // bytes per panel
    const uint32_t lane_off = (uint32_t)((lane & 15) * 64 + (lane >> 4) * 16);
    const int8_t *ab = g.a + lane_off, *wb = g.w + (size_t)(n0 + 16 * wave) * 64 + lane_off;
    v4i fw[U], acc[MT];
    auto load = [&](int u, int s) { fw[u] = *(const v4i *)(wb + (size_t)s * pw); };
    auto mul = [&](int u, int s) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const v4i f = *(const v4i *)(s_a + ((s * MT + i) * 64 + lane) * 16);
            acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[u], f, acc[i], 0, 0, 0);
        }
    };
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < U; u++) load(u, u < steps ? u : steps - 1);
    for (int c = wave; c < steps * MT; c += WAVES)
        __builtin_amdgcn_global_load_lds((const void *)(ab + (size_t)(c / MT) * pa + (c % MT) * 1024),
                                         (lds_void *)(s_a + c * 1024), 16, 0, 0);
    wait_vmcnt<0>();  // this wave's part landed (the barrier shows it to all)
    lds_barrier();
    // the lane's 4 columns (n4 is below n_pad: the multipliers are padded)
    const int n4 = n0 + 16 * wave + 4 * (lane >> 4);
    const v4i mult = *(const v4i *)(g.mult + n4);
    int s = 0;
    for (; s + U < steps; s += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            mul(u, s + u);
            load(u, s + u + U < steps ? s + u + U : steps - 1);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
        if (s + u < steps) mul(u, s + u);
    // logit = clamp(rescale(acc, m, s), +-2^40) (ops.rs:229-234): |acc m| < 2^62; NARROW (shift 31
    // or more): an i32
    const int s_eff = g.shift < 63 ? g.shift : 63;
    const int64_t half = s_eff ? (int64_t)1 << (s_eff - 1) : 0;
    L l[MT][4];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        L mx = LMIN;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t r = ((int64_t)acc[i][e] * mult[e] + half) >> s_eff;
            l[i][e] = n4 + e < g.n ? (NARROW ? (L)r : (L)clamp64(r, -((int64_t)1 << 40), (int64_t)1 << 40)) : LMIN;
            mx = l[i][e] > mx ? l[i][e] : mx;
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) {  // the 4 lanes of a row
            const L u = __shfl_xor(mx, o, 64);
            mx = u > mx ? u : mx;
        }
        if (lane < 16) s_max[wave][16 * i + lane] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int m = 16 * i + (lane & 15);
        const int w0 = wave & ~3;  // the 4 waves of a 64-column tile
        L mx = s_max[w0][m];
#pragma unroll
        for (int w = 1; w < 4; w++) mx = s_max[w0 + w][m] > mx ? s_max[w0 + w][m] : mx;
        if (m >= g.m || n0 + 16 * w0 >= g.n) continue;
        if (wave == w0 && lane < 16) g.tmax[(size_t)m * g.tmax_ld + n0 / 64 + w0 / 4] = (int64_t)mx;
        // distances capped as the fused epilogue caps them: 65535 (NARROW), else cap16
        uint16_t d[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (NARROW) {
                const uint32_t u = (uint32_t)mx - (uint32_t)l[i][e];
                d[e] = (uint16_t)(u < 65535u ? u : 65535u);
            } else {
                const int64_t u = (int64_t)mx - (int64_t)l[i][e];
                d[e] = (uint16_t)(u < g.cap16 ? u : g.cap16);
            }
        }
        uint16_t *o = (uint16_t *)g.out + (size_t)m * g.ldo + n4;
        if (n4 + 4 <= g.n) {
            *(uint2 *)o = make_uint2(d[0] | ((uint32_t)d[1] << 16), d[2] | ((uint32_t)d[3] << 16));
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n4 + e < g.n) o[e] = d[e];
        }
    }
}

// Up to 64 rows whose A fits in LDS beside the row maxima, 8-byte output groups, padded multipliers.
// (launch_gemm has checked that the panels hold 256 rows and round_up(n, 256) columns: a workgroup
// reads 16 MT of the rows and at most 256 columns.)
static int head_tiles(const GemmArgs &g) { return g.m <= 16 ? 1 : g.m <= 32 ? 2 : 4; }
static size_t head_lds(const GemmArgs &g) { return (size_t)g.k_pad * 16 * head_tiles(g); }

bool head_rows_fits(const GemmArgs &g) {
    return g.m <= 64 && head_lds(g) <= (size_t)144 * 1024 && g.params_padded && g.ldo % 4 == 0 &&
           ((uintptr_t)g.out & 7) == 0;
}

template <int MT, int WAVES>
static hipError_t head_rows_run(const GemmArgs &g, hipStream_t stream) {
    auto run = [&](auto kernel) {
        const size_t lds = head_lds(g);
        const hipError_t e = allow_dynamic_lds((const void *)kernel, lds);
        if (e != hipSuccess) return e;
        launch_k(kernel, dim3((g.n + 16 * WAVES - 1) / (16 * WAVES)), dim3(64 * WAVES), lds, stream, g);
        return hipGetLastError();
    };
    return g.shift >= 31 ? run(k_head_rows<MT, true, WAVES>) : run(k_head_rows<MT, false, WAVES>);
}

// 8 waves a workgroup while two or more fit a CU's LDS, else 16: 16 waves of one workgroup read W
// as two of 8 would (64 rows at width 1600: 27.0 us with 8 waves, 22.2 with 16; at width 768 12.2 and
// 13.3).
hipError_t launch_head_rows(const GemmArgs &g, hipStream_t stream) {
    const int mt = head_tiles(g);
    if (head_lds(g) <= (size_t)64 * 1024) {
        return mt == 1 ? head_rows_run<1, 8>(g, stream) : mt == 2 ? head_rows_run<2, 8>(g, stream)
                                                                  : head_rows_run<4, 8>(g, stream);
    }
    return mt == 1 ? head_rows_run<1, 16>(g, stream) : mt == 2 ? head_rows_run<2, 16>(g, stream)
                                                               : head_rows_run<4, 16>(g, stream);
}

}  // namespace hs
