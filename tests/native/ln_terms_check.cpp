// Host build of the 64-bit LayerNorm row terms and the single-precision element rule
// (taco_amd/csrc/intmath.h: ln_terms_small, ln_elem_z with ln_margin) against __int128 arithmetic:
// rows at the edges of the domain, beta with and without a fraction, quotients on and beside a
// half. Prints "ok <n>" or the first mismatch and exits 1.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../taco_amd/csrc/intmath.h"

using hs::i128;
using hs::u128;

static uint64_t st = 0x7E57;
static uint64_t next() {  // splitmix64
    uint64_t z = (st += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

static i128 floor_div(i128 a, i128 b) {  // b > 0
    const i128 q = a / b;
    return a % b < 0 ? q - 1 : q;
}

int main() {
    long count = 0, taken = 0;
    const int32_t L = 1 << 24;
    for (int i = 0; i < 20000; i++) {
        const int n = (next() & 3) ? 4 * (1 + (int)(next() % 512)) : 2048;
        std::vector<int32_t> x(n);
        const int mode = (int)(next() % 5);
        const uint32_t span = 1 + (uint32_t)(next() >> (39 + next() % 25));  // up to 2^25
        const int32_t base = (int32_t)(next() % (2 * (uint64_t)L + 1)) - L;
        for (int j = 0; j < n; j++) {
            int64_t v;
            if (mode == 0) v = base;                                            // constant
            else if (mode == 1) v = (next() & 1) ? L : -L;                      // the bound
            else if (mode == 2) v = j == 0 ? L : base / 16;                     // an outlier
            else v = base / 2 + (int64_t)(next() % span) - span / 2;
            x[j] = (int32_t)(v > L ? L : (v < -L ? -L : v));
        }
        int64_t sum = 0;
        uint64_t Q = 0;
        for (int32_t v : x) sum += v, Q += (uint64_t)((int64_t)v * v);
        const uint32_t k = (next() & 3) ? 48 : (uint32_t)(next() % 49), j = (next() & 3) ? 8 : (uint32_t)(next() % 17);
        const uint64_t eps = (next() & 1) ? 1ull << 43 : 1 + (next() >> (next() % 64));
        const hs::LnTerms t = hs::ln_terms_small(sum, Q, n, 1.0 / (double)n, k, j, eps);
        count++;
        if (!t.ok) continue;
        taken++;
        const i128 mean = floor_div(sum, n);
        i128 sq = 0;
        for (int32_t v : x) sq += ((i128)v - mean) * ((i128)v - mean);
        const uint64_t inv = hs::ln_inv((u128)sq, (uint32_t)n, k, j, eps);
        if ((i128)t.mean != mean || t.inv != inv) {
            std::printf("ln_terms_small n %d mode %d k %u j %u: mean %d inv %u, want %lld %llu\n", n, mode, k, j,
                        t.mean, t.inv, (long long)mean, (unsigned long long)inv);
            return 1;
        }
    }
    if (taken < count / 2) {
        std::printf("ln_terms_small declined too often (%ld of %ld)\n", count - taken, count);
        return 1;
    }
    // the element rule: beta in units of 2^-f, |beta| <= B 2^f with the margin of that B
    long kept = 0, elems = 0;
    auto elem = [&](int64_t p, uint32_t s, int32_t beta, uint32_t f, float B) -> bool {
        // p = c inv gamma m as c = 1 or -1, inv = |p|: k = float(inv 2^-s)
        const int32_t c = p < 0 ? -1 : 1;
        const float kf = (float)std::ldexp((double)(p < 0 ? -p : p), -(int)s);
        const float z = hs::ln_elem_z(c, kf, 128.0f + (float)beta * std::ldexp(1.0f, -(int)f));
        elems++;
        if (std::fabs(hs::ln_half_dist(z)) < hs::ln_margin(B)) return true;
        kept++;
        const i128 v = (i128)p + ((i128)beta << (s - f)) + (s ? (i128)1 << (s - 1) : 0);
        i128 want = v >> s;
        want = want < -127 ? -127 : (want > 127 ? 127 : want);
        return (i128)((int32_t)std::rint(z) - 128) == want;
    };
    for (int i = 0; i < 2000000; i++) {
        const uint32_t f = (next() & 1) ? 8 : 0, s = 8 + (uint32_t)(next() % 50);
        const float B = (next() & 1) ? 16.0f : 256.0f;
        const int32_t lim = (int32_t)B << f, beta = (int32_t)(next() % (2 * (uint64_t)lim + 1)) - lim;
        int64_t p = (int64_t)(next() >> (1 + next() % 40));
        if (s < 54) p %= (int64_t)1 << (s + 9);
        if (next() & 1) {  // on or beside a half of X + beta
            const int64_t q = (int64_t)(next() % 512) - 256;
            const i128 v = ((i128)q << s) - ((i128)beta << (s - f)) + ((i128)1 << (s - 1)) + (int64_t)(next() % 5) - 2;
            if (v < ((i128)1 << 62) && v > -((i128)1 << 62)) p = (int64_t)v;
        }
        if (next() & 1) p = -p;
        if (!elem(p, s, beta, f, B)) {
            std::printf("ln_elem_z p %lld s %u beta %d f %u\n", (long long)p, s, beta, f);
            return 1;
        }
        count++;
    }
    if (kept < elems / 4) {
        std::printf("ln_elem_z declined too often\n");
        return 1;
    }
    // rescale_wide47 against the i128 rule: |v| < 2^47, shifts 16 .. 62, on and beside rounding steps
    for (int i = 0; i < 1000000; i++) {
        const uint32_t s = 16 + (uint32_t)(next() % 47);
        int64_t v = (int64_t)(next() >> (17 + next() % 46));
        int32_t m = (int32_t)(uint32_t)next();
        if (i % 16 == 0) v = (1ll << 47) - 1;
        if (i % 16 == 1) m = INT32_MIN;
        if (i % 16 == 2) m = 1, v = ((1ll << (s < 47 ? s : 46)) >> 1) + (int64_t)(next() % 3) - 1;
        if (next() & 1) v = -v;
        if ((i128)hs::rescale_wide47(v, m, s) != hs::rescale_full(v, m, s)) {
            std::printf("rescale_wide47 v %lld m %d s %u\n", (long long)v, m, s);
            return 1;
        }
        count++;
    }
    std::printf("ok %ld (terms %ld, elements %ld of %ld)\n", count, taken, kept, elems);
    return 0;
}
