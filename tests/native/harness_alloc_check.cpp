// tc_fold_blocks after an allocation that failed: the harness (taco/harness.cpp) is linked with a
// stand-in backend and an operator new that can fail once. The call that fails throws; the next
// call on the same thread must hand the backend arrays that hold its rows. argv[1]: how many of the
// row arrays are allocated before the one that fails. Prints "ok".
#include <cstdio>
#include <cstdlib>
#include <map>
#include <new>
#include <string>
#include <vector>

#include "common.h"
#include "hardshell_hip.h"
#include "taco_hip.h"

static std::map<const void *, size_t, std::less<const void *>> *g_blocks;  // the large allocations that live
static long g_fail_after = -1;  // large allocations that succeed before one fails (-1: none fails)
constexpr size_t LARGE = 1 << 14;

void *operator new(size_t n) {
    if (n >= LARGE && g_fail_after >= 0 && g_fail_after-- == 0) throw std::bad_alloc();
    void *p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    if (n >= LARGE && g_blocks) {
        auto *b = g_blocks;
        g_blocks = nullptr;
        (*b)[p] = n;
        g_blocks = b;
    }
    return p;
}
void operator delete(void *p) noexcept {
    if (g_blocks && p) {
        auto *b = g_blocks;
        g_blocks = nullptr;
        b->erase(p);
        g_blocks = b;
    }
    std::free(p);
}
void operator delete(void *p, size_t) noexcept { operator delete(p); }

namespace hs {
hs_status fail(hs_status s, int, const std::string &) { return s; }
void clear_error() {}
void sha256(const uint8_t *, size_t, uint8_t[32]) {}
}  // namespace hs

static bool g_bad = false;
static void holds(const void *p, size_t bytes, const char *what) {
    auto it = g_blocks->find(p);
    if (it != g_blocks->end() && it->second >= bytes) return;
    std::printf("the %s do not hold %zu bytes\n", what, bytes);
    g_bad = true;
}

extern "C" {
const hs_model *hs_batch_model(const hs_batch *) { return nullptr; }
void hs_batch_reset(hs_batch *, size_t) {}
hs_status hs_batch_set_overlap(hs_batch *, uint32_t) { return HS_OK; }
size_t hs_batch_slots(const hs_batch *) { return 4; }
uint32_t hs_model_eot(const hs_model *) { return 0; }
uint32_t hs_model_n_ctx(const hs_model *) { return 4096; }
uint32_t hs_model_vocab(const hs_model *) { return 2; }
void hs_model_hash(const hs_model *, uint8_t[32]) {}
hs_status hs_model_token(const hs_model *, uint32_t, const uint8_t **, size_t *) { return HS_OK; }
size_t hs_model_merges(const hs_model *, const uint32_t **) { return 0; }
hs_status hs_batch_run_coded(hs_batch *, const hs_input *in, const hs_query *q, size_t n, uint32_t,
                             hs_interval *out) {
    holds(in, n * sizeof *in, "inputs");
    holds(q, n * sizeof *q, "queries");
    holds(out, n * sizeof *out, "answers");
    if (g_bad) std::exit(1);  // before anything writes through them
    for (size_t i = 0; i < n; i++) out[i] = hs_interval{q[i].value, 0, 1ull << 31};
    return HS_OK;
}
}

int main(int argc, char **argv) {
    g_blocks = new std::map<const void *, size_t, std::less<const void *>>();
    std::vector<uint32_t> tokens(8192, 1);
    const size_t offsets[3] = {0, 4096, 8192};
    std::vector<uint8_t> out(1 << 20);
    size_t lens[2];
    auto fold = [&] {
        return tc_fold_blocks((hs_batch *)&tokens, 0, tokens.data(), offsets, 2, nullptr, out.data(), out.size(), lens);
    };
    g_fail_after = argc > 1 ? std::atol(argv[1]) : 0;
    bool threw = false;
    try {
        fold();
    } catch (const std::bad_alloc &) {
        threw = true;
    }
    if (!threw) {
        std::printf("no allocation failed\n");
        return 1;
    }
    g_fail_after = -1;
    if (fold() != HS_OK) return 1;
    std::printf("ok\n");
    return 0;
}
