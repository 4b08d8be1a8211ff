// fixed_registry.cpp -- lookup tables of the compiled fixed-plan and chirp-z
// kernels.
#include <mutex>
#include <vector>

#include "chirp.h"
#include "fixed.h"

namespace sfft {

static std::vector<FixedKernel> &registry() {
    static std::vector<FixedKernel> r;
    return r;
}
static std::mutex &registry_mutex() {
    static std::mutex m;
    return m;
}

void register_fixed(const FixedKernel &k) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    registry().push_back(k);
}

const FixedKernel *find_fixed(int n, int prec, int real, int variant) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    const int want = variant < 0 ? 0 : variant;
    for (const auto &k : registry())
        if (k.n == n && k.prec == prec && k.real == real && k.variant == want) return &k;
    return nullptr;
}

int fixed_variant_count(int n, int prec, int real) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    int c = 0;
    for (const auto &k : registry())
        if (k.n == n && k.prec == prec && k.real == real) ++c;
    return c;
}

static std::vector<ChirpKernel> &chirp_registry() {
    static std::vector<ChirpKernel> r;
    return r;
}

void register_chirp(const ChirpKernel &k) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    chirp_registry().push_back(k);
}

const ChirpKernel *find_chirp(size_t n, int prec) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    const ChirpKernel *best = nullptr;
    for (const auto &k : chirp_registry())
        if (k.part == kChirpWhole && k.prec == prec && (size_t)k.m + 1 >= 2 * n &&
            (!best || k.m < best->m))
            best = &k;
    return best;
}

bool find_chirp_split(size_t n, int prec, const ChirpKernel *&cols, const ChirpKernel *&rows) {
    std::lock_guard<std::mutex> lock(registry_mutex());
    size_t best = 0;
    cols = rows = nullptr;
    for (const auto &c : chirp_registry()) {
        if (c.part != kChirpCols || c.prec != prec) continue;
        for (const auto &r : chirp_registry()) {
            if (r.part != kChirpRows || r.prec != prec || r.m % c.tpw) continue;
            const size_t m = (size_t)c.m * (size_t)r.m;
            if (m + 1 < 2 * n) continue;
            if (best && (m > best || (m == best && c.m < cols->m))) continue;
            best = m;
            cols = &c;
            rows = &r;
        }
    }
    return best != 0;
}

}  // namespace sfft
