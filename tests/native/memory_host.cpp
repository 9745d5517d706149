// The context's device allocations over a counted stand-in memory: what the context counts is what it holds, and that stays
// within its budget.  Exit status 0, or a message and 3.
#include "device_stub.hpp"

#include <random>

#include "bh_internal.hpp"

extern "C" {

hipError_t hipMalloc(void** p, size_t n) {
    *p = std::malloc(1);  // an address
    stub::mem[*p] = n;
    stub::held += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    const auto it = stub::mem.find(p);
    stub::check(it != stub::mem.end(), "hipFree: not a block");
    stub::held -= it->second;
    stub::mem.erase(it);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t*) { return hipErrorUnknown; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t*, int) { return hipErrorUnknown; }

}  // extern "C"

static constexpr size_t MB = size_t(1) << 20;

static void same(const bh_ctx* c) {
    stub::check(c->used + c->spare_bytes + c->scratch_bytes == stub::held, "counted bytes differ from the bytes held");
    stub::check(stub::held <= c->budget, "over the budget");
}

// sectors of shrinking size, each released before the next: a kept block must not pass for a smaller one
static void shrinking() {
    bh_ctx* c = nullptr;
    stub::check(bh_ctx_create(0, 1024 * MB, &c) == BH_OK, "context");
    void* p = nullptr;
    for (size_t mb : {250, 170, 115, 78, 53, 36, 33}) {
        stub::check(bh_dev_alloc(c, &p, mb * MB) == BH_OK, "allocation");
        same(c);
        bh_dev_free(c, p, mb * MB);
        same(c);
    }
    // a block of the same size is the kept one
    stub::check(bh_dev_alloc(c, &p, 80 * MB) == BH_OK, "allocation");
    void* first = p;
    bh_dev_free(c, p, 80 * MB);
    stub::check(bh_dev_alloc(c, &p, 80 * MB) == BH_OK && p == first, "the kept block is reused");
    same(c);
    bh_dev_free(c, p, 80 * MB);
    bh_ctx_destroy(c);
    stub::check(stub::held == 0, "memory left behind");
}

// blocks and builders' scratch in any order, sizes that repeat and that lie close together
static void mixed(unsigned seed) {
    bh_ctx* c = nullptr;
    stub::check(bh_ctx_create(0, 600 * MB, &c) == BH_OK, "context");
    std::mt19937 rng(seed);
    const size_t sizes[] = {MB, 31 * MB, 32 * MB, 40 * MB, 48 * MB, 60 * MB, 64 * MB, 65 * MB, 90 * MB, 128 * MB, 192 * MB, 256 * MB, 300 * MB};
    std::vector<std::pair<void*, size_t>> held;
    for (int i = 0; i < 4000; ++i) {
        const size_t n = sizes[rng() % (sizeof(sizes) / sizeof(sizes[0]))];
        const unsigned what = rng() % 4;
        if (what < 2) {
            size_t live = 0;
            for (const auto& h : held) live += h.second;
            void* p = nullptr;
            const int rc = bh_dev_alloc(c, &p, n);
            stub::check(rc == (live + n <= 600 * MB ? BH_OK : BH_EBUDGET), "kept memory stands in the way of an allocation that fits");
            if (rc == BH_OK) held.push_back({p, n});
        } else if (what == 2 && !held.empty()) {
            std::swap(held[rng() % held.size()], held.back());
            bh_dev_free(c, held.back().first, held.back().second);
            held.pop_back();
        } else {
            BhScratch s;
            if (s.open(c, n) == BH_OK) same(c);
        }
        same(c);
    }
    for (const auto& h : held) bh_dev_free(c, h.first, h.second);
    stub::check(c->used == 0, "bytes counted for no block");
    bh_ctx_destroy(c);
    stub::check(stub::held == 0, "memory left behind");
}

int main() {
    shrinking();
    for (unsigned seed = 1; seed <= 8; ++seed) mixed(seed);
    std::puts("ok");
    return 0;
}
