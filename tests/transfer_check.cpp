// Host-side check of the copies of glac_amd/csrc/transfer.hpp, built by tests/test_transfer_route.py against
// tests/host_hip: which arrays travel through the pinned slices and which the runtime copies by itself, and that
// the bytes arrive, also when no memory is left on the host (a C entry cannot pass an exception on).  Prints
// "ok <case>" per case, exits non-zero on the first violation.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../glac_amd/csrc/transfer.hpp"

using namespace glacx;

// While `no_memory` is set every allocation fails.
static bool no_memory = false;
void *operator new(std::size_t n)
{
    void *p = no_memory ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

#define REQUIRE(cond)                                                          \
    do {                                                                       \
        if (!(cond)) {                                                         \
            std::printf("FAIL %s:%d (%s): %s\n", __FILE__, __LINE__, name, #cond); \
            std::exit(1);                                                      \
        }                                                                      \
    } while (0)

constexpr int kArrays = 4;

struct Case {
    const char *name;
    size_t bytes;                  // of each array
    unsigned known;                // bit k: the runtime knows array k
    hipMemoryType type;            // as what
    bool no_pinned, unknown_is_error;
    unsigned sliced;               // bit k: array k goes through the slices
};

static void check(const Case &c, bool up, bool starved)
{
    const char *name = c.name;
    std::vector<char> host[kArrays], dev((size_t)kArrays * c.bytes);
    for (int k = 0; k < kArrays; k++) {
        host[k].resize(c.bytes);
        for (size_t i = 0; i < c.bytes; i++) {
            const char v = (char)(i * 31 + i / 1021 + k * 7 + up);
            (up ? host[k][i] : dev[k * c.bytes + i]) = v;
        }
    }
    rt.n = rt.syncs = rt.n_known = 0;
    rt.slices = nullptr;
    rt.slice_bytes = 0;
    rt.known_type = c.type;
    rt.no_pinned = c.no_pinned;
    rt.unknown_is_error = c.unknown_is_error;
    std::vector<HostSpan> spans;
    for (int k = 0; k < kArrays; k++) {
        if (c.known >> k & 1) rt.known[rt.n_known++] = host[k].data();
        spans.push_back({host[k].data(), dev.data() + k * c.bytes, c.bytes});
    }
    {
        Transfer t;
        no_memory = starved;
        bool thrown = false;
        hipError_t e = hipSuccess;
        try {
            e = t.run(spans.data(), (int)spans.size(), up, 0, nullptr);
        } catch (...) {
            thrown = true;
        }
        no_memory = false;
        REQUIRE(!thrown && e == hipSuccess);
        for (int k = 0; k < kArrays; k++) {
            size_t direct = 0;
            for (int i = 0; i < rt.n; i++) {
                const char *at = up ? rt.copies[i].src : rt.copies[i].dst;
                if (at >= host[k].data() && at < host[k].data() + c.bytes) direct += rt.copies[i].bytes;
            }
            REQUIRE(direct == (c.sliced >> k & 1 ? 0 : c.bytes));
        }
        if (!up) REQUIRE(rt.syncs > 0);  // complete on return
        REQUIRE(hipGetLastError() == hipSuccess);
    }
    for (int k = 0; k < kArrays; k++) REQUIRE(std::memcmp(host[k].data(), dev.data() + k * c.bytes, c.bytes) == 0);
    std::printf("ok %s %s%s\n", name, up ? "up" : "down", starved ? " starved" : "");
}

int main()
{
    constexpr size_t mib = (size_t)1 << 20, large = 9 * mib + 4097 * 8;
    const Case cases[] = {
        {"ordinary", large, 0, hipMemoryTypeHost, false, false, 0xF},
        {"ordinary_error", large, 0, hipMemoryTypeHost, false, true, 0xF},
        {"small", mib, 0, hipMemoryTypeHost, false, false, 0},
        {"no_slices", large, 0, hipMemoryTypeHost, true, false, 0},
        {"pinned", large, 0xF, hipMemoryTypeHost, false, false, 0},
        {"managed", large, 0xF, hipMemoryTypeManaged, false, false, 0},
        {"device", large, 0xF, hipMemoryTypeDevice, false, true, 0},
        {"mixed", large, 0x5, hipMemoryTypeHost, false, false, 0xA},
    };
    for (const Case &c : cases)
        for (const bool up : {true, false})
            for (const bool starved : {false, true}) check(c, up, starved);
    return 0;
}
