// HostLink (csrc/pm_xfer.cpp) over the runtime model in hip/hip_runtime.h: one check
// by name, exit status 0 if it holds.
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <ctime>
#include <memory>
#include <string>
#include <vector>

#include "pm_xfer.h"

using hp3d::HostLink;
typedef std::vector<unsigned char> Bytes;

static uint32_t rng_state = 12345;
static uint32_t rnd() { return rng_state = rng_state * 1664525u + 1013904223u, rng_state >> 8; }
static Bytes noise(size_t n)
{
    Bytes b(n);
    for (size_t i = 0; i < n; ++i) b[i] = (unsigned char)(i * 2654435761u >> 13 ^ i / 251);
    return b;
}

#define CHECK(c)                                                            \
    do {                                                                    \
        if (!(c)) {                                                         \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);             \
            return false;                                                   \
        }                                                                   \
    } while (0)

static bool both_ways(HostLink& link, hipStream_t st, size_t n)
{
    const Bytes src = noise(n);
    Bytes dev(n), dst(n + 2);
    const size_t half = n / 2;
    unsigned char* from = const_cast<unsigned char*>(src.data());
    CHECK(link.upload({{from, dev.data(), half}, {from + half, dev.data() + half, n - half}}, st) == hipSuccess);
    CHECK(hipStreamSynchronize(st) == hipSuccess);
    CHECK(dev == src);
    std::fill(dev.begin(), dev.end(), 0);
    CHECK(link.upload({{from, dev.data(), n}}, st) == hipSuccess);
    CHECK(hipStreamSynchronize(st) == hipSuccess);
    CHECK(dev == src);
    CHECK(link.download({{dst.data() + 1, dev.data(), n}}, st) == hipSuccess);
    CHECK(std::memcmp(dst.data() + 1, src.data(), n) == 0 && !dst[0] && !dst[n + 1]);
    CHECK(hipGetLastError() == hipSuccess);   // no query's answer left behind
    return true;
}

// The lines of the present layout: 1 MiB pieces, copies by the calling thread alone up
// to 3 MiB, pieces of 2 MiB from 4, of 4 from 24, one turn of the ring at 32.
static bool sizes()
{
    HostLink link;
    StubStream st;
    const size_t M = 1 << 20;
    for (size_t line : {M, 2 * M, 3 * M, 4 * M, 24 * M, 32 * M, 64 * M})
        for (size_t n : {line - 1, line, line + 1}) CHECK(both_ways(link, &st, n));
    for (size_t n : {(size_t)1, (size_t)63, (size_t)257}) CHECK(both_ways(link, &st, n));
    link.close();
    return both_ways(link, &st, 5 * M + 3);   // opened again
}

// One segment below 24 MiB goes up by the runtime's copy, without the ring; from there
// on, and two segments, through it.
static bool lone()
{
    HostLink link;
    StubStream st;
    const size_t line = 24u << 20;
    Bytes src = noise(line), dev(line);
    const auto up = [&](size_t a, size_t b) {
        std::fill(dev.begin(), dev.end(), 0);
        stub().pinned_copies = stub().pageable_copies = 0;
        const HostLink::Seg segs[] = {{src.data(), dev.data(), a}, {src.data() + a, dev.data() + a, b}};
        return link.upload(segs, b ? 2 : 1, &st) == hipSuccess && hipStreamSynchronize(&st) == hipSuccess &&
               std::memcmp(dev.data(), src.data(), a + b) == 0;
    };
    CHECK(up(1, 0) && stub().pageable_copies == 1 && stub().pinned_copies == 0);
    CHECK(up(line - 1, 0) && stub().pageable_copies == 1 && stub().pinned_copies == 0);
    CHECK(up(line, 0) && stub().pageable_copies == 0 && stub().pinned_copies == 6);
    CHECK(up(100, 200) && stub().pageable_copies == 0 && stub().pinned_copies == 1);
    return true;
}

// Many odd segments, adjacent on the device or not, more of them to a piece than it has
// places for, some page-locked, some empty.
static bool parts()
{
    HostLink link;
    StubStream st;
    for (int round = 0; round < 40; ++round) {
        const int n = 1 + rnd() % 60;
        const size_t big = round % 4 == 3 ? 300000 : 700;
        Bytes dev;
        std::vector<size_t> size(n), off(n);
        for (int i = 0; i < n; ++i) {
            size[i] = rnd() % 8 ? 1 + rnd() % big : 0;
            off[i] = dev.size() + (rnd() % 5 == 0 ? rnd() % 9 : 0);
            dev.resize(off[i] + size[i]);
        }
        const Bytes image = noise(dev.size());
        std::vector<Bytes> host(n);
        std::vector<unsigned char*> ptr(n);
        std::vector<void*> locked;
        std::vector<HostLink::Seg> segs;
        for (int i = 0; i < n; ++i) {
            if (rnd() % 6 == 0) {
                void* p;
                CHECK(hipHostMalloc(&p, size[i] + 1, 0) == hipSuccess);
                locked.push_back(p);
                ptr[i] = static_cast<unsigned char*>(p);
            } else {
                host[i].resize(size[i] + 1);
                ptr[i] = host[i].data();
            }
            ptr[i][size[i]] = 77;
            segs.push_back({ptr[i], dev.data() + off[i], size[i]});
        }
        std::memcpy(dev.data(), image.data(), dev.size());
        CHECK(link.download(segs, &st) == hipSuccess && hipStreamSynchronize(&st) == hipSuccess);
        for (int i = 0; i < n; ++i)
            CHECK(std::memcmp(ptr[i], image.data() + off[i], size[i]) == 0 && ptr[i][size[i]] == 77);
        std::fill(dev.begin(), dev.end(), 0);
        CHECK(link.upload(segs, &st) == hipSuccess && hipStreamSynchronize(&st) == hipSuccess);
        for (int i = 0; i < n; ++i)
            CHECK(std::memcmp(dev.data() + off[i], image.data() + off[i], size[i]) == 0);
        for (void* p : locked) (void)hipHostFree(p);
    }
    return true;
}

// Without page-locked memory to be had, the runtime's own copies.
static bool no_ring()
{
    HostLink link;
    StubStream st;
    stub().refuse_host_malloc = true;
    for (size_t n : {(size_t)1, (size_t)(3 << 20) + 1, (size_t)(33 << 20) + 5}) CHECK(both_ways(link, &st, n));
    CHECK(stub().pinned_copies == 0 && stub().pageable_copies > 0);
    stub().refuse_host_malloc = false;
    CHECK(both_ways(link, &st, 5 << 20));
    CHECK(stub().pinned_copies > 0);
    return true;
}

// Without heap memory for the lists likewise, and no exception leaves.
static bool refuse_new = false;
static bool no_heap()
{
    HostLink link;
    StubStream st;
    const size_t n = 100000;
    const Bytes src = noise(n);
    Bytes dev(n), a(n / 2), b(n - n / 2);
    CHECK(both_ways(link, &st, 9 << 20));
    HostLink bare;   // no ring, no threads, no lists yet
    for (HostLink* l : {&link, &bare}) {
        for (size_t upto = 0; upto < 2; ++upto) {
            unsigned char* from = const_cast<unsigned char*>(src.data());
            const HostLink::Seg up[] = {{from, dev.data(), 1}, {from + 1, dev.data() + 1, n - 1}};
            const HostLink::Seg down[] = {{a.data(), dev.data(), n / 2},
                                          {b.data(), dev.data() + n / 2, n - n / 2}};
            std::fill(a.begin(), a.end(), 0);
            refuse_new = true;
            const bool ok = l->upload(up, 2, &st) == hipSuccess && l->download(down, 2, &st) == hipSuccess;
            refuse_new = false;
            CHECK(ok);
            CHECK(std::memcmp(a.data(), src.data(), n / 2) == 0);
            CHECK(std::memcmp(b.data(), src.data() + n / 2, n - n / 2) == 0);
        }
    }
    return true;
}
// (only the calling thread's allocations are refused, not the model's streams')
static const std::thread::id main_thread = std::this_thread::get_id();
static thread_local int in_model = 0;
StubModel::StubModel() { ++in_model; }
StubModel::~StubModel() { --in_model; }
void* operator new(size_t n)
{
    if (refuse_new && !in_model && std::this_thread::get_id() == main_thread) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// An upload of more than the ring holds, behind a second of other work on its stream:
// the copy threads sleep meanwhile.
static bool sleeps()
{
    HostLink link;
    StubStream st;
    const size_t n = 64u << 20;
    CHECK(both_ways(link, &st, n));   // threads made, pages touched
    const Bytes src = noise(n);
    Bytes dev(n, 1);
    bool slept = true;
    for (int again = 0; again < 2; ++again) {   // the second begins with slots in flight
        st.push([] { std::this_thread::sleep_for(std::chrono::seconds(1)); });
        const std::clock_t t0 = std::clock();   // processor time of all threads
        CHECK(link.upload({{const_cast<unsigned char*>(src.data()), dev.data(), n}}, &st) == hipSuccess);
        const double cpu = double(std::clock() - t0) / CLOCKS_PER_SEC;
        std::printf("processor time %.3f s\n", cpu);
        slept = slept && cpu < 0.5;   // a thread that never sleeps takes a second
    }
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(hipStreamSynchronize(&st) == hipSuccess);
    CHECK(slept);
    CHECK(dev == src);
    return true;
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    const bool ok = what == "sizes" ? sizes() : what == "parts" ? parts() : what == "lone" ? lone() : what == "no_ring" ? no_ring()
                    : what == "no_heap" ? no_heap()
                    : what == "sleeps" ? sleeps() : false;
    std::puts(ok ? "ok" : "failed");
    return ok ? 0 : 1;
}
