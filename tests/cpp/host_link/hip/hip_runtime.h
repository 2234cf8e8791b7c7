// The few runtime calls that HostLink makes, over host memory: a stream is a thread
// that runs its work in order, "device" memory is any other host memory.
#pragma once
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess, hipErrorInvalidValue, hipErrorOutOfMemory, hipErrorNotReady };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
struct hipPointerAttribute_t { hipMemoryType type; };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct StubModel {   // the model at work: its own allocations are not the product's
    StubModel();
    ~StubModel();
};

struct StubStream {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> work;
    size_t queued = 0, done = 0;
    bool stop = false;
    std::thread th{[this] {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            cv.wait(lk, [&] { return stop || !work.empty(); });
            if (work.empty()) return;
            auto f = std::move(work.front());
            work.pop_front();
            lk.unlock();
            f();
            lk.lock();
            ++done;
            cv.notify_all();
        }
    }};
    size_t push(std::function<void()> f)
    {
        StubModel m;
        std::lock_guard<std::mutex> lk(mu);
        work.push_back(std::move(f));
        cv.notify_all();
        return ++queued;
    }
    bool reached(size_t n)
    {
        std::lock_guard<std::mutex> lk(mu);
        return done >= n;
    }
    void wait(size_t n)
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return done >= n; });
    }
    ~StubStream()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        th.join();
    }
};
struct StubEvent { StubStream* st = nullptr; size_t at = 0; };
typedef StubStream* hipStream_t;
typedef StubEvent* hipEvent_t;

struct StubState {
    std::mutex mu;
    std::map<char*, size_t> pinned;
    bool refuse_host_malloc = false;
    size_t pinned_copies = 0, pageable_copies = 0;
    hipError_t last = hipSuccess;   // of the one calling thread
};
inline StubState& stub()
{
    static StubState s;
    return s;
}
inline bool stub_pinned(const void* p)
{
    std::lock_guard<std::mutex> lk(stub().mu);
    char* c = static_cast<char*>(const_cast<void*>(p));
    auto it = stub().pinned.upper_bound(c);
    if (it == stub().pinned.begin()) return false;
    --it;
    return c < it->first + it->second;
}
inline hipError_t stub_set(hipError_t e)
{
    if (e != hipSuccess) stub().last = e;
    return e;
}

inline hipError_t hipGetLastError()
{
    const hipError_t e = stub().last;
    stub().last = hipSuccess;
    return e;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    a->type = stub_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    StubModel m;
    if (stub().refuse_host_malloc) return stub_set(hipErrorOutOfMemory);
    *p = std::malloc(n);
    std::lock_guard<std::mutex> lk(stub().mu);
    stub().pinned[static_cast<char*>(*p)] = n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lk(stub().mu);
    if (!stub().pinned.erase(static_cast<char*>(p))) return hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    StubModel m;
    *e = new StubEvent;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st)
{
    e->st = st;
    e->at = st->push([] {});
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e)
{
    return !e->st || e->st->reached(e->at) ? hipSuccess : stub_set(hipErrorNotReady);
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (e->st) e->st->wait(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st)
{
    st->wait(st->push([] {}));
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st)
{
    const bool pinned = stub_pinned(kind == hipMemcpyHostToDevice ? s : d);
    StubModel m;
    const size_t at = st->push([=] { std::memcpy(d, s, n); });
    ++(pinned ? stub().pinned_copies : stub().pageable_copies);
    if (!pinned) st->wait(at);   // the runtime's copy of pageable memory blocks
    return hipSuccess;
}
