// pm_xfer.cpp -- see pm_xfer.h.
#include "pm_xfer.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <new>
#include <system_error>
#include <utility>

namespace hp3d {

namespace {

// Whether the runtime knows the host memory (page-locked, managed): the link
// reaches it without a slot.
bool known_to_runtime(const void* p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // an answer here, not an error
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

bool HostLink::overlap(const Seg* segs, size_t n)
{
    if (n < 2) return false;
    std::vector<std::pair<const char*, size_t>> r;
    for (size_t i = 0; i < n; ++i) r.emplace_back(static_cast<const char*>(segs[i].host), segs[i].bytes);
    std::sort(r.begin(), r.end());
    for (size_t i = 1; i < r.size(); ++i)
        if (r[i - 1].first + r[i - 1].second > r[i].first) return true;
    return false;
}

bool HostLink::open()
{
    if (ring_) return true;
    void* p = nullptr;
    if (hipHostMalloc(&p, kSlots * kSlotBytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    for (int k = 0; k < kSlots; ++k)
        if (hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            while (k-- > 0) (void)hipEventDestroy(ev_[k]);
            (void)hipHostFree(p);
            return false;
        }
    ring_ = static_cast<char*>(p);
    return true;
}

void HostLink::start_workers()
{
    if (!workers_.empty()) return;
    const int n = std::max(1, std::min(kMaxWorkers, (int)std::thread::hardware_concurrency() / 2));
    try {
        for (int k = 0; k < n; ++k) workers_.emplace_back([this] { worker(); });
    } catch (const std::system_error&) {
        // fewer, or none: the calling thread copies too
    } catch (const std::bad_alloc&) {
    }
}

void HostLink::close()
{
    {
        std::lock_guard<std::mutex> lk(mu_);
        stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : workers_) t.join();
    workers_.clear();
    stop_ = false;
    if (!ring_) return;
    for (int k = 0; k < kSlots; ++k) {
        (void)slot_ready(k);
        (void)hipEventDestroy(ev_[k]);
        ev_[k] = nullptr;
    }
    (void)hipHostFree(ring_);
    ring_ = nullptr;
}

// The pieces of the segments in pageable memory; the others are copied here.
hipError_t HostLink::split(const Seg* segs, size_t n, bool to_host, hipStream_t st)
{
    pieces_.clear();
    size_t total = 0;
    std::vector<const Seg*> mine;
    for (size_t i = 0; i < n; ++i) {
        const Seg& s = segs[i];
        if (!s.bytes) continue;
        if (known_to_runtime(s.host)) {
            const hipError_t e =
                to_host ? hipMemcpyAsync(s.host, s.dev, s.bytes, hipMemcpyDeviceToHost, st)
                        : hipMemcpyAsync(s.dev, s.host, s.bytes, hipMemcpyHostToDevice, st);
            if (e != hipSuccess) return e;
        } else {
            mine.push_back(&s);
            total += s.bytes;
        }
    }
    const size_t chunk = piece_bytes(total);
    alone_ = total <= kAloneBytes;
    for (const Seg* s : mine) {
        char* host = static_cast<char*>(s->host);
        char* dev = static_cast<char*>(s->dev);
        for (size_t at = 0; at < s->bytes;) {
            Piece* p = pieces_.empty() ? nullptr : &pieces_.back();
            if (!p || p->dev + p->bytes != dev + at || p->bytes >= chunk || p->parts == kMaxParts) {
                pieces_.emplace_back();
                p = &pieces_.back();
                p->dev = dev + at;
            }
            const size_t share = std::min(s->bytes - at, chunk - p->bytes);
            p->part[p->parts++] = {host + at, p->bytes, share};
            p->bytes += share;
            at += share;
        }
    }
    return hipSuccess;
}

// The copies by the runtime alone, in order: where there is no memory for the ring,
// page-locked, or for the lists.
hipError_t HostLink::plain(const Seg* segs, size_t n, bool to_host, hipStream_t st)
{
    for (const Seg* s = segs; s != segs + n; ++s) {
        if (!s->bytes) continue;
        const hipError_t e =
            to_host ? hipMemcpyAsync(s->host, s->dev, s->bytes, hipMemcpyDeviceToHost, st)
                    : hipMemcpyAsync(s->dev, s->host, s->bytes, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(st);
}

// The pieces that split() made, and the segments that it copied itself.
hipError_t HostLink::through_ring(const Seg* segs, size_t n, bool to_host, hipStream_t st)
{
    const hipError_t e = split(segs, n, to_host, st);
    if (e != hipSuccess || pieces_.empty()) return e;
    if (!open()) return plain(segs, n, to_host, st);
    if (!alone_) start_workers();
    begin(to_host);
    return to_host ? drain(st) : fill(st);
}

// Task i: a share of piece i / kTasks.
void HostLink::copy_task(size_t i)
{
    const Piece& p = pieces_[i / kTasks];
    char* slot = slot_ptr(i / kTasks);
    const size_t share = (p.bytes + kTasks * 64 - 1) / (kTasks * 64) * 64;
    const size_t lo = std::min(p.bytes, (i % kTasks) * share), hi = std::min(p.bytes, lo + share);
    for (int k = 0; k < p.parts; ++k) {
        const size_t b = std::max(lo, p.part[k].off);
        const size_t e = std::min(hi, p.part[k].off + p.part[k].bytes);
        if (b >= e) continue;
        char* host = p.part[k].host + (b - p.part[k].off);
        if (to_host_) std::memcpy(host, slot + b, e - b);
        else std::memcpy(slot + b, host, e - b);
    }
    left_[(i / kTasks) % kSlots].fetch_sub(1, std::memory_order_acq_rel);
}

// Take and do one handed-out task; false if there is none.
bool HostLink::work_one()
{
    size_t i = taken_.load(std::memory_order_relaxed);
    while (i < ready_.load(std::memory_order_acquire))
        if (taken_.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel)) {
            copy_task(i);
            return true;
        }
    return false;
}

// The calling thread while it waits: it copies until a worker has come; then
// it only keeps the link busy.
void HostLink::help()
{
    if (came_.load(std::memory_order_relaxed) || !work_one()) std::this_thread::yield();
}

void HostLink::worker()
{
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
        cv_.wait(lk, [&] { return stop_ || active_.load(std::memory_order_relaxed); });
        if (stop_) return;
        ++inside_;
        lk.unlock();
        came_.store(true, std::memory_order_relaxed);
        // tasks come every few microseconds while a copy is on: no sleeping (and
        // where it has to wait for its stream, slot_ready ends this)
        while (active_.load(std::memory_order_acquire))
            if (!work_one()) std::this_thread::yield();
        lk.lock();
        if (--inside_ == 0) cv_.notify_all();
        // the copy is over for everybody before the next one begins (end())
    }
}

void HostLink::begin(bool to_host)
{
    to_host_ = to_host;
    came_.store(false, std::memory_order_relaxed);
    ready_.store(0, std::memory_order_relaxed);
    taken_.store(0, std::memory_order_relaxed);
}

void HostLink::wake()
{
    if (workers_.empty()) return;
    std::lock_guard<std::mutex> lk(mu_);
    active_.store(true, std::memory_order_release);
    cv_.notify_all();
}

// The tasks of the next piece, in order.
void HostLink::hand_out(size_t piece)
{
    left_[piece % kSlots].store(kTasks, std::memory_order_relaxed);
    ready_.store((piece + 1) * kTasks, std::memory_order_release);
}

// Finishes the handed-out tasks; no worker touches the pieces on return (until wake()).
void HostLink::end()
{
    while (work_one()) {}
    for (auto& l : left_)
        while (l.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    if (!active_.load(std::memory_order_relaxed)) return;
    std::unique_lock<std::mutex> lk(mu_);
    active_.store(false, std::memory_order_release);
    cv_.wait(lk, [&] { return inside_ == 0; });
}

// The copy out of the slot, over on return.  While copies follow each other (flowing)
// that takes tens of microseconds; where it takes longer, the stream is still at the
// work before them (an earlier view's passes), and the threads sleep until it has come.
hipError_t HostLink::slot_ready(int slot, bool flowing)
{
    if (!in_flight_[slot]) return hipSuccess;
    in_flight_[slot] = false;
    if (flowing) return hipEventSynchronize(ev_[slot]);
    const auto patience = std::chrono::steady_clock::now() + std::chrono::microseconds(kPatienceUs);
    hipError_t e;
    while ((e = hipEventQuery(ev_[slot])) == hipErrorNotReady) {
        (void)hipGetLastError();   // an answer here, not an error
        if (std::chrono::steady_clock::now() < patience) {
            help();
            continue;
        }
        const bool awake = active_.load(std::memory_order_relaxed);
        if (awake) end();
        e = hipEventSynchronize(ev_[slot]);
        came_.store(false, std::memory_order_relaxed);
        if (awake) wake();
        break;
    }
    return e;
}

hipError_t HostLink::download(const Seg* segs, size_t n, hipStream_t st)
{
    try {
        if (!overlap(segs, n)) return through_ring(segs, n, true, st);
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < n && e == hipSuccess; ++i) e = through_ring(segs + i, 1, true, st);
        return e;
    } catch (const std::bad_alloc&) {   // of a list: no piece is under way
        return plain(segs, n, true, st);
    }
}

hipError_t HostLink::drain(hipStream_t st)
{
    const size_t n = pieces_.size();
    hipError_t e = hipSuccess;
    size_t issued = 0, handed = 0;
    while (handed < n && e == hipSuccess) {
        // keep the link busy: a copy into every free slot
        while (issued < n && issued < handed + kSlots && e == hipSuccess) {
            const int slot = (int)(issued % kSlots);
            if (left_[slot].load(std::memory_order_acquire) > 0) break;
            e = slot_ready(slot);
            if (e == hipSuccess)
                e = hipMemcpyAsync(slot_ptr(issued), pieces_[issued].dev, pieces_[issued].bytes,
                                   hipMemcpyDeviceToHost, st);
            // (a lone piece is waited for by its stream: 7 us less than by an event)
            if (e == hipSuccess && n > 1) e = hipEventRecord(ev_[slot], st);
            if (e == hipSuccess) ++issued;
        }
        if (e != hipSuccess) break;
        if (issued == handed) {   // every slot is being emptied: help
            help();
            continue;
        }
        if (n == 1) {
            e = hipStreamSynchronize(st);
        } else if (handed == 0) {
            e = hipEventSynchronize(ev_[0]);   // the work before the copy, however long
        } else {
            while ((e = hipEventQuery(ev_[handed % kSlots])) == hipErrorNotReady) help();
        }
        if (e != hipSuccess) break;
        hand_out(handed++);
        if (handed == 1 && !alone_) wake();
    }
    (void)hipGetLastError();   // the queries' "not ready"
    end();
    if (e != hipSuccess) (void)hipStreamSynchronize(st);   // no copy into the ring outlives the call
    return e;
}

hipError_t HostLink::upload(const Seg* segs, size_t n, hipStream_t st)
{
    if (n == 1 && segs->bytes < kLoneUpload)
        return hipMemcpyAsync(segs->dev, segs->host, segs->bytes, hipMemcpyHostToDevice, st);
    try {
        return through_ring(segs, n, false, st);
    } catch (const std::bad_alloc&) {
        return plain(segs, n, false, st);
    }
}

hipError_t HostLink::fill(hipStream_t st)
{
    const size_t n = pieces_.size();
    hipError_t e = hipSuccess;
    if (!alone_) wake();
    size_t handed = 0, issued = 0;
    while (issued < n && e == hipSuccess) {
        // without threads a piece at a time, so that the link starts early
        const size_t ahead = active_.load(std::memory_order_relaxed) ? kSlots : 1;
        while (handed < n && handed < issued + ahead && e == hipSuccess) {
            // (behind its first slot's copy the stream is at this call's)
            e = slot_ready((int)(handed % kSlots), handed > kSlots);
            if (e == hipSuccess) hand_out(handed++);
        }
        if (e != hipSuccess) break;
        const int slot = (int)(issued % kSlots);
        while (left_[slot].load(std::memory_order_acquire) > 0) help();
        e = hipMemcpyAsync(pieces_[issued].dev, slot_ptr(issued), pieces_[issued].bytes,
                           hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipEventRecord(ev_[slot], st);
        in_flight_[slot] = e == hipSuccess;
        ++issued;
    }
    end();
    if (e != hipSuccess) (void)hipStreamSynchronize(st);
    return e;
}

}  // namespace hp3d
