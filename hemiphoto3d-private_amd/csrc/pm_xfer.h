// pm_xfer.h -- copies between pageable host memory and the device.
//
// The runtime's own copy of pageable memory stages it through one thread: 17
// GB/s to the host, 36 GB/s from it, and 60 us for a small view's maps, against
// 57 GB/s and 11 us from page-locked memory; a caller's fresh arrays, whose
// pages are touched for the first time, take 4 to 14 GB/s a thread.  A HostLink
// keeps a ring of page-locked slots: the link fills or drains them in order on
// a stream while a few threads copy between the slots and the caller's memory,
// or, for copies of up to a few slots, the calling thread alone.  Page-locked
// host memory is copied by the link directly, and one segment of less than
// kLoneUpload bytes goes to the device by the runtime's copy, which is the faster
// one there (64 KiB 12 against 18 us, 1 MiB 40 and 51, 8 MiB 234 and 260, 20 MiB 564
// and 566, 24 MiB 675 and 610; an image upload is such a copy).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <initializer_list>
#include <mutex>
#include <thread>
#include <vector>

namespace hp3d {

// One host thread at a time.  Ring and threads are made by the first copy that
// needs them and given back by close().
class HostLink {
public:
    // `bytes` of host memory and of device memory.  Neighbouring segments that
    // are adjacent on the device share slots.
    struct Seg {
        void* host;
        void* dev;
        size_t bytes;
    };

    HostLink() = default;
    HostLink(const HostLink&) = delete;
    HostLink& operator=(const HostLink&) = delete;
    ~HostLink() { close(); }

    // Device to host, after the work queued on st.  Where segments overlap in
    // host memory the later one's bytes stay.  Returns when pageable
    // destinations are written; page-locked ones are once st is synchronised.
    hipError_t download(const Seg* segs, size_t n, hipStream_t st);
    // Host to device on st.  Returns when pageable sources are read; page-locked
    // ones are once st is synchronised.
    hipError_t upload(const Seg* segs, size_t n, hipStream_t st);
    // (neither throws: without memory for their lists the runtime copies)

    typedef std::initializer_list<Seg> SegList;
    hipError_t download(SegList s, hipStream_t st) { return download(s.begin(), s.size(), st); }
    hipError_t upload(SegList s, hipStream_t st) { return upload(s.begin(), s.size(), st); }
    hipError_t download(const std::vector<Seg>& s, hipStream_t st) { return download(s.data(), s.size(), st); }
    hipError_t upload(const std::vector<Seg>& s, hipStream_t st) { return upload(s.data(), s.size(), st); }
    // Whether segments share host memory.
    static bool overlap(const Seg* segs, size_t n);
    // Waits for the ring's copies and gives everything back.
    void close();

private:
    // The link spends 10 to 15 us on each copy besides its bytes, so pieces are
    // as large as still lets the threads work beside it (38 MB at 36 GB/s in
    // pieces of 2 MiB, 42 in 4; 10 MB at 26 in 1 MiB, 31 in 2).  A copy of up to
    // 3 MiB is over before threads have woken.
    static constexpr int kSlots = 8;
    static constexpr size_t kSlotBytes = 4u << 20;
    static constexpr size_t kAloneBytes = 3u << 20;
    static constexpr size_t kLoneUpload = 24u << 20;
    static size_t piece_bytes(size_t total)
    {
        return total < (4u << 20) ? 1u << 20 : total < (24u << 20) ? 2u << 20 : kSlotBytes;
    }
    static constexpr int kTasks = 4;       // a piece's shares among the threads
    static constexpr int kPatienceUs = 300;   // a 4 MiB piece takes 75 us, waking threads 50
    static constexpr int kMaxParts = 4;
    static constexpr int kMaxWorkers = 6;

    struct Piece {   // one slot's worth: adjacent device memory, its host parts
        char* dev = nullptr;
        size_t bytes = 0;
        int parts = 0;
        struct { char* host; size_t off, bytes; } part[kMaxParts];
    };

    bool open();
    void start_workers();
    hipError_t split(const Seg* segs, size_t n, bool to_host, hipStream_t st);
    static hipError_t plain(const Seg* segs, size_t n, bool to_host, hipStream_t st);
    hipError_t through_ring(const Seg* segs, size_t n, bool to_host, hipStream_t st);
    hipError_t drain(hipStream_t st);
    hipError_t fill(hipStream_t st);
    void copy_task(size_t i);
    bool work_one();
    void help();
    void worker();
    void begin(bool to_host);
    void wake();
    void hand_out(size_t piece);
    void end();
    hipError_t slot_ready(int slot, bool flowing = false);
    char* slot_ptr(size_t piece) { return ring_ + (piece % kSlots) * kSlotBytes; }

    char* ring_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    bool in_flight_[kSlots] = {};   // ev_ of a copy out of the slot, not waited for yet
    std::vector<Piece> pieces_;
    bool alone_ = true;             // no threads for this copy
    std::atomic<int> left_[kSlots] = {};   // tasks of the slot's piece not done yet

    // the copy the threads are at: tasks [0, ready_) may be taken
    bool to_host_ = false;
    std::atomic<size_t> ready_{0}, taken_{0};
    std::atomic<bool> active_{false}, came_{false};   // came_: a worker has
    std::mutex mu_;
    std::condition_variable cv_;
    bool stop_ = false;
    int inside_ = 0;                // workers in the copy (mu_)
    std::vector<std::thread> workers_;
};

}  // namespace hp3d
