// Device results into pageable host memory and host arrays to the device, in
// chunks through pinned staging.
//
// A plain copy into memory the caller has just allocated runs at the speed of
// one thread taking its page faults (about 10 GB/s here, against about 50
// over PCIe). Here several host threads each own a staging slot (4 MiB of
// pinned memory), take chunks in turn, queue the kernel that fills the slot on
// the domain's stream, wait for their own event and copy the chunk out, so
// faults and copies of different chunks overlap. Kernels write and read the
// slot over PCIe themselves; a copy between it and device memory was one more
// launch per chunk, and the transfer only began when the kernel had ended
// (per call: 16^3 cells 57 -> 42 us, 160^3 3.5 -> 3.0 ms). Slots come from a process-wide pool of at most kKept idle
// ones, given back when the last domain is destroyed, so a call allocates
// nothing after the first.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm_amd {

struct StagingSlot {
    static constexpr size_t kBytes = size_t{4} << 20;
    int device = -1;
    void* host = nullptr;
    void* dev = nullptr;  // the same memory as the device addresses it
    hipEvent_t done = nullptr;
};

class StagingPool {
public:
    static StagingPool& get() {
        static StagingPool* p = new StagingPool;  // never destroyed: no HIP calls at process exit
        return *p;
    }
    // The calling thread's current device must be `device`.
    hipError_t acquire(int device, StagingSlot& s) {
        {
            std::lock_guard<std::mutex> lock(m_);
            for (size_t i = idle_.size(); i-- > 0;)
                if (idle_[i].device == device) {
                    s = idle_[i];
                    idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(i));
                    return hipSuccess;
                }
        }
        s = StagingSlot{};
        s.device = device;
        hipError_t e = hipHostMalloc(&s.host, StagingSlot::kBytes, hipHostMallocMapped | hipHostMallocCoherent);
        if (e == hipSuccess) e = hipHostGetDevicePointer(&s.dev, s.host, 0);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
        if (e != hipSuccess) destroy(s);
        return e;
    }
    void release(const StagingSlot& s) {
        {
            std::lock_guard<std::mutex> lock(m_);
            if (domains_ > 0 && idle_.size() < kKept) {
                idle_.push_back(s);
                return;
            }
        }
        destroy(s);
    }
    void domain_created() {
        std::lock_guard<std::mutex> lock(m_);
        ++domains_;
    }
    void domain_destroyed() {
        std::vector<StagingSlot> out;
        {
            std::lock_guard<std::mutex> lock(m_);
            if (--domains_ > 0) return;
            out.swap(idle_);
        }
        for (const StagingSlot& s : out) destroy(s);
    }

private:
    static constexpr size_t kKept = 16;
    StagingPool() { idle_.reserve(kKept); }
    static void destroy(const StagingSlot& s) {
        (void)hipHostFree(s.host);
        if (s.done) (void)hipEventDestroy(s.done);
    }
    std::mutex m_;
    std::vector<StagingSlot> idle_;
    int64_t domains_ = 0;
};

// Runs chunks(slot, first item, items) for consecutive ranges of `items`
// items of `item_bytes` each, on several host threads with a slot each.
// Returns when all ranges are done.
template <class Chunk>
hipError_t staged(int device, hipStream_t stream, int64_t items, size_t item_bytes, Chunk one_chunk) {
    const int64_t most = static_cast<int64_t>(StagingSlot::kBytes / item_bytes);
    // one thread per MiB, up to 12 of the host's: 226 MB of moments take
    // 22 ms as one plain copy, 6 ms here
    const int64_t bytes = items * static_cast<int64_t>(item_bytes);
    const int64_t host = std::max<int64_t>(1, static_cast<int64_t>(std::thread::hardware_concurrency()));
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>({bytes >> 20, 12, host}));
    const int64_t chunk = std::max<int64_t>(1, std::min(most, (items + want - 1) / want));
    std::atomic<int64_t> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](bool first) {
        hipError_t e = first ? hipSuccess : hipSetDevice(device);
        StagingSlot s;
        bool have = false;
        while (e == hipSuccess && error.load() == hipSuccess) {
            if (!have) {
                e = StagingPool::get().acquire(device, s);
                // without a slot of its own a helper leaves the rest to the others
                if (e != hipSuccess && !first) {
                    (void)hipGetLastError();
                    return;
                }
                if (e != hipSuccess) break;
                have = true;
            }
            const int64_t i = next.fetch_add(chunk);
            if (i >= items) break;
            e = one_chunk(s, i, std::min(chunk, items - i));
        }
        if (have) {
            if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing in flight uses the slot
            StagingPool::get().release(s);
        }
        if (e != hipSuccess) error.store(e);
    };
    std::vector<std::thread> helpers;
    try {
        helpers.reserve(static_cast<size_t>(want));
        for (int64_t k = 1; k < want; ++k) helpers.emplace_back(work, false);
    } catch (...) {  // no more threads: those there are do the work
    }
    work(true);
    for (std::thread& t : helpers) t.join();
    return static_cast<hipError_t>(error.load());
}

// fill(slot, first item, items, stream) queues the kernels that write a
// chunk's result; out(slot in host memory, first item, items) takes it.
template <class Fill, class Out>
hipError_t staged_read(int device, hipStream_t stream, int64_t items, size_t item_bytes, Fill fill, Out out) {
    return staged(device, stream, items, item_bytes, [&](const StagingSlot& s, int64_t i, int64_t n) {
        hipError_t e = fill(s.dev, i, n, stream);
        if (e == hipSuccess) e = hipEventRecord(s.done, stream);
        if (e == hipSuccess) e = hipEventSynchronize(s.done);
        if (e == hipSuccess) out(static_cast<const char*>(s.host), i, n);
        return e;
    });
}

// in(slot in host memory, first item, items) writes a chunk; use(slot, first
// item, items, stream) queues the kernels that take it.
template <class In, class Use>
hipError_t staged_write(int device, hipStream_t stream, int64_t items, size_t item_bytes, In in, Use use) {
    return staged(device, stream, items, item_bytes, [&](const StagingSlot& s, int64_t i, int64_t n) {
        in(static_cast<char*>(s.host), i, n);
        hipError_t e = use(s.dev, i, n, stream);
        if (e == hipSuccess) e = hipEventRecord(s.done, stream);
        if (e == hipSuccess) e = hipEventSynchronize(s.done);
        return e;
    });
}

}  // namespace lbm_amd
