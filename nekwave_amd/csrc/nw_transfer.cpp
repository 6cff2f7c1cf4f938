// nw_transfer.cpp -- states between the caller's host arrays and the device.
//
// A plain hipMemcpy of pageable memory runs at 18 GB/s from the device and 38 GB/s to
// it (one copying thread inside the runtime), and a download moves FP64 where the
// device holds FP32.  Here a state goes in chunks of nodes: a kernel reads or writes
// the node-major fields on one side and a pinned slot on the other (55 GB/s over the
// link), and a few host threads copy between slots and the caller's array (30 GB/s
// per thread), each thread its own slot, so kernels and threads overlap; downloads
// cross the link in the device's precision.
// Measured, plain -> staged: 805 MB of host array (FP32 on the device) up 28.7 -> 16.6,
// down 46.7 -> 8.6 ms; 100 MB (FP64) 3.7 -> 2.2, 6.1 -> 2.2; 83 kB down 29 -> 19 us (one
// launch and one wait instead of a kernel, a copy and a wait).
#include "nw_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include <xmmintrin.h>

#include "nw_plain.hpp"

namespace nw {

namespace {

// One transfer's chunks.  Whoever is running takes the next one, so a helper that
// the system does not schedule in time delays nobody: the caller does its chunks
// and waits for those that took one.  (Threads started and joined per transfer
// waited whole time slices behind another library's spinning threads: 12.6 MB in
// 3.3 ms instead of 0.4.)
struct Job {
    int device = 0, workers = 1;
    long long chunks = 0;
    std::atomic<long long> next{0};
    std::atomic<int> running{0};
    std::atomic<int> bad{hipSuccess};
    // chunk c by worker w (in its slot); then, once, the end of worker w's share
    std::function<hipError_t(int, long long)> chunk;
    std::function<hipError_t(int)> end;

    void run(int w) {
        running.fetch_add(1);
        long long c = next.fetch_add(1);
        if (c < chunks) {
            hipError_t e = hipSetDevice(device);
            for (; c < chunks && e == hipSuccess; c = next.fetch_add(1)) e = chunk(w, c);
            const hipError_t f = end(w);
            if (e == hipSuccess) e = f;
            if (e != hipSuccess) {
                next.store(chunks);
                bad.store(e);
            }
        }
        running.fetch_sub(1);
    }
};

// A pinned slot and the event of the kernel that last used it.
struct Slot {
    void* p = nullptr;
    hipEvent_t ev = nullptr;
};

// Staging of one device.  A large transfer takes slot[] and the helpers for its whole
// length, one at a time (two would share the link).  A small one (one worker) takes one
// of small[] instead: it does not wait for another solver's large one (83 kB beside
// downloads of 340 MB: 14 ms when it did).
struct Stage {
    std::mutex mu;  // of slot[] and the job
    Slot slot[kStageSlots];
    std::mutex small_mu[kSmallSlots];
    Slot small[kSmallSlots];
    std::atomic<unsigned> turn{0};
    std::mutex users_mu;
    int users = 0;
    // helpers 1 .. kStageSlots - 1, started when a transfer first wants them
    std::vector<std::thread> helpers;
    std::mutex jm;
    std::condition_variable wake;
    std::shared_ptr<Job> job;
    unsigned long long posted = 0;
    bool quit = false;

    void help(int w) {
        unsigned long long seen = 0;
        for (;;) {
            std::shared_ptr<Job> j;
            {
                std::unique_lock<std::mutex> lk(jm);
                wake.wait(lk, [&] { return quit || posted != seen; });
                if (quit) return;
                seen = posted;
                j = job;
            }
            if (j && w < j->workers) j->run(w);
        }
    }
    // A small slot that is free, or the next one in turn when it is.
    std::unique_lock<std::mutex> take_small(int* which) {
        for (int x = 0; x < kSmallSlots; ++x) {
            std::unique_lock<std::mutex> lk(small_mu[x], std::try_to_lock);
            if (lk.owns_lock()) {
                *which = x;
                return lk;
            }
        }
        *which = static_cast<int>(turn.fetch_add(1) % kSmallSlots);
        return std::unique_lock<std::mutex>(small_mu[*which]);
    }
};
Stage& stage(int device) {
    static Stage* s = new Stage[kMaxDevices];  // never destroyed: no HIP calls after main
    return s[device];
}

// A slot's memory and its event on the current device; with the slot's mutex held.
hipError_t ready_slot(Slot& s) {
    if (!s.p) {
        const hipError_t e = hipHostMalloc(&s.p, kStageBytes, hipHostMallocPortable);
        if (e != hipSuccess) {
            s.p = nullptr;
            return e;
        }
    }
    if (!s.ev) return hipEventCreateWithFlags(&s.ev, hipEventDisableTiming);
    return hipSuccess;
}
void free_slot(Slot& s) {
    if (s.p) (void)hipHostFree(s.p);
    if (s.ev) (void)hipEventDestroy(s.ev);
    s = Slot();
}

// Waits for an event by asking for it: the runtime's own wait yields the CPU, and
// beside spinning threads of another library a yield costs a time slice (100 MB in
// 3 - 6 ms instead of 2.3).  Past 2 ms the runtime's wait.
hipError_t wait_event(hipEvent_t ev) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    for (;;) {
        const hipError_t e = hipEventQuery(ev);
        if (e != hipErrorNotReady) return e;
        if (std::chrono::steady_clock::now() > until) return hipEventSynchronize(ev);
        for (int x = 0; x < 64; ++x) __builtin_ia32_pause();
    }
}

// The conversion below reads FP32 subnormals, which a thread whose MXCSR has
// denormals-are-zero set (an option of some numerical libraries, inherited by the threads
// it starts) would read as zeros.
struct DefaultMxcsr {
    const unsigned was = _mm_getcsr();
    DefaultMxcsr() { _mm_setcsr(0x1f80); }
    ~DefaultMxcsr() { _mm_setcsr(was); }
};

// Component block of n values from the slot (R) to the caller's array (FP64).
template <typename R>
void block_from_slot(double* host, const R* slot, size_t n) {
    if constexpr (sizeof(R) == 8) {
        std::memcpy(host, slot, n * 8);
    } else {
        const DefaultMxcsr mode;
        for (size_t x = 0; x < n; ++x) host[x] = static_cast<double>(slot[x]);
    }
}

// A state in chunks of nodes, taken by up to kStageSlots workers, each through its own
// slot.  Kernels of all workers go to the one stream.
template <typename R, bool UP>
int move_state(int device, hipStream_t s, std::conditional_t<UP, const double*, double*> host, long long P,
               const DeviceState& d) {
    Stage& st = stage(device);
    const long long most = (long long)(kStageBytes / (6 * (UP ? 8 : sizeof(R))) / 64 * 64);
    // Helpers cost more where other threads want the CPUs, so no more than pay: on the
    // way out one worker per 6 MB of host array (FP32 leaves the link as twice that to
    // write; 805 MB: four 11.3, eight 8.6 ms), on the way in four (a worker's copy and
    // its slot's crossing take turns; 805 MB: two 29, three 19.7, four 16.6 ms).
    const int hw = std::max(1, static_cast<int>(std::thread::hardware_concurrency()));
    const long long want = 1 + P * 48 / (6 << 20);
    int workers = static_cast<int>(std::min<long long>(std::min(UP ? 4 : kStageSlots, hw), want));
    // two chunks or more per worker, so that kernels and copies overlap
    const long long per = P <= most && workers == 1 ? P : std::min(most, std::max<long long>(4096, P / (2 * workers) / 64 * 64));
    const long long chunks = (P + per - 1) / per;
    workers = static_cast<int>(std::min<long long>(workers, chunks));
    int which = 0;
    const std::unique_lock<std::mutex> lk = workers > 1 ? std::unique_lock<std::mutex>(st.mu) : st.take_small(&which);
    Slot* const slots = workers > 1 ? st.slot : st.small + which;
    for (int w = 0; w < workers; ++w) {
        const hipError_t e = ready_slot(slots[w]);
        if (e != hipSuccess && w > 0) {  // fewer slots do
            (void)hipGetLastError();
            workers = w;
        } else if (e != hipSuccess) {
            set_error(std::string("host staging: ") + hipGetErrorString(e));
            return NW_ERR_ALLOC;
        }
    }
    auto job = std::make_shared<Job>();
    job->device = device;
    job->workers = workers;
    job->chunks = chunks;
    bool waits[kStageSlots] = {};  // a kernel that reads the worker's slot is in flight
    job->chunk = [&](int w, long long c) -> hipError_t {
        typedef std::conditional_t<UP, double, R> V;
        V* slot = static_cast<V*>(slots[w].p);
        hipEvent_t ev = slots[w].ev;
        const long long p0 = c * per, n = std::min(per, P - p0);
        hipError_t e = hipSuccess;
        if constexpr (UP) {
            if (waits[w]) e = wait_event(ev);
            if (e != hipSuccess) return e;
            for (int f = 0; f < 6; ++f) std::memcpy(slot + f * n, host + f * P + p0, size_t(n) * 8);
            e = launch_state_in<R>(static_cast<R*>(d.data), d.cs, d.ns, p0, n, slot, s);
            if (e == hipSuccess) e = hipEventRecord(ev, s);
            waits[w] = e == hipSuccess;
        } else {
            e = launch_state_out<R>(static_cast<const R*>(d.data), d.cs, d.ns, p0, n, slot, s);
            if (e == hipSuccess) e = hipEventRecord(ev, s);
            if (e == hipSuccess) e = wait_event(ev);
            if (e != hipSuccess) return e;
            for (int f = 0; f < 6; ++f) block_from_slot(host + f * P + p0, slot + f * n, size_t(n));
        }
        return e;
    };
    job->end = [&](int w) -> hipError_t { return waits[w] ? wait_event(slots[w].ev) : hipSuccess; };
    if (workers > 1) {
        std::lock_guard<std::mutex> jl(st.jm);
        try {
            while (static_cast<int>(st.helpers.size()) < workers - 1) {
                const int w = static_cast<int>(st.helpers.size()) + 1;
                st.helpers.emplace_back([&st, w] { st.help(w); });
            }
        } catch (...) {  // no more threads: those there are, and this one
        }
        st.job = job;
        ++st.posted;
        st.wake.notify_all();
    }
    job->run(0);
    while (job->running.load() > 0) __builtin_ia32_pause();
    // a helper that wakes up from here on finds no chunk left and touches only the job
    if (workers > 1) {
        std::lock_guard<std::mutex> jl(st.jm);
        st.job.reset();
    }
    if (job->bad.load() != hipSuccess) {
        (void)hipStreamSynchronize(s);
        set_error(std::string("state transfer: ") + hipGetErrorString(static_cast<hipError_t>(job->bad.load())));
        return NW_ERR_HIP;
    }
    return NW_OK;
}

}  // namespace

void stage_retain(int device) {
    Stage& st = stage(device);
    std::lock_guard<std::mutex> lk(st.users_mu);
    ++st.users;
}

void stage_release(int device) {
    Stage& st = stage(device);
    std::lock_guard<std::mutex> lk(st.users_mu);  // no solver of the device is left to transfer
    if (--st.users > 0) return;
    {
        std::lock_guard<std::mutex> jl(st.jm);
        st.quit = true;
        st.wake.notify_all();
    }
    for (std::thread& t : st.helpers) t.join();
    st.helpers.clear();
    st.quit = false;
    for (Slot& s : st.slot) free_slot(s);
    for (Slot& s : st.small) free_slot(s);
}

bool device_pointer(const void* p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();  // plain host memory
        return false;
    }
    return at.type == hipMemoryTypeDevice;
}

int upload_state(int device, hipStream_t s, const double* host, long long P, const DeviceState& d) {
    return d.f64 ? move_state<double, true>(device, s, host, P, d) : move_state<float, true>(device, s, host, P, d);
}

int download_state(int device, hipStream_t s, double* host, long long P, const DeviceState& d) {
    return d.f64 ? move_state<double, false>(device, s, host, P, d) : move_state<float, false>(device, s, host, P, d);
}

int download_bytes(int device, hipStream_t s, void* host, const void* dev, size_t bytes) {
    int which = 0;
    std::unique_lock<std::mutex> lk;
    void* slot = nullptr;
    if (bytes <= kStageBytes && !device_pointer(host)) {
        lk = stage(device).take_small(&which);
        if (ready_slot(stage(device).small[which]) == hipSuccess) slot = stage(device).small[which].p;
        else (void)hipGetLastError();
    }
    NW_TRY_HIP(hipMemcpyAsync(slot ? slot : host, dev, bytes, hipMemcpyDefault, s));
    NW_TRY_HIP(hipStreamSynchronize(s));
    if (slot) std::memcpy(host, slot, bytes);
    return NW_OK;
}

}  // namespace nw
