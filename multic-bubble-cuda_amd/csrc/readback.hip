#include "readback.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace mcb {

namespace {

// A copy into pageable memory runs through the runtime's staging buffers on
// one thread: 64 MiB 3.9 ms, 6.4 ms into memory whose pages are not there yet,
// against 1.2 ms on the link. Here chunks into the ring follow one another on
// the link while several threads move what has arrived, kSlice at a time, and
// share the page faults: 64 MiB 1.6 ms, 1.7 ms into new pages. A chunk costs
// about 10 us beside its bytes and the last one's move is not hidden: 4 MiB
// chunks for large reads (64 MiB in 2 MiB chunks 1.8 ms), 2 MiB below (4 MiB
// 155 us against 190 with twice the threads and 247 direct, 8 MiB 275 against
// 490).
constexpr size_t kSlots = 4, kSlice = 256u << 10, kLarge = 16u << 20;
constexpr size_t chunk_of(size_t bytes) { return bytes >= kLarge ? 4u << 20 : 2u << 20; }
constexpr unsigned threads_of(size_t bytes) { return bytes >= kLarge ? 8 : 4; }
// Below this the direct copy is about as fast (2 MiB: 123 us), and starting
// threads costs what it could gain.
constexpr size_t kMinBytes = 4u << 20;
// Rows below this share one wait (19 rows of 16 KiB 405 us against 513 with a
// wait each, into pinned memory 88 against 224); from there on waiting for each
// is the faster (54 KiB 225 against 251 and 181 against 200).
constexpr size_t kOneWait = 32u << 10;

struct Events {
    hipEvent_t e[kSlots] = {};
    bool create() {
        for (auto& x : e)
            if (hipEventCreateWithFlags(&x, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                x = nullptr;
                return false;
            }
        return true;
    }
    ~Events() {
        for (auto x : e)
            if (x) (void)hipEventDestroy(x);
    }
};

// Ordinary memory that HIP does not know: the ring only helps there.
bool pageable(const void* host) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

std::shared_ptr<Readback> Readback::shared() noexcept try {
    static std::mutex mu;
    static std::weak_ptr<Readback> one;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<Readback> r = one.lock();
    if (!r) one = r = std::make_shared<Readback>();
    return r;
} catch (const std::exception&) {
    return nullptr;
}

Readback::~Readback() {
    if (ring_) (void)hipHostFree(ring_);
}

// Room for a read of `bytes`; pinning costs 30 us per MiB and more.
bool Readback::ready(size_t bytes) {
    const size_t chunk = chunk_of(bytes), need = std::min((bytes + chunk - 1) / chunk, kSlots) * chunk;
    if (ring_bytes_ >= need) return true;
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
    if (hipHostMalloc(reinterpret_cast<void**>(&ring_), need, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        ring_ = nullptr;
        return false;
    }
    ring_bytes_ = need;
    return true;
}

hipError_t Readback::copy(Readback* r, void* host, const void* dev, size_t bytes, hipStream_t stream) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (r && bytes >= kMinBytes && pageable(host) && hipStreamIsCapturing(stream, &cs) == hipSuccess &&
        cs == hipStreamCaptureStatusNone) {
        std::unique_lock<std::mutex> lk(r->mu_, std::try_to_lock);
        Events ev;
        int device = 0;
        if (lk.owns_lock() && r->ready(bytes) && hipGetDevice(&device) == hipSuccess && ev.create())
            return r->staged(static_cast<char*>(host), static_cast<const char*>(dev), bytes, stream, device, ev.e);
    }
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
}

hipError_t Readback::copy_rows(Readback* r, void* host, const void* dev, size_t bytes, size_t pitch, int rows,
                               hipStream_t stream) {
    char* const h = static_cast<char*>(host);
    const char* const d = static_cast<const char*>(dev);
    hipError_t e = hipSuccess;
    for (int i = 0; i < rows && e == hipSuccess; ++i)
        e = bytes >= kOneWait ? copy(r, h + i * bytes, d + i * pitch, bytes, stream)
                              : hipMemcpyAsync(h + i * bytes, d + i * pitch, bytes, hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess || bytes >= kOneWait) return e;
    return hipStreamSynchronize(stream);
}

hipError_t Readback::staged(char* host, const char* dev, size_t bytes, hipStream_t stream, int device,
                            const hipEvent_t* ev) {
    const size_t chunk = chunk_of(bytes), per = chunk / kSlice;
    const size_t chunks = (bytes + chunk - 1) / chunk, slices = (bytes + kSlice - 1) / kSlice;
    // Slices are claimed in order. Chunk i may enter its slot when the slices
    // of chunk i - kSlots have left it (moved[slot] counts them): whoever moves
    // the last of those sends chunk i. The slices before any claimed one are
    // claimed too, so every wait below ends, with any number of threads.
    std::atomic<size_t> next{0};
    std::atomic<size_t> moved[kSlots] = {};
    std::atomic<size_t> sent[kSlots] = {};   // chunks sent through a slot
    std::atomic<int> error{hipSuccess};
    auto send = [&](size_t i) {
        const size_t s = i % kSlots, at = i * chunk;
        hipError_t r = hipMemcpyAsync(ring_ + s * chunk, dev + at, std::min(chunk, bytes - at), hipMemcpyDeviceToHost, stream);
        if (r == hipSuccess) r = hipEventRecord(ev[s], stream);
        if (r != hipSuccess) error = r;
        sent[s].store(i / kSlots + 1, std::memory_order_release);
    };
    auto work = [&] {
        size_t here = chunks;   // the last chunk this thread has waited for
        for (size_t q; error.load() == hipSuccess && (q = next.fetch_add(1)) < slices;) {
            const size_t i = q / per, s = i % kSlots, at = q * kSlice;
            while (sent[s].load(std::memory_order_acquire) <= i / kSlots && error.load() == hipSuccess)
                std::this_thread::yield();
            if (error.load() != hipSuccess) return;
            if (i != here) {
                const hipError_t r = hipEventSynchronize(ev[s]);
                if (r != hipSuccess) {
                    error = r;
                    return;
                }
                here = i;
            }
            std::memcpy(host + at, ring_ + s * chunk + (at - i * chunk), std::min(kSlice, bytes - at));
            if (moved[s].fetch_add(1, std::memory_order_acq_rel) + 1 == per) {
                moved[s].store(0, std::memory_order_relaxed);   // before the next chunk is sent
                if (i + kSlots < chunks) send(i + kSlots);
            }
        }
    };
    for (size_t i = 0; i < std::min(chunks, kSlots); ++i) send(i);

    std::vector<std::thread> helpers;
    const size_t want = std::min<size_t>({threads_of(bytes), std::max(1u, std::thread::hardware_concurrency()), slices});
    try {
        helpers.reserve(want);
        while (helpers.size() + 1 < want)
            helpers.emplace_back([&] {
                if (hipSetDevice(device) == hipSuccess) work();
            });
    } catch (const std::exception&) {
        // fewer helpers: the loop below moves what they do not
    }
    work();
    for (auto& t : helpers) t.join();
    const hipError_t r = hipStreamSynchronize(stream);   // also after an error: the ring is in use until then
    return error.load() != hipSuccess ? static_cast<hipError_t>(error.load()) : r;
}

}  // namespace mcb
