// Device-to-host copies of large fields into ordinary (pageable) memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>
#include <mutex>

namespace mcb {

// A ring of pinned memory that large copies pass through. Contexts and
// batches share one ring: it grows to what the largest read needs (16 MiB at
// most), serves one read at a time (a second one meanwhile copies without it)
// and is freed with the last context or batch.
class Readback {
public:
    static std::shared_ptr<Readback> shared() noexcept;   // null where memory is short
    ~Readback();

    // host[0, bytes) = dev[0, bytes) behind the work queued on `stream` (of
    // the current device); returns when the copy is complete. r may be null.
    static hipError_t copy(Readback* r, void* host, const void* dev, size_t bytes, hipStream_t stream);
    // The same for `rows` rows of `bytes`, `pitch` bytes apart on the device and
    // dense on the host; small rows share one wait.
    static hipError_t copy_rows(Readback* r, void* host, const void* dev, size_t bytes, size_t pitch, int rows,
                                hipStream_t stream);

private:
    bool ready(size_t bytes);
    // ev: an event per slot, of the current device.
    hipError_t staged(char* host, const char* dev, size_t bytes, hipStream_t stream, int device, const hipEvent_t* ev);

    std::mutex mu_;
    char* ring_ = nullptr;
    size_t ring_bytes_ = 0;
};

}  // namespace mcb
