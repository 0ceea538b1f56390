// Copies between host buffers of any kind and device memory through pinned
// staging memory (internal to libhpl_hip.so).
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

namespace hplx {

// A few pinned buffers with an event each, owned by one context, slot or batch
// and used by one thread at a time.  Made on first use, given back by free().
//
// The runtime moves a pitched copy from ordinary host memory row by row, each
// row pinned and queued by itself (about 10 us a row: 27 ms for the three
// transfers of a 1024 x 1024 solve, 1.3 ms through these buffers).  Here rows are
// packed at the device's pitch by the host while the previous piece is on its
// way, so the device sees plain copies from pinned memory.  Longer transfers of
// buffers that the runtime knows -- the caller's own pinned, managed or device
// memory -- are copied from or to directly: a copy through the host's caches halves
// their rate (n = 4096 up 1.2 ms direct and 2.2 staged, down 1.2 and 2.9; 16384 19
// and 36, 19 and 45).
class HostStage {
   public:
    ~HostStage() { free(); }
    // `rows` rows of `width` bytes, `pitch` apart on each side.  to_device: the
    // copies run on `s`; an ordinary host buffer may be reused on return (of such a
    // one the device rows' bytes between width and pitch become zero where the
    // pitch fits a staging buffer, the last row's excepted), one that the runtime
    // knows once `s` has got there.  to_host: returns when the rows are in place,
    // after everything enqueued on `s` before.
    hipError_t to_device(hipStream_t s, void* dev, size_t dev_pitch, const void* host,
                         size_t host_pitch, size_t width, size_t rows);
    hipError_t to_host(hipStream_t s, void* host, size_t host_pitch, const void* dev,
                       size_t dev_pitch, size_t width, size_t rows);
    // contiguous bytes
    hipError_t to_device(hipStream_t s, void* dev, const void* host, size_t bytes);
    hipError_t to_host(hipStream_t s, void* host, const void* dev, size_t bytes);
    // the large buffers, which serve every size, for who cannot fail later (both
    // sets cost a server of four slots 1.1 ms more); free() gives them back
    hipError_t make() { return large_.make(); }
    void free() {
        small_.free();
        large_.free();
    }

   private:
    static constexpr int kBufs = 4;
    // Up to 64 KiB (status words, norms, vectors of small orders) through small
    // buffers while there are no large ones, so that only a context that moves more
    // holds their 4 MiB.  Those are 1 MiB each: packed in 30 us, on its way for 20
    // us; shorter pieces pay the launch of a copy, longer ones the wait for the
    // first and last piece.
    static constexpr size_t kSmall = 64u << 10, kLarge = 1u << 20;
    struct Ring {
        size_t bytes;  // of one buffer
        char* mem = nullptr;
        hipEvent_t ev[kBufs] = {};
        int next = 0;
        hipError_t make();
        void free();
    };
    Ring& ring(size_t bytes) { return bytes <= kSmall && !large_.mem ? small_ : large_; }
    Ring small_{kSmall}, large_{kLarge};
};

}  // namespace hplx
