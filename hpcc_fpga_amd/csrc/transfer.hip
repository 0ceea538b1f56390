#include "transfer.hpp"

#include <algorithm>
#include <cstring>

namespace hplx {

namespace {

// Memory that the runtime made or has registered (pinned, managed, device): its
// copies need no staging.  Asking costs 3 us, more than a host copy of a small
// buffer, so it is for longer transfers.
bool runtime_knows(const void* p) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t HostStage::Ring::make() {
    if (mem) return hipSuccess;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&mem), kBufs * bytes,
                                 hipHostMallocDefault);
    if (e != hipSuccess) {
        mem = nullptr;
        return e;
    }
    for (hipEvent_t& v : ev) {
        e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
        if (e != hipSuccess) {
            v = nullptr;
            free();
            return e;
        }
    }
    return hipSuccess;
}

void HostStage::Ring::free() {
    for (hipEvent_t& v : ev) {
        if (v) {
            (void)hipEventSynchronize(v);  // its last copy
            (void)hipEventDestroy(v);
        }
        v = nullptr;
    }
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
}

hipError_t HostStage::to_device(hipStream_t s, void* dev, size_t dev_pitch, const void* host,
                                size_t host_pitch, size_t width, size_t rows) {
    if (!width || !rows) return hipSuccess;
    // bytes from a row's start to the next one's (or to its own end)
    const size_t span = rows > 1 ? dev_pitch : width;
    if (width > span) return hipErrorInvalidValue;
    const size_t total = (rows - 1) * span + width;
    if (total > kSmall && runtime_knows(host))
        return hipMemcpy2DAsync(dev, dev_pitch, host, host_pitch, width, rows,
                                hipMemcpyHostToDevice, s);
    Ring& R = ring(total);
    hipError_t e = R.make();
    if (e != hipSuccess) return e;
    if (span > kLarge) {  // row by row, each in pieces
        for (size_t r = 0; r < rows && e == hipSuccess; ++r)
            e = to_device(s, static_cast<char*>(dev) + r * dev_pitch,
                          static_cast<const char*>(host) + r * host_pitch, width);
        return e;
    }
    const size_t per = std::max<size_t>(1, R.bytes / span);
    for (size_t r = 0; r < rows; r += per) {
        const size_t nr = std::min(per, rows - r);
        const int b = R.next;
        R.next = (R.next + 1) % kBufs;
        e = hipEventSynchronize(R.ev[b]);  // the buffer's previous copy
        if (e != hipSuccess) return e;
        char* buf = R.mem + b * R.bytes;
        for (size_t i = 0; i < nr; ++i) {
            std::memcpy(buf + i * span, static_cast<const char*>(host) + (r + i) * host_pitch,
                        width);
            if (i + 1 < nr || r + nr < rows) std::memset(buf + i * span + width, 0, span - width);
        }
        const size_t bytes = r + nr < rows ? nr * span : (nr - 1) * span + width;
        e = hipMemcpyAsync(static_cast<char*>(dev) + r * span, buf, bytes, hipMemcpyHostToDevice,
                           s);
        if (e == hipSuccess) e = hipEventRecord(R.ev[b], s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t HostStage::to_device(hipStream_t s, void* dev, const void* host, size_t bytes) {
    if (bytes > kSmall && runtime_knows(host))
        return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    const size_t whole = bytes / kLarge, done = whole * kLarge;
    hipError_t e = to_device(s, dev, kLarge, host, kLarge, kLarge, whole);
    if (e != hipSuccess || done == bytes) return e;
    return to_device(s, static_cast<char*>(dev) + done, bytes - done,
                     static_cast<const char*>(host) + done, bytes - done, bytes - done, 1);
}

hipError_t HostStage::to_host(hipStream_t s, void* host, const void* dev, size_t bytes) {
    if (bytes > kSmall && runtime_knows(host)) {
        hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    const size_t whole = bytes / kLarge, done = whole * kLarge;
    hipError_t e = to_host(s, host, kLarge, dev, kLarge, kLarge, whole);
    if (e != hipSuccess || done == bytes) return e;
    return to_host(s, static_cast<char*>(host) + done, bytes - done,
                   static_cast<const char*>(dev) + done, bytes - done, bytes - done, 1);
}

hipError_t HostStage::to_host(hipStream_t s, void* host, size_t host_pitch, const void* dev,
                              size_t dev_pitch, size_t width, size_t rows) {
    if (!width || !rows) return hipSuccess;
    const size_t span = rows > 1 ? dev_pitch : width;
    if (width > span) return hipErrorInvalidValue;
    const size_t total = (rows - 1) * span + width;
    if (total > kSmall && runtime_knows(host)) {
        hipError_t e = hipMemcpy2DAsync(host, host_pitch, dev, dev_pitch, width, rows,
                                        hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    Ring& R = ring(total);
    hipError_t e = R.make();
    if (e != hipSuccess) return e;
    if (span > kLarge) {
        for (size_t r = 0; r < rows && e == hipSuccess; ++r)
            e = to_host(s, static_cast<char*>(host) + r * host_pitch,
                        static_cast<const char*>(dev) + r * dev_pitch, width);
        return e;
    }
    const size_t per = std::max<size_t>(1, R.bytes / span);
    const size_t pieces = (rows + per - 1) / per;
    const int first = R.next;
    // up to kBufs pieces on their way while the oldest is unpacked
    for (size_t p = 0, q = 0; q < pieces; ++q) {
        for (; p < pieces && p < q + kBufs; ++p) {
            const size_t nr = std::min(per, rows - p * per);
            const size_t bytes = p + 1 < pieces ? nr * span : (nr - 1) * span + width;
            const int b = (int)((first + p) % kBufs);
            if (p < (size_t)kBufs) {  // what an earlier call left in the buffer
                e = hipEventSynchronize(R.ev[b]);
                if (e != hipSuccess) return e;
            }
            e = hipMemcpyAsync(R.mem + b * R.bytes, static_cast<const char*>(dev) + p * per * span,
                               bytes, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(R.ev[b], s);
            if (e != hipSuccess) return e;
        }
        const int b = (int)((first + q) % kBufs);
        e = hipEventSynchronize(R.ev[b]);
        if (e != hipSuccess) return e;
        const size_t nr = std::min(per, rows - q * per);
        for (size_t i = 0; i < nr; ++i)
            std::memcpy(static_cast<char*>(host) + (q * per + i) * host_pitch,
                        R.mem + b * R.bytes + i * span, width);
    }
    R.next = (int)((first + pieces) % kBufs);
    return hipSuccess;
}

}  // namespace hplx
