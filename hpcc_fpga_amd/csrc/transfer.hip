#include "transfer.hpp"

#include <algorithm>
#include <cstring>

namespace hplx {

namespace {

// Memory that the runtime made or has registered (pinned, managed, device): its
// copies need no staging.
bool runtime_knows(const void* p) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t HostStage::make() {
    if (mem_) return hipSuccess;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&mem_), kBufs * kBytes,
                                 hipHostMallocDefault);
    if (e != hipSuccess) {
        mem_ = nullptr;
        return e;
    }
    for (hipEvent_t& ev : ev_) {
        e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) {
            ev = nullptr;
            free();
            return e;
        }
    }
    return hipSuccess;
}

void HostStage::free() {
    for (hipEvent_t& ev : ev_) {
        if (ev) {
            (void)hipEventSynchronize(ev);  // its last copy
            (void)hipEventDestroy(ev);
        }
        ev = nullptr;
    }
    if (mem_) (void)hipHostFree(mem_);
    mem_ = nullptr;
}

hipError_t HostStage::to_device(hipStream_t s, void* dev, size_t dev_pitch, const void* host,
                                size_t host_pitch, size_t width, size_t rows) {
    if (!width || !rows) return hipSuccess;
    // bytes from a row's start to the next one's (or to its own end)
    const size_t span = rows > 1 ? dev_pitch : width;
    if (width > span) return hipErrorInvalidValue;
    if (runtime_knows(host))
        return hipMemcpy2DAsync(dev, dev_pitch, host, host_pitch, width, rows,
                                hipMemcpyHostToDevice, s);
    hipError_t e = make();
    if (e != hipSuccess) return e;
    if (span > kBytes) {  // row by row, each in pieces
        for (size_t r = 0; r < rows && e == hipSuccess; ++r)
            e = to_device(s, static_cast<char*>(dev) + r * dev_pitch,
                          static_cast<const char*>(host) + r * host_pitch, width);
        return e;
    }
    const size_t per = std::max<size_t>(1, kBytes / span);
    for (size_t r = 0; r < rows; r += per) {
        const size_t nr = std::min(per, rows - r);
        const int b = next_;
        next_ = (next_ + 1) % kBufs;
        e = hipEventSynchronize(ev_[b]);  // the buffer's previous copy
        if (e != hipSuccess) return e;
        char* buf = mem_ + b * kBytes;
        for (size_t i = 0; i < nr; ++i) {
            std::memcpy(buf + i * span, static_cast<const char*>(host) + (r + i) * host_pitch,
                        width);
            if (i + 1 < nr || r + nr < rows) std::memset(buf + i * span + width, 0, span - width);
        }
        const size_t bytes = r + nr < rows ? nr * span : (nr - 1) * span + width;
        e = hipMemcpyAsync(static_cast<char*>(dev) + r * span, buf, bytes, hipMemcpyHostToDevice,
                           s);
        if (e == hipSuccess) e = hipEventRecord(ev_[b], s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t HostStage::to_device(hipStream_t s, void* dev, const void* host, size_t bytes) {
    if (runtime_knows(host)) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    const size_t whole = bytes / kBytes, done = whole * kBytes;
    hipError_t e = to_device(s, dev, kBytes, host, kBytes, kBytes, whole);
    if (e != hipSuccess || done == bytes) return e;
    return to_device(s, static_cast<char*>(dev) + done, bytes - done,
                     static_cast<const char*>(host) + done, bytes - done, bytes - done, 1);
}

hipError_t HostStage::to_host(hipStream_t s, void* host, const void* dev, size_t bytes) {
    if (runtime_knows(host)) {
        hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    const size_t whole = bytes / kBytes, done = whole * kBytes;
    hipError_t e = to_host(s, host, kBytes, dev, kBytes, kBytes, whole);
    if (e != hipSuccess || done == bytes) return e;
    return to_host(s, static_cast<char*>(host) + done, bytes - done,
                   static_cast<const char*>(dev) + done, bytes - done, bytes - done, 1);
}

hipError_t HostStage::to_host(hipStream_t s, void* host, size_t host_pitch, const void* dev,
                              size_t dev_pitch, size_t width, size_t rows) {
    if (!width || !rows) return hipSuccess;
    const size_t span = rows > 1 ? dev_pitch : width;
    if (width > span) return hipErrorInvalidValue;
    if (runtime_knows(host)) {
        hipError_t e = hipMemcpy2DAsync(host, host_pitch, dev, dev_pitch, width, rows,
                                        hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    hipError_t e = make();
    if (e != hipSuccess) return e;
    if (span > kBytes) {
        for (size_t r = 0; r < rows && e == hipSuccess; ++r)
            e = to_host(s, static_cast<char*>(host) + r * host_pitch,
                        static_cast<const char*>(dev) + r * dev_pitch, width);
        return e;
    }
    const size_t per = std::max<size_t>(1, kBytes / span);
    const size_t pieces = (rows + per - 1) / per;
    const int first = next_;
    // up to kBufs pieces on their way while the oldest is unpacked
    for (size_t p = 0, q = 0; q < pieces; ++q) {
        for (; p < pieces && p < q + kBufs; ++p) {
            const size_t nr = std::min(per, rows - p * per);
            const size_t bytes = p + 1 < pieces ? nr * span : (nr - 1) * span + width;
            const int b = (int)((first + p) % kBufs);
            if (p < (size_t)kBufs) {  // what an earlier call left in the buffer
                e = hipEventSynchronize(ev_[b]);
                if (e != hipSuccess) return e;
            }
            e = hipMemcpyAsync(mem_ + b * kBytes, static_cast<const char*>(dev) + p * per * span,
                               bytes, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[b], s);
            if (e != hipSuccess) return e;
        }
        const int b = (int)((first + q) % kBufs);
        e = hipEventSynchronize(ev_[b]);
        if (e != hipSuccess) return e;
        const size_t nr = std::min(per, rows - q * per);
        for (size_t i = 0; i < nr; ++i)
            std::memcpy(static_cast<char*>(host) + (q * per + i) * host_pitch,
                        mem_ + b * kBytes + i * span, width);
    }
    next_ = (int)((first + pieces) % kBufs);
    return hipSuccess;
}

}  // namespace hplx
