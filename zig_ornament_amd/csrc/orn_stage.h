// orn_stage.h -- copies between the caller's host memory and the device
// through a pinned buffer the device context keeps.
//
// The runtime copies pageable memory through a staging buffer of its own, one
// part after the other: 33 MB (a 1080p framebuffer) take 1.9 ms where the link
// needs 0.6. Here the link fills parts of the buffer while threads empty the
// parts already there, which also spreads the page faults of a fresh
// destination: 33 MB in 0.88 ms, a million rays and their hits 4.1 -> 3.1 ms,
// a 1080p radiance-cache frame with its framebuffer 2.7 -> 1.8 ms, 500x500 at
// 1 spp 0.51 -> 0.45 ms. One buffer per context, allocated by the first copy, freed
// with the context. Memory the runtime knows (pinned, managed, a device's) is
// reached by the copy engines without it and may not be the host's to touch:
// its copies go straight there.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

namespace orn_rt {

class HostStage {
public:
    static constexpr size_t kBytes = size_t(32) << 20;      // pinned memory
    static constexpr size_t kKeepDevice = size_t(64) << 20;  // device workspace kept at most
    static constexpr int kParts = 8;
    static constexpr size_t kPart = kBytes / kParts;

    std::mutex mutex;  // held for a whole call: the buffer has one user at a time

    // Whether p is ordinary host memory.
    static bool pageable(const void *p)
    {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // not known
        return true;
    }

    // The calls below need the mutex. Copies are ordered on `st` after the
    // work already there.

    // Pinned memory, or null (none to be had: the callers copy directly).
    char *pinned()
    {
        if (!pin_ && !tried_) {
            tried_ = true;
            if (hipHostMalloc(reinterpret_cast<void **>(&pin_), kBytes, hipHostMallocDefault) != hipSuccess) pin_ = nullptr;
            for (hipEvent_t &e : events_)
                if (pin_ && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) release_pinned();
            (void)hipGetLastError();
        }
        return pin_;
    }

    // Device memory of at least `bytes` for the length of a call; kept up to
    // kKeepDevice, larger ones belong to the caller (*own).
    hipError_t workspace(size_t bytes, void **p, bool *own)
    {
        *own = bytes > kKeepDevice;
        if (*own) return hipMalloc(p, bytes);
        if (bytes > dev_bytes_) {
            if (dev_) (void)hipFree(dev_);
            dev_ = nullptr;
            dev_bytes_ = 0;
            const hipError_t e = hipMalloc(&dev_, bytes);
            if (e != hipSuccess) return e;
            dev_bytes_ = bytes;
        }
        *p = dev_;
        return hipSuccess;
    }

    // Device to host; returns when dst is filled.
    hipError_t to_host(void *dst, const void *src, size_t bytes, int device, hipStream_t st)
    {
        if (!pageable(dst) || !pinned()) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
            return e != hipSuccess ? e : hipStreamSynchronize(st);
        }
        for (size_t at = 0; at < bytes; at += kBytes) {
            const hipError_t e = part_to_host(static_cast<char *>(dst) + at, static_cast<const char *>(src) + at,
                                              std::min(kBytes, bytes - at), device, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

    // Host to device in pieces of at most `piece` bytes (at most kPart);
    // after(begin, bytes) enqueues what follows each piece. src and the buffer may
    // be reused after `st` has been waited for.
    template <typename After>
    hipError_t to_device(void *dst, const void *src, size_t bytes, size_t piece, hipStream_t st, After after)
    {
        hipError_t e = hipSuccess;
        const bool staged = pageable(src) && pinned();
        size_t i = 0;
        for (size_t at = 0; at < bytes && e == hipSuccess; at += piece, i++) {
            const size_t n = std::min(piece, bytes - at);
            const char *from = static_cast<const char *>(src) + at;
            if (staged) {
                char *p = pin_ + (i % kParts) * kPart;
                if (i >= kParts) e = hipEventSynchronize(events_[i % kParts]);
                if (e == hipSuccess) {
                    std::memcpy(p, from, n);
                    e = hipMemcpyAsync(static_cast<char *>(dst) + at, p, n, hipMemcpyHostToDevice, st);
                }
                if (e == hipSuccess) e = hipEventRecord(events_[i % kParts], st);
            } else {
                e = hipMemcpyAsync(static_cast<char *>(dst) + at, from, n, hipMemcpyHostToDevice, st);
            }
            if (e == hipSuccess) e = after(at, n);
        }
        return e;
    }

    // With the context's device current and its stream idle.
    void release()
    {
        release_pinned();
        if (dev_) (void)hipFree(dev_);
        dev_ = nullptr;
        dev_bytes_ = 0;
    }

private:
    // One bufferful, in parts of at least 1 MB (a part costs some 12 us to
    // enqueue): helpers and, once all parts are on their way, this thread copy
    // out what has arrived.
    hipError_t part_to_host(char *dst, const char *src, size_t bytes, int device, hipStream_t st)
    {
        constexpr size_t kLeast = size_t(1) << 20, kHelped = size_t(6) << 20;
        const size_t part = std::max(kLeast, bytes / kParts / 4096 * 4096 + 4096);  // at most kParts of them
        const int parts = static_cast<int>((bytes + part - 1) / part);
        std::atomic<int> next{0}, issued{0};
        std::atomic<hipError_t> error{hipSuccess};
        auto drain = [&] {
            for (int i = next++; i < parts; i = next++) {
                while (issued.load(std::memory_order_acquire) <= i) std::this_thread::yield();
                const hipError_t e = error.load() != hipSuccess ? error.load() : hipEventSynchronize(events_[i]);
                if (e != hipSuccess) error.store(e);
                else std::memcpy(dst + part * i, pin_ + part * i, std::min(part, bytes - part * i));
            }
        };
        std::thread helpers[2];
        if (bytes >= kHelped) {
            for (std::thread &h : helpers) {
                try {
                    h = std::thread([&] {
                        (void)hipSetDevice(device);
                        drain();
                    });
                } catch (...) {  // fewer threads, then
                    break;
                }
            }
        }
        for (int i = 0; i < parts; i++) {
            const size_t at = part * i;
            hipError_t e = error.load();
            if (e == hipSuccess)
                e = hipMemcpyAsync(pin_ + at, src + at, std::min(part, bytes - at), hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(events_[i], st);
            if (e != hipSuccess) error.store(e);
            issued.store(i + 1, std::memory_order_release);
        }
        drain();
        for (std::thread &h : helpers)
            if (h.joinable()) h.join();
        if (error.load() != hipSuccess) (void)hipStreamSynchronize(st);
        return error.load();
    }

    void release_pinned()
    {
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
        for (hipEvent_t &e : events_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    char *pin_ = nullptr;
    bool tried_ = false;
    hipEvent_t events_[kParts] = {};
    void *dev_ = nullptr;
    size_t dev_bytes_ = 0;
};

}  // namespace orn_rt
