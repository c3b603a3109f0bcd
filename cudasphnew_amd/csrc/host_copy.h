// host_copy.h -- device results into a caller's pageable array.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstring>

namespace sph {

// A copy straight into pageable memory goes through the runtime's own path,
// which costs more than the bytes: measured into fresh pages, 45 us for 64
// KiB, 220 for 384 KiB, 1000 for 4 MiB, 2910 for 12 MiB.  Through pinned slots
// (a chunk crosses the bus while the host copies the one before it) 19, 71,
// 750 and 2220 us; up to a chunk there is nothing to overlap and one copy is
// the fastest.  Each owner has its own slots, allocated on first use -- one
// for reads of up to a chunk, all with the first larger one -- and freed with
// it.  Where they cannot be had the runtime's own path serves.
struct HostCopy {
    static constexpr size_t kChunk = 512u << 10;
    static constexpr int kSlots = 4;
    static constexpr size_t kTail = 64;   // the status word, behind the slots

    char* pin = nullptr;
    int slots = 0;
    hipEvent_t done[kSlots] = {};

    HostCopy() = default;
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;

    hipError_t init(size_t bytes) {
        const int want = bytes <= kChunk ? 1 : kSlots;
        if (slots >= want) return hipSuccess;
        release();
        for (int i = 0; i < want && want > 1; ++i) {
            hipError_t e = hipEventCreateWithFlags(&done[i], hipEventDisableTiming);
            if (e != hipSuccess) return e;
        }
        hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&pin), kChunk * want + kTail, 0);
        if (e == hipSuccess) slots = want;
        return e;
    }

    void release() {
        if (pin) (void)hipHostFree(pin);
        for (hipEvent_t& e : done) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        pin = nullptr;
        slots = 0;
    }

    // bytes of device memory src into dst, after the work on st; waits for
    // them.  word (may be null): a device status word, copied first; nothing
    // is written to dst unless accept takes its value.
    template <class Accept>
    hipError_t read(hipStream_t st, void* dst, const void* src, size_t bytes, const uint32_t* word, Accept accept) {
        if (init(bytes) != hipSuccess) {
            (void)hipGetLastError();
            return read_direct(st, dst, src, bytes, word, accept);
        }
        hipError_t e = hipSuccess;
        if (word) {
            e = hipMemcpyAsync(pinned_word(), word, sizeof(uint32_t), hipMemcpyDeviceToHost, st);
            if (e != hipSuccess) return e;
        }
        const size_t n = (bytes + kChunk - 1) / kChunk;
        auto size = [&](size_t k) { return std::min(kChunk, bytes - k * kChunk); };
        auto send = [&](size_t k) {
            hipError_t r = hipMemcpyAsync(pin + k % kSlots * kChunk, static_cast<const char*>(src) + k * kChunk,
                                          size(k), hipMemcpyDeviceToHost, st);
            return r == hipSuccess && n > 1 ? hipEventRecord(done[k % kSlots], st) : r;
        };
        for (size_t k = 0; k < std::min<size_t>(n, kSlots) && e == hipSuccess; ++k) e = send(k);
        if (n <= 1 && e == hipSuccess) e = hipStreamSynchronize(st);
        for (size_t k = 0; k < n && e == hipSuccess; ++k) {
            if (n > 1) e = hipEventSynchronize(done[k % kSlots]);
            if (e != hipSuccess) break;
            if (k == 0 && word && !accept(*pinned_word())) return hipStreamSynchronize(st);
            std::memcpy(static_cast<char*>(dst) + k * kChunk, pin + k % kSlots * kChunk, size(k));
            if (k + kSlots < n) e = send(k + kSlots);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(st);   // nothing still writes the slots
        return e;
    }

    hipError_t read(hipStream_t st, void* dst, const void* src, size_t bytes) {
        return read(st, dst, src, bytes, nullptr, [](uint32_t) { return true; });
    }

  private:
    template <class Accept>
    static hipError_t read_direct(hipStream_t st, void* dst, const void* src, size_t bytes, const uint32_t* word,
                                  Accept accept) {
        uint32_t value = 0;
        hipError_t e = hipSuccess;
        if (word) {
            e = hipMemcpyAsync(&value, word, sizeof(value), hipMemcpyDeviceToHost, st);
            const hipError_t w = hipStreamSynchronize(st);
            if (e == hipSuccess) e = w;
            if (e != hipSuccess || !accept(value)) return e;
        }
        e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        const hipError_t w = hipStreamSynchronize(st);
        return e == hipSuccess ? w : e;
    }

    uint32_t* pinned_word() const { return reinterpret_cast<uint32_t*>(pin + kChunk * slots); }
};

}  // namespace sph
