// host_stage.cpp - the ring of pinned chunks behind HostStage.
#include "host_stage.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "crt_runtime.h"

namespace crt {

int HostStage::init(int device) {
    device_ = device;
    HIP_TRY(hipHostMalloc((void**)&pin_, kChunk * kSlots, hipHostMallocDefault));
    for (hipEvent_t& e : ev_) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return CRT_OK;
}

void HostStage::release() {
    for (int k = 0; k < kSlots; ++k) {
        if (used_[k]) (void)hipEventSynchronize(ev_[k]);
        if (ev_[k]) (void)hipEventDestroy(ev_[k]);
        ev_[k] = nullptr;
        used_[k] = false;
    }
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
}

// The ring's next slot, once its last copy has completed.
hipError_t HostStage::claim(int& slot) {
    slot = next_;
    next_ = (next_ + 1) % kSlots;
    if (!used_[slot]) return hipSuccess;
    used_[slot] = false;
    return hipEventSynchronize(ev_[slot]);
}

hipError_t HostStage::push(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    if (bytes > kChunk) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    int slot;
    hipError_t e = claim(slot);
    if (e != hipSuccess) return e;
    std::memcpy(pin_ + slot * kChunk, src, bytes);
    e = hipMemcpyAsync(dst, pin_ + slot * kChunk, bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
    used_[slot] = true;
    return e;
}

hipError_t HostStage::fetch(const Copy* list, int n, hipStream_t s) {
    struct Piece { char* host; const char* dev; size_t bytes; };
    size_t total = 0;
    for (int k = 0; k < n; ++k) total += list[k].bytes;
    if (total == 0) return hipStreamSynchronize(s);
    if (total <= kChunk) {
        // one slot for everything
        int slot;
        hipError_t e = claim(slot);
        size_t off = 0;
        for (int k = 0; k < n && e == hipSuccess; ++k) {
            if (list[k].bytes) e = hipMemcpyAsync(pin_ + slot * kChunk + off, list[k].dev, list[k].bytes, hipMemcpyDeviceToHost, s);
            off += list[k].bytes;
        }
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        if (e != hipSuccess) return e;
        off = 0;
        for (int k = 0; k < n; ++k) {
            if (list[k].bytes) std::memcpy(list[k].host, pin_ + slot * kChunk + off, list[k].bytes);
            off += list[k].bytes;
        }
        return hipSuccess;
    }
    // pieces of at most a chunk; short ones share a slot (a slot's event and its wait cost more than the
    // copy of a 64x64 image)
    std::vector<Piece> pieces;
    std::vector<size_t> first;   // first piece of each slotful
    size_t room = 0;
    for (int k = 0; k < n; ++k)
        for (size_t off = 0; off < list[k].bytes; off += kChunk) {
            const size_t b = std::min(kChunk, list[k].bytes - off);
            if (b > room) { first.push_back(pieces.size()); room = kChunk; }
            room -= b;
            pieces.push_back(Piece{(char*)list[k].host + off, (const char*)list[k].dev + off, b});
        }
    const size_t np = first.size();
    first.push_back(pieces.size());
    for (int k = 0; k < kSlots; ++k) {   // the ring is this call's
        if (!used_[k]) continue;
        used_[k] = false;
        const hipError_t e = hipEventSynchronize(ev_[k]);
        if (e != hipSuccess) return e;
    }
    std::atomic<size_t> queued{0}, taken{0}, err{0};
    std::vector<std::atomic<char>> done(np);
    for (auto& d : done) d.store(0, std::memory_order_relaxed);
    // takes queued slotfuls in order: waits for the copies into the ring, copies them out
    auto drain_one = [&](size_t k) {
        const int slot = (int)(k % kSlots);
        const hipError_t e = hipEventSynchronize(ev_[slot]);
        if (e != hipSuccess) err.store((size_t)e);
        const char* from = pin_ + slot * kChunk;
        for (size_t p = first[k]; p < first[k + 1] && e == hipSuccess; from += pieces[p++].bytes)
            std::memcpy(pieces[p].host, from, pieces[p].bytes);
        done[k].store(1, std::memory_order_release);
    };
    auto worker = [&]() {
        (void)hipSetDevice(device_);
        for (;;) {
            const size_t k = taken.fetch_add(1);
            if (k >= np) return;
            while (queued.load(std::memory_order_acquire) <= k) std::this_thread::yield();
            drain_one(k);
        }
    };
    std::thread helper[kThreads];
    int started = 0;
    try {
        const int want = total >= kParallel ? (int)std::min<size_t>(kThreads, np / 2) : 0;
        for (; started < want; ++started) helper[started] = std::thread(worker);
    } catch (const std::system_error&) {
        // fewer threads, or none: this one drains below
    }
    for (size_t k = 0; k < np; ++k) {
        // what the slot held must be out; without helpers this thread takes it
        while (k >= (size_t)kSlots && !done[k - kSlots].load(std::memory_order_acquire)) {
            if (started) { std::this_thread::yield(); continue; }
            drain_one(taken.fetch_add(1));
        }
        const int slot = (int)(k % kSlots);
        hipError_t e = (hipError_t)err.load();
        char* to = pin_ + slot * kChunk;
        for (size_t p = first[k]; p < first[k + 1] && e == hipSuccess; to += pieces[p++].bytes)
            e = hipMemcpyAsync(to, pieces[p].dev, pieces[p].bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
        if (e != hipSuccess) err.store((size_t)e);   // the slots left are handed out and fail with it
        queued.store(k + 1, std::memory_order_release);
    }
    worker();
    for (int k = 0; k < started; ++k) helper[k].join();
    next_ = 0;
    if (err.load()) { (void)hipStreamSynchronize(s); return (hipError_t)err.load(); }
    return hipSuccess;
}

}  // namespace crt
