// Large device results to the caller's pageable memory through pinned slots:
// the order of the steps.  The runtime's part (queueing a transfer into a
// slot, waiting for it) is an Io, so that the order can be checked on the
// host without a GPU:
//   Err                        an error, Err{} for none
//   Err plain(dst, bytes)      the runtime's own copy
//   bool pinned(dst)           the destination is pinned memory
//   bool ready()               the slots are there, or could be made
//   Err begin()                once in every thread, before its transfers
//   Err queue(slot, at, len)   starts the transfer of len bytes at offset at
//   Err wait(slot)             waits for the slot's last transfer
//   void drain()               waits for every transfer queued so far
//   unsigned char* slot(s)     a slot's memory
//   std::thread thread(f)      a thread that runs f
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace flgpu {

constexpr size_t kStageSlot = 1 << 20;
constexpr size_t kStageMin = 4 << 20;              // smaller copies go the runtime's way
constexpr int kStageThreads = 4, kStageDepth = 3;  // slots in flight per thread
constexpr int kStageSlots = kStageThreads * kStageDepth;

// Each thread takes every T-th chunk of a slot's size: the transfer (55 GB/s
// into pinned memory) then overlaps the copies to the destination, and
// several threads share the page faults of memory the caller has just
// allocated.  No transfer into a slot is in flight when this returns: after
// an error the queued ones are waited for, since the next copy -- of another
// context, on another stream -- takes the same slots.
template <class Io>
typename Io::Err staged_copy(Io& io, void* dst, size_t bytes) {
    using Err = typename Io::Err;
    const int64_t nch = (int64_t)((bytes + kStageSlot - 1) / kStageSlot);
    const int T = (int)std::min<int64_t>(kStageThreads, (nch + 1) / 2);
    Err err[kStageThreads] = {};
    auto size = [&](int64_t ch) { return std::min(kStageSlot, bytes - (size_t)ch * kStageSlot); };
    auto work = [&](int t) {
        auto slot = [&](int64_t q) { return t * kStageDepth + (int)(q % kStageDepth); };
        Err e = io.begin();
        const int64_t mine = (nch - t + T - 1) / T;
        for (int64_t q = 0; q < mine + kStageDepth - 1 && e == Err{}; q++) {
            if (q < mine) {  // queue chunk q of this thread
                const int64_t ch = t + q * T;
                e = io.queue(slot(q), (size_t)ch * kStageSlot, size(ch));
            }
            const int64_t r = q - (kStageDepth - 1);
            if (r >= 0 && r < mine && e == Err{}) {  // and take the one queued kStageDepth - 1 before it
                const int64_t ch = t + r * T;
                e = io.wait(slot(r));
                if (e == Err{})
                    std::memcpy((unsigned char*)dst + ch * kStageSlot, io.slot(slot(r)), size(ch));
            }
        }
        err[t] = e;
    };
    std::thread pool[kStageThreads];
    int started = 1;
    try {
        for (; started < T; started++) pool[started] = io.thread([&work, started] { work(started); });
    } catch (const std::exception&) {  // no more threads, or no memory for one: this one takes their share
    }
    work(0);
    for (int t = 1; t < started; t++) pool[t].join();
    for (int t = started; t < T; t++) work(t);
    for (int t = 0; t < T; t++)
        if (err[t] != Err{}) {
            io.drain();
            return err[t];
        }
    return Err{};
}

// A copy of any size: through the slots, guarded by mu, when it is large and
// goes to pageable memory; the runtime's way to pinned memory (one direct
// transfer), and when another thread has the slots or the memory for them is
// not to be had.
template <class Io>
typename Io::Err copy_to_host(Io& io, std::mutex& mu, void* dst, size_t bytes) {
    if (bytes > kStageMin && !io.pinned(dst)) {
        std::unique_lock<std::mutex> lk(mu, std::try_to_lock);
        if (lk.owns_lock() && io.ready()) return staged_copy(io, dst, bytes);
    }
    return bytes ? io.plain(dst, bytes) : typename Io::Err{};
}

}  // namespace flgpu
