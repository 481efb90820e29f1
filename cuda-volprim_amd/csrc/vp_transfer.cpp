// vp_transfer.cpp — device scratch kept between calls, and copies between
// device memory and ordinary host memory.
//
// A call allocates nothing once its context has served one of its size: an
// allocation and its free cost up to 100 us each, against 60 us of kernels in
// the smallest renders.  Ordinary host memory goes through pinned slots of
// the context: the runtime's own path for it runs at the speed of one host
// thread, 3.4 of the 5.1 ms of building and exporting 250000 primitives.
#include <atomic>
#include <cstring>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "vp_internal.h"

namespace {

vp_status fail(vp_status code, const std::string& msg) {
    vp_set_error(msg);
    return code;
}

// Pinned slots of ctx, allocated on first use: one for copies that fit it,
// all of them with an event each for longer ones.  Held under ctx->mu.
bool ensure_stage(vp_context* ctx, uint32_t slots) {
    if (ctx->stage_slots >= slots) return true;
    for (uint32_t k = 0; slots > 1 && k < kStageSlots; ++k)
        if (!ctx->stage_ev[k] && hipEventCreateWithFlags(&ctx->stage_ev[k], hipEventDisableTiming) != hipSuccess) {
            ctx->stage_ev[k] = nullptr;
            return false;
        }
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    ctx->stage = nullptr;
    ctx->stage_slots = 0;
    void* p = nullptr;
    if (hipHostMalloc(&p, slots * kStageSlot, hipHostMallocDefault) != hipSuccess) return false;
    ctx->stage = static_cast<char*>(p);
    ctx->stage_slots = slots;
    return true;
}

// Memory that the runtime knows (pinned, device, managed) is copied directly.
bool ordinary(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess && a.type != hipMemoryTypeUnregistered) return false;
    (void)hipGetLastError();
    return true;
}

// Runs work on this thread and on up to kStageThreads - 1 more.
template <typename F>
void on_threads(int device, size_t chunks, F&& work) {
    std::vector<std::thread> pool;
    const size_t extra = std::max<size_t>(1, std::min<size_t>(kStageThreads, chunks / 2)) - 1;
    try {
        pool.reserve(extra);
        for (size_t k = 0; k < extra; ++k)
            pool.emplace_back([&work, device] {
                (void)hipSetDevice(device);
                work();
            });
    } catch (const std::exception&) {  // fewer threads, the same work
    }
    work();
    for (auto& t : pool) t.join();
}

// Waits for s where a function returns (an error, an exception) with copies
// under way, before the lock of the slots is released: they are the next
// call's then, and the caller's memory its own again.
struct WaitOnFailure {
    hipStream_t s;
    bool armed = true;
    ~WaitOnFailure() {
        if (armed) (void)hipStreamSynchronize(s);
    }
};

struct Slots {
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};
    std::atomic<size_t> queued[kStageSlots];  // chunk last queued in the slot, plus one
    Slots() {
        for (auto& q : queued) q.store(0, std::memory_order_relaxed);
    }
    void note(hipError_t e) {
        if (e != hipSuccess) err.store(e, std::memory_order_relaxed);
    }
    bool good() const { return err.load(std::memory_order_relaxed) == hipSuccess; }
    // until chunk c has been queued in its slot; chunks are taken in order, so
    // its holder waits for none after it
    void wait_queued(size_t c) const {
        while (queued[c % kStageSlots].load(std::memory_order_acquire) != c + 1) std::this_thread::yield();
    }
    void set_queued(size_t c) { queued[c % kStageSlots].store(c + 1, std::memory_order_release); }
};

}  // namespace

bool vp_give_back_scratch(vp_context* ctx) {
    if (ctx->scratch_busy.exchange(true, std::memory_order_acquire)) return false;
    const bool any = ctx->scratch != nullptr;
    if (any) (void)hipFree(ctx->scratch);
    ctx->scratch = nullptr;
    ctx->scratch_bytes = 0;
    ctx->scratch_busy.store(false, std::memory_order_release);
    return any;
}

hipError_t vp_device_malloc(vp_context* ctx, void** p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess || !vp_give_back_scratch(ctx)) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

void ScratchLease::release() {
    if (!p) return;
    if (!done) (void)hipStreamSynchronize(stream);
    if (owned)
        (void)hipFree(p);
    else
        ctx->scratch_busy.store(false, std::memory_order_release);
    p = nullptr;
}

vp_status vp_lease_scratch(vp_context* ctx, size_t bytes, hipStream_t s, ScratchLease& lease) {
    lease.ctx = ctx;
    lease.stream = s;
    const bool mine = bytes <= kScratchKeep && !ctx->scratch_busy.exchange(true, std::memory_order_acquire);
    if (mine && ctx->scratch_bytes < bytes) {
        if (ctx->scratch) (void)hipFree(ctx->scratch);
        ctx->scratch_bytes = 0;
        if (hipMalloc(&ctx->scratch, bytes) == hipSuccess)
            ctx->scratch_bytes = bytes;
        else
            ctx->scratch = nullptr;
    }
    if (mine) {
        lease.p = ctx->scratch;
        if (!lease.p) ctx->scratch_busy.store(false, std::memory_order_release);
    } else {
        lease.owned = vp_device_malloc(ctx, &lease.p, bytes) == hipSuccess;
        if (!lease.owned) lease.p = nullptr;
    }
    if (lease.p) return VP_OK;
    (void)hipGetLastError();
    return fail(VP_ERR_OOM, "cannot allocate " + std::to_string(bytes) + " bytes of device memory");
}

vp_status vp_copy_out(vp_context* ctx, const HostCopy* copies, size_t n, hipStream_t s) {
    std::lock_guard<std::mutex> lk(ctx->mu);
    WaitOnFailure wait{s};
    // what leaves the device in one copy: a part, a slot's worth of a longer
    // one, or several short ones that lie one after the other
    struct Piece {
        char* dst;
        size_t offset, bytes;  // in its run
    };
    struct Run {
        const char* src;
        size_t bytes, first, end;  // pieces
    };
    std::vector<Piece> pieces;
    std::vector<Run> runs;
    for (size_t i = 0; i < n; ++i) {
        const char* src = static_cast<const char*>(copies[i].src);
        if (copies[i].bytes == 0) continue;
        if (!ordinary(copies[i].dst)) {
            VP_HIP_TRY(hipMemcpyAsync(copies[i].dst, src, copies[i].bytes, hipMemcpyDeviceToHost, s));
            continue;
        }
        for (size_t o = 0; o < copies[i].bytes; o += kStageSlot) {
            const size_t bytes = std::min(kStageSlot, copies[i].bytes - o);
            const bool joins = o == 0 && copies[i].joins && !runs.empty() && src >= runs.back().src + runs.back().bytes &&
                               src < runs.back().src + runs.back().bytes + 256 &&
                               src + bytes <= runs.back().src + kStageSlot;
            if (!joins) runs.push_back({src + o, 0, pieces.size(), pieces.size()});
            Run& r = runs.back();
            pieces.push_back({static_cast<char*>(copies[i].dst) + o, static_cast<size_t>(src + o - r.src), bytes});
            r.bytes = pieces.back().offset + bytes;
            ++r.end;
        }
    }
    size_t total = 0;
    for (const Run& r : runs) total += (r.bytes + 15) / 16 * 16;
    if (!ensure_stage(ctx, total <= kStageSlot ? 1u : kStageSlots)) {
        (void)hipGetLastError();
        for (const Run& r : runs)
            for (size_t k = r.first; k < r.end; ++k)
                VP_HIP_TRY(hipMemcpyAsync(pieces[k].dst, r.src + pieces[k].offset, pieces[k].bytes, hipMemcpyDeviceToHost,
                                          s));
        VP_HIP_TRY(hipStreamSynchronize(s));
        wait.armed = false;
        return VP_OK;
    }
    const auto deliver = [&](const Run& r, const char* from) {
        for (size_t k = r.first; k < r.end; ++k) std::memcpy(pieces[k].dst, from + pieces[k].offset, pieces[k].bytes);
    };
    if (total <= kStageSlot) {
        // everything in one slot, written there by a kernel: one launch and
        // one wait (a copy through the runtime takes two of its launches)
        char* at = ctx->stage;
        for (size_t i = 0; i < runs.size(); i += kCopyParts) {
            CopyParts cp{};
            for (uint32_t k = 0; k < kCopyParts && i + k < runs.size(); ++k) {
                cp.src[k] = reinterpret_cast<const uint32_t*>(runs[i + k].src);
                cp.dst[k] = reinterpret_cast<uint32_t*>(at);
                cp.words[k] = static_cast<uint32_t>(runs[i + k].bytes / 4);
                at += (runs[i + k].bytes + 15) / 16 * 16;
            }
            VP_HIP_TRY(vp_launch_copy_parts(cp, s));
        }
        VP_HIP_TRY(hipStreamSynchronize(s));
        wait.armed = false;
        at = ctx->stage;
        for (const Run& r : runs) {
            deliver(r, at);
            at += (r.bytes + 15) / 16 * 16;
        }
        return VP_OK;
    }
    Slots S;
    auto queue = [&](size_t c) {
        char* slot = ctx->stage + (c % kStageSlots) * kStageSlot;
        if (S.good()) S.note(hipMemcpyAsync(slot, runs[c].src, runs[c].bytes, hipMemcpyDeviceToHost, s));
        if (S.good()) S.note(hipEventRecord(ctx->stage_ev[c % kStageSlots], s));
        S.set_queued(c);
    };
    for (size_t c = 0; c < kStageSlots && c < runs.size(); ++c) queue(c);
    on_threads(ctx->device, runs.size(), [&] {
        for (size_t c; (c = S.next.fetch_add(1)) < runs.size();) {
            S.wait_queued(c);
            if (S.good()) S.note(hipEventSynchronize(ctx->stage_ev[c % kStageSlots]));
            if (S.good()) deliver(runs[c], ctx->stage + (c % kStageSlots) * kStageSlot);
            if (c + kStageSlots < runs.size()) queue(c + kStageSlots);
        }
    });
    VP_HIP_TRY(static_cast<hipError_t>(S.err.load()));
    VP_HIP_TRY(hipStreamSynchronize(s));
    wait.armed = false;
    return VP_OK;
}

vp_status vp_copy_in(vp_context* ctx, void* dst, const void* src, size_t elem, size_t count,
                     bool (*check)(const void* rows, size_t count), bool* good, hipStream_t s) {
    std::lock_guard<std::mutex> lk(ctx->mu);
    WaitOnFailure wait{s};
    const char* from = static_cast<const char*>(src);
    char* to = static_cast<char*>(dst);
    const size_t rows = kStageSlot / elem;
    if (count <= rows || !ensure_stage(ctx, kStageSlots)) {
        (void)hipGetLastError();
        *good = check(src, count);
        if (*good) VP_HIP_TRY(hipMemcpyAsync(dst, src, elem * count, hipMemcpyHostToDevice, s));
        wait.armed = false;
        return VP_OK;
    }
    const size_t chunks = (count + rows - 1) / rows;
    Slots S;
    std::atomic<bool> ok{true};
    on_threads(ctx->device, chunks, [&] {
        for (size_t c; (c = S.next.fetch_add(1)) < chunks;) {
            const size_t m = std::min(rows, count - c * rows);
            char* slot = ctx->stage + (c % kStageSlots) * kStageSlot;
            if (c >= kStageSlots) {
                S.wait_queued(c - kStageSlots);
                if (S.good()) S.note(hipEventSynchronize(ctx->stage_ev[c % kStageSlots]));
            }
            if (!check(from + c * rows * elem, m)) ok.store(false, std::memory_order_relaxed);
            if (S.good()) {
                std::memcpy(slot, from + c * rows * elem, m * elem);
                S.note(hipMemcpyAsync(to + c * rows * elem, slot, m * elem, hipMemcpyHostToDevice, s));
            }
            if (S.good()) S.note(hipEventRecord(ctx->stage_ev[c % kStageSlots], s));
            S.set_queued(c);
        }
    });
    *good = ok.load();
    VP_HIP_TRY(static_cast<hipError_t>(S.err.load()));
    VP_HIP_TRY(hipStreamSynchronize(s));  // the slots are the next call's
    wait.armed = false;
    return VP_OK;
}
