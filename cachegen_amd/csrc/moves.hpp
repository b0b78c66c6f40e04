// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Bytes between pinned host memory and device memory, and how far they have got.
#pragma once

#include <new>
#include <vector>

namespace {

// The container's sections cross the bus by the copy engines.  A kernel that does the same is faster on a quiet GPU: a
// copy is set apart from the kernels before and after it (1 MB down behind a kernel 20 us more than its bytes, up before
// one 11) and from the copy before it (5 to 15).  But beside a model that keeps the compute units busy every launch waits
// until the model's kernel has no more workgroups to send.  By kernel / by copies, us: beside matrix products of
// 0.8 ms each, one behind another, eight chunks (59 MB) decoded 12600 / 2000, one chunk 4500 / 1230, eight chunks
// stored 15400 / 2920, one 4230 / 390; on a quiet GPU one chunk to bytes and back 442 / 493, a chunk of counts from bytes
// 130 / 147, store and retrieve of 59 MB 3070 / 3340, merge of 44 MB 1011 / 907.
//
// How far they are the host sees by asking an event, which takes 0.1 us and needs no compute unit either; an event's record
// is 1 us.  Events are kept, up to kKeptEvents a device: a new one takes 9 us.
class Events {
public:
    static hipEvent_t take(int device)
    {
        Kept &k = kept(device);
        {
            std::lock_guard<std::mutex> lock(k.mutex);
            if (!k.events.empty()) {
                const hipEvent_t e = k.events.back();
                k.events.pop_back();
                return e;
            }
        }
        hipEvent_t e = nullptr;
        return hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess ? e : nullptr;
    }

    static void give(int device, hipEvent_t e)
    {
        Kept &k = kept(device);
        {
            std::lock_guard<std::mutex> lock(k.mutex);
            if (k.events.size() < kKeptEvents) {
                k.events.push_back(e);
                return;
            }
        }
        (void)hipEventDestroy(e);
    }

private:
    static constexpr size_t kKeptEvents = 64;
    struct Kept {
        std::mutex mutex;
        std::vector<hipEvent_t> events;
        Kept() { events.reserve(kKeptEvents); }             // giving one back cannot fail
    };
    static Kept &kept(int device)
    {
        static Kept *const all = new Kept[64];              // for the process: a thread may still be at work when it ends
        return all[device & 63];
    }
};

// Places of a stream, in order, each with a number that *mark (an ordinary word of the host, ascending) shows once the stream
// is through with what was queued before.  One thread at a time asks; any may read the mark.
class Watch {
public:
    Watch(int32_t *mark, int device) : mark_(mark), device_(device) {}
    ~Watch()
    {
        for (; next_ < places_.size(); ++next_) Events::give(device_, places_[next_].event);
    }
    Watch(const Watch &) = delete;
    Watch &operator=(const Watch &) = delete;

    int add(int32_t value, hipStream_t stream)
    {
        hipEvent_t e = nullptr;
        try {
            if (places_.size() == places_.capacity()) places_.reserve(2 * places_.size() + 8);
            if (!(e = Events::take(device_))) return failed(hipGetLastError());
        } catch (const std::exception &what) {
            return fail(CG_ERR_LAUNCH, "moves: %s", what.what());
        }
        const hipError_t rc = hipEventRecord(e, stream);
        if (rc != hipSuccess) {
            Events::give(device_, e);
            return failed(rc);
        }
        places_.push_back({e, value});
        return CG_OK;
    }

    // Brings the mark up to date; an error if nothing is left that could bring it to `value`.
    int look(int32_t value)
    {
        while (next_ < places_.size()) {
            const hipError_t rc = query_event(places_[next_].event);
            if (rc == hipErrorNotReady) {
                (void)hipGetLastError();
                return CG_OK;
            }
            if (rc != hipSuccess) return failed(rc);
            passed();
        }
        return __atomic_load_n(mark_, __ATOMIC_ACQUIRE) < value ? nothing() : CG_OK;
    }

    int wait(int32_t value)
    {
        while (__atomic_load_n(mark_, __ATOMIC_ACQUIRE) < value) {
            if (next_ == places_.size()) return nothing();
            const hipError_t rc = hipEventSynchronize(places_[next_].event);
            if (rc != hipSuccess) return failed(rc);
            passed();
        }
        return CG_OK;
    }

private:
    struct Place {
        hipEvent_t event;
        int32_t value;
    };
    void passed()
    {
        __atomic_store_n(mark_, places_[next_].value, __ATOMIC_RELEASE);
        Events::give(device_, places_[next_].event);
        ++next_;
    }
    static int nothing() { return fail(CG_ERR_ARG, "moves: no place of the stream has that number"); }
    static int failed(hipError_t rc)
    {
        (void)hipGetLastError();
        return fail(CG_ERR_LAUNCH, "moves: %s", hipGetErrorString(rc));
    }

    int32_t *mark_;
    int device_;
    std::vector<Place> places_;
    size_t next_ = 0;
};

int move_bytes(const void *src, void *dst, int64_t n, bool to_host, hipStream_t stream)
{
    const hipError_t rc = hipMemcpyAsync(dst, src, (size_t)n, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, stream);
    if (rc == hipSuccess) return CG_OK;
    (void)hipGetLastError();
    return fail(CG_ERR_LAUNCH, "move_bytes: %s", hipGetErrorString(rc));
}

}  // namespace
