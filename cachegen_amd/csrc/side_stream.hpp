// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  A second stream for the launches of one call that need not wait for one another.
#pragma once

namespace {

// Forks from the caller's stream when made and joins it when it goes out of scope, also after a failed launch: whatever was
// queued on it is behind the caller's work before the call and before the caller's work after it, so the caller's memory
// is used as on its own stream.  One stream and two events per device, kept, and lent to one call at a time: a call that
// finds them lent (ok() false), or with work of another stream still on them (it would wait for that: two calls on two
// streams, the first behind 40 ms of other work, ended after 42 ms both), or whose stream is being captured (a lent
// stream would belong to that capture until its end), queues everything on its own stream.
class SideStream {
public:
    explicit SideStream(hipStream_t caller) : caller_(caller)
    {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(caller, &capture) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        int dev = -1;
        if (capture != hipStreamCaptureStatusNone || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return;
        Kept &k = kept_[dev];
        if (k.lent.exchange(true, std::memory_order_acquire)) return;
        if (!(k.stream || make(k)) || !free_for(k, caller)) {
            (void)hipGetLastError();
            k.lent.store(false, std::memory_order_release);
            return;
        }
        if (hipEventRecord(k.fork, caller_) != hipSuccess || hipStreamWaitEvent(k.stream, k.fork, 0) != hipSuccess) {
            (void)hipGetLastError();
            k.lent.store(false, std::memory_order_release);
            return;
        }
        k.user = caller;
        kept = &k;
    }

    ~SideStream()
    {
        if (!kept) return;
        if (hipEventRecord(kept->join, kept->stream) != hipSuccess || hipStreamWaitEvent(caller_, kept->join, 0) != hipSuccess)
            (void)hipStreamSynchronize(kept->stream);
        kept->lent.store(false, std::memory_order_release);
    }

    SideStream(const SideStream &) = delete;
    SideStream &operator=(const SideStream &) = delete;

    bool ok() const { return kept != nullptr; }
    hipStream_t stream() const { return kept->stream; }

private:
    struct Kept {
        std::atomic<bool> lent{false};
        hipStream_t stream = nullptr;
        hipEvent_t fork = nullptr, join = nullptr;
        hipStream_t user = nullptr;         // the last caller's, whose work the stream and `join` stand for
    };

    // Whether nothing is on the kept stream but what is before this call on the caller's anyway.  hipStreamPerThread is one
    // handle for the streams of all threads.
    static bool free_for(Kept &k, hipStream_t caller)
    {
        if (k.user == caller && caller != hipStreamPerThread) return true;
        return query_event(k.join) == hipSuccess;                       // never recorded: through
    }

    static bool make(Kept &k)
    {
        if (!k.fork && hipEventCreateWithFlags(&k.fork, hipEventDisableTiming) != hipSuccess) return false;
        if (!k.join && hipEventCreateWithFlags(&k.join, hipEventDisableTiming) != hipSuccess) return false;
        return hipStreamCreateWithFlags(&k.stream, hipStreamNonBlocking) == hipSuccess;
    }

    static constexpr int kDevices = 64;
    static Kept kept_[kDevices];
    hipStream_t caller_;
    Kept *kept = nullptr;
};

SideStream::Kept SideStream::kept_[SideStream::kDevices];

}  // namespace
