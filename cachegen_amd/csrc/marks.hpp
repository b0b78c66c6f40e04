// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Marks and words that kernels store to pinned memory for a host that looks at them: only
// where a kernel runs that can do it, since beside a busy GPU each launch waits its turn.
#pragma once

namespace {

// Sets *mark (pinned host memory) to `value`.  A stream runs its launches one behind the other, so the host that
// reads the value knows that all launches before this one are through.  What they stored to device memory the launches behind
// them see; what they stored to host memory the host sees only if the threads that stored it have released it to the
// system (host_stores_done): the release here is of this thread's XCD, and theirs may be another.
__device__ __forceinline__ void set_mark(int32_t *mark, int32_t value)
{
    __hip_atomic_store(mark, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void mark_kernel(int32_t *mark, int32_t value) { set_mark(mark, value); }

// Ends a kernel's stores to host memory that a mark will stand for, in the threads that made them.
__device__ __forceinline__ void host_stores_done() { __threadfence_system(); }

// Up to four words of device memory, as 64-bit numbers, to pinned memory, and a mark behind them: 8 us until the host has
// them, where a copy of one word and its wait are 14.
struct WordsArgs {
    const void *at[4];
    int32_t bytes[4];           // 4 (signed) or 8
    int32_t n;
    int64_t *out;
    int32_t *mark;
    int32_t value;
};

__global__ void read_words_kernel(WordsArgs a)
{
    for (int i = 0; i < a.n; ++i) a.out[i] = a.bytes[i] == 8 ? *static_cast<const int64_t *>(a.at[i]) : *static_cast<const int32_t *>(a.at[i]);
    set_mark(a.mark, a.value);
}

// The largest of two vectors' values (NaN where there is one), which sizes the tables of an encode: one launch where a
// maximum, its reduction and a copy of the result took the host 27 us.  One wavefront; a vector has a value a layer.
__global__ __launch_bounds__(64) void largest_kernel(const float *a, const float *b, int64_t n, float *out, int32_t *mark, int32_t value)
{
    float m = -INFINITY;
    bool nan = false;
    for (int64_t i = threadIdx.x; i < n; i += 64) {
        const float x = a[i], y = b[i];
        nan |= __builtin_isnan(x) || __builtin_isnan(y);
        m = fmaxf(m, fmaxf(x, y));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (__ballot(nan) != 0) m = __builtin_nanf("");
    if (threadIdx.x == 0) {
        *out = m;
        set_mark(mark, value);
    }
}

// hipEventQuery, also while another thread captures a graph: asked in that thread's way it counts among the calls that a
// capture in the global mode refuses and is broken by.
hipError_t query_event(hipEvent_t e)
{
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool changed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    const hipError_t rc = hipEventQuery(e);
    if (changed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    return rc;
}

// The word is read for so long, then the stream is waited for, which also finds out about a launch that failed.
constexpr std::chrono::milliseconds kMarkPatience{200};

// Until *mark >= value.
int wait_for_mark(const int32_t *mark, int32_t value, hipStream_t stream)
{
    const auto start = std::chrono::steady_clock::now();
    for (;;) {
        for (int i = 0; i < 64; ++i) {
            if (__atomic_load_n(mark, __ATOMIC_ACQUIRE) >= value) return CG_OK;
            __builtin_ia32_pause();
        }
        if (std::chrono::steady_clock::now() - start > kMarkPatience) break;
    }
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return fail(CG_ERR_LAUNCH, "wait_mark: %s", hipGetErrorString(e));
    if (__atomic_load_n(mark, __ATOMIC_ACQUIRE) >= value) return CG_OK;
    return fail(CG_ERR_ARG, "wait_mark: nothing on this stream sets the mark");
}

}  // namespace
