// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Bytes between pinned host memory and device memory, and marks that
// tell the host how far a stream has got.
#pragma once

namespace {

// The container's sections cross the bus by a kernel and not by hipMemcpyAsync.  What bounds either is the bus
// (57 GB/s), but a copy is set apart from what the stream does before and after it: one behind another costs
// 7 to 10 us besides its bytes, where one kernel starts right behind another, and a host that waits for a kernel's
// event wakes 13 us after its end, where it sees a word that a kernel stores to pinned memory as soon as
// it is there.  One after the other, copies / this kernel: 64 KB 10.4 / 7.8 us, 1 MB 27.5 / 21, 4 MB 83 / 77, 6 MB 119 /
// 114, 14 MB 265 / 260 up; six pieces of 1 MB down with an event behind each 206 / 153.
// 64 blocks, one 16-byte load in flight a thread: 256 KB under way, twice what the bus needs for its round trip of
// about 2 us.  Upwards more blocks are slower (4 MB: 77 us with 64 blocks, 80 with 256, 102 with 1024: reads
// that arrive out of order), downwards they make no difference.
constexpr int kMoveThreads = 256, kMoveBlocks = 64;
constexpr int64_t kMovePart = 1 << 30;      // bytes a launch: offsets from a buffer descriptor's base are 32 bits

// Cache policy of an access at system scope (sc0 sc1): a load of host memory does not take a line that an earlier kernel
// left in the GPU's caches, a store to it goes through to it.
constexpr int kSystemScope = 1 | 16;

__global__ void mark_kernel(int32_t *mark, int32_t value) { set_mark(mark, value); }

// n bytes, n <= kMovePart.  mark (may be null): set first, for what was queued before.
template <bool TO_HOST>
__global__ __launch_bounds__(kMoveThreads) void move_bytes_kernel(const uint8_t *src, uint8_t *dst, uint32_t n, int32_t *mark, int32_t value)
{
    if (mark && blockIdx.x == 0 && threadIdx.x == 0) set_mark(mark, value);
    constexpr int kLoad = TO_HOST ? 0 : kSystemScope, kStore = TO_HOST ? kSystemScope : 0;
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, (int)n, kBufferWord3);
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc((void *)dst, 0, (int)n, kBufferWord3);
    const uint32_t step = gridDim.x * kMoveThreads, tid = blockIdx.x * kMoveThreads + threadIdx.x;
    // bytes up to the first 16-byte boundary of both, whole 16-byte units, bytes behind them; memory whose
    // addresses differ inside such a unit goes byte by byte
    const uint32_t skew = (uint32_t)(uintptr_t)dst & 15u;
    uint32_t head = (16u - skew) & 15u;
    if ((((uintptr_t)src ^ (uintptr_t)dst) & 15u) != 0 || head > n) head = n;
    const uint32_t units = (n - head) >> 4;
    for (uint32_t i = tid; i < units; i += step) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(from, (int)(head + 16u * i), 0, kLoad);
        __builtin_amdgcn_raw_buffer_store_b128(v, to, (int)(head + 16u * i), 0, kStore);
    }
    const uint32_t tail = head + 16u * units;
    for (uint32_t i = tid; i < head + (n - tail); i += step) {
        const int at = (int)(i < head ? i : tail + (i - head));
        __builtin_amdgcn_raw_buffer_store_b8(__builtin_amdgcn_raw_buffer_load_b8(from, at, 0, kLoad), to, at, 0, kStore);
    }
    if (TO_HOST) host_stores_done();                     // there before the launch behind this one sets its mark
}

int launch_move_bytes(const uint8_t *src, uint8_t *dst, int64_t n, bool to_host, int32_t *mark, int32_t value, hipStream_t stream)
{
    for (int64_t at = 0; at < n; at += kMovePart) {
        const uint32_t part = (uint32_t)(n - at < kMovePart ? n - at : kMovePart);
        const int64_t blocks = ceil_div(part, 16 * kMoveThreads);
        const dim3 grid((unsigned)(blocks < kMoveBlocks ? blocks : kMoveBlocks));
        if (to_host) move_bytes_kernel<true><<<grid, dim3(kMoveThreads), 0, stream>>>(src + at, dst + at, part, at ? nullptr : mark, value);
        else move_bytes_kernel<false><<<grid, dim3(kMoveThreads), 0, stream>>>(src + at, dst + at, part, at ? nullptr : mark, value);
    }
    return check_launch("move_bytes");
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

// The same for a caller that does something else meanwhile.
class MarkWatch {
public:
    MarkWatch(const int32_t *mark, hipStream_t stream) : mark_(mark), stream_(stream), last_(__atomic_load_n(mark, __ATOMIC_RELAXED)) {}

    // Whether the mark is short of `value` and has not moved for that long.
    bool overdue(int32_t value)
    {
        const int32_t now = __atomic_load_n(mark_, __ATOMIC_ACQUIRE);
        if (++looks_ % 64 && now == last_) return false;
        const auto t = std::chrono::steady_clock::now();
        if (now != last_) since_ = t;
        last_ = now;
        return now < value && t - since_ > kMarkPatience;
    }

    int settle()
    {
        since_ = std::chrono::steady_clock::now();
        const hipError_t e = hipStreamSynchronize(stream_);
        return e == hipSuccess ? CG_OK : fail(CG_ERR_LAUNCH, "moves: %s", hipGetErrorString(e));
    }

private:
    const int32_t *mark_;
    hipStream_t stream_;
    int32_t last_;
    uint32_t looks_ = 0;
    std::chrono::steady_clock::time_point since_ = std::chrono::steady_clock::now();
};

}  // namespace
