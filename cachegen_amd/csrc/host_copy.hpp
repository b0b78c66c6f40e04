// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip.  Copies between ordinary
// and pinned host memory by several threads, in step with what crosses the bus; plain C++, without HIP.
#pragma once

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdint>
#include <cstring>
#include <functional>
#include <vector>
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#include <emmintrin.h>
#endif

#include "cachegen_hip.h"

namespace {

// A container is copied once on the host each way, out of the pinned memory that its sections reach or into the one they
// leave from.  Done with one library call a section, each a fork and join of its own, a chunk's five copies took 190 us
// of which the bytes are 60, and the bus waited meanwhile.  Here a call's copies are one job, cut into blocks; the blocks of
// what has arrived are copied while the rest is on the bus, and what is staged leaves while the rest is staged.
//
// The threads are the caller's team: the OpenMP runtime that torch's own copies run on.  Threads of this library's
// own, beside sixteen of that runtime that still look for work after a torch operation, are more than the cores that a
// process has here, and a job then waits for a thread that waits for a core (53 MB: 3 to 10 ms instead of 1.2).
// A block has an owner among the threads, by its address in ordinary memory: a blob that is read back soon lies in the
// caches of the threads that wrote it.  Owners are dealt before the team is there, and the runtime may give a smaller one
// (a thread limit, dynamic teams, a caller inside a parallel region) or none.  So every thread goes through the job step
// by step, its own blocks of a step first and then what nobody has begun of it: who waits for a pinned slot has seen
// every block of the steps before taken, those are copied without waiting for this one, and the move that frees the slot
// is launched.  A job ends with any team, on its caller alone too.
//
// Staged and moved to the GPU, one thread / eight: 1 MB 57 / 52 us, 2.7 MB 96 / 86, 6 MB 168 / 152, 14 MB 343 / 326, 53 MB 1532 / 1152;
// copied out of pinned memory just written: 1.4 MB 40 / 20, 6 MB 157 / 61, 14 MB 364 / 130.  Sixteen are no faster (a chunk to
// bytes and back 476 us, 458 with eight), but the team is of all of torch's threads, of which the others return at once: the
// runtime ends the threads that a smaller one leaves out and has to start them again for torch's next operation.
constexpr int64_t kHostBlock = 64 << 10;
constexpr int kHostThreads = 8;

struct HostBlock {
    uint8_t *dst;
    const uint8_t *src;
    int32_t bytes;
    int32_t owner;
    int32_t value;                          // to be copied when the job's mark is this far
    int32_t step;                           // counts towards this step's completion
};

struct HostJob {
    std::vector<HostBlock> blocks;          // by steps
    std::vector<size_t> ends;               // behind each step's blocks
    std::vector<std::atomic<uint8_t>> taken;
    std::vector<std::atomic<int32_t>> left; // blocks to come, per step
    std::atomic<int32_t> done{0};           // blocks that are through
    std::atomic<bool> stop{false};
    const int32_t *mark = nullptr;          // how far what the blocks wait for has got
    int nthreads = 1;
    bool large = false;                     // kPastCaches or more

    bool reached(int32_t value) const { return __atomic_load_n(mark, __ATOMIC_ACQUIRE) >= value; }
};

inline void host_pause()
{
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
    __builtin_ia32_pause();
#endif
}

// memcpy with stores past the caches, whole 64-byte lines of them: what is staged is read by the bus next, a large blob by
// whoever asks for it later.  memcpy copies blocks of this size by the processor's string instruction, through the caches,
// and that is slow out of blobs that a store has just left in them, the slower the more threads' caches they are in:
// 53 MB staged right after they were stored, 4 / 8 / 16 threads, 985 / 1120 / 1757 us, by this 762 / 590 / 585.  Small jobs
// are faster through the caches (kPastCaches): copied out of pinned memory, memcpy / this, 1.4 MB 24 / 34 us, 2.7 MB 28 / 54,
// 6 MB 54 / 79, 14 MB 156 / 158; staged and moved, 2.7 MB 95 / 99, 6 MB 162 / 170, 14 MB 350 / 337.  Whole calls: store and
// retrieve of 59 MB in blobs of 6 MB 3735 / 3315, merge of 44 MB 814 / 766, a 14 MB pickle to bytes and back 1731 / 1587.
constexpr int64_t kPastCaches = 8 << 20;

inline void copy_past_caches(uint8_t *dst, const uint8_t *src, size_t n)
{
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
    const size_t head = std::min<size_t>(n, (64 - ((uintptr_t)dst & 63)) & 63);
    memcpy(dst, src, head);
    dst += head;
    src += head;
    n -= head;
    for (; n >= 64; n -= 64, dst += 64, src += 64) {
        __m128i v[4];
        for (int i = 0; i < 4; ++i) v[i] = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src) + i);
        for (int i = 0; i < 4; ++i) _mm_stream_si128(reinterpret_cast<__m128i *>(dst) + i, v[i]);
    }
    memcpy(dst, src, n);
    _mm_sfence();                           // the block counts as copied only behind its stores
#else
    memcpy(dst, src, n);
#endif
}

inline void copy_block(uint8_t *dst, const uint8_t *src, size_t n) { memcpy(dst, src, n); }

// Block i, if it is still to be had.  `idle` runs while the mark is waited for.
inline void take_block(HostJob &job, size_t i, const std::function<void()> *idle)
{
    if (job.taken[i].load(std::memory_order_relaxed) || job.taken[i].exchange(1, std::memory_order_acq_rel)) return;
    const HostBlock &b = job.blocks[i];
    while (!job.reached(b.value) && !job.stop.load(std::memory_order_relaxed)) {
        if (idle) (*idle)();
        host_pause();
    }
    if (!job.stop.load(std::memory_order_relaxed)) (job.large ? copy_past_caches : copy_block)(b.dst, b.src, (size_t)b.bytes);
    job.left[(size_t)b.step].fetch_sub(1, std::memory_order_acq_rel);
    job.done.fetch_add(1, std::memory_order_acq_rel);
}

inline void work_on(HostJob &job, int me, const std::function<void()> *idle)
{
    size_t first = 0;
    for (const size_t end : job.ends) {
        for (int mine = 1; mine >= 0; --mine)
            for (size_t i = first; i < end; ++i) {
                if (mine && job.blocks[i].owner != me) continue;
                take_block(job, i, idle);
                if (idle) (*idle)();
            }
        first = end;
    }
}

// The job on the team's threads; `idle` (may be null) is run by the caller now and then.
struct HostRun {
    HostJob *job;
    const std::function<void()> *idle;
    int (*thread_num)();
};

inline void host_member(void *run)
{
    const HostRun &r = *static_cast<HostRun *>(run);
    const int me = r.thread_num();
    if (me >= r.job->nthreads) return;
    const std::function<void()> *const idle = me == 0 ? r.idle : nullptr;       // the caller is thread 0
    work_on(*r.job, me, idle);
    // another thread's block may wait for what only the caller's idle() brings about: it stays until all are through
    while (idle && r.job->done.load(std::memory_order_acquire) < (int32_t)r.job->blocks.size()) {
        (*idle)();
        host_pause();
    }
}

inline int host_threads(const CgHostTeam *team)
{
    if (!team || !team->parallel || !team->thread_num || team->threads < 1) return 1;
    return std::min(team->threads, kHostThreads);
}

inline void run_job(HostJob &job, const CgHostTeam *team, const std::function<void()> *idle)
{
    if (job.nthreads > 1 && job.blocks.size() > 2) {
        HostRun r = {&job, idle, team->thread_num};
        team->parallel(&host_member, &r, (unsigned)team->threads, 0u);
    } else {
        work_on(job, 0, idle);
    }
}

// Blocks of one copy; `home`: the address by which they are dealt to the threads, which moves with the copy.
inline void add_blocks(HostJob &job, uint8_t *dst, const uint8_t *src, int64_t n, uintptr_t home, int32_t value, int32_t step)
{
    while (n > 0) {
        const int64_t m = std::min<int64_t>(n, kHostBlock - (int64_t)(home % kHostBlock));
        job.blocks.push_back({dst, src, (int32_t)m, (int32_t)(home / kHostBlock % (uintptr_t)job.nthreads), value, step});
        dst += m;
        src += m;
        home += (uintptr_t)m;
        n -= m;
    }
}

inline void seal(HostJob &job, int steps)
{
    job.taken = std::vector<std::atomic<uint8_t>>(job.blocks.size());
    job.left = std::vector<std::atomic<int32_t>>((size_t)steps);
    const auto earlier = [](const HostBlock &a, const HostBlock &b) { return a.step < b.step; };
    if (!std::is_sorted(job.blocks.begin(), job.blocks.end(), earlier)) std::stable_sort(job.blocks.begin(), job.blocks.end(), earlier);
    int64_t bytes = 0;
    for (const HostBlock &b : job.blocks) {
        job.left[(size_t)b.step].fetch_add(1, std::memory_order_relaxed);
        bytes += b.bytes;
    }
    job.large = bytes >= kPastCaches;
    size_t end = 0;
    for (const auto &n : job.left) job.ends.push_back(end += (size_t)n.load(std::memory_order_relaxed));
}

// Where the steps of an upload begin: the first is a quarter of one so that the bus has something to do soon.
struct HostSteps {
    int64_t step;
    int64_t start(int64_t k) const { return k == 0 ? 0 : k == 1 ? step / 4 : (k - 1) * step; }
    int64_t of(int64_t at) const { return at < step / 4 ? 0 : at < step ? 1 : at / step + 1; }
};

// cg_host_stage's steps, launched by launch(from, offset in the area, bytes); through() gives the number of them that are
// through, or an error (negative).
template <typename Launch, typename Through>
int stage_job(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, int64_t bytes, const CgHostTeam *team, int *moves,
              Launch launch, Through through)
{
    const HostSteps at_step = {step};
    const int64_t ring_bytes = nslots * step;
    auto pinned = [&](int64_t at) { return static_cast<uint8_t *>(slots[at / step % nslots]) + at % step; };
    const int32_t steps = (int32_t)at_step.of(bytes - 1) + 1;
    int32_t known = 0;                      // steps that are through, as the other threads read it
    HostJob job;
    job.mark = &known;
    job.nthreads = host_threads(team);
    for (int i = 0; i < n; ++i) {
        const CgHostPart &p = parts[i];
        for (int64_t at = p.dst, end = p.dst + p.bytes; at < end;) {
            const int64_t k = at_step.of(at), stop = std::min(end, at_step.start(k + 1));
            // a slot is free once the step that it held is through
            const int32_t need = at < ring_bytes ? 0 : (int32_t)at_step.of(stop - 1 - ring_bytes) + 1;
            add_blocks(job, pinned(at), reinterpret_cast<const uint8_t *>(p.src) + (at - p.dst), stop - at,
                       (uintptr_t)p.src + (uintptr_t)(at - p.dst), need, (int32_t)k);
            at = stop;
        }
    }
    seal(job, steps);
    const bool in_turn = bytes > ring_bytes;
    int rc = 0;
    int32_t launched = 0;
    const std::function<void()> idle = [&] {
        while (!rc && launched < steps && job.left[(size_t)launched].load(std::memory_order_acquire) <= 0) {
            const int64_t at = at_step.start(launched), end = std::min(bytes, at_step.start(launched + 1));
            rc = launch(pinned(at), at, end - at);
            if (!rc) ++launched;
        }
        if (!rc && in_turn && launched < steps && known < launched) {
            const int32_t now = through();
            if (now < 0) rc = now;
            else if (now > known) __atomic_store_n(&known, now, __ATOMIC_RELEASE);
        }
        if (rc) job.stop.store(true);
    };
    run_job(job, team, &idle);
    while (!rc && launched < steps) idle();
    *moves = launched;
    return rc;
}

// Whether cg_host_stage's arguments describe something that it can do; null, or what is wrong.
inline const char *stage_fault(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, const void *area, int64_t bytes,
                               const int *moves)
{
    if (!parts || n < 0 || !slots || !area || !moves || bytes <= 0) return "null pointer or nothing to move";
    if (step < 64 || step % 64) return "steps are multiples of 64 bytes";
    if (nslots < 2 && nslots * step < bytes) return "pinned memory too small";
    for (int64_t i = 0; i < nslots && i * step < bytes; ++i)
        if (!slots[i]) return "null slot";
    for (int i = 0; i < n; ++i)
        if (parts[i].bytes < 0 || (parts[i].bytes && !parts[i].src) || parts[i].dst < 0 || parts[i].dst + parts[i].bytes > bytes) return "bad part";
    return nullptr;
}

}  // namespace
