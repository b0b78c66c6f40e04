// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Tables <-> histogram counts, for containers that store the
// counts instead of the tables.
//
// A table is a function of its histogram (cal_cdf.cu:29-49 in LMCache/third_party/torchac_cuda):
//   cdf[i] = (0xFFFF - max_bins) * cum[i] / n + i,   cum = running sum of the counts, n = tokens
// and for n <= 256 the running sums are recovered from the table exactly, because the scale
// exceeds n: cum[i] = ceil((cdf[i] - i) * n / scale).  A "group" is one (chunk, row): C channels
// that share a token count and, in the ragged form, a number of stored symbols.
#pragma once

namespace {

constexpr int kWireThreads = 256;

__global__ void clear_ints_kernel(int32_t *a, int64_t na, int32_t *b)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na) a[i] = 0;
    if (i == 0 && b) *b = 0;
}

// What the host has to know of an encoded tensor before it can lay blobs out, stored straight into
// host memory (pinned: the host reads it once a mark behind this launch is there, without a
// copy of its own): out = [status, wide, inexact, payload offset at each of nbounds sub-chunk
// boundaries, nsym[0 .. ngroups)].  One block; a few hundred values.
__global__ __launch_bounds__(kWireThreads) void wire_meta_kernel(
    const int32_t *__restrict__ status, const int64_t *__restrict__ offsets, int64_t per_sub, int64_t nbounds,
    const int32_t *__restrict__ wide, const int32_t *__restrict__ inexact, const int32_t *__restrict__ nsym, int64_t ngroups, int64_t *out)
{
    if (threadIdx.x == 0) {
        out[0] = *status;
        out[1] = wide ? *wide : 0;
        out[2] = inexact ? *inexact : 0;
    }
    for (int64_t i = threadIdx.x; i < nbounds; i += kWireThreads) out[3 + i] = offsets[i * per_sub];
    for (int64_t i = threadIdx.x; i < ngroups; i += kWireThreads) out[3 + nbounds + i] = nsym[i];
    host_stores_done();
}

// Stream lengths as 16-bit words; *wide (zero before the launch) is set where one does not fit.
__global__ __launch_bounds__(kWireThreads) void lengths_to_u16_kernel(
    const int32_t *__restrict__ lengths, int64_t n, uint16_t *__restrict__ out, int32_t *wide)
{
    const int64_t i = (int64_t)blockIdx.x * kWireThreads + threadIdx.x;
    if (i >= n) return;
    const int32_t v = lengths[i];
    out[i] = (uint16_t)v;
    if (v < 0 || v > 0xFFFF) atomicOr(wide, 1);
}

// The three kernels below have a wave per block and a channel per lane.  A channel's counts and its
// table are contiguous, so the lanes' walks over them are strided, but the 64 channels of a block
// are contiguous as a whole: they pass through LDS, which the wave fills and empties in order.  What
// is left is latency (64 groups of 1024 channels, lp = 33, data not in cache: tables to counts 18.6 ->
// 12.7 us, counts to tables 18.7 -> 6.7).
// kMaxTable bounds the LDS: 16.5 KB for the tables of a block, 8 KB for its counts.
constexpr int kTableChannels = 64;
constexpr int kMaxTable = CG_MAX_LP;

__device__ __forceinline__ void wave_copy(void *dst, const void *src, int bytes)
{
    const int lane = threadIdx.x;
    int done = 0;
    if (((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0) {
        const int words = bytes >> 4;
#pragma unroll 5
        for (int i = lane; i < words; i += kTableChannels) static_cast<uint4 *>(dst)[i] = static_cast<const uint4 *>(src)[i];
        done = words << 4;
    }
#pragma unroll 8
    for (int i = done + lane; i < bytes; i += kTableChannels) static_cast<uint8_t *>(dst)[i] = static_cast<const uint8_t *>(src)[i];
}

__device__ __forceinline__ int block_channels(int64_t first, int64_t C)
{
    return (int)(C - first < kTableChannels ? C - first : kTableChannels);
}

// x / d for a d that the wave shares: 2^32 / d, rounded up, exceeds 2^32 / d by e / d with e <= d, so
// the product with x is less than one too large.
struct SharedDivisor {
    uint32_t d, inverse;
    __device__ explicit SharedDivisor(uint32_t divisor) : d(divisor), inverse(0xFFFFFFFFu / divisor + 1u) {}
    __device__ uint32_t operator()(uint32_t x) const
    {
        const uint32_t q = d == 1u ? x : __umulhi(x, inverse);
        return q * d > x ? q - 1u : q;
    }
};

// counts: uint8 [ngroups, C, lp - 1], clamped to 255; nsym[g]: one more than the largest symbol that
// occurs in group g (at least 1); inexact: set to 1 if some table is not what the formula gives for
// any histogram.
__global__ __launch_bounds__(kTableChannels) void tables_to_counts_kernel(
    const uint16_t *__restrict__ cdf, int lp, int64_t C, const int32_t *__restrict__ tokens,
    uint8_t *__restrict__ counts, int32_t *nsym, int32_t *inexact)
{
    __shared__ alignas(16) uint16_t table[kTableChannels * kMaxTable];
    __shared__ alignas(16) uint8_t count[kTableChannels * (kMaxTable - 1)];
    const int64_t g = blockIdx.y, first = (int64_t)blockIdx.x * kTableChannels;
    const int channels = block_channels(first, C), lane = threadIdx.x;
    wave_copy(table, cdf + (g * C + first) * lp, channels * lp * 2);
    __syncthreads();
    int last = 1;
    if (lane < channels) {
        const uint32_t n = (uint32_t)tokens[g];
        const uint32_t scale = 0xFFFFu - (uint32_t)(lp - 1);
        const SharedDivisor by_scale(scale), by_n(n);
        const uint16_t *t = table + lane * lp;
        uint8_t *out = count + lane * (lp - 1);
        bool exact = t[0] == 0;
        uint32_t prev = 0;
#pragma unroll 4
        for (int i = 1; i < lp; ++i) {
            const uint32_t c = t[i];
            const uint32_t q = c - (uint32_t)i;                    // wraps if c < i: caught below
            const bool fits = c >= (uint32_t)i;
            const uint32_t cum = fits ? by_scale(q * n + scale - 1u) : 0u;      // q < 2^16, n <= 256
            exact &= fits & (cum >= prev) & (cum <= n) & (by_n(scale * (cum <= n ? cum : n)) + (uint32_t)i == c);      // no branches
            const uint32_t c1 = cum >= prev ? cum - prev : 0u;
            out[i - 1] = (uint8_t)(c1 > 255u ? 255u : c1);
            last = c1 ? i : last;
            prev = cum;
        }
        if (!exact || prev != n) *inexact = 1;                                  // everybody who writes writes the same
    }
    __syncthreads();
    wave_copy(counts + (g * C + first) * (lp - 1), count, channels * (lp - 1));
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const int other = __shfl_xor(last, o, 64);
        last = other > last ? other : last;
    }
    if (lane == 0) atomicMax(nsym + g, last);
}

// Ragged form: group g's channels in turn, nsym[g] counts each, from byte starts[g] on.  starts ==
// null: the groups follow one another, and every block adds up the symbol counts before its group's
// (the host does not have to see them first).
__global__ __launch_bounds__(kTableChannels) void pack_counts_kernel(
    const uint8_t *__restrict__ counts, int lp, int64_t C, const int32_t *__restrict__ nsym,
    const int64_t *__restrict__ starts, uint8_t *__restrict__ out)
{
    __shared__ alignas(16) uint8_t count[kTableChannels * (kMaxTable - 1)];
    __shared__ alignas(16) uint8_t packed[kTableChannels * (kMaxTable - 1)];
    const int64_t g = blockIdx.y, first = (int64_t)blockIdx.x * kTableChannels;
    const int channels = block_channels(first, C), lane = threadIdx.x;
    wave_copy(count, counts + (g * C + first) * (lp - 1), channels * (lp - 1));
    int32_t before = 0;                                             // at most 65535 groups of 128 symbols
    if (!starts) {
        for (int64_t i = lane; i < g; i += kTableChannels) before += nsym[i];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o, 64);
    }
    __syncthreads();
    const int k = nsym[g] < lp - 1 ? nsym[g] : lp - 1;
    if (lane < channels)
#pragma unroll 8
        for (int j = 0; j < k; ++j) packed[lane * k + j] = count[lane * (lp - 1) + j];
    __syncthreads();
    wave_copy(out + (starts ? starts[g] : (int64_t)before * C) + first * k, packed, channels * k);
}

// The inverse: ragged counts -> tables.  A count of 256 (one symbol for all n = 256 tokens)
// was stored as 255: the one token missing from the sum goes back to that entry.  invalid is
// set if a channel's counts cannot be completed to its group's token count that way.
__global__ __launch_bounds__(kTableChannels) void counts_to_tables_kernel(
    const uint8_t *__restrict__ data, int64_t data_bytes, int lp, int64_t C,
    const int32_t *__restrict__ tokens, const uint8_t *__restrict__ nsym,
    const int64_t *__restrict__ starts, uint16_t *__restrict__ cdf, int32_t *invalid)
{
    __shared__ alignas(16) uint8_t count[kTableChannels * (kMaxTable - 1)];
    __shared__ alignas(16) uint16_t table[kTableChannels * kMaxTable];
    const int64_t g = blockIdx.y, first = (int64_t)blockIdx.x * kTableChannels;
    const int channels = block_channels(first, C), lane = threadIdx.x;
    const int k = nsym[g];
    const int64_t at = starts[g] + first * k;
    const bool inside = k >= 1 && k <= lp - 1 && at >= 0 && at + (int64_t)channels * k <= data_bytes;
    if (inside) wave_copy(count, data + at, channels * k);           // never read outside the section
    __syncthreads();
    if (lane < channels) {
        const uint32_t n = (uint32_t)tokens[g];
        const uint32_t scale = 0xFFFFu - (uint32_t)(lp - 1);
        const SharedDivisor by_n(n ? n : 1u);
        const uint8_t *src = count + lane * k;
        uint16_t *t = table + lane * lp;
        uint32_t sum = 0, full = 0;
#pragma unroll 8
        for (int j = 0; j < (inside ? k : 0); ++j) {
            sum += src[j];
            full += src[j] == 255u;
        }
        const uint32_t missing = n - sum;                           // wraps if the sum is too large
        if (!inside || !(missing == 0u || (missing == 1u && full == 1u))) {
            *invalid = 1;                                           // everybody who writes writes the same; may be host memory
            host_stores_done();
        }
        uint32_t cum = 0;
        t[0] = 0;
        const int stored = inside ? k : 0;
        const uint32_t clipped = missing == 1u ? 255u : 256u;       // the count that stands for one more
#pragma unroll 8
        for (int i = 1; i <= stored; ++i) {
            const uint32_t c = src[i - 1];
            cum += c + (c == clipped ? 1u : 0u);
            t[i] = (uint16_t)(by_n(scale * cum) + (uint32_t)i);
        }
        const uint32_t last = by_n(scale * cum);
#pragma unroll 8
        for (int i = stored + 1; i < lp; ++i) t[i] = (uint16_t)(last + (uint32_t)i);
    }
    __syncthreads();
    wave_copy(cdf + (g * C + first) * lp, table, channels * lp * 2);
}

}  // namespace
