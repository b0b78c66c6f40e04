// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Running sums of stream lengths and compaction of the encoder scratch into the payload.
//
// Paths in the comments are relative to LMCache/ in the reference tree:
//   enc_new.cu = third_party/torchac_cuda/torchac_kernel_enc_new.cu
//   dec_new.cu = third_party/torchac_cuda/torchac_kernel_dec_new.cu
//   cal_cdf.cu = third_party/torchac_cuda/cal_cdf.cu
//   encoder.py = lmcache/storage_backend/serde/cachegen_encoder.py
//   decoder.py = lmcache/storage_backend/serde/cachegen_decoder.py
#pragma once

namespace {

// ------------------------------------------------------------------------------------
// Exclusive running sum of the stream lengths (replaces the cumsum of decoder.py:70 and
// the index arithmetic of encoder.py:214-221): per-block sums, a one-block scan of
// those, then a per-block scan with the block's base added.
// ------------------------------------------------------------------------------------
constexpr int kScanThreads = 256;
constexpr int kScanPerThread = 8;
constexpr int kScanTile = kScanThreads * kScanPerThread;

// The block's exclusive running sum: wavefront shuffles and one exchange of the four wavefronts' totals
// through `lds` (at least 4 values).  A sum in LDS, halving the distance eight times with two barriers
// each, kept a launch of one block 1 us longer.
template <typename T>
__device__ __forceinline__ T block_exclusive_scan_256(T v, T *lds, T &total)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    T incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T up = __shfl_up(incl, o, 64);
        if (lane >= o) incl += up;
    }
    if (lane == 63) lds[wave] = incl;
    __syncthreads();
    T before = incl - v;
    total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const T t = lds[w];
        if (w < wave) before += t;
        total += t;
    }
    __syncthreads();
    return before;
}

__global__ __launch_bounds__(kScanThreads) void scan_tile_sums_kernel(
    const int32_t *__restrict__ lengths, int64_t n, int32_t clamp, int64_t *__restrict__ sums)
{
    __shared__ int64_t lds[kScanThreads];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
    int64_t s = 0;
    for (int j = 0; j < kScanPerThread; ++j)
        if (base + j < n) {
            int32_t v = lengths[base + j];
            v = v < 0 ? 0 : (v > clamp ? clamp : v);
            s += v;
        }
    int64_t total;
    block_exclusive_scan_256(s, lds, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// In place, one block: every thread owns a contiguous run of the sums, adds it up, the block
// scans the 256 run totals, and every thread rewrites its run as exclusive running sums.
// Runs are handled 16 values at a time from registers so that the loads are in flight together.
__global__ __launch_bounds__(kScanThreads) void scan_sums_kernel(int64_t *sums, int64_t ntiles)
{
    __shared__ int64_t lds[kScanThreads];
    constexpr int kBatch = 16;
    const int64_t per = (ntiles + kScanThreads - 1) / kScanThreads;
    const int64_t lo = (int64_t)threadIdx.x * per;
    const int64_t hi = lo + per < ntiles ? lo + per : ntiles;
    int64_t mine = 0;
    for (int64_t i0 = lo; i0 < hi; i0 += kBatch) {
        int64_t v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) v[j] = i0 + j < hi ? sums[i0 + j] : 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) mine += v[j];
    }
    int64_t total;
    int64_t run = block_exclusive_scan_256(mine, lds, total);
    for (int64_t i0 = lo; i0 < hi; i0 += kBatch) {
        int64_t v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) v[j] = i0 + j < hi ? sums[i0 + j] : 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (i0 + j < hi) sums[i0 + j] = run;
            run += v[j];
        }
    }
}

__global__ __launch_bounds__(kScanThreads) void scan_apply_kernel(
    const int32_t *__restrict__ lengths, int64_t n, int32_t clamp,
    const int64_t *__restrict__ sums, int64_t *__restrict__ offsets)
{
    __shared__ int64_t lds[kScanThreads];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
    int32_t v[kScanPerThread];
    int64_t s = 0;
    for (int j = 0; j < kScanPerThread; ++j) {
        int32_t x = base + j < n ? lengths[base + j] : 0;
        x = x < 0 ? 0 : (x > clamp ? clamp : x);
        v[j] = x;
        s += x;
    }
    int64_t total;
    // sums == nullptr: the input is a single tile and this kernel is the whole scan
    int64_t run = (sums ? sums[blockIdx.x] : 0) + block_exclusive_scan_256(s, lds, total);
    for (int j = 0; j < kScanPerThread; ++j) {
        if (base + j < n) offsets[base + j] = run;
        run += v[j];
        if (base + j == n - 1) offsets[n] = run;
    }
}

// The whole running sum in one launch of one block, for up to kScanSmallMax values (the byte
// counts of the encoder's tiles): every thread owns up to 16 consecutive values, the block scans
// the 1024 thread totals with wavefront shuffles, and every thread writes its run.
constexpr int kScanSmallThreads = 1024;
constexpr int kScanSmallPer = 16;
constexpr int kScanSmallMax = kScanSmallThreads * kScanSmallPer;

// COLLECT: and what the host has to know of padded streams of these lengths (collect_sizes_kernel), stored with a mark.
template <bool COLLECT>
__device__ __forceinline__ void scan_small(const int32_t *__restrict__ lengths, int32_t n, int32_t clamp, int64_t *__restrict__ offsets,
                                           int64_t nslots, int64_t cap, int64_t *out, int32_t *mark, int32_t value)
{
    __shared__ int64_t wave_totals[kScanSmallThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (n + kScanSmallThreads - 1) / kScanSmallThreads;      // <= kScanSmallPer
    const int lo = tid * per;
    int32_t v[kScanSmallPer];
    int64_t mine = 0;
#pragma unroll
    for (int j = 0; j < kScanSmallPer; ++j) {
        int32_t x = (j < per && lo + j < n) ? lengths[lo + j] : 0;
        x = x < 0 ? 0 : (x > clamp ? clamp : x);
        v[j] = x;
        mine += x;
    }
    // inclusive running sum over the wavefront, then over the 16 wavefront totals
    int64_t incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t up = __shfl_up(incl, o, 64);
        if (lane >= o) incl += up;
    }
    if (lane == 63) wave_totals[wave] = incl;
    __syncthreads();
    int64_t before = 0;
    for (int w = 0; w < wave; ++w) before += wave_totals[w];
    int64_t run = before + incl - mine;
#pragma unroll
    for (int j = 0; j < kScanSmallPer; ++j) {
        if (j < per && lo + j < n) {
            offsets[lo + j] = run;
            run += v[j];
            if (lo + j == n - 1) offsets[n] = run;
            if (COLLECT && lo + j == n - 1) {
                out[0] = run;
                host_stores_done();
            }
        }
    }
    if (!COLLECT) return;
    int unfit = 0;
#pragma unroll
    for (int j = 0; j < kScanSmallPer; ++j)
        if (j < per && lo + j < n) unfit |= v[j] > (lo + j < nslots ? cap : 0);
    unfit = __syncthreads_or(unfit);
    if (tid == 0) {
        out[1] = unfit ? 1 : 0;
        set_mark(mark, value);
    }
}

__global__ __launch_bounds__(kScanSmallThreads) void scan_small_kernel(
    const int32_t *__restrict__ lengths, int32_t n, int32_t clamp, int64_t *__restrict__ offsets)
{
    scan_small<false>(lengths, n, clamp, offsets, 0, 0, nullptr, nullptr, 0);
}

// The sums, the sizes' check and the mark of a collect_bytes in one launch where two and an event were 7 us and the host's
// 13 us to wake from it.
__global__ __launch_bounds__(kScanSmallThreads) void scan_collect_kernel(
    const int32_t *__restrict__ lengths, int32_t n, int64_t *__restrict__ offsets, int64_t nslots, int64_t cap, int64_t *out, int32_t *mark, int32_t value)
{
    scan_small<true>(lengths, n, INT_MAX, offsets, nslots, cap, out, mark, value);
}

// ------------------------------------------------------------------------------------
// collect_bytes (encoder.py:209-222).  A block owns 256 consecutive streams, i.e. one
// contiguous range of the payload, and assembles it in LDS, 16 KiB at a time: every thread
// copies its own stream from its slot to the stream's place in the range (two quads of words in
// flight, aligned words by a byte permute, single bytes at the two ends), then the block writes the
// tile out as aligned 32-bit words.  Only the first and last word of a block's range are written
// byte by byte, so neighbouring blocks never write the same byte.  All positions are
// 32-bit offsets from the range's start.
// ------------------------------------------------------------------------------------
constexpr int kCompactStreams = 256;
constexpr int kCompactTile = 16384;

// SCAN: the offsets are not known yet; `offsets` is written here from the streams' lengths and
// the exclusive running sum of the tiles' byte counts, instead of being read.  That sum comes
// from tile_base (a scan launch made it), or is added up here: from the sums of the groups of
// kTileGroup tiles before this block's group (at most kMaxTileGroups, left by the coder) and the
// counts of the tiles before this one in its group (group_sums != null), or from the counts of all
// tiles before this one (neither: calls of at most kDirectTiles tiles, where that is a few loads per
// thread and saves the scan launch, 5 us and its gap).
constexpr int kDirectTiles = 1024;
// Bound by the trips to memory of a wavefront's longest stream and by HBM: what the words of long streams
// cost among short ones.  Word by word (word w of stream t at w * 256 + t) each of them was a line of its own, read and written
// for four bytes; a quad of four words is loaded by one instruction, and its words share the line.  32
// layers x 8192 tokens x 1024 channels 63.9 -> 45.6 us (183 -> 137 MB read), and the coder 274.9 -> 271.5 (220 -> 151 MB written); the
// whole encode 626 -> 607, 80 layers x 32768 tokens 6100 -> 5850, four levels of 4096 tokens 1043 -> 1008, 4096 channels 2540 ->
// 2470 (each pair on one machine).  Sub-chunks of at most kShortStreams tokens lie word by word.
// SLICES > 1: the block has SLICES x 256 threads, and a stream's words are dealt to SLICES threads, eight in
// turn.
struct CompactArgs {
    const uint8_t *slots;
    int32_t cap;
    int64_t *offsets;
    const int32_t *lengths;
    const int64_t *tile_base;
    int64_t nstreams;
    uint8_t *payload;
    int64_t payload_cap;
    int32_t skew;
    int32_t *status;
    const int32_t *group_sums, *tile_sums;
    uint32_t place;         // kQuadPlace or kWordPlace
};

template <bool SCAN, int SLICES>
__device__ __forceinline__ void compact_streams(const CompactArgs &a, int32_t *rel, uint32_t *buf)
{
    const uint8_t *__restrict__ const slots = a.slots;
    const int32_t *__restrict__ const lengths = a.lengths, *__restrict__ const group_sums = a.group_sums, *__restrict__ const tile_sums = a.tile_sums;
    const int64_t *__restrict__ const tile_base = a.tile_base;
    int64_t *__restrict__ const offsets = a.offsets;
    uint8_t *__restrict__ const payload = a.payload;
    int32_t *const status = a.status;
    const int64_t nstreams = a.nstreams, payload_cap = a.payload_cap;
    const int32_t cap = a.cap, skew = a.skew;
    const int tid = threadIdx.x % 256, slice = SLICES > 1 ? threadIdx.x / 256 : 0;
    const bool lead_slice = slice == 0;                // the threads that stand for the streams
    const int64_t sbase = (int64_t)blockIdx.x * kCompactStreams;
    const int count = (nstreams - sbase < kCompactStreams) ? (int)(nstreams - sbase) : kCompactStreams;
    int64_t o0;
    if (SCAN) {
        int32_t mine = 0;
        if (lead_slice && tid < count) {
            mine = lengths[sbase + tid];
            mine = mine < 0 ? 0 : (mine > cap ? cap : mine);
        }
        int32_t total32;
        if (!group_sums && !tile_base) {
            int32_t part = 0;
#pragma unroll
            for (int i = 0; i < kDirectTiles / 256; ++i) {
                const int t = tid + i * 256;
                if (lead_slice && t < (int)blockIdx.x) part += tile_sums[t];
            }
            int32_t sum;
            block_exclusive_scan_256(part, reinterpret_cast<int32_t *>(buf), sum);
            o0 = sum;
        } else if (group_sums) {
            const int g = (int)(blockIdx.x / kTileGroup), r = (int)(blockIdx.x % kTileGroup);
            int32_t part = lead_slice && tid < g ? group_sums[tid] : 0;
            if (lead_slice && tid < r) part += tile_sums[(int64_t)g * kTileGroup + tid];
            int32_t sum;
            block_exclusive_scan_256(part, reinterpret_cast<int32_t *>(buf), sum);     // at most 16384 tiles of 64 KiB: fits
            o0 = sum;
        } else {
            o0 = tile_base[blockIdx.x];
        }
        const int32_t before = block_exclusive_scan_256(mine, reinterpret_cast<int32_t *>(buf), total32);    // buf is free until the copy
        const int64_t total64 = total32;                       // at most 256 streams of `cap` <= 256 bytes
        if (lead_slice) rel[tid] = before;
        if (lead_slice && tid == 0) rel[kCompactStreams] = total32;
        if (lead_slice && tid < count) offsets[sbase + tid] = o0 + before;
        if (sbase + count == nstreams && lead_slice && tid == 0) offsets[nstreams] = o0 + total64;
        __syncthreads();
        // threads past the last stream carry the total, like the padding of the other form
    } else {
        o0 = offsets[sbase];
        for (int i = threadIdx.x; i <= kCompactStreams; i += 256 * SLICES)
            rel[i] = (int32_t)(offsets[sbase + (i < count ? i : count)] - o0);
        __syncthreads();
    }
    const int total = rel[count];
    if (o0 + total > payload_cap) {                    // never write past the caller's buffer
        if (threadIdx.x == 0 && status) atomicOr(status, 2);
        return;
    }
    // x = position in the range + lead: aligned words of the payload are at multiples of 4
    const int lead = (int)((o0 + skew) & 3);
    uint8_t *const dst = payload + o0 - lead;
    const int end = lead + total;
    const int my0 = rel[tid] + lead, my1 = rel[tid + 1] + lead;     // rel[] is padded with the total
    // this thread's stream, quad by quad or word by word (kQuadRow in encoder.hpp)
    const bool quads = a.place == kQuadPlace;
    const uint8_t *const mine_at = slots + sbase * (int64_t)cap + tid * (quads ? 16 : 4);
    const int nquads = (my1 - my0 + 15) >> 4, nwords = (my1 - my0 + 3) >> 2;
    uint8_t *const bytes = reinterpret_cast<uint8_t *>(buf);
    // Aligned word first + i of the range holds the end of the stream's word i - 1 and the beginning of word i:
    // four of their eight bytes, the same four for every i.
    const int first = my0 >> 2;
    const uint32_t pick_bytes = 0x07060504u - (uint32_t)(my0 & 3) * 0x01010101u;

    for (int t0 = 0; t0 < end; t0 += kCompactTile) {
        const int t1 = t0 + kCompactTile < end ? t0 + kCompactTile : end;
        const int xs = my0 > t0 ? my0 : t0;
        const int xe = my1 < t1 ? my1 : t1;
        if (xs < xe) {
            const int whole0 = (xs + 3) >> 2, whole1 = xe >> 2;         // the range's words that are all this stream's
            uint32_t head = 0, tail = 0, prev = 0;
            bool ends_here = false;                                     // this thread has the word that the stream ends inside
            const int i_first = ((xs >> 2) - first) & ~7;
            for (int i0 = i_first + 8 * slice; 4 * (first + i0) < xe; i0 += 8 * SLICES) {
                uint32_t w[8];
                const bool want_prev = i0 > 0 && (SLICES > 1 || i0 == i_first);
                if (quads) {
                    const int g = i0 >> 2;
                    uint4 q0 = make_uint4(0, 0, 0, 0), q1 = q0;
                    if (g < nquads) q0 = *reinterpret_cast<const uint4 *>(mine_at + g * kQuadRow);
                    if (g + 1 < nquads) q1 = *reinterpret_cast<const uint4 *>(mine_at + (g + 1) * kQuadRow);
                    if (want_prev) prev = *reinterpret_cast<const uint32_t *>(mine_at + (g - 1) * kQuadRow + 12);
                    w[0] = q0.x, w[1] = q0.y, w[2] = q0.z, w[3] = q0.w;
                    w[4] = q1.x, w[5] = q1.y, w[6] = q1.z, w[7] = q1.w;
                } else {
#pragma unroll
                    for (int u = 0; u < 8; ++u) w[u] = i0 + u < nwords ? *reinterpret_cast<const uint32_t *>(mine_at + (i0 + u) * kWordRow) : 0u;
                    if (want_prev) prev = *reinterpret_cast<const uint32_t *>(mine_at + (i0 - 1) * kWordRow);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (u == 4 && 4 * (first + i0 + u) >= xe) break;    // short streams (chunks of 8 tokens, 32 layers x 4096 x 1024 channels): 239 -> 231 us
                    const uint32_t v = __builtin_amdgcn_perm(w[u], u ? w[u - 1] : prev, pick_bytes);
                    const int j = first + i0 + u;
                    if (u == 0 && i0 == 0) head = v;
                    if (j == whole1) tail = v, ends_here = true;
                    if (j >= whole0 && j < whole1) buf[j - (t0 >> 2)] = v;
                }
                prev = w[7];
            }
            // the words that this stream shares with its neighbours, byte by byte
            if (slice == 0 && xs == my0 && first < whole0)
                for (int c = 0; c < 4; ++c)
                    if (4 * first + c >= xs && 4 * first + c < xe) bytes[4 * first + c - t0] = (uint8_t)(head >> (8 * c));
            if (ends_here && whole1 >= whole0)
                for (int c = 0; c < 3; ++c)
                    if (4 * whole1 + c < xe) bytes[4 * whole1 + c - t0] = (uint8_t)(tail >> (8 * c));
        }
        __syncthreads();
        for (int w = (t0 >> 2) + (int)threadIdx.x; 4 * w < t1; w += 256 * SLICES) {
            const int x0 = 4 * w;
            const uint32_t v = buf[w - (t0 >> 2)];
            if (x0 >= lead && x0 + 4 <= end) {
                *reinterpret_cast<uint32_t *>(dst + x0) = v;
            } else {
                for (int j = 0; j < 4; ++j)
                    if (x0 + j >= lead && x0 + j < end) dst[x0 + j] = (uint8_t)(v >> (8 * j));
            }
        }
        __syncthreads();
    }
}

template <bool SCAN>
__global__ __launch_bounds__(256) void compact_streams_kernel(CompactArgs a)
{
    __shared__ int32_t rel[kCompactStreams + 1];       // stream offsets relative to the block's first byte
    __shared__ __align__(16) uint32_t buf[kCompactTile / 4];
    compact_streams<SCAN, 1>(a, rel, buf);
}

// A launch of few blocks lasts as long as its longest stream: 160 bytes are five rounds of loads for one
// thread, each as long as a trip to memory.
template <bool SCAN>
__global__ __launch_bounds__(1024) void compact_few_kernel(CompactArgs a)
{
    __shared__ int32_t rel[kCompactStreams + 1];
    __shared__ __align__(16) uint32_t buf[kCompactTile / 4];
    compact_streams<SCAN, 4>(a, rel, buf);
}

// The streams of several quantization levels of one tensor: level v has the blocks of y index v.
struct CompactLevelsArgs {
    CompactArgs level[kMaxLevels];
};

template <bool SCAN, int SLICES>
__global__ __launch_bounds__(256 * SLICES) void compact_levels_kernel(CompactLevelsArgs p)
{
    __shared__ int32_t rel[kCompactStreams + 1];
    __shared__ __align__(16) uint32_t buf[kCompactTile / 4];
    compact_streams<SCAN, SLICES>(p.level[blockIdx.y], rel, buf);
}

// collect_bytes for streams in a padded buffer (encoder.py:209-222): stream g = row * nc + channel
// goes to out[offsets[g] ...].  A wavefront copies four streams, a byte per lane: the streams are
// some tens of bytes long and begin anywhere.
constexpr int kCollectPerWave = 4;

__global__ __launch_bounds__(256) void collect_bytes_kernel(
    const uint8_t *__restrict__ padded, int64_t cap, int64_t p0, int64_t p1, const int64_t *__restrict__ offsets,
    int64_t nc, int64_t nstreams, uint8_t *__restrict__ out, int64_t out_bytes)
{
    const int lane = threadIdx.x & 63;
    const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kCollectPerWave;
#pragma unroll
    for (int i = 0; i < kCollectPerWave; ++i) {
        const int64_t g = first + i;
        if (g >= nstreams) return;
        const int64_t at = offsets[g];
        int64_t n = offsets[g + 1] - at;
        n = n < cap ? n : cap;
        if (at < 0 || at + n > out_bytes) continue;          // never write past the caller's buffer
        const uint8_t *src = padded + g / nc * p0 + g % nc * p1;
        for (int64_t j = lane; j < n; j += 64) out[at + j] = src[j];
    }
}

// What the host has to know before it makes room for those streams, stored straight into pinned
// memory (no copy, no second launch that reduces): out[0] = their bytes; out[1], zero before the
// launch, is set where the offsets do not begin at 0, a stream is longer than its slot, or a stream
// that is not empty has no slot among the buffer's nslots.  One load a thread, bound by its launch and
// the host's wait, which takes the place of reading the total back.  Without / with the check the four
// functions on one sub-chunk take 167.7 / 168.5 us (2 layers x 512 channels x 256 tokens), 111.0 / 111.5
// (36 layers, 86 tokens), 69.3 / 74.6 (2 layers x 1024 channels x 35 tokens: the host is the slower side).
__global__ __launch_bounds__(256) void collect_sizes_kernel(
    const int64_t *__restrict__ offsets, int64_t n, int64_t nslots, int64_t cap, int64_t *out)
{
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= n) return;
    const int64_t at = offsets[g], size = offsets[g + 1] - at;
    const bool last = g == n - 1, unfit = (g == 0 && at != 0) || size < 0 || size > (g < nslots ? cap : 0);
    if (last) out[0] = at + size;
    if (unfit) out[1] = 1;                               // everybody who writes writes the same
    if (last || unfit) host_stores_done();
}

__global__ void clear_status_kernel(int32_t *status) { *status = 0; }

}  // namespace
