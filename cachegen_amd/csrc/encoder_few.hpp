// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Range encoder for calls of few wavefronts: encode_few_kernel.
//
// Paths in the comments are relative to LMCache/ in the reference tree:
//   enc_new.cu = third_party/torchac_cuda/torchac_kernel_enc_new.cu
//   encoder.py = lmcache/storage_backend/serde/cachegen_encoder.py
#pragma once

namespace {

// A call of few wavefronts lasts as long as one stream's chain of symbols.  One wavefront alone on its
// SIMD issues a dependent instruction every 4.5 to 7 cycles and waits 49 for an LDS round trip, but 36 at every branch
// on a mask that a vector instruction made (issue_probe.hip): encode_streams_kernel, which takes one such
// branch a symbol (bits that do not fit, or a carry that runs far) and more with the store code, and
// reads a symbol's table entries when it comes to code it, takes 114 ns a symbol alone where this takes 93.  Here
//   - four symbols are coded without a branch: their bits are counted, and if a lane has more than
//     its register holds, or meets the full range, the wavefront codes the four again one by one,
//     exactly (tables of up to 64 symbols need 7.75 bits a symbol for that; a stream's first four
//     symbols go that way);
//   - the entries of eight symbols are read in one round trip, from tables of 32-bit entries;
//   - a sub-chunk's symbols are in registers before the first is coded;
//   - the store code runs once per eight symbols.
// 256 symbols of 65536 streams (one wavefront a SIMD; 32 layers x 1024 channels), encode_streams_kernel / here: 36 / 30 us, with
// the tables counted in the kernel 44 / 34, from byte symbols 52 / 38; of 128 symbols 21 / 18, 26 / 21, 30 / 22.
// The stream is the same number, written the same way (see encoder.hpp): the interval's lower end with
// its carries.
template <int BS, bool SLOTS, bool TILE>
struct FewEncoder {
    static constexpr int kRow = 4 * BS;     // bytes of a row of the tables: entry e << 16 of lane c at word e * BS + c
    lds_char *col;          // this lane's entry 0
    lds_char *top;          // the entry of the last symbol, whose upper bound is 2^16
    uint32_t span;          // the interval's width modulo 2^32: 0 is the full range
    uint64_t tail;          // the window in the lower half; above it the bits moved out of it since the last keep(), and a carry
    uint64_t out;           // `waiting` bits that wait to be written, and a carry (0 or 1) above them
    uint32_t waiting;       // at most 31 after take_words()
    uint32_t cache;         // the last complete word, not yet written: a carry may still reach it
    uint32_t ones;          // words of all ones that follow it
    WordWriter<true, SLOTS, TILE> w;

    __device__ __forceinline__ void init(const uint32_t *column, int lp)
    {
        col = (lds_char *)column;
        top = col + (lp - 2) * kRow;
        span = 0;
        tail = 0;
        out = 0;
        waiting = 0;
        cache = 0;
        ones = 0;
    }

    __device__ __forceinline__ lds_char *entry(uint32_t s) const { return col + s * (uint32_t)kRow; }
    static __device__ __forceinline__ uint32_t value(lds_char *at) { return *(lds_u32 *)at; }

    // the held-back word, raised by the carry, and the words of all ones behind it (which the
    // carry turns into zeros)
    __device__ __forceinline__ void release(uint32_t carry)
    {
        w.store_word(cache + carry);
        for (; ones; --ones) w.store_word(carry ? 0u : 0xFFFFFFFFu);
    }

    // writes the first 32 waiting bits of the lanes that have so many
    __device__ __forceinline__ void take_words()
    {
        if (waiting < 32u) return;
        waiting -= 32u;
        const uint64_t first = out >> waiting;
        const uint32_t word = (uint32_t)first, carry = (uint32_t)(first >> 32);
        out = __builtin_amdgcn_ubfe((uint32_t)out, 0u, waiting);
        if (__builtin_expect((word != 0xFFFFFFFFu) & (ones == 0u), 1)) {
            w.store_word(cache + carry);
            cache = word;
        } else if (!carry && word == 0xFFFFFFFFu) {
            ones++;
        } else {
            release(carry);
            cache = word;
        }
    }

    // the k <= 31 bits above the window join the waiting ones
    __device__ __forceinline__ void keep(uint32_t k)
    {
        out = (out << k) + (tail >> 32);
        waiting += k;
        tail = (uint32_t)tail;
    }

    // the interval becomes [low + t_lo, low + t_hi); returns the bits that leave the window
    __device__ __forceinline__ uint32_t narrow(uint32_t t_lo, uint32_t t_hi)
    {
        tail += t_lo;
        const uint32_t width = t_hi - t_lo, d = width - 1u, low = (uint32_t)tail;
        const int n = step_count(low, low + d, d);
        tail <<= n;
        span = width << n;
        return (uint32_t)n;
    }

    // one symbol, any interval: T(c) is c << 16 for the full range.  At most 31 bits may wait.
    template <bool SENTINEL>
    __device__ __forceinline__ void put_one(lds_char *at)
    {
        const uint32_t c_lo = value(at), c_hi = value(at + kRow);
        const uint32_t t_lo = span ? __umulhi(span, c_lo) : c_lo;
        uint32_t t_hi = span ? __umulhi(span, c_hi) : c_hi;
        if (SENTINEL && at == top) t_hi = span;
        keep(narrow(t_lo, t_hi));
        take_words();
    }

    // four symbols, whose entries are lo[j] and hi[j]
    template <bool SENTINEL>
    __device__ __forceinline__ void put_four(lds_char *const *at, const uint32_t *lo, const uint32_t *hi)
    {
        const uint32_t tail0 = (uint32_t)tail, span0 = span;
        const uint32_t most = 63u - waiting < 31u ? 63u - waiting : 31u;       // bits that fit above the window and behind the waiting ones
        uint32_t k = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t t_lo = __umulhi(span, lo[j]);
            uint32_t t_hi = __umulhi(span, hi[j]);
            if (SENTINEL && at[j] == top) t_hi = span;
            k += narrow(t_lo, t_hi);
        }
        // an interval that is the full range (span 0) stays it in these steps, so it is seen here
        const uint32_t bits = span ? k : 255u;
        if (__builtin_expect(__ballot(bits > most) != 0, 0)) {
            tail = tail0;
            span = span0;
            take_words();               // the second four of a group: put_one() wants room for its bits
#pragma unroll
            for (int j = 0; j < 4; ++j) put_one<SENTINEL>(at[j]);
            k = 0;
        }
        keep(k);
    }

    __device__ __forceinline__ int finish()
    {
        // the closing bits (enc_new.cu:309-317): the two bits of the number that follow plus a quarter
        // of the window
        tail = (tail + 0x40000000u) << 2;
        keep(2u);
        take_words();
        const uint32_t nbits = waiting & 31u;
        release((uint32_t)(out >> nbits));
        return w.finish(nbits ? (uint32_t)out << (32u - nbits) : 0u, (int)nbits);
    }
};

// The forms and arguments of encode_streams_kernel; streams begin at multiples of four bytes.
template <int BS, bool PACKED, bool FUSE_CDF, bool SLOTS, bool TILE>
__device__ __forceinline__ void encode_few(const EncodeArgs &a, uint32_t *entries, uint32_t z)
{
    const int tid = threadIdx.x;
    const StreamId id = locate<BS>(a.sg, z);
    const int lp = a.lp;
    uint32_t *col = entries + tid;
    uint16_t *mine = a.cdf + ((id.chunk * a.sg.rows + id.row) * a.sg.nc + id.ch) * lp;      // this lane's table in memory
    const uint32_t smax = (uint32_t)(lp - 2);
    // the row's alphabet: as in encode_streams_kernel
    bool sentinel = true;
    int mode = kBytes;
    float cq = 0.0f;
    const bool levels_known = PACKED && a.key_bins;
    if (levels_known) {
        const int64_t kvi = id.row >= a.L ? 1 : 0, l = id.row - kvi * a.L;       // 2L rows: keys, then values
        cq = floorf((kvi ? a.value_bins : a.key_bins)[l] * 0.5f) - 1.0f;
        sentinel = !(cq >= 0.0f && 2.0f * cq + 1.0f <= (float)(lp - 2));
        if (a.nibbles && narrow_alphabet(cq, lp)) mode = kNibbles;
    }
    // all of the sub-chunk's symbols, four to a word, in two halves of 32 words
    typedef uint32_t words32 __attribute__((ext_vector_type(32)));
    words32 words, later;
    const int nwords = (id.n + 3) >> 2;
    if (PACKED) {
        const uint32_t row_bytes = (uint32_t)a.sg.nc * (mode == kNibbles ? 2u : 4u);
        const int64_t first = ((id.row * a.nsub + id.sub) * kWordsPerSub) * a.sg.nc;        // uniform over the block
        const uint32_t lo32 = __builtin_amdgcn_readfirstlane((uint32_t)first);
        const uint32_t hi32 = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)first >> 32));
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.sym4 + (int64_t)(((uint64_t)hi32 << 32) | lo32)), 0, (int)((uint32_t)nwords * row_bytes), kBufferWord3);
        const uint32_t voff = !id.active ? 0xFFFFFFFCu : (uint32_t)(mode == kBytes ? id.ch : id.ch >> 1) * 4u;
#pragma unroll
        for (int w = 0; w < 32; ++w) words[w] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)voff, (int)((uint32_t)w * row_bytes), 0);
#pragma unroll
        for (int w = 0; w < 32; ++w) later[w] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)voff, (int)((uint32_t)(32 + w) * row_bytes), 0);
        if (mode == kNibbles && (id.ch & 1)) {
#pragma unroll
            for (int w = 0; w < 32; ++w) words[w] >>= 16, later[w] >>= 16;
        }
    }

    if (levels_known && a.maxima) {
        int saturates = 0;
        for (int i = tid; i < id.n; i += BS) {
            const uint32_t bits = a.maxima[id.row * a.sg.g.T + id.t0 + i];
            const float m = a.max_dt == CG_DT_BF16 ? load16f<CG_DT_BF16>(bits) : load16f<CG_DT_F16>(bits);
            saturates |= scale_overflows(cq, m);
        }
        if (__syncthreads_or(saturates)) sentinel = true;       // the last symbol does occur
    }
    if (mode == kNibbles && sentinel) mode = kNibblesEscaped;

    // Token t of the sub-chunk, from its word.
    auto symbol = [&](auto tag, uint32_t x, int j) {
        constexpr int MODE = decltype(tag)::MODE;
        const uint32_t s = packed_symbol<MODE>(x, j, smax);
        return MODE == kBytes && s > smax ? smax : s;           // table reads stay inside the table
    };
    if (FUSE_CDF) {
        // one counter per entry and lane, in the lane's own column: no barrier
        for (int i = 0; i < lp; ++i) col[i * BS] = 0;
        if (id.active) {
            auto count = [&](auto tag) {
                auto add = [&](uint32_t x, int j) { atomicAdd(col + (symbol(tag, x, j) + 1) * BS, 1u); };
                auto half = [&](const words32 &v, int w0) {
                    const int whole = (id.n >> 2) - w0;         // words of four tokens from here on
                    const int wn = __builtin_amdgcn_readfirstlane(whole < 32 ? whole : 32);
#pragma unroll 1
                    for (int w = 0; w < wn; ++w) {
                        const uint32_t x = v[w];
#pragma unroll
                        for (int j = 0; j < 4; ++j) add(x, j);
                    }
                    if (whole >= 0 && whole < 32)
                        for (int j = 0; j < (id.n & 3); ++j) add(v[__builtin_amdgcn_readfirstlane(whole)], j);
                };
                half(words, 0);
                half(later, 32);
            };
            if (mode == kNibbles) count(CodeTag<false, kNibbles>());
            else if (mode == kNibblesEscaped) count(CodeTag<false, kNibblesEscaped>());
            else count(CodeTag<false, kBytes>());
            normalize_counts(lp, 0xFFFFu - (uint32_t)(lp - 1), (uint32_t)id.n, [&](int i) { return col[i * BS]; },
                             [&](int i, uint32_t c) { col[i * BS] = c << 16; });
            // to memory: two entries per 32-bit store, one where the table starts or ends off a word boundary
            const int first = (int)((reinterpret_cast<uintptr_t>(mine) >> 1) & 1u);
            if (first) mine[0] = (uint16_t)(col[0] >> 16);
            const int npairs = (lp - first) >> 1;
            const uint32_t *src = col + first * BS;
            uint32_t *dst = reinterpret_cast<uint32_t *>(mine + first);
            constexpr int kPairs = 8;
            int i = 0;
#pragma unroll 1
            for (; i + kPairs <= npairs; i += kPairs) {
                uint32_t v[kPairs];
#pragma unroll
                for (int j = 0; j < kPairs; ++j) v[j] = src[2 * (i + j) * BS] >> 16 | src[(2 * (i + j) + 1) * BS];
#pragma unroll
                for (int j = 0; j < kPairs; ++j) dst[i + j] = v[j];
            }
            for (; i < npairs; ++i) dst[i] = src[2 * i * BS] >> 16 | src[(2 * i + 1) * BS];
            if ((lp - first) & 1) mine[lp - 1] = (uint16_t)(col[(lp - 1) * BS] >> 16);
        }
    } else if (id.active) {
        // every lane copies its own table; a lane reads its own column only: no barrier
        constexpr int kBatch = 16;
        int e0 = 0;
        for (; e0 + kBatch <= lp; e0 += kBatch) {
            uint16_t v[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) v[j] = mine[e0 + j];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) col[(e0 + j) * BS] = (uint32_t)v[j] << 16;
        }
        for (; e0 < lp; ++e0) col[e0 * BS] = (uint32_t)mine[e0] << 16;
    }
    asm volatile("" ::: "memory");          // LDS serves a wavefront's accesses in order
    if (!id.active) return;

    FewEncoder<BS, SLOTS, TILE> enc;
    const int64_t stream = (id.sub * a.sg.rows + id.row) * a.sg.nc + id.ch;
    enc.init(col, lp);
    if (TILE) {
        enc.w.init(nullptr, a.cap, a.place, (uint32_t)tid);
        enc.w.tile = __builtin_amdgcn_make_buffer_rsrc((void *)(a.out + (int64_t)linear_block(z) * ((int64_t)kSlotTile * a.cap)), 0,
                                                       kSlotTile * a.cap, kBufferWord3);
    } else if (SLOTS) {
        enc.w.init(a.out + (stream / kSlotTile) * ((int64_t)kSlotTile * a.cap), a.cap, a.place, (uint32_t)(stream % kSlotTile));
    } else {
        enc.w.init(a.out + id.row * a.o0 + id.ch * a.o1, a.cap);
    }

    auto code = [&](auto tag) {
        constexpr bool SENTINEL = decltype(tag)::SENTINEL;
        // eight symbols: the words x0 and x1
        auto group = [&](uint32_t x0, uint32_t x1) {
            lds_char *at[8];
            uint32_t lo[8], hi[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) at[j] = enc.entry(symbol(tag, j < 4 ? x0 : x1, j & 3));
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                lo[j] = enc.value(at[j]);
                hi[j] = enc.value(at[j] + enc.kRow);
            }
            enc.template put_four<SENTINEL>(at, lo, hi);
            enc.template put_four<SENTINEL>(at + 4, lo + 4, hi + 4);
            enc.take_words();
        };
        const int full = (id.n >> 3) * 2;                  // words of full groups
        if (PACKED) {
            for (int h = 0; h * 32 < full; ++h) {
                // uniform; kept in a scalar register so that the loop test is scalar too
                const int wn = __builtin_amdgcn_readfirstlane(full - h * 32 < 32 ? full - h * 32 : 32);
#pragma unroll 1
                for (int w = 0; w < wn; w += 2) group(words[w], words[w + 1]);
                if (h == 0 && full >= 32) words = later;
            }
            // the fewer than eight symbols behind the last full group, whose words are in `words` by now
#pragma unroll 1
            for (int t = full * 4; t < id.n; ++t) enc.template put_one<SENTINEL>(enc.entry(symbol(tag, words[(t >> 2) & 31], t & 3)));
        } else {
            // byte symbols: parts of 64 tokens, the next part's loads in flight while one is coded, one copy of
            // the code for all parts (straight-line code for 256 loads took a lone wavefront 24 us).  A
            // part's last loads may repeat the sub-chunk's last token.
            constexpr int kPart = 64;
            typedef uint32_t part_words __attribute__((ext_vector_type(kPart / 4)));
            const uint8_t *sp = a.sym + id.row * a.s0 + id.t0 * a.s1;             // uniform over the block
            const uint32_t voff = (uint32_t)id.ch * (uint32_t)a.s2;               // the host checks that this fits
            uint32_t bytes[kPart];
            auto fetch = [&](int t0) {
                const uint8_t *row = sp + (int64_t)t0 * a.s1;
#pragma unroll
                for (int j = 0; j < kPart; ++j) {
                    bytes[j] = row[voff];
                    if (t0 + j + 1 < id.n) row += a.s1;
                }
            };
            if (id.n > 0) fetch(0);
#pragma unroll 1
            for (int t0 = 0; t0 < id.n; t0 += kPart) {
                part_words part;
#pragma unroll
                for (int w = 0; w < kPart / 4; ++w)
                    part[w] = bytes[4 * w] | bytes[4 * w + 1] << 8 | bytes[4 * w + 2] << 16 | bytes[4 * w + 3] << 24;
                if (t0 + kPart < id.n) fetch(t0 + kPart);
                const int left = id.n - t0 < kPart ? id.n - t0 : kPart;
                const int wn = __builtin_amdgcn_readfirstlane((left >> 3) * 2);
#pragma unroll 1
                for (int w = 0; w < wn; w += 2) group(part[w], part[w + 1]);
#pragma unroll 1
                for (int t = wn * 4; t < left; ++t) enc.template put_one<SENTINEL>(enc.entry(symbol(tag, part[t >> 2], t & 3)));
            }
        }
    };
    if (PACKED && mode == kNibbles) code(CodeTag<false, kNibbles>());
    else if (PACKED && mode == kNibblesEscaped) code(CodeTag<true, kNibblesEscaped>());
    else if (PACKED && !sentinel) code(CodeTag<false, kBytes>());
    else code(CodeTag<true, kBytes>());
    const int len = enc.finish();
    a.lengths[stream] = len;
    if (len > a.cap && a.status) atomicOr(a.status, 1);
    if (SLOTS && a.tile_sums) {
        __shared__ int32_t wave_sums[BS / 64];
        leave_tile_sum<BS>(a, wave_sums, linear_block(z), tid, len);
    }
}

template <int BS, bool PACKED, bool FUSE_CDF, bool SLOTS, bool TILE = false>
__global__ __launch_bounds__(BS) void encode_few_kernel(EncodeArgs a)
{
    extern __shared__ uint32_t entries[];
    encode_few<BS, PACKED, FUSE_CDF, SLOTS, TILE>(a, entries, blockIdx.z);
}

template <int BS, bool FUSE_CDF, bool TILE>
__global__ __launch_bounds__(BS) void encode_few_levels_kernel(EncodeLevelsArgs p)
{
    extern __shared__ uint32_t entries[];
    uint32_t z = blockIdx.z;
    const EncodeArgs a = level_args(p, z);
    encode_few<BS, true, FUSE_CDF, true, TILE>(a, entries, z);
}

}  // namespace
