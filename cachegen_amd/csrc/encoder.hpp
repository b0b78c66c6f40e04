// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Range encoder: word writer, coder state, encode_streams_kernel.
//
// Paths in the comments are relative to LMCache/ in the reference tree:
//   enc_new.cu = third_party/torchac_cuda/torchac_kernel_enc_new.cu
//   dec_new.cu = third_party/torchac_cuda/torchac_kernel_dec_new.cu
//   cal_cdf.cu = third_party/torchac_cuda/cal_cdf.cu
//   encoder.py = lmcache/storage_backend/serde/cachegen_encoder.py
//   decoder.py = lmcache/storage_backend/serde/cachegen_decoder.py
#pragma once

namespace {

// ---- encoder (enc_new.cu:21-97, 253-307) -------------------------------------------
// The reference's coder emits a bit for every E1/E2 step and counts E3 (underflow) steps as
// pending bits that follow the next emitted bit as its complements (enc_new.cu:86-97,
// 275-305).  That output is the binary expansion of the interval's lower end, written with
// carries: after a total of n renormalisation steps the bits emitted or pending are the
// lower end's first n bits, a pending run 0111..1 being a run of ones that a later carry may
// still turn into 1000..0, and the closing `pending + 2` bits (enc_new.cu:309-317) are the
// next two bits of the lower end plus a quarter of the window.  So the lower end is kept
// here as one long number: its last 32 bits (`low`, the coder's window; bit 31 can differ
// from the reference's, where an underflow step clears it, and nothing reads it) below 64
// bits that are waiting to be written (`out`).  A symbol adds its offset to the number and
// shifts it left by the step count n = clz(low ^ high) + (underflow steps); nothing is
// counted or spliced per symbol.  Words leave at fixed points, once per eight symbols (every
// lane of a wavefront runs the store code whenever one lane has a word ready); a carry out
// of the waiting bits is added to the last word, which is therefore held back one round
// (`cache`), and a word of all ones is only counted (`ones`) until the word after it shows
// whether the carry comes.  n <= 18 for any table whose symbols all have non-zero width,
// because the span stays above 2^30 between symbols.
constexpr int kSlotTile = 256;      // streams per tile of the encoder's scratch
// Tiles whose byte counts the coder's blocks also add up into one sum per group, so that the
// compaction finds a tile's place in the payload from at most kMaxTileGroups group sums and
// kTileGroup - 1 tile counts; calls with more groups run a scan launch over the tile counts.
constexpr int kTileGroup = 64;
constexpr int kMaxTileGroups = 256;

// Streams of a tile lie interleaved by quads of four words: word w of the tile's stream t is the tile's
// word (w / 4 * kSlotTile + t) * 4 + w % 4.  The words that a wavefront writes at about the same time share
// a few lines, and the many words of a long stream among short ones share theirs.  Streams that hardly fill a quad are
// interleaved word by word (word w of stream t is word w * kSlotTile + t): quads are four times the lines for
// a stream of one word.
constexpr int kQuadRow = kSlotTile * 16;        // bytes from one quad of a stream to the next
constexpr int kWordRow = kSlotTile * 4;         // bytes from one word of a stream to the next
// Symbols of a call's longest sub-chunk up to which its streams are interleaved word by word.  By words / by quads, the whole
// encode, us, 32 layers x 4096 tokens in chunks of   16         24         32         40         48         56         64         96
//   1024 channels, tables of 17 entries               700/724    556/569    441/444    415/416    383/385    364/364    338/338    313/312
//                            33                       897/941    731/759    546/556    526/533    469/473    448/449    402/401    359/357
//                            65                     1908/1944  1500/1522  1068/1076  1022/1028   879/883    814/819    692/695    601/600
//   400 channels, 33 entries                          490/505    377/384    288/291               244/244               198/198    187/186
// one chunk of so many tokens, 74 layers x 1536 ch.  51.8/52.1  53.9/53.9  54.6/54.8             58.9/58.8             62.2/61.7  69.4/69.3
constexpr int kShortStreams = 48;
// The bits of a word's offset in its tile that are the stream's place there; the others count the stream's words.
constexpr uint32_t kQuadPlace = kQuadRow - 16, kWordPlace = kWordRow - 4;

// TILE: the stream's words go to a tile of the scratch through a buffer descriptor that covers exactly the
// tile: a word or byte past the stream's capacity falls outside the descriptor and is dropped by the
// hardware, so nothing is compared or counted per word.  SLOTS without TILE: a tile through pointers, for blocks that
// are not whole tiles.  Neither: the stream's words lie one behind the other.
template <bool ALIGNED, bool SLOTS, bool TILE>
struct WordWriter {
    uint32_t place;         // SLOTS: kQuadPlace or kWordPlace (uniform)
    uint8_t *wptr;          // where the next word goes
    int cap;
    uint32_t whole;         // places a whole word can start at: cap - 3, or none
    int nbytes;             // bytes written so far; -4 before the held-back word's first, empty turn
    __amdgpu_buffer_rsrc_t tile;    // TILE: the block's tile
    uint32_t voff;                  // TILE: byte offset in the tile of the next word (of stream t's first: 16 t)

    // bytes from one word to the next inside a quad, and from its last word to the next quad's first
    __device__ __forceinline__ int step() const { return SLOTS && place == kWordPlace ? kWordRow : 4; }
    __device__ __forceinline__ int last_step() const { return !SLOTS ? 4 : place == kWordPlace ? kWordRow : kQuadRow - 12; }

    // SLOTS: dst is the tile and t the stream's place in it
    __device__ __forceinline__ void init(uint8_t *dst, int capacity, uint32_t tile_place = 0, uint32_t t = 0)
    {
        place = tile_place;
        // the first word stored is the empty held-back word: it goes one word before the
        // stream (TILE: the offset wraps and the hardware drops the store)
        wptr = dst + first(t) - last_step();
        cap = capacity;
        whole = capacity >= 4 ? (uint32_t)capacity - 3u : 0u;
        nbytes = -4;
        voff = (first(t) | ~place) & ~3u;
    }
    __device__ __forceinline__ uint32_t first(uint32_t t) const { return !SLOTS ? 0u : place == kWordPlace ? t * 4u : t * 16u; }

    __device__ __forceinline__ void store_word(uint32_t word)
    {
        if (TILE) {
            __builtin_amdgcn_raw_buffer_store_b32((int)__builtin_bswap32(word), tile, (int)voff, 0, 0);
            // the stream's place is all ones while 4 is added: the carry out of the bits below passes over it
            const uint32_t next = (voff | place) + 4u;
            asm("v_bitop3_b32 %0, %1, %0, %2 bitop3:0xD8" : "+v"(voff) : "v"(next), "s"(place));    // the place of voff, the rest of next
            return;
        }
        // one test on the common path: nbytes in [0, cap - 4]
        if (__builtin_expect((uint32_t)nbytes < whole, 1)) {
            if (ALIGNED) {
                *reinterpret_cast<uint32_t *>(wptr) = __builtin_bswap32(word);
            } else {
                wptr[0] = (uint8_t)(word >> 24);
                wptr[1] = (uint8_t)(word >> 16);
                wptr[2] = (uint8_t)(word >> 8);
                wptr[3] = (uint8_t)word;
            }
        } else if (nbytes >= 0) {
            // the last words of a stream that does not fit its slot: keep what fits
            for (int j = 0; j < 4; ++j)
                if (nbytes + j < cap) wptr[j] = (uint8_t)(word >> (24 - 8 * j));
        }
        wptr += SLOTS && (nbytes & 12) == 12 ? last_step() : step();
        nbytes += 4;
    }

    // the stream's last `nbits` bits (fewer than 32, left-aligned in `word`), byte by byte
    // (enc_new.cu:42-55); returns the stream length
    __device__ __forceinline__ int finish(uint32_t word, int nbits)
    {
        if (TILE) nbytes = place == kWordPlace ? (int)(voff / kWordRow * 4) : (int)((voff / kQuadRow << 4) | (voff & 12u));
        for (int left = nbits, j = 0; left > 0; left -= 8, ++j) {
            if (TILE) __builtin_amdgcn_raw_buffer_store_b8((char)(word >> 24), tile, (int)(voff + j), 0, 0);
            else if (nbytes < cap) wptr[j] = (uint8_t)(word >> 24);
            nbytes++;
            word <<= 8;
        }
        return nbytes;
    }
};

// The coder state is the number described above plus the interval's width less one,
// `span_less_one`: the full range 2^32 (the initial state, and any later interval that is exactly
// a binary fraction) is 2^32 - 1 there, and floor(span * c / 2^16) is the high word of
// span_less_one * (c << 16) + (c << 16) for every span, one 64-bit multiply-add with nothing set
// apart for the full range.  Renormalising by n bits maps span to span << n for E1/E2 and E3
// steps alike, span_less_one to itself with n ones moved in: the upper half of a 64-bit shift of
// `width_ones`, which holds the width less one above 32 ones.
//
// What bounds the coding loop is the issue of its vector instructions, 3.5 cycles each.  The width less one comes by one
// subtraction with a borrow that is always there, the next span by that shift, a symbol's table address by a shift and one
// v_bitop3 (RowPlace below), what a symbol's bits and its carry ask for by one branch, and a power of two of lanes a
// table row leaves no LDS bank conflicts (36.6 M cycles before): 169.2 -> 160.9 M instructions for 32 layers x
// 8192 tokens x 1024 channels, coder 272 -> 263 us, encode 606 -> 601; 80 layers x 32768 tokens 5918 -> 5839, four levels of
// 4096 tokens 1013 -> 987 (all of it together, each pair on one machine).  Forms in which the last symbol may occur
// (SENTINEL) compare the symbol and so extract it first.
template <int BS, bool ALIGNED, bool SLOTS, bool TILE, int kS>
struct RangeEncoder {
    static constexpr int kRow = 2 * kS;     // bytes from an entry to the next of the same table
    uint32_t col;           // LDS byte of this lane's table column: entry e at col + e * kRow
    uint32_t smax;          // lp - 2: the largest symbol
    uint64_t span;          // span_less_one in its upper half
    uint64_t width_ones;    // the coded symbol's width less one, above 32 ones
    // the number's last 96 bits: `tail` holds the window (its lower half, called low in the
    // comments) and above it the first 32 of the bits waiting to be written, `out_hi` the rest
    // of them: 63 - room bits wait, and above them there may be a carry (0 or 1) that belongs
    // to the held-back word
    uint64_t tail;
    uint32_t out_hi;
    // counted this way, the subtraction that books a shift borrows exactly when the bits (and
    // the place for a carry above them) do not fit, and that borrow is the test
    uint32_t room;
    uint32_t cache;         // the last complete word, not yet written: a carry may still reach it
    uint32_t ones;          // words of all ones that follow it
    uint32_t plain;         // 0xFFFFFFFF while `ones` is 0, else 0: a word below it is stored the short way
    // the coded symbol's two table entries, each shifted left by 16: only ever written by
    // loads into the upper half, so that the lower halves stay zero
    uint64_t bound_lo, bound_hi;
    WordWriter<ALIGNED, SLOTS, TILE> w;

    __device__ __forceinline__ void init(const uint16_t *column, int lp)
    {
        col = (uint32_t)(uintptr_t)(lds_char *)column;
        bound_lo = 0;
        bound_hi = 0;
        smax = (uint32_t)(lp - 2);
        span = ~0ull;
        width_ones = 0xFFFFFFFFu;
        tail = 0;
        out_hi = 0;
        room = 63;
        cache = 0;
        ones = 0;
        plain = 0xFFFFFFFFu;
    }

    // the held-back word, raised by the carry, and the words of all ones behind it (which the
    // carry turns into zeros); not on the common path
    __device__ __forceinline__ void release(uint32_t carry)
    {
        w.store_word(cache + carry);
        for (; ones; --ones) w.store_word(carry ? 0u : 0xFFFFFFFFu);
        plain = 0xFFFFFFFFu;
    }

    // takes the top 32 waiting bits (and the carry above them); needs at least 32 waiting
    __device__ __forceinline__ void flush_word()
    {
        const uint32_t sh = 31u - room;                 // waiting bits that stay
        const uint32_t out_lo = (uint32_t)(tail >> 32);
        const uint64_t top = (((uint64_t)out_hi << 32) | out_lo) >> sh;
        const uint32_t word = (uint32_t)top, carry = (uint32_t)(top >> 32);
        tail = ((uint64_t)__builtin_amdgcn_ubfe(out_lo, 0u, sh) << 32) | (uint32_t)tail;
        out_hi = 0;
        room += 32u;
        if (__builtin_expect(word < plain, 1)) {
            w.store_word(cache + carry);
            cache = word;
        } else {
            asm volatile("");
            if (carry) {
                release(1u);
                cache = word;
            } else if (word == 0xFFFFFFFFu) {
                ones++;
                plain = 0u;
            } else {
                release(0u);
                cache = word;
            }
        }
    }

    // The two steps below are written out instruction by instruction, on fixed registers
    // (tail in v[56:57], out_hi in v59, v58 as the lower half of the pair that shifts out_hi):
    // the 96-bit add is one carry chain and the 96-bit shift two 64-bit shifts and a move, which
    // the compiler does not find from C (it compares for the carry and shuffles the halves).

    // the number grows by `add` (a carry may run into the waiting bits)
    __device__ __forceinline__ void add_low(uint32_t add)
    {
        asm("v_add_co_u32 v56, vcc, v56, %2\n\ts_nop 1\n\t"
            "v_addc_co_u32 v57, vcc, 0, v57, vcc\n\ts_nop 1\n\t"
            "v_addc_co_u32 v59, vcc, 0, v59, vcc"
            : "+{v[56:57]}"(tail), "+{v59}"(out_hi)
            : "v"(add)
            : "vcc");
    }

    // the same for the lower bound (lo_pair's upper half) of a symbol with upper bound `hi`, without the third add (a carry out
    // of the 64 low bits needs 32 waiting ones: the lanes that have one are left in `carry`): leaves the width less
    // one in width_ones and gives the step count of the interval [low, low + width - 1], as step_count() has
    // it (common.hpp), four instructions after the window's add
    __device__ __forceinline__ int add_and_count(uint64_t lo_pair, uint32_t hi, uint64_t &carry)
    {
        int n;
        // (a carry that a vector instruction wrote is read no sooner than two instructions later, the distance that the
        // compiler keeps everywhere for this GPU; it sees nothing of what is written out here.  No change in time:
        // 599 -> 598 us an encode)
        asm("s_mov_b64 vcc, -1\n\tv_subb_co_u32 v61, vcc, %5, v63, vcc\n\t"
            "v_add_co_u32 v56, vcc, v56, v63\n\ts_nop 0\n\t"
            "v_add_u32 v62, v61, v56\n\t"
            "v_addc_co_u32 v57, %2, 0, v57, vcc\n\t"
            "v_bitop3_b32 v62, v62, v56, v61 bitop3:0x82\n\t"
            "v_lshl_or_b32 v62, v62, 1, v61\n\t"
            "v_ffbh_u32 %0, v62"
            : "=&v"(n), "+{v[62:63]}"(lo_pair), "=&s"(carry), "+{v[56:57]}"(tail), "+{v[60:61]}"(width_ones)
            : "v"(hi)
            : "vcc");
        return n;
    }
    __device__ __forceinline__ void add_carry(uint64_t carry)
    {
        asm("v_addc_co_u32 v59, %0, 0, v59, %0" : "+s"(carry), "+{v59}"(out_hi));
    }

    // n <= 31 bits more will wait; what is to happen for a carry out of the low bits and, unless ROOM (the
    // caller knows that the bits fit), where more than 32 bits were waiting already is left to one branch on
    // both, which is next to never taken
    template <bool ROOM>
    __device__ __forceinline__ void book(int n, uint64_t carry)
    {
        uint64_t full = 0;
        if (ROOM) room -= (uint32_t)n;
        else asm("v_sub_co_u32 %0, %1, %0, %2" : "+v"(room), "=s"(full) : "v"(n));
        if (__builtin_expect((carry | full) != 0, 0)) {
            add_carry(carry);
            if (!ROOM && (int32_t)room < 0) {
                room += (uint32_t)n;
                flush_word();
                room -= (uint32_t)n;
            }
        }
    }
    // the number moves left by n bits
    __device__ __forceinline__ void move(int n)
    {
        asm("v_mov_b32 v58, v57\n\t"
            "v_lshlrev_b64 v[58:59], %2, v[58:59]\n\t"
            "v_lshlrev_b64 v[56:57], %2, v[56:57]"
            : "+{v[56:57]}"(tail), "+{v59}"(out_hi)
            : "v"(n)
            : "v58");
    }

    // FIRST: the symbol directly follows a flush (the first of a group)
    // at: the LDS byte of the symbol's lower bound; top: the symbol is smax, whose upper bound is 2^16 and not
    // the table's last entry (enc_new.cu:270)
    template <bool FIRST>
    __device__ __forceinline__ void put_at(uint32_t at, bool top)
    {
        // both entries into the upper halves of the lower registers of two pairs whose upper
        // registers stay 0: the pairs are the entries shifted left by 16, as 64-bit values
        asm volatile("ds_read_u16_d16_hi v52, %2\n\tds_read_u16_d16_hi v54, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
                     : "+{v[52:53]}"(bound_lo), "+{v[54:55]}"(bound_hi)
                     : "v"(at), "n"(kRow));
        // T(c) = (span * c) >> 16 = high word of span * (c << 16) = high word of
        // span_less_one * (c << 16) + (c << 16): one 64-bit multiply-add, right for the full range
        // (span_less_one = 2^32 - 1) as for every other span, so no case is set apart
        // (the second product takes the span's place)
        const uint32_t all = top ? (uint32_t)(span >> 32) + 1u : 0u;            // T(2^16) is the span
        uint64_t prod;
        asm("v_mad_u64_u32 v[62:63], vcc, v51, v52, v[52:53]\n\tv_mad_u64_u32 v[50:51], vcc, v51, v54, v[54:55]"
            : "=&{v[62:63]}"(prod), "+{v[50:51]}"(span)
            : "{v[52:53]}"(bound_lo), "{v[54:55]}"(bound_hi)
            : "vcc");
        uint64_t carry;
        const int n = add_and_count(prod, top ? all : (uint32_t)(span >> 32), carry);
        book<FIRST>(n, carry);
        move(n);
        span = width_ones << n;
    }

    // SENTINEL: symbol smax may occur
    // CLAMP: the symbol may lie outside the table (it is kept inside; symbols that are known to
    // be table symbols skip the compare)
    template <bool SENTINEL, bool FIRST, bool CLAMP = true>
    __device__ __forceinline__ void put_symbol(uint32_t s)
    {
        if (CLAMP) s = s < smax ? s : smax;             // keep table reads inside the table
        put_at<FIRST>(col + s * (uint32_t)kRow, SENTINEL && s == smax);
    }

    // one group of symbols is through: write a word if 32 bits are waiting
    __device__ __forceinline__ void end_group()
    {
        if (room <= 31u) flush_word();
    }

    __device__ __forceinline__ int finish()
    {
        // the closing bits (enc_new.cu:309-317): the two bits below `out` of the number plus a
        // quarter of the window
        add_low(0x40000000u);
        book<false>(2, 0);
        move(2);
        end_group();
        const uint32_t nbits = 63u - room;              // fewer than 32 are left
        const uint32_t out_lo = (uint32_t)(tail >> 32);
        release(out_lo >> nbits);
        return w.finish(nbits ? out_lo << (32u - nbits) : 0u, (int)nbits);
    }
};

struct EncodeArgs {
    uint16_t *cdf;          // [chunk][row][channel][lp]; written when the histogram is fused
    int32_t lp;
    const uint8_t *sym;     // byte symbols: sym[row*s0 + token*s1 + channel*s2]
    int64_t s0, s1, s2;
    const uint32_t *sym4;   // or packed symbols
    int32_t nibbles;        // rows of at most 15 symbols are packed four bits a symbol (quantize_pack_kernel)
    const uint16_t *maxima; // the row maxima [2L, T] and their type, to know the rows that saturate (or null)
    int32_t max_dt;
    int64_t nsub;
    uint8_t *out;           // out[row*o0 + channel*o1 + byte], or the scratch tiles (SLOTS)
    int64_t o0, o1;
    int32_t cap;
    int32_t *lengths;       // [sub][row][channel]
    int32_t *status;        // may be null
    int32_t *tile_sums;     // SLOTS, one block per tile of kSlotTile streams: stored bytes per tile, or null
    int32_t *group_sums;    // with tile_sums, or null: the tile's bytes are also added to the sum of its
                            // group of kTileGroup tiles (zero before the launch)
    const float *key_bins, *value_bins;     // float32 [L] each, or null when the levels are not known
    int64_t L;
    StreamGrid sg;
    int32_t last_first;     // encode_streams_kernel: the last sub-chunk's blocks are the launch's first (code_last_first)
    uint32_t place;         // SLOTS: kQuadPlace or kWordPlace
};

// Several quantization levels of one tensor in one launch: what they share, and what differs.  Level v has the
// launch's blocks of z index v * nsub and up.
struct EncodeLevel {
    uint16_t *cdf;
    const uint32_t *sym4;
    uint8_t *out;
    int32_t *lengths, *status, *tile_sums, *group_sums;
    const float *key_bins, *value_bins;
    int32_t lp;
};
struct EncodeLevelsArgs {
    EncodeArgs all;
    EncodeLevel level[kMaxLevels];
};

// The arguments of the level that this block belongs to; z becomes the block's sub-chunk (uniform: at most seven
// subtractions on the scalar unit, once per block).
__device__ __forceinline__ EncodeArgs level_args(const EncodeLevelsArgs &p, uint32_t &z)
{
    int v = 0;
    while (z >= (uint32_t)p.all.nsub) {
        z -= (uint32_t)p.all.nsub;
        ++v;
    }
    const EncodeLevel &o = p.level[v];
    EncodeArgs a = p.all;
    a.cdf = o.cdf;
    a.sym4 = o.sym4;
    a.out = o.out;
    a.lengths = o.lengths;
    a.status = o.status;
    a.tile_sums = o.tile_sums;
    a.group_sums = o.group_sums;
    a.key_bins = o.key_bins;
    a.value_bins = o.value_bins;
    a.lp = o.lp;
    return a;
}

// How a packed word holds its four symbols: kBytes, a byte each (any value; kept inside the
// table where it is used); kNibbles, four bits each, every one a table symbol; kNibblesEscaped,
// four bits each where 15 stands for a saturated byte, i.e. the table's last symbol.
enum { kBytes = 0, kNibbles = 1, kNibblesEscaped = 2 };

template <bool SENTINEL_, int MODE_>
struct CodeTag {
    static constexpr bool SENTINEL = SENTINEL_;
    static constexpr int MODE = MODE_;
};

template <int MODE>
__device__ __forceinline__ uint32_t packed_symbol(uint32_t v, int j, uint32_t smax)
{
    if (MODE == kBytes) return (v >> (8 * j)) & 0xFFu;
    uint32_t s = __builtin_amdgcn_ubfe(v, (uint32_t)(4 * j), 4u);
    if (MODE == kNibblesEscaped) s = s == 15u ? smax : s;
    return s;
}

// The bytes that the block's streams occupy in the payload, for the compaction.  Every lane of the block
// is active where this is called (the host asks for tile sums only when a block is exactly one tile).
// wave_sums: BS / 64 words of LDS.
template <int BS>
__device__ __forceinline__ void leave_tile_sum(const EncodeArgs &a, int32_t *wave_sums, uint32_t tile, int tid, int len)
{
    int32_t v = len < a.cap ? len : a.cap;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((tid & 63) == 0) wave_sums[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) {
        int32_t total = 0;
        for (int w = 0; w < BS / 64; ++w) total += wave_sums[w];
        a.tile_sums[tile] = total;                            // at most 256 streams of 256 bytes
        if (a.group_sums) __hip_atomic_fetch_add(a.group_sums + tile / kTileGroup, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Entries of the coder's tables in LDS from one entry of a lane to its next.  Packed symbols: every lane reads and
// writes its own column only, so the row is the block's lanes and a power of two: a symbol's bits, moved to their place, and
// the column's make an entry's address without an add.  Byte symbols, whose tables are staged transposed: TableStride.
template <int BS, bool PACKED>
struct EncodeTable {
    static constexpr int kS = PACKED ? BS : TableStride<BS>::k16;
};
// Words of LDS behind the tables: one a wavefront for whether a row saturates, one a wavefront for the streams' bytes.
constexpr int kEncodeLdsWords = 8;
template <int BS, bool PACKED>
constexpr size_t encode_lds(int lp)
{
    return (size_t)lp * EncodeTable<BS, PACKED>::kS * sizeof(uint16_t) + kEncodeLdsWords * sizeof(uint32_t);
}

// Where the four symbols of a word go in an entry's address.  The tables begin at LDS byte 0 (no static
// LDS: the build checks it), a lane's column is below kRow and a symbol's entry a multiple of it, so
// the address is one v_bitop3 of the moved word, the symbol's bits there and the column.
template <int BS, int MODE>
struct RowPlace {
    static constexpr int kBit = BS == 256 ? 9 : BS == 128 ? 8 : 7;          // 2 BS bytes a row
    static_assert(2 * BS == 1 << kBit, "");
    static constexpr uint32_t kMask = (MODE == kBytes ? 0xFFu : 0xFu) << kBit;
    // a word of four-bit symbols is turned first, so that the lane's half begins at bit kBit: half_shift + turn
    static constexpr uint32_t kTurn = 32u - kBit;

    static __device__ __forceinline__ uint32_t entry(uint32_t v, int j, uint32_t col)
    {
        // the mask from a vector register: with a scalar operand the instruction takes a turn of its own (605 -> 600 us an encode)
        uint32_t x;
        const int left = MODE == kBytes ? kBit - 8 * j : -4 * j;
        if (left == 1) asm("v_add_u32 %0, %1, %1" : "=v"(x) : "v"(v));       // issues beside other wavefronts', a left shift does not
        else x = left >= 0 ? v << left : v >> -left;
        asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0xEA" : "=v"(x) : "v"(x), "v"(kMask), "v"(col));     // (x & mask) | col
        return x;
    }
};

// PACKED: symbols come from sym4.  FUSE_CDF (PACKED only, one sub-chunk per chunk): the
// block first builds its own tables from the same words and writes them out.
// SLOTS: stream g of the launch is written to out[g * cap ...] (the fused path's scratch).
// z: the block's sub-chunk, counted in the launch's order.
template <int BS, bool ALIGNED, bool PACKED, bool FUSE_CDF, bool SLOTS, bool TILE>
__device__ __forceinline__ void encode_streams(const EncodeArgs &a, uint16_t *tab, uint32_t z)
{
    const int tid = threadIdx.x;
    const uint32_t coder_sub = a.last_first ? (uint32_t)a.nsub - 1 - z : z;
    const StreamId id = locate<BS>(a.sg, coder_sub);
    const int lp = a.lp;
    const int64_t ch0 = (int64_t)blockIdx.x * BS;
    constexpr int kS = EncodeTable<BS, PACKED>::kS;
    uint16_t *col = tab + table_column<BS>(tid);
    int32_t *const lds_words = reinterpret_cast<int32_t *>(tab + lp * kS);          // kEncodeLdsWords
    uint16_t *cdf_block = a.cdf + ((id.chunk * a.sg.rows + id.row) * a.sg.nc + ch0) * lp;
    const int nwords = (id.n + 3) >> 2;
    // The row's alphabet (2C + 1 symbols for `bins` levels, encoder.py:44-52): it may leave the
    // table's last symbol unused (then its special upper bound is never needed), and with at
    // most 15 symbols the quantizer may have packed it four bits a symbol, two channels to a
    // word.  A token row whose scale overflowed (a maximum so small that MAX / max is infinite)
    // saturates its bytes to 255, which the reference's coder reads as the table's last symbol:
    // such bytes arrive as the value 15.  All uniform over the block.
    bool sentinel = true;
    int mode = kBytes;
    uint32_t half_shift = 0;
    float cq = 0.0f;
    const bool levels_known = PACKED && a.key_bins;
    if (levels_known) {
        const int64_t kvi = id.row >= a.L ? 1 : 0, l = id.row - kvi * a.L;       // 2L rows: keys, then values
        cq = floorf((kvi ? a.value_bins : a.key_bins)[l] * 0.5f) - 1.0f;
        sentinel = !(cq >= 0.0f && 2.0f * cq + 1.0f <= (float)(lp - 2));
        if (a.nibbles && narrow_alphabet(cq, lp)) {
            mode = kNibbles;
            half_shift = (uint32_t)(id.ch & 1) * 16u;
        }
    }

    // PACKED: the sub-chunk's words ([word][channel]) are read through a buffer descriptor that
    // ends with its last word row: the lane's channel is the vector offset, the word row the
    // scalar one, and a row past the end (or the offset of a lane without a channel) reads
    // zero, so a load costs no address arithmetic, compare or branch.
    __amdgpu_buffer_rsrc_t symbols_rsrc;
    uint32_t symbols_voff = 0xFFFFFFFCu;
    const uint32_t row_bytes = (uint32_t)a.sg.nc * (mode == kNibbles ? 2u : 4u);
    if (PACKED) {
        const int64_t first = ((id.row * a.nsub + id.sub) * kWordsPerSub) * a.sg.nc;        // uniform over the block
        const uint32_t lo32 = __builtin_amdgcn_readfirstlane((uint32_t)first);
        const uint32_t hi32 = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)first >> 32));
        symbols_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(a.sym4 + (int64_t)(((uint64_t)hi32 << 32) | lo32)), 0,
                                                         (int)((uint32_t)nwords * row_bytes), kBufferWord3);
        if (id.active) symbols_voff = (uint32_t)(mode == kNibbles ? id.ch >> 1 : id.ch) * 4u;
    }
    // Half a sub-chunk (32 words = 128 symbols) at a time is loaded into registers and indexed
    // by the (uniform) loop counter, so the coding loop has no loads to wait for and its stores
    // never hold it up.
    typedef uint32_t words32 __attribute__((ext_vector_type(32)));
    words32 words;
    auto load_half = [&](int h) {
#pragma unroll
        for (int w = 0; w < 32; ++w)
            words[w] = __builtin_amdgcn_raw_buffer_load_b32(symbols_rsrc, (int)symbols_voff,
                                                            (int)((uint32_t)(h * 32 + w) * row_bytes), 0);
    };

    if (levels_known && a.maxima) {
        int saturates = 0;
        // every token row of the sub-chunk, whatever the block size
        for (int i = tid; i < id.n; i += BS) {
            const uint32_t bits = a.maxima[id.row * a.sg.g.T + id.t0 + i];
            const float m = a.max_dt == CG_DT_BF16 ? load16f<CG_DT_BF16>(bits) : load16f<CG_DT_F16>(bits);
            saturates |= scale_overflows(cq, m);
        }
        // by hand: __syncthreads_or() takes LDS of its own, which would sit in front of the tables
        const bool wave_saturates = __any(saturates);
        if ((tid & 63) == 0) lds_words[tid >> 6] = wave_saturates;
        __syncthreads();
        int any = 0;
#pragma unroll
        for (int w = 0; w < BS / 64; ++w) any |= lds_words[w];
        if (__builtin_amdgcn_readfirstlane(any)) sentinel = true;       // the last symbol does occur
    }
    if (mode == kNibbles && sentinel) mode = kNibblesEscaped;

    if (FUSE_CDF) {
        for (int i = 0; i < lp; ++i) col[i * kS] = 0;
        __syncthreads();                     // another lane, of another wavefront, shares this lane's words
        if (id.active) {
            const uint32_t smax = (uint32_t)(lp - 2);
            // two lanes share a 32-bit LDS word: each adds to its own half with one atomic that
            // returns nothing (a count is at most 256, so the low half never carries over)
            uint32_t *const pair = reinterpret_cast<uint32_t *>(tab) + (table_column<BS>(tid) >> 1);
            const uint32_t one = (table_column<BS>(tid) & 1) ? 0x10000u : 1u;
            auto count = [&](auto tag) {
                constexpr int MODE = decltype(tag)::MODE;
                for (int h = 0; h * 32 < nwords; ++h) {
                    load_half(h);
                    // uniform; kept in a scalar register so that the loop test is scalar too
                    const int wn = __builtin_amdgcn_readfirstlane(nwords - h * 32 < 32 ? nwords - h * 32 : 32);
#pragma unroll 1
                    for (int w = 0; w < wn; ++w) {
                        const uint32_t v = MODE == kBytes ? words[w] : words[w] >> half_shift;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            uint32_t s = packed_symbol<MODE>(v, j, smax);
                            if (MODE == kBytes) s = s < smax ? s : smax;
                            if ((h * 32 + w) * 4 + j < id.n) atomicAdd(pair + (s + 1) * (kS / 2), one);
                        }
                    }
                }
            };
            if (mode == kNibbles) count(CodeTag<false, kNibbles>());
            else if (mode == kNibblesEscaped) count(CodeTag<false, kNibblesEscaped>());
            else count(CodeTag<false, kBytes>());
        }
        __syncthreads();                     // the other lane's counts are all in
        if (id.active) {
            normalize_column16_stride<kS>(col, lp, lp - 1, (uint32_t)id.n);
            write_column16_stride<kS>(col, cdf_block + (int64_t)tid * lp, lp);
        }
    } else if (!PACKED) {
        stage_tables16<BS>(tab, cdf_block, lp, ch0, a.sg.nc);
        __syncthreads();
    } else if (id.active) {
        // Packed symbols: every lane copies its own table (the transposed copy costs a division and a
        // dozen instructions an entry; this one costs the coder under one a symbol).  A lane reads
        // its own column only and LDS serves a wavefront's accesses in order: no barrier, but the
        // compiler must not move the coder's reads up.
        stage_column16_stride<kS>(col, cdf_block + (int64_t)tid * lp, lp);
        asm volatile("" ::: "memory");
    }
    if (!id.active) return;

    RangeEncoder<BS, ALIGNED, SLOTS, TILE, kS> enc;
    const int64_t stream = (id.sub * a.sg.rows + id.row) * a.sg.nc + id.ch;
    // SLOTS: the scratch is cut into tiles of kSlotTile streams
    if (TILE) {
        // the block is exactly one tile (the host launches this form only then): its number is
        // the tile, tid the stream's place in it
        enc.init(col, lp);
        enc.w.init(nullptr, a.cap, a.place, (uint32_t)tid);
        enc.w.tile = __builtin_amdgcn_make_buffer_rsrc((void *)(a.out + (int64_t)linear_block(coder_sub) * ((int64_t)kSlotTile * a.cap)), 0,
                                                       kSlotTile * a.cap, kBufferWord3);
    } else if (SLOTS) {
        enc.init(col, lp);
        enc.w.init(a.out + (stream / kSlotTile) * ((int64_t)kSlotTile * a.cap), a.cap, a.place, (uint32_t)(stream % kSlotTile));
    } else {
        enc.init(col, lp);
        enc.w.init(a.out + id.row * a.o0 + id.ch * a.o1, a.cap);
    }

    auto code = [&](auto tag) {
        constexpr bool SENTINEL = decltype(tag)::SENTINEL;
        constexpr int MODE = decltype(tag)::MODE;
        // a byte can lie outside the table only where the table's last symbol can occur at all
        // (a saturated row, a table shorter than the row's alphabet, symbols handed in by a caller)
        constexpr bool CLAMP = MODE == kBytes && SENTINEL;
        const uint32_t smax = (uint32_t)(lp - 2);
        if (PACKED) {
            typedef RowPlace<BS, MODE> Place;
            const uint32_t turn = half_shift + (SENTINEL ? 0u : Place::kTurn);          // modulo 32
            auto word = [&](uint32_t x) { return MODE == kBytes ? x : __builtin_amdgcn_alignbit(x, x, turn); };
            const int full = (id.n >> 3) * 2;              // words of full groups
            for (int h = 0; h == 0 || h * 32 < full; ++h) {
                load_half(h);
                // uniform; kept in a scalar register so that the loop test is scalar too
                const int wn = __builtin_amdgcn_readfirstlane(full - h * 32 < 32 ? full - h * 32 : 32);
                // two words = eight symbols between two visits of the store code, and no test per
                // symbol of whether there is one
                auto put = [&](auto first_tag, uint32_t v, int j) {
                    constexpr bool FIRST = decltype(first_tag)::value;
                    if (SENTINEL) enc.template put_symbol<SENTINEL, FIRST, CLAMP>(packed_symbol<MODE>(v, j, smax));
                    else enc.template put_at<FIRST>(Place::entry(v, j, enc.col), false);
                };
#pragma unroll 1
                for (int w = 0; w < wn; w += 2) {
                    const uint32_t v = word(words[w]);
                    put(BoolTag<true>(), v, 0);
                    put(BoolTag<false>(), v, 1);
                    put(BoolTag<false>(), v, 2);
                    put(BoolTag<false>(), v, 3);
                    // fetched only here: there is no register to hold it earlier
                    int w1 = w + 1;
                    asm volatile("" : "+s"(w1));
                    const uint32_t u = word(words[w1]);
                    put(BoolTag<false>(), u, 0);
                    put(BoolTag<false>(), u, 1);
                    put(BoolTag<false>(), u, 2);
                    put(BoolTag<false>(), u, 3);
                    enc.end_group();
                }
            }
            // the fewer than eight symbols behind the last full group, loaded again one at a time
            // (keeping the registers indexed up to here costs the kernel its eighth wavefront)
#pragma unroll 1
            for (int t = full * 4; t < id.n; ++t) {
                const uint32_t x = __builtin_amdgcn_raw_buffer_load_b32(symbols_rsrc, (int)symbols_voff, (int)((uint32_t)(t >> 2) * row_bytes), 0);
                const uint32_t v = word(x) >> (MODE == kBytes || SENTINEL ? 0 : Place::kBit);
                enc.template put_symbol<SENTINEL, false, CLAMP>(packed_symbol<MODE>(v, t & 3, smax));
            }
            enc.end_group();
        } else {
            const uint8_t *sp = a.sym + id.row * a.s0 + id.t0 * a.s1 + id.ch * a.s2;
            uint32_t nxt[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) nxt[j] = (j < id.n) ? sp[(int64_t)j * a.s1] : 0u;
            for (int i0 = 0; i0 < id.n; i0 += 8) {
                uint32_t cur[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) cur[j] = nxt[j];
#pragma unroll
                for (int j = 0; j < 8; ++j) nxt[j] = (i0 + 8 + j < id.n) ? sp[(int64_t)(i0 + 8 + j) * a.s1] : 0u;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if (j == 0) enc.template put_symbol<SENTINEL, true>(cur[j]);
                    else if (i0 + j < id.n) enc.template put_symbol<SENTINEL, false>(cur[j]);
                }
                enc.end_group();
            }
        }
    };
    if (PACKED && mode == kNibbles) code(CodeTag<false, kNibbles>());
    else if (PACKED && mode == kNibblesEscaped) code(CodeTag<true, kNibblesEscaped>());
    else if (PACKED && !sentinel) code(CodeTag<false, kBytes>());
    else code(CodeTag<true, kBytes>());
    const int len = enc.finish();
    // the lane's place by its index alone: nothing of the channel's number is kept in registers through the loop
    a.lengths[(id.sub * a.sg.rows + id.row) * a.sg.nc + ch0 + (uint32_t)tid] = len;
    if (len > a.cap && a.status) atomicOr(a.status, 1);
    if (SLOTS && a.tile_sums) leave_tile_sum<BS>(a, lds_words + BS / 64, linear_block(coder_sub), tid, len);
}

template <int BS, bool ALIGNED, bool PACKED, bool FUSE_CDF, bool SLOTS, bool TILE = false>
__global__ __launch_bounds__(BS) void encode_streams_kernel(EncodeArgs a)
{
    extern __shared__ uint16_t tab[];
    encode_streams<BS, ALIGNED, PACKED, FUSE_CDF, SLOTS, TILE>(a, tab, blockIdx.z);
}

// Packed symbols of several levels, into the scratch.
template <int BS, bool FUSE_CDF, bool TILE>
__global__ __launch_bounds__(BS) void encode_streams_levels_kernel(EncodeLevelsArgs p)
{
    extern __shared__ uint16_t tab[];
    uint32_t z = blockIdx.z;
    const EncodeArgs a = level_args(p, z);
    encode_streams<BS, true, true, FUSE_CDF, true, TILE>(a, tab, z);
}

}  // namespace
