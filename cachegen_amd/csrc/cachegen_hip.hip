// CacheGen KV codec for MI355X (gfx950): hand-written HIP kernels behind a C ABI.
//
// The codec is HBM/ALU-bound integer work with no dense contraction, so there is
// no MFMA here.  The mapping everywhere is one lane = one (row, channel) stream
// and one wavefront = 64 adjacent channels of one row, which keeps every symbol
// and KV access of a wave on one contiguous segment; per-block tables live in LDS
// as 16-bit entries, one row of lanes per table entry (every lane has a column of its
// own; lanes whose symbols differ still meet on LDS banks now and then, which measured
// at 40 to 60 % of the LDS-busy cycles and does not limit these kernels: they are bound
// by vector instruction issue).  This file is the one translation unit: it includes the
// kernels and the launch helpers and defines the C ABI.
//
// Paths in the comments are relative to LMCache/ in the reference tree:
//   enc_new.cu = third_party/torchac_cuda/torchac_kernel_enc_new.cu
//   dec_new.cu = third_party/torchac_cuda/torchac_kernel_dec_new.cu
//   cal_cdf.cu = third_party/torchac_cuda/cal_cdf.cu
//   encoder.py = lmcache/storage_backend/serde/cachegen_encoder.py
//   decoder.py = lmcache/storage_backend/serde/cachegen_decoder.py
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <atomic>
#include <chrono>
#include <mutex>
#include <type_traits>

#include "cachegen_hip.h"

// The float32 steps of quantisation and dequantisation are rounded one by one, as eager
// tensor code rounds them: no fused multiply-add anywhere in this file.
#pragma clang fp contract(off)


#include "common.hpp"
#include "marks.hpp"
#include "quantize.hpp"
#include "tables.hpp"
#include "quantize_tables.hpp"
#include "encoder.hpp"
#include "encoder_few.hpp"
#include "decoder.hpp"
#include "scan_compact.hpp"
#include "launch.hpp"
#include "side_stream.hpp"
#include "host_lengths.hpp"
#include "host_copy.hpp"
#include "moves.hpp"
#include "tables_wire.hpp"

// ======================================================================================
// Scratch of the entry point that allocates nothing (cg_scan_lengths_static): the partial sums
// of the multi-block running sum, one int64 per 2048 lengths plus one.  Every GPU the library
// runs on holds its own copy of this array, at its own address, until the process ends.  In host
// code the array's name is only a handle for hipGetSymbolAddress: kernels and copies get the
// device address looked up once per device below, never the name.
// ======================================================================================
constexpr int64_t kStaticScanMaxLengths = CG_SCAN_STATIC_MAX_LENGTHS;
constexpr size_t kStaticScanBytes = (size_t)(kStaticScanMaxLengths / kScanTile + 2) * sizeof(int64_t);
static __device__ __align__(256) unsigned char scratch[kStaticScanBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_static_scratch_mutex;
void *g_static_scratch[kMaxDevices];          // device address of `scratch` on each GPU, once looked up

// Device address of `scratch` on the current device (looked up on the first call per device).
int static_scratch(void **ptr)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(CG_ERR_LAUNCH, "scan_lengths_static: hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(CG_ERR_ARG, "scan_lengths_static: device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (!g_static_scratch[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(CG_ERR_LAUNCH, "scan_lengths_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
        g_static_scratch[dev] = p;
    }
    *ptr = g_static_scratch[dev];
    return CG_OK;
}

}  // namespace

// ======================================================================================
// C ABI
// ======================================================================================
extern "C" {

const char *cg_last_error(void) { return g_error; }
int cg_abi_version(void) { return 5; }

int64_t cg_num_chunks(int64_t T, int64_t chunk_tokens)
{
    if (T <= 0 || chunk_tokens <= 0) return 0;
    return ceil_div(T, chunk_tokens);
}

int64_t cg_num_subchunks(int64_t T, int64_t chunk_tokens)
{
    if (T <= 0 || chunk_tokens <= 0) return 0;
    const int64_t nchunks = ceil_div(T, chunk_tokens);
    const int64_t last = T - (nchunks - 1) * chunk_tokens;
    return (nchunks - 1) * ceil_div(chunk_tokens, kSub) + ceil_div(last, kSub);
}

int cg_calculate_cdf(const int8_t *sym, int64_t nl, int64_t nt, int64_t nc, int64_t s0, int64_t s1,
                     int64_t s2, int max_bins, int16_t *cdf, void *stream)
{
    if (!sym || !cdf) return fail(CG_ERR_ARG, "calculate_cdf: null pointer");
    if (nl <= 0 || nt <= 0 || nc <= 0) return fail(CG_ERR_ARG, "calculate_cdf: empty input");
    if (max_bins < 1 || max_bins + 1 > CG_MAX_LP) return fail(CG_ERR_ARG, "Max bins must be less than %d", CG_MAX_LP);
    if (nt > 65535) return fail(CG_ERR_ARG, "calculate_cdf: at most 65535 tokens per table (16-bit counters)");
    return launch_cdf(reinterpret_cast<const uint8_t *>(sym), nullptr, 0, nl, nt, nc, s0, s1, s2, max_bins, nt,
                      reinterpret_cast<uint16_t *>(cdf), static_cast<hipStream_t>(stream));
}

int cg_encode_fast_new(const int16_t *cdf, int lp, const int8_t *sym, int64_t nl, int64_t nt, int64_t nc,
                       int64_t s0, int64_t s1, int64_t s2, uint8_t *out, int64_t cap, int64_t o0,
                       int64_t o1, int32_t *lengths, void *stream)
{
    if (!cdf || (!sym && nt > 0) || !out || !lengths) return fail(CG_ERR_ARG, "encode: null pointer");
    if (int rc = check_lp(lp, "encode")) return rc;
    if (nl <= 0 || nc <= 0 || nt < 0) return fail(CG_ERR_ARG, "encode: empty input");
    if (nt > kSub) return fail(CG_ERR_ARG, "Number of tokens should be less than or equal to %d", kSub);
    if (cap <= 0 || cap > INT_MAX) return fail(CG_ERR_ARG, "encode: bad output buffer length");
    const int block = pick_block(nc, lp);
    EncodeArgs a;
    memset(&a, 0, sizeof(a));
    a.cdf = reinterpret_cast<uint16_t *>(const_cast<int16_t *>(cdf));      // only read here
    a.lp = lp;
    a.sym = reinterpret_cast<const uint8_t *>(sym);
    a.s0 = s0;
    a.s1 = s1;
    a.s2 = s2;
    a.out = out;
    a.o0 = o0;
    a.o1 = o1;
    a.cap = (int32_t)cap;
    a.lengths = lengths;
    a.status = nullptr;
    int64_t nblocks;
    // nt == 0 still writes the two closing bits of every stream
    if (int rc = make_grid(nl, nc, nt ? nt : 1, nt ? nt : 1, 1, block, a.sg, nblocks)) return rc;
    if (nt == 0) a.sg.g.T = 0;
    const bool aligned = aligned_to(out, 4) && o0 % 4 == 0 && o1 % 4 == 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid = stream_grid(a.sg, nblocks);
    if (aligned) {
        // that form reaches a channel from its token row with a 32-bit offset
        const bool few = few_encode(nblocks, ENC_BYTES, lp, block, false) && s2 >= 0 && s2 <= 0x7FFFFFFFll / nc;
        CG_DISPATCH_BS(block, return (launch_encode<BS, false, false, false>(a, grid, few, st)));
    }
    CG_DISPATCH_BS(block, (encode_streams_kernel<BS, false, false, false, false><<<grid, dim3(block), encode_lds<BS, false>(lp), st>>>(a)));
    return check_launch("encode");
}

int cg_decode_fast_new(const int16_t *cdf, int lp, const uint8_t *padded, int64_t cap, int64_t p0,
                       int64_t p1, const int32_t *lengths, int64_t nl, int64_t nt, int64_t nc,
                       uint8_t *out, int64_t o0, int64_t o1, int64_t o2, void *stream)
{
    if (!cdf || !padded || !lengths || !out) return fail(CG_ERR_ARG, "decode: null pointer");
    if (int rc = check_lp(lp, "decode")) return rc;
    if (nl <= 0 || nc <= 0 || nt <= 0) return fail(CG_ERR_ARG, "decode: empty input");
    if (nt > kSub) return fail(CG_ERR_ARG, "Number of tokens should be less than or equal to %d", kSub);
    if (cap <= 0 || cap > INT_MAX) return fail(CG_ERR_ARG, "decode: bad padded buffer length");
    const bool few = few_wavefronts(nl, nc, 1, lp);
    const int block = few ? 64 : pick_block(nc, lp);
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    a.cdf = reinterpret_cast<const uint16_t *>(cdf);
    a.lp = lp;
    if (int rc = set_byte_window(a, padded, (nl - 1) * p0 + (nc - 1) * p1 + cap, "decode")) return rc;
    a.p0 = p0;
    a.p1 = p1;
    a.out_sym = out;
    a.o0 = o0;
    a.o1 = o1;
    a.o2 = o2;
    a.last_round_first = 0xFFFFFFFFu;     // one sub-chunk: a single round of blocks
    int64_t nblocks;
    if (int rc = make_grid(nl, nc, nt, nt, 1, block, a.sg, nblocks)) return rc;
    return launch_decode_symbols<SRC_PADDED>(a, nblocks, block, few, static_cast<hipStream_t>(stream));
}

int cg_decode_fast_prefsum(const int16_t *cdf, int lp, const uint8_t *bytes, int64_t nbytes,
                           const int64_t *prefix, int64_t nl, int64_t nt, int64_t nc, uint8_t *out,
                           int64_t o0, int64_t o1, int64_t o2, void *stream)
{
    if (!cdf || !prefix || !out || !bytes) return fail(CG_ERR_ARG, "decode: null pointer");
    if (int rc = check_lp(lp, "decode")) return rc;
    if (nl <= 0 || nc <= 0 || nt <= 0) return fail(CG_ERR_ARG, "decode: empty input");
    if (nt > kSub) return fail(CG_ERR_ARG, "Number of tokens should be less than or equal to %d", kSub);
    const bool few = few_wavefronts(nl, nc, 1, lp);
    const int block = few ? 64 : pick_block(nc, lp);
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    a.cdf = reinterpret_cast<const uint16_t *>(cdf);
    a.lp = lp;
    if (int rc = set_byte_window(a, bytes, nbytes, "decode")) return rc;
    a.offsets = prefix;
    a.out_sym = out;
    a.o0 = o0;
    a.o1 = o1;
    a.o2 = o2;
    a.last_round_first = 0xFFFFFFFFu;     // one sub-chunk: a single round of blocks
    int64_t nblocks;
    if (int rc = make_grid(nl, nc, nt, nt, 1, block, a.sg, nblocks)) return rc;
    return launch_decode_symbols<SRC_PREFIX>(a, nblocks, block, few, static_cast<hipStream_t>(stream));
}

int cg_quantize_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl,
                   int64_t skv, int64_t st, int64_t sh, const float *key_bins, const float *value_bins,
                   uint8_t *sym, void *maxima, void *stream)
{
    if (!kv || !key_bins || !value_bins || !sym || !maxima) return fail(CG_ERR_ARG, "quantize: null pointer");
    if (int rc = check_dt(kv_dt, "quantize")) return rc;
    if (L <= 0 || T <= 0 || H <= 0 || D <= 0) return fail(CG_ERR_ARG, "quantize: empty input");
    return launch_quantize(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, sym, maxima,
                           static_cast<hipStream_t>(stream));
}

int cg_collect_bytes(const uint8_t *padded, int64_t cap, int64_t p0, int64_t p1, const int64_t *offsets, int64_t nl, int64_t nc,
                     uint8_t *out, int64_t out_bytes, void *stream)
{
    if (!padded || !offsets || !out) return fail(CG_ERR_ARG, "collect_bytes: null pointer");
    if (nl <= 0 || nc <= 0 || cap <= 0 || out_bytes <= 0) return fail(CG_ERR_ARG, "collect_bytes: empty input");
    const int64_t nblocks = ceil_div(nl * nc, 4 * kCollectPerWave);
    if (nblocks > INT_MAX) return fail(CG_ERR_ARG, "collect_bytes: too many streams");
    collect_bytes_kernel<<<dim3((unsigned)nblocks), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(padded, cap, p0, p1, offsets, nc,
                                                                                                     nl * nc, out, out_bytes);
    return check_launch("collect_bytes");
}

int cg_collect_sizes(const int64_t *offsets, int64_t n, int64_t nslots, int64_t cap, int64_t *out, void *stream)
{
    if (!offsets || !out) return fail(CG_ERR_ARG, "collect_sizes: null pointer");
    const int64_t nblocks = ceil_div(n, 256);
    if (n <= 0 || nslots <= 0 || cap <= 0 || nblocks > INT_MAX) return fail(CG_ERR_ARG, "collect_sizes: bad count");
    collect_sizes_kernel<<<dim3((unsigned)nblocks), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(offsets, n, nslots, cap, out);
    return check_launch("collect_sizes");
}

size_t cg_scan_workspace(int64_t n) { return align_up((size_t)(ceil_div(n > 0 ? n : 1, kScanTile) + 1) * sizeof(int64_t), 256); }

int cg_scan_lengths(const int32_t *lengths, int64_t n, int64_t *offsets, void *scratch,
                    size_t scratch_bytes, void *stream)
{
    if (!lengths || !offsets || !scratch) return fail(CG_ERR_ARG, "scan: null pointer");
    if (n <= 0) return fail(CG_ERR_ARG, "scan: empty input");
    if (scratch_bytes < cg_scan_workspace(n)) return fail(CG_ERR_WORKSPACE, "scan: scratch too small");
    return launch_scan(lengths, n, INT_MAX, offsets, scratch, static_cast<hipStream_t>(stream));
}

int cg_scan_lengths_static(const int32_t *lengths, int64_t n, int64_t *offsets, void *stream)
{
    if (!lengths || !offsets) return fail(CG_ERR_ARG, "scan_lengths_static: null pointer");
    if (n <= 0) return fail(CG_ERR_ARG, "scan_lengths_static: empty input");
    if (n > kStaticScanMaxLengths)
        return fail(CG_ERR_WORKSPACE, "scan_lengths_static: %lld lengths exceed the built-in scratch (at most %lld); "
                                      "use cg_scan_lengths with a workspace", (long long)n, (long long)kStaticScanMaxLengths);
    void *ptr = nullptr;
    if (int rc = static_scratch(&ptr)) return rc;
    // every partial sum the second and third kernel read is written by the first kernel of this
    // same call, so nothing of the previous call's contents has to be cleared
    return launch_scan(lengths, n, INT_MAX, offsets, ptr, static_cast<hipStream_t>(stream));
}

}  // extern "C"

namespace {

// Workspace of the fused encoder, carved in this order: `nlevels` symbol areas (a 256-token
// slot per stream each); `areas` times the coder's scratch tiles and the small arrays of the two running
// sums; the group sums of all levels.  The pointers are level 0's; level(v) has those of level v.
// areas: one for each level, or one that levels coded one behind the other share.
struct EncodeWorkspace {
    size_t symbols_bytes;       // one level's symbols
    size_t area_bytes;          // one area's scratch and sums
    int areas;
    uint8_t *symbols, *scratch;
    void *scan_scratch, *tile_scan_scratch;
    int32_t *tile_sums, *group_sums;
    int64_t *tile_base;
    int64_t nsub, nstreams, ntiles;
    uint32_t place;             // how streams lie in their tile
    size_t total;

    EncodeWorkspace(void *base, int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels, int nareas = 1) : areas(nareas)
    {
        nsub = cg_num_subchunks(T, chunk_tokens);
        nstreams = nsub * 2 * L * C;
        ntiles = ceil_div(nstreams, kSlotTile);
        place = chunk_tokens <= kShortStreams || T <= kShortStreams ? kWordPlace : kQuadPlace;
        symbols_bytes = align_up((size_t)nstreams * kSub, 256);
        uint8_t *ws = static_cast<uint8_t *>(base);
        symbols = ws;
        ws += symbols_bytes * (size_t)nlevels;
        scratch = ws;           // kStreamCap bytes per stream, in tiles of kSlotTile streams (kQuadPlace, kWordPlace)
        ws += (size_t)ntiles * kSlotTile * kStreamCap;
        scan_scratch = ws;
        ws += cg_scan_workspace(nstreams);
        tile_sums = reinterpret_cast<int32_t *>(ws);           // bytes per tile of streams
        ws += align_up((size_t)ntiles * sizeof(int32_t), 256);
        tile_base = reinterpret_cast<int64_t *>(ws);           // their running sums
        ws += align_up((size_t)(ntiles + 1) * sizeof(int64_t), 256);
        tile_scan_scratch = ws;
        ws += cg_scan_workspace(ntiles);
        area_bytes = align_up((size_t)(ws - scratch), 256);
        ws = scratch + area_bytes * (size_t)areas;
        group_sums = reinterpret_cast<int32_t *>(ws);          // bytes per group of kTileGroup tiles
        ws += align_up((size_t)nlevels * kMaxTileGroups * sizeof(int32_t), 256);
        total = (size_t)(ws - static_cast<uint8_t *>(base));
    }

    EncodeWorkspace level(int v) const
    {
        EncodeWorkspace w = *this;
        const size_t by = areas > 1 ? area_bytes * (size_t)v : 0;
        w.symbols += symbols_bytes * (size_t)v;
        w.scratch += by;
        w.scan_scratch = static_cast<uint8_t *>(scan_scratch) + by;
        w.tile_scan_scratch = static_cast<uint8_t *>(tile_scan_scratch) + by;
        w.tile_sums += by / sizeof(int32_t);
        w.tile_base += by / sizeof(int64_t);
        w.group_sums += (size_t)v * kMaxTileGroups;
        return w;
    }
};

// Tiles of a level up to which several levels have an area of scratch each, so that they can share launches: that is
// 1 GB of scratch for one level and 3 more for four.  Beyond, the launches' ends matter little and the memory much.  Four levels
// of 1024 channels, one behind the other with one scratch / shared, us: 32 layers x 4096 tokens in chunks of 128 (8192 tiles)
// 1381 / 1305, 8192 tokens in chunks of 256 2155 / 2060, 16384 tokens (16384 tiles) 4250 / 4100 and 4720 / 4407 with one
// table over them; 2048 tokens in chunks of 16 (32768 tiles) 2958 / 2984, 4096 tokens (65536) 5957 / 5950, 80 layers x 32768
// tokens in chunks of 256 (81920) 20480 / 20380 with 27 GB of workspace / 43.
constexpr int64_t kApartTiles = 16384;

int level_areas(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels)
{
    return ceil_div(cg_num_subchunks(T, chunk_tokens) * 2 * L * C, kSlotTile) <= kApartTiles ? nlevels : 1;
}

}  // namespace

extern "C" {

size_t cg_encode_kv_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens)
{
    return EncodeWorkspace(nullptr, L, T, C, chunk_tokens, 1).total;
}

size_t cg_encode_kv_levels_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels)
{
    if (nlevels < 1 || nlevels > CG_MAX_LEVELS) return 0;
    return EncodeWorkspace(nullptr, L, T, C, chunk_tokens, nlevels, level_areas(L, T, C, chunk_tokens, nlevels)).total;
}

size_t cg_encode_kv_levels_least_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels)
{
    if (nlevels < 1 || nlevels > CG_MAX_LEVELS) return 0;
    return EncodeWorkspace(nullptr, L, T, C, chunk_tokens, nlevels).total;
}

}  // extern "C"

namespace {

// What one quantization level's outputs are.
struct LevelOut {
    const float *key_bins, *value_bins;
    int max_bins;
    int16_t *cdf;
    int32_t *lengths;
    int64_t *offsets;
    uint8_t *payload;
    int64_t payload_cap;
    int32_t *status;
};

// The compaction's arguments, after the scan launches that it needs.  fused_scan: the coder left its tiles' byte
// counts; grouped: and their sums by groups of tiles.
int scan_for_compaction(const LevelOut &o, const EncodeWorkspace &w, bool fused_scan, bool grouped, const int32_t *group_sums, CompactArgs &c, hipStream_t s)
{
    const int32_t skew = (int32_t)(reinterpret_cast<uintptr_t>(o.payload) & 3u);
    const int64_t *tile_base = nullptr;
    if (fused_scan && !grouped && w.ntiles > kDirectTiles) {
        if (int rc = launch_scan(w.tile_sums, w.ntiles, INT_MAX, w.tile_base, w.tile_scan_scratch, s)) return rc;
        tile_base = w.tile_base;
    } else if (!fused_scan) {
        if (int rc = launch_scan(o.lengths, w.nstreams, kStreamCap, o.offsets, w.scan_scratch, s)) return rc;
    }
    c = {w.scratch, kStreamCap, o.offsets, fused_scan ? o.lengths : nullptr, tile_base, w.nstreams, o.payload,
         o.payload_cap, skew, o.status, grouped ? group_sums : nullptr, fused_scan ? w.tile_sums : nullptr, w.place};
    return CG_OK;
}

// Tables, streams and payload of one level from its symbols (packed words `sym4`, or byte
// symbols [2L, T, C]): calculate_cdf + encode_fast_new + collect_bytes for every chunk
// (encoder.py:265-292, 209-222).
// The level's status word has been set to zero by an earlier launch of the same call.
// maxima, max_dt: the row maxima (packed symbols only); nibbles: the quantizer packed the rows
// of at most 15 symbols four bits a symbol (see narrow_alphabet).
// tables_ready: the tables were written by an earlier launch of the call (quantize_tables_kernel).
// group_sums: kMaxTileGroups words that an earlier launch of the call set to zero, or null.  may_be_few: false keeps encode_few_kernel out.
int code_and_compact(const LevelOut &o, const uint32_t *sym4, const uint8_t *sym_bytes, const EncodeWorkspace &w,
                     int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, hipStream_t s,
                     const void *maxima = nullptr, int max_dt = 0, bool nibbles = false, bool tables_ready = false,
                     int32_t *group_sums = nullptr, bool may_be_few = true)
{
    const int64_t rows = 2 * L;
    const int lp = o.max_bins + 1;
    uint16_t *tables = reinterpret_cast<uint16_t *>(o.cdf);

    const int block = pick_block(C, lp);
    EncodeArgs a;
    memset(&a, 0, sizeof(a));
    a.cdf = tables;
    a.lp = lp;
    a.nsub = w.nsub;
    a.out = w.scratch;
    a.cap = kStreamCap;
    a.lengths = o.lengths;
    a.status = o.status;
    a.key_bins = o.key_bins;
    a.value_bins = o.value_bins;
    a.L = L;
    int64_t nblocks;
    if (int rc = make_grid(rows, C, T, chunk_tokens, w.nsub, block, a.sg, nblocks)) return rc;
    const dim3 grid = stream_grid(a.sg, nblocks);
    // when every encoder block is exactly one tile of the scratch, the blocks leave their byte
    // counts behind and the compaction computes the stream offsets itself
    const bool fused_scan = block == kSlotTile && C % kSlotTile == 0;
    a.tile_sums = fused_scan ? w.tile_sums : nullptr;
    // few enough tiles: no scan launch either, the coder's blocks add the counts up by groups of
    // tiles (the sums were cleared by the call's quantizer) and the compaction adds up what lies before
    // each tile: four levels of 32 layers x 4096 tokens x 1024 channels 1164 -> 1153 us, 32 layers x 4096
    // tokens x 4096 channels 1292 -> 1280 (both through quantize_pack_kernel)
    const bool grouped = fused_scan && group_sums && ceil_div(w.ntiles, kTileGroup) <= kMaxTileGroups;
    a.group_sums = grouped ? group_sums : nullptr;
    a.last_first = code_last_first(w.ntiles);
    a.place = w.place;

    if (sym4) {
        // four tokens per word, read by one lane per channel
        a.sym4 = sym4;
        a.nibbles = nibbles ? 1 : 0;
        a.maxima = static_cast<const uint16_t *>(maxima);
        a.max_dt = max_dt;
        const EncodeSource source = tables_ready ? ENC_QUANTIZER_TABLES : chunk_tokens <= kSub ? ENC_COUNTED : ENC_TABLES;
        const bool few = may_be_few && few_encode(nblocks, source, lp, block, fused_scan);
        int rc = CG_OK;
        if (source == ENC_COUNTED) {
            // one sub-chunk per chunk: the encoder builds the tables itself
            if (fused_scan) rc = launch_encode<kSlotTile, true, true, true, true>(a, grid, few, s);
            else CG_DISPATCH_BS(block, rc = (launch_encode<BS, true, true, true>(a, grid, few, s)));
        } else {
            if (!tables_ready)
                rc = launch_cdf(nullptr, sym4, w.nsub, rows, T, C, 0, 0, 0, o.max_bins, chunk_tokens, tables, s,
                                nibbles ? o.key_bins : nullptr, nibbles ? o.value_bins : nullptr);
            if (rc) return rc;
            if (fused_scan) rc = launch_encode<kSlotTile, true, false, true, true>(a, grid, few, s);
            else CG_DISPATCH_BS(block, rc = (launch_encode<BS, true, false, true>(a, grid, few, s)));
        }
        if (rc) return rc;
    } else {
        // any shape or alignment: byte symbols [2L, T, C]
        if (int rc = launch_cdf(sym_bytes, nullptr, 0, rows, T, C, T * C, C, 1, o.max_bins, chunk_tokens, tables, s)) return rc;
        a.sym = sym_bytes;
        a.s0 = T * C;
        a.s1 = C;
        a.s2 = 1;
        CG_DISPATCH_BS(block, (encode_streams_kernel<BS, true, false, false, true><<<grid, dim3(block), encode_lds<BS, false>(lp), s>>>(a)));
        if (int rc = check_launch("encode_kv")) return rc;
    }

    const int64_t cblocks = ceil_div(w.nstreams, kCompactStreams);
    if (cblocks > INT_MAX) return fail(CG_ERR_ARG, "encode_kv: too many streams");
    CompactArgs c;
    if (int rc = scan_for_compaction(o, w, fused_scan, grouped, group_sums, c, s)) return rc;
    const dim3 cgrid((unsigned)cblocks);
    if (cblocks <= sliced_compact_blocks()) {
        if (fused_scan) compact_few_kernel<true><<<cgrid, dim3(1024), 0, s>>>(c);
        else compact_few_kernel<false><<<cgrid, dim3(1024), 0, s>>>(c);
    } else {
        if (fused_scan) compact_streams_kernel<true><<<cgrid, dim3(256), 0, s>>>(c);
        else compact_streams_kernel<false><<<cgrid, dim3(256), 0, s>>>(c);
    }
    return check_launch("compact");
}

// Whether levels of these table sizes can share launches: blocks of 256 lanes for all of them, and sub-chunks of
// all levels are one grid dimension.
bool levels_alike(const int *max_bins, int n, int64_t nsub, int64_t C)
{
    bool alike = n > 1 && nsub * n <= 65535;
    for (int v = 0; v < n; ++v) alike = alike && pick_block(C, max_bins[v] + 1) == kSlotTile;
    return alike;
}

// Several levels of one tensor from their packed symbols (level v's in w.level(v)): as code_and_compact for each,
// with a launch for all of them where they can share one.  A launch of one level ends with its slowest streams
// while the next waits, and a small one does not fill the GPU: it lasts as long as one stream's chain of symbols,
// as often as there are levels.  Tables of 9, 17, 33 and 65 entries, a launch per level / shared, the whole call, us:
//                     chunks of 256 tokens    300 tokens      one chunk
//   1024 channels  32 layers x 4096 tokens  1153 / 1070   1504 / 1436   1255 / 1144
//                  32 x 1024                 382 /  328    493 /  434    416 /  345
//                  32 x  256                 178 /  102
//                   4 x  256                 155 /   59
//    512 channels  32 x 4096                 695 /  618    918 /  830    785 /  668
//                   4 x 2048                 169 /   71    199 /  101    244 /   89
//   4096 channels  32 x 1024                1348 / 1250   1877 / 1806   1467 / 1385
// Other tables, 1024 channels in chunks of 256 tokens, with every length that a compute unit holds another number of blocks of
// in a launch of its own (below):
//                         32 layers x 4096 tokens     32 x 1024     4 x 256
//   41, 49, 57, 65                  1713 / 1600       555 / 519    213 /  69
//   17, 41, 57, 65                  1574 / 1449       515 / 480    195 /  66
//   13, 21, 33                       978 /  894       328 / 266    125 /  60
//   65, 65                           965 /  907       276 / 263    109 /  60
//   9 to 65, eight levels           2890 / 2667       977 / 823    372 /  76
int code_and_compact_levels(const LevelOut *o, int n, const EncodeWorkspace &w, int64_t L, int64_t T, int64_t C,
                            int64_t chunk_tokens, hipStream_t s, const void *maxima, int max_dt, bool sums_cleared)
{
    const int64_t rows = 2 * L;
    int max_lp = 0, max_bins[kMaxLevels];
    for (int v = 0; v < n; ++v) {
        max_bins[v] = o[v].max_bins;
        if (max_bins[v] + 1 > max_lp) max_lp = max_bins[v] + 1;
    }
    if (w.areas != n || !levels_alike(max_bins, n, w.nsub, C)) {
        for (int v = 0; v < n; ++v) {
            const EncodeWorkspace wv = w.level(v);
            if (int rc = code_and_compact(o[v], reinterpret_cast<uint32_t *>(wv.symbols), nullptr, wv, L, T, C, chunk_tokens, s, maxima, max_dt,
                                          true, false, sums_cleared ? wv.group_sums : nullptr)) return rc;
        }
        return CG_OK;
    }
    EncodeLevelsArgs p;
    memset(&p, 0, sizeof(p));
    EncodeArgs &a = p.all;
    a.nsub = w.nsub;
    a.cap = kStreamCap;
    a.L = L;
    a.nibbles = 1;
    a.maxima = static_cast<const uint16_t *>(maxima);
    a.max_dt = max_dt;
    a.last_first = code_last_first(w.ntiles);
    a.place = w.place;
    int64_t nblocks;
    if (int rc = make_grid(rows, C, T, chunk_tokens, w.nsub, kSlotTile, a.sg, nblocks)) return rc;
    if (nblocks > INT_MAX / kMaxLevels) return fail(CG_ERR_ARG, "encode_kv_levels: too many streams");
    const bool fused_scan = C % kSlotTile == 0;             // as in code_and_compact
    const bool grouped = fused_scan && sums_cleared && ceil_div(w.ntiles, kTileGroup) <= kMaxTileGroups;
    const bool counted = chunk_tokens <= kSub;              // the coder makes the tables
    if (!counted) {
        CdfLevelsArgs t;
        memset(&t, 0, sizeof(t));
        t.all.nsub = w.nsub;
        t.all.nibbles = 1;
        t.all.L = L;
        t.all.rows = rows;
        t.all.nc = C;
        t.all.g = a.sg.g;
        for (int v = 0; v < n; ++v)
            t.level[v] = {reinterpret_cast<const uint32_t *>(w.level(v).symbols), o[v].key_bins, o[v].value_bins,
                          reinterpret_cast<uint16_t *>(o[v].cdf), o[v].max_bins};
        CdfGrid g;
        if (int rc = make_cdf_grid(t.all, true, n, max_lp, g)) return rc;
        if (g.sliced) CG_DISPATCH_BS(g.block, (calculate_cdf_levels_kernel<BS, 4><<<g.grid, dim3(BS * 4), g.shmem, s>>>(t)));
        else CG_DISPATCH_BS(g.block, (calculate_cdf_levels_kernel<BS, 1><<<g.grid, dim3(BS), g.shmem, s>>>(t)));
        if (int rc = check_launch("calculate_cdf levels")) return rc;
    }
    // The coder's launches: all levels together where that is a call of few wavefronts, or where even
    // blocks with the longest table's LDS are all resident at once; else those levels together of whose tables a
    // compute unit holds equally many blocks (with the LDS of a 65-entry table the shorter ones would run at half
    // the wavefronts).
    const dim3 grid = stream_grid(a.sg, nblocks);
    const EncodeSource source = counted ? ENC_COUNTED : ENC_TABLES;
    const bool few = few_encode(nblocks * n, source, max_lp, kSlotTile, fused_scan);
    const bool together = few || nblocks * n <= (int64_t)compute_units() * resident_encode_blocks(max_lp);
    // the levels by launches: members[i], longest tables first
    int members[kMaxLevels][kMaxLevels], sizes[kMaxLevels], nlaunches = 0;
    for (int64_t resident = 1; resident <= 8; ++resident) {
        int count = 0;
        for (int v = n - 1; v >= 0; --v)
            if (together || resident_encode_blocks(o[v].max_bins + 1) == resident) members[nlaunches][count++] = v;
        if (!count) continue;
        sizes[nlaunches++] = count;
        if (together) break;
    }
    auto code = [&](int launch, hipStream_t on) {
        int lp = 0;
        for (int i = 0; i < sizes[launch]; ++i) {
            const int v = members[launch][i];
            const EncodeWorkspace wv = w.level(v);
            p.level[i] = {reinterpret_cast<uint16_t *>(o[v].cdf), reinterpret_cast<const uint32_t *>(wv.symbols), wv.scratch,
                          o[v].lengths, o[v].status, fused_scan ? wv.tile_sums : nullptr, grouped ? wv.group_sums : nullptr,
                          o[v].key_bins, o[v].value_bins, o[v].max_bins + 1};
            if (o[v].max_bins + 1 > lp) lp = o[v].max_bins + 1;
        }
        if (counted) return fused_scan ? launch_encode_levels<true, true>(p, sizes[launch], lp, grid, few, on)
                                       : launch_encode_levels<true, false>(p, sizes[launch], lp, grid, few, on);
        return fused_scan ? launch_encode_levels<false, true>(p, sizes[launch], lp, grid, few, on)
                          : launch_encode_levels<false, false>(p, sizes[launch], lp, grid, few, on);
    };
    const int64_t cblocks = ceil_div(w.nstreams, kCompactStreams);
    auto compact = [&](const int *levels, int count, hipStream_t on) {
        CompactLevelsArgs c;
        for (int i = 0; i < count; ++i) {
            const EncodeWorkspace wv = w.level(levels[i]);
            if (int rc = scan_for_compaction(o[levels[i]], wv, fused_scan, grouped, wv.group_sums, c.level[i], on)) return rc;
        }
        const dim3 cgrid((unsigned)cblocks, (unsigned)count);
        if (cblocks * count <= sliced_compact_blocks()) {
            if (fused_scan) compact_levels_kernel<true, 4><<<cgrid, dim3(1024), 0, on>>>(c);
            else compact_levels_kernel<false, 4><<<cgrid, dim3(1024), 0, on>>>(c);
        } else {
            if (fused_scan) compact_levels_kernel<true, 1><<<cgrid, dim3(256), 0, on>>>(c);
            else compact_levels_kernel<false, 1><<<cgrid, dim3(256), 0, on>>>(c);
        }
        return check_launch("compact levels");
    };
    if (nlaunches > 1) {
        const SideStream side(s);
        if (side.ok()) {
            // the launch of the longest tables beside the other levels' coder and their compaction.  Their LDS (four blocks of
            // 65 entries are 135 of 160 KB) leaves half of a compute unit's wavefront slots empty, but room for one block
            // more with the LDS of 33 entries: on large caches the coders take as long as one behind the other (796 us
            // and 812), and what is won is the compaction of the shorter tables, which runs beside the longest
            // tables' coder.  Four levels, one behind the other / beside, us: 32 layers x 4096 tokens
            // x 1024 channels 1070 / 1049, x 1024 tokens 328 / 308, 512 channels 205 / 178, 400 channels 242 / 190; 4 layers x
            // 2048 tokens in chunks of 1500 162 / 135
            if (int rc = code(0, side.stream())) return rc;
            if (int rc = compact(members[0], sizes[0], side.stream())) return rc;
            for (int i = 1; i < nlaunches; ++i) {
                if (int rc = code(i, s)) return rc;
                if (int rc = compact(members[i], sizes[i], s)) return rc;
            }
            return CG_OK;
        }
    }
    for (int i = nlaunches - 1; i >= 0; --i)
        if (int rc = code(i, s)) return rc;
    int all[kMaxLevels];
    for (int v = 0; v < n; ++v) all[v] = v;
    return compact(all, n, s);
}

int check_kv_geometry(const char *what, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t chunk_tokens)
{
    if (int rc = check_dt(kv_dt, what)) return rc;
    if (L <= 0 || T <= 0 || H <= 0 || D <= 0) return fail(CG_ERR_ARG, "%s: empty input", what);
    if (chunk_tokens <= 0) return fail(CG_ERR_ARG, "%s: chunk_tokens must be positive", what);
    if (chunk_tokens > 65535) return fail(CG_ERR_ARG, "%s: at most 65535 tokens per chunk (16-bit counters)", what);
    // refused here, before the first launch of the call has written anything
    return check_grid_limits(2 * L, cg_num_subchunks(T, chunk_tokens));
}

// cg_encode_kv.  `flags` (CG_TEST_*, 0 from cg_encode_kv) switch the internal choices that have
// two forms to the form the call would not take by itself; the results are the same.
int encode_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl,
              int64_t skv, int64_t st, int64_t sh, const float *key_bins, const float *value_bins,
              int max_bins, int64_t chunk_tokens, int delta_group, int16_t *cdf, void *maxima,
              int32_t *lengths, int64_t *offsets, uint8_t *payload, int64_t payload_cap,
              int32_t *status, void *workspace, size_t workspace_bytes, void *stream, int flags)
{
    const bool four_bit_words = !(flags & CG_TEST_BYTE_SYMBOLS), may_be_few = !(flags & CG_TEST_MANY_WAVEFRONTS);
    if (!kv || !key_bins || !value_bins || !cdf || !maxima || !lengths || !offsets || !payload || !status || !workspace)
        return fail(CG_ERR_ARG, "encode_kv: null pointer");
    if (int rc = check_kv_geometry("encode_kv", kv_dt, L, T, H, D, chunk_tokens)) return rc;
    if (int rc = check_lp(max_bins + 1, "encode_kv")) return rc;
    if (delta_group < 0 || delta_group > kSub) return fail(CG_ERR_ARG, "encode_kv: delta_group must be in [0, %d]", kSub);
    const int64_t C = H * D;
    const EncodeWorkspace w(workspace, L, T, C, chunk_tokens, 1);
    if (workspace_bytes < w.total) return fail(CG_ERR_WORKSPACE, "encode_kv: workspace too small");
    if (!aligned_to(workspace, 256)) return fail(CG_ERR_ARG, "encode_kv: workspace must be 256-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const LevelOut o = {key_bins, value_bins, max_bins, cdf, lengths, offsets, payload, payload_cap, status};

    const bool packed = kv_vectorizable(kv, D, C, sl, skv, st, sh) && C % 8 == 0;
    if (delta_group > 0 && !packed)
        return fail(CG_ERR_ARG, "encode_kv: delta groups need head sizes and strides that are multiples of 8 and a 16-byte aligned tensor");
    if (packed) {
        uint32_t *sym4 = reinterpret_cast<uint32_t *>(w.symbols);
        const bool nibbles = four_bit_words && delta_group == 0;
        // The quantizer counts the symbols as it makes them and writes the tables, where the
        // tables fit its LDS and there are chunks enough to fill the GPU; the coder then only codes.
        QuantTablesShape shape;
        const int64_t nchunks = cg_num_chunks(T, chunk_tokens);
        const int64_t reach = chunk_tokens < T ? chunk_tokens : T;       // tokens of the longest chunk
        // Few (row, chunk) pairs but long chunks (one table over a whole context): the chunks are
        // cut into parts of whole sub-chunks, a block each, whose counters are summed in memory
        // (in the stream slots of the workspace, which nothing uses before the coder runs).
        int64_t part_tokens = 0;
        if ((flags & CG_TEST_SPLIT_CHUNKS) && reach > kSub) part_tokens = kSub;
        else if (2 * L * nchunks < kQuantTablesPartBlocks && reach > kSub) {
            const int64_t want = ceil_div(kQuantTablesPartBlocks, 2 * L * nchunks);     // parts per chunk
            part_tokens = reach / want / kSub * kSub;
            if (part_tokens < kSub) part_tokens = kSub;
        }
        const int64_t nparts = part_tokens ? ceil_div(reach, part_tokens) : 1;
        const bool enough_blocks = (flags & CG_TEST_TABLES_IN_QUANTIZER) || 2 * L * nchunks * nparts >= kQuantTablesMinBlocks;
        // the table builder addresses a chunk's token rows with a 32-bit offset from the chunk's first
        const bool addressable = st >= 0 && sh >= 0 && ((H - 1) * sh + (D - 1) + (reach - 1) * st) * 2 + 16 <= 0xFFFFFFF0ll;
        if (delta_group == 0 && !(flags & CG_TEST_TABLES_IN_CODER) && enough_blocks && addressable &&
            quantize_tables_shape(C / 8, max_bins + 1, sh == D, shape)) {
            const size_t slots_bytes = (size_t)w.ntiles * kSlotTile * kStreamCap;
            if (nparts > 1 && (size_t)nchunks * 2 * L * shape.lds > slots_bytes) part_tokens = 0;       // one block per chunk after all
            if (int rc = launch_quantize_tables(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, sym4, maxima,
                                                reinterpret_cast<uint16_t *>(cdf), w.nsub, chunk_tokens, nibbles, status, shape, s,
                                                nparts > 1 ? part_tokens : 0, nparts > 1 && part_tokens ? w.scratch : nullptr, slots_bytes,
                                                w.group_sums)) return rc;
            return code_and_compact(o, sym4, nullptr, w, L, T, C, chunk_tokens, s, maxima, kv_dt, nibbles, true, w.group_sums, may_be_few);
        }
        int32_t *const group_sums = w.ntiles > kDirectTiles ? w.group_sums : nullptr;
        if (int rc = launch_quantize_pack(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, sym4,
                                          maxima, w.nsub, chunk_tokens, delta_group, s, status, 0, nullptr, nullptr, 0,
                                          nibbles, nullptr, max_bins + 1, group_sums)) return rc;
        return code_and_compact(o, sym4, nullptr, w, L, T, C, chunk_tokens, s, maxima, kv_dt, nibbles, false, group_sums, may_be_few);
    }
    clear_status_kernel<<<1, 1, 0, s>>>(status);
    if (int rc = launch_quantize(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, w.symbols, maxima, s)) return rc;
    return code_and_compact(o, nullptr, w.symbols, w, L, T, C, chunk_tokens, s);
}

}  // namespace

extern "C" {

int cg_encode_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl,
                 int64_t skv, int64_t st, int64_t sh, const float *key_bins, const float *value_bins,
                 int max_bins, int64_t chunk_tokens, int delta_group, int16_t *cdf, void *maxima,
                 int32_t *lengths, int64_t *offsets, uint8_t *payload, int64_t payload_cap,
                 int32_t *status, void *workspace, size_t workspace_bytes, void *stream)
{
    return encode_kv(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, max_bins, chunk_tokens, delta_group,
                     cdf, maxima, lengths, offsets, payload, payload_cap, status, workspace, workspace_bytes, stream, 0);
}

int cg_test_encode_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl,
                      int64_t skv, int64_t st, int64_t sh, const float *key_bins, const float *value_bins,
                      int max_bins, int64_t chunk_tokens, int delta_group, int16_t *cdf, void *maxima,
                      int32_t *lengths, int64_t *offsets, uint8_t *payload, int64_t payload_cap,
                      int32_t *status, void *workspace, size_t workspace_bytes, void *stream, int flags)
{
    return encode_kv(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins, value_bins, max_bins, chunk_tokens, delta_group,
                     cdf, maxima, lengths, offsets, payload, payload_cap, status, workspace, workspace_bytes, stream, flags);
}

int cg_test_few_encode_blocks(int source, int lp, int block, int tile)
{
    if (source < ENC_BYTES || source > ENC_QUANTIZER_TABLES || lp < 2 || lp > CG_MAX_LP || (block != 64 && block != 128 && block != 256)) return -1;
    return (int)few_encode_blocks(static_cast<EncodeSource>(source), lp, block, tile != 0);
}

int cg_encode_kv_levels_together(const void *kv, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl, int64_t skv, int64_t st, int64_t sh,
                                 int nlevels, const int *max_bins, int64_t chunk_tokens)
{
    if (!max_bins || nlevels < 1 || nlevels > CG_MAX_LEVELS || chunk_tokens <= 0) return 0;
    const int64_t C = H * D;
    return kv_vectorizable(kv, D, C, sl, skv, st, sh) && C % 8 == 0 && level_areas(L, T, C, chunk_tokens, nlevels) > 1 &&
           levels_alike(max_bins, nlevels, cg_num_subchunks(T, chunk_tokens), C);
}

int cg_encode_kv_levels(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D, int64_t sl,
                        int64_t skv, int64_t st, int64_t sh, int nlevels, const float *const *key_bins,
                        const float *const *value_bins, const int *max_bins, int64_t chunk_tokens,
                        int16_t *const *cdf, void *maxima, int32_t *const *lengths, int64_t *const *offsets,
                        uint8_t *const *payload, const int64_t *payload_cap, int32_t *status,
                        void *workspace, size_t workspace_bytes, void *stream)
{
    if (!kv || !key_bins || !value_bins || !max_bins || !cdf || !maxima || !lengths || !offsets || !payload ||
        !payload_cap || !status || !workspace)
        return fail(CG_ERR_ARG, "encode_kv_levels: null pointer");
    if (nlevels < 1 || nlevels > CG_MAX_LEVELS)
        return fail(CG_ERR_ARG, "encode_kv_levels: between 1 and %d levels, got %d", CG_MAX_LEVELS, nlevels);
    if (int rc = check_kv_geometry("encode_kv_levels", kv_dt, L, T, H, D, chunk_tokens)) return rc;
    int lp_lv[CG_MAX_LEVELS];
    LevelOut outs[CG_MAX_LEVELS];
    for (int v = 0; v < nlevels; ++v) {
        if (!key_bins[v] || !value_bins[v] || !cdf[v] || !lengths[v] || !offsets[v] || !payload[v])
            return fail(CG_ERR_ARG, "encode_kv_levels: null pointer for level %d", v);
        if (int rc = check_lp(max_bins[v] + 1, "encode_kv_levels")) return rc;
        lp_lv[v] = max_bins[v] + 1;
        outs[v] = {key_bins[v], value_bins[v], max_bins[v], cdf[v], lengths[v], offsets[v], payload[v], payload_cap[v], status + v};
    }
    const int64_t C = H * D;
    int areas = level_areas(L, T, C, chunk_tokens, nlevels);
    if (workspace_bytes < EncodeWorkspace(nullptr, L, T, C, chunk_tokens, nlevels, areas).total) areas = 1;
    const EncodeWorkspace w(workspace, L, T, C, chunk_tokens, nlevels, areas);
    if (workspace_bytes < w.total) return fail(CG_ERR_WORKSPACE, "encode_kv_levels: workspace too small");
    if (!aligned_to(workspace, 256)) return fail(CG_ERR_ARG, "encode_kv_levels: workspace must be 256-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);

    const bool packed = kv_vectorizable(kv, D, C, sl, skv, st, sh) && C % 8 == 0;
    if (packed) {
        // one pass over the tensor: every row is loaded once, its maximum found once, and its
        // symbols written once per level
        int32_t *const group_sums = w.ntiles > kDirectTiles ? w.group_sums : nullptr;
        if (int rc = launch_quantize_pack(kv, kv_dt, L, T, H, D, sl, skv, st, sh, nullptr, nullptr, reinterpret_cast<uint32_t *>(w.symbols),
                                          maxima, w.nsub, chunk_tokens, 0, s, status, nlevels, key_bins, value_bins,
                                          (int64_t)(w.symbols_bytes / 4), true, lp_lv, 0, group_sums)) return rc;
        return code_and_compact_levels(outs, nlevels, w, L, T, C, chunk_tokens, s, maxima, kv_dt, group_sums != nullptr);
    }
    // shapes the vector loads cannot take: one plain quantization pass per level
    for (int v = 0; v < nlevels; ++v) {
        const EncodeWorkspace wv = w.level(v);
        clear_status_kernel<<<1, 1, 0, s>>>(status + v);
        if (int rc = launch_quantize(kv, kv_dt, L, T, H, D, sl, skv, st, sh, key_bins[v], value_bins[v], wv.symbols, maxima, s)) return rc;
        if (int rc = code_and_compact(outs[v], nullptr, wv.symbols, wv, L, T, C, chunk_tokens, s)) return rc;
    }
    return CG_OK;
}

int cg_decode_kv(const int16_t *cdf, int max_bins, const void *maxima, int max_dt, const int64_t *offsets,
                 const uint8_t *payload, int64_t payload_bytes, const float *key_bins,
                 const float *value_bins, int64_t L, int64_t T, int64_t H, int64_t D,
                 int64_t chunk_tokens, int delta_group, void *out, int out_dt, int64_t ol, int64_t okv,
                 int64_t ot, int64_t oh, void *stream)
{
    if (!cdf || !maxima || !offsets || !key_bins || !value_bins || !out || !payload)
        return fail(CG_ERR_ARG, "decode_kv: null pointer");
    if (int rc = check_dt(max_dt, "decode_kv")) return rc;
    if (L <= 0 || T <= 0 || H <= 0 || D <= 0 || chunk_tokens <= 0) return fail(CG_ERR_ARG, "decode_kv: empty input");
    if (int rc = check_lp(max_bins + 1, "decode_kv")) return rc;
    if (delta_group < 0 || delta_group > kSub) return fail(CG_ERR_ARG, "decode_kv: delta_group must be in [0, %d]", kSub);
    const int64_t C = H * D, rows = 2 * L;
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    if (int rc = set_output(a, "decode_kv", out, out_dt, H, D, ol, okv, ot, oh)) return rc;
    a.cdf = reinterpret_cast<const uint16_t *>(cdf);
    a.lp = max_bins + 1;
    if (int rc = set_byte_window(a, payload, payload_bytes, "decode_kv")) return rc;
    a.offsets = offsets;
    a.L = L;
    a.maxima = static_cast<const uint16_t *>(maxima);
    a.max_dt = max_dt;
    a.delta_group = delta_group;
    a.key_bins = key_bins;
    a.value_bins = value_bins;
    const bool few = few_wavefronts(rows, C, cg_num_subchunks(T, chunk_tokens), a.lp);
    const int block = few ? 64 : decode_kv_block(C, a.lp);
    int64_t nblocks;
    if (int rc = make_grid(rows, C, T, chunk_tokens, cg_num_subchunks(T, chunk_tokens), block, a.sg, nblocks)) return rc;
    return launch_decode_kv<SRC_OFFSETS>(a, nblocks, block, few, out_dt, static_cast<hipStream_t>(stream));
}

int cg_decode_listed(const CgListedSub *subs, int64_t nsub, int max_bins, int64_t L, int64_t H, int64_t D,
                     int delta_group, void *out, int out_dt, int64_t ol, int64_t okv, int64_t ot, int64_t oh, void *stream)
{
    if (!subs || !out) return fail(CG_ERR_ARG, "decode_listed: null pointer");
    if (L <= 0 || H <= 0 || D <= 0 || nsub <= 0) return fail(CG_ERR_ARG, "decode_listed: empty input");
    if (int rc = check_lp(max_bins + 1, "decode_listed")) return rc;
    if (delta_group < 0 || delta_group > kSub) return fail(CG_ERR_ARG, "decode_listed: delta_group must be in [0, %d]", kSub);
    const int64_t C = H * D, rows = 2 * L;
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    if (int rc = set_output(a, "decode_listed", out, out_dt, H, D, ol, okv, ot, oh)) return rc;
    a.lp = max_bins + 1;
    a.L = L;
    a.delta_group = delta_group;
    a.listed = subs;
    const bool few = few_wavefronts(rows, C, nsub, a.lp);
    const int block = few ? 64 : decode_kv_block(C, a.lp);
    int64_t nblocks;
    // the entries hold the token geometry; the grid only needs its size
    if (int rc = make_grid(rows, C, nsub, 1, nsub, block, a.sg, nblocks)) return rc;
    return launch_decode_kv<SRC_LISTED>(a, nblocks, block, few, out_dt, static_cast<hipStream_t>(stream));
}

int cg_host_tile_starts(const void *lengths, int itemsize, int64_t nsub, int64_t rows, int64_t C,
                        uint32_t *tile_starts, int64_t *sub_bytes)
{
    if (!lengths || !tile_starts || !sub_bytes) return fail(CG_ERR_ARG, "host_tile_starts: null pointer");
    if (nsub <= 0 || rows <= 0 || C <= 0 || rows > (1 << 24) / C || (itemsize != 2 && itemsize != 4))
        return fail(CG_ERR_ARG, "host_tile_starts: bad shape");
    const bool fine = itemsize == 2 ? host_tile_starts<uint16_t>(lengths, nsub, rows, C, kStreamCap, tile_starts, sub_bytes)
                                    : host_tile_starts<int32_t>(lengths, nsub, rows, C, kStreamCap, tile_starts, sub_bytes);
    return fine ? CG_OK : fail(CG_ERR_ARG, "host_tile_starts: negative length");
}

int cg_host_list(const CgHostContainer *items, int n, const void *const *lengths, const int64_t *array_subs,
                 int64_t L, int64_t C, uint32_t *tile_starts, int64_t starts_at, CgListedSub *subs, int *bad)
{
    if (!items || !lengths || !array_subs || !tile_starts || !subs || !bad) return fail(CG_ERR_ARG, "host_list: null pointer");
    if (n <= 0 || L <= 0 || C <= 0 || 2 * L > (1 << 24) / C) return fail(CG_ERR_ARG, "host_list: bad shape");
    const int64_t rows = 2 * L, tiles = ceil_div(C, 64);
    int64_t sum;
    for (int i = 0; i < n; ++i) {
        const CgHostContainer &c = items[i];
        *bad = i;
        if (c.tokens <= 0 || c.chunk_tokens <= 0 || c.payload_bytes <= 0) return fail(CG_ERR_ARG, "host_list: empty container");
        const int64_t nsub = cg_num_subchunks(c.tokens, c.chunk_tokens), nsc = ceil_div(c.chunk_tokens, kSub);
        const int64_t skew = c.payload & 3;
        int64_t first = skew, g = 0;
        for (int k = 0; k < c.narrays; ++k, ++lengths, ++array_subs) {
            const int size = c.lengths_u16 ? 2 : 4;
            const char *p = static_cast<const char *>(*lengths);
            for (int64_t j = 0; j < *array_subs; ++j, ++g, ++subs, p += rows * C * size, tile_starts += rows * tiles, starts_at += rows * tiles * 4) {
                if (g >= nsub) return fail(CG_ERR_ARG, "host_list: more lengths than sub-chunks");
                if (int rc = cg_host_tile_starts(p, size, 1, rows, C, tile_starts, &sum)) return rc;
                const int64_t chunk = g / nsc, t0 = chunk * c.chunk_tokens + (g - chunk * nsc) * kSub;
                int64_t end = (chunk + 1) * c.chunk_tokens;
                if (end > c.tokens) end = c.tokens;
                subs->cdf = reinterpret_cast<const int16_t *>(c.tables + chunk * rows * C * (c.max_bins + 1) * 2);
                subs->maxima = reinterpret_cast<const void *>(c.maxima + t0 * 2);
                subs->lengths = reinterpret_cast<const void *>(c.lengths + g * rows * C * size);
                subs->bytes = reinterpret_cast<const uint8_t *>(c.payload - skew);
                subs->last_word = (skew + c.payload_bytes - 1) & ~3ll;
                subs->first = first;
                subs->tile_starts = reinterpret_cast<const uint32_t *>(starts_at);
                subs->key_bins = reinterpret_cast<const float *>(c.key_bins);
                subs->value_bins = reinterpret_cast<const float *>(c.value_bins);
                subs->t_out = c.t_out + t0;
                subs->n = (int32_t)(end - t0 < kSub ? end - t0 : kSub);
                subs->maxima_pitch = (int32_t)c.tokens;
                subs->max_dt = c.max_dt;
                subs->lengths_u16 = c.lengths_u16;
                first += sum;
            }
        }
        if (g != nsub || first - skew != c.payload_bytes)
            return fail(CG_ERR_ARG, "host_list: lengths do not add up to the payload");
    }
    return CG_OK;
}

void *cg_watch_new(int32_t *mark)
{
    int device = 0;
    if (!mark || hipGetDevice(&device) != hipSuccess) return nullptr;
    return new (std::nothrow) Watch(mark, device);
}

void cg_watch_free(void *watch) { delete static_cast<Watch *>(watch); }

int cg_watch_add(void *watch, int32_t value, void *stream)
{
    if (!watch) return fail(CG_ERR_ARG, "watch_add: null pointer");
    return static_cast<Watch *>(watch)->add(value, static_cast<hipStream_t>(stream));
}

int cg_watch_wait(void *watch, int32_t value)
{
    if (!watch) return fail(CG_ERR_ARG, "watch_wait: null pointer");
    return static_cast<Watch *>(watch)->wait(value);
}

int cg_move_bytes(const void *src, void *dst, int64_t n, int to_host, void *watch, int32_t value, void *stream)
{
    if (!src || !dst || n <= 0) return fail(CG_ERR_ARG, "move_bytes: null pointer or nothing to move");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = move_bytes(src, dst, n, to_host != 0, s)) return rc;
    return watch ? static_cast<Watch *>(watch)->add(value, s) : CG_OK;
}

int cg_mark(int32_t *mark, int32_t value, void *stream)
{
    if (!mark || !aligned_to(mark, 4)) return fail(CG_ERR_ARG, "mark: null or misaligned pointer");
    mark_kernel<<<1, 1, 0, static_cast<hipStream_t>(stream)>>>(mark, value);
    return check_launch("mark");
}

int cg_wait_mark(const int32_t *mark, int32_t value, void *stream)
{
    if (!mark || !aligned_to(mark, 4)) return fail(CG_ERR_ARG, "wait_mark: null or misaligned pointer");
    return wait_for_mark(mark, value, static_cast<hipStream_t>(stream));
}

// Pinned words of one reader at a time: eight 64-bit numbers, of which the last holds the mark.
static int32_t *words_mark(void *words) { return reinterpret_cast<int32_t *>(static_cast<int64_t *>(words) + 7); }

int cg_read_words(const void *const *at, const int32_t *bytes, int n, void *words, int32_t value, void *stream)
{
    if (!at || !bytes || !words || n < 1 || n > 4) return fail(CG_ERR_ARG, "read_words: between 1 and 4 words");
    WordsArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < n; ++i) {
        if (!at[i] || (bytes[i] != 4 && bytes[i] != 8) || !aligned_to(at[i], (size_t)bytes[i])) return fail(CG_ERR_ARG, "read_words: bad word");
        a.at[i] = at[i];
        a.bytes[i] = bytes[i];
    }
    a.n = n;
    a.out = static_cast<int64_t *>(words);
    a.mark = words_mark(words);
    a.value = value;
    read_words_kernel<<<1, 1, 0, static_cast<hipStream_t>(stream)>>>(a);
    if (int rc = check_launch("read_words")) return rc;
    return wait_for_mark(a.mark, value, static_cast<hipStream_t>(stream));
}

int cg_largest(const float *a, const float *b, int64_t n, void *words, int32_t value, void *stream)
{
    if (!a || !b || !words || n < 1) return fail(CG_ERR_ARG, "largest: null pointer or no values");
    largest_kernel<<<1, 64, 0, static_cast<hipStream_t>(stream)>>>(a, b, n, static_cast<float *>(words), words_mark(words), value);
    if (int rc = check_launch("largest")) return rc;
    return wait_for_mark(words_mark(words), value, static_cast<hipStream_t>(stream));
}

int cg_scan_collect(const int32_t *lengths, int64_t n, int64_t *offsets, void *scratch, size_t scratch_bytes, int64_t nslots, int64_t cap,
                    void *words, int32_t value, void *stream)
{
    if (!words) return fail(CG_ERR_ARG, "scan_collect: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    int64_t *const out = static_cast<int64_t *>(words);
    if (lengths && offsets && n > 0 && n <= kScanSmallMax && nslots > 0 && cap > 0) {
        scan_collect_kernel<<<1, kScanSmallThreads, 0, s>>>(lengths, (int32_t)n, offsets, nslots, cap, out, words_mark(words), value);
        return check_launch("scan_collect");
    }
    out[0] = out[1] = 0;
    if (int rc = cg_scan_lengths(lengths, n, offsets, scratch, scratch_bytes, stream)) return rc;
    if (int rc = cg_collect_sizes(offsets, n, nslots, cap, out, stream)) return rc;
    return cg_mark(words_mark(words), value, stream);
}

int cg_decode_fast_lengths(const int16_t *cdf, int lp, const uint8_t *bytes, int64_t nbytes, const int32_t *lengths, int64_t nl, int64_t nt,
                           int64_t nc, uint8_t *out, int64_t o0, int64_t o1, int64_t o2, int64_t *offsets, void *scratch, size_t scratch_bytes,
                           void *stream)
{
    if (nl <= 0 || nc <= 0) return fail(CG_ERR_ARG, "decode: empty input");
    if (int rc = cg_scan_lengths(lengths, nl * nc, offsets, scratch, scratch_bytes, stream)) return rc;
    return cg_decode_fast_prefsum(cdf, lp, bytes, nbytes, offsets + 1, nl, nt, nc, out, o0, o1, o2, stream);
}

int cg_host_fill(const CgHostPart *parts, int n, const int32_t *mark, const CgHostTeam *team, void *watch)
{
    if (!parts || n <= 0 || !mark) return fail(CG_ERR_ARG, "host_fill: null pointer or nothing to copy");
    try {
        HostJob job;
        job.mark = mark;
        job.nthreads = host_threads(team);
        for (int i = 0; i < n; ++i) {
            const CgHostPart &p = parts[i];
            if (p.bytes < 0 || (p.bytes && (!p.dst || !p.src))) return fail(CG_ERR_ARG, "host_fill: bad part");
            add_blocks(job, reinterpret_cast<uint8_t *>(p.dst), reinterpret_cast<const uint8_t *>(p.src), p.bytes, (uintptr_t)p.dst, p.value, 0);
        }
        seal(job, 1);
        int32_t last = INT_MIN;
        for (const HostBlock &b : job.blocks) last = std::max(last, b.value);
        int rc = CG_OK;
        const std::function<void()> idle = [&] {
            if (!rc && watch && (rc = static_cast<Watch *>(watch)->look(last))) job.stop.store(true);
        };
        run_job(job, team, &idle);
        return rc;
    } catch (const std::exception &e) {
        return fail(CG_ERR_ARG, "host_fill: %s", e.what());
    }
}

int cg_host_stage(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, void *area, int64_t bytes, void *watch,
                  int32_t value, const CgHostTeam *team, int *moves, void *stream)
{
    if (moves) *moves = 0;
    if (const char *what = stage_fault(parts, n, slots, nslots, step, area, bytes, moves)) return fail(CG_ERR_ARG, "host_stage: %s", what);
    try {
        hipStream_t s = static_cast<hipStream_t>(stream);
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess) return fail(CG_ERR_LAUNCH, "host_stage: no device");
        // a place behind each move whose slot is used again (the copy engine stops for 4 us at each)
        int32_t through = 0;
        Watch steps(&through, device);
        int32_t launched = 0;
        const int rc = stage_job(parts, n, slots, nslots, step, bytes, team, moves,
                                 [&](const uint8_t *from, int64_t at, int64_t size) {
                                     const int bad = move_bytes(from, static_cast<uint8_t *>(area) + at, size, false, s);
                                     if (bad) return bad;
                                     ++launched;
                                     return at + nslots * step < bytes ? steps.add(launched, s) : CG_OK;
                                 },
                                 [&] {
                                     const int bad = steps.look(through);
                                     return bad ? bad : through;
                                 });
        *moves = launched;
        if (rc || !watch) return rc;
        return static_cast<Watch *>(watch)->add(value, s);
    } catch (const std::exception &e) {
        return fail(CG_ERR_ARG, "host_stage: %s", e.what());
    }
}

int cg_test_host_stage(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, void *area, int64_t bytes,
                       const CgHostTeam *team, int *moves)
{
    if (moves) *moves = 0;
    if (const char *what = stage_fault(parts, n, slots, nslots, step, area, bytes, moves)) return fail(CG_ERR_ARG, "host_stage: %s", what);
    try {
        // a move reads its slot as late as it may: when the one behind it is launched
        struct { const uint8_t *from; uint8_t *to; int64_t size; } last = {nullptr, nullptr, 0};
        int32_t through = 0;
        const int rc = stage_job(parts, n, slots, nslots, step, bytes, team, moves,
                                 [&](const uint8_t *from, int64_t at, int64_t size) {
                                     if (last.size) {
                                         memcpy(last.to, last.from, (size_t)last.size);
                                         ++through;
                                     }
                                     last = {from, static_cast<uint8_t *>(area) + at, size};
                                     return 0;
                                 },
                                 [&] { return through; });
        if (last.size) memcpy(last.to, last.from, (size_t)last.size);
        return rc;
    } catch (const std::exception &e) {
        return fail(CG_ERR_ARG, "host_stage: %s", e.what());
    }
}

int cg_tables_to_counts(const int16_t *cdf, int max_bins, int64_t ngroups, int64_t C, const int32_t *tokens,
                        uint8_t *counts, int32_t *nsym, int32_t *inexact, void *stream)
{
    if (!cdf || !tokens || !counts || !nsym || !inexact) return fail(CG_ERR_ARG, "tables_to_counts: null pointer");
    if (int rc = check_lp(max_bins + 1, "tables_to_counts")) return rc;
    if (ngroups <= 0 || C <= 0 || ngroups > 65535) return fail(CG_ERR_ARG, "tables_to_counts: bad group or channel count");
    hipStream_t s = static_cast<hipStream_t>(stream);
    clear_ints_kernel<<<dim3((unsigned)ceil_div(ngroups, kWireThreads)), dim3(kWireThreads), 0, s>>>(nsym, ngroups, inexact);
    const dim3 grid((unsigned)ceil_div(C, kTableChannels), (unsigned)ngroups);
    tables_to_counts_kernel<<<grid, dim3(kTableChannels), 0, s>>>(reinterpret_cast<const uint16_t *>(cdf), max_bins + 1, C,
                                                               tokens, counts, nsym, inexact);
    return check_launch("tables_to_counts");
}

int cg_pack_counts(const uint8_t *counts, int max_bins, int64_t ngroups, int64_t C, const int32_t *nsym,
                   const int64_t *starts, uint8_t *out, void *stream)
{
    if (!counts || !nsym || !out) return fail(CG_ERR_ARG, "pack_counts: null pointer");
    if (int rc = check_lp(max_bins + 1, "pack_counts")) return rc;
    if (ngroups <= 0 || C <= 0 || ngroups > 65535) return fail(CG_ERR_ARG, "pack_counts: bad group or channel count");
    const dim3 grid((unsigned)ceil_div(C, kTableChannels), (unsigned)ngroups);
    pack_counts_kernel<<<grid, dim3(kTableChannels), 0, static_cast<hipStream_t>(stream)>>>(counts, max_bins + 1, C, nsym,
                                                                                         starts, out);
    return check_launch("pack_counts");
}

int cg_wire_meta(const int32_t *status, const int64_t *offsets, int64_t per_sub, int64_t nbounds, const int32_t *wide,
                 const int32_t *inexact, const int32_t *nsym, int64_t ngroups, int64_t *out, void *stream)
{
    if (!status || !offsets || !out || (ngroups > 0 && !nsym)) return fail(CG_ERR_ARG, "wire_meta: null pointer");
    if (per_sub <= 0 || nbounds <= 0 || ngroups < 0) return fail(CG_ERR_ARG, "wire_meta: bad count");
    wire_meta_kernel<<<dim3(1), dim3(kWireThreads), 0, static_cast<hipStream_t>(stream)>>>(status, offsets, per_sub, nbounds, wide,
                                                                                           inexact, nsym, ngroups, out);
    return check_launch("wire_meta");
}

int cg_lengths_to_u16(const int32_t *lengths, int64_t n, uint16_t *out, int32_t *wide, void *stream)
{
    if (!lengths || !out || !wide) return fail(CG_ERR_ARG, "lengths_to_u16: null pointer");
    const int64_t nblocks = ceil_div(n, kWireThreads);
    if (n <= 0 || nblocks > INT_MAX) return fail(CG_ERR_ARG, "lengths_to_u16: bad count");
    hipStream_t s = static_cast<hipStream_t>(stream);
    clear_ints_kernel<<<dim3(1), dim3(kWireThreads), 0, s>>>(wide, 1, nullptr);
    lengths_to_u16_kernel<<<dim3((unsigned)nblocks), dim3(kWireThreads), 0, s>>>(lengths, n, out, wide);
    return check_launch("lengths_to_u16");
}

int cg_counts_to_tables(const uint8_t *data, int64_t data_bytes, int max_bins, int64_t ngroups, int64_t C,
                        const int32_t *tokens, const uint8_t *nsym, const int64_t *starts, int16_t *cdf,
                        int32_t *invalid, void *stream)
{
    if (!invalid) return fail(CG_ERR_ARG, "counts_to_tables: null pointer");
    clear_ints_kernel<<<dim3(1), dim3(kWireThreads), 0, static_cast<hipStream_t>(stream)>>>(invalid, 1, nullptr);
    return cg_rebuild_tables(data, data_bytes, max_bins, ngroups, C, tokens, nsym, starts, cdf, invalid, stream);
}

int cg_rebuild_tables(const uint8_t *data, int64_t data_bytes, int max_bins, int64_t ngroups, int64_t C,
                      const int32_t *tokens, const uint8_t *nsym, const int64_t *starts, int16_t *cdf,
                      int32_t *invalid, void *stream)
{
    if (!data || !tokens || !nsym || !starts || !cdf || !invalid) return fail(CG_ERR_ARG, "counts_to_tables: null pointer");
    if (int rc = check_lp(max_bins + 1, "counts_to_tables")) return rc;
    if (ngroups <= 0 || C <= 0 || data_bytes < 0)
        return fail(CG_ERR_ARG, "counts_to_tables: bad group or channel count");
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int64_t g = 0; g < ngroups; g += 65535) {                   // a grid's limit in y
        const dim3 grid((unsigned)ceil_div(C, kTableChannels), (unsigned)(ngroups - g < 65535 ? ngroups - g : 65535));
        counts_to_tables_kernel<<<grid, dim3(kTableChannels), 0, s>>>(data, data_bytes, max_bins + 1, C, tokens + g, nsym + g, starts + g,
                                                                     reinterpret_cast<uint16_t *>(cdf) + g * C * (max_bins + 1), invalid);
        if (int rc = check_launch("counts_to_tables")) return rc;
    }
    return CG_OK;
}

}  // extern "C"
