/*
 * cachegen_hip.h -- C ABI of the MI355X (gfx950) CacheGen KV codec library.
 *
 * Plain pointers and sizes only; every pointer named "device" must be memory the
 * GPU can access, `stream` is a hipStream_t passed as void* (NULL = the null
 * stream).  All functions are asynchronous with respect to the host, keep no
 * state between calls and return CG_OK or a negative CG_ERR_* code;
 * cg_last_error() then holds a message for the calling thread.
 *
 * The encode and decode entry points launch one block per (channel tile, row,
 * sub-chunk of 256 tokens) on a three-dimensional grid: at most 65535 rows
 * (layers, or 2 x layers for the *_kv functions) and 65535 sub-chunks per call,
 * CG_ERR_ARG beyond.
 *
 * Paths in the comments are relative to LMCache/ in the reference tree:
 *   enc_new.cu = third_party/torchac_cuda/torchac_kernel_enc_new.cu
 *   dec_new.cu = third_party/torchac_cuda/torchac_kernel_dec_new.cu
 *   cal_cdf.cu = third_party/torchac_cuda/cal_cdf.cu
 *   main.cpp   = third_party/torchac_cuda/main.cpp
 *   encoder.py = lmcache/storage_backend/serde/cachegen_encoder.py
 *   decoder.py = lmcache/storage_backend/serde/cachegen_decoder.py
 */
#ifndef CACHEGEN_HIP_H
#define CACHEGEN_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define CG_OK 0
#define CG_ERR_ARG (-1)      /* bad shape, stride, dtype or limit */
#define CG_ERR_LAUNCH (-2)   /* the HIP runtime refused a launch */
#define CG_ERR_WORKSPACE (-3)/* workspace too small */

#define CG_DT_F16 0
#define CG_DT_BF16 1

#define CG_MAX_TOKENS_PER_STREAM 256 /* cachegen_basics.py:8, enc_new.cu:9-15 */
#define CG_MAX_LP 129                /* table length limit of this library (reference: 48 / 64) */
#define CG_MAX_LEVELS 8              /* quantization levels one cg_encode_kv_levels call takes */

/* Message for the last error returned on this thread ("" if none). */
const char *cg_last_error(void);
/* ABI version of the library: bumped when a signature changes. */
int cg_abi_version(void);

/* ---------------------------------------------------------------------------
 * The four entry points of the reference's extension module (main.cpp:14-17).
 * Strides are in elements.  Tables are int16 bit patterns of uint16 values.
 * ------------------------------------------------------------------------- */

/* torchac_cuda.calculate_cdf (cal_cdf.cu:68-129).
 * sym  device int8  [nl, nt, nc], strides (s0, s1, s2), values in [0, max_bins)
 * cdf  device int16 [nl, nc, max_bins + 1], contiguous, written
 * Counters are 16 bits wide as in the reference, so nt <= 65535 is required. */
int cg_calculate_cdf(const int8_t *sym, int64_t nl, int64_t nt, int64_t nc,
                     int64_t s0, int64_t s1, int64_t s2, int max_bins,
                     int16_t *cdf, void *stream);

/* torchac_cuda.encode_fast_new (enc_new.cu:355-451).
 * cdf      device int16 [nl, nc, lp] contiguous
 * sym      device int8  [nl, nt, nc], strides (s0, s1, s2), nt <= 256
 * out      device uint8 [nl, nc, cap], strides (o0, o1, 1); stream (l, c) is written
 *          to out[l, c, 0:length]; bytes past the length are left untouched
 * lengths  device int32 [nl, nc] contiguous, written.  A stream longer than `cap`
 *          is truncated to `cap` stored bytes while its full length is reported. */
int cg_encode_fast_new(const int16_t *cdf, int lp, const int8_t *sym,
                       int64_t nl, int64_t nt, int64_t nc,
                       int64_t s0, int64_t s1, int64_t s2,
                       uint8_t *out, int64_t cap, int64_t o0, int64_t o1,
                       int32_t *lengths, void *stream);

/* torchac_cuda.decode_fast_new (dec_new.cu:314-393): streams in a padded buffer.
 * padded   device uint8 [nl, nc, cap], strides (p0, p1, 1)
 * lengths  device int32 [nl, nc] contiguous (kept for the reference's signature: the
 *          decoder stops after nt symbols and does not need them)
 * out      device uint8 [nl, nt, nc], strides (o0, o1, o2), written */
int cg_decode_fast_new(const int16_t *cdf, int lp, const uint8_t *padded, int64_t cap,
                       int64_t p0, int64_t p1, const int32_t *lengths,
                       int64_t nl, int64_t nt, int64_t nc,
                       uint8_t *out, int64_t o0, int64_t o1, int64_t o2, void *stream);

/* torchac_cuda.decode_fast_prefsum (dec_new.cu:403-479): streams concatenated in
 * (layer, channel) order.
 * bytes    device uint8 [nbytes]; the decoder loads whole aligned 32-bit
 *          words, so up to 3 bytes on either side of the buffer (inside the same aligned
 *          words) are read but never used
 * prefix   device int64 [nl, nc] contiguous: INCLUSIVE running sum of the stream
 *          lengths (decoder.py:70); stream g = l*nc + c is bytes[prefix[g-1]:prefix[g]] */
int cg_decode_fast_prefsum(const int16_t *cdf, int lp, const uint8_t *bytes, int64_t nbytes,
                           const int64_t *prefix, int64_t nl, int64_t nt, int64_t nc,
                           uint8_t *out, int64_t o0, int64_t o1, int64_t o2, void *stream);

/* ---------------------------------------------------------------------------
 * Fused forms of the Python-side tensor code around those kernels.
 *
 * A KV cache is a 16-bit float tensor indexed (layer, k|v, token, head, dim) with
 * element strides (sl, skv, st, sh, 1): [L,2,T,H,D] ("vllm") and [L,2,H,T,D]
 * ("huggingface") are both expressible (encoder.py:341-342, decoder.py:169-173).
 * C = H*D channels; "2L" rows are the L key layers followed by the L value layers
 * (encoder.py:263).  Tokens are cut into chunks of `chunk_tokens` (one table per
 * chunk, layer and channel: one `to_bytes` call of the reference each) and every
 * chunk into sub-chunks of at most 256 tokens (encoder.py:279-292); sub-chunks
 * are numbered consecutively over the whole tensor (nsub of them).  A stream is
 * one (sub-chunk, row of 2L, channel), numbered in that order.
 * ------------------------------------------------------------------------- */

/* torch_quant_vectorized on K and V (encoder.py:42-59, 72-83, 258-263).
 * kv          device fp16/bf16 KV cache (kv_dt, strides above)
 * key_bins    device float32 [L], value_bins likewise (encoder.py:311-322)
 * sym         device uint8 [2L, T, C] contiguous, written
 * maxima      device 16-bit [2, L, T] contiguous in kv_dt, written: row maxima,
 *             maxima[0] = max_tensors_key, maxima[1] = max_tensors_value */
int cg_quantize_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                   int64_t sl, int64_t skv, int64_t st, int64_t sh,
                   const float *key_bins, const float *value_bins,
                   uint8_t *sym, void *maxima, void *stream);

/* Number of sub-chunks / chunks for T tokens cut every chunk_tokens. */
int64_t cg_num_chunks(int64_t T, int64_t chunk_tokens);
int64_t cg_num_subchunks(int64_t T, int64_t chunk_tokens);

/* Bytes of device workspace cg_encode_kv needs. */
size_t cg_encode_kv_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens);

/* encode_function for every chunk at once (encoder.py:247-301), including
 * collect_bytes (encoder.py:209-222).
 * cdf         device int16 [nchunks, 2L, C, max_bins+1], written
 * maxima      device 16-bit [2, L, T] in kv_dt, written
 * lengths     device int32 [nsub, 2L, C], written: bytes of every stream
 * offsets     device int64 [nsub*2L*C + 1], written: exclusive running sum of the
 *             lengths; offsets[last] = total payload bytes
 * payload     device uint8 [payload_cap], written: all streams back to back in
 *             stream order; the streams of sub-chunk g are
 *             payload[offsets[g*2L*C] : offsets[(g+1)*2L*C]] = that sub-chunk's
 *             `bytestream` tensor.  payload_cap >= 256 * number of streams is
 *             always enough.
 * status      device int32 [1], written: 0, or 1 if a stream exceeded 256 bytes
 *             (the reference overruns its buffer there; here the stream is cut).
 * workspace   device scratch of cg_encode_kv_workspace(...) bytes, 256-aligned
 * delta_group 0 for the reference's codec.  > 0 (no counterpart in the reference): inside
 *             every sub-chunk, tokens form groups of this many; the first row of a group
 *             (the anchor) is quantized as is, every other row as its float32 difference
 *             from the anchor row, with the row maximum of the differences rounded to the
 *             16-bit format; cg_decode_kv with the same value adds the reconstructed
 *             anchor back. */
int cg_encode_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                 int64_t sl, int64_t skv, int64_t st, int64_t sh,
                 const float *key_bins, const float *value_bins, int max_bins,
                 int64_t chunk_tokens, int delta_group,
                 int16_t *cdf, void *maxima, int32_t *lengths, int64_t *offsets,
                 uint8_t *payload, int64_t payload_cap, int32_t *status,
                 void *workspace, size_t workspace_bytes, void *stream);

/* Test hook: cg_encode_kv with the internal choices that have two forms switched by `flags` to
 * the form the call would not take by itself.  Same arguments and the same results as
 * cg_encode_kv, which is what the tests that call it check.  No counterpart in the reference.
 * CG_TEST_BYTE_SYMBOLS          every row's symbols cross from the quantizer to the coder a byte a
 *                               symbol (cg_encode_kv packs rows of at most 15 symbols four bits a symbol)
 * CG_TEST_TABLES_IN_QUANTIZER   the quantizer counts the symbols and writes the tables, however few
 *                               chunks the call has (cg_encode_kv does so from 512 (row, chunk) pairs on,
 *                               where the tables of all channels fit the LDS of one block; calls with
 *                               fewer pairs and chunks of more than 256 tokens cut the chunks into parts)
 * CG_TEST_SPLIT_CHUNKS          with the form above: every chunk of more than 256 tokens is counted in
 *                               parts of 256 tokens by separate blocks, whose counters are summed in memory
 * CG_TEST_TABLES_IN_CODER       never: the coder (one table per sub-chunk) or a separate pass over
 *                               the symbols (longer chunks) builds the tables
 * CG_TEST_MANY_WAVEFRONTS       the coder's form for calls of many wavefronts, however few there are
 */
#define CG_TEST_BYTE_SYMBOLS 1
#define CG_TEST_TABLES_IN_QUANTIZER 2
#define CG_TEST_TABLES_IN_CODER 4
#define CG_TEST_SPLIT_CHUNKS 8
#define CG_TEST_MANY_WAVEFRONTS 16
int cg_test_encode_kv(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                      int64_t sl, int64_t skv, int64_t st, int64_t sh,
                      const float *key_bins, const float *value_bins, int max_bins,
                      int64_t chunk_tokens, int delta_group,
                      int16_t *cdf, void *maxima, int32_t *lengths, int64_t *offsets,
                      uint8_t *payload, int64_t payload_cap, int32_t *status,
                      void *workspace, size_t workspace_bytes, void *stream, int flags);

/* Test hook, no GPU work: blocks of `block` (64, 128 or 256) lanes a compute unit up to which an encode with
 * tables of lp entries takes the coder's form for few wavefronts; -1 for arguments out of range.
 * source: 0 byte symbols, 1 packed symbols with tables made by the coder, 2 by a pass of their own, 3 by
 * the quantizer.  tile: the channels are a multiple of 256 and a block is 256 lanes. */
int cg_test_few_encode_blocks(int source, int lp, int block, int tile);

/* The same KV cache encoded at `nlevels` quantization levels from ONE read of the tensor: the
 * adaptive-streaming use of the reference, which pre-encodes every chunk at QUANT_LEVEL 1..3
 * by calling the serializer once per level (run_adaptation.py:63-72, src/utils.py:357-377).
 * Every row is loaded once and its maximum found once; its symbols are written once per level
 * and each level is then coded exactly as cg_encode_kv codes it, so level v's tables, lengths,
 * offsets and payload are byte-identical to a cg_encode_kv call with key_bins[v],
 * value_bins[v], max_bins[v].
 * key_bins, value_bins   HOST arrays of nlevels device pointers (float32 [L] each)
 * max_bins               HOST array of nlevels ints
 * cdf, lengths, offsets, payload   HOST arrays of nlevels device pointers, shaped as in
 *                        cg_encode_kv (cdf[v]: [nchunks, 2L, C, max_bins[v]+1]); payload_cap
 *                        a HOST array of nlevels capacities
 * maxima                 device 16-bit [2, L, T]: the row maxima do not depend on the level
 * status                 device int32 [nlevels]
 * workspace              cg_encode_kv_levels_workspace(...) bytes, 256-aligned: symbols for every level and, up to
 *                        16384 tiles of 256 streams a level, stream scratch for every level, so that levels can share
 *                        launches; with less, down to cg_encode_kv_levels_least_workspace(...), whose levels share one
 *                        scratch, they are coded one behind the other.  32 layers x 4096 tokens x 1024 channels, four
 *                        levels: 2.15 GB and 1.35 GB
 * 1 <= nlevels <= CG_MAX_LEVELS.  Tensors whose head size or strides are not multiples of 8
 * are quantized once per level instead. */
size_t cg_encode_kv_levels_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels);
size_t cg_encode_kv_levels_least_workspace(int64_t L, int64_t T, int64_t C, int64_t chunk_tokens, int nlevels);
/* Whether the levels of a call with these arguments share launches where the workspace is the larger one (tensors that the
 * vector loads take, tables of at most 80 entries, more than 128 channels): the least one is as good otherwise. */
int cg_encode_kv_levels_together(const void *kv, int64_t L, int64_t T, int64_t H, int64_t D,
                                 int64_t sl, int64_t skv, int64_t st, int64_t sh,
                                 int nlevels, const int *max_bins, int64_t chunk_tokens);
int cg_encode_kv_levels(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                        int64_t sl, int64_t skv, int64_t st, int64_t sh,
                        int nlevels, const float *const *key_bins, const float *const *value_bins,
                        const int *max_bins, int64_t chunk_tokens,
                        int16_t *const *cdf, void *maxima, int32_t *const *lengths,
                        int64_t *const *offsets, uint8_t *const *payload, const int64_t *payload_cap,
                        int32_t *status, void *workspace, size_t workspace_bytes, void *stream);

/* collect_bytes (encoder.py:209-222): the streams of a padded buffer, back to back.
 * padded   device uint8 [nl, nc, cap], strides (p0, p1, 1)
 * offsets  device int64 [nl*nc + 1]: exclusive running sum of the lengths (cg_scan_lengths)
 * out      device uint8 [out_bytes], written; nothing is written past it
 * The lengths have to fit the slots: cg_collect_sizes says whether they do. */
int cg_collect_bytes(const uint8_t *padded, int64_t cap, int64_t p0, int64_t p1, const int64_t *offsets,
                     int64_t nl, int64_t nc, uint8_t *out, int64_t out_bytes, void *stream);

/* Looks n streams over before cg_collect_bytes: offsets device int64 [n + 1], nslots and cap the
 * padded buffer's slots and their size.
 * out  int64 [2] that the GPU can write, pinned host memory as a rule; out[0] is written: offsets[n];
 *      out[1] (zero it first) is set to 1 if offsets[0] is not 0, a stream does not fit its slot, or
 *      one behind the last slot is not empty */
int cg_collect_sizes(const int64_t *offsets, int64_t n, int64_t nslots, int64_t cap, int64_t *out, void *stream);

/* Exclusive running sum of stream lengths: offsets[0] = 0, offsets[i+1] =
 * offsets[i] + lengths[i] (the inclusive sums of decoder.py:70 are offsets[1:]).
 * scratch: device, cg_scan_workspace(n) bytes. */
size_t cg_scan_workspace(int64_t n);
int cg_scan_lengths(const int32_t *lengths, int64_t n, int64_t *offsets,
                    void *scratch, size_t scratch_bytes, void *stream);

/* cg_scan_lengths for callers that cannot allocate device memory and have no workspace to
 * pass (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * No counterpart in the reference.  Same results as cg_scan_lengths; the partial sums live
 * in an array that is part of the library's device image (about 64 KiB on every GPU the
 * library runs on, held until the process ends), so the call allocates and frees nothing.
 * n <= CG_SCAN_STATIC_MAX_LENGTHS, CG_ERR_WORKSPACE otherwise.  All calls on one GPU share that
 * array: two calls whose kernels overlap on the same GPU (different streams, or different
 * threads on different streams) race; calls queued on one stream do not.  The first call on a
 * device looks the array's address up (hipGetSymbolAddress) with that device current. */
#define CG_SCAN_STATIC_MAX_LENGTHS (16 * 1024 * 1024)
int cg_scan_lengths_static(const int32_t *lengths, int64_t n, int64_t *offsets, void *stream);

/* decode_function_gpu + do_dequantize + the final cast and layout (decoder.py:
 * 77-112, 24-34, 159-173) for every chunk at once.
 * cdf, maxima, offsets, payload: as written by cg_encode_kv (maxima in max_dt);
 *             whole aligned 32-bit words of the payload are loaded, see
 *             cg_decode_fast_prefsum
 * out         device fp16/bf16 KV cache (out_dt, strides (ol, okv, ot, oh, 1)), written.
 *             ot and oh must not be negative, and 256 token rows of one layer's keys or
 *             values must span less than 4 GiB (((H-1)*oh + D-1 + 255*ot) * 2 + 2 bytes):
 *             the kernel addresses them with a 32-bit offset from a per-block base;
 *             CG_ERR_ARG otherwise */
int cg_decode_kv(const int16_t *cdf, int max_bins, const void *maxima, int max_dt,
                 const int64_t *offsets, const uint8_t *payload, int64_t payload_bytes,
                 const float *key_bins, const float *value_bins,
                 int64_t L, int64_t T, int64_t H, int64_t D, int64_t chunk_tokens,
                 int delta_group,
                 void *out, int out_dt, int64_t ol, int64_t okv, int64_t ot, int64_t oh,
                 void *stream);

/* cg_decode_kv for chunks that lie in several places, each with tables, maxima, lengths, payload
 * and quantization levels of its own, decoded by one launch into token ranges of one tensor: the
 * containers a store hands back, without bringing their sections together first.  One entry per
 * sub-chunk; every pointer is a device pointer.  No counterpart in the reference, which decodes
 * chunk by chunk and concatenates (cache_engine.py:229-293). */
typedef struct CgListedSub {
    const int16_t *cdf;             /* [2L, C, max_bins+1]: tables of the sub-chunk's chunk */
    const void *maxima;             /* 16-bit: row r's maximum of the sub-chunk's token i at r*maxima_pitch + i */
    const void *lengths;            /* [2L, C] int32, or uint16 (lengths_u16): bytes of every stream */
    const uint8_t *bytes;           /* 4-byte aligned; the payload's words are loaded from here ... */
    int64_t last_word;              /* ... up to the word at this byte offset */
    int64_t first;                  /* byte offset from `bytes` of the sub-chunk's first stream */
    const uint32_t *tile_starts;    /* [2L, ceil(C/64)]: bytes from the first stream to stream (row, 64*i) */
    const float *key_bins, *value_bins;     /* float32 [L] each */
    int64_t t_out;                  /* the sub-chunk's first token in the output tensor */
    int32_t n;                      /* its tokens, 1..256 */
    int32_t maxima_pitch;
    int32_t max_dt;                 /* CG_DT_* of the maxima */
    int32_t lengths_u16;
} CgListedSub;

/* subs: device array of nsub entries; the same max_bins, geometry and delta_group for all of them.
 * The output arguments and limits are those of cg_decode_kv. */
int cg_decode_listed(const CgListedSub *subs, int64_t nsub, int max_bins, int64_t L, int64_t H, int64_t D,
                     int delta_group, void *out, int out_dt, int64_t ol, int64_t okv, int64_t ot, int64_t oh,
                     void *stream);

/* HOST memory, no GPU work: the entries of cg_decode_listed and the running sums they point to, for
 * containers whose sections are (or will be) in device memory. */
typedef struct CgHostContainer {
    int64_t tables, maxima, lengths, payload;       /* device addresses of the sections: [nchunks, 2L, C, max_bins+1],
                                                       [2, L, T], [nsub, 2L, C], bytes back to back */
    int64_t payload_bytes;
    int64_t key_bins, value_bins;                   /* device addresses, float32 [L] each */
    int64_t t_out;                                  /* first token in the output tensor */
    int64_t tokens, chunk_tokens;
    int32_t max_bins, max_dt, lengths_u16;
    int32_t narrays;                                /* host arrays that hold the lengths, consecutive sub-chunks each */
} CgHostContainer;

/* lengths      HOST array of the containers' length arrays (narrays each, one after the other), array_subs
 *              the sub-chunks of each
 * tile_starts  HOST uint32, written; starts_at: its device address (see CgListedSub)
 * subs         HOST, written: one entry per sub-chunk, containers in order
 * bad          written: the number of the first container whose lengths are negative or do not add
 *              up to its payload (CG_ERR_ARG then) */
int cg_host_list(const CgHostContainer *items, int n, const void *const *lengths, const int64_t *array_subs,
                 int64_t L, int64_t C, uint32_t *tile_starts, int64_t starts_at, CgListedSub *subs, int *bad);

/* HOST memory, no GPU work: the running sums of stream lengths that cg_decode_listed starts from.
 * lengths      [nsub, rows, C] int32, or uint16 (itemsize 2), at any byte address
 * tile_starts  uint32 [nsub, rows, ceil(C/64)], written: bytes of the sub-chunk's streams before
 *              stream (row, 64*i), a stream counting min(length, 256) bytes
 * sub_bytes    int64 [nsub], written: bytes of every sub-chunk
 * CG_ERR_ARG if a length is negative. */
int cg_host_tile_starts(const void *lengths, int itemsize, int64_t nsub, int64_t rows, int64_t C,
                        uint32_t *tile_starts, int64_t *sub_bytes);

/* ---------------------------------------------------------------------------
 * Tables as histogram counts, for containers that store the counts (no counterpart in
 * the reference, whose container pickles the tables; the relation inverted here is
 * cal_cdf.cu:29-49).  A group is one (chunk, row): C channels sharing a token count
 * tokens[g] <= 256.
 * ------------------------------------------------------------------------- */

/* cdf     device int16 [ngroups, C, max_bins+1]
 * tokens  device int32 [ngroups]: tokens the tables of group g were built over (1..256)
 * counts  device uint8 [ngroups, C, max_bins], written: histogram counts, 256 stored as 255
 * nsym    device int32 [ngroups], written: 1 + the largest symbol that occurs in the group
 * inexact device int32 [1], written: 1 if some table is not the table of any histogram */
int cg_tables_to_counts(const int16_t *cdf, int max_bins, int64_t ngroups, int64_t C,
                        const int32_t *tokens, uint8_t *counts, int32_t *nsym, int32_t *inexact,
                        void *stream);

/* Ragged form of `counts`: out[starts[g] + ch*nsym[g] + j] = counts[g, ch, j], j < nsym[g].
 * starts may be null: the groups then follow one another (starts[g] = C * sum of nsym[0..g)). */
int cg_pack_counts(const uint8_t *counts, int max_bins, int64_t ngroups, int64_t C,
                   const int32_t *nsym, const int64_t *starts, uint8_t *out, void *stream);

/* Ragged counts back to tables.
 * data    device uint8 [data_bytes]: as written by cg_pack_counts (never read outside)
 * nsym    device uint8 [ngroups]; starts device int64 [ngroups]
 * cdf     device int16 [ngroups, C, max_bins+1], written
 * invalid device int32 [1], written: 1 if some channel's counts do not add up to tokens[g] */
int cg_counts_to_tables(const uint8_t *data, int64_t data_bytes, int max_bins, int64_t ngroups, int64_t C,
                        const int32_t *tokens, const uint8_t *nsym, const int64_t *starts, int16_t *cdf,
                        int32_t *invalid, void *stream);

/* The same for groups that lie in several containers (starts: byte offsets from `data`), with the verdict
 * stored to *invalid (device or pinned host memory, zero before the call) only where it is bad. */
int cg_rebuild_tables(const uint8_t *data, int64_t data_bytes, int max_bins, int64_t ngroups, int64_t C,
                      const int32_t *tokens, const uint8_t *nsym, const int64_t *starts, int16_t *cdf,
                      int32_t *invalid, void *stream);

/* What a host that lays out containers has to read back of an encoded tensor, in one piece:
 * out[0] = *status, out[1] = *wide (0 if null), out[2] = *inexact (0 if null), out[3 + i] =
 * offsets[i * per_sub] for i < nbounds, out[3 + nbounds + g] = nsym[g] for g < ngroups.
 * out  int64, device or pinned host memory (then no copy is needed: wait for the stream) */
int cg_wire_meta(const int32_t *status, const int64_t *offsets, int64_t per_sub, int64_t nbounds,
                 const int32_t *wide, const int32_t *inexact, const int32_t *nsym, int64_t ngroups,
                 int64_t *out, void *stream);

/* out[i] = lengths[i] as 16 bits; *wide (device int32, written) = 1 if some length does not fit. */
int cg_lengths_to_u16(const int32_t *lengths, int64_t n, uint16_t *out, int32_t *wide, void *stream);

/* ---------------------------------------------------------------------------
 * Between pinned host memory and device memory (no counterpart in the reference, which copies
 * tensor by tensor and waits).
 * ------------------------------------------------------------------------- */

/* A watch: places of a stream, in order, each with a number, that *mark shows (a word of ordinary host memory, ascending)
 * once the stream is through with what was queued before the place; brought up to date by the functions that wait.  One
 * thread at a time; made for the current device.  Null if there is no memory for it. */
void *cg_watch_new(int32_t *mark);
void cg_watch_free(void *watch);
/* A place, here. */
int cg_watch_add(void *watch, int32_t value, void *stream);
/* HOST: returns when *mark >= value; CG_ERR_ARG if no place has such a number. */
int cg_watch_wait(void *watch, int32_t value);

/* n > 0 bytes from src to dst, one of them in pinned host memory (to_host: dst) and the other in device
 * memory, queued on the stream.  Both stay valid until it is through.
 * watch  or null: a place behind it, with the number `value` */
int cg_move_bytes(const void *src, void *dst, int64_t n, int to_host, void *watch, int32_t value, void *stream);

/* Sets *mark (pinned host int32) to `value` when everything queued on the stream before this call is through, together with
 * what this library's launches among it stored to host memory (others': what they have themselves released to
 * the system). */
int cg_mark(int32_t *mark, int32_t value, void *stream);

/* HOST: returns when *mark >= value; CG_ERR_ARG if the stream is through and it is not. */
int cg_wait_mark(const int32_t *mark, int32_t value, void *stream);

/* The functions below store to `words`: 64 bytes of pinned memory, 8-byte aligned, one reader's at a time, whose last
 * int64 begins with the mark; the mark is set to `value`, which differs from call to call, behind everything else. */

/* HOST, returns when they are there: words[i] = the 4-byte (signed) or 8-byte number at at[i], device memory; n <= 4. */
int cg_read_words(const void *const *at, const int32_t *bytes, int n, void *words, int32_t value, void *stream);

/* HOST, returns when it is there: the first float of words = the largest value of the device vectors a and b, n each; NaN
 * if there is one. */
int cg_largest(const float *a, const float *b, int64_t n, void *words, int32_t value, void *stream);

/* cg_scan_lengths and cg_collect_sizes, with its numbers in words[0] and words[1]; does not wait. */
int cg_scan_collect(const int32_t *lengths, int64_t n, int64_t *offsets, void *scratch, size_t scratch_bytes,
                    int64_t nslots, int64_t cap, void *words, int32_t value, void *stream);

/* cg_decode_fast_prefsum from the stream lengths (device int32 [nl, nc]): offsets (device int64 [nl*nc + 1]) is written
 * by cg_scan_lengths, whose scratch is scratch. */
int cg_decode_fast_lengths(const int16_t *cdf, int lp, const uint8_t *bytes, int64_t nbytes, const int32_t *lengths,
                           int64_t nl, int64_t nt, int64_t nc, uint8_t *out, int64_t o0, int64_t o1, int64_t o2,
                           int64_t *offsets, void *scratch, size_t scratch_bytes, void *stream);

/* The threads of a host function: those of an OpenMP runtime, through its documented entry points, at most `threads`
 * of them (the runtime may give fewer).  Null, or null pointers: the caller alone. */
typedef struct CgHostTeam {
    void (*parallel)(void (*fn)(void *), void *data, unsigned num_threads, unsigned flags);      /* GOMP_parallel */
    int (*thread_num)(void);                                                                     /* omp_get_thread_num */
    int32_t threads;
    int32_t reserved;
} CgHostTeam;

/* One copy on the host. */
typedef struct CgHostPart {
    int64_t dst, src;               /* addresses; cg_host_stage: dst is an offset in the area */
    int64_t bytes;
    int32_t value;                  /* cg_host_fill: src is there when the mark is this far */
    int32_t reserved;
} CgHostPart;

/* HOST: the copies, by the team, each part as soon as *mark says that it has arrived; returns when all
 * are done.  watch: the mark's, which has places up to the largest number; or null: somebody else sets the mark. */
int cg_host_fill(const CgHostPart *parts, int n, const int32_t *mark, const CgHostTeam *team, void *watch);

/* HOST and the stream: `bytes` bytes of device memory at `area` from the parts (ascending, not overlapping; what lies
 * between them is undefined), staged in pinned memory by the team and moved in steps, each as soon as it is staged.
 * step   bytes of a step, a multiple of 64 (the first is a quarter of one)
 * slots  HOST array of nslots addresses of pinned memory, a step each, used in turn: two at least, or as many as
 *        there are steps (the last of them then no larger than what is left); stays valid until the moves are through
 * watch, value  as in cg_move_bytes, behind the last move
 * moves  written: the moves queued (all of them, or those before an error) */
int cg_host_stage(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, void *area, int64_t bytes,
                  void *watch, int32_t value, const CgHostTeam *team, int *moves, void *stream);

/* Test hook, no GPU work: cg_host_stage with a copy on the host in the place of each move, done as late as a move may be;
 * `area` is host memory. */
int cg_test_host_stage(const CgHostPart *parts, int n, void *const *slots, int nslots, int64_t step, void *area, int64_t bytes,
                       const CgHostTeam *team, int *moves);

#ifdef __cplusplus
}
#endif
#endif /* CACHEGEN_HIP_H */
