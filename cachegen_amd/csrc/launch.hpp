// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip, which
// is the one translation unit.  Host-side launch helpers: block size, grids, kernel dispatch.
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
// host-side launch helpers
// ------------------------------------------------------------------------------------
// Lanes per block: as many adjacent channels as possible while the per-block table
// (lp words per lane) stays well inside the default dynamic LDS window.
int pick_block(int64_t nc, int lp)
{
    int block = 256;
    if (lp > 80) block = 128;
    while (block > 64 && nc <= block / 2) block /= 2;
    return block;
}

// The stream kernels run on a three-dimensional grid (channel tile, row, sub-chunk), so that a
// block reads its place from its index instead of dividing for it: rows and sub-chunks are grid
// dimensions and must fit one.
int check_grid_limits(int64_t rows, int64_t nsub)
{
    if (rows > 65535 || nsub > 65535)
        return fail(CG_ERR_ARG, "%lld rows and %lld sub-chunks: at most 65535 of each in one call", (long long)rows, (long long)nsub);
    return CG_OK;
}

int make_grid(int64_t rows, int64_t nc, int64_t T, int64_t S, int64_t nsub, int block,
              StreamGrid &sg, int64_t &nblocks)
{
    sg.rows = rows;
    sg.nc = nc;
    sg.ctiles = (int32_t)ceil_div(nc, block);
    sg.g.T = T;
    sg.g.S = S;
    sg.g.nsc = (int32_t)ceil_div(S, kSub);
    nblocks = nsub * rows * sg.ctiles;
    if (nblocks <= 0 || nblocks > INT_MAX) return fail(CG_ERR_ARG, "grid of %lld blocks is out of range", (long long)nblocks);
    return check_grid_limits(rows, nsub);
}

dim3 stream_grid(const StreamGrid &sg, int64_t nblocks)
{
    return dim3((unsigned)sg.ctiles, (unsigned)sg.rows, (unsigned)(nblocks / (sg.rows * sg.ctiles)));
}

// Compute units of the current device (asked once per device).
int compute_units()
{
    static std::atomic<int> known[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = known[dev].load(std::memory_order_relaxed);
    if (!n) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        known[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Run `launch` with the block size as a compile-time constant.
#define CG_DISPATCH_BS(block, ...)                      \
    do {                                                \
        if ((block) == 256) { constexpr int BS = 256; __VA_ARGS__; } \
        else if ((block) == 128) { constexpr int BS = 128; __VA_ARGS__; } \
        else { constexpr int BS = 64; __VA_ARGS__; }    \
    } while (0)

// Lanes (channels of all rows and chunks, up to a block's width) up to which the tables are counted by
// four slices of a block (calculate_cdf_kernel).  The slices wait for their loads side by side, which is
// what a call of few blocks or long chunks is made of; a block of four times the lanes costs more to
// start and, from 640 blocks of 256 lanes on, leaves a second round of blocks.  Unsliced / sliced, 512 to
// 4096 channels, 4 to 512 rows, tables of 33 entries, us:
//   symbols as bytes, chunks of   32 tokens    64 k lanes 10.0 /  9.9   128 k 10.8 / 11.2   160 k 12.2 / 17.3
//                                 64                      11.4 / 10.4         12.1 / 12.0         13.6 / 18.7
//                                256                      19.5 / 13.1         22.1 / 17.9         26.6 / 26.9   250 k 29.9 / 32.2
//                                512                      31.1 / 17.6         39.5 / 26.6         42.4 / 36.8         47.1 / 46.0
//                               1024                      67.5 / 28.0         69.5 / 42.0         74.2 / 57.0         101.8 / 79.0
// Packed symbols, whole encode call, tables of 17 / 33 / 65 entries: with slices a chunk of 300 tokens takes
// 1.02 / 1.03 / 1.05 times as long at 72 k to 128 k lanes and 1.08 / 1.08 / 1.1 at 160 k, one of 512 tokens
// 1.00 / 1.01 / 1.02 and 1.06, one of 700 tokens 0.985 / 0.985 / 1.02 and 1.05, one of 1000 to 1500 0.98 /
// 0.98 / 1.02 and 1.04; at 64 k lanes and below less time throughout (1500 tokens 0.89, 512 tokens 0.94).
int64_t sliced_lanes(bool packed, int64_t chunk_tokens)
{
    if (packed) return (chunk_tokens >= 640 ? 128 : 64) << 10;
    return (chunk_tokens >= 512 ? 256 : chunk_tokens >= 64 ? 128 : 64) << 10;
}

// The blocks of a table pass over `nlevels` levels (1 for byte symbols) and their LDS, the longest table's.
struct CdfGrid {
    int block;
    bool sliced;
    dim3 grid;
    size_t shmem;
};

int make_cdf_grid(CdfArgs &a, bool packed, int nlevels, int max_lp, CdfGrid &g)
{
    const int64_t S = a.g.S, T = a.g.T;
    int block = pick_block(a.nc, max_lp);
    while (!packed && block > 64 && (size_t)max_lp * (block + 1) * sizeof(uint32_t) > 64 * 1024) block /= 2;
    a.ctiles = (int32_t)ceil_div(a.nc, block);
    int64_t nblocks = ceil_div(T, S) * a.rows * a.ctiles;
    if (nblocks <= 0 || nblocks > INT_MAX) return fail(CG_ERR_ARG, "calculate_cdf: grid out of range");
    // Narrower blocks where that is how more compute units get one: a block's lanes and slices all count
    // through one unit's LDS.  512 channels x 4 rows: 512 tokens 13.1 -> 8.6 us, 256 tokens of byte symbols 11.1 -> 7.6.
    while (block > 64 && nblocks * nlevels * 2 <= compute_units()) {
        block /= 2;
        a.ctiles = (int32_t)ceil_div(a.nc, block);
        nblocks = ceil_div(T, S) * a.rows * a.ctiles;
    }
    g.block = block;
    g.shmem = packed ? (size_t)max_lp * (block + 2) * sizeof(uint16_t)
                     : (size_t)max_lp * (block + 1) * sizeof(uint32_t);     // TableStride
    g.sliced = nblocks * nlevels * block <= sliced_lanes(packed, S < T ? S : T);
    g.grid = dim3((unsigned)nblocks, (unsigned)nlevels);
    return CG_OK;
}

// key_bins, value_bins (packed symbols only, may be null): the rows of at most 15 symbols hold
// four bits a symbol.
int launch_cdf(const uint8_t *sym, const uint32_t *sym4, int64_t nsub, int64_t rows, int64_t T,
               int64_t nc, int64_t s0, int64_t s1, int64_t s2, int max_bins, int64_t S,
               uint16_t *cdf, hipStream_t stream, const float *key_bins = nullptr, const float *value_bins = nullptr)
{
    CdfArgs a;
    a.sym = sym;
    a.s0 = s0;
    a.s1 = s1;
    a.s2 = s2;
    a.sym4 = sym4;
    a.nsub = nsub;
    a.nibbles = (sym4 && key_bins && value_bins) ? 1 : 0;
    a.key_bins = key_bins;
    a.value_bins = value_bins;
    a.L = rows / 2;
    a.cdf = cdf;
    a.rows = rows;
    a.nc = nc;
    a.max_bins = max_bins;
    a.g.T = T;
    a.g.S = S;
    a.g.nsc = (int32_t)ceil_div(S, kSub);
    CdfGrid g;
    if (int rc = make_cdf_grid(a, sym4 != nullptr, 1, max_bins + 1, g)) return rc;
    const dim3 grid = g.grid, blk(g.sliced ? g.block * 4 : g.block);
    const size_t shmem = g.shmem;
    if (g.sliced) {
        if (sym4) CG_DISPATCH_BS(g.block, (calculate_cdf_kernel<BS, true, 4><<<grid, blk, shmem, stream>>>(a)));
        else CG_DISPATCH_BS(g.block, (calculate_cdf_kernel<BS, false, 4><<<grid, blk, shmem, stream>>>(a)));
    } else {
        if (sym4) CG_DISPATCH_BS(g.block, (calculate_cdf_kernel<BS, true, 1><<<grid, blk, shmem, stream>>>(a)));
        else CG_DISPATCH_BS(g.block, (calculate_cdf_kernel<BS, false, 1><<<grid, blk, shmem, stream>>>(a)));
    }
    return check_launch("calculate_cdf");
}

int launch_scan(const int32_t *lengths, int64_t n, int32_t clamp, int64_t *offsets, void *scratch,
                hipStream_t stream)
{
    const int64_t ntiles = ceil_div(n, kScanTile);
    int64_t *sums = static_cast<int64_t *>(scratch);
    if (ntiles > 1 && n <= kScanSmallMax) {
        // a few thousand values: one block does it all, two launches fewer
        scan_small_kernel<<<dim3(1), dim3(kScanSmallThreads), 0, stream>>>(lengths, (int32_t)n, clamp, offsets);
        return check_launch("scan_lengths");
    }
    if (ntiles == 1) {
        scan_apply_kernel<<<dim3(1), dim3(kScanThreads), 0, stream>>>(lengths, n, clamp, nullptr, offsets);
        return check_launch("scan_lengths");
    }
    scan_tile_sums_kernel<<<dim3((unsigned)ntiles), dim3(kScanThreads), 0, stream>>>(lengths, n, clamp, sums);
    scan_sums_kernel<<<dim3(1), dim3(kScanThreads), 0, stream>>>(sums, ntiles);
    scan_apply_kernel<<<dim3((unsigned)ntiles), dim3(kScanThreads), 0, stream>>>(lengths, n, clamp, sums, offsets);
    return check_launch("scan_lengths");
}

int check_dt(int dt, const char *what)
{
    if (dt != CG_DT_F16 && dt != CG_DT_BF16) return fail(CG_ERR_ARG, "%s: dtype must be CG_DT_F16 or CG_DT_BF16", what);
    return CG_OK;
}

int check_lp(int lp, const char *what)
{
    if (lp < 2 || lp > CG_MAX_LP) return fail(CG_ERR_ARG, "%s: CDF length should be in [2, %d], got %d", what, CG_MAX_LP, lp);
    return CG_OK;
}

bool kv_vectorizable(const void *kv, int64_t D, int64_t C, int64_t sl, int64_t skv, int64_t st, int64_t sh)
{
    return (D % 8 == 0) && (sl % 8 == 0) && (skv % 8 == 0) && (st % 8 == 0) && (sh % 8 == 0) &&
           aligned_to(kv, 16) && (C / 8 <= 64 * kMaxUnits);
}

int launch_quantize(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                    int64_t sl, int64_t skv, int64_t st, int64_t sh, const float *key_bins,
                    const float *value_bins, uint8_t *sym, void *maxima, hipStream_t stream)
{
    const int64_t C = H * D;
    const int64_t nrows = 2 * L * T;
    const int64_t nblocks = ceil_div(nrows, 4);
    if (nblocks > INT_MAX || C > INT_MAX) return fail(CG_ERR_ARG, "quantize: tensor too large for one launch");
    const bool vec = kv_vectorizable(kv, D, C, sl, skv, st, sh) && aligned_to(sym, 8);
    const uint16_t *p = static_cast<const uint16_t *>(kv);
    uint16_t *mx = static_cast<uint16_t *>(maxima);
    dim3 grid((unsigned)nblocks), block(256);
    if (vec) {
        const int nunits = (int)(C / 8);
        const bool contiguous = (sh == D);
#define CG_LAUNCH_Q(DT, HC) quantize_kv_kernel<DT, HC><<<grid, block, 0, stream>>>( \
        p, L, T, (int)D, sl, skv, st, sh, key_bins, value_bins, sym, mx, nunits, nrows)
        if (kv_dt == CG_DT_F16) { if (contiguous) CG_LAUNCH_Q(CG_DT_F16, true); else CG_LAUNCH_Q(CG_DT_F16, false); }
        else { if (contiguous) CG_LAUNCH_Q(CG_DT_BF16, true); else CG_LAUNCH_Q(CG_DT_BF16, false); }
#undef CG_LAUNCH_Q
    } else {
        if (kv_dt == CG_DT_F16)
            quantize_kv_generic_kernel<CG_DT_F16><<<grid, block, 0, stream>>>(
                p, L, T, (int)D, (int)C, sl, skv, st, sh, key_bins, value_bins, sym, mx, nrows);
        else
            quantize_kv_generic_kernel<CG_DT_BF16><<<grid, block, 0, stream>>>(
                p, L, T, (int)D, (int)C, sl, skv, st, sh, key_bins, value_bins, sym, mx, nrows);
    }
    return check_launch("quantize_kv");
}

template <int DT, bool HC>
void launch_quantize_pack_nu(const PackedQuantArgs &a, int64_t nblocks, hipStream_t stream)
{
    const dim3 grid((unsigned)nblocks), block(256);
    if (a.delta_group > 0) {
        if (a.nunits <= 128) quantize_pack_delta_kernel<DT, HC, 2><<<grid, block, 0, stream>>>(a);
        else if (a.nunits <= 256) quantize_pack_delta_kernel<DT, HC, 4><<<grid, block, 0, stream>>>(a);
        else quantize_pack_delta_kernel<DT, HC, 8><<<grid, block, 0, stream>>>(a);
        return;
    }
    if (a.nlevels > 0) {
        if (a.nunits <= 128) quantize_pack_kernel<DT, HC, 2, true><<<grid, block, 0, stream>>>(a);
        else if (a.nunits <= 256) quantize_pack_kernel<DT, HC, 4, true><<<grid, block, 0, stream>>>(a);
        else quantize_pack_kernel<DT, HC, 8, true><<<grid, block, 0, stream>>>(a);
        return;
    }
    if (a.nunits <= 128) quantize_pack_kernel<DT, HC, 2><<<grid, block, 0, stream>>>(a);
    else if (a.nunits <= 256) quantize_pack_kernel<DT, HC, 4><<<grid, block, 0, stream>>>(a);
    else quantize_pack_kernel<DT, HC, 8><<<grid, block, 0, stream>>>(a);
}

// nlevels > 0: key_bins_lv / value_bins_lv hold that many bins vectors and level v's words go
// to sym4 + v * level_words (one read of the tensor for all levels); nlevels == 0: one level,
// key_bins / value_bins.
int launch_quantize_pack(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                         int64_t sl, int64_t skv, int64_t st, int64_t sh, const float *key_bins,
                         const float *value_bins, uint32_t *sym4, void *maxima, int64_t nsub,
                         int64_t S, int delta_group, hipStream_t stream, int32_t *status, int nlevels = 0,
                         const float *const *key_bins_lv = nullptr, const float *const *value_bins_lv = nullptr,
                         int64_t level_words = 0, bool nibbles = false, const int *lp_lv = nullptr, int lp = 0,
                         int32_t *group_sums = nullptr)
{
    PackedQuantArgs a;
    memset(&a, 0, sizeof(a));
    // status: one word per level (one word when nlevels == 0), consecutive
    a.nstatus = nlevels > 0 ? nlevels : 1;
    for (int v = 0; v < a.nstatus; ++v) a.status[v] = status + v;
    a.group_sums = group_sums;          // kMaxTileGroups words per level
    a.ngroup_sums = group_sums ? kMaxTileGroups * a.nstatus : 0;
    a.nlevels = nlevels;
    for (int v = 0; v < nlevels; ++v) {
        a.key_bins_lv[v] = key_bins_lv[v];
        a.value_bins_lv[v] = value_bins_lv[v];
        a.lp_lv[v] = lp_lv ? lp_lv[v] : 0;
    }
    a.lp = lp;
    a.level_words = level_words;
    a.nibbles = nibbles ? 1 : 0;
    a.kv = static_cast<const uint16_t *>(kv);
    a.L = L;
    a.sl = sl;
    a.skv = skv;
    a.st = st;
    a.sh = sh;
    a.D = (int32_t)D;
    a.key_bins = key_bins;
    a.value_bins = value_bins;
    a.sym4 = sym4;
    a.maxima = static_cast<uint16_t *>(maxima);
    a.nunits = (int32_t)(H * D / 8);
    a.nsub = nsub;
    a.delta_group = delta_group;
    a.g.T = T;
    a.g.S = S;
    a.g.nsc = (int32_t)ceil_div(S, kSub);
    const int64_t nblocks = 2 * L * nsub * 16;
    if (nblocks > INT_MAX) return fail(CG_ERR_ARG, "quantize: tensor too large for one launch");
    const bool contiguous = (sh == D);
    if (kv_dt == CG_DT_F16) {
        if (contiguous) launch_quantize_pack_nu<CG_DT_F16, true>(a, nblocks, stream);
        else launch_quantize_pack_nu<CG_DT_F16, false>(a, nblocks, stream);
    } else {
        if (contiguous) launch_quantize_pack_nu<CG_DT_BF16, true>(a, nblocks, stream);
        else launch_quantize_pack_nu<CG_DT_BF16, false>(a, nblocks, stream);
    }
    return check_launch("quantize_pack");
}

// The quantizer that also builds the tables (quantize_tables_kernel): which of its forms takes a tensor of `nunits` units of 8 channels and tables of `lp` entries,
// if any.
// Long chunks of a call with fewer (row, chunk) pairs than this are cut into parts, whole
// sub-chunks each, until the launch has about this many blocks (measured on one table over
// 8192 tokens of 32 layers: parts of 256 tokens 0.765 ms, of 512 tokens 0.807, the whole encode).
constexpr int64_t kQuantTablesPartBlocks = 2048;

struct QuantTablesShape {
    int nu, lp;
    size_t lds;
};

constexpr size_t kMaxLdsPerBlock = 160 * 1024;      // gfx950
// fewer (row, chunk) blocks than this leave compute units idle: the two-kernel form is used instead
constexpr int64_t kQuantTablesMinBlocks = 512;

bool quantize_tables_shape(int64_t nunits, int lp, bool heads_contiguous, QuantTablesShape &shape)
{
    // 2048 channels: only tensors whose heads follow one another (the other form runs out of registers)
    const int nu = nunits <= 64 ? 1 : nunits <= 128 ? 2 : (nunits <= 256 && heads_contiguous) ? 4 : 0;
    if (!nu || (lp != 9 && lp != 17 && lp != 33 && lp != 65)) return false;
    shape.nu = nu;
    shape.lp = lp;
    shape.lds = (size_t)nu * 4 * lp * 256;
    return shape.lds <= kMaxLdsPerBlock;
}

// A kernel that wants more than 64 KiB of dynamic LDS has to be allowed to, once per device;
// `asked` holds one bit per device for that kernel.
int allow_dynamic_lds(const void *kernel, int bytes, std::atomic<uint64_t> &asked)
{
    if (bytes <= 64 * 1024) return CG_OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return fail(CG_ERR_LAUNCH, "dynamic LDS: hipGetDevice");
    if (asked.load(std::memory_order_relaxed) >> dev & 1) return CG_OK;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(CG_ERR_LAUNCH, "dynamic LDS: hipFuncSetAttribute: %s", hipGetErrorString(e));
    asked.fetch_or(1ull << dev, std::memory_order_relaxed);
    return CG_OK;
}

template <int DT, bool HC, int NU, int LP>
int launch_quantize_tables_form(const QuantTablesArgs &a, dim3 grid, hipStream_t stream)
{
    typedef CountLayout<NU, LP> Layout;
    if (Layout::kBytes > (int)kMaxLdsPerBlock) return fail(CG_ERR_ARG, "quantize_tables: tables do not fit the LDS");
    static std::atomic<uint64_t> asked{0}, asked_for_sums{0};       // per form of the kernel: these are templates
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(&quantize_tables_kernel<DT, HC, NU, LP>), Layout::kBytes, asked)) return rc;
    if (!a.partial) {
        quantize_tables_kernel<DT, HC, NU, LP><<<grid, dim3(QuantTablesBlock<NU>::kThreads), Layout::kBytes, stream>>>(a);
        return check_launch("quantize_tables");
    }
    // chunks cut into parts: counters summed in memory, then one block per (chunk, row) for the tables
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(&tables_from_partial_kernel<NU, LP>), Layout::kBytes, asked_for_sums)) return rc;
    const int64_t nquads = (int64_t)grid.x * grid.y * (Layout::kBytes / 16);
    clear_quads_kernel<<<dim3((unsigned)ceil_div(nquads, 256)), dim3(256), 0, stream>>>(reinterpret_cast<uint4 *>(a.partial), nquads);
    quantize_tables_kernel<DT, HC, NU, LP><<<grid, dim3(QuantTablesBlock<NU>::kThreads), Layout::kBytes, stream>>>(a);
    tables_from_partial_kernel<NU, LP><<<dim3(grid.x, grid.y), dim3(QuantTablesBlock<NU>::kThreads), Layout::kBytes, stream>>>(
        a.partial, a.cdf, a.nunits, a.g);
    return check_launch("quantize_tables");
}

template <int DT, bool HC, int LP>
int launch_quantize_tables_nu(const QuantTablesArgs &a, const QuantTablesShape &shape, dim3 grid, hipStream_t stream)
{
    if (shape.nu == 1) return launch_quantize_tables_form<DT, HC, 1, LP>(a, grid, stream);
    if (shape.nu == 2) return launch_quantize_tables_form<DT, HC, 2, LP>(a, grid, stream);
    if (HC && LP <= 33) return launch_quantize_tables_form<DT, true, 4, (LP <= 33 ? LP : 33)>(a, grid, stream);
    return fail(CG_ERR_ARG, "quantize_tables: shape not built");
}

template <int DT, bool HC>
int launch_quantize_tables_shape(const QuantTablesArgs &a, const QuantTablesShape &shape, dim3 grid, hipStream_t stream)
{
    switch (shape.lp) {
    case 9: return launch_quantize_tables_nu<DT, HC, 9>(a, shape, grid, stream);
    case 17: return launch_quantize_tables_nu<DT, HC, 17>(a, shape, grid, stream);
    case 33: return launch_quantize_tables_nu<DT, HC, 33>(a, shape, grid, stream);
    case 65: return launch_quantize_tables_nu<DT, HC, 65>(a, shape, grid, stream);
    }
    return fail(CG_ERR_ARG, "quantize_tables: shape not built");
}

// Quantization, row maxima, packed symbols and the tables of every chunk in one launch.
int launch_quantize_tables(const void *kv, int kv_dt, int64_t L, int64_t T, int64_t H, int64_t D,
                           int64_t sl, int64_t skv, int64_t st, int64_t sh, const float *key_bins,
                           const float *value_bins, uint32_t *sym4, void *maxima, uint16_t *cdf, int64_t nsub, int64_t S,
                           bool nibbles, int32_t *status,
                           const QuantTablesShape &shape, hipStream_t stream,
                           int64_t part_tokens = 0, void *partial = nullptr, size_t partial_bytes = 0,
                           int32_t *group_sums = nullptr)
{
    QuantTablesArgs a;
    memset(&a, 0, sizeof(a));
    a.kv = static_cast<const uint16_t *>(kv);
    a.L = L;
    a.sl = sl;
    a.skv = skv;
    a.st = st;
    a.sh = sh;
    a.D = (int32_t)D;
    a.key_bins = key_bins;
    a.value_bins = value_bins;
    a.status = status;
    a.group_sums = group_sums;          // kMaxTileGroups words of the workspace
    a.ngroups = kMaxTileGroups;
    a.sym4 = sym4;
    a.maxima = static_cast<uint16_t *>(maxima);
    a.cdf = cdf;
    a.nunits = (int32_t)(H * D / 8);
    a.nsub = nsub;
    a.nibbles = nibbles ? 1 : 0;
    a.g.T = T;
    a.g.S = S;
    a.g.nsc = (int32_t)ceil_div(S, kSub);
    const int64_t nchunks = ceil_div(T, S);
    if (nchunks > INT_MAX || 2 * L > 65535) return fail(CG_ERR_ARG, "quantize_tables: grid out of range");
    dim3 grid((unsigned)nchunks, (unsigned)(2 * L));
    if (partial) {
        const int64_t nparts = ceil_div(S < T ? S : T, part_tokens);
        if (part_tokens <= 0 || part_tokens % kSub || nparts > 65535 || !aligned_to(partial, 16) ||
            (size_t)nchunks * 2 * L * shape.lds > partial_bytes)
            return fail(CG_ERR_ARG, "quantize_tables: parts of chunks out of range");
        grid.z = (unsigned)nparts;
        a.part_tokens = (int32_t)part_tokens;
        a.partial = static_cast<uint32_t *>(partial);
    }
    const bool contiguous = (sh == D);
    if (kv_dt == CG_DT_F16) {
        if (contiguous) return launch_quantize_tables_shape<CG_DT_F16, true>(a, shape, grid, stream);
        return launch_quantize_tables_shape<CG_DT_F16, false>(a, shape, grid, stream);
    }
    if (contiguous) return launch_quantize_tables_shape<CG_DT_BF16, true>(a, shape, grid, stream);
    return launch_quantize_tables_shape<CG_DT_BF16, false>(a, shape, grid, stream);
}

// Where the symbols and tables of an encode come from.
enum EncodeSource {
    ENC_BYTES,              // byte symbols, tables in memory (the reference's entry point)
    ENC_COUNTED,            // packed symbols, tables made by the coder
    ENC_TABLES,             // packed symbols, tables made by a pass of their own
    ENC_QUANTIZER_TABLES,   // packed symbols, tables made by the quantizer
};

// Wavefronts a compute unit up to which an encode is bound by one stream's chain of symbols
// (encode_few_kernel).  tile: every block is a whole tile of the scratch (TILE).  Measured on make_kv's caches,
// encode_streams_kernel / encode_few_kernel, the whole call in a graph, us, by wavefronts a SIMD (a quarter of a unit's):
//   1024 channels, tables of      17           33           41           65           97          129 entries
//   byte symbols        1      49 /  29     52 /  39     53 /  43     58 /  49     67 /  60     70 /  61
//   (256 tokens)        1.5    53 /  37     55 /  47     56 /  52     62 /  61     67 /  62     70 / 102
//                       2      53 /  38     56 /  48     57 /  52     62 /  61     68 / 104     71 / 113
//                       2.5    58 /  48     61 /  61     62 /  64     69 /  93     74 / 119    133 / 148
//                       3      58 /  48     61 /  61     63 /  66     70 / 104     82 / 124    139 / 165
//   tables by the       0.5    53 /  39     62 /  51     64 /  55     69 /  60     81 /  80     84 /  83
//   coder (256 tokens)  1      60 /  45     69 /  57     71 /  62     76 /  66     92 /  94     96 /  97
//                       1.5    66 /  57     73 /  68     77 /  73     82 /  80     97 / 102    102 / 146
//                       2      71 /  62     81 /  76     85 /  81     91 /  88    107 / 149    113 / 166
//   by a pass of their  1      62 /  53     69 /  64     71 /  67     77 /  74     95 / 101    102 / 108
//   own (512 tokens)    1.5    70 /  66     76 /  75     79 /  82     88 /  93    103 / 112    112 / 162
//                       2      75 /  71     85 /  87     88 /  92     98 / 104    111 / 160    122 / 178
//   by the quantizer    1      80 /  69     87 /  82                 102 / 100
//   (512 tokens)        2      84 /  79     95 /  97                 114 / 119
//   (256 tokens)        1      74 /  63     80 /  75                  89 /  87
//                       2                   86 /  86
//   400, 128, 64 channels (blocks of 256, 128, 64 lanes), packed symbols, at the line taken and above it:
//   by the coder        25 entries: 400  87 / 83 at 2;  128  97 / 95 at 1, 106 / 111 at 1.25;  64  91 / 91 at 0.5, 119 / 122 at 1
//                       65 entries: 400  86 / 81 at 1, 90 / 92 at 1.25
//   by a pass           17 entries: 400  84 / 82 at 2;  128  95 / 94 at 1, 110 / 111 at 1.5;  64  78 / 81 at 0.25
//                       29 entries: 400  80 / 79 at 1, 85 / 87 at 1.25;  33 entries: 400  68 / 69 at 0.25, 80 / 80 at 1
//   by the quantizer    17 entries: 400  85 / 83 at 2;  128  93 / 92 at 1, 115 / 118 at 2;  64  87 / 89 at 0.5, 115 / 121 at 1
//                       33 entries: 400  89 / 89 at 1, 91 / 95 at 1.25;  128  88 / 93 at 0.25
//   byte symbols of 64 channels and 25 to 29 entries, the worst of that form: 65 / 69 at 2.25, 71 / 73 at 2.5, 74 / 74 at 3
// (the last column of byte symbols is 128 entries).  Longer tables cost encode_few_kernel more: it copies
// those that are in memory entry by entry, at twice the width.
int few_encode_wavefronts(EncodeSource source, int lp, int block, bool tile)
{
    if (source == ENC_BYTES) return lp <= 33 ? 12 : 8;
    if (source == ENC_COUNTED) return lp > 80 || block == 64 ? 2 : block == 128 || (lp > 33 && !tile) ? 4 : 8;
    if (tile) return lp <= (source == ENC_TABLES ? 17 : 33) ? 8 : 4;
    if (block == 256) return lp <= 17 ? 8 : lp <= (source == ENC_TABLES ? 29 : 33) ? 4 : 0;
    return block == 128 && lp <= 17 ? 4 : 0;
}

// Blocks a compute unit up to which it is taken: those wavefronts, and no more than its LDS holds at once,
// or a second round of blocks waits for the first (65 entries from byte symbols, blocks of 65 KB, two a
// unit: 61 us for two wavefronts a SIMD, 91 for 2.25).  LDS is given out by 1280 bytes (of blocks of 53 x 1024
// bytes a unit holds two, not three); a block of packed symbols has 272 besides its tables.
int64_t few_encode_blocks(EncodeSource source, int lp, int block, bool tile)
{
    const size_t lds = align_up((size_t)lp * block * sizeof(uint32_t) + (source == ENC_BYTES ? 0 : 272), 1280);
    const int64_t fit = (int64_t)(kMaxLdsPerBlock / lds), chain = (int64_t)few_encode_wavefronts(source, lp, block, tile) * 64 / block;
    return fit < chain ? fit : chain;
}

bool few_encode(int64_t nblocks, EncodeSource source, int lp, int block, bool tile)
{
    return nblocks <= (int64_t)compute_units() * few_encode_blocks(source, lp, block, tile);
}

// Output buffers whose streams begin at multiples of four bytes.
template <int BS, bool PACKED, bool FUSE_CDF, bool SLOTS, bool TILE = false>
int launch_encode(const EncodeArgs &a, dim3 grid, bool few, hipStream_t stream)
{
    if (few) {
        static std::atomic<uint64_t> asked{0};          // per form of the kernel: these are templates
        const size_t lds = (size_t)a.lp * BS * sizeof(uint32_t);
        if (lds > 64 * 1024)
            if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(&encode_few_kernel<BS, PACKED, FUSE_CDF, SLOTS, TILE>),
                                           CG_MAX_LP * BS * (int)sizeof(uint32_t), asked)) return rc;
        encode_few_kernel<BS, PACKED, FUSE_CDF, SLOTS, TILE><<<grid, dim3(BS), lds, stream>>>(a);
    } else {
        const size_t lds = encode_lds<BS, PACKED>(a.lp);
        encode_streams_kernel<BS, true, PACKED, FUSE_CDF, SLOTS, TILE><<<grid, dim3(BS), lds, stream>>>(a);
    }
    return check_launch("encode");
}

// Blocks of tables of `lp` entries that a compute unit holds at once (eight of 256 lanes are all its wavefronts).
int64_t resident_encode_blocks(int lp)
{
    const int64_t fit = (int64_t)(kMaxLdsPerBlock / align_up(encode_lds<kSlotTile, true>(lp), 1280));
    return fit < 8 ? fit : 8;
}

// `count` levels in one launch of blocks of 256 lanes; their tables' LDS is the longest's.
template <bool FUSE_CDF, bool TILE>
int launch_encode_levels(const EncodeLevelsArgs &p, int count, int max_lp, dim3 grid, bool few, hipStream_t stream)
{
    constexpr int BS = kSlotTile;
    grid.z *= (unsigned)count;
    if (few) {
        static std::atomic<uint64_t> asked{0};          // per form of the kernel: these are templates
        const size_t lds = (size_t)max_lp * BS * sizeof(uint32_t);
        if (lds > 64 * 1024)
            if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(&encode_few_levels_kernel<BS, FUSE_CDF, TILE>),
                                           CG_MAX_LP * BS * (int)sizeof(uint32_t), asked)) return rc;
        encode_few_levels_kernel<BS, FUSE_CDF, TILE><<<grid, dim3(BS), lds, stream>>>(p);
    } else {
        encode_streams_levels_kernel<BS, FUSE_CDF, TILE><<<grid, dim3(BS), encode_lds<BS, true>(max_lp), stream>>>(p);
    }
    return check_launch("encode levels");
}

// Whether the coder begins with the last sub-chunk: the compaction behind it begins with the first, and so
// finds what the coder wrote last in the last-level cache (256 MB; the scratch of 8192 tiles is 0.22 GB of
// partial lines) instead of pushing it out before it gets there.  Forward / last first, 32 layers x 1024
// channels, us: 4096 tokens (4096 tiles), tables of 65 entries 904 / 896, four levels 1157 / 1153; 8192 tokens
// 659 / 652, under one table 676 / 654; 12288 tokens 948 / 939, 16384 tokens 1286 / 1286; 8192 tokens x 4096
// channels (32768 tiles) 2551-2573 / 2535-2546; up to 2048 tokens, whose scratch the cache holds anyway, no
// difference.  80 layers x 32768 tokens (83840 tiles, of which it holds a tenth) 6220-6250 / 6240-6350.  Rows
// outermost as well (the quantizer's order, mirrored) is slower: four levels 1186.
bool code_last_first(int64_t ntiles) { return ntiles <= 32768; }

// Tiles up to which the compaction deals a stream's words to four threads (compact_few_kernel): four a
// compute unit.  16 tiles 16.9 -> 8.6 us, 256 tiles 12.2 -> 7.4; at 1024 tiles (32 layers x 1024 channels x
// 1024 tokens) the encode takes 116.3 / 116.0 us, at 768 99.3 / 98.1.
int64_t sliced_compact_blocks() { return (int64_t)compute_units() * 4; }

// Describe the readable byte window [bytes, bytes + nbytes) to the bit reader, which
// loads aligned words at 32-bit offsets from the window's 4-byte-aligned base.
int set_byte_window(DecodeArgs &a, const uint8_t *bytes, int64_t nbytes, const char *what)
{
    if (nbytes <= 0) return fail(CG_ERR_ARG, "%s: empty byte buffer", what);
    const uint32_t skew = (uint32_t)(reinterpret_cast<uintptr_t>(bytes) & 3u);
    a.bytes = bytes - skew;
    a.bytes_skew = skew;
    a.last_word = (skew + nbytes - 1) & ~3ll;
    return CG_OK;
}

size_t decode_few_shmem(int lp) { return (size_t)lp * 64 * sizeof(uint32_t) + (size_t)(kSub + lp) * sizeof(float); }

size_t decode_shmem(int lp, int block) { return align_up((size_t)lp * block * sizeof(uint16_t), 4) + (size_t)(lp + kSub) * sizeof(float); }

size_t decode_float_shmem(int lp, int block) { return (size_t)lp * block * sizeof(uint16_t) + (size_t)(lp + kSub + block / 64) * sizeof(float); }

// Whether a dequantising decode takes the float search (decode_float_kernel): tables of 64 symbols always, of
// 8, 16 and 32 up to twelve wavefronts a SIMD.  It takes fewer cycles a symbol, but more energy, and a large
// decode runs within some 10 to 40 W of this GPU's power limit (1400 W), where the energy is what counts:
// 32 layers x 8192 tokens x 1024 channels 519 us at 2.34 GHz / 546 at 2.19, x 16384 tokens x 4096 channels
// 3822 at 2.26 / 4051 at 2.04.  (Tables of 64 symbols leave room for half the wavefronts, which stay below
// that limit: 1332 W at 2.39 GHz.)  The same for both layouts of the output.  Measured with 32 layers x 1024
// channels, decode_streams_kernel / decode_float_kernel, us:
//   wavefronts a SIMD          4            6            8           12           16           24           32
//   tables of  8 symbols   73 /  67     86 /  82    107 / 105    175 / 172    224 / 220    320 / 322    416 / 423
//             16           88 /  72    104 /  92    128 / 121    204 / 194    263 / 252    368 / 368    479 / 483
//             32          100 /  83    119 / 105    146 / 138    218 / 212    280 / 270    394 / 396    511 / 522
//             64          122 / 101    199 / 171    231 / 212    343 / 319    452 / 407    656 / 590    861 / 773
// On other data (bench.py's four levels of 4096 tokens, sixteen wavefronts) 8, 16, 32 symbols 247 / 252, 271 / 274,
// 285 / 288, 64 symbols 450 / 406: the line is below sixteen.  Calls with symbol output have no such form.
constexpr int64_t kFloatWavefronts = 12;
bool float_search(int64_t rows, int64_t nc, int64_t nsub, int lp)
{
    if (lp == 65) return true;
    return (lp == 9 || lp == 17 || lp == 33) && rows * ceil_div(nc, 64) * nsub <= (int64_t)compute_units() * 4 * kFloatWavefronts;
}

// Tables of 2^k symbols (lp = 2^k + 1) take the kernel with the unrolled search.
template <int BS, int SRC, int OUT>
void launch_decode_log2(const DecodeArgs &a, dim3 grid, size_t shmem, hipStream_t stream, bool flt = false)
{
    const dim3 blk(BS);
    if constexpr (OUT != OUT_SYMBOLS) {
        if (flt) {
            const size_t lds = decode_float_shmem(a.lp, BS);
            switch (a.lp) {
            case 9: decode_float_kernel<BS, 3, SRC, OUT><<<grid, blk, lds, stream>>>(a); return;
            case 17: decode_float_kernel<BS, 4, SRC, OUT><<<grid, blk, lds, stream>>>(a); return;
            case 33: decode_float_kernel<BS, 5, SRC, OUT><<<grid, blk, lds, stream>>>(a); return;
            case 65: decode_float_kernel<BS, 6, SRC, OUT><<<grid, blk, lds, stream>>>(a); return;
            }
        }
    }
    if constexpr (OUT == OUT_SYMBOLS) {
        if (a.lp == 65) {
            decode_streams_kernel<BS, 6, SRC, OUT><<<grid, blk, shmem, stream>>>(a);
            return;
        }
    }
    switch (a.lp) {
    case 9: decode_streams_kernel<BS, 3, SRC, OUT><<<grid, blk, shmem, stream>>>(a); break;
    case 17: decode_streams_kernel<BS, 4, SRC, OUT><<<grid, blk, shmem, stream>>>(a); break;
    case 33: decode_streams_kernel<BS, 5, SRC, OUT><<<grid, blk, shmem, stream>>>(a); break;
    default: decode_streams_kernel<BS, -1, SRC, OUT><<<grid, blk, shmem, stream>>>(a); break;
    }
}

// Whether a decode of these wavefronts is bound by one stream's chain of symbols (decode_few_kernel,
// blocks of 64): tables of 16 and 32 symbols up to three wavefronts a SIMD, of 64 up to two (its tables
// of 32-bit entries take 18 KB of LDS a block, so a third round of blocks would wait for the first).  Measured
// with 32 layers x 1024 channels, the form for more wavefronts (decode_float_kernel; below, decode_streams_kernel
// for one wavefront) / decode_few_kernel, us, one wavefront a SIMD (256 tokens), two, three, four:
//   tables of 32 symbols   93 / 49    67 / 62    81 / 79    82 / 99
//   of 16                  82 / 45    59 / 54    71 / 69    71 / 88
//   of 64                 107 / 55    80 / 74    97 / 129
// Symbol output (rows of 1024 channels, 256 tokens; decode_streams_kernel / decode_few_kernel), where there is no
// float search, by wavefronts a SIMD:
//                          1          2          2.125       2.5         3          3.5         4
//   tables of 16 symbols   77 / 43    81 / 55    90 / 68     89 / 71     90 / 72    99 / 90    101 / 93
//   of 32                  86 / 48    88 / 61    96 / 76     97 / 80     98 / 80   108 / 102   110 / 103
//   of 64                  97 / 53   103 / 73   113 / 115   113 / 131   114 / 141  126 / 174   128 / 179
// The same lines do for both: symbols spread evenly over the alphabet take 89.6 / 86.3 at 3.25 and 90.8 / 96.3 at four for 16.
// Tables of 8 symbols have no instantiation; other lengths search by bisection.
int64_t few_wavefronts_a_simd(int lp) { return lp == 17 || lp == 33 ? 3 : lp == 65 ? 2 : 0; }
bool few_wavefronts(int64_t rows, int64_t nc, int64_t nsub, int lp)
{
    const int64_t most = (int64_t)compute_units() * 4 * few_wavefronts_a_simd(lp);
    const int64_t tiles = ceil_div(nc, 64);
    return rows <= most && tiles <= most && nsub <= most && rows * tiles <= most && rows * tiles * nsub <= most;
}

template <int SRC, int OUT>
void launch_decode_few(const DecodeArgs &a, dim3 grid, size_t shmem, hipStream_t stream)
{
    switch (a.lp) {
    case 17: decode_few_kernel<4, SRC, OUT><<<grid, 64, shmem, stream>>>(a); break;
    case 33: decode_few_kernel<5, SRC, OUT><<<grid, 64, shmem, stream>>>(a); break;
    default: decode_few_kernel<6, SRC, OUT><<<grid, 64, shmem, stream>>>(a); break;
    }
}

template <int SRC>
int launch_decode_symbols(const DecodeArgs &a, int64_t nblocks, int block, bool few, hipStream_t stream)
{
    const dim3 grid = stream_grid(a.sg, nblocks);
    const size_t shmem = few ? decode_few_shmem(a.lp) : decode_shmem(a.lp, block);
    if (few) launch_decode_few<SRC, OUT_SYMBOLS>(a, grid, shmem, stream);
    else CG_DISPATCH_BS(block, (launch_decode_log2<BS, SRC, OUT_SYMBOLS>(a, grid, shmem, stream)));
    return check_launch("decode");
}

// Dequantised output (SRC_OFFSETS, SRC_LISTED): blocks of at most 128 lanes.
template <int SRC>
int launch_decode_kv(DecodeArgs &a, int64_t nblocks, int block, bool few, int out_dt, hipStream_t stream)
{
    const size_t shmem = few ? decode_few_shmem(a.lp) : decode_shmem(a.lp, block);
    const dim3 grid = stream_grid(a.sg, nblocks);
    // the blocks that are resident together at the launch's end (32 wavefronts per compute unit
    // where registers and LDS allow it, which they do for tables of up to 33 entries)
    const int64_t resident = (int64_t)compute_units() * (2048 / block);
    a.last_round_first = (uint32_t)(nblocks > resident ? nblocks - resident : 0);
    const bool flt = !few && float_search(a.sg.rows, a.sg.nc, nblocks / (a.sg.rows * a.sg.ctiles), a.lp);
    if (few) {
        if (out_dt == CG_DT_BF16) launch_decode_few<SRC, OUT_BF16>(a, grid, shmem, stream);
        else launch_decode_few<SRC, OUT_F16>(a, grid, shmem, stream);
    } else if (block == 128) {
        if (out_dt == CG_DT_BF16) launch_decode_log2<128, SRC, OUT_BF16>(a, grid, shmem, stream, flt);
        else launch_decode_log2<128, SRC, OUT_F16>(a, grid, shmem, stream, flt);
    } else {
        if (out_dt == CG_DT_BF16) launch_decode_log2<64, SRC, OUT_BF16>(a, grid, shmem, stream, flt);
        else launch_decode_log2<64, SRC, OUT_F16>(a, grid, shmem, stream, flt);
    }
    return check_launch("decode_kv");
}

// What the dequantising decoder's output has to satisfy, and its part of the arguments.
int set_output(DecodeArgs &a, const char *what, void *out, int out_dt, int64_t H, int64_t D, int64_t ol, int64_t okv, int64_t ot, int64_t oh)
{
    if (int rc = check_dt(out_dt, what)) return rc;
    if (D > INT_MAX) return fail(CG_ERR_ARG, "%s: head size too large", what);
    // the kernel stores through a buffer descriptor per block: a channel's byte offset plus a
    // token row's byte offset inside one stream's token range must fit 32 bits
    if (ot < 0 || oh < 0 || ((H - 1) * oh + (D - 1) + (int64_t)(kSub - 1) * ot) * 2 + 2 > 0xFFFFFFFFll)
        return fail(CG_ERR_ARG, "%s: negative output strides, or %d token rows of one layer's keys or values "
                                "span 4 GiB or more", what, kSub);
    a.out_kv = static_cast<uint16_t *>(out);
    a.ol = ol;
    a.okv = okv;
    a.ot = ot;
    a.oh = oh;
    a.D = (int32_t)D;
    return CG_OK;
}

// two wavefronts per block: a block's slot is held until its slowest wavefront is through
// its 256 symbols, and smaller blocks leave fewer finished wavefronts waiting for that
// (one wavefront per block loses more to the per-block set-up than it gains)
int decode_kv_block(int64_t C, int lp)
{
    const int block = pick_block(C, lp);
    return block > 128 ? 128 : block;
}

}  // namespace
