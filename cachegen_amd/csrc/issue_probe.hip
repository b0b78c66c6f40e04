// Calibration probe of the CacheGen KV codec library for MI355X (gfx950): how fast one SIMD
// issues vector instructions, and at which engine clock.  Not part of the codec: bench.py uses it
// to price the decoder's instruction count against what this GPU really issues, at the clock it
// really runs at, instead of against 4 cycles per instruction at the data-sheet clock.
//
// The two range coders are bound by the issue of vector instructions.  On this GPU a wave64
// instruction takes a SIMD 4 cycles, except that adds, subtracts, bitwise operations, right
// shifts, moves and float32 add/multiply take 2 when their operands are registers (no scalar
// register, SDWA or DPP operand).  The probe measures both classes, and a sequence with the
// decoder's own mix and order of instructions, with 8 wavefronts per SIMD and two independent
// dependency chains per wavefront, and reads the engine clock from inside the kernel (the shader
// clock counter against the constant 100 MHz counter).
//
// The second half takes single instructions: two of them in turn on full SIMDs (whether they issue
// beside each other, and, read beside the card's power, what each costs), and chains of dependent ones in a
// wavefront that is alone on its compute unit (what a call of few wavefronts waits for).  What the instructions compute is of no
// account there: a select may read a mask sooner than it may be relied on.
#include <hip/hip_runtime.h>

#include <cstdint>

extern "C" {

// kind: 0 = cheap class (v_add_u32, v_xor_b32, v_lshrrev_b32, v_and_b32 in turn)
//       1 = full-rate class (v_mul_u32_u24, v_cndmask_b32, v_lshlrev_b32, v_add3_u32 in turn)
//       2 = one decoded symbol of decode_streams_kernel (rows of at most 16 levels): 23 instructions
//           of the full class and 12 of the cheap class in the order the compiler emits them
// iters: loop trips of 64 (kinds 0, 1) or 70 (kind 2: two symbols of 35) instructions per wavefront
// ns_per_instruction: time one SIMD takes per wave64 instruction, 8 wavefronts resident
// clock_mhz: engine clock while the probe ran
// Returns 0, or the hipError_t that stopped it.
int cg_probe_issue_rate(int kind, int iters, double *ns_per_instruction, double *clock_mhz);

// The engine clock averaged over about `microseconds` of wall time, sampled by ONE wavefront that
// idles between two readings: launched on `stream` next to other work (a side stream of the
// benchmark), it reports the clock the GPU ran at while that work was running.  The result is
// read with cg_probe_clock_result after the stream has been synchronized.
int cg_probe_clock_start(int microseconds, void *stream);
int cg_probe_clock_result(double *clock_mhz, double *window_us);

// Instructions of the probe, numbered from 0; null past the last.
const char *cg_probe_op(int op);
// Launches `launches` kernels of `iters` trips of 32 pairs "a a b b" on the null stream: full SIMDs.
int cg_probe_pair_start(int a, int b, int iters, int launches);
// Waits for them: ns a SIMD took for an instruction, the engine clock of the last launch.
int cg_probe_pair_wait(double *ns_per_instruction, double *clock_mhz);
// Chains of one wavefront alone on its compute unit, numbered from 0; null past the last.
const char *cg_probe_chain(int chain);
// Cycles of a link of the chain.
int cg_probe_chain_cycles(int chain, double *cycles);
// PCI address of the current device, for the card's own power reading (at least 16 bytes).
int cg_probe_pci(char *address, int size);

}  // extern "C"

namespace {

struct ClockSample {
    uint64_t cycles0, ticks0, cycles1, ticks1;      // shader clock counter, 100 MHz counter
};

__device__ __forceinline__ void read_clocks(uint64_t &cycles, uint64_t &ticks)
{
    cycles = clock64();
    ticks = wall_clock64();
}

template <int KIND>
__global__ __launch_bounds__(256) void issue_rate_kernel(uint32_t *sink, ClockSample *sample, int iters, uint32_t seed)
{
    uint32_t a = threadIdx.x + seed, b = (blockIdx.x * 3 + 1) & 15, c = seed ^ 0x1234567u, d = a * 7 + 1;
    uint64_t w = ((uint64_t)a << 32) | b, w2 = ((uint64_t)c << 32) | d;
    uint64_t cycles0 = 0, ticks0 = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) read_clocks(cycles0, ticks0);
    for (int i = 0; i < iters; ++i) {
        if (KIND == 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                asm volatile("v_add_u32 %0, %0, %2\n\tv_add_u32 %1, %1, %2\n\t"
                             "v_xor_b32 %0, %0, %3\n\tv_xor_b32 %1, %1, %3\n\t"
                             "v_lshrrev_b32 %0, 1, %0\n\tv_lshrrev_b32 %1, 1, %1\n\t"
                             "v_and_b32 %0, %0, %3\n\tv_and_b32 %1, %1, %3"
                             : "+v"(a), "+v"(c) : "v"(b), "v"(d));
        } else if (KIND == 1) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                asm volatile("v_mul_u32_u24 %0, %0, %2\n\tv_mul_u32_u24 %1, %1, %2\n\t"
                             "v_cndmask_b32 %0, %0, %3, vcc\n\tv_cndmask_b32 %1, %1, %3, vcc\n\t"
                             "v_lshlrev_b32 %0, 1, %0\n\tv_lshlrev_b32 %1, 1, %1\n\t"
                             "v_add3_u32 %0, %0, %2, %3\n\tv_add3_u32 %1, %1, %2, %3"
                             : "+v"(a), "+v"(c) : "v"(b), "v"(d) : "vcc");
        } else {
            // the symbol loop of decode_streams_kernel<128, 5, OFFSETS, F16>, rows of at most 16
            // levels, as compiled: search (two probes on registers, two on table entries), bounds
            // and the one test, dequantisation, state update, bit window, and the wait states before a mask is read;
            // LDS reads and the store left out (they are not vector-ALU instructions); twice, on two sets of registers
#define CG_PROBE_SYMBOL(x, y, p, q)                                                         \
            "v_mul_u32_u24 " p ", " x ", %8\n\tv_cmp_gt_u32 vcc, " p ", " y "\n\t"              \
            "s_nop 1\n\tv_cndmask_b32 " q ", %8, %9, vcc\n\tv_cndmask_b32 " p ", %9, %8, vcc\n\t" \
            "v_mul_u32_u24 " q ", " q ", " x "\n\tv_cmp_gt_u32 vcc, " q ", " y "\n\t"           \
            "v_add_u32 " q ", 0x410, " p "\n\ts_nop 0\n\tv_cndmask_b32 " p ", " q ", " p ", vcc\n\t" \
            "v_add_u32 " q ", 0x208, " p "\n\tv_mul_u32_u24 " p ", " x ", " p "\n\t"            \
            "v_cmp_gt_u32 vcc, " p ", " y "\n\ts_nop 1\n\tv_cndmask_b32 " p ", " q ", " p ", vcc\n\t" \
            "v_add_u32 " q ", 0x104, " p "\n\tv_mul_u32_u24 " p ", " x ", " p "\n\t"            \
            "v_cmp_gt_u32 vcc, " p ", " y "\n\ts_nop 1\n\tv_cndmask_b32 " p ", " q ", " p ", vcc\n\t" \
            "v_add_u32 " q ", " p ", %9\n\t"                                                    \
            "v_mul_hi_u32 " p ", " p ", " x "\n\tv_mul_hi_u32 " q ", " q ", " x "\n\t"          \
            "v_sub_u32 " q ", " q ", " p "\n\tv_sub_u32 " y ", " y ", " p "\n\t"                \
            "v_cmp_ge_u32 vcc, " y ", " q "\n\t"                                                \
            "v_mul_f32 " p ", " p ", " q "\n\tv_cvt_f16_f32 " p ", " p "\n\t"                   \
            "v_add_u32 " p ", " p ", " x "\n\tv_add_u32 " q ", -1, " q "\n\t"                   \
            "v_add_u32 " y ", " p ", " q "\n\tv_bitop3_b32 " y ", " q ", " p ", " y " bitop3:0x90\n\t" \
            "v_lshl_or_b32 " q ", " y ", 1, " q "\n\tv_ffbh_u32 " q ", " q "\n\t"               \
            "v_sub_co_u32 " p ", vcc, " p ", " q "\n\tv_mov_b32 " y ", " p "\n\t"
            uint32_t t0 = a, t1 = c, t2 = b, t3 = d;
            asm volatile(CG_PROBE_SYMBOL("%0", "%1", "%4", "%5")
                         "v_lshlrev_b64 %2, %5, %2\n\tv_lshlrev_b64 %3, %5, %3\n\tv_lshlrev_b64 %2, %5, %2\n\t"
                         CG_PROBE_SYMBOL("%1", "%0", "%6", "%7")
                         "v_lshlrev_b64 %2, %7, %2\n\tv_lshlrev_b64 %3, %7, %3\n\tv_lshlrev_b64 %2, %7, %2"
                         : "+v"(a), "+v"(c), "+v"(w), "+v"(w2), "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3)
                         : "v"(b), "v"(d)
                         : "vcc");
#undef CG_PROBE_SYMBOL
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sample->cycles0 = cycles0;
        sample->ticks0 = ticks0;
        read_clocks(sample->cycles1, sample->ticks1);
    }
    sink[blockIdx.x * 256 + threadIdx.x] = a + c + d + (uint32_t)w + (uint32_t)(w >> 32) + (uint32_t)w2 + (uint32_t)(w2 >> 32);
}

// One wavefront that sleeps between two readings of the clocks, for about `ticks` ticks of the
// 100 MHz counter; bounded by that counter, so it always ends.
__global__ __launch_bounds__(64) void clock_window_kernel(ClockSample *sample, uint64_t ticks)
{
    uint64_t cycles0, ticks0, cycles1, ticks1;
    read_clocks(cycles0, ticks0);
    do {
        __builtin_amdgcn_s_sleep(64);
        read_clocks(cycles1, ticks1);
    } while (ticks1 - ticks0 < ticks);
    if (threadIdx.x == 0) {
        sample->cycles0 = cycles0;
        sample->ticks0 = ticks0;
        sample->cycles1 = cycles1;
        sample->ticks1 = ticks1;
    }
}

ClockSample *g_window = nullptr;        // the sampler's result, device memory kept for the process

}  // namespace

#define CG_PROBE_CHECK(x)                  \
    do {                                   \
        const hipError_t e_ = (x);         \
        if (e_ != hipSuccess) return (int)e_; \
    } while (0)

extern "C" int cg_probe_issue_rate(int kind, int iters, double *ns_per_instruction, double *clock_mhz)
{
    if (kind < 0 || kind > 2 || iters <= 0 || !ns_per_instruction || !clock_mhz) return (int)hipErrorInvalidValue;
    int dev = 0, cus = 0;
    CG_PROBE_CHECK(hipGetDevice(&dev));
    CG_PROBE_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int blocks = cus * 8 * 4;          // 8 blocks of 4 wavefronts per compute unit, 4 rounds
    uint32_t *sink = nullptr;
    ClockSample *sample = nullptr;
    CG_PROBE_CHECK(hipMalloc(&sink, (size_t)blocks * 256 * sizeof(uint32_t)));
    CG_PROBE_CHECK(hipMalloc(&sample, sizeof(ClockSample)));
    hipEvent_t e0, e1;
    CG_PROBE_CHECK(hipEventCreate(&e0));
    CG_PROBE_CHECK(hipEventCreate(&e1));
    float ms = 0.0f;
    for (int rep = 0; rep < 2; ++rep) {      // the first run brings the clock up
        CG_PROBE_CHECK(hipEventRecord(e0, nullptr));
        if (kind == 0) issue_rate_kernel<0><<<blocks, 256>>>(sink, sample, iters, rep + 1);
        else if (kind == 1) issue_rate_kernel<1><<<blocks, 256>>>(sink, sample, iters, rep + 1);
        else issue_rate_kernel<2><<<blocks, 256>>>(sink, sample, iters, rep + 1);
        CG_PROBE_CHECK(hipGetLastError());
        CG_PROBE_CHECK(hipEventRecord(e1, nullptr));
        CG_PROBE_CHECK(hipDeviceSynchronize());
        CG_PROBE_CHECK(hipEventElapsedTime(&ms, e0, e1));
    }
    ClockSample host;
    CG_PROBE_CHECK(hipMemcpy(&host, sample, sizeof(host), hipMemcpyDeviceToHost));
    CG_PROBE_CHECK(hipFree(sink));
    CG_PROBE_CHECK(hipFree(sample));
    CG_PROBE_CHECK(hipEventDestroy(e0));
    CG_PROBE_CHECK(hipEventDestroy(e1));
    const double per_trip = kind == 2 ? 70.0 : 64.0;     // instructions per loop trip and wavefront
    const double per_simd = (double)blocks * 4.0 * iters * per_trip / (cus * 4.0);
    *ns_per_instruction = (double)ms * 1e6 / per_simd;
    const double ticks = (double)(host.ticks1 - host.ticks0);
    *clock_mhz = ticks > 0 ? (double)(host.cycles1 - host.cycles0) / ticks * 100.0 : 0.0;
    return 0;
}

extern "C" int cg_probe_clock_start(int microseconds, void *stream)
{
    if (microseconds <= 0 || microseconds > 10 * 1000 * 1000) return (int)hipErrorInvalidValue;
    if (!g_window) CG_PROBE_CHECK(hipMalloc(&g_window, sizeof(ClockSample)));
    clock_window_kernel<<<1, 64, 0, static_cast<hipStream_t>(stream)>>>(g_window, (uint64_t)microseconds * 100u);
    return (int)hipGetLastError();
}

extern "C" int cg_probe_clock_result(double *clock_mhz, double *window_us)
{
    if (!g_window || !clock_mhz || !window_us) return (int)hipErrorInvalidValue;
    ClockSample host;
    CG_PROBE_CHECK(hipMemcpy(&host, g_window, sizeof(host), hipMemcpyDeviceToHost));
    const double ticks = (double)(host.ticks1 - host.ticks0);
    *window_us = ticks / 100.0;
    *clock_mhz = ticks > 0 ? (double)(host.cycles1 - host.cycles0) / ticks * 100.0 : 0.0;
    return 0;
}

namespace {

// The probe's instructions: d and w are the results, of 32 and 64 bits, a b f q two sets of operands that no
// instruction writes; %8 and %10 are operands of both sets, %14 an LDS address, %15 a shift count.
#define CG_ASM_s_nop(d, w, a, b, f, q) "s_nop 0\n\t"
#define CG_ASM_v_add_u32(d, w, a, b, f, q) "v_add_u32 " d ", " a ", " b "\n\t"
#define CG_ASM_v_xor_b32(d, w, a, b, f, q) "v_xor_b32 " d ", " a ", " b "\n\t"
#define CG_ASM_v_lshrrev_b32(d, w, a, b, f, q) "v_lshrrev_b32 " d ", 6, " a "\n\t"
#define CG_ASM_v_ashrrev_i32(d, w, a, b, f, q) "v_ashrrev_i32 " d ", 31, " a "\n\t"
#define CG_ASM_v_bitop3_b32(d, w, a, b, f, q) "v_bitop3_b32 " d ", " a ", " b ", %8 bitop3:0xca\n\t"
#define CG_ASM_v_mov_b32(d, w, a, b, f, q) "v_mov_b32 " d ", " a "\n\t"
#define CG_ASM_v_add_f32(d, w, a, b, f, q) "v_add_f32 " d ", " f ", %10\n\t"
#define CG_ASM_v_mul_f32(d, w, a, b, f, q) "v_mul_f32 " d ", " f ", %10\n\t"
#define CG_ASM_v_fma_f32(d, w, a, b, f, q) "v_fma_f32 " d ", " f ", %10, -%8\n\t"
#define CG_ASM_v_cndmask_b32(d, w, a, b, f, q) "v_cndmask_b32_e64 " d ", " a ", " b ", vcc\n\t"
#define CG_ASM_v_sub_co_u32(d, w, a, b, f, q) "v_sub_co_u32 " d ", vcc, " a ", " b "\n\t"
#define CG_ASM_v_cmp_gt_u32(d, w, a, b, f, q) "v_cmp_gt_u32 vcc, " a ", " b "\n\t"
#define CG_ASM_v_lshlrev_b32(d, w, a, b, f, q) "v_lshlrev_b32 " d ", 6, " a "\n\t"
#define CG_ASM_v_add3_u32(d, w, a, b, f, q) "v_add3_u32 " d ", " a ", " b ", %8\n\t"
#define CG_ASM_v_lshl_or_b32(d, w, a, b, f, q) "v_lshl_or_b32 " d ", " a ", 1, " b "\n\t"
#define CG_ASM_v_ffbh_u32(d, w, a, b, f, q) "v_ffbh_u32 " d ", " a "\n\t"
#define CG_ASM_v_cvt_f32_u32(d, w, a, b, f, q) "v_cvt_f32_u32 " d ", " a "\n\t"
#define CG_ASM_v_mul_hi_u32(d, w, a, b, f, q) "v_mul_hi_u32 " d ", " a ", " b "\n\t"
#define CG_ASM_v_lshlrev_b64(d, w, a, b, f, q) "v_lshlrev_b64 " w ", %15, " q "\n\t"
#define CG_ASM_v_mad_u64_u32(d, w, a, b, f, q) "v_mad_u64_u32 " w ", vcc, " a ", " b ", " q "\n\t"
#define CG_ASM_v_mul_u32_u24(d, w, a, b, f, q) "v_mul_u32_u24 " d ", " a ", " b "\n\t"
#define CG_ASM_ds_read_u16(d, w, a, b, f, q) "ds_read_u16 " d ", %14\n\t"
#define CG_PROBE_OPS(X) \
    X(s_nop) X(v_add_u32) X(v_xor_b32) X(v_lshrrev_b32) X(v_ashrrev_i32) X(v_bitop3_b32) X(v_mov_b32) X(v_add_f32) X(v_mul_f32) X(v_fma_f32) \
    X(v_cndmask_b32) X(v_sub_co_u32) X(v_cmp_gt_u32) X(v_lshlrev_b32) X(v_add3_u32) X(v_lshl_or_b32) X(v_ffbh_u32) X(v_cvt_f32_u32) \
    X(v_mul_hi_u32) X(v_lshlrev_b64) X(v_mad_u64_u32) X(v_mul_u32_u24) X(ds_read_u16)
// the same list beside another instruction
#define CG_PROBE_BESIDE(X, a) \
    X(a, s_nop) X(a, v_add_u32) X(a, v_xor_b32) X(a, v_lshrrev_b32) X(a, v_ashrrev_i32) X(a, v_bitop3_b32) X(a, v_mov_b32) X(a, v_add_f32) \
    X(a, v_mul_f32) X(a, v_fma_f32) X(a, v_cndmask_b32) X(a, v_sub_co_u32) X(a, v_cmp_gt_u32) X(a, v_lshlrev_b32) X(a, v_add3_u32) \
    X(a, v_lshl_or_b32) X(a, v_ffbh_u32) X(a, v_cvt_f32_u32) X(a, v_mul_hi_u32) X(a, v_lshlrev_b64) X(a, v_mad_u64_u32) X(a, v_mul_u32_u24) \
    X(a, ds_read_u16)
#define CG_PROBE_NUMBER(name) OP_##name,
enum { CG_PROBE_OPS(CG_PROBE_NUMBER) kOps };

struct Operands {
    uint32_t a, b, c, e, lds, count;
    float f, g, h, k;
    uint64_t q, r;
};

struct Results {
    uint32_t d0, d1;
    uint64_t w0, w1;
};

// 32 pairs in one statement: between two the compiler sets s_nop
template <int A, int B> __device__ void issue(Results &r, const Operands &o);
#define CG_FIRST(OP) OP("%0", "%2", "%4", "%5", "%9", "%12")
#define CG_SECOND(OP) OP("%1", "%3", "%6", "%7", "%11", "%13")
#define CG_FOUR(A, B) CG_FIRST(A) CG_SECOND(A) CG_SECOND(B) CG_FIRST(B)
#define CG_SIXTEEN(A, B) CG_FOUR(A, B) CG_FOUR(A, B) CG_FOUR(A, B) CG_FOUR(A, B)
#define CG_PROBE_PAIR(x, y)                                                                                                        \
    template <> __device__ __forceinline__ void issue<OP_##x, OP_##y>(Results &r, const Operands &o)                             \
    {                                                                                                                              \
        asm volatile(CG_SIXTEEN(CG_ASM_##x, CG_ASM_##y) CG_SIXTEEN(CG_ASM_##x, CG_ASM_##y) CG_SIXTEEN(CG_ASM_##x, CG_ASM_##y)    \
                     CG_SIXTEEN(CG_ASM_##x, CG_ASM_##y) "s_waitcnt lgkmcnt(0)"                                                    \
                     : "+v"(r.d0), "+v"(r.d1), "+v"(r.w0), "+v"(r.w1)                                                             \
                     : "v"(o.a), "v"(o.b), "v"(o.c), "v"(o.e), "v"(o.k), "v"(o.f), "v"(o.g), "v"(o.h), "v"(o.q), "v"(o.r),        \
                       "v"(o.lds), "v"(o.count)                                                                                    \
                     : "vcc", "memory");                                                                                           \
    }
#define CG_PROBE_ROW(x) CG_PROBE_BESIDE(CG_PROBE_PAIR, x)
CG_PROBE_OPS(CG_PROBE_ROW)

__device__ __forceinline__ uint32_t scrambled(uint32_t &h)
{
    h ^= h << 13;
    h ^= h >> 17;
    h ^= h << 5;
    return h;
}

template <int A, int B>
__global__ __launch_bounds__(256) void pair_kernel(uint32_t *sink, ClockSample *sample, int iters, uint32_t seed)
{
    __shared__ uint32_t table[1024];
    for (int i = threadIdx.x; i < 1024; i += 256) table[i] = i * 2654435761u;
    __syncthreads();
    uint32_t h = (threadIdx.x + blockIdx.x * 256 + seed) * 2654435761u | 1u;
    Operands o;
    o.a = scrambled(h), o.b = scrambled(h), o.c = scrambled(h), o.e = scrambled(h);
    o.f = (float)scrambled(h), o.g = (float)scrambled(h) * 0x1p-32f, o.h = (float)scrambled(h), o.k = (float)scrambled(h);
    o.q = (uint64_t)scrambled(h) << 32 | scrambled(h), o.r = (uint64_t)scrambled(h) << 32 | scrambled(h);
    o.lds = (scrambled(h) & 15u) * 256u + (threadIdx.x & 63u) * 4u;            // inside the table: no two lanes of one word
    o.count = scrambled(h) & 3u;
    Results r = {0, 0, 0, 0};
    uint64_t cycles0 = 0, ticks0 = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) read_clocks(cycles0, ticks0);
    for (int i = 0; i < iters; ++i) issue<A, B>(r, o);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sample->cycles0 = cycles0;
        sample->ticks0 = ticks0;
        read_clocks(sample->cycles1, sample->ticks1);
    }
    sink[blockIdx.x * 256 + threadIdx.x] = r.d0 + r.d1 + (uint32_t)r.w0 + (uint32_t)(r.w0 >> 32) + (uint32_t)r.w1 + (uint32_t)(r.w1 >> 32);
}

typedef void (*PairKernel)(uint32_t *, ClockSample *, int, uint32_t);

// a <= b
template <int A, int B>
PairKernel pick_pair(int a, int b)
{
    if (a == A && b == B) return pair_kernel<A, B>;
    if constexpr (B + 1 < kOps) return pick_pair<A, B + 1>(a, b);
    else if constexpr (A + 1 < kOps) return pick_pair<A + 1, A + 1>(a, b);
    else return nullptr;
}

// ---- one wavefront alone ------------------------------------------------------------------
enum { CHAIN_ADD, CHAIN_BITOP3, CHAIN_MUL_HI, CHAIN_SHIFT64, CHAIN_LDS, CHAIN_SCALAR_BRANCH, CHAIN_MASK_BRANCH, kChains };

constexpr int kLinks = 64;          // a trip

template <int CHAIN>
__global__ __launch_bounds__(64) void chain_kernel(uint32_t *sink, ClockSample *sample, int iters, uint32_t seed)
{
    __shared__ uint32_t table[64];
    table[threadIdx.x] = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)&table[threadIdx.x];      // every word holds its own address
    __syncthreads();
    uint32_t a = table[threadIdx.x], b = a + seed, one = 1;
    const uint32_t c = seed * 7u + 3u;
    uint64_t w = b;
    const uint64_t cycles0 = clock64();
#define CG_LINKS16(text) text text text text text text text text text text text text text text text text
#define CG_LINKS(text) CG_LINKS16(text) CG_LINKS16(text) CG_LINKS16(text) CG_LINKS16(text)
    for (int i = 0; i < iters; ++i) {
        if (CHAIN == CHAIN_ADD) asm volatile(CG_LINKS("v_add_u32 %0, %0, %1\n\t") : "+v"(b) : "v"(c));
        if (CHAIN == CHAIN_BITOP3) asm volatile(CG_LINKS("v_bitop3_b32 %0, %0, %1, %2 bitop3:0xca\n\t") : "+v"(b) : "v"(c), "v"(one));
        if (CHAIN == CHAIN_MUL_HI) asm volatile(CG_LINKS("v_mul_hi_u32 %0, %0, %1\n\t") : "+v"(b) : "v"(c));
        if (CHAIN == CHAIN_SHIFT64) asm volatile(CG_LINKS("v_lshlrev_b64 %0, %1, %0\n\t") : "+v"(w) : "v"(one));
        if (CHAIN == CHAIN_LDS) asm volatile(CG_LINKS("ds_read_b32 %0, %0\n\ts_waitcnt lgkmcnt(0)\n\t") : "+v"(a) : : "memory");
        // branches to the next instruction, whichever way they go
#pragma unroll
        for (int j = 0; j < kLinks; ++j) {
            if (CHAIN == CHAIN_SCALAR_BRANCH) asm volatile("s_cmp_eq_u32 %0, 0\n\ts_cbranch_scc1 L%=\n\tL%=:" : : "s"(seed) : "scc");
            if (CHAIN == CHAIN_MASK_BRANCH) asm volatile("v_cmp_eq_u32 vcc, 0, %0\n\ts_cbranch_vccnz L%=\n\tL%=:" : : "v"(one) : "vcc");
        }
    }
#undef CG_LINKS
#undef CG_LINKS16
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sample->cycles0 = cycles0;
        sample->cycles1 = clock64();
    }
    sink[blockIdx.x * 64 + threadIdx.x] = a + b + one + (uint32_t)w + (uint32_t)(w >> 32);
}

struct PairRun {
    uint32_t *sink;
    ClockSample *sample;
    hipEvent_t e0, e1;
    double per_simd;            // instructions of all launches a SIMD
};
PairRun g_pair = {};

}  // namespace

extern "C" const char *cg_probe_op(int op)
{
#define CG_PROBE_NAME(name) #name,
    static const char *const names[] = {CG_PROBE_OPS(CG_PROBE_NAME)};
    return op >= 0 && op < kOps ? names[op] : nullptr;
}

extern "C" int cg_probe_pair_start(int a, int b, int iters, int launches)
{
    if (a < 0 || b < 0 || a >= kOps || b >= kOps || iters <= 0 || launches <= 0) return (int)hipErrorInvalidValue;
    const PairKernel kernel = a <= b ? pick_pair<0, 0>(a, b) : pick_pair<0, 0>(b, a);
    int dev = 0, cus = 0;
    CG_PROBE_CHECK(hipGetDevice(&dev));
    CG_PROBE_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int blocks = cus * 8 * 4;          // 8 blocks of 4 wavefronts per compute unit, 4 rounds
    if (!g_pair.sink) {
        CG_PROBE_CHECK(hipMalloc(&g_pair.sink, (size_t)blocks * 256 * sizeof(uint32_t)));
        CG_PROBE_CHECK(hipMalloc(&g_pair.sample, sizeof(ClockSample)));
        CG_PROBE_CHECK(hipEventCreate(&g_pair.e0));
        CG_PROBE_CHECK(hipEventCreate(&g_pair.e1));
    }
    g_pair.per_simd = (double)blocks * 4.0 * iters * 64.0 * launches / (cus * 4.0);
    CG_PROBE_CHECK(hipEventRecord(g_pair.e0, nullptr));
    for (int i = 0; i < launches; ++i) kernel<<<blocks, 256>>>(g_pair.sink, g_pair.sample, iters, (uint32_t)i + 1);
    CG_PROBE_CHECK(hipGetLastError());
    return (int)hipEventRecord(g_pair.e1, nullptr);
}

extern "C" int cg_probe_pair_wait(double *ns_per_instruction, double *clock_mhz)
{
    if (!g_pair.sink || !ns_per_instruction || !clock_mhz) return (int)hipErrorInvalidValue;
    float ms = 0.0f;
    ClockSample host;
    CG_PROBE_CHECK(hipEventSynchronize(g_pair.e1));
    CG_PROBE_CHECK(hipEventElapsedTime(&ms, g_pair.e0, g_pair.e1));
    CG_PROBE_CHECK(hipMemcpy(&host, g_pair.sample, sizeof(host), hipMemcpyDeviceToHost));
    *ns_per_instruction = (double)ms * 1e6 / g_pair.per_simd;
    const double ticks = (double)(host.ticks1 - host.ticks0);
    *clock_mhz = ticks > 0 ? (double)(host.cycles1 - host.cycles0) / ticks * 100.0 : 0.0;
    return 0;
}

extern "C" const char *cg_probe_chain(int chain)
{
    static const char *const names[] = {"v_add_u32 (32-bit encoding)", "v_bitop3_b32 (64-bit encoding)", "v_mul_hi_u32", "v_lshlrev_b64", "ds_read_b32 and its wait",
                                        "s_cmp and a branch on it", "v_cmp and a branch on its mask"};
    return chain >= 0 && chain < kChains ? names[chain] : nullptr;
}

extern "C" int cg_probe_chain_cycles(int chain, double *cycles)
{
    if (chain < 0 || chain >= kChains || !cycles) return (int)hipErrorInvalidValue;
    static void (*const kernels[])(uint32_t *, ClockSample *, int, uint32_t) = {
        chain_kernel<CHAIN_ADD>, chain_kernel<CHAIN_BITOP3>, chain_kernel<CHAIN_MUL_HI>, chain_kernel<CHAIN_SHIFT64>, chain_kernel<CHAIN_LDS>,
        chain_kernel<CHAIN_SCALAR_BRANCH>, chain_kernel<CHAIN_MASK_BRANCH>};
    constexpr int kBlocks = 64, kIters = 100;          // far fewer blocks than compute units: each has one to itself
    uint32_t *sink = nullptr;
    ClockSample *sample = nullptr, host;
    CG_PROBE_CHECK(hipMalloc(&sink, (size_t)kBlocks * 64 * sizeof(uint32_t)));
    CG_PROBE_CHECK(hipMalloc(&sample, sizeof(ClockSample)));
    for (int rep = 0; rep < 3; ++rep) kernels[chain]<<<kBlocks, 64>>>(sink, sample, kIters, (uint32_t)rep + 1);
    CG_PROBE_CHECK(hipGetLastError());
    CG_PROBE_CHECK(hipMemcpy(&host, sample, sizeof(host), hipMemcpyDeviceToHost));
    CG_PROBE_CHECK(hipFree(sink));
    CG_PROBE_CHECK(hipFree(sample));
    *cycles = (double)(host.cycles1 - host.cycles0) / ((double)kIters * kLinks);
    return 0;
}

extern "C" int cg_probe_pci(char *address, int size)
{
    int dev = 0;
    if (!address || size < 16) return (int)hipErrorInvalidValue;
    CG_PROBE_CHECK(hipGetDevice(&dev));
    return (int)hipDeviceGetPCIBusId(address, size, dev);
}
