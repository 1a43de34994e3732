// Decode kernels for gfx950 (MI355X), behind the launcher names of the reference's
// src/kernels.cuh. Wave64 throughout: a GEMV row is one wave whose lanes stream 16-byte chunks
// (global_load_dwordx4, non-temporal for weights and the KV cache) and meet in an xor-butterfly
// tree; RMSNorm rows up to 8192 wide are one wave held in registers; a RoPE head is a group of
// D/16 lanes that each hold the chunk [8L, 8L+8) and its rotation partner [D/2+8L, ...), so the
// rotation is lane-local. Arithmetic is fp32 with bf16 stores at the reference's rounding points
// (src/kernels.cu), in the summation orders the CPU oracle restates.
#include <limits.h>
#include <math.h>
#include <stdarg.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include "common.h"
#include "internal.h"
#include "rope.h"

using namespace llm;

// ------------------------------------------------------------------------------------------
// error handling (src/common.cuh:11-22 semantics, switchable to recording)
// ------------------------------------------------------------------------------------------

static int g_exit_on_error = 1;
static thread_local char g_err[1024];
static thread_local bool g_has_err = false;

bool llm_fail(const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (g_exit_on_error) {
        fprintf(stderr, "%s\n", buf);
        exit(EXIT_FAILURE);
    }
    if (!g_has_err) {  // keep the first error until it is cleared
        strncpy(g_err, buf, sizeof g_err - 1);
        g_err[sizeof g_err - 1] = 0;
        g_has_err = true;
    }
    return false;
}

bool llm_has_error() { return g_has_err; }

extern "C" int llm_set_exit_on_error(int enable) {
    int old = g_exit_on_error;
    g_exit_on_error = enable ? 1 : 0;
    return old;
}
extern "C" const char *llm_last_error(void) { return g_has_err ? g_err : nullptr; }
extern "C" void llm_clear_error(void) {
    g_has_err = false;
    g_err[0] = 0;
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// ------------------------------------------------------------------------------------------
// embedding (src/kernels.cu:7-23)
// ------------------------------------------------------------------------------------------

// One workgroup copies the row in 16-byte chunks. With vocab > 0 a token outside [0, vocab)
// sets *err and copies nothing (the step uses this for tokens fed back on the device).
__global__ __launch_bounds__(256) void embedding_kernel(bf16 *out, const bf16 *table,
                                                        const int *d_token, int hidden, int vocab,
                                                        int *err) {
    const int token = *d_token;
    if (vocab > 0 && (token < 0 || token >= vocab)) {
        if (err && threadIdx.x == 0) *err = 1;
        return;
    }
    const bf16 *row = table + (size_t)token * hidden;
    if ((hidden & 7) == 0) {
        for (int c = threadIdx.x; c < hidden / 8; c += blockDim.x) st16(out + 8 * c, ld16(row + 8 * c));
    } else {
        for (int i = threadIdx.x; i < hidden; i += blockDim.x) out[i] = row[i];
    }
}

static void launch_embedding(bf16 *out, const bf16 *table, const int *d_token, int hidden,
                             int vocab, int *err, hipStream_t stream) {
    if (hidden <= 0) {
        llm_fail("embedding: hidden %d must be positive", hidden);
        return;
    }
    if ((hidden & 7) == 0 && (!aligned16(out) || !aligned16(table))) {
        llm_fail("embedding: out and table must be 16-byte aligned");
        return;
    }
    embedding_kernel<<<1, 256, 0, stream>>>(out, table, d_token, hidden, vocab, err);
    LAUNCH_OK();
}

extern "C" void embedding_forward(bf16 *out, const bf16 *table, const int *d_token, int hidden,
                                  hipStream_t stream) {
    launch_embedding(out, table, d_token, hidden, 0, nullptr, stream);
}

// Used by the step for device-fed tokens.
void embedding_checked(bf16 *out, const bf16 *table, const int *d_token, int hidden, int vocab,
                       int *err, hipStream_t stream) {
    launch_embedding(out, table, d_token, hidden, vocab, err, stream);
}

// ------------------------------------------------------------------------------------------
// RMSNorm (src/kernels.cu:25-71)
// ------------------------------------------------------------------------------------------

// One wave per row, the row in registers: lane l holds chunks l, l+64, ... (NC of them).
// sum of squares: per-lane fma in chunk/element order, then the wave tree. The row, its output
// and the weights are buffers: chunks past the end read as zeros and are not written, with no
// branch around the loads and stores (with per-chunk bounds branches and plain loads the
// 4096 x 2560 sweep took 10.5 us instead of 7.3; two or four rows per wave with the next row
// requested early measured slower still).
template <int NC>
__global__ __launch_bounds__(256) void rmsnorm_wave_kernel(bf16 *out, const bf16 *in,
                                                           const bf16 *weight, int rows, int dim,
                                                           float eps) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= rows) return;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(in + (size_t)row * dim), (short)0, dim * 2, BUFFER_FLAGS);
    const __amdgpu_buffer_rsrc_t wr =
        __builtin_amdgcn_make_buffer_rsrc((void *)weight, (short)0, dim * 2, BUFFER_FLAGS);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(out + (size_t)row * dim), (short)0, dim * 2, BUFFER_FLAGS);
    u32x4 xv[NC], wv[NC];
#pragma unroll
    for (int k = 0; k < NC; k++)
        xv[k] = __builtin_amdgcn_raw_buffer_load_b128(xr, 16 * (lane + 64 * k), 0, BUFFER_NT);
#pragma unroll
    for (int k = 0; k < NC; k++)
        wv[k] = __builtin_amdgcn_raw_buffer_load_b128(wr, 16 * (lane + 64 * k), 0, 0);
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) acc = dot8(xv[k], xv[k], acc);
    const float total = wave_sum(acc);
    const float inv = 1.0f / sqrtf(total / (float)dim + eps);
#pragma unroll
    for (int k = 0; k < NC; k++) {
        float r[8];
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = round_bf(elem(xv[k], e) * inv) * elem(wv[k], e);
        __builtin_amdgcn_raw_buffer_store_b128(
            u32x4{pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]), pack2(r[6], r[7])}, yr,
            16 * (lane + 64 * k), 0, BUFFER_NT);
    }
}

// Rows that rmsnorm_wave_kernel does not take: wider than 8192, of a dim that is no multiple of 8,
// or not 16-byte aligned. T threads per row (64 W, W = max(1, min(16, ceil(chunks / 1024))); four rows
// per workgroup when W = 1), thread t holds chunks t, t + T, ... (NC of them) in registers and sums
// its squares in chunk/element order; the dim % 8 elements behind the last whole chunk belong to the
// thread that chunk index falls to, last in its order. Wave trees, then the waves added in order
// through LDS. Chunks past the row are the last one read again and left out of the sum, and the
// elements behind the chunks come from the row's last 8, so no branch surrounds a load.
//
// Bound by memory: 16-byte accesses at whatever element the row begins (rows of odd dims cross more
// cache lines than those that begin on a multiple of 4 or 16 bytes). The element-by-element form it
// replaces read each row twice with a bounds test per element: 1000 x 9000 31.0 -> 7.4 us (4.9 TB/s),
// 1000 x 9001 32.2 -> 9.2, 1000 x 30000 71.9 -> 24.9, 4096 x 8190 80.3 -> 27.5, 4096 x 2561 26.9 -> 10.5,
// 1 x 9000 16.8 -> 3.4, 4096 x 101 3.9 -> 3.8. Over 32768 wide a row takes 5 to 16 waves, whose 128
// registers a thread do not hold 16 chunks and the arithmetic: 26 of them go to scratch (108 bytes a
// thread), still 1000 x 32769 65.9 -> 45.3, 1000 x 40000 83.9 -> 38.6, 1000 x 65536 108 -> 57.5,
// 500 x 131072 110 -> 62.7. Up to two chunks per thread the stores are plain: such rows end inside cache
// lines that others begin in (4096 x 101 4.2 us with non-temporal ones, 4096 x 1025 5.7 against 5.5;
// 1000 x 9000 8.4 with plain ones).
template <int NC, int THREADS>
__global__ __launch_bounds__(THREADS) void rmsnorm_rows_kernel(bf16 *out, const bf16 *in,
                                                               const bf16 *weight, int rows,
                                                               int dim, int waves, float eps) {
    typedef u32x4 chunk_t __attribute__((aligned(2)));  // 16 bytes at an element boundary
    __shared__ float part[16];
    const bool alone = waves == 1;  // a wave per row, four rows per workgroup: no sync
    const int T = 64 * waves;
    const int t = alone ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
    const int row = alone ? (int)blockIdx.x * 4 + wave_id() : (int)blockIdx.x;
    if (row >= rows) return;
    const LLM_GLOBAL bf16 *x = gptr(in + (size_t)row * dim), *g = gptr(weight);
    LLM_GLOBAL bf16 *y = gptr(out + (size_t)row * dim);
    const int full = dim >> 3, rem = dim & 7;  // whole chunks (at least one), elements behind them
    u32x4 xv[NC], wv[NC];
#pragma unroll
    for (int k = 0; k < NC; k++)
        xv[k] = __builtin_nontemporal_load(
            (const LLM_GLOBAL chunk_t *)(x + 8 * min(t + T * k, full - 1)));
    const u32x4 xl = *(const LLM_GLOBAL chunk_t *)(x + dim - 8);  // the row's last 8 elements
    // the weights with the row, or where 16 waves' registers do not hold both, at their use
    constexpr bool EARLY = THREADS <= 256;
    const auto weights = [&](int k) {
        return (u32x4)*(const LLM_GLOBAL chunk_t *)(g + 8 * min(t + T * k, full - 1));
    };
#pragma unroll
    for (int k = 0; k < NC && EARLY; k++) wv[k] = weights(k);
    const u32x4 wl = *(const LLM_GLOBAL chunk_t *)(g + dim - 8);
    const bool tail = rem != 0 && t == full % T;
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const float sum = dot8(xv[k], xv[k], acc);
        acc = t + T * k < full ? sum : acc;
    }
#pragma unroll
    for (int e = 1; e < 8; e++) {
        const float sum = fmaf(elem(xl, e), elem(xl, e), acc);
        acc = tail && e >= 8 - rem ? sum : acc;
    }
    float total = wave_sum(acc);
    if (!alone) {
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = total;
        __syncthreads();
        total = part[0];
        for (int w = 1; w < waves; w++) total = total + part[w];
    }
    const float inv = 1.0f / sqrtf(total / (float)dim + eps);
    const auto store = [&](int at, const u32x4 &xc, const u32x4 &wc) {
        float r[8];
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = round_bf(elem(xc, e) * inv) * elem(wc, e);
        const u32x4 v{pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]), pack2(r[6], r[7])};
        if constexpr (NC <= 2)
            *(LLM_GLOBAL chunk_t *)(y + at) = v;
        else
            __builtin_nontemporal_store(v, (LLM_GLOBAL chunk_t *)(y + at));
    };
#pragma unroll
    for (int k = 0; k < NC; k++)
        if (t + T * k < full) store(8 * (t + T * k), xv[k], EARLY ? wv[k] : weights(k));
    if (tail) store(dim - 8, xl, wl);  // over elements of the last chunk too: the same values
}

// The rest (dim < 8, or over 16 chunks per thread: dim > 131079): the same sums, element by element.
__global__ __launch_bounds__(1024) void rmsnorm_generic_kernel(bf16 *out, const bf16 *in,
                                                               const bf16 *weight, int dim,
                                                               float eps) {
    __shared__ float part[16];
    const int row = blockIdx.x;
    const int T = blockDim.x;
    const bf16 *x = in + (size_t)row * dim;
    const int n_chunks = (dim + 7) / 8;
    float acc = 0.0f;
    for (int c = threadIdx.x; c < n_chunks; c += T)
        for (int e = 0; e < 8; e++) {
            const int i = 8 * c + e;
            if (i < dim) {
                const float v = bf2f(x[i]);
                acc = fmaf(v, v, acc);
            }
        }
    const float ws = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ws;
    __syncthreads();
    float total = part[0];
    for (int w = 1; w < T / 64; w++) total = total + part[w];
    const float inv = 1.0f / sqrtf(total / (float)dim + eps);
    bf16 *y = out + (size_t)row * dim;
    for (int i = threadIdx.x; i < dim; i += T)
        y[i] = f2bf(round_bf(bf2f(x[i]) * inv) * bf2f(weight[i]));
}

static int rms_waves(int dim) {
    int n_chunks = (dim + 7) / 8;
    int w = (n_chunks + 64 * 16 - 1) / (64 * 16);
    return w < 1 ? 1 : (w > 16 ? 16 : w);
}

extern "C" void rmsnorm_forward(bf16 *out, const bf16 *in, const bf16 *weight, int rows, int dim,
                                float eps, hipStream_t stream) {
    if (rows <= 0 || dim <= 0) {
        llm_fail("rmsnorm: rows %d and dim %d must be positive", rows, dim);
        return;
    }
    const int per_lane = (dim / 8 + 63) / 64;
    const bool fast = (dim & 7) == 0 && per_lane <= 16 && aligned16(out) && aligned16(in) &&
                      aligned16(weight);
    if (fast) {
        const int blocks = (rows + 3) / 4;
#define RMS(NC_)                                                                            \
    if (per_lane <= NC_) {                                                                  \
        rmsnorm_wave_kernel<NC_><<<blocks, 256, 0, stream>>>(out, in, weight, rows, dim, eps); \
        LAUNCH_OK();                                                                        \
        return;                                                                             \
    }
        RMS(1) RMS(2) RMS(3) RMS(4) RMS(5) RMS(6) RMS(8) RMS(12) RMS(16)
#undef RMS
    }
    const int waves = rms_waves(dim), held = (dim / 8 + 64 * waves - 1) / (64 * waves);
    if (dim >= 8 && held <= 16) {
        // over 4 waves a row has more than 12 chunks per thread
        const int blocks = waves == 1 ? (rows + 3) / 4 : rows, threads = waves == 1 ? 256 : 64 * waves;
#define RMS(NC_, THREADS_)                                                                     \
    if (held <= NC_ && threads <= THREADS_) {                                                  \
        rmsnorm_rows_kernel<NC_, THREADS_>                                                     \
            <<<blocks, threads, 0, stream>>>(out, in, weight, rows, dim, waves, eps);          \
        LAUNCH_OK();                                                                           \
        return;                                                                                \
    }
        RMS(1, 256) RMS(2, 256) RMS(4, 256) RMS(6, 256) RMS(8, 256) RMS(10, 256) RMS(12, 256)
        RMS(16, 256) RMS(16, 1024)
#undef RMS
    }
    rmsnorm_generic_kernel<<<rows, 64 * waves, 0, stream>>>(out, in, weight, dim, eps);
    LAUNCH_OK();
}

// ------------------------------------------------------------------------------------------
// GEMV family (src/kernels.cu:79-212, :215-298)
// ------------------------------------------------------------------------------------------

// A launch covers up to three weight matrices against one input vector (qkv stacks
// [wq; wk; wv]); each segment owns a contiguous range of waves.
struct GemvSeg {
    const bf16 *w;
    bf16 *out;
    int rows;
    int wave_begin;
};

struct GemvArgs {
    GemvSeg seg[3];
    int n_seg;
    const bf16 *x;
    int cols;
    bf16 *tap;             // residual epilogue: optional copy of y
    const bf16 *norm_w;    // fused RMSNorm prologue: gamma (NORM kernels only)
    float eps;
};

// The fused RMSNorm prologue of a one-panel GEMV: the wave's input chunks (lane l: chunks
// l + 64k, the layout of rmsnorm_wave_kernel<NC>) normalised in registers with that kernel's
// arithmetic, so the GEMV sees exactly the bf16 vector rmsnorm_forward would have written. The
// gamma chunks are requested with the input, before the weight rows, and the arithmetic runs
// after the weight requests: loads complete in order, so it waits for the input and gamma only.
template <int NC>
__device__ __forceinline__ void norm_gamma_load(const bf16 *gamma, int cols, u32x4 (&gv)[NC]) {
    const int lane = tid_x() & 63;
    const __amdgpu_buffer_rsrc_t gr =
        __builtin_amdgcn_make_buffer_rsrc((void *)gamma, (short)0, cols * 2, BUFFER_FLAGS);
#pragma unroll
    for (int k = 0; k < NC; k++) gv[k] = __builtin_amdgcn_raw_buffer_load_b128(gr, 16 * (lane + 64 * k), 0, 0);
}
template <int NC>
__device__ __forceinline__ void norm_apply(u32x4 (&xv)[NC], const u32x4 (&gv)[NC], int cols, float eps) {
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) acc = dot8(xv[k], xv[k], acc);
    const float total = wave_sum(acc);
    const float inv = 1.0f / sqrtf(total / (float)cols + eps);
#pragma unroll
    for (int k = 0; k < NC; k++) {
        float r[8];
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = round_bf(elem(xv[k], e) * inv) * elem(gv[k], e);
        xv[k] = u32x4{pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]), pack2(r[6], r[7])};
    }
}

enum { EPI_PLAIN = 0, EPI_RESID = 1 };

// Wave `wave` computes RPW consecutive rows. Lane l streams chunks l, l+64, ... of each row
// (NC per lane per panel, panels until the row ends), fma-accumulating in order; the wave tree
// then gives every lane each row's sum and lane i stores row row0+i.
template <int NC, int RPW, int EPI, bool NORM = false>
__global__ __launch_bounds__(256) void gemv_kernel(GemvArgs a) {
    // Wide rows (NC >= 10: over 4096 columns) take the input through LDS: the workgroup loads
    // each panel of x once instead of once per wave, which at one row per wave would double the
    // L2-to-CU traffic of the weight stream.
    constexpr bool XLDS = NC >= 10 && !NORM;
    constexpr int XT = XLDS ? (64 * NC + 255) / 256 : 1;  // x chunks per thread and panel
    __shared__ u32x4 xs[XLDS ? 64 * NC : 1];
    const int lane = threadIdx.x & 63;
    // wave-uniform (scalar), so the per-row buffer descriptors below are scalar too
    const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int si = (a.n_seg > 2 && wave >= a.seg[2].wave_begin)   ? 2
                   : (a.n_seg > 1 && wave >= a.seg[1].wave_begin) ? 1
                                                                  : 0;
    const bf16 *w = si == 0 ? a.seg[0].w : si == 1 ? a.seg[1].w : a.seg[2].w;
    bf16 *out = si == 0 ? a.seg[0].out : si == 1 ? a.seg[1].out : a.seg[2].out;
    const int rows = si == 0 ? a.seg[0].rows : si == 1 ? a.seg[1].rows : a.seg[2].rows;
    const int wb = si == 0 ? a.seg[0].wave_begin : si == 1 ? a.seg[1].wave_begin : a.seg[2].wave_begin;
    const int row0 = (wave - wb) * RPW;
    // with XLDS every wave takes part in the workgroup's syncs; a wave without rows loads
    // nothing (zero-size row buffers) and stores nothing
    const bool active = row0 < rows;
    if (!XLDS && !active) return;
    const int cols = a.cols;
    const int n_chunks = cols >> 3;
    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)a.x, (short)0, cols * 2, BUFFER_FLAGS);
    float acc[RPW];
#pragma unroll
    for (int i = 0; i < RPW; i++) acc[i] = 0.0f;
    for (int c0 = 0; c0 < n_chunks; c0 += 64 * NC) {
        u32x4 wv[RPW][NC];
        u32x4 xv[NC];
        u32x4 xt[XT];
        if constexpr (XLDS) {
#pragma unroll
            for (int j = 0; j < XT; j++)
                xt[j] = __builtin_amdgcn_raw_buffer_load_b128(
                    xr, 16 * (c0 + (int)threadIdx.x + 256 * j), 0, 0);
        } else {
#pragma unroll
            for (int k = 0; k < NC; k++)
                xv[k] = __builtin_amdgcn_raw_buffer_load_b128(xr, 16 * (c0 + lane + 64 * k), 0, 0);
        }
        u32x4 gm[NC];  // one panel when NORM (host check)
        if constexpr (NORM) norm_gamma_load<NC>(a.norm_w, cols, gm);
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            // the row as a buffer: chunks past its end read as zeros with no branch around the
            // loads, so each chunk's FMAs wait only for that chunk's load
            const int r = min(row0 + i, rows - 1);
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(w + (size_t)r * cols), (short)0, active ? cols * 2 : 0, BUFFER_FLAGS);
#pragma unroll
            for (int k = 0; k < NC; k++)
                wv[i][k] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * (c0 + lane + 64 * k), 0,
                                                                 BUFFER_NT);
        }
        if constexpr (XLDS) {
            if (c0 > 0) __syncthreads();  // every wave has read the previous panel
#pragma unroll
            for (int j = 0; j < XT; j++)
                if ((int)threadIdx.x + 256 * j < 64 * NC) xs[threadIdx.x + 256 * j] = xt[j];
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NC; k++) xv[k] = xs[lane + 64 * k];
        }
        if constexpr (NORM) norm_apply<NC>(xv, gm, cols, a.eps);
#pragma unroll
        for (int i = 0; i < RPW; i++)
#pragma unroll
            for (int k = 0; k < NC; k++) acc[i] = dot8(wv[i][k], xv[k], acc[i]);
    }
    if (!active) return;
    float mine = 0.0f;
#pragma unroll
    for (int i = 0; i < RPW; i++) {
        const float t = wave_sum(acc[i]);
        if (lane == i) mine = t;
    }
    const int r = row0 + lane;
    if (lane < RPW && r < rows) {
        const uint32_t y = f2bf(mine);
        if (EPI == EPI_PLAIN) {
            out[r] = (bf16)y;
        } else {
            if (a.tap) a.tap[r] = (bf16)y;
            out[r] = (bf16)f2bf(bf2f(out[r]) + bf2f((bf16)y));
        }
    }
}

// gate and up rows together: g = bf16(wg[r].x), u = bf16(wu[r].x),
// act = bf16(bf16(silu(g)) * u) (src/kernels.cu:276-287).
template <int NC, int RPW, bool NORM = false>
__global__ __launch_bounds__(256) void gate_up_kernel(bf16 *act, const bf16 *wg, const bf16 *wu,
                                                      const bf16 *x, int rows, int cols,
                                                      bf16 *gate_tap, bf16 *up_tap,
                                                      const bf16 *norm_w = nullptr,
                                                      float eps = 0.0f) {
    const int lane = threadIdx.x & 63;
    const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = wave * RPW;
    if (row0 >= rows) return;
    const int n_chunks = cols >> 3;
    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, cols * 2, BUFFER_FLAGS);
    float ag[RPW], au[RPW];
#pragma unroll
    for (int i = 0; i < RPW; i++) ag[i] = au[i] = 0.0f;
    for (int c0 = 0; c0 < n_chunks; c0 += 64 * NC) {
        u32x4 xv[NC];
        u32x4 gv[RPW][NC], uv[RPW][NC];
#pragma unroll
        for (int k = 0; k < NC; k++)
            xv[k] = __builtin_amdgcn_raw_buffer_load_b128(xr, 16 * (c0 + lane + 64 * k), 0, 0);
        u32x4 gm[NC];  // one panel when NORM (host check)
        if constexpr (NORM) norm_gamma_load<NC>(norm_w, cols, gm);
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const size_t r = (size_t)min(row0 + i, rows - 1);
            const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(wg + r * cols), (short)0, cols * 2, BUFFER_FLAGS);
            const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(wu + r * cols), (short)0, cols * 2, BUFFER_FLAGS);
#pragma unroll
            for (int k = 0; k < NC; k++) {
                const int off = 16 * (c0 + lane + 64 * k);
                gv[i][k] = __builtin_amdgcn_raw_buffer_load_b128(rg, off, 0, BUFFER_NT);
                uv[i][k] = __builtin_amdgcn_raw_buffer_load_b128(ru, off, 0, BUFFER_NT);
            }
        }
        if constexpr (NORM) norm_apply<NC>(xv, gm, cols, eps);
#pragma unroll
        for (int i = 0; i < RPW; i++)
#pragma unroll
            for (int k = 0; k < NC; k++) {
                ag[i] = dot8(gv[i][k], xv[k], ag[i]);
                au[i] = dot8(uv[i][k], xv[k], au[i]);
            }
    }
    float g_mine = 0.0f, u_mine = 0.0f;
#pragma unroll
    for (int i = 0; i < RPW; i++) {
        const float g = wave_sum(ag[i]);
        const float u = wave_sum(au[i]);
        if (lane == i) {
            g_mine = g;
            u_mine = u;
        }
    }
    const int r = row0 + lane;
    if (lane < RPW && r < rows) {
        const bf16 g = (bf16)f2bf(g_mine);
        const bf16 u = (bf16)f2bf(u_mine);
        if (gate_tap) gate_tap[r] = g;
        if (up_tap) up_tap[r] = u;
        const float s = round_bf(silu_f32(bf2f(g)));
        act[r] = (bf16)f2bf(s * bf2f(u));
    }
}

// Per-lane chunk capacity of one panel.
static int pick_nc(int n_chunks) {
    const int per_lane = (n_chunks + 63) / 64;
    static const int ncs[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20};
    for (int v : ncs)
        if (v >= per_lane) return v;
    return 20;
}

// Rows per wave: enough loads in flight per lane (RPW*NC ~ 8-12) while keeping at least ~2048
// waves (8 per CU) when the matrix has the rows for it. Fewer rows leave the fused RMSNorm's
// arithmetic, once per wave, in front of the stream; more leave fewer waves to overlap. RMSNorm + LM
// head of 151936 rows (us, rows per wave): 1024 columns (NC 2) 8 48.0, 4 43.9 (7.1 TB/s), 2 44.0, 1
// 66.5; 2048 (NC 4) 4 93.5, 2 85.2 (7.3 TB/s), 1 116; 2560 (NC 5) 4 110, 2 106.5, 1 144; 100000 rows of
// 512 (NC 1) 8 15.6, 4 15.9, 2 20.3; of 1496 (NC 3) 4 42.0, 2 42.9. A pair of gate and up rows counts
// twice.
static int pick_rpw(int nc, long total_rows, int pairs) {
    int rpw = nc <= 1 ? 8 : nc <= 3 ? 4 : nc <= 8 ? 2 : 1;
    if (pairs) rpw = nc <= 2 ? 4 : nc <= 4 ? 2 : 1;
    while (rpw > 1 && total_rows / rpw < 2048) rpw /= 2;
    return rpw;
}

static bool check_gemv(const char *name, const void *w, const void *x, int rows, int cols) {
    if (cols % 8 != 0) return llm_fail("%s: cols %d is not a multiple of 8", name, cols);
    if (rows <= 0 || cols <= 0) return llm_fail("%s: rows %d and cols %d must be positive", name, rows, cols);
    if (!aligned16(w) || !aligned16(x))
        return llm_fail("%s: weight and input must be 16-byte aligned", name);
    return true;
}

#define GEMV_CASES(X) \
    X(1, 1) X(1, 2) X(1, 4) X(1, 8) X(2, 1) X(2, 2) X(2, 4) X(3, 1) X(3, 2) X(3, 4) \
    X(4, 1) X(4, 2) X(5, 1) X(5, 2) X(6, 1) X(6, 2) X(8, 1) X(8, 2) X(10, 1)    \
    X(12, 1) X(16, 1) X(20, 1)

template <int EPI>
static bool dispatch_gemv(const GemvArgs &a, int nc, int rpw, int blocks, hipStream_t st) {
#define X(NC_, RPW_)                                                         \
    if (nc == NC_ && rpw == RPW_) {                                          \
        if (EPI == EPI_PLAIN && a.norm_w)                                    \
            gemv_kernel<NC_, RPW_, EPI_PLAIN, true><<<blocks, 256, 0, st>>>(a); \
        else                                                                 \
            gemv_kernel<NC_, RPW_, EPI><<<blocks, 256, 0, st>>>(a);          \
        return LAUNCH_OK();                                                  \
    }
    GEMV_CASES(X)
#undef X
    return llm_fail("gemv: no kernel for nc %d rpw %d", nc, rpw);
}

static void launch_gemv(GemvArgs &a, int epi, hipStream_t stream) {
    long total_rows = 0;
    for (int i = 0; i < a.n_seg; i++) total_rows += a.seg[i].rows;
    const int nc = pick_nc(a.cols / 8);
    const int rpw = pick_rpw(nc, total_rows, 0);
    int waves = 0;
    for (int i = 0; i < a.n_seg; i++) {
        a.seg[i].wave_begin = waves;
        waves += (a.seg[i].rows + rpw - 1) / rpw;
    }
    const int blocks = (waves + 3) / 4;
    if (epi == EPI_PLAIN)
        dispatch_gemv<EPI_PLAIN>(a, nc, rpw, blocks, stream);
    else
        dispatch_gemv<EPI_RESID>(a, nc, rpw, blocks, stream);
}

extern "C" void gemv_forward(bf16 *out, const bf16 *w, const bf16 *x, int rows, int cols,
                             hipStream_t stream) {
    if (!check_gemv("gemv", w, x, rows, cols)) return;
    GemvArgs a = {};
    a.seg[0] = {w, out, rows, 0};
    a.n_seg = 1;
    a.x = x;
    a.cols = cols;
    launch_gemv(a, EPI_PLAIN, stream);
}

extern "C" void gemv_residual_forward(bf16 *x, const bf16 *w, const bf16 *in, int rows, int cols,
                                      bf16 *tap, hipStream_t stream) {
    if (!check_gemv("gemv_residual", w, in, rows, cols)) return;
    if (x == in) {
        llm_fail("gemv_residual: in must not alias x");
        return;
    }
    GemvArgs a = {};
    a.seg[0] = {w, x, rows, 0};
    a.n_seg = 1;
    a.x = in;
    a.cols = cols;
    a.tap = tap;
    launch_gemv(a, EPI_RESID, stream);
}

extern "C" void qkv_forward(bf16 *q, bf16 *k, bf16 *v, const bf16 *wq, const bf16 *wk,
                            const bf16 *wv, const bf16 *x, int q_rows, int kv_rows, int cols,
                            hipStream_t stream) {
    if (!check_gemv("qkv", wq, x, q_rows, cols) || !check_gemv("qkv", wk, x, kv_rows, cols) ||
        !check_gemv("qkv", wv, x, kv_rows, cols))
        return;
    GemvArgs a = {};
    a.seg[0] = {wq, q, q_rows, 0};
    a.seg[1] = {wk, k, kv_rows, 0};
    a.seg[2] = {wv, v, kv_rows, 0};
    a.n_seg = 3;
    a.x = x;
    a.cols = cols;
    launch_gemv(a, EPI_PLAIN, stream);
}

#define GATE_UP_CASES(X) \
    X(1, 1) X(1, 2) X(1, 4) X(2, 1) X(2, 2) X(2, 4) X(3, 1) X(3, 2) X(4, 1) X(4, 2) X(5, 1) \
    X(6, 1) X(8, 1) X(10, 1) X(12, 1) X(16, 1) X(20, 1)

static void launch_gate_up(bf16 *act, const bf16 *w_gate, const bf16 *w_up, const bf16 *x,
                           int rows, int cols, bf16 *gate_tap, bf16 *up_tap, const bf16 *norm_w,
                           float eps, hipStream_t stream) {
    const int nc = pick_nc(cols / 8);
    const int rpw = pick_rpw(nc, rows, 1);
    const int waves = (rows + rpw - 1) / rpw;
    const int blocks = (waves + 3) / 4;
#define X(NC_, RPW_)                                                                       \
    if (nc == NC_ && rpw == RPW_) {                                                        \
        if (norm_w)                                                                        \
            gate_up_kernel<NC_, RPW_, true><<<blocks, 256, 0, stream>>>(                   \
                act, w_gate, w_up, x, rows, cols, gate_tap, up_tap, norm_w, eps);          \
        else                                                                               \
            gate_up_kernel<NC_, RPW_><<<blocks, 256, 0, stream>>>(act, w_gate, w_up, x,    \
                                                                 rows, cols, gate_tap, up_tap); \
        LAUNCH_OK();                                                                       \
        return;                                                                            \
    }
    GATE_UP_CASES(X)
#undef X
    llm_fail("gate_up: no kernel for nc %d rpw %d", nc, rpw);
}

extern "C" void gate_up_forward(bf16 *act, const bf16 *w_gate, const bf16 *w_up, const bf16 *x,
                                int rows, int cols, bf16 *gate_tap, bf16 *up_tap,
                                hipStream_t stream) {
    if (!check_gemv("gate_up", w_gate, x, rows, cols) || !check_gemv("gate_up", w_up, x, rows, cols))
        return;
    launch_gate_up(act, w_gate, w_up, x, rows, cols, gate_tap, up_tap, nullptr, 0.0f, stream);
}

// The fused forms: RMSNorm of x (one row) as the GEMV's prologue, summing the squares in the
// order of rmsnorm_wave_kernel (lane l: chunks l, l+64, ..., then the wave tree), so the result
// is rmsnorm_forward's. That kernel covers rows of up to 64 * 16 chunks (8192 columns), which
// also fit one GEMV panel.
static bool check_norm_fused(const char *name, const bf16 *norm_w, int cols) {
    if (!norm_w) return llm_fail("%s: norm weights are NULL", name);
    if (!aligned16(norm_w)) return llm_fail("%s: norm weights must be 16-byte aligned", name);
    if ((cols / 8 + 63) / 64 > 16 || cols / 8 > 64 * pick_nc(cols / 8))
        return llm_fail("%s: %d columns do not fit one panel (at most 8192)", name, cols);
    return true;
}

extern "C" void rmsnorm_qkv_forward(bf16 *q, bf16 *k, bf16 *v, const bf16 *wq, const bf16 *wk,
                                    const bf16 *wv, const bf16 *x, const bf16 *norm_w, float eps,
                                    int q_rows, int kv_rows, int cols, hipStream_t stream) {
    if (!check_gemv("rmsnorm_qkv", wq, x, q_rows, cols) ||
        !check_gemv("rmsnorm_qkv", wk, x, kv_rows, cols) ||
        !check_gemv("rmsnorm_qkv", wv, x, kv_rows, cols) ||
        !check_norm_fused("rmsnorm_qkv", norm_w, cols))
        return;
    GemvArgs a = {};
    a.seg[0] = {wq, q, q_rows, 0};
    a.seg[1] = {wk, k, kv_rows, 0};
    a.seg[2] = {wv, v, kv_rows, 0};
    a.n_seg = 3;
    a.x = x;
    a.cols = cols;
    a.norm_w = norm_w;
    a.eps = eps;
    launch_gemv(a, EPI_PLAIN, stream);
}

extern "C" void rmsnorm_gemv_forward(bf16 *out, const bf16 *w, const bf16 *x, const bf16 *norm_w,
                                     float eps, int rows, int cols, hipStream_t stream) {
    if (!check_gemv("rmsnorm_gemv", w, x, rows, cols) ||
        !check_norm_fused("rmsnorm_gemv", norm_w, cols))
        return;
    GemvArgs a = {};
    a.seg[0] = {w, out, rows, 0};
    a.n_seg = 1;
    a.x = x;
    a.cols = cols;
    a.norm_w = norm_w;
    a.eps = eps;
    launch_gemv(a, EPI_PLAIN, stream);
}

extern "C" void rmsnorm_gate_up_forward(bf16 *act, const bf16 *w_gate, const bf16 *w_up,
                                        const bf16 *x, const bf16 *norm_w, float eps, int rows,
                                        int cols, hipStream_t stream) {
    if (!check_gemv("rmsnorm_gate_up", w_gate, x, rows, cols) ||
        !check_gemv("rmsnorm_gate_up", w_up, x, rows, cols) ||
        !check_norm_fused("rmsnorm_gate_up", norm_w, cols))
        return;
    launch_gate_up(act, w_gate, w_up, x, rows, cols, nullptr, nullptr, norm_w, eps, stream);
}

// ------------------------------------------------------------------------------------------
// SwiGLU elementwise (src/kernels.cu:283-286 over arrays)
// ------------------------------------------------------------------------------------------

__device__ __forceinline__ u32x4 swiglu8(const u32x4 &g, const u32x4 &u) {
    float gv[8], s[8], r[8];
#pragma unroll
    for (int e = 0; e < 8; e++) gv[e] = elem(g, e);
    silu_bf16x8(gv, s);
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = s[e] * elem(u, e);
    return u32x4{pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]), pack2(r[6], r[7])};
}

// Grid-stride over 16-byte chunks, U chunks per thread per step. One chunk per thread and a grid
// of up to 80 workgroups per CU (every chunk of a 4096 x 9728 call in one pass) measured fastest:
// 38.7 us against 47.5 with 4 chunks per thread and 8 workgroups per CU.
constexpr int SWIGLU_U = 1;
constexpr int SWIGLU_BLOCKS_PER_CU = 80;
__global__ __launch_bounds__(256) void swiglu_kernel(bf16 *act, const bf16 *gate, const bf16 *up,
                                                     size_t n) {
    constexpr int U = SWIGLU_U;
    const size_t n_chunks = n / 8;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; c + (U - 1) * stride < n_chunks; c += U * stride) {
        u32x4 g[U], u[U];
#pragma unroll
        for (int i = 0; i < U; i++) {
            g[i] = ld16_nt(gate + 8 * (c + i * stride));
            u[i] = ld16_nt(up + 8 * (c + i * stride));
        }
#pragma unroll
        for (int i = 0; i < U; i++)
            __builtin_nontemporal_store(swiglu8(g[i], u[i]), (u32x4 *)(act + 8 * (c + i * stride)));
    }
    for (; c < n_chunks; c += stride)
        __builtin_nontemporal_store(swiglu8(ld16_nt(gate + 8 * c), ld16_nt(up + 8 * c)),
                                    (u32x4 *)(act + 8 * c));
    if (blockIdx.x == 0)
        for (size_t i = n_chunks * 8 + threadIdx.x; i < n; i += blockDim.x)
            act[i] = (bf16)f2bf(round_bf(silu_f32(bf2f(gate[i]))) * bf2f(up[i]));
}

// Scalar variant for buffers that are not 16-byte aligned.
__global__ __launch_bounds__(256) void swiglu_scalar_kernel(bf16 *act, const bf16 *gate,
                                                            const bf16 *up, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        act[i] = (bf16)f2bf(round_bf(silu_f32(bf2f(gate[i]))) * bf2f(up[i]));
}

static int device_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            cus = 256;
    }
    return cus;
}

extern "C" void swiglu_forward(bf16 *act, const bf16 *gate, const bf16 *up, size_t n,
                               hipStream_t stream) {
    if (n == 0) return;
    const size_t chunks = (n + 7) / 8;
    size_t blocks = (chunks + 255) / 256;
    const size_t cap = (size_t)device_cus() * SWIGLU_BLOCKS_PER_CU;
    if (blocks > cap) blocks = cap;
    if (aligned16(act) && aligned16(gate) && aligned16(up))
        swiglu_kernel<<<(unsigned)blocks, 256, 0, stream>>>(act, gate, up, n);
    else
        swiglu_scalar_kernel<<<(unsigned)blocks, 256, 0, stream>>>(act, gate, up, n);
    LAUNCH_OK();
}

// ------------------------------------------------------------------------------------------
// QK-norm + RoPE + KV-cache write (src/kernels.cu:301-403)
// ------------------------------------------------------------------------------------------

struct RopeArgs {
    bf16 *q;
    bf16 *k;
    const bf16 *v;
    const bf16 *qn;
    const bf16 *kn;
    bf16 *kc;
    bf16 *vc;
    const int *positions;
    bf16 *q_tap;
    bf16 *k_tap;
    int n_tokens, n_heads, n_kv_heads;
    float eps;
    int qg, kg, vg;  // waves per token: q head groups, k head groups, v copy groups
    float inv_freq[128];
};

// A wave handles 64/(D/16) heads of one token: lane L of a head holds [8L, 8L+8) and
// [D/2+8L, D/2+8L+8). Sum of squares: fma over the first chunk then the second, tree over the
// D/16 lanes. The RoPE table (cos/sin of pos*inv_freq_j in double, rounded to fp32 then bf16)
// is computed one entry per lane and fetched by lane shuffles.
template <int D>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(RopeArgs a) {
    constexpr int LH = D / 16;
    constexpr int HPW = 64 / LH;
    constexpr int HALF = D / 2;
    constexpr int NJ = (HALF + 63) / 64;
    const int lane = threadIdx.x & 63;
    const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per_token = a.qg + a.kg + a.vg;
    const int t = wave / per_token;
    if (t >= a.n_tokens) return;
    const int item = wave - t * per_token;
    const int pos = a.positions[t];
    const int hg = lane / LH, L = lane % LH;
    const int q_dim = a.n_heads * D, kv_dim = a.n_kv_heads * D;
    const size_t slot = (size_t)pos * kv_dim;

    if (item >= a.qg + a.kg) {  // value rows into the cache
        const int h = (item - a.qg - a.kg) * HPW + hg;
        if (h < a.n_kv_heads) {
            const bf16 *src = a.v + (size_t)t * kv_dim + h * D;
            bf16 *dst = a.vc + slot + h * D;
            st16(dst + 8 * L, ld16(src + 8 * L));
            st16(dst + HALF + 8 * L, ld16(src + HALF + 8 * L));
        }
        return;
    }
    const bool is_k = item >= a.qg;
    // the wave's heads h0 .. h0 + HPW - 1 (those that exist) as one buffer, so the descriptor is
    // wave-uniform: loads past the last head read zeros and stores there are dropped; the
    // loads go out before the RoPE table is computed, which then overlaps them
    const int h0 = (is_k ? item - a.qg : item) * HPW;
    const int n_h = min(HPW, (is_k ? a.n_kv_heads : a.n_heads) - h0);
    const size_t off = (size_t)t * (is_k ? kv_dim : q_dim) + (size_t)h0 * D;
    bf16 *tap = is_k ? a.k_tap : a.q_tap;
    auto heads = [&](bf16 *base) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, n_h * D * 2, BUFFER_FLAGS);
    };
    const __amdgpu_buffer_rsrc_t xr = heads((is_k ? a.k : a.q) + off);
    const int oa = hg * D * 2 + 16 * L, ob = oa + 2 * HALF;
    const u32x4 xa = __builtin_amdgcn_raw_buffer_load_b128(xr, oa, 0, BUFFER_NT);
    const u32x4 xb = __builtin_amdgcn_raw_buffer_load_b128(xr, ob, 0, BUFFER_NT);
    const bf16 *w = is_k ? a.kn : a.qn;
    const u32x4 wa = ld16(w + 8 * L), wb = ld16(w + HALF + 8 * L);
    float cs[NJ], sn[NJ];
    rope_table<D>(pos, a.inv_freq, cs, sn);
    u32x4 ya, yb, va, vb;
    norm_rope<D>(xa, xb, wa, wb, a.eps, cs, sn, L, ya, yb, va, vb);
    if (tap) {
        const __amdgpu_buffer_rsrc_t tr = heads(tap + off);
        __builtin_amdgcn_raw_buffer_store_b128(ya, tr, oa, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(yb, tr, ob, 0, 0);
    }
    __builtin_amdgcn_raw_buffer_store_b128(va, xr, oa, 0, BUFFER_NT);
    __builtin_amdgcn_raw_buffer_store_b128(vb, xr, ob, 0, BUFFER_NT);
    if (is_k) {
        const __amdgpu_buffer_rsrc_t cr = heads(a.kc + slot + (size_t)h0 * D);
        __builtin_amdgcn_raw_buffer_store_b128(va, cr, oa, 0, BUFFER_NT);
        __builtin_amdgcn_raw_buffer_store_b128(vb, cr, ob, 0, BUFFER_NT);
    }
}

// inv_freq_j = 1 / fp32(pow(theta, fp32(2j / D))) as HF computes it (modeling_qwen3.py:121),
// cached per (theta, D).
void rope_inv_freq_table(float theta, int D, float *out) {
    static std::mutex mu;
    static float cached_theta = -1.0f;
    static int cached_d = -1;
    static float table[128];
    std::lock_guard<std::mutex> lock(mu);
    if (cached_theta != theta || cached_d != D) {
        for (int j = 0; j < D / 2; j++) {
            const float e = (float)(2 * j) / (float)D;
            table[j] = 1.0f / (float)pow((double)theta, (double)e);
        }
        cached_theta = theta;
        cached_d = D;
    }
    memcpy(out, table, sizeof(float) * (D / 2));
}

static void launch_qk_norm_rope(bf16 *q, bf16 *k, const bf16 *v, const bf16 *q_norm_w,
                                const bf16 *k_norm_w, bf16 *key_cache, bf16 *value_cache,
                                const int *positions, int n_tokens, int n_heads, int n_kv_heads,
                                int head_dim, float eps, float theta, bf16 *q_tap, bf16 *k_tap,
                                hipStream_t stream) {
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) {
        llm_fail("qk_norm_rope: head_dim %d is not 64, 128 or 256", head_dim);
        return;
    }
    if (n_tokens <= 0 || n_heads <= 0 || n_kv_heads <= 0) {
        llm_fail("qk_norm_rope: n_tokens %d, n_heads %d, n_kv_heads %d must be positive",
                 n_tokens, n_heads, n_kv_heads);
        return;
    }
    const void *ptrs[] = {q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, q_tap, k_tap};
    for (const void *p : ptrs)
        if (p && !aligned16(p)) {
            llm_fail("qk_norm_rope: tensors must be 16-byte aligned");
            return;
        }
    RopeArgs a;
    memset(&a, 0, sizeof a);
    a.q = q;
    a.k = k;
    a.v = v;
    a.qn = q_norm_w;
    a.kn = k_norm_w;
    a.kc = key_cache;
    a.vc = value_cache;
    a.positions = positions;
    a.q_tap = q_tap;
    a.k_tap = k_tap;
    a.n_tokens = n_tokens;
    a.n_heads = n_heads;
    a.n_kv_heads = n_kv_heads;
    a.eps = eps;
    const int hpw = 64 / (head_dim / 16);
    a.qg = (n_heads + hpw - 1) / hpw;
    a.kg = (n_kv_heads + hpw - 1) / hpw;
    a.vg = a.kg;
    rope_inv_freq_table(theta, head_dim, a.inv_freq);
    const long waves = (long)n_tokens * (a.qg + a.kg + a.vg);
    const unsigned blocks = (unsigned)((waves + 3) / 4);
    if (head_dim == 64)
        qk_norm_rope_kernel<64><<<blocks, 256, 0, stream>>>(a);
    else if (head_dim == 128)
        qk_norm_rope_kernel<128><<<blocks, 256, 0, stream>>>(a);
    else
        qk_norm_rope_kernel<256><<<blocks, 256, 0, stream>>>(a);
    LAUNCH_OK();
}

extern "C" void qk_norm_rope_forward(bf16 *q, bf16 *k, const bf16 *v, const bf16 *q_norm_w,
                                     const bf16 *k_norm_w, bf16 *key_cache, bf16 *value_cache,
                                     const int *d_pos, int n_heads, int n_kv_heads, int head_dim,
                                     float eps, float theta, bf16 *q_tap, bf16 *k_tap,
                                     hipStream_t stream) {
    launch_qk_norm_rope(q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, d_pos, 1, n_heads,
                        n_kv_heads, head_dim, eps, theta, q_tap, k_tap, stream);
}

extern "C" void qk_norm_rope_rows(bf16 *q, bf16 *k, const bf16 *v, const bf16 *q_norm_w,
                                  const bf16 *k_norm_w, bf16 *key_cache, bf16 *value_cache,
                                  const int *d_positions, int n_tokens, int n_heads,
                                  int n_kv_heads, int head_dim, float eps, float theta,
                                  bf16 *q_tap, bf16 *k_tap, hipStream_t stream) {
    launch_qk_norm_rope(q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, d_positions,
                        n_tokens, n_heads, n_kv_heads, head_dim, eps, theta, q_tap, k_tap, stream);
}

// ------------------------------------------------------------------------------------------
// decode attention, split softmax (src/kernels.cu:439-497)
// ------------------------------------------------------------------------------------------

// 16 consecutive floats of LDS (16-byte aligned), all requested at once.
__device__ __forceinline__ void ld_lds16(const float *p, float (&v)[16]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4 *q = (const f32x4 *)p;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const f32x4 a = q[i];
        v[4 * i] = a.x;
        v[4 * i + 1] = a.y;
        v[4 * i + 2] = a.z;
        v[4 * i + 3] = a.w;
    }
}

constexpr int ATT_B = 64;  // positions per block
constexpr int ATTN_MAXGRID = 8192;  // workgroups of a pass

struct AttnArgs {
    bf16 *out;
    const bf16 *q;
    const bf16 *kc;
    const bf16 *vc;
    float *scores;   // [n_heads, max_seq]
    float *stats;    // [n_heads, max_blocks, 2]: block max, block sum of exp(s - max)
    float *partial;  // [n_heads, max_blocks, D]: block sums of p v
    const int *d_pos;
    int n_heads, n_kv_heads, max_seq, max_blocks;
    float scale;
    int *err;    // the step's error flag (set to 1 for a position outside the cache), or NULL
};

// Whether the query's position (n - 1) is one that the caches hold. Where it is not, every pass leaves
// the caches and the workspace alone, `out` becomes zeros and the step's error flag is set.
__device__ __forceinline__ bool position_held(const AttnArgs &a, int n) {
    return n > 0 && n <= a.max_seq;
}
__device__ __forceinline__ void position_error(const AttnArgs &a) {
    if (a.err && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(gptr(a.err), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A block's max in the statistics. It is one of the scores, which are bf16 values: the low half of its
// word is zero after the scores pass, and for block 0 of a kv head's first query head it then counts
// the head's items that have stored their partials (attn_pv_combine_kernel).
__device__ __forceinline__ float block_max(const float *st, int b) {
    return __uint_as_float(__float_as_uint(st[2 * b]) & 0xffff0000u);
}

static size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }

// Workspace layout: scores [n_heads, max_seq], stats [n_heads, max_blocks, 2], then (from a
// 16-byte boundary) partials [n_heads, max_blocks, D].
static size_t attention_partial_offset(int n_heads, int max_seq) {
    const size_t mb = ceil_div((size_t)max_seq, ATT_B);
    return ceil_div((size_t)n_heads * max_seq + (size_t)n_heads * mb * 2, 4) * 4;
}

extern "C" size_t attention_workspace_floats(int n_heads, int head_dim, int max_seq) {
    const size_t mb = ceil_div((size_t)max_seq, ATT_B);
    return attention_partial_offset(n_heads, max_seq) + (size_t)n_heads * mb * head_dim;
}

// This lane's chunks (16 bytes at 8 L) of the rows first, first + PPW, ... of block b of a cache, kv
// head g: the block's rows below `rows` as one buffer, so that those at or past it read zeros with no
// branch around the loads.
template <int D, int ITERS>
__device__ __forceinline__ void request_rows(const bf16 *cache, int kv_dim, int b, int g, int rows,
                                             int first, int L, u32x4 (&out)[ITERS]) {
    constexpr int PPW = 512 / D;  // positions of a wave's load
    const int have = min(ATT_B, rows - b * ATT_B);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(cache + (size_t)b * ATT_B * kv_dim + g * D), (short)0,
        have <= 0 ? 0 : ((have - 1) * kv_dim + D) * 2, BUFFER_FLAGS);
#pragma unroll
    for (int it = 0; it < ITERS; it++)
        out[it] = __builtin_amdgcn_raw_buffer_load_b128(
            rs, ((first + it * PPW) * kv_dim + 8 * L) * 2, 0, BUFFER_NT);
}

// Pass 1, per (block of 64 positions, kv head): scores of the REP query heads sharing the kv
// head, s = bf16(bf16(q.k) * scale) with q.k over D/8 lanes; then per head the block max and
// the block's tree sum of exp(s - max). Work items are strided over a fixed grid because the
// position count is only known on the device.
template <int D, int REP>
__global__ __launch_bounds__(256) void attn_scores_kernel(AttnArgs a) {
    constexpr int LP = D / 8, PPW = 64 / LP, PER_WAVE = ATT_B / 4, ITERS = PER_WAVE / PPW;
    __shared__ float sc[REP][ATT_B];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int G = lane / LP, L = lane % LP;
    const int n = *a.d_pos + 1;
    if (!position_held(a, n)) return position_error(a);
    const int nb = (n + ATT_B - 1) / ATT_B;
    const int kv_dim = a.n_kv_heads * D;
    for (int item = blockIdx.x; item < nb * a.n_kv_heads; item += gridDim.x) {
        const int b = item / a.n_kv_heads, g = item - b * a.n_kv_heads;
        u32x4 qv[REP];
#pragma unroll
        for (int r = 0; r < REP; r++) qv[r] = ld16(a.q + (size_t)(g * REP + r) * D + 8 * L);
        u32x4 kv[ITERS];
        request_rows<D, ITERS>(a.kc, kv_dim, b, g, n, w * PER_WAVE + G, L, kv);
        // the ITERS * REP dot products of a lane, reduced over the LP lanes of its position group
        // LP at a time by reduce-scatter (each total bit-identical to group_sum<LP>): lane L of a
        // slice ends with product scatter_row(L) of that slice
        constexpr int NP = ITERS * REP, SL = NP < LP ? NP : LP;
        float part[NP];
#pragma unroll
        for (int it = 0; it < ITERS; it++)
#pragma unroll
            for (int r = 0; r < REP; r++) part[it * REP + r] = dot8(qv[r], kv[it], 0.0f);
#pragma unroll
        for (int s0 = 0; s0 < NP; s0 += SL) {
            float slice[SL];
#pragma unroll
            for (int j = 0; j < SL; j++) slice[j] = part[s0 + j];
            const float d = group_sum_scatter<LP, SL>(slice);
            const int j = s0 + scatter_row<SL>(L), it = j / REP, r = j - it * REP;
            const int slot = w * PER_WAVE + it * PPW + G;
            const int t = b * ATT_B + slot;
            const float s = round_bf(round_bf(d) * a.scale);
            if (L < SL) {
                sc[r][slot] = s;
                if (t < n) a.scores[(size_t)(g * REP + r) * a.max_seq + t] = s;
            }
        }
        __syncthreads();
        for (int r = w; r < REP; r += 4) {
            const bool v = b * ATT_B + lane < n;
            const float s = v ? sc[r][lane] : -__builtin_huge_valf();
            const float m = wave_max(s);
            const float e = v ? exp_f32(s - m) : 0.0f;
            const float S = wave_sum(e);
            if (lane == 0) {
                float *st = a.stats + ((size_t)(g * REP + r) * a.max_blocks + b) * 2;
                st[0] = m;
                st[1] = S;
            }
        }
        __syncthreads();
    }
}

// Pass 1 with the QK-norm + RoPE of the position folded in (qk_norm_rope_forward followed by
// attn_scores_kernel, the same bits): an item requests its key history rows (positions < pos)
// first, then normalises and rotates its kv head's REP query heads (waves 0 .. QWAVES-1, the
// qk_norm_rope_kernel lane layout) into LDS while they stream; the item of the block holding
// pos also rotates the key (next wave), which it uses for position pos and writes, with the
// value row, into the caches' row pos. Every item of a kv head computes the same roped query
// heads; nothing waits for another workgroup.
struct AttnRopeArgs {
    AttnArgs at;
    const bf16 *k, *v, *qn, *kn;  // at.q is the query before QK-norm + RoPE
    bf16 *kc_w, *vc_w;            // the caches, writable (row pos)
    const float *table;           // the RoPE table at *d_pos (rope_table_kernel), or NULL
    float eps;
    float inv_freq[128];
};

// The RoPE table at *d_pos, once for every layer of a step: table[j] = cos and table[D/2 + j] =
// sin of fp32(pos * inv_freq_j) as rope_table computes them (double sincos, rounded to fp32 and
// then to bf16), j < D/2.
struct RopeFreqArgs {
    float inv_freq[128];
};
__global__ __launch_bounds__(128) void rope_table_kernel(float *table, const int *d_pos,
                                                         RopeFreqArgs f, int half) {
    const int j = threadIdx.x;
    if (j < half) {
        const float angle = (float)*d_pos * f.inv_freq[j];
        double sn, cs;
        sincos_d((double)angle, &sn, &cs);
        table[j] = round_bf((float)cs);
        table[half + j] = round_bf((float)sn);
    }
}

bool rope_table_launch(float *table, const int *d_pos, int head_dim, float theta,
                       hipStream_t stream) {
    if (head_dim != 64 && head_dim != 128 && head_dim != 256)
        return llm_fail("rope_table: head_dim %d is not 64, 128 or 256", head_dim);
    RopeFreqArgs f;
    rope_inv_freq_table(theta, head_dim, f.inv_freq);
    rope_table_kernel<<<1, 128, 0, stream>>>(table, d_pos, f, head_dim / 2);
    return LAUNCH_OK();
}

// The rope inputs of one wave of the one-pass kernel (the raw head rows and norm weights, requested
// before the key rows so that they are not behind them: loads complete in order) and its RoPE table.
template <int D>
struct RopeIn {
    u32x4 xa, xb, wa, wb;
    float cs[RopeShape<D>::NJ], sn[RopeShape<D>::NJ];
};

// This lane's RoPE frequencies inv_freq[lane + 64 m], m < NJ, picked out of the argument table
// with scalar loads and selects. Indexed per lane, the table would be read with a vector load,
// which the compiler places at its use, after the key rows requested before it; the wait for it
// would then wait for all of those rows.
template <int D>
struct LaneFreq {
    float f[RopeShape<D>::NJ];
    __device__ float operator[](int j) const { return f[j >> 6]; }  // j = lane + 64 m
};
template <int D>
__device__ __forceinline__ LaneFreq<D> lane_freq(const float (&table)[128]) {
    constexpr int NJ = RopeShape<D>::NJ, HALF = RopeShape<D>::HALF;
    const int lane = threadIdx.x & 63;
    LaneFreq<D> out;
#pragma unroll
    for (int m = 0; m < NJ; m++) {
        float f = 0.0f;
#pragma unroll
        for (int k = 0; k < 64 && 64 * m + k < HALF; k++) f = lane == k ? table[64 * m + k] : f;
        out.f[m] = f;
    }
    return out;
}

// The rope inputs of one wave: the raw head rows and norm weights, and the lane's part of the RoPE
// table: TABLE: the entries of its rotation pairs 8 L .. 8 L + 7, read from the step's table; else the
// frequencies of the entries it computes, inv_freq[lane + 64 m].
template <int D, bool TABLE>
struct ScoresRopeIn {
    u32x4 xa, xb, wa, wb;
    u32x4 cs[TABLE ? 2 : 1], sn[TABLE ? 2 : 1];
    float freq[RopeShape<D>::NJ];
    __device__ float operator[](int j) const { return freq[j >> 6]; }  // j = lane + 64 m
};

// Waves 0 .. QWAVES-1 take the kv head's REP query heads (HPW per wave, the qk_norm_rope_kernel
// lane layout); wave QWAVES the key head. Every wave issues the requests, the others' read nothing
// (empty buffers), so no branch joins before the key rows. Returns whether the wave has heads (wave
// QWAVES: if the item holds the position).
template <int D, int REP, bool TABLE>
__device__ __forceinline__ bool rope_request(const AttnRopeArgs &r, int g, ScoresRopeIn<D, TABLE> &in) {
    constexpr int LH = D / 16, HPW = 64 / LH, HALF = D / 2;
    constexpr int QWAVES = (REP + HPW - 1) / HPW;
    static_assert(QWAVES < 4 && HPW >= 2, "rope waves");
    const int w = wave_id();
    const int lane = tid_x() & 63, hg = lane / LH, L = lane % LH;
    const bool is_k = w == QWAVES, any = w <= QWAVES;
    const int hl0 = is_k ? 0 : w * HPW;
    const int n_h = !any ? 0 : is_k ? 1 : min(HPW, REP - hl0);
    const bf16 *src = is_k ? r.k + (size_t)g * D : r.at.q + ((size_t)g * REP + hl0) * D;
    // the wave's heads as one wave-uniform buffer: loads past the last head read zeros
    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)src, (short)0, n_h * D * 2, BUFFER_FLAGS);
    const int oa = hg * D * 2 + 16 * L, ob = oa + 2 * HALF;
    in.xa = __builtin_amdgcn_raw_buffer_load_b128(xr, oa, 0, 0);
    in.xb = __builtin_amdgcn_raw_buffer_load_b128(xr, ob, 0, 0);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(is_k ? r.kn : r.qn), (short)0, any ? D * 2 : 0, BUFFER_FLAGS);
    in.wa = __builtin_amdgcn_raw_buffer_load_b128(wr, 16 * L, 0, 0);
    in.wb = __builtin_amdgcn_raw_buffer_load_b128(wr, 16 * L + 2 * HALF, 0, 0);
    if constexpr (TABLE) {
        const __amdgpu_buffer_rsrc_t tr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)r.table, (short)0, any ? 2 * HALF * 4 : 0, BUFFER_FLAGS);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            in.cs[i] = __builtin_amdgcn_raw_buffer_load_b128(tr, 32 * L + 16 * i, 0, 0);
            in.sn[i] = __builtin_amdgcn_raw_buffer_load_b128(tr, HALF * 4 + 32 * L + 16 * i, 0, 0);
        }
    } else {
        // in the argument segment itself (the address of the by-value argument would be a copy's)
        const char *args = (const char *)__builtin_amdgcn_kernarg_segment_ptr();
        const __amdgpu_buffer_rsrc_t fr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(args + offsetof(AttnRopeArgs, inv_freq)), (short)0, any ? HALF * 4 : 0,
            BUFFER_FLAGS);
#pragma unroll
        for (int m = 0; m < RopeShape<D>::NJ; m++)
            in.freq[m] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(fr, 4 * (lane + 64 * m), 0, 0));
    }
    return any;
}

// QK-norm + RoPE of the requested heads into q_out / k_out (LDS); the key wave also writes k'
// and (its next group of lanes) the value row into the caches' row pos.
template <int D, int REP, bool TABLE>
__device__ __forceinline__ void rope_finish(const AttnRopeArgs &r, int g, int pos,
                                            const ScoresRopeIn<D, TABLE> &in, u32x4 *q_out,
                                            u32x4 *k_out) {
    constexpr int LH = D / 16, HPW = 64 / LH, HALF = D / 2;
    constexpr int QWAVES = (REP + HPW - 1) / HPW;
    const int w = wave_id();
    const int lane = tid_x() & 63, hg = lane / LH, L = lane % LH;
    const bool is_k = w == QWAVES;
    const int hl0 = is_k ? 0 : w * HPW;
    const int n_h = is_k ? 1 : min(HPW, REP - hl0);
    const size_t kv_dim = (size_t)r.at.n_kv_heads * D;
    u32x4 ya, yb, va, vb;
    float c[8], s[8];
    if constexpr (TABLE) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const u32x4 &cw = in.cs[e / 4], &sw = in.sn[e / 4];
            c[e] = __uint_as_float(e % 4 == 0 ? cw.x : e % 4 == 1 ? cw.y : e % 4 == 2 ? cw.z : cw.w);
            s[e] = __uint_as_float(e % 4 == 0 ? sw.x : e % 4 == 1 ? sw.y : e % 4 == 2 ? sw.z : sw.w);
        }
    } else {
        float cs[RopeShape<D>::NJ], sn[RopeShape<D>::NJ];
        rope_table<D>(pos, in, cs, sn);
        rope_fetch<D>(cs, sn, L, c, s);
    }
    norm_rope_with<D>(in.xa, in.xb, in.wa, in.wb, r.eps, c, s, ya, yb, va, vb);
    if (hg < n_h) {
        u32x4 *dst = is_k ? k_out : q_out + (hl0 + hg) * (D / 8);
        dst[L] = va;
        dst[HALF / 8 + L] = vb;
        if (is_k) {
            bf16 *row = r.kc_w + (size_t)pos * kv_dim + (size_t)g * D;
            st16(row + 8 * L, va);
            st16(row + HALF + 8 * L, vb);
        }
    } else if (is_k && hg == 1) {  // the next group of lanes copies the value row
        const bf16 *vsrc = r.v + (size_t)g * D;
        bf16 *row = r.vc_w + (size_t)pos * kv_dim + (size_t)g * D;
        st16(row + 8 * L, ld16(vsrc + 8 * L));
        st16(row + HALF + 8 * L, ld16(vsrc + HALF + 8 * L));
    }
}

// TABLE: the RoPE table comes from r.table, each lane its own entries, instead of being computed in
// double precision by every item and fetched from the lanes that computed them. The kernel then fits 96
// registers without spills for D <= 128 and REP <= 4 (five workgroups per CU instead of four: Qwen3-4B's
// 1056 items at 8448 positions are resident in one wave of 1280 slots) and its items' rope chain is
// shorter.
//
// Bound by its chain (the heads' norm and rotation, the products, the exponentials) beside the key
// stream. With the table's entries shuffled in 16 steps, a branch around each key row's load and lane
// values held over the item loop, the Qwen3-1.7B hipGraph step took 1189 us after 5000 positions and
// 1287 after 8300, 4B 2099 after 4300 and 2249 after 8200; now 1153, 1246, 2070 and 2200. (Requesting
// the rope inputs, or the next pass's statistics, before the position is known changed nothing.)
template <int D, int REP, bool TABLE>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(TABLE && D <= 128 && REP <= 4 ? 5 : 1)))
void attn_rope_scores_kernel(AttnRopeArgs r) {
    constexpr int LP = D / 8, PPW = 64 / LP, PER_WAVE = ATT_B / 4, ITERS = PER_WAVE / PPW;
    constexpr int LH = D / 16, QWAVES = (REP + 64 / LH - 1) / (64 / LH);
    const AttnArgs &a = r.at;
    __shared__ float sc[REP][ATT_B];
    __shared__ u32x4 qk_s[(REP + 1) * (D / 8)];  // the roped query heads, then the key
    const int w = wave_id();
    const int kv_dim = a.n_kv_heads * D;
    const int pos = *a.d_pos;
    ScoresRopeIn<D, TABLE> in;
    bool roper = rope_request<D, REP>(r, (int)blockIdx.x % a.n_kv_heads, in);
    __builtin_amdgcn_sched_barrier(0);  // ahead of the key rows
    const int n = pos + 1;
    if (!position_held(a, n)) return position_error(a);
    const int nb = (n + ATT_B - 1) / ATT_B;
    for (int item = blockIdx.x; item < nb * a.n_kv_heads; item += gridDim.x) {
        const int b = item / a.n_kv_heads, g = item - b * a.n_kv_heads;
        if (item != (int)blockIdx.x) {
            __syncthreads();  // the previous item's LDS has been read
            roper = rope_request<D, REP>(r, g, in);
        }
        const int lane = tid_x() & 63, G = lane / LP, L = lane % LP;  // not held over the loop
        u32x4 kv[ITERS];
        request_rows<D, ITERS>(a.kc, kv_dim, b, g, pos, w * PER_WAVE + G, L, kv);
        asm volatile("" ::: "memory");  // the key rows are requested before the rotation
        if (roper && (w < QWAVES || b == nb - 1))
            rope_finish<D, REP, TABLE>(r, g, pos, in, qk_s, qk_s + REP * (D / 8));
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITERS; it++)
            if (b * ATT_B + w * PER_WAVE + it * PPW + G == pos) kv[it] = qk_s[REP * (D / 8) + L];
        // the scores of attn_scores_kernel
        constexpr int NP = ITERS * REP, SL = NP < LP ? NP : LP;
        float part[NP];
#pragma unroll
        for (int it = 0; it < ITERS; it++)
#pragma unroll
            for (int q = 0; q < REP; q++) part[it * REP + q] = dot8(qk_s[q * (D / 8) + L], kv[it], 0.0f);
#pragma unroll
        for (int s0 = 0; s0 < NP; s0 += SL) {
            float slice[SL];
#pragma unroll
            for (int j = 0; j < SL; j++) slice[j] = part[s0 + j];
            const float d = group_sum_scatter<LP, SL>(slice);
            const int j = s0 + scatter_row<SL>(L), it = j / REP, q = j - it * REP;
            const int slot = w * PER_WAVE + it * PPW + G;
            const int t = b * ATT_B + slot;
            const float s = round_bf(round_bf(d) * a.scale);
            if (L < SL) {
                sc[q][slot] = s;
                if (t < n) a.scores[(size_t)(g * REP + q) * a.max_seq + t] = s;
            }
        }
        __syncthreads();
        for (int q = w; q < REP; q += 4) {
            const bool v = b * ATT_B + lane < n;
            const float s = v ? sc[q][lane] : -__builtin_huge_valf();
            const float m = wave_max(s);
            const float e = v ? exp_f32(s - m) : 0.0f;
            const float S = wave_sum(e);
            if (lane == 0) {
                float *st = a.stats + ((size_t)(g * REP + q) * a.max_blocks + b) * 2;
                st[0] = m;
                st[1] = S;
            }
        }
    }
}

// Pass 2, per (block, kv head): each query head's global max M and sum (chunks of 64 block
// statistics: tree sum of S_b exp(m_b - M), chunks added in order), the block's probabilities
// p = bf16(exp(s - M) / sum), then p v accumulated per lane over its positions, tree over the
// position groups of a wave, waves added in order 0..3.
// One item of pass 2, block b of kv head g: the probabilities of the block's positions for the
// REP query heads, and the block's partial output sum p v of each head, handed over as
// store(index into the [n_heads, max_blocks, D] partials, value).
template <int D, int REP, class Store>
__device__ __forceinline__ void pv_item(const AttnArgs &a, int b, int g, int n, int nb,
                                        float (&p_s)[REP][ATT_B], float (&red)[4][REP][D],
                                        Store store) {
    constexpr int LP = D / 8, PPW = 64 / LP, PER_WAVE = ATT_B / 4, ITERS = PER_WAVE / PPW;
    // not held over attn_pv_kernel's items, in which they took up to 15 registers: a PV pass of its own is
    // 0.1 to 0.6 us shorter (8 heads on 8 of 256 at 4000 positions 13.1 -> 12.5 an attention_forward)
    const int lane = tid_x() & 63, w = wave_id();
    const int G = lane / LP, L = lane % LP;
    const int kv_dim = a.n_kv_heads * D;
    // The first head of this wave (r = w, where it has one): its score and block statistics are
    // requested before the values. Loads complete in order, so the statistics chain then waits only
    // for them and runs while the values stream. Unconditional (clamped indices), so no branch joins
    // before the value requests.
    constexpr int MAXC = 4;  // chunks of 64 block statistics held in registers
    // (which waves have heads turns with the workgroups of a CU, 256 apart, for heads of 128 and more:
    // those with REP < 4 leave waves idle here; 8 heads on 1 of 128 at 2000 positions 21.3 -> 21.1 us a
    // block, the 1.7B hipGraph step after 5000 1152 -> 1146 us; of 64 it measured 0.8% slower)
    const int wu = (wave_id() + (D >= 128 ? (int)(blockIdx.x >> 8) : 0)) & 3;
    float mv0[MAXC], sv0[MAXC], s_t0;
    {
        const int h = g * REP + (wu < REP ? wu : 0);
        const float *st = a.stats + (size_t)h * a.max_blocks * 2;
        s_t0 = a.scores[(size_t)h * a.max_seq + min(b * ATT_B + lane, n - 1)];
#pragma unroll
        for (int c = 0; c < MAXC; c++) {
            const int bi = min(c * 64 + lane, nb - 1);
            mv0[c] = block_max(st, bi);
            sv0[c] = st[2 * bi + 1];
        }
    }
    // every lane requests a value row (positions past n clamped to n - 1: the PV loop skips
    // those slots), so no load sits on some paths only and no wait is made conservative
    u32x4 vv[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
        const int t = min(b * ATT_B + w * PER_WAVE + it * PPW + G, n - 1);
        vv[it] = ld16_nt(a.vc + (size_t)t * kv_dim + g * D + 8 * L);
    }
    asm volatile("" ::: "memory");  // the requests stay ahead of the branches below
    // The probability of this lane's position from its score and the head's block statistics (at
    // most C chunks of 64). The max is exact in any order, so over the lane's chunks first and then
    // one wave_max; the chunk sums (wave_sum of each, scattered over the lanes) are added in order.
    const auto prob = [&](auto chunks, float s_t, const float (&mv)[MAXC], const float (&sv)[MAXC]) {
        constexpr int C = decltype(chunks)::value, B = C == 3 ? 4 : C;
        float ml = -__builtin_huge_valf();
#pragma unroll
        for (int c = 0; c < C; c++) ml = c * 64 + lane < nb ? fmaxf(ml, mv[c]) : ml;
        const float M = wave_max(ml);
        float term[B];
#pragma unroll
        for (int c = 0; c < B; c++)
            term[c] = c < C && c * 64 + lane < nb ? sv[c] * exp_f32(mv[c] - M) : 0.0f;
        const float totals = wave_sum_scatter<B>(term);
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < C; c++) {
            // chunk c's total is in the lane that scatter_row maps to it
            const int at = B == 4 ? ((c & 1) << 1 | c >> 1) : c;
            const float cs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(totals), at));
            sum = c == 0 ? cs : sum + cs;
        }
        return b * ATT_B + lane < n ? round_bf(exp_f32(s_t - M) / sum) : 0.0f;
    };
    const auto prob_of = [&](float s_t, const float (&mv)[MAXC], const float (&sv)[MAXC]) {
        if (nb <= 64) return prob(std::integral_constant<int, 1>{}, s_t, mv, sv);
        if (nb <= 128) return prob(std::integral_constant<int, 2>{}, s_t, mv, sv);
        if (nb <= 192) return prob(std::integral_constant<int, 3>{}, s_t, mv, sv);
        return prob(std::integral_constant<int, MAXC>{}, s_t, mv, sv);
    };
    static_assert(MAXC == 4, "chunk counts");
    for (int r = wu; r < REP; r += 4) {
        if (nb <= 64 * MAXC) {
            if (r == wu) {
                p_s[r][lane] = prob_of(s_t0, mv0, sv0);
                continue;
            }
            // a second head of the wave (REP = 8): every statistic requested at once
            const int h = g * REP + r;
            const float *st = a.stats + (size_t)h * a.max_blocks * 2;
            const float s_t = a.scores[(size_t)h * a.max_seq + min(b * ATT_B + lane, n - 1)];
            float mv[MAXC], sv[MAXC];
#pragma unroll
            for (int c = 0; c < MAXC; c++) {
                const int bi = min(c * 64 + lane, nb - 1);
                mv[c] = block_max(st, bi);
                sv[c] = st[2 * bi + 1];
            }
            p_s[r][lane] = prob_of(s_t, mv, sv);
            continue;
        }
        // more than 64 * MAXC blocks
        const int h = g * REP + r;
        const float *st = a.stats + (size_t)h * a.max_blocks * 2;
        const int t = b * ATT_B + lane;
        const float s_t = a.scores[(size_t)h * a.max_seq + min(t, n - 1)];
        float M = -__builtin_huge_valf(), sum = 0.0f;
        for (int c0 = 0; c0 < nb; c0 += 64) {
            const int bi = c0 + lane;
            M = fmaxf(M, wave_max(bi < nb ? block_max(st, bi) : -__builtin_huge_valf()));
        }
        for (int c0 = 0; c0 < nb; c0 += 64) {
            const int bi = c0 + lane;
            const float term = bi < nb ? st[2 * bi + 1] * exp_f32(block_max(st, bi) - M) : 0.0f;
            const float cs = wave_sum(term);
            sum = c0 == 0 ? cs : sum + cs;
        }
        p_s[r][lane] = t < n ? round_bf(exp_f32(s_t - M) / sum) : 0.0f;
    }
    __syncthreads();
    float acc[REP][8];
#pragma unroll
    for (int r = 0; r < REP; r++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[r][e] = 0.0f;
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
        const int slot = w * PER_WAVE + it * PPW + G;
        if (b * ATT_B + slot < n) {
#pragma unroll
            for (int r = 0; r < REP; r++) {
                const float p = p_s[r][slot];
#pragma unroll
                for (int e = 0; e < 8; e++) acc[r][e] = fmaf(p, elem(vv[it], e), acc[r][e]);
            }
        }
    }
    // the position groups (lanes LP apart) summed with the pairing of butterfly_sum<LP, 64>,
    // reduce-scattered: each lane keeps REP * 8 / (64 / LP) of the values, at offset `off`
    constexpr int NV = REP * 8, NG = 64 / LP, KEEP = NV / NG;
    float flat[NV], kept[KEEP];
#pragma unroll
    for (int r = 0; r < REP; r++)
#pragma unroll
        for (int e = 0; e < 8; e++) flat[r * 8 + e] = acc[r][e];
    scatter_keep<NV, LP, 64>(flat, kept);
    int off = 0;
#pragma unroll
    for (int k = 0, m = NV; (LP << k) < 64; k++, m >>= 1)
        if ((lane >> k) & LP) off += m / 2;
#pragma unroll
    for (int j = 0; j < KEEP; j++) {
        const int idx = off + j, r = idx / 8, e = idx % 8;
        red[w][r][8 * L + e] = kept[j];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < REP * D; i += 256) {
        const int r = i / D, d = i - r * D;
        const float v = ((red[0][r][d] + red[1][r][d]) + red[2][r][d]) + red[3][r][d];
        store(((size_t)(g * REP + r) * a.max_blocks + b) * D + d, v);
    }
}

template <int D, int REP>
__global__ __launch_bounds__(256) void attn_pv_kernel(AttnArgs a) {
    __shared__ float p_s[REP][ATT_B];
    __shared__ float red[4][REP][D];
    const int n = *a.d_pos + 1;
    if (!position_held(a, n)) return;
    const int nb = (n + ATT_B - 1) / ATT_B;
    for (int item = blockIdx.x; item < nb * a.n_kv_heads; item += gridDim.x) {
        const int b = item / a.n_kv_heads, g = item - b * a.n_kv_heads;
        pv_item<D, REP>(a, b, g, n, nb, p_s, red,
                        [&](size_t i, float v) { a.partial[i] = v; });
        __syncthreads();
    }
}

// Pass 3: out = bf16(block partials added in block order). A workgroup takes COMBINE_COLS
// columns of one query head (D / COMBINE_COLS workgroups per head, so the loads spread over
// more CUs). The additions are sequential, the loads are not: the columns' partials are staged
// in LDS by all 256 threads (every 16-byte load of a chunk of CB blocks in flight at once), then
// thread c adds column c in block order, 16 LDS reads at a time, the next 16 in flight meanwhile (with
// a test around each addition and no reads ahead, 32 heads on 8 of 128 at 8300 positions took 18.1 us
// instead of 16.6, 1 on 1 of 64 at 16000 13.8 instead of 11.1).
constexpr int COMBINE_COLS = 32;
template <int D>
__global__ __launch_bounds__(256) void attn_combine_kernel(AttnArgs a) {
    constexpr int CC = COMBINE_COLS, Q = CC / 4;  // columns; 16-byte loads per block row
    constexpr int CB = 256;                      // blocks per LDS chunk (32 KB, 16384 positions)
    static_assert(D % CC == 0, "columns per workgroup");
    __shared__ float part[CB * CC];
    const int h = blockIdx.x / (D / CC), c0 = (blockIdx.x % (D / CC)) * CC;
    const float *src = a.partial + (size_t)h * a.max_blocks * D + c0;
    float acc = -0.0f;  // -0 + x is x, also for x = -0
    // The first chunk's loads cover min(CB, max_blocks) blocks, whatever the history, and the
    // position is read after them (a per-lane load: as a uniform value it would be loaded, and
    // waited for, before them): one round trip instead of two. Blocks past the history are
    // loaded and not added. Later chunks are those of the history (loaded for caches of more than 16384
    // positions whatever the history, one cost 0.4 us at 12345).
    int nb = a.max_blocks;
    for (int b0 = 0; b0 < nb; b0 += CB) {
        if (b0 > 0) __syncthreads();  // the previous chunk has been added
        constexpr int PER = CB * Q / 256;  // 16-byte loads per thread for a full chunk
        const int n4 = min(CB, nb - b0) * Q;
        u32x4 v4[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            // load i: block b0 + i / Q, columns c0 + 4 (i % Q) .. + 3
            const int i = min((int)threadIdx.x + 256 * j, n4 - 1);
            v4[j] = *(const u32x4 *)(src + (size_t)(b0 + i / Q) * D + 4 * (i % Q));
        }
        const int n = a.d_pos[tid_x() >> 31] + 1;
        // staged before the history is looked at, so the loads above cannot be moved past it
#pragma unroll
        for (int j = 0; j < PER; j++)
            if ((int)threadIdx.x + 256 * j < n4) ((u32x4 *)part)[threadIdx.x + 256 * j] = v4[j];
        nb = __builtin_amdgcn_readfirstlane(position_held(a, n) ? (n + ATT_B - 1) / ATT_B : 0);
        const int cnt = min(CB, nb - b0);
        __syncthreads();
        if (threadIdx.x < CC) {
            // in block order; 16 are added while the next 16 are read
            const float *col = part + threadIdx.x;
            const int whole = cnt & ~15;
            float v[16], next[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = col[u * CC];
            for (int j = 0; j < whole; j += 16) {
#pragma unroll
                for (int u = 0; u < 16; u++) next[u] = col[(min(j + 16, CB - 16) + u) * CC];
#pragma unroll
                for (int u = 0; u < 16; u++) acc += v[u];
#pragma unroll
                for (int u = 0; u < 16; u++) v[u] = next[u];
            }
#pragma unroll
            for (int u = 0; u < 15; u++)
                if (whole + u < cnt) acc += v[u];
        }
    }
    if (threadIdx.x < CC) a.out[(size_t)h * D + c0 + threadIdx.x] = nb > 0 ? (bf16)f2bf(acc) : 0;
}

// ------------------------------------------------------------------------------------------
// One-pass attention of the step: QK-norm + RoPE, the scores, the split softmax, PV and the
// combine in ONE launch, with the arithmetic of qk_norm_rope_kernel followed by
// attn_scores/pv/combine (the same bits; blocks of 64 positions as there). Workgroup (g, i), i
// < ipk, of kv head g takes the blocks i, i + ipk, i + 2 ipk, ... of the history. The split
// softmax has two global steps: every block's statistics before any probability, every block's
// partial output before the combine. They are handoffs between the ipk workgroups of a kv head,
// as tagged 64-bit words (float bits << 32 | tag, agent-scope atomic stores and loads; the tag
// names the launch), so the data is its own ready signal: no counter, no fence, no grid
// barrier. The combine is split by columns: workgroup i adds, in block order, the partials of
// its columns of the kv head's query heads. Each workgroup counts its launches in a word of
// its own (one cache line each: the count every wave reads at the start is not one line that
// the whole grid queues on), so the tag is that count + 1.
//
// Workgroups wait for each other, so all must be resident: the grid never exceeds the CU count
// (one 512-thread workgroup per CU fits), and every wait is bounded (on timeout the error flag
// is set and the kernel finishes with what it read).
// ------------------------------------------------------------------------------------------

constexpr int OP_WAVES = 8, OP_THREADS = 64 * OP_WAVES;
constexpr int OP_PRE = 3;          // rounds (two blocks each) whose K/V rows are requested first
constexpr int OP_MAXJ = 16;        // blocks of one workgroup (scores and probabilities in LDS)
constexpr int OP_MAXB = 512;       // blocks of the history (32768 positions)
constexpr int OP_MAXCPI = 32;      // combine columns of one workgroup
constexpr int OP_STAGE = 8192;     // floats staged: statistics, or a chunk of combine partials
constexpr long long OP_SPIN_LIMIT = 1 << 22;
constexpr int OP_MAXGRID = 1024;   // workgroups (launch counters in the workspace)
constexpr int OP_CTR_STRIDE = 16;  // 8-byte words between two counters (128 bytes)
constexpr size_t OP_HEADER = (size_t)OP_MAXGRID * OP_CTR_STRIDE * 8;

struct OnePassArgs {
    AttnRopeArgs r;                  // r.at.q: the query before QK-norm + RoPE; r.at.out: output
    unsigned long long *tstats;      // [n_heads, max_blocks, 2] tagged block max, block sum
    unsigned long long *tpart;       // [n_heads, max_blocks, D] tagged block partial outputs
    unsigned long long *launches;    // per workgroup (OP_CTR_STRIDE words apart): its launches
    int *err;                        // set to 2 when a wait times out
    int ipk;                         // workgroups per kv head
    int cpi;                         // combine columns per workgroup
};

__device__ __forceinline__ unsigned long long op_ld(const unsigned long long *p) {
    return __hip_atomic_load(gptr((unsigned long long *)p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void op_st(unsigned long long *p, float v, uint32_t tag) {
    __hip_atomic_store(gptr(p), ((unsigned long long)__float_as_uint(v) << 32) | tag,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls the tagged words addr(idx), idx = threadIdx.x + NT k < total (NT threads in the
// workgroup, K words of a thread in flight), until every tag is `tag`, and hands each value to
// put(idx, value). Bounded: once *err is set (by another wait or an earlier error), or when its
// own polls run out (then *err = 2 unless already set), it goes on with what it read.
template <int NT = OP_THREADS, int K = 8, class Addr, class Put>
__device__ __forceinline__ void op_poll(int total, uint32_t tag, int *err, Addr addr, Put put) {
    for (int base = 0; base < total; base += NT * K) {
        unsigned long long wv[K];
        long long spins = 0;
        for (;;) {
            bool fresh = true;
#pragma unroll
            for (int k = 0; k < K; k++) {
                const int idx = base + (int)threadIdx.x + NT * k;
                wv[k] = idx < total ? op_ld(addr(idx)) : 0ull;
                fresh &= idx >= total || (uint32_t)wv[k] == tag;
            }
            if (fresh) break;
            if ((++spins & 15) == 0 && wait_gives_up(spins, OP_SPIN_LIMIT, err)) break;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int idx = base + (int)threadIdx.x + NT * k;
            if (idx < total) put(idx, __uint_as_float((uint32_t)(wv[k] >> 32)));
        }
    }
}

template <int REP>
__global__ __launch_bounds__(OP_THREADS) void attn_one_pass_kernel(OnePassArgs o) {
    constexpr int D = 128, LP = D / 8, PPW = 64 / LP, ITERS = ATT_B / 4 / PPW;
    static_assert(ITERS == 4, "a wave takes a quarter (16 positions) of a block");
    constexpr int MAXC = 4;  // chunks of 64 block statistics held in registers
    const AttnRopeArgs &r = o.r;
    const AttnArgs &a = r.at;
    __shared__ u32x4 qk_s[(REP + 1) * (D / 8)];  // the roped query heads, then the key
    __shared__ float sc[REP][OP_MAXJ][ATT_B];    // scores, then probabilities
    __shared__ float red[2][4][REP][D];          // PV quarters of a round's two blocks
    __shared__ float stage[OP_STAGE];            // statistics / a chunk of combine partials
    __shared__ float gstat[REP][2];              // each head's global max and sum
    __shared__ unsigned long long launch_s;

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = w >> 2, qtr = w & 3;  // block of a round, quarter of the block
    const int G = lane / LP, L = lane % LP;
    const int ipk = o.ipk;
    const int g = blockIdx.x / ipk, i = blockIdx.x - g * ipk;
    const int pos = *a.d_pos;
    if (pos < 0 || pos >= a.max_seq) {  // every workgroup reads the same pos: all return
        if (threadIdx.x == 0) *o.err = 1;
        return;
    }
    const int n = pos + 1;
    const int nb = (n + ATT_B - 1) / ATT_B;
    const int nj = nb > i ? (nb - i + ipk - 1) / ipk : 0;  // blocks of this workgroup
    const bool owner = (pos / ATT_B) % ipk == i;            // holds the block of pos
    const int row_bytes = a.n_kv_heads * D * 2;
    auto slot_pos = [&](int j, int it) {  // position of this lane's slot `it` in block j
        return (i + ipk * j) * ATT_B + qtr * 16 + it * PPW + G;
    };
    // The kv head's K and V history as buffers over rows 0..pos-1: a lane's load of a row at or
    // past pos, or of a block this workgroup does not have (offset past the end), returns zeros
    // without a memory access. Every load is then unconditional, so each wait below waits
    // exactly for the rows it needs (loads complete in order).
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.kc + g * D), (short)0, pos * row_bytes, BUFFER_FLAGS);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.vc + g * D), (short)0, pos * row_bytes, BUFFER_FLAGS);
    auto off = [&](int j, int it) { return (uint32_t)(slot_pos(j, it) * row_bytes + 16 * L); };
    auto rows_of = [&](const __amdgpu_buffer_rsrc_t &all, const bf16 *base, int j) {
        return j < nj ? all : __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, 0,
                                                                BUFFER_FLAGS);
    };

    // Every request is unconditional (absent data: empty buffers), issued in the order of use:
    // the launch counter, the rope inputs (wave 0: the query heads; wave 1 of the workgroup
    // holding pos: the key head, and the value row for the cache and PV), this lane's RoPE
    // frequency, then the K and V rows of the first rounds.
    const unsigned long long launches = op_ld(o.launches + (size_t)blockIdx.x * OP_CTR_STRIDE);
    constexpr int LH = D / 16, HALF = D / 2;
    static_assert(REP <= 64 / LH, "a kv head's query heads in one wave");
    const bool rq_q = w == 0, rq_k = w == 1 && owner;
    const int hg = lane / LH, Lr = lane % LH;
    RopeIn<D> in;
    {
        const bf16 *src = rq_k ? r.k + (size_t)g * D : a.q + (size_t)g * REP * D;
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)src, (short)0, rq_q ? REP * D * 2 : rq_k ? D * 2 : 0, BUFFER_FLAGS);
        in.xa = __builtin_amdgcn_raw_buffer_load_b128(xr, hg * D * 2 + 16 * Lr, 0, 0);
        in.xb = __builtin_amdgcn_raw_buffer_load_b128(xr, hg * D * 2 + 16 * Lr + D, 0, 0);
        const __amdgpu_buffer_rsrc_t nr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(rq_k ? r.kn : r.qn), (short)0, rq_q || rq_k ? D * 2 : 0, BUFFER_FLAGS);
        in.wa = __builtin_amdgcn_raw_buffer_load_b128(nr, 16 * Lr, 0, 0);
        in.wb = __builtin_amdgcn_raw_buffer_load_b128(nr, 16 * Lr + D, 0, 0);
    }
    // the value row of pos: every lane of the workgroup holding pos (PV), lanes L of wave 1's
    // second head group write it to the cache
    const __amdgpu_buffer_rsrc_t vrow = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(r.v + (size_t)g * D), (short)0, owner ? D * 2 : 0, BUFFER_FLAGS);
    const u32x4 vcur = __builtin_amdgcn_raw_buffer_load_b128(vrow, 16 * L, 0, 0);
    const u32x4 vcp_a = __builtin_amdgcn_raw_buffer_load_b128(vrow, 16 * Lr, 0, 0);
    const u32x4 vcp_b = __builtin_amdgcn_raw_buffer_load_b128(vrow, 16 * Lr + D, 0, 0);
    const LaneFreq<D> freq = lane_freq<D>(r.inv_freq);
    // the small requests stay ahead of the rows (the compiler would otherwise move them after,
    // and every wait for them would wait for all the rows too)
    __builtin_amdgcn_sched_barrier(0);
    u32x4 kpre[OP_PRE][ITERS], vpre[OP_PRE][ITERS];
#pragma unroll
    for (int rd = 0; rd < OP_PRE; rd++) {
        const __amdgpu_buffer_rsrc_t kr = rows_of(krs, a.kc, 2 * rd + half);
#pragma unroll
        for (int it = 0; it < ITERS; it++)
            kpre[rd][it] = __builtin_amdgcn_raw_buffer_load_b128(kr, off(2 * rd + half, it), 0,
                                                                 BUFFER_NT);
    }
#pragma unroll
    for (int rd = 0; rd < OP_PRE; rd++) {
        const __amdgpu_buffer_rsrc_t vr = rows_of(vrs, a.vc, 2 * rd + half);
#pragma unroll
        for (int it = 0; it < ITERS; it++)
            vpre[rd][it] = __builtin_amdgcn_raw_buffer_load_b128(vr, off(2 * rd + half, it), 0,
                                                                 BUFFER_NT);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (rq_q || rq_k) rope_table<D>(pos, freq, in.cs, in.sn);  // while the rows stream
    if (threadIdx.x == 0) launch_s = launches;
    __syncthreads();
    const uint32_t tag = (uint32_t)(launch_s % 0xffffffffull) + 1u;
    // QK-norm + RoPE (qk_norm_rope_kernel lane layout): the roped query heads and key into
    // LDS; the workgroup holding pos writes k' and v into the caches' row pos
    if (rq_q || rq_k) {
        u32x4 ya, yb, va, vb;
        norm_rope<D>(in.xa, in.xb, in.wa, in.wb, r.eps, in.cs, in.sn, Lr, ya, yb, va, vb);
        const size_t row = (size_t)pos * a.n_kv_heads * D + (size_t)g * D;
        if (rq_q && hg < REP) {
            qk_s[hg * (D / 8) + Lr] = va;
            qk_s[hg * (D / 8) + HALF / 8 + Lr] = vb;
        } else if (rq_k && hg == 0) {
            qk_s[REP * (D / 8) + Lr] = va;
            qk_s[REP * (D / 8) + HALF / 8 + Lr] = vb;
            st16(r.kc_w + row + 8 * Lr, va);
            st16(r.kc_w + row + HALF + 8 * Lr, vb);
        } else if (rq_k && hg == 1) {
            st16(r.vc_w + row + 8 * Lr, vcp_a);
            st16(r.vc_w + row + HALF + 8 * Lr, vcp_b);
        }
    }
    __syncthreads();

    // scores (attn_scores_kernel): block j's quarter qtr, 16 lanes per position
    auto scores = [&](int j, const u32x4 (&kr)[ITERS]) {
        const u32x4 kcur = qk_s[REP * (D / 8) + L];
        u32x4 qv[REP];
#pragma unroll
        for (int q = 0; q < REP; q++) qv[q] = qk_s[q * (D / 8) + L];
        constexpr int NP = ITERS * REP, SL = NP < LP ? NP : LP;
        float part[NP];
#pragma unroll
        for (int it = 0; it < ITERS; it++) {
            const u32x4 kk = slot_pos(j, it) == pos ? kcur : kr[it];
#pragma unroll
            for (int q = 0; q < REP; q++) part[it * REP + q] = dot8(qv[q], kk, 0.0f);
        }
#pragma unroll
        for (int s0 = 0; s0 < NP; s0 += SL) {
            float slice[SL];
#pragma unroll
            for (int u = 0; u < SL; u++) slice[u] = part[s0 + u];
            const float d = group_sum_scatter<LP, SL>(slice);
            const int u = s0 + scatter_row<SL>(L), it = u / REP, q = u - it * REP;
            if (L < SL) sc[q][j][qtr * 16 + it * PPW + G] = round_bf(round_bf(d) * a.scale);
        }
    };
#pragma unroll
    for (int rd = 0; rd < OP_PRE; rd++)
        if (2 * rd + half < nj) scores(2 * rd + half, kpre[rd]);
    for (int j = 2 * OP_PRE + half; j < nj; j += 2) {
        u32x4 kr[ITERS];
#pragma unroll
        for (int it = 0; it < ITERS; it++)
            kr[it] = __builtin_amdgcn_raw_buffer_load_b128(rows_of(krs, a.kc, j), off(j, it), 0,
                                                           BUFFER_NT);
        scores(j, kr);
    }
    __syncthreads();

    // block statistics (max, tree sum of exp(s - max)), published tagged; two (head, block)
    // pairs per wave at a time
    for (int p0 = w; p0 < REP * nj; p0 += 2 * OP_WAVES) {
        float s2[2], m2[2], e2[2], S2[2];
        bool v2[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int p = min(p0 + u * OP_WAVES, REP * nj - 1), q = p % REP, j = p / REP;
            v2[u] = (i + ipk * j) * ATT_B + lane < n;
            s2[u] = v2[u] ? sc[q][j][lane] : -__builtin_huge_valf();
        }
#pragma unroll
        for (int u = 0; u < 2; u++) m2[u] = wave_max(s2[u]);
#pragma unroll
        for (int u = 0; u < 2; u++) e2[u] = v2[u] ? exp_f32(s2[u] - m2[u]) : 0.0f;
#pragma unroll
        for (int u = 0; u < 2; u++) S2[u] = wave_sum(e2[u]);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int p = p0 + u * OP_WAVES;
            if (p < REP * nj && lane < 2) {
                const int q = p % REP, j = p / REP, b = i + ipk * j;
                unsigned long long *st = o.tstats + ((size_t)(g * REP + q) * a.max_blocks + b) * 2;
                op_st(st + lane, lane == 0 ? m2[u] : S2[u], tag);
            }
        }
    }

    // every block's statistics of the kv head's query heads, then each head's global max and
    // sum (attn_pv_kernel order: max over all blocks; chunks of 64 blocks summed by the wave
    // tree, the chunk sums added in order)
    op_poll(REP * nb * 2, tag, o.err,
            [&](int idx) {
                const int q = idx / (2 * nb), rest = idx - q * 2 * nb;
                return o.tstats + ((size_t)(g * REP + q) * a.max_blocks) * 2 + rest;
            },
            [&](int idx, float v) { stage[idx] = v; });
    __syncthreads();
    if (w < REP) {
        const float *st = stage + w * 2 * nb;
        float M, sum;
        if (nb <= 64 * MAXC) {
            // the chunks' terms and wave sums side by side (independent chains)
            float mv[MAXC], sv[MAXC], cs[MAXC];
#pragma unroll
            for (int c = 0; c < MAXC; c++) {
                const int bi = min(c * 64 + lane, nb - 1);
                mv[c] = st[2 * bi];
                sv[c] = st[2 * bi + 1];
            }
            float ml = -__builtin_huge_valf();
#pragma unroll
            for (int c = 0; c < MAXC; c++) ml = c * 64 + lane < nb ? fmaxf(ml, mv[c]) : ml;
            M = wave_max(ml);
#pragma unroll
            for (int c = 0; c < MAXC; c++)
                cs[c] = wave_sum(c * 64 + lane < nb ? sv[c] * exp_f32(mv[c] - M) : 0.0f);
            sum = cs[0];
#pragma unroll
            for (int c = 1; c < MAXC; c++) sum = c * 64 < nb ? sum + cs[c] : sum;
        } else {
            float ml = -__builtin_huge_valf();
            for (int c0 = 0; c0 < nb; c0 += 64)
                if (c0 + lane < nb) ml = fmaxf(ml, st[2 * (c0 + lane)]);
            M = wave_max(ml);
            sum = 0.0f;
            for (int c0 = 0; c0 < nb; c0 += 64) {
                const int bi = c0 + lane;
                const float cs =
                    wave_sum(bi < nb ? st[2 * bi + 1] * exp_f32(st[2 * bi] - M) : 0.0f);
                sum = c0 == 0 ? cs : sum + cs;
            }
        }
        if (lane == 0) {
            gstat[w][0] = M;
            gstat[w][1] = sum;
        }
    }
    __syncthreads();

    // PV (attn_pv_kernel), per round of two blocks: each wave turns the scores of its quarter
    // into probabilities p = bf16(exp(s - M) / sum) (0 past the history; only this wave reads
    // them), lane (G, L) accumulates its 4 slots, the position groups meet in the butterfly's
    // pairing (reduce-scattered), the quarters are added in order 0..3, and each block's partial
    // output is published tagged
    auto pv_round = [&](int rd, const u32x4 (&vr)[ITERS]) {
        const int j = 2 * rd + half;
        if (j < nj) {
            const int b = i + ipk * j;
#pragma unroll
            for (int u = 0; u < (REP * 16 + 63) / 64; u++) {
                const int idx = lane + 64 * u, q = idx / 16, sl = qtr * 16 + idx % 16;
                if (idx < REP * 16) {
                    const float s = sc[q][j][sl];
                    sc[q][j][sl] =
                        b * ATT_B + sl < n ? round_bf(exp_f32(s - gstat[q][0]) / gstat[q][1]) : 0.0f;
                }
            }
            float acc[REP][8];
#pragma unroll
            for (int q = 0; q < REP; q++)
#pragma unroll
                for (int e = 0; e < 8; e++) acc[q][e] = 0.0f;
#pragma unroll
            for (int it = 0; it < ITERS; it++) {
                const int t = slot_pos(j, it);
                if (t < n) {
                    const u32x4 vt = t == pos ? vcur : vr[it];
#pragma unroll
                    for (int q = 0; q < REP; q++) {
                        const float p = sc[q][j][qtr * 16 + it * PPW + G];
#pragma unroll
                        for (int e = 0; e < 8; e++) acc[q][e] = fmaf(p, elem(vt, e), acc[q][e]);
                    }
                }
            }
            constexpr int NV = REP * 8, NG = 64 / LP, KEEP = NV / NG;
            float flat[NV], kept[KEEP];
#pragma unroll
            for (int q = 0; q < REP; q++)
#pragma unroll
                for (int e = 0; e < 8; e++) flat[q * 8 + e] = acc[q][e];
            scatter_keep<NV, LP, 64>(flat, kept);
            int off0 = 0;
#pragma unroll
            for (int k = 0, m = NV; (LP << k) < 64; k++, m >>= 1)
                if ((lane >> k) & LP) off0 += m / 2;
#pragma unroll
            for (int u = 0; u < KEEP; u++) {
                const int idx = off0 + u, q = idx / 8, e = idx % 8;
                red[half][qtr][q][8 * L + e] = kept[u];
            }
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < 2 * REP * D; idx += OP_THREADS) {
            const int h2 = idx / (REP * D), rest = idx - h2 * REP * D;
            const int q = rest / D, d = rest - q * D, jb = 2 * rd + h2;
            if (jb < nj) {
                const float v = ((red[h2][0][q][d] + red[h2][1][q][d]) + red[h2][2][q][d]) +
                                red[h2][3][q][d];
                const int b = i + ipk * jb;
                op_st(o.tpart + ((size_t)(g * REP + q) * a.max_blocks + b) * D + d, v, tag);
            }
        }
        __syncthreads();
    };
#pragma unroll
    for (int rd = 0; rd < OP_PRE; rd++)
        if (2 * rd < nj) pv_round(rd, vpre[rd]);
    for (int rd = OP_PRE; 2 * rd < nj; rd++) {
        u32x4 vr[ITERS];
#pragma unroll
        for (int it = 0; it < ITERS; it++)
            vr[it] = __builtin_amdgcn_raw_buffer_load_b128(rows_of(vrs, a.vc, 2 * rd + half),
                                                           off(2 * rd + half, it), 0, BUFFER_NT);
        pv_round(rd, vr);
    }

    // combine (attn_combine_kernel): columns [c0, c1) of the kv head's REP * D, each the
    // block partials added in block order, staged in chunks of the blocks
    const int c0 = i * o.cpi, c1 = min(REP * D, c0 + o.cpi), nc = c1 - c0;
    if (nc > 0) {
        const int cb = OP_STAGE / nc;  // blocks per chunk
        float acc = 0.0f;
        for (int b0 = 0; b0 < nb; b0 += cb) {
            const int cnt = min(cb, nb - b0);
            op_poll(cnt * nc, tag, o.err,
                    [&](int idx) {
                        const int bb = idx / nc, c = c0 + idx - bb * nc, q = c / D, d = c - q * D;
                        return o.tpart + ((size_t)(g * REP + q) * a.max_blocks + b0 + bb) * D + d;
                    },
                    [&](int idx, float v) { stage[idx] = v; });
            __syncthreads();
            if ((int)threadIdx.x < nc) {
                const int c = threadIdx.x;
                int j0 = 0;
                if (b0 == 0) {
                    acc = stage[c];
                    j0 = 1;
                }
                for (; j0 + 16 <= cnt; j0 += 16) {  // 16 LDS reads in flight, then the adds
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; u++) v[u] = stage[(j0 + u) * nc + c];
#pragma unroll
                    for (int u = 0; u < 16; u++) acc += v[u];
                }
                for (; j0 < cnt; j0++) acc += stage[j0 * nc + c];
            }
            __syncthreads();
        }
        if ((int)threadIdx.x < nc) {
            const int c = c0 + threadIdx.x, q = c / D, d = c - q * D;
            a.out[(size_t)(g * REP + q) * D + d] = (bf16)f2bf(acc);
        }
    }
    if (threadIdx.x == 0)
        __hip_atomic_store(gptr(o.launches + (size_t)blockIdx.x * OP_CTR_STRIDE), launch_s + 1,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

extern "C" size_t attention_one_pass_bytes(int n_heads, int head_dim, int max_seq) {
    const size_t mb = ceil_div((size_t)max_seq, ATT_B);
    return OP_HEADER + (size_t)n_heads * mb * 2 * 8 + (size_t)n_heads * mb * head_dim * 8;
}

// The workgroups per kv head of the one-pass attention on this device (0: not supported).
static int one_pass_ipk(int n_heads, int n_kv_heads, int head_dim, int max_seq) {
    if (head_dim != 128 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0) return 0;
    const int rep = n_heads / n_kv_heads;
    if (rep != 1 && rep != 2 && rep != 4 && rep != 8) return 0;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    int ipk = (cus < OP_MAXGRID ? cus : OP_MAXGRID) / n_kv_heads;
    if (ipk > 64) ipk = 64;
    const int max_blocks = (int)ceil_div((size_t)max_seq, ATT_B);
    if ((size_t)max_seq * n_kv_heads * head_dim * 2 >= ((size_t)1 << 31)) return 0;
    if (ipk < 1 || max_blocks > OP_MAXB || max_blocks > ipk * OP_MAXJ ||
        (rep * head_dim + ipk - 1) / ipk > OP_MAXCPI)
        return 0;
    return ipk;
}

extern "C" int attention_one_pass_supported(int n_heads, int n_kv_heads, int head_dim,
                                            int max_seq) {
    return one_pass_ipk(n_heads, n_kv_heads, head_dim, max_seq) > 0;
}

bool attention_one_pass_launch(bf16 *out, const bf16 *q, const bf16 *k, const bf16 *v,
                               const bf16 *q_norm_w, const bf16 *k_norm_w, bf16 *key_cache,
                               bf16 *value_cache, void *ws, int *err, const int *d_pos,
                               int n_heads, int n_kv_heads, int head_dim, float eps, float theta,
                               int max_seq, float scale, hipStream_t stream) {
    const int ipk = one_pass_ipk(n_heads, n_kv_heads, head_dim, max_seq);
    if (ipk <= 0)
        return llm_fail("attention_one_pass: no one-pass attention for %d/%d heads of %d over %d "
                        "positions on this device", n_heads, n_kv_heads, head_dim, max_seq);
    const void *ptrs[] = {out, q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, ws, err,
                          d_pos};
    for (const void *p : ptrs)
        if (!p) return llm_fail("attention_one_pass: null pointer argument");
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(q_norm_w) ||
        !aligned16(k_norm_w) || !aligned16(key_cache) || !aligned16(value_cache) ||
        ((uintptr_t)ws & 255))
        return llm_fail("attention_one_pass: q, k, v, the norm weights and the caches must be "
                        "16-byte aligned and the workspace 256-byte aligned");
    OnePassArgs o;
    memset(&o, 0, sizeof o);
    AttnArgs &a = o.r.at;
    a.out = out;
    a.q = q;
    a.kc = key_cache;
    a.vc = value_cache;
    a.d_pos = d_pos;
    a.n_heads = n_heads;
    a.n_kv_heads = n_kv_heads;
    a.max_seq = max_seq;
    a.max_blocks = (int)ceil_div((size_t)max_seq, ATT_B);
    a.scale = scale;
    o.r.k = k;
    o.r.v = v;
    o.r.qn = q_norm_w;
    o.r.kn = k_norm_w;
    o.r.kc_w = key_cache;
    o.r.vc_w = value_cache;
    o.r.eps = eps;
    rope_inv_freq_table(theta, head_dim, o.r.inv_freq);
    o.launches = (unsigned long long *)ws;
    o.tstats = (unsigned long long *)((char *)ws + OP_HEADER);
    o.tpart = o.tstats + (size_t)n_heads * a.max_blocks * 2;
    o.err = err;
    o.ipk = ipk;
    const int rep = n_heads / n_kv_heads;
    o.cpi = (rep * head_dim + ipk - 1) / ipk;
    const int grid = n_kv_heads * ipk;
    switch (rep) {
    case 1: attn_one_pass_kernel<1><<<grid, OP_THREADS, 0, stream>>>(o); break;
    case 2: attn_one_pass_kernel<2><<<grid, OP_THREADS, 0, stream>>>(o); break;
    case 4: attn_one_pass_kernel<4><<<grid, OP_THREADS, 0, stream>>>(o); break;
    default: attn_one_pass_kernel<8><<<grid, OP_THREADS, 0, stream>>>(o); break;
    }
    return LAUNCH_OK();
}

extern "C" void qk_norm_rope_attention_one_pass(bf16 *out, const bf16 *q, const bf16 *k,
                                                const bf16 *v, const bf16 *q_norm_w,
                                                const bf16 *k_norm_w, bf16 *key_cache,
                                                bf16 *value_cache, void *ws, int *err,
                                                const int *d_pos, int n_heads, int n_kv_heads,
                                                int head_dim, float eps, float theta,
                                                int max_seq, float scale, hipStream_t stream) {
    attention_one_pass_launch(out, q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, ws, err,
                              d_pos, n_heads, n_kv_heads, head_dim, eps, theta, max_seq, scale,
                              stream);
}

// ------------------------------------------------------------------------------------------
// Passes 2 and 3 in one launch (attn_pv_kernel followed by attn_combine_kernel, the same bits).
// Every item stores its block partials with agent scope and then counts itself in the low half of the
// max of its kv head's first block (block_max; the scores pass has left a zero there). The item that
// completes the count adds the kv head's partials in block order. No workgroup waits for another one:
// the launch ends whatever else runs on the device and however few of its workgroups fit at once, and
// nothing is kept from call to call.
//
// Bound by its chain (statistics, exponentials, the products, the count, the in-order sums) rather
// than by the value stream, and at long histories by the one CU that reads a kv head's partials, at
// some 50 GB/s. The lines, from attention_forward of a full history in us, one launch / two (heads on
// kv heads of head_dim, blocks):
//   16 on 8 of 128: 8 blocks 7.8 / 8.2, 64 10.9 / 11.1, 96 12.9 / 12.8, 128 15.1 / 14.5, 160 17.0 / 15.9
//   32 on 8 of 128: 8 7.8 / 8.8, 48 11.2 / 11.2, 64 12.4 / 11.9, 96 14.8 / 13.8
//   64 on 8 of 128: 8 9.9 / 11.1, 32 11.9 / 12.6, 48 14.2 / 14.3, 64 15.0 / 14.8
//   64 on 8 of 256: 8 13.1 / 13.6, 16 14.1 / 14.3, 24 16.1 / 14.7
//   1 on 1 of 64: 48 7.3 / 7.3, 64 7.9 / 7.7, 96 8.9 / 8.2; 8 on 8 of 64: 96 10.1 / 10.2, 128 11.5 / 11.0
// The host knows the longest history only, and shorter ones in the same caches gain from one launch
// (16 on 8 of 128 at 260 positions of 4096: 6.7 / 7.4). Past PVC_MAX_ITEMS the workgroups, which stay
// until their stores are acknowledged, no longer fit the device at once: 16 on 16 of 128, 64 blocks
// 12.2 / 13.0, 96 16.2 / 15.6, 128 24.3 / 18.2.
// ------------------------------------------------------------------------------------------

constexpr int PVC_MAX_FLOATS = 32768;  // partials of a kv head: blocks of the longest history x REP * D
constexpr int PVC_MAX_BLOCKS = 96;
constexpr int PVC_MAX_ITEMS = 1280;    // blocks x kv heads
static_assert(PVC_MAX_BLOCKS < 0x10000, "the count of a kv head's items fits 16 bits");

template <int D, int REP>
__global__ __launch_bounds__(256) void attn_pv_combine_kernel(AttnArgs a) {
    constexpr int COLS = REP * D;
    constexpr int C = COLS > 256 ? COLS / 256 : 1;  // columns of a thread in the combine
    constexpr int U = 32 / C;                       // blocks it requests at a time
    __shared__ float p_s[REP][ATT_B];
    __shared__ float red[4][REP][D];
    __shared__ int s_last;
    const int n = *a.d_pos + 1;
    const int nb = (n + ATT_B - 1) / ATT_B;
    if (!position_held(a, n)) {
        if ((int)blockIdx.x < a.n_kv_heads)
            for (int i = threadIdx.x; i < COLS; i += 256) a.out[(size_t)blockIdx.x * COLS + i] = 0;
        return;
    }
    if ((int)blockIdx.x >= nb * a.n_kv_heads) return;  // the grid holds every item: one each
    const int b = blockIdx.x / a.n_kv_heads, g = blockIdx.x - b * a.n_kv_heads;
    pv_item<D, REP>(a, b, g, n, nb, p_s, red, [&](size_t i, float v) {
        __hip_atomic_store(gptr(a.partial + i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
    // The partials are written through to the level all XCDs share: once every wave's stores are
    // acknowledged there, the count needs no release of its own (which writes back the whole L2).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t *count = (uint32_t *)(a.stats + (size_t)g * REP * a.max_blocks * 2);
        s_last = (int)(__hip_atomic_fetch_add(gptr(count), 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT) & 0xffff) == nb - 1;
    }
    __syncthreads();
    if (!s_last) return;
    // the partials are read with agent scope too, past this XCD's own copies of those lines
    const int c0 = threadIdx.x * C;  // columns c0 .. c0 + C - 1 of the kv head's REP * D
    if (c0 >= COLS) return;
    // the kv head's partials as one buffer: REP heads of max_blocks rows of D
    const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.partial + (size_t)g * REP * a.max_blocks * D), (short)0,
        REP * a.max_blocks * D * 4, BUFFER_FLAGS);
    const int at = (c0 / D * a.max_blocks * D + c0 % D) * 4;
    float acc[C], v[2][U][C];
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = -0.0f;  // -0 + x is x, also for x = -0
    const auto request = [&](int b0, float (&to)[U][C]) {  // past the end: the last block again
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int row = min(b0 + u, nb - 1) * D * 4;
            if constexpr (C == 1) {
                to[u][0] =
                    __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(pr, at, row, BUFFER_SC1));
            } else if constexpr (C == 2) {
                const auto w = __builtin_amdgcn_raw_buffer_load_b64(pr, at, row, BUFFER_SC1);
                to[u][0] = __uint_as_float(w[0]);
                to[u][1] = __uint_as_float(w[1]);
            } else {
#pragma unroll
                for (int c = 0; c < C; c += 4) {
                    const u32x4 w =
                        __builtin_amdgcn_raw_buffer_load_b128(pr, at + 4 * c, row, BUFFER_SC1);
                    to[u][c] = __uint_as_float(w.x);
                    to[u][c + 1] = __uint_as_float(w.y);
                    to[u][c + 2] = __uint_as_float(w.z);
                    to[u][c + 3] = __uint_as_float(w.w);
                }
            }
        }
    };
    const auto add = [&](int b0, const float (&from)[U][C]) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (b0 + u >= nb) break;
#pragma unroll
            for (int c = 0; c < C; c++) acc[c] += from[u][c];
        }
    };
    request(0, v[0]);
    for (int b0 = 0; b0 < nb; b0 += 2 * U) {
        if (b0 + U < nb) request(b0 + U, v[1]);
        add(b0, v[0]);
        if (b0 + 2 * U < nb) request(b0 + 2 * U, v[0]);
        add(b0 + U, v[1]);
    }
#pragma unroll
    for (int c = 0; c < C; c++) a.out[(size_t)g * COLS + c0 + c] = (bf16)f2bf(acc[c]);
}

// The scores pass, then PV and combine in one launch or two.
template <int D, int REP>
static void launch_attention_t(const AttnArgs &a, int grid, hipStream_t stream,
                               const AttnRopeArgs *rope = nullptr) {
    if (rope && rope->table)
        attn_rope_scores_kernel<D, REP, true><<<grid, 256, 0, stream>>>(*rope);
    else if (rope)
        attn_rope_scores_kernel<D, REP, false><<<grid, 256, 0, stream>>>(*rope);
    else
        attn_scores_kernel<D, REP><<<grid, 256, 0, stream>>>(a);
    if (!LAUNCH_OK()) return;
    if (a.max_blocks <= PVC_MAX_BLOCKS && a.max_blocks * REP * D <= PVC_MAX_FLOATS &&
        (long)a.max_blocks * a.n_kv_heads <= PVC_MAX_ITEMS) {
        attn_pv_combine_kernel<D, REP><<<grid, 256, 0, stream>>>(a);
        LAUNCH_OK();
        return;
    }
    attn_pv_kernel<D, REP><<<grid, 256, 0, stream>>>(a);
    if (!LAUNCH_OK()) return;
    attn_combine_kernel<D><<<a.n_heads * (D / COMBINE_COLS), 256, 0, stream>>>(a);
    LAUNCH_OK();
}

// Block statistics and partial outputs of attention_forward for a caller whose `att` holds only
// the reference's [n_heads, max_seq] scores (src/forward.cu:10-51 sizes it so): a library-owned
// device array of 2^22 floats (16 MiB) per device, as argmax_forward keeps its partials. Every
// value a call reads from it was written earlier in the same call, so nothing is cleared; calls
// on one device that use it must not overlap.
constexpr size_t ATTN_BLOCK_FLOATS = (size_t)1 << 22;
static __device__ __align__(256) float g_attn_blocks[ATTN_BLOCK_FLOATS];

static float *attn_blocks_on_current_device() {
    static std::mutex mu;
    static float *addr[64];
    int dev = 0;
    if (!HIP_OK(hipGetDevice(&dev))) return nullptr;
    if (dev < 0 || dev >= 64) {
        llm_fail("attention: device %d out of range", dev);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        float *p = nullptr;
        if (!HIP_OK(hipGetSymbolAddress((void **)&p, HIP_SYMBOL(g_attn_blocks)))) return nullptr;
        addr[dev] = p;
    }
    return addr[dev];
}

// Where the split softmax keeps its block statistics and partial outputs. An `att` with room for
// attention_workspace_floats() floats holds them after the scores. An `att` sized the
// reference's way, [n_heads, max_seq] floats, holds the scores only, and the rest goes to the
// library's array. A smaller `att` is an error, not an overrun. The room is what the runtime
// knows of the allocation holding `att` (a buffer carved out of a larger allocation counts to
// that allocation's end); where it knows nothing, `att` is taken to hold the whole workspace.
static bool attention_blocks(float *att, int n_heads, int head_dim, int max_seq, float **stats,
                             float **partial) {
    *stats = att + (size_t)n_heads * max_seq;
    *partial = att + attention_partial_offset(n_heads, max_seq);
    hipDeviceptr_t base = nullptr;
    size_t bytes = 0;
    if (hipMemGetAddressRange(&base, &bytes, (hipDeviceptr_t)att) != hipSuccess || !base) {
        (void)hipGetLastError();  // not a runtime allocation: nothing to check against
        return true;
    }
    const size_t avail = bytes - (size_t)((const char *)att - (const char *)base);
    const size_t need = attention_workspace_floats(n_heads, head_dim, max_seq) * sizeof(float);
    if (avail >= need) return true;
    const size_t scores = (size_t)n_heads * max_seq * sizeof(float);
    if (avail < scores)
        return llm_fail("attention: att has room for %zu bytes, fewer than the %zu of its "
                        "[%d, %d] scores", avail, scores, n_heads, max_seq);
    const size_t mb = ceil_div((size_t)max_seq, ATT_B);
    const size_t stat_floats = ceil_div((size_t)n_heads * mb * 2, 4) * 4;
    const size_t block_floats = stat_floats + (size_t)n_heads * mb * head_dim;
    if (block_floats > ATTN_BLOCK_FLOATS)
        return llm_fail("attention: att holds the [%d, %d] scores only, and the %zu floats of "
                        "block statistics and partials exceed the library's %zu (give att "
                        "attention_workspace_floats(%d, %d, %d) floats)",
                        n_heads, max_seq, block_floats, ATTN_BLOCK_FLOATS, n_heads, head_dim,
                        max_seq);
    float *blocks = attn_blocks_on_current_device();
    if (!blocks) return false;
    *stats = blocks;
    *partial = blocks + stat_floats;
    return true;
}

static bool attention_args(AttnArgs &a, int &grid, bf16 *out, const bf16 *q,
                           const bf16 *key_cache, const bf16 *value_cache, float *att,
                           int n_heads, int n_kv_heads, int head_dim, const int *d_pos,
                           int max_seq, float scale, int *err) {
    if (head_dim != 64 && head_dim != 128 && head_dim != 256)
        return llm_fail("attention: head_dim %d is not 64, 128 or 256", head_dim);
    if (n_kv_heads <= 0 || n_heads % n_kv_heads != 0)
        return llm_fail("attention: n_heads %d is not a multiple of n_kv_heads %d", n_heads,
                        n_kv_heads);
    const int rep = n_heads / n_kv_heads;
    if (rep != 1 && rep != 2 && rep != 4 && rep != 8)
        return llm_fail("attention: n_heads / n_kv_heads = %d is not 1, 2, 4 or 8", rep);
    if (max_seq <= 0) return llm_fail("attention: max_seq %d must be positive", max_seq);
    if (!aligned16(q) || !aligned16(key_cache) || !aligned16(value_cache) || !aligned16(att))
        return llm_fail("attention: q, the caches and att must be 16-byte aligned");
    float *stats = nullptr, *partial = nullptr;
    if (!attention_blocks(att, n_heads, head_dim, max_seq, &stats, &partial)) return false;
    a.out = out;
    a.q = q;
    a.kc = key_cache;
    a.vc = value_cache;
    a.max_blocks = (int)ceil_div((size_t)max_seq, ATT_B);
    a.scores = att;
    a.stats = stats;
    a.partial = partial;
    a.d_pos = d_pos;
    a.n_heads = n_heads;
    a.n_kv_heads = n_kv_heads;
    a.max_seq = max_seq;
    a.scale = scale;
    // one workgroup per (block, kv head) of the longest history, so every item of a step runs in
    // the same wave of workgroups (a fixed cap made the last few items of a long history a second
    // wave that doubled the kernel time); items beyond the current history exit at once
    const long items = (long)a.max_blocks * n_kv_heads;
    grid = (int)(items < ATTN_MAXGRID ? items : ATTN_MAXGRID);
    a.err = err;
    return true;
}

bool attention_launch(bf16 *out, const bf16 *q, const bf16 *key_cache, const bf16 *value_cache,
                      float *att, int n_heads, int n_kv_heads, int head_dim, const int *d_pos,
                      int max_seq, float scale, hipStream_t stream, int *err) {
    AttnArgs a;
    int grid = 0;
    if (!attention_args(a, grid, out, q, key_cache, value_cache, att, n_heads, n_kv_heads,
                        head_dim, d_pos, max_seq, scale, err))
        return false;
    const int rep = n_heads / n_kv_heads;
#define ATT(D_, R_)                               \
    if (head_dim == D_ && rep == R_) {            \
        launch_attention_t<D_, R_>(a, grid, stream); \
        return !llm_has_error();                  \
    }
    ATT(64, 1) ATT(64, 2) ATT(64, 4) ATT(64, 8) ATT(128, 1) ATT(128, 2) ATT(128, 4) ATT(128, 8)
    ATT(256, 1) ATT(256, 2) ATT(256, 4) ATT(256, 8)
#undef ATT
    return false;
}

extern "C" void attention_forward(bf16 *out, const bf16 *q, const bf16 *key_cache,
                                  const bf16 *value_cache, float *att, int n_heads, int n_kv_heads,
                                  int head_dim, const int *d_pos, int max_seq, float scale,
                                  hipStream_t stream) {
    attention_launch(out, q, key_cache, value_cache, att, n_heads, n_kv_heads, head_dim, d_pos,
                     max_seq, scale, stream);
}

// Workspace of attention_forward_noalloc: a library-owned device array instead of the caller's
// `att`, for callers that cannot allocate. Each device holds its own copy until the process
// ends; it keeps the last call's scores, statistics and partial outputs (every value a call
// reads was written earlier in the same call, so nothing needs clearing). Calls that overlap on
// one device race on it.
constexpr size_t ATTN_SCRATCH_FLOATS = (size_t)1 << 20;  // 4 MiB
static __device__ __align__(256) float scratch[ATTN_SCRATCH_FLOATS];

// The device address of this device's copy of `scratch`, looked up once per device with that
// device current. In host code the array's name is only a host-side stand-in, never passed to a
// kernel.
static float *scratch_on_current_device() {
    static std::mutex mu;
    static float *addr[64];
    int dev = 0;
    if (!HIP_OK(hipGetDevice(&dev))) return nullptr;
    if (dev < 0 || dev >= 64) {
        llm_fail("attention_forward_noalloc: device %d out of range", dev);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        float *p = nullptr;
        if (!HIP_OK(hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch)))) return nullptr;
        addr[dev] = p;
    }
    return addr[dev];
}

bool qk_norm_rope_attention_launch(bf16 *out, const bf16 *q, const bf16 *k, const bf16 *v,
                                   const bf16 *q_norm_w, const bf16 *k_norm_w, bf16 *key_cache,
                                   bf16 *value_cache, float *att, const int *d_pos, int n_heads,
                                   int n_kv_heads, int head_dim, float eps, float theta,
                                   int max_seq, float scale, hipStream_t stream,
                                   const float *rope_table, int *err) {
    AttnRopeArgs r;
    memset(&r, 0, sizeof r);
    int grid = 0;
    if (!attention_args(r.at, grid, out, q, key_cache, value_cache, att, n_heads, n_kv_heads,
                        head_dim, d_pos, max_seq, scale, err))
        return false;
    const void *ptrs[] = {k, v, q_norm_w, k_norm_w};
    for (const void *p : ptrs)
        if (!p || !aligned16(p))
            return llm_fail("qk_norm_rope_attention: k, v and the norm weights must be non-null "
                            "and 16-byte aligned");
    r.k = k;
    r.v = v;
    r.qn = q_norm_w;
    r.kn = k_norm_w;
    r.kc_w = key_cache;
    r.vc_w = value_cache;
    r.table = rope_table;
    r.eps = eps;
    rope_inv_freq_table(theta, head_dim, r.inv_freq);
    const int rep = n_heads / n_kv_heads;
#define ATT(D_, R_)                                        \
    if (head_dim == D_ && rep == R_) {                     \
        launch_attention_t<D_, R_>(r.at, grid, stream, &r);          \
        return !llm_has_error();                                     \
    }
    ATT(64, 1) ATT(64, 2) ATT(64, 4) ATT(64, 8) ATT(128, 1) ATT(128, 2) ATT(128, 4) ATT(128, 8)
    ATT(256, 1) ATT(256, 2) ATT(256, 4) ATT(256, 8)
#undef ATT
    return false;
}

extern "C" void qk_norm_rope_attention_forward(bf16 *out, const bf16 *q, const bf16 *k,
                                               const bf16 *v, const bf16 *q_norm_w,
                                               const bf16 *k_norm_w, bf16 *key_cache,
                                               bf16 *value_cache, float *att, const int *d_pos,
                                               int n_heads, int n_kv_heads, int head_dim,
                                               float eps, float theta, int max_seq, float scale,
                                               hipStream_t stream) {
    qk_norm_rope_attention_launch(out, q, k, v, q_norm_w, k_norm_w, key_cache, value_cache, att,
                                  d_pos, n_heads, n_kv_heads, head_dim, eps, theta, max_seq,
                                  scale, stream);
}

extern "C" void attention_forward_noalloc(bf16 *out, const bf16 *q, const bf16 *key_cache,
                                          const bf16 *value_cache, int n_heads, int n_kv_heads,
                                          int head_dim, const int *d_pos, int max_seq,
                                          float scale, hipStream_t stream) {
    if (n_heads <= 0 || head_dim <= 0 || max_seq <= 0) {
        llm_fail("attention_forward_noalloc: n_heads %d, head_dim %d and max_seq %d must be "
                 "positive", n_heads, head_dim, max_seq);
        return;
    }
    const size_t need = attention_workspace_floats(n_heads, head_dim, max_seq);
    if (need > ATTN_SCRATCH_FLOATS) {
        llm_fail("attention_forward_noalloc: %zu floats of workspace for %d heads of %d over %d "
                 "positions; the library's scratch holds %zu",
                 need, n_heads, head_dim, max_seq, ATTN_SCRATCH_FLOATS);
        return;
    }
    float *ws = scratch_on_current_device();
    if (!ws) return;
    attention_forward(out, q, key_cache, value_cache, ws, n_heads, n_kv_heads, head_dim, d_pos,
                      max_seq, scale, stream);
}

// ------------------------------------------------------------------------------------------
// temperature sampling (src/kernels.cu:546-597)
// ------------------------------------------------------------------------------------------

// Inverse-CDF sampling from softmax(x * inv_temp). The additions keep the reference's order, so the
// chosen index follows from the weights alone: the row's max; chunk k of SAMPLE_T contiguous chunks
// [k c, k c + c) adds its weights exp((x - max) * inv_temp) in order (c = ceil(n / SAMPLE_T)); the
// chunk sums are added in order for the total and walked to the chunk holding u * total (never past
// the last), then that chunk's elements to the first whose running sum passes it (-1 if none does).
//
// Two launches for long rows: sample_kernel, one workgroup, takes the max (a row of 151936 is 300 KB,
// read from L2); sample_sums_kernel spreads the weights, which are most of the work, over SAMPLE_WGS
// workgroups, and the last of them to finish adds the chunk sums and draws. The chunk sums live in one
// of SAMPLE_SLOTS library-owned slots. A call has a number, which both of its launches are given and
// which names its slot: the first launch takes the slot and leaves the max in it, together with the
// number, once for each workgroup of the second, which exchanges that word for a spent one before it
// publishes. With the slot taken by another call the first launch draws alone, as it does for rows of up
// to SAMPLE_ALONE, and the second finds no word of its number. So calls may overlap on any streams,
// whatever they share. (Two launches of one captured graph at once have one number: one takes the slot,
// the other draws alone, and whichever second launch comes first does the sums, the same ones.)
//
// Bound by two launches and the round trips in and between them (the row's max by one workgroup, the
// work's word, the sums' arrival, the sums, the drawn chunk's logits again): the additions whose order is
// fixed, 1024 for the total and some 150 in each of two chunks, take 2.6 us at 4.6 clocks each. 151936
// logits: 105-119 us on one workgroup, 19.6 us spread over 64, 17.5 us with the chains' LDS reads four
// deep and the slot taken beside the max; 73.7 us on one workgroup now. The line at SAMPLE_ALONE: alone
// 9.0 / 10.2 / 15.3 / 22.1 us at 4096 / 12288 / 16384 / 32768 logits, spread 13.4-13.8 us at each.
constexpr int SAMPLE_T = 1024;
constexpr int SAMPLE_WGS = 64, SAMPLE_ROWS = SAMPLE_T / SAMPLE_WGS;  // chunks per workgroup
constexpr int SAMPLE_PIECE = 256;  // weights of a chunk staged at a time
constexpr int SAMPLE_SLOTS = 64;
constexpr int SAMPLE_ALONE = 12288;  // longest row drawn in one launch

struct SampleSlot {
    unsigned busy;   // taken by a call (of the library's slots)
    unsigned done;   // workgroups of the second launch that have published their sums
    float pad[30];
    unsigned long long work[SAMPLE_WGS];  // of the library's: what workgroup w of the second launch does
    float sums[SAMPLE_T];
    float maxes[SAMPLE_WGS];  // of a step's slot: parts of the row's max
};
static __device__ SampleSlot g_sample_slots[SAMPLE_SLOTS];

// The draw from the SAMPLE_T chunk sums in LDS, by the whole workgroup (every thread calls it after
// a barrier). Prefix sums of non-negative weights never decrease, so the walk over the chunks is
// done on the ends of 64 segments of 16 chunks first (lane s keeps the running sum after segment s:
// the additions of the total itself), then inside one segment. One wave runs each serial chain; a
// dependent addition takes 4.6 clocks and an LDS read some 200, so four reads of 16 sums are in flight.
__device__ __forceinline__ int sample_draw(const bf16 *x, int n, float inv_temp, float u, float mx,
                                           const float *sums, float *piece, float *share) {
    const int t = threadIdx.x, lane = t & 63;
    const int chunk = (n + SAMPLE_T - 1) / SAMPLE_T;
    float v[4][16];
    if (t < 64) {
        // segments that hold chunks with elements (the sums past them are zeros, which add nothing)
        const int segs = ((n + chunk - 1) / chunk + 15) / 16;
        float total = 0.0f, end = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) ld_lds16(sums + 16 * q, v[q]);
        for (int s = 0; s < segs; s += 4) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int j = 0; j < 16; j++) total += v[q][j];
                end = lane >= s + q ? total : end;
                ld_lds16(sums + 16 * min(s + q + 4, 63), v[q]);
            }
        }
        const float target = u * total;
        const unsigned long long past = __ballot(!(end <= target));
        const int s = past ? __ffsll(past) - 1 : 63;
        float cdf = s > 0 ? __shfl(end, s - 1) : 0.0f;
        int k = 16 * s;
        ld_lds16(sums + 16 * s, v[0]);
        bool on = true;  // never past the segment: its end is past the target, or it is the last
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const float next = cdf + v[0][j];
            on = on && 16 * s + j < SAMPLE_T - 1 && next <= target;
            cdf = on ? next : cdf;
            k += on ? 1 : 0;
        }
        if (t == 0) {
            share[0] = cdf;
            share[1] = target;
            share[2] = __int_as_float(k);
        }
    }
    __syncthreads();
    const float cdf = share[0], target = share[1];
    const int k = __float_as_int(share[2]);
    const long long start = (long long)k * chunk;
    const int count = start >= n ? 0 : (int)(n - start < chunk ? n - start : chunk);
    int chosen = -1;
    float run = 0.0f;
    for (int b = 0; b < count; b += SAMPLE_PIECE) {
        const int len = min(SAMPLE_PIECE, count - b);
        if (t < SAMPLE_PIECE)
            piece[t] = t < len ? exp_f32((bf2f(x[start + b + t]) - mx) * inv_temp) : 0.0f;
        __syncthreads();
        if (t < 64 && chosen < 0) {
            // 64 running sums at a time (past the end they add zeros), lane j keeps the j-th; then
            // the first that passes
#pragma unroll
            for (int q = 0; q < 4; q++) ld_lds16(piece + 16 * q, v[q]);
            for (int j0 = 0; j0 < len && chosen < 0; j0 += 64) {
                float mine = 0.0f;
#pragma unroll
                for (int q = 0; q < 4; q++) {
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        run += v[q][j];
                        mine = lane >= 16 * q + j ? run : mine;
                    }
                    ld_lds16(piece + min(j0 + 64 + 16 * q, SAMPLE_PIECE - 16), v[q]);
                }
                const unsigned long long hit = __ballot(j0 + lane < len && cdf + mine > target);
                if (hit) chosen = (int)(start + b + j0) + __ffsll(hit) - 1;
            }
        }
        __syncthreads();
    }
    return chosen;  // in the first wave
}

// A word of SampleSlot::work: the call's number (40 bits, never 0), whether the work is still to be
// done, and the row's max, which is one of its bf16 values.
constexpr unsigned long long SAMPLE_OPEN = 1ull << 16;
__host__ __device__ __forceinline__ unsigned long long sample_open_work(unsigned long long call) {
    return call << 24 | SAMPLE_OPEN;
}

// The max of the row, then either the work of sample_sums_kernel (call != 0) or the whole draw.
// The last wave takes the slot before it reads its part of the row. vec: x is 16-byte aligned.
__global__ __launch_bounds__(SAMPLE_T) void sample_kernel(int *out, const bf16 *x, int n,
                                                          float inv_temp, float u, int vec,
                                                          unsigned long long call) {
    __shared__ __align__(16) float sums[SAMPLE_T];
    __shared__ __align__(16) float piece[SAMPLE_PIECE];
    __shared__ float wmax[SAMPLE_T / 64];
    __shared__ float share[3];
    __shared__ int s_taken;
    const int t = threadIdx.x;
    SampleSlot &sl = g_sample_slots[call % SAMPLE_SLOTS];
    if (call && t == SAMPLE_T - 64) {
        s_taken = __hip_atomic_exchange(gptr(&sl.busy), 1u, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT) == 0;
        if (s_taken)
            __hip_atomic_store(gptr(&sl.done), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float m = -__builtin_huge_valf();
    int done = 0;
    if (vec) {
        constexpr int U = 8;  // 16-byte loads of a thread in flight (past the end: the last chunk again)
        const int n_chunks = n / 8;
        for (int c0 = 0; c0 < n_chunks; c0 += U * SAMPLE_T) {
            u32x4 v[U];
#pragma unroll
            for (int i = 0; i < U; i++)
                v[i] = ld16(x + 8 * (size_t)min(c0 + i * SAMPLE_T + t, n_chunks - 1));
#pragma unroll
            for (int i = 0; i < U; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) m = fmaxf(m, elem(v[i], e));
        }
        done = n_chunks * 8;
    }
    for (int i = done + t; i < n; i += SAMPLE_T) m = fmaxf(m, bf2f(x[i]));
    m = wave_max(m);
    if ((t & 63) == 0) wmax[t >> 6] = m;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the slot's count is zero before any work is open
    __syncthreads();
    float mx = wmax[0];
#pragma unroll
    for (int w = 1; w < SAMPLE_T / 64; w++) mx = fmaxf(mx, wmax[w]);  // max: any order
    if (call && s_taken) {
        if (t < SAMPLE_WGS)
            __hip_atomic_store(gptr(&sl.work[t]), sample_open_work(call) | __float_as_uint(mx) >> 16,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const int chunk = (n + SAMPLE_T - 1) / SAMPLE_T;
    const long long start = (long long)t * chunk, end = min(start + chunk, (long long)n);
    float acc = 0.0f;
    for (long long i = start; i < end; i++) acc += exp_f32((bf2f(x[i]) - mx) * inv_temp);
    sums[t] = acc;
    __syncthreads();
    const int chosen = sample_draw(x, n, inv_temp, u, mx, sums, piece, share);
    if (t == 0) *out = chosen;
}

// A decode step draws with a slot of its own, in which sample_max_kernel has left the row's max in
// parts (traced in a sampled 4B decode: 4.5 us, against 5.6 with one workgroup). The drawn token is
// also handed to the host, with the step's error flag, in the two pinned words at mail.
struct SampleStep {
    SampleSlot *slot;  // NULL: the library's slot of the call
    int *mail;
    const int *err;
    unsigned long long call;
};

// Workgroup w's part of the row's max. vec: x is 16-byte aligned.
__global__ __launch_bounds__(256) void sample_max_kernel(SampleSlot *slot, const bf16 *x, int n, int vec) {
    __shared__ float wmax[4];
    const int t0 = blockIdx.x * 256 + threadIdx.x, stride = SAMPLE_WGS * 256;
    float m = -__builtin_huge_valf();
    const int n_chunks = vec ? n / 8 : 0;
    for (int c = t0; c < n_chunks; c += stride) {
        const u32x4 v = ld16(x + 8 * (size_t)c);
#pragma unroll
        for (int e = 0; e < 8; e++) m = fmaxf(m, elem(v, e));
    }
    for (int i = 8 * n_chunks + t0; i < n; i += stride) m = fmaxf(m, bf2f(x[i]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        slot->maxes[blockIdx.x] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
}

// Workgroup w: the sums of chunks [w SAMPLE_ROWS, (w + 1) SAMPLE_ROWS). All threads compute the
// weights of a piece of each chunk into LDS (four chunks per wave, one lane per weight), then lane r
// of the first wave adds chunk r's in order. The workgroup that publishes last draws.
__global__ __launch_bounds__(256) void sample_sums_kernel(int *out, const bf16 *x, int n,
                                                          float inv_temp, float u,
                                                          SampleStep step) {
    constexpr int R = SAMPLE_ROWS, P = SAMPLE_PIECE, RW = R / 4;
    __shared__ __align__(16) float stage[R * (P + 1)];  // padded rows: lanes 0..R-1 read one column
    __shared__ float share[3];
    __shared__ int s_last;
    __shared__ unsigned long long s_work;
    static_assert(R * (P + 1) >= SAMPLE_T + P, "the draw reuses the staging");
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int chunk = (n + SAMPLE_T - 1) / SAMPLE_T;
    const int k0 = blockIdx.x * R;
    // this lane's elements of the piece at b, clamped into the row (those past a chunk's end or the
    // row's are not added)
    uint16_t v[RW][P / 64];
    const auto request = [&](int b) {
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int j = 0; j < P / 64; j++) {
                const long long at = (long long)(k0 + w * RW + r) * chunk + b + lane + 64 * j;
                v[r][j] = x[min(at, (long long)n - 1)];
            }
    };
    request(0);  // before the wait for the max
    SampleSlot &sl = step.slot ? *step.slot : g_sample_slots[step.call % SAMPLE_SLOTS];
    float mx;
    bool mine = true;  // (of the first wave) its sums are the ones to publish
    static_assert(SAMPLE_WGS == 64, "a lane per part");
    if (step.slot) {
        mx = wave_max(sl.maxes[lane]);
    } else {
        if (t == 0)
            s_work = __hip_atomic_load(gptr(&sl.work[blockIdx.x]), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        unsigned long long word = s_work;
        // the first launch has drawn, or this work is done
        if (word >> 16 != sample_open_work(step.call) >> 16) return;
        mx = __uint_as_float((uint32_t)word << 16);
        if (t == 0)
            mine = __hip_atomic_compare_exchange_strong(gptr(&sl.work[blockIdx.x]), &word,
                                                        word ^ SAMPLE_OPEN, __ATOMIC_RELAXED,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float acc = 0.0f;
    for (int b = 0; b < chunk; b += P) {
        const int len = min(P, chunk - b);
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int j = 0; j < P / 64; j++)
                if (64 * j < len)
                    stage[(w * RW + r) * (P + 1) + lane + 64 * j] =
                        exp_f32((bf2f(v[r][j]) - mx) * inv_temp);
        if (b + P < chunk) request(b + P);
        __syncthreads();
        if (t < R) {
            // chunk k0 + t's weights of the piece that exist, in order, 16 LDS reads in flight
            const long long at = (long long)(k0 + t) * chunk + b;
            const int have = at >= n ? 0 : (int)min((long long)len, n - at);
            const float *row = stage + t * (P + 1);
            float e[2][16];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 16; i++) e[h][i] = row[16 * h + i];
            int j = 0;
            for (; j + 32 <= have; j += 32)
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int i = 0; i < 16; i++) acc += e[h][i];
#pragma unroll
                    for (int i = 0; i < 16; i++) e[h][i] = row[min(j + 32 + 16 * h, P - 16) + i];
                }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (j + 16 * h + i < have) acc += e[h][i];
        }
        __syncthreads();
    }
    if (w == 0) mine = __builtin_amdgcn_readfirstlane(mine);
    if (t < R && mine)
        __hip_atomic_store(gptr(&sl.sums[k0 + t]), acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // The sums are written through to the level all XCDs share, by this wave alone: once they are
    // acknowledged there, the arrival needs no release of its own (which writes back the whole L2).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (t == 0)
        s_last = mine && __hip_atomic_fetch_add(gptr(&sl.done), 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!s_last) return;
    float *sums = stage, *piece = stage + SAMPLE_T;
    float got[SAMPLE_T / 256];
#pragma unroll
    for (int i = 0; i < SAMPLE_T / 256; i++)
        got[i] = __hip_atomic_load(gptr(&sl.sums[t + 256 * i]), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < SAMPLE_T / 256; i++) sums[t + 256 * i] = got[i];
    __syncthreads();
    if (t == 0) {  // every sum has been read
        if (step.slot)
            __hip_atomic_store(gptr(&sl.done), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            __hip_atomic_store(gptr(&sl.busy), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int chosen = sample_draw(x, n, inv_temp, u, mx, sums, piece, share);
    if (t == 0) {
        *out = chosen;
        if (step.mail) {
            step.mail[0] = chosen;
            step.mail[1] = *step.err;
        }
    }
}

// Gives back the slot that call's first launch has taken, where the second could not be launched.
__global__ __launch_bounds__(SAMPLE_WGS) void sample_give_back_kernel(unsigned long long call) {
    SampleSlot &sl = g_sample_slots[call % SAMPLE_SLOTS];
    unsigned long long word = sl.work[threadIdx.x];
    const bool closed =
        word >> 16 == sample_open_work(call) >> 16 &&
        __hip_atomic_compare_exchange_strong(gptr(&sl.work[threadIdx.x]), &word, word ^ SAMPLE_OPEN,
                                             __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    if (__ballot(closed) == ~0ull && threadIdx.x == 0)
        __hip_atomic_store(gptr(&sl.busy), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

extern "C" void sample_forward(int *out, const bf16 *x, int n, float inv_temp, float u,
                               hipStream_t stream) {
    if (n <= 0) {
        llm_fail("sample: n %d must be positive", n);
        return;
    }
    static std::atomic<unsigned long long> calls;
    const unsigned long long call =
        n > SAMPLE_ALONE ? 1 + calls.fetch_add(1, std::memory_order_relaxed) % ((1ull << 40) - 1) : 0;
    sample_kernel<<<1, SAMPLE_T, 0, stream>>>(out, x, n, inv_temp, u, aligned16(x) ? 1 : 0, call);
    if (!LAUNCH_OK() || !call) return;
    sample_sums_kernel<<<SAMPLE_WGS, 256, 0, stream>>>(out, x, n, inv_temp, u,
                                                       SampleStep{nullptr, nullptr, nullptr, call});
    if (!LAUNCH_OK()) sample_give_back_kernel<<<1, SAMPLE_WGS, 0, stream>>>(call);
}

extern "C" int llm_sample_slots(int set) {
    std::vector<SampleSlot> slots(SAMPLE_SLOTS);
    int taken = 0;
    const size_t bytes = sizeof(SampleSlot) * SAMPLE_SLOTS;
    if (!HIP_OK(hipMemcpyFromSymbol(slots.data(), HIP_SYMBOL(g_sample_slots), bytes))) return -1;
    for (SampleSlot &slot : slots) {
        taken += slot.busy != 0;
        if (set >= 0) slot.busy = (unsigned)set;
    }
    if (set >= 0 && !HIP_OK(hipMemcpyToSymbol(HIP_SYMBOL(g_sample_slots), slots.data(), bytes))) return -1;
    return taken;
}

size_t sample_slot_bytes() { return sizeof(SampleSlot); }
bool sample_takes_one_launch(int n) { return n <= SAMPLE_ALONE; }

bool sample_step(int *out, const bf16 *x, int n, float inv_temp, float u, void *slot, int *mail,
                 const int *err, hipStream_t stream) {
    sample_max_kernel<<<SAMPLE_WGS, 256, 0, stream>>>((SampleSlot *)slot, x, n, aligned16(x) ? 1 : 0);
    if (!LAUNCH_OK()) return false;
    sample_sums_kernel<<<SAMPLE_WGS, 256, 0, stream>>>(out, x, n, inv_temp, u,
                                                       SampleStep{(SampleSlot *)slot, mail, err, 0});
    return LAUNCH_OK();
}

__global__ __launch_bounds__(256) void exp_bits_kernel(float *out, unsigned first, unsigned n,
                                                       int branches) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float x = __uint_as_float(first + (unsigned)i);
        out[i] = branches ? exp_f32<true>(x) : exp_f32(x);
    }
}

extern "C" void llm_exp_bits(float *out, unsigned first, unsigned n, int branches, hipStream_t stream) {
    exp_bits_kernel<<<4096, 256, 0, stream>>>(out, first, n, branches);
    LAUNCH_OK();
}

// ------------------------------------------------------------------------------------------
// streaming ceiling probe (measurement helper)
// ------------------------------------------------------------------------------------------

// MODE 0: read n16 chunks of a (grid-stride, four 16-byte loads in flight per thread), each
// thread's xor of its chunks to dst (one word per thread); MODE 1: dst = a; MODE 2: dst = a ^ b
// (one chunk per thread). The shapes that measured fastest for plain reads and copies on MI355X.
template <int MODE>
__global__ __launch_bounds__(256) void stream_probe_kernel(u32x4 *dst, const u32x4 *a,
                                                           const u32x4 *b, size_t n16) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if constexpr (MODE == 0) {
        // thread (block b, lane-in-block i) reads chunks b * 1024 + i + 256 u + stride j
        const size_t stride = (size_t)gridDim.x * 256 * 4;
        uint32_t acc = 0;
        for (size_t base = (size_t)blockIdx.x * 1024 + threadIdx.x; base < n16; base += stride) {
            u32x4 v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const size_t i = base + 256 * u;
                v[u] = i < n16 ? __builtin_nontemporal_load(a + i) : u32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (int u = 0; u < 4; u++) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
        }
        ((uint32_t *)dst)[t] = acc;
    } else {
        for (size_t i = t; i < n16; i += (size_t)gridDim.x * 256) {
            u32x4 v = __builtin_nontemporal_load(a + i);
            if constexpr (MODE == 2) v ^= __builtin_nontemporal_load(b + i);
            __builtin_nontemporal_store(v, dst + i);
        }
    }
}

extern "C" void hbm_stream_probe(void *dst, const void *a, const void *b, size_t n_bytes, int mode,
                                 hipStream_t stream) {
    if (mode < 0 || mode > 2 || n_bytes % 16 != 0 || !aligned16(dst) || !aligned16(a) ||
        (mode == 2 && !aligned16(b))) {
        llm_fail("hbm_stream_probe: mode %d, %zu bytes (a multiple of 16, 16-byte aligned)", mode,
                 n_bytes);
        return;
    }
    const size_t n16 = n_bytes / 16;
    if (n16 == 0) return;
    if (mode == 0) {
        stream_probe_kernel<0><<<1024, 256, 0, stream>>>((u32x4 *)dst, (const u32x4 *)a, nullptr, n16);
    } else {
        size_t blocks = (n16 + 255) / 256;
        const size_t cap = (size_t)device_cus() * 80;
        if (blocks > cap) blocks = cap;
        if (mode == 1)
            stream_probe_kernel<1><<<(unsigned)blocks, 256, 0, stream>>>((u32x4 *)dst,
                                                                        (const u32x4 *)a, nullptr, n16);
        else
            stream_probe_kernel<2><<<(unsigned)blocks, 256, 0, stream>>>(
                (u32x4 *)dst, (const u32x4 *)a, (const u32x4 *)b, n16);
    }
    LAUNCH_OK();
}

// The device read peak (bench/bandwidth.cu:25-116 read_kernel): 16-byte chunks, U non-temporal
// loads in flight per thread per round, either grid-stride over the whole buffer (CONTIG false,
// the reference's pattern) or over one contiguous range per workgroup (CONTIG true, as a GEMV's
// workgroups read their rows). The xor of the data is stored only in the unlikely case it equals
// a constant, so the loads are not removed.
template <int U, bool CONTIG>
__global__ __launch_bounds__(1024) void read_peak_kernel(const u32x4 *a, size_t n16,
                                                         uint32_t *out) {
    size_t first = 0, end = n16, stride = (size_t)gridDim.x * blockDim.x;
    size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if constexpr (CONTIG) {
        const size_t span = (n16 + gridDim.x - 1) / gridDim.x;
        first = min(n16, (size_t)blockIdx.x * span);
        end = min(n16, first + span);
        stride = blockDim.x;
        t0 = first + threadIdx.x;
    }
    uint32_t acc = 0;
    for (size_t base = t0; base < end; base += U * stride) {
        u32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const size_t i = base + u * stride;
            v[u] = i < end ? __builtin_nontemporal_load(a + i) : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; u++) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    if (acc == 0x9e3779b9u) *out = acc;
}

extern "C" void hbm_read_peak_probe(unsigned *out, const void *a, size_t n_bytes, int blocks,
                                    int threads, int loads_in_flight, int contiguous,
                                    hipStream_t stream) {
    if (n_bytes % 16 != 0 || !aligned16(a) || out == nullptr || blocks < 1 ||
        blocks > (1 << 20) || (threads != 64 && threads != 128 && threads != 256 &&
                               threads != 512 && threads != 1024) ||
        (loads_in_flight != 4 && loads_in_flight != 8 && loads_in_flight != 16) ||
        (contiguous != 0 && contiguous != 1)) {
        llm_fail("hbm_read_peak_probe: %zu bytes (a multiple of 16, 16-byte aligned), %d blocks "
                 "of %d threads (64..1024, a power of two), %d loads in flight (4, 8 or 16), "
                 "layout %d (0 grid-stride, 1 a range per workgroup)",
                 n_bytes, blocks, threads, loads_in_flight, contiguous);
        return;
    }
    if (n_bytes == 0) return;
    const u32x4 *p = (const u32x4 *)a;
    const size_t n16 = n_bytes / 16;
#define PEAK(U, C) read_peak_kernel<U, C><<<blocks, threads, 0, stream>>>(p, n16, out)
    if (contiguous) {
        if (loads_in_flight == 4) PEAK(4, true);
        else if (loads_in_flight == 8) PEAK(8, true);
        else PEAK(16, true);
    } else {
        if (loads_in_flight == 4) PEAK(4, false);
        else if (loads_in_flight == 8) PEAK(8, false);
        else PEAK(16, false);
    }
#undef PEAK
    LAUNCH_OK();
}

// The device copy peak: a grid-stride copy, each thread requesting U non-temporal 16-byte loads
// (chunks blockDim apart) before it stores them. Every chunk index is checked against n16.
template <int U>
__global__ __launch_bounds__(1024) void copy_peak_kernel(u32x4 *__restrict__ d,
                                                         const u32x4 *__restrict__ a, size_t n16) {
    const size_t tile = (size_t)blockDim.x * U, stride = (size_t)gridDim.x * tile;
    for (size_t base = (size_t)blockIdx.x * tile + threadIdx.x; base < n16; base += stride) {
        u32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const size_t i = base + (size_t)u * blockDim.x;
            v[u] = i < n16 ? __builtin_nontemporal_load(a + i) : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const size_t i = base + (size_t)u * blockDim.x;
            if (i < n16) __builtin_nontemporal_store(v[u], d + i);
        }
    }
}

extern "C" void hbm_copy_peak_probe(void *dst, const void *a, size_t n_bytes, int blocks,
                                    int threads, int chunks_in_flight, hipStream_t stream) {
    if (n_bytes % 16 != 0 || !aligned16(a) || !aligned16(dst) || blocks < 1 ||
        blocks > (1 << 20) || (threads != 64 && threads != 128 && threads != 256 &&
                               threads != 512 && threads != 1024) ||
        (chunks_in_flight != 1 && chunks_in_flight != 2 && chunks_in_flight != 4 &&
         chunks_in_flight != 8)) {
        llm_fail("hbm_copy_peak_probe: %zu bytes (a multiple of 16, 16-byte aligned), %d blocks "
                 "of %d threads (64..1024, a power of two), %d chunks in flight (1, 2, 4 or 8)",
                 n_bytes, blocks, threads, chunks_in_flight);
        return;
    }
    if (n_bytes == 0) return;
    u32x4 *d = (u32x4 *)dst;
    const u32x4 *p = (const u32x4 *)a;
    const size_t n16 = n_bytes / 16;
    if (chunks_in_flight == 1) copy_peak_kernel<1><<<blocks, threads, 0, stream>>>(d, p, n16);
    else if (chunks_in_flight == 2) copy_peak_kernel<2><<<blocks, threads, 0, stream>>>(d, p, n16);
    else if (chunks_in_flight == 4) copy_peak_kernel<4><<<blocks, threads, 0, stream>>>(d, p, n16);
    else copy_peak_kernel<8><<<blocks, threads, 0, stream>>>(d, p, n16);
    LAUNCH_OK();
}

// ------------------------------------------------------------------------------------------
// argmax (src/kernels.cu:499-544), two stages
// ------------------------------------------------------------------------------------------

constexpr int AMAX_GROUPS = 256;
// Library-owned partial results of argmax_forward (calls on one device must not overlap).
__device__ float g_amax_val[AMAX_GROUPS];
__device__ int g_amax_idx[AMAX_GROUPS];

__device__ __forceinline__ void block_amax(float &v, int &i, float *lv, int *li) {
    wave_amax(v, i);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        lv[w] = v;
        li[w] = i;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 1; k < (int)(blockDim.x >> 6); k++) amax_pair(v, i, lv[k], li[k]);
}

// A row that one workgroup reads in less time than a second launch takes. Each thread sees its elements
// in ascending order, so its largest value keeps the lowest index (the comparison of equal values by
// index lets the first -inf in, which equals the value a thread begins with).
//
// Bound by its launch and its round trips. One launch here / two launches: 2.8 / 4.4 us at 1000 values,
// 3.5 / 4.8 at 8192, 4.6 / 4.9 at 24576, 5.2 / 4.9 at 32768.
constexpr int AMAX_ALONE = 24576, AMAX_ALONE_T = 1024;
__global__ __launch_bounds__(AMAX_ALONE_T) void argmax_alone_kernel(const bf16 *x, int n, int vec,
                                                                    int *out) {
    constexpr int U = 4;  // 16-byte loads of a thread in flight
    __shared__ float lv[AMAX_ALONE_T / 64];
    __shared__ int li[AMAX_ALONE_T / 64];
    const int t = threadIdx.x;
    float v = -__builtin_huge_valf();
    int idx = INT_MAX;
    const auto take = [&](float f, int i) {
        // -inf counts as a value (lowest index); NaN does not
        if (f > v || (f == v && i < idx)) {
            v = f;
            idx = i;
        }
    };
    int done = 0;
    if (vec) {
        const int n_chunks = n / 8;
        for (int c0 = 0; c0 < n_chunks; c0 += U * AMAX_ALONE_T) {
            u32x4 ch[U];
#pragma unroll
            for (int u = 0; u < U; u++) ch[u] = ld16(x + 8 * min(c0 + u * AMAX_ALONE_T + t, n_chunks - 1));
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + u * AMAX_ALONE_T + t;
                if (c < n_chunks)
#pragma unroll
                    for (int e = 0; e < 8; e++) take(elem(ch[u], e), 8 * c + e);
            }
        }
        done = n_chunks * 8;
    }
    for (int i = done + t; i < n; i += AMAX_ALONE_T) take(bf2f(x[i]), i);
    wave_amax(v, idx);
    if ((t & 63) == 0) {
        lv[t >> 6] = v;
        li[t >> 6] = idx;
    }
    __syncthreads();
    if (t < 64) {
        v = t < AMAX_ALONE_T / 64 ? lv[t] : -__builtin_huge_valf();
        idx = t < AMAX_ALONE_T / 64 ? li[t] : INT_MAX;
        wave_amax(v, idx);
        if (t == 0) *out = idx;
    }
}

__global__ __launch_bounds__(256) void argmax_stage1_kernel(const bf16 *x, int n, int vec,
                                                            float *pv, int *pi) {
    __shared__ float lv[4];
    __shared__ int li[4];
    float v = -__builtin_huge_valf();
    int idx = INT_MAX;
    const int stride = gridDim.x * blockDim.x;
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
    int done = 0;
    if (vec) {
        const int n_chunks = n / 8;
        for (int c = t0; c < n_chunks; c += stride) {
            const u32x4 ch = ld16(x + 8 * (size_t)c);
#pragma unroll
            for (int e = 0; e < 8; e++) amax_pair(v, idx, elem(ch, e), 8 * c + e);
        }
        done = n_chunks * 8;
    }
    for (int i = done + t0; i < n; i += stride) amax_pair(v, idx, bf2f(x[i]), i);
    block_amax(v, idx, lv, li);
    if (threadIdx.x == 0) {
        pv[blockIdx.x] = v;
        pi[blockIdx.x] = idx;
    }
}

__global__ __launch_bounds__(256) void argmax_stage2_kernel(const float *pv, const int *pi,
                                                            int groups, int *out) {
    __shared__ float lv[4];
    __shared__ int li[4];
    float v = -__builtin_huge_valf();
    int idx = INT_MAX;
    for (int k = threadIdx.x; k < groups; k += blockDim.x) amax_pair(v, idx, pv[k], pi[k]);
    block_amax(v, idx, lv, li);
    if (threadIdx.x == 0) *out = idx;
}

int argmax_partial_count() { return AMAX_GROUPS; }

static int argmax_groups(int n) {
    const int g = (n + 256 * 8 - 1) / (256 * 8);
    return g < 1 ? 1 : (g > AMAX_GROUPS ? AMAX_GROUPS : g);
}

// Shared by argmax_forward (library buffer) and the step (its own buffer).
void argmax_launch(int *out, const bf16 *x, int n, float *pv, int *pi, hipStream_t stream) {
    if (n <= AMAX_ALONE) {
        argmax_alone_kernel<<<1, AMAX_ALONE_T, 0, stream>>>(x, n, aligned16(x) ? 1 : 0, out);
        LAUNCH_OK();
        return;
    }
    const int groups = argmax_groups(n);
    argmax_stage1_kernel<<<groups, 256, 0, stream>>>(x, n, aligned16(x) ? 1 : 0, pv, pi);
    if (!LAUNCH_OK()) return;
    argmax_stage2_kernel<<<1, 256, 0, stream>>>(pv, pi, groups, out);
    LAUNCH_OK();
}

extern "C" void argmax_forward(int *out, const bf16 *x, int n, hipStream_t stream) {
    if (n <= 0) {
        llm_fail("argmax: n %d must be positive", n);
        return;
    }
    // Each device holds its own copy of the partials; look their addresses up once per device.
    static std::mutex mu;
    static float *pv_dev[64];
    static int *pi_dev[64];
    int dev = 0;
    if (!HIP_OK(hipGetDevice(&dev))) return;
    if (dev < 0 || dev >= 64) {
        llm_fail("argmax: device %d out of range", dev);
        return;
    }
    float *pv;
    int *pi;
    {
        std::lock_guard<std::mutex> lock(mu);
        if (!pv_dev[dev]) {
            if (!HIP_OK(hipGetSymbolAddress((void **)&pv_dev[dev], HIP_SYMBOL(g_amax_val))) ||
                !HIP_OK(hipGetSymbolAddress((void **)&pi_dev[dev], HIP_SYMBOL(g_amax_idx)))) {
                pv_dev[dev] = nullptr;
                return;
            }
        }
        pv = pv_dev[dev];
        pi = pi_dev[dev];
    }
    argmax_launch(out, x, n, pv, pi, stream);
}
