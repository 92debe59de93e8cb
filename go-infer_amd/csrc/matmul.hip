// Weight matrix times a batch of activations on the matrix cores: the
// O-projection that follows attention (pkg/engine/forward.go:270 and 580,
// Weights.MatMul / MatMulBatch, pkg/engine/weights.go:237-350), for weights
// of GGML type F32, F16, Q8_0 or Q4_0.
//
//   y[b][r] = sum_c W[r][c] * x[b][c]      (pkg/math/gemv.go, metal.MatMulBatch,
//                                            pkg/metal/metal_darwin.go:849-880)
//
// Weights are converted once (gi_weights_upload) from their GGUF layout into
// operand order, and activations are split into it on every call, so that
// each 16-byte operand load of a wave reads one contiguous 1 KiB run (a
// row-major load would send every quarter-wave to 16 rows, and the L1 tag
// rate -- one line per lane -- bounds that form):
//   16-bit weight matrices (F16, the F32 halves): the 16 x 32 tile (rows
//   16t.., columns 32kk..) is 512 elements in lane order, lane
//   16 * ((c / 8) % 4) + r % 16 holding columns 8 ((c / 8) % 4) .. +7 of its
//   row (op_index);
//   activation halves: the same tiles, in lane order (matmul_reg) or
//   row-major (x_index; matmul_sk's direct loads permute them);
//   Q8_0  int8 codes in the same order (512 bytes per tile), and per tile the
//         fp16 block scales of its 16 rows (scale_index), so that a row tile's
//         scales are one run: row-fastest over the whole matrix, each tile's
//         32 bytes shared their lines with workgroups of other XCDs, whose
//         L2s then each fetched them (Q4_0, 8192 x 8192, batch 1: 19.1 -> 17.9
//         us);
//   Q4_0  per tile and block, the 16 nibble bytes of each of the 16 rows
//         (byte j holds elements j and j+16, quant.go:504), 256 bytes;
//         scales as Q8_0;
//   F32   two fp16 halves, hi and lo, of W * 2^e[r] (e[r] from the row's
//         largest |w|, so both halves stay normal), and 2^-e[r] per row.
// Rows of weights are padded with zeros to multiples of 128 and those of
// activations to multiples of 64, so the product loops need no bounds checks.
//
// Activations are split into fp16 hi + lo of x * 2^e, e per batch row and
// range of k-steps, so the products keep float32 accuracy.  The matrix cores
// then compute W * x^T on 16x16x32 f16 tiles: quantised codes are exact fp16
// values, and one 32-wide k-step is exactly one quantisation block, so each
// k-step's partial product is scaled by its block scale in float32
// (DotVecQ8_0 / DotVecQ4_0 sum a block, then multiply by d).  F32 weights take
// three products (hi*hi, hi*lo, lo*hi).
//
// Three forms of the product, each described at its kernel:
//   * matmul_vec (batches of up to 16): bound by the weights' bytes and by
//     latency; one launch that splits x itself;
//   * matmul_reg (larger batches): 16 .. 64 x 32 / 64 tiles, the k-steps
//     divided over the waves of a workgroup, operands straight into registers;
//     split_x runs first;
//   * matmul_sk (F16 and F32 weights, large products): 128 x 128 tiles over
//     slices of the k-steps through LDS, the slices' partial tiles added by
//     reduce_splits; split_rows runs first.
#include "../../include/goinfer_paged.h"
#include "gi_common.h"
#include "devbuf.h"
#include "mfma_ops.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <new>
#include <string>
#include <type_traits>
#include <utility>

namespace gi {
namespace {

typedef __attribute__((address_space(3))) void *lds_void;
using mfma_ops::f4;
using mfma_ops::h8;
using mfma_ops::i8x8_to_h8;
using mfma_ops::mfma16;
using mfma_ops::u2;
using mfma_ops::u4x8_to_h8;

enum : int { W_F32 = 0, W_F16 = 1, W_Q4_0 = 2, W_Q8_0 = 8 }; // GGML type ids


// Activation rows are padded to multiples of 64, the widest batch side of
// matmul_reg's tiles and half of matmul_sk's (whose waves past the padding
// idle); weight rows to multiples of 128, the row side of the split-K tile and
// a multiple of all others.
__host__ __device__ __forceinline__ int64_t round_pad(int64_t n) { return (n + 63) / 64 * 64; }
__host__ __device__ __forceinline__ int64_t weight_rows_pad(int64_t n) { return (n + 127) / 128 * 128; }

// Element (r, c) of a 16-bit matrix (or an int8 code matrix) with KS
// k-steps of 32 columns, in operand order.
__host__ __device__ __forceinline__ int64_t op_index(int64_t r, int c, int KS)
{
    return (((r >> 4) * KS + (c >> 5)) * 64 + 16 * ((c >> 3) & 3) + (r & 15)) * 8 + (c & 7);
}

// Element (b, c) of the split-K form's activation halves: each 16 x 32 tile row-major
// (16 rows of 64 bytes), so that one batch row's k-step is one 64-byte run
// when it is written.  The direct loads read a tile's 1 KiB whole and permute
// it into lane order (operand order) on the way into LDS.
__host__ __device__ __forceinline__ int64_t x_index(int64_t b, int c, int KS)
{
    return (((b >> 4) * KS + (c >> 5)) * 16 + (b & 15)) * 32 + (c & 31);
}

// The scale of row r's quantisation block kk.
__host__ __device__ __forceinline__ int64_t scale_index(int64_t r, int kk, int KS)
{
    return ((r >> 4) * KS + kk) * 16 + (r & 15);
}

// Byte i of row r's Q4_0 block kk.
__host__ __device__ __forceinline__ int64_t q4_index(int64_t r, int kk, int i, int KS)
{
    return (((r >> 4) * KS + kk) * 16 + (r & 15)) * 16 + i;
}

// ---- conversion of GGUF weights into the operand layout ------------------

// Q8_0 / Q4_0: one thread per (row, block) of the padded rows; raw blocks
// are byte-addressed.
__global__ __launch_bounds__(256) void convert_quant(const uint8_t *__restrict__ raw, int type, int rows,
                                                    int rows_pad, int cols, uint8_t *__restrict__ codes,
                                                    uint16_t *__restrict__ scales)
{
    const int nb = cols / 32;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)rows_pad * nb)
        return;
    const int r = (int)(i / nb), kb = (int)(i - (int64_t)r * nb);
    const bool live = r < rows;
    const int bb = type == W_Q8_0 ? 34 : 18;
    const uint8_t *blk = raw + (live ? i : 0) * bb;
    scales[scale_index(r, kb, nb)] = live ? (uint16_t)(blk[0] | (blk[1] << 8)) : 0;
    if (type == W_Q8_0) {
        for (int j = 0; j < 32; j++)
            codes[op_index(r, 32 * kb + j, nb)] = live ? blk[2 + j] : 0;
    } else {
        for (int j = 0; j < 16; j++)
            codes[q4_index(r, kb, j, nb)] = live ? blk[2 + j] : 0x88; // padded rows: codes 8 (zero)
    }
}

// F16: one thread per 8 consecutive elements of the padded rows.
__global__ __launch_bounds__(256) void convert_f16(const uint16_t *__restrict__ raw, int rows, int rows_pad, int cols,
                                                  uint16_t *__restrict__ dst)
{
    const int per = cols / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)rows_pad * per)
        return;
    const int r = (int)(i / per), c = 8 * (int)(i - (int64_t)r * per);
    uint4 v = {0u, 0u, 0u, 0u};
    if (r < rows)
        v = *reinterpret_cast<const uint4 *>(raw + (int64_t)r * cols + c);
    *reinterpret_cast<uint4 *>(dst + op_index(r, c, cols / 32)) = v;
}

// F32: one workgroup per padded row; W * 2^e split into hi + lo fp16.
__global__ __launch_bounds__(256) void convert_f32(const float *__restrict__ raw, int rows, int cols,
                                                  _Float16 *__restrict__ hi, _Float16 *__restrict__ lo,
                                                  float *__restrict__ row_scale)
{
    __shared__ float s_max[256];
    const int r = blockIdx.x, KS = cols / 32;
    if (r >= rows) {
        for (int c = threadIdx.x; c < cols; c += 256) {
            hi[op_index(r, c, KS)] = (_Float16)0.0f;
            lo[op_index(r, c, KS)] = (_Float16)0.0f;
        }
        if (threadIdx.x == 0)
            row_scale[r] = 0.0f;
        return;
    }
    const float *w = raw + (int64_t)r * cols;
    float m = 0.0f;
    for (int c = threadIdx.x; c < cols; c += 256)
        m = fmaxf(m, fabsf(w[c]));
    s_max[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            s_max[threadIdx.x] = fmaxf(s_max[threadIdx.x], s_max[threadIdx.x + s]);
        __syncthreads();
    }
    const int e = pow2_exponent_for(s_max[0]);
    const float up = ldexpf(1.0f, e);
    for (int c = threadIdx.x; c < cols; c += 256) {
        const float x = w[c] * up; // exact: a power of two
        const _Float16 h = (_Float16)x;
        hi[op_index(r, c, KS)] = h;
        lo[op_index(r, c, KS)] = (_Float16)(x - (float)h);
    }
    if (threadIdx.x == 0)
        row_scale[r] = ldexpf(1.0f, -e);
}

// ---- activations: x * 2^e split into hi + lo -----------------------------------

// For the split-K form: one power of two per batch row.
// One workgroup per padded batch row (rows past the batch are zeros); each
// thread takes runs of 8 columns, so the halves go out as 16-byte stores,
// four of them one 64-byte run of a tile (x_index).
__global__ __launch_bounds__(256) void split_rows(const float *__restrict__ x, int batch, int cols,
                                                 _Float16 *__restrict__ xh, _Float16 *__restrict__ xl,
                                                 float *__restrict__ xscale)
{
    __shared__ float s_max[4];
    const int b = blockIdx.x, KS = cols / 32, runs = cols / 8;
    if (b >= batch) {
        for (int q = threadIdx.x; q < runs; q += 256) {
            *reinterpret_cast<uint4 *>(xh + x_index(b, 8 * q, KS)) = uint4{0u, 0u, 0u, 0u};
            *reinterpret_cast<uint4 *>(xl + x_index(b, 8 * q, KS)) = uint4{0u, 0u, 0u, 0u};
        }
        return;
    }
    const float *xr = x + (int64_t)b * cols;
    // a thread's first KEEP runs stay in registers between the two passes
    // (all of them for rows up to 8192 columns)
    constexpr int KEEP = 4;
    f4 ku[KEEP], kv[KEEP];
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int q = threadIdx.x + 256 * k;
        ku[k] = kv[k] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (q < runs) {
            ku[k] = *reinterpret_cast<const f4 *>(xr + 8 * q);
            kv[k] = *reinterpret_cast<const f4 *>(xr + 8 * q + 4);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(m, fmaxf(fabsf(ku[k][i]), fabsf(kv[k][i])));
    }
    for (int q = threadIdx.x + 256 * KEEP; q < runs; q += 256) {
        const f4 u = *reinterpret_cast<const f4 *>(xr + 8 * q), v = *reinterpret_cast<const f4 *>(xr + 8 * q + 4);
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(m, fmaxf(fabsf(u[i]), fabsf(v[i])));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0)
        s_max[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    const int e = pow2_exponent_for(m);
    const float up = ldexpf(1.0f, e);
    auto emit = [&](int q, const f4 &u, const f4 &v) {
        h8 hi, lo;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float t = (k < 4 ? u[k] : v[k - 4]) * up; // exact: a power of two
            const _Float16 h = (_Float16)t;
            hi[k] = h;
            lo[k] = (_Float16)(t - (float)h);
        }
        *reinterpret_cast<h8 *>(xh + x_index(b, 8 * q, KS)) = hi;
        *reinterpret_cast<h8 *>(xl + x_index(b, 8 * q, KS)) = lo;
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int q = threadIdx.x + 256 * k;
        if (q < runs)
            emit(q, ku[k], kv[k]);
    }
    for (int q = threadIdx.x + 256 * KEEP; q < runs; q += 256)
        emit(q, *reinterpret_cast<const f4 *>(xr + 8 * q), *reinterpret_cast<const f4 *>(xr + 8 * q + 4));
    if (threadIdx.x == 0)
        xscale[b] = ldexpf(1.0f, -e);
}

// For matmul_reg: each wave of a workgroup takes one contiguous segment of the
// k-steps (seg_steps of them), and x is scaled per (batch row, segment), so
// that a wave's sums carry one power of two per column.
constexpr int kRegWaves = 8, kRegWorkgroups = 256;
__host__ __device__ __forceinline__ int seg_steps(int KS) { return (KS + kRegWaves - 1) / kRegWaves; }

// One workgroup per (16 batch rows, segment): the rows' largest magnitudes
// over the segment, then the halves in operand order (op_index), whole tiles
// at a time: lane r of 16 holds row r, so 16 lanes write one 256-byte run.
// xscale[segment][batch_pad] = 2^-e.  Rows past the batch are zeros.
__global__ __launch_bounds__(256) void split_x(const float *__restrict__ x, int batch, int batch_pad, int cols,
                                              _Float16 *__restrict__ xh, _Float16 *__restrict__ xl,
                                              float *__restrict__ xscale)
{
    __shared__ float s_max[4][16];
    const int KS = cols / 32, per = seg_steps(KS), seg = blockIdx.y;
    const int r = threadIdx.x & 15, q0 = threadIdx.x >> 4, b = blockIdx.x * 16 + r;
    const int first = 4 * per * seg, runs = max(0, min(4 * per, cols / 8 - first)); // runs of 8 columns
    const float *xr = x + (int64_t)min(b, batch - 1) * cols + 8 * (int64_t)first;
    // a thread's first KEEP runs stay in registers between the two passes
    // (all of them for rows up to 8192 columns)
    constexpr int KEEP = 8;
    f4 ku[KEEP], kv[KEEP];
    float m = 0.0f;
    auto top = [&](const f4 &u, const f4 &v) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(m, fmaxf(fabsf(u[i]), fabsf(v[i])));
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int q = q0 + 16 * k;
        ku[k] = kv[k] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (q < runs && b < batch) {
            ku[k] = *reinterpret_cast<const f4 *>(xr + 8 * q);
            kv[k] = *reinterpret_cast<const f4 *>(xr + 8 * q + 4);
        }
    }
#pragma unroll
    for (int k = 0; k < KEEP; k++)
        top(ku[k], kv[k]);
    if (b < batch)
        for (int q = q0 + 16 * KEEP; q < runs; q += 16)
            top(*reinterpret_cast<const f4 *>(xr + 8 * q), *reinterpret_cast<const f4 *>(xr + 8 * q + 4));
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    if ((threadIdx.x & 48) == 0)
        s_max[threadIdx.x >> 6][r] = m;
    __syncthreads();
    m = fmaxf(fmaxf(s_max[0][r], s_max[1][r]), fmaxf(s_max[2][r], s_max[3][r]));
    const int e = pow2_exponent_for(m);
    const float up = ldexpf(1.0f, e);
    auto emit = [&](int q, const f4 &u, const f4 &v) __attribute__((always_inline)) {
        h8 hi, lo;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float t = (k < 4 ? u[k] : v[k - 4]) * up; // exact: a power of two
            const _Float16 h = (_Float16)t;
            hi[k] = h;
            lo[k] = (_Float16)(t - (float)h);
        }
        const int64_t o = op_index(b, 8 * (first + q), KS);
        *reinterpret_cast<h8 *>(xh + o) = hi;
        *reinterpret_cast<h8 *>(xl + o) = lo;
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int q = q0 + 16 * k;
        if (q < runs)
            emit(q, ku[k], kv[k]);
    }
    for (int q = q0 + 16 * KEEP; q < runs; q += 16) {
        f4 u = f4{0.0f, 0.0f, 0.0f, 0.0f}, v = u;
        if (b < batch) {
            u = *reinterpret_cast<const f4 *>(xr + 8 * q);
            v = *reinterpret_cast<const f4 *>(xr + 8 * q + 4);
        }
        emit(q, u, v);
    }
    if (threadIdx.x < 16)
        xscale[(int64_t)seg * batch_pad + b] = ldexpf(1.0f, -e);
}

// ---- the product -----------------------------------------------------------

struct MatArgs {
    int type;
    int rows, cols, batch;
    int rows_pad;           // rows padded to a multiple of 128
    const uint8_t *a;      // F16 / F32-hi / Q8 codes / Q4 nibble bytes
    const uint8_t *a_lo;   // F32 lo
    const uint16_t *scales; // Q8 / Q4 block scales (scale_index)
    const float *row_scale; // F32
    const _Float16 *xh, *xl;
    const float *xscale;
    float *y;
};

// Lane I of this lane's row of 16.
template <int I>
__device__ __forceinline__ uint32_t row_lane(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + I, 0xF, 0xF, false); // row_newbcast
}

template <int N>
using ic = std::integral_constant<int, N>;

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(ic<I>{}), ...);
}
// f(ic<0>{}), ..., f(ic<N - 1>{}): an unrolled loop whose index is a
// constant expression
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// ---- batches over 16 ---------------------------------------------------------------
//
// A workgroup of 8 waves owns 16 RT rows x 16 CT batch columns; wave w takes
// the w-th segment of the k-steps for the whole tile, its operands straight
// from memory into registers in lane order, one k-step ahead.  No two waves
// share an operand, so nothing goes through LDS and nothing synchronises
// until the eight waves' sums meet at the end; a weight fragment feeds 2 CT
// products (hi and lo), an activation pair RT.  Tiles are sized so that one
// round of workgroups covers the CUs: each re-reads its operands from the L2
// (30 TB/s measured for L2-resident runs of 1 KiB), and consecutive workgroups
// of an XCD (blockIdx mod 8) take consecutive tiles of one eighth of the rows,
// so an XCD reads an eighth of the weights.  What bounds it: 10 to 12 KiB of
// operands per 32 products against a CU's 56 bytes per cycle from the L2, and
// for quantised weights the scale multiply-adds beside the products.
//
// Per call with split_x, 4096 x 4096: batch 32 Q8_0 34.9 -> 15.4 us, F16 34.5
// -> 17.1; batch 256 Q8_0 39.0 -> 30.9, F16 33.6 -> 31.5; 8192 x 8192, batch
// 64, Q8_0: 62.8 -> 42.7.  (Before: 64 x 64 tiles staged through LDS by four
// waves, one per SIMD, on rows / 64 workgroups; F16 at batch 256 matmul_sk.)
// Weights four k-steps ahead instead of one (tiles of up to 32 rows): Q8_0,
// batch 32: 17.0 -> 15.4.
template <int WT, int RT, int CT>
__global__ __launch_bounds__(64 * kRegWaves) void matmul_reg(MatArgs a, int batch_pad)
{
#if __HIP_DEVICE_COMPILE__ // (target builtins inside generic lambdas: not for the host pass)
    constexpr bool QUANT = WT == W_Q8_0 || WT == W_Q4_0;
    constexpr int COLS = 16 * CT;
    __shared__ float red[kRegWaves][16 * RT][COLS + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = lane & 15, g = lane >> 4;
    // tile index: row tiles major, batch tiles minor; XCD x takes the x-th
    // eighth of them
    const int bts = (a.batch + COLS - 1) / COLS, tiles = (a.rows + 16 * RT - 1) / (16 * RT) * bts;
    const int per_xcd = gridDim.x / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= tiles)
        return;
    const int r0 = tile / bts * 16 * RT, b0 = tile % bts * COLS;
    const int KS = a.cols / 32, per = seg_steps(KS);
    const int k0 = w * per, k1 = min(KS, k0 + per);
    const int64_t rt0 = r0 / 16, bt0 = b0 / 16;
    f4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int c = 0; c < CT; c++)
            acc[r][c] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    // the operands of one k-step; the weights of tiles of up to 32 rows are
    // instead loaded four k-steps at a time (they come from memory, where one
    // k-step's products do not cover the latency; a larger tile has no
    // registers for it)
    constexpr bool GROUP = RT <= 2;
    struct Weights {
        h8 wh[QUANT ? 1 : RT], wl[WT == W_F32 ? RT : 1];
        u2 wq[QUANT ? RT : 1];
    };
    struct Step {
        h8 xh[CT], xl[CT];
        Weights W;
    };
    auto load_w = [&](int k, Weights &W) __attribute__((always_inline)) {
        const int kk = min(k, k1 - 1);
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const int64_t t = (rt0 + r) * KS + kk;
            if constexpr (QUANT) {
                W.wq[r] = *reinterpret_cast<const u2 *>(WT == W_Q8_0 ? a.a + t * 512 + 8 * lane
                                                                     : a.a + t * 256 + 16 * j + 8 * (g & 1));
            } else {
                W.wh[r] = *reinterpret_cast<const h8 *>(a.a + t * 1024 + 16 * lane);
                if constexpr (WT == W_F32)
                    W.wl[r] = *reinterpret_cast<const h8 *>(a.a_lo + t * 1024 + 16 * lane);
            }
        }
    };
    auto load = [&](int k, Step &S) __attribute__((always_inline)) {
        const int kk = min(k, k1 - 1);
#pragma unroll
        for (int c = 0; c < CT; c++) {
            const int64_t o = ((bt0 + c) * KS + kk) * 512 + 8 * lane;
            S.xh[c] = *reinterpret_cast<const h8 *>(a.xh + o);
            S.xl[c] = *reinterpret_cast<const h8 *>(a.xl + o);
        }
        if constexpr (!GROUP)
            load_w(k, S.W);
    };
    // scales of four k-steps from k: lane (j, g) holds rows 4g .. 4g + 3 of
    // k-step k + (j & 3)
    auto load_scales = [&](int k, u2 (&sw)[RT]) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RT; r++)
            sw[r] = *reinterpret_cast<const u2 *>(a.scales + ((rt0 + r) * KS + min(k + (j & 3), k1 - 1)) * 16 + 4 * g);
    };
    auto products = [&](auto ic_i, const Step &S, const Weights &W, const u2 (&sw)[RT]) __attribute__((always_inline)) {
        constexpr int i = decltype(ic_i)::value;
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if constexpr (QUANT) {
                const h8 aq = WT == W_Q8_0 ? i8x8_to_h8(W.wq[r]) : u4x8_to_h8(W.wq[r], (g & 2) ? 4 : 0);
                const uint32_t s01 = row_lane<i>(sw[r].x), s23 = row_lane<i>(sw[r].y);
                const _Float16 d[4] = {__builtin_bit_cast(_Float16, (uint16_t)(s01 & 0xFFFFu)),
                                       __builtin_bit_cast(_Float16, (uint16_t)(s01 >> 16)),
                                       __builtin_bit_cast(_Float16, (uint16_t)(s23 & 0xFFFFu)),
                                       __builtin_bit_cast(_Float16, (uint16_t)(s23 >> 16))};
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    f4 z = mfma16(aq, S.xh[c], f4{0.0f, 0.0f, 0.0f, 0.0f});
                    z = mfma16(aq, S.xl[c], z);
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        acc[r][c][q] = fmaf(z[q], (float)d[q], acc[r][c][q]);
                }
            } else {
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    acc[r][c] = mfma16(W.wh[r], S.xh[c], acc[r][c]);
                    acc[r][c] = mfma16(W.wh[r], S.xl[c], acc[r][c]);
                    if constexpr (WT == W_F32)
                        acc[r][c] = mfma16(W.wl[r], S.xh[c], acc[r][c]);
                }
            }
        }
    };
    if (k0 < k1) {
        Step A, B;
        Weights wc[GROUP ? 4 : 1], wn[GROUP ? 4 : 1]; // this group's and the next's
        u2 sw[RT], sn[RT];
        auto load_group = [&](int k) __attribute__((always_inline)) {
            if constexpr (GROUP) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    load_w(k + i, wn[i]);
            }
            if constexpr (QUANT)
                load_scales(k, sn);
        };
        load_group(k0);
        load(k0, A);
        for (int k = k0; k < k1; k += 4) {
            if constexpr (GROUP) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    wc[i] = wn[i];
            }
            if constexpr (QUANT) {
#pragma unroll
                for (int r = 0; r < RT; r++)
                    sw[r] = sn[r];
            }
            load_group(k + 4);
            load(k + 1, B);
            products(ic<0>{}, A, GROUP ? wc[0] : A.W, sw);
            load(k + 2, A);
            if (k + 1 < k1)
                products(ic<1>{}, B, GROUP ? wc[GROUP ? 1 : 0] : B.W, sw);
            load(k + 3, B);
            if (k + 2 < k1)
                products(ic<2>{}, A, GROUP ? wc[GROUP ? 2 : 0] : A.W, sw);
            load(k + 4, A);
            if (k + 3 < k1)
                products(ic<3>{}, B, GROUP ? wc[GROUP ? 3 : 0] : B.W, sw);
        }
    }
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const float down = a.xscale[(int64_t)w * batch_pad + b0 + 16 * c + j];
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                red[w][16 * r + 4 * g + q][16 * c + j] = acc[r][c][q] * down;
    }
    __syncthreads();
    // rows fastest: coalesced stores
    for (int e = threadIdx.x; e < 16 * RT * COLS; e += 64 * kRegWaves) {
        const int rl = e % (16 * RT), cl = e / (16 * RT), r = r0 + rl, b = b0 + cl;
        if (b >= a.batch || r >= a.rows)
            continue;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < kRegWaves; q++)
            v += red[q][rl][cl];
        a.y[(int64_t)b * a.rows + r] = WT == W_F32 ? v * a.row_scale[r] : v;
    }
#endif
}

// Tile shapes: 32 columns to batch 32, else 64, and the rows (16, 32 or 64)
// whose rounds of one workgroup per CU cost least: a tile of 64 rows takes 1.6
// and one of 32 rows 1.2 times as long as one of 16 (4096 x 4096 Q8_0 batch 256
// 28 us in 256 tiles of 64, batch 128 20 in 256 of 32; 2048 x 2048 17.7, 13.8
// and 11.9).  By the most rows that still gave each CU a workgroup, 1.5 rounds
// were common: 2048 x 2048, batch 192, F32 20.5 -> 15.5, Q8_0 18.2 -> 13.5; 4096 x
// 4096, batch 160, Q8_0 34.1 -> 27.7.
struct RegTiles {
    int ct, rt, tiles;
    RegTiles(int rows, int batch) : ct(batch <= 32 ? 2 : 4)
    {
        const int bts = (batch + 16 * ct - 1) / (16 * ct);
        int64_t best = INT64_MAX;
        for (const int r : {4, 2, 1}) {
            const int n = (rows + 16 * r - 1) / (16 * r) * bts;
            const int64_t cost = (int64_t)rounds(n) * (r == 4 ? 8 : r == 2 ? 6 : 5);
            if (cost < best) {
                best = cost;
                rt = r;
                tiles = n;
            }
        }
    }
    static int rounds(int n) { return (n + kRegWorkgroups - 1) / kRegWorkgroups; }
    // a quarter or more of the last rounds' workgroups missing
    bool uneven() const { return 4 * (int64_t)tiles <= 3 * (int64_t)rounds(tiles) * kRegWorkgroups; }
};

template <int WT>
void launch_reg(const MatArgs &a, int batch_pad, hipStream_t st)
{
    const RegTiles t(a.rows, a.batch);
    const int ct = t.ct, rt = t.rt;
    const dim3 grid((unsigned)((t.tiles + 7) / 8 * 8)), block(64 * kRegWaves);
#define GI_REG(RT, CT) hipLaunchKernelGGL((matmul_reg<WT, RT, CT>), grid, block, 0, st, a, batch_pad)
    if (ct == 2) {
        if (rt == 4)
            GI_REG(4, 2);
        else if (rt == 2)
            GI_REG(2, 2);
        else
            GI_REG(1, 2);
    } else {
        if (rt == 4)
            GI_REG(4, 4);
        else if (rt == 2)
            GI_REG(2, 4);
        else
            GI_REG(1, 4);
    }
#undef GI_REG
}

// ---- 16-bit weights, large products: split-K ---------------------------------
//
// A workgroup of four waves owns a 128 x 128 (rows x batch) output tile over
// one of S slices of the k-steps, and two workgroups share a CU.  Wave w
// takes batch rows 32w .. 32w + 31 of the tile and all 128 rows, so each
// weight fragment read from LDS feeds four products (two batch tiles, hi and
// lo) and each activation fragment eight (the row tiles).  Per k-step the
// eight weight tiles (shared by the waves, each loading two) and every wave's
// activation halves arrive by direct global->LDS loads two k-steps ahead,
// through three stages; one barrier per k-step hands a stage from the loads
// to the products.  The per-CU load volume is 24 KiB per 128 products against
// matmul_reg's 10 to 12 KiB per 32.  With S > 1 the partial tiles go to a
// workspace and reduce_splits adds them.  Quantised weights do not take it:
// their per-block scale multiply-adds need 272 registers here (one wave per
// SIMD).

struct SKArgs {
    MatArgs m;
    int splits;   // S: slices of the k-steps
    int ks_per;   // k-steps per slice (the last may have fewer)
    float *part;  // S > 1: partial tiles [S][batch_pad][rows_pad]
    int batch_pad;
};

// The k-step slices give about kSplitKWorkgroups workgroups, none shorter than
// kMinSliceSteps k-steps.  The form is taken from kSplitKMinSteps (64 x 64
// pieces of the output times k-steps) up, where matmul_reg's operand volume per
// product costs more than the reduction launch here (per call, this /
// matmul_reg):
// 8192 x 8192, batch 256: F16 93 / 101 us, F32 123 / 142; batch 127: 57 / 58,
// 81 / 88; 4096 x 4096, batch 512: 54 / 56, 69 / 72; batch 256 (below the
// line): 33.6 / 31.5, 41.8 / 41.2.
// From a quarter of that up it is taken at batches over 64 where matmul_reg's
// tiles leave a quarter of the CUs idle (4096 x 4096, batch 160: F16 28.4 / 39,
// F32 34.4 / 51; batch 320: 40.8 / 52, 60.9 / 70.4; F32 384 73 / 70), and for F32
// rows of 4096 columns and more, which matmul_reg reads in two planes (batch 65
// 28.9 / 30.7, 200 40.0 / 40.6; 2048 columns, batch 512: 28.3 / 22.3).
constexpr int kSplitKWorkgroups = 256, kMinSliceSteps = 4, kSplitKMinSteps = 65536;
constexpr int kSplitKF32Steps = 128; // 4096 columns

template <int WT>
__global__ __launch_bounds__(256) void matmul_sk(SKArgs s)
{
    static_assert(WT == W_F16 || WT == W_F32, "16-bit weight tiles (F32 as hi + lo)");
    // (device pass only: the host pass, which emits the launch stub, cannot
    // instantiate the target builtins inside the generic lambdas below)
#if __HIP_DEVICE_COMPILE__
    constexpr int NST = 3;                 // stages (k-steps in flight); the loop is unrolled by NST
    constexpr int NWV = 4;                 // waves
    constexpr int BS = 2;                  // batch tiles of 16 per wave
    constexpr int BT = 16 * BS * NWV;      // batch rows per workgroup
    constexpr int XB = 1024 * 2 * BS;      // a wave's activation halves of one k-step
    constexpr int WB = (WT == W_F32 ? 16 : 8) * 1024; // the 128 rows' weight tiles of one k-step
    // weight tiles per wave, and its direct loads of them per k-step
    constexpr int TPW = 8 / NWV, DW = (WT == W_F32 ? 2 : 1) * TPW;
    const MatArgs &a = s.m;
    // Every load in flight is a direct global->LDS load: with register loads
    // in flight beside them the compiler assumes the two kinds complete out
    // of order and waits for all of them.  Each stage is an array of its own,
    // named at compile time where it is used, so that before an LDS read the
    // compiler waits only for the loads into that array (it does not tell
    // apart offsets into one array).
    __shared__ __attribute__((aligned(16))) uint8_t w0[WB], w1[WB], w2[WB];
    __shared__ __attribute__((aligned(16))) uint8_t x0[NWV * XB], x1[NWV * XB], x2[NWV * XB];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = lane & 15, g = lane >> 4;
    const int sl = blockIdx.x, r0 = blockIdx.y * 128;
    const int bw0 = blockIdx.z * BT + 16 * BS * w; // this wave's first batch row
    const bool active = bw0 < s.batch_pad;          // uniform: the activations are padded to 64
    const int KS = a.cols / 32;
    const int k0 = sl * s.ks_per, nk = min(s.ks_per, KS - k0);
    const int64_t rt0 = r0 / 16, bt0 = bw0 / 16;
    f4 acc[8][BS];
#pragma unroll
    for (int rs = 0; rs < 8; rs++)
#pragma unroll
        for (int bs = 0; bs < BS; bs++)
            acc[rs][bs] = f4{0.0f, 0.0f, 0.0f, 0.0f};

    auto wstage = [&](auto u) __attribute__((always_inline)) -> uint8_t * {
        constexpr int U = decltype(u)::value % NST;
        return U == 0 ? w0 : U == 1 ? w1 : w2;
    };
    auto xstage = [&](auto u) __attribute__((always_inline)) -> uint8_t * {
        constexpr int U = decltype(u)::value % NST;
        return (U == 0 ? x0 : U == 1 ? x1 : x2) + XB * w;
    };
    // This wave's direct loads of k-step i of the slice (clamped to the last,
    // so every call issues the same number) into stage u: its share of the
    // weight tiles, then (ACT) its activation halves, each permuted into
    // lane order on the way (lane (j, g) fetches row j's k-elements
    // 8g .. 8g + 7, x_index).
    auto issue = [&](int i, auto u, auto act) __attribute__((always_inline)) {
        const int kk = k0 + min(i, nk - 1);
        uint8_t *d = wstage(u);
        // 1 KiB tiles TPW w .. TPW w + TPW - 1 (F32: their lo tiles too, 8 KiB
        // later)
#pragma unroll
        for (int q = 0; q < DW; q++) {
            const uint8_t *src = q >= TPW ? a.a_lo : a.a;
            const int tile = TPW * w + q % TPW;
            const int64_t t = (rt0 + tile) * KS + kk;
            __builtin_amdgcn_global_load_lds(src + t * 1024 + 16 * lane, (lds_void)(d + 1024 * (8 * (q / TPW) + tile)),
                                             16, 0, 0);
        }
        if (decltype(act)::value) {
            uint8_t *xd = xstage(u);
#pragma unroll
            for (int bs = 0; bs < BS; bs++) {
                const int64_t o = ((bt0 + bs) * KS + kk) * 512 + 32 * j + 8 * g;
                __builtin_amdgcn_global_load_lds(a.xh + o, (lds_void)(xd + 2048 * bs), 16, 0, 0);
                __builtin_amdgcn_global_load_lds(a.xl + o, (lds_void)(xd + 2048 * bs + 1024), 16, 0, 0);
            }
        }
    };
    // Loads per k-step and wave; before the barrier of k-step i a wave waits
    // until only the next stage's are in flight (its own of stage i have
    // landed).
    constexpr int VMA = (NST - 2) * (DW + 2 * BS), VMI = (NST - 2) * DW;
    // One k-step: ACT, a wave inside the batch (loads and products), else one
    // that only loads its share of the weights.
    auto body = [&](int i, auto u, auto act) __attribute__((always_inline)) {
        constexpr bool ACT = decltype(act)::value;
        if (ACT)
            __builtin_amdgcn_s_waitcnt((VMA & 15) | ((VMA >> 4) << 14) | 0x0F70);
        else
            __builtin_amdgcn_s_waitcnt((VMI & 15) | ((VMI >> 4) << 14) | 0x0F70);
        // every wave's loads of stage i have landed, and every wave is done
        // with stage i - 1, which the loads below refill.  A bare barrier:
        // __syncthreads' release fence would wait for every load in flight.
        asm volatile("s_barrier" ::: "memory");
        issue(i + NST - 1, ic<decltype(u)::value + NST - 1>{}, act);
        if (!ACT)
            return;
        const uint8_t *sp = wstage(u);
        const uint8_t *xp = xstage(u);
        h8 xh[BS], xl[BS];
#pragma unroll
        for (int bs = 0; bs < BS; bs++) {
            xh[bs] = *reinterpret_cast<const h8 *>(xp + 2048 * bs + 16 * lane);
            xl[bs] = *reinterpret_cast<const h8 *>(xp + 2048 * bs + 1024 + 16 * lane);
        }
#pragma unroll
        for (int rs = 0; rs < 8; rs++) {
            const h8 ah = *reinterpret_cast<const h8 *>(sp + 1024 * rs + 16 * lane);
            h8 al = {};
            if (WT == W_F32)
                al = *reinterpret_cast<const h8 *>(sp + 8192 + 1024 * rs + 16 * lane);
#pragma unroll
            for (int bs = 0; bs < BS; bs++) {
                acc[rs][bs] = mfma16(ah, xh[bs], acc[rs][bs]);
                acc[rs][bs] = mfma16(ah, xl[bs], acc[rs][bs]);
                if (WT == W_F32)
                    acc[rs][bs] = mfma16(al, xh[bs], acc[rs][bs]);
            }
        }
    };
    // whole rounds of NST k-steps, then the remainder
    auto run = [&](auto act) __attribute__((always_inline)) {
        static_for<NST - 1>([&](auto u) __attribute__((always_inline)) { issue(decltype(u)::value, u, act); });
        const int nfull = nk / NST * NST;
        for (int i = 0; i < nfull; i += NST)
            static_for<NST>([&](auto u) __attribute__((always_inline)) { body(i + decltype(u)::value, u, act); });
        static_for<NST - 1>([&](auto u) __attribute__((always_inline)) {
            if (nfull + decltype(u)::value < nk)
                body(nfull + decltype(u)::value, u, act);
        });
    };
    if (nk > 0) {
        if (active)
            run(std::true_type{});
        else
            run(std::false_type{});
    }
    // the trailing (unused) loads land before the workgroup ends
    __builtin_amdgcn_s_waitcnt(0x0F70);
    if (!active)
        return;
    // lane (j, g) holds rows 16 rs + 4g + i of batch row 16 bs + j
#pragma unroll
    for (int bs = 0; bs < BS; bs++) {
        const int b = bw0 + 16 * bs + j;
        if (s.splits > 1) {
            float *pp = s.part + ((int64_t)sl * s.batch_pad + b) * a.rows_pad + r0 + 4 * g;
#pragma unroll
            for (int rs = 0; rs < 8; rs++)
                *reinterpret_cast<f4 *>(pp + 16 * rs) = acc[rs][bs];
        } else if (b < a.batch) {
            const float xs = a.xscale[b];
#pragma unroll
            for (int rs = 0; rs < 8; rs++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = r0 + 16 * rs + 4 * g + i;
                    if (r < a.rows)
                        a.y[(int64_t)b * a.rows + r] =
                            acc[rs][bs][i] * xs * (WT == W_F32 ? a.row_scale[r] : 1.0f);
                }
        }
    }
#endif
}

// y[b][r] = (sum over the S slices of the partial tiles) * xscale[b]
// (* row_scale[r] for F32 weights): four consecutive rows per thread.
__global__ __launch_bounds__(256) void reduce_splits(const float *__restrict__ part, int splits, int batch,
                                                    int batch_pad, int rows, int rows_pad,
                                                    const float *__restrict__ xscale,
                                                    const float *__restrict__ row_scale, float *__restrict__ y)
{
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; // index of 4 rows
    const int per = rows_pad / 4;
    const int b = (int)(q / per), r = 4 * (int)(q - (int64_t)b * per);
    if (b >= batch)
        return;
    f4 v = *reinterpret_cast<const f4 *>(part + (int64_t)b * rows_pad + r);
#pragma unroll 4
    for (int sl = 1; sl < splits; sl++)
        v += *reinterpret_cast<const f4 *>(part + ((int64_t)sl * batch_pad + b) * rows_pad + r);
    const float xs = xscale[b];
    f4 o;
#pragma unroll
    for (int i = 0; i < 4; i++)
        o[i] = v[i] * xs * (row_scale ? row_scale[min(r + i, rows - 1)] : 1.0f);
    float *yp = y + (int64_t)b * rows + r;
    if ((rows & 3) == 0 && r + 4 <= rows) {
        *reinterpret_cast<f4 *>(yp) = o; // 16-byte aligned: rows and r are multiples of 4
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (r + i < rows)
                yp[i] = o[i];
    }
}

// ---- batches of up to 16: one launch, no workspace ---------------------------
//
// A workgroup of 16 waves owns 16 rows; wave w takes the w-th sixteenth of the
// k-steps, CH at a time, for all BP (batch padded to a power of two) rows of
// x.  Such a product is bound by reading the weights once, and its time by
// latency: 256 workgroups at 4096 rows put every weight byte in flight in the
// first instructions, before anything is waited for.  The x chunk (BP x 32 CH
// columns) is loaded once per wave (64 / BP lanes share a row), scaled by the
// chunk's own power of two per row, split into hi + lo halves and handed to
// the operand lanes through the wave's own LDS, so nothing synchronises until
// the sixteen waves' sums meet at the end.  Each x row's 64-byte k-steps are
// XOR-swizzled by row, so that the operand reads of four rows fall on all 64
// banks.
//
// Up to 8 batch rows share one 16-column operand: column b holds row b's hi
// half, column 8 + b its lo half, and the two sums are added at the end.
//
// Batch 1, per call: 4096 x 4096 Q4_0 35.1 -> 5.2 us over one matrix again and
// again and 5.7 in a run of 32 matrices, F16 32.6 -> 7.6 (4.4 TB/s of weights;
// an empty kernel called the same way takes 4.2); 8192 x 8192
// Q4_0 63 -> 13.8, F16 59 -> 22.8 (5.9 TB/s).  Batch 16, 4096 x 4096: Q4_0
// 35.4 -> 9.7, F32 41.8 -> 15.6.  (Before: x padded to 64 rows and split in a
// launch of its own, then 64 x 64 tiles on 64 workgroups.)  Above 16 rows the
// x each workgroup converts outweighs its weights.  Batch 1 over quantised
// weights fits two workgroups on a CU (64 VGPRs), so that one's loads run
// under the other's products where there are more than 256: 8192 x 8192 Q8_0
// 17.4 -> 14.5 us.
constexpr int kVecWaves = 16, kVecMaxBatch = 16;

// Bytes of LDS per wave: hi and lo planes of BP rows of CH k-steps.
template <int BP, int CH>
constexpr int kVecStage = 2 * BP * CH * 64;

template <int WT, int BP, int CH>
__global__ __launch_bounds__(64 * kVecWaves, (WT == W_Q8_0 || WT == W_Q4_0) && BP == 1 ? 8 : 1) void matmul_vec(MatArgs a, const float *__restrict__ x)
{
    static_assert(BP >= 1 && BP <= 16 && (BP & (BP - 1)) == 0, "batch rows padded to a power of two");
    static_assert(CH >= 4 && CH <= 16, "a lane of a 16-lane row per k-step's scales");
#if __HIP_DEVICE_COMPILE__ // (target builtins inside generic lambdas, as in matmul_sk)
    constexpr bool PACK = BP <= 8; // hi and lo columns in one operand
    constexpr int LPR = 64 / BP;   // lanes per x row
    constexpr int XI = CH * 32 / (4 * LPR) > 0 ? CH * 32 / (4 * LPR) : 1; // 16-byte loads per lane
    constexpr int ROW = CH * 64;   // bytes of one row of a plane
    constexpr int RED = kVecWaves * 16 * 17 * 4;
    constexpr int STG = kVecWaves * kVecStage<BP, CH>;
    __shared__ __attribute__((aligned(16))) uint8_t smem[STG > RED ? STG : RED];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = lane & 15, g = lane >> 4;
    const int r0 = blockIdx.x * 16, b0 = blockIdx.y * BP;
    const int C = a.cols, KS = C / 32;
    const int per = (KS + kVecWaves - 1) / kVecWaves;
    const int k0 = w * per, k1 = min(KS, k0 + per);
    uint8_t *mine = smem + w * kVecStage<BP, CH>;
    // this lane's x row and first column within a chunk
    const int xb = lane / LPR, xs = 4 * (lane % LPR);
    const float *xr = x + (int64_t)min(b0 + xb, a.batch - 1) * C;
    // the plane rows this lane's operand columns read
    const int ob = PACK ? (j & 7) & (BP - 1) : j;
    const uint8_t *op = mine + ob * ROW + 16 * g + (PACK && j >= 8 ? BP * ROW : 0);
    const int64_t t0 = (int64_t)blockIdx.x * KS;

    f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int kc = k0; kc < k1; kc += CH) {
        const int nk = min(CH, k1 - kc);
        // the chunk's weights (k-steps past the range repeat its last) ...
        h8 wh[CH], wl[WT == W_F32 ? CH : 1];
        u2 wq[CH], sw; // sw: lane (j, g) holds rows 4g .. 4g + 3's scales of k-step j
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const int kk = min(kc + i, k1 - 1);
            const int64_t t = t0 + kk;
            if (WT == W_F16 || WT == W_F32) {
                wh[i] = *reinterpret_cast<const h8 *>(a.a + t * 1024 + 16 * lane);
                if (WT == W_F32)
                    wl[i] = *reinterpret_cast<const h8 *>(a.a_lo + t * 1024 + 16 * lane);
            } else {
                wq[i] = *reinterpret_cast<const u2 *>(WT == W_Q8_0 ? a.a + t * 512 + 8 * lane
                                                                   : a.a + t * 256 + 16 * j + 8 * (g & 1));
            }
        }
        if (WT == W_Q8_0 || WT == W_Q4_0)
            sw = *reinterpret_cast<const u2 *>(a.scales + (t0 + min(kc + (j & (CH - 1)), k1 - 1)) * 16 + 4 * g);
        // ... and its x, the row's largest magnitude in the chunk, and the halves
        f4 xv[XI];
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int c = xs + 4 * LPR * i;
            xv[i] = f4{0.0f, 0.0f, 0.0f, 0.0f};
            if (c < 32 * nk)
                xv[i] = *reinterpret_cast<const f4 *>(xr + 32 * kc + c);
#pragma unroll
            for (int q = 0; q < 4; q++)
                m = fmaxf(m, fabsf(xv[i][q]));
        }
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1)
            m = fmaxf(m, __shfl_xor(m, o));
        const int e = pow2_exponent_for(m);
        const float up = ldexpf(1.0f, e);
        // the operand reads of the last chunk are done (they fed its products)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int c = xs + 4 * LPR * i;
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            h4 hi, lo;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float t = xv[i][q] * up; // exact: a power of two
                const _Float16 h = (_Float16)t;
                hi[q] = h;
                lo[q] = (_Float16)(t - (float)h);
            }
            uint8_t *d = mine + xb * ROW + 64 * ((c >> 5) ^ (xb & (CH - 1) & 3)) + 2 * (c & 31);
            if (c < 32 * CH) {
                *reinterpret_cast<h4 *>(d) = hi;
                *reinterpret_cast<h4 *>(d + BP * ROW) = lo;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // 2^-e of the row of this lane's operand column
        const float down = __shfl(ldexpf(1.0f, -e), ob * LPR);
        f4 z = f4{0.0f, 0.0f, 0.0f, 0.0f}; // the chunk's sums, in units of 2^-e
        static_for<CH>([&](auto ic_i) __attribute__((always_inline)) {
            constexpr int i = decltype(ic_i)::value;
            if (i >= nk)
                return;
            const uint8_t *xp = op + 64 * (i ^ (ob & (CH - 1) & 3));
            const h8 xh = *reinterpret_cast<const h8 *>(xp);
            h8 xl = {};
            if (!PACK)
                xl = *reinterpret_cast<const h8 *>(xp + BP * ROW);
            if (WT == W_F16 || WT == W_F32) {
                z = mfma16(wh[i], xh, z);
                if (!PACK)
                    z = mfma16(wh[i], xl, z);
                if (WT == W_F32)
                    z = mfma16(wl[i], xh, z);
            } else {
                const h8 aq = WT == W_Q8_0 ? i8x8_to_h8(wq[i]) : u4x8_to_h8(wq[i], (g & 2) ? 4 : 0);
                f4 p = mfma16(aq, xh, f4{0.0f, 0.0f, 0.0f, 0.0f});
                if (!PACK)
                    p = mfma16(aq, xl, p);
                // k-step i's scales, from lane i of each row of 16 lanes
                const uint32_t s01 = row_lane<i>(sw.x), s23 = row_lane<i>(sw.y);
                z[0] = fmaf(p[0], (float)__builtin_bit_cast(_Float16, (uint16_t)(s01 & 0xFFFFu)), z[0]);
                z[1] = fmaf(p[1], (float)__builtin_bit_cast(_Float16, (uint16_t)(s01 >> 16)), z[1]);
                z[2] = fmaf(p[2], (float)__builtin_bit_cast(_Float16, (uint16_t)(s23 & 0xFFFFu)), z[2]);
                z[3] = fmaf(p[3], (float)__builtin_bit_cast(_Float16, (uint16_t)(s23 >> 16)), z[3]);
            }
        });
#pragma unroll
        for (int i = 0; i < 4; i++)
            acc[i] = fmaf(z[i], down, acc[i]);
    }
    // the sixteen waves' sums: [wave][column][row]
    __syncthreads();
    float(*red)[16][17] = reinterpret_cast<float(*)[16][17]>(smem);
#pragma unroll
    for (int i = 0; i < 4; i++)
        red[w][j][4 * g + i] = acc[i];
    __syncthreads();
    // lanes 16 q + r of wave b: row r of batch row b, waves 4 q .. 4 q + 3
    if (w < BP && b0 + w < a.batch) {
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < kVecWaves / 4; q++) {
            v += red[4 * g + q][w][j];
            if (PACK)
                v += red[4 * g + q][8 + w][j];
        }
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        const int r = r0 + j;
        if (g == 0 && r < a.rows)
            a.y[(int64_t)(b0 + w) * a.rows + r] = WT == W_F32 ? v * a.row_scale[r] : v;
    }
#endif
}

// Launches matmul_vec for a.batch <= kVecMaxBatch.
template <int WT>
void launch_vec(const MatArgs &a, const float *x, hipStream_t st)
{
    const dim3 grid((unsigned)((a.rows + 15) / 16)), block(64 * kVecWaves);
    if (a.batch <= 1)
        hipLaunchKernelGGL((matmul_vec<WT, 1, 8>), grid, block, 0, st, a, x);
    else if (a.batch <= 2)
        hipLaunchKernelGGL((matmul_vec<WT, 2, 8>), grid, block, 0, st, a, x);
    else if (a.batch <= 4)
        hipLaunchKernelGGL((matmul_vec<WT, 4, 8>), grid, block, 0, st, a, x);
    else if (a.batch <= 8)
        hipLaunchKernelGGL((matmul_vec<WT, 8, WT == W_F32 ? 4 : 8>), grid, block, 0, st, a, x);
    else
        hipLaunchKernelGGL((matmul_vec<WT, 16, 4>), grid, block, 0, st, a, x);
}

int hip_fail(hipError_t e, const char *what)
{
    return set_error(GI_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

} // namespace
} // namespace gi

struct gi_weights {
    gi_paged *h = nullptr; // stream and allocation of the products
    int device = 0;        // frees need only this, so destroy does not use h
    int type = 0, rows = 0, cols = 0;
    uint8_t *a = nullptr, *a_lo = nullptr;
    uint16_t *scales = nullptr;
    float *row_scale = nullptr;
    // activation split (hi, lo halves, row scales), grown on demand
    gi::DevBuffer xsplit;
};

extern "C" {

int gi_weights_upload(gi_paged *h, int ggml_type, int rows, int cols, const void *raw, gi_weights **out)
{
    using namespace gi;
    if (!out)
        return set_error(GI_ERR_BAD_ARG, "gi_weights_upload: out is NULL");
    *out = nullptr;
    if (!h || !raw || rows <= 0 || cols <= 0 || cols % 32)
        return set_error(GI_ERR_BAD_ARG, "gi_weights_upload: need a pool handle, weights, rows > 0 and cols % 32 == 0");
    if (ggml_type != W_F32 && ggml_type != W_F16 && ggml_type != W_Q8_0 && ggml_type != W_Q4_0)
        return set_error(GI_ERR_BAD_ARG, "gi_weights_upload: GGML type " + std::to_string(ggml_type) +
                                             " has no device kernel (F32, F16, Q4_0, Q8_0 do)");
    const int64_t nb = cols / 32;
    const int64_t raw_bytes = (int64_t)rows * (ggml_type == W_F32   ? (int64_t)cols * 4
                                               : ggml_type == W_F16 ? (int64_t)cols * 2
                                               : ggml_type == W_Q8_0 ? nb * 34
                                                                     : nb * 18);
    gi_weights *wt = new (std::nothrow) gi_weights();
    if (!wt)
        return set_error(GI_ERR_OOM, "gi_weights_upload: out of host memory");
    wt->h = h;
    wt->type = ggml_type;
    wt->rows = rows;
    wt->cols = cols;
    hipStream_t st = (hipStream_t)gi_paged_stream(h);
    void *tmp = nullptr, *p = nullptr;
    int rc = GI_OK;
    auto alloc = [&](size_t n, void **dst) {
        if (rc == GI_OK)
            rc = gi_dev_alloc(h, n, dst);
    };
    const int64_t rows_pad = weight_rows_pad(rows);
    {
        alloc((size_t)raw_bytes, &tmp);
        if (rc == GI_OK)
            rc = gi_memcpy_h2d(h, tmp, raw, (size_t)raw_bytes);
        hipError_t e = hipSuccess;
        if (ggml_type == W_F16) {
            alloc((size_t)rows_pad * cols * 2, &p);
            wt->a = (uint8_t *)p;
            if (rc == GI_OK) {
                const int64_t n = rows_pad * (cols / 8);
                hipLaunchKernelGGL(convert_f16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                                   (const uint16_t *)tmp, rows, (int)rows_pad, cols, (uint16_t *)wt->a);
                e = hipGetLastError();
            }
        } else if (ggml_type == W_F32) {
            alloc((size_t)rows_pad * cols * 2, &p);
            wt->a = (uint8_t *)p;
            alloc((size_t)rows_pad * cols * 2, &p);
            wt->a_lo = (uint8_t *)p;
            alloc((size_t)rows_pad * 4, &p);
            wt->row_scale = (float *)p;
            if (rc == GI_OK) {
                hipLaunchKernelGGL(convert_f32, dim3((unsigned)rows_pad), dim3(256), 0, st, (const float *)tmp, rows,
                                   cols, (_Float16 *)wt->a, (_Float16 *)wt->a_lo, wt->row_scale);
                e = hipGetLastError();
            }
        } else {
            alloc((size_t)rows_pad * (ggml_type == W_Q8_0 ? cols : cols / 2), &p);
            wt->a = (uint8_t *)p;
            alloc((size_t)rows_pad * nb * 2, &p);
            wt->scales = (uint16_t *)p;
            if (rc == GI_OK) {
                const int64_t n = rows_pad * nb;
                hipLaunchKernelGGL(convert_quant, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                                   (const uint8_t *)tmp, ggml_type, rows, (int)rows_pad, cols, wt->a, wt->scales);
                e = hipGetLastError();
            }
        }
        if (e != hipSuccess && rc == GI_OK)
            rc = hip_fail(e, "gi_weights_upload");
        if (tmp) {
            const int rc2 = gi_dev_free(h, tmp); // waits for the conversion
            if (rc == GI_OK)
                rc = rc2;
        }
    }
    // the pool's device, which every gi_dev_alloc above made current
    (void)hipGetDevice(&wt->device);
    if (rc != GI_OK) {
        gi_weights_destroy(wt);
        return rc;
    }
    *out = wt;
    return GI_OK;
}

void gi_weights_destroy(gi_weights *w)
{
    if (!w)
        return;
    // Does not touch the pool handle, which may be gone already; waits for
    // the device's queued work (which may still read these buffers) first.
    if (hipSetDevice(w->device) == hipSuccess)
        (void)hipDeviceSynchronize();
    for (void *p : {(void *)w->a, (void *)w->a_lo, (void *)w->scales, (void *)w->row_scale})
        if (p)
            (void)hipFree(p);
    gi::devbuf_release(w->xsplit);
    delete w;
}

int gi_matmul_batch(gi_weights *w, int batch, const float *x, float *y)
{
    using namespace gi;
    if (!w || batch < 0 || (batch > 0 && (!x || !y)))
        return set_error(GI_ERR_BAD_ARG, "gi_matmul_batch: bad argument");
    if (batch == 0)
        return GI_OK;
    gi_paged *h = w->h;
    const int rows_pad = (int)weight_rows_pad(w->rows);
    hipStream_t st = (hipStream_t)gi_paged_stream(h);
    hipError_t e = hipSetDevice(w->device);
    if (e != hipSuccess)
        return hip_fail(e, "gi_matmul_batch");
    MatArgs a{};
    a.type = w->type;
    a.rows = w->rows;
    a.rows_pad = rows_pad;
    a.cols = w->cols;
    a.batch = batch;
    a.a = w->a;
    a.a_lo = w->a_lo;
    a.scales = w->scales;
    a.row_scale = w->row_scale;
    a.y = y;
    // matmul_vec writes rows of y while other workgroups still read x: buffers
    // that overlap take the form that splits x first
    const uintptr_t xa = (uintptr_t)x, ya = (uintptr_t)y;
    const bool overlap = xa < ya + (uintptr_t)batch * w->rows * 4 && ya < xa + (uintptr_t)batch * w->cols * 4;
    if (batch <= kVecMaxBatch && !overlap) {
        switch (w->type) {
        case W_F32: launch_vec<W_F32>(a, x, st); break;
        case W_F16: launch_vec<W_F16>(a, x, st); break;
        case W_Q8_0: launch_vec<W_Q8_0>(a, x, st); break;
        default: launch_vec<W_Q4_0>(a, x, st); break;
        }
        e = hipGetLastError();
        return e == hipSuccess ? GI_OK : hip_fail(e, "gi_matmul_batch");
    }
    // hi and lo halves [batch_pad][cols], their row scales (matmul_reg: per
    // segment), then (split-K) the partial tiles [splits][batch_pad][rows_pad]
    const int batch_pad = (int)round_pad(batch);
    const size_t nx = (size_t)batch_pad * w->cols * 2;
    const int KS = w->cols / 32;
    const int64_t tiles64 = (int64_t)((w->rows + 63) / 64) * (batch_pad / 64);
    const bool early = batch > 64 && (RegTiles(w->rows, batch).uneven() || (w->type == W_F32 && KS >= kSplitKF32Steps));
    const bool sk = (w->type == W_F16 || w->type == W_F32) && tiles64 * KS >= kSplitKMinSteps / (early ? 4 : 1);
    int splits = 1, ks_per = KS;
    if (sk) {
        const int tiles = (rows_pad / 128) * ((batch_pad + 127) / 128);
        splits = std::max(1, std::min((kSplitKWorkgroups + tiles - 1) / tiles, KS / kMinSliceSteps));
        ks_per = (KS + splits - 1) / splits;
        splits = (KS + ks_per - 1) / ks_per;
    }
    const size_t part_off = (2 * nx + (size_t)kRegWaves * batch_pad * 4 + 255) / 256 * 256;
    const size_t need = part_off + (splits > 1 ? (size_t)splits * batch_pad * rows_pad * 4 : 0);
    const int rc = devbuf_reserve(w->xsplit, need, st, "gi_matmul_batch");
    if (rc != GI_OK)
        return rc;
    _Float16 *xh = (_Float16 *)w->xsplit.ptr;
    _Float16 *xl = (_Float16 *)((uint8_t *)w->xsplit.ptr + nx);
    float *xscale = (float *)((uint8_t *)w->xsplit.ptr + 2 * nx);
    a.xh = xh;
    a.xl = xl;
    a.xscale = xscale;
    if (sk) {
        hipLaunchKernelGGL(split_rows, dim3((unsigned)batch_pad), dim3(256), 0, st, x, batch, w->cols, xh, xl, xscale);
        SKArgs k{};
        k.m = a;
        k.splits = splits;
        k.ks_per = ks_per;
        k.part = (float *)((uint8_t *)w->xsplit.ptr + part_off);
        k.batch_pad = batch_pad;
        dim3 grid((unsigned)splits, (unsigned)(rows_pad / 128), (unsigned)((batch_pad + 127) / 128));
        if (w->type == W_F32)
            hipLaunchKernelGGL((matmul_sk<W_F32>), grid, dim3(256), 0, st, k);
        else
            hipLaunchKernelGGL((matmul_sk<W_F16>), grid, dim3(256), 0, st, k);
        if (splits > 1) {
            const int64_t n = (int64_t)batch * (rows_pad / 4);
            hipLaunchKernelGGL(reduce_splits, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, k.part, splits,
                               batch, batch_pad, w->rows, rows_pad, xscale,
                               w->type == W_F32 ? (const float *)w->row_scale : nullptr, y);
        }
    } else {
        hipLaunchKernelGGL(split_x, dim3((unsigned)(batch_pad / 16), kRegWaves), dim3(256), 0, st, x, batch,
                           batch_pad, w->cols, xh, xl, xscale);
        switch (w->type) {
        case W_F32: launch_reg<W_F32>(a, batch_pad, st); break;
        case W_F16: launch_reg<W_F16>(a, batch_pad, st); break;
        case W_Q8_0: launch_reg<W_Q8_0>(a, batch_pad, st); break;
        default: launch_reg<W_Q4_0>(a, batch_pad, st); break;
        }
    }
    e = hipGetLastError();
    return e == hipSuccess ? GI_OK : hip_fail(e, "gi_matmul_batch");
}

} // extern "C"
