// Per-token K/V append into pages and block gather back to the reference's
// contiguous layout.
//
// Append restates, on the page layout of gi_common.h, what the reference does
// when it stores one token vector:
//   f32  : copy            (pkg/engine/kvcache.go:173-178, forward.go:236-240)
//   f16  : FP32ToFP16 per element, truncating (pkg/quant/fp16.go:38-69)
//   q8_0 : QuantizeQ8_0 of the whole kv_dim vector (kvcache.go:152-161,
//          pkg/quant/quant.go:407-456), blocks of 32 never straddle a head
//          because head_dim % 32 == 0.
//   q4_0 : QuantizeQ4_0 likewise (kvcache.go:162-171, quant.go:458-521).
// The fused form applies RoPE (pkg/math/kernels.go:22-35) to q and K first,
// as Forward does before its store (forward.go:228-240, 527-545).
// Gather (KVCache.Get / ForkAt, kvcache.go:183-284) rebuilds tokens [0, n)
// of one sequence from its block table: token t lives at
// (block_table[t / page_tokens], t % page_tokens) (paged_kv.go:107-131).
#include "gi_common.h"
#include "gi_kernels.h"
#include "mfma_ops.h"
#include "token_store.h"

#include <algorithm>

namespace gi {

namespace {

constexpr int kThreads = 256;
using mfma_ops::f4;
using mfma_ops::u2;
using mfma_ops::u4;

__device__ __forceinline__ void raise_flag(int *status, int bit)
{
    if (status)
        atomicOr(status, bit);
}

// Resolves token i's destination page and slot.  Explicit mode reads the
// caller's (block id, slot) arrays, as returned by AppendToken; decode mode
// appends at position seq_lens[i]-1 of sequence i through its block table.
struct Dest {
    const int32_t *block_ids;
    const int32_t *slots;
    const int32_t *block_tables;
    const int32_t *seq_lens;
    int max_blocks;
};

__device__ __forceinline__ bool resolve(const Dest &D, const PoolLayout &L, int i,
                                        int64_t *page, int *slot, int *status)
{
    int64_t p;
    int s;
    if (D.block_ids) {
        p = D.block_ids[i];
        s = D.slots[i];
    } else {
        int len = D.seq_lens[i];
        int pos = len - 1;
        int blk = pos >= 0 ? pos / L.page_tokens : -1;
        if (blk < 0 || blk >= D.max_blocks) {
            raise_flag(status, FLAG_BAD_SLOT);
            return false;
        }
        p = D.block_tables[(int64_t)i * D.max_blocks + blk];
        s = pos % L.page_tokens;
    }
    if (p < 0 || p >= L.num_pages) {
        raise_flag(status, FLAG_BAD_PAGE);
        return false;
    }
    if (s < 0 || s >= L.page_tokens) {
        raise_flag(status, FLAG_BAD_SLOT);
        return false;
    }
    *page = p;
    *slot = s;
    return true;
}

// f32 / f16 append: one thread per (token, element); K and V both.
// AT_LEN selects the decode-step form (position from seq_lens); it only
// names the instance so profiles tell the per-step append from bulk writes.
template <int KT, bool AT_LEN>
__global__ __launch_bounds__(kThreads) void append_plain(PoolLayout L, uint8_t *base, int n_tok,
                                                         Dest D, const float *__restrict__ k,
                                                         const float *__restrict__ v, int *status)
{
    const int hd = L.head_dim;
    const int kv_dim = L.num_kv_heads * hd;
    const int64_t total = (int64_t)n_tok * kv_dim;
    for (int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * kThreads) {
        int i = (int)(e / kv_dim);
        int j = (int)(e - (int64_t)i * kv_dim);
        int64_t page;
        int s;
        // Every thread of a token resolves the same destination; only the
        // token's first element raises a flag so each bad token counts once.
        int *st = j == 0 ? status : nullptr;
        if (!resolve(D, L, i, &page, &s, st))
            continue;
        const int kvh = j / hd;
        store_token_elem<KT>(L, base + page * L.page_bytes, s, kvh, j - kvh * hd, k[e], v[e], true);
    }
}

// q8_0 append: 32 consecutive threads quantise one block of 32 elements.
template <bool AT_LEN>
__global__ __launch_bounds__(kThreads) void append_q8(PoolLayout L, uint8_t *base, int n_tok,
                                                      Dest D, const float *__restrict__ k,
                                                      const float *__restrict__ v, int *status)
{
    const int hd = L.head_dim;
    const int kv_dim = L.num_kv_heads * hd;
    const int64_t total = (int64_t)n_tok * kv_dim; // multiple of 32
    for (int64_t e0 = (int64_t)blockIdx.x * kThreads; e0 < total;
         e0 += (int64_t)gridDim.x * kThreads) {
        int64_t e = e0 + threadIdx.x;
        // total and kThreads are multiples of 32, so a 32-lane group is
        // either wholly in range or wholly out: the shuffles below see only
        // complete groups.
        if (e >= total)
            break;
        int i = (int)(e / kv_dim);
        int j = (int)(e - (int64_t)i * kv_dim);
        int64_t page = 0;
        int s = 0;
        int *st = j == 0 ? status : nullptr;
        const bool ok = resolve(D, L, i, &page, &s, st);
        const int kvh = j / hd;
        store_token_elem<KV_Q8_0>(L, base + page * L.page_bytes, s, kvh, j - kvh * hd, k[e], v[e], ok);
    }
}

// q4_0 append: 32 consecutive threads quantise one block of 32 elements
// (QuantizeQ4_0 of the whole kv_dim vector, kvcache.go:162-171).
template <bool AT_LEN>
__global__ __launch_bounds__(kThreads) void append_q4(PoolLayout L, uint8_t *base, int n_tok,
                                                      Dest D, const float *__restrict__ k,
                                                      const float *__restrict__ v, int *status)
{
    const int kv_dim = L.num_kv_heads * L.head_dim;
    const int64_t total = (int64_t)n_tok * kv_dim; // multiple of 32
    for (int64_t e0 = (int64_t)blockIdx.x * kThreads; e0 < total;
         e0 += (int64_t)gridDim.x * kThreads) {
        int64_t e = e0 + threadIdx.x;
        // whole 32-lane groups are in or out of range (see append_q8)
        if (e >= total)
            break;
        int i = (int)(e / kv_dim);
        int j = (int)(e - (int64_t)i * kv_dim);
        int64_t page = 0;
        int s = 0;
        bool ok = resolve(D, L, i, &page, &s, j == 0 ? status : nullptr);
        quant_store_q4(L, base + page * L.page_bytes, s, j, k[e], v[e], ok);
    }
}

// Bulk append with explicit destinations (gi_paged_append, a prefill chunk):
// a workgroup takes kRowTok consecutive tokens of one kv head.  Each thread
// converts 4 consecutive elements of one token (a 32-element quantisation
// block is 8 consecutive lanes), writes them into the token's K row, and
// stages their V form in LDS transposed to [row][token]: V pages are
// dimension-major, so written element by element each V store would touch
// its own 32-byte sector.  Then each thread writes 8 tokens of one V row (or
// of one V-scale row) with one store when they sit on consecutive slots of
// one page with the store aligned (the usual chunk append), token by token
// otherwise; neighbouring lanes write the two halves of a 16-token row.
// Bytes are identical to append_plain / append_q8 / append_q4 (the same
// conversion and quantisation code).  head_dim is a multiple of 32 and at
// most kRowMaxHd.
// s_v rows are kRowPad words apart: 16 put the lanes of a token, 4 rows
// each, on one bank.
//
// ROPE (gi_paged_rope_append of a chunk): K is turned on its way, and
// workgroups of blockIdx.y >= num_kv_heads turn the tile's q, 4 pairs per
// thread and step, into q_out (which may be q: a pair's two ends are read and
// written by one thread).  Same products and sums as rope_append, which took
// one 4-byte pair per thread and stored V element by element.
constexpr int kRowTok = 16, kRowPad = 17, kRowMaxHd = 256;

// 4 consecutive elements x of a head turned with y, the other ends of their
// pairs; lo: x are the first ends (dimensions below rope_half).
__device__ __forceinline__ f4 rope4(f4 x, f4 y, const float2 *cs, bool lo)
{
    const f4 a = *reinterpret_cast<const f4 *>(cs), b = *reinterpret_cast<const f4 *>(cs + 2);
    const float c[4] = {a[0], a[2], b[0], b[2]}, s[4] = {a[1], a[3], b[1], b[3]};
    f4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float y0, y1;
        rope_pair(lo ? x[i] : y[i], lo ? y[i] : x[i], c[i], s[i], &y0, &y1);
        r[i] = lo ? y0 : y1;
    }
    return r;
}

template <int KT, bool ROPE>
__global__ __launch_bounds__(kThreads) void append_rows(PoolLayout L, uint8_t *base, int n_tok, Dest D,
                                                        const float *__restrict__ k, const float *__restrict__ v,
                                                        int *status, RopeArgs R)
{
    const int hd = L.head_dim, P = L.page_tokens, nb = hd / 32;
    const int kv_dim = L.num_kv_heads * hd;
    const int h = blockIdx.y, i0 = blockIdx.x * kRowTok, tid = threadIdx.x;
    const int nt = min(kRowTok, n_tok - i0);
    const int rh = ROPE ? R.rope_half : 0;
    if (ROPE && h >= L.num_kv_heads) {
        // q: per head rh / 4 units of 4 pairs, then the dimensions past 2 rh
        const int upr = rh / 4, per = upr + (hd - 2 * rh) / 4;
        const int total = nt * R.num_heads * per, step = (gridDim.y - L.num_kv_heads) * kThreads;
        for (int u = (h - L.num_kv_heads) * kThreads + tid; u < total; u += step) {
            const int hq = u / per, c = u - hq * per, t = hq / R.num_heads;
            const int pos = R.positions[i0 + t];
            if (pos < 0 || pos >= R.max_pos)
                continue; // reported with its K
            const int64_t o = ((int64_t)i0 * R.num_heads + hq) * hd;
            if (c < upr) {
                const float2 *cs = R.table + (int64_t)pos * rh + 4 * c;
                const f4 x = *reinterpret_cast<const f4 *>(R.q + o + 4 * c);
                const f4 y = *reinterpret_cast<const f4 *>(R.q + o + rh + 4 * c);
                *reinterpret_cast<f4 *>(R.q_out + o + 4 * c) = rope4(x, y, cs, true);
                *reinterpret_cast<f4 *>(R.q_out + o + rh + 4 * c) = rope4(y, x, cs, false);
            } else {
                const int64_t e = o + 2 * rh + 4 * (c - upr);
                *reinterpret_cast<f4 *>(R.q_out + e) = *reinterpret_cast<const f4 *>(R.q + e);
            }
        }
        return;
    }
    const int gpt = hd / 4; // 4-element groups per token
    const int ngroups = kRowTok * gpt;
    __shared__ int64_t s_page[kRowTok];
    __shared__ int s_slot[kRowTok];              // -1: token not stored
    __shared__ int s_pos[kRowTok];               // ROPE: its position
    __shared__ uint32_t s_v[kRowMaxHd * kRowPad]; // V element bits (or codes, q4 bytes) [row][token]
    __shared__ uint16_t s_vs[kRowMaxHd / 32 * kRowTok]; // V block scales [block][token]

    if (tid < kRowTok) {
        int64_t pg = 0;
        int sl = -1;
        // the kv head 0 workgroup reports each bad token once
        bool take = tid < nt;
        if (ROPE && take) {
            const int pos = R.positions[i0 + tid];
            s_pos[tid] = pos;
            if (pos < 0 || pos >= R.max_pos) { // skipped whole
                take = false;
                if (h == 0)
                    raise_flag(status, FLAG_BAD_POS);
            }
        }
        if (take && !resolve(D, L, i0 + tid, &pg, &sl, h == 0 ? status : nullptr))
            sl = -1;
        s_page[tid] = pg;
        s_slot[tid] = sl;
    }
    __syncthreads();

    // ---- K rows, and V converted into LDS ----
    for (int g0 = 0; g0 < ngroups; g0 += kThreads) {
        // whole 8-lane groups (one quantisation block) are in or out of range
        const int g = g0 + tid;
        const int t = g / gpt, a4 = g - t * gpt, d0 = 4 * a4, blk = a4 >> 3, a = a4 & 7;
        const bool in = g < ngroups && t < nt;
        f4 kx = f4{0.0f, 0.0f, 0.0f, 0.0f}, vx = kx;
        if (in) {
            const int64_t e = (int64_t)(i0 + t) * kv_dim + (int64_t)h * hd + d0;
            kx = *reinterpret_cast<const f4 *>(k + e);
            vx = *reinterpret_cast<const f4 *>(v + e);
            if (ROPE && d0 < 2 * rh && s_slot[t] >= 0) {
                const bool lo = d0 < rh;
                const f4 y = *reinterpret_cast<const f4 *>(k + e + (lo ? rh : -rh));
                kx = rope4(kx, y, R.table + (int64_t)s_pos[t] * rh + (lo ? d0 : d0 - rh), lo);
            }
        }
        const int sl = g < ngroups ? s_slot[t] : -1;
        uint8_t *pg = base + (g < ngroups ? s_page[t] : 0) * L.page_bytes;
        const bool st = in && sl >= 0;
        const int64_t krow = (int64_t)h * P + sl; // K row of the token
        uint32_t vb[4];                            // V element bits / codes for s_v
        if constexpr (KT == KV_F32) {
            if (st)
                *reinterpret_cast<f4 *>(pg + L.k_off + (krow * hd + d0) * 4) = kx;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // (copied out before the bit cast: hipcc's __builtin_bit_cast
                // of a vector element reads element 0 whatever the index)
                const float x = vx[c];
                vb[c] = __builtin_bit_cast(uint32_t, x);
            }
        } else if constexpr (KT == KV_F16) {
            uint32_t kh[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                kh[c] = float_to_half_bits_rtz(kx[c]);
                vb[c] = float_to_half_bits_rtz(vx[c]);
            }
            if (st)
                *reinterpret_cast<u2 *>(pg + L.k_off + (krow * hd + d0) * 2) =
                    u2{kh[0] | (kh[1] << 16), kh[2] | (kh[3] << 16)};
        } else {
            uint32_t kk = 0, vk = 0;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                kk = max(kk, abs_key(kx[c]));
                vk = max(vk, abs_key(vx[c]));
            }
#pragma unroll
            for (int m = 1; m < 8; m <<= 1) {
                kk = max(kk, (uint32_t)__shfl_xor((int)kk, m, 8));
                vk = max(vk, (uint32_t)__shfl_xor((int)vk, m, 8));
            }
            float kinv, vinv;
            const bool q8 = KT == KV_Q8_0;
            const uint32_t kd = q8 ? q8_scale(__builtin_bit_cast(float, kk), &kinv)
                                   : q4_scale(__builtin_bit_cast(float, kk), &kinv);
            const uint32_t vd = q8 ? q8_scale(__builtin_bit_cast(float, vk), &vinv)
                                   : q4_scale(__builtin_bit_cast(float, vk), &vinv);
            if (q8) {
                uint32_t kw = 0;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    kw |= ((uint32_t)q8_quant(kx[c], kinv) & 0xFFu) << (8 * c);
                    vb[c] = (uint32_t)q8_quant(vx[c], vinv) & 0xFFu;
                }
                if (st)
                    *reinterpret_cast<uint32_t *>(pg + L.k_off + krow * hd + d0) = kw;
                if (st && a == 0)
                    reinterpret_cast<uint16_t *>(pg + L.ks_off)[krow * nb + blk] = (uint16_t)kd;
            } else {
                // byte j of a block holds element j (low nibble) and j + 16
                // (high): lanes a < 4 take the high nibbles of lane a + 4
                uint32_t kn = 0, vn = 0;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    kn |= (uint32_t)q4_quant(kx[c], kinv) << (8 * c);
                    vn |= (uint32_t)q4_quant(vx[c], vinv) << (8 * c);
                }
                const uint32_t kh = (uint32_t)__shfl_down((int)kn, 4, 8);
                const uint32_t vh = (uint32_t)__shfl_down((int)vn, 4, 8);
                const uint32_t kw = kn | (kh << 4), vw = vn | (vh << 4);
                if (st && a < 4)
                    *reinterpret_cast<uint32_t *>(pg + L.k_off + (krow * nb + blk) * 16 + 4 * a) = kw;
                if (st && a == 0)
                    reinterpret_cast<uint16_t *>(pg + L.ks_off)[krow * nb + blk] = (uint16_t)kd;
#pragma unroll
                for (int c = 0; c < 4; c++)
                    vb[c] = (vw >> (8 * c)) & 0xFFu;
            }
            if (g < ngroups && a == 0)
                s_vs[blk * kRowTok + t] = (uint16_t)vd;
        }
        if (g < ngroups) {
            if (KT == KV_Q4_0) {
                if (a < 4) // byte rows 4a .. 4a + 3 of block blk
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        s_v[(blk * 16 + 4 * a + c) * kRowPad + t] = vb[c];
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++)
                    s_v[(d0 + c) * kRowPad + t] = vb[c];
            }
        }
    }
    __syncthreads();

    // ---- V rows and V-scale rows, 8 tokens per task ----
    constexpr int ESZ = KT == KV_F32 ? 4 : KT == KV_F16 ? 2 : 1;
    const int vrows = KT == KV_Q4_0 ? hd / 2 : hd;
    const bool quant = KT == KV_Q8_0 || KT == KV_Q4_0;
    const int ntask = (vrows + (quant ? nb : 0)) * (kRowTok / 8);
    for (int task = tid; task < ntask; task += kThreads) {
        const int row = task / (kRowTok / 8), t0 = 8 * (task % (kRowTok / 8));
        const bool scale_row = row >= vrows; // quantised pages: V-scale row of block row - vrows
        const int64_t off = scale_row ? L.vs_off + (((int64_t)h * nb + (row - vrows)) * P) * 2
                                      : L.v_off + (((int64_t)h * vrows + row) * P) * ESZ;
        const int esz = scale_row ? 2 : ESZ;
        // one store when the 8 tokens are consecutive slots of one page
        const int s0 = s_slot[t0];
        bool run = s0 >= 0;
#pragma unroll
        for (int t = 1; t < 8; t++)
            run = run && s_slot[t0 + t] == s0 + t && s_page[t0 + t] == s_page[t0];
        uint8_t *dst0 = base + s_page[t0] * L.page_bytes + off + (int64_t)s0 * esz;
        run = run && ((uintptr_t)dst0 & (uintptr_t)(8 * esz - 1)) == 0;
        uint32_t x[8];
#pragma unroll
        for (int t = 0; t < 8; t++)
            x[t] = scale_row ? (uint32_t)s_vs[(row - vrows) * kRowTok + t0 + t] : s_v[row * kRowPad + t0 + t];
        if (run) {
            if (esz == 4) {
                reinterpret_cast<u4 *>(dst0)[0] = u4{x[0], x[1], x[2], x[3]};
                reinterpret_cast<u4 *>(dst0)[1] = u4{x[4], x[5], x[6], x[7]};
            } else if (esz == 2) {
                *reinterpret_cast<u4 *>(dst0) =
                    u4{x[0] | (x[1] << 16), x[2] | (x[3] << 16), x[4] | (x[5] << 16), x[6] | (x[7] << 16)};
            } else {
                *reinterpret_cast<u2 *>(dst0) = u2{x[0] | (x[1] << 8) | (x[2] << 16) | (x[3] << 24),
                                                   x[4] | (x[5] << 8) | (x[6] << 16) | (x[7] << 24)};
            }
        } else {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int s = s_slot[t0 + t];
                if (s < 0)
                    continue;
                uint8_t *d = base + s_page[t0 + t] * L.page_bytes + off + (int64_t)s * esz;
                if (esz == 4)
                    *reinterpret_cast<uint32_t *>(d) = x[t];
                else if (esz == 2)
                    *reinterpret_cast<uint16_t *>(d) = (uint16_t)x[t];
                else
                    *d = (uint8_t)x[t];
            }
        }
    }
}

// Gather of pages of whole 16-token groups at head dimension 64 or 128.  A
// workgroup takes kGatherTok tokens of one kv head, K and V.  Bytes bound it
// (each read and written once), so every load and store is 16 bytes of one
// run: f32 and f16 K rows go straight through; V, and the codes and scales
// of quantised pages, are put together in LDS as the token rows the host's
// layout has (ROW bytes: f32 and f16 elements, 34- or 18-byte blocks), which
// leave as 16-byte (quantised rows: 4-byte) stores or widened to float4.  V
// pages are dimension-major: read element by element in output order, as
// gather_kernel does, a wave touched 64 sectors per 128 bytes.  Bytes are
// gather_kernel's.  Llama-3-8B shape, us a call, gather_kernel / here: 6001
// tokens fp16 23.75 / 8.94, q8_0 29.2 / 8.4, q4_0 15.4 / 7.2; 16000 tokens fp16
// 58.4 / 20.8, widened 64.1 / 33.7.
constexpr int kGatherTok = 32;

template <int KT, int HD, bool WIDEN>
__global__ __launch_bounds__(kThreads) void gather_tiles(PoolLayout L, const uint8_t *base,
                                                         const int32_t *__restrict__ table, int n_tok,
                                                         uint8_t *kout, uint8_t *vout, int *status)
{
    constexpr bool QUANT = KT == KV_Q8_0 || KT == KV_Q4_0;
    constexpr int NB = HD / 32;
    constexpr int ROW = KT == KV_F32 ? 4 * HD : KT == KV_F16 ? 2 * HD : KT == KV_Q8_0 ? 34 * NB : 18 * NB;
    // row stride in LDS: 16-byte aligned rows that start 4 (f32, f16) banks
    // apart, quantised rows packed
    constexpr int LROW = QUANT ? ROW : ROW + 16;
    constexpr int T = kGatherTok;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) uint8_t s_v[T * LROW];
    __shared__ __align__(16) uint8_t s_k[QUANT ? T * LROW : 16];
    __shared__ int64_t s_page[T / 16]; // page offset of each 16-token group, -1: none
    const int t0 = blockIdx.x * T, kvh = blockIdx.y, tid = threadIdx.x;
    const int P = L.page_tokens;
    if (tid < T / 16) {
        const int t = t0 + 16 * tid;
        int64_t off = -1;
        if (t < n_tok) {
            const int64_t page = table[t / P];
            if (page >= 0 && page < L.num_pages)
                off = page * L.page_bytes;
            else if (kvh == 0)
                raise_flag(status, FLAG_BAD_PAGE);
        }
        s_page[tid] = off;
    }
    __syncthreads();
    const int64_t row_out = (int64_t)L.num_kv_heads * (WIDEN ? 4 * HD : ROW); // bytes of a token vector
    const int64_t head_out = (int64_t)kvh * (WIDEN ? 4 * HD : ROW);

    // ---- K rows and V units of 16 bytes ----
    if constexpr (!QUANT) {
        constexpr int E = KT == KV_F32 ? 4 : 2, U = ROW / 16; // 16-byte units of a K row
        for (int u = tid; u < T * U; u += kThreads) {
            const int r = u / U, c = u - r * U, t = t0 + r;
            const int64_t off = s_page[r >> 4];
            if (t >= n_tok || off < 0)
                continue;
            const u4 x = *reinterpret_cast<const u4 *>(base + off + L.k_off + ((int64_t)kvh * P + t % P) * ROW + 16 * c);
            uint8_t *o = kout + t * row_out + head_out;
            if constexpr (WIDEN && KT == KV_F16) {
                float4 *w = reinterpret_cast<float4 *>(o + 32 * c);
                w[0] = float4{half_bits_to_float(x[0] & 0xFFFFu), half_bits_to_float(x[0] >> 16),
                              half_bits_to_float(x[1] & 0xFFFFu), half_bits_to_float(x[1] >> 16)};
                w[1] = float4{half_bits_to_float(x[2] & 0xFFFFu), half_bits_to_float(x[2] >> 16),
                              half_bits_to_float(x[3] & 0xFFFFu), half_bits_to_float(x[3] >> 16)};
            } else {
                *reinterpret_cast<u4 *>(o + 16 * c) = x;
            }
        }
        // V unit: TU tokens of one dimension
        constexpr int TU = 16 / E, UG = 16 / TU; // units per dimension and 16-token group
        for (int u = tid; u < T / TU * HD; u += kThreads) {
            const int grp = u / (UG * HD), d = u % (UG * HD) / UG, q = u % UG;
            const int r = 16 * grp + TU * q;
            const int64_t off = s_page[grp];
            if (off < 0)
                continue;
            const u4 x = *reinterpret_cast<const u4 *>(base + off + L.v_off +
                                                       (((int64_t)kvh * HD + d) * P + (t0 + r) % P) * E);
#pragma unroll
            for (int i = 0; i < TU; i++) {
                if constexpr (E == 4)
                    *reinterpret_cast<uint32_t *>(&s_v[(r + i) * LROW + 4 * d]) = x[i];
                else
                    *reinterpret_cast<uint16_t *>(&s_v[(r + i) * LROW + 2 * d]) = (uint16_t)(x[i / 2] >> (16 * (i & 1)));
            }
        }
    } else {
        constexpr int CB = KT == KV_Q8_0 ? 32 : 16, BB = CB + 2; // code bytes and bytes of a block
        constexpr int KU = NB * CB / 16;                         // 16-byte units of a K code row
        auto put = [&](uint8_t *row, int at, u4 x) { // 16 code bytes at an even offset
#pragma unroll
            for (int i = 0; i < 8; i++)
                *reinterpret_cast<uint16_t *>(row + at + 2 * i) = (uint16_t)(x[i / 2] >> (16 * (i & 1)));
        };
        for (int u = tid; u < T * KU; u += kThreads) {
            const int r = u / KU, c = u - r * KU;
            const int64_t off = s_page[r >> 4];
            if (off < 0)
                continue;
            const u4 x = *reinterpret_cast<const u4 *>(base + off + L.k_off +
                                                       (((int64_t)kvh * P + (t0 + r) % P) * KU + c) * 16);
            const int b = c * 16 / CB;
            put(&s_k[r * LROW], b * BB + 2 + c * 16 % CB, x);
        }
        // V unit: 16 tokens of one code row
        for (int u = tid; u < T / 16 * NB * CB; u += kThreads) {
            const int grp = u / (NB * CB), cr = u % (NB * CB);
            const int64_t off = s_page[grp];
            if (off < 0)
                continue;
            const u4 x = *reinterpret_cast<const u4 *>(base + off + L.v_off + ((int64_t)kvh * NB * CB + cr) * P +
                                                       (t0 + 16 * grp) % P);
            const int at = cr / CB * BB + 2 + cr % CB;
#pragma unroll
            for (int i = 0; i < 16; i++)
                s_v[(16 * grp + i) * LROW + at] = (uint8_t)(x[i / 4] >> (8 * (i & 3)));
        }
        for (int u = tid; u < T * NB; u += kThreads) {
            const int r = u / NB, b = u - r * NB, s = (t0 + r) % P;
            const int64_t off = s_page[r >> 4];
            if (off < 0)
                continue;
            *reinterpret_cast<uint16_t *>(&s_k[r * LROW + b * BB]) =
                reinterpret_cast<const uint16_t *>(base + off + L.ks_off)[((int64_t)kvh * P + s) * NB + b];
            *reinterpret_cast<uint16_t *>(&s_v[r * LROW + b * BB]) =
                reinterpret_cast<const uint16_t *>(base + off + L.vs_off)[((int64_t)kvh * NB + b) * P + s];
        }
    }
    __syncthreads();

    // ---- LDS rows to the output ----
    auto emit = [&](const uint8_t *rows, uint8_t *out) {
        if constexpr (!WIDEN || KT == KV_F32) {
            constexpr int OU = QUANT ? 4 : 16, U = ROW / OU;
            for (int u = tid; u < T * U; u += kThreads) {
                const int r = u / U, c = u - r * U, t = t0 + r;
                if (t >= n_tok || s_page[r >> 4] < 0)
                    continue;
                uint8_t *o = out + t * row_out + head_out + OU * c;
                if constexpr (QUANT)
                    *reinterpret_cast<uint32_t *>(o) = *reinterpret_cast<const uint32_t *>(rows + r * LROW + 4 * c);
                else
                    *reinterpret_cast<u4 *>(o) = *reinterpret_cast<const u4 *>(rows + r * LROW + 16 * c);
            }
        } else {
            constexpr int U = HD / 4;
            for (int u = tid; u < T * U; u += kThreads) {
                const int r = u / U, d = 4 * (u - r * U), t = t0 + r;
                if (t >= n_tok || s_page[r >> 4] < 0)
                    continue;
                const uint8_t *row = rows + r * LROW;
                float f[4];
                if constexpr (KT == KV_F16) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        f[i] = half_bits_to_float(*reinterpret_cast<const uint16_t *>(row + 2 * (d + i)));
                } else if constexpr (KT == KV_Q8_0) {
                    const uint8_t *blk = row + d / 32 * 34;
                    const float sc = half_bits_to_float(*reinterpret_cast<const uint16_t *>(blk));
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        f[i] = (float)(int8_t)blk[2 + d % 32 + i] * sc;
                } else {
                    const uint8_t *blk = row + d / 32 * 18;
                    const float sc = half_bits_to_float(*reinterpret_cast<const uint16_t *>(blk));
                    const int sh = d & 16 ? 4 : 0;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        f[i] = (float)(((blk[2 + (d & 15) + i] >> sh) & 15) - 8) * sc;
                }
                *reinterpret_cast<float4 *>(out + t * row_out + head_out + 4 * d) = float4{f[0], f[1], f[2], f[3]};
            }
        }
    };
    if constexpr (QUANT)
        emit(s_k, kout);
    emit(s_v, vout);
}

// Gather one sequence's tokens [0, n_tok) of one layer, element by element:
// the page sizes and output alignments gather_tiles does not take, and short
// sequences at 4 bytes an element.
//   widen == 0: stored format, the reference's bytes per token vector
//               (f32: 4*kv_dim, f16: 2*kv_dim, q8_0: kv_dim/32 blocks of
//               34 bytes = LE fp16 scale + 32 int8, quant.go:38-41).
//   widen == 1: float32 values (FP16ToFP32 / DequantizeQ8_0).
template <int KT, int WIDEN>
__global__ __launch_bounds__(kThreads) void gather_kernel(PoolLayout L, const uint8_t *base,
                                                          const int32_t *__restrict__ table,
                                                          int n_tok, uint8_t *kout, uint8_t *vout,
                                                          int *status)
{
    const int hd = L.head_dim;
    const int kv_dim = L.num_kv_heads * hd;
    const int P = L.page_tokens;
    const int nb = hd / 32;
    // Units per token: one per element, except raw q8_0 / q4_0: one per byte.
    const int per_tok = (KT == KV_Q8_0 && !WIDEN) ? (kv_dim / 32) * 34
                        : (KT == KV_Q4_0 && !WIDEN) ? (kv_dim / 32) * 18
                                                    : kv_dim;
    const int64_t total = (int64_t)n_tok * per_tok;
    for (int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * kThreads) {
        int t = (int)(e / per_tok);
        int u = (int)(e - (int64_t)t * per_tok);
        int64_t page = table[t / P];
        int s = t % P;
        if (page < 0 || page >= L.num_pages) {
            if (u == 0)
                raise_flag(status, FLAG_BAD_PAGE);
            continue;
        }
        const uint8_t *pg = base + page * L.page_bytes;
        if (KT == KV_Q4_0) {
            // 18-byte blocks: LE fp16 scale, then byte j = dim j | dim j+16 << 4
            int b, r;
            if (WIDEN) {
                b = u >> 5;
                r = 2 + (u & 15); // the byte holding dim u & 31
            } else {
                b = u / 18;
                r = u - b * 18;
            }
            const int kvh = b / nb, blk = b - kvh * nb;
            const uint16_t ks = reinterpret_cast<const uint16_t *>(pg + L.ks_off)[((int64_t)kvh * P + s) * nb + blk];
            const uint16_t vs = reinterpret_cast<const uint16_t *>(pg + L.vs_off)[((int64_t)kvh * nb + blk) * P + s];
            uint8_t kb = 0, vb = 0;
            if (r >= 2) {
                kb = pg[L.k_off + (((int64_t)kvh * P + s) * nb + blk) * 16 + (r - 2)];
                vb = pg[L.v_off + (((int64_t)kvh * nb + blk) * 16 + (r - 2)) * P + s];
            }
            if (WIDEN) { // (nibble - 8) * d (quant.go:103-110)
                const int sh = (u & 16) ? 4 : 0;
                reinterpret_cast<float *>(kout)[e] = (float)(((kb >> sh) & 15) - 8) * half_bits_to_float(ks);
                reinterpret_cast<float *>(vout)[e] = (float)(((vb >> sh) & 15) - 8) * half_bits_to_float(vs);
            } else {
                kout[e] = r == 0 ? (uint8_t)(ks & 0xFF) : r == 1 ? (uint8_t)(ks >> 8) : kb;
                vout[e] = r == 0 ? (uint8_t)(vs & 0xFF) : r == 1 ? (uint8_t)(vs >> 8) : vb;
            }
            continue;
        }
        if (KT == KV_Q8_0 && !WIDEN) {
            int b = u / 34, r = u - b * 34; // global 32-block index and byte
            int kvh = b / nb, blk = b - kvh * nb;
            uint8_t kb, vb;
            if (r < 2) {
                uint16_t ks = reinterpret_cast<const uint16_t *>(pg + L.ks_off)
                    [((int64_t)kvh * P + s) * nb + blk];
                uint16_t vs = reinterpret_cast<const uint16_t *>(pg + L.vs_off)
                    [((int64_t)kvh * nb + blk) * P + s];
                kb = (uint8_t)(r == 0 ? ks & 0xFF : ks >> 8);
                vb = (uint8_t)(r == 0 ? vs & 0xFF : vs >> 8);
            } else {
                int d = blk * 32 + (r - 2);
                kb = (pg + L.k_off)[((int64_t)kvh * P + s) * hd + d];
                vb = (pg + L.v_off)[((int64_t)kvh * hd + d) * P + s];
            }
            kout[e] = kb;
            vout[e] = vb;
            continue;
        }
        int kvh = u / hd;
        int d = u - kvh * hd;
        int64_t ki = ((int64_t)kvh * P + s) * hd + d;
        int64_t vi = ((int64_t)kvh * hd + d) * P + s;
        if (KT == KV_F32) {
            reinterpret_cast<float *>(kout)[e] = reinterpret_cast<const float *>(pg + L.k_off)[ki];
            reinterpret_cast<float *>(vout)[e] = reinterpret_cast<const float *>(pg + L.v_off)[vi];
        } else if (KT == KV_F16) {
            uint16_t kh = reinterpret_cast<const uint16_t *>(pg + L.k_off)[ki];
            uint16_t vh = reinterpret_cast<const uint16_t *>(pg + L.v_off)[vi];
            if (WIDEN) {
                reinterpret_cast<float *>(kout)[e] = half_bits_to_float(kh);
                reinterpret_cast<float *>(vout)[e] = half_bits_to_float(vh);
            } else {
                reinterpret_cast<uint16_t *>(kout)[e] = kh;
                reinterpret_cast<uint16_t *>(vout)[e] = vh;
            }
        } else { // q8_0 widened: float32(int8 q) * FP16ToFP32(d) (quant.go:207)
            int blk = d >> 5;
            float ks = half_bits_to_float(reinterpret_cast<const uint16_t *>(pg + L.ks_off)
                                              [((int64_t)kvh * P + s) * nb + blk]);
            float vs = half_bits_to_float(reinterpret_cast<const uint16_t *>(pg + L.vs_off)
                                              [((int64_t)kvh * nb + blk) * P + s]);
            int8_t kq = reinterpret_cast<const int8_t *>(pg + L.k_off)[ki];
            int8_t vq = reinterpret_cast<const int8_t *>(pg + L.v_off)[vi];
            reinterpret_cast<float *>(kout)[e] = (float)kq * ks;
            reinterpret_cast<float *>(vout)[e] = (float)vq * vs;
        }
    }
}

int grid_for(int64_t units)
{
    int64_t g = (units + kThreads - 1) / kThreads;
    if (g > 65536)
        g = 65536;
    return g < 1 ? 1 : (int)g;
}

hipError_t append_any(const PoolLayout &L, uint8_t *base, int n_tok, const Dest &D,
                      const float *k, const float *v, int *status, hipStream_t st)
{
    if (n_tok <= 0)
        return hipSuccess;
    const bool at_len = D.block_ids == nullptr;
    // the row kernel reads K/V 16 bytes at a time: inputs of any other
    // alignment (a caller's float pointer) take the per-element kernels
    const bool aligned16 = ((uintptr_t)k % 16 == 0) && ((uintptr_t)v % 16 == 0);
    if (!at_len && aligned16 && L.head_dim % 32 == 0 && L.head_dim <= kRowMaxHd) {
        dim3 rgrid((unsigned)((n_tok + kRowTok - 1) / kRowTok), (unsigned)L.num_kv_heads);
#define GI_ROWS(KT) hipLaunchKernelGGL((append_rows<KT, false>), rgrid, dim3(kThreads), 0, st, L, base, n_tok, D, k, v, status, \
                       RopeArgs{})
        switch (L.kv_type) {
        case KV_F32:
            GI_ROWS(KV_F32);
            break;
        case KV_F16:
            GI_ROWS(KV_F16);
            break;
        case KV_Q4_0:
            GI_ROWS(KV_Q4_0);
            break;
        default:
            GI_ROWS(KV_Q8_0);
            break;
        }
#undef GI_ROWS
        return hipGetLastError();
    }
    int64_t units = (int64_t)n_tok * L.num_kv_heads * L.head_dim;
    dim3 grid(grid_for(units)), block(kThreads);
#define GI_APPEND(KERNEL)                                                                    \
    hipLaunchKernelGGL(KERNEL, grid, block, 0, st, L, base, n_tok, D, k, v, status)
    switch (L.kv_type) {
    case KV_F32:
        if (at_len)
            GI_APPEND((append_plain<KV_F32, true>));
        else
            GI_APPEND((append_plain<KV_F32, false>));
        break;
    case KV_F16:
        if (at_len)
            GI_APPEND((append_plain<KV_F16, true>));
        else
            GI_APPEND((append_plain<KV_F16, false>));
        break;
    case KV_Q4_0:
        if (at_len)
            GI_APPEND(append_q4<true>);
        else
            GI_APPEND(append_q4<false>);
        break;
    default:
        if (at_len)
            GI_APPEND(append_q8<true>);
        else
            GI_APPEND(append_q8<false>);
        break;
    }
#undef GI_APPEND
    return hipGetLastError();
}

// Rotates the first 2*rh dims of each of n_heads heads of x (head stride hd)
// into y; the dims past 2*rh are copied.  Pair p = (head, j) is (j, j + rh)
// of that head.  Pairs [p0, p0 + step * k) go to the threads of the
// workgroup in turn, and y may alias x: every element is read and written
// by the one thread that owns its pair.
__device__ __forceinline__ void rope_rows(const float *x, float *y, int n_heads, int hd, int rh,
                                          const float2 *cs, int p0, int step)
{
    for (int p = p0 + threadIdx.x; p < n_heads * rh; p += step) {
        int h = p / rh, j = p - h * rh;
        const float *xh = x + (int64_t)h * hd;
        float *yh = y + (int64_t)h * hd;
        float2 t = cs[j];
        float y0, y1;
        rope_pair(xh[j], xh[j + rh], t.x, t.y, &y0, &y1);
        yh[j] = y0;
        yh[j + rh] = y1;
    }
    const int rest = hd - 2 * rh;
    if (rest > 0) {
        for (int p = p0 + threadIdx.x; p < n_heads * rest; p += step) {
            int h = p / rest, j = 2 * rh + (p - h * rest);
            y[(int64_t)h * hd + j] = x[(int64_t)h * hd + j];
        }
    }
}

// Fused RoPE + append.  Grid (n_tok, 1 + q_blocks): block (i, 0) turns
// token i's K into LDS and stores K (in the pool's format: f32 copy,
// truncated fp16, or Q8_0 blocks of the rotated vector) and V; block
// (i, 1 + b) turns kThreads pairs of token i's q into q_out, one pair per
// thread, so no thread waits on a chain of dependent loads.  A token whose
// position is outside the table is skipped whole (its q_out row is not
// written); one whose page or slot is bad has its q turned but nothing
// stored.
template <int KT, bool AT_LEN>
__global__ __launch_bounds__(kThreads) void rope_append(PoolLayout L, uint8_t *base, Dest D, RopeArgs R,
                                                        const float *__restrict__ k,
                                                        const float *__restrict__ v, int *status)
{
    extern __shared__ float sk[]; // kv_dim rotated K values
    const int i = blockIdx.x;
    const int hd = L.head_dim;
    const int kv_dim = L.num_kv_heads * hd;
    const int pos = AT_LEN ? D.seq_lens[i] - 1 : R.positions[i];
    if (pos < 0 || pos >= R.max_pos) {
        if (threadIdx.x == 0 && blockIdx.y == 0)
            raise_flag(status, FLAG_BAD_POS);
        return;
    }
    const float2 *cs = R.table + (int64_t)pos * R.rope_half;
    if (blockIdx.y > 0) {
        const int64_t qo = (int64_t)i * R.num_heads * hd;
        const int nqb = gridDim.y - 1;
        rope_rows(R.q + qo, R.q_out + qo, R.num_heads, hd, R.rope_half, cs,
                  (int)(blockIdx.y - 1) * kThreads, nqb * kThreads);
        return;
    }
    const float *kx = k + (int64_t)i * kv_dim;
    const float *vx = v + (int64_t)i * kv_dim;
    rope_rows(kx, sk, L.num_kv_heads, hd, R.rope_half, cs, 0, kThreads);
    __syncthreads();
    int64_t page;
    int s;
    // every thread resolves the same destination; thread 0 reports
    if (!resolve(D, L, i, &page, &s, threadIdx.x == 0 ? status : nullptr))
        return;
    uint8_t *pg = base + page * L.page_bytes;
    const int P = L.page_tokens;
    if (KT == KV_Q4_0) {
        // 32-lane groups are whole blocks in every iteration (see below)
        for (int e = threadIdx.x; e < kv_dim; e += kThreads)
            quant_store_q4(L, pg, s, e, sk[e], vx[e], true);
        return;
    }
    if (KT == KV_Q8_0) {
        const int nb = hd / 32;
        // kv_dim and kThreads are multiples of 32: a 32-lane group (one
        // Q8_0 block) is wholly in or out of range in every iteration.
        for (int e = threadIdx.x; e < kv_dim; e += kThreads) {
            float kv0 = sk[e], vv0 = vx[e];
            float kinv, vinv;
            uint32_t kd = q8_scale(__builtin_bit_cast(float, max32(abs_key(kv0))), &kinv);
            uint32_t vd = q8_scale(__builtin_bit_cast(float, max32(abs_key(vv0))), &vinv);
            int kvh = e / hd, d = e - kvh * hd, blk = d >> 5;
            reinterpret_cast<int8_t *>(pg + L.k_off)[((int64_t)kvh * P + s) * hd + d] = (int8_t)q8_quant(kv0, kinv);
            reinterpret_cast<int8_t *>(pg + L.v_off)[((int64_t)kvh * hd + d) * P + s] = (int8_t)q8_quant(vv0, vinv);
            if ((d & 31) == 0) {
                reinterpret_cast<uint16_t *>(pg + L.ks_off)[((int64_t)kvh * P + s) * nb + blk] = (uint16_t)kd;
                reinterpret_cast<uint16_t *>(pg + L.vs_off)[((int64_t)kvh * nb + blk) * P + s] = (uint16_t)vd;
            }
        }
        return;
    }
    for (int e = threadIdx.x; e < kv_dim; e += kThreads) {
        int kvh = e / hd, d = e - kvh * hd;
        int64_t ki = ((int64_t)kvh * P + s) * hd + d;
        int64_t vi = ((int64_t)kvh * hd + d) * P + s;
        if (KT == KV_F32) {
            reinterpret_cast<float *>(pg + L.k_off)[ki] = sk[e];
            reinterpret_cast<float *>(pg + L.v_off)[vi] = vx[e];
        } else {
            reinterpret_cast<uint16_t *>(pg + L.k_off)[ki] = (uint16_t)float_to_half_bits_rtz(sk[e]);
            reinterpret_cast<uint16_t *>(pg + L.v_off)[vi] = (uint16_t)float_to_half_bits_rtz(vx[e]);
        }
    }
}

} // namespace

hipError_t launch_append(const PoolLayout &L, uint8_t *base, int n_tok, const int32_t *block_ids,
                         const int32_t *slots, const float *k, const float *v, int *status,
                         hipStream_t st)
{
    Dest D{block_ids, slots, nullptr, nullptr, 0};
    return append_any(L, base, n_tok, D, k, v, status, st);
}

hipError_t launch_append_at_len(const PoolLayout &L, uint8_t *base, int batch,
                                const int32_t *block_tables, int max_blocks,
                                const int32_t *seq_lens, const float *k, const float *v,
                                int *status, hipStream_t st)
{
    Dest D{nullptr, nullptr, block_tables, seq_lens, max_blocks};
    return append_any(L, base, batch, D, k, v, status, st);
}

// Elements of q (or 4 x K) from which a RoPE append goes by rows: below, the
// rows' longer chain (destinations, LDS) costs more than its wider accesses
// give.  us a call, rope_append / rows: Llama-3-8B shape fp16 512 tokens 8.5 /
// 7.7, 1024 13.7 / 10.2, 2048 24.0 / 16.4, f32 2048 31.3 / 17.3, q8_0 300 9.9 /
// 10.7; TinyLlama shape f32 300 tokens with the attention behind it 24.8 /
// 25.4, 2048 tokens 13.7 / 8.6.  And fp16 and q8_0 chunks from kRopeRowsTok
// tokens only: Llama-3-70B shape fp16 256 7.1 / 7.7, 512 10.7 / 9.1, q8_0 300
// 10.4 / 11.4, 512 11.5 / 11.5 (f32 256 7.6 / 6.6, q4_0 9.7 / 8.9).
constexpr int64_t kRopeRowsMin = 512 * 4096;
constexpr int kRopeRowsTok = 512;

hipError_t launch_rope_append(const PoolLayout &L, uint8_t *base, int n_tok, const int32_t *block_ids,
                              const int32_t *slots, const int32_t *block_tables, int max_blocks,
                              const int32_t *seq_lens, const RopeArgs &R, const float *k,
                              const float *v, int *status, hipStream_t st)
{
    if (n_tok <= 0)
        return hipSuccess;
    Dest D{block_ids, slots, block_tables, seq_lens, max_blocks};
    const bool at_len = block_ids == nullptr;
    const size_t lds = sizeof(float) * (size_t)L.num_kv_heads * L.head_dim;
    // a chunk: whole rows, where 16-byte accesses and groups of 4 pairs fit
    const uintptr_t ptrs = (uintptr_t)k | (uintptr_t)v | (uintptr_t)R.q | (uintptr_t)R.q_out | (uintptr_t)R.table;
    const int64_t elems = (int64_t)n_tok * std::max(R.num_heads, 4 * L.num_kv_heads) * L.head_dim;
    const bool enough = elems >= kRopeRowsMin &&
                        (n_tok >= kRopeRowsTok || L.kv_type == KV_F32 || L.kv_type == KV_Q4_0);
    if (!at_len && enough && ptrs % 16 == 0 && R.rope_half % 4 == 0 && L.head_dim % 32 == 0 &&
        L.head_dim <= kRowMaxHd) {
        const int per = R.rope_half / 4 + (L.head_dim - 2 * R.rope_half) / 4;
        const int64_t qb = ((int64_t)kRowTok * R.num_heads * per + kThreads - 1) / kThreads;
        const dim3 rgrid((unsigned)((n_tok + kRowTok - 1) / kRowTok),
                         (unsigned)(L.num_kv_heads + std::min<int64_t>(qb, 1024)));
#define GI_ROPE_ROWS(KT) \
    hipLaunchKernelGGL((append_rows<KT, true>), rgrid, dim3(kThreads), 0, st, L, base, n_tok, D, k, v, status, R)
        switch (L.kv_type) {
        case KV_F32: GI_ROPE_ROWS(KV_F32); break;
        case KV_F16: GI_ROPE_ROWS(KV_F16); break;
        case KV_Q4_0: GI_ROPE_ROWS(KV_Q4_0); break;
        default: GI_ROPE_ROWS(KV_Q8_0); break;
        }
#undef GI_ROPE_ROWS
        return hipGetLastError();
    }
    // q blocks: one rotated pair (or copied dim past rope_dim) per thread
    const int64_t q_units = (int64_t)R.num_heads *
                            std::max(R.rope_half, L.head_dim - 2 * R.rope_half);
    const int nqb = (int)((q_units + kThreads - 1) / kThreads);
    dim3 grid((unsigned)n_tok, (unsigned)(1 + nqb)), block(kThreads);
#define GI_ROPE(KT)                                                                                \
    do {                                                                                           \
        if (at_len)                                                                                \
            hipLaunchKernelGGL((rope_append<KT, true>), grid, block, lds, st, L, base, D, R, k, v, \
                               status);                                                            \
        else                                                                                       \
            hipLaunchKernelGGL((rope_append<KT, false>), grid, block, lds, st, L, base, D, R, k,   \
                               v, status);                                                         \
    } while (0)
    switch (L.kv_type) {
    case KV_F32:
        GI_ROPE(KV_F32);
        break;
    case KV_F16:
        GI_ROPE(KV_F16);
        break;
    case KV_Q4_0:
        GI_ROPE(KV_Q4_0);
        break;
    default:
        GI_ROPE(KV_Q8_0);
        break;
    }
#undef GI_ROPE
    return hipGetLastError();
}

hipError_t launch_gather(const PoolLayout &L, const uint8_t *base, const int32_t *table, int n_tok,
                         void *k_out, void *v_out, int widen, int *status, hipStream_t st)
{
    if (n_tok <= 0)
        return hipSuccess;
    int kv_dim = L.num_kv_heads * L.head_dim;
    int64_t per_tok = (L.kv_type == KV_Q8_0 && !widen) ? (kv_dim / 32) * 34
                      : (L.kv_type == KV_Q4_0 && !widen) ? (kv_dim / 32) * 18
                                                         : kv_dim;
    dim3 grid(grid_for((int64_t)n_tok * per_tok)), block(kThreads);
    uint8_t *ko = (uint8_t *)k_out, *vo = (uint8_t *)v_out;
    // gather_tiles' 16-byte accesses: pages of whole 16-token groups, output
    // rows on 16-byte (stored quantised blocks: 4-byte) boundaries.  Where 4
    // bytes an element are written, short sequences are too few workgroups of
    // 32 tokens: element by element below these numbers of elements (us a call,
    // that / tiles, Llama-3-8B shape: widened fp16 200 tokens 4.6 / 6.6, 600
    // 5.4 / 7.1, 2000 11.2 / 8.7; widened q8_0 200 4.6 / 5.5, 600 5.9 / 5.8; f32 200
    // 4.5 / 5.0, 600 5.3 / 5.5, 2000 11.6 / 7.8, TinyLlama shape 2000 5.4 / 4.7).
    const int64_t tiles_from = !widen && L.kv_type != KV_F32 ? 0 : L.kv_type == KV_F16 ? 1 << 20 : 3 << 17;
    const uintptr_t mask = ((L.kv_type == KV_Q8_0 || L.kv_type == KV_Q4_0) && !widen) ? 3 : 15;
    if ((int64_t)n_tok * kv_dim >= tiles_from && L.page_tokens % 16 == 0 &&
        (L.head_dim == 64 || L.head_dim == 128) && (((uintptr_t)k_out | (uintptr_t)v_out) & mask) == 0 &&
        L.num_kv_heads <= 65535) {
        const dim3 tg((unsigned)((n_tok + kGatherTok - 1) / kGatherTok), (unsigned)L.num_kv_heads);
#define GI_TILES(KT, W)                                                                                            \
    do {                                                                                                           \
        if (L.head_dim == 128)                                                                                     \
            hipLaunchKernelGGL((gather_tiles<KT, 128, W>), tg, block, 0, st, L, base, table, n_tok, ko, vo, status); \
        else                                                                                                       \
            hipLaunchKernelGGL((gather_tiles<KT, 64, W>), tg, block, 0, st, L, base, table, n_tok, ko, vo, status); \
        return hipGetLastError();                                                                                  \
    } while (0)
        switch (L.kv_type) {
        case KV_F32: GI_TILES(KV_F32, false);
        case KV_F16:
            if (widen)
                GI_TILES(KV_F16, true);
            GI_TILES(KV_F16, false);
        case KV_Q4_0:
            if (widen)
                GI_TILES(KV_Q4_0, true);
            GI_TILES(KV_Q4_0, false);
        default:
            if (widen)
                GI_TILES(KV_Q8_0, true);
            GI_TILES(KV_Q8_0, false);
        }
#undef GI_TILES
    }
#define GI_GATHER(KT, W) \
    hipLaunchKernelGGL((gather_kernel<KT, W>), grid, block, 0, st, L, base, table, n_tok, ko, vo, status)
    if (L.kv_type == KV_F32) {
        GI_GATHER(KV_F32, 0);
    } else if (L.kv_type == KV_F16) {
        if (widen)
            GI_GATHER(KV_F16, 1);
        else
            GI_GATHER(KV_F16, 0);
    } else if (L.kv_type == KV_Q4_0) {
        if (widen)
            GI_GATHER(KV_Q4_0, 1);
        else
            GI_GATHER(KV_Q4_0, 0);
    } else {
        if (widen)
            GI_GATHER(KV_Q8_0, 1);
        else
            GI_GATHER(KV_Q8_0, 0);
    }
#undef GI_GATHER
    return hipGetLastError();
}

namespace {

// Page copy: grid (chunks, pairs, layers), 16 bytes per thread and step.
// Pairs with an id outside the pool are skipped and flagged.
__global__ __launch_bounds__(kThreads) void copy_pages_kernel(uint8_t *const *layer_base, int64_t page_bytes,
                                                              int64_t num_pages, const int32_t *src,
                                                              const int32_t *dst, int *status)
{
    const int pair = blockIdx.y, layer = blockIdx.z;
    const int64_t s = src[pair], d = dst[pair];
    if (s < 0 || s >= num_pages || d < 0 || d >= num_pages) {
        if (blockIdx.x == 0 && threadIdx.x == 0 && status)
            atomicOr(status, FLAG_BAD_PAGE);
        return;
    }
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    uint8_t *base = layer_base[layer];
    const u4 *sp = reinterpret_cast<const u4 *>(base + s * page_bytes);
    u4 *dp = reinterpret_cast<u4 *>(base + d * page_bytes);
    const int64_t n16 = page_bytes / 16;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n16; i += (int64_t)gridDim.x * kThreads)
        dp[i] = sp[i];
}

} // namespace

hipError_t launch_copy_pages(const PoolLayout &L, uint8_t *const *layer_base, int n, const int32_t *src,
                             const int32_t *dst, int *status, hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    const int64_t n16 = L.page_bytes / 16;
    const unsigned gx = (unsigned)std::min<int64_t>((n16 + kThreads - 1) / kThreads, 64);
    for (int i0 = 0; i0 < n; i0 += 65535) { // grid y limit
        const int cnt = std::min(n - i0, 65535);
        hipLaunchKernelGGL(copy_pages_kernel, dim3(gx, (unsigned)cnt, (unsigned)L.num_layers), dim3(kThreads),
                           0, st, layer_base, L.page_bytes, L.num_pages, src + i0, dst + i0, status);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

} // namespace gi
