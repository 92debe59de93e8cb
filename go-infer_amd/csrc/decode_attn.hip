// Paged GQA attention, vector-ALU kernel (all KV types) and the split-K
// merge.
//
// Semantics follow the reference's decode loop (pkg/engine/forward.go:
// 242-267): for q-head h, kv head h / (H/KVH); score[t] = dot(q_h, K[t]) *
// scale; softmax over t < L (pkg/math/kernels.go:48-70); out_h = sum_t
// p[t] V[t].  The softmax is evaluated online (running max / sum per head)
// so a page is read once; the result equals the two-pass form up to float
// rounding.  One workgroup owns one (query, kv head, context split) and
// serves all H/KVH query heads of the group, so each K/V element is read
// from HBM once per decode step.
#include "gi_common.h"
#include "gi_kernels.h"
#include "token_store.h"

#include <math.h>

namespace gi {

namespace {

constexpr int NT = 256;

// Eight consecutive K elements of (page, kv head, slot) starting at d0,
// widened to float32 exactly as the reference reads them.
template <int KT, int HD>
__device__ __forceinline__ void load8_k(const uint8_t *pg, const PoolLayout &L, int kvh, int s,
                                        int d0, float *o)
{
    const int64_t row = (int64_t)kvh * L.page_tokens + s;
    if (KT == KV_F32) {
        const float4 *p = reinterpret_cast<const float4 *>(pg + L.k_off + (row * HD + d0) * 4);
        float4 a = p[0], b = p[1];
        o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
        o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
    } else if (KT == KV_F16) {
        uint4 w = *reinterpret_cast<const uint4 *>(pg + L.k_off + (row * HD + d0) * 2);
        uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o[2 * i] = half_bits_to_float(u[i] & 0xFFFFu);
            o[2 * i + 1] = half_bits_to_float(u[i] >> 16);
        }
    } else if (KT == KV_Q4_0) {
        // dims d0..d0+7 of one block: the low nibbles of bytes j..j+7 when
        // d0 % 32 < 16, else the high nibbles of bytes j-16..j-9
        const int blk = d0 >> 5, j = d0 & 31;
        uint2 w = *reinterpret_cast<const uint2 *>(pg + L.k_off + (row * (HD / 32) + blk) * 16 + (j & 15));
        float sc = half_bits_to_float(reinterpret_cast<const uint16_t *>(pg + L.ks_off)[row * (HD / 32) + blk]);
        const int sh = j & 16 ? 4 : 0;
        uint32_t u[2] = {w.x, w.y};
#pragma unroll
        for (int i = 0; i < 8; i++)
            o[i] = (float)((int)((u[i >> 2] >> (8 * (i & 3) + sh)) & 15) - 8) * sc;
    } else {
        uint2 w = *reinterpret_cast<const uint2 *>(pg + L.k_off + row * HD + d0);
        float sc = half_bits_to_float(
            reinterpret_cast<const uint16_t *>(pg + L.ks_off)[row * (HD / 32) + (d0 >> 5)]);
        uint32_t u[2] = {w.x, w.y};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            int8_t q = (int8_t)((u[i >> 2] >> (8 * (i & 3))) & 0xFF);
            o[i] = (float)q * sc;
        }
    }
}

// One V element (page, kv head, dimension d, slot), widened to float32.
template <int KT, int HD>
__device__ __forceinline__ float load_v(const uint8_t *pg, const PoolLayout &L, int kvh, int d,
                                        int s)
{
    const int64_t idx = ((int64_t)kvh * HD + d) * L.page_tokens + s;
    if (KT == KV_F32)
        return reinterpret_cast<const float *>(pg + L.v_off)[idx];
    if (KT == KV_F16)
        return half_bits_to_float(reinterpret_cast<const uint16_t *>(pg + L.v_off)[idx]);
    if (KT == KV_Q4_0) {
        const int blk = d >> 5, j = d & 31;
        const int64_t bi = (int64_t)kvh * (HD / 32) + blk;
        const uint8_t b = pg[L.v_off + (bi * 16 + (j & 15)) * L.page_tokens + s];
        const float sc = half_bits_to_float(reinterpret_cast<const uint16_t *>(pg + L.vs_off)[bi * L.page_tokens + s]);
        return (float)((int)((j & 16 ? b >> 4 : b) & 15) - 8) * sc;
    }
    float sc = half_bits_to_float(reinterpret_cast<const uint16_t *>(
        pg + L.vs_off)[((int64_t)kvh * (HD / 32) + (d >> 5)) * L.page_tokens + s]);
    return (float)reinterpret_cast<const int8_t *>(pg + L.v_off)[idx] * sc;
}

// Workgroup = 256 threads over one (query, kv head, split).  Tiles of TOK
// tokens: in the score phase TPT = HD/8 threads share a token (8 elements
// each, tree-reduced with lane shuffles); the softmax phase keeps a running
// max / sum per query head in LDS; in the P*V phase thread (d, group) owns
// one output dimension for a slice of the tile's tokens, reading the
// dimension-major V tile.
template <int KT, int HD, int G>
__global__ __launch_bounds__(NT) void attn_valu(DecodeArgs a)
{
    constexpr int TPT = HD / 8;
    constexpr int TOK = NT / TPT;
    constexpr int NG = NT / HD;
    constexpr int TPG = TOK / NG;
    static_assert(G * TOK <= NT, "softmax phase needs one thread per (head, token)");
    static_assert(TOK % NG == 0, "tile tokens split evenly over P*V groups");

    const PoolLayout &L = a.L;
    const int split = blockIdx.x, kvh = blockIdx.y, qrow = blockIdx.z;
    const int b = qrow / a.n_q, qi = qrow - b * a.n_q;
    const int tid = threadIdx.x;
    const int H = a.num_heads;
    const int h0 = kvh * G;
    const int P = L.page_tokens;
    int len = a.start_pos ? a.start_pos[b] + qi + 1 : a.seq_lens[b];
    if (len > a.max_blocks * P || len < 0) {
        // More tokens than the block table maps (read what it maps), or a
        // negative length (nothing to read).
        if (tid == 0 && split == 0 && a.status)
            atomicOr(a.status, FLAG_BAD_SLOT);
        len = len < 0 ? 0 : a.max_blocks * P;
    }
    // the last split runs to the end of the sequence, so that a length
    // beyond the one the plan was sized for is still attended in full
    const int t0 = split * a.split_tokens;
    const int t1 = split == a.num_splits - 1 ? len : min(len, t0 + a.split_tokens);
    const int32_t *bt = a.block_tables + (int64_t)b * a.max_blocks;
    const int64_t qbase = (int64_t)qrow * H;

    __shared__ float s_p[G][TOK];
    __shared__ float s_alpha[G];
    __shared__ float s_m[G], s_l[G];
    __shared__ float s_acc[NG][G][HD];

    float *wsp = nullptr;
    if (a.num_splits > 1)
        wsp = a.ws + (((int64_t)qrow * L.num_kv_heads + kvh) * a.num_splits + split) * (G * (HD + 2));

    if (t0 >= t1) {
        // Empty split: partial with m = -inf, l = 0 (or zero output when the
        // whole sequence is empty).
        for (int e = tid; e < G * HD; e += NT) {
            if (wsp)
                wsp[e] = 0.0f;
            else
                a.out[(qbase + h0 + e / HD) * HD + e % HD] = 0.0f;
        }
        if (wsp && tid < G) {
            wsp[G * HD + 2 * tid] = -INFINITY;
            wsp[G * HD + 2 * tid + 1] = 0.0f;
        }
        return;
    }

    const int part = tid % TPT, tok = tid / TPT, d0 = part * 8;
    float qr[G][8];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int j = 0; j < 8; j++)
            qr[g][j] = a.q[(qbase + h0 + g) * HD + d0 + j];
    if (tid < G) {
        s_m[tid] = -INFINITY;
        s_l[tid] = 0.0f;
    }
    const int pd = tid % HD, pgp = tid / HD;
    float acc[G];
#pragma unroll
    for (int g = 0; g < G; g++)
        acc[g] = 0.0f;
    __syncthreads();

    for (int tb = t0; tb < t1; tb += TOK) {
        // ---- scores ----
        const int t = tb + tok;
        bool valid = t < t1;
        float ps[G];
#pragma unroll
        for (int g = 0; g < G; g++)
            ps[g] = 0.0f;
        if (valid) {
            int64_t page = bt[t / P];
            if (page < 0 || page >= L.num_pages) {
                if (part == 0 && a.status)
                    atomicOr(a.status, FLAG_BAD_PAGE);
                valid = false;
            } else {
                float kf[8];
                load8_k<KT, HD>(a.base + page * L.page_bytes, L, kvh, t % P, d0, kf);
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        ps[g] = fmaf(qr[g][j], kf[j], ps[g]);
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int m = TPT / 2; m >= 1; m >>= 1)
                ps[g] += __shfl_xor(ps[g], m, TPT);
#pragma unroll
        for (int g = 0; g < G; g++)
            if (part == g)
                s_p[g][tok] = valid ? ps[g] * a.scale : -INFINITY;
        __syncthreads();

        // ---- online softmax, one thread per (head, token) ----
        if (tid < G * TOK) {
            const int g = tid / TOK, tt = tid % TOK;
            const float sv = s_p[g][tt];
            float mx = sv;
#pragma unroll
            for (int m = TOK / 2; m >= 1; m >>= 1)
                mx = fmaxf(mx, __shfl_xor(mx, m, TOK));
            const float m_old = s_m[g];
            const float m_new = fmaxf(m_old, mx);
            const float p = sv == -INFINITY ? 0.0f : expf(sv - m_new);
            float sum = p;
#pragma unroll
            for (int m = TOK / 2; m >= 1; m >>= 1)
                sum += __shfl_xor(sum, m, TOK);
            s_p[g][tt] = p;
            if (tt == 0) {
                const float al = m_old == -INFINITY ? 0.0f : expf(m_old - m_new);
                s_alpha[g] = al;
                s_m[g] = m_new;
                s_l[g] = s_l[g] * al + sum;
            }
        }
        __syncthreads();

        // ---- P * V ----
#pragma unroll
        for (int g = 0; g < G; g++)
            acc[g] *= s_alpha[g];
        for (int i = 0; i < TPG; i++) {
            const int tt = pgp * TPG + i;
            const int t2 = tb + tt;
            if (t2 < t1) {
                int64_t page = bt[t2 / P];
                if (page >= 0 && page < L.num_pages) {
                    float vv = load_v<KT, HD>(a.base + page * L.page_bytes, L, kvh, pd, t2 % P);
#pragma unroll
                    for (int g = 0; g < G; g++)
                        acc[g] = fmaf(s_p[g][tt], vv, acc[g]);
                }
            }
        }
        __syncthreads();
    }

#pragma unroll
    for (int g = 0; g < G; g++)
        s_acc[pgp][g][pd] = acc[g];
    __syncthreads();
    if (tid < HD) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            float s = 0.0f;
#pragma unroll
            for (int grp = 0; grp < NG; grp++)
                s += s_acc[grp][g][pd];
            if (wsp) {
                wsp[g * HD + pd] = s;
            } else {
                const float l = s_l[g];
                a.out[(qbase + h0 + g) * HD + pd] = l > 0.0f ? s / l : 0.0f;
            }
        }
        if (wsp && tid < G) {
            wsp[G * HD + 2 * tid] = s_m[tid];
            wsp[G * HD + 2 * tid + 1] = s_l[tid];
        }
    }
}

// Merges split partials: out = sum_s acc_s e^(m_s - M) / sum_s l_s e^(m_s - M).
// W waves serve one (query row, head): wave w takes splits w, w + W, ...,
// lane i the HD / 64 dimensions from i * HD / 64, and the waves' sums meet in
// LDS.  Latency bounds it, so a wave's first kMergeAhead partials are
// requested together with the maxima of all splits: one round trip for up to
// W * kMergeAhead splits.  W is 1 (four heads per workgroup, no barrier) for
// up to kMergeAhead splits and 4 above: four waves per head on 2 splits of 52
// sequences x 32 heads cost 1 us more than one (19.9 against 18.9 us a step).
// Both also write a step's turned q (DecodeArgs.rope), which every split has
// read by then.
constexpr int kMergeAhead = 8;

template <int HD, int W>
__global__ __launch_bounds__(256) void merge_splits(float *out, const float *__restrict__ ws,
                                                    int rows, int H, int KVH, int splits,
                                                    float *q, const float2 *__restrict__ rope,
                                                    int rope_max_pos, const int32_t *__restrict__ seq_lens)
{
    constexpr int V = HD / 64, ROWS = 4 / W; // (query row, head) pairs per workgroup
    typedef float vec __attribute__((ext_vector_type(V)));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wv = wave % W;
    const int64_t row = (int64_t)blockIdx.x * ROWS + wave / W;
    if (row >= rows) // W == 1 only: a workgroup of W == 4 is one row
        return;
    const int64_t qrow = row / H;
    const int h = (int)(row - qrow * H);
    const int G = H / KVH;
    const int kvh = h / G, g = h - kvh * G;
    const int64_t stride = (int64_t)G * (HD + 2);
    const float *w0 = ws + (qrow * KVH + kvh) * splits * stride;
    const float *ml = w0 + G * HD + 2 * g; // (m, l) of split 0
    const float *wo = w0 + g * HD + V * lane;

    vec o[kMergeAhead];
    float2 t[kMergeAhead];
#pragma unroll
    for (int i = 0; i < kMergeAhead; i++) {
        const int s = wv + W * i;
        if (s < splits) {
            o[i] = *reinterpret_cast<const vec *>(wo + s * stride);
            t[i] = *reinterpret_cast<const float2 *>(ml + s * stride);
        }
    }
    if (rope && wv == 0 && lane < HD / 2) {
        const int pos = seq_lens[qrow] - 1;
        if (pos >= 0 && pos < rope_max_pos) {
            float *x = q + row * HD + lane;
            const float2 cs = rope[(int64_t)pos * (HD / 2) + lane];
            rope_pair(x[0], x[HD / 2], cs.x, cs.y, &x[0], &x[HD / 2]);
        }
    }
    float M = -INFINITY;
    for (int s = lane; s < splits; s += 64)
        M = fmaxf(M, ml[s * stride]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1)
        M = fmaxf(M, __shfl_xor(M, m));

    vec num = {};
    float den = 0.0f;
    auto add = [&](vec x, float2 y) {
        const float f = y.x == -INFINITY ? 0.0f : expf(y.x - M);
#pragma unroll
        for (int v = 0; v < V; v++)
            num[v] = fmaf(x[v], f, num[v]);
        den = fmaf(y.y, f, den);
    };
#pragma unroll
    for (int i = 0; i < kMergeAhead; i++)
        if (wv + W * i < splits)
            add(o[i], t[i]);
    for (int s = wv + W * kMergeAhead; s < splits; s += W)
        add(*reinterpret_cast<const vec *>(wo + s * stride), *reinterpret_cast<const float2 *>(ml + s * stride));

    if constexpr (W == 1) {
        vec r;
#pragma unroll
        for (int v = 0; v < V; v++)
            r[v] = den > 0.0f ? num[v] / den : 0.0f;
        *reinterpret_cast<vec *>(out + row * HD + V * lane) = r;
    } else {
        __shared__ float s_num[W][HD];
        __shared__ float s_den[W];
#pragma unroll
        for (int v = 0; v < V; v++)
            s_num[wv][V * lane + v] = num[v];
        if (lane == 0)
            s_den[wv] = den;
        __syncthreads();
        if (threadIdx.x < HD) {
            float n = 0.0f, d = 0.0f;
#pragma unroll
            for (int x = 0; x < W; x++) {
                n += s_num[x][threadIdx.x];
                d += s_den[x];
            }
            out[row * HD + threadIdx.x] = d > 0.0f ? n / d : 0.0f;
        }
    }
}

template <int KT>
hipError_t launch_valu_kt(const DecodeArgs &a, dim3 grid, hipStream_t st)
{
    const int HD = a.L.head_dim;
    const int G = a.num_heads / a.L.num_kv_heads;
#define GI_VALU(HDv, Gv)                                                                     \
    if (HD == HDv && G == Gv) {                                                              \
        hipLaunchKernelGGL((attn_valu<KT, HDv, Gv>), grid, dim3(NT), 0, st, a);              \
        return hipGetLastError();                                                            \
    }
    GI_VALU(64, 1) GI_VALU(64, 2) GI_VALU(64, 4) GI_VALU(64, 8)
    GI_VALU(128, 1) GI_VALU(128, 2) GI_VALU(128, 4) GI_VALU(128, 8) GI_VALU(128, 16)
#undef GI_VALU
    return hipErrorInvalidValue;
}

} // namespace

size_t decode_workspace_bytes(const PoolLayout &L, int batch, int num_heads, int num_splits)
{
    if (num_splits <= 1)
        return 0;
    const int G = num_heads / L.num_kv_heads;
    return (size_t)batch * L.num_kv_heads * num_splits * G * (L.head_dim + 2) * sizeof(float);
}

// f32 pages at head dimension 128 stage 32 KiB per wave, so a CU holds one
// four-wave workgroup of them; every other page type runs one eight-wave or
// two four-wave workgroups per CU (decode_waves).
static bool one_wg_per_cu(const PoolLayout &L) { return L.kv_type == KV_F32 && L.head_dim == 128; }

// Whole page pairs and a multiple of 64 tokens: the unit a split holds.
static int split_unit(const PoolLayout &L)
{
    int unit = 2 * L.page_tokens;
    while (unit % 64)
        unit += 2 * L.page_tokens;
    return unit;
}

static void set_plan(const PoolLayout &L, int max_len, int splits, int *split_tokens, int *num_splits)
{
    const int unit = split_unit(L);
    if (splits < 1)
        splits = 1;
    int per = (max_len + splits - 1) / splits;
    per = (per + unit - 1) / unit * unit;
    *split_tokens = per;
    *num_splits = (max_len + per - 1) / per;
}

// Split-K planning.  A workgroup costs about 4 us beside its tokens (query,
// table and page latencies, cross-wave merge) and a split sequence a merge
// launch, so a sequence is split only where that leaves less of the chip
// idle.  Measured on MI355X in us per layer (start: about one workgroup per
// CU, rounded up, and at least 1024 tokens per split):
//  - up to two blocks per wave (four where the pairs themselves use the
//    CUs), one split: batch 1 x 300 f16 8.6 against 10.0 in splits of 128,
//    batch 14 x 400-800 (112 pairs) 19.5 against 21.1 in two.  At head
//    dimension 64 (f32 pages apart) a third round of blocks still costs less
//    than the merge: batch 4 x 600 f16 9.2 against 9.8, q8_0 10.2 against 11.2
//    (700: 9.8 / 9.8, 11.7 / 11.2), and f16 with 64 pairs a fourth one: 800
//    9.9 against 11.0 (900 11.2 / 11.2);
//  - few (sequence, kv head) pairs: splits of 128 tokens until the CUs are
//    full.  Batch 1 f16 1000 tokens 16.1 -> 11.1, 6001 18.8 -> 13.5; f32
//    1000 29.8 -> 13.4; splits of 64 were no faster;
//  - the number of workgroups is kept at or below one (eight waves) or two
//    (four waves) per CU, whichever leaves less idle: rounded up it left a
//    few CUs with twice the work.  f16, 5000 tokens: 72 pairs 43.8 in 4
//    splits, 35.7 in 3; 96 pairs 55.9 in 3, 45.3 in 5; 160 pairs 82.5 in 2,
//    69.9 in 3.  f32 at head dimension 128 (one workgroup per CU): 136 pairs
//    161 in 2 splits, 124 in one;
//  - 1 to 2 pairs per CU: unsplit, half of the CUs hold one workgroup and
//    half two; 5 or 3 splits even that out on long sequences.  5000 tokens,
//    288 pairs: f16 150 -> 125, q4_0 76 -> 57, f32 310 -> 248, q8_0 85 -> 81;
//    384 pairs, 1500-6500 tokens: f16 157 -> 140, q4_0 87 -> 71, f32 298 ->
//    268, but q8_0 at 5000 tokens 95 -> 106, which stays unsplit, as does q8_0
//    from 9/8 pairs per CU (320 pairs, 4200 tokens 0.93 of the speed, 264 1.03);
//    equal lengths of 2600 to 4000 over 1.25 pairs per CU lose 2 to 5 % on f16
//    and f32 (q4_0 gains 0 to 9 %), from 4200 on they are even; at 1500
//    tokens splits lose everywhere, so only the caller's word for the longest
//    sequence is taken here, not the width of the tables (40 x 600 tokens under
//    tables of 4096: f16 23.0 -> 31.2, q4_0 19.0 -> 28.8);
//  - from two pairs per CU on the launch has enough rounds to even out: 480
//    and 640 pairs are fastest unsplit.
constexpr int kDecodeMinSplit = 128;

void decode_plan(const PoolLayout &L, int batch, int num_heads, int max_len, bool bound_only, int num_cus,
                 int *split_tokens, int *num_splits)
{
    (void)num_heads;
    if (max_len < 1)
        max_len = 1;
    const int64_t cus = num_cus > 0 ? num_cus : 256;
    const int64_t pairs = (int64_t)batch * L.num_kv_heads;
    const bool single = one_wg_per_cu(L);
    int64_t s = 1;
    int min_split = kDecodeMinSplit;
    int whole = single ? 256 : pairs * 4 <= cus ? 512 : 1024;
    if (L.head_dim == 64 && L.kv_type != KV_F32)
        whole = max(whole, L.kv_type == KV_F16 && pairs * 8 > cus ? 896 : 640);
    if (pairs < 1 || max_len <= whole) {
        s = 1;
    } else if (pairs <= cus / 2) {
        s = cus / pairs;
        const int64_t s2 = 2 * cus / pairs;
        if (!single && pairs * (s2 - 2 * s) * 20 > 3 * 2 * cus) // 15 % more of the chip
            s = s2;
    } else if (pairs < cus) {
        s = single || max_len <= 1024 ? 1 : 2 * cus / pairs;
        min_split = 512;
    } else if (pairs > cus && pairs < 2 * cus && !bound_only) {
        const bool near = pairs * 4 <= 5 * cus, q8 = L.kv_type == KV_Q8_0;
        if (near && max_len >= 4096 && (!q8 || pairs * 8 <= 9 * cus))
            s = 5;
        else if (pairs * 16 <= 25 * cus && !q8 && max_len >= (near || L.kv_type == KV_Q4_0 ? 2560 : 4096))
            s = 3;
    }
    set_plan(L, max_len, (int)min(s, (int64_t)(max_len + min_split - 1) / min_split), split_tokens, num_splits);
}

// The plan with the fewest partials: about one workgroup per CU, splits of
// at least 1024 tokens.  For scratch that decode_plan's partials overflow.
void decode_plan_coarse(const PoolLayout &L, int batch, int max_len, int num_cus, int *split_tokens, int *num_splits)
{
    if (max_len < 1)
        max_len = 1;
    const int64_t cus = num_cus > 0 ? num_cus : 256;
    const int64_t pairs = (int64_t)batch * L.num_kv_heads;
    const int64_t s = pairs > 0 ? (cus + pairs - 1) / pairs : 1;
    set_plan(L, max_len, (int)min(s, ((int64_t)max_len + 1023) / 1024), split_tokens, num_splits);
}

// Both plans keep to two workgroups per CU up to one (sequence, kv head) pair
// per CU; decode_plan's five splits of up to 1.25 pairs per CU are the most of
// all.
size_t decode_workspace_ahead(const PoolLayout &L, int batch, int num_heads, int num_cus)
{
    const int64_t cus = num_cus > 0 ? num_cus : 256;
    const int64_t pairs = (int64_t)batch * L.num_kv_heads;
    const int64_t slots = pairs <= cus ? 2 * cus : min(5 * pairs, 25 * cus / 4);
    const int G = num_heads / L.num_kv_heads;
    return (size_t)slots * G * (L.head_dim + 2) * sizeof(float);
}

// Whether a decode step stores its token inside the matrix-core decode
// launch (DecodeArgs.new_k) rather than in an append launch before it:
// when the grid fits the CUs at once (two workgroups each).  Measured
// same-box: batch 32 x U[512, 4096] 2.84 against 2.93 ms per step, 8 x
// 32768 (page 32) 14.64-14.69 against 14.93-14.97, batch 1 (TinyLlama,
// one graph) 5,245 against 4,315 tokens/s; but batch 256 x 8192 (four
// rounds) 42.63-42.96 against 42.09-42.42 ms, the fused launch slower by
// more than the append launch it saves.  Each 64 rows of a step cost every
// wave another look for pages that rows share (share_tokens, about 1 us for
// the first two), so steps of more than kFuseRows rows are not fused either.
constexpr int kFuseRows = 128;
bool decode_fuses_append(const PoolLayout &L, int batch, int num_splits, int num_cus)
{
    // one round: as many workgroups as the CUs hold at once (two each)
    const int64_t wgs = (int64_t)batch * L.num_kv_heads * (num_splits > 0 ? num_splits : 1);
    return batch <= kFuseRows && wgs <= (int64_t)2 * (num_cus > 0 ? num_cus : 256);
}

// The matrix-core decode turns whole heads: a pair's two elements are then
// in one lane of the query operand.  Turning q and storing the token inside
// the launch saves the one before it (4 us; 8 us at 48 sequences), and costs
// each workgroup the wait for its token's store and the q write at its end.
// With RoPE, us per layer, fused / separate:
//  - one round (two workgroups per CU): batch 1 x 6001 f16 14.9 / 19.1,
//    batch 64 x 2000 q4_0 41.0 / 45.5, q8_0 51.3 / 55.4, f16 80.1 / 80.7;
//  - q4_0, and 16-bit or 8-bit pages at head dimension 64 (three or more
//    workgroups per CU at once): up to six per CU, or three above 64 rows.
//    q4_0 48 x 1500-6500 (1152) 74.6 / 77.1, 64 x 1500-3000 (512) 53.8 /
//    56.6, 90 x 1500-3000 (720) 67.4 / 69.0, but 128 x 1500-3000 (1024)
//    98.3 / 96.5; head dimension 64 q4_0 128 x 300-600 (512) 18.6 / 19.0,
//    300 x 1000-2000 (1200) 66.2 / 59.1;
//  - f16 and f32 at head dimension 128 stream at the HBM rate from the first
//    block, so long splits hide the separate launch: f16 64 x 5000 182.9 /
//    180.6, 64 x 12000 422 / 414, f32 64 x 2000 159.8 / 154.2, 64 x 700
//    69.9 / 71.6.
bool decode_fuses_rope(const PoolLayout &L, int batch, int num_heads, int requested, int rope_half,
                       int split_tokens, int num_splits, int num_cus)
{
    if (batch > kFuseRows || rope_half != L.head_dim / 2 || decode_kernel_kind(L, num_heads, requested) != 1)
        return false;
    const int64_t cus = num_cus > 0 ? num_cus : 256;
    const int64_t wgs = (int64_t)batch * L.num_kv_heads * (num_splits > 0 ? num_splits : 1);
    if (wgs <= cus)
        return true;
    if (L.kv_type == KV_Q4_0 || (L.head_dim == 64 && L.kv_type != KV_F32))
        return wgs <= (batch <= 64 ? 6 : 3) * cus;
    if (L.head_dim == 128 && (L.kv_type == KV_F32 || L.kv_type == KV_F16) &&
        split_tokens >= (L.kv_type == KV_F32 ? 2000 : 4096))
        return false;
    return wgs <= 2 * cus;
}

int decode_waves(const PoolLayout &L, int batch, int num_splits, int num_cus)
{
    const int64_t wgs = (int64_t)batch * L.num_kv_heads * (num_splits > 0 ? num_splits : 1);
    const bool one_round = wgs <= (num_cus > 0 ? num_cus : 256);
    // f32 pages stage HD * 256 bytes per wave in LDS: eight waves at head
    // dimension 64 (128 KiB), four at 128
    if (L.kv_type == KV_F32)
        return one_round && L.head_dim == 64 ? 8 : 4;
    return one_round ? 8 : 4;
}

int decode_kernel_kind(const PoolLayout &L, int num_heads, int requested)
{
    const bool mfma = mfma_decode_supported(L, num_heads);
    if (requested == 0 || !mfma)
        return 0;
    return 1;
}

hipError_t launch_decode(const DecodeArgs &a, hipStream_t st)
{
    const PoolLayout &L = a.L;
    if (a.num_heads % L.num_kv_heads)
        return hipErrorInvalidValue;
    const int n_q = a.n_q > 0 ? a.n_q : 1;
    hipError_t e;
    if (n_q == 1 && !a.start_pos && decode_kernel_kind(L, a.num_heads, a.kernel) == 1) {
        e = launch_decode_mfma(a, st); // stores a decode step's token itself
    } else {
        if (a.new_k) { // the vector path appends in a launch of its own
            e = launch_append_at_len(L, a.append_base, a.batch, a.block_tables, a.max_blocks, a.seq_lens,
                                     a.new_k, a.new_v, a.status, st);
            if (e != hipSuccess)
                return e;
        }
        dim3 grid(a.num_splits, L.num_kv_heads, a.batch * n_q);
        switch (L.kv_type) {
        case KV_F32: e = launch_valu_kt<KV_F32>(a, grid, st); break;
        case KV_F16: e = launch_valu_kt<KV_F16>(a, grid, st); break;
        case KV_Q4_0: e = launch_valu_kt<KV_Q4_0>(a, grid, st); break;
        default: e = launch_valu_kt<KV_Q8_0>(a, grid, st); break;
        }
    }
    if (e != hipSuccess || a.num_splits <= 1)
        return e;
    const int rows = a.batch * n_q * a.num_heads;
#define GI_MERGE(HDv, Wv)                                                                              \
    hipLaunchKernelGGL((merge_splits<HDv, Wv>), dim3((unsigned)((rows + 4 / Wv - 1) / (4 / Wv))),       \
                       dim3(256), 0, st, a.out, a.ws, rows, a.num_heads, L.num_kv_heads, a.num_splits, \
                       a.q_rot, a.rope, a.rope_max_pos, a.seq_lens)
    if (a.num_splits <= kMergeAhead) {
        if (L.head_dim == 128)
            GI_MERGE(128, 1);
        else
            GI_MERGE(64, 1);
    } else {
        if (L.head_dim == 128)
            GI_MERGE(128, 4);
        else
            GI_MERGE(64, 4);
    }
#undef GI_MERGE
    return hipGetLastError();
}

hipError_t launch_prefill(const PrefillArgs &p, hipStream_t st)
{
    if (p.chunk_len <= 0 || p.batch <= 0)
        return hipSuccess;
    if (p.kernel != 0 && mfma_prefill_supported(p.L, p.num_heads))
        return launch_prefill_mfma(p, st);
    DecodeArgs a{};
    a.L = p.L;
    a.base = p.base;
    a.q = p.q;
    a.out = p.out;
    a.block_tables = p.block_tables;
    a.max_blocks = p.max_blocks;
    a.seq_lens = nullptr;
    a.batch = p.batch;
    a.n_q = p.chunk_len;
    a.start_pos = p.start_pos;
    a.num_heads = p.num_heads;
    a.scale = p.scale;
    a.split_tokens = 1 << 30;
    a.num_splits = 1;
    a.ws = nullptr;
    a.status = p.status;
    a.kernel = 0;
    if (p.chunk_len <= 0 || p.batch <= 0)
        return hipSuccess;
    return launch_decode(a, st);
}

} // namespace gi
