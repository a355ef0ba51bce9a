// attention_f32.hip -- fused fp32 attention for head_dim 128 (no mask): the op
// behind FlashAttentionOp::operator() on F32 q/k/v
// (src/nn/attention/FlashAttentionOp.cpp:84-94), O = softmax(scale Q K^T) V per
// (batch, head), with fp32 accuracy on the bf16 matrix cores.
//
// Every operand of both products is three exact bf16 parts (x = x0 + x1 + x2)
// and a product the six MFMAs x0 y0, x0 y1, x1 y0, x1 y1, x0 y2, x2 y0, as in
// the fp32 GEMM (gemm_f32.hip).  Through GEMMs the scores crossed memory four
// times and each head took launches of its own.  Python call included, 24 heads of
// 1536 x 1536: 1112 us with fp32 MFMAs, 709 with split ones, 230 here (126
// TFLOP/s, six bf16 products each); 8 heads of 1000 x 1000 318 -> 55 us, 24 of 320 x 320
// 347 -> 40 us.  Relative error against 64 bits at those three: 3.04e-7 -> 2.19e-7, 2.97e-7
// -> 1.88e-7, 2.81e-7 -> 1.71e-7.  Bound by the MFMAs and, beside them, softmax and
// the splitting of P.
//
// split_kv_kernel first writes K and V as rows of three 256-byte planes
// ([head][key][plane][128] bf16) so that the key tiles stream into LDS by
// direct DMA and each element is split once, not once per query block.
// A workgroup of four waves takes 128 queries, each wave 32 with Q's parts in
// registers (96); two workgroups per CU.  As in the bf16 kernel the transposed
// products S^T = K Q^T and O^T = V^T P^T keep a query in one lane column, P^T
// goes from the score accumulators into the MFMA's operand, and V is read
// transposed (ds_read_tr16_b64).  Per 32-key tile: the scores' x0 y0 in one
// accumulator, the small products in another; P split; each 32-d
// block of V^T P^T into a fresh accumulator, small products first, then added to
// O.  So O and the scores are rounded to fp32 once per tile or 16-d step, and the
// row sum carries its rounding error along.
// Blocks for less than half of two per CU share their keys out over several
// workgroups, whose partial O, maxima and sums attn_combine_kernel adds (64 blocks of
// the 8 heads of 1000: 182 us in one range, 55 in eight).
// One K and one V buffer (24 KB each): K of the next tile loads while softmax and
// P V run, V of the next tile while its scores are computed.
//
// A (batch, head) with operands outside the range in which the parts are normal
// numbers (|q|, |k| >= 2^50, |v| >= 2^30 or 0 < |v| < 2^-80, not finite) is taken on
// the fp32 matrix cores instead (attn_native): 24 heads of 1536 x 1536 with one such element a head
// 840 us, 8 of 1000 326, 24 of 320 176 (a query at a time by hand 18.7 ms, 6.1 and 2.4; through GEMMs
// 1112, 318 and 347 us).
#include <math.h>

#include <initializer_list>

#include "capi_util.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace dit {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t* lds_short4_p;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int D = 128, QB = 128, KB = 32;     // head dim, queries per workgroup, keys per tile
constexpr int ROWB = 3 * D * 2, TILEB = KB * ROWB;
constexpr int SPLIT_ROWS = 64;                // rows per workgroup of split_kv_kernel
constexpr float kQkMax = 1125899906842624.0f;      // 2^50
constexpr float kVMax = 1073741824.0f;             // 2^30
// A product of parts is lost below 2^-126, and a row's largest weight is at
// least 1 before the division by l: n keys lose under 6 n 2^-46 of a result of this size.
constexpr float kVMin = 8.2718061255302767e-25f;   // 2^-80

constexpr float kScaleMax = 1208925819614629174706176.0f;  // 2^80

struct F32Attn {
    const float* q;
    const float* k;
    const float* v;
    float* o;
    int64_t qs[3], ks[3], vs[3], os[3];  // batch, token, head strides (elements)
    int32_t bh, bh0, heads, seq_q, seq_kv, q_blocks, kv_blocks;  // bh (batch, head) pairs from bh0 on
    float scale, c_hi, c_lo;             // scale * log2(e) = c_hi + c_lo
    uint8_t* kp;                         // planes [bh][seq_kv][3][128] bf16
    uint8_t* vp;
    uint32_t* flags;                     // [bh][2 kv_blocks]: 1 = operands out of range
    int32_t splits;                      // key ranges per query block; > 1: partial results
    float* part;                         // [split][bh][seq_q][128]: O before its division by l
    float2* ml;                          // [split][bh][seq_q]: (m, l)
};

// 8 fp32 as three planes of 8 bf16.
__device__ __forceinline__ void split8(const float (&x)[8], uint4 (&p)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t h = pack_bf16x2(x[2 * e], x[2 * e + 1]);
        const float r0 = x[2 * e] - bf16_lo(h), r1 = x[2 * e + 1] - bf16_hi(h);
        const uint32_t m = pack_bf16x2(r0, r1);
        w[0][e] = h;
        w[1][e] = m;
        w[2][e] = pack_bf16x2(r0 - bf16_lo(m), r1 - bf16_hi(m));
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) p[i] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
}

__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}

// Block (i, bh, z): rows [64 i, + 64) of K (z = 0) or V (z = 1) of one head, and whether
// any of them is out of range.
__global__ __launch_bounds__(256) void split_kv_kernel(const F32Attn a) {
    const int bh = blockIdx.y, h = (a.bh0 + bh) % a.heads, b = (a.bh0 + bh) / a.heads;
    const bool is_v = blockIdx.z != 0;
    const float* src = is_v ? a.v + b * a.vs[0] + h * a.vs[2] : a.k + b * a.ks[0] + h * a.ks[2];
    const int64_t ts = is_v ? a.vs[1] : a.ks[1];
    uint8_t* dst = (is_v ? a.vp : a.kp) + (int64_t)bh * a.seq_kv * ROWB;
    bool odd = false;
#pragma unroll
    for (int u = 0; u < SPLIT_ROWS * (D / 8) / 256; ++u) {
        const int i = threadIdx.x + 256 * u, row = blockIdx.x * SPLIT_ROWS + (i >> 4), c = i & 15;
        if (row >= a.seq_kv) continue;
        float x[8];
        load8(src + row * ts + 8 * c, x);
        const float top = is_v ? kVMax : kQkMax;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            odd |= !(fabsf(x[e]) < top) || (is_v && x[e] != 0.f && fabsf(x[e]) < kVMin);
        uint4 p[3];
        split8(x, p);
#pragma unroll
        for (int j = 0; j < 3; ++j)
            *reinterpret_cast<uint4*>(dst + (int64_t)row * ROWB + j * 256 + 16 * c) = p[j];
    }
    const int any = __syncthreads_or(odd);
    if (threadIdx.x == 0) a.flags[((int64_t)bh * 2 + blockIdx.z) * a.kv_blocks + blockIdx.x] = any ? 1u : 0u;
}

// Queries [q0, q0 + QB) of one head on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32), for operands of any magnitude: the arithmetic of the
// GEMM path (gemm_f32.hip) tile by tile.  The keys are walked twice, for
// each query's largest score m and l = sum expf(scale s - m), then for O = sum
// (expf(scale s - m) / l) v, so no product exceeds the largest |v|.  A row whose scores are
// -inf so far keeps the weights 0; rows with a NaN or +inf score, or none above -inf, are NaN.
// K and V tiles of 32 keys pass through LDS, the next one on its way in registers.  As in the
// kernel below lane l holds query l % 32 and, of a 32 x 32 block, key (or d) 8 (i / 4) +
// 4 (l / 32) + i % 4; MFMA step 4 c + e of the scores takes d = 8 c + 4 (l / 32) + e, step i
// of P V the keys of score element i, so P goes from one to the other in place.
__device__ void attn_native(const F32Attn& a, int b, int h, int q0, float* lds) {
    constexpr int LD = D + 4;  // padded row: 16 rows' 16-byte reads hit distinct banks
    float* const Kt = lds;
    float* const Vt = lds + KB * LD;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5, q = q0 + 32 * wave + r;
    const float* kb = a.k + b * a.ks[0] + h * a.ks[2];
    const float* vb = a.v + b * a.vs[0] + h * a.vs[2];
    // Q is read again for every tile: 64 registers more would spill.
    const float* qp = a.q + b * a.qs[0] + (int64_t)min(q, a.seq_q - 1) * a.qs[1] + h * a.qs[2] + 4 * g;

    // Thread t: float4 t % 32 of rows t / 32 + 8 u; zeros past seq_kv (a masked weight
    // must not meet a NaN).
    const int srow = tid >> 5, scol = 4 * (tid & 31);
    auto fetch = [&](const float* src, int64_t ts, int k0, float4 (&x)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int key = k0 + srow + 8 * u;
            x[u] = key < a.seq_kv ? *reinterpret_cast<const float4*>(src + key * ts + scol) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto stash = [&](float* dst, const float4 (&x)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<float4*>(dst + (srow + 8 * u) * LD + scol) = x[u];
    };
    // scale s of the K tile from key k0, -inf past seq_kv; two running sums.
    auto scores = [&](int k0, float (&s)[16]) {
        f32x16_t acc[2];
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[0][e] = acc[1][e] = 0.f;
#pragma unroll 4
        for (int c = 0; c < 16; ++c) {
            const float4 kv = *reinterpret_cast<const float4*>(Kt + r * LD + 8 * c + 4 * g);
            const float4 qv = *reinterpret_cast<const float4*>(qp + 8 * c);
            const float kx[4] = {kv.x, kv.y, kv.z, kv.w}, qx[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[e], qx[e], acc[e & 1], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = a.scale * (acc[0][i] + acc[1][i]);
            if (k0 + 8 * (i >> 2) + 4 * g + (i & 3) >= a.seq_kv) s[i] = -INFINITY;
        }
    };

    float m = -INFINITY, l = 0.f, l_err = 0.f;
    float4 nk[4], nv[4];
    fetch(kb, a.ks[1], 0, nk);
    for (int k0 = 0; k0 < a.seq_kv; k0 += KB) {
        __syncthreads();  // every wave has read the tile before
        stash(Kt, nk);
        __syncthreads();
        if (k0 + KB < a.seq_kv) fetch(kb, a.ks[1], k0 + KB, nk);
        float s[16], mt = m;
        scores(k0, s);
#pragma unroll
        for (int i = 0; i < 16; ++i) mt = fmaxf(mt, s[i]);
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float ref = mt == -INFINITY ? 0.f : mt, alpha = expf(m - ref);
        float ts = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) ts += expf(s[i] - ref);
        m = mt;
        l *= alpha;
        l_err *= alpha;
        const float n = l + ts, bb = n - l;  // l + l_err += ts
        l_err += (l - (n - bb)) + (ts - bb);
        l = n;
    }
    l += l_err;
    const float inv = 1.0f / (l + __shfl_xor(l, 32)), ref = m == -INFINITY ? 0.f : m;

    f32x16_t o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    fetch(kb, a.ks[1], 0, nk);
    for (int k0 = 0; k0 < a.seq_kv; k0 += KB) {
        __syncthreads();
        stash(Kt, nk);
        __syncthreads();
        fetch(vb, a.vs[1], k0, nv);
        float p[16];
        scores(k0, p);
        stash(Vt, nv);
        __syncthreads();
        if (k0 + KB < a.seq_kv) fetch(kb, a.ks[1], k0 + KB, nk);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            p[i] = expf(p[i] - ref) * inv;
            if (k0 + 8 * (i >> 2) + 4 * g + (i & 3) >= a.seq_kv) p[i] = 0.f;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x16_t acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(Vt[(8 * (i >> 2) + 4 * g + (i & 3)) * LD + 32 * t + r], p[i], acc,
                                                           0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e) o[t][e] += acc[e];
        }
    }
    if (q >= a.seq_q) return;
    float* op = a.o + b * a.os[0] + (int64_t)q * a.os[1] + h * a.os[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
            *reinterpret_cast<float4*>(op + 32 * t + 8 * i4 + 4 * g) =
                make_float4(o[t][4 * i4], o[t][4 * i4 + 1], o[t][4 * i4 + 2], o[t][4 * i4 + 3]);
}

__device__ __forceinline__ uint2 read_tr16(const uint8_t* p) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_p)(p)));
}

// 16-byte chunk c of a plane of tile row r is stored at c ^ fswz(r): 16
// consecutive rows read at one chunk (K), and 4 consecutive rows at two adjacent
// ones (V, transposed), hit distinct banks.
__device__ __forceinline__ int fswz(int r) { return ((r & 7) << 1) | ((r >> 3) & 1); }

// exp(scale d)
__device__ __forceinline__ float score_weight(float d, const F32Attn& a) {
    return __builtin_amdgcn_exp2f(__builtin_fmaf(d, a.c_hi, d * a.c_lo));
}

// x, hidden from the optimiser: what is derived from it is computed where it is
// used and not kept in registers over the loop.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

__global__ __launch_bounds__(256, 2) void flash_attn_f32_kernel(const F32Attn a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * TILEB];  // K tile, V tile
    uint32_t bid = blockIdx.x;
    const uint32_t nb = gridDim.x;
    if ((nb & 7u) == 0) bid = (bid & 7u) * (nb >> 3) + (bid >> 3);  // a run of heads per XCD
    const int qblk = (int)(bid % (uint32_t)a.q_blocks);
    const int split = (int)(bid / (uint32_t)a.q_blocks) % a.splits, bh = (int)(bid / (uint32_t)(a.q_blocks * a.splits));
    const int h = (a.bh0 + bh) % a.heads, b = (a.bh0 + bh) / a.heads;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int q = qblk * QB + wave * 32 + r;

    // Q's parts (rows past seq_q as zeros), and whether this block's operands are
    // all in range.
    bf16x8_t qf[3][8];
    bool odd = false;
    const float* qp = a.q + b * a.qs[0] + (int64_t)min(q, a.seq_q - 1) * a.qs[1] + h * a.qs[2] + 8 * g;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        float x[8];
        load8(qp + 16 * c, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) odd |= !(fabsf(x[e]) < kQkMax);
        uint4 p[3];
        split8(x, p);
#pragma unroll
        for (int j = 0; j < 3; ++j) qf[j][c] = __builtin_bit_cast(bf16x8_t, p[j]);
    }
    for (int i = tid; i < 2 * a.kv_blocks; i += 256) odd |= a.flags[(int64_t)bh * 2 * a.kv_blocks + i] != 0;
    // Marked unlikely: with attn_native in line the compiler put a wait for every DMA in
    // flight at the top of the key loop (24 heads of 1536 244.5 -> 247.3 us, 2 of 328 26.6 ->
    // 27.2).  Behind it, it keeps the loop as it was and spills three of attn_native's registers.
    if (__builtin_expect(__syncthreads_or(odd), 0)) {
        // attn_combine_kernel leaves rows with l = NaN as they are
        if (a.splits > 1 && q < a.seq_q && g == 0)
            a.ml[((int64_t)split * a.bh + bh) * a.seq_q + q] = make_float2(0.f, NAN);
        static_assert(2 * KB * (D + 4) * (int)sizeof(float) <= 2 * TILEB, "attn_native's tiles");
        if (split == 0) attn_native(a, b, h, qblk * QB, reinterpret_cast<float*>(smem));
        return;
    }

    // DMA: a tile is 24 instructions of 1 KB, six a wave; lane i writes LDS byte
    // 1024 n + 16 i of the tile, loaded from the chunk that belongs there.  Rows
    // past seq_kv load the last one (their scores are masked).
    const uint8_t* kpl = a.kp + (int64_t)bh * a.seq_kv * ROWB;
    const uint8_t* vpl = a.vp + (int64_t)bh * a.seq_kv * ROWB;
    uint32_t src[6];
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const int at = (wave * 6 + n) * 1024 + lane * 16, row = at / ROWB, in = at % ROWB;
        src[n] = (uint32_t)(row * ROWB + (in & ~255) + ((((in & 255) >> 4) ^ fswz(row)) << 4));
    }
    auto issue = [&](const uint8_t* planes, int t, uint8_t* buf) {
        const int left = a.seq_kv - t * KB;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(planes + (int64_t)t * TILEB), 0, TILEB, 0x00020000);
        if (left >= KB) {
#pragma unroll
            for (int n = 0; n < 6; ++n)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(buf + (wave * 6 + n) * 1024), 16, src[n], 0, 0, 0);
        } else {
#pragma unroll
            for (int n = 0; n < 6; ++n) {
                const uint32_t at = opaque(src[n]), past = max((int)(at / ROWB) - (left - 1), 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(buf + (wave * 6 + n) * 1024), 16,
                                                         at - past * ROWB, 0, 0, 0);
            }
        }
    };
    uint8_t* const Kt = smem;
    uint8_t* const Vt = smem + TILEB;

    const int kbase = r * ROWB + ((g ^ fswz(r)) << 4);  // chunk 2 c + g: ^ 32 c
    // Transposed V reads: lane s of 16-lane group gi reads row 16 j + 4 (gi / 2) + s / 4 (+ 8),
    // d = 32 tt + 16 (gi % 2) + 4 (s % 4).
    const int s16 = lane & 15, gi = lane >> 4, vrow = 4 * (gi >> 1) + (s16 >> 2);
    const int vcol = 16 * (gi & 1) + 4 * (s16 & 3);
    const int vbase = vrow * ROWB + (((vcol >> 3) ^ fswz(vrow)) << 4) + 8 * ((vcol >> 2) & 1);

    f32x16_t o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f, l_err = 0.f;

    auto weight = [&](float d) { return score_weight(d, a); };
    const int tiles = (a.seq_kv + KB - 1) / KB;
    const int t0 = (int)((int64_t)tiles * split / a.splits), ntiles = (int)((int64_t)tiles * (split + 1) / a.splits);
    issue(kpl, t0, Kt);
    issue(vpl, t0, Vt);
    __builtin_amdgcn_s_waitcnt(6 | 0x0F70);  // vmcnt(6): K landed
    __builtin_amdgcn_s_barrier();
    for (int t = t0; t < ntiles; ++t) {
        const uint32_t kofs = opaque(kbase);
        f32x16_t s, low;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = low[e] = 0.f;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            bf16x8_t kf[3];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                kf[j] = *reinterpret_cast<const bf16x8_t*>(Kt + (kofs ^ (32 * c)) + 256 * j);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[0][c], s, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[1][c], low, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[0][c], low, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[1][c], low, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[2], qf[0][c], low, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[2][c], low, 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        // V of this tile has landed and every wave has read K: the K buffer takes
        // the next tile.
        __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        if (t + 1 < ntiles) issue(kpl, t + 1, Kt);

        // Element i is key 32 t + 8 (i / 4) + 4 g + i % 4.
        float mx = -INFINITY;
        const int left = a.seq_kv - t * KB;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] += low[i];
            if (8 * (i >> 2) + 4 * g + (i & 3) >= left) s[i] = -INFINITY;
            mx = fmaxf(mx, s[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // As in the bf16 kernel the reference (here a raw score) moves only when a
        // score exceeds it by more than 2^8; O and l share it.  exp2 takes the
        // difference of two scores, exact where it matters, times scale * log2(e).
        const float m_cand = fmaxf(m_run, mx);
        const bool move = !((m_cand - m_run) * a.c_hi <= 8.0f);
        if (__builtin_amdgcn_ballot_w64(move)) {
            const float m_new = move ? m_cand : m_run;
            const float alpha = m_run == -INFINITY ? 0.f : weight(m_run - m_new);
            l_run *= alpha;
            l_err *= alpha;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[tt][e] *= alpha;
            m_run = m_new;
        }
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        bf16x8_t pf[3][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[e] = weight(s[8 * j + e] - m_run);
                if (8 * ((8 * j + e) >> 2) + 4 * g + (e & 3) >= left) x[e] = 0.f;
                sum[e & 3] += x[e];
            }
            uint4 p[3];
            split8(x, p);
#pragma unroll
            for (int i = 0; i < 3; ++i) pf[i][j] = __builtin_bit_cast(bf16x8_t, p[i]);
        }
        {   // l_run += the tile's sum, its rounding error kept in l_err
            const float ts = (sum[0] + sum[1]) + (sum[2] + sum[3]);
            const float n = l_run + ts, bb = n - l_run;
            l_err += (l_run - (n - bb)) + (ts - bb);
            l_run = n;
        }
        // O^T[d][q] += V^T[d][key] P^T[key][q], by 32-d blocks.
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            const uint32_t vofs = opaque(vbase) ^ (tt << 6);
            f32x16_t acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = 0.f;
            // small products first, one plane of V at a time
            auto mac = [&](int vi, std::initializer_list<int> planes) {
                bf16x8_t vf[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint2 lo = read_tr16(Vt + vofs + 16 * j * ROWB + 256 * vi);
                    const uint2 hi = read_tr16(Vt + (vofs ^ 16) + (16 * j + 8) * ROWB + 256 * vi);
                    vf[j] = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
                }
                for (int pi : planes)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[j], pf[pi][j], acc, 0, 0, 0);
            };
            mac(2, {0});
            mac(1, {1, 0});
            mac(0, {2, 1, 0});
#pragma unroll
            for (int e = 0; e < 16; ++e) o[tt][e] += acc[e];
        }
        __builtin_amdgcn_s_setprio(0);
        // K of the next tile has landed and every wave has read V.
        __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        if (t + 1 < ntiles) issue(vpl, t + 1, Vt);
    }
    l_run += l_err;
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const float inv = a.splits > 1 ? 1.0f : 1.0f / l_tot;
    if (q < a.seq_q) {
        const int64_t row = ((int64_t)split * a.bh + bh) * a.seq_q + q;
        float* op = a.splits > 1 ? a.part + row * D : a.o + b * a.os[0] + (int64_t)q * a.os[1] + h * a.os[2];
        if (a.splits > 1 && g == 0) a.ml[row] = make_float2(m_run, l_tot);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
                *reinterpret_cast<float4*>(op + 32 * tt + 8 * i4 + 4 * g) =
                    make_float4(o[tt][4 * i4] * inv, o[tt][4 * i4 + 1] * inv, o[tt][4 * i4 + 2] * inv,
                                o[tt][4 * i4 + 3] * inv);
    }
}

// The key ranges' partial results of one row: O = sum 2^(m_s - m) O_s / sum 2^(m_s - m) l_s.
// 32 threads a row, eight rows a workgroup.
__global__ __launch_bounds__(256) void attn_combine_kernel(const F32Attn a) {
    const int64_t row = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5), rows = (int64_t)a.bh * a.seq_q;
    if (row >= rows) return;
    float m = -INFINITY;
    bool plain = false;
    for (int s = 0; s < a.splits; ++s) {
        const float2 v = a.ml[s * rows + row];
        m = fmaxf(m, v.x);
        plain |= v.y != v.y;
    }
    if (plain) return;
    const int d = (threadIdx.x & 31) * 4;
    float l = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < a.splits; ++s) {
        const float2 v = a.ml[s * rows + row];
        const float w = score_weight(v.x - m, a);
        const float4 p = *reinterpret_cast<const float4*>(a.part + (s * rows + row) * D + d);
        l += w * v.y;
        o.x += w * p.x;
        o.y += w * p.y;
        o.z += w * p.z;
        o.w += w * p.w;
    }
    const int64_t bh = row / a.seq_q, q = row - bh * a.seq_q, b = (a.bh0 + bh) / a.heads, h = a.bh0 + bh - b * a.heads;
    const float inv = 1.0f / l;
    *reinterpret_cast<float4*>(a.o + b * a.os[0] + q * a.os[1] + h * a.os[2] + d) =
        make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
}

// Key ranges per query block: as many as keep two workgroups per CU, each of at
// least two tiles.
int attn_f32_splits(int64_t bh, int64_t seq_q, int64_t seq_kv) {
    const int64_t wgs = bh * ((seq_q + QB - 1) / QB), tiles = (seq_kv + KB - 1) / KB;
    int64_t s = wgs > 0 ? 2 * cu_count() / wgs : 1;
    if (s > tiles / 2) s = tiles / 2;
    if (s > 8) s = 8;
    return s < 2 ? 1 : (int)s;
}

}  // namespace

// Largest number of (batch, head) pairs, in launches of about equal size, whose
// workspace is at most `limit`; 0: not even one's.
int64_t attn_f32_fused_heads(int64_t bh, int64_t seq_q, int64_t seq_kv, size_t limit) {
    int64_t n = (int64_t)(limit / (size_t)(2 * seq_kv * ROWB));
    if (n > bh) n = bh;
    if (n > 65535) n = 65535;  // split_kv_kernel's grid
    while (n > 0 && attn_f32_fused_bytes(n, seq_q, seq_kv) > limit) --n;
    if (n == 0) return 0;
    const int64_t launches = (bh + n - 1) / n, even = (bh + launches - 1) / launches;
    return attn_f32_fused_bytes(even, seq_q, seq_kv) <= limit ? even : n;  // fewer heads may take more key ranges
}

size_t attn_f32_fused_bytes(int64_t bh, int64_t seq_q, int64_t seq_kv) {
    const int64_t blocks = (seq_kv + SPLIT_ROWS - 1) / SPLIT_ROWS;
    const int64_t splits = attn_f32_splits(bh, seq_q, seq_kv);
    return (size_t)(bh * (2 * seq_kv * ROWB + 8 * blocks)) + (splits > 1 ? (size_t)(splits * bh * seq_q * (D * 4 + 8)) : 0);
}

bool attn_f32_fused_takes(const float* q, const float* k, const float* v, const float* o, int64_t batch, int64_t heads,
                          int64_t seq_q, int64_t seq_kv, int64_t head_dim, const int64_t* qs, const int64_t* ks,
                          const int64_t* vs, const int64_t* os, float scale) {
    // Parts of a score lost below 2^-126 stay under 2^-38 after the scale.
    if (head_dim != D || !(scale >= 0.f && scale <= kScaleMax) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o))
        return false;
    for (int i = 0; i < 3; ++i)
        if (qs[i] % 4 || ks[i] % 4 || vs[i] % 4 || os[i] % 4) return false;
    return batch * heads < (1ll << 31) && ((seq_q + QB - 1) / QB) * batch * heads < (1ll << 31) && seq_kv < (1ll << 30);
}

int attn_f32_fused(const float* q, const float* k, const float* v, float* o, int64_t batch, int64_t heads,
                   int64_t seq_q, int64_t seq_kv, const int64_t* qs, const int64_t* ks, const int64_t* vs,
                   const int64_t* os, float scale, int64_t heads_per_launch, void* workspace, hipStream_t st) {
    F32Attn a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.o = o;
    for (int i = 0; i < 3; ++i) {
        a.qs[i] = qs[i];
        a.ks[i] = ks[i];
        a.vs[i] = vs[i];
        a.os[i] = os[i];
    }
    a.heads = (int32_t)heads;
    a.seq_q = (int32_t)seq_q;
    a.seq_kv = (int32_t)seq_kv;
    a.q_blocks = (int32_t)((seq_q + QB - 1) / QB);
    a.kv_blocks = (int32_t)((seq_kv + SPLIT_ROWS - 1) / SPLIT_ROWS);
    const double c = (double)scale * 1.4426950408889634;
    a.scale = scale;
    a.c_hi = (float)c;
    a.c_lo = (float)(c - (double)a.c_hi);
    a.kp = (uint8_t*)workspace;
    for (int64_t bh0 = 0; bh0 < batch * heads; bh0 += heads_per_launch) {
        const int64_t bh = batch * heads - bh0 < heads_per_launch ? batch * heads - bh0 : heads_per_launch;
        a.bh0 = (int32_t)bh0;
        a.bh = (int32_t)bh;
        a.vp = a.kp + (size_t)bh * (size_t)seq_kv * ROWB;
        a.splits = attn_f32_splits(heads_per_launch, seq_q, seq_kv);  // what the workspace is sized for
        const size_t rows = a.splits > 1 ? (size_t)a.splits * (size_t)bh * (size_t)seq_q : 0;
        a.part = (float*)(a.vp + (size_t)bh * (size_t)seq_kv * ROWB);
        a.ml = (float2*)(a.part + rows * D);
        a.flags = (uint32_t*)(a.ml + rows);
        hipLaunchKernelGGL(split_kv_kernel, dim3((unsigned)a.kv_blocks, (unsigned)bh, 2), dim3(256), 0, st, a);
        int rc = check_launch("dt_flash_attn_f32(split)");
        if (rc) return rc;
        hipLaunchKernelGGL(flash_attn_f32_kernel, dim3((unsigned)(a.q_blocks * bh * a.splits)), dim3(256), 0, st, a);
        rc = check_launch("dt_flash_attn_f32");
        if (rc) return rc;
        if (a.splits == 1) continue;
        hipLaunchKernelGGL(attn_combine_kernel, dim3((unsigned)((bh * seq_q + 7) / 8)), dim3(256), 0, st, a);
        rc = check_launch("dt_flash_attn_f32(combine)");
        if (rc) return rc;
    }
    return DT_OK;
}

}  // namespace dit
