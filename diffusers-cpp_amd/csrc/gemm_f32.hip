// gemm_f32.hip -- fp32 Linear and attention for graphs whose weights and
// activations are both F32, the reference's own precision (Linear::forward ->
// Runtime::mul_mat with F32 weights, src/nn/Linear.cpp:17-36; ggml computes
// such products in fp32).
//
// GEMM: C[m][n] = sum_k A[m][k] * B[n][k] (+ bias[n]) (+ D[m][n]), A the
// activation [M, K] and B the weight [N, K], both K-contiguous.  The fp32
// matrix cores (157 TFLOP/s) bound this product, the bf16 ones (2.5 PFLOP/s)
// do not: each operand is split exactly into three bf16 parts, x = x0 + x1 +
// x2 (8 + 8 + 8 bits, each the rounded remainder of the last), and the product
// taken as the six bf16 MFMAs x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0 with
// fp32 accumulation.  The three left out are 2^-27.4 of |x w| in the root mean square
// (N(0, 1) operands) and at most 2^-24.05, about what fp32 rounds one product by, so a
// product that stands alone may be off by 1.85 half units instead of 1 (K = 1 and 2
// therefore run on the fp32 matrix cores); from three terms on the total, whose
// sums are rounded less often, is closer than the fp32 MFMAs' in both measures.  x0 w0 is summed by itself, in runs of 128 k
// that are then added to the tile's total, and the five small ones in an
// accumulator of their own, whose rounding is 2^-8 of the other's; so the sum
// is rounded about 8 + K/128 times where the fp32 MFMA's was 64 + K/128.
// Relative error against 64 bits (2-norm, N(0, 1) x N(0, 0.02)), fp32 MFMAs ->
// here: K = 64 1.04e-7 -> 5.0e-8, 256 1.50e-7 -> 7.1e-8, 3072 1.74e-7 ->
// 1.14e-7, 12288 2.32e-7 -> 1.91e-7.  Time at 1536 x 27648 x 3072: 3761 us (69
// TFLOP/s) -> 1472 us (177); 1536 x 3072 x 9216: 2023 -> 647 us.
//
// A workgroup of four waves computes a 128 x 128 tile, each wave 64 x 64 (2 x 2
// blocks of 32 x 32; three sets of 64 accumulators leave room for two waves
// per SIMD), through chunks of 16 k in three LDS stages.  Both operands are
// loaded into registers, split there (5.5 VALU instructions an element) and
// written to LDS as three planes, so each element is split once per workgroup
// and each plane read feeds two MFMAs of three products.  Chunk kt + 2 is split
// and chunk kt + 3 loaded while chunk kt is multiplied.  The waves run their
// MFMAs at raised priority (s_setprio), so of a SIMD's two waves one keeps
// the matrix core while the other splits: 1801 -> 1501 us at 1536 x 27648 x
// 3072.  A larger wave tile does not fit the registers; running sums without
// the separate small accumulator do (156 TFLOP/s before the priorities against
// 148), but were 10% less exact than the fp32 MFMAs.
// As in the bf16 kernels the MFMA computes C^T = B A^T: the weight rows are the
// instruction's A operand, the activation rows its B operand, so lane l holds
// C[m = l % 32][n = 8 (i / 4) + 4 (l / 32) + i % 4] of each block and stores 4
// consecutive n.
// Rows past M or N load a clamped valid row (products never stored); k past
// K loads zeros, so any K >= 1 is exact.
// Operands outside the split's range (not finite, above 2^30, or so small that
// a part of them falls below bf16's range and it would show) send their tile
// through the fp32 matrix cores instead (f32_tile_native).
//
// Attention (no mask) for head dims other than 128 or rows that are not 16-byte aligned
// (the others run attention_f32.hip's fused kernel): per (batch, head), S = Q K^T by the
// GEMM, P = softmax(scale S) row by row in fp32 (max, then expf(scale s - max),
// then the sum), O = P V by the GEMM against V^T (a transposed copy), heads
// taken eight at a time through a workspace -- the fp32 arithmetic of ggml's
// CPU flash_attn_ext for F32 operands (FlashAttentionOp.cpp:84-94), with the
// probabilities normalised before the product instead of after.
#include <type_traits>

#include "capi_util.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace dit {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kF32MaxGroup = 8;
constexpr int FT = 128;          // tile edge
constexpr int FKC = 16;          // K per chunk
constexpr int FLUSH = 8;         // chunks per run of the sum
constexpr int FKP = FKC + 4;     // padded LDS row, floats (80 bytes: 16 lanes' 16-byte reads hit distinct banks)

struct F32Problem {
    const float* A;
    const float* B;
    float* C;
    const float* D;
    const float* bias;
    int64_t lda, ldb, ldc, ldd;
    int M, N, K;
    int vec;  // 16-byte row loads allowed (f32_validate)
};

struct F32Group {
    F32Problem p[kF32MaxGroup];
    int tile_start[kF32MaxGroup + 1];
    int count;
};

// This workgroup's problem and tile; XCD-contiguous numbering (each of the 8
// XCDs takes a contiguous range of tiles), in groups of 8 tile rows that share
// their weight columns: 1536 x 27648 x 3072 took 1524 us row by row, 1482 in
// groups of 4, 1472 of 8, 1458 of 16 (one group); 1536 x 3072 x 9216 665, 660,
// 647 and 660.
constexpr int F32_GROUP_M = 8;
__device__ __forceinline__ const F32Problem& f32_locate(const F32Group& g, int* tm, int* tn) {
    uint32_t bid = blockIdx.x;
    const uint32_t nb = gridDim.x, q = nb >> 3;
    if (bid < (q << 3)) bid = (bid & 7u) * q + (bid >> 3);
    int pi = 0;
    while (pi + 1 < g.count && (int)bid >= g.tile_start[pi + 1]) ++pi;
    const F32Problem& p = g.p[pi];
    const int local = (int)bid - g.tile_start[pi];
    const int tiles_m = (p.M + FT - 1) / FT, tiles_n = (p.N + FT - 1) / FT;
    const int per_group = F32_GROUP_M * tiles_n;
    const int group = local / per_group, first_m = group * F32_GROUP_M;
    const int rows = min(tiles_m - first_m, F32_GROUP_M);
    const int in_group = local - group * per_group;
    *tm = first_m + in_group % rows;
    *tn = in_group / rows;
    return p;
}

// 4 consecutive k of one row from k0, zeros past K.
template <bool VEC>
__device__ __forceinline__ float4 load4(const float* row, int k0, int K) {
    if constexpr (VEC) return *reinterpret_cast<const float4*>(row + k0);
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k0 + e < K ? row[k0 + e] : 0.0f;
    return make_float4(v[0], v[1], v[2], v[3]);
}

// 4 fp32 as three planes of 4 bf16 (8 bytes each), x = p0 + p1 + p2.
__device__ __forceinline__ void split3(const float4& x, uint2 (&p)[3]) {
    const uint32_t h0 = pack_bf16x2(x.x, x.y), h1 = pack_bf16x2(x.z, x.w);
    const float r0 = x.x - bf16_lo(h0), r1 = x.y - bf16_hi(h0), r2 = x.z - bf16_lo(h1), r3 = x.w - bf16_hi(h1);
    const uint32_t m0 = pack_bf16x2(r0, r1), m1 = pack_bf16x2(r2, r3);
    p[0] = make_uint2(h0, h1);
    p[1] = make_uint2(m0, m1);
    p[2] = make_uint2(pack_bf16x2(r0 - bf16_lo(m0), r1 - bf16_hi(m0)), pack_bf16x2(r2 - bf16_lo(m1), r3 - bf16_hi(m1)));
}

// max(m, |a|, |b|) in one instruction (fmaxf quiets each operand first); a NaN
// is passed over.
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
    return m;
}

// A stage: 16 k of the A rows, then of the B rows, as three planes of 256 rows
// x 32 bytes; half h (8 k) of row r at half h ^ xswz(r), so that 8 (32-bank) or
// 16 (64-bank) consecutive rows at one half hit distinct banks.
constexpr int XPLANE = 2 * FT * FKC * 2, XSTAGE = 3 * XPLANE, XSTAGES = 3;
__device__ __forceinline__ int xswz(int r) { return ((r >> 2) ^ (r >> 3)) & 1; }
// Largest |operand| and smallest |sum| the split products are used for.
constexpr float kSplitMax = 1073741824.0f;  // 2^30
constexpr float kSplitMin = 8.8817841970012523e-16f;  // 2^-50
constexpr float kTiny = 2.9103830456733704e-11f;  // 2^-35

// The tile on the fp32 matrix cores (v_mfma_f32_32x32x2_f32): products and
// sums in fp32 for operands of any magnitude.  Chunks of 16 k; MFMA s of a
// chunk (s = 0..7) multiplies the k-pair {s, 8 + s}: lanes 0-31 supply k = s
// and lanes 32-63 k = 8 + s, into set s % 2 of two running sums; runs of 8 chunks
// are summed (set 0 + set 1) before they join the tile's total.
template <bool VEC>
__device__ __forceinline__ void f32_tile_native(const F32Problem& p, uint8_t* smem, int m0, int n0, int wm, int wn,
                                                f32x16_t (&tot)[2][2]) {
    constexpr int OP = FT * FKP;
    float* sm = reinterpret_cast<float*>(smem);  // [2][A | B][128][FKP]
    const int tid = threadIdx.x, lane = tid & 63;
    const int row = tid >> 1, kh = (tid & 1) * 8;
    const float* arow = p.A + (int64_t)min(m0 + row, p.M - 1) * p.lda + kh;
    const float* brow = p.B + (int64_t)min(n0 + row, p.N - 1) * p.ldb + kh;
    f32x16_t acc[2][2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[0][j][i][e] = acc[1][j][i][e] = tot[j][i][e] = 0.f;
    const int lrow = lane & 31, lk = (lane >> 5) * 8;
    const int nk = (p.K + FKC - 1) / FKC, kn = p.K - kh;
    float4 a0, a1, b0, b1;
    auto fetch = [&](int kt) {
        const int k0 = kt * FKC;
        a0 = load4<VEC>(arow, k0, kn);
        a1 = load4<VEC>(arow, k0 + 4, kn);
        b0 = load4<VEC>(brow, k0, kn);
        b1 = load4<VEC>(brow, k0 + 4, kn);
    };
    fetch(0);
    __syncthreads();  // every wave's reads of the LDS before this tile are done
    for (int kt = 0; kt < nk; ++kt) {
        // Two stages: chunk kt is written beside chunk kt - 1, which is still read.
        float* const stage = sm + (kt & 1) * 2 * OP;
        float* a = stage + row * FKP + kh;
        *reinterpret_cast<float4*>(a) = a0;
        *reinterpret_cast<float4*>(a + 4) = a1;
        *reinterpret_cast<float4*>(a + OP) = b0;
        *reinterpret_cast<float4*>(a + OP + 4) = b1;
        __syncthreads();
        if (kt + 1 < nk) fetch(kt + 1);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float4 w[2], x[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                w[j] = *reinterpret_cast<const float4*>(stage + OP + (wn + 32 * j + lrow) * FKP + lk + 4 * half);
                x[j] = *reinterpret_cast<const float4*>(stage + (wm + 32 * j + lrow) * FKP + lk + 4 * half);
            }
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        acc[st & 1][j][i] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(w[j][st], x[i][st], acc[st & 1][j][i], 0, 0, 0);
        }
        if ((kt + 1) % FLUSH == 0 || kt + 1 == nk) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        tot[j][i][e] += acc[0][j][i][e] + acc[1][j][i][e];
                        acc[0][j][i][e] = acc[1][j][i][e] = 0.f;
                    }
        }
    }
}

template <bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const F32Group grp) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[XSTAGES * XSTAGE];
    static_assert(2 * 2 * FT * FKP * 4 <= XSTAGES * XSTAGE, "the fp32 tile's stages");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    const F32Problem& p = f32_locate(grp, &tm, &tn);
    const int m0 = tm * FT, n0 = tn * FT;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // Staging: k [4 q, + 4) of two rows of both operands per thread, so four
    // consecutive lanes load (and write) one row's 64 (32) consecutive bytes.
    const int row = tid >> 2, kq = (tid & 3) * 4;
    // VEC: buffer loads, the tile's first row the scalar base, a row's 32-bit
    // byte offset per lane (f32_validate bounds it), the chunk a scalar offset.
    const float* grow[4];  // A rows, B rows
    uint32_t gofs[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int ar = min(row + 64 * i, p.M - 1 - m0), br = min(row + 64 * i, p.N - 1 - n0);
        if constexpr (VEC) {
            gofs[i] = (uint32_t)(ar * (int)p.lda + kq) * 4u;
            gofs[2 + i] = (uint32_t)(br * (int)p.ldb + kq) * 4u;
        } else {
            grow[i] = p.A + (m0 + ar) * p.lda + kq;
            grow[2 + i] = p.B + (n0 + br) * p.ldb + kq;
        }
    }
    const __amdgpu_buffer_rsrc_t rsa =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A + m0 * p.lda), 0, 0x7FFFFFFF, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B + n0 * p.ldb), 0, 0x7FFFFFFF, 0x00020000);

    f32x16_t acc[2][2], low[2][2], tot[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][i][e] = low[j][i][e] = tot[j][i][e] = 0.f;

    float big = 0.f;  // largest |operand| this thread staged
    const int nk = (p.K + FKC - 1) / FKC, K = p.K;
    const int wofs = row * 32 + (((kq >> 3) ^ xswz(row)) << 4) + 2 * (kq & 4);
    float4 raw[4];
    // Chunks past the last are staged again from it and never read.
    auto fetch = [&](int kt) {
        const int k0 = min(kt, nk - 1) * FKC;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (VEC) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(i < 2 ? rsa : rsb, gofs[i], k0 * 4, 0);
                raw[i] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                                     __uint_as_float(v[3]));
            } else {
                raw[i] = load4<false>(grow[i], k0, K - kq);
            }
        }
    };
    auto stash = [&](uint8_t* st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 x = raw[i];
            uint2 pl[3];
            split3(x, pl);
            big = max3_abs(max3_abs(big, x.x, x.y), x.z, x.w);
#pragma unroll
            for (int j = 0; j < 3; ++j)
                *reinterpret_cast<uint2*>(st + wofs + 64 * 32 * i + XPLANE * j) = pl[j];
        }
    };

    const int lrow = lane & 31, g = lane >> 5;
    const int rofs = lrow * 32 + ((g ^ xswz(lrow)) << 4);
    const int xofs = wm * 32 + rofs, yofs = (FT + wn) * 32 + rofs;
    typedef bf16x8_t frag2[2];
    auto read = [&](const uint8_t* st, int ofs, int plane, frag2& f) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            f[j] = *reinterpret_cast<const bf16x8_t*>(st + ofs + XPLANE * plane + 32 * 32 * j);
    };
    auto mac = [&](f32x16_t (&c)[2][2], const frag2& wf, const frag2& xf) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                c[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], xf[i], c[j][i], 0, 0, 0);
    };
    // Set by a thread that has staged an operand out of range, at the end of an even or
    // odd run of FLUSH chunks, and read at the end of the next one: the rest of
    // the split products is then not taken.  A chunk's barrier lies between every write
    // and the reads before and after it, so all threads read the same.
    __shared__ int out_of_range[2];
    if (tid < 2) out_of_range[tid] = 0;
    fetch(0);
    stash(smem);
    fetch(1);
    stash(smem + XSTAGE);
    fetch(2);
    __syncthreads();
    uint8_t *s0 = smem, *s1 = smem + XSTAGE, *s2 = smem + 2 * XSTAGE;  // chunk kt, kt + 1, kt + 2
    bool early = false;
    for (int kt = 0; kt < nk;) {
        const int end = min(kt + FLUSH, nk);
        for (; kt < end; ++kt) {
            frag2 w0, w1, w2, x0, x1, x2;
            read(s0, yofs, 0, w0);
            read(s0, xofs, 0, x0);
            read(s0, xofs, 1, x1);
            __builtin_amdgcn_s_setprio(1);
            mac(acc, w0, x0);
            read(s0, yofs, 1, w1);
            mac(low, w0, x1);
            read(s0, xofs, 2, x2);
            mac(low, w1, x1);
            mac(low, w1, x0);
            read(s0, yofs, 2, w2);
            mac(low, w0, x2);
            mac(low, w2, x0);
            __builtin_amdgcn_s_setprio(0);
            stash(s2);
            fetch(kt + 3);
            // Chunk kt + 2 is written, and every wave has read chunk kt's planes
            // (chunk kt + 3 takes its stage next).
            __syncthreads();
            uint8_t* t = s0;
            s0 = s1;
            s1 = s2;
            s2 = t;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    tot[j][i][e] += acc[j][i][e];
                    acc[j][i][e] = 0.f;
                }
        const int run = (kt - 1) / FLUSH & 1;
        if (!(big < kSplitMax)) out_of_range[run] = 1;
        if (out_of_range[run ^ 1]) {
            early = true;
            break;
        }
    }

    // The split products stand in for fp32 ones only where every part of
    // them is a normal number: no operand above 2^30 (or not finite), and no
    // sum small enough for a part that fell below bf16's range to show.  A
    // sum of operands that are all zero or at least 2^-35 is exact however
    // small, so a small sum first looks for smaller operands.
    bool odd = !(big < kSplitMax), small = false;
    // One or two products (element-wise loads): leaving out the smallest three of nine then
    // shows, up to 1.9 of fp32's half units instead of 1.
    if constexpr (!VEC) odd |= K < 3;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float v = tot[j][i][e] += low[j][i][e];
                odd |= !(fabsf(v) < INFINITY);
                small |= fabsf(v) < kSplitMin;
            }
    if (!early && __syncthreads_or(small)) {
        for (int kt = 0; kt < nk; ++kt) {
            fetch(kt);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) odd |= x[e] != 0.f && fabsf(x[e]) < kTiny;
            }
        }
    }
    if (__syncthreads_or(odd)) f32_tile_native<VEC>(p, smem, m0, n0, wm, wn, tot);

    // Epilogue: bias, addend, store 4 consecutive n per lane where they fit.
    const bool v4 = (p.N % 4) == 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + wm + 32 * i + lrow;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wn + 32 * j + 8 * q + 4 * g;
                if (n >= p.N) continue;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * q + e;
                    v[e] = tot[j][i][r];
                    if (p.bias && n + e < p.N) v[e] += p.bias[n + e];
                    if (p.D && n + e < p.N) v[e] += p.D[(int64_t)m * p.ldd + n + e];
                }
                float* dst = p.C + (int64_t)m * p.ldc + n;
                if (v4 && n + 4 <= p.N) {
                    *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < p.N) dst[e] = v[e];
                }
            }
        }
    }
}

// ---- few rows -----------------------------------------------------------------
// The product is a stream of the weight, and the fp32 matrix cores keep up with
// it (18432 x 3072 at 16 rows: 12 us of v_mfma_f32_16x16x4_f32 against 44 us of
// weights at 5.1 TB/s), so nothing is split into bf16 parts.  As the bf16
// kernel for few rows (gemm.hip): a workgroup owns 16 weight rows, its KS waves one K range
// each, operands go straight from memory into registers, and the partial sums
// meet in LDS and are added in wave order.  Lane l supplies row l % 16, k = 16 b +
// 4 (l / 16) + s in MFMA s of 16-k block b.  Each s has a running sum of its own over 8
// blocks; the four are added and join the wave's total (one running sum was
// 20% less exact than the tiles, this is more).  At M = 1 18432 x 3072 341 ->
// 59 us, 3072 x 3072 339 -> 18 us.
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Up to 16 rows; up to 32 with fewer than four workgroups per CU (3072 x 3072 at 20 rows
// 22.5 us against 38 in tiles; 18432 x 3072 104 against 86, its activations
// being read again for every 16 weight rows).
bool f32_skinny(int64_t M, int64_t cols) { return M <= 16 || (M <= 32 && (cols + 15) / 16 < 4 * cu_count()); }

template <int MB, int KS>
__global__ __launch_bounds__(64 * KS) void gemm_f32_skinny_kernel(const F32Group grp) {
    constexpr int LD = 16 + 4;
    __shared__ float part[KS][16 * MB * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int pi = 0;
    while (pi + 1 < grp.count && (int)blockIdx.x >= grp.tile_start[pi + 1]) ++pi;
    const F32Problem& p = grp.p[pi];
    const int n0 = ((int)blockIdx.x - grp.tile_start[pi]) * 16;
    const int r = lane & 15, g = lane >> 4;
    const int nblk = p.K / 16, per = (nblk + KS - 1) / KS;
    const int b0 = min(wave * per, nblk), b1 = min(b0 + per, nblk);
    const float* wp = p.B + (int64_t)min(n0 + r, p.N - 1) * p.ldb + 4 * g;
    const float* xp[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) xp[i] = p.A + (int64_t)min(16 * i + r, p.M - 1) * p.lda + 4 * g;
    f32x4_t tot[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) tot[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // U blocks from block b: one run.
    auto run = [&](int b, auto uc) {
        constexpr int U = decltype(uc)::value;
        float4 w[U], x[U][MB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint4 t = ld_stream(wp + (int64_t)(b + u) * 16);
            w[u] = make_float4(__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z), __uint_as_float(t.w));
#pragma unroll
            for (int i = 0; i < MB; ++i) x[u][i] = *reinterpret_cast<const float4*>(xp[i] + (int64_t)(b + u) * 16);
        }
        f32x4_t acc[MB][4];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[i][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float wv[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const float xv[4] = {x[u][i].x, x[u][i].y, x[u][i].z, x[u][i].w};
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    acc[i][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s], xv[s], acc[i][s], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) tot[i][e] += (acc[i][0][e] + acc[i][1][e]) + (acc[i][2][e] + acc[i][3][e]);
    };
    int b = b0;
    for (; b + 8 <= b1; b += 8) run(b, std::integral_constant<int, 8>{});
    for (; b + 2 <= b1; b += 2) run(b, std::integral_constant<int, 2>{});
    if (b < b1) run(b, std::integral_constant<int, 1>{});

#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[wave][(16 * i + r) * LD + 4 * g + e] = tot[i][e];
    __syncthreads();
    for (int u = tid; u < 16 * MB * 16; u += 64 * KS) {
        const int m = u >> 4, c = u & 15, n = n0 + c;
        if (m >= p.M || n >= p.N) continue;
        float v = part[0][m * LD + c];
#pragma unroll
        for (int k = 1; k < KS; ++k) v += part[k][m * LD + c];
        if (p.bias) v += p.bias[n];
        if (p.D) v += p.D[(int64_t)m * p.ldd + n];
        p.C[(int64_t)m * p.ldc + n] = v;
    }
}

template <int MB>
int f32_skinny_launch(const F32Problem* ps, int n, hipStream_t st) {
    F32Group g{};
    g.count = n;
    int64_t total = 0;
    for (int i = 0; i < n; ++i) {
        g.p[i] = ps[i];
        g.tile_start[i] = (int)total;
        total += ((int64_t)ps[i].N + 15) / 16;
    }
    DT_REQUIRE(total < (1ll << 31), "dt_gemm_f32: too many tiles");
    g.tile_start[n] = (int)total;
    // Eight waves a workgroup until there are four workgroups per CU.
    if (total >= 4 * cu_count())
        hipLaunchKernelGGL((gemm_f32_skinny_kernel<MB, 4>), dim3((unsigned)total), dim3(256), 0, st, g);
    else
        hipLaunchKernelGGL((gemm_f32_skinny_kernel<MB, 8>), dim3((unsigned)total), dim3(512), 0, st, g);
    return check_launch("dt_gemm_f32");
}

int64_t f32_tiles(const F32Problem& p) { return (int64_t)((p.M + FT - 1) / FT) * ((p.N + FT - 1) / FT); }

int f32_launch(const F32Problem* ps, int n, hipStream_t st) {
    // 16-byte row loads or not is the kernel's, so a group that holds both kinds
    // is two launches: one unaligned problem does not slow the others.
    F32Problem part[2][kF32MaxGroup];
    int np[2] = {0, 0};
    for (int i = 0; i < n; ++i) {
        const int kind = ps[i].vec != 0;
        part[kind][np[kind]++] = ps[i];
    }
    if (np[0] && np[1]) {
        const int rc = f32_launch(part[0], np[0], st);
        return rc ? rc : f32_launch(part[1], np[1], st);
    }
    const bool vec = np[1] > 0;
    int m_max = 0;
    int64_t cols = 0;
    for (int i = 0; i < n; ++i) {
        m_max = m_max > ps[i].M ? m_max : ps[i].M;
        cols += ps[i].N;
    }
    if (vec && f32_skinny(m_max, cols))
        return m_max <= 16 ? f32_skinny_launch<1>(ps, n, st) : f32_skinny_launch<2>(ps, n, st);
    F32Group g{};
    g.count = n;
    int64_t total = 0;
    for (int i = 0; i < n; ++i) {
        g.p[i] = ps[i];
        g.tile_start[i] = (int)total;
        total += f32_tiles(ps[i]);
    }
    DT_REQUIRE(total < (1ll << 31), "dt_gemm_f32: too many tiles");
    g.tile_start[n] = (int)total;
    if (total == 0) return DT_OK;
    if (vec)
        hipLaunchKernelGGL(gemm_f32_kernel<true>, dim3((unsigned)total), dim3(256), 0, st, g);
    else
        hipLaunchKernelGGL(gemm_f32_kernel<false>, dim3((unsigned)total), dim3(256), 0, st, g);
    return check_launch("dt_gemm_f32");
}

// 128 rows of it span less than 2^31 bytes.
constexpr int64_t kVecLd = (1ll << 22) - 1;

int f32_validate(const dt_gemm_problem& q, F32Problem* out) {
    DT_REQUIRE(q.M >= 0 && q.N >= 0 && q.K > 0, "dt_gemm_f32: bad shape");
    DT_REQUIRE(q.M < (1ll << 31) && q.N < (1ll << 31) && q.K < (1ll << 31), "dt_gemm_f32: shape too large");
    DT_REQUIRE(!q.b_scale, "dt_gemm_f32: F32 weights only");
    int vec = 0;
    if (q.M > 0 && q.N > 0) {
        DT_REQUIRE(q.lda >= q.K && q.ldb >= q.K && q.ldc >= q.N, "dt_gemm_f32: leading dimensions must cover the rows");
        DT_REQUIRE(!q.addend || q.ldd >= q.N, "dt_gemm_f32: ldd < N");
        DT_REQUIRE(q.A && q.B && q.C, "dt_gemm_f32: null pointer");
        DT_REQUIRE(((reinterpret_cast<uintptr_t>(q.A) | reinterpret_cast<uintptr_t>(q.B)) & 3) == 0,
                   "dt_gemm_f32: A and B must be 4-byte aligned");
        DT_REQUIRE(q.N % 4 != 0 || ((reinterpret_cast<uintptr_t>(q.C) & 15) == 0 && q.ldc % 4 == 0),
                   "dt_gemm_f32: C must be 16-byte aligned with ldc %% 4 == 0");
        vec = q.K % FKC == 0 && q.lda % 4 == 0 && q.ldb % 4 == 0 && q.lda <= kVecLd && q.ldb <= kVecLd && aligned16(q.A) && aligned16(q.B);
    }
    *out = F32Problem{(const float*)q.A, (const float*)q.B, (float*)q.C, (const float*)q.addend, q.bias,
                      q.lda, q.ldb, q.ldc, q.ldd, (int)q.M, (int)q.N, (int)q.K, vec};
    return DT_OK;
}

// ---- attention pieces ---------------------------------------------------------

// dst[r][c] = src[c * src_ld + r] for a rows x cols block: V [Skv][128]
// (token stride src_ld) -> V^T [128][Skv]; 32 x 32 tiles through LDS.
__global__ __launch_bounds__(256) void transpose_f32_kernel(const float* __restrict__ src, int64_t src_ld,
                                                            float* __restrict__ dst, int rows, int cols) {
    __shared__ float t[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    for (int k = ty; k < 32; k += 8) {
        const int c = c0 + k, r = r0 + tx;
        t[k][tx] = (c < cols && r < rows) ? src[(int64_t)c * src_ld + r] : 0.0f;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        if (r < rows && c < cols) dst[(int64_t)r * cols + c] = t[tx][k];
    }
}

// Row-wise softmax(scale * s) in place over rows of n: one workgroup per row.
__global__ __launch_bounds__(256) void softmax_rows_f32_kernel(float* __restrict__ s, int64_t n, float scale) {
    __shared__ float red[256 / kWave];
    float* row = s + (int64_t)blockIdx.x * n;
    float mx = -INFINITY;
    for (int64_t i = threadIdx.x; i < n; i += 256) mx = fmaxf(mx, scale * row[i]);
    // block max
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (lane == 0) red[wid] = mx;
    __syncthreads();
    mx = red[0];
    for (int i = 1; i < 256 / kWave; ++i) mx = fmaxf(mx, red[i]);
    float sum = 0.0f;
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const float e = expf(scale * row[i] - mx);
        row[i] = e;
        sum += e;
    }
    sum = block_sum_f32(sum, red);
    const float inv = 1.0f / sum;
    for (int64_t i = threadIdx.x; i < n; i += 256) row[i] *= inv;
}

}  // namespace
}  // namespace dit

extern "C" int dt_gemm_f32_grouped(const dt_gemm_problem* problems, int32_t count, dt_stream_t stream) {
    using namespace dit;
    DT_REQUIRE(count >= 0 && count <= kF32MaxGroup, "dt_gemm_f32_grouped: count %d outside 0..%d", count,
               kF32MaxGroup);
    DT_REQUIRE(problems || count == 0, "dt_gemm_f32_grouped: null problem list");
    F32Problem ps[kF32MaxGroup];
    int n = 0;
    for (int i = 0; i < count; ++i) {
        F32Problem p;
        const int rc = f32_validate(problems[i], &p);
        if (rc) return rc;
        if (p.M > 0 && p.N > 0) ps[n++] = p;
    }
    if (n == 0) return DT_OK;
    return f32_launch(ps, n, (hipStream_t)stream);
}

extern "C" int dt_gemm_f32(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc, int64_t M,
                           int64_t N, int64_t K, const float* bias, const float* addend, int64_t ldd,
                           dt_stream_t stream) {
    const dt_gemm_problem p{A, lda, B, ldb, C, ldc, addend, ldd, bias, M, N, K, nullptr, 0};
    return dt_gemm_f32_grouped(&p, 1, stream);
}

// K ranges of one product (1: not split), for products of at most two tiles per
// CU (a CU runs two at once): the number with the least estimated time, rounds
// of workgroups at 6.3 us per 128 k of one tile alone on its CU and 10.2 beside
// another (both measured), then the reduce, its launch and the partial sums at
// 5 TB/s.  A range has at least 512 k.  3072 x 9216, Python call included: 200 rows
// 456 us in one range, 99 in eight; 1536 rows 647 and 496 (five).
static int f32_split_count(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ((M + dit::FT - 1) / dit::FT) * ((N + dit::FT - 1) / dit::FT), cus = dit::cu_count();
    if (dit::f32_skinny(M, N) || K % 64 != 0 || tiles > 2 * cus) return 1;
    int best = 1;
    double best_t = 1e300;
    for (int64_t S = 1; S <= dit::kF32MaxGroup && (S == 1 || S <= K / 512); ++S) {
        const int64_t full = tiles * S / (2 * cus), rest = tiles * S - full * 2 * cus;
        const double rounds = (double)full * 10.2 + (rest > cus ? 10.2 : rest > 0 ? 6.3 : 0.0);
        const double t = rounds * (double)K / (double)(128 * S) +
                         (S > 1 ? 5.0 + (double)(S * M * N) * 8.0 / 5.0e6 : 0.0);
        if (t < best_t) {
            best_t = t;
            best = (int)S;
        }
    }
    return best;
}

extern "C" size_t dt_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || M >= (1ll << 31) || N >= (1ll << 31)) return 0;
    const int s = f32_split_count(M, N, K);
    return s > 1 ? (size_t)(s * M * dit::gemm_split_ld(N)) * sizeof(float) : 0;
}

extern "C" int dt_gemm_f32_ws(const dt_gemm_problem* problem, void* workspace, size_t workspace_bytes,
                              dt_stream_t stream) {
    using namespace dit;
    DT_REQUIRE(problem != nullptr, "dt_gemm_f32_ws: null problem");
    const dt_gemm_problem& q = *problem;
    const size_t need = dt_gemm_f32_workspace_bytes(q.M, q.N, q.K);
    if (need == 0 || !workspace || workspace_bytes < need || !aligned16(workspace))
        return dt_gemm_f32_grouped(problem, 1, stream);
    F32Problem p;
    const int rc = f32_validate(q, &p);
    if (rc) return rc;
    const int S = f32_split_count(q.M, q.N, q.K);
    const int64_t ldp = gemm_split_ld(q.N), blocks = q.K / 64;
    F32Problem ps[kF32MaxGroup];
    float* part = (float*)workspace;
    for (int s = 0; s < S; ++s) {
        const int64_t k0 = blocks * s / S * 64, k1 = blocks * (s + 1) / S * 64;
        ps[s] = p;
        ps[s].A = p.A + k0;
        ps[s].B = p.B + k0;
        ps[s].K = (int)(k1 - k0);
        ps[s].C = part + s * q.M * ldp;
        ps[s].ldc = ldp;
        ps[s].D = nullptr;
        ps[s].bias = nullptr;
    }
    const int rl = f32_launch(ps, S, (hipStream_t)stream);
    if (rl) return rl;
    return gemm_reduce(part, S, q.M, q.N, q.C, q.ldc, q.bias, q.addend, q.ldd, DT_TYPE_F32, (hipStream_t)stream);
}

// Workspace of dt_flash_attn_f32: per head of a group of up to 8, the
// scores [seq_q][seq_kv] and V^T [head_dim][seq_kv], fp32; or what the fused kernel
// needs, if that is more.  It takes 1536 bytes per key and head, so beyond
// kFusedWs (24 heads of 7000 keys) and the group's scores it takes fewer heads
// per launch: a call's memory does not grow with its batch.
static int64_t attn_f32_group(int64_t batch, int64_t heads) {
    const int64_t bh = batch * heads;
    return bh < dit::kF32MaxGroup ? bh : dit::kF32MaxGroup;
}
constexpr size_t kFusedWs = 256u << 20;

static size_t attn_f32_gemm_bytes(int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim) {
    const int64_t per = (seq_q * seq_kv + head_dim * seq_kv + 3) / 4 * 4;  // 16-byte aligned per head
    return (size_t)(attn_f32_group(batch, heads) * per) * sizeof(float);
}

// (batch, head) pairs per launch of the fused kernel, 0: not for these sizes.
static int64_t attn_f32_per_launch(int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim) {
    if (head_dim != 128) return 0;
    const size_t gemms = attn_f32_gemm_bytes(batch, heads, seq_q, seq_kv, head_dim);
    return dit::attn_f32_fused_heads(batch * heads, seq_q, seq_kv, gemms > kFusedWs ? gemms : kFusedWs);
}

extern "C" size_t dt_flash_attn_f32_workspace_bytes(int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_kv,
                                                     int64_t head_dim) {
    if (batch <= 0 || heads <= 0 || seq_q <= 0 || seq_kv <= 0 || head_dim <= 0) return 0;
    const size_t gemms = attn_f32_gemm_bytes(batch, heads, seq_q, seq_kv, head_dim);
    const int64_t n = attn_f32_per_launch(batch, heads, seq_q, seq_kv, head_dim);
    const size_t fused = n ? dit::attn_f32_fused_bytes(n, seq_q, seq_kv) : 0;
    return gemms > fused ? gemms : fused;
}

extern "C" int dt_flash_attn_f32(const float* q, const float* k, const float* v, float* o, int64_t batch,
                                 int64_t heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim,
                                 const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                 const int64_t* o_strides, float scale, void* workspace, size_t workspace_bytes,
                                 dt_stream_t stream) {
    using namespace dit;
    DT_REQUIRE(batch >= 0 && heads >= 0 && seq_q >= 0 && seq_kv >= 0 && head_dim > 0,
               "dt_flash_attn_f32: bad shape");
    if (batch == 0 || heads == 0 || seq_q == 0) return DT_OK;
    DT_REQUIRE(seq_kv > 0, "dt_flash_attn_f32: no keys");
    DT_REQUIRE(q && k && v && o && q_strides && k_strides && v_strides && o_strides, "dt_flash_attn_f32: null pointer");
    DT_REQUIRE(seq_q < (1ll << 31) && seq_kv < (1ll << 31) && seq_q * seq_kv < (1ll << 40),
               "dt_flash_attn_f32: sequence too long");
    const size_t need = dt_flash_attn_f32_workspace_bytes(batch, heads, seq_q, seq_kv, head_dim);
    DT_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace),
               "dt_flash_attn_f32: workspace of %zu bytes (16-byte aligned) needed", need);
    hipStream_t st = (hipStream_t)stream;
    const int64_t per_launch = attn_f32_per_launch(batch, heads, seq_q, seq_kv, head_dim);
    if (per_launch && attn_f32_fused_takes(q, k, v, o, batch, heads, seq_q, seq_kv, head_dim, q_strides, k_strides,
                                           v_strides, o_strides, scale))
        return attn_f32_fused(q, k, v, o, batch, heads, seq_q, seq_kv, q_strides, k_strides, v_strides, o_strides, scale,
                              per_launch, workspace, st);
    const int64_t per = (seq_q * seq_kv + head_dim * seq_kv + 3) / 4 * 4;
    const int64_t bh = batch * heads, gsz = attn_f32_group(batch, heads);
    float* ws = (float*)workspace;
    for (int64_t h0 = 0; h0 < bh; h0 += gsz) {
        const int n = (int)(bh - h0 < gsz ? bh - h0 : gsz);
        dt_gemm_problem sp[kF32MaxGroup], op[kF32MaxGroup];
        for (int i = 0; i < n; ++i) {
            const int64_t b = (h0 + i) / heads, h = (h0 + i) % heads;
            float* S = ws + i * per;
            float* Vt = S + seq_q * seq_kv;
            const float* qh = q + b * q_strides[0] + h * q_strides[2];
            const float* kh = k + b * k_strides[0] + h * k_strides[2];
            const float* vh = v + b * v_strides[0] + h * v_strides[2];
            float* oh = o + b * o_strides[0] + h * o_strides[2];
            // V^T [head_dim][seq_kv]
            const dim3 tg((unsigned)((seq_kv + 31) / 32), (unsigned)((head_dim + 31) / 32));
            hipLaunchKernelGGL(transpose_f32_kernel, tg, dim3(256), 0, st, vh, v_strides[1], Vt, (int)head_dim,
                               (int)seq_kv);
            int rc = check_launch("dt_flash_attn_f32(transpose)");
            if (rc) return rc;
            sp[i] = dt_gemm_problem{qh, q_strides[1], kh, k_strides[1], S, seq_kv, nullptr, 0, nullptr,
                                    seq_q, seq_kv, head_dim, nullptr, 0};
            op[i] = dt_gemm_problem{S, seq_kv, Vt, seq_kv, oh, o_strides[1], nullptr, 0, nullptr,
                                    seq_q, head_dim, seq_kv, nullptr, 0};
        }
        int rc = dt_gemm_f32_grouped(sp, n, stream);
        if (rc) return rc;
        for (int i = 0; i < n; ++i) {
            hipLaunchKernelGGL(softmax_rows_f32_kernel, dim3((unsigned)seq_q), dim3(256), 0, st, ws + i * per,
                               seq_kv, scale);
            rc = check_launch("dt_flash_attn_f32(softmax)");
            if (rc) return rc;
        }
        rc = dt_gemm_f32_grouped(op, n, stream);
        if (rc) return rc;
    }
    return DT_OK;
}
