// attention.hip -- unmasked scaled-dot-product attention for head_dim 128,
// the op behind FlashAttentionOp::operator() (src/nn/attention/FlashAttentionOp.cpp:84-94,
// ggml_flash_attn_ext with scale 1/sqrt(128), no mask in Flux2):
//   O[s, :] = sum_j softmax_j(scale * <Q[s], K[j]>) V[j, :]   per (batch, head).
//
// Formulation (gfx950, v_mfma_f32_32x32x16_bf16): each wave owns 32 queries
// and computes the TRANSPOSED products S^T = K Q^T and O^T += V^T P^T, so the
// accumulator column -- the query -- is the lane index (lane % 32) in both.
// Every per-query softmax quantity (running max, running sum, rescale factor)
// is therefore a per-lane scalar, shared only with the partner lane l ^ 32
// that holds the other half of the keys.  P^T goes from the S^T accumulator
// registers straight into the B operand of the PV product: the MFMA's
// reduction index is a permutation of 16 keys, and V^T is read from LDS in
// that same permutation (keys {4g..4g+3, 8+4g..8+4g+3} for lane half g).
//
// A 256-thread workgroup (4 waves, 128 queries) shares 64-key K and V tiles
// in LDS, double-buffered and filled by direct DMA; two workgroups per CU
// give each SIMD two waves, so one wave's softmax overlaps the other's
// MFMAs.  Workgroups are ordered so that each XCD (8 per MI355X, one L2 each)
// works through a contiguous range of (batch, head) slices.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "capi_util.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "rope_angles.hpp"

namespace dit {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int D = 128;       // head dim
constexpr int QB = 128;      // queries per workgroup

struct AttnArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    void* o;
    int64_t qs[3], ks[3], vs[3], os[3];  // batch, token, head strides (elements)
    int32_t batch, heads, seq_q, seq_kv;
    int32_t q_blocks;                     // ceil(seq_q / QB)
    float scale_log2;                     // scale * log2(e)
};

// The Q prologue's operands: q before its QK-RMSNorm + RoPE, in up to two
// token segments with their own norm weights (the txt | img concatenation of
// Flux2Attention.hpp:93-116; one segment: split = seq_q), and the RoPE
// positions of the joint sequence.
struct AttnPro {
    const uint16_t* q0;
    const uint16_t* q1;
    int64_t q0_bs, q0_ts, q0_hs, q1_bs, q1_ts, q1_hs;  // batch, token, head strides (elements)
    const float* w0;
    const float* w1;
    int32_t split;       // queries [0, split) from q0, [split, seq_q) from q1 (token - split)
    int32_t axis_dim, n_pos;
    float theta_scale, eps;
    const float* table;  // [n_pos][axis_dim] (cos, sin); NULL: angles on the device
    RopeAxisPos pos;     // position of joint token t on axis a: pos.ptr[a][t * pos.stride[a]]
};

__device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

// Position of token t on axis `axis`, through an unrolled select so the
// kernel-argument arrays are never indexed dynamically.
__device__ __forceinline__ int pro_position(const RopeAxisPos& pos, int axis, int t) {
    const int32_t* p = pos.ptr[0];
    int64_t st = pos.stride[0];
#pragma unroll
    for (int a = 1; a < kMaxRopeAxes; ++a)
        if (axis == a) {
            p = pos.ptr[a];
            st = pos.stride[a];
        }
    return p[(int64_t)t * st];
}

// ---- K/V by direct DMA, two workgroups per CU ---------------------------------
// K and V tiles move global -> LDS by direct DMA (global_load_lds_dwordx4)
// into two 32 KB buffers, so no registers are spent on staging.  At most 256 registers per lane (two waves per SIMD):
// one wave's softmax (VALU) runs while the other wave on the SIMD issues
// MFMAs.  V stays [key][d] in LDS; the V^T A operand is read with
// ds_read_tr16_b64, which gives lane i of a 16-lane group element c = i % 4
// of lane 4 j + i / 4's 4 x b16: with lane s addressing V[k0 + s / 4][d0 +
// 4 (s % 4) ..], lane i receives V[k0 + j][d0 + i] for j = 0..3, i.e. four
// keys of one d.  Rows of 256 bytes are XOR-swizzled in 16-byte chunks:
// K chunk c of row r at c ^ (r & 15) (16 rows read one logical chunk),
// V chunk c at c ^ 4 (r & 3) (4 rows x 4 consecutive chunks per transposed
// read).
constexpr int DKB = 64;                 // keys per tile
constexpr int DROW = D * 2;             // bytes per K / V row
constexpr int DTILE = DKB * DROW;       // 16 KB

__device__ __forceinline__ int kswz(int r) { return r & 15; }
__device__ __forceinline__ int vswz(int r) { return (r & 3) << 2; }

template <int N_OUT>
__device__ __forceinline__ void attn_wait_vm() {
    __builtin_amdgcn_s_waitcnt((N_OUT & 15) | ((N_OUT >> 4) << 14) | 0x0F70);
}

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t* lds_short4_p;

// ds_read_tr16_b64 of the 8 bytes at p (an LDS address).
__device__ __forceinline__ uint2 read_tr16(const uint8_t* p) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_p)(p)));
}

// Chunk c (8 dims) of queries q0 + row, + row + 4, ... (N of them) with QK-RMSNorm + RoPE
// applied, 16 lanes a query, as bf16 into their rows of `rows` in LDS (chunk c of row r at
// c ^ (r & 15)).  Every operation is the QK kernel's (qk_rope.hip), in its order: per
// 8-dim chunk the sum of squares, the 16 chunk sums added by its 16-lane DPP tree, 1 /
// sqrt(ss / 128 + eps), (x * r) * w, the rotation, one bf16 rounding -- so the q used here
// is bit-identical to the stored output of dt_qk_rmsnorm_rope.  (A lane taking half of a
// query's chunks, as its MFMA operand holds them, made 16-byte loads of 64 scattered
// lines and a long unrolled body: about 5 us of the 16.5 a 320-token attention took.)
// All N queries' loads are issued before the first is used, and the angles' loads,
// which wait for the positions, together: query by query each of a wave's eight waited
// for memory twice.  With operands from HBM (many input sets in turn): 16 heads of 1068
// 36.7 -> 33.4 us, 24 of 700 28.7 -> 25.3, 24 of 1536 56.5 -> 52.8, 24 of 320 10.1 -> 9.7.
template <int N>
__device__ __forceinline__ void q_prologue16(const AttnPro& pro, int b, int h, int q0, int row, int seq_q, int c,
                                             uint8_t* rows) {
    const int d0 = 8 * c, axis = d0 / pro.axis_dim, i0 = d0 - axis * pro.axis_dim;
    auto emit = [&](int n, const uint4& raw, const float (&cs)[8]) {
        const float* w = (min(q0 + row + 4 * n, seq_q - 1) >= pro.split ? pro.w1 : pro.w0) + d0;
        const float4 wa = *reinterpret_cast<const float4*>(w), wb = *reinterpret_cast<const float4*>(w + 4);
        const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
        float v[8], o[8];
        Io<bf16>::unpack(raw, v);
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        ss = row16_sum(ss);
        const float rs = 1.0f / sqrtf(ss / (float)D + pro.eps);
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const float x0 = mul_rn(mul_rn(v[2 * qd], rs), wv[2 * qd]);
            const float x1 = mul_rn(mul_rn(v[2 * qd + 1], rs), wv[2 * qd + 1]);
            const float cn = cs[2 * qd], sn = cs[2 * qd + 1];
            o[2 * qd] = sub_rn(mul_rn(x0, cn), mul_rn(x1, sn));
            o[2 * qd + 1] = add_rn(mul_rn(x0, sn), mul_rn(x1, cn));
        }
        const int r = row + 4 * n;
        *reinterpret_cast<uint4*>(rows + r * DROW + ((c ^ (r & 15)) << 4)) = Io<bf16>::pack(o);
    };
    int p[N];
    uint4 raw[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const int qrow = min(q0 + row + 4 * n, seq_q - 1);  // rows past the sequence are never stored
        const int seg = qrow >= pro.split, tok = seg ? qrow - pro.split : qrow;
        p[n] = pro_position(pro.pos, axis, qrow);
        raw[n] = ld16((seg ? pro.q1 + b * pro.q1_bs + (int64_t)tok * pro.q1_ts + h * pro.q1_hs
                           : pro.q0 + b * pro.q0_bs + (int64_t)tok * pro.q0_ts + h * pro.q0_hs) + d0);
    }
    bool hit = pro.table != nullptr;
#pragma unroll
    for (int n = 0; n < N; ++n) hit = hit && p[n] >= 0 && p[n] < pro.n_pos;
    if (__builtin_amdgcn_ballot_w64(!hit) == 0) {  // every angle from the table
        float cs[N][8];
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float* t = pro.table + (int64_t)p[n] * pro.axis_dim + i0;  // rope_angles' table branch
            const float4 ca = *reinterpret_cast<const float4*>(t), cb = *reinterpret_cast<const float4*>(t + 4);
            cs[n][0] = ca.x; cs[n][1] = ca.y; cs[n][2] = ca.z; cs[n][3] = ca.w;
            cs[n][4] = cb.x; cs[n][5] = cb.y; cs[n][6] = cb.z; cs[n][7] = cb.w;
        }
#pragma unroll
        for (int n = 0; n < N; ++n) emit(n, raw[n], cs[n]);
    } else {
        // Some angle off the table: unrolled for eight queries this body would
        // put their registers into scratch memory.
        constexpr int U = N <= 2 ? N : 1;
#pragma unroll U
        for (int n = 0; n < N; ++n) {
            int pn = p[0];
            uint4 rn = raw[0];
#pragma unroll
            for (int i = 1; i < N; ++i)
                if (n == i) {
                    pn = p[i];
                    rn = raw[i];
                }
            float cs[8];
            rope_angles<4>(pn, i0, pro.table, pro.n_pos, pro.axis_dim, pro.theta_scale, cs);
            emit(n, rn, cs);
        }
    }
}

template <typename TO, bool PRO>
__global__ __launch_bounds__(256, 2) void flash_attn_dma_kernel(AttnArgs a, AttnPro pro) {
    // [buffer][K | V][64 rows][256 B]
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * 2 * DTILE];

    uint32_t bid = blockIdx.x;
    const uint32_t nb = gridDim.x;
    if ((nb & 7u) == 0) bid = (bid & 7u) * (nb >> 3) + (bid >> 3);
    const int qblk = (int)(bid % (uint32_t)a.q_blocks);
    const int bh = (int)(bid / (uint32_t)a.q_blocks);
    const int h = bh % a.heads, b = bh / a.heads;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, g = lane >> 5;
    const int q0 = qblk * QB + wave * 32;

    const uint16_t* Qp = a.q + b * a.qs[0] + h * a.qs[2];
    const uint16_t* Kp = a.k + b * a.ks[0] + h * a.ks[2];
    const uint16_t* Vp = a.v + b * a.vs[0] + h * a.vs[2];

    bf16x8_t qf[8];
    if constexpr (!PRO) {
        const int qrow = q0 + r;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            uint4 u = qrow < a.seq_q ? ld16(Qp + (int64_t)qrow * a.qs[1] + 16 * c + 8 * g) : make_uint4(0, 0, 0, 0);
            qf[c] = __builtin_bit_cast(bf16x8_t, u);
        }
    }

    // DMA: wave w fills rows [16 w, 16 w + 16) of the K and the V tile, four
    // instructions of 4 rows each; lane i covers row + i / 16, stored chunk
    // i % 16, loaded from the swizzled source chunk.  Rows past seq_kv load
    // the last valid row (finite data; their scores are masked).
    const int drow = 16 * wave + (lane >> 4), dpos = lane & 15;
    const uint16_t* kq[4];
    const uint16_t* vq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = drow + 4 * j;
        kq[j] = Kp + (int64_t)row * a.ks[1] + (dpos ^ kswz(row)) * 8;
        vq[j] = Vp + (int64_t)row * a.vs[1] + (dpos ^ vswz(row)) * 8;
    }
    auto issue = [&](int kv0, int buf) {
        uint8_t* kb = smem + buf * 2 * DTILE + 16 * wave * DROW;
        uint8_t* vb = kb + DTILE;
        if (kv0 + DKB <= a.seq_kv) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                __builtin_amdgcn_global_load_lds(kq[j] + (int64_t)kv0 * a.ks[1], kb + 4 * j * DROW, 16, 0, 0);
                __builtin_amdgcn_global_load_lds(vq[j] + (int64_t)kv0 * a.vs[1], vb + 4 * j * DROW, 16, 0, 0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int row = drow + 4 * j;
                const int key = min(kv0 + row, a.seq_kv - 1);
                __builtin_amdgcn_global_load_lds(Kp + (int64_t)key * a.ks[1] + (dpos ^ kswz(row)) * 8,
                                                 kb + 4 * j * DROW, 16, 0, 0);
                __builtin_amdgcn_global_load_lds(Vp + (int64_t)key * a.vs[1] + (dpos ^ vswz(row)) * 8,
                                                 vb + 4 * j * DROW, 16, 0, 0);
            }
        }
    };

    // Per-lane LDS offsets, the same for every tile.  K: row 32 hh + r, chunk
    // 2 c + g at (2 c + g) ^ (r & 15) (32 hh is an immediate).  V (transposed
    // reads): lane s of 16-lane group gi reads row 16 j + 4 tg + s / 4 (+ 8),
    // d = 32 tt + 16 dsub + 4 (s % 4), whose swizzled chunk is
    // 4 (tt ^ s / 4) + (16 dsub + 4 (s % 4)) / 8.
    int koff[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) koff[c] = r * DROW + (((2 * c + g) ^ (r & 15)) << 4);
    const int s16 = lane & 15, gi = lane >> 4, tg = gi >> 1, dsub = gi & 1;
    const int trow = s16 >> 2, tcol = 16 * dsub + 4 * (s16 & 3);
    int voff[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
        voff[tt] = (4 * tg + trow) * DROW + ((4 * (tt ^ trow) + (tcol >> 3)) << 4) + 8 * ((tcol >> 2) & 1);

    f32x16_t o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;  // running max in units of scale * log2(e)
    const float sc = a.scale_log2;          // >= 0, so max(sc * s) = sc * max(s)

    const int ntiles = (a.seq_kv + DKB - 1) / DKB;
    auto tile = [&](int t, auto buf_c, auto mask_c) {
        constexpr int BUF = decltype(buf_c)::value;
        constexpr bool MASK = decltype(mask_c)::value;
        const int kv0 = t * DKB;
        // One barrier per tile: once every wave has this tile's DMA and has
        // finished the previous tile (its LDS reads returned), the previous
        // tile's buffer takes tile t + 1 while tile t is computed -- the same
        // slack as issuing it two tiles ahead after a second barrier at the
        // end of each tile, which measured 3% slower (271.7 -> 263.7 us at
        // 4608 x 4608 x 24 heads).
        attn_wait_vm<0>();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        if (t + 1 < ntiles) issue(kv0 + DKB, BUF ^ 1);
        const uint8_t* Kt = smem + BUF * 2 * DTILE;
        const uint8_t* Vt_ = Kt + DTILE;

        // The two 32-key halves are independent accumulator chains; issuing
        // them alternately keeps the MFMA pipe from waiting on each result.
        f32x16_t sacc[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int e = 0; e < 16; ++e) sacc[hh][e] = 0.f;
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(Kt + 32 * hh * DROW + koff[c]);
                sacc[hh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], sacc[hh], 0, 0, 0);
            }
        // Element i of sacc[hh] is key kv0 + 32 hh + 8 (i / 4) + 4 g + i % 4.
        float mx = -INFINITY;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (MASK && kv0 + 32 * hh + 8 * (i >> 2) + 4 * g + (i & 3) >= a.seq_kv) continue;
                mx = fmaxf(mx, sacc[hh][i]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // The reference max moves only when a score exceeds it by more than
        // 2^8: every exponent argument stays <= 8, so P <= 256 (exact in bf16
        // range, no fp32 overflow), and O and l share the same reference, so
        // O / l is unchanged.  Most tiles then skip the 64 rescales.
        const float m_cand = fmaxf(m_run, mx * sc);
        const bool move = m_cand > m_run + 8.0f;
        if (__builtin_amdgcn_ballot_w64(move)) {
            const float m_new = move ? m_cand : m_run;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[tt][e] *= alpha;
            m_run = m_new;
        }
        const float m_new = m_run;
        float psum = 0.f;
        bf16x8_t pf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                float p2[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int i = 8 * (j & 1) + e + u;
                    float arg = __builtin_fmaf(sacc[j >> 1][i], sc, -m_new);
                    if (MASK && kv0 + 32 * (j >> 1) + 8 * (i >> 2) + 4 * g + (i & 3) >= a.seq_kv) arg = -INFINITY;
                    p2[u] = __builtin_amdgcn_exp2f(arg);
                    psum += p2[u];
                }
                const uint32_t pk = pack_bf16x2(p2[0], p2[1]);
                pf[j][e] = __builtin_bit_cast(__bf16, (uint16_t)(pk & 0xFFFFu));
                pf[j][e + 1] = __builtin_bit_cast(__bf16, (uint16_t)(pk >> 16));
            }
        }
        l_run += psum;

        // O^T[d][q] += V^T[d][key] P^T[key][q]: MFMA j covers keys 16 j ..;
        // lane half g supplies keys {16 j + 4 g + e, 16 j + 8 + 4 g + e}.
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const uint2 lo = read_tr16(Vt_ + 16 * j * DROW + voff[tt]);
                const uint2 hi = read_tr16(Vt_ + (16 * j + 8) * DROW + voff[tt]);
                const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
                o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[j], o[tt], 0, 0, 0);
            }
        }
    };

    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    using Full = std::integral_constant<bool, false>;
    using Part = std::integral_constant<bool, true>;
    // Full tiles in pairs (the buffer of each is then a constant), then the
    // last tile, masked when seq_kv is not a multiple of the tile.
    const int nfull = a.seq_kv / DKB;
    issue(0, 0);
    if constexpr (PRO) {
        // q goes through the second K/V buffer, still idle while the first
        // tile's DMA (above) is in flight: wave w's rows at [32 w, 32 w +
        // 32) x 256 B.  Every wave has read its rows back before the
        // barrier, and the buffer's first DMA comes after it.
        uint8_t* rows = smem + 2 * DTILE + 32 * wave * DROW;
        q_prologue16<8>(pro, b, h, q0, lane >> 4, a.seq_q, lane & 15, rows);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's rows are in LDS
#pragma unroll
        for (int c = 0; c < 8; ++c)
            qf[c] = *reinterpret_cast<const bf16x8_t*>(rows + r * DROW + (((2 * c + g) ^ (r & 15)) << 4));
        __syncthreads();
    }
    int t = 0;
    for (; t + 1 < nfull; t += 2) {
        tile(t, B0{}, Full{});
        tile(t + 1, B1{}, Full{});
    }
    if (t < nfull) {
        tile(t, B0{}, Full{});
        ++t;
        if (t < ntiles) tile(t, B1{}, Part{});
    } else if (t < ntiles) {
        tile(t, B0{}, Part{});
    }

    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const float inv = 1.0f / l_tot;
    const int q = q0 + r;
    if (q < a.seq_q) {
        TO* op = reinterpret_cast<TO*>(a.o) + b * a.os[0] + (int64_t)q * a.os[1] + h * a.os[2];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const int d = 32 * tt + 8 * i4 + 4 * g;
                float v4[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v4[e] = o[tt][4 * i4 + e] * inv;
                if constexpr (sizeof(TO) == 4) {
                    *reinterpret_cast<float4*>(reinterpret_cast<float*>(op) + d) =
                        make_float4(v4[0], v4[1], v4[2], v4[3]);
                } else {
                    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(op) + d) =
                        make_uint2(pack_bf16x2(v4[0], v4[1]), pack_bf16x2(v4[2], v4[3]));
                }
            }
    }
}

// ---- few query blocks: 32 queries per workgroup, keys over its waves -------------
// With blocks of 128 queries a short sequence or few heads leave most CUs idle (24
// heads of 320 tokens: 72 workgroups), and each then walks all keys by itself.  Here
// a workgroup takes 32 queries and each of its four waves every fourth 32-key tile, from
// K and V buffers of its own (8 KB each): a wave waits only for its own DMA and there
// is no barrier until the four partial results meet in LDS.  K of the wave's next
// tile loads from the end of its scores on, V from the end of P V on.  The
// products, the softmax and its moving reference are flash_attn_dma_kernel's: every
// wave starts from the largest score of keys 0-63, so P is rounded to bf16 at the
// scale that kernel rounds it at (waves starting from their own first tile's differed from
// it by 2.7e-3 in the 2-norm, all of it that rounding).  A reference that
// is still -inf (every score so far -inf) gives its keys weight 0, not exp2(-inf + inf).
// Kernel time (launches in one HIP graph), against blocks of 128: 24 heads of 320 16.1
// -> 8.9 us, of 20 8.7 -> 6.0, 8 heads of 1000 28.8 -> 15.7, 2 of 2048 45 -> 23; past two
// workgroups per CU K and V are read too often (24 heads of 700, 528 workgroups: 24.8
// against 34.7, of 1000 31 against 43, with the older prologue's 4 us).  Eight waves a
// workgroup were slower (13.5 -> 15.8 us at 24 heads of 320).
constexpr int NW = 4, FQB = 32, FKB = 32, FTILE = FKB * DROW;  // waves; 8 KB

// The wave's 32 keys x 128 d of V as the V^T operands of both 16-key steps: lo, hi of
// block tt and step j at vf[j][tt].  The wait is in the block, so nothing reads
// the registers early; the compiler's own wait before its transposed reads would also
// drain the DMA in flight.
__device__ __forceinline__ void read_v_tile(uint32_t lds, const int (&voff)[4], bf16x8_t (&vf)[2][4]) {
    uint2 r[2][4][2];
    uint32_t at[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) at[tt] = lds + (uint32_t)voff[tt];
    asm volatile(
        "ds_read_b64_tr_b16 %0, %16\n\t"
        "ds_read_b64_tr_b16 %1, %16 offset:2048\n\t"
        "ds_read_b64_tr_b16 %2, %17\n\t"
        "ds_read_b64_tr_b16 %3, %17 offset:2048\n\t"
        "ds_read_b64_tr_b16 %4, %18\n\t"
        "ds_read_b64_tr_b16 %5, %18 offset:2048\n\t"
        "ds_read_b64_tr_b16 %6, %19\n\t"
        "ds_read_b64_tr_b16 %7, %19 offset:2048\n\t"
        "ds_read_b64_tr_b16 %8, %16 offset:4096\n\t"
        "ds_read_b64_tr_b16 %9, %16 offset:6144\n\t"
        "ds_read_b64_tr_b16 %10, %17 offset:4096\n\t"
        "ds_read_b64_tr_b16 %11, %17 offset:6144\n\t"
        "ds_read_b64_tr_b16 %12, %18 offset:4096\n\t"
        "ds_read_b64_tr_b16 %13, %18 offset:6144\n\t"
        "ds_read_b64_tr_b16 %14, %19 offset:4096\n\t"
        "ds_read_b64_tr_b16 %15, %19 offset:6144\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0][0][0]), "=&v"(r[0][0][1]), "=&v"(r[0][1][0]), "=&v"(r[0][1][1]), "=&v"(r[0][2][0]),
          "=&v"(r[0][2][1]), "=&v"(r[0][3][0]), "=&v"(r[0][3][1]), "=&v"(r[1][0][0]), "=&v"(r[1][0][1]),
          "=&v"(r[1][1][0]), "=&v"(r[1][1][1]), "=&v"(r[1][2][0]), "=&v"(r[1][2][1]), "=&v"(r[1][3][0]),
          "=&v"(r[1][3][1])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
        : "memory");
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
            vf[j][tt] = __builtin_bit_cast(bf16x8_t, make_uint4(r[j][tt][0].x, r[j][tt][0].y, r[j][tt][1].x, r[j][tt][1].y));
}

template <typename TO, bool PRO>
__global__ __launch_bounds__(256, 2) void flash_attn_few_kernel(AttnArgs a, AttnPro pro) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[NW * 2 * FTILE];  // [wave][K | V]
    __shared__ __attribute__((aligned(16))) uint8_t qrows[PRO ? FTILE : 16];
    __shared__ float ml[2][NW][FQB];
    __shared__ float first[2][FQB];  // per query: tile 0's and tile 1's largest scaled score
    uint32_t bid = blockIdx.x;
    const uint32_t nb = gridDim.x;
    if ((nb & 7u) == 0) bid = (bid & 7u) * (nb >> 3) + (bid >> 3);
    const int blocks = (a.seq_q + FQB - 1) / FQB;
    const int qblk = (int)(bid % (uint32_t)blocks), bh = (int)(bid / (uint32_t)blocks);
    const int h = bh % a.heads, b = bh / a.heads;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5, q = qblk * FQB + r;
    const uint16_t* Kp = a.k + b * a.ks[0] + h * a.ks[2];
    const uint16_t* Vp = a.v + b * a.vs[0] + h * a.vs[2];
    uint8_t* const Kt = smem + wave * 2 * FTILE;
    uint8_t* const Vt = Kt + FTILE;

    // DMA: eight instructions of 4 rows; rows past seq_kv load the last one.
    const int drow = lane >> 4, dpos = lane & 15;
    auto issue = [&](const uint16_t* src, int64_t ts, int t, uint8_t* buf, auto is_k) {
        const int k0 = t * FKB;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int row = 4 * j + drow, sw = decltype(is_k)::value ? kswz(row) : vswz(row);
            __builtin_amdgcn_global_load_lds(src + min(k0 + row, a.seq_kv - 1) * ts + (dpos ^ sw) * 8, buf + 4 * j * DROW,
                                             16, 0, 0);
        }
    };
    auto issue_k = [&](int t) { issue(Kp, a.ks[1], t, Kt, std::true_type{}); };
    auto issue_v = [&](int t) { issue(Vp, a.vs[1], t, Vt, std::false_type{}); };

    const int ntiles = (a.seq_kv + FKB - 1) / FKB;
    if (wave < ntiles) issue_k(wave);
    // Each wave prepares eight of the block's queries for all.
    bf16x8_t qf[8];
    if constexpr (PRO) {
        q_prologue16<FQB / (4 * NW)>(pro, b, h, qblk * FQB, (FQB / NW) * wave + (lane >> 4), a.seq_q, lane & 15, qrows);
        // Not __syncthreads: K's DMA stays in flight.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's rows are in LDS
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 8; ++c)
            qf[c] = *reinterpret_cast<const bf16x8_t*>(qrows + r * DROW + (((2 * c + g) ^ (r & 15)) << 4));
    } else {
        const uint16_t* Qp = a.q + b * a.qs[0] + h * a.qs[2];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            qf[c] = __builtin_bit_cast(bf16x8_t, q < a.seq_q ? ld16(Qp + (int64_t)q * a.qs[1] + 16 * c + 8 * g)
                                                             : make_uint4(0, 0, 0, 0));
    }
    if (wave < ntiles) issue_v(wave);

    int koff[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) koff[c] = r * DROW + (((2 * c + g) ^ (r & 15)) << 4);
    const int s16 = lane & 15, gi = lane >> 4, tg = gi >> 1, dsub = gi & 1;
    const int trow = s16 >> 2, tcol = 16 * dsub + 4 * (s16 & 3);
    int voff[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
        voff[tt] = (4 * tg + trow) * DROW + ((4 * (tt ^ trow) + (tcol >> 3)) << 4) + 8 * ((tcol >> 2) & 1);
    const uint32_t vlds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)Vt;

    f32x16_t o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const float sc = a.scale_log2;
    // Tile 0's and 1's maxima are in LDS.  Once per wave, whether or not it has a
    // tile; not __syncthreads: the DMA stays in flight.
    auto meet = [&]() {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's maxima are in LDS
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave >= ntiles) meet();
    for (int t = wave; t < ntiles; t += NW) {
        attn_wait_vm<8>();  // K (V's eight are younger)
        f32x16_t s[2];
#pragma unroll
        for (int e = 0; e < 16; ++e) s[0][e] = s[1][e] = 0.f;
        __builtin_amdgcn_sched_barrier(0);  // no LDS read before the wait
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(Kt + koff[c]);
            s[c & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], s[c & 1], 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): K read, its buffer is free
        __builtin_amdgcn_sched_barrier(0);
        const bool more = t + NW < ntiles;
        if (more) issue_k(t + NW);
        // Element i is key 32 t + 8 (i / 4) + 4 g + i % 4.
        const int left = a.seq_kv - t * FKB;
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[0][i] += s[1][i];
            if (8 * (i >> 2) + 4 * g + (i & 3) < left) mx = fmaxf(mx, s[0][i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (t == wave) {
            if (wave < 2 && g == 0) first[wave][r] = mx * sc;
            meet();
            m_run = ntiles > 1 ? fmaxf(first[0][r], first[1][r]) : first[0][r];
        }
        const float m_cand = fmaxf(m_run, mx * sc);
        const bool move = m_cand > m_run + 8.0f;
        if (__builtin_amdgcn_ballot_w64(move)) {
            const float m_new = move ? m_cand : m_run;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[tt][e] *= alpha;
            m_run = m_new;
        }
        const float m_sub = m_run == -INFINITY ? 0.f : m_run;
        float psum = 0.f;
        bf16x8_t pf[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t pk[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                float p2[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int i = 8 * j + e + u;
                    float arg = __builtin_fmaf(s[0][i], sc, -m_sub);
                    if (8 * (i >> 2) + 4 * g + (i & 3) >= left) arg = -INFINITY;
                    p2[u] = __builtin_amdgcn_exp2f(arg);
                    psum += p2[u];
                }
                pk[e / 2] = pack_bf16x2(p2[0], p2[1]);
            }
            pf[j] = __builtin_bit_cast(bf16x8_t, make_uint4(pk[0], pk[1], pk[2], pk[3]));
        }
        l_run += psum;
        if (more) attn_wait_vm<8>();  // V (K's next eight are younger)
        else attn_wait_vm<0>();
        bf16x8_t vf[2][4];
        read_v_tile(vlds, voff, vf);
        if (more) issue_v(t + NW);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
                o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[j][tt], pf[j], o[tt], 0, 0, 0);
    }

    // The waves' results share the largest reference: O = sum w_i O_i / sum w_i l_i.
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (g == 0) {
        ml[0][wave][r] = m_run;
        ml[1][wave][r] = l_tot;
    }
    __syncthreads();
    float m = ml[0][0][r];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, ml[0][w][r]);
    const float mine = __builtin_amdgcn_exp2f(m_run - m);
    float* part = reinterpret_cast<float*>(smem);  // [wave][128 d][32 q]
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            part[wave * D * FQB + (32 * tt + 8 * (e >> 2) + 4 * g + (e & 3)) * FQB + r] = o[tt][e] * mine;
    __syncthreads();
    const int qq = qblk * FQB + r, d0 = (tid >> 5) * (64 / NW);
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) l += __builtin_amdgcn_exp2f(ml[0][w][r] - m) * ml[1][w][r];
    const float inv = 1.0f / l;
    if (qq < a.seq_q) {
        TO* op = reinterpret_cast<TO*>(a.o) + b * a.os[0] + (int64_t)qq * a.os[1] + h * a.os[2];
#pragma unroll
        for (int d = d0; d < d0 + 64 / NW; d += 4) {
            float v4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < NW; ++w) v += part[w * D * FQB + (d + e) * FQB + r];
                v4[e] = v * inv;
            }
            if constexpr (sizeof(TO) == 4)
                *reinterpret_cast<float4*>(reinterpret_cast<float*>(op) + d) = make_float4(v4[0], v4[1], v4[2], v4[3]);
            else
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(op) + d) =
                    make_uint2(pack_bf16x2(v4[0], v4[1]), pack_bf16x2(v4[2], v4[3]));
        }
    }
}

}  // namespace
}  // namespace dit

namespace dit {
namespace {

// Shared checks of k, v, o, the sizes and the strides; q and its strides are
// checked only when given (the prologue takes its own).
int attn_prepare(const void* q, const void* k, const void* v, void* o, int64_t batch, int64_t heads,
                 int64_t seq_q, int64_t seq_kv, int64_t head_dim, const int64_t* q_strides,
                 const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides, float scale,
                 int32_t o_type, const char* who, AttnArgs* out) {
    DT_REQUIRE(head_dim == D, "%s: head_dim %lld unsupported (128 only)", who, (long long)head_dim);
    DT_REQUIRE(o_type == DT_TYPE_BF16 || o_type == DT_TYPE_F32, "%s: o_type %d unsupported", who, o_type);
    DT_REQUIRE(batch >= 0 && heads >= 0 && seq_q >= 0 && seq_kv >= 0, "%s: negative size", who);
    DT_REQUIRE(seq_kv > 0 || batch == 0 || heads == 0 || seq_q == 0, "%s: seq_kv must be positive", who);
    DT_REQUIRE(k && v && o && k_strides && v_strides && o_strides && (!q || q_strides), "%s: null pointer", who);
    DT_REQUIRE(seq_q < (1ll << 30) && seq_kv < (1ll << 30) && heads < (1 << 20) && batch < (1 << 20),
               "%s: size too large", who);
    AttnArgs a{};
    a.q = (const uint16_t*)q;
    a.k = (const uint16_t*)k;
    a.v = (const uint16_t*)v;
    a.o = o;
    for (int i = 0; i < 3; ++i) {
        a.qs[i] = q ? q_strides[i] : 0;
        a.ks[i] = k_strides[i];
        a.vs[i] = v_strides[i];
        a.os[i] = o_strides[i];
        DT_REQUIRE(a.qs[i] % 8 == 0 && a.ks[i] % 8 == 0 && a.vs[i] % 8 == 0 && a.os[i] % 4 == 0,
                   "%s: strides must keep rows 16-byte aligned", who);
    }
    DT_REQUIRE((!q || aligned16(q)) && aligned16(k) && aligned16(v) && aligned16(o),
               "%s: pointers must be 16-byte aligned", who);
    a.batch = (int32_t)batch;
    a.heads = (int32_t)heads;
    a.seq_q = (int32_t)seq_q;
    a.seq_kv = (int32_t)seq_kv;
    a.q_blocks = (int32_t)((seq_q + QB - 1) / QB);
    DT_REQUIRE(scale >= 0.f, "%s: scale must be >= 0 (got %g)", who, (double)scale);
    a.scale_log2 = scale * 1.4426950408889634f;
    DT_REQUIRE((int64_t)a.q_blocks * heads * batch < (1ll << 31), "%s: grid too large", who);
    *out = a;
    return DT_OK;
}

template <bool PRO>
int attn_launch(const AttnArgs& a, const AttnPro& pro, int32_t o_type, hipStream_t st, const char* who) {
    const int64_t blocks = (int64_t)a.q_blocks * a.heads * a.batch;
    const unsigned nblocks = (unsigned)blocks;
    if (nblocks == 0) return DT_OK;
    // Blocks of 32 queries while two per CU hold them all (see the kernel).
    const int64_t few = (int64_t)((a.seq_q + FQB - 1) / FQB) * a.heads * a.batch;
    if (few <= 2 * cu_count()) {
        const dim3 grid((unsigned)few);
        const bool f32 = o_type == DT_TYPE_F32;
        if (f32) hipLaunchKernelGGL((flash_attn_few_kernel<float, PRO>), grid, dim3(64 * NW), 0, st, a, pro);
        else hipLaunchKernelGGL((flash_attn_few_kernel<uint16_t, PRO>), grid, dim3(64 * NW), 0, st, a, pro);
        return check_launch(who);
    }
    if (o_type == DT_TYPE_F32)
        hipLaunchKernelGGL((flash_attn_dma_kernel<float, PRO>), dim3(nblocks), dim3(256), 0, st, a, pro);
    else
        hipLaunchKernelGGL((flash_attn_dma_kernel<uint16_t, PRO>), dim3(nblocks), dim3(256), 0, st, a, pro);
    return check_launch(who);
}

}  // namespace

int flash_attn_qk_launch(const AttnQk& qk, const void* k, const void* v, void* o, int64_t batch, int64_t heads,
                         int64_t seq_q, int64_t seq_kv, const int64_t* k_strides, const int64_t* v_strides,
                         const int64_t* o_strides, float scale, int32_t o_type, hipStream_t st) {
    const char* who = "dt_flash_attn_qk_bf16";
    AttnArgs a;
    int rc = attn_prepare(nullptr, k, v, o, batch, heads, seq_q, seq_kv, D, nullptr, k_strides, v_strides,
                          o_strides, scale, o_type, who, &a);
    if (rc || a.q_blocks == 0 || heads == 0 || batch == 0) return rc;
    DT_REQUIRE(qk.n_axes > 0 && qk.n_axes <= kMaxRopeAxes && qk.axis_dim > 0 && qk.axis_dim % 8 == 0 &&
                   qk.n_axes * qk.axis_dim == D,
               "%s: need n_axes <= %d, axis_dim %% 8 == 0 and n_axes * axis_dim == 128 (%d * %d)", who,
               kMaxRopeAxes, qk.n_axes, qk.axis_dim);
    DT_REQUIRE(qk.split >= 0, "%s: split < 0", who);
    const bool two = qk.split < seq_q;
    DT_REQUIRE(qk.q[0] && qk.w[0] && (!two || (qk.q[1] && qk.w[1])), "%s: null q or norm weight", who);
    for (int sgi = 0; sgi < (two ? 2 : 1); ++sgi) {
        DT_REQUIRE(aligned16(qk.q[sgi]) && aligned16(qk.w[sgi]), "%s: q / weights must be 16-byte aligned", who);
        for (int i = 0; i < 3; ++i)
            DT_REQUIRE(qk.qs[sgi][i] % 8 == 0, "%s: q strides must keep rows 16-byte aligned", who);
    }
    for (int ax = 0; ax < qk.n_axes; ++ax)
        DT_REQUIRE(qk.pos.ptr[ax] != nullptr, "%s: null position pointer for axis %d", who, ax);
    DT_REQUIRE(!qk.table || (aligned16(qk.table) && qk.n_pos >= 0), "%s: rope table must be 16-byte aligned", who);
    AttnPro pro{};
    pro.q0 = (const uint16_t*)qk.q[0];
    pro.q0_bs = qk.qs[0][0];
    pro.q0_ts = qk.qs[0][1];
    pro.q0_hs = qk.qs[0][2];
    pro.w0 = qk.w[0];
    if (two) {
        pro.q1 = (const uint16_t*)qk.q[1];
        pro.q1_bs = qk.qs[1][0];
        pro.q1_ts = qk.qs[1][1];
        pro.q1_hs = qk.qs[1][2];
        pro.w1 = qk.w[1];
    }
    pro.split = (int32_t)std::min<int64_t>(qk.split, seq_q);
    pro.axis_dim = qk.axis_dim;
    pro.n_pos = qk.table ? qk.n_pos : 0;
    pro.theta_scale = powf(qk.freq_base, -2.0f / (float)qk.axis_dim);
    pro.eps = qk.eps;
    pro.table = qk.table;
    pro.pos = qk.pos;
    for (int ax = qk.n_axes; ax < kMaxRopeAxes; ++ax) {
        pro.pos.ptr[ax] = qk.pos.ptr[0];
        pro.pos.stride[ax] = qk.pos.stride[0];
    }
    a.q = pro.q0;
    return attn_launch<true>(a, pro, o_type, st, who);
}

}  // namespace dit

extern "C" int dt_flash_attn_bf16(const void* q, const void* k, const void* v, void* o, int64_t batch,
                                  int64_t heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim,
                                  const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                  const int64_t* o_strides, float scale, int32_t o_type, dt_stream_t stream) {
    using namespace dit;
    const char* who = "dt_flash_attn_bf16";
    DT_REQUIRE(head_dim == D, "%s: head_dim %lld unsupported (128 only)", who, (long long)head_dim);
    if (batch == 0 || heads == 0 || seq_q == 0) return DT_OK;
    DT_REQUIRE(q != nullptr, "%s: null pointer", who);
    AttnArgs a;
    int rc = attn_prepare(q, k, v, o, batch, heads, seq_q, seq_kv, head_dim, q_strides, k_strides, v_strides,
                          o_strides, scale, o_type, who, &a);
    if (rc) return rc;
    return attn_launch<false>(a, AttnPro{}, o_type, (hipStream_t)stream, who);
}

extern "C" int dt_flash_attn_qk_bf16(const void* q0, const int64_t* q0_strides, const float* w0, const void* q1,
                                     const int64_t* q1_strides, const float* w1, int64_t split, float eps,
                                     const int32_t* pos, int64_t pos_stride, int32_t n_axes, int32_t axis_dim,
                                     float freq_base, const float* rope_table, int32_t n_pos, const void* k,
                                     const void* v, void* o, int64_t batch, int64_t heads, int64_t seq_q,
                                     int64_t seq_kv, int64_t head_dim, const int64_t* k_strides,
                                     const int64_t* v_strides, const int64_t* o_strides, float scale,
                                     int32_t o_type, dt_stream_t stream) {
    using namespace dit;
    const char* who = "dt_flash_attn_qk_bf16";
    DT_REQUIRE(head_dim == D, "%s: head_dim %lld unsupported (128 only)", who, (long long)head_dim);
    if (batch == 0 || heads == 0 || seq_q == 0) return DT_OK;
    DT_REQUIRE(q0_strides && (split >= seq_q || q1_strides), "%s: null q strides", who);
    DT_REQUIRE(pos != nullptr && pos_stride >= n_axes && n_axes > 0 && n_axes <= kMaxRopeAxes,
               "%s: bad positions (pos_stride %lld, n_axes %d)", who, (long long)pos_stride, n_axes);
    AttnQk qk{};
    qk.q[0] = q0;
    qk.q[1] = q1;
    qk.w[0] = w0;
    qk.w[1] = w1;
    for (int i = 0; i < 3; ++i) {
        qk.qs[0][i] = q0_strides[i];
        qk.qs[1][i] = split < seq_q ? q1_strides[i] : 0;
    }
    qk.split = split;
    qk.eps = eps;
    for (int ax = 0; ax < n_axes; ++ax) {
        qk.pos.ptr[ax] = pos + ax;
        qk.pos.stride[ax] = pos_stride;
    }
    qk.n_axes = n_axes;
    qk.axis_dim = axis_dim;
    qk.freq_base = freq_base;
    qk.table = n_pos > 0 ? rope_table : nullptr;
    qk.n_pos = n_pos;
    return flash_attn_qk_launch(qk, k, v, o, batch, heads, seq_q, seq_kv, k_strides, v_strides, o_strides, scale,
                                o_type, (hipStream_t)stream);
}
