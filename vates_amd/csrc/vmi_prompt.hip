// The decoder blocks on a prompt: full attention, Gated DeltaNet and the
// quantised projections over blocks of thousands of tokens at once
// (decode.prefill).  The reference feeds a prompt through its ordinary forward
// (mlx_streaming/mtp/generate.py:101-220, 470-520), as the verify kernels here
// would: eight tokens a pass, every weight read again for each eight (a
// 777-token prompt through two layers and the MTP layer: 34.2 ms).  Here
// the weights are read once per block and the matrix cores do the work.
//
//   k_pr_prep   a projection's input rows in MFMA operand order (RMSNorm
//               fused where there is one) and their group sums
//   k_pr_gemm   Y = X W^T for 4-bit W, exact operands, fp32 scales
//   k_pr_qkv    q and k RMSNorm and rotary; k and v into the cache
//   k_pr_flash  causal attention over the cache, online softmax
//   k_pr_conv   causal conv, SiLU, q/k normalisation and gates of the delta rule
//   k_pr_wy     per 16 tokens and value head, what their delta rule needs beside
//               the state: a 16 x 16 triangular inverse, q k products, decays
//   k_pr_chunk  the delta rule 16 tokens at a time, fp32 MFMAs
//   k_pr_scan   the delta rule token by token, fp32, one state row per 16
//               lanes: short blocks, and the last tokens of others
//   k_pr_gnorm  the gated RMSNorm, written as the out projection's operand

#include <climits>

#include "vmi_attn_device.h"
#include "vmi_internal.h"

namespace {

constexpr int kPrThreads = 256;
constexpr int kGHead = 128;     // Gated DeltaNet head dims
constexpr int kConvRing = 32;   // conv ring rows (vmi_gdn_layer)
constexpr int kPrTokPad = 128;  // rows of the transposed group sums are padded to this

// Sum over the 8 lanes of an aligned group, in every lane of it.
__device__ __forceinline__ float sum8(float v) {
    v += vmi_dpp_f32<VMI_DPP_XOR1>(v);
    v += vmi_dpp_f32<VMI_DPP_XOR2>(v);
    return v + vmi_dpp_f32<VMI_DPP_HALF_MIRROR>(v);
}

__device__ __forceinline__ float sum_bf16x8(const vmi_u4& u) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += __uint_as_float(u[i] << 16) + __uint_as_float(u[i] & 0xffff0000u);
    return s;
}

// A projection's input: xop [T][K/8] 16-byte pieces of 8 columns in the slot
// order of vmi_unpack_u4_bf16_128, xneg [K/64][Tp] = -128 times the sum of each
// 64-column group (Tp = T rounded up to kPrTokPad).
struct PrOperand {
    vmi_u4* xop;
    float* xneg;
    int Tp;
};

// One wave per token: lane l holds pieces l, l + 64, ... (K = 512 NCH).
// Bound by the bytes of x.  limit (or null) is set to INT_MAX for the kernels
// behind this one.
template <int NCH>
__global__ __launch_bounds__(kPrThreads) void k_pr_prep(const uint16_t* x, const uint16_t* w, float eps, int T,
                                                         PrOperand o, int* limit) {
    constexpr int K = 512 * NCH;
    const int lane = threadIdx.x & 63, t = blockIdx.x * (kPrThreads / 64) + at_wave();
    if (limit && blockIdx.x == 0 && threadIdx.x == 0) *limit = INT_MAX;
    if (t >= T) return;
    const vmi_u4* row = reinterpret_cast<const vmi_u4*>(x + (size_t)t * K);
    vmi_u4 u[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) u[i] = row[lane + 64 * i];
    if (w) {
        const vmi_u4* wr = reinterpret_cast<const vmi_u4*>(w);
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NCH; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = __uint_as_float(u[i][e] << 16), b = __uint_as_float(u[i][e] & 0xffff0000u);
                ss = fmaf(a, a, ss);
                ss = fmaf(b, b, ss);
            }
        ss = vmi_wave_sum_canon(ss);
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(ss * (1.0f / (float)K) + eps));
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const vmi_u4 g = wr[lane + 64 * i];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                u[i][e] = vmi_pack_bf16x2((__uint_as_float(u[i][e] << 16) * inv) * __uint_as_float(g[e] << 16),
                                          (__uint_as_float(u[i][e] & 0xffff0000u) * inv) *
                                              __uint_as_float(g[e] & 0xffff0000u));
        }
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const uint4 q = qg_operand_order(u[i]);
        o.xop[(size_t)t * (K / 8) + lane + 64 * i] = vmi_u4{q.x, q.y, q.z, q.w};
        const float s = sum8(sum_bf16x8(u[i]));
        if ((lane & 7) == 0) o.xneg[(size_t)((lane >> 3) + 8 * i) * o.Tp + t] = -128.0f * s;
    }
}

// ------------------------------------------------------------------- GEMM
struct PrGemm {
    PrOperand x;
    int T, K;
    vmi_qmat m[3];             // up to three matrices stacked along the output rows
    int rows[3], nrows;
    float* out;                // [T, out_stride], or null
    int out_stride;
    const uint16_t* residual;  // [T, out_stride] bf16, or null
    uint16_t* out_bf16;        // bf16(y + residual), or null
};

// Y[t][n] = sum_k x[t][k] (q s + b)[n][k], exact operands: bf16 x against
// bf16 128 + q, the group's MFMAs starting from C = -128 sum(x) so that D is
// sum(q x); the group's scale enters by one fp32 FMA per output, and the bias
// term sum_g b_g sum(x)_g by bf16 MFMAs on a three-way split of the sums (24
// bits), 8 groups each.  A workgroup of 2 x WN waves covers 32 WT tokens x
// 16 NT WN rows, a wave 16 WT x 16 NT: one unpacked weight operand feeds WT
// MFMAs, one x operand NT.  A stage is two groups (128 columns) of x and of the
// packed weights, moved by DMA into a ring of NS slots, NS - 1 stages
// ahead; the scales come eight groups (four stages) at a time.
//   x rows: 256 bytes, 16-byte piece c at c ^ (row & 15)
//   weight rows: 64 bytes, piece c at c ^ ((row >> 2) & 3), so that the 8-byte
//   reads of 16 rows cover the banks once
// Bound by VALU and MFMA work together (per group and wave: 4 WT NT scale
// FMAs and 14 NT unpack operations beside 2 WT NT MFMAs; 12,352 x 2048 ran
// its matrix cores 32 % and its VALU 49 % of the time, LDS 20 %; wave priorities or
// a forced interleaving of the two moved nothing).  With the weights loaded straight to
// registers, 8 bytes a lane from 16 rows, and one stage ahead, the same tiles waited
// for memory: 777 tokens, 12,352 x 2048: 98 -> 73 us, 9216 x 2048: 68 -> 47,
// 2048 x 4096: 73 -> 33, 1024 x 2048: 37 -> 12.
template <int WT_, int NT_, int WN_, int NS_>
struct PrShape {
    static constexpr int WT = WT_, NT = NT_, WN = WN_, NS = NS_;
    static constexpr int NW = 2 * WN, Threads = 64 * NW;
    static constexpr int TM = 32 * WT, TN = 16 * NT * WN;
    static constexpr int kX = TM * 256, kS = 2 * TM * 4, kW = TN * 64, kStage = kX + kS + kW;
    static constexpr int kScale = 16 * (TN < 64 ? 64 : TN);
    static constexpr int kLds = NS * kStage + 2 * kScale;
    // DMA instructions per wave and stage: x, weights, group sums
    static constexpr int NX = TM / 4 / NW, NWt = (TN / 16 + NW - 1) / NW;
    static constexpr int kIssue = NX + NWt + 1;
    static_assert(TM % (4 * NW) == 0 && kLds <= 163840, "tile");
    static_assert(TN / 16 >= NW ? (TN / 16) % NW == 0 : NW % (TN / 16) == 0, "weight pieces");
    static_assert(NS >= 3 && (NS - 2) * kIssue + (NS + 1) / 4 + 1 <= 63, "vmcnt");
};

// Output row n of the stacked matrices: which one, and its row there.
__device__ __forceinline__ int pr_row(const PrGemm& a, int n, int& mi) {
    int r = min(n, a.nrows - 1);
    mi = 0;
    if (r >= a.rows[0]) {
        r -= a.rows[0];
        mi = 1;
        if (r >= a.rows[1]) {
            r -= a.rows[1];
            mi = 2;
        }
    }
    return r;
}

template <class P>
__global__ __launch_bounds__(P::Threads, 2) void k_pr_gemm(PrGemm a) {
    constexpr int WT = P::WT, NT = P::NT, NS = P::NS, TM = P::TM, TN = P::TN, NW = P::NW;
    __shared__ __attribute__((aligned(16))) uint8_t s_ring[P::kLds];
    uint8_t* const s_scale = s_ring + NS * P::kStage;
    const int lane = threadIdx.x & 63, w = at_wave(), nl = lane & 15, q4 = lane >> 4;
    // the XCDs take equal runs of the tiles, token tiles innermost: a run's
    // weights reach its L2 once (workgroups are dealt to the 8 XCDs in turn)
    const int ty = (a.T + TM - 1) / TM, tiles = ty * ((a.nrows + TN - 1) / TN);
    const int tile = ((int)blockIdx.x & 7) * ((int)gridDim.x >> 3) + ((int)blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int t0 = (tile % ty) * TM, n0 = (tile / ty) * TN;
    const int wt = w & 1, wn = w >> 1;
    const int KC = a.K / 8, S = a.K / 128;
    // x: 4 rows per wave and instruction; tokens past T read the last row
    const vmi_u4* xsrc[P::NX];
#pragma unroll
    for (int j = 0; j < P::NX; ++j) {
        const int row = 4 * (NW * j + w) + q4;
        xsrc[j] = a.x.xop + (size_t)min(t0 + row, a.T - 1) * KC + ((lane & 15) ^ (row & 15));
    }
    // weights: 16 rows per instruction; rows past the end read the last one
    const vmi_u4* wsrc[P::NWt];
    int wpos[P::NWt];
#pragma unroll
    for (int j = 0; j < P::NWt; ++j) {
        wpos[j] = (NW * j + w) % (TN / 16);
        const int row = 16 * wpos[j] + (lane >> 2);
        int mi;
        const int r = pr_row(a, n0 + row, mi);
        const uint32_t* W = mi == 0 ? a.m[0].w : mi == 1 ? a.m[1].w : a.m[2].w;
        wsrc[j] = reinterpret_cast<const vmi_u4*>(W + (size_t)r * KC) + ((lane & 3) ^ ((row >> 2) & 3));
    }
    // scales: 64 rows per instruction (waves past the last piece repeat one)
    const int zpiece = w % (TN < 64 ? 1 : TN / 64);
    const uint16_t* zsrc;
    {
        int mi;
        const int r = pr_row(a, n0 + (64 * zpiece + lane) % TN, mi);
        zsrc = (mi == 0 ? a.m[0].s : mi == 1 ? a.m[1].s : a.m[2].s) + (size_t)r * (a.K / 64);
    }
    // the two groups' sums: 2 TM floats in pieces of 64 (Tp covers the tile), repeated by the waves past them
    const int spiece = w % (2 * TM / 64), si = 64 * spiece + lane;
    const float* ssrc = a.x.xneg + (size_t)(si / TM) * a.x.Tp + t0 + si % TM;
    auto issue_scales = [&](int blk) {
        vmi_lds_dma16_opaque(zsrc + 8 * blk, s_scale + (blk & 1) * P::kScale + 1024 * zpiece);
    };
    auto issue = [&](int st, int slot) {
        uint8_t* L = s_ring + slot * P::kStage;
#pragma unroll
        for (int j = 0; j < P::NX; ++j) vmi_lds_dma16_opaque(xsrc[j] + 16 * st, L + 1024 * (NW * j + w));
#pragma unroll
        for (int j = 0; j < P::NWt; ++j) vmi_lds_dma16_opaque(wsrc[j] + 4 * st, L + P::kX + P::kS + 1024 * wpos[j]);
        vmi_lds_dma4_opaque(ssrc + (size_t)(2 * st) * a.x.Tp, L + P::kX + 256 * spiece);
    };
    vmi_f4 acc[WT][NT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[i][nt] = vmi_f4{0.f, 0.f, 0.f, 0.f};
    // past the last stage the ring keeps moving (the last stage again, into a slot nobody
    // reads), so that every wait counts the same
#pragma unroll
    for (int st = 0; st < NS - 1; ++st) {
        if (st % 4 == 0) issue_scales(min(st / 4, S / 4 - 1));
        issue(min(st, S - 1), st);
    }
    int slot = 0, fill = NS - 1;
    const int wrow = 16 * NT * wn + nl;
#pragma unroll 1
    for (int blk = 0; blk < S / 4; ++blk) {
        vmi_u4 sc[NT];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int st = 4 * blk + u;
            // the stages st + 1 .. st + NS - 2 may be in flight, and the scales issued with them
            constexpr int kN = (NS - 2) * P::kIssue;
            constexpr auto scales_in = [](int uu) {
                int n = 0;
                for (int k = 1; k <= NS - 2; ++k) n += (uu + k) % 4 == 0;
                return n;
            };
            if (u == 0) vmi_vm_wait_c<kN + scales_in(0)>();
            if (u == 1) vmi_vm_wait_c<kN + scales_in(1)>();
            if (u == 2) vmi_vm_wait_c<kN + scales_in(2)>();
            if (u == 3) vmi_vm_wait_c<kN + scales_in(3)>();
            __syncthreads();
            if ((u + NS - 1) % 4 == 0) issue_scales(min(blk + (u + NS - 1) / 4, S / 4 - 1));
            issue(min(st + NS - 1, S - 1), fill);
            const uint8_t* X = s_ring + slot * P::kStage;
            const uint8_t* W = X + P::kX + P::kS;
            slot = slot + 1 == NS ? 0 : slot + 1;
            fill = fill + 1 == NS ? 0 : fill + 1;
            if (u == 0) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    sc[nt] = *reinterpret_cast<const vmi_u4*>(s_scale + (blk & 1) * P::kScale + 16 * (wrow + 16 * nt));
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                vmi_u4 xa[WT][2];
                vmi_f4 c0[WT];
                uint2 wq[NT];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const int r = wrow + 16 * nt, c = 2 * g + (q4 >> 1);
                    wq[nt] = *reinterpret_cast<const uint2*>(W + r * 64 + 16 * (c ^ ((r >> 2) & 3)) + 8 * (q4 & 1));
                }
#pragma unroll
                for (int i = 0; i < WT; ++i) {
                    const int row = 16 * (WT * wt + i) + nl, p = 8 * g + 2 * q4;
                    xa[i][0] = *reinterpret_cast<const vmi_u4*>(X + row * 256 + 16 * (p ^ (row & 15)));
                    xa[i][1] = *reinterpret_cast<const vmi_u4*>(X + row * 256 + 16 * ((p + 1) ^ (row & 15)));
                    c0[i] = *reinterpret_cast<const vmi_f4*>(X + P::kX + 4 * (g * TM + 16 * (WT * wt + i) + 4 * q4));
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const vmi_u4 b0 = vmi_unpack_u4_bf16_128(wq[nt].x), b1 = vmi_unpack_u4_bf16_128(wq[nt].y);
                    const float s = __uint_as_float(g ? (sc[nt][u] & 0xffff0000u) : (sc[nt][u] << 16));
                    vmi_f4 d[WT];
#pragma unroll
                    for (int i = 0; i < WT; ++i) d[i] = vmi_mfma_bf16(xa[i][0], b0, c0[i]);
#pragma unroll
                    for (int i = 0; i < WT; ++i) d[i] = vmi_mfma_bf16(xa[i][1], b1, d[i]);
#pragma unroll
                    for (int i = 0; i < WT; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][nt][e] = fmaf(s, d[i][e], acc[i][nt][e]);
                }
            }
        }
    }
    vmi_vm_wait_c<0>();  // no DMA may outlive the workgroup's LDS
    // the bias term, 8 groups per MFMA (lane block q4 carries groups 8 c + 2 q4 and + 1), the
    // operands of up to four of them requested together
    const uint16_t* brow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        int mi;
        const int r = pr_row(a, n0 + wrow + 16 * nt, mi);
        brow[nt] = (mi == 0 ? a.m[0].b : mi == 1 ? a.m[1].b : a.m[2].b) + (size_t)r * (a.K / 64) + 2 * q4;
    }
    const int nc = a.K / 512;
#pragma unroll 1
    for (int c0 = 0; c0 < nc; c0 += 4) {
        float xs[4][WT][2];
        uint32_t bs[4][NT];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = min(c0 + j, nc - 1);
            const float* x0 = a.x.xneg + (size_t)(8 * c + 2 * q4) * a.x.Tp + t0 + 16 * WT * wt + nl;
#pragma unroll
            for (int i = 0; i < WT; ++i) {
                xs[j][i][0] = x0[16 * i];
                xs[j][i][1] = x0[a.x.Tp + 16 * i];
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) bs[j][nt] = *reinterpret_cast<const uint32_t*>(brow[nt] + 8 * c);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (c0 + j >= nc) break;
            vmi_u4 ab[WT];
#pragma unroll
            for (int i = 0; i < WT; ++i) ab[i] = vmi_bias_a_operand(xs[j][i][0] * -0.0078125f, xs[j][i][1] * -0.0078125f);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const vmi_u4 bb = vmi_bias_b_operand(bs[j][nt]);
#pragma unroll
                for (int i = 0; i < WT; ++i) acc[i][nt] = vmi_mfma_bf16(ab[i], bb, acc[i][nt]);
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + wrow + 16 * nt;
        if (n >= a.nrows) continue;
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = t0 + 16 * (WT * wt + i) + 4 * q4 + e;
                if (t >= a.T) continue;
                const size_t at = (size_t)t * a.out_stride + n;
                if (a.out) a.out[at] = acc[i][nt][e];
                if (a.out_bf16)
                    a.out_bf16[at] =
                        vmi_f32_to_bf16(acc[i][nt][e] + (a.residual ? vmi_bf16_to_f32(a.residual[at]) : 0.0f));
            }
    }
}

// -------------------------------------------------------------- attention
struct PrAttn {
    const float* qkv;         // [T, stride]: q | gate per head, then k, then v
    int stride, T, n_heads, n_kv, pos0, max_len;
    int h0;                   // first head k_pr_qkv forms (0, or n_heads: keys and values only)
    const uint16_t *q_norm, *k_norm;
    int rope_dim;
    float eps;
    double rope_base;
    uint16_t *k_cache, *v_cache;
    uint16_t* q;              // [n_kv][T G][256] bf16 query rows, row t G + j of head g G + j
    uint16_t* o;              // [T][n_heads * 256] bf16 gated attention output
    int* limit;               // first position of the call whose values hold an infinity or NaN (k_pr_qkv)
};

// One workgroup per token: the verify kernel's arithmetic (norm_rope_rows) on
// every q and k head; keys and values go to the cache at the token's position.
__global__ __launch_bounds__(kPrThreads) void k_pr_qkv(PrAttn a) {
    __shared__ float s_row[kPrThreads / 64][kHeadDim];
    __shared__ float2 s_cs[kHeadDim / 2];
    const int t = blockIdx.x, lane = threadIdx.x & 63, w = at_wave(), pos = a.pos0 + t;
    if ((int)threadIdx.x < a.rope_dim / 2) s_cs[threadIdx.x] = rotary_cs(pos, threadIdx.x, a.rope_base);
    __syncthreads();
    const float* row = a.qkv + (size_t)t * a.stride;
    const int G = a.n_heads / a.n_kv, kt = pos % VMI_KV_BLOCK;
    for (int hh = a.h0 + w; hh < a.n_heads + 2 * a.n_kv; hh += kPrThreads / 64) {
        const bool is_q = hh < a.n_heads, is_v = hh >= a.n_heads + a.n_kv;
        const int col = is_q ? hh * 2 * kHeadDim : a.n_heads * 2 * kHeadDim + (hh - a.n_heads) * kHeadDim;
        float v[1][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[0][j] = row[col + lane + 64 * j];
        if (is_v) {
            const int g = hh - a.n_heads - a.n_kv;
            uint16_t* dst = a.v_cache + vmi_kv_block(g, a.max_len, pos);
            bool bad = false;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint16_t b = vmi_f32_to_bf16(v[0][j]);
                bad = bad || (b & 0x7f80u) == 0x7f80u;
                dst[vmi_v_elem(kt, lane + 64 * j)] = b;
            }
            if (__any(bad) && lane == 0) atomicMin(a.limit, pos);
            continue;
        }
        const uint16_t* nw = is_q ? a.q_norm : a.k_norm;
        float nf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) nf[j] = vmi_bf16_to_f32(nw[lane + 64 * j]);
        const float2* cs[1] = {s_cs};
        uint16_t o[1][4];
        norm_rope_rows<1>(v, nf, a.eps, cs, a.rope_dim, s_row[w], o);
        if (is_q) {
            uint16_t* dst = a.q + ((size_t)(hh / G) * a.T * G + (size_t)t * G + hh % G) * kHeadDim;
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[lane + 64 * j] = o[0][j];
        } else {
            uint16_t* dst = a.k_cache + vmi_kv_block(hh - a.n_heads, a.max_len, pos);
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[vmi_k_elem(kt, lane + 64 * j)] = o[0][j];
        }
    }
}

// grid (tiles of 64 M query rows, n_kv), four waves of 16 M rows.  Per cache block
// of 32 positions (keys and values, 32 KB, DMA'd into one of two LDS slots
// in the cache's own operand order): S^T = K Q^T, so that a lane holds 8
// consecutive keys of one query; the online softmax (Milakov and Gimelshein, 2018) in registers (the running
// maximum is exact: a block that raises it rescales the sums); the bf16
// probabilities are then the B operand of O^T = V^T P^T as they stand, and
// every sum a lane holds belongs to its own query.  Late tiles, which see the
// most keys, start first.  M = 2: bound by LDS reads and MFMAs alike (a wave reads
// 32 KB per 64 MFMAs).  M = 1 where 128-row tiles leave
// CUs idle: 777 tokens, 98 workgroups 63.6 us, 196 of half the rows 45.5.
template <int M>
__global__ __launch_bounds__(kPrThreads, 2) void k_pr_flash(PrAttn a) {
    __shared__ vmi_u4 s_kv[2][2][16 * 64];  // [slot][keys, values]
    const int lane = threadIdx.x & 63, w = at_wave(), nl = lane & 15, q4 = lane >> 4;
    const int g = blockIdx.y, G = a.n_heads / a.n_kv, R = a.T * G;
    const int r0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * (64 * M) + 16 * M * w;
    const int last_row = min(r0 - 16 * M * w + 64 * M, R) - 1;
    const int nb = (a.pos0 + last_row / G) / VMI_KV_BLOCK + 1;
    const uint16_t* kc = a.k_cache + vmi_kv_block(g, a.max_len, 0);
    const uint16_t* vc = a.v_cache + vmi_kv_block(g, a.max_len, 0);
    auto issue = [&](int b, int u) {
        const uint16_t* ks = kc + (size_t)b * (VMI_KV_BLOCK * kHeadDim) + lane * 8;
        const uint16_t* vs = vc + (size_t)b * (VMI_KV_BLOCK * kHeadDim) + lane * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            vmi_lds_dma16_opaque(ks + (4 * j + w) * 512, &s_kv[u][0][(4 * j + w) * 64]);
            vmi_lds_dma16_opaque(vs + (4 * j + w) * 512, &s_kv[u][1][(4 * j + w) * 64]);
        }
    };
    issue(0, 0);
    vmi_u4 qb[M][8];
    int last[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int row = min(r0 + 16 * m + nl, R - 1);
        last[m] = a.pos0 + row / G;
        const uint16_t* qr = a.q + ((size_t)g * R + row) * kHeadDim + 8 * q4;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) qb[m][kk] = *reinterpret_cast<const vmi_u4*>(qr + 32 * kk);
    }
    const int first = a.pos0 + min(r0, R - 1) / G;  // the wave's earliest query position
    // values from here on count as zeros: stale ones past the last position, and a
    // block's own that are not finite, since their probability of 0 for an earlier query
    // would still give a NaN; the queries that do see those end as NaN by their sums
    const int limit = *a.limit, stop = min(a.pos0 + a.T, limit);
    vmi_f4 ot[M][16];
    float mx[M], ls[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        mx[m] = -INFINITY;
        ls[m] = 0.0f;
#pragma unroll
        for (int d = 0; d < 16; ++d) ot[m][d] = vmi_f4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 1
    for (int b = 0; b < nb; ++b) {
        vmi_vm_wait_c<0>();
        __syncthreads();
        if (b + 1 < nb) issue(b + 1, (b + 1) & 1);
        const vmi_u4* K = s_kv[b & 1][0];
        const vmi_u4* V = s_kv[b & 1][1];
        vmi_f4 s[M][2];
#pragma unroll
        for (int m = 0; m < M; ++m) s[m][0] = s[m][1] = vmi_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const vmi_u4 k0 = K[kk * 64 + lane], k1 = K[(8 + kk) * 64 + lane];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                s[m][0] = vmi_mfma_bf16(k0, qb[m][kk], s[m][0]);
                s[m][1] = vmi_mfma_bf16(k1, qb[m][kk], s[m][1]);
            }
        }
        const int p0 = VMI_KV_BLOCK * b + 8 * q4;
        const bool mask = VMI_KV_BLOCK * b + VMI_KV_BLOCK - 1 > first;  // wave-uniform
        vmi_u4 pb[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = s[m][e >> 2][e & 3] * 0.09016844005556021f;  // log2(e) / sqrt(256)
            if (mask) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = p0 + e <= last[m] ? x[e] : -INFINITY;
            }
            float bm = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float nm = fmaxf(mx[m], bm);  // finite from the first block on: every query sees position 0
            if (__any(nm > mx[m])) {
                const float f = __builtin_amdgcn_exp2f(mx[m] - nm);
                ls[m] *= f;
#pragma unroll
                for (int d = 0; d < 16; ++d)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ot[m][d][e] *= f;
                mx[m] = nm;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t u = vmi_pack_bf16x2(__builtin_amdgcn_exp2f(x[2 * i] - nm),
                                                   __builtin_amdgcn_exp2f(x[2 * i + 1] - nm));
                ls[m] += __uint_as_float(u << 16);
                ls[m] += __uint_as_float(u & 0xffff0000u);
                pb[m][i] = u;
            }
        }
        const bool tail = VMI_KV_BLOCK * (b + 1) > stop;
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            vmi_u4 v = V[d * 64 + lane];
            if (tail) v = keep_first(v, stop - p0);
#pragma unroll
            for (int m = 0; m < M; ++m) ot[m][d] = vmi_mfma_bf16(v, pb[m], ot[m][d]);
        }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        float l = ls[m];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        if (last[m] >= limit) l = __builtin_nanf("");
        const int row = r0 + 16 * m + nl;
        if (row >= R) continue;
        const int t = row / G, h = g * G + row % G;
        const float* gate = a.qkv + (size_t)t * a.stride + (size_t)h * 2 * kHeadDim + kHeadDim + 4 * q4;
        uint16_t* o = a.o + ((size_t)t * a.n_heads + h) * kHeadDim + 4 * q4;
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            const vmi_f4 z = *reinterpret_cast<const vmi_f4*>(gate + 16 * d);
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = ot[m][d][e] / l / (1.0f + expf(-z[e]));
            *reinterpret_cast<uint2*>(o + 16 * d) = make_uint2(vmi_pack_bf16x2(y[0], y[1]), vmi_pack_bf16x2(y[2], y[3]));
        }
    }
}

// ---------------------------------------------------------- Gated DeltaNet
struct PrGdn {
    int T, pos0, n_k, n_v, r, per_g, conv_dim, stride, n_slots;
    const float* proj;        // [T, stride]: n_k groups [q k v.. z..] | per group b.. a..
    const uint16_t* conv_w;   // [conv_dim][4]
    const float *A_log, *dt_bias;
    uint16_t* conv_ring;
    float* state_ring;
    float* c;                 // [T][conv_dim] conv outputs, q and k normalised
    float* gb;                // [T][n_v][2] (g, beta)
    float* y;                 // [T][n_v][128]
    float* wy;                // [t0 / 16][n_v][kWyFloats] (k_pr_wy)
    int t0;                   // tokens k_pr_chunk takes; k_pr_scan takes the others
    int* limit;               // first piece with an infinity or NaN (k_pr_wy): the scan takes over there
    const uint16_t* norm_w;
    float eps;
    PrOperand o;
};

// Projection column of head hd of the conv channels (q heads, k heads, v heads).
__device__ __forceinline__ int pr_src(const PrGdn& a, int hd) {
    if (hd < a.n_k) return hd * a.per_g;
    if (hd < 2 * a.n_k) return (hd - a.n_k) * a.per_g + kGHead;
    const int h = hd - 2 * a.n_k;
    return (h / a.r) * a.per_g + 2 * kGHead + (h % a.r) * kGHead;
}

__device__ __forceinline__ vmi_f4 bf16_round4(const vmi_f4& v) {
    const uint32_t a = vmi_pack_bf16x2(v[0], v[1]), b = vmi_pack_bf16x2(v[2], v[3]);
    return vmi_f4{__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u), __uint_as_float(b << 16),
                  __uint_as_float(b & 0xffff0000u)};
}

// grid (ceil(T / kConvTok), slices of 8 heads, then one slice of gates): a
// thread owns 4 channels and slides its window over kConvTok tokens, so each
// projection row is read 1 + 3 / kConvTok times.  Bound by those bytes.
constexpr int kConvTok = 8;
__global__ __launch_bounds__(kPrThreads) void k_pr_conv(PrGdn a) {
    const int tid = threadIdx.x, t0 = blockIdx.x * kConvTok, heads = 2 * a.n_k + a.n_v;
    if (blockIdx.y == gridDim.y - 1) {
        if (blockIdx.x == 0 && tid == 0) *a.limit = INT_MAX;
        for (int i = tid; i < kConvTok * a.n_v; i += kPrThreads) {
            const int t = t0 + i / a.n_v, h = i % a.n_v;
            if (t >= a.T) return;
            const float* p = a.proj + (size_t)t * a.stride + a.n_k * a.per_g + (h / a.r) * 2 * a.r + h % a.r;
            const float x = p[a.r] + a.dt_bias[h];
            const float sp = x > 30.0f ? x : log1pf(expf(x));
            *reinterpret_cast<float2*>(a.gb + ((size_t)t * a.n_v + h) * 2) =
                make_float2(expf(-expf(a.A_log[h]) * sp), 1.0f / (1.0f + expf(-p[0])));
        }
        return;
    }
    const int hd = blockIdx.y * 8 + (tid >> 5), ch = 4 * (tid & 31);
    if (hd >= heads) return;
    const int c = hd * kGHead + ch;
    const float* src = a.proj + pr_src(a, hd) + ch;
    float cw[4][4];  // [channel][tap]
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint2 u = *reinterpret_cast<const uint2*>(a.conv_w + (size_t)(c + e) * 4);
        cw[e][0] = __uint_as_float(u.x << 16);
        cw[e][1] = __uint_as_float(u.x & 0xffff0000u);
        cw[e][2] = __uint_as_float(u.y << 16);
        cw[e][3] = __uint_as_float(u.y & 0xffff0000u);
    }
    vmi_f4 win[3 + kConvTok];
#pragma unroll
    for (int i = 0; i < 3 + kConvTok; ++i) {
        const int t = t0 - 3 + i, p = a.pos0 + t;
        win[i] = vmi_f4{0.f, 0.f, 0.f, 0.f};
        if (t >= 0) {
            if (t < a.T) win[i] = bf16_round4(*reinterpret_cast<const vmi_f4*>(src + (size_t)t * a.stride));
        } else if (p >= 0) {
            const uint2 u = *reinterpret_cast<const uint2*>(a.conv_ring + (size_t)(p % kConvRing) * a.conv_dim + c);
            win[i] = vmi_f4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                            __uint_as_float(u.y & 0xffff0000u)};
        }
    }
    const bool norm = hd < 2 * a.n_k;
    const float scale = hd < a.n_k ? 1.0f / kGHead : 0.08838834764831845f;  // 1/128, 1/sqrt(128)
#pragma unroll
    for (int j = 0; j < kConvTok; ++j) {
        if (t0 + j >= a.T) break;
        vmi_f4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float acc = 0.0f;
#pragma unroll
            for (int tap = 0; tap < 4; ++tap) acc = fmaf(cw[e][tap], win[j + tap][e], acc);
            o[e] = acc / (1.0f + expf(-acc));
        }
        if (norm) {
            float ss = fmaf(o[0], o[0], fmaf(o[1], o[1], fmaf(o[2], o[2], o[3] * o[3])));
            ss = vmi_row_sum16(ss);
            ss += __shfl_xor(ss, 16);
            const float f = __fdiv_rn(1.0f, __fsqrt_rn(ss * (1.0f / kGHead) + 1e-6f)) * scale;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] *= f;
        }
        *reinterpret_cast<vmi_f4*>(a.c + (size_t)(t0 + j) * a.conv_dim + c) = o;
    }
}

// The delta rule by 16 tokens (C = 16), in the WY form (Bischof and Van Loan,
// 1987; for this rule Yang et al., "Parallelizing Linear Transformers with the Delta
// Rule over Sequence Length", 2024).  Within a piece, with S the state
// before it, g_t the decays, G_t = g_0 .. g_t and r(t, i) = g_{i+1} .. g_t:
//   delta = X diag(beta) (V - diag(G) K S^T),  X = (I + L)^-1,
//           L[t][i] = beta_t r(t, i) k_i.k_t  (i < t)
//   y     = diag(G) Q S^T + M delta,  M[t][i] = r(t, i) k_i.q_t  (i <= t)
//   S'    = G_C S + sum_t r(C - 1, t) delta_t k_t^T
// which is the recurrence with its sums in another order; every factor is a
// product of decays (never a quotient), and X's entries are those of products of
// the contractions I - beta k k^T, so nothing grows.  An infinity or NaN would reach
// earlier tokens of its piece through the products' zeros: the pieces stop
// before the first one that holds any, and k_pr_scan takes the rest.
// One record of k_pr_wy per (piece, value head): X diag(beta) [16][16], M
// [16][16], G[16], r(C - 1, t)[16].
constexpr int kWyTok = 16, kWyFloats = 2 * 256 + 2 * 16;
constexpr int kChunkMin = 336;

__device__ __forceinline__ vmi_f4 pr_mfma_f32(float a, float b, const vmi_f4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// One wave per (piece, value head): the Gram products by fp32 MFMAs (operand
// registers of K serve as both sides), then lane c solves column c of X.
// Bound by latency; 1536 waves at 777 tokens.
__global__ __launch_bounds__(kPrThreads) void k_pr_wy(PrGdn a) {
    __shared__ __attribute__((aligned(16))) float s_l[kPrThreads / 64][16][16];
    __shared__ float s_r[kPrThreads / 64][16][16];
    __shared__ float2 s_gb[kPrThreads / 64][16];
    const int lane = threadIdx.x & 63, w = at_wave(), nl = lane & 15, q4 = lane >> 4;
    const int h = (int)blockIdx.y * (kPrThreads / 64) + w, hk = h / a.r, t0 = blockIdx.x * kWyTok;
    float* out = a.wy + ((size_t)blockIdx.x * a.n_v + h) * kWyFloats;
    const float* kr = a.c + (size_t)(t0 + nl) * a.conv_dim + (a.n_k + hk) * kGHead + 4 * q4;
    const float* qr = a.c + (size_t)(t0 + nl) * a.conv_dim + hk * kGHead + 4 * q4;
    vmi_f4 k[8], q[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        k[b] = *reinterpret_cast<const vmi_f4*>(kr + 16 * b);
        q[b] = *reinterpret_cast<const vmi_f4*>(qr + 16 * b);
    }
    const float2 gb = *reinterpret_cast<const float2*>(a.gb + ((size_t)(t0 + nl) * a.n_v + h) * 2);
    if (lane < 16) s_gb[w][lane] = gb;
    {
        const float* vr = a.c + (size_t)(t0 + nl) * a.conv_dim + (2 * a.n_k + h) * kGHead + 4 * q4;
        float z = 0.0f * gb.x + 0.0f * gb.y;  // NaN where any is not finite
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const vmi_f4 v = *reinterpret_cast<const vmi_f4*>(vr + 16 * b);
#pragma unroll
            for (int e = 0; e < 4; ++e) z = fmaf(k[b][e], 0.0f, fmaf(q[b][e], 0.0f, fmaf(v[e], 0.0f, z)));
        }
        if (__any(z != z) && lane == 0) atomicMin(a.limit, (int)blockIdx.x);
    }
    // four sums each: shorter chains, and less rounding in every entry
    vmi_f4 kk4[4], qk4[4];  // [t = 4 q4 + e][i = nl]
#pragma unroll
    for (int e = 0; e < 4; ++e) kk4[e] = qk4[e] = vmi_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            kk4[e] = pr_mfma_f32(k[b][e], k[b][e], kk4[e]);
            qk4[e] = pr_mfma_f32(q[b][e], k[b][e], qk4[e]);
        }
    const vmi_f4 kk = (kk4[0] + kk4[1]) + (kk4[2] + kk4[3]), qk = (qk4[0] + qk4[1]) + (qk4[2] + qk4[3]);
    __syncthreads();
    float r = 0.0f, G = 1.0f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {  // column nl of r (every q4 writes the same values)
        const float g = s_gb[w][t].x;
        r = t == nl ? 1.0f : r * g;  // 0 above the diagonal
        G *= g;
        s_r[w][t][nl] = r;
        if (t == nl && q4 == 0) out[512 + t] = G;
    }
    if (q4 == 0) out[528 + nl] = r;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int t = 4 * q4 + e;
        const float rt = s_r[w][t][nl];
        s_l[w][t][nl] = nl < t ? s_gb[w][t].y * rt * kk[e] : 0.0f;
        out[256 + 16 * t + nl] = rt * qk[e];
    }
    __syncthreads();
    float x[16];
    const float beta = s_gb[w][nl].y;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < t; ++i) acc = fmaf(s_l[w][t][i], x[i], acc);
        x[t] = t == nl ? 1.0f : t < nl ? 0.0f : -acc;
        if ((t >> 2) == q4) out[16 * t + nl] = x[t] * beta;
    }
}

// A workgroup per 16 state rows (grid n_v * 8, as k_pr_scan's), wave w the
// state's columns 32 w .. + 31, kept transposed in MFMA result layout: lane (s = lane
// >> 4, n = lane & 15) holds S[row n][32 w + 16 b + 4 s + e], which is also the
// operand layout of K S^T and Q S^T with the contraction taken in that
// order, and the results of one product are the next one's operand as they
// stand.  Per piece and wave 16 MFMAs for the two products (their sums over the
// waves meet in LDS, one barrier), 4 for delta, 8 for the new state, and 4
// for y on the waves in turn.  Operands come straight to registers two pieces
// ahead.  Bound by that chain.
struct PrPiece {
    vmi_f4 k[2], q[2];      // [token n][32 w + 16 b + 4 s + e]
    float kt[2][4], v[4];   // k[token 4 s + e][32 w + 16 b + n]; v[token 4 s + e][row n]
    vmi_f4 x, m, G, rc;     // record rows n (columns 4 s + e); G, r(C - 1, .) of tokens 4 s + e
    float Gc;
};

__global__ __launch_bounds__(kPrThreads, 1) void k_pr_chunk(PrGdn a) {
    __shared__ vmi_f4 s_part[2][2][kPrThreads / 64][64];  // [piece parity][k, q][wave][lane]
    const int lane = threadIdx.x & 63, w = at_wave(), nl = lane & 15, q4 = lane >> 4;
    const int h = blockIdx.x % a.n_v, rg = blockIdx.x / a.n_v, hk = h / a.r;
    const int pieces = min(a.t0 / kWyTok, *a.limit), col = 32 * w;
    if (pieces == 0) return;
    const size_t slot_elems = (size_t)a.n_v * kGHead * kGHead;
    const size_t off = ((size_t)h * kGHead + 16 * rg + nl) * kGHead + col + 4 * q4;
    vmi_f4 S[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        S[b] = vmi_f4{0.f, 0.f, 0.f, 0.f};
        if (a.pos0 > 0)
            S[b] = *reinterpret_cast<const vmi_f4*>(a.state_ring + (size_t)(a.pos0 % a.n_slots) * slot_elems + off + 16 * b);
    }
    const float* kbase = a.c + (size_t)(a.n_k + hk) * kGHead + col;
    const float* qbase = a.c + (size_t)hk * kGHead + col;
    const float* vbase = a.c + (size_t)(2 * a.n_k + h) * kGHead + 16 * rg;
    auto load = [&](int c, PrPiece& p) {
        c = min(c, pieces - 1);
        const int t = c * kWyTok;
        const size_t row = (size_t)(t + nl) * a.conv_dim;
        const float* rec = a.wy + ((size_t)c * a.n_v + h) * kWyFloats;
#pragma unroll
        for (int b = 0; b < 2; ++b) p.k[b] = *reinterpret_cast<const vmi_f4*>(kbase + row + 16 * b + 4 * q4);
#pragma unroll
        for (int b = 0; b < 2; ++b) p.q[b] = *reinterpret_cast<const vmi_f4*>(qbase + row + 16 * b + 4 * q4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const size_t te = (size_t)(t + 4 * q4 + e) * a.conv_dim + nl;
            p.v[e] = vbase[te];
            p.kt[0][e] = kbase[te];
            p.kt[1][e] = kbase[te + 16];
        }
        p.x = *reinterpret_cast<const vmi_f4*>(rec + 16 * nl + 4 * q4);
        p.m = *reinterpret_cast<const vmi_f4*>(rec + 256 + 16 * nl + 4 * q4);
        p.G = *reinterpret_cast<const vmi_f4*>(rec + 512 + 4 * q4);
        p.rc = *reinterpret_cast<const vmi_f4*>(rec + 528 + 4 * q4);
        p.Gc = rec[512 + 15];
    };
    auto piece = [&](int c, const PrPiece& p) {
        vmi_f4 ks[2], qs[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            ks[b] = qs[b] = vmi_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) ks[b] = pr_mfma_f32(p.k[b][e], S[b][e], ks[b]);
        }
        vmi_f4(*part)[kPrThreads / 64][64] = s_part[c & 1];
        part[0][w][lane] = ks[0] + ks[1];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) qs[b] = pr_mfma_f32(p.q[b][e], S[b][e], qs[b]);
        part[1][w][lane] = qs[0] + qs[1];
        __syncthreads();
        const vmi_f4 sk = (part[0][0][lane] + part[0][1][lane]) + (part[0][2][lane] + part[0][3][lane]);
        vmi_f4 d = {0.f, 0.f, 0.f, 0.f};  // delta[token 4 s + e][row n]
#pragma unroll
        for (int e = 0; e < 4; ++e) d = pr_mfma_f32(p.x[e], fmaf(-p.G[e], sk[e], p.v[e]), d);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            S[b] *= p.Gc;
#pragma unroll
            for (int e = 0; e < 4; ++e) S[b] = pr_mfma_f32(p.kt[b][e], d[e] * p.rc[e], S[b]);
        }
        if ((c & 3) == w) {
            vmi_f4 y = (part[1][0][lane] + part[1][1][lane]) + (part[1][2][lane] + part[1][3][lane]);
            y *= p.G;
#pragma unroll
            for (int e = 0; e < 4; ++e) y = pr_mfma_f32(p.m[e], d[e], y);
            float* yo = a.y + ((size_t)(c * kWyTok + 4 * q4) * a.n_v + h) * kGHead + 16 * rg + nl;
#pragma unroll
            for (int e = 0; e < 4; ++e) yo[(size_t)e * a.n_v * kGHead] = y[e];
        }
    };
    PrPiece p[3];
    load(0, p[0]);
    asm volatile("" ::: "memory");  // in this order: the loop's waits count them
    load(1, p[1]);
    asm volatile("" ::: "memory");
    for (int c = 0; c < pieces; c += 3) {
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            if (c + u < pieces) {  // uniform
                load(c + u + 2, p[(u + 2) % 3]);
                asm volatile("" ::: "memory");
                piece(c + u, p[u]);
            }
        }
    }
    // the state k_pr_scan continues from: a slot that the last n_slots tokens, all its own, write again
    float* dst = a.state_ring + (size_t)((a.pos0 + kWyTok * pieces) % a.n_slots) * slot_elems + off;
#pragma unroll
    for (int b = 0; b < 2; ++b) *reinterpret_cast<vmi_f4*>(dst + 16 * b) = S[b];
}

// The delta rule from token t0 on, token by token.  A state row's recurrence touches no other row, so the rows
// go to workgroups of 16 (grid n_v * 8, head = index mod n_v: the eight
// workgroups of a head share an XCD's L2 where n_v is a multiple of 8), 16
// lanes a row, 8 dk a lane, and the tokens run in order: one wave per SIMD
// at 32 heads.  Bound by the chain of one token (product with k, row sum,
// update) and its issue; the inputs of 16 tokens at a time come through LDS,
// loaded a piece ahead.  The state after each of the last n_slots tokens
// goes to the ring, as a run of verify batches would leave it.
constexpr int kScanTok = 16;
__global__ __launch_bounds__(kPrThreads) void k_pr_scan(PrGdn a) {
    __shared__ float s_qk[2][kScanTok][2 * kGHead];
    __shared__ float s_v[2][kScanTok][16];
    __shared__ float2 s_gb[2][kScanTok];
    __shared__ float s_y[2][kScanTok][16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int h = blockIdx.x % a.n_v, rg = blockIdx.x / a.n_v, hk = h / a.r;
    // this workgroup's share of the conv ring: the block's last 32 inputs
    {
        const int n = min(a.T, kConvRing), per = (n * (a.conv_dim / 4) + (int)gridDim.x - 1) / (int)gridDim.x;
        const int i1 = min(((int)blockIdx.x + 1) * per, n * (a.conv_dim / 4));
        for (int i = blockIdx.x * per + tid; i < i1; i += kPrThreads) {
            const int t = a.T - n + i / (a.conv_dim / 4), c = 4 * (i % (a.conv_dim / 4));
            const vmi_f4 v = *reinterpret_cast<const vmi_f4*>(a.proj + (size_t)t * a.stride + pr_src(a, c / kGHead) + c % kGHead);
            *reinterpret_cast<uint2*>(a.conv_ring + (size_t)((a.pos0 + t) % kConvRing) * a.conv_dim + c) =
                make_uint2(vmi_pack_bf16x2(v[0], v[1]), vmi_pack_bf16x2(v[2], v[3]));
        }
    }
    const int begin = a.t0 ? kWyTok * min(*a.limit, a.t0 / kWyTok) : 0;
    const int lr = tid >> 4, row = 16 * rg + lr, d0 = 4 * (lane & 15);
    const size_t slot_elems = (size_t)a.n_v * kGHead * kGHead;
    const size_t off = ((size_t)h * kGHead + row) * kGHead + d0;
    float S[8];
    {
        const int pos = a.pos0 + begin;
        const float* src = a.state_ring + (size_t)(pos % a.n_slots) * slot_elems + off;
#pragma unroll
        for (int i = 0; i < 8; ++i) S[i] = pos > 0 ? src[(i & 3) + (i >> 2) * 64] : 0.0f;
    }
    vmi_f4 rqk[4];
    float rv;
    float2 rgb;
    auto load = [&](int t0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = min(t0 + 4 * j + (tid >> 6), a.T - 1), c4 = tid & 63;
            const int head = c4 < 32 ? hk : a.n_k + hk;
            rqk[j] = *reinterpret_cast<const vmi_f4*>(a.c + (size_t)t * a.conv_dim + head * kGHead + 4 * (c4 & 31));
        }
        const int t = min(t0 + (tid >> 4), a.T - 1);
        rv = a.c[(size_t)t * a.conv_dim + (size_t)(2 * a.n_k + h) * kGHead + 16 * rg + (tid & 15)];
        rgb = *reinterpret_cast<const float2*>(a.gb + ((size_t)min(t0 + (tid & 15), a.T - 1) * a.n_v + h) * 2);
    };
    auto flush = [&](int t0, int u) {  // y of a finished piece: 16 rows of 16 tokens
        const int t = t0 + (tid >> 4);
        if (t < a.T) a.y[((size_t)t * a.n_v + h) * kGHead + 16 * rg + (tid & 15)] = s_y[u][tid >> 4][tid & 15];
    };
    load(begin);
    int u = 0;
    for (int t0 = begin; t0 < a.T; t0 += kScanTok, u ^= 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<vmi_f4*>(&s_qk[u][4 * j + (tid >> 6)][4 * (tid & 63)]) = rqk[j];
        s_v[u][tid >> 4][tid & 15] = rv;
        if (tid < kScanTok) s_gb[u][tid] = rgb;
        __syncthreads();
        if (t0 > begin) flush(t0 - kScanTok, u ^ 1);
        load(t0 + kScanTok);
        const int n = min(kScanTok, a.T - t0);
        auto token = [&](int i) {
            const vmi_f4 q0 = *reinterpret_cast<const vmi_f4*>(&s_qk[u][i][d0]);
            const vmi_f4 q1 = *reinterpret_cast<const vmi_f4*>(&s_qk[u][i][64 + d0]);
            const vmi_f4 k0 = *reinterpret_cast<const vmi_f4*>(&s_qk[u][i][kGHead + d0]);
            const vmi_f4 k1 = *reinterpret_cast<const vmi_f4*>(&s_qk[u][i][kGHead + 64 + d0]);
            const float2 gb = s_gb[u][i];
            float ka = 0.0f, kb = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[e] *= gb.x;
                S[4 + e] *= gb.x;
                ka = fmaf(S[e], k0[e], ka);
                kb = fmaf(S[4 + e], k1[e], kb);
            }
            const float delta = (s_v[u][i][lr] - vmi_row_sum16(ka + kb)) * gb.y;
            float ya = 0.0f, yb = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[e] = fmaf(k0[e], delta, S[e]);
                S[4 + e] = fmaf(k1[e], delta, S[4 + e]);
                ya = fmaf(S[e], q0[e], ya);
                yb = fmaf(S[4 + e], q1[e], yb);
            }
            const float yo = vmi_row_sum16(ya + yb);
            if ((lane & 15) == 0) s_y[u][i][lr] = yo;
            const int t = t0 + i;
            if (a.T - t <= a.n_slots) {
                float* dst = a.state_ring + (size_t)((a.pos0 + t + 1) % a.n_slots) * slot_elems + off;
                *reinterpret_cast<vmi_f4*>(dst) = vmi_f4{S[0], S[1], S[2], S[3]};
                *reinterpret_cast<vmi_f4*>(dst + 64) = vmi_f4{S[4], S[5], S[6], S[7]};
            }
        };
        if (n == kScanTok) {
#pragma unroll 4
            for (int i = 0; i < kScanTok; ++i) token(i);
        } else {
            for (int i = 0; i < n; ++i) token(i);
        }
    }
    __syncthreads();
    flush(begin + (a.T - 1 - begin) / kScanTok * kScanTok, u ^ 1);
}

// y / rms * w * silu(z) per (token, value head), 16 lanes each, rounded to bf16
// and written as the out projection's operand.  Bound by the bytes of y and z.
__global__ __launch_bounds__(kPrThreads) void k_pr_gnorm(PrGdn a) {
    const int i = blockIdx.x * (kPrThreads / 16) + (threadIdx.x >> 4), l = threadIdx.x & 15;
    if (i >= a.T * a.n_v) return;
    const int t = i / a.n_v, h = i % a.n_v;
    const float* y = a.y + (size_t)i * kGHead + 8 * l;
    const float* z = a.proj + (size_t)t * a.stride + (h / a.r) * a.per_g + (2 + a.r + h % a.r) * kGHead + 8 * l;
    const vmi_f4 y0 = *reinterpret_cast<const vmi_f4*>(y), y1 = *reinterpret_cast<const vmi_f4*>(y + 4);
    const vmi_f4 z0 = *reinterpret_cast<const vmi_f4*>(z), z1 = *reinterpret_cast<const vmi_f4*>(z + 4);
    const vmi_u4 nw = *reinterpret_cast<const vmi_u4*>(a.norm_w + 8 * l);
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(y0[e], y0[e], fmaf(y1[e], y1[e], ss));
    ss = vmi_row_sum16(ss);
    const float inv = __fdiv_rn(1.0f, __fsqrt_rn(ss * (1.0f / kGHead) + a.eps));
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float yv = e < 4 ? y0[e & 3] : y1[e & 3], zv = e < 4 ? z0[e & 3] : z1[e & 3];
        const float wv = __uint_as_float((e & 1) ? (nw[e >> 1] & 0xffff0000u) : (nw[e >> 1] << 16));
        f[e] = yv * inv * wv * (zv / (1.0f + expf(-zv)));
    }
    vmi_u4 u;
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = vmi_pack_bf16x2(f[2 * e], f[2 * e + 1]);
    const uint4 q = qg_operand_order(u);
    a.o.xop[((size_t)t * a.n_v + h) * (kGHead / 8) + l] = vmi_u4{q.x, q.y, q.z, q.w};
    const float s = sum8(sum_bf16x8(u));
    if ((l & 7) == 0) a.o.xneg[(size_t)(2 * h + (l >> 3)) * a.o.Tp + t] = -128.0f * s;
}

// ------------------------------------------------------------------- host
struct Carve {
    uint8_t* base;
    size_t off = 0;
    explicit Carve(void* p) : base(static_cast<uint8_t*>(p)) {}
    void* take(size_t bytes) {
        void* p = base + off;
        off += vmi::align256(bytes);
        return p;
    }
};

bool pr_k_ok(int K) { return K > 0 && K % 512 == 0 && K <= 4096; }
bool pr_qmat_ok(const vmi_qmat& m) {
    return vmi::qmat_ok(m) && !((reinterpret_cast<uintptr_t>(m.s) | reinterpret_cast<uintptr_t>(m.b)) & 15);
}

PrOperand pr_operand(Carve& c, int T, int K) {
    PrOperand o;
    o.Tp = (T + kPrTokPad - 1) / kPrTokPad * kPrTokPad;
    o.xop = static_cast<vmi_u4*>(c.take((size_t)T * K * 2));
    o.xneg = static_cast<float*>(c.take((size_t)(K / 64) * o.Tp * 4));
    return o;
}

hipError_t pr_prep(const uint16_t* x, const uint16_t* w, float eps, int T, int K, const PrOperand& o, hipStream_t s,
                   int* limit = nullptr) {
    const dim3 grid((T + 3) / 4), blk(kPrThreads);
    switch (K / 512) {
#define VMI_PREP(n) case n: hipLaunchKernelGGL(k_pr_prep<n>, grid, blk, 0, s, x, w, eps, T, o, limit); break;
        VMI_PREP(1) VMI_PREP(2) VMI_PREP(3) VMI_PREP(4) VMI_PREP(5) VMI_PREP(6) VMI_PREP(7) VMI_PREP(8)
#undef VMI_PREP
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class P>
hipError_t pr_gemm_as(const PrGemm& g, hipStream_t s) {
    const int tiles = ((g.T + P::TM - 1) / P::TM) * ((g.nrows + P::TN - 1) / P::TN);
    hipLaunchKernelGGL(k_pr_gemm<P>, dim3((tiles + 7) / 8 * 8), dim3(P::Threads), 0, s, g);
    return hipGetLastError();
}

// The tile shape with the least estimated time: rounds of one workgroup per
// CU times what a round measured at K = 2048 (us): 32 x 32 tiles 9, 64 x 64 11,
// 64 x 128 17 alone and 15 where two share a CU, 128 x 256 40.  Over 20 to 4096
// tokens and 1024 to 12,352 rows the shape taken is 1.03 times the best one's time
// on average: at most 1.09 at K = 2048 and 1.02 at 4096; at 1024 and 512 columns,
// where two 64 x 128 tiles on a CU take less of a round than at 2048, the largest
// tile is taken too early, up to 1.15 and 1.29.  At 777 tokens: 12,352 rows 77 us by 64 x 128 tiles (89
// by 128 x 256), 9216 rows 47 by 128 x 256 (55 by 64 x 128), 1024 rows 12 by
// 64 x 64 (18 by 64 x 128); 2048 rows of K = 4096 at 75 tokens 14.5 by 32 x 32
// (20 by 64 x 64).
hipError_t pr_gemm(const PrGemm& g, hipStream_t s) {
    const long ncu = vmi::device_cus();
    auto cost = [&](int tm, int tn, int one, int more) {
        const long tiles = (long)((g.T + tm - 1) / tm) * ((g.nrows + tn - 1) / tn), rounds = (tiles + ncu - 1) / ncu;
        return rounds == 1 ? (long)one : rounds * more;
    };
    const long c[4] = {cost(32, 32, 9, 9), cost(64, 64, 11, 11), cost(64, 128, 17, 15), cost(128, 256, 40, 40)};
    int best = 0;
    for (int i = 1; i < 4; ++i)
        if (c[i] < c[best]) best = i;
    switch (best) {
        case 0: return pr_gemm_as<PrShape<1, 1, 2, 8>>(g, s);
        case 1: return pr_gemm_as<PrShape<2, 1, 4, 4>>(g, s);
        case 2: return pr_gemm_as<PrShape<2, 2, 4, 3>>(g, s);
        default: return pr_gemm_as<PrShape<4, 4, 4, 3>>(g, s);
    }
}

constexpr int kPrMaxT = 8192;

struct AttnWs {
    PrOperand xn, on;
    float* qkv;
    uint16_t *q, *o;
    int* limit;
    size_t bytes;
};

AttnWs attn_ws(const vmi_attn_layer_desc& D, int T, void* base) {
    AttnWs w;
    Carve c(base);
    w.xn = pr_operand(c, T, D.hidden);
    w.on = pr_operand(c, T, D.n_heads * kHeadDim);
    w.qkv = static_cast<float*>(c.take((size_t)T * (D.n_heads * 2 + D.n_kv_heads * 2) * kHeadDim * 4));
    w.q = static_cast<uint16_t*>(c.take((size_t)T * D.n_heads * kHeadDim * 2));
    w.o = static_cast<uint16_t*>(c.take((size_t)T * D.n_heads * kHeadDim * 2));
    w.limit = static_cast<int*>(c.take(sizeof(int)));
    w.bytes = c.off;
    return w;
}

bool attn_form_ok(const vmi_attn_layer_desc& D, int T) {
    return T > 0 && T <= kPrMaxT && D.head_dim == kHeadDim && D.n_heads > 0 && D.n_kv_heads > 0 &&
           D.n_heads % D.n_kv_heads == 0 && pr_k_ok(D.hidden) && pr_k_ok(D.n_heads * kHeadDim) &&
           D.rope_dim >= 0 && D.rope_dim <= kHeadDim && D.rope_dim % 2 == 0 && D.bits == 4 && D.group == 64 &&
           pr_qmat_ok(D.q_proj) && pr_qmat_ok(D.k_proj) && pr_qmat_ok(D.v_proj) && pr_qmat_ok(D.o_proj) &&
           D.input_norm && D.q_norm && D.k_norm && !(reinterpret_cast<uintptr_t>(D.input_norm) & 15);
}

struct GdnWs {
    PrOperand xn, on;
    float *proj, *c, *gb, *y, *wy;
    int* limit;
    size_t bytes;
};

// Tokens that go through k_pr_chunk: all but the last n_slots, whose states
// the ring keeps, in whole pieces; none below kChunkMin, where their outputs
// are no closer to 64-bit ones than the sequential rule's: relative error of y over six
// inputs, sequential and pieces, 1e-7: 265 tokens 2.18 and 2.20, 300 2.32 and 2.36,
// 350 2.48 and 2.42, 400 2.62 and 2.57, 512 2.87 and 2.78, 777 3.23 and 3.10, 1200 3.51 and
// 3.28 (the state's is smaller at every length, 3.59 and 3.20 at 265).
int gdn_chunk_tokens(int T, int n_slots) {
    const int n = n_slots < T ? (T - n_slots) / kWyTok * kWyTok : 0;
    return n >= kChunkMin ? n : 0;
}

GdnWs gdn_ws(const vmi_gdn_layer_desc& D, int T, void* base) {
    GdnWs w;
    Carve c(base);
    const int r = D.n_v_heads / D.n_k_heads;
    const int stride = D.n_k_heads * (2 + 2 * r) * kGHead + 2 * D.n_v_heads;
    w.xn = pr_operand(c, T, D.hidden);
    w.on = pr_operand(c, T, D.n_v_heads * kGHead);
    w.proj = static_cast<float*>(c.take((size_t)T * stride * 4));
    w.c = static_cast<float*>(c.take((size_t)T * (2 * D.n_k_heads + D.n_v_heads) * kGHead * 4));
    w.gb = static_cast<float*>(c.take((size_t)T * D.n_v_heads * 2 * 4));
    w.y = static_cast<float*>(c.take((size_t)T * D.n_v_heads * kGHead * 4));
    w.limit = static_cast<int*>(c.take(sizeof(int)));
    w.wy = static_cast<float*>(c.take((size_t)(T / kWyTok) * D.n_v_heads * kWyFloats * 4));
    w.bytes = c.off;
    return w;
}

bool gdn_form_ok(const vmi_gdn_layer_desc& D, int T) {
    // n_v % 4 == 0 (as the width n_v * 128 asks): k_pr_wy's workgroups take four value
    // heads each, and the projection rows stay 16-byte aligned
    return T > 0 && T <= kPrMaxT && D.head_k_dim == kGHead && D.head_v_dim == kGHead && D.n_k_heads > 0 &&
           D.n_v_heads > 0 && D.n_v_heads % D.n_k_heads == 0 && D.n_v_heads % 4 == 0 &&
           pr_k_ok(D.hidden) && pr_k_ok(D.n_v_heads * kGHead) && D.bits == 4 && D.group == 64 &&
           pr_qmat_ok(D.in_proj_qkvz) && pr_qmat_ok(D.in_proj_ba) && pr_qmat_ok(D.out_proj) && D.input_norm &&
           D.conv_weight && D.A_log && D.dt_bias && D.norm_weight &&
           !((reinterpret_cast<uintptr_t>(D.input_norm) | reinterpret_cast<uintptr_t>(D.norm_weight) |
              reinterpret_cast<uintptr_t>(D.conv_weight)) & 15);
}

}  // namespace

extern "C" size_t vmi_attention_prompt_workspace_bytes(const vmi_attn_layer_desc* desc, int T) {
    return desc && attn_form_ok(*desc, T) ? attn_ws(*desc, T, nullptr).bytes : 0;
}

extern "C" int vmi_attention_prompt(const vmi_attn_layer_desc* desc, const uint16_t* x, int T, int pos0,
                                    uint16_t* k_cache, uint16_t* v_cache, int max_len, uint16_t* out, void* workspace,
                                    size_t workspace_bytes, void* stream) {
    vmi::clear_error();
    if (!desc) return vmi::fail(VMI_ERR_INVALID, "null desc");
    const vmi_attn_layer_desc& D = *desc;
    if (!attn_form_ok(D, T)) return vmi::fail(VMI_ERR_UNSUPPORTED, "layer form or T=%d not built for prompts", T);
    if (!x || !k_cache || !v_cache) return vmi::fail(VMI_ERR_INVALID, "null x/cache");
    if (pos0 < 0 || max_len % VMI_KV_BLOCK || T > max_len || pos0 > max_len - T)
        return vmi::fail(VMI_ERR_INVALID, "pos0=%d T=%d max_len=%d", pos0, T, max_len);
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_cache) |
         reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(workspace)) & 15)
        return vmi::fail(VMI_ERR_INVALID, "x, out, caches and workspace must be 16-byte aligned");
    const AttnWs W = attn_ws(D, T, workspace);
    if (!workspace || workspace_bytes < W.bytes)
        return vmi::fail(VMI_ERR_WORKSPACE, "workspace needs %zu bytes (got %zu)", W.bytes, workspace_bytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int heads = D.n_heads, kv = D.n_kv_heads, stride = (2 * heads + 2 * kv) * kHeadDim;
    hipError_t e = pr_prep(x, D.input_norm, D.norm_eps, T, D.hidden, W.xn, s, W.limit);
    if (e != hipSuccess) return vmi::hip_fail(e, "input norm launch");
    // without an output only the keys and values are formed (columns of the same rows)
    const int qrows = out ? heads * 2 * kHeadDim : 0;
    PrGemm p{};
    p.x = W.xn; p.T = T; p.K = D.hidden;
    p.m[0] = D.q_proj; p.m[1] = D.k_proj; p.m[2] = D.v_proj;
    p.rows[0] = qrows; p.rows[1] = kv * kHeadDim; p.rows[2] = kv * kHeadDim; p.nrows = qrows + 2 * kv * kHeadDim;
    p.out = W.qkv + (heads * 2 * kHeadDim - qrows); p.out_stride = stride;
    e = pr_gemm(p, s);
    if (e != hipSuccess) return vmi::hip_fail(e, "qkv projection launch");
    PrAttn at{};
    at.qkv = W.qkv; at.stride = stride; at.T = T; at.n_heads = heads; at.n_kv = kv; at.pos0 = pos0; at.max_len = max_len;
    at.q_norm = D.q_norm; at.k_norm = D.k_norm; at.rope_dim = D.rope_dim; at.eps = D.norm_eps;
    at.rope_base = D.rope_dim ? pow((double)D.rope_theta, -2.0 / (double)D.rope_dim) : 1.0;
    at.k_cache = k_cache; at.v_cache = v_cache; at.q = W.q; at.o = W.o; at.limit = W.limit;
    at.h0 = out ? 0 : heads;
    hipLaunchKernelGGL(k_pr_qkv, dim3(T), dim3(kPrThreads), 0, s, at);
    if (!out) {
        e = hipGetLastError();
        return e == hipSuccess ? VMI_OK : vmi::hip_fail(e, "key/value launch");
    }
    const int R = T * (heads / kv);
    if ((R + 127) / 128 * kv >= vmi::device_cus())
        hipLaunchKernelGGL(k_pr_flash<2>, dim3((R + 127) / 128, kv), dim3(kPrThreads), 0, s, at);
    else
        hipLaunchKernelGGL(k_pr_flash<1>, dim3((R + 63) / 64, kv), dim3(kPrThreads), 0, s, at);
    e = pr_prep(W.o, nullptr, 0.0f, T, heads * kHeadDim, W.on, s);
    if (e != hipSuccess) return vmi::hip_fail(e, "attention launch");
    PrGemm o{};
    o.x = W.on; o.T = T; o.K = heads * kHeadDim;
    o.m[0] = o.m[1] = o.m[2] = D.o_proj;
    o.rows[0] = o.nrows = D.hidden;
    o.out_stride = D.hidden; o.residual = x; o.out_bf16 = out;
    e = pr_gemm(o, s);
    return e == hipSuccess ? VMI_OK : vmi::hip_fail(e, "o_proj launch");
}

extern "C" size_t vmi_gdn_prompt_workspace_bytes(const vmi_gdn_layer_desc* desc, int T) {
    return desc && gdn_form_ok(*desc, T) ? gdn_ws(*desc, T, nullptr).bytes : 0;
}

extern "C" int vmi_gdn_prompt(const vmi_gdn_layer_desc* desc, const uint16_t* x, int T, int pos0, uint16_t* conv_ring,
                              float* state_ring, int n_slots, uint16_t* out, void* workspace, size_t workspace_bytes,
                              void* stream) {
    vmi::clear_error();
    if (!desc) return vmi::fail(VMI_ERR_INVALID, "null desc");
    const vmi_gdn_layer_desc& D = *desc;
    if (!gdn_form_ok(D, T)) return vmi::fail(VMI_ERR_UNSUPPORTED, "layer form or T=%d not built for prompts", T);
    if (!x || !out || !conv_ring || !state_ring) return vmi::fail(VMI_ERR_INVALID, "null x/out/ring");
    if (pos0 < 0 || n_slots < 1) return vmi::fail(VMI_ERR_INVALID, "pos0=%d n_slots=%d", pos0, n_slots);
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(state_ring) |
         reinterpret_cast<uintptr_t>(conv_ring) | reinterpret_cast<uintptr_t>(workspace)) & 15)
        return vmi::fail(VMI_ERR_INVALID, "x, out, rings and workspace must be 16-byte aligned");
    const GdnWs W = gdn_ws(D, T, workspace);
    if (!workspace || workspace_bytes < W.bytes)
        return vmi::fail(VMI_ERR_WORKSPACE, "workspace needs %zu bytes (got %zu)", W.bytes, workspace_bytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    PrGdn a{};
    a.T = T; a.pos0 = pos0; a.n_k = D.n_k_heads; a.n_v = D.n_v_heads; a.r = a.n_v / a.n_k;
    a.per_g = (2 + 2 * a.r) * kGHead; a.conv_dim = (2 * a.n_k + a.n_v) * kGHead;
    a.stride = a.n_k * a.per_g + 2 * a.n_v; a.n_slots = n_slots;
    a.proj = W.proj; a.conv_w = D.conv_weight; a.A_log = D.A_log; a.dt_bias = D.dt_bias;
    a.conv_ring = conv_ring; a.state_ring = state_ring; a.c = W.c; a.gb = W.gb; a.y = W.y;
    a.norm_w = D.norm_weight; a.eps = D.norm_eps; a.o = W.on;
    a.wy = W.wy; a.limit = W.limit;
    a.t0 = gdn_chunk_tokens(T, n_slots);
    hipError_t e = pr_prep(x, D.input_norm, D.norm_eps, T, D.hidden, W.xn, s);
    if (e != hipSuccess) return vmi::hip_fail(e, "input norm launch");
    PrGemm p{};
    p.x = W.xn; p.T = T; p.K = D.hidden;
    p.m[0] = D.in_proj_qkvz; p.m[1] = p.m[2] = D.in_proj_ba;
    p.rows[0] = a.n_k * a.per_g; p.rows[1] = 2 * a.n_v; p.nrows = a.stride;
    p.out = W.proj; p.out_stride = a.stride;
    e = pr_gemm(p, s);
    if (e != hipSuccess) return vmi::hip_fail(e, "qkvz/ba projection launch");
    hipLaunchKernelGGL(k_pr_conv, dim3((T + kConvTok - 1) / kConvTok, (2 * a.n_k + a.n_v + 7) / 8 + 1), dim3(kPrThreads),
                       0, s, a);
    if (a.t0) {
        hipLaunchKernelGGL(k_pr_wy, dim3(a.t0 / kWyTok, a.n_v / 4), dim3(kPrThreads), 0, s, a);
        hipLaunchKernelGGL(k_pr_chunk, dim3(a.n_v * (kGHead / 16)), dim3(kPrThreads), 0, s, a);
    }
    hipLaunchKernelGGL(k_pr_scan, dim3(a.n_v * (kGHead / 16)), dim3(kPrThreads), 0, s, a);
    hipLaunchKernelGGL(k_pr_gnorm, dim3((T * a.n_v + 15) / 16), dim3(kPrThreads), 0, s, a);
    PrGemm o{};
    o.x = W.on; o.T = T; o.K = a.n_v * kGHead;
    o.m[0] = o.m[1] = o.m[2] = D.out_proj;
    o.rows[0] = o.nrows = D.hidden;
    o.out_stride = D.hidden; o.residual = x; o.out_bf16 = out;
    e = pr_gemm(o, s);
    return e == hipSuccess ? VMI_OK : vmi::hip_fail(e, "out_proj launch");
}

extern "C" size_t vmi_qgemm_workspace_bytes(int T, int K, vmi_qmat w, int N, int bits, int group) {
    if (T <= 0 || T > kPrMaxT || !pr_k_ok(K) || N <= 0 || bits != 4 || group != 64 || !pr_qmat_ok(w)) return 0;
    Carve c(nullptr);
    pr_operand(c, T, K);
    return c.off;
}

extern "C" int vmi_qgemm(const uint16_t* x, int T, int K, vmi_qmat w, int N, int bits, int group,
                         const uint16_t* residual, uint16_t* out_bf16, void* workspace, size_t workspace_bytes,
                         void* stream) {
    vmi::clear_error();
    const size_t need = vmi_qgemm_workspace_bytes(T, K, w, N, bits, group);
    if (!need) return vmi::fail(VMI_ERR_UNSUPPORTED, "T=%d K=%d N=%d bits=%d group=%d", T, K, N, bits, group);
    if (!x || !out_bf16) return vmi::fail(VMI_ERR_INVALID, "null x/out");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(workspace)) & 15)
        return vmi::fail(VMI_ERR_INVALID, "x and workspace must be 16-byte aligned");
    if (!workspace || workspace_bytes < need)
        return vmi::fail(VMI_ERR_WORKSPACE, "workspace needs %zu bytes (got %zu)", need, workspace_bytes);
    Carve c(workspace);
    PrGemm g{};
    g.x = pr_operand(c, T, K);
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e = pr_prep(x, nullptr, 0.0f, T, K, g.x, s);
    if (e != hipSuccess) return vmi::hip_fail(e, "operand launch");
    g.T = T; g.K = K;
    g.m[0] = g.m[1] = g.m[2] = w;
    g.rows[0] = g.nrows = N;
    g.out_stride = N; g.residual = residual; g.out_bf16 = out_bf16;
    e = pr_gemm(g, s);
    return e == hipSuccess ? VMI_OK : vmi::hip_fail(e, "qgemm launch");
}
