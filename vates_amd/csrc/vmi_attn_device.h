// Device helpers shared by the attention kernels of the verify batch
// (vmi_attn.hip) and of the prompt (vmi_prompt.hip).
#pragma once

#include "vmi_device.h"

namespace {

constexpr int kHeadDim = 256;

__device__ __forceinline__ int at_wave() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

__device__ __forceinline__ void bf16x8f(const uint4& q, float (&v)[8]) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

__device__ __forceinline__ vmi_u4 keep_first(vmi_u4 v, int n) {  // zero bf16 elements e >= n
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] &= (2 * i < n ? 0x0000ffffu : 0u) | (2 * i + 1 < n ? 0xffff0000u : 0u);
    return v;
}

// (cos, sin) of pos * theta^(-2 fi / rd), base = theta^(-2/rd): the angle in
// turns and in double, reduced to [-1/2, 1/2] turn, then in fp32.
__device__ __forceinline__ float2 rotary_cs(int pos, int fi, double base) {
    double f = 1.0, b = base;
    for (int e = fi; e; e >>= 1) {
        if (e & 1) f *= b;
        b *= b;
    }
    const double turns = (double)pos * (f * 0.15915494309189535);  // 1 / (2 pi)
    const float r = (float)((turns - rint(turns)) * 6.283185307179586);
    float sn, cs;
    sincosf(r, &sn, &cs);
    return make_float2(cs, sn);
}

// NR head rows of one wave (dims lane + 64 j of row i in v[i]) in place:
// RMSNorm (x^2 of the lane's four dims in order, then the canonical wave
// sum), times the norm weight, rounded to bf16 (the model dtype), then the
// rotary pairs (d, d + rd/2) in fp32 with (cos, sin) of pos * theta^(-2i/rd)
// from cs[i], rounded to bf16.  The rows go through together and nothing
// branches on the lane, so their reductions and LDS reads overlap.  The
// rotary partner of dim d: for rd = 64 the lane 32 apart, for rd = 128 and
// 256 another register of the same lane; other widths go through srow, the
// wave's own LDS row, one row at a time.
template <int NR>
__device__ __forceinline__ void norm_rope_rows(float (&v)[NR][4], const float (&nw)[4], float eps,
                                               const float2* const (&cs)[NR], int rd, float* srow,
                                               uint16_t (&o)[NR][4]) {
    const int lane = threadIdx.x & 63;
    float ss[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        ss[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) ss[i] = fmaf(v[i][j], v[i][j], ss[i]);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) ss[i] = vmi_wave_sum_canon(ss[i]);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(ss[i] * (1.0f / (float)kHeadDim) + eps));
        const uint32_t u01 = vmi_pack_bf16x2((v[i][0] * inv) * nw[0], (v[i][1] * inv) * nw[1]);
        const uint32_t u23 = vmi_pack_bf16x2((v[i][2] * inv) * nw[2], (v[i][3] * inv) * nw[3]);
        v[i][0] = __uint_as_float(u01 << 16);
        v[i][1] = __uint_as_float(u01 & 0xffff0000u);
        v[i][2] = __uint_as_float(u23 << 16);
        v[i][3] = __uint_as_float(u23 & 0xffff0000u);
    }
    const int half = rd / 2;
    auto store = [&](int i, const float (&r)[4]) {
        const uint32_t a = vmi_pack_bf16x2(r[0], r[1]), b = vmi_pack_bf16x2(r[2], r[3]);
        o[i][0] = (uint16_t)a;
        o[i][1] = (uint16_t)(a >> 16);
        o[i][2] = (uint16_t)b;
        o[i][3] = (uint16_t)(b >> 16);
    };
    if (rd == 64 || rd == 128 || rd == 256) {
        // register j of every lane is rotated or not as a whole (rd is a
        // multiple of 64): the table reads need no lane mask
        float2 c[NR][4];
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int d = lane + 64 * j;
                c[i][j] = 64 * j < rd ? cs[i][d < half ? d : d - half] : make_float2(1.0f, 0.0f);
            }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            float pr[4];
            if (rd == 64) {
                pr[0] = __shfl_xor(v[i][0], 32, 64);
                pr[1] = pr[2] = pr[3] = 0.0f;
            } else if (rd == 128) {
                pr[0] = v[i][1];
                pr[1] = v[i][0];
                pr[2] = pr[3] = 0.0f;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) pr[j] = v[i][j ^ 2];
            }
            float r[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int d = lane + 64 * j;
                const float partner = d < half ? -pr[j] : pr[j];
                r[j] = 64 * j < rd ? v[i][j] * c[i][j].x + partner * c[i][j].y : v[i][j];
            }
            store(i, r);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) srow[lane + 64 * j] = v[i][j];
        __builtin_amdgcn_wave_barrier();  // srow is this wave's own row: LDS order within a wave suffices
        float r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d = lane + 64 * j;
            r[j] = v[i][j];
            if (d < rd) {
                const float2 c = cs[i][d < half ? d : d - half];
                const float partner = d < half ? -srow[d + half] : srow[d - half];
                r[j] = v[i][j] * c.x + partner * c.y;
            }
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read its partner before srow is rewritten
        store(i, r);
    }
}

// 8 bf16 values in MFMA operand order: pairs (e, e + 4), the order in which
// vmi_unpack_u4_bf16_128 yields a word's nibbles.
__device__ __forceinline__ uint4 qg_operand_order(const vmi_u4& u) {
    return make_uint4(__builtin_amdgcn_perm(u[2], u[0], 0x05040100u), __builtin_amdgcn_perm(u[2], u[0], 0x07060302u),
                      __builtin_amdgcn_perm(u[3], u[1], 0x05040100u), __builtin_amdgcn_perm(u[3], u[1], 0x07060302u));
}

}  // namespace
