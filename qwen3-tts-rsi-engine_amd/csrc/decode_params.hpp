// The parameter block of the decode attention launches (every grid's kernels take it by value),
// the helpers for its optional SDPA-style mask, and the step plan's entry points
// (decode_plan.hip).
#pragma once

#include "q3t_common.hpp"

namespace q3t {

struct DecodeParams {
    int B, Hq, Hkv, ctx, nchunks;
    int splits;             // balanced grid: workgroups per KV head (0: chunked grid)
    int bundles;            // bundled grid: workgroups per KV head (0: another grid)
    float scale_log2;
    int has_mask, mask_dtype;
    const char *q;
    int64_t q_sb, q_ss, q_sh;
    char *k, *v;
    int64_t k_sb, k_sh, k_st, v_sb, v_sh, v_st;
    const int64_t *offs;
    const int64_t *pos;     // null: every request attends all of its keys
    const char *mask;
    int64_t m_sb, m_ss, m_st;
    char *out;
    int64_t o_sb, o_ss, o_sh;
    const char *nk, *nv;
    int64_t nk_sb, nk_sh, nv_sb, nv_sh;
    const char *cs, *sn;
    int64_t cs_sb;
    float *partials;
    int *counters;
    const char *qnw, *knw;  // fused: optional RMSNorm weights (bf16, D) of query / new key rows
    float eps;
    int stream;             // read K/V rows with the non-temporal cache policy (host choice)
    int64_t nk_ss, nv_ss, cs_ss;  // fused, two tokens: token strides of new K/V and cos/sin
    const int32_t *plan;    // bundled grid: the step's plan (decode_plan.hip), null without one
};

// The step plan (decode_plan.hip): bundles per KV head, plan size in int32 and its launch.
int64_t plan_bundle_count(int64_t batch, int64_t kv_heads);
int64_t plan_ints(int64_t batch, int64_t kv_heads);
int plan_launch(const int64_t *pos, int batch, int ctx, int bundles, int32_t *plan, hipStream_t s);

// The unsplit form of the chunked grid (decode_direct.hip): one workgroup per (request, KV head).
constexpr int kDirectMaxCtx = 2048;    // longest context it takes (a mask row's words in LDS)
constexpr int kDirectOneWave = 32;     // longest context of one wave a workgroup
constexpr int kDirectManyPairs = 64;   // (request, KV head) pairs from which its workgroups are smaller
void direct_launch(const DecodeParams &p, int group, int tokens, bool fused, hipStream_t s);

// 4 bytes per lane from global memory into LDS at lds_base + 4 * lane (the mask words of a
// stage's rows); offsets past the resource's range write zeros.
Q3T_DEVICE void load_to_lds4(i32x4_t rsrc, uint32_t voffset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\t" Q3T_VMEM_SGPR_WAIT "buffer_load_dword %1, %2, 0 offen lds"
                 :: "s"(lds_base), "v"(voffset), "s"(rsrc) : "memory", "m0");
}

// A mask term (log2 units) from the 4-byte word holding it; `sub` = its byte offset in the word.
Q3T_DEVICE float mask_term(uint32_t word, uint32_t sub, int dtype) {
    const uint32_t x = word >> (8 * sub);
    switch (dtype) {
        case Q3T_BF16: return bf16_to_float(x & 0xffffu) * 1.4426950408889634f;
        case Q3T_F16: return (float)__builtin_bit_cast(_Float16, (uint16_t)(x & 0xffffu)) * 1.4426950408889634f;
        case Q3T_F32: return __uint_as_float(word) * 1.4426950408889634f;
        default: return (x & 0xffu) ? 0.0f : -INFINITY;  // bool: True attends
    }
}

Q3T_DEVICE int mask_elem_size(int dtype) { return dtype == Q3T_F32 ? 4 : dtype == Q3T_BOOL ? 1 : 2; }

Q3T_DEVICE float load_mask(const char *m, int dtype) {
    switch (dtype) {
        case Q3T_BF16: return bf16_to_float(*reinterpret_cast<const uint16_t *>(m));
        case Q3T_F16: return (float)*reinterpret_cast<const _Float16 *>(m);
        case Q3T_F32: return *reinterpret_cast<const float *>(m);
        default: return *reinterpret_cast<const uint8_t *>(m) ? 0.0f : -INFINITY;  // bool: True attends
    }
}

// Sum over each aligned group of LPK (8, 16 or 32) lanes; every lane of the group gets it.
template <int LPK>
Q3T_DEVICE float group_sum(float x) {
    x = sum8(x);
    if constexpr (LPK >= 16) x += xor8(x);
    if constexpr (LPK >= 32) x += xor16(x);
    return x;
}

// RMSNorm of one bf16 row spread over LPK lanes (8 elements per lane), as the attention
// module's q_norm / k_norm compute it: fp32 sum of squares over the row, x * rsqrt(mean + eps)
// rounded to bf16, times the bf16 weight, rounded to bf16.  The sum's order is this kernel's
// (lanes, then the DPP tree); rows agree with other orders to the last bf16 bit except near
// rounding ties.
template <int LPK>
Q3T_DEVICE U4 rms_norm8(const U4 &x, const U4 &w, float eps, int width) {
    const uint32_t v[4] = {x.x, x.y, x.z, x.w}, g[4] = {w.x, w.y, w.z, w.w};
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = bf16_lo(v[i]), b = bf16_hi(v[i]);
        ss = __builtin_fmaf(a, a, ss);
        ss = __builtin_fmaf(b, b, ss);
    }
    ss = group_sum<LPK>(ss);
    const float r = __builtin_amdgcn_rsqf(ss * (1.0f / (float)width) + eps);
    uint32_t y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t n = cvt_pk_bf16(bf16_lo(v[i]) * r, bf16_hi(v[i]) * r);
        y[i] = cvt_pk_bf16_canon(bf16_lo(n) * bf16_lo(g[i]), bf16_hi(n) * bf16_hi(g[i]));
    }
    return U4{y[0], y[1], y[2], y[3]};
}

template <typename T>
Q3T_DEVICE void store_out(char *base, float v) {
    if constexpr (sizeof(T) == 2)
        *reinterpret_cast<uint16_t *>(base) = (uint16_t)float_to_bf16(v);
    else
        *reinterpret_cast<float *>(base) = v;
}

}  // namespace q3t
