// The work of one workgroup on one (request, KV head) pair over a key range, on vector
// instructions: shared by the split grids (decode_attention.hip) and the whole-request kernel of the
// types that the MFMA kernels do not take (decode_whole.hip).
#pragma once

#include "decode_params.hpp"

namespace q3t {

constexpr int kChunkRows = 64;
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kEmpty = -1.0e30f;  // finite "no key yet" running max

// Partial score of one lane: its 16 bytes of the query row and of the key row.
template <typename T>
Q3T_DEVICE float lane_dot(const U4 &q, const U4 &k) {
    if constexpr (sizeof(T) == 2) {
        float s = dot2_bf16(q.x, k.x, 0.f);
        s = dot2_bf16(q.y, k.y, s);
        s = dot2_bf16(q.z, k.z, s);
        return dot2_bf16(q.w, k.w, s);
    } else {
        float s = __uint_as_float(q.x) * __uint_as_float(k.x);
        s += __uint_as_float(q.y) * __uint_as_float(k.y);
        s += __uint_as_float(q.z) * __uint_as_float(k.z);
        return s + __uint_as_float(q.w) * __uint_as_float(k.w);
    }
}

// Sum / max across the lane groups of a wave (lanes that differ in the bits above the group).
template <int LPK>
Q3T_DEVICE float cross_sum(float x) {
    if constexpr (LPK <= 8) x += xor8(x);
    if constexpr (LPK <= 16) x += xor16(x);
    return x + xor32(x);
}
template <int LPK>
Q3T_DEVICE float cross_max(float x) {
    if constexpr (LPK <= 8) x = fmaxf(x, xor8(x));
    if constexpr (LPK <= 16) x = fmaxf(x, xor16(x));
    return fmaxf(x, xor32(x));
}

// Sums of N values across the lane halves (permlane32_swap) and then across 16-lane rows
// (permlane16_swap), two values per swap: swap(a, b) leaves lanes 0-31 with the half-sums of
// a and lanes 32-63 with those of b, so every step halves the register count instead of
// reducing each value on its own.  Afterwards half[k] in half h holds element 2k + h summed
// over both halves, and quarter[m] in row g holds element 4m + kRowElem[g] summed over all
// four rows.
constexpr int kRowElem[4] = {0, 2, 1, 3};
template <int N>
Q3T_DEVICE void sum_halves(const float (&v)[N], float (&half)[N / 2]) {
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * k]), __float_as_uint(v[2 * k + 1]),
                                                        false, false);
        half[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
}
template <int N>
Q3T_DEVICE void sum_rows(const float (&half)[N / 2], float (&quarter)[N / 4]) {
#pragma unroll
    for (int k = 0; k < N / 4; ++k) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(half[2 * k]), __float_as_uint(half[2 * k + 1]),
                                                        false, false);
        quarter[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
}

// Reduce the lane groups' accumulators of a wave and store the wave's acc rows (R x D) to LDS.
// acc[r][e] of lane (group, cl) belongs to element e of the 16-byte chunk cl of query row r.
template <int LPK, int CW, int R, int D>
Q3T_DEVICE void store_wave_acc(float (&acc)[R][CW], float (&dst)[R][D], int lane) {
    constexpr int N = R * CW;
    float v[N];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < CW; ++e) v[r * CW + e] = acc[r][e];
    if constexpr (LPK == 32) {  // two groups: the lane halves
        float h2[N / 2];
        sum_halves<N>(v, h2);
        const int cl = lane & 31, hf = lane >> 5;
#pragma unroll
        for (int k = 0; k < N / 2; ++k) {
            const int i = 2 * k + hf;
            dst[i / CW][cl * CW + i % CW] = h2[k];
        }
    } else {
        if constexpr (LPK == 8) {  // two groups per 16-lane row first
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] += xor8(v[i]);
        }
        float h2[N / 2], q4[N / 4];
        sum_halves<N>(v, h2);
        sum_rows<N>(h2, q4);
        const int row = (lane >> 4) & 3, cl = lane & (LPK - 1);
        const int sel = kRowElem[row];
        if (LPK == 16 || (lane & 8) == 0) {
#pragma unroll
            for (int k = 0; k < N / 4; ++k) {
                const int i = 4 * k + sel;
                dst[i / CW][cl * CW + i % CW] = q4[k];
            }
        }
    }
}

// Lane geometry of a variant: one 16-byte vector of a key row per lane.
template <typename T, int D, int W = kWaves, int ROWS = kChunkRows>
struct DecodeShape {
    static constexpr int ES = sizeof(T);
    static constexpr int LPK = D * ES / 16;       // lanes per key row: 8, 16 or 32
    static constexpr int CW = 16 / ES;            // elements per lane
    static constexpr int RPW = 64 / LPK;          // rows per wave per pass
    static constexpr int RPP = RPW * W;      // rows per workgroup pass
    static constexpr int P = ROWS / RPP;    // passes per block
    static_assert(P >= 1 && ROWS % RPP == 0, "block must be whole passes");
};

// Waves per SIMD the register allocation aims for: the kernel is latency-bound, so the
// bf16 variants with at most two query rows per KV head are held to 80 VGPRs (6 waves),
// which they meet without spilling; wider variants keep the compiler's choice.
// bf16 launches of one or two query rows per KV head fit 80 VGPRs (6 waves per SIMD); the
// mask's per-key terms need a few more, which 5 waves per SIMD leave room for without spills
constexpr int decode_waves_per_eu(int es, int rows, bool mask) {
    return es == 2 && rows <= 2 ? (mask ? 5 : 6) : 1;
}

// The work of one workgroup on one (request, KV head) pair over a key range [j0, j1): the
// online softmax of the pair's G * SQ query rows, shared by both grids below.
//   load_rows  requests the rows that depend only on (request, head): the query rows and,
//              fused, the step's cos/sin rows and new key/value rows (16 bytes per lane
//              each; lane group t holds token t's new rows).  Callers issue it before the
//              request's key count is known.
//   attend     streams the arena keys of the range in 64-key blocks (every pass of a block
//              issued before any math; with PIPE the next block is requested before the
//              current one is folded in, which costs a second block of registers), folds in the step's new keys when `finisher`
//              (fused: rotated, written to the arena at L-SQ ... L-1 and attended from LDS;
//              no workgroup reads those arena rows in the same launch), and leaves the
//              range's merged state in wave 0: for output t = lane + 64 i (query row
//              t / D, dim t % D) the unnormalised accumulator A[i], the weight sum Ls[i]
//              and the running maximum Mx[i] in scaled log2 units.
// W waves work on the pair, on blocks of ROWS keys.
template <typename T, int D, int G, int SQ, int FUSE, bool MASK, bool STREAM, bool PIPE, int W = kWaves, int ROWS = kChunkRows>
struct PairWork {
    // FUSE: 0 attention only, 1 the fused step, 2 the fused step with its q/k norms (a separate
    // instance: the norm code, even unexecuted, slowed the fused bundled kernel by 1.8 us)
    static constexpr bool FUSED = FUSE > 0, NORM = FUSE > 1;
    static constexpr int R = G * SQ;
    using S = DecodeShape<T, D, W, ROWS>;
    static constexpr int LPK = S::LPK, CW = S::CW, RPW = S::RPW, RPP = S::RPP, P = S::P, ES = S::ES;
    static constexpr int OPL = R * D / 64;  // outputs per lane of wave 0
    static constexpr int HD = D;
    static_assert(!FUSED || (ES == 2 && D == 128 && SQ <= 2), "fused path: bf16, D=128, one or two tokens");

    struct Lds {
        float acc[W][R][D];
        float ml[W][R][2];
    };
    using NewRows = U4[2][FUSED ? SQ : 1][16];  // rotated new keys, new values (fused)

    U4 qr[R];
    U4 nk, nv, cv[SQ], sv[SQ];

    Q3T_DEVICE void load_rows(const DecodeParams &p, int b, int h) {
        const int lane = threadIdx.x & 63, grp = lane / LPK, cl = lane % LPK;
        if constexpr (FUSED) {
#pragma unroll
            for (int t = 0; t < SQ; ++t) {
                cv[t] = load16(p.cs + (b * p.cs_sb + t * p.cs_ss) * 2 + cl * 16);
                sv[t] = load16(p.sn + (b * p.cs_sb + t * p.cs_ss) * 2 + cl * 16);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int qi = r / G, hq = h * G + r % G;
            qr[r] = load16(p.q + (b * p.q_sb + qi * p.q_ss + hq * p.q_sh) * ES + cl * 16);
        }
        if constexpr (FUSED) {
            const int tk = grp < SQ ? grp : SQ - 1;
            nk = load16(p.nk + (b * p.nk_sb + tk * p.nk_ss + h * p.nk_sh) * ES + cl * 16);
            nv = load16(p.nv + (b * p.nv_sb + tk * p.nv_ss + h * p.nv_sh) * ES + cl * 16);
        }
    }

    // Zero output rows of a request without a valid position (it attends nothing).
    static Q3T_DEVICE void write_zeros(const DecodeParams &p, int b, int h) {
        for (int t = threadIdx.x; t < R * D; t += W * 64) {
            const int r = t / D, d = t % D, qi = r / G, hq = h * G + r % G;
            store_out<T>(p.out + (b * p.o_sb + qi * p.o_ss + hq * p.o_sh + d) * ES, 0.f);
        }
    }

    // Wave 0: final output rows A / Ls of request b.
    static Q3T_DEVICE void write_out(const DecodeParams &p, int b, int h, const float (&A)[OPL],
                                     const float (&Ls)[OPL]) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int i = 0; i < OPL; ++i) {
            const int t = lane + 64 * i, r = t / D, d = t % D, qi = r / G, hq = h * G + r % G;
            store_out<T>(p.out + (b * p.o_sb + qi * p.o_ss + hq * p.o_sh + d) * ES,
                         A[i] * __builtin_amdgcn_rcpf(Ls[i]));
        }
    }

    // The range's keys: every wave's state in LDS, the workgroup past a barrier.
    Q3T_DEVICE void stream(const DecodeParams &p, int b, int h, int L, int j0, int j1, bool finisher, Lds &lds, NewRows &snew) {
        const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
        const int grp = lane / LPK, cl = lane % LPK;
        const bool with_new = FUSED && finisher;
        const int jend = FUSED ? min(j1, L - SQ) : j1;  // arena keys of the range: [j0, jend)

        const char *kb = p.k + ((p.offs ? p.offs[b] : (int64_t)b * p.k_sb) + h * p.k_sh) * ES;
        const char *vb = p.v + ((p.offs ? p.offs[b] : (int64_t)b * p.v_sb) + h * p.v_sh) * ES;
        const int kst = (int)(p.k_st * ES), vst = (int)(p.v_st * ES);
        const bool same_stride = kst == vst;
        // K/V rows 0 .. ctx-1 of (b, h) through buffer resources (32-bit row offsets)
        const auto krs = buffer_rsrc(uniform_ptr(kb), (uint32_t)((p.ctx - 1) * kst + D * ES));
        const auto vrs = buffer_rsrc(uniform_ptr(vb), (uint32_t)((p.ctx - 1) * vst + D * ES));
        const char *mask_row = MASK ? p.mask + b * p.m_sb * mask_elem_size(p.mask_dtype) : nullptr;

        // keys of the block at jb: rows at or past jend get an offset outside the resource,
        // which reads zeros without a memory access
        auto load_block = [&](int jb, U4 (&kr)[P], U4 (&vr)[P]) {
#pragma unroll
            for (int pp = 0; pp < P; ++pp) {
                const int j = jb + pp * RPP + wave * RPW + grp;
                const bool ok = j < jend;
                const uint32_t ko = ok ? (uint32_t)(j * kst) + cl * 16 : 0xfffffff0u;
                const uint32_t vo = ok ? (same_stride ? ko : (uint32_t)(j * vst) + cl * 16) : 0xfffffff0u;
                if constexpr (STREAM) {
                    kr[pp] = buffer_load16_stream(krs, ko);
                    vr[pp] = buffer_load16_stream(vrs, vo);
                } else {
                    kr[pp] = buffer_load16(krs, ko);
                    vr[pp] = buffer_load16(vrs, vo);
                }
            }
        };

        // with PIPE the first block is requested before the query prologue and every later
        // block while the one before it is being folded in; without, each block after the
        // previous one (fewer registers: the chunked grid's rows arrive with the position)
        U4 kr[PIPE ? P : 1], vr[PIPE ? P : 1];
        if constexpr (PIPE) load_block(j0, kr, vr);

        U4 q[R];
#pragma unroll
        for (int r = 0; r < R; ++r) q[r] = qr[r];
        if constexpr (FUSED) {
            if (NORM && p.qnw) {
                const U4 w = load16(p.qnw + cl * 16);
#pragma unroll
                for (int r = 0; r < R; ++r) q[r] = rms_norm8<LPK>(q[r], w, p.eps, D);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) q[r] = rope_half8(q[r], xor8_u4(q[r]), cv[r / G], sv[r / G], cl < 8);
            if (with_new && wave == 0 && grp < SQ && L - SQ + grp >= 0) {
                // lane group t of wave 0 holds token t's whole rows, so the half exchange (and
                // the norm's row sum) sees every element
                const U4 ct = SQ == 1 || grp == 0 ? cv[0] : cv[SQ - 1];
                const U4 st = SQ == 1 || grp == 0 ? sv[0] : sv[SQ - 1];
                U4 kx = nk;
                if (NORM && p.knw) kx = rms_norm8<LPK>(nk, load16(p.knw + cl * 16), p.eps, D);
                const U4 kn = rope_half8(kx, xor8_u4(kx), ct, st, cl < 8);
                const int row = L - SQ + grp;
                buffer_store16(krs, (uint32_t)(row * kst) + cl * 16, kn);
                buffer_store16(vrs, (uint32_t)(row * vst) + cl * 16, nv);
                snew[0][grp][cl] = kn;
                snew[1][grp][cl] = nv;
            }
        }


        float m[R], l[R], acc[R][CW];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            m[r] = kEmpty;
            l[r] = 0.f;
#pragma unroll
            for (int e = 0; e < CW; ++e) acc[r][e] = 0.f;
        }

        // one online-softmax step over P key vectors per lane (invalid ones carry -inf scores)
        auto step = [&](const U4 (&kr)[P], const U4 (&vr)[P], const int (&kidx)[P], const bool (&valid)[P],
                        const float (&mk)[P][SQ], bool rescale) {
            float s[P][R];
#pragma unroll
            for (int pp = 0; pp < P; ++pp)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int qi = r / G;
                    bool ok = valid[pp];
                    // several queries of a request without a mask: causal among the last keys
                    if constexpr (SQ > 1 && !MASK) ok = ok && kidx[pp] <= L - SQ + qi;
                    float x = group_sum<LPK>(lane_dot<T>(q[r], kr[pp])) * p.scale_log2;
                    if constexpr (MASK) x += mk[pp][qi];
                    s[pp][r] = ok ? x : -INFINITY;
                }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float mb = s[0][r];
#pragma unroll
                for (int pp = 1; pp < P; ++pp) mb = fmaxf(mb, s[pp][r]);
                const float mn = fmaxf(m[r], cross_max<LPK>(mb));
                if (rescale) {  // nothing to rescale before the first block
                    const float alpha = fexp2(m[r] - mn);
                    l[r] *= alpha;
#pragma unroll
                    for (int e = 0; e < CW; ++e) acc[r][e] *= alpha;
                }
                m[r] = mn;
#pragma unroll
                for (int pp = 0; pp < P; ++pp) {
                    const float w = fexp2(s[pp][r] - mn);
                    l[r] += w;
                    const uint32_t x[4] = {vr[pp].x, vr[pp].y, vr[pp].z, vr[pp].w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (ES == 2) {
                            acc[r][2 * i] += w * bf16_lo(x[i]);
                            acc[r][2 * i + 1] += w * bf16_hi(x[i]);
                        } else {
                            acc[r][i] += w * __uint_as_float(x[i]);
                        }
                    }
                }
            }
        };

        // mask terms of keys (log2 units), requested right after the block's key and value
        // rows so that the scores wait for one round trip, not two
        auto key_mask = [&](const int (&kidx)[P], const bool (&valid)[P], float (&mk)[P][SQ]) {
#pragma unroll
            for (int pp = 0; pp < P; ++pp)
#pragma unroll
                for (int qi = 0; qi < SQ; ++qi) {
                    mk[pp][qi] = 0.f;
                    if constexpr (MASK) {
                        if (valid[pp])
                            mk[pp][qi] = load_mask(mask_row + (qi * p.m_ss + (int64_t)kidx[pp] * p.m_st) *
                                                                  mask_elem_size(p.mask_dtype),
                                                   p.mask_dtype) * kLog2e;
                    }
                }
        };
        auto block_keys = [&](int jb, int (&kidx)[P], bool (&valid)[P]) {
#pragma unroll
            for (int pp = 0; pp < P; ++pp) {
                kidx[pp] = jb + pp * RPP + wave * RPW + grp;
                valid[pp] = kidx[pp] < jend;
            }
        };
        if constexpr (PIPE) {
            // two register buffers in turn (the loop handles two blocks per trip, so neither
            // buffer is ever copied): while one block is folded in, the next one is in flight.
            // The next block is requested unconditionally (rows past the range read zeros from
            // outside the buffer resource, without a memory access), so the number of loads in
            // flight is the same on every path and each block waits only for its own loads.
            U4 kb2[P], vb2[P];
            for (int jb = j0; jb < jend; jb += 2 * ROWS) {
                int kidx[P];
                bool valid[P];
                float mk[P][SQ];
                const int j2 = jb + ROWS;
                load_block(j2, kb2, vb2);
                block_keys(jb, kidx, valid);
                key_mask(kidx, valid, mk);
                step(kr, vr, kidx, valid, mk, jb != j0);
                if (j2 >= jend) break;
                load_block(j2 + ROWS, kr, vr);
                block_keys(j2, kidx, valid);
                key_mask(kidx, valid, mk);
                step(kb2, vb2, kidx, valid, mk, true);
            }
        } else {
            for (int jb = j0; jb < jend; jb += ROWS) {
                U4 kb_[P], vb_[P];
                int kidx[P];
                bool valid[P];
                float mk[P][SQ];
                load_block(jb, kb_, vb_);
                block_keys(jb, kidx, valid);
                key_mask(kidx, valid, mk);
                step(kb_, vb_, kidx, valid, mk, jb != j0);
            }
        }
        if constexpr (FUSED) {
            if (with_new && wave == 0) {  // the new keys: token t's in lane group t of wave 0
                U4 kr[P], vr[P];
                int kidx[P];
                bool valid[P];
                float mk[P][SQ];
                const U4 zero = {0u, 0u, 0u, 0u};
                const bool mine = grp < SQ && L - SQ + grp >= 0;
#pragma unroll
                for (int pp = 0; pp < P; ++pp) {
                    kr[pp] = (pp == 0 && mine) ? snew[0][grp < SQ ? grp : 0][cl] : zero;
                    vr[pp] = (pp == 0 && mine) ? snew[1][grp < SQ ? grp : 0][cl] : zero;
                    kidx[pp] = L - SQ + grp;
                    valid[pp] = pp == 0 && mine;
                }
                key_mask(kidx, valid, mk);
                step(kr, vr, kidx, valid, mk, j0 < jend);
            }
        }

        // the wave's state: sums across its lane groups, then into LDS
#pragma unroll
        for (int r = 0; r < R; ++r) l[r] = cross_sum<LPK>(l[r]);
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                lds.ml[wave][r][0] = m[r];
                lds.ml[wave][r][1] = l[r];
            }
        }
        store_wave_acc<LPK, CW, R, D>(acc, lds.acc[wave], lane);
        __syncthreads();
    }

    // Output t (query row t / D, dim t % D) of the waves' states: accumulator, weight sum, maximum.
    static Q3T_DEVICE void merge(const Lds &lds, int t, float &sa, float &sl, float &mx) {
        const int r = t / D, d = t % D;
        mx = lds.ml[0][r][0];
#pragma unroll
        for (int w = 1; w < W; ++w) mx = fmaxf(mx, lds.ml[w][r][0]);
        sl = 0.f;
        sa = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float wt = fexp2(lds.ml[w][r][0] - mx);
            sl += lds.ml[w][r][1] * wt;
            sa += lds.acc[w][r][d] * wt;
        }
    }

    Q3T_DEVICE void attend(const DecodeParams &p, int b, int h, int L, int j0, int j1, bool finisher,
                           Lds &lds, NewRows &snew, float (&A)[OPL], float (&Ls)[OPL], float (&Mx)[OPL]) {
        stream(p, b, h, L, j0, j1, finisher, lds, snew);
        if ((threadIdx.x >> 6) != 0) return;
#pragma unroll
        for (int i = 0; i < OPL; ++i) merge(lds, (threadIdx.x & 63) + 64 * i, A[i], Ls[i], Mx[i]);
    }
};

}  // namespace q3t
