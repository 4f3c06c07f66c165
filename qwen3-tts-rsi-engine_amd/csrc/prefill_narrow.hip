// Prefill attention of one-head groups (as many KV heads as query heads) in launches of few
// workgroups, where the longest block's chain of tiles is the launch.
//
// One workgroup of 4 waves per (request, 64-query block, head), a wave its 16 queries on 16x16
// products: half the products of a 32-column wave per step, and with one head there is nothing to
// fill the other 16 columns.  The ring, the swizzles and the softmax are prefill_attention.hip's; the
// value rows (new_values) are copied by as many workgroups again, on CUs that would stay idle.
// us per layer, 128-query blocks of 32 columns / this form: one prompt of 464 rows and 16 heads 20.7 /
// 19.8, 2 x 200 16.5 / 14.4, 1 x 1024 under a bf16 mask 39.9 / 33.6 (the line: narrow_blocks).
#include "prefill_params.hpp"

namespace q3t {
namespace narrow {

constexpr int kQBlock = 64;   // queries per workgroup, 16 per wave
constexpr int kTile = kKeys;  // keys per LDS stage and per softmax step
constexpr int kStages = 3;    // LDS ring depth: loads run kStages - 1 tiles ahead

template <int D, int MB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
prefill_narrow_kernel(const int32_t *cu, const int64_t *slots, int nb, PrefillParams p) {
    constexpr int NT = 256;                       // threads
    constexpr int KK = D / 32;                    // MFMA steps over the head dimension
    constexpr int DB = D / 16;                    // 16-row blocks of O^T
    constexpr int CPR = D / 8;                    // 16-byte chunks per row
    constexpr int ROW = D * 2;                    // bytes per row
    constexpr int KBYTES = kTile * ROW;           // K part of a stage
    constexpr int RB = kTile * MB;                // mask bytes per query row of a tile
    constexpr int MBYTES = kQBlock * RB;          // mask tile of a stage
    constexpr int SBYTES = 2 * KBYTES + MBYTES;   // stage: K rows, V rows, mask rows
    constexpr int LPT = 2 * kTile * CPR / NT;     // 16-byte loads per thread per tile
    constexpr int LPR = MB ? RB / 16 : 1;         // lanes per mask row
    constexpr int RPI = 64 / LPR;                 // mask rows per wave load
    constexpr int LPTM = MB ? 16 / RPI : 0;       // mask loads per wave per tile (16 rows)
    constexpr int WAIT = LPT + LPTM;              // loads of one tile per thread
    static_assert(LPT >= 1 && (2 * kTile * CPR) % NT == 0, "a tile is whole loads per thread");
    static_assert(KBYTES % 1024 == 0, "a wave's load never straddles K and V");
    __shared__ __attribute__((aligned(1024))) uint8_t ring[kStages * SBYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    int start = 0, next = 0;
    int64_t slot_l = lane;
    if (nb <= 64 && lane < nb) {
        start = cu[lane];
        next = cu[lane + 1];
        if (slots) slot_l = slots[lane];
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: resources stay scalar
    const int g = lane >> 4, c = lane & 15;
    const bool copies = (int)blockIdx.x >= p.attn_wgs;  // past the attention grid: value rows to copy
    const int wg = copies ? (int)blockIdx.x - p.attn_wgs : place_workgroup(blockIdx.x, p.attn_wgs);
    const int h = wg % p.Hq, rest = wg / p.Hq;
    if (copies && wg >= p.attn_wgs) {  // past these: rows that no block covers
        copy_other_rows<D, false>(p, cu, slots, nb, wg - p.attn_wgs, (int64_t)p.nqb * kQBlock);
        return;
    }
    PrefillItem item;
    if (!find_item<kQBlock>(p, cu, slots, nb, start, next, slot_l, rest, item)) return;
    const int b = item.b, t0 = item.t0, n = item.n, kn = item.kn, q0 = item.qb * kQBlock;
    const int64_t slot = item.slot;
    if (copies) {
        copy_uncovered_rows<D, false>(p, h, slot, t0, q0, (int64_t)t0 + min(n, q0 + kQBlock));
        return;
    }
    // keys 0 ... kv_end-1 are visible to this block; the arena holds at most `cap` of them.
    // Causal: up to the block's last query and the request's key count; masked: every key.
    const int kv_end = MB ? (int)p.cap : (int)min((int64_t)min(min(n, kn), q0 + kQBlock), p.cap);
    const int ntiles = kv_end > 0 ? (kv_end + kTile - 1) / kTile : 0;
    const int wq0 = q0 + 16 * wave;              // first query of this wave
    // keys [0, wave_end) can be visible to the wave; steps reaching past mask_from need the
    // per-key rule (the diagonal or the end of the keys).  A wave whose queries all lie past
    // the request (the tail of its last block) scores nothing: it only loads its share of
    // every tile and joins the barriers.
    const int wave_end = wq0 >= n ? 0 : MB ? kv_end : min(wq0 + 16, kv_end);
    const int mask_from = MB ? kv_end : min(wq0 + 1, kv_end);
    const int qpos = wq0 + c;
    const bool qvalid = qpos < n;
    const int lim = MB ? kv_end - 1 : min(qpos, kv_end - 1);  // last key visible to this lane's query

    // tile loader: load i of a thread fills LDS slot s = i * NT + tid (16 bytes) of a stage:
    // row s / CPR (K rows first, then V rows), physical chunk s % CPR, holding logical chunk
    // (physical ^ swizzle(row)) of key tile * kTile + row
    const char *kbase = p.k + (slot * p.k_sb + h * p.k_sh) * 2;
    const char *vbase = MB == 0 && p.nv ? p.nv + ((int64_t)t0 * p.nv_st + h * p.nv_sh) * 2
                                        : p.v + (slot * p.v_sb + h * p.v_sh) * 2;
    const uint32_t kst = (uint32_t)(p.k_st * 2), vst = (uint32_t)((MB == 0 && p.nv ? p.nv_st : p.v_st) * 2);
    const i32x4_t krs = scalar_rsrc(kbase, kv_end > 0 ? (uint32_t)((kv_end - 1) * kst + D * 2) : 0u);
    const i32x4_t vrs = scalar_rsrc(vbase, kv_end > 0 ? (uint32_t)((kv_end - 1) * vst + D * 2) : 0u);
    // mask rows of the request's queries (rows past its queries read zeros)
    const uint32_t mrow = (uint32_t)(p.m_sq * MB);
    const i32x4_t mrs = scalar_rsrc(MB ? p.mask + b * p.m_sb * MB : kbase,
                                    MB ? (uint32_t)((n - 1) * (int64_t)mrow + p.cap * MB) : 0u);
    const uint32_t ring_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
    uint32_t row_off[LPT];
    int row_of[LPT];
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
        const int s = i * NT + tid, rall = s / CPR, pc = s % CPR;
        const bool is_v = rall >= kTile;
        const int r = rall % kTile;
        const int ch = pc ^ ((is_v ? 2 * r : r) & (CPR - 1));
        row_of[i] = r;
        row_off[i] = (uint32_t)r * (is_v ? vst : kst) + ch * 16;
    }
    auto issue = [&](int kt, int stage) {
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
            const int first_slot = i * NT + wave * 64;             // wave-uniform
            const bool is_v = first_slot / CPR >= kTile;
            const int key0 = kt * kTile;
            const uint32_t off = row_of[i] < kv_end - key0
                                     ? row_off[i] + (uint32_t)key0 * (is_v ? vst : kst)
                                     : 0xfffffff0u;
            load_to_lds16(is_v ? vrs : krs, off,
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)(ring_base + stage * SBYTES + first_slot * 16)));
        }
        if constexpr (MB > 0) {
            // the wave's own 16 query rows of the mask tile: load i covers rows RPI i ... + RPI - 1
#pragma unroll
            for (int i = 0; i < LPTM; ++i) {
                const int r = 16 * wave + i * RPI + lane / LPR;
                const uint32_t off = q0 + r < n ? (uint32_t)(q0 + r) * mrow + (uint32_t)(kt * RB + (lane % LPR) * 16)
                                                : 0xfffffff0u;
                load_to_lds16(mrs, off, (uint32_t)__builtin_amdgcn_readfirstlane(
                                            (int)(ring_base + stage * SBYTES + 2 * KBYTES + (16 * wave + i * RPI) * RB)));
            }
        }
    };

    // per-lane LDS read addresses within a stage
    uint32_t ka[KK], va[DB];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) ka[kk] = c * ROW + (((4 * kk + g) ^ (c & (CPR - 1))) * 16);
    {
        const int r = 4 * g + (c >> 2);  // key row of this lane's transposed read (+16 for keys 16..31)
        const int sw = (2 * r) & (CPR - 1);
#pragma unroll
        for (int db = 0; db < DB; ++db)
            va[db] = KBYTES + r * ROW + (((2 * db + ((c >> 1) & 1)) ^ sw) * 16) + 8 * (c & 1);
    }

    // the first tiles go out before anything else waits on memory
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
        if (s < ntiles) issue(s, s);

    // the wave's query rows as B operands: Q[query c][8g + 32kk ...], zeros past the request
    bf16x8_t qB[KK];
    // with cos/sin: the lane's RoPE rows (its query token, dims 32kk + 8g ... + 7 and the same
    // dims D/2 further)
    U4 rc1[KK / 2], rc2[KK / 2], rs1[KK / 2], rs2[KK / 2];
    if (p.cs) {
        const int64_t tr = (int64_t)(t0 + (qvalid ? qpos : 0)) * p.cs_st * 2;
#pragma unroll
        for (int kk = 0; kk < KK / 2; ++kk) {
            const int d1 = (32 * kk + 8 * g) * 2, d2 = d1 + D;  // bytes of dims d and d + D/2
            rc1[kk] = load16(p.cs + tr + d1);
            rc2[kk] = load16(p.cs + tr + d2);
            rs1[kk] = load16(p.sn + tr + d1);
            rs2[kk] = load16(p.sn + tr + d2);
        }
    }
    {
        const char *row = p.q + ((int64_t)(t0 + (qvalid ? qpos : 0)) * p.q_st + h * p.q_sh) * 2;
        U4 qv[KK];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qv[kk] = load16(row + (32 * kk + 8 * g) * 2);
        if (p.cs) {
            // rotate-half RoPE in registers (bf16-exact; the rotated rows are never stored, so NaN
            // payloads need no canonical form): the lane's dims 32kk + 8g ... + 7 pair with the same
            // dims of kk + KK/2, which the lane holds as well
#pragma unroll
            for (int kk = 0; kk < KK / 2; ++kk) {
                U4 y1, y2;
                rope8<false>(&qv[kk].x, &qv[kk + KK / 2].x, &rc1[kk].x, &rc2[kk].x, &rs1[kk].x, &rs2[kk].x,
                             &y1.x, &y2.x);
                qv[kk] = y1;
                qv[kk + KK / 2] = y2;
            }
        }
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            if (!qvalid) qv[kk] = U4{0u, 0u, 0u, 0u};
            qB[kk] = as_bf16x8(qv[kk]);
        }
    }

    f32x4_t acc[DB];
    float m = 0.f, l = 0.f;  // running maximum (scaled log2 units) and this lane's weight sum
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bool first = true;
    const float sl = p.scale_log2;

    auto step = [&](int kt, uint32_t sbase) {
        const int kb0 = kt * kTile;  // first key of the step
        if (kb0 >= wave_end) return;  // past this wave's keys
        const bool masked = kb0 + kTile > mask_from;  // the step reaches past the diagonal or the keys
        const int rel = lim - kb0;
        float mk[8];
        if constexpr (MB > 0) {
            const uint32_t mrow_lds = sbase + 2 * KBYTES + (16 * wave + c) * RB;
            float lo[4], hi[4];
            mask_values<MB>(mrow_lds + 4 * g * MB, p.mdt, lo);
            mask_values<MB>(mrow_lds + (16 + 4 * g) * MB, p.mdt, hi);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                mk[i] = lo[i];
                mk[4 + i] = hi[i];
            }
        }
        // S^T of keys kb0 + 16kb + (4g..4g+3); a wave issuing products goes
        // first, the others do their softmax meanwhile
        f32x4_t st0 = {0.f, 0.f, 0.f, 0.f}, st1 = {0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const bf16x8_t a0 = as_bf16x8(lds_read16(sbase + ka[kk]));
            const bf16x8_t a1 = as_bf16x8(lds_read16(sbase + ka[kk] + 16 * ROW));
            st0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, qB[kk], st0, 0, 0, 0);
            st1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, qB[kk], st1, 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        float x[8] = {st0[0], st0[1], st0[2], st0[3], st1[0], st1[1], st1[2], st1[3]};
        if constexpr (MB > 0) {  // scores in log2 units with the mask added
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = __builtin_fmaf(x[e], sl, mk[e]);
        }
        if (masked) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (4 * g + i > rel) x[i] = -INFINITY;
                if (16 + 4 * g + i > rel) x[4 + i] = -INFINITY;
            }
        }
        float mx = x[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = __builtin_amdgcn_fmed3f(mx, x[e], __builtin_inff());
        // the step maximum of a query is the largest of its four lanes' maxima (scaling is
        // monotonic, so it commutes with the maximum): some query exceeds its running maximum
        // by more than kRescaleLog2 exactly when some lane's own maximum does, and the
        // maximum across lanes is needed only to start and to rescale
        float mt = MB ? mx : mx * sl;
        if (first || __builtin_amdgcn_ballot_w64(mt > m + kRescaleLog2) != 0) {
            mt = __builtin_amdgcn_fmed3f(mt, xor16(mt), __builtin_inff());
            mt = __builtin_amdgcn_fmed3f(mt, xor32(mt), __builtin_inff());
            if constexpr (MB > 0) mt = fmaxf(mt, kEmptyP);  // a fully masked step keeps m finite
            if (first) {
                m = mt;
            } else {
                const float mn = fmaxf(m, mt);
                const float alpha = fexp2(m - mn);
                m = mn;
                l *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db) acc[db] *= alpha;
            }
        }
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = MB ? fexp2(x[e] - m) : fexp2(__builtin_fmaf(x[e], sl, -m));
        l += ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
        const U4 packed = {cvt_pk_bf16(pv[0], pv[1]), cvt_pk_bf16(pv[2], pv[3]),
                           cvt_pk_bf16(pv[4], pv[5]), cvt_pk_bf16(pv[6], pv[7])};
        const bf16x8_t pB = as_bf16x8(packed);
        first = false;
        // O^T += V^T . P^T
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const uint2 lo = lds_read_tr16(sbase + va[db]), hi = lds_read_tr16(sbase + va[db] + 16 * ROW);
            const bf16x8_t av = as_bf16x8(U4{lo.x, lo.y, hi.x, hi.y});
            acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, pB, acc[db], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // one ring position: wait for this tile's loads (later tiles stay in flight), barrier
    // (every wave is done with the stage the next load overwrites), issue the tile
    // kStages - 1 ahead into that stage, then the products
    auto ring_step = [&](int kt, int stage) {
        if (kt + 1 < ntiles) wait_loads<WAIT>();  // the one younger tile stays in flight
        else wait_loads<0>();
        lds_barrier();
        if (kt + kStages - 1 < ntiles) issue(kt + kStages - 1, (stage + kStages - 1) % kStages);
        step(kt, ring_base + stage * SBYTES);
    };
    static_assert(kStages == 3, "the waits above and the unrolled ring below assume three stages");
    for (int kt = 0; kt < ntiles; kt += kStages) {
        ring_step(kt, 0);
        if (kt + 1 < ntiles) ring_step(kt + 1, 1);
        if (kt + 2 < ntiles) ring_step(kt + 2, 2);
    }

    if (!qvalid) return;
    float lt = l + xor16(l);
    lt += xor32(lt);
    const float inv = lt > 0.f ? __builtin_amdgcn_rcpf(lt) : 0.f;  // no visible key: zero row
    char *orow = p.out + ((int64_t)(t0 + qpos) * p.o_st + h * p.o_sh) * 2;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        const uint2 v = {cvt_pk_bf16(acc[db][0] * inv, acc[db][1] * inv),
                         cvt_pk_bf16(acc[db][2] * inv, acc[db][3] * inv)};
        *reinterpret_cast<uint2 *>(orow + (16 * db + 4 * g) * 2) = v;
    }
}

template <int D>
static void launch(const PrefillParams &p, dim3 grid, hipStream_t s) {
    if (!p.mask) hipLaunchKernelGGL((prefill_narrow_kernel<D, 0>), grid, dim3(256), 0, s, p.cu, p.slots, p.B, p);
    else if (p.mdt == Q3T_F32) hipLaunchKernelGGL((prefill_narrow_kernel<D, 4>), grid, dim3(256), 0, s, p.cu, p.slots, p.B, p);
    else hipLaunchKernelGGL((prefill_narrow_kernel<D, 2>), grid, dim3(256), 0, s, p.cu, p.slots, p.B, p);
}

}  // namespace narrow

void launch_prefill_narrow(const PrefillParams &p, int64_t head_dim, int64_t max_seqlen, hipStream_t s) {
    using namespace narrow;
    PrefillParams q = p;
    q.nqb = (int)((max_seqlen + kQBlock - 1) / kQBlock);
    q.by_request = 0;
    q.attn_wgs = (int)prefill_workgroups(p, kQBlock, p.Hq, max_seqlen);
    const dim3 grid((uint32_t)(p.nv ? 2 * q.attn_wgs + other_row_workgroups(p) : q.attn_wgs));
    if (head_dim == 128) launch<128>(q, grid, s);
    else launch<64>(q, grid, s);
}

}  // namespace q3t
