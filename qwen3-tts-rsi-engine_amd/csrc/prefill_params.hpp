// What the prefill attention kernels share: their arguments, the numbering of their work items and
// the arena rows of tokens that no query block covers.
#pragma once

#include "q3t_common.hpp"

namespace q3t {

constexpr int kXcds = 8;        // MI355X: 8 XCDs of 32 CUs
constexpr int kCusPerXcd = 32;
constexpr int kKeys = 32;     // keys of one MFMA block of scores
constexpr float kLog2eP = 1.4426950408889634f;
constexpr float kRescaleLog2 = 8.0f;

struct PrefillParams {
    int B, Hq, Hkv, nqb, group;
    int64_t T;
    float scale_log2;
    const int32_t *cu;
    const char *q;
    int64_t q_st, q_sh;
    const char *k;
    char *v;  // written only with nv
    int64_t k_sb, k_sh, k_st, v_sb, v_sh, v_st;
    int64_t cap;
    const int64_t *slots;
    char *out;
    int64_t o_st, o_sh;
    const char *cs, *sn;  // optional cos/sin rows per token: the query rows are rotated on load
    int64_t cs_st;
    const int32_t *kvl;   // optional keys per request (a right-padded batch): query i sees keys
                          // j <= i with j < kvl[b]
    const char *mask;     // optional (B, 1, Lq, capacity) additive mask: every key is scored
    int mdt;              // mask element type (Q3T_BF16, Q3T_F16 or Q3T_F32)
    int64_t m_sb, m_sq;   // mask strides (elements) of requests and query rows; keys unit-stride
    // optional value rows of the step's tokens as the projection wrote them: the products
    // read them (key j of request b is token cu[b] + j) and each workgroup copies those of its
    // query block into the arena view `v` at their positions
    const char *nv;
    int64_t nv_st, nv_sh;
    // key rows of the step's tokens before their rotation: the launch rotates each tile in LDS
    // and writes its block's rows into the arena (instances that rotate keys only)
    const char *nk;
    int64_t nk_st, nk_sh;
    int by_request;       // work items numbered request by request
    int attn_wgs;         // narrow form: workgroups that attend (as many that copy values follow)
};

// Workgroups of a launch of `heads` head groups and blocks of `block` queries.  Items are numbered
// densely up to 64 requests: a request of L rows has ceil(L / block) blocks, so there are at most
// (T + (block - 1) B) / block of them; rounded up to whole rounds of one workgroup per CU, which
// keeps the placement of every item as in the full grid.
inline int64_t prefill_workgroups(const PrefillParams &p, int64_t block, int64_t heads, int64_t max_seqlen) {
    const int64_t wgs = p.B * ((max_seqlen + block - 1) / block) * heads;
    if (p.B > 64) return wgs;
    const int64_t items = (p.T + (block - 1) * p.B) / block, round = kXcds * kCusPerXcd;
    const int64_t bound = (items * heads + round - 1) / round * round;
    return bound < wgs ? bound : wgs;
}

// Workgroups that look for rows that no query block covers (copy_other_rows), with new rows.
inline int64_t other_row_workgroups(const PrefillParams &p) { return p.nv ? (int64_t)p.Hkv * ((p.B + 63) / 64) : 0; }

// The form for one-head groups in launches of few workgroups (prefill_narrow.hip).
void launch_prefill_narrow(const PrefillParams &p, int64_t head_dim, int64_t max_seqlen, hipStream_t s);

constexpr float kEmptyP = -1.0e30f;  // finite running maximum before any visible key (masked)

// 16 bytes of a mask tile row in LDS -> 4 (2-byte types) or 2 x 2 (fp32: two reads) values in
// log2 units; positive infinity never occurs in an additive mask, -inf (and finfo.min, which
// overflows to -inf once scaled) gives a zero weight.
template <int MB>
Q3T_DEVICE void mask_values(uint32_t addr, int mdt, float (&mv)[4]) {
    if constexpr (MB == 2) {
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
        const u32x2_t w = *(__attribute__((address_space(3))) const u32x2_t *)(uintptr_t)addr;
        const uint32_t h[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = mdt == Q3T_F16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)h[i])
                                           : bf16_to_float(h[i]);
            mv[i] = v * kLog2eP;
        }
    } else {
        const U4 w = lds_read16(addr);
        const uint32_t f[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) mv[i] = __uint_as_float(f[i]) * kLog2eP;
    }
}

// Arena rows of one KV head for packed tokens that no query block covers: tokens t0 + pos0 ... t1 - 1
// of a request starting at t0 keep their place, as the prologue gives them theirs.  Values, and
// with RK the rotated keys.  A thread takes chunks ch and ch + CPR/2 of a row.
template <int D, bool RK>
Q3T_DEVICE void copy_uncovered_rows(const PrefillParams &p, int h, int64_t slot, int t0, int pos0, int64_t t1) {
    constexpr int HALF = D / 16;  // chunks of half a row
    const int64_t end = min(t1 - t0, p.cap);
#pragma unroll 1
    for (int64_t pos = (int64_t)pos0 + threadIdx.x / HALF; pos < end; pos += 256 / HALF) {
        const int ch = threadIdx.x % HALF;
        const int64_t t = t0 + pos;
        const char *v = p.nv + (t * p.nv_st + h * p.nv_sh) * 2 + ch * 16;
        char *av = p.v + (slot * p.v_sb + h * p.v_sh + pos * p.v_st) * 2 + ch * 16;
        store16(av, load16(v));
        store16(av + D, load16(v + D));
        if constexpr (RK) {
            const char *k = p.nk + (t * p.nk_st + h * p.nk_sh) * 2 + ch * 16;
            const char *cr = p.cs + t * p.cs_st * 2 + ch * 16, *sr = p.sn + t * p.cs_st * 2 + ch * 16;
            char *ak = const_cast<char *>(p.k) + (slot * p.k_sb + h * p.k_sh + pos * p.k_st) * 2 + ch * 16;
            U4 x1 = load16(k), x2 = load16(k + D), c1 = load16(cr), c2 = load16(cr + D), s1 = load16(sr), s2 = load16(sr + D), y1, y2;
            rope8(&x1.x, &x2.x, &c1.x, &c2.x, &s1.x, &s2.x, &y1.x, &y2.x);
            store16(ak, y1);
            store16(ak + D, y2);
        }
    }
}

// Work item `item` of the rows that no query block covers, of a KV head and up to 64 requests: rows of
// requests longer than `covered`, and the tokens past the last request's end, which go on at its next
// positions.
template <int D, bool RK>
Q3T_DEVICE void copy_other_rows(const PrefillParams &p, const int32_t *cu, const int64_t *slots, int nb, int item, int64_t covered) {
    const int h = item % p.Hkv, b0 = item / p.Hkv * 64, lane = threadIdx.x & 63;
    int t0 = -1, t1 = -1;
    if (b0 + lane < nb) {
        t0 = cu[b0 + lane];
        t1 = cu[b0 + lane + 1];
    }
    const int64_t rows = t0 < 0 || t0 >= p.T ? 0 : min((int64_t)t1 - t0, p.T - t0);
    const int last = nb - 1 - b0;  // the last request's lane, past 63 in an earlier item
    const bool past = lane == last && t0 >= 0 && t1 >= t0 && t1 < p.T;
    uint64_t longer = __builtin_amdgcn_ballot_w64(rows > covered), open = __builtin_amdgcn_ballot_w64(past);
    // a request longer than covered from there to its end; then the last one from its end on
    while (longer | open) {
        const int l = __builtin_ctzll(longer ? longer : open), b = b0 + l;
        const int from = __builtin_amdgcn_readlane(t0, l), end = __builtin_amdgcn_readlane(t1, l);
        const int64_t slot = slots ? slots[b] : b;
        copy_uncovered_rows<D, RK>(p, h, slot, from, longer ? (int)covered : end - from, longer ? min((int64_t)end, p.T) : p.T);
        if (longer) longer &= longer - 1;
        else open = 0;
    }
}

// Placement: the hardware deals workgroup i to XCD i % 8 and, within an XCD, to its 32 CUs
// in turn, so CU k of an XCD holds the XCD's workgroups k, k + 32, k + 64 at once (three
// per CU).  Work items are numbered longest first; reversing the order within the second
// and third of every four rounds of 32 puts a short item next to every long one on a CU.
// Measured on the 16-prompt workload (seed 0): the most loaded CU from 27 to 20 tiles.
Q3T_DEVICE int place_workgroup(uint32_t index, int count) {
    const int xcd = index % kXcds, j = index / kXcds;
    const int rounds = count / (kXcds * kCusPerXcd);  // complete rounds on every XCD
    if (j >= rounds * kCusPerXcd) return (int)index;
    const int r = j / kCusPerXcd, pos = j % kCusPerXcd;
    const bool flip = (r & 3) == 1 || (r & 3) == 2;
    return (r * kCusPerXcd + (flip ? kCusPerXcd - 1 - pos : pos)) * kXcds + xcd;
}

struct PrefillItem {
    int b, qb, t0, n, kn;  // request, query block, the request's first token, rows and keys
    int64_t slot;
};
// Work item `rest` of this head group: a (query block qb, request b) pair, numbered with
// the longest blocks first.  Up to 64 requests the numbering is dense: only pairs with
// rows exist, so the grid's round-robin placement over shader engines sees real work
// evenly (empty slots in between would pile long blocks onto some engines and stall the
// in-order dispatch behind them).  Lane i holds request i's row range; each level counts
// the requests with a block there (ballot) and the item's request is picked by rank
// (mbcnt), all wave-uniform, with no memory access beyond the row offsets.  `start`, `next`,
// `slot_l`: the lane's request's first token, the next one's and its slot (up to 64 requests).
// False: there is no such item.
template <int QB>
Q3T_DEVICE bool find_item(const PrefillParams &p, const int32_t *cu, const int64_t *slots, int nb, int start, int next,
                          int64_t slot_l, int rest, PrefillItem &item) {
    const int lane = threadIdx.x & 63;
    int &b = item.b, &qb = item.qb, &t0 = item.t0, &n = item.n, &kn = item.kn;
    int64_t &slot = item.slot;
    if (nb <= 64) {
        int rows = 0, klen = 0;
        if (lane < nb) {
            rows = (start < 0 || start >= p.T) ? 0 : (int)min((int64_t)(next - start), p.T - start);
            klen = p.kvl ? p.kvl[lane] : rows;
        }
        const int blocks = rows > 0 ? (rows + QB - 1) / QB : 0;
        qb = -1;
        b = 0;
        if (p.by_request) {
            // blocks of requests 0 ... lane; of a request longer than the caller said, those that the
            // grid was sized for
            int before = min(blocks, p.nqb);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int y = __shfl_up(before, off);
                if (lane >= off) before += y;
            }
            const uint64_t done = __builtin_amdgcn_ballot_w64(before <= rest);  // requests wholly before the item
            if (~done) {
                b = __builtin_ctzll(~done);
                qb = __builtin_amdgcn_readlane(before, b) - 1 - rest;
            }
        } else {
            int remaining = rest;
            for (int level = p.nqb - 1; level >= 0; --level) {
                const uint64_t has = __builtin_amdgcn_ballot_w64(blocks > level);
                const int count = __builtin_popcountll(has);
                if (remaining < count) {
                    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32),
                                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
                    const uint64_t pick = __builtin_amdgcn_ballot_w64(blocks > level && (int)rank == remaining);
                    b = __builtin_ctzll(pick);
                    qb = level;
                    break;
                }
                remaining -= count;
            }
        }
        if (qb < 0) return false;  // past the last block with rows
        t0 = __builtin_amdgcn_readlane(start, b);
        n = __builtin_amdgcn_readlane(rows, b);
        kn = __builtin_amdgcn_readlane(klen, b);
        slot = ((int64_t)__builtin_amdgcn_readlane((int)(slot_l >> 32), b) << 32) |
               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)slot_l, b);
    } else {
        b = rest % p.B;
        qb = p.nqb - 1 - rest / p.B;  // the longest blocks are dispatched first
        t0 = cu[b];
        if (t0 < 0 || t0 >= p.T) return false;
        n = (int)min((int64_t)(cu[b + 1] - t0), p.T - t0);  // rows past the packed tokens do not exist
        kn = p.kvl ? p.kvl[b] : n;
        slot = slots ? slots[b] : b;
    }
    return qb * QB < n;
}

}  // namespace q3t
