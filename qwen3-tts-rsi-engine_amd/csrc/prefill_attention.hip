// Varlen causal prefill: RoPE + arena write prologue and the attention kernel.
//
// Reference behaviour: PrefillGraph.compute (prefill_graph.py:31-50) runs padded causal
// self-attention with positions cumsum(mask)-1 and mask key_valid & causal; the per-layer
// prefill KV is later copied into the request's arena slot (continuous.py:468-471,
// packed_kv.py:6-31).  Here requests are packed along the token axis by cu_seqlens, so
// only valid rows exist, and rotated keys/values go straight into the arena slot.
#include "prefill_params.hpp"

namespace q3t {

struct PrefillRopeWriteParams {
    int B, Hq, Hkv, D;
    int64_t T, capacity;
    const int32_t *cu;
    const char *q, *k, *v;
    int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh;
    const char *cs, *sn;
    int64_t cs_st;
    char *qo;
    int64_t qo_st, qo_sh;
    char *ak, *av;
    int64_t a_sb, a_sh, a_st;
    const int64_t *slots;
};

Q3T_DEVICE int request_of(const int32_t *cu, int B, int64_t t) {
    int lo = 0, hi = B - 1;  // last b with cu[b] <= t
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cu[mid] <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// One wave per token; a lane's work item is 8 dims of each half of one of the token's head
// rows.  Heads [0, Hq) are query heads (rotated into q_out; absent when q_out is null, the
// attention kernel then rotates the queries itself); the Hkv heads after them rotate the key
// and copy the value into the arena at the token's position within its request (without value
// rows, p.v null, only the keys: the attention launch copies the values).  The token's
// request, position and slot are the same for the whole wave: 12.5 -> 12.0 us per layer on
// the 16-prompt workload (keys and values) against one item per thread with per-lane lookups,
// and 12.0 -> 11.0 us with the request found by one ballot instead of a binary search of
// dependent loads; keys only, 6.5 us.  (Two tokens per wave, the next one's rows requested
// before the current one's are stored, or non-temporal stores: no gain.)
__global__ void __launch_bounds__(256) prefill_rope_write_kernel(PrefillRopeWriteParams p) {
    const int vecs = p.D / 16;
    const int qh = p.qo ? p.Hq : 0;  // without q_out only the key/value rows are handled
    const int items = (qh + p.Hkv) * vecs;
    const int half = p.D / 2;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Up to 64 requests, lane i holds request i's first token and slot, loaded once per wave in
    // one round trip; a token's request is then a ballot (the count of requests starting at or
    // before it, less one), not a binary search of dependent loads.
    int start_l = 0x7fffffff;
    int64_t slot_l = 0;
    if (p.B <= 64 && lane < p.B) {
        start_l = p.cu[lane];
        slot_l = p.slots ? p.slots[lane] : lane;
    }
    // a token's request: the last one starting at or before it
    auto locate = [&](int t, int &pos, int64_t &slot) {
        if (p.B <= 64) {
            const int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(start_l <= t));
            const int b = n > 0 ? n - 1 : 0;
            pos = t - __builtin_amdgcn_readlane(start_l, b);
            slot = ((int64_t)__builtin_amdgcn_readlane((int)(slot_l >> 32), b) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)slot_l, b);
        } else {
            const int b = request_of(p.cu, p.B, t);
            pos = t - p.cu[b];
            slot = p.slots ? p.slots[b] : b;
        }
    };
    for (int t = blockIdx.x * 4 + wave; t < (int)p.T; t += gridDim.x * 4) {
        int pos;
        int64_t slot;
        locate(t, pos, slot);
        const bool write_kv = pos >= 0 && pos < p.capacity;
        const char *crow = p.cs + (int64_t)t * p.cs_st * 2, *srow = p.sn + (int64_t)t * p.cs_st * 2;
        for (int it = lane; it < items; it += 64) {
            const int c = it % vecs, hd = it / vecs;
            U4 c1 = load16(crow + c * 16), c2 = load16(crow + (half + c * 8) * 2);
            U4 s1 = load16(srow + c * 16), s2 = load16(srow + (half + c * 8) * 2);
            if (hd < qh) {
                const char *row = p.q + ((int64_t)t * p.q_st + hd * p.q_sh) * 2;
                U4 x1 = load16(row + c * 16), x2 = load16(row + (half + c * 8) * 2), y1, y2;
                rope8(&x1.x, &x2.x, &c1.x, &c2.x, &s1.x, &s2.x, &y1.x, &y2.x);
                char *orow = p.qo + ((int64_t)t * p.qo_st + hd * p.qo_sh) * 2;
                store16(orow + c * 16, y1);
                store16(orow + (half + c * 8) * 2, y2);
            } else if (write_kv) {
                const int h = hd - qh;
                const char *krow = p.k + ((int64_t)t * p.k_st + h * p.k_sh) * 2;
                U4 x1 = load16(krow + c * 16), x2 = load16(krow + (half + c * 8) * 2), y1, y2;
                U4 w1 = {0u, 0u, 0u, 0u}, w2 = w1;
                if (p.v) {  // without value rows the attention launch copies them
                    const char *vrow = p.v + ((int64_t)t * p.v_st + h * p.v_sh) * 2;
                    w1 = load16(vrow + c * 16);
                    w2 = load16(vrow + (half + c * 8) * 2);
                }
                rope8(&x1.x, &x2.x, &c1.x, &c2.x, &s1.x, &s2.x, &y1.x, &y2.x);
                const int64_t a = (slot * p.a_sb + h * p.a_sh + pos * p.a_st) * 2;
                store16(p.ak + a + c * 16, y1);
                store16(p.ak + a + (half + c * 8) * 2, y2);
                if (p.v) {
                    store16(p.av + a + c * 16, w1);
                    store16(p.av + a + (half + c * 8) * 2, w2);
                }
            }
        }
    }
}


// ---- varlen causal attention on bf16 MFMA tiles ------------------------------------------
//
// One workgroup of 4 waves per (request, query block, GH query heads of one KV head).  A wave
// owns 32 columns: with GH = 2 the two heads' rows of 16 queries (64-query blocks), with GH = 1
// 32 queries of one head (128-query blocks); every K and V row read from LDS feeds all 32.
// Keys stream through a ring of kStages LDS stages of kTile keys (K rows then V rows), filled by
// buffer loads that write LDS directly (16 bytes per lane) kStages - 1 tiles ahead of the
// products, so the K/V reads never pass through registers.  With v_mfma_f32_32x32x16_bf16 (lane
// l = 32 hi + c holds A[c][8 hi ... 8 hi + 7], B[8 hi ... 8 hi + 7][c] and D[8 i + 4 hi ... + 3][c],
// i = 0..3), per 32 keys:
//   S^T (keys x columns) = K . Q^T   A = K rows from LDS, B = the wave's query rows (registers);
//                                    lane (hi, c) gets keys 8 i + 4 hi + {0..3} of column c;
//   O^T (dims x columns) += V^T . P^T   B = P^T straight from the S^T registers (contraction
//                                    order, per 16 keys: 4 hi + {0..3}, 8 + 4 hi + {0..3}); A = V^T
//                                    read by ds_read_b64_tr_b16 in that order: within a 16-lane
//                                    group, lane i reads 4 dims of key row i/4 and receives, after
//                                    the transpose, 4 keys of dim i.
// A lane keeps the online softmax of one column, and one column's keys sit in two lanes, so a
// step costs one maximum, one threshold and one sum per lane and 24 LDS reads for 16 products.
// (The same tiles as 16x16x32 products, a head after the other, took 40 LDS reads, 32 products and
// two softmax states per step.)
// What bounds it: where the launch fills the card, memory and the workgroups' start as much as the
// products (16 prompts of 32..512 with no tile at all: 19 of 25.8 us, the query, value and output
// rows at ~3.6 TB/s); where it does not, the longest block's chain of tiles.  us per layer for the
// whole step, before -> after this form: one prompt of 464 22.1 -> 17.9, of 2048 66.8 -> 45.1, 4 of
// 100..300 20.3 -> 17.4, 8 x 256 under a mask 21.1 -> 17.2, 32 of 500 102 -> 94.7, 16 of 32..512 32.7 ->
// 32.2.
// Rows are stored unpadded with their 16-byte chunks XOR-swizzled (K chunk ch of row r at
// ch ^ (r & 15), V at ch ^ 4 (r & 3) for rows of 256 bytes), which keeps the 16-byte K reads of
// 32 rows and the transposing V reads of 4 rows x 64 bytes on distinct banks; over whole launches
// 8.7% of the LDS cycles are in conflict (16 prompts of 32..512).
// The causal mask is applied only on the steps that straddle the wave's diagonal or the end of
// the keys.  The running maximum moves only when a step's maximum exceeds it by more than
// kRescaleLog2 (log2 units), so the accumulators are rescaled rarely and unnormalised weights
// stay below 2^kRescaleLog2 (well inside bf16 and fp32 range).
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// Queries per workgroup.
constexpr int query_block(int gh) { return 4 * (32 / gh); }

// A wave's share of a tile's K or V rows: N loads of 1 KiB, consecutive in LDS.
template <int N>
Q3T_DEVICE void load_tile(i32x4_t rs, const uint32_t (&o)[N], uint32_t at, uint32_t base) {
    static_assert(N == 1 || N == 2 || N == 4, "");
    if constexpr (N == 4)
        asm volatile("s_mov_b32 m0, %0\n\t" Q3T_VMEM_SGPR_WAIT "buffer_load_dwordx4 %1, %5, 0 offen lds\n\t"
                     "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %5, 0 offen lds\n\t"
                     "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %5, 0 offen lds\n\t"
                     "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds"
                     :: "s"(base), "v"(o[0] + at), "v"(o[1] + at), "v"(o[2] + at), "v"(o[3] + at), "s"(rs) : "memory", "m0", "scc");
    else if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %0\n\t" Q3T_VMEM_SGPR_WAIT "buffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
                     "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
                     :: "s"(base), "v"(o[0] + at), "v"(o[1] + at), "s"(rs) : "memory", "m0", "scc");
    else
        load_to_lds16(rs, o[0] + at, base);
}

// 16 bytes to an address of 8-byte alignment, as output rows may have (a store of four dwords needs
// dword alignment only).
Q3T_DEVICE void store16_at8(char *p, const U4 &v) {
    typedef uint32_t u32x4_at8_t __attribute__((ext_vector_type(4), aligned(8)));
    *reinterpret_cast<u32x4_at8_t *>(p) = u32x4_at8_t{v.x, v.y, v.z, v.w};
}

Q3T_DEVICE void lds_write8(uint32_t byte_addr, uint32_t lo, uint32_t hi) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    *(__attribute__((address_space(3))) u32x2_t *)(uintptr_t)byte_addr = u32x2_t{lo, hi};
}

// MB: bytes per mask element (0: no mask, 2: bf16 / fp16, 4: fp32).  Without a mask the
// causal rule (and the optional per-request key counts) bounds the key tiles of each query
// block; with a mask every key tile of the view is scored and the mask alone decides, its
// tile (the block's query rows x 32 keys) staged through the same LDS ring as the keys and
// values.  RK: the keys arrive unrotated (the step's own projection rows).  `cu`, `slots`, `nb`
// and `attn_wgs` lead the arguments: they are preloaded into scalar registers, so a wave asks for its row
// offsets without waiting for the argument block.  With new rows, workgroups past attn_wgs look for
// those that no query block covers.  Looked for in the blocks, ahead of their first loads, they cost a
// prompt of 45 rows 1.3% (28 layers 257.6 us without, 261.1), at the blocks' ends 3.4%; so 255.8.
// SUB: 32-key blocks per tile.  One (three stages of 16 KiB and the mask tile; without a mask 168
// VGPRs and three workgroups per CU for two heads, else at most 256 and two) where the launch fills
// the card; two (two stages of 32 KiB, the blocks' score chains independent of one another, one
// maximum, barrier and wait for both) where it does not and the longest block's chain of tiles is
// the launch: kFewGroups.  Three waves per SIMD asked of a masked instance, whose LDS does not let
// them in, had the compiler keep to no bound: 276-280 registers, one workgroup per CU (us per layer,
// so / with two asked for: 32 x 256 61.6 / 41.0, 16 x 512 98 / 59); one head without a mask spills
// under it (32 prompts of 500 128 / 150).
template <int D, int GH, int MB, int SUB, bool RK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SUB == 2 || GH == 1 || MB > 0 ? 2 : 3)))
prefill_attention_kernel(const int32_t *cu, const int64_t *slots, int nb, int attn_wgs, PrefillParams p) {
    constexpr int QPW = 32 / GH;                  // queries per wave
    constexpr int QB = query_block(GH);           // queries per workgroup
    constexpr int KK = D / 16;                    // MFMA steps over the head dimension
    constexpr int DB = D / 32;                    // 32-row blocks of O^T
    constexpr int CPR = D / 8;                    // 16-byte chunks per row
    constexpr int ROW = D * 2;                    // bytes per row
    constexpr int kTile = kKeys * SUB;            // keys of a tile
    constexpr int kStages = SUB == 2 ? 2 : 3;     // LDS ring depth: loads run kStages - 1 tiles ahead
    constexpr int KBYTES = kTile * ROW;           // K part of a stage
    constexpr int RB = kTile * MB;                // mask bytes per query row of a tile
    constexpr int MBYTES = QB * RB;               // mask tile of a stage
    constexpr int SBYTES = 2 * KBYTES + MBYTES;   // stage: K rows, V rows, mask rows
    constexpr int NL = D / 64 * SUB;              // K (and V) loads per wave and tile
    constexpr int LPR = MB ? RB / 16 : 1;         // lanes per mask row
    constexpr int RPI = 64 / LPR;                 // mask rows per wave load
    constexpr int LPTM = MB ? QPW / RPI : 0;      // mask loads per wave per tile
    constexpr int WAIT = 2 * NL + LPTM;           // loads of one tile per wave
    __shared__ __attribute__((aligned(1024))) uint8_t ring[kStages * SBYTES];

    if constexpr (MB == 0) {
        if (__builtin_expect((int)blockIdx.x >= attn_wgs, false)) {
            copy_other_rows<D, RK>(p, cu, slots, nb, (int)blockIdx.x - attn_wgs, (int64_t)p.nqb * QB);
            return;
        }
    }
    const int tid = threadIdx.x, lane = tid & 63;
    int start = 0, next = 0;
    int64_t slot_l = lane;
    if (nb <= 64 && lane < nb) {
        start = cu[lane];
        next = cu[lane + 1];
        if (slots) slot_l = slots[lane];
    }
    prefetch_kernargs<24 + sizeof(PrefillParams)>();
    // the wave index through readfirstlane: wave-uniform for the compiler too, so that the
    // per-wave load resources stay in scalar registers
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hi = lane >> 5, col = lane & 31;
    const int hgroups = p.Hq / GH;
    const int wg = place_workgroup(blockIdx.x, attn_wgs);
    const int hq0 = (wg % hgroups) * GH;  // the workgroup's first query head
    const int h = hq0 / p.group;          // the workgroup's KV head
    const int rest = wg / hgroups;
    // one workgroup per KV head and query block writes the new rows into the arena
    const bool writes = MB == 0 && p.nv && hq0 % p.group == 0;
    PrefillItem item;
    if (!find_item<QB>(p, cu, slots, nb, start, next, slot_l, rest, item)) return;
    const int b = item.b, qb = item.qb, t0 = item.t0, n = item.n, kn = item.kn, q0 = qb * QB;
    const int64_t slot = item.slot;
    // keys 0 ... kv_end-1 are visible to this block; the arena holds at most `cap` of them.
    // Causal: up to the block's last query and the request's key count; masked: every key.
    const int kv_end = MB ? (int)p.cap : (int)min((int64_t)min(min(n, kn), q0 + QB), p.cap);
    const int ntiles = kv_end > 0 ? (kv_end + kTile - 1) / kTile : 0;
    const int wq0 = q0 + QPW * wave;             // first query of this wave
    // keys [0, wave_end) can be visible to the wave; steps reaching past mask_from need the
    // per-key rule (the diagonal or the end of the keys).  A wave whose queries all lie past
    // the request (the tail of its last block) scores nothing: it only loads its share of
    // every tile and joins the barriers.
    const int wave_end = wq0 >= n ? 0 : MB ? kv_end : min(wq0 + QPW, kv_end);
    const int mask_from = MB ? kv_end : min(wq0 + 1, kv_end);
    const int qpos = wq0 + col % QPW;
    const int hq = hq0 + col / QPW;              // the column's query head
    const bool qvalid = qpos < n;
    const int lim = MB ? kv_end - 1 : min(qpos, kv_end - 1);  // last key visible to this lane's column

    // tile loader: a wave's loads fill 8 SUB K rows and V rows of a stage; physical chunk pc of row
    // r holds logical chunk pc ^ swizzle(r).  The resources end with key kv_end - 1: rows past it
    // read zeros.
    const bool own_values = MB == 0 && p.nv;
    const char *kbase = RK ? p.nk + ((int64_t)t0 * p.nk_st + h * p.nk_sh) * 2 : p.k + (slot * p.k_sb + h * p.k_sh) * 2;
    const char *vbase = own_values ? p.nv + ((int64_t)t0 * p.nv_st + h * p.nv_sh) * 2
                                   : p.v + (slot * p.v_sb + h * p.v_sh) * 2;
    const uint32_t kst = (uint32_t)((RK ? p.nk_st : p.k_st) * 2), vst = (uint32_t)((own_values ? p.nv_st : p.v_st) * 2);
    const i32x4_t krs = scalar_rsrc(kbase, kv_end > 0 ? (uint32_t)((kv_end - 1) * kst + D * 2) : 0u);
    const i32x4_t vrs = scalar_rsrc(vbase, kv_end > 0 ? (uint32_t)((kv_end - 1) * vst + D * 2) : 0u);
    // mask rows of the request's queries (rows past its queries read zeros)
    const uint32_t mrow = (uint32_t)(p.m_sq * MB);
    const i32x4_t mrs = scalar_rsrc(MB ? p.mask + b * p.m_sb * MB : kbase,
                                    MB ? (uint32_t)((n - 1) * (int64_t)mrow + p.cap * MB) : 0u);
    auto v_swizzle = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); };
    const uint32_t ring_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
    uint32_t koff[NL], voff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int r = 8 * SUB * wave + i * (64 / CPR) + lane / CPR, pc = lane % CPR;
        koff[i] = (uint32_t)r * kst + ((pc ^ r) & (CPR - 1)) * 16;
        voff[i] = (uint32_t)r * vst + (pc ^ v_swizzle(r)) * 16;
    }
    const uint32_t load_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ring_base + wave * 8 * SUB * ROW));
    auto issue = [&](int kt, int stage) {
        const uint32_t at = load_base + stage * SBYTES;
        load_tile<NL>(krs, koff, (uint32_t)(kt * kTile) * kst, at);
        load_tile<NL>(vrs, voff, (uint32_t)(kt * kTile) * vst, at + KBYTES);
        if constexpr (MB > 0) {
            // the wave's own query rows of the mask tile: load i covers rows RPI i ... + RPI - 1
#pragma unroll
            for (int i = 0; i < LPTM; ++i) {
                const int r = QPW * wave + i * RPI + lane / LPR;
                const uint32_t off = q0 + r < n ? (uint32_t)(q0 + r) * mrow + (uint32_t)(kt * RB + (lane % LPR) * 16)
                                                : 0xfffffff0u;
                load_to_lds16(mrs, off, (uint32_t)__builtin_amdgcn_readfirstlane(
                                            (int)(ring_base + stage * SBYTES + 2 * KBYTES + (QPW * wave + i * RPI) * RB)));
            }
        }
    };

    // per-lane LDS read addresses within a stage: K row `col`, chunk 2 kk + hi (its XOR with the
    // row moves only the address's low bits, so step kk is an XOR of the first); V key row
    // 4 hi + i/4 (i = lane % 16), 4 dims of the 16-lane group's 16 (likewise for dim block db)
    const uint32_t ka = ring_base + col * ROW + ((hi ^ col) & (CPR - 1)) * 16;
    uint32_t va;
    {
        const int i = lane & 15, r = 4 * hi + (i >> 2), chunk = 2 * ((lane >> 4) & 1) + ((i >> 1) & 1);
        va = ring_base + KBYTES + r * ROW + (chunk ^ v_swizzle(r)) * 16 + 8 * (i & 1);
    }

    // The column's query row as B operands (dims 16 kk + 8 hi ... + 7, zeros past the request) and,
    // with cos/sin, its RoPE.  Rows are loaded whole (CPR lanes of 16 bytes each), staged in the
    // wave's 32 rows of the ring past its first stage and read back in operand order: loaded
    // in operand order they came in 32-byte pieces of 32 rows at once, each line four times over.
    // The first tile is in flight meanwhile; the block's own value rows, if they go to the arena,
    // come with the queries.
    constexpr int RPL = 64 / CPR;                 // rows per load
    const int lr = lane / CPR, lc = lane % CPR;   // row and chunk of a row load
    auto token = [&](int i) { return t0 + min(wq0 + i, n - 1); };  // the wave's i-th query's token
    U4 qrow[32 / RPL], crow[QPW / RPL], srow[QPW / RPL], vrow[QPW / RPL];
#pragma unroll
    for (int i = 0; i < 32 / RPL; ++i) {
        const int r = i * RPL + lr;               // column r: query r % QPW of head r / QPW
        qrow[i] = load16(p.q + ((int64_t)token(r % QPW) * p.q_st + (hq0 + r / QPW) * p.q_sh) * 2 + lc * 16);
    }
    if (p.cs) {
#pragma unroll
        for (int i = 0; i < QPW / RPL; ++i) {
            const int64_t at = (int64_t)token(i * RPL + lr) * p.cs_st * 2 + lc * 16;
            crow[i] = load16(p.cs + at);
            srow[i] = load16(p.sn + at);
        }
    }
    // RK: cos/sin of a tile's keys
    constexpr int RPT = RK ? 512 / CPR : 1, RKN = RK ? kTile / RPT : 1;  // key rows per pass, passes
    const int rk_row = tid / (CPR / 2), rk_chunk = tid % (CPR / 2);
    U4 rkc[RKN][4];
    auto load_rotation = [&](int kt, int u) {
        const int key = min(kt * kTile + u * RPT + rk_row, n - 1);
        const int64_t at = (int64_t)(t0 + key) * p.cs_st * 2 + rk_chunk * 16;
        rkc[u][0] = load16(p.cs + at);
        rkc[u][1] = load16(p.cs + at + D);
        rkc[u][2] = load16(p.sn + at);
        rkc[u][3] = load16(p.sn + at + D);
    };
    const bool copy_values = writes && !RK;
    if (copy_values) {
#pragma unroll
        for (int i = 0; i < QPW / RPL; ++i)
            vrow[i] = load16(p.nv + ((int64_t)token(i * RPL + lr) * p.nv_st + h * p.nv_sh) * 2 + lc * 16);
    }
    if (ntiles > 0) issue(0, 0);
    const uint32_t stage_row = ring_base + SBYTES + wave * 32 * ROW;  // the wave's staging rows
    auto stage_rows = [&](auto &rows) {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(rows) / sizeof(U4)); ++i) {
            const int r = i * RPL + lr;
            lds_write16(stage_row + r * ROW + ((lc ^ r) & (CPR - 1)) * 16, rows[i]);
        }
    };
    // chunk 2 kk + hi of staged row r
    auto staged = [&](int r, int kk) { return lds_read16(stage_row + r * ROW + (((2 * kk + hi) ^ r) & (CPR - 1)) * 16); };
    bf16x8_t qB[KK];
    {
        U4 qv[KK];
        stage_rows(qrow);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qv[kk] = staged(col, kk);
        if (p.cs) {
            // rotate-half RoPE in registers (bf16-exact; the rotated rows are never stored, so NaN
            // payloads need no canonical form): dims of kk pair with those of kk + KK/2
            U4 c[KK], t[KK];
            stage_rows(crow);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) c[kk] = staged(col % QPW, kk);
            stage_rows(srow);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) t[kk] = staged(col % QPW, kk);
#pragma unroll
            for (int kk = 0; kk < KK / 2; ++kk) {
                U4 y1, y2;
                rope8<false>(&qv[kk].x, &qv[kk + KK / 2].x, &c[kk].x, &c[kk + KK / 2].x, &t[kk].x, &t[kk + KK / 2].x,
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
    if (copy_values) {
#pragma unroll
        for (int i = 0; i < QPW / RPL; ++i) {
            const int64_t pos = wq0 + i * RPL + lr;
            if (pos < n && pos < p.cap) store16(p.v + (slot * p.v_sb + h * p.v_sh + pos * p.v_st) * 2 + lc * 16, vrow[i]);
        }
    }
    if constexpr (RK) {  // the first tile's, in flight over the barriers
#pragma unroll
        for (int u = 0; u < RKN; ++u) load_rotation(0, u);
    }
    lds_barrier();  // every wave is done with its staging rows
    if (kStages == 3 && ntiles > 1) issue(1, 1);

    f32x16_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = f32x16_t{};
    float m = 0.f, l = 0.f;  // running maximum (scaled log2 units) and this lane's weight sum
    bool first = true;
    const float sl = p.scale_log2;

    // Every 32-key block of the tile (one past the wave's keys is masked out: a second instance of
    // the step for half a tile cost 33 register moves in each).  A block's weights go into the
    // products while the next block's are computed.
    auto step = [&](int kt, uint32_t stage) {
        constexpr int NS = SUB;
        if (kt * kTile >= wave_end) return;  // past this wave's keys
        const int kb0 = kt * kTile;  // first key of the step
        const uint32_t so = stage * SBYTES;
        f32x16_t st[NS];
#pragma unroll
        for (int u = 0; u < NS; ++u) st[u] = f32x16_t{};
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int u = 0; u < NS; ++u)
                st[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(lds_read16((ka ^ (32 * kk)) + so + u * 32 * ROW)), qB[kk], st[u], 0, 0, 0);
        if constexpr (SUB == 2) {
            // K fragments three products ahead: left alone, the compiler reads each fragment right in
            // front of its product and waits a whole LDS latency for every one (one prompt of 2048 43.2 ->
            // 41.0 us; with one block per tile the registers for it spill)
            constexpr int MFMA = 0x8, DS_READ = 0x100, AHEAD = 3;
            __builtin_amdgcn_sched_group_barrier(DS_READ, AHEAD * NS, 0);
#pragma unroll
            for (int kk = 0; kk < KK - AHEAD; ++kk) {
                __builtin_amdgcn_sched_group_barrier(MFMA, NS, 0);
                __builtin_amdgcn_sched_group_barrier(DS_READ, NS, 0);
            }
            __builtin_amdgcn_sched_group_barrier(MFMA, AHEAD * NS, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        float x[16 * NS];
#pragma unroll
        for (int e = 0; e < 16 * NS; ++e) x[e] = st[e / 16][e % 16];
        if constexpr (MB > 0) {  // scores in log2 units with the mask added
            const uint32_t mrow_lds = ring_base + so + 2 * KBYTES + (QPW * wave + col % QPW) * RB;
#pragma unroll
            for (int i = 0; i < 4 * NS; ++i) {
                float mk[4];
                mask_values<MB>(mrow_lds + (8 * i + 4 * hi) * MB, p.mdt, mk);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * i + e] = __builtin_fmaf(x[4 * i + e], sl, mk[e]);
            }
        }
        if (kb0 + 32 * NS > mask_from) {  // the step reaches past the diagonal or the keys
            int rel = lim - kb0 - 4 * hi;
            asm volatile("" : "+v"(rel));  // keeps the comparisons inside the branch
#pragma unroll
            for (int e = 0; e < 16 * NS; ++e)
                if (8 * (e / 4) + e % 4 > rel) x[e] = -INFINITY;
        }
        float mx = x[0];
#pragma unroll
        for (int e = 1; e < 16 * NS; ++e) mx = __builtin_amdgcn_fmed3f(mx, x[e], __builtin_inff());
        // a column's step maximum is the larger of its two lanes' (scaling is monotonic, so it
        // commutes with the maximum): some column exceeds its running maximum by more than
        // kRescaleLog2 exactly when some lane's own maximum does, and the maximum across lanes is
        // needed only to start and to rescale
        float mt = MB ? mx : mx * sl;
        if (first || __builtin_amdgcn_ballot_w64(mt > m + kRescaleLog2) != 0) {
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
            first = false;
        }
#pragma unroll
        for (int u = 0; u < 2 * NS; ++u) {
            float pv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) pv[e] = MB ? fexp2(x[8 * u + e] - m) : fexp2(__builtin_fmaf(x[8 * u + e], sl, -m));
            l += ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
            const bf16x8_t pB = as_bf16x8(U4{cvt_pk_bf16(pv[0], pv[1]), cvt_pk_bf16(pv[2], pv[3]),
                                             cvt_pk_bf16(pv[4], pv[5]), cvt_pk_bf16(pv[6], pv[7])});
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const uint32_t at = (va ^ (64 * db)) + so + 16 * u * ROW;
                const uint2 lo = lds_read_tr16(at), up = lds_read_tr16(at + 8 * ROW);
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(U4{lo.x, lo.y, up.x, up.y}), pB, acc[db], 0, 0, 0);
            }
        }
    };
    // RK: a landed tile's keys are rotated in LDS, a thread taking chunks pc and pc + CPR/2 of row
    // tid / (CPR/2) of every RPT; the block's own rows go to the arena, keys and values
    auto rotate_keys = [&](int kt, uint32_t stage) {
#pragma unroll
        for (int u = 0; u < RKN; ++u) {
            const int r = u * RPT + rk_row, key = kt * kTile + r;
            if (key >= kv_end) continue;
            if (kt > 0) load_rotation(kt, u);
            const uint32_t row = ring_base + stage * SBYTES + r * ROW;
            const uint32_t k1 = row + ((rk_chunk ^ r) & (CPR - 1)) * 16, k2 = row + (((rk_chunk + CPR / 2) ^ r) & (CPR - 1)) * 16;
            const U4 x1 = lds_read16(k1), x2 = lds_read16(k2);
            U4 y1, y2;
            rope8(&x1.x, &x2.x, &rkc[u][0].x, &rkc[u][1].x, &rkc[u][2].x, &rkc[u][3].x, &y1.x, &y2.x);
            lds_write16(k1, y1);
            lds_write16(k2, y2);
            if (key >= q0 && writes) {
                char *ak = const_cast<char *>(p.k) + (slot * p.k_sb + h * p.k_sh + (int64_t)key * p.k_st) * 2 + rk_chunk * 16;
                char *av = p.v + (slot * p.v_sb + h * p.v_sh + (int64_t)key * p.v_st) * 2 + rk_chunk * 16;
                store16(ak, y1);
                store16(ak + D, y2);
                store16(av, lds_read16(row + KBYTES + (rk_chunk ^ v_swizzle(r)) * 16));
                store16(av + D, lds_read16(row + KBYTES + ((rk_chunk + CPR / 2) ^ v_swizzle(r)) * 16));
            }
        }
    };
    // one ring position: wait for this tile's loads (a younger tile stays in flight with three
    // stages), barrier (every wave is done with the stage the next load overwrites), issue the
    // tile kStages - 1 ahead into that stage, then the products
    auto ring_step = [&](int kt, int stage) {
        if (kStages == 3 && kt + 1 < ntiles) wait_loads<WAIT>();
        else wait_loads<0>();
        lds_barrier();
        if (kt + kStages - 1 < ntiles) issue(kt + kStages - 1, (stage + kStages - 1) % kStages);
        if constexpr (RK) {
            rotate_keys(kt, stage);
            lds_barrier();
        }
        step(kt, stage);
    };
    if constexpr (RK) {  // one tile, unless a request is longer than the caller said
        for (int kt = 0; kt < ntiles; ++kt) ring_step(kt, kt % kStages);
    } else {
        for (int kt = 0; kt < ntiles; kt += kStages) {
            ring_step(kt, 0);
            if (kt + 1 < ntiles) ring_step(kt + 1, 1);
            if (kStages == 3 && kt + 2 < ntiles) ring_step(kt + 2, kStages - 1);
        }
    }

    // The output rows go through LDS (the wave's 32 rows, swizzled chunks) so that each is stored
    // whole, CPR lanes of 16 bytes, and not in 16-byte pieces of 32 rows at once.
    lds_barrier();  // every wave is done with the ring
    {
        const float lt = l + xor32(l);
        const float inv = lt > 0.f ? __builtin_amdgcn_rcpf(lt) : 0.f;  // no visible key: zero row
        const uint32_t rows = ring_base + wave * 32 * ROW;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                lds_write8(rows + col * ROW + (((4 * db + i) ^ col) & (CPR - 1)) * 16 + 8 * hi,
                           cvt_pk_bf16(acc[db][4 * i] * inv, acc[db][4 * i + 1] * inv),
                           cvt_pk_bf16(acc[db][4 * i + 2] * inv, acc[db][4 * i + 3] * inv));
#pragma unroll
        for (int i = 0; i < 32 / RPL; ++i) {
            const int r = i * RPL + lr, pos = wq0 + r % QPW;
            const U4 v = lds_read16(rows + r * ROW + ((lc ^ r) & (CPR - 1)) * 16);
            if (pos < n) store16_at8(p.out + ((int64_t)(t0 + pos) * p.o_st + (hq0 + r / QPW) * p.o_sh) * 2 + lc * 16, v);
        }
    }
}

}  // namespace q3t

using namespace q3t;

// Validates the arguments and fills the kernel's; `empty`: there is nothing to write.
static int rope_write_params(const q3t_prefill_rope_write_args *a, PrefillRopeWriteParams &p, bool &empty) {
    empty = false;
    if (!a) return Q3T_EINVAL;
    if (a->batch < 1 || a->total_tokens < 0 || a->q_heads < 1 || a->kv_heads < 1 ||
        a->capacity < 1 || a->batch > (1 << 20))
        return Q3T_EINVAL;
    if (a->head_dim != 64 && a->head_dim != 128) return Q3T_EUNSUPPORTED;
    if (a->total_tokens > (1 << 30)) return Q3T_EUNSUPPORTED;  // 32-bit token indices
    empty = a->total_tokens == 0;
    if (empty) return Q3T_OK;
    // q_out == NULL: keys and values only (the attention kernel rotates the queries itself)
    const bool with_q = a->q_out != nullptr;
    // value == NULL: keys only (q3t_prefill_attention then copies the values, new_values)
    const bool with_v = a->value != nullptr;
    if (!a->cu_seqlens || (with_q && !a->query) || !a->key || !a->cos || !a->sin || !a->arena_keys ||
        (with_v && !a->arena_values))
        return Q3T_EINVAL;
    const int64_t st[] = {with_q ? a->q_stride_t : 0, with_q ? a->q_stride_h : 0, a->k_stride_t, a->k_stride_h,
                          with_v ? a->v_stride_t : 0, with_v ? a->v_stride_h : 0, a->cs_stride_t,
                          with_q ? a->qo_stride_t : 0, with_q ? a->qo_stride_h : 0, a->a_stride_b,
                          a->a_stride_h, a->a_stride_t};
    for (int64_t s : st)
        if ((s * 2) % 16) return Q3T_EINVAL;
    const void *ptrs[] = {with_q ? a->query : a->key, a->key, with_v ? a->value : a->key, a->cos, a->sin,
                          with_q ? a->q_out : a->key, a->arena_keys, with_v ? a->arena_values : a->key};
    for (const void *q : ptrs)
        if (!aligned(q, 16)) return Q3T_EINVAL;
    p.B = (int)a->batch; p.Hq = (int)a->q_heads; p.Hkv = (int)a->kv_heads; p.D = (int)a->head_dim;
    p.T = a->total_tokens; p.capacity = a->capacity; p.cu = a->cu_seqlens;
    p.q = (const char *)a->query; p.k = (const char *)a->key; p.v = (const char *)a->value;
    p.q_st = a->q_stride_t; p.q_sh = a->q_stride_h; p.k_st = a->k_stride_t; p.k_sh = a->k_stride_h;
    p.v_st = a->v_stride_t; p.v_sh = a->v_stride_h;
    p.cs = (const char *)a->cos; p.sn = (const char *)a->sin; p.cs_st = a->cs_stride_t;
    p.qo = (char *)a->q_out; p.qo_st = a->qo_stride_t; p.qo_sh = a->qo_stride_h;
    p.ak = (char *)a->arena_keys; p.av = with_v ? (char *)a->arena_values : nullptr;
    p.a_sb = a->a_stride_b; p.a_sh = a->a_stride_h; p.a_st = a->a_stride_t;
    p.slots = a->kv_slots;
    return Q3T_OK;
}

static int launch_rope_write(const PrefillRopeWriteParams &p, hipStream_t s) {
    int64_t blocks = (p.T + 3) / 4;  // one token per wave
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(prefill_rope_write_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p);
    return launch_status();
}

extern "C" int q3t_prefill_rope_write(const q3t_prefill_rope_write_args *a, void *stream) {
    PrefillRopeWriteParams p;
    bool empty;
    const int st = rope_write_params(a, p, empty);
    if (st != Q3T_OK || empty) return st;
    return launch_rope_write(p, (hipStream_t)stream);
}


// Workgroups from which a launch fills the card (two per CU).  Below, the longest block's chain of
// tiles bounds it.  us per layer, one / two 32-key blocks per tile: one prompt of 464 21.9 / 18.8 (64
// workgroups), of 2048 58.2 / 41.0 (256); 16 prompts of 32..512 (664) 33.5 / 39.3, 8 of 1024..2048
// 102.7 / 103.8.  Under a bf16 mask 8 x 256 16.1 / 14.8 (256), 2 x 1024 41.3 / 36.1 (256), 16 x 256
// 25.3 / 25.2 (512), 32 x 256 41.0 / 40.7 (1024), 64 x 128 31.0 / 30.9; rows of 64 8 x 256 12.5 / 11.4
// (256), 32 x 256 25.7 / 28.2 (1024).
// Two blocks' mask rows cost their gain where they leave one workgroup on a CU: fp32 masks (8 x 256
// 15.7 / 16.9, 16 x 256 25.9 / 36.1, 2 x 1024 38.4 / 42.8; rows of 64 8 x 256 11.6 / 12.5) and one head's
// rows of 128 under a mask (8 x 256 16.7 / 17.2, 16 x 256 25.2 / 34.4) always take one.
constexpr int64_t kFewGroups = 512;
// One-head groups take blocks of 64 queries on 16-column products (prefill_narrow.hip) where the query
// rows of all heads are fewer than this many blocks of 128 would hold; there the chain of the longest
// block is the launch, and a wave's is half as long.  us per layer, blocks of 128 / of 64 (16 heads
// unless said): one prompt of 464 20.7 / 19.8, 8 x 250 23.9 / 22.9 (250 blocks), 8 heads 16 of 32..512
// 28.5 / 27.4 (300), 12 x 500 32.8 / 32.1 (375), 16 x 500 39.5 / 42.2 (500), rows of 64 12 x 500 21.9 /
// 20.7 and 16 x 500 25.4 / 26.0; bf16 mask 2 x 1024 42.1 / 40.0 (256), 12 x 256 22.3 / 26.9 (384), rows of
// 64 14.1 / 13.4, 8 x 512 23.7 / 25.4 (512); fp32 mask, one workgroup of 128 per CU, 12 x 256 30.9 / 26.4,
// 8 x 512 51.3 / 45.2 (512), 16 x 256 34.0 / 34.8, 32 x 256 62.1 / 66.0 (1024).
static bool narrow_blocks(const PrefillParams &p, int head_dim, int64_t wgs) {
    const int64_t blocks = !p.mask || head_dim == 64 ? 384 : p.mdt == Q3T_F32 ? 512 : 256;
    return p.T * p.Hq <= blocks * 128 && wgs <= 16 * blocks;  // the grid too: requests of no rows count in it
}
// Bytes of one KV head's rows of the whole step from which its L2 share no longer holds them.
constexpr int64_t kL2Rows = 3 << 20;

template <int D, int GH, int MB, int SUB, bool RK = false>
static void launch_tiles(const PrefillParams &p, const int64_t *slots, dim3 grid, hipStream_t s) {
        hipLaunchKernelGGL((prefill_attention_kernel<D, GH, MB, SUB, RK>), dim3(grid.x + (uint32_t)other_row_workgroups(p)), dim3(256), 0, s, p.cu, slots, p.B,
                       (int)grid.x, p);
}

template <int D, int GH>
static void launch_prefill(const PrefillParams &p, int64_t max_seqlen, const int64_t *slots, hipStream_t s) {
    constexpr int QB = query_block(GH);
    PrefillParams q = p;
    q.nqb = (int)((max_seqlen + QB - 1) / QB);
    const int64_t wgs = prefill_workgroups(p, QB, p.Hq / GH, max_seqlen);
    if constexpr (GH == 1) {
        if (!p.nk && narrow_blocks(p, D, wgs)) {
            launch_prefill_narrow(p, D, max_seqlen, s);
            return;
        }
    }
    // Longest blocks first over all requests ends the launch evenly, but every request's rows are
    // then in use at once; request by request keeps the rows in use in the XCD's L2.  The latter
    // where the rows exceed it and the blocks are many against one request's, so that the last
    // request's chain is a small part of the launch (us per layer, by length / by request: 32
    // prompts of 500 85.9 / 79.2, 16 of 512 52.5 / 46.4, 8 of 1024..2048 93.7 / 103).
    q.by_request = p.T * D * 4 > kL2Rows && (int64_t)q.nqb * 8 <= (p.T + QB - 1) / QB;
    const dim3 grid((uint32_t)wgs);
    const bool few = wgs <= kFewGroups;
    if (p.nk) launch_tiles<D, GH, 0, 2, true>(q, slots, grid, s);
    else if (p.mask && p.mdt == Q3T_F32) launch_tiles<D, GH, 4, 1>(q, slots, grid, s);
    else if (p.mask) {
        if constexpr (D == 128 && GH == 1) launch_tiles<D, GH, 2, 1>(q, slots, grid, s);
        else if (few) launch_tiles<D, GH, 2, 2>(q, slots, grid, s);
        else launch_tiles<D, GH, 2, 1>(q, slots, grid, s);
    } else if (few) launch_tiles<D, GH, 0, 2>(q, slots, grid, s);
    else launch_tiles<D, GH, 0, 1>(q, slots, grid, s);
}

static int launch_prefill_sizes(const PrefillParams &p, int64_t head_dim, int64_t max_seqlen, const int64_t *slots, hipStream_t s) {
    // the query heads of a KV head pair up in one workgroup and share its staged K/V tiles
    if (p.group % 2 == 0) {
        if (head_dim == 128) launch_prefill<128, 2>(p, max_seqlen, slots, s);
        else launch_prefill<64, 2>(p, max_seqlen, slots, s);
    } else {
        if (head_dim == 128) launch_prefill<128, 1>(p, max_seqlen, slots, s);
        else launch_prefill<64, 1>(p, max_seqlen, slots, s);
    }
    return launch_status();
}

// Validates the arguments and fills the kernel's; `empty`: there is nothing to attend.
static int prefill_params(const q3t_prefill_args *a, PrefillParams &p, bool &empty) {
    empty = false;
    if (!a) return Q3T_EINVAL;
    if (a->batch < 1 || a->batch > (1 << 20) || a->total_tokens < 0 || a->total_tokens > INT32_MAX ||
        a->max_seqlen < 0 || a->capacity < 1 || a->q_heads < 1 || a->kv_heads < 1 ||
        a->q_heads % a->kv_heads)
        return Q3T_EINVAL;
    if (a->head_dim != 64 && a->head_dim != 128) return Q3T_EUNSUPPORTED;
    const int64_t G = a->q_heads / a->kv_heads;
    if (G != 1 && G != 2 && G != 4) return Q3T_EUNSUPPORTED;
    empty = a->total_tokens == 0 || a->max_seqlen == 0;
    if (empty) return Q3T_OK;
    if (!a->cu_seqlens || !a->query || !a->keys || !a->values || !a->out) return Q3T_EINVAL;
    const int64_t st[] = {a->q_stride_t, a->q_stride_h, a->k_stride_b, a->k_stride_h, a->k_stride_t,
                          a->v_stride_b, a->v_stride_h, a->v_stride_t, a->o_stride_t, a->o_stride_h};
    for (int64_t v : st)
        if (v < 0 || (v * 2) % 16) return Q3T_EINVAL;
    if (!aligned(a->query, 16) || !aligned(a->keys, 16) || !aligned(a->values, 16) || !aligned(a->out, 8))
        return Q3T_EINVAL;
    if ((a->cos != nullptr) != (a->sin != nullptr)) return Q3T_EINVAL;
    if (a->cos && (!aligned(a->cos, 16) || !aligned(a->sin, 16) || a->cs_stride_t < 0 || (a->cs_stride_t * 2) % 16))
        return Q3T_EINVAL;
    // key rows of one (slot, head) are addressed by 32-bit byte offsets
    const int64_t max_st = a->k_stride_t > a->v_stride_t ? a->k_stride_t : a->v_stride_t;
    if (a->capacity * max_st * 2 + a->head_dim * 2 > INT32_MAX) return Q3T_EUNSUPPORTED;
    if (a->mask) {
        // rows of 16-byte aligned keys, addressed by 32-bit offsets from a request's base
        if (a->mask_dtype != Q3T_BF16 && a->mask_dtype != Q3T_F16 && a->mask_dtype != Q3T_F32) return Q3T_EUNSUPPORTED;
        const int64_t es = a->mask_dtype == Q3T_F32 ? 4 : 2;
        if (!aligned(a->mask, 16) || a->mask_stride_q < 0 || a->mask_stride_b < 0 || (a->mask_stride_q * es) % 16 ||
            (a->mask_stride_b * es) % 16)
            return Q3T_EINVAL;
        if ((a->max_seqlen - 1) * a->mask_stride_q * es + a->capacity * es > INT32_MAX) return Q3T_EUNSUPPORTED;
    }
    if (a->new_values) {
        // value rows of the step's tokens: only for the causal rule (a mask scores every key
        // of the arena view, beyond the step's rows); 32-bit row offsets from a request's
        // first token
        if (a->mask) return Q3T_EINVAL;
        if (!aligned(a->new_values, 16) || a->nv_stride_t < 0 || a->nv_stride_h < 0 || (a->nv_stride_t * 2) % 16 ||
            (a->nv_stride_h * 2) % 16)
            return Q3T_EINVAL;
        const int64_t rows = a->capacity < a->max_seqlen ? a->capacity : a->max_seqlen;
        if (rows * a->nv_stride_t * 2 + a->head_dim * 2 > INT32_MAX) return Q3T_EUNSUPPORTED;
    }
    p = PrefillParams{};
    p.B = (int)a->batch; p.Hq = (int)a->q_heads; p.Hkv = (int)a->kv_heads;
    p.group = (int)G;
    // blocks of 64 queries (128 where a workgroup takes one head)
    const int64_t blocks = (a->max_seqlen + 63) / 64;
    if ((int64_t)p.B * blocks * p.Hq > INT32_MAX) return Q3T_EUNSUPPORTED;
    p.scale_log2 = a->scale * kLog2eP;
    p.cu = a->cu_seqlens;
    p.q = (const char *)a->query; p.q_st = a->q_stride_t; p.q_sh = a->q_stride_h;
    p.k = (const char *)a->keys; p.v = (char *)a->values;
    p.k_sb = a->k_stride_b; p.k_sh = a->k_stride_h; p.k_st = a->k_stride_t;
    p.v_sb = a->v_stride_b; p.v_sh = a->v_stride_h; p.v_st = a->v_stride_t;
    p.slots = a->kv_slots;
    p.cap = a->capacity;
    p.T = a->total_tokens;
    p.out = (char *)a->out; p.o_st = a->o_stride_t; p.o_sh = a->o_stride_h;
    p.cs = (const char *)a->cos; p.sn = (const char *)a->sin; p.cs_st = a->cs_stride_t;
    p.kvl = a->kv_lens;
    p.mask = (const char *)a->mask;
    p.mdt = (int)a->mask_dtype;
    p.m_sb = a->mask_stride_b; p.m_sq = a->mask_stride_q;
    p.nv = (const char *)a->new_values; p.nv_st = a->nv_stride_t; p.nv_sh = a->nv_stride_h;
    return Q3T_OK;
}

extern "C" int q3t_prefill_attention(const q3t_prefill_args *a, void *stream) {
    PrefillParams p;
    bool empty;
    const int st = prefill_params(a, p, empty);
    if (st != Q3T_OK || empty) return st;
    return launch_prefill_sizes(p, a->head_dim, a->max_seqlen, a->kv_slots, (hipStream_t)stream);
}

// Whether one launch does the whole layer: the attention's workgroups rotate the keys they read
// and write their own block's rows, so the keys of a request's earlier blocks are rotated once
// more in every later one.  Worth it up to kRotateRows rows a request (us per layer, two launches /
// one: a prompt of 45 rows 10.0 / 8.6, 16 of 64 14.5 / 12.3, 60 of 60 23.7 / 20.3; 3 of 100, two blocks,
// 12.2 / 13.3).
constexpr int64_t kRotateRows = 64;
static bool rotates_keys(const q3t_prefill_rope_write_args *w, const PrefillRopeWriteParams &r,
                         const q3t_prefill_args *a, const PrefillParams &p) {
    return a->max_seqlen <= kRotateRows && !a->mask && !a->kv_lens && p.nv && p.cs && !w->q_out && !w->value &&
           w->arena_keys == a->keys && w->cu_seqlens == a->cu_seqlens && w->kv_slots == a->kv_slots &&
           w->cos == a->cos && w->sin == a->sin && w->cs_stride_t == a->cs_stride_t && r.B == p.B && r.T == p.T &&
           r.Hkv == p.Hkv && r.capacity == p.cap && w->head_dim == a->head_dim && r.a_sb == p.k_sb && r.a_sh == p.k_sh &&
           r.a_st == p.k_st && r.k_st >= 0 && r.k_sh >= 0 && kRotateRows * r.k_st * 2 + a->head_dim * 2 <= INT32_MAX;
}

extern "C" int q3t_prefill_step(const q3t_prefill_rope_write_args *w, const q3t_prefill_args *a, void *stream) {
    PrefillRopeWriteParams r;
    PrefillParams p;
    bool nothing_to_write, nothing_to_attend;
    int st = rope_write_params(w, r, nothing_to_write);
    if (st != Q3T_OK) return st;
    st = prefill_params(a, p, nothing_to_attend);
    if (st != Q3T_OK) return st;
    hipStream_t s = (hipStream_t)stream;
    if (!nothing_to_write && !nothing_to_attend && rotates_keys(w, r, a, p)) {
        p.nk = r.k;
        p.nk_st = r.k_st;
        p.nk_sh = r.k_sh;
        return launch_prefill_sizes(p, a->head_dim, a->max_seqlen, a->kv_slots, s);
    }
    if (!nothing_to_write) st = launch_rope_write(r, s);
    if (st != Q3T_OK || nothing_to_attend) return st;
    return launch_prefill_sizes(p, a->head_dim, a->max_seqlen, a->kv_slots, s);
}
