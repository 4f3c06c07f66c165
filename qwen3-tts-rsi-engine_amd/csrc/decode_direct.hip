// Decode attention with one workgroup per (request, KV head): the chunked grid's unsplit form,
// for short arenas and few requests (the code predictor's 16-row caches, a lone talker request,
// the drop-in call under a full-arena mask).
//
// Bound by latency, not bytes: a launch is one chain of memory round trips (arguments and
// position, rows, keys, output), and splitting a short request over workgroups adds three more
// (publish, count, collect).  So nothing is split: the W waves of a workgroup share the
// request's keys and merge in LDS.
//   * the position and every line of the argument block come in one scalar round trip (the
//     position array is the leading argument, preloaded into scalar registers);
//   * the last wave loads the rows that depend only on (request, head), rotates them in LDS
//     (fused) while the first keys are in flight, and one barrier hands them to the others;
//   * wave w owns keys 16 w ... 16 w + 15 of every 16 W keys.  Its K and V rows go straight to
//     LDS (16 bytes per lane, rows of 16-byte chunks XOR-swizzled as in the bundled grid), two
//     stages of its own in flight, with no barrier in the stream;
//   * S^T = K . Q^T and O^T += V^T . P^T run on bf16 MFMA tiles whose 16 columns are mostly
//     empty, so the weights keep all 24 bits of their float32: columns 0 ... R-1 carry the weights
//     rounded to bf16, columns R ... 2R-1 (the same queries again) the remainders rounded to bf16
//     and columns 2R ... 3R-1 what is left of those, which is exact; the three are added at the
//     end.  Eight query rows (R = 8) leave no columns for the third part: a second product of the
//     same V fragments adds it;
// A wave issues one instruction every four cycles here (one wave per SIMD), so the instructions
// on the chain count as much as its round trips: arguments straight into scalar registers,
// 32-bit row offsets, resources that end at the last key instead of per-lane bounds, four loads
// per M0 write and address arithmetic placed under the loads' latency took the 16-row launch
// from 6.2 to 3.8 us.
// Measured, us per layer (28-layer graphs of fused steps, 16/8 heads), split kernel -> this one:
// 64 requests x 16 rows 6.5 -> 3.8; 1 x 300 keys 10.7 -> 6.1; 21 x 30..511 keys 16.6 -> 9.2;
// 64 x 32..511 keys 18.0 -> 15.7; 128 x 32..512 keys 32.0 -> 26.6; 1 x 1750 keys 22.5 -> 13.4.
//   * masked launches bring the request's whole mask row into LDS once and stop at its last
//     visible key.  Each wave's first two stages are on their way before the mask is looked at, so
//     of the keys that the mask hides behind it, those stages' are read and no others; none reaches
//     the output, also where it is not finite: their scores are dropped and their value rows zeroed.
#include "decode_params.hpp"

#include <type_traits>

namespace q3t {
namespace direct {

constexpr int kRow = 256;                      // bytes of a bf16 row of D = 128
constexpr int kKeys = 16;                      // keys of a wave's stage
constexpr int kStage = 2 * kKeys * kRow;       // K rows then V rows: 8 KiB
constexpr int kLoads = kStage / 1024;          // 1 KiB loads per stage
constexpr int kStages = 2;                     // stages of a wave: one scored, one in flight
constexpr int kMaskWords = kDirectMaxCtx;      // 4-byte words of a mask row
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kEmpty = -1.0e30f;             // running maximum before any visible key

// The launch's arguments as they sit in the argument block after the position array: 54 dwords
// that a wave loads into scalar registers in one round trip.  Strides are in bytes, those of the
// arena planes in 16-byte units (a plane can exceed 4 GiB; a batch of rows cannot).
struct DirectParams {
    const char *q;
    char *k, *v, *out;
    const char *nk, *nv, *cs, *sn;
    const char *mask;
    const int64_t *offs;
    const char *qnw, *knw;
    uint32_t q_sb, q_ss, q_sh, o_sb;
    uint32_t o_ss, o_sh, nk_sb, nk_sh;
    uint32_t nv_sb, nv_sh, nk_ss, nv_ss;
    uint32_t cs_sb, cs_ss, k_st, v_st;
    float scale_log2, eps;
    int32_t ctx, mask_dtype;
    uint32_t k_sb16, k_sh16, v_sb16, v_sh16;
    int64_t m_sb, m_ss;  // elements
    int32_t stream, vec_out;
};
static_assert(sizeof(DirectParams) == 54 * 4, "loaded as 3 x 16 + 4 + 2 dwords");

template <int ROWS, int R, int MASKS, int W>
struct DirectLds {
    char ring[kStages][W][kStage];
    char head[ROWS][kRow];
    float ml[W][R][2];
    alignas(16) uint32_t maskw[MASKS ? MASKS : 1][MASKS ? kMaskWords + 64 : 4];  // whole 64-word loads
};

Q3T_DEVICE uint32_t lds_read4(uint32_t byte_addr) {
    return *(__attribute__((address_space(3))) const uint32_t *)(uintptr_t)byte_addr;
}
// Four mask elements of one type from an LDS byte address, in log2 units: the type is looked at once
// for the four (looked at for each, and with a division for each in the search of the last visible key, 8
// requests over 2000 rows took 28.8 us a launch, 21.7 on the split kernel; now 21.4).
Q3T_DEVICE void mask_terms(uint32_t at, int dtype, float (&x)[4]) {
    auto elements = [&](auto element, auto term) {
        using E = decltype(element);
        const auto *e = (__attribute__((address_space(3))) const E *)(uintptr_t)at;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = term(e[i]);
    };
    if (dtype == Q3T_BF16) elements(uint16_t{}, [](uint16_t e) { return bf16_to_float(e) * kLog2e; });
    else if (dtype == Q3T_F32) elements(float{}, [](float e) { return e * kLog2e; });
    else if (dtype == Q3T_F16) elements(uint16_t{}, [](uint16_t e) { return (float)__builtin_bit_cast(_Float16, e) * kLog2e; });
    else elements(uint8_t{}, [](uint8_t e) { return e ? 0.0f : -INFINITY; });  // bool: True attends
}
// What rounding to bf16 left of two floats (exact).
Q3T_DEVICE void bf16_rest(float &a, float &b, uint32_t rounded) {
    a -= bf16_lo(rounded);
    b -= bf16_hi(rounded);
}

// Four 1 KiB loads of a stage's K or V rows (rows 4i + lane / 16, chunk lane % 16) into LDS.  The
// instruction's offset moves the memory and the LDS address alike, so load i's voffset is 1024 i
// short of its row; rows past the resource's range write zeros.
#define Q3T_LOAD4(POLICY)                                                                          \
    asm volatile("s_mov_b32 m0, %0\n\t" Q3T_VMEM_SGPR_WAIT                                         \
                 "buffer_load_dwordx4 %1, %5, 0 offen" POLICY " lds\n\t"                           \
                 "buffer_load_dwordx4 %2, %5, 0 offen offset:1024" POLICY " lds\n\t"               \
                 "buffer_load_dwordx4 %3, %5, 0 offen offset:2048" POLICY " lds\n\t"               \
                 "buffer_load_dwordx4 %4, %5, 0 offen offset:3072" POLICY " lds"                   \
                 :: "s"(base), "v"(v[0] + at), "v"(v[1] + at), "v"(v[2] + at), "v"(v[3] + at), "s"(rsrc) : "memory", "m0")
Q3T_DEVICE void load_rows(i32x4_t rsrc, const uint32_t (&v)[4], uint32_t at, uint32_t base, bool stream) {
    if (stream) Q3T_LOAD4(" nt");
    else Q3T_LOAD4("");
}
#undef Q3T_LOAD4
// 16 bytes per lane at base + voffset into LDS at lds_base + 16 lane.
Q3T_DEVICE void load_row16(const char *base, uint32_t voffset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\t" Q3T_VMEM_SGPR_WAIT "global_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_base), "v"(voffset), "s"(base) : "memory", "m0");
}

// Global memory through pointers that the compiler sees only as loaded integers (it would use
// flat accesses, which also count as LDS accesses).
#define Q3T_GLOBAL __attribute__((address_space(1)))
Q3T_DEVICE void global_store16(char *p, const U4 &v) { *(Q3T_GLOBAL i32x4_t *)(uintptr_t)p = __builtin_bit_cast(i32x4_t, v); }
Q3T_DEVICE void global_store2(char *p, uint32_t v) { *(Q3T_GLOBAL uint16_t *)(uintptr_t)p = (uint16_t)v; }
Q3T_DEVICE void global_store4(char *p, uint32_t v) { *(Q3T_GLOBAL uint32_t *)(uintptr_t)p = v; }
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
Q3T_DEVICE void global_store8(char *p, uint32_t lo, uint32_t hi) { *(Q3T_GLOBAL u32x2_t *)(uintptr_t)p = u32x2_t{lo, hi}; }

// A scalar resource without a detour over vector registers: base and bytes are uniform.
Q3T_DEVICE i32x4_t uniform_rsrc(const char *base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return i32x4_t{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xffffu), (int)bytes, 0x00020000};
}

template <int G, int SQ, int FUSE, bool MASK, int W>
__global__ void __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(2)))
decode_direct_kernel(const int64_t *pos, DirectParams) {
    constexpr bool FUSED = FUSE > 0, NORM = FUSE > 1;
    constexpr int R = G * SQ;               // query rows
    // columns of a query row: its weights in two or three bf16 parts
    constexpr bool THIRD = 3 * R <= 16;
    constexpr int COLS = (THIRD ? 3 : 2) * R;
    static_assert(2 * R <= 16, "each query row takes two of the 16 columns at least");
    // rows in LDS: queries, then (fused) cos, sin, new keys and new values of each token, and
    // the norm weights
    constexpr int COS = R, SIN = R + SQ, NEWK = R + 2 * SQ, NEWV = R + 3 * SQ, QNW = R + 4 * SQ, KNW = QNW + 1;
    constexpr int ROWS = R + (FUSED ? 4 * SQ : 0) + (NORM ? 2 : 0);
    constexpr int SK = W * kKeys;           // keys of a stage of the whole workgroup
    constexpr int RW = W - 1;               // the wave that loads and rotates the rows
    __shared__ __attribute__((aligned(1024))) DirectLds<ROWS, R, MASK ? SQ : 0, W> s;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = blockIdx.x, b = blockIdx.y;

    typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    struct Block { u32x16_t a, b, c; u32x4_t d; uint64_t e; } block;
    uint64_t pb;
    asm volatile("s_load_dwordx2 %[pb], %[pa], 0x0\n\ts_load_dwordx16 %[a], %[ka], 0x8\n\t"
                 "s_load_dwordx16 %[b], %[ka], 0x48\n\ts_load_dwordx16 %[c], %[ka], 0x88\n\t"
                 "s_load_dwordx4 %[d], %[ka], 0xc8\n\ts_load_dwordx2 %[e], %[ka], 0xd8\n\ts_waitcnt lgkmcnt(0)"
                 : [pb] "=&s"(pb), [a] "=&s"(block.a), [b] "=&s"(block.b), [c] "=&s"(block.c), [d] "=&s"(block.d),
                   [e] "=&s"(block.e)
                 : [pa] "s"(pos ? (uint64_t)(uintptr_t)(pos + b) : (uint64_t)(uintptr_t)__builtin_amdgcn_kernarg_segment_ptr()), [ka] "s"(__builtin_amdgcn_kernarg_segment_ptr())
                 : "memory");
    struct Packed { uint32_t w[54]; } words;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        words.w[i] = block.a[i];
        words.w[16 + i] = block.b[i];
        words.w[32 + i] = block.c[i];
        if (i < 4) words.w[48 + i] = block.d[i];
    }
    words.w[52] = (uint32_t)block.e;
    words.w[53] = (uint32_t)(block.e >> 32);
    const DirectParams p = __builtin_bit_cast(DirectParams, words);

    // without positions every request attends all of its keys
    const int L = !pos ? p.ctx : (int64_t)pb >= 0 && (int64_t)pb < p.ctx ? (int)pb + 1 : 0;
    char *out = p.out + (b * p.o_sb + h * G * p.o_sh);
    if (L == 0) {  // no valid position: attends nothing, zero rows
        for (int t = tid; t < R * 128; t += W * 64) {
            const int r = t / 128;
            global_store2(out + ((r / G) * p.o_ss + (r % G) * p.o_sh + t % 128 * 2), 0u);
        }
        return;
    }
    auto lds = [](const void *x) { return (uint32_t)(uintptr_t)x; };
    auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };

    // the wave's keys: 16 wave ... + 15 of every SK.  Resources end at the last key to read, so
    // rows past it read zeros without a memory access; fused, rows from L - SQ on are the step's
    // own.
    const char *kp, *vp;
    if (p.offs) {
        const int64_t o = *(Q3T_GLOBAL const int64_t *)(uintptr_t)(p.offs + b) * 2;
        kp = p.k + o + (uint64_t)h * p.k_sh16 * 16;
        vp = p.v + o + (uint64_t)h * p.v_sh16 * 16;
    } else {
        kp = p.k + ((uint64_t)b * p.k_sb16 + (uint64_t)h * p.k_sh16) * 16;
        vp = p.v + ((uint64_t)b * p.v_sb16 + (uint64_t)h * p.v_sh16) * 16;
    }
    const int jend = FUSED ? L - SQ : L;
    const uint32_t kbytes = jend > 0 ? (uint32_t)(jend - 1) * p.k_st + kRow : 0u;
    const uint32_t vbytes = jend > 0 ? (uint32_t)(jend - 1) * p.v_st + kRow : 0u;
    const i32x4_t krs = uniform_rsrc(kp, kbytes), vrs = uniform_rsrc(vp, vbytes);

    // the words of each query token's mask row, 64 per load, the loads dealt to the waves
    int mbase[SQ] = {}, mes = 0;  // byte of a row's first element within its first word; element size
    if constexpr (MASK) {
        mes = mask_elem_size(p.mask_dtype);
#pragma unroll
        for (int q = 0; q < SQ; ++q) {
            const int64_t first = ((int64_t)b * p.m_sb + q * p.m_ss) * mes;
            mbase[q] = (int)(first & 3);
            const int bytes = mbase[q] + p.ctx * mes;
            const i32x4_t mrs = uniform_rsrc(p.mask + (first - mbase[q]), (uint32_t)((bytes + 3) & ~3));
            for (int w0 = wave * 64; w0 * 4 < mbase[q] + L * mes; w0 += W * 64)
                load_to_lds4(mrs, (uint32_t)((w0 + lane) * 4), uniform(lds(&s.maskw[q][w0])));
        }
    }
    // the rows that depend only on (request, head)
    if (wave == RW) {
        const uint32_t lane16 = c * 16, head = lds(&s.head[0][0]);
        const uint32_t qo = b * p.q_sb + h * G * p.q_sh;
#pragma unroll
        for (int i = 0; i < (R + 3) / 4; ++i) {
            const int r = 4 * i + g;
            const uint32_t ro = SQ == 1 ? r * p.q_sh : (r / G) * p.q_ss + (r % G) * p.q_sh;
            if (R % 4 == 0 || r < R) load_row16(p.q, qo + ro + lane16, head + i * 1024);
        }
        if constexpr (FUSED) {
            if (lane < 16 * SQ) {
                const uint32_t co = b * p.cs_sb + (SQ == 1 ? 0 : g * p.cs_ss) + lane16;
                load_row16(p.cs, co, head + COS * kRow);
                load_row16(p.sn, co, head + SIN * kRow);
                load_row16(p.nk, b * p.nk_sb + h * p.nk_sh + (SQ == 1 ? 0 : g * p.nk_ss) + lane16, head + NEWK * kRow);
                load_row16(p.nv, b * p.nv_sb + h * p.nv_sh + (SQ == 1 ? 0 : g * p.nv_ss) + lane16, head + NEWV * kRow);
            }
            if constexpr (NORM) {
                if (p.qnw && lane < 16) load_row16(p.qnw, lane16, head + QNW * kRow);
                if (p.knw && lane < 16) load_row16(p.knw, lane16, head + KNW * kRow);
            }
        }
    }

    // voffsets of a stage's four K and four V loads (row 4i + g, chunk c swizzled), each 1024 i short
    uint32_t kv[4], vv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        kv[i] = (uint32_t)(wave * kKeys + 4 * i + g) * p.k_st + ((c ^ g) ^ (4 * i)) * 16 - 1024 * i;
        vv[i] = (uint32_t)(wave * kKeys + 4 * i + g) * p.v_st + ((c ^ (2 * g)) ^ (8 * i & 15)) * 16 - 1024 * i;
    }
    const uint32_t ring = lds(&s.ring[0][0][0]) + wave * kStage;
    auto issue = [&](int t) {
        const uint32_t base = uniform(ring + (t % kStages) * (W * kStage));
        load_rows(krs, kv, t * SK * p.k_st, base, p.stream);
        load_rows(vrs, vv, t * SK * p.v_st, base + kKeys * kRow, p.stream);
    };
    auto stages = [&](int keys) { return max(0, (keys - wave * kKeys + SK - 1) / SK); };
    int mine = stages(L), issued = min(mine, kStages);
    if (issued > 0) issue(0);
    if (issued > 1) issue(1);

    // per-lane LDS offsets within a stage: K rows as the A operand of S^T (row c, dims 32 kk +
    // 8 g ...), V rows for the transposing read (row 4g + c/4, 4 dims)
    uint32_t ka[4], va[8];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) ka[kk] = ring + c * kRow + (((4 * kk + g) ^ c) & 15) * 16;
    {
        const int r = 4 * g + (c >> 2);
#pragma unroll
        for (int db = 0; db < 8; ++db)
            va[db] = ring + kKeys * kRow + r * kRow + (((2 * db + ((c >> 1) & 1)) ^ (2 * r)) & 15) * 16 + 8 * (c & 1);
    }
    const int part = c / R;                     // the column's part of the weights
    const int cq = c < COLS ? c % R : 0;        // the column's query row
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(va[i]));  // computed here, while the loads are in flight
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ka[i]));

    // the rows (and mask words) landed before the stages, which stay in flight
    if (wave == RW || MASK) {
        if (issued == 2) wait_loads<2 * kLoads>();
        else if (issued == 1) wait_loads<kLoads>();
        else wait_loads<0>();
    }
    if constexpr (FUSED) {
        if (wave == RW) {
            // lane group: one row, lane c its chunk c; normalised, rotated and written back
#pragma unroll
            for (int i = 0; i < (R + SQ + 3) / 4; ++i) {
                const int item = 4 * i + g;
                const bool ok = item < R + SQ, is_key = item >= R;
                const int tk = SQ == 1 || !ok ? 0 : is_key ? item - R : item / G;
                const int row = !ok ? 0 : is_key ? NEWK + tk : item;
                U4 x = lds_read16(lds(&s.head[row][c * 16]));
                if constexpr (NORM) {
                    // a missing weight leaves its rows as they are
                    const U4 w = lds_read16(lds(&s.head[is_key ? KNW : QNW][c * 16]));
                    const U4 y = rms_norm8<16>(x, w, p.eps, 128);
                    if (is_key ? p.knw != nullptr : p.qnw != nullptr) x = y;
                }
                const U4 cv = lds_read16(lds(&s.head[COS + tk][c * 16])), sv = lds_read16(lds(&s.head[SIN + tk][c * 16]));
                const U4 y = rope_half8(x, xor8_u4(x), cv, sv, c < 8);
                if (ok) lds_write16(lds(&s.head[row][c * 16]), y);
            }
        }
    }
    lds_barrier();

    int Lv = L;  // keys [0, Lv) can be visible
    if constexpr (MASK) {
        // the last key that a token's row shows: 64 words at a time from the end (the whole row is
        // in LDS); a row that hides every key is scored in full, as any other mask is
        int shown = 0;
        bool all = false;
#pragma unroll
        for (int q = 0; q < SQ; ++q) {
            const int last_word = (mbase[q] + L * mes - 1) >> 2, shift = mes >> 1;  // log2 of 1, 2 or 4 bytes
            int row = 0;
            for (int w0 = last_word & ~63; w0 >= 0 && row == 0; w0 -= 64) {
                const int w = w0 + lane;
                int seen = -1;  // the last visible key of the lane's word
                if (w <= last_word) {
                    const uint32_t word = lds_read4(lds(&s.maskw[q][w]));
                    for (int sub = 0; sub < 4; sub += mes) {
                        const int j = (w * 4 + sub - mbase[q]) >> shift;
                        if (w * 4 + sub >= mbase[q] && j < L && mask_term(word, (uint32_t)sub, p.mask_dtype) != -INFINITY) seen = j;
                    }
                }
                const uint64_t any = __builtin_amdgcn_ballot_w64(seen >= 0);
                if (any) row = __builtin_amdgcn_readlane(seen, 63 - __builtin_clzll(any)) + 1;
            }
            all = all || row == 0;
            shown = max(shown, row);
        }
        Lv = all ? L : shown;
        mine = stages(Lv);
    }

    bf16x8_t qB[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const U4 x = lds_read16(lds(&s.head[cq][(4 * kk + g) * 16])), zero = {0u, 0u, 0u, 0u};
        qB[kk] = as_bf16x8(c < COLS ? x : zero);
    }
    // one past the column's last visible key: without a mask two tokens attend causally
    const int lim = SQ > 1 && !MASK ? L - SQ + cq / G + 1 : Lv;
    float mx = kEmpty, l = 0.f;
    f32x4_t acc[8];
#pragma unroll
    for (int db = 0; db < 8; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < mine; ++t) {
        // the next stage, into the slot scored last (the first two went out above), once the wave's
        // reads of that slot have returned: the products that use them order nothing against the
        // loads, which the compiler does not see as writes of the slot
        if (issued < mine && issued <= t + 1) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(issued++);
        }
        if (issued > t + 1) wait_loads<kLoads>();
        else wait_loads<0>();
        const uint32_t slot = (t % kStages) * (W * kStage);
        const int w0 = t * SK + wave * kKeys;  // the stage's first key
        if constexpr (FUSED) {
            // the step's keys and values enter the stage at their rows (the loads left zeros)
            const int r = L - SQ + g - w0;
            if (g < SQ && L - SQ + g >= 0 && r >= 0 && r < kKeys) {
                const uint32_t sb = ring + slot + r * kRow;
                lds_write16(sb + ((c ^ r) & 15) * 16, lds_read16(lds(&s.head[NEWK + g][c * 16])));
                lds_write16(sb + kKeys * kRow + ((c ^ (2 * r)) & 15) * 16, lds_read16(lds(&s.head[NEWV + g][c * 16])));
            }
        }
        if constexpr (MASK) {
            // value rows behind the last visible key: their weights are zero, but zero times an
            // infinity or a NaN is not
            if (w0 + kKeys > Lv) {
                const U4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (w0 + 4 * i + g >= Lv) lds_write16(ring + slot + kKeys * kRow + (4 * i + g) * kRow + c * 16, zero);
            }
        }
        f32x4_t st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(lds_read16(ka[kk] + slot)), qB[kk], st, 0, 0, 0);
        const int j0 = w0 + 4 * g;  // the lane's keys: j0 ... j0 + 3
        float x[4];
        if constexpr (MASK) {
            // the terms of keys past the row are whatever follows it in LDS, and not used
            const int tk = SQ > 1 && cq / G ? SQ - 1 : 0;  // the column's token
            mask_terms(lds(&s.maskw[tk][0]) + mbase[tk] + j0 * mes, p.mask_dtype, x);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = st[i] * p.scale_log2;
            if constexpr (MASK) v += x[i];
            x[i] = j0 + i < lim ? v : -INFINITY;
        }
        float mb = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
        if (t == 0 || __builtin_amdgcn_ballot_w64(mb > mx)) {
            mb = fmaxf(mb, xor16(mb));
            mb = fmaxf(mb, xor32(mb));
            const float mn = fmaxf(mx, mb);
            if (t > 0) {
                const float alpha = fexp2(mx - mn);
                l *= alpha;
#pragma unroll
                for (int db = 0; db < 8; ++db) acc[db] *= alpha;
            }
            mx = mn;
        }
        float pw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) pw[i] = fexp2(x[i] - mx);
        l += (pw[0] + pw[1]) + (pw[2] + pw[3]);
        uint2 pp = {cvt_pk_bf16(pw[0], pw[1]), cvt_pk_bf16(pw[2], pw[3])};
        bf16_rest(pw[0], pw[1], pp.x);
        bf16_rest(pw[2], pw[3], pp.y);
        const uint2 second = {cvt_pk_bf16(pw[0], pw[1]), cvt_pk_bf16(pw[2], pw[3])};
        bf16_rest(pw[0], pw[1], second.x);
        bf16_rest(pw[2], pw[3], second.y);
        uint2 third = {cvt_pk_bf16(pw[0], pw[1]), cvt_pk_bf16(pw[2], pw[3])};
        if constexpr (!THIRD) third = part == 0 ? third : uint2{0u, 0u};  // a product of its own
        const uint2 rest = THIRD && part == 2 ? third : second;
        pp = part == 0 ? pp : rest;
        const s16x4_t pv = __builtin_bit_cast(s16x4_t, pp);
#pragma unroll
        for (int db = 0; db < 8; ++db) {
            const s16x4_t v = __builtin_bit_cast(s16x4_t, lds_read_tr16(va[db] + slot));
            acc[db] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v, pv, acc[db], 0, 0, 0);
            if constexpr (!THIRD)
                acc[db] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v, __builtin_bit_cast(s16x4_t, third), acc[db], 0, 0, 0);
        }
    }
    // nothing of the wave's is in flight into LDS from here on (a mask can end the stream early)
    wait_loads<0>();

    if constexpr (FUSED) {
        // the step's rows into the arena, by the wave with the fewest keys
        if (wave == RW && g < SQ) {
            const int row = L - SQ + g;
            if (row >= 0) {
                global_store16(const_cast<char *>(kp) + (uint64_t)((uint32_t)row * p.k_st + c * 16), lds_read16(lds(&s.head[NEWK + g][c * 16])));
                global_store16(const_cast<char *>(vp) + (uint64_t)((uint32_t)row * p.v_st + c * 16), lds_read16(lds(&s.head[NEWV + g][c * 16])));
            }
        }
    }
    // the wave's state: the weight sums over its lane groups and every column's accumulators, into
    // the wave's own (drained) first stage; then the merge of the waves.  Dims 16 db + 4 g ... + 3
    // of column c are chunk (4 db + g) ^ c of its 512 bytes: distinct banks for the columns.
    float lt = l + xor16(l);
    lt += xor32(lt);
    if (c < COLS) {
        if (c < R && g == 0) {
            if (W > 1) s.ml[wave][c][0] = mx;
            s.ml[wave][c][1] = lt;
        }
        const uint32_t state = ring + c * 512 + (g ^ c) * 16;
#pragma unroll
        for (int db = 0; db < 8; ++db)
            lds_write16(state ^ (db * 64), __builtin_bit_cast(U4, acc[db]));
    }
    lds_barrier();
    // The merge: V dims of a query row per thread.  With eight waves so few that all threads take one
    // pass: four dims each, one wave at work for two rows, added up eight waves' three parts in 1-2% of a
    // launch more (28 layers, one request of 200..400 keys 173.4 us, now 171.1).  With four it is the same.
    constexpr int V = W < 8 || 2 * R / W >= 4 ? 4 : 2 * R / W >= 2 ? 2 : 1;
    for (int t = tid; t < R * 128 / V; t += W * 64) {
        const int r = t / (128 / V), d = t % (128 / V) * V;
        const uint32_t from = lds(&s.ring[0][0][0]) + d % 4 * 4;
        // a wave's sums: the parts of the weights added up (unless a sum is infinite, whose
        // remainder may be 0 x inf)
        auto sums = [&](int w, float (&x)[V]) {
            auto column = [&](int c, float (&v)[V]) {
                typedef float floats_t __attribute__((ext_vector_type(V)));
                const floats_t f = *(__attribute__((address_space(3))) const floats_t *)(uintptr_t)(
                    from + w * kStage + c * 512 + ((d / 4) ^ c) * 16);
                __builtin_memcpy(v, &f, sizeof(v));
            };
            float rest[V];
            column(r, x);
            column(r + R, rest);
            if constexpr (THIRD) {
                float third[V];
                column(r + 2 * R, third);
#pragma unroll
                for (int i = 0; i < V; ++i) rest[i] += third[i];
            }
#pragma unroll
            for (int i = 0; i < V; ++i) x[i] = __builtin_fabsf(x[i]) < INFINITY ? x[i] + rest[i] : x[i];
        };
        float sl, sa[V];
        if constexpr (W == 1) {
            sl = s.ml[0][r][1];
            sums(0, sa);
        } else {
            auto merge = [&](auto count) {
                constexpr int N = decltype(count)::value;
                float mm = s.ml[0][r][0];
#pragma unroll
                for (int w = 1; w < N; ++w) mm = fmaxf(mm, s.ml[w][r][0]);
                sl = 0.f;
#pragma unroll
                for (int i = 0; i < V; ++i) sa[i] = 0.f;
#pragma unroll
                for (int w = 0; w < N; ++w) {
                    const float wt = fexp2(s.ml[w][r][0] - mm);
                    float x[V];
                    sums(w, x);
                    sl += s.ml[w][r][1] * wt;
#pragma unroll
                    for (int i = 0; i < V; ++i) sa[i] += x[i] * wt;
                }
            };
            // waves past the keys hold nothing
            if (W > 2 && Lv <= W / 2 * kKeys) merge(std::integral_constant<int, W / 2>{});
            else merge(std::integral_constant<int, W>{});
        }
        const float inv = __builtin_amdgcn_rcpf(sl);
        char *o = out + ((r / G) * p.o_ss + (r % G) * p.o_sh + d * 2);
        uint32_t y[(V + 1) / 2];
#pragma unroll
        for (int i = 0; i < V; i += 2) y[i / 2] = cvt_pk_bf16_canon(sa[i] * inv, sa[V > 1 ? i + 1 : 0] * inv);
        if constexpr (V == 4) {
            if (p.vec_out) {
                global_store8(o, y[0], y[1]);
                continue;
            }
        } else if constexpr (V == 2) {
            if (p.vec_out) {
                global_store4(o, y[0]);
                continue;
            }
        }
#pragma unroll
        for (int i = 0; i < V; ++i) global_store2(o + 2 * i, i % 2 ? y[i / 2] >> 16 : y[i / 2]);
    }
}

// Launch sizes and the arguments that pick an instance.
struct Call {
    int B, Hkv, waves;
    bool mask, norm;
    const int64_t *pos;
    hipStream_t stream;
};

template <int G, int SQ, int FUSE, bool MASK>
static void launch_waves(const Call &a, const DirectParams &p) {
    const dim3 grid((uint32_t)a.Hkv, (uint32_t)a.B);
    if (a.waves == 1) hipLaunchKernelGGL((decode_direct_kernel<G, SQ, FUSE, MASK, 1>), grid, dim3(64), 0, a.stream, a.pos, p);
    else if (a.waves == 4) hipLaunchKernelGGL((decode_direct_kernel<G, SQ, FUSE, MASK, 4>), grid, dim3(256), 0, a.stream, a.pos, p);
    else hipLaunchKernelGGL((decode_direct_kernel<G, SQ, FUSE, MASK, 8>), grid, dim3(512), 0, a.stream, a.pos, p);
}

template <int G, int SQ, int FUSE>
static void launch_mask(const Call &a, const DirectParams &p) {
    if (a.mask) launch_waves<G, SQ, FUSE, true>(a, p);
    else launch_waves<G, SQ, FUSE, false>(a, p);
}

template <int G, int SQ>
static void launch_fuse(const Call &a, bool fused, const DirectParams &p) {
    if (!fused) launch_mask<G, SQ, 0>(a, p);
    else if (a.norm) launch_mask<G, SQ, 2>(a, p);
    else launch_mask<G, SQ, 1>(a, p);
}

template <int G>
static void launch_tokens(const Call &a, int tokens, bool fused, const DirectParams &p) {
    if (tokens == 1) launch_fuse<G, 1>(a, fused, p);
    else launch_fuse<G, 2>(a, fused, p);
}

// Waves per workgroup.  One where the arena's rows are one or two stages of a wave (the code
// predictor's 16-row caches): no merge.  Eight for a few pairs, where a workgroup's own loads in
// flight bound it; four from kDirectManyPairs, where two workgroups share a CU (us per layer, eight /
// four waves: one request of 1750 keys 13.4 / 17.8, 4 of 100..500 7.4 / 7.9, 8 of 30..511 9.0 / 8.5, 64 of
// them 18.4 / 15.8).
static int waves(const DecodeParams &p) {
    static_assert(kDirectOneWave == 2 * kKeys, "two stages");
    if (p.ctx <= kDirectOneWave) return 1;
    return (int64_t)p.B * p.Hkv >= kDirectManyPairs ? 4 : 8;
}

}  // namespace direct

void direct_launch(const DecodeParams &d, int group, int tokens, bool fused, hipStream_t stream) {
    using namespace direct;
    DirectParams p = {};
    p.q = d.q; p.k = d.k; p.v = d.v; p.out = d.out;
    p.nk = d.nk; p.nv = d.nv; p.cs = d.cs; p.sn = d.sn;
    p.mask = d.mask; p.offs = d.offs; p.qnw = d.qnw; p.knw = d.knw;
    auto bytes = [](int64_t elements) { return (uint32_t)(elements * 2); };
    p.q_sb = bytes(d.q_sb); p.q_ss = bytes(d.q_ss); p.q_sh = bytes(d.q_sh);
    p.o_sb = bytes(d.o_sb); p.o_ss = bytes(d.o_ss); p.o_sh = bytes(d.o_sh);
    p.nk_sb = bytes(d.nk_sb); p.nk_sh = bytes(d.nk_sh); p.nk_ss = bytes(d.nk_ss);
    p.nv_sb = bytes(d.nv_sb); p.nv_sh = bytes(d.nv_sh); p.nv_ss = bytes(d.nv_ss);
    p.cs_sb = bytes(d.cs_sb); p.cs_ss = bytes(d.cs_ss);
    p.k_st = bytes(d.k_st); p.v_st = bytes(d.v_st);
    p.k_sb16 = (uint32_t)(d.k_sb / 8); p.k_sh16 = (uint32_t)(d.k_sh / 8);
    p.v_sb16 = (uint32_t)(d.v_sb / 8); p.v_sh16 = (uint32_t)(d.v_sh / 8);
    p.scale_log2 = d.scale_log2; p.eps = d.eps;
    p.ctx = d.ctx; p.mask_dtype = d.mask_dtype; p.m_sb = d.m_sb; p.m_ss = d.m_ss; p.stream = d.stream;
    p.vec_out = ((reinterpret_cast<uintptr_t>(d.out) | p.o_sb | p.o_ss | p.o_sh) & 7) == 0;
    const Call a = {d.B, d.Hkv, waves(d), d.has_mask != 0, d.qnw || d.knw, d.pos, stream};
    switch (group) {
        case 1: launch_tokens<1>(a, tokens, fused, p); break;
        case 2: launch_tokens<2>(a, tokens, fused, p); break;
        default: launch_tokens<4>(a, tokens, fused, p); break;
    }
}

}  // namespace q3t
