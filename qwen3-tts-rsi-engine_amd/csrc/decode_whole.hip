// Decode attention with one workgroup per (request, KV head) on vector instructions: the chunked
// grid's unsplit form for fp32 rows and bf16 rows of 64 (decode_direct.hip takes bf16 rows of 128).
//
// For few requests over short arenas, where the split kernel's workgroups spend more on merging a
// request through memory (publish, count, collect: three device-scope round trips) than on its
// keys.  The waves of a workgroup share the request's keys, all loads of a block issued before any
// math, and merge in LDS, one output per thread.  fp32 throughout, as the split kernel.  Bound by
// the round trips of position, first block and each later block, and, in fp32, by what one CU
// streams of the longest request.
// us per launch, split -> whole (uniform contexts up to the capacity): fp32 rows of 128: 16 requests
// x 512 rows 17.2 -> 14.9, 16 x 128 9.5 -> 6.6, 32 x 256 15.3 -> 11.5, 1 x 512 11.1 -> 8.9; fp32 rows of
// 64: 16 x 512 14.3 -> 8.7, 4 x 1000 13.8 -> 8.3; bf16 rows of 64: 16 x 512 12.3 -> 7.1, 1 x 2000 18.8 ->
// 12.9.
#include "decode_pair.hpp"

namespace q3t {
namespace whole {

constexpr int kWholeWaves = 16;  // bf16 rows of 64

template <typename T, int D, int G, int SQ, bool MASK>
__global__ void __launch_bounds__(kWholeWaves * 64) decode_whole_kernel(DecodeParams p) {
    constexpr int kRows = 64 / DecodeShape<T, D>::LPK * kWholeWaves * 2;  // two passes of the workgroup
    using Work = PairWork<T, D, G, SQ, 0, MASK, false, false, kWholeWaves, kRows>;
    __shared__ typename Work::Lds lds;
    __shared__ typename Work::NewRows snew;
    const int h = blockIdx.x % p.Hkv, b = blockIdx.x / p.Hkv;
    const int64_t pb = p.pos ? p.pos[b] : p.ctx - 1;
    Work work;
    work.load_rows(p, b, h);
    const int L = (pb >= 0 && pb < p.ctx) ? (int)pb + 1 : 0;
    if (L == 0) {
        Work::write_zeros(p, b, h);
        return;
    }
    work.stream(p, b, h, L, 0, L, false, lds, snew);
    for (int t = threadIdx.x; t < Work::R * D; t += kWholeWaves * 64) {
        float a, l, m;
        Work::merge(lds, t, a, l, m);
        const int r = t / D, d = t % D, qi = r / G, hq = h * G + r % G;
        store_out<T>(p.out + (b * p.o_sb + qi * p.o_ss + hq * p.o_sh + d) * (int64_t)sizeof(T), a * __builtin_amdgcn_rcpf(l));
    }
}

// fp32 rows.  Eight lanes hold a key, CH 16-byte chunks each (lane c of the eight: chunks c, c + 8,
// ..., so that a load reads 128 bytes of a row), and a wave scores eight keys at once: the sum of a
// key's partial products crosses three lane exchanges for eight keys, where one chunk per lane took
// five for two.  Bound by vector instructions on the longest requests: a key costs about 12 of a
// wave's (25 with one chunk per lane).
template <int D, int G, int SQ, bool MASK>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) decode_whole_f32_kernel(DecodeParams p) {
    constexpr int W = 8, R = G * SQ, CH = D / 32, P = R > 2 ? 2 : 4;  // passes per block of keys
    constexpr int N = R * CH * 4;                                     // accumulators per lane
    __shared__ float sacc[W][R][D], sml[W][R][2];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 3, c = lane & 7;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x % p.Hkv, b = blockIdx.x / p.Hkv;
    const int64_t pb = p.pos ? p.pos[b] : p.ctx - 1;
    float4 q[R][CH];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < CH; ++j)
            q[r][j] = *reinterpret_cast<const float4 *>(p.q + (b * p.q_sb + (r / G) * p.q_ss + (h * G + r % G) * p.q_sh) * 4 + (c + 8 * j) * 16);
    const int L = (pb >= 0 && pb < p.ctx) ? (int)pb + 1 : 0;
    auto out_at = [&](int r, int d) {
        return reinterpret_cast<float *>(p.out + (b * p.o_sb + (r / G) * p.o_ss + (h * G + r % G) * p.o_sh + d) * 4);
    };
    if (L == 0) {
        for (int t = tid; t < R * D; t += W * 64) *out_at(t / D, t % D) = 0.f;
        return;
    }
    const char *kb = p.k + ((p.offs ? p.offs[b] : (int64_t)b * p.k_sb) + h * p.k_sh) * 4;
    const char *vb = p.v + ((p.offs ? p.offs[b] : (int64_t)b * p.v_sb) + h * p.v_sh) * 4;
    const int kst = (int)(p.k_st * 4), vst = (int)(p.v_st * 4);
    const auto krs = buffer_rsrc(uniform_ptr(kb), (uint32_t)((p.ctx - 1) * kst + D * 4));
    const auto vrs = buffer_rsrc(uniform_ptr(vb), (uint32_t)((p.ctx - 1) * vst + D * 4));
    const int mes = MASK ? mask_elem_size(p.mask_dtype) : 0;
    const char *mask_row = MASK ? p.mask + b * p.m_sb * mes : nullptr;
    float m[R], l[R], acc[R][CH][4];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        m[r] = kEmpty;
        l[r] = 0.f;
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r][j][e] = 0.f;
    }
    for (int jb = wave * 8; jb < L; jb += W * 8 * P) {
        // the block's rows, all loads before any math (rows at or past L read zeros without an access)
        float4 kr[P][CH], vr[P][CH];
        float mk[P][SQ];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const int key = jb + u * W * 8 + g;
            const uint32_t ko = key < L ? (uint32_t)(key * kst) + c * 16 : 0xffff0000u, vo = key < L ? (uint32_t)(key * vst) + c * 16 : 0xffff0000u;
#pragma unroll
            for (int j = 0; j < CH; ++j) kr[u][j] = __builtin_bit_cast(float4, buffer_load16(krs, ko + 128 * j));
#pragma unroll
            for (int j = 0; j < CH; ++j) vr[u][j] = __builtin_bit_cast(float4, buffer_load16(vrs, vo + 128 * j));
#pragma unroll
            for (int qi = 0; qi < SQ; ++qi) {
                mk[u][qi] = 0.f;
                if (MASK && key < L) mk[u][qi] = load_mask(mask_row + (qi * p.m_ss + (int64_t)key * p.m_st) * mes, p.mask_dtype) * kLog2e;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float x[P];
#pragma unroll
            for (int u = 0; u < P; ++u) {
                float s = 0.f;
                if (jb + u * W * 8 < L)  // uniform: passes past the request's keys cost nothing
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    s += q[r][j].x * kr[u][j].x;
                    s += q[r][j].y * kr[u][j].y;
                    s += q[r][j].z * kr[u][j].z;
                    s += q[r][j].w * kr[u][j].w;
                }
                const int key = jb + u * W * 8 + g;
                // several queries of a request without a mask: causal among the last keys
                const bool seen = key < L && (MASK || SQ == 1 || key <= L - SQ + r / G);
                x[u] = seen ? sum8(s) * p.scale_log2 + mk[u][r / G] : -INFINITY;
            }
            float mb = x[0];
#pragma unroll
            for (int u = 1; u < P; ++u) mb = fmaxf(mb, x[u]);
            const float mn = fmaxf(m[r], cross_max<8>(mb)), alpha = fexp2(m[r] - mn);
            l[r] *= alpha;
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][j][e] *= alpha;
            m[r] = mn;
#pragma unroll
            for (int u = 0; u < P; ++u) {
                if (jb + u * W * 8 >= L) break;
                const float w = fexp2(x[u] - mn);
                l[r] += w;
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    acc[r][j][0] += w * vr[u][j].x;
                    acc[r][j][1] += w * vr[u][j].y;
                    acc[r][j][2] += w * vr[u][j].z;
                    acc[r][j][3] += w * vr[u][j].w;
                }
            }
        }
    }
    // the wave's state, summed over its eight keys, and the merge of the waves
    float v[N], h2[N / 2], q4[N / 4];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float a = acc[i / (CH * 4)][i / 4 % CH][i % 4];
        v[i] = a + xor8(a);
    }
    sum_halves<N>(v, h2);
    sum_rows<N>(h2, q4);
    if ((lane & 8) == 0) {
        const int sel = kRowElem[lane >> 4];
#pragma unroll
        for (int k = 0; k < N / 4; ++k) sacc[wave][k / CH][(c + 8 * (k % CH)) * 4 + sel] = q4[k];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float lt = cross_sum<8>(l[r]);
        if (lane == 0) {
            sml[wave][r][0] = m[r];
            sml[wave][r][1] = lt;
        }
    }
    __syncthreads();
    for (int t = tid; t < R * D; t += W * 64) {
        const int r = t / D, d = t % D;
        float mx = sml[0][r][0];
#pragma unroll
        for (int w = 1; w < W; ++w) mx = fmaxf(mx, sml[w][r][0]);
        float sl = 0.f, sa = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float wt = fexp2(sml[w][r][0] - mx);
            sl += sml[w][r][1] * wt;
            sa += sacc[w][r][d] * wt;
        }
        *out_at(r, d) = sa * __builtin_amdgcn_rcpf(sl);
    }
}

// Both kernels' launches: bf16 rows of 64 (T = uint16_t) and fp32 rows.
template <typename T, int D, int G, int SQ, bool MASK>
static void launch_one(const DecodeParams &p, hipStream_t s) {
    const dim3 grid((uint32_t)p.B * p.Hkv);
    if constexpr (sizeof(T) == 2) hipLaunchKernelGGL((decode_whole_kernel<T, D, G, SQ, MASK>), grid, dim3(kWholeWaves * 64), 0, s, p);
    else hipLaunchKernelGGL((decode_whole_f32_kernel<D, G, SQ, MASK>), grid, dim3(512), 0, s, p);
}

template <typename T, int D, int G>
static void launch(const DecodeParams &p, int tokens, hipStream_t s) {
    if (tokens == 1) {
        if (p.has_mask) launch_one<T, D, G, 1, true>(p, s);
        else launch_one<T, D, G, 1, false>(p, s);
    } else if constexpr (G <= 2) {  // eight query rows do not fit a wave's registers
        if (p.has_mask) launch_one<T, D, G, 2, true>(p, s);
        else launch_one<T, D, G, 2, false>(p, s);
    }
}

template <typename T, int D>
static void launch_group(const DecodeParams &p, int group, int tokens, hipStream_t s) {
    if (group == 1) launch<T, D, 1>(p, tokens, s);
    else if (group == 2) launch<T, D, 2>(p, tokens, s);
    else launch<T, D, 4>(p, tokens, s);
}

}  // namespace whole

void whole_launch(const DecodeParams &p, bool f32, int head_dim, int group, int tokens, hipStream_t s) {
    if (!f32) whole::launch_group<uint16_t, 64>(p, group, tokens, s);
    else if (head_dim == 128) whole::launch_group<float, 128>(p, group, tokens, s);
    else whole::launch_group<float, 64>(p, group, tokens, s);
}

}  // namespace q3t
