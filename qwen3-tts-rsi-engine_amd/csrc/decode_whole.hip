// Decode attention with one workgroup per (request, KV head) on vector instructions: the chunked
// grid's unsplit form for bf16 rows of 64 (decode_direct.hip takes bf16 rows of 128).
//
// For few requests over short arenas, where the split kernel's workgroups spend more on merging a
// request through memory (publish, count, collect: three device-scope round trips) than on its
// keys.  The waves of a workgroup share the request's keys, all loads of a block issued before any
// math, and merge in LDS, one output per thread.  fp32 sums, as the split kernel.  Bound by the
// round trips of position, first block and each later block.
// us per launch, split -> whole (uniform contexts up to the capacity): 16 requests x 512 rows 12.3 ->
// 7.1, 1 x 2000 18.8 -> 12.9.
// fp32 rows stay split: eight lanes to a key took an fp32 step of 16 requests from 218 to 202 us, but
// in its order of the sums the relative error against float64 was 1-3% above the split kernel's
// (64 calls of rows of 64 under a mask: 1.409 against 1.370e-7).
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
    const int64_t pb = p.pos[b];
    Work work;
    work.load_rows(p, b, h);
    const int L = keys_of(p, pb);
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

template <typename T, int D, int G, int SQ, bool MASK>
static void launch_one(const DecodeParams &p, hipStream_t s) {
    hipLaunchKernelGGL((decode_whole_kernel<T, D, G, SQ, MASK>), dim3((uint32_t)p.B * p.Hkv), dim3(kWholeWaves * 64), 0, s, p);
}

template <typename T, int D, int G>
static void launch(const DecodeParams &p, int tokens, hipStream_t s) {
    if (tokens == 1) {
        if (p.mask) launch_one<T, D, G, 1, true>(p, s);
        else launch_one<T, D, G, 1, false>(p, s);
    } else if constexpr (G <= 2) {  // eight query rows do not fit a wave's registers
        if (p.mask) launch_one<T, D, G, 2, true>(p, s);
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

void whole_launch(const DecodeParams &p, int group, int tokens, hipStream_t s) {
    whole::launch_group<uint16_t, 64>(p, group, tokens, s);
}

}  // namespace q3t
