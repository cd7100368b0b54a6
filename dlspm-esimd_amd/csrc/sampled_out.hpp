// SDDMM: where results go, and the sampled dot products of a run of one row's nonzeros (sddmm.hip, sddmm_tiles.hip).
#pragma once

#include "common.hpp"
#include "launch.hpp"

namespace dlspm {

// Where the results go. Results of more than one and a half times what one L2 holds (6 MiB on an MI355X) are stored with
// the non-temporal hint: ordinary stores are held in the L2 as dirty lines and written back later, hinted ones drain as
// they are issued. (The L2's hit rate and the bytes fetched do not change by it; the time does.) Measured with both
// kinds of store in one process, D = 32 / 128: 24576 x 8192 at density 0.3 (230 MiB of results) 443 -> 297 us /
// 1287 -> 1089 us; 8192 x 2048 at 0.3 (19 MiB) 32.5 -> 28.1 us / 90.6 -> 88.3 us; 6144 x 2048 at 0.2 (9.6 MiB) -3.5 % /
// -4.4 %; 6.4 MiB -1.2 % / -1.8 %; 4.8 MiB +0.4 ... +2.2 % / equal. Small results lose by the hint -- neighbouring waves
// share cache lines here, and a kernel ends when its stores have reached memory -- (2048 x 2048 at 5 %, 0.8 MiB: +8 % /
// +4 %) and keep ordinary stores.
struct SampledOut {
    float* __restrict__ at;
    int streaming;
    __device__ __forceinline__ void store(int j, float v) const
    {
        // (wave-uniform) The hinted store is written out as an instruction: __builtin_nontemporal_store on one side of
        // this branch and a plain store on the other are merged into one store by the compiler, and the hint is lost.
        // (A vector store like any other; the wait counts that the compiler inserts can only become stricter by it.)
        if (streaming) asm volatile("global_store_dword %0, %1, off nt" : : "v"(at + j), "v"(v) : "memory");
        else at[j] = v;
    }
};
static inline SampledOut sampled_out(const SddmmArgs& x)
{
    const int forced = tuning().stream_results;  // -1: the size rule (sweeps and tests switch it off or on)
    const long long l2 = x.l2_bytes;
    const bool by_rule = (long long)x.nnz * (long long)sizeof(float) > l2 + l2 / 2;
    return SampledOut{x.out, (forced < 0 ? by_rule : forced != 0) ? 1 : 0};
}

// out[j] = <lhs_row, rhs[col_indices[j]]> for the nonzeros j in [p, q) of one row (p < q, wave-uniform), 64 at a time: all of
// them, or (several waves in turn) every `step`-th 64.
template <int VEC, int G1, int DS, int MASKED, int FLIGHT = 8, typename Out>
__device__ __forceinline__ void sddmm_segment(int p, int q, int D, const int* __restrict__ col_indices,
                                              const float* __restrict__ lhs_row, const float* __restrict__ rhs,
                                              Out out, int lane, int step = 1)
{
    using VecT = Vec<VEC>;
    const int g = lane % G1;
    VecT lq[DS > 0 ? DS : 1];
    if constexpr (DS > 0) {
#pragma unroll
        for (int s = 0; s < DS; ++s) {
            const int d = (s * G1 + g) * VEC;
            if constexpr (MASKED) lq[s] = d < D ? VecT::gload_clip(lhs_row, d, D) : VecT::zero();
            else lq[s] = VecT::gload(lhs_row + d);
        }
    }
    // 64 column indices per pass, one per lane; the next 64 are requested (index clamped, no condition) before
    // the rhs rows of the current ones
    int c_nxt = col_indices[min(p + lane, q - 1)];
    for (int base = p; base < q; base += step * kWave) {
        const int c = base + lane < q ? c_nxt : 0;
        c_nxt = col_indices[min(base + step * kWave + lane, q - 1)];
        const int cnt = min(kWave, q - base);
        const float o = sddmm_chunk<VEC, G1, DS, MASKED, FLIGHT>(D, lane, cnt, c, lhs_row, lq, rhs);
        if (base + lane < q) out.store(base + lane, o);
    }
}

}  // namespace dlspm
