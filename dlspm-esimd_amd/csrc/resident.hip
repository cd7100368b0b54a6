// SpMM on matrices dense enough that every row of B is used by many rows of a workgroup: B is gathered from LDS.
//
// What bounds the row-block kernels (spmm.hip) is a compute unit's vector-memory path, 64 bytes per clock: every nonzero
// gathers its row of B through it. LDS delivers four times as much, so here a workgroup of sixteen waves owns 64 RR rows and
// one tile of 64 columns, and goes through the columns of the matrix in slices of KS: the slice's KS x 64 floats of B lie
// in LDS (two buffers: the next slice is fetched while the current one is worked on), and the waves gather from there.
//   * Sixteen lanes (one DPP row) work on one row of the matrix, four floats of the tile each; a wave works on four
//     rows at a time. The sixteen lanes hold 16 x 4 consecutive (column, value) pairs of their row, and the pair in
//     use is handed to the whole group by DPP row_newbcast inside the instruction that uses it: the address of the LDS
//     read is one v_add_u32_dpp, the four products are v_fmac_f32_dpp. No ds_bpermute (it would share the LDS pipe with
//     the reads) and no v_readlane (four rows have four different pairs).
//   * A row's pairs are consumed in CSR order through all slices, so its sum is the plain sequential one, whatever RR and
//     KS are: deterministic, no partial rows, no second kernel, no workspace.
//   * Where a slice ends in a row is found on the way (the first column of the row's next pairs that lies past the slice), so
//     nothing is needed beforehand. Columns that do not ascend are stopped at: what is left of such a row after the last
//     slice is gathered from memory, in order.
//   * The rows of a workgroup are sorted by length and dealt to the waves in quads, so that the four rows a wave works on are
//     about equally long and the four SIMDs have about the same to do.
// Measured (three operand sets in turn): 8192 x 8192, N = 128, density 0.1 119 -> 88 us; 32768 x 8192, density 0.3 1587 -> 612 us;
// 2048 x 512, N = 392, 102 nonzeros per row 14.9 -> 12.0 us (more at spmm_resident_choose). A step (four nonzeros x 64 columns
// of one wave) costs 7.4 clocks of a compute unit, where its LDS read by itself would cost 4.9 and its five vector
// instructions 5.3; in the row-block kernels the same four nonzeros cost 22. Matrix cores on a densified A were slower (16384 x
// 8192, density 0.3, N = 128: 505 us, this 335): the scatter and its barriers, not the products, set the time there.
// The reference has no counterpart (SPMM/spmmesimd2.hpp:63-147 gathers every row of B from memory).
#include <algorithm>
#include <cmath>
#include <utility>

#include "common.hpp"
#include "launch.hpp"

namespace dlspm {

constexpr int kResidentWaves = 16, kResidentThreads = kResidentWaves * 64;
constexpr int kResidentRows = 4 * kResidentWaves;  // rows of a workgroup and RR
constexpr int kResidentTile = 64;                  // columns of B
constexpr int kTileRowBytes = kResidentTile * (int)sizeof(float);
constexpr int kResidentMaxSlice = 304;  // two buffers of 304 rows of 256 bytes, a row of zeros: 152 of 160 KiB
constexpr int kLanePairs = 4, kChunk = 16 * kLanePairs;  // pairs per lane and load, pairs of a row per load

template <int LANE> __device__ __forceinline__ int row_bcast(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, 0x150 + LANE, 0xF, 0xF, true);
}

// acc += a[lane LANE of the DPP row] * b. The first of a run waits out the two states that a DPP operand needs after a
// vector write of its register (the compiler does not see the DPP operand inside the asm).
template <int LANE, bool FIRST> __device__ __forceinline__ void fmac_bcast(float4& acc, float a, const float4& b)
{
#define DLSPM_FMAC_BCAST                                                                                              \
    "v_fmac_f32_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"                                        \
    "v_fmac_f32_dpp %1, %4, %6 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"                                        \
    "v_fmac_f32_dpp %2, %4, %7 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"                                        \
    "v_fmac_f32_dpp %3, %4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
    if constexpr (FIRST)
        asm("s_nop 1\n\t" DLSPM_FMAC_BCAST
            : "+v"(acc.x), "+v"(acc.y), "+v"(acc.z), "+v"(acc.w)
            : "v"(a), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w), "n"(LANE));
    else
        asm(DLSPM_FMAC_BCAST
            : "+v"(acc.x), "+v"(acc.y), "+v"(acc.z), "+v"(acc.w)
            : "v"(a), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w), "n"(LANE));
#undef DLSPM_FMAC_BCAST
}

// The pairs of lanes LANE0 .. LANE0 + LANES - 1 of every group, in order: `at` = byte offset of each pair's row in `tiles`
template <int LANE0, int... I>
__device__ __forceinline__ void resident_steps(const char* tiles, const int* at, int lane_bytes, const float* a, float4& acc,
                                               std::integer_sequence<int, I...>)
{
    float4 b[sizeof...(I)];
    ((b[I] = *reinterpret_cast<const float4*>(tiles + (row_bcast<LANE0 + I / kLanePairs>(at[I % kLanePairs]) + lane_bytes))), ...);
    (fmac_bcast<LANE0 + I / kLanePairs, I == 0>(acc, a[I % kLanePairs], b[I]), ...);
}
// ... of all sixteen lanes, two lanes' eight pairs in flight at a time
template <int... L>
__device__ __forceinline__ void resident_full_chunk(const char* tiles, const int* at, int lane_bytes, const float* a, float4& acc,
                                                    std::integer_sequence<int, L...>)
{
    (resident_steps<2 * L>(tiles, at, lane_bytes, a, acc, std::make_integer_sequence<int, 2 * kLanePairs>{}), ...);
}
// ... of the lanes of which some group has pairs: a prefix, one bit per lane in `lanes`
template <int L>
__device__ __forceinline__ bool resident_lane(const char* tiles, const int* at, int lane_bytes, const float* a, float4& acc, unsigned lanes)
{
    if ((lanes >> L & 1) == 0) return false;
    resident_steps<L>(tiles, at, lane_bytes, a, acc, std::make_integer_sequence<int, kLanePairs>{});
    return true;
}
template <int... L>
__device__ __forceinline__ void resident_part_chunk(const char* tiles, const int* at, int lane_bytes, const float* a, float4& acc,
                                                    unsigned lanes, std::integer_sequence<int, L...>)
{
    (void)(resident_lane<L>(tiles, at, lane_bytes, a, acc, lanes) && ...);
}

// QC: chunks of 64 pairs of a row that are loaded ahead (a slice's share of a row is to fit them: what exceeds it is loaded
// when it is needed, with nothing to hide the latency behind). SLICE rows of B per slice.
template <int RR, int QC>
__global__ __launch_bounds__(kResidentThreads) void spmm_resident_kernel(int M, int K, int N, int nnz, int slice, int col_tiles,
                                                                         int tiles_per_xcd, int streaming, const int* __restrict__ row_offsets,
                                                                         const int* __restrict__ col_indices,
                                                                         const float* __restrict__ values,
                                                                         const float* __restrict__ B, float* __restrict__ C)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    constexpr int kRows = kResidentRows * RR;
    extern __shared__ __attribute__((aligned(1024))) char tiles[];  // two slices of B, one row of zeros
    const int buffer_bytes = slice * kTileRowBytes, zeros = 2 * buffer_bytes;

    const int t = threadIdx.x, lane = t & 63, g = lane >> 4, l = lane & 15, lane_bytes = l * 16;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    int ct, row0;
    if (tiles_per_xcd) {
        // the column tiles of a row block go to the same XCD (workgroup 8 j + x runs on XCD x) one after the other: the
        // second finds the CSR arrays in that XCD's L2 (16384 x 8192 at density 0.3, N = 128: 351 -> 335 us)
        const int at_xcd = (int)(blockIdx.x >> 3);
        ct = at_xcd % col_tiles;
        row0 = ((at_xcd / col_tiles) * 8 + (int)(blockIdx.x & 7)) * kRows;
        if (row0 >= M) return;  // (the grid is rounded up to whole XCDs)
    } else {
        const int row_blocks = (M - 1) / kRows + 1;
        ct = (int)blockIdx.x / row_blocks;
        row0 = ((int)blockIdx.x - ct * row_blocks) * kRows;
    }
    const int col = min(ct * kResidentTile + l * 4, N - 4);  // a lane past the width moves back to end with it, as everywhere

    const __amdgpu_buffer_rsrc_t columns_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(col_indices), 0, nnz * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t values_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(values), 0, nnz * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t B_buffer =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, (int)((unsigned)K * (unsigned)N * 4u), 0x00020000);

    // ---- fetching a slice of B: 64 rows per pass of the workgroup
    constexpr int kPasses = (kResidentMaxSlice + kResidentRows - 1) / kResidentRows;
    u4 fetched[kPasses];
    const unsigned fetch_at = (unsigned)(t >> 4) * (unsigned)N * 4u + (unsigned)col * 4u;
    auto fetch = [&](int s) {  // (rows past K: the buffer's range check returns zeros)
#pragma unroll
        for (int q = 0; q < kPasses; ++q)
            if (q * kResidentRows + 4 * w < slice)
                fetched[q] = __builtin_amdgcn_raw_buffer_load_b128(B_buffer, fetch_at, (unsigned)(s * slice + q * kResidentRows) * (unsigned)N * 4u, 0);
    };
    auto put = [&](int buffer) {
#pragma unroll
        for (int q = 0; q < kPasses; ++q)
            if (q * kResidentRows + 4 * w < slice)
                *reinterpret_cast<u4*>(tiles + buffer * buffer_bytes + (q * kResidentRows + (t >> 4)) * kTileRowBytes + lane_bytes) = fetched[q];
    };
    fetch(0);

    // ---- the rows, longest first: every row counts the rows in front of it
    int* const lengths = reinterpret_cast<int*>(tiles);
    int* const order = lengths + kRows;
    if (t < kRows) lengths[t] = row0 + t < M ? row_offsets[row0 + t + 1] - row_offsets[row0 + t] : -1;
    __syncthreads();
    if (t < kRows) {
        const int mine = lengths[t];
        int before = 0;
        for (int i = 0; i < kRows; i += 4) {
            const int4 x = *reinterpret_cast<const int4*>(lengths + i);
            before += (x.x > mine || (x.x == mine && i < t)) + (x.y > mine || (x.y == mine && i + 1 < t)) +
                      (x.z > mine || (x.z == mine && i + 2 < t)) + (x.w > mine || (x.w == mine && i + 3 < t));
        }
        order[before] = row0 + t;
    }
    __syncthreads();
    int row[RR], p[RR], end[RR], c[RR][QC][kLanePairs];
    float a[RR][QC][kLanePairs];
    float4 acc[RR];
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
        // quads of four rows, longest first, dealt to the four SIMDs (wave w runs on SIMD w mod 4) forwards and backwards in turn
        const int quad = rr * kResidentWaves + w, turn = quad >> 2;
        const int dealt = (turn & 1) ? (turn << 2) + 3 - (quad & 3) : quad;
        row[rr] = order[dealt * 4 + g];
        const bool exists = row[rr] < M;
        p[rr] = exists ? row_offsets[row[rr]] : 0;  // (the group's position; each lane's first pair is 4 l behind it)
        end[rr] = exists ? row_offsets[row[rr] + 1] : 0;
        acc[rr] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    auto load_pairs = [&](int rr) {
#pragma unroll
        for (int q = 0; q < QC; ++q) {
            const unsigned at = (unsigned)(p[rr] + kLanePairs * l) * 4u + (unsigned)(q * kChunk * 4);
            const u4 x = __builtin_amdgcn_raw_buffer_load_b128(columns_buffer, at, 0, 0), y = __builtin_amdgcn_raw_buffer_load_b128(values_buffer, at, 0, 0);
#pragma unroll
            for (int i = 0; i < kLanePairs; ++i) {
                c[rr][q][i] = (int)x[i];
                a[rr][q][i] = __uint_as_float(y[i]);
            }
        }
    };
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) load_pairs(rr);
    __syncthreads();  // (`order` is read; the slices may be written over it)
    put(0);
    if (t < 16) *reinterpret_cast<float4*>(tiles + zeros + t * 16) = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();

    constexpr unsigned long long kFirstLanes = 0x0001000100010001ull, kLastLanes = 0x8000800080008000ull;  // of the four groups
    unsigned stuck = 0;  // bit rr: the row's columns do not ascend; the rest of it is done at the end
    const int slices = (K + slice - 1) / slice;
    for (int s = 0; s < slices; ++s) {
        if (s + 1 < slices) fetch(s + 1);
        const int k0 = s * slice, base = (s & 1) * buffer_bytes;
#pragma unroll
        for (int rr = 0; rr < RR; ++rr) {
            bool more = (stuck >> rr & 1) == 0;
            unsigned long long stopped = 0;  // lanes of the groups that have met the end of the slice (or of their row)
            while (more) {
                more = false;
                bool next = true;
                const int left0 = end[rr] - p[rr] - kLanePairs * l;
#pragma unroll
                for (int q = 0; q < QC; ++q) {
                    if (!next) continue;
                    int at[kLanePairs];
                    unsigned long long in[kLanePairs], all = ~0ull;  // which lanes' pairs lie in this slice
                    const int left = left0 - q * kChunk;             // pairs of the row from the lane's first on
#pragma unroll
                    for (int i = 0; i < kLanePairs; ++i) {
                        const int k = c[rr][q][i] - k0;
                        in[i] = __ballot((unsigned)k < (unsigned)slice) & __ballot(i < left);
                        all &= in[i];
                        at[i] = k * kTileRowBytes + base;
                    }
                    if (all == ~0ull) {
                        resident_full_chunk(tiles, at, lane_bytes, a[rr][q], acc[rr], std::make_integer_sequence<int, 8>{});
                        p[rr] += kChunk;
                        if (q == QC - 1) more = true;
                        continue;
                    }
                    // in CSR order the pairs of this slice come first; anything else is left for the end
                    unsigned long long disorder = (in[0] & stopped) | (in[0] & ~(in[kLanePairs - 1] << 1) & ~kFirstLanes);
#pragma unroll
                    for (int i = 1; i < kLanePairs; ++i) disorder |= in[i] & ~in[i - 1];
                    if (disorder != 0) {
                        stuck |= 1u << rr;
                        next = false;
                        continue;
                    }
                    const unsigned long long open = ~in[kLanePairs - 1] & kLastLanes;
                    stopped = (open - (open >> 15)) | open;
                    unsigned lanes = (unsigned)in[0] | (unsigned)(in[0] >> 32);
                    lanes = (lanes | (lanes >> 16)) & 0xffffu;
                    int n = 0;
                    float av[kLanePairs];
#pragma unroll
                    for (int i = 0; i < kLanePairs; ++i) {
                        const bool mine = __builtin_amdgcn_inverse_ballot_w64(in[i]);
                        n += mine ? 1 : 0;
                        at[i] = mine ? at[i] : zeros;
                        av[i] = mine ? a[rr][q][i] : 0.f;
                    }
                    n += __builtin_amdgcn_update_dpp(0, n, 0x128, 0xf, 0xf, true);  // row_ror: the sum over the group
                    n += __builtin_amdgcn_update_dpp(0, n, 0x124, 0xf, 0xf, true);
                    n += __builtin_amdgcn_update_dpp(0, n, 0x122, 0xf, 0xf, true);
                    n += __builtin_amdgcn_update_dpp(0, n, 0x121, 0xf, 0xf, true);
                    p[rr] += n;
                    resident_part_chunk(tiles, at, lane_bytes, av, acc[rr], lanes, std::make_integer_sequence<int, 16>{});
                    next = (in[kLanePairs - 1] & kLastLanes) != 0;  // some group goes on
                    if (q == QC - 1) more = next;
                }
                load_pairs(rr);
            }
        }
        if (s + 1 < slices) put((s + 1) & 1);
        __syncthreads();
    }

#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
        if (row[rr] >= M) continue;
        for (int j = p[rr]; j < end[rr]; ++j) {
            const float v = values[j];
            Vec<4> b = Vec<4>::gload(B + (size_t)col_indices[j] * N + col), sum{acc[rr]};
            sum.fma(v, b);
            acc[rr] = sum.v;
        }
        if (ct * kResidentTile + l * 4 < N) Vec<4>{acc[rr]}.gstore(C + (size_t)row[rr] * N + col, streaming != 0);
    }
}

template <int RR, int QC> static hipError_t launch_one(const SpmmArgs& x, const ResidentPlan& plan, hipStream_t stream)
{
    const int col_tiles = (int)ceil_div(x.N, kResidentTile);
    const long long row_blocks = ceil_div(x.M, kResidentRows * RR);
    const bool tiles_per_xcd = col_tiles > 1 && row_blocks >= 64;  // (rounding few row blocks up to eight would leave XCDs idle)
    const long long blocks = (tiles_per_xcd ? (row_blocks + 7) / 8 * 8 : row_blocks) * col_tiles;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const size_t lds = (size_t)(2 * plan.slice + 1) * kTileRowBytes;
    const auto kernel = &spmm_resident_kernel<RR, QC>;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                          (2 * kResidentMaxSlice + 1) * kTileRowBytes);
    if (allowed != hipSuccess) return allowed;
    const int stream_rule = tuning().stream_results;
    const bool streaming = stream_rule < 0 ? (long long)x.M * x.N >= 1024 * 1024 : stream_rule != 0;  // (as dense_rows_window)
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kResidentThreads), lds, stream, x.M, x.K, x.N, x.nnz, plan.slice, col_tiles,
                       tiles_per_xcd ? 1 : 0, streaming ? 1 : 0, x.row_offsets, x.col_indices, x.values, x.B, x.C);
    return hipGetLastError();
}

// The resident schedule for these sizes, or rr == 0: where its estimated time is below 0.9 of the row-block kernels'.
// Both estimates (us) are fits to three operand sets worked on in turn, M = 128 ... 32768, K = 512 ... 8192, N = 48 ... 3136,
// density 0.05 ... 0.5 (700 timings, the second within 6 % of them):
//   row-block   2 + nnz width x 1.55e-7 (8192 x 8192, N = 128, density 0.1 / 0.2 / 0.3: 119 ... 136 / 291 / 428);
//   resident    rounds of one workgroup per compute unit x (3.6 + 1.2 rr + 0.55 slices + K / 304 rr (1.0 + 15.6 density)): the
//               start, what a slice costs whatever is in it (its barrier, the ends of its rows), and its steps (the same
//               cases at rr = 1: 95 / 153 / 189; 32768 x 8192 at rr = 2: 310 / 499 / 617, row-block 588 / 1077 / 1587).
// Rows per workgroup: as many as keep the compute units in step. The four rows that a wave works on wait for the longest
// of them and all waves of a workgroup for the slowest, so uneven rows take longer, the more the fewer rows a workgroup has
// and the shorter they are (lognormal rows, sigma 0.6, against Bernoulli rows: rr = 1 2.2 / 1.7 / 1.35 / 1.0 of the time at
// density 0.1 / 0.2 / 0.3 / 0.5, rr = 2 1.75 / 1.3 / 1.05 / 1.0): calls with a row plan or a cut plan count that in full, calls
// that say nothing about their rows against the 1.2 that such rows cost the row-block kernels, and calls with the
// even-rows hint not at all.
ResidentPlan spmm_resident_choose(const DeviceInfo& dev, int M, int K, int N, int nnz, bool rows_even, bool planned)
{
    const Tuning& t = tuning();
    const ResidentPlan none{0, 0, 0};
    if (!rule_on(kRuleResidentSlices) || N < 4 || M <= 0 || K <= 0 || nnz <= 0 || nnz >= (1 << 29) || !dense_fits_buffer(K, N)) return none;
    // (a schedule that was asked for by name)
    if (t.split_w > 0 || t.flat >= 0 || t.slices >= 0 || t.tile_major >= 0 || t.tile_width > 0 || t.plan_order > 0 || t.xcd_contiguous) return none;
    const double density = (double)nnz / ((double)M * K);
    const long long slices = ceil_div(K, kResidentMaxSlice), col_tiles = ceil_div(N, kResidentTile);
    const int slice = (int)(ceil_div(ceil_div(K, slices), 16) * 16);  // (at most the largest: 304 is a multiple of 16)
    // two chunks of 64 pairs ahead where a slice's share of a row exceeds one: mean and two deviations of a Bernoulli row
    const double share = density * slice;
    const int chunks = share + 2.0 * std::sqrt(share * (1.0 - density)) > (double)kChunk ? 2 : 1;
    // what a dense row costs the row-block kernels: half of the lanes that its layout leaves idle count
    const double width = N <= 32 ? 32 : N <= 64 ? 64 : N <= 128 ? 0.5 * (N + 128) : N <= 256 ? 0.5 * (N + 256) : N;
    const double row_block_us = 2.0 + (double)nnz * width * 1.55e-7;
    ResidentPlan best = none;
    double best_us = 0.9 * row_block_us;
    for (int rr = 1; rr <= (chunks == 1 ? 4 : 3); ++rr) {
        const long long workgroups = ceil_div(M, kResidentRows * rr) * col_tiles, rounds = ceil_div(workgroups, dev.cus);
        if (8 * workgroups < 5ll * dev.cus) break;  // (the others' vector-memory paths would go unused)
        double us = (double)rounds * (3.6 + 1.2 * rr + 0.55 * (double)slices + K / 304.0 * rr * (1.0 + 15.6 * density));
        const double uneven = std::max(1.0, rr == 1 ? 1.0 + 3.5 * (0.45 - density) : 1.0 + 3.8 * (0.3 - density));
        if (planned) us *= uneven;
        else if (!rows_even) us *= std::max(1.0, uneven / (M <= 16 * dev.cus ? 1.5 : 1.15));
        if (us < best_us) {
            best_us = us;
            best = ResidentPlan{rr, chunks, slice};
        }
    }
    return best;
}

hipError_t spmm_resident_launch(const SpmmArgs& x, const ResidentPlan& plan, hipStream_t stream)
{
    if (plan.chunks == 1) {
        if (plan.rr == 1) return launch_one<1, 1>(x, plan, stream);
        if (plan.rr == 2) return launch_one<2, 1>(x, plan, stream);
        if (plan.rr == 3) return launch_one<3, 1>(x, plan, stream);
        if (plan.rr == 4) return launch_one<4, 1>(x, plan, stream);
    } else {
        if (plan.rr == 1) return launch_one<1, 2>(x, plan, stream);
        if (plan.rr == 2) return launch_one<2, 2>(x, plan, stream);
        if (plan.rr == 3) return launch_one<3, 2>(x, plan, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace dlspm
