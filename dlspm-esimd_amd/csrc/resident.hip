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
//   * A row's pairs are consumed in CSR order through all slices, in chunks of up to 64 that end where the slice does. A chunk is
//     summed in two chains (four where two chunks are loaded ahead), the chunks' sums are added in 64 bits: no partial rows, no
//     second kernel, no workspace, the same bits whatever RR is, and an error against 64 bits of 6.6e-8 ... 7.8e-8 for rows of 50
//     ... 2500 nonzeros (the row-block kernels' 2 ... 128 chains per row: 7.7e-8 ... 5.7e-7 on the same calls). One chain per
//     row costs 4 % less (8192 x 8192 at 0.1 87.5 us, here 91.1; 32768 x 8192 at 0.3 615 and 642) and has 1.6e-7 ... 6.3e-7.
//   * Where a slice ends in a row is found on the way (the first column of the row's next pairs that lies past the slice), so
//     nothing is needed beforehand. Columns that do not ascend are stopped at: what is left of such a row after the last
//     slice is gathered from memory, in order.
//   * The rows of a workgroup are sorted by length and dealt to the waves in quads, so that the four rows a wave works on are
//     about equally long and the four SIMDs have about the same to do.
// Measured (three operand sets in turn): 8192 x 8192, N = 128, density 0.1 119 -> 91 us; 32768 x 8192, density 0.3 1587 -> 642 us;
// 2048 x 512, N = 392, 102 nonzeros per row 14.9 -> 12.3 us (more at spmm_resident_choose). What bounds it (counters, 32768 x 8192
// at 0.3): an LDS read of a wave (four nonzeros x 64 columns) comes every 8.7 clocks of a compute unit, of which the LDS is
// busy 4.1 (no bank conflicts) and the vector units 6.1 (six instructions, 4 clocks on one of four SIMDs); in the row-block
// kernels the same four nonzeros take 22 clocks. At 0.1 a third of the lanes in a slice's last chunk hold no pair and the
// vector units are busy 46 % of the time, the LDS 33 %: what is left is the start and the barrier of each slice.
// The reference has no counterpart (SPMM/spmmesimd2.hpp:63-147 gathers every row of B from memory).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <utility>

#include "common.hpp"
#include "launch.hpp"
#include "resident_walk.hpp"

namespace dlspm {

constexpr int kResidentWaves = 16, kResidentThreads = kResidentWaves * 64;
constexpr int kResidentRows = 4 * kResidentWaves;  // rows of a workgroup and RR
constexpr int kResidentTile = 64;                  // columns of B
constexpr int kTileRowBytes = kResidentTile * (int)sizeof(float);

template <int LANE> __device__ __forceinline__ int row_bcast(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, 0x150 + LANE, 0xF, 0xF, true);
}

// A chunk's sum of a row, four columns: CHAINS sequential ones, pair i in chain i mod CHAINS.
template <int CHAINS> struct ChunkSum { float4 chain[CHAINS]; };

// sum += a[i] of lane LANE of the DPP row * b[i], i = 0 ... 3 (lane 0: the chains begin with their products). One block of
// instructions, so that nothing can come between its waits and its reads: a DPP operand may be read two wait states after
// a vector instruction wrote its register (the CDNA3 instruction set's table of manually inserted wait states: VALU writes
// VGPR, VALU DPP reads that VGPR: 2), and the compiler, which inserts such waits for instructions of its own, does not look
// into the block.
template <int LANE, int CHAINS> __device__ __forceinline__ void fmac_lane(ChunkSum<CHAINS>& sum, const float* a, const float4* b)
{
#define DLSPM_DPP(op, c, a, b, xyzw) op " %[" c xyzw "], %[" a "], %[" b xyzw "] row_newbcast:%[lane] row_mask:0xf bank_mask:0xf\n\t"
#define DLSPM_DPP4(op, c, a, b) DLSPM_DPP(op, c, a, b, "x") DLSPM_DPP(op, c, a, b, "y") DLSPM_DPP(op, c, a, b, "z") DLSPM_DPP(op, c, a, b, "w")
#define DLSPM_OPERANDS(c, name, v) [name##x] c(v.x), [name##y] c(v.y), [name##z] c(v.z), [name##w] c(v.w)
#define DLSPM_IN                                                                                                                    \
    [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), DLSPM_OPERANDS("v", b0, b[0]), DLSPM_OPERANDS("v", b1, b[1]), \
        DLSPM_OPERANDS("v", b2, b[2]), DLSPM_OPERANDS("v", b3, b[3]), [lane] "n"(LANE)
    static_assert(kLanePairs == 4 && (CHAINS == 2 || CHAINS == 4), "the blocks are written for four pairs");
    if constexpr (CHAINS == 2) {
        if constexpr (LANE == 0)
            asm("s_nop 1\n\t" DLSPM_DPP4("v_mul_f32_dpp", "c0", "a0", "b0") DLSPM_DPP4("v_mul_f32_dpp", "c1", "a1", "b1")
                    DLSPM_DPP4("v_fmac_f32_dpp", "c0", "a2", "b2") DLSPM_DPP4("v_fmac_f32_dpp", "c1", "a3", "b3")
                : DLSPM_OPERANDS("=&v", c0, sum.chain[0]), DLSPM_OPERANDS("=&v", c1, sum.chain[1])
                : DLSPM_IN);
        else
            asm("s_nop 1\n\t" DLSPM_DPP4("v_fmac_f32_dpp", "c0", "a0", "b0") DLSPM_DPP4("v_fmac_f32_dpp", "c1", "a1", "b1")
                    DLSPM_DPP4("v_fmac_f32_dpp", "c0", "a2", "b2") DLSPM_DPP4("v_fmac_f32_dpp", "c1", "a3", "b3")
                : DLSPM_OPERANDS("+v", c0, sum.chain[0]), DLSPM_OPERANDS("+v", c1, sum.chain[1])
                : DLSPM_IN);
    } else {
        if constexpr (LANE == 0)
            asm("s_nop 1\n\t" DLSPM_DPP4("v_mul_f32_dpp", "c0", "a0", "b0") DLSPM_DPP4("v_mul_f32_dpp", "c1", "a1", "b1")
                    DLSPM_DPP4("v_mul_f32_dpp", "c2", "a2", "b2") DLSPM_DPP4("v_mul_f32_dpp", "c3", "a3", "b3")
                : DLSPM_OPERANDS("=&v", c0, sum.chain[0]), DLSPM_OPERANDS("=&v", c1, sum.chain[1]),
                  DLSPM_OPERANDS("=&v", c2, sum.chain[2]), DLSPM_OPERANDS("=&v", c3, sum.chain[3])
                : DLSPM_IN);
        else
            asm("s_nop 1\n\t" DLSPM_DPP4("v_fmac_f32_dpp", "c0", "a0", "b0") DLSPM_DPP4("v_fmac_f32_dpp", "c1", "a1", "b1")
                    DLSPM_DPP4("v_fmac_f32_dpp", "c2", "a2", "b2") DLSPM_DPP4("v_fmac_f32_dpp", "c3", "a3", "b3")
                : DLSPM_OPERANDS("+v", c0, sum.chain[0]), DLSPM_OPERANDS("+v", c1, sum.chain[1]),
                  DLSPM_OPERANDS("+v", c2, sum.chain[2]), DLSPM_OPERANDS("+v", c3, sum.chain[3])
                : DLSPM_IN);
    }
#undef DLSPM_DPP
#undef DLSPM_DPP4
#undef DLSPM_OPERANDS
#undef DLSPM_IN
}

// The row's sum so far, in 64 bits: what the chunks' sums add up to has no rounding of its own.
struct RowSum {
    double x = 0.0, y = 0.0, z = 0.0, w = 0.0;
    template <int CHAINS> __device__ __forceinline__ void add(const ChunkSum<CHAINS>& s)
    {
        auto plus = [](float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); };
        float4 c = plus(s.chain[0], s.chain[1]);
        if constexpr (CHAINS == 4) c = plus(c, plus(s.chain[2], s.chain[3]));
        x += c.x;
        y += c.y;
        z += c.z;
        w += c.w;
    }
};

// The pairs of lanes LANE0 .. LANE0 + LANES - 1 of every group, in order: `at` = byte offset of each pair's row in `tiles`
template <int LANE0, int CHAINS, int... L>
__device__ __forceinline__ void resident_steps(const char* tiles, const int* at, int lane_bytes, const float* a, ChunkSum<CHAINS>& sum,
                                               std::integer_sequence<int, L...>)
{
    float4 b[sizeof...(L)][kLanePairs];
    auto load = [&](auto lane, int i) {
        constexpr int kLane = decltype(lane)::value;
        b[kLane][i] = *reinterpret_cast<const float4*>(tiles + (row_bcast<LANE0 + kLane>(at[i]) + lane_bytes));
    };
    ((load(std::integral_constant<int, L>{}, 0), load(std::integral_constant<int, L>{}, 1), load(std::integral_constant<int, L>{}, 2),
      load(std::integral_constant<int, L>{}, 3)), ...);
    (fmac_lane<LANE0 + L>(sum, a, b[L]), ...);
}
// ... of all sixteen lanes, FLIGHT lanes' pairs in flight at a time
template <int FLIGHT, int CHAINS, int... L>
__device__ __forceinline__ void resident_full_chunk(const char* tiles, const int* at, int lane_bytes, const float* a, ChunkSum<CHAINS>& sum,
                                                    std::integer_sequence<int, L...>)
{
    (resident_steps<FLIGHT * L>(tiles, at, lane_bytes, a, sum, std::make_integer_sequence<int, FLIGHT>{}), ...);
}
// ... of the lanes of which some group has pairs: a prefix, one bit per lane in `lanes`
template <int L, int CHAINS>
__device__ __forceinline__ bool resident_lane(const char* tiles, const int* at, int lane_bytes, const float* a, ChunkSum<CHAINS>& sum, unsigned lanes)
{
    if ((lanes >> L & 1) == 0) return false;
    resident_steps<L>(tiles, at, lane_bytes, a, sum, std::make_integer_sequence<int, 1>{});
    return true;
}
template <int CHAINS, int... L>
__device__ __forceinline__ void resident_part_chunk(const char* tiles, const int* at, int lane_bytes, const float* a, ChunkSum<CHAINS>& sum,
                                                    unsigned lanes, std::integer_sequence<int, L...>)
{
    (void)(resident_lane<L>(tiles, at, lane_bytes, a, sum, lanes) && ...);
}

// What is left of a wave's four rows, sixteen lanes each, whose columns do not ascend: from memory, in CSR order, in 64 bits. Sixteen
// pairs of a row at a time and eight of their rows of B on their way together (16384 x 8192 at density 0.3, N = 128, all rows shuffled: 2962
// -> 1149 us; one nonzero after the other before). With selects: what is behind a branch here makes the compiler order the loop over the
// slices anew.
template <int... L>
__device__ __forceinline__ void gather_rest(int p, int end, int l, int N, const int* __restrict__ col_indices, const float* __restrict__ values,
                                            const float* __restrict__ B, RowSum& sum, std::integer_sequence<int, L...>)
{
    auto pair = [&](int j) { return max(min(j + l, end - 1), 0); };
    int column = col_indices[pair(p)];
    float value = values[pair(p)];
    for (; __ballot(p < end) != 0; p += 16) {
        const int c = column;
        const float a = value;
        column = col_indices[pair(p + 16)];
        value = values[pair(p + 16)];
        auto some = [&](auto first) {  // eight of the sixteen
            constexpr int kFirst = decltype(first)::value;
            const Vec<4> b[] = {Vec<4>::gload(B + (size_t)row_bcast<kFirst + L>(c) * N)...};
            auto add = [&](int i, float v) {
                const bool in = p + kFirst + i < end;
                sum.x = in ? fma((double)v, (double)b[i].v.x, sum.x) : sum.x;
                sum.y = in ? fma((double)v, (double)b[i].v.y, sum.y) : sum.y;
                sum.z = in ? fma((double)v, (double)b[i].v.z, sum.z) : sum.z;
                sum.w = in ? fma((double)v, (double)b[i].v.w, sum.w) : sum.w;
            };
            (add(L, __int_as_float(row_bcast<kFirst + L>(__float_as_int(a)))), ...);
        };
        some(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);  // (eight rows of B take the registers there are)
        some(std::integral_constant<int, 8>{});
    }
}

// QC: chunks of 64 pairs of a row that are loaded ahead (a slice's share of a row is to fit them: what exceeds it is loaded
// when it is needed, with nothing to hide the latency behind). CHAINS: see ChunkSum.
template <int RR, int QC, int CHAINS>
__global__ __launch_bounds__(kResidentThreads) void spmm_resident_kernel(
    int M, int K, int N, int nnz, int slice, int col_tiles, int tiles_per_xcd, int streaming, const int* __restrict__ row_offsets,
    const int* __restrict__ col_indices, const float* __restrict__ values, const float* __restrict__ B, float* __restrict__ C)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    constexpr int kRows = kResidentRows * RR, kFlight = RR <= 2 ? 2 : 1;
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
    static_assert(kResidentFetchRows * 16 == kResidentThreads, "a pass of the workgroup");
    constexpr int kPasses = (kResidentMaxSlice + kResidentFetchRows - 1) / kResidentFetchRows;
    // in phases, one after each of the wave's quads, so that few registers hold what is on its way
    constexpr int kPhase = RR == 1 ? kPasses : RR == 2 ? 3 : 2, kPhases = (kPasses + kPhase - 1) / kPhase;
    static_assert(kPhases <= RR, "every phase has a quad to hide behind");
    struct Fetched { u4 pass[kPhase]; };
    // (resident_fetch_row with the row of the slice and pass as the scalar offset: no address lies outside B, whatever a buffer's range
    // check covers)
    const unsigned row_bytes = (unsigned)N * 4u, fetch_at = (unsigned)(t >> 4) * row_bytes + (unsigned)col * 4u;
    auto passes = [&](int phase, auto&& each) {
#pragma unroll
        for (int q = phase * kPhase; q < min((phase + 1) * kPhase, kPasses); ++q)
            if (resident_fetches(q, w * kWave, slice)) each(q, q - phase * kPhase);
    };
    auto fetch = [&](Fetched& f, int s, int phase) {
        passes(phase, [&](int q, int i) {
            f.pass[i] = __builtin_amdgcn_raw_buffer_load_b128(B_buffer, fetch_at, (unsigned)resident_fetch_row(s, q, 0, slice, K) * row_bytes, 0);
        });
    };
    auto fetch_first = [&](Fetched& f, int phase) {
        if (slice <= K) return fetch(f, 0, phase);
        passes(phase, [&](int q, int i) {  // (the only slice)
            f.pass[i] = __builtin_amdgcn_raw_buffer_load_b128(B_buffer, (unsigned)resident_fetch_row(0, q, t, slice, K) * row_bytes + (unsigned)col * 4u, 0, 0);
        });
    };
    auto put = [&](const Fetched& f, int buffer, int phase) {
        passes(phase, [&](int q, int i) {
            *reinterpret_cast<u4*>(tiles + buffer * buffer_bytes + (q * kResidentFetchRows + (t >> 4)) * kTileRowBytes + lane_bytes) = f.pass[i];
        });
    };
    Fetched fetched;
    fetch_first(fetched, 0);

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
    RowSum total[RR];
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
        // quads of four rows, longest first, dealt to the four SIMDs (wave w runs on SIMD w mod 4) forwards and backwards in turn
        const int quad = rr * kResidentWaves + w, turn = quad >> 2;
        const int dealt = (turn & 1) ? (turn << 2) + 3 - (quad & 3) : quad;
        row[rr] = order[dealt * 4 + g];
        const bool exists = row[rr] < M;
        p[rr] = exists ? row_offsets[row[rr]] : 0;  // (the group's position; each lane's first pair is 4 l behind it)
        end[rr] = exists ? row_offsets[row[rr] + 1] : 0;
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
    put(fetched, 0, 0);
#pragma unroll
    for (int phase = 1; phase < kPhases; ++phase) {
        fetch_first(fetched, phase);
        put(fetched, 0, phase);
    }
    if (t < 16) *reinterpret_cast<float4*>(tiles + zeros + t * 16) = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();

    unsigned stuck = 0;  // bit rr: the row's columns do not ascend; the rest of it is done at the end
    const int slices = (K + slice - 1) / slice;
    for (int s = 0; s < slices; ++s) {
        if (s + 1 < slices) fetch(fetched, s + 1, 0);
        const int k0 = resident_slice_start(s, slice, K), base = (s & 1) * buffer_bytes;
#pragma unroll
        for (int rr = 0; rr < RR; ++rr) {
            bool more = (stuck >> rr & 1) == 0;
            ChunkSum<CHAINS> sum;  // (declared inside the branches that fill it, it costs 40 registers' worth of spills)
            unsigned long long stopped = 0;  // lanes of the groups that have met the end of the slice (or of their row)
            while (more) {
                more = false;
                bool next = true;
                const int left0 = end[rr] - p[rr] - kLanePairs * l;
#pragma unroll
                for (int q = 0; q < QC; ++q) {
                    if (!next) continue;
                    int at[kLanePairs];
                    unsigned long long in[kLanePairs];    // which lanes' pairs lie in this slice
                    const int left = left0 - q * kChunk;  // pairs of the row from the lane's first on
#pragma unroll
                    for (int i = 0; i < kLanePairs; ++i) {
                        const int k = c[rr][q][i] - k0;
                        in[i] = __ballot((unsigned)k < (unsigned)slice) & __ballot(i < left);
                        at[i] = k * kTileRowBytes + base;
                    }
                    unsigned lanes = 0;
                    const ResidentStep step = resident_step(in, stopped, lanes);
                    if (step == kResidentFull) {
                        resident_full_chunk<kFlight>(tiles, at, lane_bytes, a[rr][q], sum, std::make_integer_sequence<int, 16 / kFlight>{});
                        total[rr].add(sum);
                        p[rr] += kChunk;
                        if (q == QC - 1) more = true;
                        continue;
                    }
                    if (step == kResidentDisorder) {
                        stuck |= 1u << rr;
                        next = false;
                        continue;
                    }
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
                    if (lanes != 0) {
                        resident_part_chunk(tiles, at, lane_bytes, av, sum, lanes, std::make_integer_sequence<int, 16>{});
                        total[rr].add(sum);
                    }
                    next = resident_goes_on(in);
                    if (q == QC - 1) more = next;
                }
                load_pairs(rr);
            }
            if (rr < kPhases && s + 1 < slices) {
                put(fetched, (s + 1) & 1, rr);
                if (rr + 1 < kPhases) fetch(fetched, s + 1, rr + 1);
            }
        }
        __syncthreads();
    }

    // (the lane's place once more: kept through the loop, it would be spilled)
    const int l_end = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) & 15, col_end = min(ct * kResidentTile + l_end * 4, N - 4);
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
        RowSum& sum = total[rr];
        // (Where nothing is left. A branch that is not expected to be taken keeps the gathering out of the way of the kernel's end, which
        // the short calls notice (2048 x 2048 at 0.1, N = 392 12.5 -> 12.3 us); at two chunks ahead it also makes the compiler order the loop
        // above for fewer registers, 2 ... 7 % slower (27241 x 5786 at 0.2, N = 128, lognormal rows 417 -> 443), and there it stays away.)
        if (QC == 2 || __builtin_expect(__ballot(p[rr] < end[rr]) != 0, 0))
            gather_rest(p[rr], end[rr], l_end, N, col_indices, values, B + col_end, sum, std::make_integer_sequence<int, 8>{});
        if (row[rr] >= M) continue;
        const Vec<4> out{make_float4((float)sum.x, (float)sum.y, (float)sum.z, (float)sum.w)};
        if (ct * kResidentTile + l_end * 4 < N) out.gstore(C + (size_t)row[rr] * N + col_end, streaming != 0);
    }
}

template <int RR, int QC, int CHAINS> static hipError_t launch_one(const SpmmArgs& x, const ResidentPlan& plan, hipStream_t stream)
{
    const int col_tiles = (int)ceil_div(x.N, kResidentTile);
    const long long row_blocks = ceil_div(x.M, kResidentRows * RR);
    const bool tiles_per_xcd = col_tiles > 1 && row_blocks >= 64;  // (rounding few row blocks up to eight would leave XCDs idle)
    const long long blocks = (tiles_per_xcd ? (row_blocks + 7) / 8 * 8 : row_blocks) * col_tiles;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const size_t lds = (size_t)(2 * plan.slice + 1) * kTileRowBytes;
    const auto kernel = &spmm_resident_kernel<RR, QC, CHAINS>;
    // (once per kernel and device: the attribute belongs to the function as loaded on one device)
    static std::atomic<unsigned long long> allowed[2];
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (device & 63);
    if (device >= 128 || (allowed[device >> 6].load(std::memory_order_relaxed) & bit) == 0) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (2 * kResidentMaxSlice + 1) * kTileRowBytes);
        if (e != hipSuccess) return e;
        if (device < 128) allowed[device >> 6].fetch_or(bit, std::memory_order_relaxed);
    }
    const int stream_rule = tuning().stream_results;
    const bool streaming = stream_rule < 0 ? (long long)x.M * x.N >= 1024 * 1024 : stream_rule != 0;  // (as dense_rows_window)
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kResidentThreads), lds, stream, x.M, x.K, x.N, x.nnz, plan.slice, col_tiles,
                       tiles_per_xcd ? 1 : 0, streaming ? 1 : 0, x.row_offsets, x.col_indices, x.values, x.B, x.C);
    return hipGetLastError();
}

// The resident schedule for these sizes, or rr == 0: where its estimated time is below 0.9 of the row-block kernels'.
// Both estimates (us) are fits to three operand sets worked on in turn, M = 128 ... 32768, K = 512 ... 8192, N = 32 ... 12544,
// density 0.05 ... 0.5, Bernoulli rows (122 cases; row-block estimate / measured 0.96 in the geometric mean, 0.74 ... 1.17 in nine of
// ten; resident, 416 timings, 0.99 and 0.88 ... 1.14). Over these cases and as many with lognormal rows the schedule was
// never chosen where it is slower; it takes 0.50 ... 0.60 of the row-block kernels' time where chosen:
//   row-block   2 + nnz width x 1.55e-7 (8192 x 8192, N = 128, density 0.1 / 0.2 / 0.3: 130 ... 138 / 292 / 437);
//   resident    rounds of one workgroup per compute unit x (3.6 + 1.2 rr + 0.55 slices + K / 304 rr (1.0 + 15.6 density)): the
//               start, what a slice costs whatever is in it (its barrier, the ends of its rows), and its steps (the same
//               cases at rr = 1: 99 / 151 / 188; 32768 x 8192 at rr = 2: 306 / 521 / 649, row-block 579 / 1076 / 1586).
// Rows per workgroup: as many as keep the compute units in step. The four rows that a wave works on wait for the longest
// of them and all waves of a workgroup for the slowest, so uneven rows take longer, the more the fewer rows a workgroup has
// and the shorter they are (lognormal rows, sigma 0.6, against Bernoulli rows at density 0.1 / 0.2 / 0.3 / 0.5: rr = 1 1.6 / 1.5 / 1.3 /
// 1.0 of the time in the mean and up to 2.4 / 1.7 / 1.3 / 1.0, rr = 2 1.4 / 1.1 / 1.0 / 1.0 and up to 2.0 / 1.2 / 1.1 / 1.0): calls with a
// row plan, a cut plan or DLSPM_HINT_ROWS_SKEWED count the most of that, calls that say nothing about their rows count it
// against the 1.2 that such rows cost the row-block kernels, and calls with the even-rows hint not at all.
ResidentPlan spmm_resident_choose(const DeviceInfo& dev, int M, int K, int N, int nnz, bool rows_even, bool uneven_rows)
{
    const Tuning& t = tuning();
    ResidentPlan none{0, 0, 0, 0.0};
    if (!rule_on(kRuleResidentSlices) || N < 4 || M <= 0 || K <= 0 || nnz <= 0 || nnz >= (1 << 29) || !dense_fits_buffer(K, N)) return none;
    // (a schedule that was asked for by name)
    if (t.split_w > 0 || t.flat >= 0 || t.slices >= 0 || t.tile_major >= 0 || t.tile_width > 0 || t.plan_order > 0 || t.xcd_contiguous) return none;
    const double density = (double)nnz / ((double)M * K);
    const long long slices = ceil_div(K, kResidentMaxSlice), col_tiles = ceil_div(N, kResidentTile);
    const int slice = resident_slice_rows(K);
    // two chunks of 64 pairs ahead where a slice's share of a row exceeds one: mean and two deviations of a Bernoulli row
    const double share = density * slice;
    const int chunks = share + 2.0 * std::sqrt(share * (1.0 - density)) > (double)kChunk ? 2 : 1;
    // what a dense row costs the row-block kernels: half of the lanes that its layout leaves idle count
    const double width = N <= 32 ? 32 : N <= 64 ? 64 : N <= 128 ? 0.5 * (N + 128) : N <= 256 ? 0.5 * (N + 256) : N;
    const double row_block_us = 2.0 + (double)nnz * width * 1.55e-7;
    none.us = row_block_us;
    ResidentPlan best = none;
    double best_us = 0.9 * row_block_us;
    for (int rr = 1; rr <= (chunks == 1 ? 4 : 3); ++rr) {
        const long long workgroups = ceil_div(M, kResidentRows * rr) * col_tiles, rounds = ceil_div(workgroups, dev.cus);
        if (8 * workgroups < 5ll * dev.cus) break;  // (the others' vector-memory paths would go unused)
        double us = (double)rounds * (3.6 + 1.2 * rr + 0.55 * (double)slices + K / 304.0 * rr * (1.0 + 15.6 * density));
        const double uneven = std::max(1.0, rr == 1 ? 1.0 + 3.5 * (0.45 - density) : 1.0 + 3.8 * (0.3 - density));
        if (uneven_rows) us *= uneven;
        else if (!rows_even) us *= std::max(1.0, uneven / (M <= 16 * dev.cus ? 1.5 : 1.15));
        if (us < best_us) {
            best_us = us;
            best = ResidentPlan{rr, chunks, slice, us};
        }
    }
    return best;
}

int resident_rows_per_workgroup(const ResidentPlan& plan) { return kResidentRows * plan.rr; }

hipError_t spmm_resident_launch(const SpmmArgs& x, const ResidentPlan& plan, hipStream_t stream)
{
    if (plan.chunks == 1) {
        if (plan.rr == 1) return launch_one<1, 1, 2>(x, plan, stream);
        if (plan.rr == 2) return launch_one<2, 1, 2>(x, plan, stream);
        if (plan.rr == 3) return launch_one<3, 1, 2>(x, plan, stream);
        if (plan.rr == 4) return launch_one<4, 1, 2>(x, plan, stream);
    } else {
        if (plan.rr == 1) return launch_one<1, 2, 4>(x, plan, stream);
        if (plan.rr == 2) return launch_one<2, 2, 4>(x, plan, stream);
        if (plan.rr == 3) return launch_one<3, 1, 4>(x, plan, stream);  // (two chunks ahead of three quads do not fit the registers)
    }
    return hipErrorInvalidValue;
}

}  // namespace dlspm
