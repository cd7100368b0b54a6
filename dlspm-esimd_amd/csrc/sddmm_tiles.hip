// SDDMM on masks dense enough that the dot products of whole tiles cost less than the sampled ones gathered one by one.
//
// What bounds the gathering kernels (sddmm.hip) is a compute unit's vector-memory path, 64 bytes per clock: every nonzero reads its
// row of rhs through it, 2 clocks at D = 32, 8 at D = 128. Here a workgroup of eight waves computes all dot products of 64 rows of
// lhs with 256 rows of rhs on the bf16 matrix cores (dense_tiles.hpp), puts them into LDS and picks the sampled ones from there:
//   * Wave w computes the tile's columns 32 w ... + 31. It reads its rows of rhs 128 bytes of a row at a time, passes them through
//     LDS so that a lane then holds one row's floats, and splits them into their parts once for all 64 rows of lhs, whose parts
//     stay in LDS while the workgroup goes through the tiles of its range of columns.
//   * Wave w samples the rows 8 w ... + 7: the row's next 128 columns are in registers, those that lie in the tile are
//     a prefix of them, and their results go to their slots. A row's position is carried from tile to tile; where a range does not
//     begin with the row it is found by a binary search. Any position is a correct one: what a row has left at the end of a range,
//     because its columns do not ascend, is computed as in sddmm.hip, and so are results that are not finite (dense_tiles.hpp).
//   * Rows whose first 64 columns do not ascend, and rows of lhs with a nonzero value below 2^-109, are left out of the tiles. A
//     workgroup that finds more than half of its rows to be such gathers all of them instead, otherwise its waves share them behind the
//     tiles (us, gathering kernels / all rows shuffled / every sixteenth, at 8192 x 8192: D = 128 at 0.2 250 / 274 / 126, D = 64 at 0.2
//     125 / 137 / 78, D = 32 at 0.3 110 / 119 / 61; while the wave of such a row finished it alone: 1565 / 307, 654 / 158, 481 / 131;
//     2048 x 2048 at 0.3, D = 128, 24 / 31 / 16, was 187 / 62).
//   * Such a value in a row of rhs is noted for the end, where results of its column that are small enough to show what its parts lost,
//     and results that are not finite, are gathered: a value of 1e-36 in every row of rhs takes the three from 104 / 66 / 56 to 133 / 92 /
//     80 us (1175 / 605 / 388 while its parts were NaN and every result of the column was computed again).
//   * Up to D = 32 two workgroups share a compute unit, one sampling while the other computes. Above, the parts of lhs take the
//     LDS of the second one, and the splits of a step of sixteen, the loads and the passage through LDS stand between the products
//     of the step before it instead.
// Measured (us, gathering kernels -> tiles): 24576 x 8192 at density 0.2, D = 32, three operand sets in turn 237 -> 163; one set, plain
// calls: 8192 x 8192, D = 32 at 0.3 115 -> 58, D = 64 at 0.2 / 0.3 131 / 194 -> 69 / 74, D = 128 at 0.1 / 0.2 / 0.3 134 / 255 / 386 -> 109 /
// 108 / 116; 30000 x 4093 at 0.2, D = 50 304 -> 139; 2048 x 2048 at 0.3, D = 128 24.7 -> 14.2. Against 64 bits the results are off by
// 3.8 / 4.3 / 4.8 / 5.2e-8 at D = 32 / 64 / 96 / 128, the gathering kernels' by 6.2 / 7.2 / 8.0 / 8.8e-8; operands of one sign 3.4 / 3.8 / 3.9 /
// 4.4e-8 and 4.1 / 4.2 / 4.3 / 4.5e-8. For the latter hi x hi has two chains of every second step above D = 32, and the last step's goes
// behind the small products: in one chain of all steps the sums grow as they go, and so do their roundings (3.4 / 5.2 / 5.7 / 6.9e-8).
// That is 1 % of the time in the mean of 17 sizes, up to 4 % at D = 65 ... 95.
// What bounds it: D = 128, the products (a wave spends 6 of the 7 us of a tile in them; 3 at the rate of products of constants, 4.5 at
// what a large bf16 product of random numbers reaches here, 1.2 ... 1.35 PFLOP/s of 2.5: the chip lowers its clocks); D = 32, the
// turns of computing (1.5 ... 2.5 us of 4 ... 5), waiting at the barrier and sampling, which two workgroups overlap only in part.
// Measured and not kept: tiles of D = 32 in turn in two buffers, half of the waves sampling while the others compute (175 against
// 152); sixteen lanes with four columns each per row (equal); ordinary stores (+20 %); columns touched two tiles ahead (+12 %).
// The reference has no counterpart (SDDMM/sddmm-esimd-fromfile.hpp:59-131 gathers every row).
#include <algorithm>

#include "dense_tiles.hpp"
#include "launch.hpp"
#include "sampled_out.hpp"

namespace dlspm {

constexpr int kTileWaves = 8, kTileRows = 64, kTileCols = 32 * kTileWaves;
constexpr int kRowsPerWave = kTileRows / kTileWaves;
constexpr int kAhead = 2;  // columns of a row loaded ahead, times 64
constexpr int kFewWords = 32 * kTileWaves;

// Element (row, col) of a tile lies at row * kTileCols + (col ^ turned(row)): eight lanes that write four columns each of eight
// rows fall on all banks
__device__ __forceinline__ constexpr int turned(int row) { return (row & 7) << 2; }
static_assert(kRowsPerWave == 8, "row i of a wave is turned by turned(i)");

// the first of the columns [p, e) that is not below `column` (where the columns do not ascend: some position, and none before it for
// a higher column, so that the ranges of a row neither overlap nor leave anything out)
__device__ __forceinline__ int first_not_below(const int* __restrict__ col_indices, int p, int e, int column)
{
    while (p < e) {
        const int middle = p + (e - p) / 2;
        if (col_indices[middle] < column) p = middle + 1;
        else e = middle;
    }
    return p;
}

// (in front of the scores: an LDS access holds an offset of 64 KiB, and behind them every part would take an address register of its own)
template <int PARTS> struct LhsParts { bf16x8 lhs_parts[PARTS][kWave]; };
template <int N> struct Stage { float stage[N][32 * 32]; };
template <> struct Stage<0> {};
template <int STAGES, int PARTS> struct __attribute__((aligned(16))) TileLds : LhsParts<PARTS>, Stage<STAGES> {
    float scores[kTileRows * kTileCols];
    int first[kTileRows], end[kTileRows], done[kTileRows];  // nonzeros of the rows in the range of columns, and how far the tiles got
    unsigned long long apart[kTileWaves];  // rows that each wave has found to be none for the tiles
    unsigned few[kFewWords];               // columns of the range, modulo 32 kFewWords, whose row of rhs has a value below 2^-109
    int any_few;
};

struct ScaledOut {
    float* __restrict__ at;
    float scale;
    __device__ __forceinline__ void store(int j, float v) const { at[j] = v * scale; }
};

// SEGMENTS: of 32 floats, of a row of lhs and rhs. FULL: D == 32 SEGMENTS
template <int SEGMENTS, bool FULL, bool STREAM>
__global__ __launch_bounds__(kTileWaves * 64) __attribute__((amdgpu_waves_per_eu(SEGMENTS == 1 ? 4 : 2, SEGMENTS == 1 ? 4 : 2))) void sddmm_tiles_kernel(
    int M, int K, int D, int nnz, int row_blocks, int range_tiles, const int* __restrict__ row_offsets, const int* __restrict__ col_indices,
    const float* __restrict__ lhs, const float* __restrict__ rhs, float scale, float* __restrict__ out)
{
    constexpr int KS = 2 * SEGMENTS;  // steps of sixteen floats
    constexpr bool kTwoPerUnit = SEGMENTS == 1;  // workgroups per compute unit: rhs goes through the wave's own columns of the tile
    constexpr int kStagePitch = kTwoPerUnit ? kTileCols : 32;
    __shared__ TileLds<kTwoPerUnit ? 0 : kTileWaves, 2 * KS * 3> lds;

    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), l = lane & 31, h = lane >> 5;
    const int range = (int)(blockIdx.x / (unsigned)row_blocks), row0 = ((int)blockIdx.x - range * row_blocks) * kTileRows;
    const int first_column = range * range_tiles * kTileCols, columns_end = min(K, first_column + range_tiles * kTileCols);
    const int tiles = (columns_end - first_column + kTileCols - 1) / kTileCols;

    // ---- a segment of the wave's 32 rows of rhs: eight lanes read 128 bytes of a row; from LDS every lane then takes sixteen floats
    // of row l, in two steps of eight
    Vec<4> raw[4];
    // (rows behind the last: the buffer's range check, with the whole offset in the vector part, makes them zeros)
    const __amdgpu_buffer_rsrc_t rhs_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rhs), 0, (int)((unsigned)K * (unsigned)D * 4u), 0x00020000);
    const unsigned row_bytes = (unsigned)D * 4u, rhs_from = (unsigned)(first_column + 32 * w + (lane >> 3)) * row_bytes;
    auto load_rhs = [&](int tile, int s) {
        const int d = 32 * s + 4 * (lane & 7), last = D - 4;
        const bool partial = !FULL && s == SEGMENTS - 1;
        const unsigned from = rhs_from + (unsigned)(min(tile, tiles - 1) * kTileCols) * row_bytes + (unsigned)(partial ? min(d, last) : d) * 4u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            raw[i] = Vec<4>::bload(rhs_buffer, from + (unsigned)(8 * i) * row_bytes, 0);
            if (partial) raw[i].zero_first(d - last);
        }
    };
    float* stage;
    if constexpr (kTwoPerUnit) stage = lds.scores + 32 * w;
    else stage = lds.stage[w];
    float* const stage_to = stage + (lane >> 3) * kStagePitch + (((lane & 7) ^ (lane >> 3)) << 2);
    auto put = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[i].store(stage_to + i * 8 * kStagePitch);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    auto get = [&](float* x, int step) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const Vec<4> v = Vec<4>::load(stage + l * kStagePitch + (((4 * step + 2 * h + q) ^ (l & 7)) << 2));
            x[4 * q] = v.v.x, x[4 * q + 1] = v.v.y, x[4 * q + 2] = v.v.z, x[4 * q + 3] = v.v.w;
        }
    };
    load_rhs(0, 0);

    // ---- the rows' nonzeros in the range of columns
    const __amdgpu_buffer_rsrc_t columns = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(col_indices), 0, nnz * 4, 0x00020000);
    const int offsets = row_offsets[min(row0 + w * kRowsPerWave + min(lane, kRowsPerWave), M)];  // of the wave's rows
    const int searched = min(row0 + (t & (kTileRows - 1)), M), from = row_offsets[searched], to = row_offsets[min(searched + 1, M)];
    int leading[kRowsPerWave];
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i)
        leading[i] = __builtin_amdgcn_raw_buffer_load_b32(columns, (unsigned)(__builtin_amdgcn_readlane(offsets, i) + lane) * 4u, 0, 0);
    if (t < 2 * kTileRows) {
        const int column = t < kTileRows ? first_column : columns_end;
        (t < kTileRows ? lds.first : lds.end)[t & (kTileRows - 1)] = column == 0 ? from : column >= K ? to : first_not_below(col_indices, from, to, column);
    }
    // ---- the parts of lhs: lane l holds row l % 32, floats 16 ks + 8 (l / 32) ... + 7
    unsigned long long apart = 0;
    for (int i = w; i < 2 * KS; i += kTileWaves) {
        const float* from = lhs + (size_t)min(row0 + 32 * (i / KS) + l, M - 1) * D;
        float x[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int d = 16 * (i % KS) + 8 * h + 4 * q;
            const Vec<4> v = FULL ? Vec<4>::gload(from + d) : d < D ? Vec<4>::gload_clip(from, d, D) : Vec<4>::zero();
            x[4 * q] = v.v.x, x[4 * q + 1] = v.v.y, x[4 * q + 2] = v.v.z, x[4 * q + 3] = v.v.w;
        }
        unsigned long long few = 0;
        const Parts q = split_parts(x, few);
        apart |= (unsigned long long)((unsigned)few | (unsigned)(few >> 32)) << 32 * (i / KS);
        lds.lhs_parts[3 * i + 0][lane] = q.hi;
        lds.lhs_parts[3 * i + 1][lane] = q.mid;
        lds.lhs_parts[3 * i + 2][lane] = q.lo;
    }
    auto lhs_at = [&](int rt, int ks) {
        const int i = 3 * (rt * KS + ks);
        return Parts{lds.lhs_parts[i][lane], lds.lhs_parts[i + 1][lane], lds.lhs_parts[i + 2][lane]};
    };
    // Rows that are left out of the tiles: those whose columns do not ascend, told by the first 64, and rows of lhs with a value below
    // 2^-109. Every range of columns comes to the same ones; they share their nonzeros evenly.
    int unordered = 0;
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) {
        const int length = __builtin_amdgcn_readlane(offsets, i + 1) - __builtin_amdgcn_readlane(offsets, i);
        const int next = __builtin_amdgcn_update_dpp(0, leading[i], 0x130, 0xf, 0xf, true);  // wave_shl:1
        if (__ballot(lane < min(length, kWave) - 1 && leading[i] > next) != 0) unordered |= 1 << i;
    }
    if (lane == 0) lds.apart[w] = apart | (unsigned long long)unordered << w * kRowsPerWave;
    if (t < kFewWords) lds.few[t] = 0;
    if (t == 0) lds.any_few = 0;
    __syncthreads();
    const unsigned long long found = lds.apart[lane & (kTileWaves - 1)];
    apart = 0;
    if (__ballot(found != 0) != 0) {
#pragma unroll
        for (int i = 0; i < kTileWaves; ++i)
            apart |= (unsigned)__builtin_amdgcn_readlane((int)found, i) | (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(found >> 32), i) << 32;
        const int length = lane_get(offsets, lane + 1) - offsets, row = w * kRowsPerWave + (lane & (kRowsPerWave - 1));
        if (lane < kRowsPerWave && (apart >> row & 1) != 0) {
            const int ranges = (int)(gridDim.x / (unsigned)row_blocks), share = (length - 1) / ranges + 1;
            lds.first[row] = offsets + min(share * range, length);
            lds.end[row] = offsets + min(share * (range + 1), length);
        }
    }
    const unsigned mine_apart = (unsigned)(apart >> w * kRowsPerWave) & ((1u << kRowsPerWave) - 1);
    const int my_first = lds.first[w * kRowsPerWave + (lane & (kRowsPerWave - 1))], my_end = lds.end[w * kRowsPerWave + (lane & (kRowsPerWave - 1))];
    int p[kRowsPerWave], e[kRowsPerWave];
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) {
        p[i] = __builtin_amdgcn_readlane(my_first, i);
        e[i] = mine_apart >> i & 1 ? p[i] : __builtin_amdgcn_readlane(my_end, i);
    }
    const bool gather = __builtin_popcountll(apart) > kTileRows / 2;  // (uniform) all rows are gathered: their tiles would cost more than they save
    int c[kRowsPerWave][kAhead];
    auto load_columns = [&](int i) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q) c[i][q] = __builtin_amdgcn_raw_buffer_load_b32(columns, (unsigned)(p[i] + lane) * 4u + q * kWave * 4, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) load_columns(i);

    // ---- the wave's part of a tile: 64 rows x 32 columns
    // the products of one step with the parts q0, q1 of the lhs rows 0 ... 31, 32 ... 63, smallest first; hi x hi into `sum`, or none
    auto multiply = [&](const Parts& r, const Parts& q0, const Parts& q1, f32x16* small, f32x16* sum) {
        small[0] = mfma(r.lo, q0.hi, small[0]);
        small[1] = mfma(r.lo, q1.hi, small[1]);
        if (sum && sum != small) {
            sum[0] = mfma(r.hi, q0.hi, sum[0]);
            sum[1] = mfma(r.hi, q1.hi, sum[1]);
        }
        small[0] = mfma(r.mid, q0.mid, small[0]);
        small[1] = mfma(r.mid, q1.mid, small[1]);
        small[0] = mfma(r.hi, q0.lo, small[0]);
        small[1] = mfma(r.hi, q1.lo, small[1]);
        small[0] = mfma(r.mid, q0.hi, small[0]);
        small[1] = mfma(r.mid, q1.hi, small[1]);
        small[0] = mfma(r.hi, q0.mid, small[0]);
        small[1] = mfma(r.hi, q1.mid, small[1]);
        if (sum == small) {
            sum[0] = mfma(r.hi, q0.hi, sum[0]);
            sum[1] = mfma(r.hi, q1.hi, sum[1]);
        }
    };
    auto write_scores = [&](const f32x16* sum) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4*>(lds.scores + (32 * rt + l) * kTileCols + 32 * w + ((8 * q + 4 * h) ^ turned(l))) =
                    make_float4(sum[rt][4 * q], sum[rt][4 * q + 1], sum[rt][4 * q + 2], sum[rt][4 * q + 3]);
    };
    // the lanes whose rows of rhs have a value below 2^-109, for the end
    auto note_few = [&](int tile, unsigned long long few) {
        if (few == 0) return;
        lds.few[(tile * kTileWaves + w) % kFewWords] |= (unsigned)few | (unsigned)(few >> 32);
        lds.any_few = 1;
    };
    // D <= 32: the small products of both steps come first, in one accumulator
    auto compute_short = [&](int tile) {
        f32x16 sum[2] = {};
        __syncthreads();  // (the previous tile has been read)
        put();
        load_rhs(tile + 1, 0);
        Parts r[2];
        float x[2][8];
        unsigned long long few = 0;
        get(x[0], 0);
        get(x[1], 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            r[ks] = split_parts(x[ks], few);
            multiply(r[ks], lhs_at(0, ks), lhs_at(1, ks), sum, nullptr);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) sum[rt] = mfma(r[ks].hi, lhs_at(rt, ks).hi, sum[rt]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        write_scores(sum);
        note_few(tile, few);
    };
    // D > 32: `ready` and `of_lhs` are the parts of the step at hand, `next` the floats of the one after it. Between the products
    // stand the split of the next step, the segment after it on its way through LDS, and the loads of the one behind that
    Parts ready, of_lhs[2];
    unsigned long long few_ahead = 0;
    float next[8];
    if constexpr (!kTwoPerUnit) {
        put();
        float x[8];
        get(x, 0);
        get(next, 1);
        ready = split_parts(x, few_ahead);
        of_lhs[0] = lhs_at(0, 0), of_lhs[1] = lhs_at(1, 0);
        load_rhs(0, 1);
    }
    auto compute_long = [&](int tile) {
        f32x16 small[2] = {}, sum[2][2] = {};
        unsigned long long few = few_ahead;
        few_ahead = 0;
#pragma unroll
        for (int s = 0; s < SEGMENTS; ++s) {
            float staged[2][8];
#pragma unroll
            for (int step = 0; step < 2; ++step) {
                const int ks = 2 * s + step;
                const Parts now = ready, q0 = of_lhs[0], q1 = of_lhs[1];
                of_lhs[0] = lhs_at(0, (ks + 1) % KS), of_lhs[1] = lhs_at(1, (ks + 1) % KS);
                if (step == 0) {
                    put();
                    get(staged[0], 0);
                    get(staged[1], 1);
                    ready = split_parts(next, few);
                    load_rhs(tile + (s + 2) / SEGMENTS, (s + 2) % SEGMENTS);
                } else {
                    ready = split_parts(staged[0], s + 1 < SEGMENTS ? few : few_ahead);
#pragma unroll
                    for (int i = 0; i < 8; ++i) next[i] = staged[1][i];
                }
                multiply(now, q0, q1, small, ks == KS - 1 ? small : sum[step]);
#pragma unroll
                for (int g = 0; g < 12; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product,
                    __builtin_amdgcn_sched_group_barrier(0x300, 1, 0);  // one LDS access,
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);  // six vector instructions in its 32 clocks
                }
                __builtin_amdgcn_sched_barrier(0);  // (across steps the compiler would move loads far ahead, and spill)
            }
        }
        f32x16 scores[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) scores[rt] = (small[rt] + sum[1][rt]) + sum[0][rt];
        __syncthreads();  // (the previous tile has been read)
        write_scores(scores);
        note_few(tile, few);
    };

    // ---- the sampled ones. All reads, then all loads for the next tile, then all stores: loads and stores complete in order
    float all_finite = 0.f;  // NaN once a result is not finite
    auto sample = [&](int tile) {
        const int k0 = first_column + tile * kTileCols;
        const float* const mine = lds.scores + w * kRowsPerWave * kTileCols;
        int n[kRowsPerWave], at[kRowsPerWave];
        float v[kRowsPerWave][kAhead];
        bool full = false;
        auto leading = [&](int i, int q) {  // how many of the 64 lie in the tile, in front of the first that does not
            const unsigned long long in = __ballot((unsigned)(c[i][q] - k0) < (unsigned)kTileCols) & __ballot(lane < e[i] - p[i] - q * kWave);
            return in == ~0ull ? kWave : __builtin_ctzll(~in);
        };
        auto read = [&](int i, int q) { v[i][q] = mine[i * kTileCols + ((int)min((unsigned)(c[i][q] - k0), (unsigned)kTileCols - 1) ^ turned(i))]; };
        auto store = [&](int i, int q) {
            v[i][q] *= scale;
            all_finite = fmaf(v[i][q], 0.f, all_finite);
            if (lane + q * kWave < n[i]) {
                float* const to = out + at[i] + q * kWave;
                if constexpr (STREAM) __builtin_nontemporal_store(v[i][q], to + lane);
                else to[lane] = v[i][q];
            }
        };
#pragma unroll
        for (int i = 0; i < kRowsPerWave; ++i) {
            n[i] = leading(i, 0);
            read(i, 0);
            if (n[i] == kWave) {
                n[i] += leading(i, 1);
                read(i, 1);
            }
            full = full || n[i] == kAhead * kWave;
        }
#pragma unroll
        for (int i = 0; i < kRowsPerWave; ++i) {
            at[i] = p[i];
            p[i] += n[i];
            load_columns(i);
        }
#pragma unroll
        for (int i = 0; i < kRowsPerWave; ++i) {
            store(i, 0);
            if (n[i] >= kWave) store(i, 1);
        }
        if (!full) return;
#pragma unroll
        for (int i = 0; i < kRowsPerWave; ++i) {
            bool more = n[i] == kAhead * kWave;
            while (more) {  // (the next columns were requested just now)
                n[i] = leading(i, 0);
                read(i, 0);
                at[i] = p[i];
                p[i] += n[i];
                load_columns(i);
                store(i, 0);
                more = n[i] == kWave;
            }
        }
    };

    for (int tile = 0; tile < (gather ? 0 : tiles); ++tile) {
        if constexpr (kTwoPerUnit) compute_short(tile);
        else compute_long(tile);
        __syncthreads();
        sample(tile);
    }

    // ---- what is left: rows whose columns do not ascend, and results that are not finite
    const ScaledOut plain{out, scale};
    const int at_end = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));  // (the lane; kept through the loop, it would be spilled)
    auto gathered = [&](int row, int from, int to, int step) {
        sddmm_segment<4, 8, SEGMENTS, FULL ? kExactWidth : kMaskedBySelect, kTwoPerUnit ? 8 : 16>(from, to, D, col_indices, lhs + (size_t)(row0 + row) * D, rhs,
                                                                                                 plain, at_end, step);
    };
    int left = 0;
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) {
        const int row = w * kRowsPerWave + i;
        if (at_end == 0) lds.done[row] = (mine_apart >> i & 1) != 0 ? lds.first[row] : p[i];
        left |= e[i] - p[i];
    }
    if (apart != 0 || left != 0) {
        // all rows: whole ones, dealt to the waves of the row block's workgroups; some: each by all waves, 64 nonzeros in turn; rows
        // that are found not to ascend on the way: by their own wave
        const bool shared = apart != 0 && !gather;
        if (shared) __syncthreads();
        const unsigned ranges = gridDim.x / (unsigned)row_blocks, row = at_end;  // (a row per lane)
        const int from = gather ? row_offsets[min(row0 + at_end, M)] : lds.done[row], to = gather ? row_offsets[min(row0 + at_end + 1, M)] : lds.end[row];
        const bool mine = gather ? row % ranges == (unsigned)range && row / ranges % kTileWaves == (unsigned)w : shared || row / kRowsPerWave == (unsigned)w;
        int turn = shared ? w : 0;
        for (unsigned long long rows = __ballot(mine && from < to); rows != 0; rows &= rows - 1) {
            const int at = __builtin_ctzll(rows), p_row = __builtin_amdgcn_readlane(from, at), e_row = __builtin_amdgcn_readlane(to, at);
            const int own = p_row + turn * kWave;
            // (the lines of its columns, all at once)
            const int touched = gather ? col_indices[min(own + 32 * at_end, e_row - 1)] : 0;
            if (own < e_row) gathered(at, own, e_row, shared ? kTileWaves : 1);
            asm volatile("" : : "v"(touched));
            if (shared) turn = (turn - (e_row - p_row + kWave - 1) / kWave) & (kTileWaves - 1);
        }
        if (gather) return;
    }
    // Parts of values below 2^-109 are off by 2^-134 at most, which does not show in a result from 2^34 times what that can come to on:
    // smaller ones of such a column are gathered too.
    const bool any_few = __builtin_amdgcn_readfirstlane(lds.any_few) != 0;
    if (__ballot(!(all_finite == 0.f)) == 0 && !any_few) return;
    float bound = 0.f;
    if (any_few) {
        unsigned most = 0;
#pragma unroll 1
        for (int i = 0; i < 2 * KS; ++i) {
            const uint4 hi = __builtin_bit_cast(uint4, lds.lhs_parts[3 * i][at_end]);
            for (unsigned x : {hi.x, hi.x << 16, hi.y, hi.y << 16, hi.z, hi.z << 16, hi.w, hi.w << 16}) {
                x &= 0x7fff0000u;
                most = max(most, x < 0x7f800000u ? x : 0u);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, o));
        bound = (float)D * __uint_as_float(most) * 0x1p-99f * fabsf(scale);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // (this wave's own stores)
    constexpr int kLoads = 4;
#pragma unroll 1
    for (int row = w * kRowsPerWave; row < (w + 1) * kRowsPerWave; ++row) {
        const int done = __builtin_amdgcn_readfirstlane(lds.done[row]);
        for (int at = __builtin_amdgcn_readfirstlane(lds.first[row]); at < done; at += kLoads * kWave) {
            float x[kLoads];
            int column[kLoads];
            unsigned bad = 0;
#pragma unroll
            for (int q = 0; q < kLoads; ++q) {
                x[q] = out[min(at + q * kWave + at_end, done - 1)];
                column[q] = col_indices[min(at + q * kWave + at_end, done - 1)];
            }
#pragma unroll
            for (int q = 0; q < kLoads; ++q) {
                const unsigned of_few = lds.few[((unsigned)(column[q] - first_column) >> 5) % kFewWords] >> (column[q] - first_column & 31) & 1;
                const float least = of_few != 0 ? bound : 0.f;
                bad |= (__ballot(!(fabsf(x[q]) >= least && fabsf(x[q]) < __builtin_inff())) != 0 ? 1u : 0u) << q;
            }
            if (bad != 0) gathered(row, at + __builtin_ctz(bad) * kWave, min(at + (32 - __builtin_clz(bad)) * kWave, done), 1);
        }
    }
}

template <int SEGMENTS> static hipError_t launch_one(const SddmmArgs& x, float scale, const TilePlan& plan, hipStream_t stream)
{
    const long long row_blocks = ceil_div(x.M, kTileRows), blocks = row_blocks * plan.ranges;
    if (blocks <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const bool full = x.D == 32 * SEGMENTS, streaming = sampled_out(x).streaming != 0;
    const auto kernel = full ? streaming ? &sddmm_tiles_kernel<SEGMENTS, true, true> : &sddmm_tiles_kernel<SEGMENTS, true, false>
                             : streaming ? &sddmm_tiles_kernel<SEGMENTS, false, true> : &sddmm_tiles_kernel<SEGMENTS, false, false>;
    const int range_tiles = (int)ceil_div(ceil_div(x.K, kTileCols), plan.ranges);
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kTileWaves * 64), 0, stream, x.M, x.K, x.D, x.nnz, (int)row_blocks, range_tiles,
                       x.row_offsets, x.col_indices, x.lhs, x.rhs, scale, x.out);
    return hipGetLastError();
}

// The ranges of columns with which tiles are estimated to take the least time, and that time (sddmm_tiles_plan; ranges == 0: not for
// these sizes, or tuning overrides name a schedule), and whether SDDMM runs on them: where it is below 0.9 of the gathering kernels',
// whatever the call brings with it (so that the bits of a result depend on the sizes alone). Both estimates (us) are fits to one operand
// set worked on over and over:
//   gathering   2 + nnz (2.2 + 0.122 D) 1e-6, D rounded up to a whole access of eight lanes, a fifth more where lanes past D are masked
//               one by one (a twenty-fifth up to D = 24; 8192 x 8192 at density 0.1, D = 32 / 50 / 64 / 128 38 / 82 / 63 / 125, estimate
//               43 / 79 / 69 / 121);
//   tiles       rounds of one workgroup per compute unit (D <= 32: two) x (6, with a search 8, D <= 32 one more, + tiles of a range x
//               (D <= 32: 4.4 + 6 density, from 0.3 on 18 density, where rows have more than 64 columns in a tile; above: 0.1 + 1.42
//               segments + 5.5 density)): 8192 x 8192 at 0.3, D = 32 58 (measured 58), D = 128 at 0.1 110 (109), 24576 x 8192 at 0.3,
//               D = 128 378 (381). The tiles of a last round of two workgroups per unit that fills half of the slots, one on
//               each unit, take about 0.75 of a full one's.
// 56 masks of 500 ... 8200 rows near the line, gathering / tiles: 0.91 ... 2.7; the five below 1.1 were D = 17 ... 22 on 2000 ... 6000 rows
// (2952 x 1702 at 0.47, D = 19, lognormal rows, 14.7 / 16.6), for which the additions up to D = 32 are.
TilePlan sddmm_tiles_plan(const DeviceInfo& dev, int M, int K, int D, int nnz)
{
    TilePlan best{0, 0.0};
    const Tuning& t = tuning();
    if (t.split_w > 0 || t.flat >= 0 || t.flat_chunk > 0 || t.slices >= 0 || t.plan_order > 0 || t.xcd_contiguous) return best;  // (a schedule that was asked for by name)
    if (!rule_on(kRuleDenseGroups) || D < 17 || D > 128 || M <= 0 || K <= 0 || nnz <= 0 || nnz >= (1 << 29) || !dense_fits_buffer(K + 256ll, D)) return best;
    const double density = (double)nnz / ((double)M * K);
    const int segments = (int)ceil_div(D, 32);
    const long long row_blocks = ceil_div(M, kTileRows), tiles = ceil_div(K, kTileCols), slots = (segments == 1 ? 2ll : 1ll) * dev.cus;
    const double tile_us = segments == 1 ? 4.4 + 6.0 * density + 12.0 * std::max(0.0, density - 0.3) : 0.1 + 1.42 * segments + 5.5 * density;
    for (long long wanted = 1; wanted <= tiles && wanted <= 64; ++wanted) {
        const long long per = ceil_div(tiles, wanted), ranges = ceil_div(tiles, per), units = row_blocks * ranges;
        double rounds = (double)(units / slots);
        const double last = (double)(units % slots) / (double)slots;
        if (last > 0.0) rounds += segments > 1 ? 1.0 : 0.75 + 0.5 * std::max(0.0, last - 0.5);
        const double start_us = (ranges > 1 ? 8.0 : 6.0) + (segments == 1 ? 1.0 : 0.0);
        const double us = (double)ceil_div(units, slots) * start_us + rounds * (double)per * tile_us;
        if (best.ranges == 0 || us < best.us) best = TilePlan{(int)ranges, us};
    }
    return best;
}
TilePlan sddmm_tiles_choose(const DeviceInfo& dev, int M, int K, int D, int nnz)
{
    const TilePlan best = sddmm_tiles_plan(dev, M, K, D, nnz);
    const double gathered = 32.0 * (double)ceil_div(D, 32) * (D % 4 == 0 ? 1.0 : D <= 24 ? 1.04 : 1.2);
    return rule_on(kRuleSddmmTiles) && best.us < 0.9 * (2.0 + (double)nnz * (2.2 + 0.122 * gathered) * 1e-6) ? best : TilePlan{0, 0.0};
}

void sddmm_tile_shape(int* rows, int* columns)
{
    *rows = kTileRows;
    *columns = kTileCols;
}

hipError_t sddmm_tiles_launch(const SddmmArgs& x, float scale, const TilePlan& plan, hipStream_t stream)
{
    const int segments = (int)ceil_div(x.D, 32);
    if (segments == 1) return launch_one<1>(x, scale, plan, stream);
    if (segments == 2) return launch_one<2>(x, scale, plan, stream);
    if (segments == 3) return launch_one<3>(x, scale, plan, stream);
    if (segments == 4) return launch_one<4>(x, scale, plan, stream);
    return hipErrorInvalidValue;
}

}  // namespace dlspm
