// SpMM on matrices dense enough that the products of whole tiles cost less than those of the nonzeros one by one.
//
// What bounds the resident schedule (resident.hip) is the LDS and the vector units: every nonzero reads its row of B from LDS, 512 bytes
// at N = 128, 600 us of LDS time for the 80 million of 32768 x 8192 at 0.3. Here a workgroup of eight waves computes 64 x 128
// results as dense products on the bf16 matrix cores (dense_tiles.hpp), the zeros of A included:
//   * A goes through LDS in slices of 128 columns, in two buffers. Every wave owns eight rows: sixteen lanes hold a row's next 64 (column,
//     value) pairs, those that lie in the slice are a prefix of them, and each is split into its three parts and written to its place
//     in a cleared row, whose 16 bytes beyond the slice take what is not in it. The pairs of the slice after are then on their way.
//   * B is split by a kernel of its own into the caller's memory, in the order in which lanes read it: split by every workgroup
//     instead, it would take more vector instructions than the matrix cores leave free.
//   * Wave w computes columns 32 (w mod 4) ... + 31 of all 64 rows, in the slice's first or last four steps of sixteen: one read of a
//     part of B serves two row blocks. (With one, the reads of B alone need all that a compute unit's vector-memory path carries.)
//     The products of a slice and the scatter of the next one are one stream of instructions, a product, four others and two writes in turn.
//   * hi x hi of a slice's steps is added up in 32 bits and goes to 64 bits slice by slice; the five smaller products have sums of
//     their own. The two halves of the steps meet in LDS at the end.
// Values of B that are not finite have zeros for parts and are added at the end, to the rows that use them (one NaN in B, 16384 x 8192,
// N = 128 at 0.3: 1601 us while it went through the products and made every row of its column one to compute again, now 245).
// Rows whose columns do not ascend, other results that are not finite, and results that are not large against what values too small for
// their parts may have lost are computed once more from the floats, row by row (three values of 1e-36 in every row of that matrix: 206
// us; 1598 while every row with one was computed again).
// Measured (us, three operand sets in turn, resident -> tiles): 32768 x 8192, N = 128 at 0.2 / 0.3 527 / 647 -> 392 / 420; 16384 x 8192 at 0.2 / 0.3 / 0.5
// 266 / 327 / 496 -> 204 / 206 / 291; 4096 x 4096, N = 512 at 0.5 245 -> 134; 16384 x 2048, N = 256 at 0.3 173 -> 113; 2000 x 4608, N = 3136 at 0.3
// 703 -> 440. Against 64 bits the results are off by 3.0 ... 3.4e-8, the resident schedule's by 6.9 ... 7.1e-8.
// What bounds it: the products and the power they take. 6 x 2 M K N in 206 us are 1.0 PFLOP/s of bf16, where a large bf16 product of random
// numbers reaches 1.2 ... 1.35 here; single launches take 5-10 % less than launches one after the other.
// Measured and not kept (16384 x 8192 at 0.3): B split in the kernel 388; 32 rows per workgroup, two workgroups per compute unit 267; eight
// waves that only scatter beside eight that only multiply 235, sums in 32 bits, off by 2e-7, because their registers do not hold more.
// The reference has no counterpart (SPMM/spmmesimd2.hpp:63-147 gathers every row of B from memory).
#include <algorithm>
#include <atomic>
#include <cstddef>

#include "dense_tiles.hpp"
#include "launch.hpp"

namespace dlspm {

constexpr int kTileWaves = 8, kTileThreads = kTileWaves * 64;
constexpr int kFragmentBytes = 3 * kWave * 16;

// ---- B: split once, in the order in which the products read it: [strip of 32 columns][step][part][lane][8]
// A value that is not finite, or that bf16 rounds to infinity, would make every result of its column NaN, through the zeros of A as
// well: its parts are zeros, and the rows that have its column get it from the float (spmm_tiles_kernel). Per strip and step, in a word:
// bits 0 ... 31 the columns with a nonzero value below 2^-109, 32 ... 47 the rows of B with a value that has no parts, 48 ... 55 the
// exponent of the largest of the others.
constexpr unsigned kTooLarge = 0xfeff0000u;  // twice the bits of a value, from this on: no parts
__global__ __launch_bounds__(256) void split_dense_kernel(int K, int N, int steps, const float* __restrict__ B, bf16x8* __restrict__ parts,
                                                          unsigned long long* __restrict__ notes)
{
    const int lane = threadIdx.x & 63, l = lane & 31, h = lane >> 5;
    const long long fragment = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int strip = (int)(fragment / steps), step = (int)(fragment - (long long)strip * steps);
    if (strip * 32 >= N) return;
    const int n = strip * 32 + l, k0 = 16 * step + 8 * h;
    float x[8], most = 0.f;
    unsigned without = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        x[j] = n < N && k0 + j < K ? B[(size_t)(k0 + j) * N + n] : 0.f;
        const bool none = (__float_as_uint(x[j]) << 1) >= kTooLarge;
        without |= none ? 1u << j : 0u;
        x[j] = none ? 0.f : x[j];
        most = fmaxf(most, fabsf(x[j]));
    }
    unsigned least;
    const Parts p = split_parts(x, least);
    bf16x8* const to = parts + fragment * 3 * kWave + lane;
    to[0] = p.hi;
    to[kWave] = p.mid;
    to[2 * kWave] = p.lo;
    const unsigned long long few = __ballot(least < kTooSmall);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o));
    unsigned long long note = (unsigned)few | (unsigned)(few >> 32) | (unsigned long long)(__float_as_uint(most) >> 23) << 48;
    if (__ballot(without != 0) != 0)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned long long in = __ballot((without >> j & 1) != 0);
            note |= (unsigned long long)((unsigned)in != 0 ? 1 : 0) << (32 + j) | (unsigned long long)((unsigned)(in >> 32) != 0 ? 1 : 0) << (40 + j);
        }
    if (lane == 0) notes[fragment] = note;
}

constexpr int kRows = 64, kCols = 128;                     // of C per workgroup
constexpr int kSlice = 128, kSteps = kSlice / 16;          // columns of A worked on at a time, in steps of sixteen
constexpr int kRowBytes = kSlice * 2 + 16, kPartBytes = kRows * kRowBytes, kBuffer = 3 * kPartBytes;
constexpr int kMostColumns = 1 << 22;                      // (a strip's parts are read as a buffer)
constexpr int kMine = kSteps / 2;                          // steps per wave: two waves share a strip
constexpr int kAhead = 2;                                  // steps of B loaded ahead
// the end, in the same LDS: the sums of one way (then what values of B without parts add), and behind them
constexpr int kSumBytes = 4 * 32 * kWave * (int)sizeof(double), kLoad = 4 * kWave;
struct EndLds {
    int again[kRows];  // the row is computed from the floats
    int tiny[kRows];   // ... has a value below 2^-109
    unsigned without, few, most;  // some strip of the tile has values of B without parts, below 2^-109; the bits of the rows' largest value
};
constexpr int kMarkSteps = (kSumBytes - kRows * kCols * (int)sizeof(float)) / (int)sizeof(unsigned short);
static_assert(kMarkSteps % kTileThreads == 0, "steps that share a mark are one thread's");

__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void spmm_tiles_kernel(
    int M, int K, int N, int nnz, int col_tiles, int streaming, const int* __restrict__ row_offsets, const int* __restrict__ col_indices,
    const float* __restrict__ values, const float* __restrict__ B, const bf16x8* __restrict__ parts,
    const unsigned long long* __restrict__ notes, float* __restrict__ C)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) char shared[];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), l = lane & 31, h = lane >> 5, l16 = lane & 15;
    const int at_xcd = (int)(blockIdx.x >> 3), ct = at_xcd % col_tiles, row0 = ((at_xcd / col_tiles) * 8 + (int)(blockIdx.x & 7)) * kRows;
    if (row0 >= M) return;
    const int col0 = ct * kCols, slices = (K + kSlice - 1) / kSlice, steps = slices * kSteps;
    const int strip = w & 3, way = w >> 2;

    // ---- A: eight rows per wave, in two groups of four, sixteen lanes to a row, four pairs to a lane
    const __amdgpu_buffer_rsrc_t columns_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(col_indices), 0, nnz * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t values_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(values), 0, nnz * 4, 0x00020000);
    int p[2], e[2], n[2], at[2][4];
    u4 c[2], a[2];
    bool wrong[2] = {false, false}, tiny[2] = {false, false};
    auto load_pairs = [&](int g) {
        const unsigned from = (unsigned)(p[g] + 4 * l16) * 4u;
        c[g] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(columns_buffer, from, 0, 0));
        a[g] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(values_buffer, from, 0, 0));
    };
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int row = row0 + 8 * w + 4 * g + (lane >> 4);
        p[g] = row_offsets[min(row, M)];
        e[g] = row_offsets[min(row + 1, M)];
        load_pairs(g);
    }
    auto place = [&](int g, int k0, int last) {
        int before = __builtin_amdgcn_update_dpp(last, (int)c[g][3], 0x111, 0xf, 0xf, false);  // row_shr:1
        const int left = e[g] - p[g] - 4 * l16;
        int m = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kk = (int)c[g][i] - k0;
            const bool in_row = i < left, in = in_row && (unsigned)kk < (unsigned)kSlice;
            wrong[g] |= in_row && (int)c[g][i] <= before;
            before = (int)c[g][i];
            m += in ? 1 : 0;
            at[g][i] = in ? kk : kSlice;
        }
        m += __builtin_amdgcn_update_dpp(0, m, 0x128, 0xf, 0xf, true);  // row_ror: the sum over the row
        m += __builtin_amdgcn_update_dpp(0, m, 0x124, 0xf, 0xf, true);
        m += __builtin_amdgcn_update_dpp(0, m, 0x122, 0xf, 0xf, true);
        n[g] = m + __builtin_amdgcn_update_dpp(0, m, 0x121, 0xf, 0xf, true);
    };
    const int own_row = 8 * w + (lane >> 4);
    auto put = [&](int g, int buffer) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        auto round2 = [](float x, float y) { return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x, y}, bf16x2)); };
        char* const row = shared + buffer * kBuffer + own_row * kRowBytes + g * 4 * kRowBytes;
        unsigned least = ~0u;
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const float x = __uint_as_float(a[g][i]), y = __uint_as_float(a[g][i + 1]);
            const unsigned hi = round2(x, y);
            const float rx = x - __uint_as_float(hi << 16), ry = y - __uint_as_float(hi & 0xffff0000u);
            const unsigned mid = round2(rx, ry);
            const unsigned lo = round2(rx - __uint_as_float(mid << 16), ry - __uint_as_float(mid & 0xffff0000u));
            unsigned short* const px = reinterpret_cast<unsigned short*>(row + at[g][i] * 2);
            unsigned short* const py = reinterpret_cast<unsigned short*>(row + at[g][i + 1] * 2);
            px[0] = (unsigned short)hi;
            px[kPartBytes / 2] = (unsigned short)mid;
            px[kPartBytes] = (unsigned short)lo;
            py[0] = (unsigned short)(hi >> 16);
            py[kPartBytes / 2] = (unsigned short)(mid >> 16);
            py[kPartBytes] = (unsigned short)(lo >> 16);
            least = min(least, min((a[g][i] << 1) - 1u, (a[g][i + 1] << 1) - 1u));
        }
        tiny[g] |= least < kTooSmall;
    };
    auto clear = [&](int buffer) {
#pragma unroll
        for (int i = 0; i < 6; ++i)
            *reinterpret_cast<uint4*>(shared + buffer * kBuffer + (i >> 1) * kPartBytes + (own_row + 4 * (i & 1)) * kRowBytes + l16 * 16) = uint4{0u, 0u, 0u, 0u};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    auto rest = [&](int g, int slice, int buffer, int last) {  // rows with more pairs in the slice than one load
        while (__ballot(n[g] == 64) != 0) {
            place(g, slice * kSlice, n[g] == 64 ? last : -1);
            put(g, buffer);
            last = __builtin_amdgcn_update_dpp(0, (int)c[g][3], 0x15f, 0xf, 0xf, true);
            p[g] += n[g];
            load_pairs(g);
        }
    };

    // ---- the products
    const __amdgpu_buffer_rsrc_t parts_buffer = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16x8*>(parts) + (size_t)min(col0 / 32 + strip, (N - 1) / 32) * steps * 3 * kWave, 0, steps * kFragmentBytes, 0x00020000);
    Parts b[kAhead];
    auto load_b = [&](int slot, int slice, int m) {  // the wave's m-th step from that slice's first on
        const int from = (min(slice + m / kMine, slices - 1) * kSteps + way * kMine + m % kMine) * kFragmentBytes;
        auto part = [&](int i) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(parts_buffer, lane * 16, from + i * kWave * 16, 0)); };
        b[slot] = Parts{part(0), part(1), part(2)};
    };
    f32x16 sum[2] = {}, small[2] = {};
    double total[2][16];
#pragma unroll
    for (int i = 0; i < 32; ++i) total[i / 16][i % 16] = 0.0;
#pragma unroll
    for (int m = 0; m < kAhead; ++m) load_b(m, 0, m);
    clear(0);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        place(g, 0, -1);
        put(g, 0);
        const int last = __builtin_amdgcn_update_dpp(0, (int)c[g][3], 0x15f, 0xf, 0xf, true);
        p[g] += n[g];
        load_pairs(g);
        rest(g, 0, 0, last);
    }
    __syncthreads();
    const char* const mine_at = shared + l * kRowBytes + way * kMine * 32 + h * 16;
    for (int s = 0; s < slices; ++s) {
        const int next = (s + 1) & 1;
        int last[2];
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            Parts q[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const char* const from = mine_at + (s & 1) * kBuffer + r * 32 * kRowBytes + m * 32;
                q[r] = Parts{*reinterpret_cast<const bf16x8*>(from), *reinterpret_cast<const bf16x8*>(from + kPartBytes), *reinterpret_cast<const bf16x8*>(from + 2 * kPartBytes)};
            }
            if (m == 0) clear(next);
            const Parts now = b[m % kAhead];
            const int g = m >> 1;
            if ((m & 1) == 0) place(g, (s + 1) * kSlice, -1);
            else {
                put(g, next);
                last[g] = __builtin_amdgcn_update_dpp(0, (int)c[g][3], 0x15f, 0xf, 0xf, true);
                p[g] += n[g];
                load_pairs(g);
            }
            if (m == 0)
#pragma unroll
                for (int i = 0; i < 32; ++i) total[i / 16][i % 16] += (double)sum[i / 16][i % 16];
            // (the two row blocks' products in turn: none waits for the one before it)
            auto both = [&](f32x16 (&to)[2], const bf16x8 Parts::*x, const bf16x8 Parts::*y) {
#pragma unroll
                for (int r = 0; r < 2; ++r) to[r] = mfma(now.*x, q[r].*y, to[r]);
            };
            both(small, &Parts::lo, &Parts::hi);
            both(small, &Parts::mid, &Parts::mid);
            both(small, &Parts::hi, &Parts::lo);
            both(small, &Parts::mid, &Parts::hi);
            both(small, &Parts::hi, &Parts::mid);
            if (m == 0) sum[0] = sum[1] = f32x16{};
            both(sum, &Parts::hi, &Parts::hi);
            load_b(m % kAhead, s, m + kAhead);
            // the reads of A first, then a product, four vector instructions and two writes in turn
            __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
            for (int i = 0; i < 12; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g)
            if (s + 1 < slices) rest(g, s + 1, next, last[g]);
        __syncthreads();
    }

    {
        // (the thread's place once more: kept through the loop, it would be spilled)
        const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), t = w * kWave + lane, l = lane & 31, h = lane >> 5, l16 = lane & 15;
        const int own_row = 8 * w + (lane >> 4);
        // ---- the two ways' sums
        double* const sums = reinterpret_cast<double*>(shared);
        EndLds& end = *reinterpret_cast<EndLds*>(shared + kSumBytes);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            total[i / 16][i % 16] += (double)sum[i / 16][i % 16] + (double)small[i / 16][i % 16];
            if (way > 0) sums[(strip * 32 + i) * kWave + lane] = total[i / 16][i % 16];
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const unsigned long long bad = __ballot(wrong[g] || p[g] < e[g]), few = __ballot(tiny[g]);
            if (l16 == 0) {
                end.again[own_row + 4 * g] = (bad >> (lane & 48) & 0xffff) != 0 ? 1 : 0;
                end.tiny[own_row + 4 * g] = (few >> (lane & 48) & 0xffff) != 0 ? 1 : 0;
            }
        }
        if (t == 0) end.without = end.few = end.most = 0;
        __syncthreads();
        const unsigned long long* const strip_notes = notes + (size_t)min(col0 / 32 + strip, (N - 1) / 32) * steps;
        unsigned few = 0;  // columns of the strip with a value of B that its parts do not hold
        float bound = 0.f, bound_tiny = 0.f;
        if (way == 0) {
            unsigned without = 0, exponent = 0;
            for (int i = lane; i < steps; i += kWave) {
                const unsigned long long note = strip_notes[i];
                few |= (unsigned)note;
                without |= (unsigned)(note >> 32) & 0xffffu;
                exponent = max(exponent, (unsigned)(note >> 48));
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                few |= __shfl_xor(few, o);
                without |= __shfl_xor(without, o);
                exponent = max(exponent, (unsigned)__shfl_xor((int)exponent, o));
            }
            if (lane == 0) {
                if (few != 0) end.few = 1;
                if (without != 0) end.without = 1;
            }
            // A value below 2^-109 is off by 2^-134 at most in its parts: of no account for results from 2^34 times what that can come to on.
            bound_tiny = ldexpf((float)K, (int)exponent - 126 - 100);
#pragma unroll
            for (int i = 0; i < 32; ++i) total[i / 16][i % 16] += sums[(strip * 32 + i) * kWave + lane];
        }
        __syncthreads();
        if (end.few != 0) {  // (uniform) the largest value of the 64 rows
            const int from = row_offsets[row0], to = row_offsets[min(row0 + kRows, M)];
            unsigned most = 0;
            for (int j = from + w * 2 * kLoad; j < to; j += kTileWaves * 2 * kLoad) {
                u4 x[2];
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    x[q] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(values_buffer, (unsigned)(j + q * kLoad + 4 * lane) * 4u, 0, 0));
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const unsigned v = x[i / 4][i % 4] & 0x7fffffffu;  // (a row with an infinity has no finite result to be bounded)
                    if (j + i / 4 * kLoad + 4 * lane + i % 4 < to && v < 0x7f800000u) most = max(most, v);
                }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, o));
            if (lane == 0) __hip_atomic_fetch_max(&end.most, most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __syncthreads();
            bound = (float)K * __uint_as_float(end.most) * 0x1p-100f;
        }
        if (way == 0) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const float least_row = end.tiny[32 * r + l] != 0 ? bound_tiny : 0.f;
                bool bad = false;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float x = fabsf((float)total[r][i]);
                    const int n = 8 * (i / 4) + 4 * h + i % 4;
                    const float least = fmaxf(least_row, (few >> n & 1) != 0 ? bound : 0.f);
                    bad |= (col0 + 32 * strip + n < N) & !((x >= least) & (x < __builtin_inff()));
                }
                if (bad) end.again[32 * r + l] = 1;
            }
        }
        __syncthreads();

        // ---- two columns of a row of the tile per lane
        const int c0 = col0 + 2 * lane, c0_at = min(c0, N - 2);
        const bool in0 = c0 < N, in1 = c0 + 1 < N;
        typedef float f2 __attribute__((ext_vector_type(2), aligned(4)));
        auto load_two = [&](int column) {
            f2 b = *reinterpret_cast<const f2*>(B + (size_t)column * N + c0_at);
            b.x = c0 == c0_at ? b.x : b.y;
            return b;
        };
        // ---- what the values of B without parts add: to the rows that have their columns, and to no others
        float* const extra = reinterpret_cast<float*>(shared);  // [row][column of the tile]
        if (end.without != 0) {  // (uniform)
            unsigned short* const of_step = reinterpret_cast<unsigned short*>(extra + kRows * kCols);  // which rows of B, per step modulo kMarkSteps
            for (int at = t; at < min(steps, kMarkSteps); at += kTileThreads) {
                unsigned long long any = 0;
                for (int i = at; i < steps; i += kMarkSteps)
#pragma unroll
                    for (int q = 0; q < kCols / 32; ++q) any |= notes[(size_t)min(col0 / 32 + q, (N - 1) / 32) * steps + i];
                of_step[at] = (unsigned short)(any >> 32);
            }
            __syncthreads();
            for (int i = w; i < kRows; i += kTileWaves) {
                double x0 = 0.0, x1 = 0.0;
                if (end.again[i] == 0 && row0 + i < M) {
                    const int from = __builtin_amdgcn_readfirstlane(row_offsets[row0 + i]), to = __builtin_amdgcn_readfirstlane(row_offsets[row0 + i + 1]);
                    bool large = false;  // a finite value: the sum is wanted as a whole
                    constexpr int kLoads = 4;
                    for (int j = from; j < to; j += kLoads * kLoad) {
                        u4 k[kLoads];
#pragma unroll
                        for (int q = 0; q < kLoads; ++q)
                            k[q] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(columns_buffer, (unsigned)(j + q * kLoad + 4 * lane) * 4u, 0, 0));
                        unsigned hits = 0;  // of the lane's pairs
#pragma unroll
                        for (int i = 0; i < 4 * kLoads; ++i) {
                            const unsigned mine = j + i / 4 * kLoad + 4 * lane + i % 4 < to ? 1u : 0u, column = k[i / 4][i % 4];
                            hits |= ((unsigned)of_step[mine * (column >> 4) % kMarkSteps] >> (column & 15) & mine) << i;
                        }
                        for (unsigned long long left; (left = __ballot(hits != 0)) != 0;) {
                            const int of = __builtin_ctzll(left), i = __builtin_ctz(__builtin_amdgcn_readlane(hits, of)), at = j + i / 4 * kLoad + 4 * of + i % 4;
                            if (lane == of) hits &= hits - 1;
                            const f2 b = load_two(col_indices[at]);
                            const double v = values[at];
                            const bool none0 = in0 && (__float_as_uint(b.x) << 1) >= kTooLarge, none1 = in1 && (__float_as_uint(b.y) << 1) >= kTooLarge;
                            large = large || (none0 && fabsf(b.x) < __builtin_inff()) || (none1 && fabsf(b.y) < __builtin_inff());
                            if (none0) x0 = fma(v, (double)b.x, x0);
                            if (none1) x1 = fma(v, (double)b.y, x1);
                        }
                        // (nothing changes any more)
                        if (__ballot(large) != 0 || __ballot((in0 && x0 == x0) || (in1 && x1 == x1)) == 0) break;
                    }
                    if (__ballot(large) != 0) end.again[i] = 1;
                }
                *reinterpret_cast<float2*>(extra + i * kCols + 2 * lane) = make_float2((float)x0, (float)x1);
            }
            __syncthreads();
        }
        if (way == 0)
#pragma unroll
            for (int r = 0; r < 2; ++r)
                if (row0 + 32 * r + l < M && end.again[32 * r + l] == 0)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int at = 32 * strip + 8 * q + 4 * h, n = col0 + at;
                        float* const to = C + (size_t)(row0 + 32 * r + l) * N + n;
                        Vec<4> x{make_float4((float)total[r][4 * q], (float)total[r][4 * q + 1], (float)total[r][4 * q + 2], (float)total[r][4 * q + 3])};
                        if (end.without != 0) {
                            const float4 y = *reinterpret_cast<const float4*>(extra + (32 * r + l) * kCols + at);
                            x.v = make_float4(x.v.x + y.x, x.v.y + y.y, x.v.z + y.z, x.v.w + y.w);
                        }
                        if (n + 3 < N) x.gstore(to, streaming != 0);
                        else {
                            if (n < N) to[0] = x.v.x;
                            if (n + 1 < N) to[1] = x.v.y;
                            if (n + 2 < N) to[2] = x.v.z;
                        }
                    }
        // ---- rows whose columns do not ascend, and results that the parts do not give: from the floats, in CSR order, in 64 bits
        for (int i = w; i < kRows; i += kTileWaves) {
            if (end.again[i] == 0 || row0 + i >= M) continue;
            const int from = __builtin_amdgcn_readfirstlane(row_offsets[row0 + i]), to = __builtin_amdgcn_readfirstlane(row_offsets[row0 + i + 1]);
            double x0 = 0.0, x1 = 0.0;
            int next_column = from < to ? col_indices[min(from + lane, to - 1)] : 0;
            float next_value = from < to ? values[min(from + lane, to - 1)] : 0.f;
            for (int j = from; j < to; j += kWave) {
                const int count = min(to - j, kWave), column = next_column;
                const int2 value = __builtin_bit_cast(int2, (double)next_value);  // (a conversion takes as long as four products)
                next_column = col_indices[min(j + kWave + lane, to - 1)];
                next_value = values[min(j + kWave + lane, to - 1)];
                constexpr int kFlight = 16;
                auto add = [&](const f2& b, int k) {
                    const double v = __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(value.x, k), __builtin_amdgcn_readlane(value.y, k)));
                    x0 = fma(v, (double)b.x, x0);
                    x1 = fma(v, (double)b.y, x1);
                };
                int k = 0;
                for (; k + kFlight <= count; k += kFlight) {
                    f2 b[kFlight];
#pragma unroll
                    for (int u = 0; u < kFlight; ++u) b[u] = load_two(__builtin_amdgcn_readlane(column, k + u));
#pragma unroll
                    for (int u = 0; u < kFlight; ++u) add(b[u], k + u);
                }
#pragma unroll 1
                for (; k < count; ++k) add(load_two(__builtin_amdgcn_readlane(column, k)), k);
            }
            float* const to_row = C + (size_t)(row0 + i) * N + c0;
            if (in0) to_row[0] = (float)x0;
            if (in1) to_row[1] = (float)x1;
        }
    }
}

// Tiles for these sizes: where their estimated time is below 0.9 of `other_us`, that of the schedule which needs no memory. The estimate
// (us): the split of B, and rounds of one workgroup per compute unit x (5 + slices x (2.95, from a density of 0.3 on 7 more per unit of
// density, where rows have more than 64 pairs in a slice)). Measured / estimated, and the resident schedule: 16384 x 8192, N = 128 at 0.2 /
// 0.3 / 0.5 204 / 206 / 291 (203 / 203 / 293) and 266 / 327 / 496; 8192 x 8192 at 0.3, N = 128 190 (203, on half of the units) and 187, N = 256
// 194 (206) and 323; 32768 x 8192 at 0.3, N = 64 400 (395) and 340; 2000 x 4608 at 0.3, N = 3136 440 (494) and 703. Uneven rows (lognormal,
// sigma 0.6) gain less, since a row of many pairs makes its wave come back to four rows and the others wait: 32768 x 8192 at 0.3 660 -> 545,
// 12288 x 4096 at 0.3, N = 200 241 -> 240. The row blocks are dealt to the XCDs with all their column tiles: 85 of them in three make 33
// workgroups for the 32 units of some, two rounds (5408 x 1340 at 0.25, N = 311: 79, estimated 82, resident 60).
double spmm_tiles_us(const DeviceInfo& dev, int M, int K, int N, int nnz)
{
    const double density = (double)nnz / ((double)M * K), slice_us = 2.95 + 7.0 * std::max(0.0, density - 0.3);
    // (eight XCDs: each has its row blocks' column tiles)
    const long long slices = ceil_div(K, kSlice), rounds = ceil_div(ceil_div(ceil_div(M, kRows), 8) * ceil_div(N, kCols), std::max(dev.cus / 8, 1));
    return 6.0 + (double)K * N * 3e-6 + (double)rounds * (5.0 + (double)slices * slice_us);
}
bool spmm_tiles_choose(const DeviceInfo& dev, int M, int K, int N, int nnz, double other_us)
{
    const Tuning& t = tuning();
    if (!rule_on(kRuleDenseGroups) || !rule_on(kRuleSpmmTiles) || N < 4 || M <= 0 || K <= 0 || nnz <= 0 || nnz >= (1 << 29) || K > kMostColumns || !dense_fits_buffer(K, N)) return false;
    // (a schedule that was asked for by name)
    if (t.split_w > 0 || t.flat >= 0 || t.slices >= 0 || t.tile_major >= 0 || t.tile_width > 0 || t.plan_order > 0 || t.xcd_contiguous) return false;
    return spmm_tiles_us(dev, M, K, N, nnz) < 0.9 * other_us;
}

static long long fragments_of(int K, int N) { return ceil_div(N, 32) * ceil_div(K, kSlice) * kSteps; }
size_t spmm_tiles_bytes(int K, int N) { return (size_t)fragments_of(K, N) * (kFragmentBytes + sizeof(unsigned long long)); }

void spmm_tile_shape(int* rows, int* columns)
{
    *rows = kRows;
    *columns = kCols;
}

hipError_t spmm_tiles_launch(const SpmmArgs& x, void* memory, hipStream_t stream)
{
    const int col_tiles = (int)ceil_div(x.N, kCols), steps = (int)ceil_div(x.K, kSlice) * kSteps;
    const long long fragments = fragments_of(x.K, x.N), blocks = (ceil_div(x.M, kRows) + 7) / 8 * 8 * col_tiles;
    if (blocks > 0x7fffffffLL || fragments > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    bf16x8* const parts = static_cast<bf16x8*>(memory);
    unsigned long long* const notes = reinterpret_cast<unsigned long long*>(static_cast<char*>(memory) + fragments * kFragmentBytes);
    hipLaunchKernelGGL(split_dense_kernel, dim3((unsigned)ceil_div(fragments, 4)), dim3(256), 0, stream, x.K, x.N, steps, x.B, parts, notes);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    constexpr size_t lds = 2 * kBuffer;
    static_assert(lds >= kSumBytes + sizeof(EndLds), "what the kernel ends with");
    // (once per device, as spmm_resident_launch)
    static std::atomic<unsigned long long> allowed[2];
    int device = 0;
    e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (device & 63);
    if (device >= 128 || (allowed[device >> 6].load(std::memory_order_relaxed) & bit) == 0) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&spmm_tiles_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        if (device < 128) allowed[device >> 6].fetch_or(bit, std::memory_order_relaxed);
    }
    const int stream_rule = tuning().stream_results;
    const bool streaming = stream_rule < 0 ? (long long)x.M * x.N >= 1024 * 1024 : stream_rule != 0;  // (as dense_rows_window)
    hipLaunchKernelGGL(spmm_tiles_kernel, dim3((unsigned)blocks), dim3(kTileThreads), lds, stream, x.M, x.K, x.N, x.nnz, col_tiles, streaming ? 1 : 0,
                       x.row_offsets, x.col_indices, x.values, x.B, parts, notes, x.C);
    return hipGetLastError();
}

}  // namespace dlspm
