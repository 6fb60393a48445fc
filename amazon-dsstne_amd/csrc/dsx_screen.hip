// dsx_screen.hip — 16-bit screening of candidates for the fp32 searches (nearest neighbours, output layer with top-K).
//
// A search wants, per row, the k columns of the highest fp32 scores.  The fp32 matrix instructions form every product at 1/16 of the
// f16 ones' rate (157 TFLOP/s against 2.5 PFLOP/s), so here all columns are looked at in f16 (dsx_f16.hip), as upper bounds of their
// scores, and only what the f16 operands' error leaves open is scored in fp32.  Scores and results are fp32 sums, all of them formed by
// one function in one order (equal columns tie, wherever they lie); the f16 sums only decide what cannot be a result.
//
// Error of a screened sum s' = sum x'_i w'_i against the fp32 sum s of the same row and column, x', w' rounded to f16 (unit
// roundoff u = 2^-11, 2^-25 absolute below the normal range), fp32 accumulation:
//   |s' - s| <= (2u + u^2) |x| |w| + 2^-25 sqrt(d) (|x| + |w|) + d 2^-50 + (1.1 d + 16) 2^-24 |x| |w|      (Cauchy-Schwarz; |.| = 2-norm)
// (d 2^-50: both operands' absolute roundings together, all there is to go by where every component is near 2^-25; the last term: d
// roundings of the matrix instructions' sums and d / 16 + 5 of screen_finish's)
// With the column's norm |w| kept in the table and e1, e0 per row, that is e1 |w| + e0.  A sum starts from its column's bias, raised by
// b_raise |b| for the roundings of a sum that holds it; z is that sum plus e1 |w|.  z + e0 is never below the score, whatever the
// spread of the norms, and the score lies above z - width(z, |w|) (screen_width).  So:
//   the k-th largest z - width bounds the k-th score from below, and only columns with z + e0 at or above that (as pre-activation
//   sums: preactivation_bound) can be results.  For normally distributed scores of 512 products that leaves about 1.2 k columns.
// Exceptions: a column whose norm is above 60,000 gets zeros and an infinite start (it always passes); a row above 65,504 is flagged,
// as is one whose lists fill up (thousands of scores tied at the top): its caller computes it again in fp32.
//
// Two ways (screen_stored).  Few columns, or few rows: the sums are stored as halves, rounded up, and a workgroup per row takes what
// reaches the bound from there.  Many of both: only a first block's are; the rest are compared with the rows' bounds where they are
// formed (raised by their errors, or against bounds lowered by the largest: screen_even), in ranges that grow by a factor, after
// each of which the lists are cut back to what can still be a result.
// Candidates of earlier ranges are not scored until the last one is through: what is scored in fp32 is about 1.2 k columns a row.
//
// Searches of long tables that are kept go in bytes (screen_in_bytes): the matrix instructions form products of bytes at twice
// the rate of halves, and read half as much.  x' = u q, w' = v r with whole numbers q, r of 127 at most; u is a row's unit, v one of 32 columns.  With
// what the bytes leave out, x = x' + x", w = w' + w", the sum of the products of the bytes is exact and
//   |s' - s| <= |x"| |w| + |x'| |w"| + (1.25 d + 64) 2^-24 |x| |w| + 3 u v      (the last two: a score's roundings in whatever order, and a start's)
// which is some fifteen times what halves leave open.  A word holds s' as an upper bound, and lies above it by
//   |word - s'| <= 50 u v + 1e-3 |word|
// at most: the lowest five bits of the float of 1.5 * 2^23 u v + s' say whose it is, and are taken for the largest they could be (33 units of its last place, a
// rounding of the start and one of the product counted in: 49.5 u v + 4e-6 |s'|), and it is rounded up to a half.  Where both operands are nearly whole numbers
// of their units that is more than the error.  So columns are not told apart by estimates of their scores on both sides: the columns of the k largest
// sums are scored at once, and their k-th score is what the others' upper bounds are held against (i8_finish_kernel): 1.2 to 4 k columns a row are
// scored.  No ranges, whose bounds and lists would take as long as the products do, and no lists that fill up.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include "dsx_screen.h"

namespace dsx {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
constexpr float kF16Max = 65504.0f, kScreenMax = 60000.0f;
constexpr uint32_t kPickWords = 2048;    // candidates of a row (part) that its workgroup holds
constexpr uint32_t kKeepWords = 1024;    // candidates of a row that outlive a column range
constexpr uint32_t kListWords = 4096;    // words of all of a row's lists of one column range
constexpr uint32_t kPickBlocks = 2048;   // blocks of 32 columns that a workgroup reads

uint32_t screen_ld(uint32_t dim) { return knn_f16_ld(dim); }
uint32_t screen_pitch32(uint32_t dim) { return (dim + 3) / 4 * 4; }

// Relative part of the error, with room for the rounding of the norms themselves; what a bias is raised by, per unit.
__host__ __device__ __forceinline__ float screen_relative(uint32_t dim) { return 9.765625e-4f * 1.01f + (1.25f * (float)dim + 64.0f) * 5.9604645e-8f; }
__host__ __device__ __forceinline__ float screen_bias_raise(uint32_t dim) { return ((float)dim + 64.0f) * 6.6e-8f; }

// stats (nearest neighbours): [0] largest norm of a column (the bits of a non-negative float; NaN columns have no part in it: their
// scores are NaN on every path); [1] sum of the norms of one column in 256, [2] their number; [4], [5], [7] I8ItemsArgs::error_most; [6] I8ItemsArgs::stats
struct ScreenItemsArgs {
    const float* W;       // [dim][ldw]
    uint64_t ldw;
    uint32_t n, dim, ld, pitch32;
    _Float16* out16;      // [n rounded up to 256][ld], zero filled
    float* out32;         // [n][pitch32], zero filled beyond dim
    float* norm;          // [n rounded up to 256]; infinite for columns that always pass
    float* seg_norm;      // [n rounded up to 256 / 64] largest of 64 columns
    uint32_t* stats;
};

// A workgroup takes 64 columns, 64 components at a time through LDS: reads are contiguous along the columns, writes along the
// components.  Bound by memory.
__global__ __launch_bounds__(256) void screen_items_kernel(ScreenItemsArgs a)
{
    __shared__ float sTile[64][65];
    __shared__ float sSum[4][64];
    const uint32_t col0 = blockIdx.x * 64, l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const bool valid = col0 + l < a.n;
    float sum = 0.0f;
    for (uint32_t d0 = 0; d0 < a.ld; d0 += 64) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t d = d0 + 4 * i + q;
            float x = (valid && d < a.dim) ? a.W[(uint64_t)d * a.ldw + col0 + l] : 0.0f;
            sTile[l][4 * i + q] = x;
            sum += x * x;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; i++) {   // 64 columns x 8 pieces of 8 halves
            const uint32_t c = (threadIdx.x >> 3) + 32 * i, p = (threadIdx.x & 7) * 8;
            half8 h;
#pragma unroll
            for (int e = 0; e < 8; e++) h[e] = (_Float16)sTile[c][p + e];
            *reinterpret_cast<half8*>(a.out16 + (uint64_t)(col0 + c) * a.ld + d0 + p) = h;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {   // 64 columns x 16 pieces of 4 floats
            const uint32_t c = (threadIdx.x >> 4) + 16 * i, p = (threadIdx.x & 15) * 4;
            if (col0 + c < a.n && d0 + p < a.pitch32)
                *reinterpret_cast<float4*>(a.out32 + (uint64_t)(col0 + c) * a.pitch32 + d0 + p) =
                    make_float4(sTile[c][p], sTile[c][p + 1], sTile[c][p + 2], sTile[c][p + 3]);
        }
    }
    sSum[q][l] = sum;
    __syncthreads();
    const float norm = sqrtf(sSum[0][l] + sSum[1][l] + sSum[2][l] + sSum[3][l]);   // of column l, in all four wavefronts
    const bool always = norm > kScreenMax;
    if (always)   // (its components may be infinite in f16; what the loop above wrote was ordered before by the barrier)
        for (uint32_t p = 8 * q; p < a.ld; p += 32) *reinterpret_cast<half8*>(a.out16 + (uint64_t)(col0 + l) * a.ld + p) = half8{};
    if (q == 0) {
        const float kept = always ? __builtin_inff() : norm;
        a.norm[col0 + l] = kept;
        float finite = always ? 0.0f : fmaxf(kept, 0.0f), most = fmaxf(norm, 0.0f);   // (drops NaN)
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            finite = fmaxf(finite, __shfl_xor(finite, d));
            most = fmaxf(most, __shfl_xor(most, d));
        }
        if (l == 0) {
            a.seg_norm[blockIdx.x] = finite;   // (a column that always passes counts for no bound)
            if (__float_as_uint(most) > *(volatile uint32_t*)&a.stats[0]) atomicMax(&a.stats[0], __float_as_uint(most));
        }
    }
    if (q == 1 && blockIdx.x % 256 == 0) {
        float some = (valid && norm <= kF16Max) ? norm : 0.0f;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) some += __shfl_xor(some, d);
        const uint32_t number = (uint32_t)__popcll(__ballot(valid && norm <= kF16Max));
        if (l == 0) {
            unsafeAtomicAdd(reinterpret_cast<float*>(&a.stats[1]), some);   // (the instruction; plain atomicAdd is a loop, 36 us of it here)
            atomicAdd(&a.stats[2], number);
        }
    }
}

struct ScreenRowsArgs {
    const float* X;
    uint32_t ldx, batch, dim, ld;
    int whole;              // X is 16-byte aligned and its pitch a multiple of 4
    _Float16* out16;        // [batch rounded up to 256][ld], zero filled
    float* e1;              // [batch]
    float* e0;              // [batch]
    float* scale;           // [batch]
    int scaled;             // the scale follows the norms (else 1)
    uint32_t* row_flag;     // [batch] set where the error has no bound, else cleared
    uint32_t* told;         // host-visible word set with it (may be NULL)
    uint32_t* cand_count;   // [batch] cleared, and so is
    uint32_t* clear;        // [clear_words]
    uint32_t clear_words;
    const uint32_t* stats;
    ScreenNotes* notes;     // host-visible: what the table's columns and the rows are like (nearest neighbours)
};

// One wavefront per row, which holds up to 1,024 components of it between the two passes.  Bound by latency, one round trip so (256 x 1,024:
// 9.7 us when a lane read its components one by one, twice; 4.5 so; 4,096 x 1,024 28 / 14 beside other kernels).
__global__ __launch_bounds__(256) void screen_rows_kernel(ScreenRowsArgs a)
{
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const bool valid = row < a.batch;
    const float* x = a.X + (uint64_t)row * a.ldx;
    auto part = [&](uint32_t d) __attribute__((always_inline)) -> float4 {
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (!valid || d >= a.dim) return v;
        if (a.whole) {
            v = *reinterpret_cast<const float4*>(x + d);
            if (d + 1 >= a.dim) v.y = 0.0f;
            if (d + 2 >= a.dim) v.z = 0.0f;
            if (d + 3 >= a.dim) v.w = 0.0f;
        } else {
            v.x = x[d];
            if (d + 1 < a.dim) v.y = x[d + 1];
            if (d + 2 < a.dim) v.z = x[d + 2];
            if (d + 3 < a.dim) v.w = x[d + 3];
        }
        return v;
    };
    constexpr int G = 4;
    float4 held[G];
#pragma unroll
    for (int g = 0; g < G; g++) held[g] = part(g * 4 * kWave + 4 * lane);
    float sum = 0.0f;
    auto add = [&](const float4& v) __attribute__((always_inline)) { sum += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w); };
#pragma unroll
    for (int g = 0; g < G; g++) add(held[g]);
#pragma unroll 4
    for (uint32_t d = G * 4 * kWave + 4 * lane; d < a.dim; d += 4 * kWave) add(part(d));
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) sum += __shfl_xor(sum, d);
    const float norm = sqrtf(sum);
    const bool bad = norm > kF16Max;   // (a NaN in the row: its scores are NaN everywhere, there is nothing to miss)
    auto put = [&](uint32_t d, const float4& v) __attribute__((always_inline)) {
        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
        half4 h = {};
        if (!bad) h = half4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
        if (d < a.ld) *reinterpret_cast<half4*>(a.out16 + (uint64_t)row * a.ld + d) = h;
    };
#pragma unroll
    for (int g = 0; g < G; g++) put(g * 4 * kWave + 4 * lane, held[g]);
#pragma unroll 4
    for (uint32_t d = G * 4 * kWave + 4 * lane; d < a.ld; d += 4 * kWave) put(d, part(d));
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < a.clear_words; i += 256) a.clear[i] = 0;
    if (!valid || lane != 0) return;
    a.cand_count[row] = 0;
    a.row_flag[row] = bad ? 1u : 0u;
    if (row == 0 && a.notes) {
        a.notes->largest = __uint_as_float(a.stats[0]);
        a.notes->sum = __uint_as_float(a.stats[1]);
        a.notes->number = a.stats[2];
    }
    const float absolute = 2.9802322e-8f * 1.01f * sqrtf((float)a.dim + 4.0f);
    a.e1[row] = bad ? 0.0f : (screen_relative(a.dim) + screen_bias_raise(a.dim)) * norm + absolute + 1e-30f;
    a.e0[row] = bad ? 0.0f : absolute * norm + (float)a.dim * 8.8817842e-16f * 1.01f + 1e-30f;
    // Stored as halves, sums without a bias are scaled by a power of two that takes the largest there can be to about 1,024 (products of
    // tiny vectors would all be the same few subnormal halves).
    float scale = 1.0f;
    if (a.scaled) {
        const float most = norm * __uint_as_float(a.stats[0]);
        if (most > 1e-30f && most < 1e30f) scale = ldexpf(1.0f, 10 - ilogbf(most));
    }
    a.scale[row] = scale;
    if (bad && a.told) *(volatile uint32_t*)a.told = 1u;
}

// ---- bytes
// The unit of a vector's bytes: 127 of it are the largest component, and the bytes' own norm stays below 2,000 and their roundings (2,032 with
// 4,096 components), so that a sum of products of two vectors' bytes is below 2^22.
__device__ __forceinline__ float i8_unit(float largest, float norm) { return fmaxf(largest * (1.0f / 127.0f) * 1.000001f, norm * (1.0f / 2000.0f)); }

// Norms whose squares are too small to be summed count as what the largest component allows (also what bytes leave out: half a unit each, or
// everything where the unit is too small to divide by).
__device__ __forceinline__ float i8_norm(float norm, float largest, uint32_t dim) { return norm < 1e-15f ? largest * 1.01f * sqrtf((float)dim) : norm; }
__device__ __forceinline__ float i8_left(float left, float unit, float largest, uint32_t dim)
{
    const float most = (unit > 1e-35f ? 0.5f * unit : largest) * sqrtf((float)dim);
    return 1.01f * (unit < 1e-15f ? most : sqrtf(left));
}

struct I8ItemsArgs {
    const float* rows32;    // [n][pitch32]
    const _Float16* rows16; // or [n rounded up to 256][ld16]
    uint32_t ld16;
    float* norm;            // [n]; from rows16 it is made here
    uint32_t* stats;        // [6] whether a norm is no number (from rows16: no finite one); from rows16 [0], the largest, as well
    uint32_t n, dim, pitch32, ld8;
    int8_t* items8;         // [n rounded up to 256][ld8], zero filled
    float* unit;            // [n rounded up to 256 / 32]
    float* side;            // [n rounded up to 256 / 32][kI8Side]
    float2* error;          // [n rounded up to 256 / 128] largest norm, and largest norm of what the bytes leave out, of 128 columns
    uint32_t* error_most;   // the largest two of these, and ([3]) the largest unit (the bits of non-negative floats)
};

// A workgroup takes 128 columns, 32 after each other: their largest component, then their bytes; a wavefront eight columns.  Bound by memory (the second
// reading comes from L2).
template <bool HALVES>
__global__ __launch_bounds__(256) void i8_items_kernel(I8ItemsArgs a)
{
    __shared__ float sLargest[4], sNorm[4], sLeft[4];
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    float norm_most = 0.0f, left_most = 0.0f, unit_most = 0.0f;
    auto four = [&](uint32_t c, uint32_t d) __attribute__((always_inline)) -> float4 {
        if constexpr (HALVES) {
            typedef _Float16 half4 __attribute__((ext_vector_type(4)));
            if (d >= a.ld16) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const half4 h = *reinterpret_cast<const half4*>(a.rows16 + (uint64_t)c * a.ld16 + d);
            return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
        } else {
            if (d >= a.pitch32) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            return *reinterpret_cast<const float4*>(a.rows32 + (uint64_t)c * a.pitch32 + d);
        }
    };
    for (uint32_t block = blockIdx.x * 4; block < blockIdx.x * 4 + 4; block++) {
        const uint32_t c0 = block * 32 + wave * 8;
        float largest = 0.0f, norms = 0.0f;
        for (uint32_t c = c0; c < min(c0 + 8, a.n); c++) {
            float norm, most = 0.0f, sum = 0.0f;
            if constexpr (!HALVES) {
                norm = a.norm[c];
                if (norm != norm && lane == 0) a.stats[6] = 1u;
                if (!(norm < __builtin_inff())) continue;   // always passes, or never: no bytes
            }
            for (uint32_t d = 4 * lane; d < a.ld8; d += 4 * kWave) {
                const float4 v = four(c, d);
                most = fmaxf(fmaxf(most, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
                if constexpr (HALVES) sum += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
            }
            if constexpr (HALVES) {
#pragma unroll
                for (int d = 1; d < kWave; d *= 2) sum += __shfl_xor(sum, d);
                norm = sqrtf(sum);
                if (lane == 0) {
                    a.norm[c] = norm;
                    if (!(norm < __builtin_inff())) a.stats[6] = 1u;
                }
                if (!(norm < __builtin_inff())) continue;
            }
            norms = fmaxf(norms, norm);
            largest = fmaxf(largest, most);
        }
#pragma unroll
        for (int d = 1; d < kWave; d *= 2) largest = fmaxf(largest, __shfl_xor(largest, d));
        if (lane == 0) {
            sLargest[wave] = largest;
            sNorm[wave] = norms;
        }
        __syncthreads();
        const float norm32 = fmaxf(fmaxf(sNorm[0], sNorm[1]), fmaxf(sNorm[2], sNorm[3]));
        const float largest32 = fmaxf(fmaxf(sLargest[0], sLargest[1]), fmaxf(sLargest[2], sLargest[3])), unit = i8_unit(largest32, norm32);
        const float inverse = unit > 1e-35f ? 1.0f / unit : 0.0f;   // (all bytes 0: what they leave out is everything)
        norm_most = fmaxf(norm_most, i8_norm(norm32, largest32, a.dim));
        unit_most = fmaxf(unit_most, unit);
        for (uint32_t c = c0; c < c0 + 8; c++) {
            const bool some = c < a.n && a.norm[min(c, a.n - 1)] < __builtin_inff();   // (this wavefront's own, and behind a barrier)
            float left = 0.0f;
            for (uint32_t d = 4 * lane; d < a.ld8; d += 4 * kWave) {
                float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if (some) *reinterpret_cast<float4*>(v) = four(c, d);
                uint32_t bytes = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float b = fminf(fmaxf(rintf(v[e] * inverse), -127.0f), 127.0f), rest = fmaf(-b, unit, v[e]);
                    bytes |= ((uint32_t)(int32_t)b & 255u) << (8 * e);
                    left = fmaf(rest, rest, left);
                }
                *reinterpret_cast<uint32_t*>(a.items8 + (uint64_t)c * a.ld8 + d) = bytes;
            }
#pragma unroll
            for (int d = 1; d < kWave; d *= 2) left += __shfl_xor(left, d);
            // (three units of the sums' last place for the roundings of a sum that has started from something: i8_rows_kernel's |x| is 127 of its units at least)
            left_most = fmaxf(left_most, i8_left(left, unit, largest32, a.dim) + unit * (4.0f / 127.0f) + 1e-30f);
        }
        if (threadIdx.x == 0) a.unit[block] = unit;
        if (threadIdx.x < kI8Side) {
            const uint32_t c = block * 32 + threadIdx.x;
            a.side[(uint64_t)block * kI8Side + threadIdx.x] = threadIdx.x == 32 ? unit : (threadIdx.x > 32 || c >= a.n) ? -3e37f : i8_start(0.0f, a.norm[c], 0.0f);
        }
        __syncthreads();
    }
    if (lane == 0) sLeft[wave] = left_most;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float left = fmaxf(fmaxf(sLeft[0], sLeft[1]), fmaxf(sLeft[2], sLeft[3]));
        a.error[blockIdx.x] = make_float2(norm_most, left);
        if (HALVES && __float_as_uint(norm_most) > *(volatile uint32_t*)&a.stats[0]) atomicMax(&a.stats[0], __float_as_uint(norm_most));
        if (__float_as_uint(norm_most) > *(volatile uint32_t*)&a.error_most[0]) atomicMax(&a.error_most[0], __float_as_uint(norm_most));
        if (__float_as_uint(left) > *(volatile uint32_t*)&a.error_most[1]) atomicMax(&a.error_most[1], __float_as_uint(left));
        if (__float_as_uint(unit_most) > *(volatile uint32_t*)&a.error_most[3]) atomicMax(&a.error_most[3], __float_as_uint(unit_most));
    }
}

struct I8RowsArgs {
    const float* X;
    uint32_t ldx, batch, dim, ld8;
    int8_t* rows8;          // [batch rounded up to 256][ld8], zero filled
    float* unit;            // [batch] times scale
    float4* error;          // [batch] a column's sum is wrong by x times its norm, y times the norm of what its bytes leave out, and z at most; w: 1 / scale
    const uint32_t* stats;  // (the table's) where sums are scaled before they are stored as halves, NULL: they are not
    uint32_t* row_flag;     // as screen_rows_kernel
    uint32_t* told;
    uint32_t* clear;
    uint32_t clear_words;
    int halves;             // the rows are rounded to halves first
    const float* bias;      // with row_blocks: the side of i8_wide_run, made by the workgroups behind the rows' (NULL: not)
    const float* norm;
    float bias_raise;
    uint32_t row_blocks, n;
    const float* table_side;
    float* side;
};

// One wavefront per row, which it reads twice.  Bound by latency.
__global__ __launch_bounds__(256) void i8_rows_kernel(I8RowsArgs a)
{
    if (blockIdx.x >= a.row_blocks) {
        for (uint64_t i = (uint64_t)(blockIdx.x - a.row_blocks) * 256 + threadIdx.x; i < ((uint64_t)a.n + 255) / 256 * 8 * kI8Side; i += (uint64_t)(gridDim.x - a.row_blocks) * 256) {
            const uint32_t block = (uint32_t)(i / kI8Side), e = (uint32_t)(i % kI8Side), c = block * 32 + e;
            a.side[i] = (e >= 32 || c >= a.n) ? a.table_side[i] : i8_start(a.bias[c], a.norm[c], a.bias_raise);
        }
        return;
    }
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const bool valid = row < a.batch;
    const float* x = a.X + (uint64_t)row * a.ldx;
    auto part = [&](uint32_t d, float (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = (valid && d + e < a.dim) ? x[d + e] : 0.0f;
            if (a.halves) v[e] = (float)(_Float16)v[e];
        }
    };
    constexpr int G = 4;
    float held[G][4];
#pragma unroll
    for (int g = 0; g < G; g++) part(4 * (g * kWave + lane), held[g]);
    float sum = 0.0f, largest = 0.0f;
    auto add = [&](const float (&v)[4]) __attribute__((always_inline)) {
        sum += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
        largest = fmaxf(fmaxf(largest, fmaxf(fabsf(v[0]), fabsf(v[1]))), fmaxf(fabsf(v[2]), fabsf(v[3])));
    };
#pragma unroll
    for (int g = 0; g < G; g++) add(held[g]);
    for (uint32_t d = G * 4 * kWave + 4 * lane; d < a.dim; d += 4 * kWave) {
        float v[4];
        part(d, v);
        add(v);
    }
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
        sum += __shfl_xor(sum, d);
        largest = fmaxf(largest, __shfl_xor(largest, d));
    }
    const float norm = sqrtf(sum);
    const bool bad = norm > kF16Max;   // (a NaN in the row: its unit is one too, and the row has no results)
    const float unit = (norm != norm) ? norm : bad ? 0.0f : i8_unit(largest, norm), inverse = unit > 1e-35f ? 1.0f / unit : 0.0f;
    float left = 0.0f;
    auto put = [&](uint32_t d, const float (&v)[4]) __attribute__((always_inline)) {
        uint32_t bytes = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float b = inverse > 0.0f ? fminf(fmaxf(rintf(v[e] * inverse), -127.0f), 127.0f) : 0.0f, rest = fmaf(-b, unit, v[e]);
            bytes |= ((uint32_t)(int32_t)b & 255u) << (8 * e);
            left = fmaf(rest, rest, left);
        }
        if (d < a.ld8) *reinterpret_cast<uint32_t*>(a.rows8 + (uint64_t)row * a.ld8 + d) = bytes;
    };
#pragma unroll
    for (int g = 0; g < G; g++) put(4 * (g * kWave + lane), held[g]);
    for (uint32_t d = G * 4 * kWave + 4 * lane; d < a.ld8; d += 4 * kWave) {
        float v[4];
        part(d, v);
        put(d, v);
    }
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) left += __shfl_xor(left, d);
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < a.clear_words; i += 256) a.clear[i] = 0;
    if (!valid || lane != 0) return;
    a.row_flag[row] = bad ? 1u : 0u;
    float scale = 1.0f;
    if (a.stats) {
        const float most = norm * __uint_as_float(a.stats[0]);
        if (most > 1e-30f && most < 1e30f) scale = ldexpf(1.0f, 10 - ilogbf(most));
    }
    const float rest = i8_left(left, unit, largest, a.dim), length = i8_norm(norm, largest, a.dim);
    a.unit[row] = unit * scale;
    a.error[row] = make_float4(rest + ((1.25f * (float)a.dim + 64.0f) * 5.9604645e-8f + screen_bias_raise(a.dim)) * length + 1e-30f, (length + rest) * 1.01f + 1e-30f,
                               1e-30f, 1.0f / scale);
    if (bad && a.told) *(volatile uint32_t*)a.told = 1u;
}

// What the kernels below have in common.
struct ScreenFoldArgs {
    uint32_t batch, k, n;
    const float* e1;
    const float* e0;
    float width_bias;        // share of width per unit of e1 |w| beyond 2.02 (the bias's roundings)
    float width_z;           // and per unit of |z|
    const float* norm;       // by column
    const float* seg_norm;
    const float* largest;    // norm whose error the ranges' bounds are lowered by (NULL: the sums are raised)
    uint32_t act;
    float slope, alpha, lambda;
    uint32_t* row_flag;
    uint32_t* told;
    uint32_t* open;
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;    // NULL: no filter
    // candidates that outlive the range, and the next range's bound
    uint64_t* keep;          // [batch][kKeepWords]
    uint32_t* keep_count;    // [batch]
    uint32_t* admit;         // [batch]
    // lists
    uint64_t* seg;           // [batch][lists][seg_cap]
    uint32_t* seg_count;     // [batch][kF16ListStride]
    uint32_t lists, seg_cap;
    uint64_t* cand;          // [batch][cap]
    uint32_t* cand_count;
    uint32_t cap;
    // pick
    const _Float16* Z;
    const _Float16* M;
    uint64_t ldz;
    const float* scale;
    uint32_t stored;         // columns of Z
    // in bytes
    const uint32_t* words;   // [batch][ldw]
    uint64_t ldw;
    const float2* error_items;
    const float4* error_rows;
    const _Float16* rows16;  // scores are products of halves (else NULL)
    uint32_t ld16;
    const uint2* near;       // i8_near_kernel's
    const uint2* near_found;
    // final
    const float* X;
    uint32_t ldx, dim, pitch32;
    const float* rows32;
    const float* bias;
    float* keys;
    uint32_t* values;
    float* keys2;
    uint32_t* values2;
};

// A score lies above z less this.  (z: rounded up when it was stored as a half, which width_z and the last term cover; half_step: 1 /
// scale of the row, as halves below the normal range are 2^-24 apart)
__device__ __forceinline__ float screen_width(const ScreenFoldArgs& a, float z, float norm, float e1, float e0, float half_step)
{
    return e1 * (2.02f + a.width_bias) * norm + 1.01f * e0 + a.width_z * fabsf(z) + 2e-7f * half_step;
}

// A listed sum, raised by its column's norm.  (A column of infinite norm has an infinite sum.)
__device__ __forceinline__ uint64_t screen_raised(const ScreenFoldArgs& a, uint64_t word, float e1)
{
    const float x = key_score((uint32_t)(word >> 32)), norm = a.norm[~(uint32_t)word];
    return ((uint64_t)score_key(norm < __builtin_inff() ? fmaf(e1, norm, x) : __builtin_inff()) << 32) | (uint32_t)word;
}

// The sum z below which nothing can be a result when k columns have scores of at least this key.  (Args: what knows the activation)
template <class Args> __device__ __forceinline__ float screen_cut_key(const Args& a, uint32_t key, float e0)
{
    const float z = preactivation_bound(key, a.act, a.slope, a.alpha, a.lambda);
    const float cut = z - e0 * 1.001f - fabsf(z) * 2.3841858e-7f;   // (the subtraction itself is rounded)
    return (cut == cut) ? cut : -__builtin_inff();
}

// The same when k columns score at least t (as a sum); -inf: anything can.
__device__ __forceinline__ float screen_cut(const ScreenFoldArgs& a, float t, float e0)
{
    if (!(t > -__builtin_inff())) return -__builtin_inff();
    return screen_cut_key(a, score_key(activate_rt(t, a.act, a.slope, a.alpha, a.lambda)), e0);
}

__device__ __forceinline__ void screen_flag(const ScreenFoldArgs& a, uint32_t b)
{
    a.row_flag[b] = 1;
    if (a.told) *(volatile uint32_t*)a.told = 1u;
    if (a.admit) a.admit[b] = 0xffffffffu;   // a NaN: nothing more of the row is wanted
}

// What bytes leave too much of open; halves may not.
__device__ __forceinline__ void screen_open(const ScreenFoldArgs& a, uint32_t b)
{
    a.row_flag[b] = 1;
    if (a.open) *(volatile uint32_t*)a.open = 1u;
}

// The row itself into LDS, zero filled to whole rounds of the loop below; first: the caller's component threadIdx.x of it.
template <int T> __device__ __forceinline__ void screen_row(const ScreenFoldArgs& a, uint32_t b, float* sX, float first)
{
    const uint32_t dpad = (a.dim + 63) / 64 * 64;
    if (threadIdx.x < dpad) sX[threadIdx.x] = first;
    for (uint32_t d = T + threadIdx.x; d < dpad; d += T) sX[d] = (d < a.dim) ? a.X[(uint64_t)b * a.ldx + d] : 0.0f;
}

// The same as halves, as items of an fp16 table are laid out.
template <int T> __device__ __forceinline__ void screen_row_halves(const ScreenFoldArgs& a, uint32_t b, _Float16* sX, float first)
{
    if (threadIdx.x < a.ld16) sX[threadIdx.x] = (_Float16)first;
    for (uint32_t d = T + threadIdx.x; d < a.ld16; d += T) sX[d] = (d < a.dim) ? (_Float16)a.X[(uint64_t)b * a.ldx + d] : (_Float16)0.0f;
}

// The row's candidates sList[from .. count) scored in fp32: their words get the scores' keys, and become 0 where a score is no number.  Sixteen lanes per
// candidate; the order of a sum depends on nothing but its length.  Every lane of the workgroup calls this.
template <int T, int STEPS = 2> __device__ __forceinline__ void screen_score(const ScreenFoldArgs& a, uint64_t* sList, uint32_t from, uint32_t count, const float* sX)
{
    // (four candidates of a group of lanes at a time: their rows are waited for together)
    constexpr int U = 4;
    const uint32_t sub = threadIdx.x % 16;
    for (uint32_t e0 = from + threadIdx.x / 16; e0 < count; e0 += T / 16 * U) {
        uint32_t col[U];
        float sum[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            col[u] = ~(uint32_t)sList[min(e0 + T / 16 * u, count - 1)];
            sum[u] = 0.0f;
        }
#pragma unroll STEPS
        for (uint32_t d = 4 * sub; d < a.pitch32; d += 64) {
            const float4 x = *reinterpret_cast<const float4*>(sX + d);
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (u == 0 || e0 + T / 16 * u < count) v[u] = *reinterpret_cast<const float4*>(a.rows32 + (uint64_t)col[u] * a.pitch32 + d);
#pragma unroll
            for (int u = 0; u < U; u++)
                if (u == 0 || e0 + T / 16 * u < count) {
                    sum[u] = fmaf(x.x, v[u].x, sum[u]);
                    sum[u] = fmaf(x.y, v[u].y, sum[u]);
                    sum[u] = fmaf(x.z, v[u].z, sum[u]);
                    sum[u] = fmaf(x.w, v[u].w, sum[u]);
                }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int d = 1; d < 16; d *= 2) sum[u] += __shfl_xor(sum[u], d);
            if (sub == 0 && e0 + T / 16 * u < count) {
                const float y = activate_rt(sum[u] + (a.bias ? a.bias[col[u]] : 0.0f), a.act, a.slope, a.alpha, a.lambda);
                sList[e0 + T / 16 * u] = (y == y) ? ((uint64_t)score_key(y) << 32) | (uint32_t)~col[u] : 0ull;
            }
        }
    }
}

// The same of an fp16 table: exact products, summed by the matrix instruction of the searches that are not screened, in their order (dsx_f16.hip), so that a
// score has the same bits whichever way a search goes.  A wavefront takes 32 candidates, as the row operand; every column of the other one is the query.
// Bound by the latency of the candidates' rows.  4,096 rows x 1,000,000 x 128 top 100: i8_finish_kernel 146 to 158 us (sixteen lanes a candidate, sums in an order of
// their own: 152).
template <int T> __device__ __forceinline__ void screen_score_halves(const ScreenFoldArgs& a, uint64_t* sList, uint32_t from, uint32_t count, const _Float16* sX)
{
    const uint32_t lane = threadIdx.x % kWave, l32 = lane % 32, lhi = lane / 32;
    for (uint32_t e0 = from + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * 32; e0 < count; e0 += T / kWave * 32) {
        const uint32_t col = ~(uint32_t)sList[e0 + l32 < count ? e0 + l32 : e0];   // (no other wavefront's words, which change)
        const _Float16* row = a.rows16 + (uint64_t)col * a.ld16 + 8 * lhi;
        floatx16 sums;
#pragma unroll
        for (int v = 0; v < 16; v++) sums[v] = 0.0f;
        auto pieces = [&](half8 (&item)[4], uint32_t d) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 4; s++) item[s] = *reinterpret_cast<const half8*>(row + d + 16 * s);
        };
        auto add = [&](const half8 (&item)[4], uint32_t d) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 4; s++)
                sums = __builtin_amdgcn_mfma_f32_32x32x16_f16(item[s], *reinterpret_cast<const half8*>(sX + d + 16 * s + 8 * lhi), sums, 0, 0, 0);
        };
        // (ld16 is a multiple of 64; the next 64 components are on their way while these are multiplied, the last ones twice)
        half8 now[4], next[4];
        pieces(now, 0);
#pragma unroll 1
        for (uint32_t d = 0; d < a.ld16; d += 128) {
            pieces(next, min(d + 64, a.ld16 - 64));
            __builtin_amdgcn_sched_barrier(0);
            add(now, d);
            if (d + 64 >= a.ld16) break;
            pieces(now, min(d + 128, a.ld16 - 64));
            __builtin_amdgcn_sched_barrier(0);
            add(next, d + 64);
        }
        // Result v of a lane is candidate v % 4 + v / 4 * 8 + 4 lhi, the same in all 32 lanes: lane v of them takes it.
        float y = sums[0];
#pragma unroll
        for (int v = 1; v < 16; v++) y = l32 == (uint32_t)v ? sums[v] : y;
        const uint32_t at = e0 + l32 % 4 + l32 / 4 * 8 + 4 * lhi;
        if (l32 < 16 && at < count) sList[at] = (y == y) ? ((uint64_t)score_key(y) << 32) | (uint32_t)sList[at] : 0ull;
    }
}

// The k best of the scored words sList[0 .. count) written.  sBest: 256 words, cleared before the caller's last barrier.
template <int T>
__device__ __forceinline__ void screen_results(const ScreenFoldArgs& a, uint32_t b, const uint64_t* sList, uint32_t count, uint64_t* sBest, bool listed)
{
    for (uint32_t i = threadIdx.x; i < count; i += T) {
        const uint64_t w = sList[i];
        if (w == 0) continue;
        uint32_t rank = 0;
        for (uint32_t j = 0; j < count; j++) rank += sList[j] > w;
        if (rank < a.k) sBest[rank] = w;
    }
    __syncthreads();
    if (threadIdx.x < a.k) {
        const uint64_t w = sBest[threadIdx.x], at = (uint64_t)b * a.k + threadIdx.x;
        const float key = w != 0 ? key_score((uint32_t)(w >> 32)) : -kMaxValue;   // engine/kernels.cu:3221-3224: unfilled slots
        const uint32_t col = w != 0 ? ~(uint32_t)w : 0u;
        a.keys[at] = key;
        a.values[at] = col;
        if (a.keys2) {
            a.keys2[at] = key;
            a.values2[at] = col;
        }
    }
    // A listed column scores 0, not nothing (utils/Filters.cpp:62 multiplies, kCalculateTopK then sees the zero): when the row's k-th
    // score is not above 0, or the row has fewer than k scores, such a zero belongs in the result, and the row is computed again.
    if (threadIdx.x == 0 && listed && (uint32_t)(sBest[a.k - 1] >> 32) <= score_key(0.0f)) screen_flag(a, b);
}

// The row's candidates sList[0 .. count) scored and its k best written.  Every lane of the workgroup calls this.
// first: the caller's component threadIdx.x of the row; listed: whether the row has a listed column (the same for the workgroup).
template <int T>
__device__ __forceinline__ void screen_finish(const ScreenFoldArgs& a, uint32_t b, uint64_t* sList, uint32_t count, float* sX, float first, bool listed)
{
    __shared__ uint64_t sBest[256];   // by rank (k is 256 at most)
    screen_row<T>(a, b, sX, first);
    if (threadIdx.x < 256) sBest[threadIdx.x] = 0;
    __syncthreads();
    screen_score<T>(a, sList, 0, count, sX);
    __syncthreads();
    screen_results<T>(a, b, sList, count, sBest, listed);
}

// A lower bound of the k-th largest of the workgroup's keys (0: dead ones, not counted), exact in its upper 24 bits; 0 where there are
// fewer than k.  Radix select, a byte at a time.  T: lanes; total: keys beyond that many are 0.  s: 258 words.
template <int N, int T = 256> __device__ __forceinline__ uint32_t block_kth_key(const uint32_t (&key)[N], uint32_t total, uint32_t k, uint32_t* s)
{
    uint32_t prefix = 0, need = k;
    for (int shift = 24; shift >= 8; shift -= 8) {
        if (threadIdx.x < 256) s[threadIdx.x] = 0;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < N; u++)
            if (u * T < total && key[u] != 0 && (shift == 24 || (key[u] >> (shift + 8)) == (prefix >> (shift + 8)))) atomicAdd(&s[(key[u] >> shift) & 255], 1u);
        __syncthreads();
        if (threadIdx.x < kWave) {
            const uint32_t lane = threadIdx.x;
            uint32_t h[4], sum = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                h[i] = s[4 * lane + i];
                sum += h[i];
            }
            uint32_t above = sum;   // of this lane's bins and all higher ones
#pragma unroll
            for (int d = 1; d < kWave; d *= 2) {
                const uint32_t up = __shfl_down(above, d);
                if (lane + d < kWave) above += up;
            }
            above -= sum;
            if (lane == 0 && above + sum < need) s[256] = 0xffffffffu;
            if (above < need && need <= above + sum) {
                uint32_t digit = 0, rest = need - above;
                bool found = false;
#pragma unroll
                for (int i = 3; i >= 0; i--) {
                    if (!found && rest <= h[i]) {
                        digit = 4 * lane + i;
                        found = true;
                    }
                    if (!found) rest -= h[i];
                }
                s[256] = digit;
                s[257] = rest;
            }
        }
        __syncthreads();
        if (s[256] == 0xffffffffu) return 0;   // (only in the first pass)
        prefix |= s[256] << shift;
        need = s[257];
    }
    return prefix;
}

// The k-th largest of 64 * N keys of a wavefront, exact but for its LAST lowest bits, 0 if there are fewer.  (As the top-K kernels' key search.)
template <int N, int LAST = 12> __device__ __forceinline__ uint32_t screen_wave_kth(const uint32_t (&key)[N], uint32_t k)
{
    uint32_t t = 0;
#pragma unroll 1
    for (int bit = 30; bit >= LAST; bit -= 2) {
        const uint32_t c1 = t | (1u << bit), c2 = t | (2u << bit), c3 = t | (3u << bit);
        uint32_t n1 = 0, n2 = 0, n3 = 0;
#pragma unroll
        for (int n = 0; n < N; n++) {
            n1 += (uint32_t)__popcll(__ballot(key[n] >= c1));
            n2 += (uint32_t)__popcll(__ballot(key[n] >= c2));
            n3 += (uint32_t)__popcll(__ballot(key[n] >= c3));
        }
        t = (n3 >= k) ? c3 : (n2 >= k) ? c2 : (n1 >= k) ? c1 : t;
    }
    return t;
}

enum { kPickFinal, kPickKeep };

// What a range's sums are compared with.
__device__ __forceinline__ uint32_t screen_admit(const ScreenFoldArgs& a, float cut, float e1)
{
    if (!a.largest) return score_key(cut);
    const float lowered = fmaf(-e1, *a.largest, cut);
    return score_key(lowered - (fabsf(lowered) + fabsf(cut)) * 2.4e-7f);   // (below what the roundings of the raised sum reach)
}

// Sums stored as halves: what reaches the bound.  The maxima of the row's blocks of 32 columns say which blocks can hold a result: the k-th
// of R maxima per lane (over blocks without a listed column, each less its width) bounds the k-th score, and only blocks whose largest
// sum reaches the bound are read.  Bound by latency: two round trips, a key search and, in the form that ends with the results, one
// round trip for the candidates' rows.  T lanes, E blocks each.  1,024 rows x 27,278 top 10, 144 listed columns each: 15.4 us; with all
// of the row in registers and the maxima taken from there, 27.6.
template <int T, int R, int E, int MODE>
__global__ __launch_bounds__(T, T == 256 ? 5 : 4) void screen_pick_kernel(ScreenFoldArgs a)
{
    __builtin_amdgcn_s_setprio(3);   // short kernels issue ahead of a GEMM's wavefronts that share their SIMD
    __shared__ uint64_t sList[kPickWords];
    __shared__ uint32_t sMax[R * T];
    __shared__ uint16_t sBlock[kPickBlocks];
    __shared__ uint32_t sHist[MODE == kPickFinal ? 258 : 1];
    __shared__ uint32_t sCount, sBlocks, sClean, sListed;
    __shared__ float sCut;
    extern __shared__ __attribute__((aligned(16))) uint32_t sDyn[];   // bitmap of the listed columns, a word a block; afterwards the row (kPickFinal)
    constexpr int C = E < 8 ? E : 8;
    static_assert(E * T <= 65536 && E % C == 0, "block numbers are 16 bits wide");
    const uint32_t b = blockIdx.x, lane = threadIdx.x % kWave;
    const uint32_t blocks = (a.stored + 31) / 32;
    if (a.row_flag[b] != 0) {
        if (MODE == kPickKeep && threadIdx.x == 0) {
            a.admit[b] = 0xffffffffu;
            a.keep_count[b] = 0;
        }
        return;
    }
    uint64_t fs = 0, fe = 0;
    if (a.fidx) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    const _Float16* src = a.Z + (uint64_t)b * a.ldz;
    const _Float16* maxima = a.M + (uint64_t)b * (a.ldz / 32);
    // blocks' maxima, and the largest norms of the 64 columns that they lie in: held, or asked for again, C blocks at a time
    _Float16 most[C];
    float norms[C];
    auto ask = [&](int from) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < C; e++) {
            const uint32_t i = min((from + e) * T + threadIdx.x, blocks - 1);
            most[e] = maxima[i];
            norms[e] = a.seg_norm[i / 2];
        }
    };
    if constexpr (C == E) ask(0);
    float first = 0.0f;
    if (MODE == kPickFinal && threadIdx.x < a.dim) first = a.X[(uint64_t)b * a.ldx + threadIdx.x];
    if (fe > fs)
        for (uint32_t i = threadIdx.x; i < blocks; i += T) sDyn[i] = 0;
    if (threadIdx.x == 0) sCount = sBlocks = sClean = sListed = 0;
    const float e1 = a.e1[b], e0 = a.e0[b], step = 1.0f / a.scale[b];   // (a power of two)
    __syncthreads();
    if (fe > fs) {
        bool any = false;
        for (uint64_t t = fs + threadIdx.x; t < fe; t += T) {
            const uint32_t c = a.fidx[t];
            if (c < a.stored) atomicOr(&sDyn[c >> 5], 1u << (c & 31));
            any |= c < a.n;
        }
        if (MODE == kPickFinal && __ballot(any) != 0 && lane == 0) atomicOr(&sListed, 1u);
        __syncthreads();
        // A block with a listed column has no part in the bound, unless too few others are left: then its other columns are looked at.
        uint32_t clean = 0;
#pragma unroll 4
        for (int e = 0; e < E; e++) clean += (uint32_t)__popcll(__ballot(e * T + threadIdx.x < blocks && sDyn[min(e * T + threadIdx.x, blocks - 1)] == 0));
        if (lane == 0) atomicAdd(&sClean, clean);
        __syncthreads();
    }
    const bool exact = fe > fs && sClean < min(4 * a.k, blocks);   // the same for the whole workgroup
    {
        float low[R];
#pragma unroll
        for (int i = 0; i < R; i++) low[i] = -__builtin_inff();
#pragma unroll 1
        for (int from = 0; from < E; from += C) {
            if (from * T >= blocks) break;
            if constexpr (C != E) ask(from);
#pragma unroll
            for (int u = 0; u < C; u++) {
                const uint32_t i = (from + u) * T + threadIdx.x, listed = (fe > fs && i < blocks) ? sDyn[i] : 0u;
                float m = (float)most[u];
                if (listed != 0) {
                    m = -65504.0f;
                    if (exact)
                        for (uint32_t c = 0; c < 32; c += 8) {
                            const half8 z = *reinterpret_cast<const half8*>(src + (uint64_t)i * 32 + c);
#pragma unroll
                            for (int x = 0; x < 8; x++)
                                if (!((listed >> (c + x)) & 1u)) m = fmaxf(m, (float)z[x]);
                        }
                }
                const float norm = norms[u], raised = fmaf(m, step, e1 * norm);
                // (what does not fit a half says nothing: rounded up to infinity, or held at the lowest half)
                if (i < blocks && m < 65504.0f && m > -65504.0f) low[u % R] = fmaxf(low[u % R], raised - screen_width(a, raised, norm, e1, e0, step));
            }
        }
#pragma unroll
        for (int i = 0; i < R; i++) sMax[i * T + threadIdx.x] = score_key(low[i]);
    }
    __syncthreads();
    // (one wavefront searches, a different one from row to row, so that the four SIMDs of a compute unit share the searches)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave) == ((b >> 8) & 3u)) {
        constexpr int K = R * T / kWave;
        uint32_t all[K];
#pragma unroll
        for (int i = 0; i < K; i++) all[i] = sMax[i * kWave + lane];
        const uint32_t t = screen_wave_kth<K>(all, a.k);
        if (lane == 0) sCut = screen_cut(a, t > score_key(-__builtin_inff()) ? key_score(t) : -__builtin_inff(), e0);
    }
    __syncthreads();
    const float cut = sCut;
#pragma unroll 1
    for (int from = 0; from < E; from += C) {
        if (from * T >= blocks) break;
        if constexpr (C != E) ask(from);
#pragma unroll
        for (int u = 0; u < C; u++) {
            const uint32_t i = (from + u) * T + threadIdx.x;
            const bool hot = i < blocks && fmaf((float)most[u], step, e1 * norms[u]) >= cut;
            const uint64_t m = __ballot(hot);
            if (m == 0) continue;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&sBlocks, (uint32_t)__popcll(m));
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (hot && at < kPickBlocks) sBlock[at] = (uint16_t)i;
        }
    }
    __syncthreads();
    const uint32_t hot_blocks = sBlocks;
    const bool many = hot_blocks > kPickBlocks;   // (thousands of tied scores: the row is given up below)
    // four lanes a block, eight columns each
    for (uint32_t p0 = 0; p0 < hot_blocks && !many; p0 += T / 4) {
        const uint32_t p = p0 + threadIdx.x / 4;
        const uint32_t block = sBlock[min(p, hot_blocks - 1)], c0 = block * 32 + threadIdx.x % 4 * 8;
        half8 z = {};
        if (p < hot_blocks) z = *reinterpret_cast<const half8*>(src + c0);   // (rows of Z are padded to whole tiles)
        const float raise = e1 * a.seg_norm[block / 2];
        uint32_t listed = (fe > fs) ? sDyn[block] >> (threadIdx.x % 4 * 8) : 0u;
        if (p >= hot_blocks) listed = 0xffu;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float h = (float)z[e];
            const bool ok = fmaf(h, step, raise) >= cut && c0 + e < a.stored && !((listed >> e) & 1u);
            const uint64_t m = __ballot(ok);
            if (m == 0) continue;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&sCount, (uint32_t)__popcll(m));
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (ok && at < kPickWords) sList[at] = ((uint64_t)score_key(h * step) << 32) | (uint32_t)~(c0 + e);   // (not raised: screen_raised)
        }
    }
    __syncthreads();
    const uint32_t count = sCount;
    if (many || count > (MODE == kPickKeep ? kKeepWords : kPickWords)) {   // the same for the whole workgroup
        if (threadIdx.x == 0) {
            screen_flag(a, b);
            if constexpr (MODE == kPickKeep) a.keep_count[b] = 0;
        }
        return;
    }
    if constexpr (MODE == kPickKeep) {
        for (uint32_t i = threadIdx.x; i < count; i += T) a.keep[(uint64_t)b * kKeepWords + i] = screen_raised(a, sList[i], e1);
        if (threadIdx.x == 0) {
            a.keep_count[b] = count;
            a.admit[b] = screen_admit(a, cut, e1);
        }
    } else {
        // With many candidates of long rows, the k-th of the candidates' own bounds (by column and not by block) first: a third of them go.
        uint32_t left = count;
        if (a.k > 32 && a.dim >= 256 && count > a.k) {   // the same for the whole workgroup
            constexpr int W = kPickWords / T;
            uint64_t word[W];
            uint32_t low[W];
#pragma unroll
            for (int u = 0; u < W; u++) {
                const uint32_t i = u * T + threadIdx.x;
                word[u] = 0;
                low[u] = 0;
                if (i >= count) continue;
                word[u] = screen_raised(a, sList[i], e1);
                const float z = key_score((uint32_t)(word[u] >> 32)), l = z - screen_width(a, z, a.norm[~(uint32_t)word[u]], e1, e0, step);
                low[u] = (l > -__builtin_inff()) ? score_key(l) : 0u;
            }
            const uint32_t t = block_kth_key<W, T>(low, count, a.k, sHist);
            if (threadIdx.x == 0) {
                sCut = screen_cut(a, t != 0 ? key_score(t) : -__builtin_inff(), e0);
                sCount = 0;
            }
            __syncthreads();
            const float closer = sCut;
#pragma unroll
            for (int u = 0; u < W; u++)
                if (word[u] != 0 && key_score((uint32_t)(word[u] >> 32)) >= closer) sList[atomicAdd(&sCount, 1u)] = word[u];
            __syncthreads();
            left = sCount;
        }
        screen_finish<T>(a, b, sList, left, reinterpret_cast<float*>(sDyn), first, sListed != 0);
    }
}

// A column range's lists, and what earlier ranges left: the listed columns struck out, cut back to what can still be a result, and the
// bound for the next range; in the last one (FINAL) scored and written.
template <bool FINAL>
__global__ __launch_bounds__(256, 4) void screen_fold_kernel(ScreenFoldArgs a)
{
    __builtin_amdgcn_s_setprio(3);
    constexpr int NW = 8;   // words per lane at a time
    constexpr uint32_t kSlots = 4096;
    constexpr uint32_t kEmpty = 0xffffffffu;   // (no column has this number: widths stay below 2^32 - 2)
    __shared__ uint32_t sTable[kSlots];        // listed columns
    constexpr uint32_t room = FINAL ? kPickWords : kKeepWords;
    __shared__ uint64_t left[room];            // candidates that are left
    __shared__ uint32_t sStart[257];
    __shared__ uint32_t sHist[258];
    __shared__ uint32_t sCount, sWave[4];
    __shared__ float sCut;
    extern __shared__ __attribute__((aligned(16))) uint32_t sDyn[];   // the row (FINAL)
    const uint32_t b = blockIdx.x, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t shared = a.cand_count[b];
    const bool flagged = a.row_flag[b] != 0;
    uint32_t incl = (threadIdx.x < a.lists) ? min(a.seg_count[(uint64_t)b * kF16ListStride + threadIdx.x], a.seg_cap) : 0u;
    const uint32_t kept = a.keep_count[b];
    const float e1 = a.e1[b], e0 = a.e0[b], step = 1.0f / a.scale[b];
    uint64_t fs = 0, fe = 0;
    if (a.fidx) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
        const uint32_t below = __shfl_up(incl, d);
        if (lane >= (uint32_t)d) incl += below;
    }
    if (lane == kWave - 1) sWave[wave] = incl;
    if (threadIdx.x == 0) {
        sStart[0] = 0;
        sCount = 0;
    }
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; w++) before += sWave[w];
    sStart[threadIdx.x + 1] = before + incl;
    __syncthreads();
    if (threadIdx.x == 0) a.cand_count[b] = 0;
    if (flagged) return;
    const uint32_t in_lists = sStart[256], fresh_words = shared + in_lists, total = kept + fresh_words;
    if (shared > a.cap) {   // (the lists of a row's own hold as many again)
        if (threadIdx.x == 0) screen_flag(a, b);
        return;
    }
    auto where = [&](uint32_t e) -> const uint64_t* {
        if (e < kept) return a.keep + (uint64_t)b * kKeepWords + e;
        if (e < kept + shared) return a.cand + (uint64_t)b * a.cap + (e - kept);
        const uint32_t s = e - kept - shared;
        uint32_t l = 0, h = 256;   // the last list that starts at or before s (empty ones start where the next one does)
        while (h - l > 1) {
            const uint32_t mid = (l + h) / 2;
            if (sStart[mid] <= s) l = mid;
            else h = mid;
        }
        return a.seg + ((uint64_t)b * a.lists + l) * a.seg_cap + (s - sStart[l]);
    };
    // Up to 2,048 words at a time (most rows: once), what is left of the ones before among them.  The listed columns go, 2,048 at a time,
    // into a table (at most half full, linear probing) that new words are looked up in.  Of a word its key and that of what its
    // score lies above stay in registers (0: none).
    uint32_t carried = 0;
    for (uint32_t pos = 0;;) {
        const uint32_t fresh = min(total - pos, (uint32_t)NW * 256 - carried), here = carried + fresh;
        uint32_t key[NW], low[NW], col[NW];
        uint64_t f0 = fs;
        bool first = true;
        do {
            const uint32_t some = (uint32_t)min((uint64_t)(kSlots / 2), fe - f0);
            uint32_t bits = 6;
            while ((1u << bits) < 2 * some) bits++;
            const uint32_t mask = (1u << bits) - 1, shift = 32 - bits;
            if (some != 0 && (pos == 0 || fe - fs > kSlots / 2)) {
                if (!first || pos != 0) __syncthreads();
                for (uint32_t i = threadIdx.x; i <= mask; i += 256) sTable[i] = kEmpty;
                __syncthreads();
                for (uint32_t i = threadIdx.x; i < some; i += 256) {
                    const uint32_t c = a.fidx[f0 + i];
                    uint32_t h = (c * 2654435761u) >> shift;
                    for (;;) {   // (a column listed twice takes one place)
                        const uint32_t was = atomicCAS(&sTable[h], kEmpty, c);
                        if (was == kEmpty || was == c) break;
                        h = (h + 1) & mask;
                    }
                }
                __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < NW; u++) {
                const uint32_t i = u * 256 + threadIdx.x;
                if (first) key[u] = low[u] = col[u] = 0;
                if (u * 256 >= here || i >= here || (!first && key[u] == 0)) continue;
                const uint32_t e = pos + (i - carried);
                const bool new_word = i >= carried && e >= kept;
                if (first) {
                    uint64_t word = (i < carried) ? left[i] : *where(e);
                    if (word == 0) continue;
                    col[u] = ~(uint32_t)word;
                    const float norm = a.norm[col[u]];
                    if (new_word) word = screen_raised(a, word, e1);
                    const float z = key_score((uint32_t)(word >> 32)), l = z - screen_width(a, z, norm, e1, e0, step);
                    key[u] = (uint32_t)(word >> 32);
                    low[u] = (l > -__builtin_inff()) ? score_key(l) : 0u;   // (an infinite sum, and one of an infinite norm, says nothing)
                }
                if (some != 0 && new_word) {
                    uint32_t h = (col[u] * 2654435761u) >> shift;
                    for (;;) {
                        const uint32_t v = sTable[h];
                        if (v == kEmpty) break;
                        if (v == col[u]) {
                            key[u] = low[u] = 0;
                            break;
                        }
                        h = (h + 1) & mask;
                    }
                }
            }
            f0 += some;
            first = false;
        } while (f0 < fe);
        pos += fresh;
        const uint32_t t = block_kth_key<NW>(low, here, a.k, sHist);   // (its barriers: every lane has its words)
        if (threadIdx.x == 0) {
            sCut = screen_cut(a, t != 0 ? key_score(t) : -__builtin_inff(), e0);
            sCount = 0;
        }
        __syncthreads();
        const float cut = sCut;
#pragma unroll
        for (int u = 0; u < NW; u++) {
            if (u * 256 >= here) continue;
            const bool ok = key[u] != 0 && key_score(key[u]) >= cut;
            const uint64_t m = __ballot(ok);
            if (m == 0) continue;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&sCount, (uint32_t)__popcll(m));
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (ok && at < room) left[at] = ((uint64_t)key[u] << 32) | (uint32_t)~col[u];
        }
        __syncthreads();
        carried = sCount;
        if (carried > (pos < total ? min(room, NW * 256u - 256u) : room)) {   // the same for the whole workgroup
            if (threadIdx.x == 0) screen_flag(a, b);
            return;
        }
        if (pos >= total) break;
        __syncthreads();
    }
    const uint32_t count = carried;
    if constexpr (FINAL) {
        float x = 0.0f;
        if (threadIdx.x < a.dim) x = a.X[(uint64_t)b * a.ldx + threadIdx.x];
        bool any = false;
        for (uint64_t t = fs + threadIdx.x; t < fe; t += 256) any |= a.fidx[t] < a.n;
        screen_finish<256>(a, b, left, count, reinterpret_cast<float*>(sDyn), x, __syncthreads_or(any) != 0);
    } else {
        for (uint32_t i = threadIdx.x; i < count; i += 256) a.keep[(uint64_t)b * kKeepWords + i] = left[i];
        if (threadIdx.x == 0) {
            a.keep_count[b] = count;
            a.admit[b] = screen_admit(a, sCut, e1);
        }
    }
}

constexpr uint32_t kBestWords = 2048;    // candidates of a row at a time
constexpr uint32_t kBestMost = 16384;    // candidates of a row beyond the first k (and as many as it has listed columns): with more it is left open
constexpr uint32_t kBestColumns = 1u << 20;
constexpr uint32_t kNearWords = 4096;    // words of a row that are listed
constexpr uint32_t kAloneColumns = 32768;   // up to here i8_finish_kernel looks through a row's words itself

// Sums of bytes: a word for every 32 columns says what the largest of their sums is at most, whose it is, and what the others are at most.  The columns
// of the k largest words are scored first; then all columns whose words reach the k-th of those scores, and where the others of a block
// reach it, all of the block.  So a row's bound is a score and not an estimate of one: e1 |w| + e2 |w's rest| is open on one side of it only.
//
// Two kernels.  i8_near_kernel reads a row's words, once, and lists those that can reach the bound whatever it will be: the k-th word less twice the
// largest error, where the activation is not flat.  i8_finish_kernel scores.  (In one kernel of sixteen wavefronts a row, 604 us for 4,096 rows of 1,000,000 columns, 128 components and 100
// results, 137 + 177 so: two rows to a compute unit, and all sixteen wavefronts went through the searches and lists of a few hundred words.)
struct I8NearArgs {
    uint32_t batch, k, n;
    const uint32_t* words;
    uint64_t ldw;
    const float4* error_rows;
    const float* unit;       // the rows', by the rows' scale
    const float4* error_most;   // I8ItemsArgs::error_most
    uint32_t act;
    float slope, alpha, lambda;
    const uint32_t* row_flag;
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;
    uint2* near;             // [batch][kNearWords] block (kNearDead: its largest sum is a listed column's) and word, as an integer in the order of halves
    uint2* near_found;       // [batch] how many there are; the word that k columns reach and the least that is listed (upper halves)
};
constexpr uint32_t kNearDead = 0x80000000u;
constexpr int32_t kNoWord = INT32_MIN;

// A word as an integer in the order of its first half, and back.
__device__ __forceinline__ int32_t i8_sortable(int32_t word) { return word ^ ((word >> 31) & 0x7fff0000); }

// A row per workgroup, 4 V words a lane.  Bound by reading them: their first halves alone stay in registers, two in one, so that three or four rows
// are on a compute unit; what is listed is read once more.  4,096 rows x 1,000,000 columns: 137 us, 3.7 TB/s (255 with whole words in registers, two rows to a compute
// unit; 191 with four rows and 88 bytes of scratch a lane).
// V: reads a lane; R: registers of keys that a lane has in the search; ROOM: words that out has room for.  Returns near_found's two; any: whether this lane saw
// a listed column.
template <int V, int T, int R, uint32_t ROOM> __device__ __forceinline__ uint2 i8_near(const I8NearArgs& a, uint32_t b, uint2* out, bool& any)
{
    constexpr int B = V * T * 4 / 32;   // words of a bitmap of blocks
    typedef int16_t short2v __attribute__((ext_vector_type(2)));
    __shared__ uint32_t sDead[B], sTop[2 * R * T];
    __shared__ uint16_t sNear[ROOM];
    __shared__ uint32_t sNears, sKth;
    __shared__ int32_t sNearest;
    const uint32_t tid = threadIdx.x;
    const uint32_t blocks = (a.n + 31) / 32;
    const uint32_t* words = a.words + (uint64_t)b * a.ldw;
    uint64_t fs = 0, fe = 0;
    if (a.fidx) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    const float4 error = a.error_rows[b];
    const float4 most = *a.error_most;
    if (tid == 0) sNears = 0;
    const bool some_dead = fe > fs || a.n % 256 != 0;   // the same for the workgroup
    if (some_dead) {
        for (uint32_t i = tid; i < B; i += T) sDead[i] = (i + 1) * 32 <= blocks ? 0u : i * 32 >= blocks ? ~0u : ~0u << (blocks % 32);   // (no blocks)
        __syncthreads();
        for (uint64_t t = fs + tid; t < fe; t += T) {
            const uint32_t c = a.fidx[t];
            any |= c < a.n;
            if (c < a.n && (words[c >> 5] & 31u) == (c & 31u)) atomicOr(&sDead[c >> 10], 1u << ((c >> 5) & 31u));
        }
        // (the largest sum of the last block may be one of a column beyond it)
        if (tid == 0 && a.n % 32 != 0 && (words[blocks - 1] & 31u) >= a.n % 32) atomicOr(&sDead[(blocks - 1) >> 5], 1u << ((blocks - 1) & 31u));
        __syncthreads();
    }
    // Halves in the order of integers of 16 bits, blocks 4 q and 4 q + 1 in one register, the next two in another; -32768: no words.
    short2v held[2 * V];
    constexpr int G = V < 4 ? V : 4;   // reads in flight
#pragma unroll
    for (int g = 0; g < V; g += G) {
        uint4 w[G];
#pragma unroll
        for (int v = 0; v < G; v++) {
            const uint32_t at = ((g + v) * T + tid) * 4;
            w[v] = make_uint4(~0u, ~0u, ~0u, ~0u);   // (in that order the least half)
            if (at < a.ldw) w[v] = *reinterpret_cast<const uint4*>(words + at);   // (ldw is a multiple of 8)
        }
#pragma unroll
        for (int v = 0; v < G; v++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const short2v x = __builtin_bit_cast(short2v, h ? __builtin_amdgcn_perm(w[v].w, w[v].z, 0x07060302u) : __builtin_amdgcn_perm(w[v].y, w[v].x, 0x07060302u));
                held[2 * (g + v) + h] = x ^ ((x >> (short2v){15, 15}) & (short2v){0x7fff, 0x7fff});
            }
        asm volatile("" ::: "memory");   // (no more reads in flight than that: the halves have the registers)
    }
    // (An infinite half says nothing of its column's score - a norm that f16 does not hold, a sum that a half does not - so it counts for no bound: raised
    // by kUp, the numbers stay in order and infinity becomes the least.)
    constexpr short kUp = 0x400;
    typedef uint16_t ushort2v __attribute__((ext_vector_type(2)));
    auto up = [](short2v x) __attribute__((always_inline)) { return __builtin_bit_cast(short2v, __builtin_bit_cast(ushort2v, x) + (ushort2v){kUp, kUp}); };
    short2v top[R];
#pragma unroll
    for (int r = 0; r < R; r++) top[r] = short2v{INT16_MIN, INT16_MIN};
    if (!some_dead) {
#pragma unroll
        for (int e = 0; e < 2 * V; e++) top[e % R] = __builtin_elementwise_max(top[e % R], up(held[e]));
    } else {
#pragma unroll
        for (int e = 0; e < 2 * V; e++) {
            const uint32_t q = e / 2 * T + tid, dead = sDead[q / 8] >> (q % 8 * 4 + e % 2 * 2);
            short2v x = up(held[e]);
            if (dead & 1u) x[0] = INT16_MIN;
            if (dead & 2u) x[1] = INT16_MIN;
            top[e % R] = __builtin_elementwise_max(top[e % R], x);
        }
    }
    // One wavefront searches.  The k-th of the lanes' largest is a word that k columns reach, and seldom much below the k-th of all.
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int x = top[r][h];
            sTop[(2 * r + h) * T + tid] = x > INT16_MIN + kUp ? ((uint32_t)(x - kUp) << 16) ^ 0x80000000u : 0u;
        }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(tid / kWave) == (b >> 8) % (T / kWave)) {
        // (as screen_wave_kth, but for the keys, which stay in LDS)
        uint32_t t = 0;
#pragma unroll 1
        for (int bit = 30; bit >= 16; bit -= 2) {
            const uint32_t c1 = t | (1u << bit), c2 = t | (2u << bit), c3 = t | (3u << bit);
            uint32_t n1 = 0, n2 = 0, n3 = 0;
#pragma unroll 8
            for (int i = 0; i < 2 * R * T / kWave; i++) {
                const uint32_t key = sTop[i * kWave + tid % kWave];
                n1 += (uint32_t)__popcll(__ballot(key >= c1));
                n2 += (uint32_t)__popcll(__ballot(key >= c2));
                n3 += (uint32_t)__popcll(__ballot(key >= c3));
            }
            t = (n3 >= a.k) ? c3 : (n2 >= a.k) ? c2 : (n1 >= a.k) ? c1 : t;
        }
        // What can reach the bound, whatever it will be.  The k columns' sums lie no further below their words than what a word is raised by and the
        // error; their scores, the sums activated, are what another column's score has to reach, and its word lies no further below that than the error.
        int32_t near = kNoWord + 0x10000;   // (everything)
        if (t != 0) {
            const float step = error.w, z = i8_first((uint32_t)i8_sortable((int32_t)(t ^ 0x80000000u))) * step, wide = 1.01f * fmaf(error.x, most.x, error.y * most.y);
            const float low = z - fabsf(z) * 1.0e-3f - 2e-7f * step - 50.0f * (a.unit[b] * step) * most.w - wide - error.z;
            // (i8_finish_kernel knows its k-th key but for the lowest 8 bits)
            const float cut = low > -__builtin_inff() ? screen_cut_key(a, score_key(activate_rt(low, a.act, a.slope, a.alpha, a.lambda)) & ~255u, error.z) : low;
            const float least = (cut - wide) / step;
            if (least > -65000.0f && z < 60000.0f * step) {
                const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)(least - fabsf(least) * 1.0e-3f - 1.2e-7f));
                near = i8_sortable((int32_t)(h << 16));
            }
        }
        if (tid % kWave == 0) {
            sKth = t;
            sNearest = near;
        }
    }
    __syncthreads();
    const uint32_t kth = sKth;
    const int32_t t0 = kth != 0 ? (int32_t)(kth ^ 0x80000000u) : kNoWord + 1;
    int32_t near = sNearest;
    auto listed = [&](int e) __attribute__((always_inline)) -> bool {   // the lane's e-th block (in registers)
        const uint32_t two = __builtin_bit_cast(uint32_t, held[e / 2]);
        return (int32_t)(e % 2 ? two & 0xffff0000u : two << 16) >= near;
    };
    uint32_t mine = 0;
#pragma unroll
    for (int e = 0; e < 4 * V; e++) mine += listed(e);
    uint32_t at = mine;
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
        const uint32_t below = __shfl_up(at, d);
        if (tid % kWave >= (uint32_t)d) at += below;
    }
    uint32_t base = 0;
    if (tid % kWave == kWave - 1) base = atomicAdd(&sNears, at);
    at += __shfl(base, kWave - 1) - mine;
    asm volatile("" : "+v"(near));   // (compared again: the results of the comparisons above would not fit the scalar registers)
#pragma unroll
    for (int e = 0; e < 4 * V; e++)
        if (listed(e)) {
            if (at < ROOM) sNear[at] = (uint16_t)((e / 4 * T + tid) * 4 + e % 4);
            at++;
        }
    __syncthreads();
    const uint32_t nears = sNears;
    if (nears <= ROOM)
        for (uint32_t i = tid; i < nears; i += T) {
            const uint32_t block = sNear[i], dead = some_dead ? (sDead[block >> 5] >> (block & 31u) & 1u) * kNearDead : 0u;
            out[i] = make_uint2(block | dead, (uint32_t)i8_sortable((int32_t)words[block]));
        }
    return make_uint2(nears, ((uint32_t)t0 & 0xffff0000u) | (uint32_t)sNearest >> 16);
}

template <int V>
__global__ __launch_bounds__(512, V == 16 ? 6 : 8) void i8_near_kernel(I8NearArgs a)
{
    __builtin_amdgcn_s_setprio(3);
    const uint32_t b = blockIdx.x;
    if (a.row_flag[b] != 0) return;
    bool any = false;
    const uint2 found = i8_near<V, 512, 1, kNearWords>(a, b, a.near + (uint64_t)b * kNearWords, any);
    if (threadIdx.x == 0) a.near_found[b] = found;
}

// The k-th largest key of the list's first `count` words (256 * N at most), exact but for the lowest 8 bits; 0: fewer.  The wavefront that calls it.
template <int N> __device__ __forceinline__ uint32_t list_kth(const uint64_t* sList, uint32_t count, uint32_t k)
{
    uint32_t key[N];
#pragma unroll
    for (int i = 0; i < N; i++) key[i] = (i * kWave + threadIdx.x < count) ? (uint32_t)(sList[i * kWave + threadIdx.x] >> 32) : 0u;
    return screen_wave_kth<N, 8>(key, k);
}

// A row per workgroup; several of them to a compute unit hide each other's latency: candidates' rows, twice, and a search after each.  Nothing fills up:
// what a round's list has no room for comes with the next one, against a bound that only rises.
// NEAR: not 0 for up to 32,768 columns, whose words this workgroup looks through itself (NEAR registers of keys a lane): both kernels are bound by latency
// then (4,096 and 1,904 rows x 1,024 x 27,278 top 10 with a filter, two batches: 806 us with two kernels, 727 so).
template <bool HALVES, int NEAR>
__global__ __launch_bounds__(256, 4) void i8_finish_kernel(ScreenFoldArgs a, I8NearArgs e)
{
    __builtin_amdgcn_s_setprio(3);
    constexpr int T = 256, B = NEAR ? T * 4 / 32 : kBestColumns / 32 / 32;
    __shared__ uint2 sNearWords[NEAR ? T * 4 : 1];
    constexpr uint32_t kOpen = 32;               // blocks of which all columns are looked at, per round
    __shared__ uint64_t sList[kBestWords];
    __shared__ uint64_t sBest[256];
    __shared__ uint32_t sDead[B], sHot[B], sMore[B];   // blocks whose largest sum is a listed column's (for `all`); is one to be scored; of which the others are
    __shared__ uint32_t sHist[258];
    __shared__ uint32_t sOpen[kOpen], sMask[kOpen];
    __shared__ uint32_t sCount, sOpened, sKth, sAhead;
    extern __shared__ __attribute__((aligned(16))) uint32_t sDyn[];   // the row
    float* sX = reinterpret_cast<float*>(sDyn);
    const uint32_t b = blockIdx.x, tid = threadIdx.x;
    if (a.row_flag[b] != 0) return;
    const uint32_t blocks = (a.n + 31) / 32, bitmap = (blocks + 31) / 32;
    const uint32_t* words = a.words + (uint64_t)b * a.ldw;
    const uint2* near = NEAR ? sNearWords : a.near + (uint64_t)b * kNearWords;
    uint64_t fs = 0, fe = 0;
    if (a.fidx) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    const float4 error = a.error_rows[b];
    const float e1 = error.x, e2 = error.y, e0 = error.z, step = error.w;
    const float first = (tid < a.dim) ? a.X[(uint64_t)b * a.ldx + tid] : 0.0f;
    for (uint32_t i = tid; i < bitmap; i += T) sHot[i] = sMore[i] = 0;
    sBest[tid] = 0;
    if (tid == 0) sCount = sAhead = 0;
    if constexpr (HALVES) screen_row_halves<T>(a, b, reinterpret_cast<_Float16*>(sDyn), first);
    else screen_row<T>(a, b, sX, first);
    bool any = false;
    uint2 found;
    if constexpr (NEAR != 0) found = i8_near<1, T, NEAR, T * 4>(e, b, sNearWords, any);
    else {
        found = a.near_found[b];
        for (uint64_t t = fs + tid; t < fe; t += T) any |= a.fidx[t] < a.n;
    }
    const bool listed = __syncthreads_or(any) != 0;
    if (!(e1 == e1)) {   // a row that is no number has no scores
        screen_results<T>(a, b, sList, 0, sBest, listed);
        return;
    }
    const uint32_t nears = found.x;
    const int32_t t0 = (int32_t)(found.y & 0xffff0000u), least = (int32_t)(found.y << 16);
    const bool all = NEAR ? false : nears > kNearWords;   // (more than there was room for: the words are read again; the same for the whole workgroup, as are all of these)
    if (all) {
        for (uint32_t i = tid; i < bitmap; i += T) sDead[i] = 0;
        __syncthreads();
        for (uint64_t t = fs + tid; t < fe; t += T) {
            const uint32_t c = a.fidx[t];
            if (c < a.n && (words[c >> 5] & 31u) == (c & 31u)) atomicOr(&sDead[c >> 10], 1u << ((c >> 5) & 31u));
        }
        if (tid == 0 && a.n % 32 != 0 && (words[blocks - 1] & 31u) >= a.n % 32) atomicOr(&sDead[(blocks - 1) >> 5], 1u << ((blocks - 1) & 31u));
        __syncthreads();
    }
    // Every block that can reach the bound, with its word in the order of integers (and its errors), eight a lane at a time: their loads are waited
    // for together.
    auto each = [&](auto errors, auto&& look) __attribute__((always_inline)) {
        constexpr int G = 8;
        const uint32_t total = all ? blocks : nears;
        for (uint32_t base = tid; base < total; base += G * T) {
            uint2 x[G];
            float2 e[G];
#pragma unroll
            for (int g = 0; g < G; g++) {
                const uint32_t i = base + g * T;
                x[g] = make_uint2(0, (uint32_t)kNoWord);
                if (g == 0 || i < total) x[g] = all ? make_uint2(i, words[i]) : near[i];
            }
            if constexpr (errors.value) {
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (g == 0 || base + g * T < total) e[g] = a.error_items[(x[g].x & ~kNearDead) / 4];
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                if (base + g * T >= total) break;
                const uint32_t block = x[g].x & ~kNearDead;
                look(block, all ? i8_sortable((int32_t)x[g].y) : (int32_t)x[g].y, all ? ((sDead[block >> 5] >> (block & 31u)) & 1u) != 0 : (x[g].x & kNearDead) != 0, e[g]);
            }
        }
    };
    each(std::false_type{}, [&](uint32_t block, int32_t x, bool dead, float2) {
        if (x >= t0 && !dead) {
            const uint32_t at = atomicAdd(&sCount, 1u);
            if (at < kBestWords) sList[at] = (uint32_t)~(block * 32 + ((uint32_t)x & 31u));
        }
    });
    __syncthreads();
    uint32_t count = sCount, kept = 0;
    if (count > kBestWords) {
        if (tid == 0) screen_open(a, b);
        return;
    }
    float cut = 0.0f;
    bool begun = false;
    constexpr int W = (B + T - 1) / T;
    uint32_t hot[W], more[W];
    for (;;) {
        // Scores of what is new, and what is left of the list: what is no worse than its k-th.
        if constexpr (HALVES) screen_score_halves<T>(a, sList, kept, count, reinterpret_cast<const _Float16*>(sDyn));
        else screen_score<T, 4>(a, sList, kept, count, sX);
        __syncthreads();
        constexpr int L = kBestWords / T;
        uint64_t word[L];
        uint32_t key[L];
#pragma unroll
        for (int u = 0; u < L; u++) {
            word[u] = (u * T + tid < count) ? sList[u * T + tid] : 0ull;
            key[u] = (uint32_t)(word[u] >> 32);
        }
        uint32_t t;
        if (count <= 8 * kWave) {
            if (tid < kWave) {
                t = count <= 2 * kWave ? list_kth<2>(sList, count, a.k) : count <= 4 * kWave ? list_kth<4>(sList, count, a.k) : list_kth<8>(sList, count, a.k);
                if (tid == 0) sKth = t;
            }
            __syncthreads();
            t = sKth;
        } else t = block_kth_key<L, T>(key, count, a.k, sHist);   // (its barriers: every lane has its words)
        if (tid == 0) sCount = 0;
        cut = (t != 0) ? screen_cut_key(a, t, e0) : -__builtin_inff();
        __syncthreads();
#pragma unroll
        for (int u = 0; u < L; u++)
            if (word[u] != 0 && key[u] >= t) sList[atomicAdd(&sCount, 1u)] = word[u];
        __syncthreads();
        kept = sCount;
        if (!begun) {
            begun = true;
            // What is listed was decided by words; now that there are scores it is known whether it was enough.  (A column of the k without a score,
            // a sum that was raised by more than it should have been.)
            const float4 most = *e.error_most;
            if (!all && least > kNoWord + 0x10000 && fmaf(i8_first((uint32_t)i8_sortable(least)), step, fmaf(e1, most.x, e2 * most.y) * 1.000001f) >= cut) {
                if (tid == 0) screen_open(a, b);
                return;
            }
            each(std::true_type{}, [&](uint32_t block, int32_t x, bool dead, float2 e) {
                const float wide = fmaf(e1, e.x, e2 * e.y) * 1.000001f;
                const uint32_t word = (uint32_t)i8_sortable(x);
                if (!(fmaf(i8_first(word), step, wide) >= cut)) return;
                if (x < t0 && !dead) atomicOr(&sHot[block >> 5], 1u << (block & 31u));
                if (fmaf(i8_second(word), step, wide) >= cut) atomicOr(&sMore[block >> 5], 1u << (block & 31u));
            });
            __syncthreads();
#pragma unroll
            for (int u = 0; u < W; u++) {
                const uint32_t i = u * T + tid;
                hot[u] = i < bitmap ? sHot[i] : 0u;
                more[u] = i < bitmap ? sMore[i] : 0u;
            }
            // All of that will be scored but for listed columns and those behind the last one.
            uint32_t ahead = 0;
#pragma unroll
            for (int u = 0; u < W; u++) ahead += (uint32_t)__popc(hot[u]) + 31 * (uint32_t)__popc(more[u]);
            if (ahead != 0) atomicAdd(&sAhead, ahead);
        }
        uint32_t pending = 0;
#pragma unroll
        for (int u = 0; u < W; u++) pending |= hot[u] | more[u];
        if (tid == 0) sOpened = 0;
        if (!__syncthreads_or(pending != 0)) break;
        // (what is too much is not begun: 1,000,000 x 128 along one direction, 4,096 queries, top 10, given up behind the limit 7.9 ms with the search in halves,
        // 3.3 so)
        if (sAhead > kBestMost + (fe - fs) || kept > kBestWords / 2) {
            if (tid == 0) screen_open(a, b);
            return;
        }
#pragma unroll
        for (int u = 0; u < W; u++)
            while (hot[u] != 0) {
                const uint32_t at = atomicAdd(&sCount, 1u);
                if (at >= kBestWords) break;
                const uint32_t block = (u * T + tid) * 32 + (uint32_t)__builtin_ctz(hot[u]);
                sList[at] = (uint32_t)~(block * 32 + (words[block] & 31u));
                hot[u] &= hot[u] - 1;
            }
        __syncthreads();
        count = min(sCount, kBestWords);
        __syncthreads();
        if (count <= kBestWords - kOpen * 32) {
#pragma unroll
            for (int u = 0; u < W; u++)
                while (more[u] != 0) {
                    const uint32_t at = atomicAdd(&sOpened, 1u);
                    if (at >= kOpen) break;
                    const uint32_t block = (u * T + tid) * 32 + (uint32_t)__builtin_ctz(more[u]);
                    sOpen[at] = block;
                    sMask[at] = 1u << (words[block] & 31u);   // (scored, or not wanted)
                    more[u] &= more[u] - 1;
                }
            __syncthreads();
            const uint32_t opened = min(sOpened, kOpen);
            if (opened != 0) {
                for (uint64_t t = fs + tid; t < fe; t += T) {
                    const uint32_t c = a.fidx[t];
                    for (uint32_t o = 0; o < opened; o++)
                        if (sOpen[o] == c >> 5) atomicOr(&sMask[o], 1u << (c & 31u));
                }
                __syncthreads();
                for (uint32_t i = tid; i < opened * 32; i += T) {
                    const uint32_t col = sOpen[i / 32] * 32 + i % 32;
                    if (!((sMask[i / 32] >> (i % 32)) & 1u) && col < a.n) sList[atomicAdd(&sCount, 1u)] = (uint32_t)~col;
                }
                __syncthreads();
                count = min(sCount, kBestWords);
                __syncthreads();
            }
        }
    }
    screen_results<T>(a, b, sList, kept, sBest, listed);
}

// What can be screened with copies of the table made in the call: the preparation costs what about 130 rows' fp32 products do.  Limits: the row in LDS,
// and 8 GiB for the two copies.  A layer that is taken is faster so than in fp32 ranges: 714 calls of dsx_fc_topk, 512 to 4,096 rows, 64 to 1,024
// components, 16,384 to 1,000,000 columns, k 10 to 256, with and without a filter, take 0.16 to 0.81 of the time (us, fp32 / screened: 512 x 1,024 x
// 40,000 top 10 397 / 310, 512 x 256 x 16,384 top 10 87 / 67, 1,024 x 128 x 65,536 top 100 363 / 133, 4,096 x 1,024 x 27,278 top 256 2,552 / 920,
// 4,096 x 512 x 1,000,000 top 10 31,177 / 5,081).
bool screen_takes(uint32_t batch, uint32_t dim, uint64_t n, bool layer)
{
    if (ctx().knobs.screen == 2) return false;
    const uint64_t bytes = knn_f16_rows(n) * ((uint64_t)screen_ld(dim) * 2 + (uint64_t)screen_pitch32(dim) * 4);
    return batch >= 512 && dim >= 32 && dim <= 4096 && (!layer || (uint64_t)batch * dim >= 131072) && n >= (layer ? 16384 : 65536) && bytes <= ((uint64_t)8 << 30);
}

// Nearest neighbours: whether screening is the faster way, the copies' making included.  Fitted to 752 searches of 512 to 4,096 queries, 32 to 1,024
// components, 65,536 to 1,000,000 items, k 1 to 256: none is slower, 0.3 % of the time they could take is left (us, fp32 / screened: 512 x 32 x 65,536
// top 10 79 / 98, 512 x 64 x 65,536 top 10 90 / 105, 512 x 32 x 131,072 top 10 145 / 129, 512 x 128 x 65,536 top 10 129 / 104, 1,024 x 32 x 65,536 top
// 10 151 / 103, 512 x 32 x 140,000 top 10 149 / 144, 2,048 x 128 x 150,000 top 10 767 / 260, 4,096 x 128 x 1,000,000 top 100 8,788 / 1,915).  These were
// random vectors: beyond 131,072 items, where columns may go through lists, the line is held back for large k (512 x 32 x 140,000 top 256 225 / 160),
// whose lists fill first where neighbours lie closer together.
// So it is for norms that differ: 360 searches of tables with a lognormal spread (0.5) or an item 3 or 50 times as long as the others take 0.28 of the
// time that fp32 does in all.
bool screen_search_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k)
{
    return ctx().knobs.screen == 1 || (double)batch * (dim + 32 + (n <= 131072 ? 0.25 : -0.125) * k) * (double)n >= 5.2e9;
}

static inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// Whether all columns' sums are stored.  (They are compared with bounds only where a bound keeps most columns out, and where there
// are rows for the whole GPU: a workgroup of that kind has 256 rows, and 64 share a row's columns at most.)  A workgroup reads the maxima of
// 131,072 columns; few rows have one of four times as many wavefronts each, which takes the bitmap of a million columns' filter.  More than 2^28
// sums are not stored: writing them takes what it takes, ranges leave most of them in registers (us, stored / in ranges, top 10, kept tables: 4,096 x
// 128 x 131,072 551 / 280, 512 x 64 x 1,000,000 445 / 295, 4,096 x 512 x 100,000 719 / 546).  For small k, of which few pass a bound, ranges are ahead
// from fewer sums on, if a first block is a small part of the columns (819 layers and as many searches of 2^24 to 2^28 sums measured both ways, k 1 to 64:
// 1.7 and 1.3 % of the time they could take are left, 8 and 7 with 2^28 alone; none loses more than 3 %): 4,096 x 64 x 65,536 top 1 248 / 166, 1,024 x 128 x
// 131,072 top 10 151 / 119, 512 x 128 x 131,072 top 1 108 / 93, but 4,096 x 64 x 32,768 top 1 124 / 140, 2,048 x 64 x 65,536 top 32 124 / 141,
// 256 x 256 x 524,288 top 10 204 / 243, 256 x 128 x 1,000,000 top 100 272 / 414.
static bool screen_stored(uint32_t batch, uint64_t n, uint32_t k)
{
    if (ctx().knobs.fc_topk_first_columns) return false;
    const uint64_t sums = (uint64_t)batch * n;
    if (batch > 256 && n >= 49152 + 512 * k && sums > ((uint64_t)1 << 26) + ((uint64_t)k << 22)) return false;
    return (n <= 131072 || (batch <= 512 && n <= 1048576)) && sums <= ((uint64_t)1 << 28);
}

static uint32_t screen_first_columns(uint32_t n, uint32_t k)
{
    // (two blocks of maxima for each of the k best: with fewer the bound is far below the k-th score; sixteen chunks of whole tiles)
    uint32_t c = ctx().knobs.fc_topk_first_columns ? ctx().knobs.fc_topk_first_columns : (std::max(8192u, 64 * k) + 4095) / 4096 * 4096;
    c = std::max(256u, std::min(c, 32768u)) / 256 * 256;
    return std::min(c, n);
}

// (what i8_wide_kernel takes, or a whole number of f16_sweep_kernel's pairs of stages)
static uint32_t i8_ld(uint32_t dim) { return dim > 256 && dim <= 512 ? 512 : (dim + 127) / 128 * 128; }

// What of that is known of a table alone: whether one that is kept holds a copy in bytes.  (Vectors of up to 64 and of 257 to 320 components are mostly padding:
// 128 bytes beside the 96 to 384 of the other copies, which nothing would read.)
static bool screen_has_bytes(uint32_t dim, uint64_t n)
{
    return n <= kBestColumns && (ctx().knobs.screen_bytes == 1 || (n >= 20000 && 3 * i8_ld(dim) <= 4 * screen_ld(dim)));
}

// Whether a search with a kept table goes in bytes: many products of a long table, whose bytes are not mostly padding, of which k columns are a small part (else
// blocks with one candidate hold a second one, and all 32 columns are scored).  Fitted to 1,814 searches and layers (12,000 to 1,000,000 columns, 16 to
// 1,024 components, 1 to 4,096 rows, k 1 to 200) measured both ways: 3.1 % of the time they could
// take is left, 6.3 % with halves alone; nine are slower by more than 3 %, by 22 % at most (130 x 393 x 118,322 top 30 92 / 112).  us, halves / bytes, the whole call:
// 4,096 x 512 x 1,000,000 top 100 with a filter 4,140 / 2,550, 4,096 x 128 x 1,000,000 top 100 1,780 / 1,240, 256 x 128 x 1,000,000 top 100 304 / 169, 128 x 256 x
// 500,000 top 50 168 / 121, 4,096 x 1,024 x 27,278 top 10 and then 1,904 rows 790 / 727; but 4,096 x 32 x 1,000,000 top 10 738 / 975, 1,024 x 128 x 27,278 top 10 49 / 50,
// 8 x 256 x 500,000 top 50 114 / 115, 256 x 1,024 x 27,278 top 100 87 / 276.
bool screen_in_bytes(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k)
{
    if (!screen_has_bytes(dim, n) || n < 64 * (uint64_t)k || ctx().knobs.screen_bytes == 2) return false;
    if (ctx().knobs.screen_bytes == 1) return true;
    return !ctx().knobs.fc_topk_first_columns && n >= 2500 * (uint64_t)k && (dim <= 512 || batch >= 1024) &&
           (double)batch * (double)n * screen_ld(dim) >= (n < 65536 ? 2e10 : 4e9);
}

ScreenTable screen_table(void* base, uint32_t dim, uint64_t n, bool kept)
{
    ScreenTable t;
    char* p = (char*)base;
    const uint64_t rows = knn_f16_rows(n);
    t.items16 = p;
    p += align256(rows * screen_ld(dim) * 2);
    t.rows32 = (float*)p;
    p += align256(n * screen_pitch32(dim) * sizeof(float));
    t.norm = (float*)p;
    p += align256(rows * sizeof(float));
    t.seg_norm = (float*)p;
    p += align256(rows / 64 * sizeof(float));
    t.stats = (uint32_t*)p;
    p += 256;
    t.items8 = nullptr;
    t.unit8 = nullptr;
    t.error8 = nullptr;
    t.side8 = nullptr;
    if (kept && screen_has_bytes(dim, n)) {
        t.items8 = p;
        p += align256(rows * i8_ld(dim));
        t.unit8 = (float*)p;
        p += align256(rows / 32 * sizeof(float));
        t.error8 = (float2*)p;
        p += align256(rows / 128 * sizeof(float2));
        t.side8 = (float*)p;
        p += align256(rows / 32 * kI8Side * sizeof(float) + kI8SideSlack);
    }
    t.bytes = (size_t)(p - (char*)base);
    return t;
}

ScreenTable screen_table_halves(void* base, uint32_t dim, uint64_t n)
{
    ScreenTable t{};
    char* p = (char*)base;
    const uint64_t rows = knn_f16_rows(n);
    t.norm = (float*)p;
    p += align256(rows * sizeof(float));
    t.stats = (uint32_t*)p;
    p += 256;
    t.items8 = p;
    p += align256(rows * i8_ld(dim));
    t.unit8 = (float*)p;
    p += align256(rows / 32 * sizeof(float));
    t.error8 = (float2*)p;
    p += align256(rows / 128 * sizeof(float2));
    t.side8 = (float*)p;
    p += align256(rows / 32 * kI8Side * sizeof(float) + kI8SideSlack);
    t.bytes = (size_t)(p - (char*)base);
    return t;
}

// Words of a row, and how many rows' words (and lists) there is room for: 1 GiB of them (6,144 rows of a million columns), else as many as leave equal parts.
constexpr uint64_t kWordsRoom = (uint64_t)1 << 30;
static uint64_t i8_row_words(uint64_t n) { return (n + 255) / 256 * 8; }
static uint32_t i8_rows(uint32_t batch, uint64_t n)
{
    const uint64_t row = i8_row_words(n) * sizeof(uint32_t) + (n > kAloneColumns ? (kNearWords + 1) * sizeof(uint2) : 0), most = std::max<uint64_t>(512, kWordsRoom / row / 512 * 512);
    if (batch <= most) return batch;
    const uint64_t parts = (batch + most - 1) / most;
    return (uint32_t)((batch + parts * 512 - 1) / (parts * 512) * 512);   // (whole workgroups' rows)
}

ScreenWorkspace screen_layout(void* base, uint32_t batch, uint32_t dim, uint64_t n, uint32_t k, bool kept)
{
    ScreenWorkspace w{};
    char* p = (char*)base;
    if (kept && screen_in_bytes(batch, dim, n, k)) {
        w.columns = (uint32_t)n;
        w.rows8 = p;
        p += align256(knn_f16_rows(batch) * i8_ld(dim));
        w.unit8 = (float*)p;
        p += align256((size_t)batch * sizeof(float));
        w.error8 = (float4*)p;
        p += align256((size_t)batch * sizeof(float4));
        w.side8 = (float*)p;
        p += align256(knn_f16_rows(n) / 32 * kI8Side * sizeof(float) + kI8SideSlack);
        w.rows = i8_rows(batch, n);
        w.words = (uint32_t*)p;
        p += align256(w.rows * i8_row_words(n) * sizeof(uint32_t));
        if (n > kAloneColumns) {
            w.near = (uint2*)p;
            p += align256((size_t)w.rows * kNearWords * sizeof(uint2));
            w.near_found = (uint2*)p;
            p += align256((size_t)w.rows * sizeof(uint2));
        }
        w.bytes = std::max((size_t)(p - (char*)base), screen_layout(nullptr, batch, dim, n, k, false).bytes);
        return w;
    }
    // (decided here for every search in this workspace, which may be of fewer columns: pad rows of an item table)
    const uint64_t columns = w.columns = screen_stored(batch, n, k) ? (uint32_t)n : screen_first_columns((uint32_t)n, k);
    w.rows16 = p;
    p += align256(knn_f16_rows(batch) * screen_ld(dim) * 2);
    w.e1 = (float*)p;
    p += align256((size_t)batch * sizeof(float));
    w.e0 = (float*)p;
    p += align256((size_t)batch * sizeof(float));
    w.scale = (float*)p;
    p += align256((size_t)batch * sizeof(float));
    w.sums = p;
    p += align256(batch * ((columns + 255) / 256 * 256) * 2);
    w.most = p;
    p += align256(batch * ((columns + 255) / 256 * 8) * 2);
    w.admit = (uint32_t*)p;
    p += align256((size_t)batch * sizeof(uint32_t));
    w.keep = (uint64_t*)p;
    p += align256((size_t)batch * kKeepWords * sizeof(uint64_t));
    w.keep_count = (uint32_t*)p;
    p += align256((size_t)batch * sizeof(uint32_t));
    w.seg = (uint64_t*)p;
    p += align256((size_t)batch * kListWords * sizeof(uint64_t));
    w.seg_count = (uint32_t*)p;
    p += align256((size_t)batch * kF16ListStride * sizeof(uint32_t));
    w.bytes = (size_t)(p - (char*)base);
    return w;
}

__global__ void screen_clear_kernel(uint32_t* stats) { stats[threadIdx.x] = 0; }

int screen_build(const ScreenTable& t, const float* W, uint64_t ldw, uint64_t n, uint32_t dim)
{
    hipStream_t s = ctx().stream;
    hipLaunchKernelGGL(screen_clear_kernel, dim3(1), dim3(64), 0, s, t.stats);
    ScreenItemsArgs i{};
    i.W = W; i.ldw = ldw; i.n = (uint32_t)n; i.dim = dim;
    i.ld = screen_ld(dim); i.pitch32 = screen_pitch32(dim);
    i.out16 = (_Float16*)t.items16; i.out32 = t.rows32; i.norm = t.norm; i.seg_norm = t.seg_norm; i.stats = t.stats;
    hipLaunchKernelGGL(screen_items_kernel, dim3((uint32_t)(knn_f16_rows(n) / 64)), dim3(256), 0, s, i);
    DSX_LAUNCH_CHECK("screen_items_kernel");
    if (t.items8) {
        I8ItemsArgs e{};
        e.rows32 = t.rows32; e.norm = t.norm; e.stats = t.stats; e.n = (uint32_t)n; e.dim = dim; e.pitch32 = i.pitch32; e.ld8 = i8_ld(dim);
        e.items8 = (int8_t*)t.items8; e.unit = t.unit8; e.side = t.side8; e.error = t.error8; e.error_most = t.stats + 4;
        hipLaunchKernelGGL((i8_items_kernel<false>), dim3((uint32_t)(knn_f16_rows(n) / 128)), dim3(256), 0, s, e);
        DSX_LAUNCH_CHECK("i8_items_kernel");
    }
    return DSX_OK;
}

int screen_build_halves(const ScreenTable& t, const void* items16, uint64_t n, uint32_t dim)
{
    hipStream_t s = ctx().stream;
    hipLaunchKernelGGL(screen_clear_kernel, dim3(1), dim3(64), 0, s, t.stats);
    I8ItemsArgs e{};
    e.rows16 = (const _Float16*)items16; e.ld16 = knn_f16_ld(dim); e.norm = t.norm; e.stats = t.stats; e.n = (uint32_t)n; e.dim = dim; e.ld8 = i8_ld(dim);
    e.items8 = (int8_t*)t.items8; e.unit = t.unit8; e.side = t.side8; e.error = t.error8; e.error_most = t.stats + 4;
    hipLaunchKernelGGL((i8_items_kernel<true>), dim3((uint32_t)(knn_f16_rows(n) / 128)), dim3(256), 0, s, e);
    DSX_LAUNCH_CHECK("i8_items_kernel");
    return DSX_OK;
}

int screen_rows(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w, ScreenNotes* notes)
{
    if (w.words) {
        I8RowsArgs r{};
        r.X = j.X; r.ldx = j.ldx; r.batch = j.batch; r.dim = j.dim; r.ld8 = i8_ld(j.dim);
        r.halves = j.rows16 != nullptr;
        r.rows8 = (int8_t*)w.rows8; r.unit = w.unit8; r.error = w.error8;
        r.stats = j.bias ? nullptr : t.stats;
        r.row_flag = j.row_flag; r.told = j.told; r.clear = j.clear; r.clear_words = j.clear_words;
        r.row_blocks = (uint32_t)(knn_f16_rows(j.batch) / 4);
        uint32_t more = 0;
        if (j.bias && i8_wide_takes(r.ld8, j.batch)) {
            r.bias = j.bias; r.norm = t.norm; r.bias_raise = screen_bias_raise(j.dim); r.n = j.n; r.table_side = t.side8; r.side = w.side8;
            more = std::min(1024u, (j.n + 1023) / 1024);
        }
        hipLaunchKernelGGL(i8_rows_kernel, dim3(r.row_blocks + more), dim3(256), 0, ctx().stream, r);
        DSX_LAUNCH_CHECK("i8_rows_kernel");
        return DSX_OK;
    }
    ScreenRowsArgs r{};
    r.whole = (uintptr_t)j.X % 16 == 0 && j.ldx % 4 == 0;
    r.X = j.X; r.ldx = j.ldx; r.batch = j.batch; r.dim = j.dim; r.ld = screen_ld(j.dim);
    r.out16 = (_Float16*)w.rows16; r.e1 = w.e1; r.e0 = w.e0; r.scale = w.scale; r.scaled = j.bias == nullptr; r.row_flag = j.row_flag; r.told = notes ? &notes->flag : j.told;
    r.cand_count = j.cand_count; r.clear = j.clear; r.clear_words = j.clear_words;
    r.stats = t.stats; r.notes = notes;
    hipLaunchKernelGGL(screen_rows_kernel, dim3((uint32_t)(knn_f16_rows(j.batch) / 4)), dim3(256), 0, ctx().stream, r);
    DSX_LAUNCH_CHECK("screen_rows_kernel");
    return DSX_OK;
}

template <int T, int R, int E, int MODE> static int launch_pick_as(const ScreenFoldArgs& a, size_t lds)
{
    // More LDS than a kernel gets unasked, for the bitmap of 262,144 columns and more.  Asked for once per device, as much as there can
    // be: threads that come here together ask for the same.
    if (lds > 65536 - 32768) {
        static std::atomic<bool> asked[64] = {};
        const int dev = ctx().device;
        if (dev < 0 || dev >= 64 || !asked[dev].load(std::memory_order_acquire)) {
            DSX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&screen_pick_kernel<T, R, E, MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
            if (dev >= 0 && dev < 64) asked[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL((screen_pick_kernel<T, R, E, MODE>), dim3(a.batch), dim3(T), lds, ctx().stream, a);
    DSX_LAUNCH_CHECK("screen_pick_kernel");
    return DSX_OK;
}

static int launch_pick(const ScreenFoldArgs& a, bool keep)
{
    const size_t bitmap = a.fidx ? ((size_t)a.stored + 31) / 32 * 4 : 0, row = keep ? 0 : (size_t)(a.dim + 63) / 64 * 256;
    const size_t lds = std::max<size_t>(16, std::max(bitmap, row));
    // Maxima: a lane's only one for small k, four where more than one of the k best are likely to share a lane.  Sixteen wavefronts a row
    // where there is a compute unit for each: with four, what is in flight of the candidates' rows does not cover the latency
    // (256 x 1,024 x 27,278 top 100: 47.7 us / 31.1); with more rows than that four of them pass through at a time (512 x 128 x 27,278 top 10, four
    // batches: 153 us / 214 with sixteen).
    const bool one = a.k <= 32;
    if (keep) return one ? launch_pick_as<256, 1, 4, kPickKeep>(a, lds) : launch_pick_as<256, 4, 4, kPickKeep>(a, lds);
    if (a.batch > (uint32_t)ctx().num_cus && a.stored <= 32768) return one ? launch_pick_as<256, 1, 4, kPickFinal>(a, lds) : launch_pick_as<256, 4, 4, kPickFinal>(a, lds);
    if (a.batch > 512) return one ? launch_pick_as<256, 1, 16, kPickFinal>(a, lds) : launch_pick_as<256, 4, 16, kPickFinal>(a, lds);
    if (a.stored <= 131072) return launch_pick_as<1024, 1, 4, kPickFinal>(a, lds);
    return launch_pick_as<1024, 1, 32, kPickFinal>(a, lds);
}

// What a search in bytes and one in halves tell the kernels that end with results.
static ScreenFoldArgs fold_args(const ScreenJob& j, const ScreenTable& t)
{
    ScreenFoldArgs a{};
    a.batch = j.batch; a.k = j.k; a.n = j.n;
    a.act = j.act; a.slope = j.slope; a.alpha = j.alpha; a.lambda = j.lambda;
    a.row_flag = j.row_flag; a.told = j.told; a.open = j.open;
    a.position = j.position; a.index = j.index; a.fstart = j.fstart; a.fend = j.fend; a.fidx = j.fidx;
    a.X = j.X; a.ldx = j.ldx; a.dim = j.dim; a.pitch32 = screen_pitch32(j.dim); a.rows32 = t.rows32; a.bias = j.bias;
    a.keys = j.keys; a.values = j.values; a.keys2 = j.keys2; a.values2 = j.values2;
    return a;
}

static int screen_run_bytes(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w)
{
    F16Job f{};
    f.items = t.items8; f.ld = i8_ld(j.dim) / 2; f.n = j.n;
    f.norm = t.norm; f.bias = j.bias; f.bias_raise = screen_bias_raise(j.dim);
    f.unit = t.unit8; f.words = w.words; f.ldw = i8_row_words(j.n);
    ScreenFoldArgs a = fold_args(j, t);
    a.words = w.words; a.ldw = f.ldw; a.error_items = t.error8; a.near = w.near; a.near_found = w.near_found;
    if (j.rows16) {
        a.rows16 = (const _Float16*)j.rows16;
        a.ld16 = knn_f16_ld(j.dim);
    }
    I8NearArgs e{};
    e.k = j.k; e.n = j.n; e.words = w.words; e.ldw = f.ldw;
    e.error_most = reinterpret_cast<const float4*>(t.stats + 4);
    e.index = j.index; e.fstart = j.fstart; e.fend = j.fend; e.fidx = j.fidx;
    e.near = w.near; e.near_found = w.near_found;
    e.act = j.act; e.slope = j.slope; e.alpha = j.alpha; e.lambda = j.lambda;
    const bool starts = j.bias || !j.even;
    const size_t row_lds = (size_t)(j.dim + 127) / 128 * 512;
    const bool alone = j.n <= kAloneColumns;   // (no kernel of its own for the words)
    for (uint32_t r = 0; r < j.batch; r += w.rows) {
        const uint32_t rows = std::min(w.rows, j.batch - r);
        const uint64_t results = (uint64_t)r * j.k;
        f.Q = (const int8_t*)w.rows8 + (uint64_t)r * i8_ld(j.dim); f.scale = w.unit8 + r; f.batch = rows;
        if (int rc = i8_wide_takes(f.ld * 2, rows) ? i8_wide_run(f, j.bias ? w.side8 : t.side8, starts) : i8_best_run(f, starts)) return rc;
        a.batch = e.batch = rows;
        a.X = j.X + (uint64_t)r * j.ldx;
        e.error_rows = a.error_rows = w.error8 + r;
        e.unit = w.unit8 + r;
        e.row_flag = a.row_flag = j.row_flag + r;
        a.position = e.position = j.position + r;
        a.keys = j.keys + results; a.values = j.values + results;
        if (j.keys2) {
            a.keys2 = j.keys2 + results;
            a.values2 = j.values2 + results;
        }
        if (j.before_last && r + rows == j.batch) j.before_last(j.before_last_arg);
        if (!alone) {
            if (j.n <= kBestColumns / 4) hipLaunchKernelGGL((i8_near_kernel<4>), dim3(rows), dim3(512), 0, ctx().stream, e);
            else hipLaunchKernelGGL((i8_near_kernel<16>), dim3(rows), dim3(512), 0, ctx().stream, e);
            DSX_LAUNCH_CHECK("i8_near_kernel");
        }
        auto finish = [&](auto halves) {
            constexpr bool H = decltype(halves)::value;
            if (!alone) hipLaunchKernelGGL((i8_finish_kernel<H, 0>), dim3(rows), dim3(256), row_lds, ctx().stream, a, e);
            else if (j.k <= 32) hipLaunchKernelGGL((i8_finish_kernel<H, 1>), dim3(rows), dim3(256), row_lds, ctx().stream, a, e);
            else hipLaunchKernelGGL((i8_finish_kernel<H, 2>), dim3(rows), dim3(256), row_lds, ctx().stream, a, e);
        };
        if (j.rows16) finish(std::true_type{});
        else finish(std::false_type{});
        DSX_LAUNCH_CHECK("i8_finish_kernel");
    }
    return DSX_OK;
}

int screen_run(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w)
{
    if (w.words) return screen_run_bytes(j, t, w);
    hipStream_t s = ctx().stream;
    const uint32_t ld = screen_ld(j.dim), n = j.n;
    // (a first block that is everything, of a narrow table and many rows, is a search of stored sums too: there is no range to end with)
    const uint32_t n0 = std::min(w.columns, n);
    const bool stored = n0 == n;
    F16Job f{};
    f.Q = w.rows16; f.items = t.items16; f.ld = ld; f.batch = j.batch; f.n = n0;
    f.norm = t.norm; f.bias = j.bias; f.e1 = w.e1; f.bias_raise = screen_bias_raise(j.dim);
    f.Z = w.sums; f.M = w.most; f.ldz = (n0 + 255) / 256 * 256; f.scale = w.scale;
    int rc = f16_store_run(f);
    if (rc) return rc;
    ScreenFoldArgs a = fold_args(j, t);
    a.e1 = w.e1; a.e0 = w.e0;
    a.width_bias = 2.3f * screen_bias_raise(j.dim) / (screen_relative(j.dim) + screen_bias_raise(j.dim));
    a.norm = t.norm; a.seg_norm = t.seg_norm;
    a.largest = j.even ? reinterpret_cast<const float*>(t.stats) : nullptr;
    a.keep = w.keep; a.keep_count = w.keep_count; a.admit = w.admit;
    a.seg = w.seg; a.seg_count = w.seg_count;
    a.cand = j.cand; a.cand_count = j.cand_count; a.cap = j.cap;
    a.Z = (const _Float16*)w.sums; a.M = (const _Float16*)w.most; a.ldz = f.ldz; a.scale = w.scale; a.stored = n0;
    a.width_z = 2.1f * f.bias_raise + 1.0e-3f;   // (rounding up to a half: 9.9e-4 of it at most)
    if (stored && j.before_last) j.before_last(j.before_last_arg);
    if ((rc = launch_pick(a, !stored)) || stored) return rc;
    const size_t row_lds = (size_t)(j.dim + 63) / 64 * 256;
    // A bound taken over `done` columns lets about k * width / done of the next `width` columns pass: ranges grow by a factor that keeps that near an
    // eighth of the lists (the sample's own items, which score high and pass as well, come on top), by twelve times at most, but for a last
    // range of up to twenty: survivors cost more than another range's launches then (top 10, us, 51 times / 12: searches 4,096 x 32 x 1,000,000 984 / 834,
    // 512 x 128 x 1,000,000 648 / 558; top 1, one range of 16 times / two: layers 4,096 x 64 x 140,000 245 / 279), and where scores rise along the table, or a filter lists the
    // best columns of the first block, lists do not fill up that do with 51 times (4,096 x 64 x 1,000,000 top 10, 144 such columns a row: 23.8 ms / 1.1;
    // what it costs: 1,024 x 64 x 300,000 top 1 172 / 192).
    const uint32_t growth = std::max(4u, std::min(j.cap / (8 * j.k), 12u)), last = std::max(4u, std::min(j.cap / (8 * j.k), 20u));
    for (uint32_t done = n0; done < n;) {
        uint32_t ncols = (uint32_t)((uint64_t)done * last >= n - done ? n - done : (uint64_t)done * growth);
        if (n - done - ncols < 256) ncols = n - done;   // no sliver of a last range
        f.items = (const char*)t.items16 + (uint64_t)done * ld * 2;
        f.norm = t.norm + done;
        f.bias = j.bias ? j.bias + done : nullptr;
        f.n = ncols;
        f.cand = CandArgs{w.admit, j.cand, j.cand_count, j.cap, done, j.overflow};
        f.seg = w.seg; f.seg_count = w.seg_count; f.seg_words = kListWords;
        // Vectors that fit a wavefront's registers go through the kernel that keeps the queries there, which raises no sums (1,000,000 x
        // 128 x 4,096 queries, top 100: 1,461 us in three ranges, 1,361 so).
        a.lists = 0;
        if (j.even && (rc = knn_f16_wide_run(f.Q, f.items, ld, j.batch, ncols, f.cand, f.seg, f.seg_count, f.seg_words, false, &a.lists))) return rc;
        if (!a.lists && (rc = f16_sweep_run(f, true, &a.lists))) return rc;
        a.seg_cap = kListWords / a.lists;
        done += ncols;
        if (done >= n && j.before_last) j.before_last(j.before_last_arg);
        // (the sums of the first block, rounded up to halves, are among what is kept: their width is the others' from here on)
        if (done < n) hipLaunchKernelGGL((screen_fold_kernel<false>), dim3(j.batch), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((screen_fold_kernel<true>), dim3(j.batch), dim3(256), row_lds, s, a);
        DSX_LAUNCH_CHECK("screen_fold_kernel");
    }
    return DSX_OK;
}

}  // namespace dsx

using namespace dsx;

extern "C" int dsx_testing_screen_columns(uint32_t batch, uint32_t dim, uint32_t rows_padded, uint32_t padding, uint32_t k, uint64_t* room, uint64_t* stored,
                                          int* ranges)
{
    DSX_CHECK_ARG(room && stored && ranges, "dsx_testing_screen_columns: null pointer");
    DSX_CHECK_ARG(batch > 0 && dim > 0 && padding < rows_padded && k >= 1, "dsx_testing_screen_columns: batch %u, dim %u, rows_padded %u, padding %u, k = %u", batch,
                  dim, rows_padded, padding, k);
    const ScreenWorkspace w = screen_layout(nullptr, batch, dim, rows_padded, k, false);
    const uint32_t n0 = std::min(w.columns, rows_padded - padding);   // as screen_run
    *room = (uint64_t)((char*)w.most - (char*)w.sums) / 2 / batch;
    *stored = (n0 + 255) / 256 * 256;
    *ranges = n0 < rows_padded - padding;
    return DSX_OK;
}
