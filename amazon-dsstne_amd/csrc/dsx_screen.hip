// dsx_screen.hip — 16-bit screening of candidates for the fp32 searches (nearest neighbours, output layer with top-K).
//
// A search wants, per row, the k columns of the highest fp32 scores.  The fp32 matrix instructions form every product at 1/16 of the
// f16 ones' rate (157 TFLOP/s against 2.5 PFLOP/s), so here all columns are looked at in f16 (dsx_f16.hip), as upper bounds of their
// scores, and only what the f16 operands' error leaves open is scored in fp32.  Scores and results are fp32 sums, all of them formed by
// one function in one order (equal columns tie, wherever they lie); the f16 sums only decide what cannot be a result.
//
// Error of a screened sum s' = sum x'_i w'_i against the fp32 sum s of the same row and column, x', w' rounded to f16 (unit
// roundoff u = 2^-11, 2^-25 absolute below the normal range), fp32 accumulation:
//   |s' - s| <= (2u + u^2) |x| |w| + 2^-25 sqrt(d) (|x| + |w|) + d 2^-50 + (3 d + 16) 2^-24 |x| |w|      (Cauchy-Schwarz; |.| = 2-norm)
// (d 2^-50: both operands' absolute roundings together, all there is to go by where every component is near 2^-25)
// With the column's norm |w| kept in the table and e1, e0 per row, that is e1 |w| + e0.  A sum starts from its column's bias, raised by
// b_raise |b| for the roundings of a sum that holds it; z is that sum plus e1 |w|.  z + e0 is never below the score, whatever the
// spread of the norms, and the score lies above z - width(z, |w|) (screen_width).  So:
//   the k-th largest z - width bounds the k-th score from below, and only columns with z + e0 at or above that (as pre-activation
//   sums: preactivation_bound) can be results.  For normally distributed scores of 512 products that leaves about 1.2 k columns.
// Exceptions: a column whose norm is above 60,000 gets zeros and an infinite start (it always passes); a row above 65,504 is flagged,
// as is one whose lists fill up (thousands of scores tied at the top): its caller computes it again in fp32.
//
// Two ways (screen_stored).  Few columns, or few rows: the sums are stored as halves, rounded up, and a workgroup per row (or part of
// one) takes what reaches the bound from there.  Many of both: only a first block's are; the rest are compared with the rows' bounds
// where they are formed, in ranges that grow by a factor, after each of which the lists are cut back to what can still be a result.
// Candidates of earlier ranges are not scored until the last one is through: what is scored in fp32 is about 1.2 k columns a row.
#include <algorithm>
#include <cmath>
#include "dsx_screen.h"

namespace dsx {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
constexpr float kF16Max = 65504.0f, kScreenMax = 60000.0f;
constexpr uint32_t kPickWords = 2048;    // candidates of a row (part) that its workgroup holds
constexpr uint32_t kKeepWords = 1024;    // candidates of a row that outlive a column range
constexpr uint32_t kListWords = 4096;    // words of all of a row's lists of one column range
constexpr uint32_t kPickGroups = 14;     // groups of 2,048 columns that a workgroup of 256 lanes holds in registers
constexpr uint32_t kPickColumns = kPickGroups * 2048;

uint32_t screen_ld(uint32_t dim) { return knn_f16_ld(dim); }
uint32_t screen_pitch32(uint32_t dim) { return (dim + 3) / 4 * 4; }

// Relative part of the error, with room for the rounding of the norms themselves; what a bias is raised by, per unit.
__host__ __device__ __forceinline__ float screen_relative(uint32_t dim) { return 9.765625e-4f * 1.01f + (4.0f * (float)dim + 64.0f) * 5.9604645e-8f; }
__host__ __device__ __forceinline__ float screen_bias_raise(uint32_t dim) { return ((float)dim + 64.0f) * 1.2e-7f; }

// stats (nearest neighbours): [0] largest norm of a column (the bits of a non-negative float; NaN columns have no part in it: their
// scores are NaN on every path); [1] sum of the norms of one column in 256, [2] their number
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
    _Float16* out16;        // [batch rounded up to 256][ld], zero filled
    float* e1;              // [batch]
    float* e0;              // [batch]
    float* scale;           // [batch]
    int scaled;             // the scale follows the norms (else 1)
    uint32_t* row_flag;     // [batch] set where the error has no bound
    uint32_t* told;         // host-visible word set with it (may be NULL)
    const uint32_t* stats;
    ScreenNotes* notes;     // host-visible: what the table's columns and the rows are like (nearest neighbours)
};

// One wavefront per row.
__global__ __launch_bounds__(256) void screen_rows_kernel(ScreenRowsArgs a)
{
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const bool valid = row < a.batch;
    float sum = 0.0f;
    if (valid)
        for (uint32_t d = lane; d < a.dim; d += kWave) {
            const float x = a.X[(uint64_t)row * a.ldx + d];
            sum += x * x;
        }
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) sum += __shfl_xor(sum, d);
    const float norm = sqrtf(sum);
    const bool bad = norm > kF16Max;   // (a NaN in the row: its scores are NaN everywhere, there is nothing to miss)
    for (uint32_t d = lane; d < a.ld; d += kWave) {
        const float x = (valid && !bad && d < a.dim) ? a.X[(uint64_t)row * a.ldx + d] : 0.0f;
        a.out16[(uint64_t)row * a.ld + d] = (_Float16)x;
    }
    if (!valid || lane != 0) return;
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
    if (bad) {
        a.row_flag[row] = 1;
        if (a.told) *(volatile uint32_t*)a.told = 1u;
    }
}

// What the two kernels below have in common.
struct ScreenFoldArgs {
    uint32_t batch, k, n;
    const float* e1;
    const float* e0;
    float width_bias;        // share of width per unit of e1 |w| beyond 2.02 (the bias's roundings)
    float width_z;           // and per unit of |z|
    const float* norm;       // by column
    const float* seg_norm;
    uint32_t act;
    float slope, alpha, lambda;
    uint32_t* row_flag;
    uint32_t* told;
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
    int fresh;               // fold: nothing is kept from earlier ranges
    // pick
    const _Float16* Z;
    uint64_t ldz;
    const float* scale;
    uint32_t stored;         // columns of Z
    uint32_t parts, part_columns;
    // final
    const float* X;
    uint32_t ldx, dim, pitch32;
    const float* rows32;
    const float* bias;
    float* keys;
    uint32_t* values;
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

// The sum z below which nothing can be a result when k columns score at least t (as a sum); -inf: anything can.
__device__ __forceinline__ float screen_cut(const ScreenFoldArgs& a, float t, float e0)
{
    if (!(t > -__builtin_inff())) return -__builtin_inff();
    const float y = activate_rt(t, a.act, a.slope, a.alpha, a.lambda);
    const float z = preactivation_bound(score_key(y), a.act, a.slope, a.alpha, a.lambda);
    const float cut = z - e0 * 1.001f - fabsf(z) * 2.3841858e-7f;   // (the subtraction itself is rounded)
    return (cut == cut) ? cut : -__builtin_inff();
}

__device__ __forceinline__ void screen_flag(const ScreenFoldArgs& a, uint32_t b)
{
    a.row_flag[b] = 1;
    if (a.told) *(volatile uint32_t*)a.told = 1u;
    if (a.admit) a.admit[b] = 0xffffffffu;   // a NaN: nothing more of the row is wanted
}

// The row's candidates sList[0 .. count) scored in fp32 and its k best written.  Sixteen lanes per candidate; the order of a sum depends on
// nothing but its length.  Every lane of the workgroup calls this.
__device__ __forceinline__ void screen_finish(const ScreenFoldArgs& a, uint32_t b, uint64_t* sList, uint32_t count, float* sX, uint64_t fs, uint64_t fe)
{
    __shared__ uint32_t sValid, sListed;
    __shared__ uint64_t sKth;
    const uint32_t dpad = (a.dim + 63) / 64 * 64;
    for (uint32_t d = threadIdx.x; d < dpad; d += 256) sX[d] = (d < a.dim) ? a.X[(uint64_t)b * a.ldx + d] : 0.0f;
    if (threadIdx.x == 0) {
        sValid = sListed = 0;
        sKth = 0;
    }
    __syncthreads();
    const uint32_t sub = threadIdx.x % 16;
    for (uint32_t e0 = 0; e0 < count; e0 += 16) {
        const uint32_t e = e0 + threadIdx.x / 16;
        const uint32_t col = ~(uint32_t)sList[min(e, count - 1)];
        float sum = 0.0f;
        if (e < count) {
            const float* w = a.rows32 + (uint64_t)col * a.pitch32;
#pragma unroll 4
            for (uint32_t d = 4 * sub; d < a.pitch32; d += 64) {
                const float4 v = *reinterpret_cast<const float4*>(w + d), x = *reinterpret_cast<const float4*>(sX + d);
                sum = fmaf(x.x, v.x, sum);
                sum = fmaf(x.y, v.y, sum);
                sum = fmaf(x.z, v.z, sum);
                sum = fmaf(x.w, v.w, sum);
            }
        }
#pragma unroll
        for (int d = 1; d < 16; d *= 2) sum += __shfl_xor(sum, d);
        if (sub == 0 && e < count) {
            const float y = activate_rt(sum + (a.bias ? a.bias[col] : 0.0f), a.act, a.slope, a.alpha, a.lambda);
            sList[e] = (y == y) ? ((uint64_t)score_key(y) << 32) | (uint32_t)~col : 0ull;
        }
    }
    __syncthreads();
    float* keys = a.keys + (uint64_t)b * a.k;
    uint32_t* values = a.values + (uint64_t)b * a.k;
    for (uint32_t i = threadIdx.x; i < count; i += 256) {
        const uint64_t w = sList[i];
        if (w == 0) continue;
        uint32_t rank = 0;
        for (uint32_t j = 0; j < count; j++) rank += sList[j] > w;
        atomicAdd(&sValid, 1u);
        if (rank == a.k - 1) sKth = w;
        if (rank < a.k) {
            keys[rank] = key_score((uint32_t)(w >> 32));
            values[rank] = ~(uint32_t)w;
        }
    }
    // A listed column scores 0, not nothing (utils/Filters.cpp:62 multiplies, kCalculateTopK then sees the zero): when the row's k-th
    // score is not above 0, or the row has fewer than k scores, such a zero belongs in the result, and the row is computed again.
    if (fe > fs) {
        bool listed = false;
        for (uint64_t t = fs + threadIdx.x; t < fe; t += 256) listed |= a.fidx[t] < a.n;
        if (__ballot(listed) != 0 && threadIdx.x % kWave == 0) atomicOr(&sListed, 1u);
    }
    __syncthreads();
    for (uint32_t p = sValid + threadIdx.x; p < a.k; p += 256) {   // engine/kernels.cu:3221-3224: unfilled slots
        keys[p] = -kMaxValue;
        values[p] = 0;
    }
    if (threadIdx.x == 0 && sListed != 0 && (sKth == 0 || (uint32_t)(sKth >> 32) <= score_key(0.0f))) screen_flag(a, b);
}

// A lower bound of the k-th largest of the workgroup's keys (0: dead ones, not counted), exact in its upper 24 bits; 0 where there are
// fewer than k.  Radix select, a byte at a time.  total: keys beyond that many are 0.  s: 258 words.
template <int N> __device__ __forceinline__ uint32_t block_kth_key(const uint32_t (&key)[N], uint32_t total, uint32_t k, uint32_t* s)
{
    uint32_t prefix = 0, need = k;
    for (int shift = 24; shift >= 8; shift -= 8) {
        s[threadIdx.x] = 0;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < N; u++)
            if (u * 256 < total && key[u] != 0 && (shift == 24 || (key[u] >> (shift + 8)) == (prefix >> (shift + 8)))) atomicAdd(&s[(key[u] >> shift) & 255], 1u);
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

// The k-th largest of 64 * N keys of a wavefront, exact in its upper 20 bits, 0 if there are fewer.  (As the top-K kernels' key search.)
template <int N> __device__ __forceinline__ uint32_t screen_wave_kth(const uint32_t (&key)[N], uint32_t k)
{
    uint32_t t = 0;
#pragma unroll 1
    for (int bit = 30; bit >= 12; bit -= 2) {
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

enum { kPickFinal, kPickKeep, kPickList };

// Sums stored as halves: what reaches the bound, of a row or a part of one.  Everything is requested at once and held in registers; the
// bound is the k-th of R maxima per lane (over groups of eight columns that hold no listed one, each less its width).
template <int R, int G, int MODE>
__global__ __launch_bounds__(256, 4) void screen_pick_kernel(ScreenFoldArgs a)
{
    __builtin_amdgcn_s_setprio(3);   // short kernels issue ahead of a GEMM's wavefronts that share their SIMD
    __shared__ uint64_t sList[kPickWords];
    __shared__ uint32_t sMax[R * 256];
    __shared__ uint32_t sCount;
    __shared__ float sCut;
    extern __shared__ __attribute__((aligned(16))) uint32_t sDyn[];   // bitmap of the part's listed columns; afterwards the row (kPickFinal)
    const uint32_t b = blockIdx.x, part = blockIdx.y, lane = threadIdx.x % kWave;
    const uint32_t lo = part * a.part_columns, hi = min(a.stored, lo + a.part_columns);
    if (a.row_flag[b] != 0) {
        if (threadIdx.x == 0) {
            if constexpr (MODE == kPickKeep) {
                a.admit[b] = 0xffffffffu;
                a.keep_count[b] = 0;
            }
            if constexpr (MODE == kPickList) a.seg_count[(uint64_t)b * kF16ListStride + part] = 0;
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
    half8 z[G];
    float norms[G];   // largest of the 64 columns that the group lies in
    const _Float16* src = a.Z + (uint64_t)b * a.ldz + lo;
#pragma unroll
    for (int u = 0; u < G; u++) {
        const uint32_t c = (u * 256 + threadIdx.x) * 8;
        if (lo + c < hi) z[u] = *reinterpret_cast<const half8*>(src + c);   // (rows of Z are padded to whole tiles)
        else
#pragma unroll
            for (int e = 0; e < 8; e++) z[u][e] = (_Float16)(-65504.0f);
    }
#pragma unroll
    for (int u = 0; u < G; u++) {
        const uint32_t c = lo + (u * 256 + threadIdx.x) * 8;
        norms[u] = a.seg_norm[(c < hi ? c : lo) / 64];
    }
    const uint32_t words = (hi - lo + 31) / 32;
    if (fe > fs)
        for (uint32_t i = threadIdx.x; i < words; i += 256) sDyn[i] = 0;
    if (threadIdx.x == 0) sCount = 0;
    const float e1 = a.e1[b], e0 = a.e0[b], step = 1.0f / a.scale[b];   // (a power of two)
    __syncthreads();
    if (fe > fs) {
        for (uint64_t t = fs + threadIdx.x; t < fe; t += 256) {
            const uint32_t c = a.fidx[t];
            if (c >= lo && c < hi) atomicOr(&sDyn[(c - lo) >> 5], 1u << ((c - lo) & 31));
        }
        __syncthreads();
        // a group of eight columns is a byte of the bitmap: listed ones have no part in the bound
#pragma unroll
        for (int u = 0; u < G; u++) {
            const uint32_t c = (u * 256 + threadIdx.x) * 8;
            const uint32_t listed = (lo + c < hi) ? reinterpret_cast<const unsigned char*>(sDyn)[c / 8] : 0u;
            if (__ballot(listed != 0) == 0) continue;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if ((listed >> e) & 1) z[u][e] = (_Float16)(-65504.0f);
        }
    }
    auto largest = [&](int u) __attribute__((always_inline)) -> float {
        const half2v x = __builtin_elementwise_max(__builtin_elementwise_max(half2v{z[u][0], z[u][1]}, half2v{z[u][2], z[u][3]}),
                                                   __builtin_elementwise_max(half2v{z[u][4], z[u][5]}, half2v{z[u][6], z[u][7]}));
        return (float)__builtin_elementwise_max(x[0], x[1]);
    };
    {
        float low[R];
#pragma unroll
        for (int i = 0; i < R; i++) low[i] = -__builtin_inff();
#pragma unroll
        for (int u = 0; u < G; u++) {
            const float m = largest(u), raised = fmaf(m, step, e1 * norms[u]);
            // (what does not fit a half says nothing: rounded up to infinity, or held at the lowest half, as the places beyond the end are)
            const float l = (m < 65504.0f && m > -65504.0f) ? raised - screen_width(a, raised, norms[u], e1, e0, step) : -__builtin_inff();
            low[u % R] = fmaxf(low[u % R], l);
        }
#pragma unroll
        for (int i = 0; i < R; i++) sMax[i * 256 + threadIdx.x] = score_key(low[i]);
    }
    __syncthreads();
    // (one wavefront searches, a different one from row to row, so that the four SIMDs of a compute unit share the searches)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave) == ((b >> 8) & 3u)) {
        uint32_t all[4 * R];
#pragma unroll
        for (int i = 0; i < 4 * R; i++) all[i] = sMax[i * kWave + lane];
        const uint32_t t = screen_wave_kth<4 * R>(all, a.k);
        if (lane == 0) sCut = screen_cut(a, t > score_key(-__builtin_inff()) ? key_score(t) : -__builtin_inff(), e0);
    }
    __syncthreads();
    const float cut = sCut;
#pragma unroll
    for (int u = 0; u < G; u++) {
        uint32_t at0 = lo + (u * 256 + threadIdx.x) * 8;
        asm volatile("" : "+v"(at0));   // (the norm is read again, from the cache, and not kept)
        const float raise = e1 * a.seg_norm[(at0 < hi ? at0 : lo) / 64];
        if (__ballot(fmaf(largest(u), step, raise) >= cut) == 0) continue;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t c = (u * 256 + threadIdx.x) * 8 + e;
            uint32_t bits = __builtin_bit_cast(u32x4s, z[u])[e / 2];
            asm volatile("" : "+v"(bits));   // (unpacked here, where one is needed, and not for all groups at once)
            const half2v two = __builtin_bit_cast(half2v, bits);
            const float h = (float)two[e & 1];
            bool ok = fmaf(h, step, raise) >= cut && lo + c < hi;
            if (ok && fe > fs) ok = !((sDyn[c >> 5] >> (c & 31)) & 1u);
            const uint64_t m = __ballot(ok);
            if (m == 0) continue;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&sCount, (uint32_t)__popcll(m));
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (ok && at < kPickWords) sList[at] = ((uint64_t)score_key(h * step) << 32) | (uint32_t)~(lo + c);   // (not raised: screen_raised)
        }
    }
    __syncthreads();
    const uint32_t count = sCount;
    if (count > (MODE == kPickKeep ? kKeepWords : kPickWords)) {   // the same for the whole workgroup
        if (threadIdx.x == 0) {
            screen_flag(a, b);
            if constexpr (MODE == kPickKeep) a.keep_count[b] = 0;
            if constexpr (MODE == kPickList) a.seg_count[(uint64_t)b * kF16ListStride + part] = 0;
        }
        return;
    }
    if constexpr (MODE == kPickKeep)
        for (uint32_t i = threadIdx.x; i < count; i += 256) sList[i] = screen_raised(a, sList[i], e1);   // (a lane reads below what it writes here)
    if constexpr (MODE == kPickFinal) {
        screen_finish(a, b, sList, count, reinterpret_cast<float*>(sDyn), fs, fe);
    } else if constexpr (MODE == kPickKeep) {
        for (uint32_t i = threadIdx.x; i < count; i += 256) a.keep[(uint64_t)b * kKeepWords + i] = sList[i];
        if (threadIdx.x == 0) {
            a.keep_count[b] = count;
            a.admit[b] = score_key(cut);
        }
    } else {
        uint64_t* mine = a.seg + ((uint64_t)b * a.lists + part) * a.seg_cap;
        for (uint32_t i = threadIdx.x; i < count; i += 256) {
            if (i < a.seg_cap) mine[i] = sList[i];
            else {   // the row's shared list
                const uint32_t p = atomicAdd(&a.cand_count[b], 1u);
                if (p < a.cap) a.cand[(uint64_t)b * a.cap + p] = sList[i];
            }
        }
        if (threadIdx.x == 0) a.seg_count[(uint64_t)b * kF16ListStride + part] = min(count, a.seg_cap);
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
    const uint32_t kept = a.fresh ? 0u : a.keep_count[b];
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
    if (fresh_words > a.cap) {
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
                if (first) key[u] = low[u] = 0;
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
        screen_finish(a, b, left, count, reinterpret_cast<float*>(sDyn), fs, fe);
    } else {
        for (uint32_t i = threadIdx.x; i < count; i += 256) a.keep[(uint64_t)b * kKeepWords + i] = left[i];
        if (threadIdx.x == 0) {
            a.keep_count[b] = count;
            a.admit[b] = score_key(sCut);
        }
    }
}

// The same for a layer in ranges (dsx_fc_topk), fitted to 320 layers of 512 to 4,096 rows, 64 to 1,024 components, 16,384 to 1,000,000
// columns, k 10 to 256, without filters: fp32 within 23 %, screened within 31 %; none is slower than in fp32, 1.3 % are left (us,
// screened / fp32: 512 x 256 x 16,384 top 10 105 / 80, 4,096 x 1,024 x 27,278 top 256 3,977 / 2,591, 512 x 256 x 131,072 top 100
// 539 / 539, 1,000 x 256 x 131,072 top 100 658 / 831, 4,096 x 512 x 300,000 top 100 3,578 / 10,343).
bool screen_layer_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k)
{
    if (ctx().knobs.screen == 1) return true;
    const double q = batch, d = dim, ld = screen_ld(dim), m = (double)n;
    const double growth = std::max(4u, 512 / std::max(1u, k)), fold = std::log(std::max(m / 2048.0, 1.0)) / std::log(growth + 1.0);   // as fc_topk_common's ranges
    const double ranges = std::ceil(fold), candidates = k * growth * fold;
    const double fp32 = 28.0 + 17.6 * ranges + 1.553e-8 * q * m * d + 2.61e-7 * q * m + 7.7e-5 * q * candidates + 0.49 * k * ranges;
    const double screened = 13.0 + 35.0 * ranges + 3.8e-6 * m * ld + 1.39e-9 * q * m * ld + 6e-8 * q * m + q * candidates * (7.6e-5 + 3.1e-7 * ld) + 0.57 * k * ranges;
    return fp32 > 1.1 * screened;
}

// What can be screened: the preparation costs what about 130 rows' fp32 products do.  Limits: the row in LDS, and 8 GiB for the two
// copies of the table.
bool screen_takes(uint32_t batch, uint32_t dim, uint64_t n, bool layer)
{
    if (ctx().knobs.screen == 2) return false;
    const uint64_t bytes = knn_f16_rows(n) * ((uint64_t)screen_ld(dim) * 2 + (uint64_t)screen_pitch32(dim) * 4);
    return batch >= 512 && dim >= 32 && dim <= 4096 && (!layer || (uint64_t)batch * dim >= 131072) && n >= (layer ? 16384 : 65536) && bytes <= ((uint64_t)8 << 30);
}

// Nearest neighbours: whether screening is the faster way.  Both sides as fitted to 336 measured searches of normalised random vectors (us;
// 512 to 4,096 queries, 32 to 1,024 components, 65,536 to 1,000,000 items, k 10 to 256): fp32 within 13 %, block by block or with
// candidate lists; screened within 45 %, which is why it has to be ahead by a tenth.  None of the 336 is slower than without
// screening, 1.4 % of the time they could take is left (512 x 32 x 65,536 top 256 486 screened / 140 fp32, 2,048 x 32 x 300,000 top
// 100 821 / 681, 512 x 128 x 300,000 top 100 544 / 569, 2,048 x 128 x 150,000 top 10 385 / 755, 4,096 x 128 x 1,000,000 top 100 2,368 /
// 8,789).
// norm_ratio: the largest norm of an item over the average one.  A bound is lowered by 2^-10 of the largest, about
// 2^-10 sqrt(dim) norm_ratio of the scores' spread; where the k best lie, about four of it out, that many more candidates pass:
// exp(4 * 2^-10 sqrt(dim) norm_ratio) times as many.  A first range leaves 5 k of them; lists hold 4,096.
bool screen_search_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k, bool blocks, float norm_ratio)
{
    const double q = batch, d = dim, ld = std::max(d, 64.0), m = (double)n;
    const double more = std::exp(std::min(20.0, 4.0 * std::sqrt(d) * (double)norm_ratio / 1024.0));
    if (5.0 * k * more > 3600.0) return false;
    if (ctx().knobs.screen == 1) return true;
    const double ranges = 1.0 + std::max(1.0, std::ceil(std::log(m / 40960.0) / std::log(5.0))), fold = std::log(m / 8192.0) / std::log(5.0);
    const double fp32 = blocks ? 1.464e-8 * q * m * d + 1.656e-6 * q * m + 4.3e-5 * q * k + 0.265 * k
                               : 120.0 + 1.447e-8 * q * m * d + 2.56e-7 * q * m + 2.37e-4 * q * k + 0.6 * k;
    const double screened = 90.0 + 30.0 * ranges + 3.2e-6 * m * ld + 2e-9 * q * m * ld + 1e-7 * q * m +
                            more * (q * k * fold * (4e-4 + 1.9e-6 * ld) + 0.5 * k * ranges);
    return fp32 > 1.1 * screened;
}

static inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// Whether all columns' sums are stored.  (They are compared with bounds only where a bound keeps most columns out, and where there
// are rows for the whole GPU: a workgroup of that kind has 256 rows, and 64 share a row's columns at most.)
static bool screen_stored(uint32_t batch, uint64_t n)
{
    if (ctx().knobs.fc_topk_first_columns) return false;
    return (n <= 131072 || (batch <= 512 && n <= 64 * kPickColumns)) && (uint64_t)batch * n <= ((uint64_t)1 << 30);
}

static uint32_t screen_first_columns(uint32_t n)
{
    uint32_t c = ctx().knobs.fc_topk_first_columns ? ctx().knobs.fc_topk_first_columns : 8192;
    c = std::max(256u, std::min(c, kPickColumns)) / 256 * 256;
    return std::min(c, n);
}

// Workgroups per row of the stored sums.
static uint32_t screen_parts(uint32_t batch, uint32_t n)
{
    const uint32_t least = (n + kPickColumns - 1) / kPickColumns;
    const uint32_t wanted = std::min((2 * (uint32_t)ctx().num_cus + batch - 1) / batch, std::max(1u, n / 8192));
    return std::min(64u, std::max(least, wanted));
}

ScreenTable screen_table(void* base, uint32_t dim, uint64_t n)
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
    t.bytes = (size_t)(p - (char*)base);
    return t;
}

ScreenWorkspace screen_layout(void* base, uint32_t batch, uint32_t dim, uint64_t n)
{
    ScreenWorkspace w;
    char* p = (char*)base;
    const uint64_t columns = screen_stored(batch, n) ? n : screen_first_columns((uint32_t)n);
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
    return DSX_OK;
}

int screen_rows(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w, ScreenNotes* notes)
{
    ScreenRowsArgs r{};
    r.X = j.X; r.ldx = j.ldx; r.batch = j.batch; r.dim = j.dim; r.ld = screen_ld(j.dim);
    r.out16 = (_Float16*)w.rows16; r.e1 = w.e1; r.e0 = w.e0; r.scale = w.scale; r.scaled = j.bias == nullptr; r.row_flag = j.row_flag; r.told = notes ? &notes->flag : j.told;
    r.stats = t.stats; r.notes = notes;
    hipLaunchKernelGGL(screen_rows_kernel, dim3((uint32_t)(knn_f16_rows(j.batch) / 4)), dim3(256), 0, ctx().stream, r);
    DSX_LAUNCH_CHECK("screen_rows_kernel");
    return DSX_OK;
}

template <int R, int G> static int launch_pick_mode(const ScreenFoldArgs& a, int mode, size_t lds)
{
    const dim3 grid(a.batch, a.parts);
    hipStream_t s = ctx().stream;
    switch (mode) {
    case kPickFinal: hipLaunchKernelGGL((screen_pick_kernel<R, G, kPickFinal>), grid, dim3(256), lds, s, a); break;
    case kPickKeep: hipLaunchKernelGGL((screen_pick_kernel<R, G, kPickKeep>), grid, dim3(256), lds, s, a); break;
    default: hipLaunchKernelGGL((screen_pick_kernel<R, G, kPickList>), grid, dim3(256), lds, s, a); break;
    }
    DSX_LAUNCH_CHECK("screen_pick_kernel");
    return DSX_OK;
}

static int launch_pick(const ScreenFoldArgs& a, int mode)
{
    const size_t bitmap = a.fidx ? ((size_t)a.part_columns + 31) / 32 * 4 : 0, row = mode == kPickFinal ? (size_t)(a.dim + 63) / 64 * 256 : 0;
    const size_t lds = std::max<size_t>(16, std::max(bitmap, row));
    // (maxima: a lane's only one for small k, four where more than one of the k best are likely to share a lane)
    if (a.part_columns <= 8192) return a.k <= 32 ? launch_pick_mode<1, 4>(a, mode, lds) : launch_pick_mode<4, 4>(a, mode, lds);
    return a.k <= 32 ? launch_pick_mode<1, kPickGroups>(a, mode, lds) : launch_pick_mode<4, kPickGroups>(a, mode, lds);
}

int screen_run(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w)
{
    hipStream_t s = ctx().stream;
    const uint32_t ld = screen_ld(j.dim), n = j.n;
    const bool stored = screen_stored(j.batch, n);
    const uint32_t n0 = stored ? n : screen_first_columns(n);
    F16Job f{};
    f.Q = w.rows16; f.items = t.items16; f.ld = ld; f.batch = j.batch; f.n = n0;
    f.norm = t.norm; f.bias = j.bias; f.e1 = w.e1; f.bias_raise = screen_bias_raise(j.dim);
    f.Z = w.sums; f.ldz = (n0 + 255) / 256 * 256; f.scale = w.scale;
    int rc = f16_store_run(f);
    if (rc) return rc;
    ScreenFoldArgs a{};
    a.batch = j.batch; a.k = j.k; a.n = n;
    a.e1 = w.e1; a.e0 = w.e0;
    a.width_bias = 2.3f * screen_bias_raise(j.dim) / (screen_relative(j.dim) + screen_bias_raise(j.dim));
    a.norm = t.norm; a.seg_norm = t.seg_norm;
    a.act = j.act; a.slope = j.slope; a.alpha = j.alpha; a.lambda = j.lambda;
    a.row_flag = j.row_flag; a.told = j.told;
    a.position = j.position; a.index = j.index; a.fstart = j.fstart; a.fend = j.fend; a.fidx = j.fidx;
    a.keep = w.keep; a.keep_count = w.keep_count; a.admit = w.admit;
    a.seg = w.seg; a.seg_count = w.seg_count;
    a.cand = j.cand; a.cand_count = j.cand_count; a.cap = j.cap;
    a.Z = (const _Float16*)w.sums; a.ldz = f.ldz; a.scale = w.scale; a.stored = n0;
    a.X = j.X; a.ldx = j.ldx; a.dim = j.dim; a.pitch32 = screen_pitch32(j.dim); a.rows32 = t.rows32; a.bias = j.bias;
    a.keys = j.keys; a.values = j.values;
    a.width_z = 2.1f * f.bias_raise + 1.0e-3f;   // (rounding up to a half: 9.9e-4 of it at most)
    a.parts = stored ? screen_parts(j.batch, n) : 1;
    a.part_columns = ((n0 + a.parts - 1) / a.parts + 63) / 64 * 64;
    a.parts = (n0 + a.part_columns - 1) / a.part_columns;
    a.lists = a.parts; a.seg_cap = kListWords / a.parts;
    const bool whole = stored && a.parts == 1;
    if ((rc = launch_pick(a, whole ? kPickFinal : stored ? kPickList : kPickKeep))) return rc;
    if (whole) return DSX_OK;
    const size_t row_lds = (size_t)(j.dim + 63) / 64 * 256;
    if (stored) {
        a.fresh = 1;
        hipLaunchKernelGGL((screen_fold_kernel<true>), dim3(j.batch), dim3(256), row_lds, s, a);
        DSX_LAUNCH_CHECK("screen_fold_kernel");
        return DSX_OK;
    }
    // A bound taken over `done` columns lets about k * width / done of the next `width` columns pass: ranges grow by a factor that
    // keeps that near an eighth of the lists (the sample's own items, which score high and pass as well, come on top).
    const uint32_t growth = std::max(4u, j.cap / (8 * j.k));
    a.fresh = 0;
    for (uint32_t done = n0; done < n;) {
        uint32_t ncols = (uint32_t)std::min<uint64_t>((uint64_t)n - done, (uint64_t)done * growth);
        if (n - done - ncols < 256) ncols = n - done;   // no sliver of a last range
        f.items = (const char*)t.items16 + (uint64_t)done * ld * 2;
        f.norm = t.norm + done;
        f.bias = j.bias ? j.bias + done : nullptr;
        f.n = ncols;
        f.cand = CandArgs{w.admit, j.cand, j.cand_count, j.cap, done, j.overflow};
        f.seg = w.seg; f.seg_count = w.seg_count; f.seg_words = kListWords;
        if ((rc = f16_sweep_run(f, true, &a.lists))) return rc;
        a.seg_cap = kListWords / a.lists;
        done += ncols;
        // (the sums of the first block, rounded up to halves, are among what is kept: their width is the others' from here on)
        if (done < n) hipLaunchKernelGGL((screen_fold_kernel<false>), dim3(j.batch), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((screen_fold_kernel<true>), dim3(j.batch), dim3(256), row_lds, s, a);
        DSX_LAUNCH_CHECK("screen_fold_kernel");
    }
    return DSX_OK;
}

}  // namespace dsx
