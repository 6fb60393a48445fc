// dsx_screen.hip — 16-bit screening of candidates for the fp32 searches (nearest neighbours, output layer with top-K).
//
// A search keeps, per row, the columns whose fp32 score reaches the row's bound: a few hundred of a million.  The fp32 matrix
// instructions form every product at 1/16 of the f16 ones' rate (157 TFLOP/s against 2.5 PFLOP/s), so here the columns are looked at
// in f16 first, with a bound lowered by what the f16 operands can be wrong by, and what passes is scored in fp32.  Scores and
// results are fp32 sums, all of them formed by screen_rescore_kernel in one order (equal columns tie, wherever they lie); the f16
// products only decide what cannot be a result, and the first block's fp32 matrix only gives the first bounds.
//
// Error of a screened sum s' = sum x'_i w'_i against the fp32 sum s of the same row and column, x', w' rounded to f16 (unit
// roundoff u = 2^-11, 2^-25 absolute below the normal range), fp32 accumulation:
//   |s' - s| <= (2u + u^2) |x| |w| + 2^-25 sqrt(d) (|x| + |w|) + d 2^-50 + (3 d + 16) 2^-24 |x| |w|      (Cauchy-Schwarz; |.| = 2-norm)
// (d 2^-50: both operands' absolute roundings together, all there is to go by where every component is near 2^-25)
// The matrix instructions keep subnormal operands.  A row's norm above 65,504 (a component might overflow) sets a flag instead.
//
//   ITEM_NORM = false (nearest neighbours): |w| is taken at its largest over all columns, and a norm above 65,504 sets the flag too; the
//     search reads the flag and, where lists filled up for it, runs again without screening.
//   ITEM_NORM = true (layers): one more component adds (2u + ...) |x| |w| of its own column to every sum, which makes the sums upper
//     bounds of the scores whatever the spread of the columns' norms; three more components carry the bias in three f16 pieces, raised
//     by what a sum with it can be wrong by.  Items are masked with biases of -1e9 or -inf: a bias below -60,000 is taken as that, which
//     bounds the score from above all the same.  A column above 60,000 (bias or norm) gets a bias of +inf and always passes.
//
// Preparing a table of n columns of d components reads 4 and writes 6 bytes per element, on every call (nothing is kept that could
// go stale).  4,096 queries x 1,000,000 x 128, top 100: search 8.9 ms in fp32 -> 2.9 (0.28 preparation, 1.3 f16 products at
// 0.8 PFLOP/s, 0.55 fp32 scores of 1,200 candidates per query); output layer 4,096 x 512 x 1,000,000, top 100: 31.4 ms -> 9.3 (1.3,
// 6.3, 0.9).  What bounds it: the sweep of dsx_knn_f16.hip.
#include <algorithm>
#include <cmath>
#include "dsx_device.h"
#include "dsx_internal.h"

namespace dsx {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
constexpr float kF16Max = 65504.0f, kScreenMax = 60000.0f;
constexpr int kScreenExtra = 4;   // components a layer adds: bias in three pieces, the error term

uint32_t screen_ld(uint32_t dim, bool layer) { return knn_f16_ld(dim + (layer ? kScreenExtra : 0)); }
uint32_t screen_pitch32(uint32_t dim) { return (dim + 3) / 4 * 4; }

// Relative part of the error, with room for the rounding of the norms themselves.
__device__ __forceinline__ float screen_relative(uint32_t dim) { return 9.765625e-4f * 1.01f + (4.0f * (float)dim + 64.0f) * 5.9604645e-8f; }

// stats: [0] largest norm of a column, of a layer's first block's columns only (the bits of a non-negative float; NaN columns have no
// part in it: their scores are NaN on every path); [1] sum of the norms of one column in 256, [2] their number (nearest neighbours)
struct ScreenItemsArgs {
    const float* W;       // [dim][ldw]
    const float* bias;    // layers: [n], or NULL
    uint64_t ldw;
    uint32_t n, dim, ld, pitch32;
    uint32_t first;       // columns that stats[0] is taken over
    _Float16* out16;      // [n rounded up to 256][ld], zero filled
    float* out32;         // [n][pitch32], zero filled beyond dim
    uint32_t* stats;
};

// A workgroup takes 64 columns, 64 components at a time through LDS: reads are contiguous along the columns, writes along the
// components.  Bound by memory.
template <bool ITEM_NORM>
__global__ __launch_bounds__(256) void screen_items_kernel(ScreenItemsArgs a)
{
    __shared__ float sTile[64][65];
    __shared__ float sSum[4][64];
    const uint32_t col0 = blockIdx.x * 64, l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const bool valid = col0 + l < a.n;
    float sum = 0.0f;
    const uint32_t whole = ITEM_NORM ? a.dim / 8 * 8 : a.ld;   // a layer's pieces behind this wait for the norm
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
            if (d0 + p < whole) *reinterpret_cast<half8*>(a.out16 + (uint64_t)(col0 + c) * a.ld + d0 + p) = h;
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
    auto raise = [&](uint32_t* to, float v) {
        v = fmaxf(v, 0.0f);   // (drops NaN)
#pragma unroll
        for (int d = 1; d < 64; d *= 2) v = fmaxf(v, __shfl_xor(v, d));
        if (l == 0 && __float_as_uint(v) > *(volatile uint32_t*)to) atomicMax(to, __float_as_uint(v));
    };
    if (q == 0) raise(&a.stats[0], col0 + l < a.first ? norm : 0.0f);
    if constexpr (!ITEM_NORM) {
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
    if constexpr (ITEM_NORM) {
        const float given = (a.bias && valid) ? a.bias[col0 + l] : 0.0f;
        const bool always = norm > kScreenMax || given > kScreenMax;
        float b = fmaxf(given, -kScreenMax);
        // upwards by: the roundings of a sum that holds it, and the absolute roundings of x against this column
        b += fabsf(b) * (((float)a.dim + 64.0f) * 2.3841858e-7f + 1e-6f) + 2.9802322e-8f * 1.01f * sqrtf((float)a.dim + 4.0f) * norm;
        const _Float16 hi = always ? (_Float16)__builtin_inff() : (_Float16)b;
        const float r1 = always ? 0.0f : b - (float)hi;
        const _Float16 mid = (_Float16)r1, lo = (_Float16)(r1 - (float)mid);
        const _Float16 error = always ? (_Float16)0.0f : (_Float16)(norm * 0.03125f * 1.002f + 1e-7f);   // rounded up: half an ulp is at most 2^-11
        if (always)   // (its components may be infinite in f16; what the loop above wrote was ordered before by the barrier)
            for (uint32_t p = 8 * q; p < whole; p += 32) *reinterpret_cast<half8*>(a.out16 + (uint64_t)(col0 + l) * a.ld + p) = half8{};
        for (uint32_t p = whole + 8 * q; p < a.ld; p += 32) {
            half8 h;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t d = p + e;
                if (d < a.dim) h[e] = valid && !always ? (_Float16)a.W[(uint64_t)d * a.ldw + col0 + l] : (_Float16)0.0f;
                else h[e] = d == a.dim ? hi : d == a.dim + 1 ? mid : d == a.dim + 2 ? lo : d == a.dim + 3 ? error : (_Float16)0.0f;
            }
            *reinterpret_cast<half8*>(a.out16 + (uint64_t)(col0 + l) * a.ld + p) = h;
        }
    }
}

struct ScreenRowsArgs {
    const float* X;
    uint32_t ldx, batch, dim, ld;
    _Float16* out16;        // [batch rounded up to 256][ld], zero filled
    const uint32_t* stats;
    float* eps;             // [batch] what a bound is lowered by
    float* slack;           // [batch] layers: and by how much more where it comes from another kernel's sums
    uint32_t* flag;         // one word (nearest neighbours) or one per row (layers): set where the error has no bound
    uint32_t* told;         // host-visible word set with it (may be NULL)
    ScreenNotes* notes;     // host-visible: what the table's columns are like (nearest neighbours)
};

// One wavefront per row.
template <bool ITEM_NORM>
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
    for (uint32_t d = lane; d < a.ld; d += kWave) {
        float x = (valid && d < a.dim) ? a.X[(uint64_t)row * a.ldx + d] : 0.0f;
        if constexpr (ITEM_NORM) {
            if (valid && d >= a.dim && d < a.dim + 3) x = 1.0f;
            if (valid && d == a.dim + 3) x = norm * 32.0f * screen_relative(a.dim) * 1.002f + 1e-7f;
        }
        a.out16[(uint64_t)row * a.ld + d] = (_Float16)x;
    }
    if (!valid || lane != 0) return;
    if (!ITEM_NORM && row == 0 && a.notes) {
        a.notes->largest = __uint_as_float(a.stats[0]);
        a.notes->sum = __uint_as_float(a.stats[1]);
        a.notes->number = a.stats[2];
    }
    const float most = __uint_as_float(a.stats[0]);
    float eps = 2.9802322e-8f * 1.01f * sqrtf((float)a.dim + 4.0f) * (ITEM_NORM ? norm : norm + most);
    if constexpr (ITEM_NORM) eps += 1e-7f;   // (the bias: its last piece is good to 2^-25)
    else eps += screen_relative(a.dim) * norm * most + (float)a.dim * 8.8817842e-16f * 1.01f;   // (a layer's 1e-7 covers the last term)
    a.eps[row] = eps;
    // The k columns that set the first bound are scored again in another order: d + d / 16 + 5 roundings of 2^-24 of |x| |w| apart at most,
    // and for the bias 2^-22 of |b| <= |x| |w| + |z|, whose |z| part the bounds' kernel takes off (a column that lies above the bound
    // keeps above it by less |z| than it has more).  (Nearest neighbours: inside the 4 d + 64 of screen_relative.)
    if constexpr (ITEM_NORM) a.slack[row] = (1.25f * (float)a.dim + 24.0f) * 5.9604645e-8f * 1.01f * norm * most;
    // (a NaN in the row: its scores are NaN everywhere, there is nothing to miss)
    const bool bad = norm > kF16Max || (!ITEM_NORM && most > kF16Max);
    if (bad) {
        a.flag[ITEM_NORM ? row : 0] = 1;
        if (a.told) *(volatile uint32_t*)a.told = 1u;
    }
}

// The bounds the screened sums are compared with: the rows' bounds, as pre-activation sums, less the error.
__global__ __launch_bounds__(256) void screen_bounds_kernel(const uint32_t* row_bound, const float* eps, const float* slack, uint32_t batch, uint32_t act,
                                                            float slope, float alpha, float lambda, uint32_t* admit)
{
    const uint32_t row = blockIdx.x * 256 + threadIdx.x;
    if (row >= batch) return;
    const uint32_t key = row_bound[row];
    const float z = preactivation_bound(key, act, slope, alpha, lambda);
    const float b = z - (eps[row] + (slack ? slack[row] : 0.0f)) * 1.001f - fabsf(z) * 2.3841858e-7f;   // (the subtraction itself is rounded)
    // a ReLU's k-th score this close to 0 may come out as 0 in the other order, and everything below 0 then ties with it
    const bool flat = slack && act == DSX_ACT_RELU && z <= slack[row];
    // no bound yet, or none that can be lowered: everything that is a number passes
    admit[row] = (key == 0 || flat || !(b >= -__builtin_inff())) ? 0u : score_key(b);
}

// Scores what passed in fp32: one workgroup per row, sixteen lanes per candidate.  The row's shared list is rewritten in place, the
// chunks' lists go behind it; a row that does not fit has a count above cap.
struct ScreenRescoreArgs {
    const float* X;
    uint32_t ldx, dim, pitch32;
    const float* rows32;
    const float* bias;
    uint32_t act;
    float slope, alpha, lambda;
    uint64_t* cand;          // [batch][cap]
    uint32_t* cand_count;
    uint32_t cap;
    uint32_t* overflow;      // nearest neighbours: set for a row that does not fit (or NULL)
    const uint64_t* seg;     // [batch][chunks][seg_cap]
    uint32_t* seg_count;     // [batch][64]
    uint32_t chunks, seg_cap;
};

__global__ __launch_bounds__(256) void screen_rescore_kernel(ScreenRescoreArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float sX[];   // the row, zeros up to a multiple of 64
    __shared__ uint32_t sStart[kWave + 1];
    const uint32_t b = blockIdx.x, lane = threadIdx.x % kWave;
    const uint32_t dpad = (a.dim + 63) / 64 * 64;
    for (uint32_t d = threadIdx.x; d < dpad; d += 256) sX[d] = (d < a.dim) ? a.X[(uint64_t)b * a.ldx + d] : 0.0f;
    const uint32_t shared = a.cand_count[b];
    if (threadIdx.x < kWave) {
        const uint32_t mine = (lane < a.chunks) ? min(a.seg_count[(uint64_t)b * kWave + lane], a.seg_cap) : 0u;
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < kWave; d *= 2) {
            const uint32_t below = __shfl_up(incl, d);
            if (lane >= (uint32_t)d) incl += below;
        }
        if (lane == 0) sStart[0] = 0;
        sStart[lane + 1] = incl;
    }
    __syncthreads();
    const uint32_t total = shared + sStart[kWave];
    if (total > a.cap) {   // the same for the whole workgroup
        if (threadIdx.x == 0) {
            a.cand_count[b] = total;
            if (a.overflow) *a.overflow = 1u;
        }
        return;
    }
    uint64_t* out = a.cand + (uint64_t)b * a.cap;
    const uint32_t sub = threadIdx.x % 16;
    for (uint32_t e0 = 0; e0 < total; e0 += 16) {
        const uint32_t e = e0 + threadIdx.x / 16;
        uint64_t word = 0;
        if (e < shared) word = out[e];
        else if (e < total) {
            const uint32_t s = e - shared;
            uint32_t lo = 0, hi = kWave;   // the last chunk that starts at or before s (empty chunks start where the next one does)
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) / 2;
                if (sStart[mid] <= s) lo = mid;
                else hi = mid;
            }
            word = a.seg[((uint64_t)b * a.chunks + lo) * a.seg_cap + (s - sStart[lo])];
        }
        const uint32_t col = ~(uint32_t)word;
        float sum = 0.0f;
        if (e < total) {
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
        if (sub == 0 && e < total) {
            const float y = activate_rt(sum + (a.bias ? a.bias[col] : 0.0f), a.act, a.slope, a.alpha, a.lambda);
            out[e] = (y == y) ? ((uint64_t)score_key(y) << 32) | (uint32_t)word : 0ull;
        }
    }
    if (threadIdx.x == 0) a.cand_count[b] = total;
}

// The same for a layer in ranges (dsx_fc_topk), fitted to 320 layers of 512 to 4,096 rows, 64 to 1,024 components, 16,384 to 1,000,000
// columns, k 10 to 256, without filters: fp32 within 23 %, screened within 31 %; none is slower than in fp32, 1.3 % are left (us,
// screened / fp32: 512 x 256 x 16,384 top 10 105 / 80, 4,096 x 1,024 x 27,278 top 256 3,977 / 2,591, 512 x 256 x 131,072 top 100
// 539 / 539, 1,000 x 256 x 131,072 top 100 658 / 831, 4,096 x 512 x 300,000 top 100 3,578 / 10,343).
bool screen_layer_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k)
{
    if (ctx().knobs.screen == 1) return true;
    const double q = batch, d = dim, ld = screen_ld(dim, true), m = (double)n;
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
    const uint64_t bytes = knn_f16_rows(n) * ((uint64_t)screen_ld(dim, layer) * 2 + (uint64_t)screen_pitch32(dim) * 4);
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

ScreenWorkspace screen_layout(void* base, uint32_t batch, uint32_t dim, uint64_t n, bool layer, uint32_t list_words)
{
    ScreenWorkspace w;
    char* p = (char*)base;
    w.items16 = p;
    p += align256(knn_f16_rows(n) * screen_ld(dim, layer) * 2);
    w.rows32 = (float*)p;
    p += align256(n * screen_pitch32(dim) * sizeof(float));
    w.queries16 = p;
    p += align256(knn_f16_rows(batch) * screen_ld(dim, layer) * 2);
    w.eps = (float*)p;
    p += align256((size_t)batch * sizeof(float));
    w.slack = (float*)p;
    p += align256((size_t)batch * sizeof(float));
    w.admit = (uint32_t*)p;
    p += align256((size_t)batch * sizeof(uint32_t));
    w.stats = (uint32_t*)p;
    p += 256;
    w.seg = (uint64_t*)p;
    p += align256((size_t)batch * list_words * sizeof(uint64_t));
    w.seg_count = (uint32_t*)p;
    p += align256((size_t)batch * 64 * sizeof(uint32_t));
    w.list_words = list_words;
    w.bytes = (size_t)(p - (char*)base);
    return w;
}

__global__ void screen_clear_kernel(uint32_t* stats) { stats[threadIdx.x] = 0; }

int screen_prepare(const ScreenWorkspace& w, const float* X, uint32_t ldx, uint32_t batch, const float* W, uint64_t ldw, const float* bias,
                   uint64_t n, uint32_t dim, bool layer, uint32_t first, uint32_t* flag, uint32_t* told, ScreenNotes* notes)
{
    hipStream_t s = ctx().stream;
    hipLaunchKernelGGL(screen_clear_kernel, dim3(1), dim3(64), 0, s, w.stats);
    ScreenItemsArgs i{};
    i.W = W; i.bias = bias; i.ldw = ldw; i.n = (uint32_t)n; i.dim = dim; i.first = layer ? first : (uint32_t)n;
    i.ld = screen_ld(dim, layer); i.pitch32 = screen_pitch32(dim);
    i.out16 = (_Float16*)w.items16; i.out32 = w.rows32; i.stats = w.stats;
    const dim3 grid((uint32_t)(knn_f16_rows(n) / 64));
    if (layer) hipLaunchKernelGGL((screen_items_kernel<true>), grid, dim3(256), 0, s, i);
    else hipLaunchKernelGGL((screen_items_kernel<false>), grid, dim3(256), 0, s, i);
    DSX_LAUNCH_CHECK("screen_items_kernel");
    ScreenRowsArgs r{};
    r.X = X; r.ldx = ldx; r.batch = batch; r.dim = dim; r.ld = i.ld;
    r.out16 = (_Float16*)w.queries16; r.stats = w.stats; r.eps = w.eps; r.slack = w.slack; r.flag = flag; r.told = told; r.notes = notes;
    const dim3 rgrid((uint32_t)(knn_f16_rows(batch) / 4));
    if (layer) hipLaunchKernelGGL((screen_rows_kernel<true>), rgrid, dim3(256), 0, s, r);
    else hipLaunchKernelGGL((screen_rows_kernel<false>), rgrid, dim3(256), 0, s, r);
    DSX_LAUNCH_CHECK("screen_rows_kernel");
    return DSX_OK;
}

int screen_candidates(const ScreenWorkspace& w, const float* X, uint32_t ldx, uint32_t batch, uint32_t dim, bool layer, const float* bias,
                      uint32_t ncols, const CandArgs& cand, bool report_overflow, bool first)
{
    hipStream_t s = ctx().stream;
    const uint32_t ld = screen_ld(dim, layer), act = layer ? cand.act : (uint32_t)DSX_ACT_LINEAR;
    hipLaunchKernelGGL(screen_bounds_kernel, dim3((batch + 255) / 256), dim3(256), 0, s, cand.row_bound, w.eps, layer && first ? w.slack : nullptr, batch, act,
                       cand.slope, cand.alpha, cand.lambda, w.admit);
    DSX_LAUNCH_CHECK("screen_bounds_kernel");
    CandArgs screened = cand;
    screened.row_bound = w.admit;
    uint32_t chunks = 0;
    int rc = knn_f16_candidates_run(w.queries16, (const char*)w.items16 + (uint64_t)cand.col_offset * ld * 2, ld, batch, ncols, screened, w.seg,
                                    w.seg_count, w.list_words, 1, &chunks);
    if (rc) return rc;
    ScreenRescoreArgs a{};
    a.X = X; a.ldx = ldx; a.dim = dim; a.pitch32 = screen_pitch32(dim);
    a.rows32 = w.rows32; a.bias = bias;
    a.act = act; a.slope = cand.slope; a.alpha = cand.alpha; a.lambda = cand.lambda;
    a.cand = cand.cand; a.cand_count = cand.cand_count; a.cap = cand.cand_cap;
    a.overflow = report_overflow ? cand.overflow : nullptr;
    a.seg = w.seg; a.seg_count = w.seg_count; a.chunks = chunks; a.seg_cap = chunks ? w.list_words / chunks : 0;
    hipLaunchKernelGGL(screen_rescore_kernel, dim3(batch), dim3(256), (dim + 63) / 64 * 64 * sizeof(float), s, a);
    DSX_LAUNCH_CHECK("screen_rescore_kernel");
    return DSX_OK;
}

}  // namespace dsx
