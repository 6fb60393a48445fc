// dsx_screen.h — 16-bit screening of the fp32 searches' candidates (dsx_screen.hip) and the f16 products behind it (dsx_f16.hip).
#pragma once
#include "dsx_device.h"
#include "dsx_internal.h"

namespace dsx {

// f16 products of a batch of rows with a range of items (dsx_f16.hip; layouts of knn_f16_ld / knn_f16_rows).
constexpr int kF16Scores = 0, kF16Layer = 1, kF16Store = 2, kI8Scores = 3, kI8Layer = 4;
constexpr uint32_t kF16ListStride = 256;   // seg_count's pitch: lists per row at most
struct F16Job {
    const void* Q;
    const void* items;        // of the range's first item, which is a multiple of 256
    uint32_t ld, batch, n;
    const float* norm;        // layers and stored sums
    const float* bias;
    const float* e1;
    float bias_raise;
    CandArgs cand;            // lists (the shared ones, which full lists spill into)
    uint64_t* seg;            // [batch][*lists][seg_words / *lists]
    uint32_t* seg_count;      // [batch][kF16ListStride]
    uint32_t seg_words;
    void* Z;                  // stored sums: halves, [batch][ldz], ldz a multiple of 256
    void* M;                  // the largest of every 32 of them, [batch][ldz / 32]
    uint64_t ldz;
    const float* scale;       // [batch] what a row's sums are multiplied by before they are stored; products of bytes: the rows' units
    const float* unit;        // products of bytes: the items' units, one for every 32 of them
    uint32_t* words;          // products of bytes: [batch][ldw], a word for every 32 items, ldw a multiple of 8
    uint64_t ldw;
};
int f16_sweep_run(const F16Job& j, bool layer, uint32_t* lists);
int f16_store_run(const F16Job& j);
// Products of bytes (Q and items of ld / 2 pairs of bytes): a word for every 32 items and row.  starts: of the biases and the columns that always pass.
int i8_best_run(const F16Job& j, bool starts);
// The same from vectors of 128, 256 or 512 bytes, for more than 256 rows (dsx_i8.hip).  side: for every 32 items what their sums start from, their unit, and
// three words of nothing; kI8SideSlack bytes more than that are read.
constexpr uint32_t kI8Side = 36, kI8SideSlack = 1024;
bool i8_wide_takes(uint32_t ld8, uint32_t batch);
int i8_wide_run(const F16Job& j, const float* side, bool starts);

// The integer sums start from this: the bits of 1.5 * 2^23, whose last one is worth 1, so that the sums are floats as they are (and in the order
// of floats): magnitudes below 2^22 (i8_unit).
constexpr int32_t kI8Start = 0x4B400000;
constexpr float kI8StartValue = 12582912.0f;
constexpr float kI8Most = 3.3e38f;   // above every sum

// What an item's sum starts from.  (Finite, as its lowest bits are taken; an item or a bias that is no number: never.)
__device__ __forceinline__ float i8_start(float bias, float norm, float bias_raise)
{
    return (bias != bias || norm != norm) ? -3e37f : (norm == __builtin_inff()) ? 3e37f : fminf(fmaxf(bias + fabsf(bias) * bias_raise, -3e37f), 3e37f);
}

// A row's word for 32 items: the largest of their sums as a half (upper 16 bits), the second largest as the upper 11 bits of a half, and in between
// the lowest 5 bits the place of the largest.  Both are upper bounds: i8_first, i8_second.
__device__ __forceinline__ uint32_t i8_word(uint32_t first, uint32_t second, uint32_t place) { return first << 16 | (second & 0xffe0u) | place; }
// Of a query's two lanes: the largest sums m0, m1 of 16 items each, their places in the lowest bits, and the second largest; p: the product of the units.
template <bool STARTS> __device__ __forceinline__ uint32_t i8_block_word(uint32_t m0, uint32_t m1, uint32_t s0, uint32_t s1, float p)
{
    const float a = __uint_as_float(m0), b = __uint_as_float(m1 | 4u);
    const float top = fmaxf(a, b), next = fmaxf(fmaxf(fminf(a, b), __uint_as_float(s0)), __uint_as_float(s1));
    const auto value = [&](float v) __attribute__((always_inline)) -> uint32_t {
        const uint32_t bits = __float_as_uint(v);
        const float raised = __uint_as_float(v < 0.0f ? bits & ~31u : bits | 31u);   // (of those with these bits but the place's, the largest)
        const float x = STARTS ? raised - kI8StartValue * p : (raised - kI8StartValue) * p;
        const _Float16 up = (_Float16)fmaxf(fmaf(fabsf(x), 4.932e-4f, x) + 6.0e-8f, -65504.0f);
        return __builtin_bit_cast(uint16_t, up);
    };
    return i8_word(value(top), value(next), __float_as_uint(top) & 31u);
}
__device__ __forceinline__ float i8_first(uint32_t word) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(word >> 16)); }
__device__ __forceinline__ float i8_second(uint32_t word)
{
    if ((word & 0x7c00u) == 0x7c00u) return (word & 0x8000u) ? -65504.0f : __builtin_inff();
    return (float)__builtin_bit_cast(_Float16, (uint16_t)((word & 0x8000u) ? word & 0xffe0u : word | 31u));
}

// The table of a screened search: two row-major copies (f16, fp32), the columns' norms and what they are like; one that is kept holds a copy in bytes
// as well where searches may go by it.  Laid out in screen_table(...).bytes bytes at base, filled by screen_build from W [dim][ldw].
struct ScreenTable {
    void* items16;
    float* rows32;
    float* norm;
    float* seg_norm;
    uint32_t* stats;
    void* items8;             // NULL: no bytes
    float* unit8;
    float2* error8;
    float* side8;             // i8_wide_run's, without biases
    size_t bytes;
};
ScreenTable screen_table(void* base, uint32_t dim, uint64_t n, bool kept);
int screen_build(const ScreenTable& t, const float* W, uint64_t ldw, uint64_t n, uint32_t dim);
// The bytes alone, of a table that is kept as halves (items16 [n rounded up to 256][knn_f16_ld(dim)], which searches score from); [6] of stats is set if
// it holds something that is no finite number, which such a search cannot take.
ScreenTable screen_table_halves(void* base, uint32_t dim, uint64_t n);
int screen_build_halves(const ScreenTable& t, const void* items16, uint64_t n, uint32_t dim);

// What a call works in.  columns: how many columns' sums there is room for, all of them or a first block's; screen_run goes by that and not by its
// own number of columns.  kept: the table has bytes, and the search goes by them where screen_in_bytes says so; one that has to be done again in halves works
// in the same bytes, laid out with kept = false.
struct ScreenWorkspace {
    uint32_t columns;
    void* rows16;
    float* e1;
    float* e0;
    float* scale;
    void* sums;
    void* most;
    uint32_t* admit;
    uint64_t* keep;
    uint32_t* keep_count;
    uint64_t* seg;
    uint32_t* seg_count;
    void* rows8;              // screened in bytes (only these are there then, else they are NULL)
    float* unit8;
    float4* error8;
    float* side8;             // i8_wide_run's, with the call's biases
    uint32_t rows;            // whose words there is room for
    uint32_t* words;
    uint2* near;
    uint2* near_found;
    size_t bytes;
};
ScreenWorkspace screen_layout(void* base, uint32_t batch, uint32_t dim, uint64_t n, uint32_t k, bool kept);

// Nearest neighbours, in pinned memory: the largest norm of the table, a sample of the norms and how many they are; whether a row
// cannot be screened, or not in bytes.
struct ScreenNotes {
    float largest, sum;
    uint32_t number, flag, open;
};

struct ScreenJob {
    const float* X;           // [batch][ldx]
    uint32_t ldx, batch, dim, n, k;
    const float* bias;        // [n] or NULL
    uint32_t act;
    float slope, alpha, lambda;
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;     // NULL: no filter
    float* keys;              // [batch][k]
    uint32_t* values;
    float* keys2;             // the same once more, in host memory that the device can write (or NULL)
    uint32_t* values2;
    uint32_t* row_flag;       // [batch] set for rows without a result (the caller computes them again), 0 for the others
    uint32_t* told;           // word that is set to 1 with the first of them (may be host memory; may be NULL)
    uint32_t* open;           // the same for those that a search in halves may have results of, as bytes alone left too much of them open (may be NULL)
    uint64_t* cand;           // [batch][cap]
    uint32_t* cand_count;     // [batch]
    uint32_t cap;
    uint32_t* overflow;       // scratch word
    uint32_t* clear;          // [clear_words] set to 0 on the way
    uint32_t clear_words;
    void (*before_last)(void*);   // called before the kernel that ends with the (last) results is launched (NULL: not)
    void* before_last_arg;
    const void* rows16;       // the table as halves: scores are products of these and of the rows rounded to halves (NULL: of floats); for searches in bytes
    bool even;                // no bias, no column that always passes or (where the table has bytes) is no number, and norms close together (screen_even)
};
// The rows in f16 (and notes of the table and the rows, NULL: none), then the search itself.
int screen_rows(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w, ScreenNotes* notes);
int screen_run(const ScreenJob& j, const ScreenTable& t, const ScreenWorkspace& w);

// Whether the bounds may be lowered by the error that the largest norm has, instead of raising every sum by its own: what passes beyond that
// is a factor of exp(4 * 2^-10 sqrt(dim) (largest / average - 1)) at most, 1.07 for 256 components.
inline bool screen_even(float largest, float average) { return largest < 60000.0f && largest <= 2.0f * average; }

// Whether an item table is fit for screening: no norm beyond f16's range, and none so far above the others that its share of the error (of the
// columns next to it, which are judged by the largest of 32 or 64) would let everything pass.
inline bool screen_fits(float largest, float average) { return largest <= 65504.0f && largest <= 64.0f * average; }

bool screen_takes(uint32_t batch, uint32_t dim, uint64_t n, bool layer);
bool screen_in_bytes(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k);
bool screen_search_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k);

}  // namespace dsx
