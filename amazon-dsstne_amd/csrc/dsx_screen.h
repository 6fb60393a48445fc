// dsx_screen.h — 16-bit screening of the fp32 searches' candidates (dsx_screen.hip) and the f16 products behind it (dsx_f16.hip).
#pragma once
#include "dsx_device.h"
#include "dsx_internal.h"

namespace dsx {

// f16 products of a batch of rows with a range of items (dsx_f16.hip; layouts of knn_f16_ld / knn_f16_rows).
constexpr int kF16Scores = 0, kF16Layer = 1, kF16Store = 2;
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
    const float* scale;       // [batch] what a row's sums are multiplied by before they are stored
};
int f16_sweep_run(const F16Job& j, bool layer, uint32_t* lists);
int f16_store_run(const F16Job& j);

// The table of a screened search: two row-major copies (f16, fp32), the columns' norms and what they are like.  Laid out in
// screen_table(...).bytes bytes at base, filled by screen_build from W [dim][ldw].
struct ScreenTable {
    void* items16;
    float* rows32;
    float* norm;
    float* seg_norm;
    uint32_t* stats;
    size_t bytes;
};
ScreenTable screen_table(void* base, uint32_t dim, uint64_t n);
int screen_build(const ScreenTable& t, const float* W, uint64_t ldw, uint64_t n, uint32_t dim);

// What a call works in.  columns: how many columns' sums there is room for, all of them or a first block's; screen_run goes by that and not by its
// own number of columns.
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
    size_t bytes;
};
ScreenWorkspace screen_layout(void* base, uint32_t batch, uint32_t dim, uint64_t n, uint32_t k);

// Nearest neighbours, in pinned memory: the largest norm of the table, a sample of the norms and how many they are; whether a row
// cannot be screened.
struct ScreenNotes {
    float largest, sum;
    uint32_t number, flag;
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
    uint64_t* cand;           // [batch][cap]
    uint32_t* cand_count;     // [batch]
    uint32_t cap;
    uint32_t* overflow;       // scratch word
    uint32_t* clear;          // [clear_words] set to 0 on the way
    uint32_t clear_words;
    void (*before_last)(void*);   // called before the kernel that ends with the results is launched (NULL: not)
    void* before_last_arg;
    bool even;                // no bias, no column that always passes, and norms close together (screen_even)
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
bool screen_search_pays(uint32_t batch, uint32_t dim, uint64_t n, uint32_t k);

}  // namespace dsx
