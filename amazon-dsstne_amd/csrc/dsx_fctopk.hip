// dsx_fctopk.hip — a fully connected output layer and the (filtered) top-K of its result in one call: the [batch x n] result is
// never stored.
//
// The reference runs the output layer into its unit buffer (cublasSgemm + bias + activation, engine/NNLayer.cpp:994-1167), copies
// the buffer to the host, multiplies the sample's own items by 0 there and runs kCalculateTopK over all n columns
// (utils/NNRecsGenerator.cpp:83-150).  Here only the first few thousand columns are produced as a matrix (a scratch block) and
// scanned: that leaves, per row, a best list and the key of its k-th score.  Every later column range, each several times as
// wide as everything before it, runs the same GEMM kernel in candidate mode: the tile's pre-activation sums are compared with
// the rows' bounds in registers and only the few survivors are activated and appended to per-row lists, which a small kernel
// folds into the best lists after dropping the columns the row's filter names (a row whose result a listed column's score * 0
// could enter - fewer than k scores above 0 - is recomputed with those zeros in place).  Exact for any input: admission is a superset
// of "score >= current k-th score" (preactivation_bound in dsx_device.h), lists are merged under the total order (score
// descending, column ascending), and a row whose list fills up is recomputed from scratch on the device.
#include <algorithm>
#include "dsx_screen.h"

namespace dsx {

constexpr uint32_t kLayerCandCap = 4096;       // candidate words per row and column range
static LibScratch g_layer_ws_of[DSX_MAX_LANES];   // per lane
// Pinned host memory: the device stores 1 in a word when it flags a row.  One word per weight matrix (the layer a call belongs
// to), so that one layer's tied scores say nothing about another's; kFlagWords matrices at a time, the oldest gives way.
constexpr int kFlagWords = 64;
static uint32_t* g_layer_flagged = nullptr;
static const void* g_flag_owner[kFlagWords] = {};
static int g_flag_next = 0;
// Behind them, per matrix too, a word that is stored when bytes leave rows open, and what follows from it: how many calls are still to go in halves, and
// how many were to when it last happened (KnnData does the same).
constexpr uint32_t kHalvesMost = 1024;
static uint32_t g_halves_left[kFlagWords] = {}, g_halves_next[kFlagWords] = {};
static bool g_bytes_last[kFlagWords] = {};   // the last call went in bytes

static void layer_flags_release()
{
    if (g_layer_flagged) hipHostFree(g_layer_flagged);
    g_layer_flagged = nullptr;
    for (auto& o : g_flag_owner) o = nullptr;
    g_flag_next = 0;
}

static int layer_flag_slot(const void* W, bool create)
{
    for (int i = 0; i < kFlagWords; i++)
        if (g_flag_owner[i] == W) return i;
    if (!create) return -1;
    const int i = g_flag_next;
    g_flag_next = (g_flag_next + 1) % kFlagWords;
    g_flag_owner[i] = W;
    *(volatile uint32_t*)&g_layer_flagged[i] = 0;
    *(volatile uint32_t*)&g_layer_flagged[kFlagWords + i] = 0;
    g_halves_left[i] = g_halves_next[i] = 0;
    g_bytes_last[i] = false;
    return i;
}

// Whether a call that could go in bytes goes in halves, as rows of a call before it were left open.  (Rows that bytes leave open are computed again in fp32,
// 32 at a time: little for one of them, several times what halves take where all of a batch are.)
static bool layer_in_halves(int slot)
{
    volatile uint32_t* open = g_layer_flagged + kFlagWords + slot;
    if (g_halves_left[slot] != 0) {
        g_halves_left[slot]--;
        return true;
    }
    const bool was_open = *open != 0, before = g_bytes_last[slot];
    g_bytes_last[slot] = !was_open;
    if (!was_open) {   // (the call before may not have come that far)
        if (before) g_halves_next[slot] /= 2;
        return false;
    }
    *open = 0;
    g_halves_next[slot] = std::min(kHalvesMost, std::max(1u, 4 * g_halves_next[slot]));
    g_halves_left[slot] = g_halves_next[slot] - 1;
    return true;
}

__global__ __launch_bounds__(256) void layer_clear_kernel(uint32_t* p, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

static inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

static uint32_t layer_first_columns(uint32_t n, uint32_t k)
{
    uint32_t c = ctx().knobs.fc_topk_first_columns ? ctx().knobs.fc_topk_first_columns : 2048;
    c = std::max(c, (k + 127) / 128 * 128);   // at least k candidates for the first bound
    c = (c + 127) / 128 * 128;
    // when the first block would be most of the layer anyway, the whole layer goes through the scratch matrix
    return (n <= c + c / 2) ? n : c;
}

struct LayerWorkspace {
    float* block_scores;   // [batch][ld0]
    uint64_t* best;        // [batch][k]
    uint32_t* row_bound;   // [batch]   (row_bound, cand_count, row_flag, overflow and redo_done are cleared together)
    uint32_t* cand_count;  // [batch]
    uint32_t* row_flag;    // [batch]
    uint32_t* overflow;    // [64] unused flag word of the shared epilogue
    uint32_t* redo_done;   // [layer_redo_groups]
    uint64_t* cand;        // [batch][cap]; after the last range: the lists of rows that are computed again
    ScreenTable table;     // where the layer is screened in 16 bits: the table, if the caller keeps none, and what the call works in
    ScreenWorkspace screen;
    size_t bytes;
};

static size_t layer_clear_words(uint32_t batch) { return (size_t)3 * batch + 64 + layer_redo_groups(batch); }

// screened: 0 no, 1 yes, 2 yes and the caller has the table
static LayerWorkspace layer_layout(void* base, uint32_t batch, uint32_t n0, uint32_t k, uint32_t cap, bool ranges, int screened,
                                   uint32_t kdim, uint32_t n)
{
    LayerWorkspace w;
    char* p = (char*)base;
    const uint32_t ld0 = (n0 + 3) / 4 * 4;
    w.block_scores = (float*)p;
    if (!screened) p += align256((size_t)batch * ld0 * sizeof(float));
    w.best = (uint64_t*)p;
    if (!screened) p += align256((size_t)batch * k * sizeof(uint64_t));
    w.row_bound = (uint32_t*)p;
    w.cand_count = w.row_bound + batch;
    w.row_flag = w.cand_count + batch;
    w.overflow = w.row_flag + batch;
    w.redo_done = w.overflow + 64;
    p += align256(layer_clear_words(batch) * sizeof(uint32_t));
    w.cand = (uint64_t*)p;
    if (ranges) p += align256(std::max<size_t>((size_t)batch * cap, layer_redo_words(batch, k)) * sizeof(uint64_t));
    w.table = ScreenTable{};
    w.screen = ScreenWorkspace{};
    if (screened) {
        w.screen = screen_layout(p, batch, kdim, n, k, screened == 2);
        p += w.screen.bytes;
    }
    if (screened == 1) {
        w.table = screen_table(p, kdim, n, false);
        p += w.table.bytes;
    }
    w.bytes = (size_t)(p - (char*)base);
    return w;
}

static bool layer_activation_supported(uint32_t act, const dsx_act_params* params)
{
    switch (act) {
    case DSX_ACT_SIGMOID:
    case DSX_ACT_TANH:
    case DSX_ACT_RELU:
    case DSX_ACT_LINEAR: return true;
    case DSX_ACT_LRELU: return (params ? params->slope : 0.01f) > 0.0f;
    default: return false;
    }
}

}  // namespace dsx

using namespace dsx;

extern "C" {

int dsx_testing_set_fc_topk_first_columns(uint32_t columns)
{
    ctx().knobs.fc_topk_first_columns = std::min(columns, 131072u);   // the first block's filter bitmap lives in LDS
    return DSX_OK;
}

int dsx_testing_set_fc_topk_candidate_capacity(uint32_t words)
{
    DSX_CHECK_ARG(words == 0 || (words >= 64 && words <= kLayerCandCap), "dsx_testing_set_fc_topk_candidate_capacity: %u words (64..%u)", words, kLayerCandCap);
    ctx().knobs.fc_topk_candidate_capacity = words;
    return DSX_OK;
}

int dsx_fc_topk_flagged(int reset)
{
    if (!g_layer_flagged) return 0;
    int seen = 0;
    for (int i = 0; i < kFlagWords; i++) {
        seen |= *(volatile uint32_t*)&g_layer_flagged[i] != 0;
        if (reset) *(volatile uint32_t*)&g_layer_flagged[i] = 0;
    }
    return seen;
}

int dsx_fc_topk_flagged_for(const float* W, int reset)
{
    if (!g_layer_flagged) return 0;
    const int i = layer_flag_slot(W, false);
    if (i < 0) return 0;
    const int seen = *(volatile uint32_t*)&g_layer_flagged[i] != 0;
    if (reset) *(volatile uint32_t*)&g_layer_flagged[i] = 0;
    return seen;
}

// Where the line lies (us, layer stored and guided top-K / this call, filter of 144 columns a row that score high):
//   From 131,072 columns on always, but for batches of up to 64: those are bound by reading the layer's weights once; storing their
//   scores and maxima adds little to that, and this call's tiles of 128 rows a lot (8 x 256 x 500,000, top 50: 135 / 440).  It is the memory that the
//   scores would take as much as the time: 512 x 256 x 131,072 top 10 347 / 229, but layers too small to be screened take longer (512 x 64 x 131,072
//   top 10 147 / 347).
//   Narrower layers where they are screened, and large: 4,096 x 1,024 x 27,278 top 10 1,861 / 524, 2,048 x 512 x 27,278 529 / 187, 4,096 x 128 x
//   60,000 734 / 305; top 100 4,096 x 1,024 x 27,278 1,927 / 718, 4,096 x 512 x 60,000 2,108 / 654.  (Smaller ones gain too, 1,024 x 1,024 x 27,278 530 / 262,
//   but pay for the table with every batch; with a kept one the line is the one below.)  Sigmoids only: their scores are above 0, so that no row has
//   to be computed again for a listed column's zero.
int dsx_fc_topk_pays(uint32_t batch, uint32_t k_dim, uint32_t n, uint32_t activation, uint32_t k)
{
    if (n >= 131072) return batch > 64;
    const double products = (double)batch * k_dim * n;
    return activation == DSX_ACT_SIGMOID && screen_takes(batch, k_dim, n, true) &&
           ((k <= 32 && batch >= 1536 && products >= 2e10) || (k <= 128 && batch >= 2048 && products >= 1e11));
}

// Where the line lies (us a batch; the layer stored and its guided top-K, or ranges in fp32 / screened by a kept table; filter of 144
// columns a row, nets of one hidden layer, four batches after each other or, up to 128 rows of top 20, one by itself):
//   More than 128 rows: 169 nets of 64 to 1,024 hidden units, 8,192 to 100,000 columns, 512 to 4,096 rows, top 10 and top 100, fitted:
//   what is gained grows with the columns' scores that are not stored as floats (0.6 us a million) and with the products (2.5 us
//   a thousand million); what it costs is three more launches and, for large k, candidates of long rows.  512 x 64 x 8,192 top 100 40 / 48 and top
//   10 27 / 30, 512 x 128 x 8,192 top 10 32 / 32, 512 x 64 x 16,384 top 100 57 / 51, 512 x 512 x 8,192 top 100 76 / 65, 1,024 x 128 x
//   27,278 top 10 98 / 51, 4,096 x 64 x 8,192 top 10 95 / 85, 1,024 x 1,024 x 60,000 top 10 979 / 220.
//   65 to 128 rows: where the layer is wide.  128 x 1,024 x 8,192 91 / 110, 128 x 64 x 27,278 59 / 68, 128 x 256 x 27,278 83 / 81, 128 x
//   1,024 x 27,278 141 / 94, 128 x 64 x 100,000 77 / 70, 128 x 256 x 500,000 461 / 170.
//   Up to 64 rows: both read the weights once, and half as many bytes of them only pay where they come from memory and there are tiles for
//   the whole GPU.  32 x 1,024 x 27,278 73 / 83, 1 x 64 x 100,000 55 / 55, 8 x 64 x 500,000 81 / 85, 8 x 256 x 100,000 73 / 65, 8 x
//   256 x 500,000 154 / 114, 8 x 1,024 x 100,000 145 / 98.
// Sigmoids only, as above, but for layers that are never stored; with few rows the rest of the weights' cost would be paid again for one.
int dsx_fc_topk_screened_pays(uint32_t batch, uint32_t k_dim, uint32_t n, uint32_t activation, uint32_t k)
{
    if (batch == 0 || k > 256 || n < 64 * k || n < 8192 || n >= 1u << 28 || k_dim < 32 || k_dim > 4096) return 0;
    if (activation != DSX_ACT_SIGMOID && (n < 131072 || batch <= 64)) return 0;
    const double q = batch, d = k_dim, m = n;
    if (batch <= 64) return n >= 65536 && k_dim >= 128 && m * d >= 2.5e7;
    if (batch <= 128) return n >= 24576 && m * d >= 6e6;
    return q * m * (6e-7 + 2.5e-9 * d) > 6.0 + 0.013 * k;
}

int dsx_fc_topk_supported(uint32_t ldx, const float* X, uint32_t activation, const dsx_act_params* params, const float* filter_mul)
{
    return layer_activation_supported(activation, params) && filter_mul == nullptr && ((uintptr_t)X % 16) == 0 && (ldx % 4) == 0;
}

}  // extern "C"

static int layer_flags_ready()
{
    if (g_layer_flagged) return DSX_OK;
    DSX_HIP(hipHostMalloc((void**)&g_layer_flagged, 2 * kFlagWords * sizeof(uint32_t), hipHostMallocMapped));
    for (int i = 0; i < 2 * kFlagWords; i++) g_layer_flagged[i] = 0;
    at_shutdown(layer_flags_release);
    return DSX_OK;
}

// x_planes / w_planes (both or neither): the operands as dsx_fc_split leaves them; the products then come from the split-product
// kernel.  X and W are needed either way (rows whose lists fill up are recomputed from them, in fp32).
static int fc_topk_common(const float* X, uint32_t ldx, const float* W, const float* bias, uint32_t batch, uint32_t kdim, uint32_t n,
                          uint32_t activation, const dsx_act_params* params, uint32_t k, float* keys, uint32_t* values, uint32_t position,
                          const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end, const uint32_t* filter_index,
                          const void* x_planes, const void* w_planes, const void* table)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(X && W && keys && values, "dsx_fc_topk: null device pointer");
    DSX_CHECK_ARG(kdim > 0 && n > 0 && ldx >= kdim, "dsx_fc_topk: k = %u, n = %u, ldx = %u", kdim, n, ldx);
    DSX_CHECK_ARG(k >= 1 && k <= 256, "dsx_fc_topk: k = %u is outside 1..256", k);
    DSX_CHECK_ARG(!filter_index || (filter_start && filter_end), "dsx_fc_topk: filter_index without filter_start / filter_end");
    if (!dsx_fc_topk_supported(ldx, X, activation, params, nullptr))
        return set_error(DSX_EUNSUPPORTED, "dsx_fc_topk: activation %u is not monotone (sigmoid, tanh, ReLU, leaky ReLU with a positive slope, "
                         "linear are), or X is not 16-byte aligned with a pitch that is a multiple of 4: use dsx_fc_forward + dsx_topk_filtered",
                         activation);
    if (batch == 0) return DSX_OK;
    if (int rc = layer_flags_ready()) return rc;
    const int slot = layer_flag_slot(W, true);
    uint32_t* const flag_word = g_layer_flagged + slot;
    const uint32_t cap = ctx().knobs.fc_topk_candidate_capacity ? ctx().knobs.fc_topk_candidate_capacity : kLayerCandCap;   // tests lower it to reach the overflow path with small inputs
    const uint32_t n0 = layer_first_columns(n, k);
    const bool ranges = n0 < n;
    int screened = x_planes ? 0 : table ? 2 : (ranges && screen_takes(batch, kdim, n, true)) ? 1 : 0;
    LibScratch& ws = g_layer_ws_of[current_lane()];
    int reserved = lib_scratch_reserve(ws, layer_layout(nullptr, batch, n0, k, cap, ranges || screened, screened, kdim, n).bytes, "dsx_fc_topk workspace", screened);
    if (reserved == DSX_ENOMEM && screened) {   // the 16-bit copies (up to 8 GiB) or the sums do not fit beside what is there: fp32 ranges need none
        screened = 0;
        reserved = lib_scratch_reserve(ws, layer_layout(nullptr, batch, n0, k, cap, ranges, screened, kdim, n).bytes, "dsx_fc_topk workspace");
    }
    if (reserved) return reserved;
    LayerWorkspace w = layer_layout(ws.ptr, batch, n0, k, cap, ranges || screened, screened, kdim, n);
    if (w.screen.words && layer_in_halves(slot)) w.screen = screen_layout(w.screen.rows8, batch, kdim, n, k, false);
    LayerRedo redo{};
    redo.X = X; redo.W = W; redo.bias = bias; redo.ldx = ldx; redo.ldw = n; redo.kdim = kdim; redo.n = n; redo.k = k;
    redo.act = activation;
    redo.slope = params ? params->slope : 0.01f;
    redo.alpha = params ? params->alpha : 1.0f;
    redo.lambda = params ? params->lambda : 1.0f;
    redo.position = position; redo.index = index; redo.fstart = filter_start; redo.fend = filter_end; redo.fidx = filter_index;
    redo.row_flag = w.row_flag; redo.partial = w.cand; redo.done = w.redo_done; redo.keys = keys; redo.values = values;
    if (screened) {
        const ScreenTable t = table ? screen_table(const_cast<void*>(table), kdim, n, true) : w.table;
        int rc = table ? DSX_OK : screen_build(t, W, n, n, kdim);
        if (rc) return rc;
        ScreenJob j{};
        j.X = X; j.ldx = ldx; j.batch = batch; j.dim = kdim; j.n = n; j.k = k;
        j.bias = bias; j.act = activation; j.slope = redo.slope; j.alpha = redo.alpha; j.lambda = redo.lambda;
        j.position = position; j.index = index; j.fstart = filter_start; j.fend = filter_end; j.fidx = filter_index;
        j.keys = keys; j.values = values;
        j.row_flag = w.row_flag; j.told = flag_word; j.open = flag_word + kFlagWords;
        j.cand = w.cand; j.cand_count = w.cand_count; j.cap = cap; j.overflow = w.overflow;
        j.clear = w.overflow; j.clear_words = 64 + layer_redo_groups(batch);   // (overflow and redo_done)
        if ((rc = screen_rows(j, t, w.screen, nullptr))) return rc;
        if ((rc = screen_run(j, t, w.screen))) return rc;
        return layer_redo_run(redo, batch);
    }
    const uint32_t ld0 = (n0 + 3) / 4 * 4;
    hipStream_t s = ctx().stream;

    // first block: the layer as a matrix, then the scanning top-K (filtered: indexes beyond the block are ignored)
    const uint32_t wrows = split_rows_padded(n);
    FcOrder order;
    order.as_candidates = ranges;
    int rc = x_planes ? fc_split_run(x_planes, w_planes, wrows, 0, bias, w.block_scores, ld0, batch, kdim, n0, 0, activation, params, nullptr, nullptr)
                      : fc_run(X, ldx, W, n, 0, bias, w.block_scores, ld0, batch, kdim, n0, 0, activation, params, nullptr, nullptr, nullptr, order);
    if (rc) return rc;
    if (!ranges)
        return topk_run(w.block_scores, ld0, n0, batch, k, keys, values, position, index, filter_start, filter_end, filter_index, nullptr, 0,
                        nullptr, 0, 0, 0);
    const uint32_t clear_words = (uint32_t)layer_clear_words(batch);
    hipLaunchKernelGGL(layer_clear_kernel, dim3((clear_words + 255) / 256), dim3(256), 0, s, w.row_bound, clear_words);
    DSX_LAUNCH_CHECK("layer_clear_kernel");
    rc = topk_run(w.block_scores, ld0, n0, batch, k, nullptr, nullptr, position, index, filter_start, filter_end, filter_index, nullptr, 0,
                  w.best, 1, 0, 1, w.row_bound);
    if (rc) return rc;

    // A bound taken over `done` columns lets about k * width / done of the next `width` columns pass: ranges grow by a factor that
    // keeps that near an eighth of a list (the sample's own items, which score high and pass as well, come on top).
    const uint32_t growth = std::max(4u, cap / (8 * k));
    uint32_t done = n0;
    while (done < n) {
        uint32_t ncols = (uint32_t)std::min<uint64_t>((uint64_t)n - done, (uint64_t)done * growth / 128 * 128);
        if (n - done - ncols < 128) ncols = n - done;   // no sliver of a last range
        CandArgs cand{};
        cand.row_bound = w.row_bound;
        cand.cand = w.cand;
        cand.cand_count = w.cand_count;
        cand.cand_cap = cap;
        cand.col_offset = done;
        cand.overflow = w.overflow;
        cand.act = activation;
        cand.slope = params ? params->slope : 0.01f;
        cand.alpha = params ? params->alpha : 1.0f;
        cand.lambda = params ? params->lambda : 1.0f;
        rc = x_planes ? fc_split_candidates_run(x_planes, w_planes, wrows, done, batch, kdim, ncols, cand, true, bias ? bias + done : nullptr)
                      : fc_layer_candidates_run(X, ldx, W + done, n, bias ? bias + done : nullptr, batch, kdim, ncols, cand);
        if (rc) return rc;
        done += ncols;
        LayerRefresh r{};
        r.best = w.best; r.cand = w.cand; r.cand_count = w.cand_count; r.cap = cap; r.k = k;
        r.row_bound = w.row_bound; r.row_flag = w.row_flag; r.flagged_total = flag_word;
        r.position = position; r.index = index; r.fstart = filter_start; r.fend = filter_end; r.fidx = filter_index;
        if (done == n) {
            r.keys = keys;
            r.values = values;
        }
        r.n = n; r.first_columns = n0;
        rc = layer_refresh_run(r, batch);
        if (rc) return rc;
    }
    return layer_redo_run(redo, batch);
}

extern "C" {

int dsx_fc_topk(const float* X, uint32_t ldx, const float* W, const float* bias, uint32_t batch, uint32_t kdim, uint32_t n,
                uint32_t activation, const dsx_act_params* params, uint32_t k, float* keys, uint32_t* values, uint32_t position,
                const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end, const uint32_t* filter_index)
{
    return fc_topk_common(X, ldx, W, bias, batch, kdim, n, activation, params, k, keys, values, position, index, filter_start, filter_end,
                          filter_index, nullptr, nullptr, nullptr);
}

uint64_t dsx_screen_table_bytes(uint32_t n, uint32_t kdim)
{
    return screen_table(nullptr, kdim, n, true).bytes;
}

int dsx_screen_table_build(const float* W, uint32_t ldw, uint32_t n, uint32_t kdim, void* table)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(W && table, "dsx_screen_table_build: null device pointer");
    DSX_CHECK_ARG(((uintptr_t)table % 256) == 0, "dsx_screen_table_build: the table is not 256-byte aligned");
    DSX_CHECK_ARG(n > 0 && n < 1u << 28 && kdim > 0 && kdim <= 4096 && ldw >= n, "dsx_screen_table_build: n = %u, k = %u, ldw = %u", n, kdim, ldw);
    return screen_build(screen_table(table, kdim, n, true), W, ldw, n, kdim);
}

int dsx_fc_topk_screened_reserve(int lane, uint32_t batch, uint32_t kdim, uint32_t n, uint32_t k)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(lane >= 0 && lane < DSX_MAX_LANES, "dsx_fc_topk_screened_reserve: lane %d (0..%d)", lane, DSX_MAX_LANES - 1);
    DSX_CHECK_ARG(batch > 0 && kdim > 0 && kdim <= 4096 && n > 0 && n < 1u << 28 && k >= 1 && k <= 256, "dsx_fc_topk_screened_reserve: batch %u, k_dim %u, n %u, k %u",
                  batch, kdim, n, k);
    if (int rc = layer_flags_ready()) return rc;
    const uint32_t cap = ctx().knobs.fc_topk_candidate_capacity ? ctx().knobs.fc_topk_candidate_capacity : kLayerCandCap;
    LibScratch& ws = g_layer_ws_of[lane];
    size_t bytes = layer_layout(nullptr, batch, layer_first_columns(n, k), k, cap, true, 2, kdim, n).bytes;
    // (a shorter last batch may go in halves where full ones go in bytes, whose scratch is not always the larger)
    if (screen_in_bytes(batch, kdim, n, k))
        for (uint32_t b = 1; b < batch; b++) bytes = std::max(bytes, layer_layout(nullptr, b, layer_first_columns(n, k), k, cap, true, 2, kdim, n).bytes);
    if (ws.ptr && bytes > ws.bytes)
        if (int rc = dsx_sync()) return rc;   // (the lane need not be the selected one, which is what growing waits for)
    return lib_scratch_reserve(ws, bytes, "dsx_fc_topk workspace", true);
}

int dsx_fc_topk_screened(const float* X, uint32_t ldx, const float* W, const void* table, const float* bias, uint32_t batch, uint32_t kdim,
                         uint32_t n, uint32_t activation, const dsx_act_params* params, uint32_t k, float* keys, uint32_t* values,
                         uint32_t position, const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end,
                         const uint32_t* filter_index)
{
    DSX_CHECK_ARG(table && ((uintptr_t)table % 256) == 0, "dsx_fc_topk_screened: the table is missing or not 256-byte aligned");
    DSX_CHECK_ARG(kdim <= 4096 && n < 1u << 28, "dsx_fc_topk_screened: k = %u (4,096 at most), n = %u (below 2^28)", kdim, n);
    return fc_topk_common(X, ldx, W, bias, batch, kdim, n, activation, params, k, keys, values, position, index, filter_start, filter_end,
                          filter_index, nullptr, nullptr, table);
}

int dsx_fc_topk_split(const float* X, uint32_t ldx, const float* W, const void* x_planes, const void* w_planes, const float* bias,
                      uint32_t batch, uint32_t kdim, uint32_t n, uint32_t activation, const dsx_act_params* params, uint32_t k, float* keys,
                      uint32_t* values, uint32_t position, const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end,
                      const uint32_t* filter_index)
{
    DSX_CHECK_ARG(x_planes && w_planes, "dsx_fc_topk_split: null planes");
    DSX_CHECK_ARG(((uintptr_t)x_planes % 16) == 0 && ((uintptr_t)w_planes % 16) == 0, "dsx_fc_topk_split: planes must be 16-byte aligned");
    return fc_topk_common(X, ldx, W, bias, batch, kdim, n, activation, params, k, keys, values, position, index, filter_start, filter_end,
                          filter_index, x_planes, w_planes, nullptr);
}

}  // extern "C"
