// dsx_knn.hip — device part of the exact KNN search: scores = queries . items^T, then the k best items per query.
//
// The first column block of the item table goes through the fp32 MFMA GEMM into a scratch score matrix and the scanning
// top-K; its k-th score per query is a lower bound of the query's final k-th score.  From there on the score matrix is never
// written: the same GEMM kernel runs in candidate mode, where a tile is only compared with the rows' bounds and the few
// scores that reach them are appended to per-query candidate lists.  After every column range (each four times as wide as
// everything before it, so that a range leaves about 4 k candidates per query) a small kernel folds the candidates into
// the query's best list and raises its bound.  Results are exact for any input: a list that fills up (items sorted by
// score, say) raises a flag that the host reads at the end, and the search is then redone block by block — GEMM into the
// scratch matrix, scanning top-K into packed partial lists with the running bound, one merge — which is also the path
// taken while the stream is being captured into a graph (no host read-back there; the caller then passes its own workspace,
// the library's would have to be allocated inside the capture) and for operands that are not 16-byte aligned, unless they are screened
// (dsx_screen.hip).  With fp16 storage (dsx_knn_search_f16) the scores come from the f16 MFMA kernel of dsx_knn_f16.hip instead, through
// the same three steps.
#include <algorithm>
#include <cstring>
#include <vector>
#include <hip/hip_runtime.h>
#include "dsx_screen.h"

namespace dsx {

static LibScratch g_knn_ws_of[DSX_MAX_LANES];   // per lane

static int g_knn_last_path = 0;            // how the last search ran: DSX_KNN_PATH_*
static int g_knn_last_repeated = 0;   // it was screened for nothing (1), or in bytes for nothing (2)

static uint32_t knn_block_columns(uint32_t rows_padded, uint32_t num_queries)
{
    // about 1 GiB of scores per block, a multiple of 1024 columns
    uint64_t cols = ((uint64_t)1 << 30) / ((uint64_t)std::max(1u, num_queries) * sizeof(float));
    if (ctx().knobs.knn_block_columns) cols = ctx().knobs.knn_block_columns;
    cols = std::max<uint64_t>(1024, cols / 1024 * 1024);
    cols = std::min<uint64_t>(cols, ((uint64_t)rows_padded + 1023) / 1024 * 1024);
    return (uint32_t)cols;
}

static inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// a fill kernel rather than hipMemsetAsync (memset nodes of a captured graph are not trusted on this hardware pool)
__global__ __launch_bounds__(256) void knn_clear_kernel(uint32_t* p, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

constexpr uint32_t kCandCap = 4096;   // candidate words per query and column range

struct KnnWorkspace {
    float* block_scores;
    float* seg_max;         // [queries][block columns / 64], few queries only: maxima of the block's 64-column segments
    uint64_t* partial;      // block path: [queries][lists of all blocks][k]; candidate path: [queries][k], the best lists
    uint32_t* row_bound;    // [queries] key of a score that k items seen so far reach; later columns admit nothing below it
    uint32_t* cand_count;   // [queries]
    uint32_t* overflow;     // [1] (+ padding)
    uint64_t* cand;         // [queries][kCandCap]
    void* queries16;        // fp16 storage: the query batch, [queries rounded up to 256][ld] halves; split products: its bf16 planes
    uint64_t* seg;          // fp16 storage only: [queries][lists][kCandCap / lists], the lists of a sweep in f16
    uint32_t* seg_count;    // fp16 storage only: [queries][kF16ListStride]
    ScreenTable table;      // fp32 storage, where screen_takes says so: at the workspace's start, whatever the number of queries
    ScreenWorkspace screen;
    uint32_t* row_flag;     // [queries] screened: rows without a result
    size_t bytes;
};

// A search of few queries is bound by reading the table once: its scores are stored (64 queries x 1,000,000 items: 256 MB against
// 512 MB of table at 128 components) by the kernel for few rows, which leaves segment maxima for the top-K.
static bool knn_few_queries(uint32_t num_queries) { return num_queries <= 64; }

// Lists per query that the top-K of a block of ncols columns leaves: enough workgroups per query to fill the GPU.
static bool knn_block_guided(uint32_t num_queries, uint32_t ncols, uint32_t k) { return knn_few_queries(num_queries) && topk_guided_pays(num_queries, ncols, k); }
static uint32_t knn_block_lists(uint32_t num_queries, uint32_t ncols, uint32_t k)
{
    return knn_block_guided(num_queries, ncols, k) ? topk_guided_parts(ncols, num_queries) : topk_segments(num_queries, ncols, false);
}

static bool knn_screens(uint32_t rows_padded, uint32_t num_queries, uint32_t k, uint32_t dim)
{
    return screen_takes(num_queries, dim, rows_padded, false) && screen_search_pays(num_queries, dim, rows_padded, k);
}

static KnnWorkspace knn_layout(void* base, uint32_t rows_padded, uint32_t num_queries, uint32_t k, bool f16 = false, uint32_t dim = 0,
                               bool split = false, bool screen = true, bool table = false)
{
    const uint32_t cb = knn_block_columns(rows_padded, num_queries);
    const uint32_t blocks = (rows_padded + cb - 1) / cb;
    KnnWorkspace w;
    char* p = (char*)base;
    screen = screen && !f16 && !split && (table || knn_screens(rows_padded, num_queries, k, dim));
    w.table = ScreenTable{};
    if (screen || table) {
        w.table = screen_table(p, dim, rows_padded, table);
        p += w.table.bytes;
    }
    w.block_scores = (float*)p;
    p += align256((size_t)num_queries * cb * sizeof(float));
    w.seg_max = knn_few_queries(num_queries) ? (float*)p : nullptr;
    if (w.seg_max) p += align256((size_t)num_queries * ((cb + 63) / 64) * sizeof(float));
    w.partial = (uint64_t*)p;
    // (a last block narrower than the others may be cut into more parts than they are, but not into more than fill half the GPU)
    const uint32_t lists = std::max(knn_block_lists(num_queries, cb, k), std::max(topk_segments(num_queries, cb, false), (uint32_t)ctx().num_cus / (2 * std::max(1u, num_queries)) + 2));
    p += align256((size_t)num_queries * blocks * lists * k * sizeof(uint64_t));
    w.row_bound = (uint32_t*)p;             // row_bound, cand_count, row_flag and overflow are cleared together
    w.cand_count = w.row_bound + num_queries;
    w.row_flag = w.cand_count + num_queries;
    w.overflow = w.row_flag + num_queries;
    p += align256(((size_t)3 * num_queries + 64) * sizeof(uint32_t));
    w.cand = (uint64_t*)p;
    p += align256((size_t)num_queries * kCandCap * sizeof(uint64_t));
    w.queries16 = p;
    w.seg = nullptr;
    w.seg_count = nullptr;
    if (f16) {
        p += align256((size_t)knn_f16_rows(num_queries) * knn_f16_ld(dim) * 2);
        w.seg = (uint64_t*)p;
        p += align256((size_t)num_queries * kCandCap * sizeof(uint64_t));
        w.seg_count = (uint32_t*)p;
        p += align256((size_t)num_queries * kF16ListStride * sizeof(uint32_t));
    }
    if (split) p += align256((size_t)split_plane_bytes(num_queries, dim));
    w.screen = ScreenWorkspace{};
    if (screen) {
        w.screen = screen_layout(p, num_queries, dim, rows_padded, k, table);
        p += w.screen.bytes;
    }
    w.bytes = (size_t)(p - (char*)base);
    return w;
}

// What a search of any number of queries up to num_queries needs: a workspace of a batch is used for smaller ones too, and fewer
// queries may need more (5,000 rows, k = 100: 64 queries 3.634 MB, 65 queries 3.618, because 64 leave more lists per query).
// About 40 ns per query count, once per table.
static size_t knn_workspace_most(uint32_t rows_padded, uint32_t num_queries, uint32_t k, bool f16, uint32_t dim, bool split, bool screen = true)
{
    size_t most = 0;
    for (uint64_t q = std::min(1u, num_queries); q <= num_queries; q++)
        most = std::max(most, knn_layout(nullptr, rows_padded, (uint32_t)q, k, f16, dim, split, screen).bytes);
    return most;
}

// Where the scores of a column range come from: the fp32 table through fc_gemm_kernel, or the fp16 table through knn_f16_kernel.
struct KnnOperands {
    bool f16 = false;
    bool split = false;                 // fp32 products from bf16 matrix instructions: item_planes / query_planes (dsx_fc_split)
    const void* item_planes = nullptr;
    const void* query_planes = nullptr;
    const float* items = nullptr;       // fp32: column-major [dim][rows_padded]
    const float* queries = nullptr;     // fp32: [queries][dim]
    const char* items16 = nullptr;      // fp16: [rows rounded up to 256][ld]
    const void* queries16 = nullptr;
    uint32_t rows_padded = 0, dim = 0, ld16 = 0;

    // order: what the fp32 sums have to agree with (the other column blocks, or the candidate ranges behind this one)
    int into_matrix(uint32_t c0, uint32_t ncols, uint32_t num_queries, float* Z, uint32_t ldz, const FcOrder& order, float* seg_max = nullptr,
                    uint32_t* seg_width = nullptr) const
    {
        if (f16) return knn_f16_scores_run(queries16, items16 + (uint64_t)c0 * ld16 * 2, ld16, num_queries, ncols, Z, ldz, nullptr);
        if (split)
            return fc_split_run(query_planes, item_planes, split_rows_padded(rows_padded), c0, nullptr, Z, ldz, num_queries, dim, ncols, 0,
                                DSX_ACT_LINEAR, nullptr, nullptr, nullptr);
        return fc_run(queries, dim, items + c0, rows_padded, 0, nullptr, Z, ldz, num_queries, dim, ncols, 0, DSX_ACT_LINEAR, nullptr, seg_max, seg_width,
                      nullptr, order);
    }
    // *chunks_used: how many (row, chunk) lists of seg the range filled besides the shared lists (0: none)
    int into_candidates(uint32_t c0, uint32_t ncols, uint32_t num_queries, const CandArgs& cand, uint64_t* seg, uint32_t* seg_count,
                        uint32_t* chunks_used) const
    {
        *chunks_used = 0;
        if (f16)
            return knn_f16_candidates_run(queries16, items16 + (uint64_t)c0 * ld16 * 2, ld16, num_queries, ncols, cand, seg, seg_count, kCandCap,
                                          ctx().knobs.knn_f16_sweep, chunks_used);
        if (split) return fc_split_candidates_run(query_planes, item_planes, split_rows_padded(rows_padded), c0, num_queries, dim, ncols, cand);
        return fc_candidates_run(queries, dim, items + c0, rows_padded, num_queries, dim, ncols, cand);
    }
};

// Times of the stages, added up once the search is through: a stage ends where the next one starts, and the host waits for none of
// them (4 queries x 1,000,000 x 128 through KnnExactGpu::search: 204 us with a wait per stage, 189 without).
struct KnnTimer {
    bool on = false;
    float gemm = 0.0f, topk = 0.0f;
    std::vector<hipEvent_t> marks;   // stage i lies between marks i and i + 1
    std::vector<float*> into;
    int mark(hipStream_t s)
    {
        hipEvent_t e = nullptr;
        if (ctx().knobs.knn_no_events) return set_error(DSX_EHIP, "KnnTimer: no events");
        DSX_HIP(hipEventCreate(&e));
        marks.push_back(e);
        DSX_HIP(hipEventRecord(e, s));
        return DSX_OK;
    }
    void start(hipStream_t s) { if (on && marks.empty()) on = mark(s) == DSX_OK; }
    void stop(hipStream_t s, float& t)
    {
        if (!on) return;
        on = mark(s) == DSX_OK;
        if (on) into.push_back(&t);
    }
    // True if the stream's work up to the last mark is through, and nothing has been launched without one.
    bool finish()
    {
        if (into.empty()) return false;
        const bool through = hipEventSynchronize(marks[into.size()]) == hipSuccess && on;
        for (size_t i = 0; i < into.size(); i++) {
            float ms = 0.0f;
            hipEventElapsedTime(&ms, marks[i], marks[i + 1]);
            *into[i] += ms;
        }
        into.clear();
        return through;
    }
    ~KnnTimer()
    {
        for (auto& e : marks) hipEventDestroy(e);
    }
};

// Where the results go; host_*: once more, into host memory that the device can write (or NULL).
struct KnnResults {
    float* scores;
    uint32_t* indexes;
    float* host_scores;
    uint32_t* host_indexes;
};

// Block by block through the scratch score matrix; exact for any input, no host read-back.
static int knn_search_blocks(const KnnWorkspace& w, const KnnOperands& op, uint32_t M, uint32_t num_queries, uint32_t k, const KnnResults& out, KnnTimer& t)
{
    hipStream_t s = ctx().stream;
    const uint32_t cb = knn_block_columns(op.rows_padded, num_queries);
    const uint32_t blocks = (M + cb - 1) / cb;
    FcOrder order;
    order.plan_n = blocks > 1 ? cb : 0;
    const uint32_t lists_per_block = knn_block_lists(num_queries, cb, k);
    const uint32_t lists = (blocks - 1) * lists_per_block + knn_block_lists(num_queries, M - (blocks - 1) * cb, k);
    hipLaunchKernelGGL(knn_clear_kernel, dim3((num_queries + 255) / 256), dim3(256), 0, s, w.row_bound, num_queries);
    for (uint32_t blk = 0; blk < blocks; blk++) {
        const uint32_t c0 = blk * cb;
        const uint32_t ncols = std::min(cb, M - c0);
        t.start(s);
        uint32_t seg_width = 0;
        const bool guided = knn_block_guided(num_queries, ncols, k);
        int rc = op.into_matrix(c0, ncols, num_queries, w.block_scores, cb, order, guided ? w.seg_max : nullptr, guided ? &seg_width : nullptr);
        if (rc) return rc;
        t.stop(s, t.gemm);
        t.start(s);
        if (seg_width != 0)
            rc = topk_guided_launch(w.block_scores, cb, ncols, num_queries, k, nullptr, nullptr, w.seg_max, 0, nullptr, nullptr, nullptr, nullptr,
                                    nullptr, c0, w.partial, lists, blk * lists_per_block, w.row_bound);
        else
            rc = topk_run(w.block_scores, cb, ncols, num_queries, k, nullptr, nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, c0,
                          w.partial, lists, blk * lists_per_block, knn_block_lists(num_queries, ncols, k), w.row_bound);
        if (rc) return rc;
        t.stop(s, t.topk);
    }
    t.start(s);
    int rc = topk_merge(w.partial, lists, k, out.scores, out.indexes, num_queries, out.host_scores, out.host_indexes);
    t.stop(s, t.topk);
    return rc;
}

// What the preparation of a screened search finds, stored by it in pinned memory and read before the search goes on.
static ScreenNotes* g_knn_notes = nullptr;
static hipEvent_t g_knn_noted = nullptr;

static void knn_notes_release()
{
    if (g_knn_notes) hipHostFree(g_knn_notes);
    if (g_knn_noted) hipEventDestroy(g_knn_noted);
    g_knn_notes = nullptr;
    g_knn_noted = nullptr;
}

// Whether what the preparation found speaks against screening.
static bool knn_unfit(const ScreenNotes& notes)
{
    return notes.flag != 0 || !screen_fits(notes.largest, notes.number != 0 ? notes.sum / (float)notes.number : 0.0f);
}

static int knn_notes_ready()
{
    if (!g_knn_noted) {
        at_shutdown(knn_notes_release);
        if (!g_knn_notes) DSX_HIP(hipHostMalloc((void**)&g_knn_notes, sizeof(ScreenNotes), hipHostMallocMapped));
        DSX_HIP(hipEventCreateWithFlags(&g_knn_noted, hipEventDisableTiming));
    }
    *g_knn_notes = ScreenNotes{};   // (a search is over when its call returns: nothing writes to them now)
    return DSX_OK;
}

// First block as above, the rest in candidate mode.  *overflowed tells the caller to redo the search block by block.
static int knn_search_candidates(const KnnWorkspace& w, const KnnOperands& op, uint32_t M, uint32_t num_queries, uint32_t k, const KnnResults& out,
                                 KnnTimer& t, bool* overflowed)
{
    hipStream_t s = ctx().stream;
    const uint32_t cb = knn_block_columns(op.rows_padded, num_queries);
    const uint32_t clear_words = 3 * num_queries + 64;
    hipLaunchKernelGGL(knn_clear_kernel, dim3((clear_words + 255) / 256), dim3(256), 0, s, w.row_bound, clear_words);
    // The first block only has to give every query a usable bound; a quarter of a column block does (measured on 2 M items x 4,096
    // queries: 8 K to 32 K columns are level, the full 64 K cost 0.1 ms more in stores and scan).  A width set by the caller is kept.
    uint32_t done = std::min(cb, M);
    if (!ctx().knobs.knn_block_columns) done = std::min<uint32_t>(done, std::max<uint32_t>(1024, cb / 4 / 1024 * 1024));
    t.start(s);
    FcOrder order;
    order.as_candidates = true;
    int rc = op.into_matrix(0, done, num_queries, w.block_scores, cb, order);
    if (rc) return rc;
    t.stop(s, t.gemm);
    t.start(s);
    rc = topk_run(w.block_scores, cb, done, num_queries, k, nullptr, nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, 0, w.partial, 1, 0,
                  1, w.row_bound);
    if (rc) return rc;
    t.stop(s, t.topk);
    while (done < M) {
        // a multiple of the tile width keeps every range's first column 16-byte aligned (done is a multiple of 1,024)
        const uint32_t ncols = (uint32_t)std::min<uint64_t>((uint64_t)M - done, (uint64_t)done * 4);
        t.start(s);
        const CandArgs cand{w.row_bound, w.cand, w.cand_count, kCandCap, done, w.overflow};
        uint32_t lists = 0;
        rc = op.into_candidates(done, ncols, num_queries, cand, w.seg, w.seg_count, &lists);
        if (rc) return rc;
        t.stop(s, t.gemm);
        t.start(s);
        rc = knn_refresh(w.partial, w.cand, w.cand_count, kCandCap, k, w.row_bound, num_queries, lists ? w.seg : nullptr, w.seg_count, lists,
                         lists ? kCandCap / lists : 0);
        if (rc) return rc;
        t.stop(s, t.topk);
        done += ncols;
    }
    t.start(s);
    rc = topk_merge(w.partial, 1, k, out.scores, out.indexes, num_queries, out.host_scores, out.host_indexes);
    if (rc) return rc;
    t.stop(s, t.topk);
    uint32_t flag = 0;
    DSX_HIP(hipMemcpyAsync(&flag, w.overflow, sizeof(flag), hipMemcpyDeviceToHost, s));
    DSX_HIP(hipStreamSynchronize(s));
    *overflowed = flag != 0;
    return DSX_OK;
}

// Screened in 16 bits (fp32 storage).  built: the workspace's table is there already (dsx_knn_prepare), and what it is like has been
// looked at.  *overflowed tells the caller to redo the search without screening; *unfit, that the table or the queries were found unfit
// for it first (norms beyond f16's range, or one so large that the others' bounds would be worth little); *open, that it was bytes that were not enough,
// so that halves may be.
static int knn_search_screened(const KnnWorkspace& w, const KnnOperands& op, uint32_t M, uint32_t num_queries, uint32_t k, const KnnResults& out,
                               KnnTimer& t, bool built, bool even, bool* overflowed, bool* unfit, bool* open)
{
    hipStream_t s = ctx().stream;
    int rc = knn_notes_ready();
    if (rc) return rc;
    ScreenJob j{};
    j.X = op.queries; j.ldx = op.dim; j.batch = num_queries; j.dim = op.dim; j.n = M; j.k = k;
    j.act = DSX_ACT_LINEAR;
    j.even = even;
    j.keys = out.scores; j.values = out.indexes; j.keys2 = out.host_scores; j.values2 = out.host_indexes;
    j.row_flag = w.row_flag; j.told = &g_knn_notes->flag; j.open = &g_knn_notes->open;
    j.cand = w.cand; j.cand_count = w.cand_count; j.cap = kCandCap; j.overflow = w.overflow;
    j.clear = w.overflow; j.clear_words = 64;
    t.start(s);
    if (!built) {
        if ((rc = screen_build(w.table, op.items, op.rows_padded, M, op.dim))) return rc;
    }
    if ((rc = screen_rows(j, w.table, w.screen, built ? nullptr : g_knn_notes))) return rc;
    if (!built) {
        DSX_HIP(hipEventRecord(g_knn_noted, s));
        hipError_t noted;   // (asked again and again: a wait that sleeps wakes up late)
        while ((noted = hipEventQuery(g_knn_noted)) == hipErrorNotReady) {}
        (void)hipGetLastError();   // (not ready is not an error of the next launch)
        DSX_HIP(noted);
        *unfit = knn_unfit(*g_knn_notes);
        if (*unfit) return DSX_OK;
        j.even = g_knn_notes->number != 0 && screen_even(g_knn_notes->largest, g_knn_notes->sum / (float)g_knn_notes->number);
    }
    // (candidates are cut back between the ranges too: what is counted as top-K is the kernel that scores and sorts what is left)
    if (t.on) {
        j.before_last = [](void* p) { static_cast<KnnTimer*>(p)->stop(ctx().stream, static_cast<KnnTimer*>(p)->gemm); };
        j.before_last_arg = &t;
    }
    if ((rc = screen_run(j, w.table, w.screen))) return rc;
    t.stop(s, t.topk);
    DSX_HIP(hipStreamSynchronize(s));
    const bool flagged = *(volatile uint32_t*)&g_knn_notes->flag != 0;
    *open = !flagged && *(volatile uint32_t*)&g_knn_notes->open != 0;
    *overflowed = flagged || *open;
    return DSX_OK;
}

// fp16 storage, screened in bytes: the workspace starts with the bytes (screen_table_halves); behind them lies what an unscreened search works in, or what
// this one does, as they come after each other.  *overflowed as above.
static int knn_search_halves(const ScreenTable& table, void* rest, const KnnOperands& op, const float* queries, uint32_t M, uint32_t num_queries, uint32_t k,
                             const KnnResults& out, KnnTimer& t, bool* overflowed)
{
    hipStream_t s = ctx().stream;
    int rc = knn_notes_ready();
    if (rc) return rc;
    const ScreenWorkspace w = screen_layout((char*)rest + align256((size_t)num_queries * sizeof(uint32_t)), num_queries, op.dim, op.rows_padded, k, true);
    ScreenJob j{};
    j.X = queries; j.ldx = op.dim; j.batch = num_queries; j.dim = op.dim; j.n = M; j.k = k;
    j.act = DSX_ACT_LINEAR;
    j.even = true;   // (every item is finite)
    j.rows16 = op.items16;
    j.keys = out.scores; j.values = out.indexes; j.keys2 = out.host_scores; j.values2 = out.host_indexes;
    j.row_flag = (uint32_t*)rest; j.told = j.open = &g_knn_notes->flag;
    t.start(s);
    if ((rc = screen_rows(j, table, w, nullptr))) return rc;
    if (t.on) {
        j.before_last = [](void* p) { static_cast<KnnTimer*>(p)->stop(ctx().stream, static_cast<KnnTimer*>(p)->gemm); };
        j.before_last_arg = &t;
    }
    if ((rc = screen_run(j, table, w))) return rc;
    t.stop(s, t.topk);
    DSX_HIP(hipStreamSynchronize(s));
    *overflowed = *(volatile uint32_t*)&g_knn_notes->flag != 0;
    return DSX_OK;
}

// Bytes of a workspace behind the bytes of the table, for this number of queries.
static size_t knn_halves_rest(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    const size_t unscreened = knn_layout(nullptr, rows_padded, num_queries, k, true, dim, false).bytes;
    if (!screen_in_bytes(num_queries, dim, rows_padded, k)) return unscreened;
    return std::max(unscreened, align256((size_t)num_queries * sizeof(uint32_t)) + screen_layout(nullptr, num_queries, dim, rows_padded, k, true).bytes);
}

// Whether a table of halves is worth its bytes for some number of queries.
static bool knn_prepares_halves(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return num_queries > 0 && ctx().knobs.screen != 2 && dim >= 16 && dim <= 4096 && k >= 1 && k <= 256 && screen_in_bytes(num_queries, dim, rows_padded, k);
}

}  // namespace dsx

using namespace dsx;

extern "C" {

int dsx_testing_set_knn_block_columns(uint32_t columns)
{
    ctx().knobs.knn_block_columns = columns;
    return DSX_OK;
}

int dsx_testing_set_screen(int mode)
{
    DSX_CHECK_ARG(mode >= 0 && mode <= 2, "dsx_testing_set_screen: mode %d (0 to 2)", mode);
    ctx().knobs.screen = mode;
    return DSX_OK;
}

int dsx_testing_set_screen_bytes(int mode)
{
    DSX_CHECK_ARG(mode >= 0 && mode <= 2, "dsx_testing_set_screen_bytes: mode %d (0 to 2)", mode);
    ctx().knobs.screen_bytes = mode;
    return DSX_OK;
}

int dsx_testing_set_knn_no_events(int none)
{
    ctx().knobs.knn_no_events = none;
    return DSX_OK;
}

int dsx_knn_last_search_path(void) { return g_knn_last_path; }

int dsx_knn_last_search_repeated(void) { return g_knn_last_repeated; }

int dsx_testing_set_knn_f16_sweep(int mode)
{
    DSX_CHECK_ARG(mode >= 0 && mode <= 3, "dsx_testing_set_knn_f16_sweep: mode %d (0 to 3)", mode);
    ctx().knobs.knn_f16_sweep = mode;
    return DSX_OK;
}

size_t dsx_knn_workspace_bytes(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return knn_workspace_most(rows_padded, num_queries, k, false, dim, false);
}

size_t dsx_knn_workspace_bytes_least(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return knn_workspace_most(rows_padded, num_queries, k, false, dim, false, false);
}

// Where a kept table is used: everywhere but for tables so small that k blocks of 32 items are a large part of them, vectors whose halves are
// mostly padding, and tables of more than 8 GiB.  us a search, in fp32 / so (both with their results written
// to host memory): 1 query, 8,192 x 256 top 10 46 / 43, 70,000 x 256 61 / 51, 400,000 x 256 141 / 83; 32 queries, 20,000 x 16 top 100 54 / 44; 128
// queries, 70,000 x 64 top 10 74 / 53; 512 queries, 8,192 x 64 top 100 138 / 127, 400,000 x 64 643 / 239; 4,096 queries, 8,192 x 16 top 10
// 228 / 205, 70,000 x 256 1,658 / 563.  None of 88 is slower but few short queries of a long table (knn_search_common).
static bool knn_prepares(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return num_queries > 0 && ctx().knobs.screen != 2 && dim >= 16 && dim <= 4096 && rows_padded >= 8192 && rows_padded >= 64 * k &&
           screen_table(nullptr, dim, rows_padded, false).bytes <= ((uint64_t)8 << 30) && k <= 256;
}

size_t dsx_knn_workspace_bytes_prepared(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    if (!knn_prepares(rows_padded, dim, num_queries, k)) return dsx_knn_workspace_bytes(rows_padded, dim, num_queries, k);
    size_t most = 0;
    for (uint64_t q = 1; q <= num_queries; q++) most = std::max(most, knn_layout(nullptr, rows_padded, (uint32_t)q, k, false, dim, false, true, true).bytes);
    return most;
}

size_t dsx_knn_workspace_bytes_f16(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return knn_workspace_most(rows_padded, num_queries, k, true, dim, false);
}

size_t dsx_knn_workspace_bytes_f16_prepared(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    if (!knn_prepares_halves(rows_padded, dim, num_queries, k)) return dsx_knn_workspace_bytes_f16(rows_padded, dim, num_queries, k);
    size_t most = 0;
    for (uint64_t q = 1; q <= num_queries; q++) most = std::max(most, knn_halves_rest(rows_padded, dim, (uint32_t)q, k));
    return screen_table_halves(nullptr, dim, rows_padded).bytes + most;
}

size_t dsx_knn_workspace_bytes_split(uint32_t rows_padded, uint32_t dim, uint32_t num_queries, uint32_t k)
{
    return knn_workspace_most(rows_padded, num_queries, k, false, dim, true);
}

size_t dsx_knn_f16_table_bytes(uint32_t rows_padded, uint32_t dim) { return (size_t)knn_f16_rows(rows_padded) * knn_f16_ld(dim) * 2; }

int dsx_knn_f16_convert_items(const float* items, uint32_t rows_padded, uint32_t padding, uint32_t dim, void* items_f16)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(items && items_f16, "dsx_knn_f16_convert_items: null device pointer");
    DSX_CHECK_ARG(padding < rows_padded && dim > 0, "dsx_knn_f16_convert_items: rows_padded %u, padding %u, dim %u", rows_padded, padding, dim);
    DSX_CHECK_ARG(((uintptr_t)items_f16 % 16) == 0, "dsx_knn_f16_convert_items: the fp16 table is not 16-byte aligned");
    return knn_to_f16(items, true, rows_padded, rows_padded - padding, dim, items_f16, (uint32_t)knn_f16_rows(rows_padded));
}

}  // extern "C"

// Both precisions: workspace, the two paths, timing.  screening: whether candidates may be screened; table: the workspace holds a prepared table, which
// screening uses and everything else leaves as it is; bytes: whether it may go in bytes.
static int knn_search_common(KnnOperands& op, uint32_t padding, uint32_t num_queries, uint32_t k, const KnnResults& out, void* workspace,
                             size_t workspace_bytes, float* elapsed_ms, bool aligned, const float* queries_f32, bool screening = false, bool table = false, bool even = false,
                             bool bytes = true)
{
    const bool built = screening && table;
    const size_t full = knn_layout(nullptr, op.rows_padded, num_queries, k, op.f16, op.dim, op.split, screening, table).bytes;
    const size_t need = knn_layout(nullptr, op.rows_padded, num_queries, k, op.f16, op.dim, op.split, false, table).bytes;
    bool screen = full != need;   // the screening's copies of the table (up to 8 GiB) where there is room for them: fp32 needs none
    if (workspace) {
        DSX_CHECK_ARG(workspace_bytes >= need, "dsx_knn_search: workspace of %zu bytes, %zu needed", workspace_bytes, need);
        screen = screen && workspace_bytes >= full;
        DSX_CHECK_ARG(((uintptr_t)workspace % 256) == 0, "dsx_knn_search: workspace is not 256-byte aligned");
    } else {
        LibScratch& ws = g_knn_ws_of[current_lane()];
        int reserved = screen ? lib_scratch_reserve(ws, full, "dsx_knn_search workspace", true) : DSX_ENOMEM;
        if (reserved == DSX_ENOMEM) {
            screen = false;
            reserved = lib_scratch_reserve(ws, need, "dsx_knn_search workspace");
        }
        if (reserved) return reserved;
        workspace = ws.ptr;
    }
    KnnWorkspace w = knn_layout(workspace, op.rows_padded, num_queries, k, op.f16, op.dim, op.split, screen, table);
    auto in_halves = [&] { w.screen = screen_layout(w.screen.rows8, num_queries, op.dim, op.rows_padded, k, false); };
    if (w.screen.words && !bytes) in_halves();
    const uint32_t M = op.rows_padded - padding;
    hipStream_t s = ctx().stream;
    KnnTimer t;
    t.on = elapsed_ms != nullptr;
    int rc = DSX_OK;
    if (op.f16) {   // the query batch in the table's format (knn/KnnExactGpu.cu:108-116); counted as GEMM time like the copy it replaces
        t.start(s);
        rc = knn_to_f16(queries_f32, false, op.dim, num_queries, op.dim, w.queries16, (uint32_t)knn_f16_rows(num_queries));
        if (rc) return rc;
        t.stop(s, t.gemm);
        op.queries16 = w.queries16;
    }
    if (op.split) {   // the query batch as bf16 planes, counted as GEMM time too
        t.start(s);
        rc = fc_split_planes_run(queries_f32, op.dim, 1, num_queries, op.dim, w.queries16);
        if (rc) return rc;
        t.stop(s, t.gemm);
        op.query_planes = w.queries16;
    }
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    hipStreamIsCapturing(s, &capturing);
    // (few queries against an fp32 table stay with the blocks, however many there are; a width set by the caller is kept)
    const bool few = knn_few_queries(num_queries) && !op.f16 && !op.split && !ctx().knobs.knn_block_columns;
    const bool may = aligned && (!few || built) && capturing == hipStreamCaptureStatusNone;
    // (screened searches need no alignment: vectors of 215 components, say, whose fp32 products would be formed block by block)
    const bool narrow = built && op.dim < 32 && op.rows_padded > 131072 && knn_few_queries(num_queries);   // (16 x 400,000, 32 queries: 65 us / 69)
    const bool may_screen = (!few || built) && !narrow && capturing == hipStreamCaptureStatusNone;
    const bool many = M > knn_block_columns(op.rows_padded, num_queries);
    bool screened = may_screen && w.screen.bytes != 0 && !ctx().knobs.knn_block_columns;
    bool redo = true, unfit = false, open = false;
    if (rc == DSX_OK && screened) rc = knn_search_screened(w, op, M, num_queries, k, out, t, built, even, &redo, &unfit, &open);
    if (unfit) screened = false;
    // What bytes leave open halves may settle, at a fifth of what fp32 takes (4,096 x 128 x 1,000,000 top 100: 1.8 and 8.8 ms).
    const bool again = open;
    if (rc == DSX_OK && again) {
        in_halves();
        rc = knn_search_screened(w, op, M, num_queries, k, out, t, built, even, &redo, &unfit, &open);
    }
    g_knn_last_repeated = screened && redo ? 1 : again ? 2 : 0;
    const bool candidates = screened || (may && many);
    if (rc == DSX_OK && may && (!screened || redo) && many)
        rc = knn_search_candidates(w, op, M, num_queries, k, out, t, &redo);
    g_knn_last_path = !candidates ? DSX_KNN_PATH_BLOCKS : (redo ? DSX_KNN_PATH_CANDIDATES_REDONE : DSX_KNN_PATH_CANDIDATES);
    if (rc == DSX_OK && redo) rc = knn_search_blocks(w, op, M, num_queries, k, out, t);
    bool through = false;
    if (elapsed_ms) {
        through = t.finish();
        elapsed_ms[0] = t.gemm;
        elapsed_ms[1] = t.topk;
    }
    // the results are complete when the call returns (the other ways have waited by now; where the last kernel's event has come the stream is not
    // waited for as well: 209 queries x 551,602 x 41 in halves 285 us, 311 with both)
    if (rc == DSX_OK && redo && !through && capturing == hipStreamCaptureStatusNone) DSX_HIP(hipStreamSynchronize(s));
    return rc;
}

static int knn_search_fp32(const float* items, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                           uint32_t num_queries, uint32_t k, const KnnResults& out, void* workspace, size_t workspace_bytes, float* elapsed_ms,
                           bool screening, bool table, bool even, bool bytes)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(items && queries && out.scores && out.indexes, "dsx_knn_search: null device pointer");
    DSX_CHECK_ARG(padding < rows_padded, "dsx_knn_search: padding %u leaves no item of %u", padding, rows_padded);
    DSX_CHECK_ARG(dim > 0, "dsx_knn_search: dim is 0");
    DSX_CHECK_ARG(k >= 1 && k <= 256, "dsx_knn_search: k = %u is outside 1..256", k);
    if (num_queries == 0) return DSX_OK;
    KnnOperands op;
    op.items = items;
    op.queries = queries;
    op.rows_padded = rows_padded;
    op.dim = dim;
    const bool aligned = ((uintptr_t)items % 16) == 0 && ((uintptr_t)queries % 16) == 0 && (rows_padded % 4) == 0 && (dim % 4) == 0;
    return knn_search_common(op, padding, num_queries, k, out, workspace, workspace_bytes, elapsed_ms, aligned, nullptr, screening, table, even, bytes);
}

static int knn_search_split(const void* item_planes, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                            uint32_t num_queries, uint32_t k, const KnnResults& out, void* workspace, size_t workspace_bytes, float* elapsed_ms)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(item_planes && queries && out.scores && out.indexes, "dsx_knn_search_split: null device pointer");
    DSX_CHECK_ARG(((uintptr_t)item_planes % 16) == 0, "dsx_knn_search_split: the item planes are not 16-byte aligned");
    DSX_CHECK_ARG(padding < rows_padded, "dsx_knn_search_split: padding %u leaves no item of %u", padding, rows_padded);
    DSX_CHECK_ARG(dim > 0, "dsx_knn_search_split: dim is 0");
    DSX_CHECK_ARG(k >= 1 && k <= 256, "dsx_knn_search_split: k = %u is outside 1..256", k);
    DSX_CHECK_ARG((uint64_t)split_plane_bytes(rows_padded, dim) / 3 < (1ull << 32), "dsx_knn_search_split: a plane of the item table of 4 GiB or more");
    if (num_queries == 0) return DSX_OK;
    KnnOperands op;
    op.split = true;
    op.item_planes = item_planes;
    op.rows_padded = rows_padded;
    op.dim = dim;
    return knn_search_common(op, padding, num_queries, k, out, workspace, workspace_bytes, elapsed_ms, true, queries);
}

// prepared: the workspace starts with the bytes of the table, which are used where that is faster (screening) and else left as they are.
static int knn_search_f16(const void* items_f16, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                          uint32_t num_queries, uint32_t k, const KnnResults& out, void* workspace, size_t workspace_bytes, float* elapsed_ms,
                          bool prepared = false, bool screening = false)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(items_f16 && queries && out.scores && out.indexes, "dsx_knn_search_f16: null device pointer");
    DSX_CHECK_ARG(((uintptr_t)items_f16 % 16) == 0, "dsx_knn_search_f16: the fp16 table is not 16-byte aligned");
    DSX_CHECK_ARG(padding < rows_padded, "dsx_knn_search_f16: padding %u leaves no item of %u", padding, rows_padded);
    DSX_CHECK_ARG(dim > 0, "dsx_knn_search_f16: dim is 0");
    DSX_CHECK_ARG(k >= 1 && k <= 256, "dsx_knn_search_f16: k = %u is outside 1..256", k);
    if (num_queries == 0) return DSX_OK;
    KnnOperands op;
    op.f16 = true;
    op.items16 = (const char*)items_f16;
    op.rows_padded = rows_padded;
    op.dim = dim;
    op.ld16 = knn_f16_ld(dim);
    if (prepared) {
        const ScreenTable table = screen_table_halves(workspace, dim, rows_padded);
        const size_t rest = knn_halves_rest(rows_padded, dim, num_queries, k);
        DSX_CHECK_ARG(((uintptr_t)workspace % 256) == 0, "dsx_knn_search: workspace is not 256-byte aligned");
        DSX_CHECK_ARG(workspace_bytes >= table.bytes + rest, "dsx_knn_search: workspace of %zu bytes, %zu needed", workspace_bytes, table.bytes + rest);
        workspace = (char*)workspace + table.bytes;
        workspace_bytes -= table.bytes;
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        hipStreamIsCapturing(ctx().stream, &capturing);
        if (screening && capturing == hipStreamCaptureStatusNone && !ctx().knobs.knn_block_columns && knn_prepares_halves(rows_padded, dim, num_queries, k)) {
            KnnTimer t;
            t.on = elapsed_ms != nullptr;
            bool redo = true;
            if (int rc = knn_search_halves(table, workspace, op, queries, rows_padded - padding, num_queries, k, out, t, &redo)) return rc;
            if (!redo) {
                g_knn_last_path = DSX_KNN_PATH_CANDIDATES;
                g_knn_last_repeated = 0;
                if (elapsed_ms) {
                    t.finish();
                    elapsed_ms[0] = t.gemm;
                    elapsed_ms[1] = t.topk;
                }
                return DSX_OK;
            }
            const int rc = knn_search_common(op, padding, num_queries, k, out, workspace, workspace_bytes, elapsed_ms, true, queries);
            g_knn_last_repeated = 1;
            return rc;
        }
    }
    return knn_search_common(op, padding, num_queries, k, out, workspace, workspace_bytes, elapsed_ms, true, queries);
}

extern "C" {

int dsx_knn_search(const float* items, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                   uint32_t num_queries, uint32_t k, float* scores, uint32_t* indexes, void* workspace, size_t workspace_bytes,
                   float* elapsed_ms)
{
    return knn_search_fp32(items, rows_padded, padding, dim, queries, num_queries, k, KnnResults{scores, indexes, nullptr, nullptr}, workspace,
                           workspace_bytes, elapsed_ms, true, false, false, false);
}

int dsx_knn_search_split(const void* item_planes, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                         uint32_t num_queries, uint32_t k, float* scores, uint32_t* indexes, void* workspace, size_t workspace_bytes,
                         float* elapsed_ms)
{
    return knn_search_split(item_planes, rows_padded, padding, dim, queries, num_queries, k, KnnResults{scores, indexes, nullptr, nullptr}, workspace,
                            workspace_bytes, elapsed_ms);
}

int dsx_knn_search_f16(const void* items_f16, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                       uint32_t num_queries, uint32_t k, float* scores, uint32_t* indexes, void* workspace, size_t workspace_bytes,
                       float* elapsed_ms)
{
    return knn_search_f16(items_f16, rows_padded, padding, dim, queries, num_queries, k, KnnResults{scores, indexes, nullptr, nullptr}, workspace,
                          workspace_bytes, elapsed_ms);
}

int dsx_knn_prepare(const float* items, uint32_t rows_padded, uint32_t padding, uint32_t dim, uint32_t num_queries, uint32_t k, void* workspace,
                    size_t workspace_bytes, int* prepared)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(items && workspace && prepared, "dsx_knn_prepare: null pointer");
    DSX_CHECK_ARG(padding < rows_padded && k >= 1 && k <= 256, "dsx_knn_prepare: rows_padded %u, padding %u, k = %u", rows_padded, padding, k);
    DSX_CHECK_ARG(((uintptr_t)workspace % 256) == 0, "dsx_knn_prepare: workspace is not 256-byte aligned");
    *prepared = 0;
    if (!knn_prepares(rows_padded, dim, num_queries, k) || workspace_bytes < dsx_knn_workspace_bytes_prepared(rows_padded, dim, num_queries, k)) return DSX_OK;
    const uint32_t M = rows_padded - padding;
    ScreenTable t = screen_table(workspace, dim, rows_padded, true);
    if (!screen_in_bytes(num_queries, dim, rows_padded, k)) t.items8 = nullptr;   // (no search of so few goes by them; their place is the table's all the same)
    if (int rc = screen_build(t, items, rows_padded, M, dim)) return rc;
    uint32_t stats[8];
    DSX_HIP(hipMemcpyAsync(stats, t.stats, sizeof(stats), hipMemcpyDeviceToHost, ctx().stream));
    DSX_HIP(hipStreamSynchronize(ctx().stream));
    ScreenNotes notes{};
    std::memcpy(&notes.largest, &stats[0], sizeof(float));
    std::memcpy(&notes.sum, &stats[1], sizeof(float));
    notes.number = stats[2];
    // as where a search makes its own copies
    const float average = notes.number != 0 ? notes.sum / (float)notes.number : 0.0f;
    // (in bytes an item that is no number adds up to 0, unless sums start from something)
    const bool even = screen_even(notes.largest, average) && !(t.items8 && stats[6] != 0);
    if (screen_fits(notes.largest, average)) *prepared = even ? DSX_KNN_FP32_PREPARED_EVEN : DSX_KNN_FP32_PREPARED;
    return DSX_OK;
}

int dsx_knn_prepare_f16(const void* items_f16, uint32_t rows_padded, uint32_t padding, uint32_t dim, uint32_t num_queries, uint32_t k, void* workspace,
                        size_t workspace_bytes, int* prepared)
{
    DSX_REQUIRE_INIT();
    DSX_CHECK_ARG(items_f16 && workspace && prepared, "dsx_knn_prepare_f16: null pointer");
    DSX_CHECK_ARG(((uintptr_t)items_f16 % 16) == 0, "dsx_knn_prepare_f16: the fp16 table is not 16-byte aligned");
    DSX_CHECK_ARG(padding < rows_padded && k >= 1 && k <= 256, "dsx_knn_prepare_f16: rows_padded %u, padding %u, k = %u", rows_padded, padding, k);
    DSX_CHECK_ARG(((uintptr_t)workspace % 256) == 0, "dsx_knn_prepare_f16: workspace is not 256-byte aligned");
    *prepared = 0;
    if (!knn_prepares_halves(rows_padded, dim, num_queries, k) || workspace_bytes < dsx_knn_workspace_bytes_f16_prepared(rows_padded, dim, num_queries, k)) return DSX_OK;
    const ScreenTable t = screen_table_halves(workspace, dim, rows_padded);
    if (int rc = screen_build_halves(t, items_f16, rows_padded - padding, dim)) return rc;
    uint32_t stats[8];
    DSX_HIP(hipMemcpyAsync(stats, t.stats, sizeof(stats), hipMemcpyDeviceToHost, ctx().stream));
    DSX_HIP(hipStreamSynchronize(ctx().stream));
    if (stats[6] == 0) *prepared = DSX_KNN_FP16_PREPARED;
    return DSX_OK;
}

int dsx_knn_search_host(int storage, const void* items, uint32_t rows_padded, uint32_t padding, uint32_t dim, const float* queries,
                        uint32_t num_queries, uint32_t k, float* scores, uint32_t* indexes, float* host_scores, uint32_t* host_indexes,
                        void* workspace, size_t workspace_bytes, float* elapsed_ms)
{
    DSX_CHECK_ARG((host_scores == nullptr) == (host_indexes == nullptr), "dsx_knn_search_host: host_scores and host_indexes go together");
    const size_t host_bytes = (size_t)num_queries * k * sizeof(float);
    DSX_CHECK_ARG(!host_scores || host_bytes == 0 || (dsx_host_is_pinned(host_scores, host_bytes) && dsx_host_is_pinned(host_indexes, host_bytes)),
                  "dsx_knn_search_host: the device cannot write to the host memory for %u x %u results", num_queries, k);
    const bool halves = storage == DSX_KNN_FP32_PREPARED_HALVES || storage == DSX_KNN_FP32_PREPARED_EVEN_HALVES;
    const bool table = halves || storage == DSX_KNN_FP32_PREPARED || storage == DSX_KNN_FP32_PREPARED_EVEN || storage == DSX_KNN_FP32_PREPARED_UNSCREENED;
    DSX_CHECK_ARG(!table || workspace, "dsx_knn_search_host: no prepared workspace");
    const bool bytes = storage == DSX_KNN_FP16_PREPARED || storage == DSX_KNN_FP16_PREPARED_UNSCREENED;
    DSX_CHECK_ARG(!bytes || workspace, "dsx_knn_search_host: no prepared workspace");
    const KnnResults out{scores, indexes, host_scores, host_indexes};
    switch (storage) {
    case DSX_KNN_FP32:
    case DSX_KNN_FP32_PREPARED_UNSCREENED:
    case DSX_KNN_FP32_PREPARED:
    case DSX_KNN_FP32_PREPARED_EVEN:
    case DSX_KNN_FP32_PREPARED_HALVES:
    case DSX_KNN_FP32_PREPARED_EVEN_HALVES:
        return knn_search_fp32((const float*)items, rows_padded, padding, dim, queries, num_queries, k, out, workspace, workspace_bytes, elapsed_ms,
                               storage != DSX_KNN_FP32_PREPARED_UNSCREENED, table,
                               storage == DSX_KNN_FP32_PREPARED_EVEN || storage == DSX_KNN_FP32_PREPARED_EVEN_HALVES, !halves);
    case DSX_KNN_FP16: return knn_search_f16(items, rows_padded, padding, dim, queries, num_queries, k, out, workspace, workspace_bytes, elapsed_ms);
    case DSX_KNN_FP16_PREPARED:
    case DSX_KNN_FP16_PREPARED_UNSCREENED:
        return knn_search_f16(items, rows_padded, padding, dim, queries, num_queries, k, out, workspace, workspace_bytes, elapsed_ms, true,
                              storage == DSX_KNN_FP16_PREPARED);
    case DSX_KNN_SPLIT: return knn_search_split(items, rows_padded, padding, dim, queries, num_queries, k, out, workspace, workspace_bytes, elapsed_ms);
    default: return set_error(DSX_EINVAL, "dsx_knn_search_host: storage %d", storage);
    }
}

}  // extern "C"
