// dsx_topk.hip — per-row top-K of a score matrix, plain, KNN-padded, key/value and filtered.
//
// Design (wave64, one 256-lane workgroup per (row, column segment)):
//   * every (score, column) pair is packed into one 64-bit unsigned word, order-preserving for the score in the high half
//     and the complemented column in the low half, so "largest word" == "highest score, then lowest column": the whole
//     selection runs on unsigned 64-bit max/min and the result order is total and reproducible;
//   * each wavefront streams 128-bit loads of its share of the row, two spans of eight loads per lane in flight, and keeps
//     a running top-L list (L = 64, 128 or 256 >= k) in registers, one to four words per lane, sorted descending across
//     (register, lane);
//   * a score enters only if it beats the list's current k-th word; the common case costs three vector instructions per
//     16-byte group; survivors are compacted with a 64-bit ballot into a per-wave LDS staging area and, once L of them are
//     waiting, bitonic-sorted (cross-lane exchanges) and merged into the register list, which tightens the threshold;
//   * for k <= 128 the threshold is primed before the scan from the k-th best of the lanes' first-span maxima (a binary
//     search over key bits), so a 27k-column row stages about forty words, no wave ever sorts, and the final order comes
//     from counting, for each staged word, how many staged words are larger;
//   * the kernel is bound by instruction issue as much as by HBM (four waves per SIMD run the same phases in step), so the
//     code keeps rarely-taken work (packing, filter lookups) inside wave-uniform branches;
//   * the filter (items to multiply, normally by 0, e.g. the sample's own inputs) is a per-segment bitmap in LDS:
//     listed columns are dropped from the scan and injected once, after the scan, with score * multiplier;
//   * rows split over several segments write packed partial lists that a second small kernel merges.
#include <algorithm>
#include <type_traits>
#include "dsx_screen.h"

namespace dsx {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));   // 128-bit loads of any row

constexpr int kTopkThreads = 256;
constexpr int kTopkWaves = kTopkThreads / kWave;
constexpr uint32_t kMaxBitmapBits = 256 * 1024;   // 32 KiB of LDS per workgroup

__device__ __forceinline__ uint64_t pack_score(float key, uint32_t col)
{
    return ((uint64_t)score_key(key) << 32) | (uint32_t)~col;
}

// A lower bound of the k-th largest of the wave's 64*N keys, exact in its upper 20 bits (0 if k > 64*N): at least k keys are
// >= the result.  A radix-4 search over key bits 31..12; each step is three vector compares per key and scalar bookkeeping.
// Twelve bits of slack admit a handful of extra candidates, and save a third of a dependent chain that every wave runs
// before it can ask for more data.
// LOW = 0 searches all bits: the k-th largest key itself.
template <int N, int LOW = 12> __device__ __forceinline__ uint32_t wave_kth_key(const uint32_t (&key)[N], uint32_t k)
{
    uint32_t t = 0;
#pragma unroll 1
    for (int bit = 30; bit >= LOW; bit -= 2) {
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

__device__ __forceinline__ void unpack_score(uint64_t p, float& key, uint32_t& col)
{
    key = key_score((uint32_t)(p >> 32));
    col = ~(uint32_t)p;
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int mask)
{
    uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, mask, kWave);
    uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), mask, kWave);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src)
{
    uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, src, kWave);
    uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src, kWave);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t umax64(uint64_t a, uint64_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint64_t umin64(uint64_t a, uint64_t b) { return a > b ? b : a; }

// One compare-exchange layer of a bitonic network over 64*R words held as v[r] in lane `lane` (position r*64 + lane).
// J: partner distance, K: size of the monotone blocks being built, DESC: direction of the final order.
template <int R, bool DESC, int K, int J>
__device__ __forceinline__ void bitonic_layer(uint64_t (&v)[R], uint32_t lane)
{
    if constexpr (J >= kWave) {
        constexpr int JR = J / kWave;
#pragma unroll
        for (int r = 0; r < R; r++) {
            if ((r & JR) == 0) {
                const int r2 = r | JR;
                const bool desc_block = (((r * kWave) & K) == 0) == DESC;
                const uint64_t a = v[r], b = v[r2];
                const uint64_t mx = umax64(a, b), mn = umin64(a, b);
                v[r] = desc_block ? mx : mn;
                v[r2] = desc_block ? mn : mx;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t p = r * kWave + lane;
            const bool desc_block = ((p & K) == 0) == DESC;
            const bool lower = (lane & J) == 0;
            const uint64_t other = shfl_xor_u64(v[r], J);
            v[r] = (lower == desc_block) ? umax64(v[r], other) : umin64(v[r], other);
        }
    }
}

template <int R, bool DESC, int K, int J> struct BitonicJ {
    static __device__ __forceinline__ void run(uint64_t (&v)[R], uint32_t lane)
    {
        bitonic_layer<R, DESC, K, J>(v, lane);
        if constexpr (J > 1) BitonicJ<R, DESC, K, J / 2>::run(v, lane);
    }
};

template <int R, bool DESC, int K> struct BitonicK {
    static __device__ __forceinline__ void run(uint64_t (&v)[R], uint32_t lane)
    {
        if constexpr (K > 2) BitonicK<R, DESC, K / 2>::run(v, lane);
        BitonicJ<R, DESC, K, K / 2>::run(v, lane);
    }
};

// Full sort of 64*R words.
template <int R, bool DESC> __device__ __forceinline__ void bitonic_sort(uint64_t (&v)[R], uint32_t lane)
{
    BitonicK<R, DESC, kWave * R>::run(v, lane);
}

// Sorts a bitonic sequence of 64*R words descending.
template <int R> __device__ __forceinline__ void bitonic_merge_desc(uint64_t (&v)[R], uint32_t lane)
{
    BitonicJ<R, true, kWave * R, kWave * R / 2>::run(v, lane);
}

// Running top-L list of one wavefront plus its LDS staging area.
template <int R> struct WaveTopK {
    static constexpr int L = kWave * R;
    static constexpr int kBurst = 5 * kWave;            // most words staged between two checks of the fill level
    // Words that may wait before they are merged into the list.  A workgroup none of whose wavefronts ever merged finishes by
    // counting instead of sorting (finish_row), so there is room for about three times k of them in the four wavefronts.
    static constexpr int kDrainAt = (R == 1) ? 128 : 192;
    static constexpr int kStageWords = kDrainAt + kBurst;
    static constexpr int kCountWords = (R == 4) ? 512 : 256;   // most words of a workgroup that finish_row counts

    uint64_t q[R];        // sorted descending over position r*64 + lane; 0 = empty slot
    uint64_t thr;         // current k-th word: candidates must be strictly larger
    float thr_key;        // its score: cheap first test is score >= thr_key
    float thr_above;      // the next score above thr_key
    uint32_t thr_col;     // the k-th word's column (0xffffffff while the threshold is a bare score bound)
    uint32_t count;       // staged candidates (wave-uniform)
    bool flushed;         // the register list holds something
    uint64_t* stage;      // LDS, kStageWords words, private to this wave
    uint32_t lane;
    uint32_t k;

    __device__ __forceinline__ void init(uint64_t* stage_, uint32_t lane_, uint32_t k_)
    {
#pragma unroll
        for (int r = 0; r < R; r++) q[r] = 0;
        thr = 0;
        thr_key = -__builtin_inff();
        thr_above = -__builtin_inff();
        thr_col = 0xffffffffu;
        count = 0;
        flushed = false;
        stage = stage_;
        lane = lane_;
        k = k_;
    }

    // Merge the first min(count, L) staged words into the list.
    __device__ __forceinline__ void flush()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint64_t c[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t p = r * kWave + lane;
            c[r] = (p < count) ? stage[p] : 0;
        }
        bitonic_sort<R, false>(c, lane);                       // ascending
#pragma unroll
        for (int r = 0; r < R; r++) q[r] = umax64(q[r], c[r]);   // top L of the union, bitonic
        bitonic_merge_desc<R>(q, lane);
        // k-th word -> threshold
        flushed = true;
        const uint32_t kr = (k - 1) / kWave, kl = (k - 1) % kWave;
        uint64_t t = q[0];
#pragma unroll
        for (int r = 1; r < R; r++) t = (kr == (uint32_t)r) ? q[r] : t;
        raise_threshold(shfl_u64(t, (int)kl));
        // keep what did not fit: move it to the front, 64 words at a time (source and destination of one step never overlap
        // because L >= 64, and later sources lie above every earlier destination)
        const uint32_t rest = (count > (uint32_t)L) ? count - L : 0;
        for (uint32_t i = 0; i < rest; i += kWave) {
            uint64_t keep = 0;
            if (i + lane < rest) keep = stage[L + i + lane];
            __builtin_amdgcn_wave_barrier();
            if (i + lane < rest) stage[i + lane] = keep;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        count = rest;
    }

    // Words at or below t can no longer reach the top k.
    __device__ __forceinline__ void raise_threshold(uint64_t t)
    {
        if (t > thr) {
            thr = t;
            float key;
            uint32_t col;
            unpack_score(t, key, col);
            thr_key = key;
            thr_above = key_score((uint32_t)(t >> 32) + 1u);   // above +inf this is NaN, which nothing reaches
            thr_col = col;
        }
    }

    // Lowest score a column at or beyond first_col needs.  A score equal to the k-th one wins only with a smaller column, so once
    // the k-th word's column lies before first_col, ties are out: in a row of saturated scores (thousands of columns at exactly
    // 1.0) the scan then skips every group with one compare, like any other row.
    __device__ __forceinline__ float admission_score(uint32_t first_col) const
    {
        return (thr_col < first_col) ? thr_above : thr_key;
    }

    // Every word whose score key is below t can no longer reach the top k (t must be the key of a real score).
    __device__ __forceinline__ void prime(uint32_t t)
    {
        const uint64_t w = ((uint64_t)t << 32) - 1;
        if (w > thr) {
            thr = w;
            thr_key = key_score(t);
            thr_col = 0xffffffffu;
        }
    }

    // The same with a column: at least k real words are >= w (w need not be a real word itself).  Scores equal to w's then only
    // pass with a column at or before w's, which admission_score turns into "strictly above" for everything that lies behind it.
    __device__ __forceinline__ void prime_word(uint64_t w)
    {
        if (w - 1 > thr) {
            thr = w - 1;
            float key;
            uint32_t col;
            unpack_score(w, key, col);
            thr_key = key;
            thr_above = key_score((uint32_t)(w >> 32) + 1u);
            thr_col = col;
        }
    }

    // Stage the lanes' words that beat the threshold.  All 64 lanes must call this together.  Nothing is merged here: after
    // at most five calls the caller runs drain(), which keeps count < kDrainAt between bursts.
    __device__ __forceinline__ void stage_only(bool valid, uint64_t word)
    {
        const bool cand = valid && (word > thr);
        const uint64_t m = __ballot(cand);
        if (m == 0) return;
        const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (cand) stage[count + before] = word;
        count += (uint32_t)__popcll(m);
    }

    __device__ __forceinline__ void drain()
    {
        while (count >= (uint32_t)kDrainAt) flush();
    }

    // Offer one word per lane (valid lanes only) and merge when kDrainAt are waiting.
    __device__ __forceinline__ void offer(bool valid, uint64_t word)
    {
        stage_only(valid, word);
        drain();
    }

    __device__ __forceinline__ void finish()
    {
        while (count > 0) flush();
    }
};

struct TopKArgs {
    const float* in;        // [batch][pitch]
    uint32_t pitch;         // elements between rows
    uint32_t width;         // candidate columns per row (<= pitch)
    uint32_t k;
    uint32_t segments;      // workgroups per row
    uint32_t col_offset;    // added to the reported column (column blocks of a larger matrix)
    // filter (all NULL when unfiltered)
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;
    const float* fmul;
    // results: either final (keys/values, pitch k) or packed partial lists
    float* keys;
    uint32_t* values;
    float* keys2;               // the final results once more (pinned host memory): finish_row<R, true>
    uint32_t* values2;
    uint64_t* partial;          // [batch][partial_slots][k]
    uint32_t partial_slots;
    uint32_t partial_slot0;     // this launch writes slots partial_slot0 + segment
    // column blocks of one wide matrix (KNN): key of a score that k earlier columns of the row reach, 0 = none yet; raised here
    uint32_t* row_bound;        // [batch]
    // guided variant: maxima of the row's 64-column segments, left by the producer of `in`
    const float* seg_max;       // [batch][nseg]
    uint32_t nseg;
    uint32_t part_segs;         // segments per workgroup (nseg: one workgroup per row)
};

template <int R>
__device__ __forceinline__ void write_final(const uint64_t (&q)[R], uint32_t lane, uint32_t k, uint32_t col_offset, float* keys,
                                            uint32_t* values)
{
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t p = r * kWave + lane;
        if (p < k) {
            float key = -kMaxValue;   // engine/kernels.cu:3221-3224: unfilled slots
            uint32_t col = 0;
            if (q[r] != 0) {
                unpack_score(q[r], key, col);
                col += col_offset;
            }
            keys[p] = key;
            values[p] = col;
        }
    }
}

// End of a (row, segment): merges the lists of the four waves into wave 0 and writes the result (final pairs, or packed words
// for the merge kernel).  Every lane of the workgroup must call it.
template <int R, bool TWICE = false>
__device__ __forceinline__ void finish_row(WaveTopK<R>& list, uint64_t (*sStage)[WaveTopK<R>::kStageWords], const TopKArgs& a,
                                           uint32_t b, uint32_t seg, uint32_t wave, uint32_t lane)
{
    // Merge the four waves into wave 0.  A wave that never had to flush hands over its staged words as they are (they
    // already sit in LDS); a wave with a register list flushes what is left and publishes its first k words.
    constexpr int kCount = WaveTopK<R>::kCountWords, M = kCount / kWave;
    __shared__ uint32_t sPublished[kTopkWaves];
    __shared__ uint32_t sFlushed[kTopkWaves];
    __shared__ uint32_t sPlace[kCount];
    if (wave != 0 && list.flushed) {
        list.finish();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t p = r * kWave + lane;
            if (p < a.k) sStage[wave][p] = list.q[r];
        }
    }
    if (lane == 0) {
        sPublished[wave] = (wave != 0 && list.flushed) ? a.k : list.count;
        sFlushed[wave] = list.flushed ? 1u : 0u;
    }
    for (uint32_t i = wave * kWave + lane; i < (uint32_t)kCount; i += kTopkThreads) sPlace[i] = 0;
    __syncthreads();

    uint64_t* partial = a.partial ? a.partial + ((uint64_t)b * a.partial_slots + a.partial_slot0 + seg) * a.k : nullptr;
    float* keys = a.keys + (uint64_t)b * a.k;
    uint32_t* values = a.values + (uint64_t)b * a.k;
    // result slot p of this (row, segment): a packed word for the merge kernel, or the final (score, column) pair
    auto write_slot = [&](uint32_t p, uint64_t word) {
        float key = -kMaxValue;   // engine/kernels.cu:3221-3224: unfilled slots
        uint32_t col = 0;
        if (word != 0) {
            unpack_score(word, key, col);
            col += a.col_offset;
        }
        if (partial) {
            partial[p] = (word != 0) ? ((word & 0xffffffff00000000ull) | (uint32_t)~col) : 0ull;
        } else {
            keys[p] = key;
            values[p] = col;
            if constexpr (TWICE) {
                a.keys2[(uint64_t)b * a.k + p] = key;
                a.values2[(uint64_t)b * a.k + p] = col;
            }
        }
    };

    uint32_t n0 = sPublished[0], n1 = sPublished[1], n2 = sPublished[2], n3 = sPublished[3];
    uint32_t total = n0 + n1 + n2 + n3;
    const bool any_flushed = (sFlushed[0] | sFlushed[1] | sFlushed[2] | sFlushed[3]) != 0;   // the same for every wave
    auto fetch = [&](uint32_t i) -> uint64_t {   // the i-th of all staged words
        if (i >= total) return 0ull;   // never larger than anything
        const uint32_t w = (i >= n0) + (i >= n0 + n1) + (i >= n0 + n1 + n2);
        const uint32_t first = (w == 0) ? 0 : (w == 1) ? n0 : (w == 2) ? n0 + n1 : n0 + n1 + n2;
        return sStage[w][i - first];
    };
    if (R > 1 && !any_flushed && total > (uint32_t)(R == 2 ? 4 : 5) * kWave && total > a.k) {
        // The general scan stages up to twice k words, and counting costs their number squared: the exact k-th key first (one
        // wavefront searches; which one depends on the row, so that the four SIMDs of a compute unit share the work of the
        // workgroups on it), then every wave drops its words below it.
        constexpr int N = (4 * WaveTopK<R>::kDrainAt) / kWave;
        __shared__ uint32_t sKth;
        if (wave == ((b >> 8) & 3u)) {
            uint32_t t;
            auto search = [&](auto lanes_words) __attribute__((always_inline)) {
                constexpr int C = decltype(lanes_words)::value;
                uint32_t key[C];
#pragma unroll
                for (int m = 0; m < C; m++) key[m] = (uint32_t)(fetch(m * kWave + lane) >> 32);
                return wave_kth_key<C, 0>(key, a.k);
            };
            if (total <= 4 * kWave) t = search(std::integral_constant<int, 4>());
            else if (total <= 6 * kWave) t = search(std::integral_constant<int, 6>());
            else t = search(std::integral_constant<int, N>());
            if (lane == 0) sKth = t;
        }
        __syncthreads();
        const uint32_t t = sKth, had = sPublished[wave];
        uint32_t kept = 0;
        for (uint32_t i0 = 0; i0 < had; i0 += kWave) {   // (in place: nothing moves to a later position)
            const uint64_t word = (i0 + lane < had) ? sStage[wave][i0 + lane] : 0ull;
            const bool keep = (uint32_t)(word >> 32) >= t && word != 0;
            const uint64_t m = __ballot(keep);
            __builtin_amdgcn_wave_barrier();
            if (keep) sStage[wave][kept + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = word;
            kept += (uint32_t)__popcll(m);
        }
        if (lane == 0) sPublished[wave] = kept;
        list.count = kept;
        __syncthreads();
        n0 = sPublished[0], n1 = sPublished[1], n2 = sPublished[2], n3 = sPublished[3];
        total = n0 + n1 + n2 + n3;
    }
    if (!any_flushed && total <= (uint32_t)kCount) {
        // Common case: a few words more than k in all, none of them merged yet.  The number of staged words that are larger is a
        // word's place in the result, so no sorting network runs at all.  Every lane holds the i-th, (64 + i)-th, ... of the words,
        // every wave compares them with its own staged ones and adds its counts in LDS.
        const uint32_t mine = sPublished[wave];
        auto count = [&](auto lanes_words) __attribute__((always_inline)) {
            constexpr int N = decltype(lanes_words)::value;   // words per lane
            uint64_t word[N];
            uint32_t part[N];
#pragma unroll
            for (int m = 0; m < N; m++) {
                word[m] = fetch(m * kWave + lane);
                part[m] = 0;
            }
            for (uint32_t i = 0; i < mine; i += 4) {   // broadcast reads, four in flight (a staging row has room beyond any count)
                uint64_t o[4];
#pragma unroll
                for (int u = 0; u < 4; u++) o[u] = sStage[wave][i + u];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (i + u >= mine) o[u] = 0ull;   // stale words beyond the count
#pragma unroll
                    for (int m = 0; m < N; m++) part[m] += (o[u] > word[m]) ? 1u : 0u;
                }
            }
#pragma unroll
            for (int m = 0; m < N; m++)
                if (part[m] != 0) atomicAdd(&sPlace[m * kWave + lane], part[m]);
        };
        if (total <= kWave) count(std::integral_constant<int, 1>());   // the same for the whole workgroup
        else if (total <= 2 * kWave) count(std::integral_constant<int, 2>());
        else if (total <= 3 * kWave) count(std::integral_constant<int, 3>());
        else if (M <= 4 || total <= 4 * kWave) count(std::integral_constant<int, 4>());
        else if (total <= 5 * kWave) count(std::integral_constant<int, 5>());
        else count(std::integral_constant<int, M>());
        __syncthreads();
        for (uint32_t i = wave * kWave + lane; i < total; i += kTopkThreads) {
            const uint64_t word = fetch(i);
            const uint32_t place = sPlace[i];
            if (word == 0 || place >= a.k) continue;
            write_slot(place, word);
            // this block's k-th score bounds the row's final k-th from below
            if (a.row_bound && place == a.k - 1) atomicMax(&a.row_bound[b], (uint32_t)(word >> 32));
        }
        for (uint32_t p = total + wave * kWave + lane; p < a.k; p += kTopkThreads) write_slot(p, 0ull);
        return;
    }
    if (wave != 0) return;

    for (uint32_t w = 1; w < kTopkWaves; w++) {
        const uint32_t n = sPublished[w];
        for (uint32_t p0 = 0; p0 < n; p0 += kWave) {
            const uint32_t p = p0 + lane;
            uint64_t word = 0;
            if (p < n) word = sStage[w][p];
            list.offer(word != 0, word);
        }
    }
    list.finish();
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t p = r * kWave + lane;
        if (p < a.k) write_slot(p, list.q[r]);
        if (a.row_bound && p == a.k - 1 && list.q[r] != 0) atomicMax(&a.row_bound[b], (uint32_t)(list.q[r] >> 32));
    }
}

// The scan of a (row, segment) of any width: sBitmap holds a bit for every column of the segment when FILTERED.
template <int R, bool FILTERED>
__device__ __forceinline__ void scan_segment(const TopKArgs& a, uint64_t (*sStage)[WaveTopK<R>::kStageWords], uint32_t* sBitmap)
{
    using List = WaveTopK<R>;
    const uint32_t b = blockIdx.x;
    const uint32_t seg = blockIdx.y;
    const uint32_t wave = threadIdx.x / kWave;
    const uint32_t lane = threadIdx.x % kWave;
    const float* row = a.in + (uint64_t)b * a.pitch;

    // Split the row into an unaligned head (< 4 columns), a body of 16-byte groups and a tail (< 4 columns).
    const uint32_t mis = (uint32_t)(((uintptr_t)row >> 2) & 3);
    uint32_t head = (4 - mis) & 3;
    if (head > a.width) head = a.width;
    const uint32_t nvec = (a.width - head) / 4;
    const uint32_t tail0 = head + nvec * 4;
    const uint32_t gps = (nvec + a.segments - 1) / a.segments;      // groups per segment
    const uint32_t g0 = min(seg * gps, nvec), g1 = min(g0 + gps, nvec);
    const uint32_t lo = (seg == 0) ? 0 : head + 4 * g0;
    const uint32_t hi = (seg == a.segments - 1) ? a.width : head + 4 * g1;

    List list;
    list.init(sStage[wave], lane, a.k);
    if (a.row_bound) {
        const uint32_t t = a.row_bound[b];   // k columns of earlier blocks of this row reach this score
        if (t > score_key(-__builtin_inff())) list.prime(t);
    }

    // Software pipeline: the lane's first 2 * CH 16-byte groups are requested before anything else happens (the filter's
    // chain of dependent loads would otherwise sit in front of the scan), and inside the loop two spans are in flight while
    // one is examined.  Groups beyond the segment are filled with NaN, which fails every comparison below.
    constexpr int CH = 8;
    const float4* body = reinterpret_cast<const float4*>(row + head);
    const uint32_t step = kTopkThreads;
    auto load_span = [&](float4 (&d)[CH], uint32_t first) {   // first: block-uniform group number
        const uint32_t g = first + threadIdx.x;
        if (first + CH * step <= g1) {
#pragma unroll
            for (int u = 0; u < CH; u++) d[u] = body[g + u * step];
        } else {
            const float nan = __uint_as_float(0x7fc00000u);
#pragma unroll
            for (int u = 0; u < CH; u++) {
                d[u] = make_float4(nan, nan, nan, nan);
                if (g + u * step < g1) d[u] = body[g + u * step];
            }
        }
    };
    // the filter's row range first: it heads a chain of dependent loads
    uint64_t fs = 0, fe = 0;
    if constexpr (FILTERED) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    uint32_t span = g0;
    float4 cur[CH], nxt[CH];
    load_span(cur, span);
    // Head (segment 0) and tail (last segment): at most 3 + 3 columns, taken by wave 0 and examined after the scan.
    uint32_t ht_col = 0xffffffffu;
    float ht_val = 0.0f;
    if (wave == 0) {
        if (seg == 0 && lane < head) ht_col = lane;
        if (seg == a.segments - 1 && lane >= 32 && (lane - 32) < a.width - tail0) ht_col = tail0 + (lane - 32);
        if (ht_col != 0xffffffffu) ht_val = row[ht_col];
    }

    // Filter, part one: mark the listed columns in the bitmap, note which lanes hold a listed column in their first CH groups
    // (they sit out the priming below), and request the scores of the first kFU * 256 listed columns.  The listed items
    // themselves are injected after the scan, when the threshold is tight and nearly all of them fail the first compare.
    // Vector loads complete in the order they were issued, so the column numbers are requested between the first and the
    // second span: waiting for them then costs no more than waiting for the first span, which priming needs anyway, and the
    // listed scores (requested last) are not waited for until the scan is over.
    constexpr int kFU = (R >= 2) ? 2 : 4;   // (the longer lists of k > 64 need the registers: fewer listed columns are held at once)
    __shared__ uint32_t sTaint[kTopkThreads / 2];   // 16 bits per lane: bit u = group u of the first two spans holds a listed column
    uint32_t fcol[kFU];
    float fm[kFU], fv[kFU];
    if constexpr (FILTERED) {
#pragma unroll
        for (int u = 0; u < kFU; u++) {
            const uint64_t t = fs + (uint64_t)u * kTopkThreads + threadIdx.x;
            fcol[u] = 0xffffffffu;
            fm[u] = 0.0f;   // utils/Filters.cpp:62 with the default multiplier
            if (t < fe) {
                fcol[u] = a.fidx[t];
                if (a.fmul) fm[u] = a.fmul[t];
            }
        }
    }
    load_span(nxt, span + CH * step);
    if constexpr (FILTERED) {
        const uint32_t words = (hi - lo + 31) / 32;
        for (uint32_t i = threadIdx.x; i < words; i += kTopkThreads) sBitmap[i] = 0;
        if (threadIdx.x < kTopkThreads / 2) sTaint[threadIdx.x] = 0;
        __syncthreads();
        auto mark = [&](uint32_t c) {
            if (c >= lo && c < hi) {
                atomicOr(&sBitmap[(c - lo) >> 5], 1u << ((c - lo) & 31));
                if (c >= head && c < tail0) {
                    const uint32_t gi = (c - head) / 4 - g0;
                    if (gi < 2 * CH * step) atomicOr(&sTaint[(gi % step) >> 1], 1u << (((gi % step) & 1) * 16 + gi / step));
                }
            }
        };
        // With the default multiplier (every listed column is multiplied by 0) the listed scores are only of interest to a
        // wavefront whose k-th score is not above 0 by the end of the scan: they are then read at that point, not up here.
#pragma unroll
        for (int u = 0; u < kFU; u++) {
            fv[u] = 0.0f;
            if (a.fmul && fcol[u] >= lo && fcol[u] < hi) fv[u] = row[fcol[u]];
            mark(fcol[u]);
        }
        for (uint64_t t = fs + (uint64_t)kFU * kTopkThreads + threadIdx.x; t < fe; t += kTopkThreads) mark(a.fidx[t]);
        __syncthreads();
    }

    auto filtered_out = [&](uint32_t col) -> bool {
        if constexpr (FILTERED) {
            return (sBitmap[(col - lo) >> 5] >> ((col - lo) & 31)) & 1u;
        } else {
            return false;
        }
    };

    // Priming: before anything is admitted, every lane takes the best score of its groups in each of the first two spans.
    // The k-th best of a wave's 128 maxima is a score that at least k unfiltered items reach, so nothing below it can be in the
    // result; the k-th best of the 4k scores the four waves publish is a bound for the whole workgroup.  It is found by
    // binary search on the key bits (no sorting), and the scan then admits a few dozen items per row instead of a few
    // hundred.  Groups that hold a listed column are left out, and a lane with nothing else contributes -inf, which only
    // weakens the bound.
    // The two maxima of a lane are those of its groups in the first and in the second span: together the first 2 * CH * 4 KiB of
    // the segment, 60 % of a 27,278-column row.  (A bound from the first span alone admits twice as many items on average
    // and, in the unlucky row of a large batch, ten times as many: the slowest row sets the kernel's time.)
    __shared__ uint32_t sPrime[kTopkWaves][2 * kWave];
    __shared__ uint32_t sPrimeKey;
    auto prime_from_first_spans = [&]() {
        constexpr int PV = 2;
        uint32_t taint = 0;
        if constexpr (FILTERED) taint = (sTaint[threadIdx.x >> 1] >> ((threadIdx.x & 1) * 16)) & 0xffffu;
        uint32_t key[PV];
#pragma unroll
        for (int v = 0; v < PV; v++) {
            float m = -__builtin_inff();
#pragma unroll
            for (int u = 0; u < CH; u++) {
                const float4& g = (v == 0) ? cur[u] : nxt[u];
                const float gm = fmaxf(fmaxf(g.x, g.y), fmaxf(g.z, g.w));   // fmaxf drops NaN
                m = fmaxf(m, ((taint >> (v * CH + u)) & 1u) ? -__builtin_inff() : gm);
            }
            key[v] = score_key(m);
        }
        uint32_t t;
        if constexpr (R == 1) {
            const uint32_t tw = wave_kth_key<PV>(key, a.k);
            uint32_t published = 0;   // wave-uniform
#pragma unroll
            for (int v = 0; v < PV; v++) {
                const bool pub = key[v] >= tw;   // at least k values of the wavefront
                const uint64_t pm = __ballot(pub);
                const uint32_t pos = published + __builtin_amdgcn_mbcnt_hi((uint32_t)(pm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)pm, 0u));
                if (pub && pos < a.k) sPrime[wave][pos] = key[v];
                published += (uint32_t)__popcll(pm);
            }
            __syncthreads();
            uint32_t all[4];   // the 4k published keys, side by side
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const uint32_t i = n * kWave + lane;
                all[n] = (i < kTopkWaves * a.k) ? sPrime[i / a.k][i % a.k] : 0u;
            }
            if (a.k <= 16) t = wave_kth_key<1>(reinterpret_cast<const uint32_t(&)[1]>(all), a.k);
            else if (a.k <= 32) t = wave_kth_key<2>(reinterpret_cast<const uint32_t(&)[2]>(all), a.k);
            else t = wave_kth_key<4>(all, a.k);
        } else {
            // k is a large part of the 512 maxima: they are searched at once, by one wavefront (a different one from row to row, so
            // that the four SIMDs of a compute unit share the searches of the workgroups on it)
#pragma unroll
            for (int v = 0; v < PV; v++) sPrime[wave][v * kWave + lane] = key[v];
            __syncthreads();
            if (wave == ((b >> 8) & 3u)) {
                uint32_t all[4 * PV];
#pragma unroll
                for (int n = 0; n < 4 * PV; n++) all[n] = sPrime[n / PV][(n % PV) * kWave + lane];
                const uint32_t found = wave_kth_key<4 * PV>(all, a.k);
                if (lane == 0) sPrimeKey = found;
            }
            __syncthreads();
            t = sPrimeKey;
        }
        if (t > score_key(-__builtin_inff())) {
            list.prime(t);
            // Rows whose best scores tie in their hundreds (saturated sigmoids: exactly 1.0f in every eighth column) would
            // otherwise stage every group that holds one of them until a list fills up and is sorted.  Among equal scores the
            // lower column wins, so the bound gets a column: a wavefront's first group is 256 consecutive columns, the lowest it
            // will see; if k of them reach the bound, the k-th such column X closes the bound — a score equal to it passes at or
            // before X only, and every later group fails the one compare of the scan.
            const float S = key_score(t);
            const float4& g = cur[0];
            const float e[4] = {g.x, g.y, g.z, g.w};
            const uint32_t col = head + 4 * (span + threadIdx.x);
            bool ok[4];
            uint32_t before = 0, mine = 0, total = 0;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                ok[c] = e[c] >= S;
                if constexpr (FILTERED) {
                    if (ok[c]) ok[c] = !filtered_out(col + c);
                }
                const uint64_t q = __ballot(ok[c]);
                before += __builtin_amdgcn_mbcnt_hi((uint32_t)(q >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)q, 0u));
                mine += ok[c] ? 1u : 0u;
                total += (uint32_t)__popcll(q);
            }
            if (total >= a.k) {   // wave-uniform
                const bool has = before < a.k && a.k <= before + mine;   // exactly one lane
                uint32_t need = has ? a.k - before : 0u, colX = 0;
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (ok[c] && need != 0 && --need == 0) colX = col + c;
                const uint64_t hm = __ballot(has);
                const uint32_t X = (uint32_t)__builtin_amdgcn_readlane((int)colX, __builtin_ctzll(hm));
                list.prime_word(pack_score(S, X));
            }
        }
    };
    if (g0 < g1) prime_from_first_spans();

    // The four scores of one 16-byte group; at most 4 * 64 words are staged.
    auto stage_group = [&](const float4& v, uint32_t col) {
        float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            asm volatile("" : "+v"(e[c]));   // keeps the packing below inside the (rarely taken) branch instead of hoisted for all groups
            bool ok = e[c] >= list.thr_key;
            if (__ballot(ok) == 0) continue;
            if constexpr (FILTERED) {
                if (ok) ok = !filtered_out(col + c);
            }
            list.stage_only(ok, pack_score(e[c], col + c));
        }
    };
    static_assert(CH == 8, "the scan selects among eight groups");
    static_assert(List::kBurst >= 4 * kWave, "a group stages up to 256 words between drains");

    // Body: the block walks the segment in spans of CH * 4 KiB, wave w takes the w-th KiB of each 4 KiB.  The common case
    // costs three vector instructions per group (maximum of four, one compare); groups with a survivor somewhere in the wave
    // are then walked one at a time.
    while (span < g1) {
        const uint32_t gbase = span + threadIdx.x;
        uint32_t hot = 0;
        {
            const float t = list.admission_score(head + 4 * span);   // every column of this span and after is at or beyond that
            const float t1 = list.admission_score(head + 4 * (span + step));   // ... and every column of its groups 1 to 7 at or beyond this
#pragma unroll
            for (int u = 0; u < CH; u++) {
                const float m = fmaxf(fmaxf(cur[u].x, cur[u].y), fmaxf(cur[u].z, cur[u].w));
                if (__ballot(m >= (u == 0 ? t : t1)) != 0) hot |= 1u << u;
            }
        }
        while (hot != 0) {
            const int u = __ffs(hot) - 1;
            hot &= hot - 1;
            const uint32_t col = head + 4 * (gbase + (uint32_t)u * step);
            switch (u) {
            case 0: stage_group(cur[0], col); break;
            case 1: stage_group(cur[1], col); break;
            case 2: stage_group(cur[2], col); break;
            case 3: stage_group(cur[3], col); break;
            case 4: stage_group(cur[4], col); break;
            case 5: stage_group(cur[5], col); break;
            case 6: stage_group(cur[6], col); break;
            default: stage_group(cur[7], col); break;
            }
            list.drain();
        }
#pragma unroll
        for (int u = 0; u < CH; u++) cur[u] = nxt[u];
        span += CH * step;
        load_span(nxt, span + CH * step);
    }

    // Head and tail columns (requested at the start of the kernel).
    if (wave == 0) {
        const bool ok = (ht_col != 0xffffffffu) && (ht_val >= list.thr_key) && !filtered_out(ht_col);
        list.stage_only(ok, pack_score(ht_val, ht_col));
    }

    // Filter, part two: every listed column is injected once with score * multiplier.  The lane that clears a column's bit
    // owns it (a column listed twice is injected once).  The bitmap is no longer consulted after the barrier.
    if constexpr (FILTERED) {
        __syncthreads();
        // A listed column multiplied by 0 scores 0 (or nothing at all, if its score is not finite): it cannot enter the list of
        // a wavefront that already holds k scores above 0, and the final k-th score is at least that wavefront's.
        const bool zeros_matter = a.fmul != nullptr || !(list.thr_key > 0.0f);   // wave-uniform
        for (uint64_t base = fs; base < fe && zeros_matter; base += (uint64_t)kFU * kTopkThreads) {
            if (base != fs || !a.fmul) {
                if (base != fs) {
#pragma unroll
                    for (int u = 0; u < kFU; u++) {
                        const uint64_t t = base + (uint64_t)u * kTopkThreads + threadIdx.x;
                        fcol[u] = 0xffffffffu;
                        fm[u] = 0.0f;
                        if (t < fe) {
                            fcol[u] = a.fidx[t];
                            if (a.fmul) fm[u] = a.fmul[t];
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < kFU; u++) {
                    fv[u] = 0.0f;
                    if (fcol[u] >= lo && fcol[u] < hi) fv[u] = row[fcol[u]];
                }
            }
#pragma unroll
            for (int u = 0; u < kFU; u++) {
                if (base + (uint64_t)u * kTopkThreads + wave * kWave >= fe) break;   // wave-uniform
                bool own = false;
                if (fcol[u] >= lo && fcol[u] < hi) {
                    const uint32_t bit = 1u << ((fcol[u] - lo) & 31);
                    own = (atomicAnd(&sBitmap[(fcol[u] - lo) >> 5], ~bit) & bit) != 0;
                }
                const float v = fm[u] * fv[u];   // utils/Filters.cpp:62
                list.stage_only(own && v == v, pack_score(v, fcol[u]));   // NaN never enters (it fails every comparison)
            }
            list.drain();
        }
    }

    finish_row<R>(list, sStage, a, b, seg, wave, lane);
}

// Four workgroups per compute unit for every R.  (R = 4 filtered spills 12 bytes a lane at that and none at two workgroups, which are
// slower where a batch fills the GPU: 1,024 x 60,000 k = 200 96 us against 131, 256 x 200,000 k = 256 111 against 147; 1,024 x
// 200,000 k = 256 343 against 342.)
template <int R, bool FILTERED>
__global__ __launch_bounds__(kTopkThreads, 4) void topk_scan_kernel(TopKArgs a)
{
    __shared__ uint64_t sStage[kTopkWaves][WaveTopK<R>::kStageWords];
    extern __shared__ uint32_t sBitmap[];
    scan_segment<R, FILTERED>(a, sStage, sBitmap);
}

// The same for a segment of at most G * 1,024 columns, which the workgroup holds in registers: every score is requested before
// anything else happens, and the bound is taken over all of them, so that little more than k words pass it (the scan's bound has
// seen 60 % of a 27,278-column row when it starts to admit words, and admits 1.9 k).  With 1,024 rows on the GPU at once a compute
// unit's four workgroups get their data one after the other, and one's selection runs under the next one's loads.
// Steps: R maxima per lane over its 16-byte groups that hold no listed column; their k-th largest is the bound; every wavefront
// stages its scores that reach it, then strikes out the listed ones, and finish_row puts the words in order.  A segment that this
// does not settle (fewer than k scores above 0 besides the listed ones, more survivors than the staging area holds: ties by the
// hundred) is scanned again in the general way.
template <int R, bool FILTERED, int G>
__global__ __launch_bounds__(kTopkThreads, 4) void topk_block_kernel(TopKArgs a)
{
    using List = WaveTopK<R>;
    __shared__ uint64_t sStage[kTopkWaves][List::kStageWords];
    __shared__ uint32_t sMax[R * kTopkThreads];
    __shared__ uint32_t sTaint[FILTERED ? kTopkThreads : 1];   // bit u: the lane's group u holds a listed column
    __shared__ uint32_t sBound, sNeed, sReach, sStaged;
    extern __shared__ uint32_t sBitmap[];
    const uint32_t b = blockIdx.x, seg = blockIdx.y;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const float* row = a.in + (uint64_t)b * a.pitch;
    // (the segment is cut as the general scan cuts it: at most 6 columns more than its 16-byte groups hold)
    const uint32_t head = min((4 - (uint32_t)(((uintptr_t)row >> 2) & 3)) & 3u, a.width);
    const uint32_t nvec = (a.width - head) / 4, gps = (nvec + a.segments - 1) / a.segments;
    const uint32_t g0 = min(seg * gps, nvec), g1 = min(g0 + gps, nvec);
    const uint32_t lo = (seg == 0) ? 0 : head + 4 * g0, hi = (seg == a.segments - 1) ? a.width : head + 4 * g1;

    uint64_t fs = 0, fe = 0;
    if constexpr (FILTERED) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    f32x4 v[G];
#pragma unroll
    for (int u = 0; u < G; u++) {
        const uint32_t first = lo + u * 4 * kTopkThreads;   // uniform
        const uint32_t col = first + 4 * threadIdx.x;
        if (first + 4 * kTopkThreads <= hi) {
            v[u] = *reinterpret_cast<const float4u*>(row + col);
        } else {
            const float nan = __uint_as_float(0x7fc00000u);   // fails every comparison below
            v[u] = f32x4{nan, nan, nan, nan};
            if (col + 4 <= hi) v[u] = *reinterpret_cast<const float4u*>(row + col);
            else {
                if (col < hi) v[u].x = row[col];
                if (col + 1 < hi) v[u].y = row[col + 1];
                if (col + 2 < hi) v[u].z = row[col + 2];
            }
        }
    }
    uint32_t taint = 0;
    if constexpr (FILTERED) {
        const uint32_t words = (hi - lo + 31) / 32;
        for (uint32_t i = threadIdx.x; i < words; i += kTopkThreads) sBitmap[i] = 0;
        sTaint[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) sReach = sStaged = 0;
    if constexpr (FILTERED) {
        __syncthreads();
        for (uint64_t t = fs + threadIdx.x; t < fe; t += kTopkThreads) {
            const uint32_t c = a.fidx[t];
            if (c >= lo && c < hi) {
                atomicOr(&sBitmap[(c - lo) >> 5], 1u << ((c - lo) & 31));
                atomicOr(&sTaint[((c - lo) / 4) % kTopkThreads], 1u << ((c - lo) / (4 * kTopkThreads)));
            }
        }
        __syncthreads();
        taint = sTaint[threadIdx.x];
    }
    // maximum i of a lane: its groups i, i + R, ...
#pragma unroll
    for (int i = 0; i < R; i++) {
        float m = -__builtin_inff();
#pragma unroll
        for (int u = i; u < G; u += R) {
            float g = fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w));   // fmaxf drops NaN
            if constexpr (FILTERED) g = __uint_as_float(__float_as_uint(g) | (uint32_t)__builtin_amdgcn_sbfe((int)taint, u, 1));   // listed: NaN
            m = fmaxf(m, g);
        }
        sMax[i * kTopkThreads + threadIdx.x] = score_key(m);
    }
    __syncthreads();
    // (one wavefront searches, a different one from row to row, so that the four SIMDs of a compute unit share the searches)
    if (wave == ((b >> 8) & 3u)) {
        uint32_t t;
        if (R == 1 && a.k <= 16) {   // the largest of each lane's four: the exact bound unless two of the k best share a lane
            uint32_t best[1] = {0u};
#pragma unroll
            for (int n = 0; n < 4; n++) best[0] = max(best[0], sMax[n * kWave + lane]);
            t = wave_kth_key<1>(best, a.k);
        } else {
            uint32_t all[4 * R];
#pragma unroll
            for (int n = 0; n < 4 * R; n++) all[n] = sMax[n * kWave + lane];
            t = wave_kth_key<4 * R>(all, a.k);
        }
        if (lane == 0) {
            sBound = t;
            // a bound from the row's other columns (fewer than k words may pass it); read once: other workgroups of the row raise it
            // meanwhile, and the counts below are taken by all wavefronts against one bound
            sNeed = a.row_bound ? max(t, a.row_bound[b]) : t;
        }
    }
    __syncthreads();
    const uint32_t own = sBound, t = sNeed;
    bool failed = own <= score_key(-__builtin_inff());       // fewer than k maxima
    if (FILTERED && own <= score_key(0.0f)) failed = true;   // listed columns score 0 and may belong in the result
    // Saturated activations have thousands of scores at exactly 1.0.  Among equal scores the lower column wins: when k of the
    // segment's first 1,024 columns reach the bound, later ones have to lie above it.
    const float bound = key_score(t);
    float later = bound;
    {
        uint32_t reach = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            bool ok = v[0][c] >= bound;
            if constexpr (FILTERED) {
                const uint32_t off = 4 * threadIdx.x + c;
                if (ok) ok = !((sBitmap[off >> 5] >> (off & 31)) & 1u);
            }
            reach += (uint32_t)__popcll(__ballot(ok));
        }
        if (lane == 0 && reach != 0) atomicAdd(&sReach, reach);
        __syncthreads();
        if (sReach >= a.k) later = key_score(t + 1u);   // (above +inf this is NaN, which nothing reaches)
    }
    uint32_t count = 0;   // wave-uniform
    if (!failed) {
#pragma unroll
        for (int u = 0; u < G; u++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float need = (u == 0) ? bound : later;
                const uint64_t m = __ballot(v[u][c] >= need);
                if (m == 0) continue;
                const uint32_t at = count + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (v[u][c] >= need && at < (uint32_t)List::kStageWords) sStage[wave][at] = pack_score(v[u][c], lo + (u * kTopkThreads + threadIdx.x) * 4 + c);
                count += (uint32_t)__popcll(m);
            }
        }
    }
    const bool full = count > (uint32_t)List::kStageWords - 4;   // (finish_row reads up to three words beyond the last)
    if (full) count = 0;
    if constexpr (FILTERED) {   // the listed ones are struck out, 64 at a time and in place
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint32_t kept = 0;
        for (uint32_t i0 = 0; i0 < count; i0 += kWave) {
            const uint64_t word = (i0 + lane < count) ? sStage[wave][i0 + lane] : 0ull;
            bool keep = word != 0;
            if (keep) {
                const uint32_t off = ~(uint32_t)word - lo;
                keep = !((sBitmap[off >> 5] >> (off & 31)) & 1u);
            }
            const uint64_t m = __ballot(keep);
            __builtin_amdgcn_wave_barrier();
            if (keep) sStage[wave][kept + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = word;
            kept += (uint32_t)__popcll(m);
        }
        count = kept;
    }
    List list;
    list.init(sStage[wave], lane, a.k);
    list.count = count;
    if (lane == 0) atomicAdd(&sStaged, full ? 0x10000u : count);
    __syncthreads();
    failed = failed || sStaged > ((R == 1) ? (uint32_t)List::kCountWords : 4u * (uint32_t)List::kDrainAt);   // the same for the whole workgroup
    if (!failed) {
        finish_row<R>(list, sStage, a, b, seg, wave, lane);
        return;
    }
    scan_segment<R, FILTERED>(a, sStage, sBitmap);
}

// Guided top-K: the producer of the scores also left the maximum of every 64-column segment of every row (the
// dense layer's epilogue has them in registers anyway).  The k-th largest of a row's segment maxima is a score that at least
// k items reach, so only segments whose maximum reaches it can hold a result: about k of them.  The kernel reads the
// row's maxima (1/64 of the row), picks that bound with the same key-bit search the scan uses for priming, and then reads
// just those segments.  With the filter, a maximum that is the score of a listed column says nothing about the unlisted
// ones: it is left out of the bound (its segment is still read).  Rows full of ties read more segments and still come out
// right: the survivors go through the same lists as in the scan.
constexpr uint32_t kGuidedSegWidth = 64;
constexpr uint32_t kGuidedMaxSegs = 2048;   // per workgroup

// E: segment maxima per lane (256 * E >= number of segments); the key search costs in proportion.  R: length of the lists / 64.
// Wide rows are cut into parts of a.part_segs segments, a workgroup each (blockIdx.y); the parts' lists are merged afterwards.
template <int R, bool FILTERED, int E>
__global__ __launch_bounds__(kTopkThreads, R <= 2 ? 4 : 2) void topk_guided_kernel(TopKArgs a)
{
    __builtin_amdgcn_s_setprio(3);   // short kernels issue ahead of a GEMM's wavefronts that share their SIMD
    using List = WaveTopK<R>;
    static_assert(E * kTopkThreads <= kGuidedMaxSegs, "at most kGuidedMaxSegs segments");
    __shared__ uint64_t sStage[kTopkWaves][List::kStageWords];
    __shared__ uint32_t sPrime[kTopkWaves][R * kWave];
    __shared__ uint32_t sListCount, sBound;
    __shared__ uint32_t sChunk[8 * kTopkWaves];   // listed segments per group of 64 maxima
    extern __shared__ uint32_t sDyn[];   // segments to read [nseg] | their maxima [nseg] | best listed score per segment [nseg] | bitmap of listed columns
    const uint32_t b = blockIdx.x;
    const uint32_t seg0 = blockIdx.y * a.part_segs, nseg = min(a.nseg - seg0, a.part_segs);   // this part's segments
    const uint32_t lo = seg0 * kGuidedSegWidth, hi = min(a.width, lo + nseg * kGuidedSegWidth);
    uint32_t* sList = sDyn;
    uint32_t* sListKey = sDyn + nseg;
    uint32_t* sFiltMax = sDyn + 2 * nseg;
    uint32_t* sBitmap = sDyn + 3 * nseg;

    const uint32_t wave = threadIdx.x / kWave;
    const uint32_t lane = threadIdx.x % kWave;
    const float* row = a.in + (uint64_t)b * a.pitch;
    List list;
    list.init(sStage[wave], lane, a.k);
    if (a.row_bound) {
        const uint32_t t = a.row_bound[b];   // k columns of earlier blocks of this row reach this score
        if (t > score_key(-__builtin_inff())) list.prime(t);
    }

    uint64_t fs = 0, fe = 0;
    if constexpr (FILTERED) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    uint32_t mk[E];   // keys of this lane's segment maxima; 0 = no such segment
    {
        const float* mrow = a.seg_max + (uint64_t)b * a.nseg + seg0;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t idx = e * kTopkThreads + threadIdx.x;
            mk[e] = (idx < nseg) ? score_key(mrow[idx]) : 0u;
        }
    }
    
#pragma unroll
    for (int r = 0; r < R; r++) sPrime[wave][r * kWave + lane] = 0;
    if (threadIdx.x == 0) sListCount = 0;

    constexpr int kFU = 4;
    uint32_t fcol[kFU];
    float fm[kFU], fv[kFU];
    // A row with few listed columns and the default multiplier does not read their scores at all (one round trip less on the
    // way to the bound): a segment that holds a listed column is simply left out of the bound, and a listed column's zero is
    // only looked at when zeros can still enter a list.  A long list would leave too few segments for a good bound: such rows,
    // and rows with multipliers, read the listed scores first and leave out only the segments whose maximum is one of them.
    bool light = false;   // the same for the whole workgroup
    if constexpr (FILTERED) {
        light = !a.fmul && (fe - fs) * 2 <= nseg;
        // (the listed columns are requested before the barrier below, which waits for everything in flight: the row's range,
        // the maxima and the first listed columns then cost two round trips, not three)
#pragma unroll
        for (int u = 0; u < kFU; u++) {
            const uint64_t t = fs + (uint64_t)u * kTopkThreads + threadIdx.x;
            fcol[u] = 0xffffffffu;
            fm[u] = 0.0f;   // utils/Filters.cpp:62 with the default multiplier
            if (t < fe) {
                fcol[u] = a.fidx[t];
                if (a.fmul) fm[u] = a.fmul[t];
            }
        }
        const uint32_t words = (hi - lo + 31) / 32;
        for (uint32_t i = threadIdx.x; i < words; i += kTopkThreads) sBitmap[i] = 0;
        for (uint32_t i = threadIdx.x; i < nseg; i += kTopkThreads) sFiltMax[i] = 0;
        __syncthreads();
        auto mark = [&](uint32_t c, float v) {
            atomicOr(&sBitmap[(c - lo) >> 5], 1u << ((c - lo) & 31));
            if (v == v) atomicMax(&sFiltMax[(c - lo) / kGuidedSegWidth], score_key(v));   // a NaN is never a segment's maximum
        };
        if (light) {   // (at most nseg / 2 <= 1024 listed columns: they are all in fcol)
#pragma unroll
            for (int u = 0; u < kFU; u++) {
                fv[u] = 0.0f;
                if (fcol[u] >= lo && fcol[u] < hi) {
                    atomicOr(&sBitmap[(fcol[u] - lo) >> 5], 1u << ((fcol[u] - lo) & 31));
                    sFiltMax[(fcol[u] - lo) / kGuidedSegWidth] = 0xffffffffu;   // equal to no key of a maximum that takes part (NaN patterns aside, which are 0 here)
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < kFU; u++) {
                fv[u] = 0.0f;
                if (fcol[u] >= lo && fcol[u] < hi) fv[u] = row[fcol[u]];
            }
#pragma unroll
            for (int u = 0; u < kFU; u++)
                if (fcol[u] >= lo && fcol[u] < hi) mark(fcol[u], fv[u]);
            for (uint64_t t = fs + (uint64_t)kFU * kTopkThreads + threadIdx.x; t < fe; t += kTopkThreads) {
                const uint32_t c = a.fidx[t];
                if (c >= lo && c < hi) mark(c, row[c]);
            }
        }
    }
    __syncthreads();

    auto filtered_out = [&](uint32_t col) -> bool {
        if constexpr (FILTERED) {
            return (sBitmap[(col - lo) >> 5] >> ((col - lo) & 31)) & 1u;
        } else {
            return false;
        }
    };

    // The bound: k-th largest of the maxima that are not a listed column's score, first per wave, then over the 4k the waves
    // publish.  With fewer than k such maxima there is no bound and every segment is read.
    uint32_t bound = 0;
    {
        uint32_t tk[E];
#pragma unroll
        for (int e = 0; e < E; e++) {
            tk[e] = mk[e];
            if constexpr (FILTERED) {
                const uint32_t idx = e * kTopkThreads + threadIdx.x;
                if (idx < nseg && (light ? sFiltMax[idx] != 0 : sFiltMax[idx] == mk[e])) tk[e] = 0;
            }
        }
        if (a.k <= 16) {   // the same for the whole workgroup
            // Small k: the maxima go to LDS, one wavefront takes the largest of each lane's share (every 64th) and searches
            // those 64.  The k-th largest of them is reached by k real items as well; it is the exact k-th maximum unless two of
            // the k best share a lane (then it is the next one down, and a segment more is read) — one short search instead of
            // a search per wavefront and a second one over what they publish.
#pragma unroll
            for (int e = 0; e < E; e++) {
                const uint32_t idx = e * kTopkThreads + threadIdx.x;
                if (idx < nseg) sListKey[idx] = tk[e];   // (the list of segments is built later)
            }
            __syncthreads();
            if (wave == 0) {
                uint32_t best[1] = {0u};
                for (uint32_t i = lane; i < nseg; i += kWave) best[0] = max(best[0], sListKey[i]);
                const uint32_t t = wave_kth_key<1>(best, a.k);
                if (lane == 0) sBound = t;
            }
        } else if (R > 1 && E <= 4) {
            // k is a large part of the maxima: all of them are searched at once
#pragma unroll
            for (int e = 0; e < E; e++) {
                const uint32_t idx = e * kTopkThreads + threadIdx.x;
                if (idx < nseg) sListKey[idx] = tk[e];
            }
            __syncthreads();
            if (wave == 0) {
                uint32_t all[4 * E];
#pragma unroll
                for (int n = 0; n < 4 * E; n++) all[n] = (n * kWave + lane < nseg) ? sListKey[n * kWave + lane] : 0u;
                const uint32_t t = wave_kth_key<4 * E>(all, a.k);
                if (lane == 0) sBound = t;
            }
        } else {
            const uint32_t tw = wave_kth_key<E>(tk, a.k);
            uint32_t published = 0;   // wave-uniform
#pragma unroll
            for (int e = 0; e < E; e++) {
                const bool pub = tk[e] != 0 && tk[e] >= tw;
                const uint64_t pm = __ballot(pub);
                const uint32_t pos = published + __builtin_amdgcn_mbcnt_hi((uint32_t)(pm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)pm, 0u));
                if (pub && pos < a.k) sPrime[wave][pos] = tk[e];
                published += (uint32_t)__popcll(pm);
            }
            __syncthreads();
            // (one wavefront searches, the others wait: four workgroups share a CU, and what the searches of sixteen wavefronts
            // cost is instruction issue, not latency)
            if (wave == 0) {
                uint32_t all[4 * R];
#pragma unroll
                for (int n = 0; n < 4 * R; n++) {
                    const uint32_t i = n * kWave + lane;
                    all[n] = (i < kTopkWaves * a.k) ? sPrime[i / a.k][i % a.k] : 0u;
                }
                uint32_t t;
                if (R == 1 && a.k <= 32) t = wave_kth_key<2>(reinterpret_cast<const uint32_t(&)[2]>(all), a.k);
                else t = wave_kth_key<4 * R>(all, a.k);
                if (lane == 0) sBound = t;
            }
        }
        __syncthreads();
        const uint32_t t = sBound;
        if (t > score_key(-__builtin_inff())) {
            bound = t;
            list.prime(t);
        }
    }

    // Segments whose maximum (listed or not) reaches the bound.
    uint64_t listed[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const uint32_t idx = e * kTopkThreads + threadIdx.x;
        const bool flagged = idx < nseg && mk[e] >= bound;
        const uint64_t m = __ballot(flagged);
        listed[e] = m;
        if (m == 0) continue;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&sListCount, (uint32_t)__popcll(m));
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
        if (flagged) {
            const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            sList[pos] = idx;
            sListKey[pos] = mk[e];
        }
    }
    __syncthreads();
    const uint32_t count = sListCount;
    constexpr int kSegsInFlight = (R == 1) ? 8 : 16;   // per wavefront
    // More segments than one round of reads takes, and many more than k (rows of tied scores, mostly): the list is written again in ascending
    // order, so that the first round reads the lowest columns and what only ties behind them can be left out.  Lane j holds
    // the count of the j-th group of 64 maxima; a scan over the first lanes gives every group its place.
    const bool heavy = bound != 0 && count > max((uint32_t)(kTopkWaves * kSegsInFlight), 2 * a.k);   // the same for the whole workgroup
    if (heavy) {
        if (lane == 0) {
#pragma unroll
            for (int e = 0; e < E; e++) sChunk[e * kTopkWaves + wave] = (uint32_t)__popcll(listed[e]);
        }
        __syncthreads();   // (everyone has read the count and is done with the unordered list)
        const uint32_t mine = (lane < (uint32_t)(E * kTopkWaves)) ? sChunk[lane] : 0u;
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < E * kTopkWaves; d *= 2) {
            const uint32_t up = (uint32_t)__shfl_up((int)incl, d);
            if (lane >= (uint32_t)d) incl += up;
        }
        const uint32_t excl = incl - mine;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t base = (uint32_t)__shfl((int)excl, e * kTopkWaves + (int)wave);
            const uint64_t m = listed[e];
            if ((m >> lane) & 1ull) {
                const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                sList[pos] = e * kTopkThreads + threadIdx.x;
                sListKey[pos] = mk[e];
            }
        }
        __syncthreads();
    }

    // One lane per column of a segment, eight segments in flight per wave: the usual dozen or two of segments are one round
    // trip.  A segment whose maximum no longer reaches what its columns need is not read: in a row of saturated scores every
    // segment reaches the bound, but once a wavefront holds k of them, later segments that only tie are out.
    bool first_round = heavy;
    // (the listed segments are dealt out one at a time: the usual dozen or two then keep all four wavefronts busy)
    for (uint32_t i0 = wave; i0 < count; i0 += kTopkWaves * kSegsInFlight) {
        float v[kSegsInFlight];
        uint32_t col[kSegsInFlight];
#pragma unroll
        for (int u = 0; u < kSegsInFlight; u++) {
            v[u] = __uint_as_float(0x7fc00000u);   // NaN fails the compare below
            col[u] = 0;
            const uint32_t i = i0 + u * kTopkWaves;
            if (i < count) {
                const uint32_t first = lo + sList[i] * kGuidedSegWidth;
                if (key_score(sListKey[i]) >= list.admission_score(first)) {   // wave-uniform
                    col[u] = first + lane;
                    if (col[u] < hi) v[u] = row[col[u]];
                }
            }
        }
        // Rows of tied scores (saturated activations): when the wavefront's first segments already hold k columns that reach
        // the bound, the largest column among the first k of them goes into the bound, and what only ties behind it is
        // neither staged here nor read later.
        if (first_round) {   // wave-uniform
            first_round = false;
            uint64_t qm[kSegsInFlight];   // lanes whose score reaches the bound and whose column is not listed
            uint32_t reach = 0;
#pragma unroll
            for (int u = 0; u < kSegsInFlight; u++) {
                bool q = v[u] >= list.thr_key;
                qm[u] = 0;
                if (__ballot(q) == 0) continue;
                if (q) q = !filtered_out(col[u]);
                qm[u] = __ballot(q);
                reach += (uint32_t)__popcll(qm[u]);
            }
            if (reach >= a.k) {
                const float S = list.thr_key;
                uint32_t need = a.k, X = 0;
                bool found = false;
#pragma unroll
                for (int u = 0; u < kSegsInFlight; u++) {
                    const uint32_t c = (uint32_t)__popcll(qm[u]);
                    if (found || c == 0) continue;
                    int at;
                    if (need > c) {
                        need -= c;
                        at = 63 - __builtin_clzll(qm[u]);
                    } else {
                        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(qm[u] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)qm[u], 0u));
                        at = __builtin_ctzll(__ballot(((qm[u] >> lane) & 1ull) && rank + 1 == need));
                        found = true;
                    }
                    const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)col[u], at);
                    X = x > X ? x : X;
                }
                list.prime_word(pack_score(S, X));
            }
#pragma unroll
            for (int u = 0; u < kSegsInFlight; u++) {
                if (qm[u] != 0) list.stage_only((qm[u] >> lane) & 1ull, pack_score(v[u], col[u]));
                if ((u & 3) == 3) list.drain();
            }
            list.drain();
            continue;
        }
#pragma unroll
        for (int u = 0; u < kSegsInFlight; u++) {
            bool ok = v[u] >= list.thr_key;
            if (__ballot(ok) == 0) continue;
            if (ok) ok = !filtered_out(col[u]);
            list.stage_only(ok, pack_score(v[u], col[u]));
            if ((u & 3) == 3) list.drain();   // at most four stagings of 64 words between two checks of the fill level
        }
        list.drain();
    }

    // Every listed column is injected once with score * multiplier; the lane that clears a column's bit owns it.  A listed
    // column multiplied by 0 scores 0 (or nothing at all, if its score is not finite): it cannot enter the list of a
    // wavefront that already holds k scores above 0, and the final k-th score is at least that wavefront's.
    if constexpr (FILTERED) {
        __syncthreads();
        const bool zeros_matter = a.fmul != nullptr || !(list.thr_key > 0.0f);   // wave-uniform
        for (uint64_t base = fs; base < fe && zeros_matter; base += (uint64_t)kFU * kTopkThreads) {
            if (base != fs || light) {
                if (base != fs) {
#pragma unroll
                    for (int u = 0; u < kFU; u++) {
                        const uint64_t t = base + (uint64_t)u * kTopkThreads + threadIdx.x;
                        fcol[u] = 0xffffffffu;
                        fm[u] = 0.0f;
                        if (t < fe) {
                            fcol[u] = a.fidx[t];
                            if (a.fmul) fm[u] = a.fmul[t];
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < kFU; u++) {
                    fv[u] = 0.0f;
                    if (fcol[u] >= lo && fcol[u] < hi) fv[u] = row[fcol[u]];
                }
            }
#pragma unroll
            for (int u = 0; u < kFU; u++) {
                if (base + (uint64_t)u * kTopkThreads + wave * kWave >= fe) break;   // wave-uniform
                bool own = false;
                if (fcol[u] >= lo && fcol[u] < hi) {
                    const uint32_t bit = 1u << ((fcol[u] - lo) & 31);
                    own = (atomicAnd(&sBitmap[(fcol[u] - lo) >> 5], ~bit) & bit) != 0;
                }
                const float v = fm[u] * fv[u];   // utils/Filters.cpp:62
                list.stage_only(own && v == v, pack_score(v, fcol[u]));
            }
            list.drain();
        }
    }
    finish_row<R>(list, sStage, a, b, blockIdx.y, wave, lane);
}

// Second stage: one workgroup per row merges `slots` packed partial lists of k words each (every list best first).  A bound
// comes first: if q lists have a d-th word of at least t, then q * d words of the row reach t, so the ceil(k / d)-th largest of
// the lists' d-th words bounds the k-th word; with d about 2 k / slots that rank is in the middle of the lists, and what
// passes is little more than k words, which finish_row puts in order by counting.  (61 lists of 50 words, one row: 27 -> 6 us
// against one wavefront that sorts and merges 64 words at a time.)
// TWICE: the results go to keys2 and values2 too.  (With a test at run time instead the scans and merges of a search's top 100 took 2 to 3 us more,
// 64 x 200 x 100,000 in halves 45.5 against 42.5.)
template <int R, bool TWICE>
__global__ __launch_bounds__(kTopkThreads) void topk_merge_kernel(const uint64_t* partial, uint32_t slots, uint32_t k, float* keys,
                                                                  uint32_t* values, float* keys2, uint32_t* values2)
{
    __builtin_amdgcn_s_setprio(3);   // short kernels issue ahead of a GEMM's wavefronts that share their SIMD
    using List = WaveTopK<R>;
    __shared__ uint64_t sStage[kTopkWaves][List::kStageWords];
    const uint32_t b = blockIdx.x;
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint64_t* src = partial + (uint64_t)b * slots * k;
    TopKArgs a{};
    a.k = k;
    a.keys = keys;
    a.values = values;
    a.keys2 = keys2;
    a.values2 = values2;
    if (slots == 1) {   // already in order
        for (uint32_t p = threadIdx.x; p < k; p += kTopkThreads) {
            float key = -kMaxValue;
            uint32_t col = 0;
            if (src[p] != 0) unpack_score(src[p], key, col);
            keys[(uint64_t)b * k + p] = key;
            values[(uint64_t)b * k + p] = col;
            if constexpr (TWICE) {
                keys2[(uint64_t)b * k + p] = key;
                values2[(uint64_t)b * k + p] = col;
            }
        }
        return;
    }
    List list;
    list.init(sStage[wave], lane, k);
    const uint32_t total = slots * k;
    constexpr int U = 4;
    uint64_t word[U], next[U];
    auto load = [&](uint64_t (&w)[U], uint32_t p0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t p = p0 + u * kTopkThreads + threadIdx.x;
            w[u] = (p < total) ? src[p] : 0ull;
        }
    };
    load(word, 0);
    {
        const uint32_t d = min(k, max((2 * k + slots - 1) / slots, (k + 31) / 32));   // (64 lanes: a rank of 32 at most)
        uint32_t best[1] = {0u};   // a lane's best d-th word (its lists are every 64th)
        for (uint32_t s = lane; s < slots; s += kWave) best[0] = max(best[0], (uint32_t)(src[(uint64_t)s * k + d - 1] >> 32));
        const uint32_t t = wave_kth_key<1>(best, (k + d - 1) / d);
        if (t > score_key(-__builtin_inff())) list.prime(t);
    }
    for (uint32_t p0 = 0; p0 < total; p0 += U * kTopkThreads) {
        if (p0 + U * kTopkThreads < total) load(next, p0 + U * kTopkThreads);
#pragma unroll
        for (int u = 0; u < U; u++) list.stage_only(word[u] != 0, word[u]);
        list.drain();
#pragma unroll
        for (int u = 0; u < U; u++) word[u] = next[u];
    }
    finish_row<R, TWICE>(list, sStage, a, b, 0, wave, lane);
}

// In-place payload gather for the key/value overloads: values[b][j] holds a column number on entry.
template <typename V>
__global__ __launch_bounds__(256) void topk_gather_kernel(const V* in_values, V* values, uint32_t batch, uint32_t width, uint32_t k)
{
    const uint64_t pos = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= (uint64_t)batch * k) return;
    const uint32_t b = (uint32_t)(pos / k), j = (uint32_t)(pos % k);
    const uint32_t col = reinterpret_cast<const uint32_t*>(values)[pos];
    values[pos] = (j < width) ? in_values[(uint64_t)b * width + col] : (V)0;
}

static LibScratch g_partial_of[DSX_MAX_LANES];   // per lane: lanes may run a split top-K at the same time

static int ensure_partial(size_t bytes, uint64_t** out)
{
    LibScratch& buf = g_partial_of[current_lane()];
    if (int rc = lib_scratch_reserve(buf, bytes, "top-K partial lists")) return rc;
    *out = static_cast<uint64_t*>(buf.ptr);
    return DSX_OK;
}

template <int R, int G> static void launch_block(const TopKArgs& a, uint32_t batch, bool filtered, size_t bitmap_bytes)
{
    const dim3 grid(batch, a.segments);
    if (filtered) hipLaunchKernelGGL((topk_block_kernel<R, true, G>), grid, dim3(kTopkThreads), bitmap_bytes, ctx().stream, a);
    else hipLaunchKernelGGL((topk_block_kernel<R, false, G>), grid, dim3(kTopkThreads), 0, ctx().stream, a);
}

template <int R> static int launch_scan(const TopKArgs& a, uint32_t batch, bool filtered, size_t bitmap_bytes)
{
    dim3 grid(batch, a.segments);
    // Segments that fit a workgroup's registers (multipliers other than 0 need the listed scores: the general scan).  A group of 1,024
    // columns is four registers of a lane, of the 128 that four workgroups per compute unit leave, which is what ends the ladder: 27 or
    // 28 groups fit for k <= 128, 29 spill scores (k > 128 spills 20 bytes a lane at 27; filtered forms keep 8 to 44 bytes of the
    // fallback, which few rows reach, in scratch).  The rungs below spare narrower rows the registers and compares they do not need.
    const uint32_t columns = ((a.width / 4 + 1 + a.segments - 1) / a.segments) * 4 + 8;   // an upper bound of a segment's
    if (!a.fmul && columns <= 27 * 4 * kTopkThreads) {
        if (columns <= 2 * 4 * kTopkThreads) launch_block<R, 2>(a, batch, filtered, bitmap_bytes);
        else if (columns <= 8 * 4 * kTopkThreads) launch_block<R, 8>(a, batch, filtered, bitmap_bytes);
        else if (columns <= 16 * 4 * kTopkThreads) launch_block<R, 16>(a, batch, filtered, bitmap_bytes);
        else launch_block<R, 27>(a, batch, filtered, bitmap_bytes);
        DSX_LAUNCH_CHECK("topk_block_kernel");
        return DSX_OK;
    }
    if (filtered)
        hipLaunchKernelGGL((topk_scan_kernel<R, true>), grid, dim3(kTopkThreads), bitmap_bytes, ctx().stream, a);
    else
        hipLaunchKernelGGL((topk_scan_kernel<R, false>), grid, dim3(kTopkThreads), 0, ctx().stream, a);
    DSX_LAUNCH_CHECK("topk_scan_kernel");
    return DSX_OK;
}

template <int R> static int launch_merge(const uint64_t* partial, uint32_t slots, uint32_t k, float* keys, uint32_t* values, uint32_t batch, float* keys2,
                                         uint32_t* values2)
{
    if (keys2) hipLaunchKernelGGL((topk_merge_kernel<R, true>), dim3(batch), dim3(kTopkThreads), 0, ctx().stream, partial, slots, k, keys, values, keys2, values2);
    else hipLaunchKernelGGL((topk_merge_kernel<R, false>), dim3(batch), dim3(kTopkThreads), 0, ctx().stream, partial, slots, k, keys, values, keys2, values2);
    DSX_LAUNCH_CHECK("topk_merge_kernel");
    return DSX_OK;
}

// Number of workgroups per row: enough to fill the device, and small enough segments for the LDS bitmap.
uint32_t topk_segments(uint32_t batch, uint32_t width, bool filtered)
{
    uint32_t s = 1;
    const uint32_t target_blocks = (uint32_t)ctx().num_cus * 4;
    if (batch < target_blocks) s = (target_blocks + batch - 1) / batch;
    const uint32_t max_by_size = std::max(1u, width / 8192);   // keep at least 8192 columns per segment
    s = std::min(s, max_by_size);
    if (filtered) {
        const uint32_t need = (width + (kMaxBitmapBits - 64) - 1) / (kMaxBitmapBits - 64);
        s = std::max(s, need);
    }
    return std::max(1u, s);
}

int topk_run(const float* in, uint32_t pitch, uint32_t width, uint32_t batch, uint32_t k, float* keys, uint32_t* values,
             uint32_t position, const uint32_t* index, const uint64_t* fstart, const uint64_t* fend, const uint32_t* fidx,
             const float* fmul, uint32_t col_offset, uint64_t* partial, uint32_t partial_slots, uint32_t partial_slot0,
             uint32_t forced_segments, uint32_t* row_bound, uint64_t* fixed_scratch, size_t fixed_scratch_words)
{
    const bool filtered = fidx != nullptr;
    TopKArgs a{};
    a.in = in;
    a.pitch = pitch;
    a.width = width;
    a.k = k;
    a.col_offset = col_offset;
    a.position = position;
    a.index = index;
    a.fstart = fstart;
    a.fend = fend;
    a.fidx = fidx;
    a.fmul = fmul;
    a.keys = keys;
    a.values = values;
    a.row_bound = row_bound;
    a.segments = forced_segments ? forced_segments : topk_segments(batch, width, filtered);
    if (fixed_scratch && !partial && a.segments > 1 && (size_t)batch * a.segments * k > fixed_scratch_words)
        return set_error(DSX_EINVAL, "top-K: %u rows x %u segments x k = %u need %zu bytes of partial lists, the fixed scratch holds %zu",
                         batch, a.segments, k, (size_t)batch * a.segments * k * sizeof(uint64_t), fixed_scratch_words * sizeof(uint64_t));
    const uint32_t nvec_max = width / 4 + 1;
    const uint32_t gps = (nvec_max + a.segments - 1) / a.segments;
    const size_t bitmap_bytes = filtered ? ((size_t)(4 * gps + 8 + 31) / 32) * 4 + 16 : 0;
    if (partial) {
        a.partial = partial;
        a.partial_slots = partial_slots;
        a.partial_slot0 = partial_slot0;
    } else if (a.segments > 1) {
        uint64_t* lists = fixed_scratch;
        if (!lists) {
            int rc = ensure_partial((size_t)batch * a.segments * k * sizeof(uint64_t), &lists);
            if (rc) return rc;
        }
        a.partial = lists;
        a.partial_slots = a.segments;
        a.partial_slot0 = 0;
    }
    int rc;
    if (k <= 64)
        rc = launch_scan<1>(a, batch, filtered, bitmap_bytes);
    else if (k <= 128)
        rc = launch_scan<2>(a, batch, filtered, bitmap_bytes);
    else
        rc = launch_scan<4>(a, batch, filtered, bitmap_bytes);
    if (rc) return rc;
    if (!partial && a.segments > 1) return topk_merge(a.partial, a.segments, k, keys, values, batch);
    return DSX_OK;
}

int topk_merge(const uint64_t* partial, uint32_t slots, uint32_t k, float* keys, uint32_t* values, uint32_t batch, float* keys2, uint32_t* values2)
{
    if (k <= 64) return launch_merge<1>(partial, slots, k, keys, values, batch, keys2, values2);
    if (k <= 128) return launch_merge<2>(partial, slots, k, keys, values, batch, keys2, values2);
    return launch_merge<4>(partial, slots, k, keys, values, batch, keys2, values2);
}

// Exact KNN with candidate lists: merges a row's running best list (k packed words, best first) with the candidates the last
// column range left behind, writes the best k back, raises the row's bound to their k-th key and empties the candidate
// lists.  One wavefront per row.  The candidates are the row's shared list (cand, cand_count) and, after a sweep in f16, its `lists`
// private ones, seg[row][list][seg_cap] with fill counts seg_count[row][kF16ListStride].
template <int R>
__global__ __launch_bounds__(kWave) void knn_refresh_kernel(uint64_t* best, const uint64_t* cand, uint32_t* cand_count, uint32_t cap,
                                                            uint32_t k, uint32_t* row_bound, const uint64_t* seg, uint32_t* seg_count,
                                                            uint32_t lists, uint32_t seg_cap)
{
    using List = WaveTopK<R>;
    __shared__ uint64_t sStage[List::kStageWords];
    __shared__ uint32_t sStart[kF16ListStride + 1];
    const uint32_t b = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    List list;
    list.init(sStage, lane, k);
    uint64_t* mine = best + (uint64_t)b * k;
    for (uint32_t p0 = 0; p0 < k; p0 += kWave) {
        const uint32_t p = p0 + lane;
        const uint64_t word = (p < k) ? mine[p] : 0ull;
        list.offer(word != 0, word);
    }
    const uint32_t n = min(cand_count[b], cap);
    const uint64_t* src = cand + (uint64_t)b * cap;
    for (uint32_t p0 = 0; p0 < n; p0 += kWave) {
        const uint32_t p = p0 + lane;
        const uint64_t word = (p < n) ? src[p] : 0ull;
        list.offer(word != 0, word);
    }
    if (seg) {
        // entry e of the lists laid end to end: sStart[l] is where list l starts
        const uint32_t* counts = seg_count + (uint64_t)b * kF16ListStride;
        uint32_t before = 0;
        if (lane == 0) sStart[0] = 0;
        for (uint32_t l0 = 0; l0 < lists; l0 += kWave) {
            uint32_t incl = (l0 + lane < lists) ? min(counts[l0 + lane], seg_cap) : 0u;
#pragma unroll
            for (int d = 1; d < kWave; d *= 2) {
                const uint32_t below = __shfl_up(incl, d);
                if (lane >= (uint32_t)d) incl += below;
            }
            sStart[l0 + lane + 1] = before + incl;
            before += __shfl(incl, kWave - 1);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const uint32_t total = sStart[lists];
        const uint64_t* from = seg + (uint64_t)b * lists * seg_cap;
        for (uint32_t e0 = 0; e0 < total; e0 += kWave) {
            const uint32_t e = e0 + lane;
            uint64_t word = 0;
            if (e < total) {
                uint32_t lo = 0, hi = lists;   // the last list that starts at or before e (empty ones start where the next one does)
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) / 2;
                    if (sStart[mid] <= e) lo = mid;
                    else hi = mid;
                }
                word = from[(uint64_t)lo * seg_cap + (e - sStart[lo])];
            }
            list.offer(word != 0, word);
        }
    }
    list.finish();
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t p = r * kWave + lane;
        if (p < k) mine[p] = list.q[r];
        if (p == k - 1 && list.q[r] != 0) row_bound[b] = max(row_bound[b], (uint32_t)(list.q[r] >> 32));
    }
    if (lane == 0) cand_count[b] = 0;
}

int knn_refresh(uint64_t* best, const uint64_t* cand, uint32_t* cand_count, uint32_t cap, uint32_t k, uint32_t* row_bound, uint32_t batch,
                const uint64_t* seg, uint32_t* seg_count, uint32_t lists, uint32_t seg_cap)
{
    hipStream_t s = ctx().stream;
    if (seg && (lists == 0 || lists > kF16ListStride || !seg_count))
        return set_error(DSX_EINVAL, "knn_refresh: %u lists (1..%u)", lists, kF16ListStride);
    if (k <= 64)
        hipLaunchKernelGGL((knn_refresh_kernel<1>), dim3(batch), dim3(kWave), 0, s, best, cand, cand_count, cap, k, row_bound, seg, seg_count,
                           lists, seg_cap);
    else if (k <= 128)
        hipLaunchKernelGGL((knn_refresh_kernel<2>), dim3(batch), dim3(kWave), 0, s, best, cand, cand_count, cap, k, row_bound, seg, seg_count,
                           lists, seg_cap);
    else
        hipLaunchKernelGGL((knn_refresh_kernel<4>), dim3(batch), dim3(kWave), 0, s, best, cand, cand_count, cap, k, row_bound, seg, seg_count,
                           lists, seg_cap);
    DSX_LAUNCH_CHECK("knn_refresh_kernel");
    return DSX_OK;
}

// ---------------------------------------------------------------------------------------------------------------------
// Output layer fused with its top-K (dsx_fc_topk): the row's best list so far (k packed words) is merged with the candidates
// the layer's last column range appended, minus the columns the row's filter lists (multiplier 0: the sample's own items).
// One wavefront per row.  The filter is applied by hashing the candidates' columns into an LDS table (at most half full,
// linear probing), striking out every listed column found there, and then offering only the candidates still present.
// A row whose candidate list filled up is flagged, and layer_redo_kernel computes flagged rows from scratch after the last range.
constexpr uint32_t kLayerTableSlots = 8192;   // twice the candidate capacity the layer search uses
constexpr uint32_t kLayerEmpty = 0xffffffffu, kLayerStruck = 0xfffffffeu;   // (no column has these numbers: widths stay below 2^32 - 2)

struct LayerRefreshArgs {
    uint64_t* best;            // [batch][k] packed words, best first, 0 = empty
    const uint64_t* cand;      // [batch][cap]
    uint32_t* cand_count;      // [batch], reset to 0 here
    uint32_t cap;
    uint32_t k;
    uint32_t* row_bound;       // [batch] key of the row's k-th best score, raised here
    uint32_t* row_flag;        // [batch] != 0: the row's list overflowed in this or an earlier range
    uint32_t* flagged_total;   // host-visible word that is set to 1 when a row is flagged (may be NULL)
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;      // NULL: no filter
    float* keys;               // final range only (else NULL): [batch][k] results
    uint32_t* values;
    uint32_t n;                // columns of the layer
    uint32_t first_columns;    // columns of the first block, whose listed columns the scanning top-K has dealt with
};

__device__ __forceinline__ uint32_t layer_hash(uint32_t col, uint32_t shift) { return (col * 2654435761u) >> shift; }

template <int R>
__global__ __launch_bounds__(kWave) void layer_refresh_kernel(LayerRefreshArgs a)
{
    __builtin_amdgcn_s_setprio(3);   // short kernels issue ahead of a GEMM's wavefronts that share their SIMD
    using List = WaveTopK<R>;
    __shared__ uint64_t sStage[List::kStageWords];
    __shared__ uint32_t sTable[kLayerTableSlots];
    const uint32_t b = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const uint32_t count = a.cand_count[b];
    bool flagged = a.row_flag[b] != 0;
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) a.cand_count[b] = 0;
    if (!flagged && count > a.cap) {
        flagged = true;
        if (lane == 0) {
            a.row_flag[b] = 1;
            if (a.flagged_total) *(volatile uint32_t*)a.flagged_total = 1u;
        }
    }
    const bool final_range = a.keys != nullptr;
    if (flagged) return;
    uint64_t fs = 0, fe = 0;
    if (a.fidx && (count > 0 || final_range)) {
        uint32_t r = a.position + b;
        if (a.index) r = a.index[r];
        fs = a.fstart[r];
        fe = a.fend[r];
    }
    List list;
    list.init(sStage, lane, a.k);
    const uint64_t* src = a.cand + (uint64_t)b * a.cap;
    const bool filtering = fe > fs && count > 0;   // wave-uniform
    // table size: a power of two, at least twice the candidates
    uint32_t bits = 7;
    while ((1u << bits) < 2 * count) bits++;
    const uint32_t mask = (1u << bits) - 1, shift = 32 - bits;
    if (filtering) {
        for (uint32_t i = lane; i <= mask; i += kWave) sTable[i] = kLayerEmpty;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (uint32_t p = lane; p < count; p += kWave) {
            const uint32_t col = ~(uint32_t)src[p];
            uint32_t h = layer_hash(col, shift);
            while (atomicCAS(&sTable[h], kLayerEmpty, col) != kLayerEmpty) h = (h + 1) & mask;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (uint64_t t = fs + lane; t < fe; t += kWave) {
            const uint32_t col = a.fidx[t];
            uint32_t h = layer_hash(col, shift);
            for (;;) {
                const uint32_t v = sTable[h];
                if (v == kLayerEmpty) break;
                if (v == col) {
                    sTable[h] = kLayerStruck;
                    break;
                }
                h = (h + 1) & mask;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    uint64_t* mine = a.best + (uint64_t)b * a.k;
    for (uint32_t p0 = 0; p0 < a.k; p0 += kWave) {
        const uint32_t p = p0 + lane;
        const uint64_t word = (p < a.k) ? mine[p] : 0ull;
        list.offer(word != 0, word);
    }
    for (uint32_t p0 = 0; p0 < count; p0 += kWave) {
        const uint32_t p = p0 + lane;
        const uint64_t word = (p < count) ? src[p] : 0ull;
        bool live = word != 0;
        if (filtering && live) {
            const uint32_t col = ~(uint32_t)word;
            uint32_t h = layer_hash(col, shift);
            for (;;) {
                const uint32_t v = sTable[h];
                if (v == col) break;
                if (v == kLayerEmpty) {   // struck out: the chain ends without the column
                    live = false;
                    break;
                }
                h = (h + 1) & mask;
            }
        }
        list.offer(live, word);
    }
    list.finish();
    if (final_range) {
        // The listed columns beyond the first block were struck out above, but a listed column scores 0, not nothing
        // (utils/Filters.cpp:62 multiplies, kCalculateTopK then sees the zero): when the row's k-th score is not above 0, or the
        // row has fewer than k scores, such a zero belongs in the result.  Those rows are computed again (layer_redo_kernel).
        uint64_t kth = 0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint64_t w = shfl_u64(list.q[r], (int)((a.k - 1) & (kWave - 1)));
            if ((int)((a.k - 1) / kWave) == r) kth = w;
        }
        bool zeros_matter = false;
        if (fe > fs && (kth == 0 || (uint32_t)(kth >> 32) <= score_key(0.0f))) {
            bool beyond = false;
            for (uint64_t t = fs + lane; t < fe; t += kWave) {
                const uint32_t col = a.fidx[t];
                beyond |= col >= a.first_columns && col < a.n;
            }
            zeros_matter = __ballot(beyond) != 0;
        }
        if (zeros_matter) {
            if (lane == 0) {
                a.row_flag[b] = 1;
                if (a.flagged_total) *(volatile uint32_t*)a.flagged_total = 1u;
            }
            return;
        }
        write_final<R>(list.q, lane, a.k, 0, a.keys + (uint64_t)b * a.k, a.values + (uint64_t)b * a.k);
        return;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t p = r * kWave + lane;
        if (p < a.k) mine[p] = list.q[r];
        if (p == a.k - 1 && list.q[r] != 0) a.row_bound[b] = max(a.row_bound[b], (uint32_t)(list.q[r] >> 32));
    }
}

int layer_refresh_run(const LayerRefresh& r, uint32_t batch)
{
    if (2 * r.cap > kLayerTableSlots) return set_error(DSX_EINVAL, "layer_refresh: candidate capacity %u exceeds %u", r.cap, kLayerTableSlots / 2);
    LayerRefreshArgs a{};
    a.best = r.best; a.cand = r.cand; a.cand_count = r.cand_count; a.cap = r.cap; a.k = r.k;
    a.row_bound = r.row_bound; a.row_flag = r.row_flag; a.flagged_total = r.flagged_total;
    a.position = r.position; a.index = r.index; a.fstart = r.fstart; a.fend = r.fend; a.fidx = r.fidx;
    a.keys = r.keys; a.values = r.values;
    a.n = r.n;
    a.first_columns = r.first_columns;
    hipStream_t s = ctx().stream;
    if (a.k <= 64) hipLaunchKernelGGL((layer_refresh_kernel<1>), dim3(batch), dim3(kWave), 0, s, a);
    else if (a.k <= 128) hipLaunchKernelGGL((layer_refresh_kernel<2>), dim3(batch), dim3(kWave), 0, s, a);
    else hipLaunchKernelGGL((layer_refresh_kernel<4>), dim3(batch), dim3(kWave), 0, s, a);
    DSX_LAUNCH_CHECK("layer_refresh_kernel");
    return DSX_OK;
}

// Rows of a layer whose lists filled up (thousands of scores tied at the top), or whose result needs the zeros of listed columns: the
// whole row once more, without any list that could fill up.  The flagged rows are gathered 32 at a time and the columns cut into as many
// parts as keep the GPU busy; a workgroup walks its part in steps of 512 columns, 128 per wavefront, sums in ascending pairs of k
// (bias last: as a stored layer), W from memory straight into registers one chunk of eight k ahead.  The scores go through LDS, 128
// columns at a time, to the wavefront that keeps the row's list, which merges what beats the row's k-th word when more than 32 words wait; the last
// workgroup of 32 rows to finish merges their parts.  Bound by reading W once per 32 rows from the caches; where no row is flagged, by
// the launch.
// 4,096 x 1,024 x 27,278 saturated, every row flagged: 2.8 ms, 80 TFLOP/s, of a call of 8 (4.7 of them the sweep, all of whose
// scores pass); a wavefront per row that read W for itself took 0.5 s.
constexpr uint32_t kRedoGrid = 256;   // (a grid that finds nothing to do takes its place beside another lane's GEMM first: 512 of 62 KiB of LDS 25 us, these of 34 KiB 6)
constexpr int kRedoBlocks = 4;        // blocks of 32 columns per wavefront and step
constexpr uint32_t kRedoRows = 32, kRedoCols = 128, kRedoSpan = 1024, kRedoWait = 32, kRedoParts = 128;

struct LayerRedoArgs {
    const float* X;
    const float* W;
    const float* bias;
    uint32_t ldx, ldw, batch, kdim, n, k;
    uint32_t act;
    float slope, alpha, lambda;
    uint32_t position;
    const uint32_t* index;
    const uint64_t* fstart;
    const uint64_t* fend;
    const uint32_t* fidx;       // NULL: no filter
    const uint32_t* row_flag;   // [batch]
    uint64_t* partial;          // [work items][kRedoRows][k]
    uint32_t* done;             // [groups of kRedoRows] finished parts, 0 before the launch
    float* keys;
    uint32_t* values;
};

template <int R>
__global__ __launch_bounds__(256, 2) void layer_redo_kernel(LayerRedoArgs a)
{
    using List = WaveTopK<R>;
    __shared__ float sScore[kRedoRows][kRedoCols + 4];
    __shared__ uint64_t sWait[kRedoRows][kRedoWait];        // words of a row that wait to be merged
    __shared__ uint64_t sStage[4][kRedoWait + kRedoCols];   // per wavefront: what is merged
    __shared__ uint64_t sThr[kRedoRows];                    // the row's k-th word so far
    __shared__ uint32_t sCount[kRedoRows], sMerged[kRedoRows];   // its staged words, whether it has a list yet
    __shared__ uint32_t sBits[kRedoRows][kRedoSpan / 32];   // listed columns of the span
    __shared__ uint32_t sRows[kRedoRows], sWave[4], sAny, sLast;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint32_t l32 = lane & 31, lhi = lane >> 5;
    __builtin_amdgcn_s_setprio(3);
    if (threadIdx.x == 0) sAny = 0;
    __syncthreads();
    uint32_t mine = 0;
    for (uint32_t b = threadIdx.x; b < a.batch; b += 256) mine += a.row_flag[b] != 0 ? 1u : 0u;
    if (mine != 0) atomicAdd(&sAny, mine);
    __syncthreads();
    const uint32_t flagged = sAny;
    if (flagged == 0) return;   // the same for the whole grid
    const uint32_t groups = (flagged + kRedoRows - 1) / kRedoRows, spans = (a.n + kRedoSpan - 1) / kRedoSpan;
    const uint32_t most = max(1u, min(kRedoParts, gridDim.x / groups)), per = (spans + most - 1) / most, parts = (spans + per - 1) / per;

    for (uint32_t item = blockIdx.x; item < groups * parts; item += gridDim.x) {
        const uint32_t group = item / parts, part = item % parts;
        const uint32_t rows = min(flagged - group * kRedoRows, kRedoRows);
        // the rows themselves: the flagged ones in ascending order, from the (32 group)-th on
        uint32_t before = 0;
        for (uint32_t b0 = 0; b0 < a.batch && before < (group + 1) * kRedoRows; b0 += 256) {
            const bool f = b0 + threadIdx.x < a.batch && a.row_flag[b0 + threadIdx.x] != 0;
            const uint64_t m = __ballot(f);
            __syncthreads();   // (sWave and sRows have been read)
            if (lane == 0) sWave[wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t at = before;
            for (uint32_t w = 0; w < 4; w++) {
                if (w < wave) at += sWave[w];
                before += sWave[w];
            }
            at += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (f && at / kRedoRows == group) sRows[at % kRedoRows] = b0 + threadIdx.x;
        }
        if (threadIdx.x < kRedoRows) {
            sThr[threadIdx.x] = 0;
            sCount[threadIdx.x] = sMerged[threadIdx.x] = 0;
        }
        __syncthreads();
        const float* x = a.X + (uint64_t)sRows[min(l32, rows - 1)] * a.ldx;   // (lanes beyond the rows repeat the last one)
        uint64_t* lists = a.partial + (uint64_t)item * kRedoRows * a.k;
        // (a row's waiting words, their number, its k-th word and its list belong to one wavefront)
        auto merge = [&](uint32_t r, uint32_t staged) {
            const bool has = sMerged[r] != 0;
            List list;
            list.init(sStage[wave], lane, a.k);
            uint64_t* mem = lists + (uint64_t)r * a.k;
#pragma unroll
            for (int q = 0; q < R; q++) {
                const uint32_t p = q * kWave + lane;
                if (has && p < a.k) list.q[q] = mem[p];
            }
            list.count = staged;
            list.finish();
#pragma unroll
            for (int q = 0; q < R; q++) {
                const uint32_t p = q * kWave + lane;
                if (p < a.k) mem[p] = list.q[q];
            }
            if (lane == 0) {
                sThr[r] = list.thr;
                sMerged[r] = 1;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        const uint32_t end = min(a.n, (part + 1) * per * kRedoSpan);
        for (uint32_t span = part * per * kRedoSpan; span < end; span += kRedoSpan) {
            if (a.fidx) {   // (the bits of the span before were last read before the barrier at the end of its last step)
                for (uint32_t i = threadIdx.x; i < kRedoRows * kRedoSpan / 32; i += 256) (&sBits[0][0])[i] = 0;
                __syncthreads();
                for (uint32_t r = wave; r < rows; r += 4) {
                    uint32_t f = a.position + sRows[r];
                    if (a.index) f = a.index[f];
                    const uint64_t fe = a.fend[f];
                    for (uint64_t t = a.fstart[f] + lane; t < fe; t += kWave) {
                        const uint32_t c = a.fidx[t];
                        if (c >= span && c - span < kRedoSpan) atomicOr(&sBits[r][(c - span) >> 5], 1u << ((c - span) & 31));
                    }
                }
                // (the barrier behind the first step's scores comes before they are read)
            }
            const uint32_t span_end = min(end, span + kRedoSpan);
            for (uint32_t step = span; step < span_end; step += kRedoBlocks * kRedoCols) {
                // block j of a wavefront: columns step + 128 j + 32 wave + l32
                const float* w = a.W + (uint64_t)lhi * a.ldw;
                uint32_t wcol[kRedoBlocks];
#pragma unroll
                for (int j = 0; j < kRedoBlocks; j++) wcol[j] = min(step + kRedoCols * j + 32 * wave + l32, a.n - 1);
                struct Stage {
                    float x[8], w[4][kRedoBlocks];
                };
                auto load = [&](Stage& s, uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
                    for (int t = 0; t < 4; t++)
#pragma unroll
                        for (int j = 0; j < kRedoBlocks; j++) s.w[t][j] = w[(uint64_t)(k0 + 2 * t) * a.ldw + wcol[j]];
#pragma unroll
                    for (int e = 0; e < 8; e += 4) {
                        const float4u v = *reinterpret_cast<const float4u*>(x + k0 + e);
                        s.x[e] = v.x; s.x[e + 1] = v.y; s.x[e + 2] = v.z; s.x[e + 3] = v.w;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                floatx16 acc[kRedoBlocks];
#pragma unroll
                for (int j = 0; j < kRedoBlocks; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[j][v] = 0.0f;
                auto multiply = [&](const Stage& s) __attribute__((always_inline)) {
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const float xv = lhi ? s.x[2 * t + 1] : s.x[2 * t];
#pragma unroll
                        for (int j = 0; j < kRedoBlocks; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv, s.w[t][j], acc[j], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                const uint32_t chunks = a.kdim / 8, rest = a.kdim - chunks * 8;
                if (chunks != 0) {
                    const uint32_t last = (chunks - 1) * 8;
                    Stage s0, s1;
                    load(s0, 0);
                    uint32_t k0 = 0, left = chunks;
                    for (; left >= 2; left -= 2) {   // (the last chunk is requested again and not used)
                        load(s1, k0 + 8);
                        multiply(s0);
                        load(s0, min(k0 + 16, last));
                        multiply(s1);
                        k0 += 16;
                    }
                    if (left) multiply(s0);
                }
                if (rest != 0) {
                    Stage s;
#pragma unroll
                    for (int t = 0; t < 4; t++)
#pragma unroll
                        for (int j = 0; j < kRedoBlocks; j++) s.w[t][j] = (2 * t + lhi < rest) ? w[(uint64_t)(chunks * 8 + 2 * t) * a.ldw + wcol[j]] : 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) s.x[e] = ((uint32_t)e < rest) ? x[chunks * 8 + e] : 0.0f;
                    multiply(s);
                }
#pragma unroll
                for (int j = 0; j < kRedoBlocks; j++) {
                    const uint32_t c0 = step + kRedoCols * j;
                    if (c0 >= span_end) break;   // the same for the whole workgroup
#pragma unroll
                    for (int v = 0; v < 16; v++) sScore[8 * (v / 4) + 4 * lhi + v % 4][32 * wave + l32] = acc[j][v];
                    __syncthreads();
                    float bias[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) bias[h] = (a.bias && c0 + h * kWave + lane < span_end) ? a.bias[c0 + h * kWave + lane] : 0.0f;
#pragma unroll 1
                    for (uint32_t r = wave; r < rows; r += 4) {
                        const uint64_t thr = sThr[r];
                        const uint32_t waiting = sCount[r];   // wave-uniform
                        uint64_t word[2], m[2];
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const uint32_t c = c0 + h * kWave + lane;
                            float y = activate_rt(sScore[r][h * kWave + lane] + bias[h], a.act, a.slope, a.alpha, a.lambda);
                            // a listed column keeps its place with score * 0 (utils/Filters.cpp:62), once however often it is listed
                            if (a.fidx && ((sBits[r][(c - span) >> 5] >> (c & 31)) & 1u)) y *= 0.0f;
                            word[h] = pack_score(y, c);
                            m[h] = __ballot(c < span_end && y == y && word[h] > thr);
                        }
                        if ((m[0] | m[1]) == 0) continue;
                        const uint32_t first = (uint32_t)__popcll(m[0]), count = waiting + first + (uint32_t)__popcll(m[1]);
                        const bool full = count > kRedoWait;
                        uint64_t* to = full ? sStage[wave] : sWait[r];
                        if (full && lane < waiting) to[lane] = sWait[r][lane];
#pragma unroll
                        for (int h = 0; h < 2; h++)
                            if ((m[h] >> lane) & 1ull)
                                to[waiting + (h ? first : 0u) + __builtin_amdgcn_mbcnt_hi((uint32_t)(m[h] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[h], 0u))] = word[h];
                        if (full) merge(r, count);
                        if (lane == 0) sCount[r] = full ? 0u : count;
                    }
                    __syncthreads();   // the scores have been read
                }
            }
        }
        for (uint32_t r = wave; r < rows; r += 4) {
            const uint32_t waiting = sCount[r];
            if (lane < waiting) sStage[wave][lane] = sWait[r][lane];
            merge(r, waiting);
        }
        // The last part of the group to finish merges them all.  (Release: the lists are in memory before the count; acquire: they are
        // read after it.  Workgroups of a group may run on different XCDs, whose L2s are not kept coherent.)
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) sLast = atomicAdd(&a.done[group], 1u) + 1 == parts ? 1u : 0u;
        __syncthreads();
        if (sLast != 0) {
            __threadfence();
            for (uint32_t r = wave; r < rows; r += 4) {
                List list;
                list.init(sStage[wave], lane, a.k);
                for (uint32_t s = 0; s < parts; s++) {
                    const uint64_t* src = a.partial + ((uint64_t)(group * parts + s) * kRedoRows + r) * a.k;
                    for (uint32_t p0 = 0; p0 < a.k; p0 += kWave) {
                        const uint64_t word = (p0 + lane < a.k) ? src[p0 + lane] : 0ull;
                        list.stage_only(word != 0, word);
                        list.finish();
                    }
                }
                const uint64_t row = sRows[r];
                write_final<R>(list.q, lane, a.k, 0, a.keys + row * a.k, a.values + row * a.k);
            }
        }
        __syncthreads();   // (sRows is written again)
    }
}

uint64_t layer_redo_words(uint32_t batch, uint32_t k) { return (uint64_t)std::max(kRedoGrid, (batch + kRedoRows - 1) / kRedoRows) * kRedoRows * k; }
uint32_t layer_redo_groups(uint32_t batch) { return (batch + kRedoRows - 1) / kRedoRows; }

int layer_redo_run(const LayerRedo& r, uint32_t batch)
{
    LayerRedoArgs a{};
    a.X = r.X; a.W = r.W; a.bias = r.bias; a.ldx = r.ldx; a.ldw = r.ldw; a.batch = batch; a.kdim = r.kdim; a.n = r.n; a.k = r.k;
    a.act = r.act; a.slope = r.slope; a.alpha = r.alpha; a.lambda = r.lambda;
    a.position = r.position; a.index = r.index; a.fstart = r.fstart; a.fend = r.fend; a.fidx = r.fidx;
    a.row_flag = r.row_flag; a.partial = r.partial; a.done = r.done; a.keys = r.keys; a.values = r.values;
    hipStream_t s = ctx().stream;
    if (a.k <= 64) hipLaunchKernelGGL((layer_redo_kernel<1>), dim3(kRedoGrid), dim3(256), 0, s, a);
    else if (a.k <= 128) hipLaunchKernelGGL((layer_redo_kernel<2>), dim3(kRedoGrid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((layer_redo_kernel<4>), dim3(kRedoGrid), dim3(256), 0, s, a);
    DSX_LAUNCH_CHECK("layer_redo_kernel");
    return DSX_OK;
}

// Segments per workgroup of the guided top-K: up to 2,048, and down to 512 where that would leave three quarters of the compute
// units without a workgroup (4 x 1,000,000 k = 10: 10.8 -> 9.7 us; a merge is the price, 100 x 60,000: 7.5 us whole, 10.2 cut).
static uint32_t guided_part_segs(uint32_t nseg, uint32_t batch)
{
    uint32_t most = kGuidedMaxSegs;
    while (most > kGuidedMaxSegs / 4 && 4ull * batch * ((nseg + most - 1) / most) <= (uint64_t)ctx().num_cus) most /= 2;
    const uint32_t parts = (nseg + most - 1) / most;
    return (nseg + parts - 1) / parts;
}

uint32_t topk_guided_parts(uint32_t width, uint32_t batch)
{
    const uint32_t nseg = (width + kGuidedSegWidth - 1) / kGuidedSegWidth, per = guided_part_segs(nseg, batch);
    return (nseg + per - 1) / per;
}

template <int R, bool FILTERED> static void launch_guided(const TopKArgs& a, uint32_t batch, uint32_t parts)
{
    size_t lds = (size_t)a.part_segs * 8;
    if (FILTERED) lds += (size_t)a.part_segs * (4 + kGuidedSegWidth / 8);
    const dim3 grid(batch, parts), block(kTopkThreads);
    hipStream_t s = ctx().stream;
    if (a.part_segs <= 2 * kTopkThreads) hipLaunchKernelGGL((topk_guided_kernel<R, FILTERED, 2>), grid, block, lds, s, a);
    else if (a.part_segs <= 4 * kTopkThreads) hipLaunchKernelGGL((topk_guided_kernel<R, FILTERED, 4>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((topk_guided_kernel<R, FILTERED, 8>), grid, block, lds, s, a);
}

// Guided top-K over in[batch][pitch] with the maxima of its 64-column segments; with partial != NULL the parts' packed lists go to
// partial[b][partial_slot0 + part] (as topk_run).
int topk_guided_launch(const float* in, uint32_t pitch, uint32_t width, uint32_t batch, uint32_t k, float* keys, uint32_t* values,
                       const float* seg_max, uint32_t position, const uint32_t* index, const uint64_t* fstart, const uint64_t* fend,
                       const uint32_t* fidx, const float* fmul, uint32_t col_offset, uint64_t* partial, uint32_t partial_slots,
                       uint32_t partial_slot0, uint32_t* row_bound)
{
    TopKArgs a{};
    a.in = in;
    a.pitch = pitch;
    a.width = width;
    a.k = k;
    a.segments = 1;
    a.col_offset = col_offset;
    a.position = position;
    a.index = index;
    a.fstart = fstart;
    a.fend = fend;
    a.fidx = fidx;
    a.fmul = fmul;
    a.keys = keys;
    a.values = values;
    a.row_bound = row_bound;
    a.seg_max = seg_max;
    a.nseg = (width + kGuidedSegWidth - 1) / kGuidedSegWidth;
    a.part_segs = guided_part_segs(a.nseg, batch);
    if (!partial && a.part_segs < a.nseg && a.nseg <= kGuidedMaxSegs) {
        // (a graph keeps no address of the library's scratch, which may have to be allocated now and may move when it grows)
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        DSX_HIP(hipStreamIsCapturing(ctx().stream, &capturing));
        if (capturing != hipStreamCaptureStatusNone) a.part_segs = a.nseg;
    }
    const uint32_t parts = (a.nseg + a.part_segs - 1) / a.part_segs;
    if (partial) {
        a.partial = partial;
        a.partial_slots = partial_slots;
        a.partial_slot0 = partial_slot0;
    } else if (parts > 1) {
        if (int rc = ensure_partial((size_t)batch * parts * k * sizeof(uint64_t), &a.partial)) return rc;
        a.partial_slots = parts;
    }
    if (k <= 64) {
        if (fidx) launch_guided<1, true>(a, batch, parts);
        else launch_guided<1, false>(a, batch, parts);
    } else {
        if (fidx) launch_guided<2, true>(a, batch, parts);
        else launch_guided<2, false>(a, batch, parts);
    }
    DSX_LAUNCH_CHECK("topk_guided_kernel");
    if (!partial && parts > 1) return topk_merge(a.partial, parts, k, keys, values, batch);
    return DSX_OK;
}

// Whether the guided top-K is the faster one, given segment maxima: k <= 64 and at least 3 k segments (us, guided / scan, filtered:
// 1,024 x 27,278 k = 10 8.1 / 23, k = 64 20.8 / 26; 300 x 5,000 k = 32 11.0 / 10.7); up to 128, where k segments are a large part of
// the row, for score matrices that do not stay in the caches anyway (4,096 x 27,278 k = 100 76 / 96, k = 128 94 / 99; 64 x 27,278
// k = 100 19.5 / 17.6); never above (8 x 500,000 k = 200 40 / 34).
bool topk_guided_pays(uint32_t batch, uint32_t width, uint32_t k)
{
    const uint32_t nseg = (width + kGuidedSegWidth - 1) / kGuidedSegWidth;
    if (k <= 64) return nseg >= 3 * k;
    return k <= 128 && nseg >= 4 * k && (uint64_t)batch * nseg >= 100000;
}

int topk_guided_run(const float* in, uint32_t width, uint32_t batch, uint32_t k, float* keys, uint32_t* values, const float* seg_max,
                    uint32_t seg_width, uint32_t position, const uint32_t* index, const uint64_t* fstart, const uint64_t* fend,
                    const uint32_t* fidx, const float* fmul)
{
    bool guided = seg_max && seg_width == kGuidedSegWidth && topk_guided_pays(batch, width, k);
    if (guided && width > kGuidedMaxSegs * kGuidedSegWidth) {
        // (these rows are always cut, and a graph may keep no address of the library's scratch: the scan takes most of them whole)
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        DSX_HIP(hipStreamIsCapturing(ctx().stream, &capturing));
        guided = capturing == hipStreamCaptureStatusNone;
    }
    if (!guided)
        return topk_run(in, width, width, batch, k, keys, values, position, index, fstart, fend, fidx, fmul, 0, nullptr, 0, 0, 0);
    return topk_guided_launch(in, width, width, batch, k, keys, values, seg_max, position, index, fstart, fend, fidx, fmul, 0, nullptr, 0, 0,
                              nullptr);
}

// Fixed scratch of dsx_topk_filtered_static: the packed partial lists of rows split over several workgroups,
// [batch][segments][k] words.  Every device the library runs on holds its own copy of the array at its own address; host code
// must use the address hipGetSymbolAddress reports for the current device, never the array's name.
constexpr size_t kStaticScratchWords = (size_t)1 << 21;   // 16 MiB
static __device__ __align__(256) uint64_t scratch[kStaticScratchWords];
constexpr int kStaticMaxDevices = 64;
static uint64_t* g_static_scratch[kStaticMaxDevices] = {};

int topk_static_setup(int device)
{
    if (device < 0 || device >= kStaticMaxDevices) return set_error(DSX_EINVAL, "dsx_init: device %d is beyond the %d this library keeps scratch for", device, kStaticMaxDevices);
    if (g_static_scratch[device]) return DSX_OK;
    void* p = nullptr;
    DSX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return set_error(DSX_EHIP, "dsx_init: the fixed top-K scratch has no device address");
    g_static_scratch[device] = static_cast<uint64_t*>(p);
    return DSX_OK;
}

static int check_topk(const char* fn, const float* in, const float* keys, const void* values, uint32_t width, uint32_t k)
{
    DSX_CHECK_ARG(in && keys && values, "%s: null device pointer", fn);
    DSX_CHECK_ARG(k >= 1 && k <= 256, "%s: k = %u is outside 1..256", fn, k);
    DSX_CHECK_ARG(width >= 1, "%s: width is 0", fn);
    return DSX_OK;
}

}  // namespace dsx

using namespace dsx;

extern "C" {

int dsx_topk(const float* in, float* keys, uint32_t* values, uint32_t batch, uint32_t width, uint32_t k)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk", in, keys, values, width, k);
    if (rc) return rc;
    if (batch == 0) return DSX_OK;
    return topk_run(in, width, width, batch, k, keys, values, 0, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0, 0, 0);
}

int dsx_knn_topk(const float* in, float* keys, uint32_t* values, uint32_t batch, uint32_t width, uint32_t width_padding, uint32_t k)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_knn_topk", in, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(width_padding < width, "dsx_knn_topk: padding %u leaves no column of %u", width_padding, width);
    if (batch == 0) return DSX_OK;
    return topk_run(in, width, width - width_padding, batch, k, keys, values, 0, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr,
                    0, 0, 0);
}

int dsx_topk_filtered(const float* in, float* keys, uint32_t* values, uint32_t batch, uint32_t width, uint32_t k, uint32_t position,
                      const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end, const uint32_t* filter_index,
                      const float* filter_mul)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk_filtered", in, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(filter_start && filter_end && filter_index, "dsx_topk_filtered: null filter arrays (use dsx_topk for an unfiltered call)");
    if (batch == 0) return DSX_OK;
    return topk_run(in, width, width, batch, k, keys, values, position, index, filter_start, filter_end, filter_index, filter_mul, 0,
                    nullptr, 0, 0, 0);
}

int dsx_topk_filtered_static(const float* in, float* keys, uint32_t* values, uint32_t batch, uint32_t width, uint32_t k, uint32_t position,
                             const uint32_t* index, const uint64_t* filter_start, const uint64_t* filter_end,
                             const uint32_t* filter_index, const float* filter_mul)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk_filtered_static", in, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(!filter_index || (filter_start && filter_end), "dsx_topk_filtered_static: filter_index without filter_start / filter_end");
    uint64_t* lists = g_static_scratch[ctx().device];
    if (!lists) return set_error(DSX_ENOTINIT, "dsx_topk_filtered_static: no scratch address for device %d", ctx().device);
    if (batch == 0) return DSX_OK;
    // Every (row, segment) workgroup writes all k words of its list before the merge reads them: nothing in the scratch has
    // to start at zero, whatever the previous call left there.
    return topk_run(in, width, width, batch, k, keys, values, position, index, filter_start, filter_end, filter_index, filter_mul, 0,
                    nullptr, 0, 0, 0, nullptr, lists, kStaticScratchWords);
}

int dsx_topk_guided(const float* in, float* keys, uint32_t* values, uint32_t batch, uint32_t width, uint32_t k, const float* seg_max,
                    uint32_t seg_width, uint32_t position, const uint32_t* index, const uint64_t* filter_start,
                    const uint64_t* filter_end, const uint32_t* filter_index, const float* filter_mul)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk_guided", in, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(!filter_index || (filter_start && filter_end), "dsx_topk_guided: filter_index without filter_start / filter_end");
    if (batch == 0) return DSX_OK;
    return topk_guided_run(in, width, batch, k, keys, values, seg_max, seg_width, position, index, filter_start, filter_end,
                           filter_index, filter_mul);
}

int dsx_topk_kv_f32(const float* in_keys, const float* in_values, float* keys, float* values, uint32_t batch, uint32_t width, uint32_t k)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk_kv_f32", in_keys, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(in_values, "dsx_topk_kv_f32: null input values");
    if (batch == 0) return DSX_OK;
    rc = topk_run(in_keys, width, width, batch, k, keys, reinterpret_cast<uint32_t*>(values), 0, nullptr, nullptr, nullptr, nullptr,
                  nullptr, 0, nullptr, 0, 0, 0);
    if (rc) return rc;
    const uint64_t n = (uint64_t)batch * k;
    hipLaunchKernelGGL(topk_gather_kernel<float>, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, ctx().stream, in_values, values, batch,
                       width, k);
    DSX_LAUNCH_CHECK("topk_gather_kernel");
    return DSX_OK;
}

int dsx_topk_kv_u32(const float* in_keys, const uint32_t* in_values, float* keys, uint32_t* values, uint32_t batch, uint32_t width,
                    uint32_t k)
{
    DSX_REQUIRE_INIT();
    int rc = check_topk("dsx_topk_kv_u32", in_keys, keys, values, width, k);
    if (rc) return rc;
    DSX_CHECK_ARG(in_values, "dsx_topk_kv_u32: null input values");
    if (batch == 0) return DSX_OK;
    rc = topk_run(in_keys, width, width, batch, k, keys, values, 0, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0, 0, 0);
    if (rc) return rc;
    const uint64_t n = (uint64_t)batch * k;
    hipLaunchKernelGGL(topk_gather_kernel<uint32_t>, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, ctx().stream, in_values, values,
                       batch, width, k);
    DSX_LAUNCH_CHECK("topk_gather_kernel");
    return DSX_OK;
}

}  // extern "C"
