// dsx_f16.hip — f16 products of a few hundred to a few thousand rows ("queries") with a long table of items, on the matrix cores.
//
// Operands are row-major halves, a row's components contiguous: queries [rows rounded up to 256][ld], items [items rounded up to
// 256][ld], ld a multiple of 64, zero filled.  Products are exact in fp32, sums are fp32, added in ascending k: the same bits as
// knn_f16_kernel's.  Uses (MODE):
//   kF16Scores   sums compared with the queries' bounds, survivors to lists (exact nearest neighbours, fp16 storage and screening)
//   kF16Layer    sums that start from the items' biases, raised by the error they can have (dsx_screen.hip), against the bounds
//   kF16Store    sums that start from the biases stored as halves, rounded up, and the largest of every 32 of them
//   kI8Scores    operands are bytes (rows of 2 ld of them, a unit per query and per 32 items), sums are whole numbers; of every 32 items a word is
//                stored (i8_word): the largest sum, whose it is, and the second largest.  Nothing is compared and nothing listed.
//   kI8Layer     the same with the items' starts added
//
// A wavefront owns 128 items x 64 queries: four row operands and two column operands per 16 components feed eight matrix
// instructions, 48 LDS cycles for 64 cycles of each SIMD's matrix core (a 64 x 64 tile needs as many LDS cycles as there are).
// WI x WQ wavefronts make a workgroup; with 2 x 4 it has 256 x 256 tiles, one workgroup per compute unit.  Operands go from memory
// straight to LDS (no registers, no LDS store instructions), 32 components a stage, STAGES stages in a ring: while stage s is
// multiplied, s + 1 is there (its first operands are read in s's last step, so that no barrier leaves the matrix cores idle) and the
// ones behind it are on their way; what is asked for next crosses the border from one tile to the next.  What does not run on across it in the
// forms for layers and stored sums: memory answers in order and a wait for any other load is a wait for the stages before it, so ask's loads (of which
// it makes the sums' starts on the spot) and the storing form's scales empty the ring; its compiled loop has seven or eight waits for everything, a
// large part of the time where a tile is four stages (128 components).  A stage's rows are 64 bytes; the 16-byte piece c of
// row r lies at place c ^ (r / 2 % 4) of its row (the lanes ask memory for their pieces in that order).  LDS is not what bounds the kernel:
// with r / 4 % 4 the counters' bank conflicts go from 45 % of its cycles to 1 %, and the times stay (4,411 us against 4,350 for 4,096 x
// 512 x 1,000,000 with its candidates, 796 against 805 for 6,000 x 1,024 x 27,278; two runs of one side differ by as much).
// A workgroup keeps its queries and sweeps a chunk of the item tiles.  The items are the row operand: a lane's sixteen results of a block
// are sixteen items of ONE query, so a block without survivors costs ten three-way maxima and one compare.  A lane with survivors puts
// its sixteen results in the wavefront's queue in LDS; when that is full, all lanes go through it, four results of two entries each, and
// survivors go to lists owned by one (query, chunk, wavefront row) with the fill counts in LDS.  (Looked through on the spot, result by
// result, a block with two survivors took some 700 cycles of a wavefront: 245,760 items x 128 x 4,096 queries with 500 survivors each
// 541 us, 430 so, 275 without survivors.)
// 4,096 queries x 1,000,000 items: 1.09 PFLOP/s with 512 components (a large product of the matrix library reaches 1.16 on this part),
// 0.90 with 128, where the compares are a third of the issued instructions.  (128 x 128 tiles through registers: 0.72 with 576.)
#include <algorithm>
#include <type_traits>
#include "dsx_screen.h"

namespace dsx {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

constexpr int kF16Xcds = 8;
constexpr uint32_t kF16Step = 32;   // components a stage

struct F16SweepArgs {
    const _Float16* Q;
    const _Float16* I;      // of the range's first item
    uint32_t ld;            // halves per row
    uint32_t batch, n;      // valid queries, valid items of this range
    uint32_t tiles_q, tiles_i, chunks, tiles_per_chunk;
    uint32_t group;         // query tiles that sit on one XCD together
    uint64_t* seg;          // [query][chunks * WI][seg_cap]
    uint32_t* seg_count;    // [query][kF16ListStride]
    uint32_t seg_cap;
    CandArgs cand;          // bounds, column offset, and the shared lists a full list spills into
    const float* norm;      // layers: norms of the range's items
    const float* bias;      // layers: [n], or NULL
    const float* e1;        // layers: [batch] error of a query's sum per unit of an item's norm
    float bias_raise;       // layers: what a bias is raised by, per unit of it
    _Float16* Z;            // kF16Store: [batch][ldz]
    uint64_t ldz;
    _Float16* M;            // kF16Store: [batch][ldz / 32] the largest of every 32 of them
    const float* scale;     // kF16Store: [batch] what a query's sums are multiplied by (a power of two); kI8*: a query's unit
    const float* unit;      // kI8*: units of the items' components, one for every 32 items
    uint32_t* words;        // kI8*: [batch][ldw] a word for every 32 items (i8_word)
    uint64_t ldw;
};

constexpr uint32_t kF16Queue = 32;   // entries of a wavefront's queue

// Whether a mode's sums start from something, and whether they go to lists.
constexpr bool f16_starts(int mode) { return mode != kF16Scores && mode != kI8Scores; }
constexpr bool f16_lists(int mode) { return mode == kF16Scores || mode == kF16Layer; }

template <int WI, int WQ, int STAGES> constexpr uint32_t f16_sweep_lds(int mode)
{
    return STAGES * (128 * WI + 64 * WQ) * 64 + (f16_starts(mode) ? 4 * (128 + 4) * WI * 4 : 0) +
           (f16_lists(mode) ? WI * WQ * (kF16Queue * 80 + 64 * 4) : 0);
}

template <int WI, int WQ, int STAGES, int MODE>
__global__ __launch_bounds__(64 * WI * WQ) __attribute__((amdgpu_waves_per_eu(WI * WQ == 8 ? 2 : 1, 2))) void f16_sweep_kernel(F16SweepArgs a)
{
    constexpr uint32_t WAVES = WI * WQ, BI = 128 * WI, BQ = 64 * WQ, STAGE = (BI + BQ) * 64;
    constexpr uint32_t PI = BI / 16 / WAVES, PQ = BQ / 16 / WAVES;   // 1 KiB pieces (16 rows) of a stage per wavefront
    static_assert(PI * WAVES * 16 == BI && PQ * WAVES * 16 == BQ, "whole pieces");
    extern __shared__ __attribute__((aligned(16))) unsigned char f16_lds[];
    // layers, four tiles each: what the items' sums start from, and the largest norm of 32 items
    float* sStart = reinterpret_cast<float*>(f16_lds + STAGES * STAGE);
    float* sMost = sStart + 4 * BI;
    constexpr bool EIGHT = MODE == kI8Scores || MODE == kI8Layer;
    // the wavefronts' queues (sixteen results; then the bound, e1, the largest norm, the item and the query) and their lists' fill counts
    unsigned char* after = f16_lds + STAGES * STAGE + (f16_starts(MODE) ? 4 * (128 + 4) * WI * 4 : 0);
    float (*sResult)[16] = reinterpret_cast<float (*)[16]>(after) + (threadIdx.x >> 6) * kF16Queue;
    uint4* sEntry = reinterpret_cast<uint4*>(after + WAVES * kF16Queue * 64) + (threadIdx.x >> 6) * kF16Queue;
    uint32_t* sFill = reinterpret_cast<uint32_t*>(after + WAVES * kF16Queue * 80) + (threadIdx.x & ~63u);

    const uint32_t total = a.tiles_q * a.chunks;
    uint32_t wg = blockIdx.x;
    {
        const uint32_t per_xcd = (total + kF16Xcds - 1) / kF16Xcds;
        const uint32_t xcd = wg % kF16Xcds, local = wg / kF16Xcds;
        wg = xcd * per_xcd + local;
        if (local >= per_xcd || wg >= total) return;
    }
    // groups of query tiles one after the other, all chunks of a group together
    const uint32_t block = wg / (a.group * a.chunks), in_block = wg - block * a.group * a.chunks;
    const uint32_t members = min(a.group, a.tiles_q - block * a.group);
    const uint32_t tq = block * a.group + in_block % members, chunk = in_block / members;
    const uint32_t row0 = tq * BQ;
    const uint32_t t0 = chunk * a.tiles_per_chunk, t1 = min(t0 + a.tiles_per_chunk, a.tiles_i);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wi = wave / WQ, wq = wave % WQ, l32 = lane & 31, lhi = lane >> 5;

    uint32_t q[2];
    const uint32_t list = chunk * WI + wi;
    float bound[2];
#pragma unroll
    for (int j = 0; j < 2; j++) q[j] = row0 + wq * 64 + j * 32 + l32;
    if constexpr (f16_lists(MODE)) {
        if (t0 >= t1) {   // more chunks than tiles: empty lists (the same for the whole workgroup)
            const uint32_t r = row0 + wq * 64 + lane;
            if (r < a.batch) a.seg_count[(uint64_t)r * kF16ListStride + list] = 0;
            return;
        }
        sFill[lane] = 0;   // (the wavefront's own)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            bound[j] = __uint_as_float(0x7fc00000u);   // queries beyond the batch: NaN, which nothing reaches
            if (q[j] < a.batch) {
                const uint32_t key = a.cand.row_bound[q[j]];
                bound[j] = key ? key_score(key) : -__builtin_inff();   // key 0: no bound yet, every number passes
            }
        }
    } else if (t0 >= t1) return;

    // What an item's sum starts from (its bias, raised by the roundings of a sum that holds it; an item of infinite norm always passes)
    // and its norm, asked for a tile ahead.
    float e1[2] = {0.0f, 0.0f};
    constexpr uint32_t OWN = (BI + 64 * WAVES - 1) / (64 * WAVES);   // items of a tile per lane
    float start_next[OWN], norm_next[OWN];
    auto ask = [&](uint32_t t) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t o = 0; o < OWN; o++) {
            const uint32_t i = o * 64 * WAVES + tid, c = t * BI + i;
            start_next[o] = -__builtin_inff();
            norm_next[o] = 0.0f;
            if constexpr (EIGHT) start_next[o] = -3e37f;
            if (i >= BI || t >= t1 || c >= a.n) continue;
            const float b = a.bias ? a.bias[c] : 0.0f, norm = a.norm[c];
            if constexpr (EIGHT) start_next[o] = i8_start(b, norm, a.bias_raise);
            else
                start_next[o] = (norm == __builtin_inff() && b == b) ? norm : b == -__builtin_inff() ? b : b + fabsf(b) * a.bias_raise;
            norm_next[o] = (norm == __builtin_inff()) ? 0.0f : norm;
        }
    };
    auto put = [&](uint32_t t) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t o = 0; o < OWN; o++) {
            const uint32_t i = o * 64 * WAVES + tid;
            if (i >= BI) continue;   // (whole wavefronts)
            sStart[(t & 3) * BI + i] = start_next[o];
            if constexpr (MODE == kF16Layer) {
                float m = norm_next[o];
#pragma unroll
                for (int d = 1; d < 32; d *= 2) m = fmaxf(m, __shfl_xor(m, d));
                if (l32 == 0) sMost[(t & 3) * (BI / 32) + i / 32] = m;
            }
        }
    };
    if constexpr (f16_starts(MODE)) {
        if constexpr (MODE == kF16Layer) {
#pragma unroll
            for (int j = 0; j < 2; j++)
                if (q[j] < a.batch) e1[j] = a.e1[q[j]];
        }
        ask(t0);
        put(t0);
        ask(t0 + 1);
        put(t0 + 1);
        ask(t0 + 2);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (before the barrier below)
    }

    // Operands on their way: the stage of cursor (dt, dk) goes into ring place dp.  The cursor stops at the last stage (what is asked for
    // beyond it is that stage again, and never used).
    const uint32_t nk = a.ld / kF16Step;
    const uint32_t voff = ((lane >> 2) * a.ld + (((lane & 3) ^ ((lane >> 3) & 3)) * 8)) * 2;   // this lane's bytes into a piece
    const uint64_t piece_bytes = (uint64_t)a.ld * 32;   // 16 rows
    const char* gI = reinterpret_cast<const char*>(a.I) + ((uint64_t)t0 * BI / 16 + wave * PI) * piece_bytes + voff;
    const char* gQ = reinterpret_cast<const char*>(a.Q) + ((uint64_t)row0 / 16 + wave * PQ) * piece_bytes + voff;
    uint32_t dt = t0, dk = 0, dp = 0;
    auto request = [&]() __attribute__((always_inline)) {
        typedef const __attribute__((address_space(1))) void* Src;
        typedef __attribute__((address_space(3))) void* Dst;
        unsigned char* place = f16_lds + dp * STAGE;
#pragma unroll
        for (uint32_t p = 0; p < PI; p++)
            __builtin_amdgcn_global_load_lds((Src)(gI + p * piece_bytes), (Dst)(place + (wave * PI + p) * 1024), 16, 0, 0);
#pragma unroll
        for (uint32_t p = 0; p < PQ; p++)
            __builtin_amdgcn_global_load_lds((Src)(gQ + p * piece_bytes), (Dst)(place + BI * 64 + (wave * PQ + p) * 1024), 16, 0, 0);
        dp = (dp + 1 == STAGES) ? 0 : dp + 1;
        if (dk + 1 < nk) {
            dk++;
            gI += kF16Step * 2;
            gQ += kF16Step * 2;
        } else if (dt + 1 < t1) {
            dt++;
            dk = 0;
            gI += (uint64_t)BI * a.ld * 2 - (nk - 1) * kF16Step * 2;
            gQ -= (nk - 1) * kF16Step * 2;
        }
    };
    constexpr int PER = PI + PQ;
    // waits until at most `stages` of the stages asked for last are outstanding, then for the other wavefronts
#define F16_WAIT(STAGES_LEFT)                                                                    \
    do {                                                                                         \
        if constexpr ((STAGES_LEFT) * PER == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); \
        else if constexpr ((STAGES_LEFT) * PER == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  \
        else if constexpr ((STAGES_LEFT) * PER == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  \
        else if constexpr ((STAGES_LEFT) * PER == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  \
        else if constexpr ((STAGES_LEFT) * PER == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); \
        else if constexpr ((STAGES_LEFT) * PER == 30) asm volatile("s_waitcnt vmcnt(30)" ::: "memory"); \
        else if constexpr ((STAGES_LEFT) * PER == 40) asm volatile("s_waitcnt vmcnt(40)" ::: "memory"); \
        else static_assert((STAGES_LEFT) * PER == 0, "a count for this many requests");          \
        __builtin_amdgcn_s_barrier();                                                            \
        asm volatile("" ::: "memory");                                                           \
    } while (0)

    const uint32_t swz = (lhi ^ ((l32 >> 1) & 3)) * 16;
    const uint32_t offI = (wi * 128 + l32) * 64 + swz, offQ = BI * 64 + (wq * 64 + l32) * 64 + swz;
    half8 fi[2][4], fq[2][2];
    auto fetch = [&](int set, uint32_t place, int ks) __attribute__((always_inline)) {
        const unsigned char* pi = f16_lds + place * STAGE + (ks ? (offI ^ 32u) : offI);
        const unsigned char* pq = f16_lds + place * STAGE + (ks ? (offQ ^ 32u) : offQ);
#pragma unroll
        for (int i = 0; i < 4; i++) fi[set][i] = *reinterpret_cast<const half8*>(pi + i * 2048);
#pragma unroll
        for (int j = 0; j < 2; j++) fq[set][j] = *reinterpret_cast<const half8*>(pq + j * 2048);
    };
    typedef int32_t intx16 __attribute__((ext_vector_type(16)));
    typedef int32_t intx4 __attribute__((ext_vector_type(4)));
    typedef std::conditional_t<EIGHT, intx16, floatx16> Acc;
    Acc acc[4][2];
    // (a multiplication first, whose wait is then for the reads of the step before and not for the first of these; then the next
    // step's six reads among the others)
    auto order = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 6; r++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    };
    auto multiply = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (EIGHT)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(intx4, fi[set][i]), __builtin_bit_cast(intx4, fq[set][j]), acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fi[set][i], fq[set][j], acc[i][j], 0, 0, 0);
            }
    };

    float mine[2] = {0.0f, 0.0f};   // the queries' units
    uint32_t word[2][2];
    if constexpr (EIGHT) {
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (q[j] < a.batch) mine[j] = a.scale[q[j]];
    }

    uint32_t queued = 0;   // wave-uniform
    auto settle = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // (both halves of the queue at once: their reads, and their counts, are waited for together)
        constexpr int H = kF16Queue / 16;
        float x[H][4];
        uint32_t ql[H], col0[H], at[H], passes[H];
#pragma unroll
        for (int h = 0; h < H; h++) {
            const uint32_t p = h * 16 + lane / 4;
            const float4 v = *reinterpret_cast<const float4*>(&sResult[p][lane % 4 * 4]);
            const uint4 w = sEntry[p];
            x[h][0] = v.x; x[h][1] = v.y; x[h][2] = v.z; x[h][3] = v.w;
            ql[h] = MODE == kF16Layer ? w.w % 64 : w.y % 64;
            col0[h] = (MODE == kF16Layer ? w.w / 64 * 4 : w.w) + lane % 4 * 8;
            passes[h] = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float raised = MODE == kF16Layer ? fmaf(__uint_as_float(w.y), __uint_as_float(w.z), x[h][e]) : x[h][e];
                if (raised >= __uint_as_float(w.x) && col0[h] + e < a.n) passes[h] |= 1u << e;   // (items beyond the range are zero padding)
            }
            if (p >= queued) passes[h] = 0;
        }
#pragma unroll
        for (int h = 0; h < H; h++)
            if (passes[h] != 0) at[h] = atomicAdd(&sFill[ql[h]], (uint32_t)__popc(passes[h])) & 0x7fffffffu;
#pragma unroll
        for (int h = 0; h < H; h++) {
            if (passes[h] == 0) continue;
            const uint32_t r = row0 + wq * 64 + ql[h];
            uint64_t* mine = a.seg + ((uint64_t)r * (a.chunks * WI) + list) * a.seg_cap;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (!((passes[h] >> e) & 1)) continue;
                const uint64_t word = ((uint64_t)score_key(x[h][e]) << 32) | (uint32_t)~(a.cand.col_offset + col0[h] + e);
                if (at[h] < a.seg_cap) mine[at[h]] = word;
                else {   // this list is full: the query's shared list
                    const uint32_t s = atomicAdd(&a.cand.cand_count[r], 1u);
                    if (s < a.cand.cand_cap) a.cand.cand[(uint64_t)r * a.cand.cand_cap + s] = word;
                    else {
                        *a.cand.overflow = 1u;
                        atomicOr(&sFill[ql[h]], 0x80000000u);   // (the row is done otherwise: nothing more of it is wanted)
                    }
                }
                at[h]++;
            }
        }
        queued = 0;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (sFill[j * 32 + l32] & 0x80000000u) bound[j] = __uint_as_float(0x7fc00000u);
    };
    // most: largest norm of the block's items, which stands for theirs here: what passes is listed as it is, and raised by its own
    // norm where the lists are read.  (No item's raised sum is above its sum raised by most: the multiply-add rounds monotonically.)
    auto compare = [&](const floatx16& s, int j, uint32_t item0, float most) __attribute__((always_inline)) {
        float top = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
        for (int v = 3; v < 15; v += 2) top = fmaxf(fmaxf(top, s[v]), s[v + 1]);
        top = fmaxf(top, s[15]);
        if constexpr (MODE == kF16Layer) top = fmaf(e1[j], most, top);
        uint64_t hot = __builtin_amdgcn_ballot_w64(top >= bound[j]);
        while (hot != 0) {
            if (queued == kF16Queue) settle();
            // the lowest lanes, as many as there is room for
            const uint32_t place = queued + __builtin_amdgcn_mbcnt_hi((uint32_t)(hot >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hot, 0u));
            const bool mine = ((hot >> lane) & 1) != 0 && place < kF16Queue;
            if (mine) {
#pragma unroll
                for (int g = 0; g < 4; g++) *reinterpret_cast<float4*>(&sResult[place][4 * g]) = make_float4(s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]);
                if constexpr (MODE == kF16Layer)   // (fewer than 2^28 items: their table would not fit otherwise; item0 is a multiple of 4)
                    sEntry[place] = make_uint4(__float_as_uint(bound[j]), __float_as_uint(e1[j]), __float_as_uint(most), item0 * 16 + j * 32 + l32);
                else sEntry[place] = make_uint4(__float_as_uint(bound[j]), j * 32 + l32, 0, item0);
            }
            const uint64_t taken = __builtin_amdgcn_ballot_w64(mine);
            queued += (uint32_t)__builtin_popcountll(taken);
            hot &= ~taken;
        }
    };

#pragma unroll
    for (int s = 0; s < STAGES - 1; s++) request();
    F16_WAIT(STAGES - 2);   // stage 0 is there
    fetch(0, 0, 0);
    uint32_t cp = 0;   // ring place of the stage that is multiplied
    auto stage = [&]() __attribute__((always_inline)) {
        F16_WAIT(STAGES - 3);   // the next stage is there, and every wavefront is done with the one before this
        request();
        const uint32_t np = (cp + 1 == STAGES) ? 0 : cp + 1;
        fetch(1, cp, 1);
        multiply(0);
        order();
        fetch(0, np, 0);
        multiply(1);
        order();
        cp = np;
    };
    for (uint32_t t = t0; t < t1; t++) {
        if constexpr (MODE == kF16Scores || EIGHT) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        if constexpr (EIGHT) acc[i][j][v] = kI8Start;
                        else acc[i][j][v] = 0.0f;
                    }
        } else {
            const float* from = sStart + (t & 3) * BI + wi * 128 + 4 * lhi;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float4 s = *reinterpret_cast<const float4*>(from + i * 32 + 8 * g);
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        acc[i][j][4 * g] = s.x; acc[i][j][4 * g + 1] = s.y; acc[i][j][4 * g + 2] = s.z; acc[i][j][4 * g + 3] = s.w;
                    }
                }
        }
        __builtin_amdgcn_s_setprio(1);
        stage();
        stage();   // (ld is a multiple of 64: two stages at least)
        if constexpr (f16_starts(MODE)) {
            // Two tiles ahead, into the places of the tile before last: a whole tile's barriers and waits lie before they are read.  (After the
            // tile's second stage: 4 x 128 x 1,000,000 73.5 us; after its first 77.)
            put(t + 2);
            ask(t + 3);
        }
        for (uint32_t kt = 2; kt < nk; kt++) stage();
        __builtin_amdgcn_s_setprio(0);
        if constexpr (EIGHT) {
            // The largest two of a block's 32 sums per query: a lane's sixteen first, each with its place in its lowest bits, then the two lanes of the
            // query, two blocks at a time.  (med3 where a maximum would do: fmaxf costs an instruction more, which quiets a NaN; there is none.)
            const __attribute__((address_space(4))) float* units = (const __attribute__((address_space(4))) float*)(a.unit + (uint64_t)t * (BI / 32) + wi * 4);
            float unit[4];
#pragma unroll
            for (int i = 0; i < 4; i++) unit[i] = units[i];
#pragma unroll
            for (int half = 0; half < 2; half++) {   // blocks half and half + 2
                float most[2][2], second[2][2];
#pragma unroll
                for (int x = 0; x < 2; x++) {
                    const int i = half + 2 * x;
                    float start[16];
                    if constexpr (MODE == kI8Layer) {
                        const float* from = sStart + (t & 3) * BI + wi * 128 + 4 * lhi + i * 32;
#pragma unroll
                        for (int g = 0; g < 4; g++) {
                            const float4 s = *reinterpret_cast<const float4*>(from + 8 * g);
                            start[4 * g] = s.x; start[4 * g + 1] = s.y; start[4 * g + 2] = s.z; start[4 * g + 3] = s.w;
                        }
                    }
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const float p = mine[j] * unit[i];
                        float h[2] = {-kI8Most, -kI8Most}, l[2] = {-kI8Most, -kI8Most};
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            int32_t bits = acc[i][j][v];
                            if constexpr (MODE == kI8Layer) bits = __float_as_int(fmaf(__int_as_float(bits), p, start[v]));
                            const float s = __int_as_float((bits & ~31) | (v / 4 * 8 + v % 4));
                            l[v % 2] = __builtin_amdgcn_fmed3f(h[v % 2], l[v % 2], s);
                            h[v % 2] = __builtin_amdgcn_fmed3f(h[v % 2], s, kI8Most);
                        }
                        most[x][j] = __builtin_amdgcn_fmed3f(h[0], h[1], kI8Most);
                        second[x][j] = fmaxf(fmaxf(__builtin_amdgcn_fmed3f(h[0], h[1], -kI8Most), l[0]), l[1]);
                    }
                }
                const float lower = unit[half], upper = unit[half + 2], own = lhi ? upper : lower;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    // (after the exchange the lower half's lanes hold both halves' of block `half`, the others of block half + 2)
                    const auto m = __builtin_amdgcn_permlane32_swap(__float_as_uint(most[0][j]), __float_as_uint(most[1][j]), false, false);
                    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(second[0][j]), __float_as_uint(second[1][j]), false, false);
                    word[half][j] = i8_block_word<MODE == kI8Layer>(m[0], m[1], s[0], s[1], mine[j] * own);
                }
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
                const u32x2v w = {word[0][j], word[1][j]};
                if (q[j] < a.batch) *reinterpret_cast<u32x2v*>(a.words + (uint64_t)q[j] * a.ldw + t * (BI / 32) + wi * 4 + 2 * lhi) = w;
            }
        } else if constexpr (MODE != kF16Store) {
            const uint32_t item0 = t * BI + wi * 128 + 4 * lhi;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float most = MODE == kF16Layer ? sMost[(t & 3) * (BI / 32) + wi * 4 + i] : 0.0f;
#pragma unroll
                for (int j = 0; j < 2; j++) compare(acc[i][j], j, item0 + i * 32, most);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (q[j] >= a.batch) continue;
                const float scale = a.scale[q[j]];
                // (both halves of a lane pair take the same branch: they hold the same query)
                _Float16* dst = a.Z + (uint64_t)q[j] * a.ldz + (uint64_t)t * BI + wi * 128 + lhi * 16;
                typedef _Float16 half2v __attribute__((ext_vector_type(2)));
                // raised by half a unit in the last place and a subnormal's, and no lower than the lowest half: what rounds to nearest then
                // lies above
                auto up = [&](float v) __attribute__((always_inline)) -> _Float16 {
                    const float x = v * scale;
                    return (_Float16)fmaxf(fmaf(fabsf(x), 4.932e-4f, x) + 6.0e-8f, -65504.0f);
                };
                half2v most[2];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const floatx16& v = acc[i][j];
                    float top = fmaxf(fmaxf(v[0], v[1]), v[2]);
#pragma unroll
                    for (int e = 3; e < 15; e += 2) top = fmaxf(fmaxf(top, v[e]), v[e + 1]);
                    top = fmaxf(top, v[15]);
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(top), __float_as_uint(top), false, false);
                    most[i / 2][i % 2] = up(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
                }
                if (lhi == 0) {
                    typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
                    u32x2v w = {__builtin_bit_cast(uint32_t, most[0]), __builtin_bit_cast(uint32_t, most[1])};
                    *reinterpret_cast<u32x2v*>(a.M + (uint64_t)q[j] * (a.ldz / 32) + t * (BI / 32) + wi * 4) = w;
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint32_t w[4][2];
#pragma unroll
                    for (int g = 0; g < 4; g++)
#pragma unroll
                        for (int p = 0; p < 2; p++) {
                            const half2v h = {up(acc[i][j][4 * g + 2 * p]), up(acc[i][j][4 * g + 2 * p + 1])};
                            w[g][p] = __builtin_bit_cast(uint32_t, h);
                        }
                    // a lane holds items 8 g + 4 lhi + 0..3: after the exchange the lower half's lanes hold items 0..15, the others 16..31
#pragma unroll
                    for (int g = 0; g < 2; g++) {
                        u32x4v out;
#pragma unroll
                        for (int p = 0; p < 2; p++) {
                            const auto r = __builtin_amdgcn_permlane32_swap(w[g][p], w[g + 2][p], false, false);
                            out[p] = r[0];
                            out[2 + p] = r[1];
                        }
                        *reinterpret_cast<u32x4v*>(dst + i * 32 + g * 8) = out;
                    }
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (what was asked for beyond the end must not arrive in another workgroup's LDS)
    if constexpr (f16_lists(MODE)) {
        settle();
        const uint32_t r = row0 + wq * 64 + lane;
        if (r < a.batch) a.seg_count[(uint64_t)r * kF16ListStride + list] = min(sFill[lane] & 0x7fffffffu, a.seg_cap);
    }
#undef F16_WAIT
}

template <int WI, int WQ, int STAGES, int MODE> static int launch_f16_sweep(F16SweepArgs& a)
{
    constexpr uint32_t lds = f16_sweep_lds<WI, WQ, STAGES>(MODE);
    static bool sized[64] = {};   // per device: the kernel's LDS limit is raised once
    const int dev = ctx().device;
    if (dev < 0 || dev >= 64 || !sized[dev]) {
        DSX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&f16_sweep_kernel<WI, WQ, STAGES, MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        if (dev >= 0 && dev < 64) sized[dev] = true;
    }
    const uint32_t total = a.tiles_q * a.chunks, grid = (total + kF16Xcds - 1) / kF16Xcds * kF16Xcds;
    hipLaunchKernelGGL((f16_sweep_kernel<WI, WQ, STAGES, MODE>), dim3(grid), dim3(64 * WI * WQ), lds, ctx().stream, a);
    DSX_LAUNCH_CHECK("f16_sweep_kernel");
    return DSX_OK;
}

static F16SweepArgs f16_args(const F16Job& j)
{
    F16SweepArgs a{};
    a.Q = (const _Float16*)j.Q; a.I = (const _Float16*)j.items;
    a.ld = j.ld; a.batch = j.batch; a.n = j.n;
    a.norm = j.norm; a.bias = j.bias; a.e1 = j.e1; a.bias_raise = j.bias_raise;
    a.cand = j.cand;
    a.Z = (_Float16*)j.Z; a.M = (_Float16*)j.M; a.ldz = j.ldz; a.scale = j.scale;
    a.unit = j.unit; a.words = j.words; a.ldw = j.ldw;
    a.tiles_q = (j.batch + 255) / 256;   // (one where tiles are lower)
    return a;
}

// Eight query tiles to an XCD: with 512 components their operands are half of its L2 (4, 8 and 16 are level within 2 %).
constexpr uint32_t kF16Group = 8;

int f16_sweep_run(const F16Job& j, bool layer, uint32_t* lists)
{
    F16SweepArgs a = f16_args(j);
    a.tiles_i = (j.n + 255) / 256;
    // (one workgroup per compute unit and no more than there are: two too many take as long again)
    a.chunks = std::min(std::min(kF16ListStride / 2, a.tiles_i), std::max(1u, (uint32_t)ctx().num_cus / a.tiles_q));
    a.tiles_per_chunk = (a.tiles_i + a.chunks - 1) / a.chunks;
    a.group = std::min(a.tiles_q, kF16Group);
    *lists = a.chunks * 2;
    a.seg = j.seg; a.seg_count = j.seg_count; a.seg_cap = j.seg_words / *lists;
    return layer ? launch_f16_sweep<2, 4, 4, kF16Layer>(a) : launch_f16_sweep<2, 4, 4, kF16Scores>(a);
}

template <int MODE> static int launch_f16_tiles(const F16Job& j)
{
    F16SweepArgs a = f16_args(j);
    // Few rows are bound by reading the items: as many of them in flight as LDS holds, and no matrix work for rows that are not there
    // (8 x 256 x 500,000: 56 us, 4.5 TB/s; 4 x 128 x 1,000,000: 73.5, as half as many stages lie between two tiles' stores; a copy
    // reaches 5.1 TB/s.  Seven stages in flight instead of six: 59 and 77).  128 items x 256 rows where 256 x 256 tiles leave half
    // the GPU without work (256 x 1,024 x 27,278: 28 us against 35).
    const int shape = j.batch <= 64 ? 0 : j.batch <= 128 ? 1 : a.tiles_q * ((j.n + 255) / 256) < (uint32_t)ctx().num_cus ? 2 : 3;
    const uint32_t items = shape == 2 ? 128 : 256;
    a.tiles_i = (j.n + items - 1) / items;
    a.chunks = std::min(a.tiles_i, std::max(1u, (uint32_t)ctx().num_cus / a.tiles_q));
    a.tiles_per_chunk = (a.tiles_i + a.chunks - 1) / a.chunks;
    a.chunks = (a.tiles_i + a.tiles_per_chunk - 1) / a.tiles_per_chunk;
    a.group = std::min(a.tiles_q, kF16Group);
    switch (shape) {
    case 0: return launch_f16_sweep<2, 1, 6, MODE>(a);
    case 1: return launch_f16_sweep<2, 2, 4, MODE>(a);
    case 2: return launch_f16_sweep<1, 4, 4, MODE>(a);
    default: return launch_f16_sweep<2, 4, 4, MODE>(a);
    }
}

int f16_store_run(const F16Job& j) { return launch_f16_tiles<kF16Store>(j); }

int i8_best_run(const F16Job& j, bool starts) { return starts ? launch_f16_tiles<kI8Layer>(j) : launch_f16_tiles<kI8Scores>(j); }

}  // namespace dsx
