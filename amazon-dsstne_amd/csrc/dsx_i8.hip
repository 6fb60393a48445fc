// dsx_i8.hip — products of bytes of a few hundred to a few thousand rows ("queries") with a long table of items of up to 512 components, on the matrix
// cores: of every 32 items a word per query (i8_word).  What it says is explained in dsx_screen.hip; the same words come from f16_sweep_kernel
// (dsx_f16.hip) for fewer rows and longer vectors.
//
// A wavefront keeps the operands of its 64 queries for all components in registers (8 KS of them), a workgroup of eight those of 512, and walks a chunk of
// the items: 16 KiB of whole rows a stage, from memory straight to LDS in a ring.  So the items are all that moves, once per workgroup, and one
// 16-byte LDS read feeds two matrix instructions: a stage takes half the LDS cycles that it takes matrix cycles.  (f16_sweep_kernel reads both operands from LDS,
// 0.75 of a cycle for each matrix cycle, and writes 0.25: 4,096 x 512 x 1,000,000 with starts 2,464 us, 1,907 here; 4,096 x 128 x 1,000,000 without 866, 753.)
// What bounds it: matrix and vector instructions of a SIMD hardly overlap (128 components, two wavefronts a SIMD or four: 0.50 million cycles of matrix cores busy
// and 1.09 of vector instructions, at four each, in a kernel of 1.52), and
// a block's words take 70 vector instructions for each 32 queries, whatever the number of components.
// The items are the row operand: a lane's sixteen results are sixteen items of one query.  While a block of 32 items is multiplied the sums of the one before
// it become words; the ring keeps a stage longer for that, for what its sums start from.
// Row r's 16-byte piece c lies at place c ^ (r % 8) of its row (the lanes ask memory for their pieces in that order), so that eight lanes, which read the
// same piece of eight rows, reach all banks.  (The counters show conflicts in 45 % of the LDS's cycles all the same, which are 0.25 of the kernel's.)  A lane's words are
// written 16 bytes at a time, rows apart, for which memory sees three times the bytes; 64 at a time, from registers, 753 us became 798.
#include <algorithm>
#include <atomic>
#include "dsx_screen.h"

namespace dsx {

typedef int32_t intx4 __attribute__((ext_vector_type(4)));
typedef int32_t intx16 __attribute__((ext_vector_type(16)));

struct I8WideArgs {
    const int8_t* Q;        // [queries rounded up to 256][LD]
    const int8_t* I;        // [items rounded up to 256][LD]
    const float* side;      // [items / 32][kI8Side]
    const float* unit;      // [batch]
    uint32_t batch;
    uint32_t tiles_q, chunks, quads, quads_per_chunk;   // a quad: 128 items
    uint32_t* words;        // [batch][ldw]
    uint64_t ldw;
};

constexpr uint32_t kI8Stage = 16384, kI8Place = kI8Stage + 768, kI8Stages = 8;

template <int KS, bool STARTS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void i8_wide_kernel(I8WideArgs a)
{
    constexpr uint32_t LD = KS * 32, P = LD / 16;                      // bytes and pieces of a row
    constexpr uint32_t NB = kI8Stage / (32 * LD), NQ = 4 / NB;         // blocks of a stage, stages of a quad
    constexpr uint32_t SIDES = (NB * kI8Side + 63) / 64;               // wavefronts' requests that hold a stage's side
    static_assert(NB >= 1 && NB <= 4 && SIDES * 256 <= kI8Place - kI8Stage, "a stage is one to four blocks");
    extern __shared__ __attribute__((aligned(16))) unsigned char i8_lds[];

    // Workgroups that walk the same chunk sit on the same XCD: a stage comes from memory once, and from that XCD's L2 for the others.
    const uint32_t total = a.tiles_q * a.chunks;
    uint32_t wg = blockIdx.x;
    {
        const uint32_t per_xcd = (total + 7) / 8;
        const uint32_t xcd = wg % 8, local = wg / 8;
        wg = xcd * per_xcd + local;
        if (local >= per_xcd || wg >= total) return;
    }
    const uint32_t tq = wg % a.tiles_q, chunk = wg / a.tiles_q;
    const uint32_t t0 = chunk * a.quads_per_chunk, t1 = min(t0 + a.quads_per_chunk, a.quads);
    if (t0 >= t1) return;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, lhi = lane >> 5;
    const uint32_t row0 = tq * 512 + wave * 64, stored = (a.batch + 255) / 256 * 256;

    intx4 bq[2][KS];
    float mine[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t q = row0 + j * 32 + l32;
        const int8_t* from = a.Q + (uint64_t)min(q, stored - 1) * LD + lhi * 16;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) bq[j][ks] = *reinterpret_cast<const intx4*>(from + ks * 32);
        mine[j] = q < a.batch ? a.unit[q] : 0.0f;
    }
    const float own = lhi ? mine[1] : mine[0];   // of query row0 + lane, whose words this lane has in the end

    // Items on their way: 1 KiB pieces, two a wavefront.
    const uint32_t in_piece = lane / P, row = wave * (1024 / LD) + in_piece;
    const char* gI = reinterpret_cast<const char*>(a.I) + (uint64_t)t0 * 128 * LD + wave * 1024 + in_piece * LD + ((lane % P) ^ (row & 7)) * 16;
    const char* gS = reinterpret_cast<const char*>(a.side) + (uint64_t)t0 * 4 * kI8Side * 4 + (wave % SIDES) * 256 + lane * 4;
    uint32_t asked = 0, dp = 0;
    const uint32_t stages = (t1 - t0) * NQ;
    auto request = [&]() __attribute__((always_inline)) {
        typedef const __attribute__((address_space(1))) void* Src;
        typedef __attribute__((address_space(3))) void* Dst;
        unsigned char* place = i8_lds + dp * kI8Place;
        __builtin_amdgcn_global_load_lds((Src)gI, (Dst)(place + wave * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((Src)(gI + 8192), (Dst)(place + 8192 + wave * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((Src)gS, (Dst)(place + kI8Stage + (wave % SIDES) * 256), 4, 0, 0);
        dp = (dp + 1 == kI8Stages) ? 0 : dp + 1;
        if (++asked < stages) {   // (what is asked for beyond the end is the last stage again, and never used)
            gI += kI8Stage;
            gS += NB * kI8Side * 4;
        }
    };

    // This lane's pieces of a block: four places, the others lie multiples of 128 bytes behind them.
    uint32_t at[4];
#pragma unroll
    for (int k = 0; k < 4; k++) at[k] = l32 * LD + (((2 * k + lhi) ^ (l32 & 7)) * 16);

    intx16 acc[2][2];
    intx16 start;
#pragma unroll
    for (int v = 0; v < 16; v++) start[v] = kI8Start;
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[s][j] = start;
    uint32_t word[4] = {0, 0, 0, 0};

    // The largest two of a block's 32 sums: a lane's sixteen first, each with its place in its lowest bits, then the two lanes of a query, both queries at once.
    // (med3 where a maximum would do: fmaxf costs an instruction more, which quiets a NaN; there is none.)
    auto settle = [&](const intx16 (&sums)[2], const float* side) __attribute__((always_inline)) -> uint32_t {
        const float unit = side[32];
        float most[2], second[2];
        float from[16];
        if constexpr (STARTS) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 s = *reinterpret_cast<const float4*>(side + 8 * g + 4 * lhi);
                from[4 * g] = s.x; from[4 * g + 1] = s.y; from[4 * g + 2] = s.z; from[4 * g + 3] = s.w;
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float p = mine[j] * unit;
            float h[2] = {-kI8Most, -kI8Most}, l[2] = {-kI8Most, -kI8Most};
#pragma unroll
            for (int v = 0; v < 16; v++) {
                int32_t bits = sums[j][v];
                if constexpr (STARTS) bits = __float_as_int(fmaf(__int_as_float(bits), p, from[v]));
                const float s = __int_as_float((bits & ~31) | (v / 4 * 8 + v % 4));
                l[v % 2] = __builtin_amdgcn_fmed3f(h[v % 2], l[v % 2], s);
                h[v % 2] = __builtin_amdgcn_fmed3f(h[v % 2], s, kI8Most);
            }
            most[j] = __builtin_amdgcn_fmed3f(h[0], h[1], kI8Most);
            second[j] = fmaxf(fmaxf(__builtin_amdgcn_fmed3f(h[0], h[1], -kI8Most), l[0]), l[1]);
        }
        // (after the exchange the lower lanes hold both halves of the first query, the upper ones of the second)
        const auto m = __builtin_amdgcn_permlane32_swap(__float_as_uint(most[0]), __float_as_uint(most[1]), false, false);
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(second[0]), __float_as_uint(second[1]), false, false);
        return i8_block_word<STARTS>(m[0], m[1], s[0], s[1], own * unit);
    };

#pragma unroll
    for (uint32_t s = 0; s + 2 < kI8Stages; s++) request();
    uint32_t cp = 0;   // ring place of the stage that is multiplied
    const float* side = reinterpret_cast<const float*>(i8_lds + kI8Stage);   // of the block before
    uint32_t* out = a.words + (uint64_t)(row0 + lane) * a.ldw + (uint64_t)t0 * 4;
    const bool real = row0 + lane < a.batch;
    for (uint32_t t = t0; t < t1; t++) {
#pragma unroll
        for (uint32_t b = 0; b < 4; b++) {
            const uint32_t in_stage = b % NB;
            if (in_stage == 0) {
                // The stage is there (three requests each for those behind it may not be), and every wavefront is done with the one before the last: also with
                // what it has asked LDS for, as the side of that one's last block, whose sums become words behind this barrier as the compiler has it.
                asm volatile("s_waitcnt vmcnt(15) lgkmcnt(0)" ::: "memory");
                static_assert(kI8Stages == 8, "3 (kI8Stages - 3) requests");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                request();
            }
            const unsigned char* place = i8_lds + cp * kI8Place;
            const unsigned char* rows = place + in_stage * 32 * LD;
            auto piece = [&](int ks) __attribute__((always_inline)) { return *reinterpret_cast<const intx4*>(rows + at[ks % 4] + ks / 4 * 128); };
            constexpr int AHEAD = 4;
            intx4 item[AHEAD];
#pragma unroll
            for (int ks = 0; ks < AHEAD; ks++) item[ks] = piece(ks);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const intx4 now = item[ks % AHEAD];
                if (ks + AHEAD < KS) item[ks % AHEAD] = piece(ks + AHEAD);
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[b % 2][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(now, bq[j][ks], ks == 0 ? start : acc[b % 2][j], 0, 0, 0);
            }
            word[(b + 3) % 4] = settle(acc[(b + 1) % 2], side);
            if (b == 0) {
                if (real && t != t0) *reinterpret_cast<uint4*>(out - 4) = make_uint4(word[0], word[1], word[2], word[3]);
                out += 4;
            }
            side = reinterpret_cast<const float*>(place + kI8Stage) + in_stage * kI8Side;
            if (in_stage == NB - 1) cp = (cp + 1 == kI8Stages) ? 0 : cp + 1;
        }
    }
    word[3] = settle(acc[1], side);
    if (real) *reinterpret_cast<uint4*>(out - 4) = make_uint4(word[0], word[1], word[2], word[3]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (what was asked for beyond the end must not arrive in another workgroup's LDS)
}

template <int KS, bool STARTS> static int launch_wide(const I8WideArgs& a)
{
    constexpr uint32_t lds = kI8Stages * kI8Place;
    static std::atomic<bool> sized[64] = {};   // per device: the kernel's LDS limit is raised once (threads that come here together ask for the same)
    const int dev = ctx().device;
    if (dev < 0 || dev >= 64 || !sized[dev].load(std::memory_order_acquire)) {
        DSX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&i8_wide_kernel<KS, STARTS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        if (dev >= 0 && dev < 64) sized[dev].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((i8_wide_kernel<KS, STARTS>), dim3((a.tiles_q * a.chunks + 7) / 8 * 8), dim3(512), lds, ctx().stream, a);
    DSX_LAUNCH_CHECK("i8_wide_kernel");
    return DSX_OK;
}

// Whether i8_wide_run takes vectors of ld8 bytes and so many rows.
bool i8_wide_takes(uint32_t ld8, uint32_t batch) { return batch > 256 && (ld8 == 128 || ld8 == 256 || ld8 == 512); }

int i8_wide_run(const F16Job& j, const float* side, bool starts)
{
    I8WideArgs a{};
    a.Q = (const int8_t*)j.Q; a.I = (const int8_t*)j.items; a.side = side; a.unit = j.scale; a.batch = j.batch; a.words = j.words; a.ldw = j.ldw;
    a.tiles_q = (j.batch + 511) / 512;
    a.quads = (j.n + 127) / 128;
    a.chunks = std::min(a.quads, std::max(1u, (uint32_t)ctx().num_cus / a.tiles_q));
    a.quads_per_chunk = (a.quads + a.chunks - 1) / a.chunks;
    a.chunks = (a.quads + a.quads_per_chunk - 1) / a.quads_per_chunk;
    switch (j.ld * 2) {
    case 128: return starts ? launch_wide<4, true>(a) : launch_wide<4, false>(a);
    case 256: return starts ? launch_wide<8, true>(a) : launch_wide<8, false>(a);
    default: return starts ? launch_wide<16, true>(a) : launch_wide<16, false>(a);
    }
}

}  // namespace dsx
