// dsx_fc_rows.hip — dense forward for few rows, or for few output tiles: the shapes whose time is reading W once, or a chain of
// k-steps on a nearly empty GPU, and not multiplying.
//
// The tiled kernel (dsx_fc.hip) gives a batch of 8 rows a tile of 64 or 128 and walks all of k in one workgroup.  Here a
// wavefront owns a tile of 32 MI rows x 32 NJ columns of Z and one share of k: W goes from memory straight into registers (every
// element is used by one wavefront only, so LDS would add a copy and a barrier per step), one chunk of eight k ahead of
// the multiplications, and no barrier is reached before the wavefront's share of k is done.  With KS > 1 the KS wavefronts of
// a workgroup share one tile, take the chunks of k in turn and add their tiles up through LDS; with KS = 1 a workgroup's four
// wavefronts own four neighbouring tiles and nothing is exchanged.
#include "dsx_device.h"
#include "dsx_internal.h"

namespace dsx {

template <int N>
__device__ __forceinline__ void activate_all(float (&o)[N], uint32_t act, float slope, float alpha, float lambda)
{
    switch (act) {
#define DSX_ACT_CASE(A)                                                                     \
    case A:                                                                                 \
        _Pragma("unroll") for (int j = 0; j < N; j++) o[j] = activate<A>(o[j], slope, alpha, lambda); \
        break;
        DSX_ACT_CASE(DSX_ACT_SIGMOID)
        DSX_ACT_CASE(DSX_ACT_TANH)
        DSX_ACT_CASE(DSX_ACT_RELU)
        DSX_ACT_CASE(DSX_ACT_LRELU)
        DSX_ACT_CASE(DSX_ACT_ELU)
        DSX_ACT_CASE(DSX_ACT_SELU)
#undef DSX_ACT_CASE
    default: break;
    }
}

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));

struct FcRowsArgs {
    const float* X;
    const float* W;
    const float* bias;
    float* Z;
    uint32_t ldx, ldw, ldz;
    uint32_t batch, k, n;
    int accumulate;
    uint32_t act;
    float slope, alpha, lambda;
    float* seg_max;    // optional, NJ = 4: [batch][nseg] maxima of the activated outputs over 64-column segments
    uint32_t nseg;
};

// WV: width in floats of the loads of W (n is a multiple of it; four-byte alignment is enough).  A lane's WV neighbouring columns belong to WV different MFMAs: MFMA j of a
// wavefront covers columns (j / WV) * 32 WV + WV * lane + j % WV, so a lane ends up with WV neighbouring outputs and stores them
// at once.  An output's products are added in ascending pairs of k (lane half h supplies k = 2t + h), as in the tiled kernel: a
// sum that is not split (KS = 1) has the tiled kernel's bits.
template <int NJ, int MI, int KS, int WV>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS, (MI * NJ > 4) ? 2 : 4) void fc_rows_kernel(FcRowsArgs a)
{
    static_assert(NJ % WV == 0 && 16 % KS == 0, "");
    constexpr int T = 4, CK = 2 * T;   // MFMA steps and k per chunk
    constexpr int NG = NJ / WV;
    __builtin_amdgcn_s_setprio(2);     // (ahead of another stream's GEMM on the same SIMD)
    const int lane = threadIdx.x & 63, l32 = lane & 31, lhi = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = (KS == 1) ? blockIdx.x * 4 + wave : blockIdx.x;
    const uint32_t col0 = tile * (32 * NJ), row0 = blockIdx.y * (32 * MI);
    if (col0 >= a.n) return;   // (KS = 1 only: the last workgroup's surplus wavefronts; there is no barrier in that form)

    uint32_t xoff[MI];   // byte offset of the lane's row of X; rows beyond the batch repeat the last one
#pragma unroll
    for (int i = 0; i < MI; i++) xoff[i] = min(row0 + i * 32 + l32, a.batch - 1) * a.ldx * 4u;
    uint32_t off[NG];   // byte offset of the lane's columns from the start of a pair of rows of W; columns beyond n repeat the last ones
#pragma unroll
    for (int g = 0; g < NG; g++) off[g] = (lhi * a.ldw + min(col0 + g * 32 * WV + l32 * WV, (a.n - 1) / WV * WV)) * 4u;

    struct Stage {
        float x[MI][CK];
        float w[T][NJ];
    };
    auto load = [&](Stage& s, uint32_t chunk) __attribute__((always_inline)) {
        const uint32_t k0 = chunk * CK;
#pragma unroll
        for (int t = 0; t < T; t++) {
            const char* base = reinterpret_cast<const char*>(a.W) + (uint64_t)(k0 + 2 * t) * a.ldw * 4;
#pragma unroll
            for (int g = 0; g < NG; g++) {
                if constexpr (WV == 4) {
                    const float4u v = *reinterpret_cast<const float4u*>(base + off[g]);
                    s.w[t][4 * g] = v.x; s.w[t][4 * g + 1] = v.y; s.w[t][4 * g + 2] = v.z; s.w[t][4 * g + 3] = v.w;
                } else if constexpr (WV == 2) {
                    const float2u v = *reinterpret_cast<const float2u*>(base + off[g]);
                    s.w[t][2 * g] = v.x; s.w[t][2 * g + 1] = v.y;
                } else {
                    s.w[t][g] = *reinterpret_cast<const float*>(base + off[g]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const char* base = reinterpret_cast<const char*>(a.X) + (uint64_t)k0 * 4;
#pragma unroll
            for (int e = 0; e < CK; e += 4) {
                const float4u v = *reinterpret_cast<const float4u*>(base + xoff[i] + 4 * e);
                s.x[i][e] = v.x; s.x[i][e + 1] = v.y; s.x[i][e + 2] = v.z; s.x[i][e + 3] = v.w;
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // (left to itself the scheduler sinks the loads to where they are waited for)
    };
    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    auto multiply = [&](const Stage& s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const float x = lhi ? s.x[i][2 * t + 1] : s.x[i][2 * t];
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, s.w[t][j], acc[i][j], 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    {
        const uint32_t chunks = a.k / CK;   // whole ones; this wavefront takes every KS-th
        const uint32_t first = (KS == 1) ? 0 : wave;
        if (first < chunks) {
            const uint32_t mine = (chunks - first + KS - 1) / KS, last = first + (mine - 1) * KS;
            Stage s0, s1;
            load(s0, first);
            uint32_t c = first, left = mine;
            // (the loads are unconditional, so that the stages stay in registers: the last chunk is requested again and not used)
            for (; left >= 2; left -= 2) {
                load(s1, c + KS);
                multiply(s0);
                load(s0, min(c + 2 * KS, last));
                multiply(s1);
                c += 2 * KS;
            }
            if (left) multiply(s0);
        }
        const uint32_t rest = a.k - chunks * CK;   // fewer than eight k beyond the last whole chunk: zeros behind them
        if (rest != 0 && wave == ((KS == 1) ? wave : chunks % KS)) {
            Stage s;
            const uint32_t k0 = chunks * CK;
#pragma unroll
            for (int t = 0; t < T; t++) {
                const bool ok = 2 * t + lhi < (int)rest;
                const char* base = reinterpret_cast<const char*>(a.W) + (uint64_t)(k0 + 2 * t) * a.ldw * 4;
#pragma unroll
                for (int g = 0; g < NG; g++)
#pragma unroll
                    for (int e = 0; e < WV; e++) s.w[t][g * WV + e] = ok ? reinterpret_cast<const float*>(base + off[g])[e] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int e = 0; e < CK; e++)
                    s.x[i][e] = (e < (int)rest) ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.X) + (uint64_t)(k0 + e) * 4 + xoff[i]) : 0.0f;
            multiply(s);
        }
    }

    float bias[NJ];   // by column, requested before the exchange below
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const uint32_t col = col0 + (j / WV) * 32 * WV + l32 * WV + j % WV;
        bias[j] = (a.bias && col < a.n) ? a.bias[col] : 0.0f;
    }
    // One row of the tile at a time and lane half: the lane's NJ sums, bias, activation, store, segment maxima.  (All of it is
    // done from LDS and in a loop over the rows: unrolled over the accumulator registers, with the activation chosen at run
    // time, it would be most of the kernel's code and its registers.)
    auto finish_row = [&](uint32_t row, float (&o)[NJ]) __attribute__((always_inline)) {
        const bool row_ok = row < a.batch;
        float* zrow = a.Z + (uint64_t)row * a.ldz;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint32_t col = col0 + (j / WV) * 32 * WV + l32 * WV + j % WV;
            o[j] += bias[j];
            if (a.accumulate && row_ok && col < a.n) o[j] += zrow[col];
        }
        activate_all<NJ>(o, a.act, a.slope, a.alpha, a.lambda);
        if (row_ok) {
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const uint32_t col = col0 + g * 32 * WV + l32 * WV;
                if (WV > 1 && col + WV <= a.n) {
                    if constexpr (WV == 4) *reinterpret_cast<float4u*>(zrow + col) = float4u{o[4 * g], o[4 * g + 1], o[4 * g + 2], o[4 * g + 3]};
                    else if constexpr (WV == 2) *reinterpret_cast<float2u*>(zrow + col) = float2u{o[2 * g], o[2 * g + 1]};
                } else {
#pragma unroll
                    for (int e = 0; e < WV; e++)
                        if (col + e < a.n) zrow[col + e] = o[g * WV + e];
                }
            }
        }
        if constexpr (NJ == 4) {
            if (a.seg_max) {
                // the 64 columns of a segment are 16 neighbouring lanes (WV = 4), or all 32 of a half, two segments one after the other
                float m[2] = {-__builtin_inff(), -__builtin_inff()};
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    if (col0 + (j / WV) * 32 * WV + l32 * WV + j % WV < a.n) m[WV == 4 ? 0 : j / 2] = fmaxf(m[WV == 4 ? 0 : j / 2], o[j]);
#pragma unroll
                for (int h = 0; h < (WV == 4 ? 1 : 2); h++) {
#pragma unroll
                    for (int d = 1; d < (WV == 4 ? 16 : 32); d *= 2) m[h] = fmaxf(m[h], __shfl_xor(m[h], d));
                    const uint32_t seg = col0 / 64 + (WV == 4 ? l32 / 16 : h);
                    if ((l32 & (WV == 4 ? 15 : 31)) == 0 && row_ok && seg < a.nseg) a.seg_max[(uint64_t)row * a.nseg + seg] = m[h];
                }
            }
        }
    };
    if constexpr (KS == 1) {
        __shared__ float sRows[4][4][NJ][kWave];   // per wavefront: four accumulator registers of every block at a time
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) sRows[wave][v][j][lane] = acc[i][j][4 * r + v];
                // (a lane reads what it wrote itself: no wait but the counter's)
#pragma unroll 1
                for (int v = 0; v < 4; v++) {
                    float o[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; j++) o[j] = sRows[wave][v][j][lane];
                    finish_row(row0 + i * 32 + 8 * r + 4 * lhi + v, o);
                }
            }
    } else {
        // KS accumulator registers of every block at a time; wavefront w adds up and finishes the w-th of them
        __shared__ float sPart[KS][KS][NJ][kWave];   // [register][wavefront]
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int r = 0; r < 16 / KS; r++) {
                if (i + r > 0) __syncthreads();   // the round before has been read
#pragma unroll
                for (int v = 0; v < KS; v++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) sPart[v][wave][j][lane] = acc[i][j][r * KS + v];
                __syncthreads();
                float o[NJ];
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    float p[KS];
#pragma unroll
                    for (int w = 0; w < KS; w++) p[w] = sPart[wave][w][j][lane];
#pragma unroll
                    for (int d = 1; d < KS; d *= 2)
#pragma unroll
                        for (int w = 0; w < KS; w += 2 * d) p[w] += p[w + d];
                    o[j] = p[0];
                }
                const uint32_t v = r * KS + wave;
                finish_row(row0 + i * 32 + 8 * (v / 4) + 4 * lhi + v % 4, o);
            }
    }
}

template <int NJ, int MI, int KS> static void launch_fc_rows(const FcRowsArgs& a)
{
    const uint32_t tiles = (a.n + 32 * NJ - 1) / (32 * NJ);
    const dim3 grid(KS == 1 ? (tiles + 3) / 4 : tiles, (a.batch + 32 * MI - 1) / (32 * MI)), block(KS == 1 ? 256 : 64 * KS);
    hipStream_t s = ctx().stream;
    if (NJ >= 4 && a.n % 4 == 0) hipLaunchKernelGGL((fc_rows_kernel<NJ, MI, KS, NJ >= 4 ? 4 : 1>), grid, block, 0, s, a);
    else if (NJ >= 2 && a.n % 2 == 0) hipLaunchKernelGGL((fc_rows_kernel<NJ, MI, KS, NJ >= 2 ? 2 : 1>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fc_rows_kernel<NJ, MI, KS, 1>), grid, block, 0, s, a);
}

constexpr uint32_t kRowsWide = 4096;   // from this width on a wavefront takes 128 columns, below it 32

// Where the line lies (us, this kernel against the tiled one, both back to back):
//   wide layers: up to 64 rows always (8 x 512 x 27,278: 15.4 / 38.8; 64 x 1,024 x 27,278: 45 / 87; 4 x 128 x 1,000,000: 110 / 287).
//   Up to 128 rows for long sums, until the 128-row tiles fill the GPU (128 x 1,024 x 27,278: 87 / 110); with short ones the
//   64 x 64 tiles are level or better (100 x 128 x 27,278: 19.1 / 17.1; 128 x 256 x 60,000: 48 / 42), and from 160 rows on always.
//   narrow layers: while the 64 x 64 tiles leave more than half of the compute units without one (1 x 1,024 x 1,024: 8.0 / 32;
//   256 x 1,024 x 1,024: 11 / 22; 256 x 300 x 300: 4.6 / 17); above that a tenth at most is to be had (512 x 1,024 x 1,024: 20.8 / 23,
//   1,024 x 512 x 512: 12.1 / 12.7).  Sums of at most 32 products stay where they are: there is nothing to split.  So do sums
//   of more than 4,096: cut into sixteen they would be five times closer to the exact sums than those of the split-products mode, which is to be as
//   close as this one.
bool fc_rows_takes(uint32_t batch, uint32_t k, uint32_t n, uint32_t ldx, uint32_t ldw, int transposed)
{
    if (transposed || (8ull * ldw + n) * 4 >= (1ull << 32) || (uint64_t)batch * ldx * 4 >= (1ull << 32)) return false;   // the lanes' 32-bit byte offsets
    const uint64_t cus = (uint64_t)ctx().num_cus;
    if (n >= kRowsWide) return batch <= 64 || (batch <= 128 && k >= 512 && (n + 127) / 128 < 2 * cus);
    return k > 32 && k <= 4096 && (uint64_t)((batch + 63) / 64) * ((n + 63) / 64) < cus / 2;
}

int fc_rows_run(const float* X, uint32_t ldx, const float* W, uint32_t ldw, const float* bias, float* Z, uint32_t ldz, uint32_t batch,
                uint32_t k, uint32_t n, int accumulate, uint32_t activation, const dsx_act_params* params, float* seg_max,
                uint32_t* seg_width, uint32_t plan_n)
{
    FcRowsArgs a{};
    a.X = X; a.W = W; a.bias = bias; a.Z = Z;
    a.ldx = ldx; a.ldw = ldw; a.ldz = ldz;
    a.batch = batch; a.k = k; a.n = n;
    a.accumulate = accumulate;
    a.act = activation;
    a.slope = params ? params->slope : 0.01f;
    a.alpha = params ? params->alpha : 1.0f;
    a.lambda = params ? params->lambda : 1.0f;
    const uint64_t cus = (uint64_t)ctx().num_cus;
    if (plan_n >= kRowsWide) {   // (how a sum is split depends on plan_n alone: column blocks of one product agree)
        if (seg_max && seg_width && !accumulate) {
            a.seg_max = seg_max;
            a.nseg = (n + 63) / 64;
            *seg_width = 64;
        }
        // Four wavefronts share a tile's k unless there are tiles enough to keep every SIMD busy without (8 x 256 x 500,000: 103 us
        // against 110; 8 x 512 x 27,278: 15.4 us with four, 16.1 with eight).  32 rows per wavefront where a second block would be
        // mostly padding.
        const bool split = k > 32 && (plan_n + 127) / 128 < 8 * cus;
        if (((batch - 1) / 32) % 2 == 0) {
            if (split) launch_fc_rows<4, 1, 4>(a);
            else launch_fc_rows<4, 1, 1>(a);
        } else {
            if (split) launch_fc_rows<4, 2, 4>(a);
            else launch_fc_rows<4, 2, 1>(a);
        }
    } else {
        // as many wavefronts per tile as the number of tiles asks for (us with 4, 8, 16: 200 x 512 x 2,000 12.4, 12.7, 13.2;
        // 64 x 1,024 x 1,024 -, 10.8, 11.1; 100 x 300 x 1,000 5.4, 4.9, 4.6; 1 x 1,024 x 1,024 -, 8.4, 8.0)
        const uint64_t tiles = ((uint64_t)(batch + 31) / 32) * ((plan_n + 31) / 32);
        if (tiles >= 128) launch_fc_rows<1, 1, 4>(a);
        else if (tiles >= 64) launch_fc_rows<1, 1, 8>(a);
        else launch_fc_rows<1, 1, 16>(a);
    }
    DSX_LAUNCH_CHECK("fc_rows_kernel");
    return DSX_OK;
}

}  // namespace dsx
