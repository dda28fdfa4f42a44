// F32 weights (the projections a Q4_K_M file keeps unquantized, e.g. the DeltaNet alpha/beta of
// docs/model.md:328): y[t][r] = sum_k W[r][k] x[t][k], replacing the reference's F32 instantiation
// of its GEMV/GEMM (qwen_cuda/kernels.cu:74-78, 397) and the CPU path's F32 rows used as stored
// (qwen_cpu/ops.h:60-67, quants.h:193-203).  W stays row-major as in the file (no dequant, no
// repack), every product and sum is fp32, and up to four matrices that share x take one launch.
//
// The matrices are small (5120 x 48 in the model), so what bounds a call is how many CUs its loads
// are spread over, not the bytes.  Two kernels, both without a workspace (F32 calls need none, so they
// may come first on a stream under capture):
//  * k_f32_rows: one work-group per 1, 2 or 4 rows, k split over its 256 threads (rows of up to 768 elements:
//    over a wave), up to 16 tokens per pass.  n = 48, k = 5120 (us per call, graph-timed, one wave per row before): one token 10.4 ->
//    2.6 (~2 of them the launch), 13 tokens 66 -> 3.3, 512 tokens 3540 -> 12.3.
//  * k_f32_tile: fp32 MFMA on tiles of 16 x 16 or 32 x 32 (rows x tokens), k split over the sixteen waves of the
//    work-group, their sums added through LDS in wave order.  n = 1024, m = 512 58 us (93 TFLOP/s);
//    bounded by the operand loads (a lane's 16 bytes are a line of their own) as much as by the MFMAs.
#include <algorithm>
#include <type_traits>

#include "qk_device.h"
#include "qk_internal.h"

namespace qk {
namespace {

// Eight consecutive activations of a token, elements e .. e + 7 (e % 8 == 0), as loaded: 16 bytes where x
// is fp16 (the xperm layout keeps aligned runs of eight together), 32 where it is fp32.
template <int FMT>
struct X8 {
    std::conditional_t<FMT == ACT_F32, f4, h8> v[FMT == ACT_F32 ? 2 : 1];
    __device__ void load(const void* x, size_t row, int e) {
        if constexpr (FMT == ACT_F32) {
            const float* p = (const float*)x + row + e;
            v[0] = *(const f4*)p;
            v[1] = *(const f4*)(p + 4);
        } else {
            v[0] = *(const h8*)((const _Float16*)x + row + (FMT == ACT_F16_XPERM ? xperm_pos(e) : e));
        }
    }
    __device__ float at(int q) const {
        if constexpr (FMT == ACT_F32) return v[q >> 2][q & 3];
        else return (float)v[0][q];
    }
};

// Sum over the wave's 64 lanes on the VALU (every lane gets it).
__device__ inline float wave_sum(float v) { return xor32_sum(xor16_sum(sum16(v))); }

// Tokens MT * blockIdx.y .. + MT - 1 of rows of matrix blockIdx.z (rows and tokens past the ends re-read the last
// one and are not stored), RW rows at a time with k over KT threads.
// KT = 256: the work-group's rows are RW * blockIdx.x .. + RW - 1; thread i takes elements 4 i .. 4 i + 3 of every
// 1024.  KT = 64: each wave has RW rows of its own and thread i elements 4 i .. of every 256, for rows too
// short to occupy 256 threads.
template <int FMT, int RW, int MT, int KT>
__global__ __launch_bounds__(256) void k_f32_rows(const F32Mats M, int k, const void* __restrict__ x, int m) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int z = blockIdx.z, n = M.n[z], t0 = blockIdx.y * MT;
    const int row0 = KT == 256 ? blockIdx.x * RW : (blockIdx.x * 4 + wave) * RW;
    if (row0 >= n) return;  // KT = 64: no barrier follows
    const float* wr[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) wr[i] = M.w[z] + (size_t)min(row0 + i, n - 1) * k;
    float acc[RW][MT];
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[i][t] = 0.0f;
    // passes whose loads go out together
    constexpr int U = KT == 64 ? 1 : MT == 1 ? 5 : MT == 4 && RW == 1 ? 2 : 1;
#pragma unroll U
    for (int e = 4 * (KT == 256 ? threadIdx.x : lane); e < k; e += 4 * KT) {
        f4 wv[RW], xv[MT];
#pragma unroll
        for (int i = 0; i < RW; i++) wv[i] = *(const f4*)(wr[i] + e);
#pragma unroll
        for (int t = 0; t < MT; t++) xv[t] = load_act4(x, FMT, k, min(t0 + t, m - 1), e);
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                acc[i][t] = fmaf(wv[i].x, xv[t].x, fmaf(wv[i].y, xv[t].y, fmaf(wv[i].z, xv[t].z, fmaf(wv[i].w, xv[t].w, acc[i][t]))));
    }
    // sum t RW + i: over the wave's lanes, and over the four waves where they share a row
    float sum = 0.0f;
    int o = lane;
    if constexpr (KT == 256) {
        __shared__ float part[4][RW * MT];
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const float v = wave_sum(acc[i][t]);
                if (lane == 0) part[wave][t * RW + i] = v;
            }
        __syncthreads();
        o = threadIdx.x;
        if (o < RW * MT) sum = (part[0][o] + part[1][o]) + (part[2][o] + part[3][o]);
    } else {
        static_assert(RW * MT <= 64, "a lane per sum");
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const float v = wave_sum(acc[i][t]);
                if (lane == t * RW + i) sum = v;
            }
    }
    const int t = t0 + o / RW, row = row0 + o % RW;
    if (o < RW * MT && row < n && t < m) M.y[z][(size_t)t * n + row] = sum;
}

// D(16x16 f32) += A(16x4 f32) * B(4x16 f32).  Lane l holds A[l & 15][l >> 4], B[l >> 4][l & 15] and
// D[4 (l >> 4) + i][l & 15].
__device__ inline f4 mfma_f32(float a, float b, const f4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int TILE_WAVES = 16;
// A work-group of WV = 16 waves computes 16 R rows (A operand) x 16 R tokens (B operand) of matrix blockIdx.z.
// Wave w takes 32 of every 32 WV elements of k: lane (r, g) loads elements 8 g .. 8 g + 7 of them for
// row / token r of each tile (four lanes one 128-byte line), and MFMA e multiplies element 8 g + e of
// every lane, so the four k-slots of an MFMA are the lanes' own elements.  Rows and tokens past the
// ends re-read the last one and are not stored.  Each pass's 32 products an output are summed from zero and
// then added: one chain of MFMAs over a wave's k / 16 products rounds at the size of its whole sum
// (error against float64 at k = 5120: 3.3e-7, with the pass sums 1.4e-7; the time is the same).
template <int FMT, int R>
__global__ __launch_bounds__(64 * TILE_WAVES) void k_f32_tile(const F32Mats M, int k, const void* __restrict__ x, int m) {
    constexpr int WV = TILE_WAVES;
    const int z = blockIdx.z, n = M.n[z], row0 = blockIdx.x * 16 * R, t0 = blockIdx.y * 16 * R;
    if (row0 >= n) return;
    __shared__ __align__(16) float part[WV * R * R * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const float* wr[R];
    size_t xr[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        wr[i] = M.w[z] + (size_t)min(row0 + 16 * i + r, n - 1) * k;
        xr[i] = (size_t)min(t0 + 16 * i + r, m - 1) * k;
    }
    f4 acc[R][R];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < R; j++) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int e = 32 * wave + 8 * g; e < k; e += 32 * WV) {  // k % 256 == 0
        f4 wa[R][2];
        X8<FMT> xv[R];
#pragma unroll
        for (int i = 0; i < R; i++) {
            wa[i][0] = *(const f4*)(wr[i] + e);
            wa[i][1] = *(const f4*)(wr[i] + e + 4);
            xv[i].load(x, xr[i], e);
        }
#pragma unroll
        for (int i = 0; i < R; i++)
#pragma unroll
            for (int j = 0; j < R; j++) {
                f4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 0; q < 8; q++) d = mfma_f32(wa[i][q >> 2][q & 3], xv[j].at(q), d);
                acc[i][j] += d;
            }
    }
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < R; j++) *(f4*)(part + ((wave * R + i) * R + j) * 256 + 4 * lane) = acc[i][j];
    __syncthreads();
    for (int o = threadIdx.x; o < 256 * R * R; o += 64 * WV) {
        float v = part[o];
#pragma unroll
        for (int w = 1; w < WV; w++) v += part[w * 256 * R * R + o];
        const int i = (o >> 8) / R, j = (o >> 8) % R;
        const int row = row0 + 16 * i + 4 * ((o >> 6) & 3) + (o & 3), t = t0 + 16 * j + ((o >> 2) & 15);
        if (row < n && t < m) M.y[z][(size_t)t * n + row] = v;
    }
}

constexpr int MAX_GRID_Y = 65535;

template <int FMT, int RW, int MT, int KT = 256>
void launch_rows(const F32Mats& M, int nmax, int cnt, int k, const void* x, int m, hipStream_t s) {
    constexpr int ROWS = RW * (256 / KT);
    hipLaunchKernelGGL((k_f32_rows<FMT, RW, MT, KT>), dim3((nmax + ROWS - 1) / ROWS, (m + MT - 1) / MT, cnt), dim3(256), 0, s,
                       M, k, x, m);
}
template <int FMT, int R>
void launch_tile(const F32Mats& M, int nmax, int cnt, int k, const void* x, int m, hipStream_t s) {
    constexpr int T = 16 * R;
    hipLaunchKernelGGL((k_f32_tile<FMT, R>), dim3((nmax + T - 1) / T, (m + T - 1) / T, cnt), dim3(64 * TILE_WAVES), 0, s, M, k,
                       x, m);
}

template <int FMT>
void launch_fmt(const F32Mats& M, int cnt, int k, const void* x, int m, hipStream_t s) {
    int nmax = 0;
    for (int z = 0; z < cnt; z++) nmax = std::max(nmax, M.n[z]);
    long long rows = 0;
    for (int z = 0; z < cnt; z++) rows += M.n[z];
    // The lines between the forms, measured at k = 5120 on fp16 x (us per call):
    //  * MFMA tiles pay from ~96 Ki outputs, whose tiles fill the CUs (n = 48: 30.9 against 32.7 on rows at
    //    m = 2048, 30.1 against 20.1 at m = 1000; n = 1024: 31.0 against 37.7 at m = 128), with more
    //    than the 16 tokens that one pass of the row kernel takes (n = 17408: 115.7 against 100.0 at
    //    m = 16, 118.8 against 183.8 at m = 20).
    //  * Tiles of 16 x 16 pay from 44 Ki outputs while they run in one round over the CUs (256 tiles): a
    //    work-group's time is its own 32 lines of k, whatever the call (us, rows / tiles on fp16 x: n = 48, m =
    //    1000 21.0 / 16.3, n = 128, m = 512 24.5 / 16.4, n = 1024, m = 64 24.1 / 16.3, n = 4096, m = 13 29.8 /
    //    23.1, at k = 1024 11.9 / 6.7; on fp32 x 29.3 / 20.4 for the first; below the line n = 48, m = 760 23.3 /
    //    20.4 but n = 128, m = 300 18.2 / 20.4; two rounds, n = 48, m = 1500: 29.6 / 31.2).  One rule for
    //    every format, so that they give the same bits.
    //  * Weights beyond the L2s (32 MiB) are read once: 16 tokens a pass (n = 17408, m = 16: 100.0
    //    against 138.1 with eight, 232.0 with four).
    //  * Four tokens a pass spread a small call over the most work-groups; eight pay once 8192 passes are
    //    there (n = 1024, m = 32 13.5 against 13.6, n = 4096, m = 8 17.5 against 25.8; n = 48, m = 512 13.5
    //    against 12.3).
    //  * Rows share the loads of x as soon as the work-groups left still cover the CUs (n = 48: m = 16 one
    //    row 3.29, two 3.78; m = 64 4.50 / 4.41 / four 4.61; m = 256 10.8 / 7.9 / 7.25).
    //  * Rows of up to 768 elements leave a quarter and more of 256 threads without any: a wave per two or four rows
    //    where a call has enough of them to fill the CUs (us, one wave per row / 256 threads / this: k = 256, n =
    //    65536, m = 1 19.2 / 25.3 / 11.1, m = 5 40.3 / 47.7 / 17.2, m = 13 81.2 / 110 / 33.2; n = 4096, m = 5 5.5 /
    //    5.1 / 3.6; k = 768, n = 65536, m = 1 36.1 / 41.4 / 34.0; at k = 1024 44.9 / 43.2 / 45.5).
    // (Past 2^23 rows a work-group per row would exceed a grid's 2^32 threads.)
    if ((m > 16 && rows * m >= 96 * 1024) || nmax > (1 << 23)) return launch_tile<FMT, 2>(M, nmax, cnt, k, x, m, s);
    long long tiles = 0;
    for (int z = 0; z < cnt; z++) tiles += (long long)((M.n[z] + 15) / 16) * ((m + 15) / 16);
    if (rows * m >= 44 * 1024 && tiles <= 256) return launch_tile<FMT, 1>(M, nmax, cnt, k, x, m, s);
    const long long passes = rows * ((m + 3) / 4);
    if (k <= 768 && passes >= 4096) {
        if (m == 1) return launch_rows<FMT, 2, 1, 64>(M, nmax, cnt, k, x, m, s);
        if (m <= 4) return launch_rows<FMT, 2, 4, 64>(M, nmax, cnt, k, x, m, s);
        return launch_rows<FMT, 4, 8, 64>(M, nmax, cnt, k, x, m, s);
    }
    if (m == 1) return launch_rows<FMT, 1, 1>(M, nmax, cnt, k, x, m, s);
    if (m > 8 && m <= 16 && rows * k > (8ll << 20)) return launch_rows<FMT, 4, 16>(M, nmax, cnt, k, x, m, s);
    if (m > 4 && passes >= 8192) return launch_rows<FMT, 4, 8>(M, nmax, cnt, k, x, m, s);
    if (passes >= 2048) return launch_rows<FMT, 4, 4>(M, nmax, cnt, k, x, m, s);
    if (passes >= 512) return launch_rows<FMT, 2, 4>(M, nmax, cnt, k, x, m, s);
    return launch_rows<FMT, 1, 4>(M, nmax, cnt, k, x, m, s);
}

}  // namespace

int launch_f32(const F32Mats& mats, int cnt, int k, const void* x, int xfmt, int m, hipStream_t s) {
    constexpr int CHUNK = 4 * MAX_GRID_Y;  // tokens per launch (the grid's second dimension; at least four a pass)
    F32Mats M = mats;
    for (int t0 = 0; t0 < m; t0 += CHUNK) {
        const int mt = std::min(CHUNK, m - t0);
        if (xfmt == ACT_F32) launch_fmt<ACT_F32>(M, cnt, k, (const float*)x + (size_t)t0 * k, mt, s);
        else if (xfmt == ACT_F16) launch_fmt<ACT_F16>(M, cnt, k, (const _Float16*)x + (size_t)t0 * k, mt, s);
        else launch_fmt<ACT_F16_XPERM>(M, cnt, k, (const _Float16*)x + (size_t)t0 * k, mt, s);
        if (hipGetLastError() != hipSuccess) return -1;
        for (int z = 0; z < cnt; z++) M.y[z] += (size_t)mt * M.n[z];
    }
    return 0;
}

}  // namespace qk
