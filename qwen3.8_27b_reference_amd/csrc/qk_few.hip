// Few-token GEMM (5 to 16 tokens by default): weight-streaming form of the prefill GEMM's math for batched decode.
//
// Same operands and numerics class as k_gemm (weights dequantized to fp16 with fp16-rounded scales, fp16 x,
// fp32 accumulate; the reference's tolerance path, qwen_cuda/kernels.cu:127-181), but organised like
// the decode GEMV: at few tokens k_gemm's step (a barrier, two pairs' dequant per compute wave, one
// such wave per SIMD) is a latency chain of ~0.45 us that leaves the memory system waiting, whatever is
// in flight (6, 8 and 10 stages measured 5..8 % slower than 4).  Here every wave streams its own units
// through a private LDS-DMA ring and no barrier lies inside the loop:
//
//  * A unit is one 16-row T16 tile x one super-block, 8 v_mfma_f32_16x16x32_f16 on its 16 rows x 16 token
//    columns.  The lanes take the weight bytes as the T16 planes hold them for 16-byte loads, so a lane
//    group's k-slots belong to the group's own sub-blocks and a lane applies two scales per unit
//    (Q4_K, Q5_K) instead of eight.
//  * k is cut into S slices.  A work-group holds one slice of x in LDS for the whole call, as fp16 B
//    operands brought there by LDS-DMA in the order the MFMAs read them (fp16 x, plain or xperm, where
//    it lies; fp32 x after k_gemm_cvt_x), and a contiguous range of the tiles.  Its waves cut the
//    range's units evenly; a tile cut between waves is summed through LDS in wave order.
//  * Slices are added by the split-K sum (or the gate/up pair's k_glu_sum) in slice order.
//
// What bounds it: the weight stream and the call's ends.  Q4_K 17408 x 5120 at 13 tokens takes 16.8 us (50 MB;
// 10.3 at the rate of a long stream), of which ~2 are the launch, ~4 the second launch that adds the
// slices and ~2 the x image before the first unit; the output projection at 8 tokens streams 5.5 TB/s.
#include <algorithm>

#include "qk_device.h"
#include "qk_dma.h"
#include "qk_internal.h"

namespace qk {
namespace {

constexpr int LDS_PER_CU = 160 * 1024;
constexpr int DEPTH = 2;        // units in flight per wave
constexpr int MAX_WAVES = 12;
constexpr int MAX_SLICES = 32;
constexpr int XREC = 32;        // 16-byte pieces of x per token and super-block

template <int STEP, int K>
__device__ inline void wait_units(int k) {  // at most min(k, K) units of STEP DMAs in flight
    if constexpr (K == 0) {
        wait_vm<0>();
    } else {
        if (k >= K) wait_vm<K * STEP>();
        else wait_units<STEP, K - 1>(k);
    }
}

// k-slots 8 g .. 8 g + 7 of MFMA f multiply the eight elements of piece P (elements 8 P .. 8 P + 7) of the
// super-block:
//   Q4_K / Q5_K: lane group g holds qs bytes 32 g .. 32 g + 31: f = 4 hi + 2 i + h is nibble hi of bytes
//     16 i + 8 h + j, i.e. sub-block 2 g + hi: P = 8 g + f.
//   Q6_K: f = 4 n + 2 hi + h of half n: crumb s = (g >> 1) + 2 hi, l = 16 (g & 1) + 8 h + j, sub-block
//     8 n + 4 hi + g: P = 8 (f >> 1) + 2 g + h.
//   Q8_0: f = 2 t + h: block 2 t + (g >> 1): P = 8 (f >> 1) + 2 g + h.
// In memory a token's super-block is four 128-byte lines of eight pieces: line P >> 3, place P & 7 in plain
// x; line P & 3, place P >> 2 in the xperm layout (qk_device.h xperm_pos).  The image keeps whole
// lines, so that eight lanes of a DMA take one (lanes that each took 16 bytes of another token's row
// cost a line lookup apiece: 6144 for a 96 KiB image, ~2.7 us): line v of token t at (v XT + t) 128,
// its place q at slot q ^ ((t >> 1) & 7), so that the 16 lanes of an LDS cycle read 16 different
// 16-byte bank groups.
template <int TYPE, int XT, bool XPERM>
struct XImg {
    static constexpr bool K4 = TYPE == T_Q4_K || TYPE == T_Q5_K;
    // byte offset of lane (t, g)'s operand of MFMA f in a super-block's image: (base ^ flip(f)) + add(f)
    __device__ static int base(int t, int g) {
        int line, place;
        if constexpr (K4) line = XPERM ? 0 : g, place = XPERM ? 2 * g : 0;
        else line = XPERM ? 2 * (g & 1) : 0, place = XPERM ? g >> 1 : 2 * g;
        return (line * XT + t) * 128 + 16 * (place ^ ((t >> 1) & 7));
    }
    static constexpr int flip(int f) { return 16 * (K4 ? (XPERM ? f >> 2 : f) : (XPERM ? 2 * (f >> 1) : f & 1)); }
    static constexpr int add(int f) { return 128 * XT * (K4 ? (XPERM ? f & 3 : 0) : (XPERM ? f & 1 : f >> 1)); }
};

// acc += W x for one unit: G its group in the ring, X its super-block's image, xl = XI::base of this lane.
template <int TYPE, typename XI>
__device__ inline f4 few_unit(const uint8_t* G, const uint8_t* X, int xl, int lane, f4 acc) {
    const int r = lane & 15, g = lane >> 4;
    auto b = [&](int f) __attribute__((always_inline)) { return *(const h8*)(X + (xl ^ XI::flip(f)) + XI::add(f)); };
    if constexpr (TYPE == T_Q4_K || TYPE == T_Q5_K) {
        const u4 q[2] = {ld16(G + 16 * lane), ld16(G + 1024 + 16 * lane)};
        const uint32_t s0 = ld4(G + 2112 + 12 * r), s1 = ld4(G + 2116 + 12 * r), s2 = ld4(G + 2120 + 12 * r);
        const uint32_t dd = ld4(G + 2048 + 4 * r);
        // 6-bit scales and mins of sub-blocks 2 g, 2 g + 1 (qwen_cpu/quants.h:33-41, four at a time), then
        // (half(d sc), half(-dmin m)): fp16 products of exact factors, one rounding
        const uint32_t S = g < 2 ? s0 & 0x3F3F3F3Fu : (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
        const uint32_t M = g < 2 ? s1 & 0x3F3F3F3Fu : ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
        const uint32_t sel = 0x0C040C00u + 0x00020002u * (g & 1);  // bytes (S[b], 0, M[b], 0), b = 2 (g & 1)
        const h2 dmn = as_h2(dd ^ 0x80000000u), m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
        auto qh = [&](int i) {
            if constexpr (TYPE == T_Q5_K) return ld16(G + 2304 + 256 * i + 16 * r) >> (2 * g);
            else return u4{0u, 0u, 0u, 0u};
        };
        const u4 H[2] = {qh(0), qh(1)};
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const h2 v = (as_h2(__builtin_amdgcn_perm(M, S, sel + 0x00010001u * hi) | 0x64006400u) + m1024) * dmn;
            const h2 ds = {v.x, v.x}, dm = {v.y, v.y};
#pragma unroll
            for (int i = 0; i < 2; i++) {
                u4 n = (hi ? q[i] >> 4 : q[i]) & 0x0F0F0F0Fu;
                if constexpr (TYPE == T_Q5_K) n |= ((H[i] >> hi) & 0x01010101u) << 4;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    h8 a;
                    if constexpr (TYPE == T_Q4_K) {
                        a = make_h8(pk_fma(nib_pair_lo(n[2 * h]), ds, dm), pk_fma(nib_pair_hi(n[2 * h]), ds, dm),
                                    pk_fma(nib_pair_lo(n[2 * h + 1]), ds, dm), pk_fma(nib_pair_hi(n[2 * h + 1]), ds, dm));
                    } else {
                        auto w = [&](uint32_t p) { return as_u32(__builtin_elementwise_fma(as_h2(p) + m1024, ds, dm)); };
                        a = make_h8(w(perm_lo(n[2 * h])), w(perm_hi(n[2 * h])), w(perm_lo(n[2 * h + 1])),
                                    w(perm_hi(n[2 * h + 1])));
                    }
                    acc = mfma(a, b(4 * hi + 2 * i + h), acc);
                }
            }
        }
    } else if constexpr (TYPE == T_Q6_K) {
        const float d = h2f_bits(*(const uint16_t*)(G + 3328 + 2 * r));
        const h2 m1056 = {(_Float16)-1056.0f, (_Float16)-1056.0f};
#pragma unroll
        for (int n = 0; n < 2; n++) {
            const u4 L = ld16(G + 1024 * n + 16 * lane), Q = ld16(G + 2048 + 512 * n + 16 * (r + 16 * (g & 1)));
            const u4 C = Q >> (2 * (g >> 1));  // crumb g >> 1 in the low bits, 2 + (g >> 1) four above
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                const int sc = *(const int8_t*)(G + 3072 + 128 * n + 32 * (r >> 2) + 4 * (4 * hi + g) + (r & 3));
                const _Float16 ds = (_Float16)(d * (float)sc);
                const h2 vds = {ds, ds};
                const u4 v = hi ? ((L >> 4) & 0x0F0F0F0Fu) | (C & 0x30303030u)
                                : (L & 0x0F0F0F0Fu) | ((C << 4) & 0x30303030u);
                // (1024 + q) - 1056 = q - 32 exactly, then one rounding of (q - 32) * half(d * sc)
                auto w = [&](uint32_t p) { return as_u32((as_h2(p) + m1056) * vds); };
#pragma unroll
                for (int h = 0; h < 2; h++)
                    acc = mfma(make_h8(w(perm_lo(v[2 * h])), w(perm_hi(v[2 * h])), w(perm_lo(v[2 * h + 1])),
                                       w(perm_hi(v[2 * h + 1]))),
                               b(4 * n + 2 * hi + h), acc);
            }
        }
    } else {
        const u2 dd = ld8(G + 4096 + 16 * r + 8 * (g >> 1));  // d of blocks g >> 1, 2 + .., 4 + .., 6 + ..
        const h2 m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const u4 q = ld16(G + 1024 * t + 16 * lane) ^ 0x80808080u;
            const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)(dd[t >> 1] >> (16 * (t & 1))));
            const h2 vd = {d, d};
            // int8 b as (1024 + (b ^ 0x80)) - 1152, exact; one rounding of q * d
            auto w = [&](uint32_t p) { return as_u32((as_h2(p) + m1152) * vd); };
#pragma unroll
            for (int h = 0; h < 2; h++)
                acc = mfma(make_h8(w(perm_lo(q[2 * h])), w(perm_hi(q[2 * h])), w(perm_lo(q[2 * h + 1])),
                                   w(perm_hi(q[2 * h + 1]))),
                           b(2 * t + h), acc);
        }
    }
    return acc;
}

// Tokens' slots of the x image: 8 (columns 8..15 repeat 0..7) or 16.
template <int TYPE, int XT, bool XPERM>
__global__ __launch_bounds__(64 * MAX_WAVES) void k_few(const FewParams P) {
    using XI = XImg<TYPE, XT, XPERM>;
    constexpr int GB = group_bytes(TYPE), NDMA = (GB + 1023) / 1024, XSB = XREC * XT * 16;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = P.waves;
    // slice s of k, and tiles [t0, t0 + nt) of all the matrices' tiles
    const int s = blockIdx.x / P.wgs, j = blockIdx.x - s * P.wgs;
    const int sb0 = s * P.nsb / P.slices, cs = (s + 1) * P.nsb / P.slices - sb0;
    const int t0 = (int)((long long)j * P.ntiles / P.wgs), nt = (int)((long long)(j + 1) * P.ntiles / P.wgs) - t0;
    const int nu = nt * cs;
    auto first_unit = [&](int w) { return w * nu / W; };  // nu * W < 2^31, see few_plan
    const int u0 = first_unit(wave), n = first_unit(wave + 1) - u0;
    uint8_t* const img = smem;
    uint8_t* const ring = smem + P.lds_ring + wave * (DEPTH * GB);

    // x first: DMA d brings line (d / (XT / 8)) & 3 of eight tokens (tokens past m repeat the last; their
    // columns are not stored)
    for (int d = wave; d < cs * (XSB / 1024); d += W) {
        const int sb = sb0 + d / (XSB / 1024), line = (d / (XT / 8)) & 3, t = 8 * (d & (XT / 8 - 1)) + (lane >> 3);
        const int place = (lane & 7) ^ ((t >> 1) & 7);
        const int at = XPERM ? (sb & ~3) * 256 + 256 * line + 64 * (sb & 3) + 8 * place : sb * 256 + 64 * line + 8 * place;
        dma16(P.x + (size_t)min(t, P.m - 1) * P.k + at, img + 1024 * d);
    }
    // the wave's units, tile by tile: the issue cursor runs ahead of the compute cursor
    auto matrix_of = [&](int tile) {
        return (P.cnt > 1 && tile >= P.tile0[1]) + (P.cnt > 2 && tile >= P.tile0[2]) + (P.cnt > 3 && tile >= P.tile0[3]);
    };
    auto tile_ptr = [&](int tile) {
        tile = min(tile, P.ntiles - 1);
        const int z = matrix_of(tile);
        const uint8_t* w = z == 0 ? P.w[0] : z == 1 ? P.w[1] : z == 2 ? P.w[2] : P.w[3];
        const int base = z == 0 ? 0 : z == 1 ? P.tile0[1] : z == 2 ? P.tile0[2] : P.tile0[3];
        return w + ((size_t)(tile - base) * P.nsb + sb0) * GB;
    };
    int itile = t0 + u0 / cs, isb = u0 - (itile - t0) * cs, islot = 0;
    const uint8_t* ip = tile_ptr(itile) + (size_t)isb * GB;
    auto issue = [&]() __attribute__((always_inline)) {
        dma_group<GB>(ip, ring + islot, lane);
        islot = islot == (DEPTH - 1) * GB ? 0 : islot + GB;
        ip += GB;
        if (++isb == cs) {
            isb = 0;
            ip = tile_ptr(++itile);
        }
    };
    const int ahead = min(DEPTH, n);
    for (int i = 0; i < ahead; i++) issue();
    wait_units<NDMA, DEPTH>(ahead);  // the x DMAs, older than the units', have landed
    lds_barrier();

    // results: matrix z's slice s at y[z] + s * m * n[z] (slices = 1: the result itself)
    const int g = lane >> 4;
    const int tok = lane & 15;
    auto store = [&](int tile, const f4& v) {
        if (tok >= P.m) return;
        const int z = matrix_of(tile);
        float* y = z == 0 ? P.y[0] : z == 1 ? P.y[1] : z == 2 ? P.y[2] : P.y[3];
        const int base = z == 0 ? 0 : z == 1 ? P.tile0[1] : z == 2 ? P.tile0[2] : P.tile0[3];
        const int rows = z == 0 ? P.n[0] : z == 1 ? P.n[1] : z == 2 ? P.n[2] : P.n[3];
        *(f4*)(y + ((size_t)s * P.m + tok) * rows + 16 * (tile - base) + 4 * g) = v;
    };
    const int xl = XI::base(lane & (XT - 1), g);
    int ctile = t0 + u0 / cs, csb = u0 - (ctile - t0) * cs, cslot = 0;
    bool whole = csb == 0;  // the piece being summed starts its tile
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, head = acc, tail = acc;
    bool has_tail = false;
    for (int i = 0; i < n; i++) {
        if (i > 0 && i + DEPTH - 1 < n) {
            // the slot of unit i - 1: its LDS reads have returned
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue();
        }
        wait_units<NDMA, DEPTH - 1>(n - 1 - i);
        acc = few_unit<TYPE, XI>(ring + cslot, img + csb * XSB, xl, lane, acc);
        asm volatile("" ::: "memory");
        cslot = cslot == (DEPTH - 1) * GB ? 0 : cslot + GB;
        if (++csb == cs || i == n - 1) {
            if (csb < cs && whole) {  // the tile goes on in the next wave, which continues this piece
                tail = acc;
                has_tail = true;
            } else if (!whole) {  // the rest (or a middle part) of an earlier wave's tile
                head = acc;
            } else {
                store(ctile, acc);
            }
            acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
            whole = true;
            csb = 0;
            ctile++;
        }
    }
    // tiles cut between waves: the wave that began one adds the later waves' pieces in wave order
    lds_barrier();  // every wave is done with the image
    f4* const pieces = (f4*)img;
    pieces[wave * 64 + lane] = head;
    lds_barrier();
    if (has_tail) {
        const int tile = t0 + (u0 + n - 1) / cs, end = (tile - t0 + 1) * cs;
        for (int w = wave + 1; w < W && first_unit(w) < end; w++)
            if (first_unit(w + 1) > first_unit(w)) tail += pieces[w * 64 + lane];
        store(tile, tail);
    }
}

template <int TYPE, int XT>
int launch_xt(const FewParams& p, size_t lds, hipStream_t s) {
    const dim3 grid(p.slices * p.wgs), block(64 * p.waves);
    if (p.xperm) hipLaunchKernelGGL((k_few<TYPE, XT, true>), grid, block, lds, s, p);
    else hipLaunchKernelGGL((k_few<TYPE, XT, false>), grid, block, lds, s, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <int TYPE>
int launch_few_type(const FewParams& p, size_t lds, hipStream_t s) {
    return p.m <= 8 ? launch_xt<TYPE, 8>(p, lds, s) : launch_xt<TYPE, 16>(p, lds, s);
}

}  // namespace

// Plan: the K-slices of least estimated time (us), fitted to every slice count with 8 and 12 waves on 50 sizes of
// the four types at 5 and 13 tokens, single and as gate/up pairs (the slices chosen are 1.1 % slower than the best
// in the geometric mean, 13 % at most): the busiest CU's units at 24 KB/us, its image of x at 50 KB/us, 1.1 us where
// a tile is cut between waves, and for the second launch 1.7 us, 1.1 us per MB of partials (each part written, then
// read) and 1.1 us for the parts its threads load together (four; a single matrix's of more than four, eight): a
// pair of 8192 x 512 at 5 tokens in 32 slices took 13.7 us, in four 8.4.
// Eight waves (two per SIMD) with two units each in flight beat every larger ring on every shape (Q6_K
// 17408 x 5120 at 13 tokens: 8 waves x 2 units 20.4 us, 8 x 3 21.4, 12 x 2 21.3, 16 x 3 24.1; Q4_K 5120 x 17408
// at 8 tokens 15.4 / 15.6 / 15.3 / 18.9); twelve where a CU has many units (the gate/up pair of 5120 x 17408
// at 13 tokens 26.4 -> 25.8).
// No plan, so the GEMM, for Q4_K and Q8_0 beyond eight tokens where its work-groups of eight tile pairs fill 93 %
// and more of whole rounds of the CUs and a tile holds 36 KB: there its one barrier a step is hidden and its
// activations need no image (us, this kernel / the GEMM at 16 tokens: Q4_K 4096 x 128256 68.5 / 58.9, 4096 x 65536
// 36.3 / 33.0, Q8_0 3072 x 65536 44.6 / 40.5; over k = 4096..8192 and 65536, 128256 and 248320 rows at 9, 12 and 16 tokens
// the GEMM is 1.06x for both types).  Below the lines this kernel is ahead: rounds of 77 %, Q4_K 4096 x 151936
// 1.03x..1.24x, tiles of 28 KB, Q4_K 3072 x 65536 1.03x..1.14x, eight tokens 1.06x, Q5_K 1.17x, Q6_K 1.34x.
bool few_plan(int type, FewParams& p, int cus, size_t rows, size_t part_cap, bool sums, size_t& lds) {
    const int gb = group_bytes(type), xsb = XREC * (p.m <= 8 ? 8 : 16) * 16;
    if ((type == T_Q4_K || type == T_Q8_0) && p.m > 8 && p.cnt == 1 && !sums && p.nsb * gb >= 36000) {
        const long long wgs = (p.ntiles + 15) / 16, rounds = (wgs + cus - 1) / cus;
        if (100 * wgs >= 93 * rounds * cus) return false;
    }
    double best = 0.0;
    for (int S = 1; S <= p.nsb && S <= cus && S <= MAX_SLICES; S++) {
        const bool parts = S > 1 || sums;
        if (parts && (size_t)S * p.m * rows > part_cap) break;
        const int cs = (p.nsb + S - 1) / S, wgs = std::min(p.ntiles, cus / S), tiles = (p.ntiles + wgs - 1) / wgs;
        const long long units = (long long)tiles * cs;
        const size_t img = std::max((size_t)cs * xsb, (size_t)MAX_WAVES * 1024);  // also holds the pieces
        int waves = units >= 128 ? 12 : 8;
        if (img + (size_t)waves * DEPTH * gb > LDS_PER_CU) waves = 8;
        if (img + (size_t)waves * DEPTH * gb > LDS_PER_CU || units * waves >= (1ll << 31)) continue;
        bool cut = false;  // a wave of the largest range starts inside a tile
        for (int w = 1; w < waves; w++) cut |= w * units / waves % cs != 0;
        const int loads = sums ? (S + 3) / 4 : S <= 4 ? 1 : (S + 7) / 8 * 2;
        const double t = units * gb / 24e3 + cs * xsb / 50e3 + (cut ? 1.1 : 0.0) +
                         (parts ? 1.7 + S * 4.0 * p.m * (double)rows * 1.1e-6 + 1.1 * loads : 0.0);
        if (best == 0.0 || t < best) {
            best = t;
            p.slices = S;
            p.wgs = wgs;
            p.waves = waves;
            p.lds_ring = (int)img;
            lds = img + (size_t)waves * DEPTH * gb;
        }
    }
    return best > 0.0;
}

int launch_few(int type, const FewParams& p, size_t lds, hipStream_t s) {
    if (type == T_Q4_K) return launch_few_type<T_Q4_K>(p, lds, s);
    if (type == T_Q5_K) return launch_few_type<T_Q5_K>(p, lds, s);
    if (type == T_Q6_K) return launch_few_type<T_Q6_K>(p, lds, s);
    if (type == T_Q8_0) return launch_few_type<T_Q8_0>(p, lds, s);
    return -1;
}

}  // namespace qk
