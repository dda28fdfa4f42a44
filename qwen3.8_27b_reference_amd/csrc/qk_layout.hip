// Weight-placement kernels: GGUF <-> T16 repack, bit-exact row dequant, synthetic block fill.
//
//   repack    plays the role of k_repack (qwen_cuda/kernels.cu:945-961) driven by repack_weights
//             (qwen_cuda/qwen.cpp:185-193), with the T16 group layout of qk_device.h.
//   dequant   is the selftest vehicle k_dq_* (qwen_cuda/kernels.cu:363-373, qwen_cuda/qwen.cpp:1317):
//             fp32 results identical to qwen_cpu/quants.h Ref::q8_0 / q4_k / q5_k / q6_k (:45-121).
//   embed     is k_embed_* (qwen_cuda/kernels.cu:375-389): token rows through the same expressions
//             (a run's block gathered into LDS, four elements per lane), or a caller's embedding row
//             under a mask.
#include "qk_device.h"
#include "qk_internal.h"

namespace qk {
namespace {

// Repack: one work-group per (chunk of up to REPACK_SBS super-blocks, tile).  The chunk's 16 row windows
// go through LDS in GGUF byte order, so that both sides of HBM see 16-byte accesses: GGUF rows as the
// aligned words that cover them (a row of Q6_K blocks starts at any even byte; a tile's 16
// rows, and so the tensor, end on a 16-byte boundary, so the words stay inside it), T16 groups as they
// lie, one after another.  An LDS row keeps the window's offset in its word, so words move unshifted;
// its stride is an odd number of words, so that the 16 rows a group's neighbouring pieces come from
// fall into different banks.
// Bound: HBM, each byte read and written once.  Measured (us, GGUF -> T16 / back; one byte per thread and
// access before): Q4_K 5120 x 17408 60.8 -> 18.9 (5.3 TB/s) / 62.5 -> 21.5, Q6_K 17408 x 5120 103.5 -> 34.6 /
// 119.8 -> 46.1, Q6_K 5120 x 248320 1460 -> 378 / 1636 -> 459.  A chunk is 1, 2, 4 or 8 super-blocks, the fewest
// that leave at most 1152 work-groups: smaller tensors are bound by one chunk's time (Q6_K 17408 x 48 to GGUF in
// chunks of 8, 4, 2, 1: 10.1 7.3 4.7 4.0, a byte per thread before 6.4; x 512 12.4 9.6 7.8 9.1; 6144 x 1024 10.2 8.6 6.4
// 7.7), larger ones by the words that a window shares with its neighbours (17408 x 5120 42.4 44.7 48.4 66.2).
constexpr int REPACK_SBS = 8;
template <int TYPE>
struct Repack {
    static constexpr int BS = sb_bytes(TYPE), GB = group_bytes(TYPE), PIECES = GB / 16;
    static constexpr int STRIDE = ((REPACK_SBS * BS + 15) / 16 + 1) / 2 * 32 + 16;  // bytes, an odd count of 16
    // first byte past the planes whose 16-byte pieces are 16 bytes of one row (qs, ql, qh)
    static constexpr int PLANES = TYPE == T_Q6_K ? 3072 : TYPE == T_Q8_0 ? 4096 : 2048;
    // bytes that stay together outside the planes (d, dmin, scales)
    static constexpr int UNIT = TYPE == T_Q6_K ? 1 : TYPE == T_Q8_0 ? 2 : 4;
    static_assert(STRIDE >= REPACK_SBS * BS + (BS % 16 ? 16 : 0) && STRIDE / 16 % 2 == 1, "LDS row");
    __device__ static bool plane(int o) { return o < PLANES || (TYPE == T_Q5_K && o >= 2304); }
};

// Bytes between LDS and registers at 2-byte alignment (16-byte where the type's blocks allow it).
template <int TYPE>
__device__ inline u4 lds_get16(const uint8_t* p) {
    if constexpr (TYPE == T_Q4_K || TYPE == T_Q5_K) return *(const u4*)p;
    u4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *(const uint16_t*)(p + 4 * i) | ((uint32_t)*(const uint16_t*)(p + 4 * i + 2) << 16);
    return v;
}
template <int TYPE>
__device__ inline void lds_put16(uint8_t* p, const u4& v) {
    if constexpr (TYPE == T_Q4_K || TYPE == T_Q5_K) {
        *(u4*)p = v;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            *(uint16_t*)(p + 4 * i) = (uint16_t)v[i];
            *(uint16_t*)(p + 4 * i + 2) = (uint16_t)(v[i] >> 16);
        }
    }
}

template <int TYPE, bool TO_T16>
__global__ __launch_bounds__(256) void k_repack(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int nsb) {
    using R = Repack<TYPE>;
    using unit_t = std::conditional_t<R::UNIT == 4, uint32_t, std::conditional_t<R::UNIT == 2, uint16_t, uint8_t>>;
    __shared__ __align__(16) uint8_t row[16 * R::STRIDE];
    const uint64_t rb = (uint64_t)nsb * R::BS, tile = blockIdx.y;
    const int s0 = (int)((uint64_t)blockIdx.x * nsb / gridDim.x), s1 = (int)((uint64_t)(blockIdx.x + 1) * nsb / gridDim.x);
    const int len = (s1 - s0) * R::BS, words = (len + 15) / 16 + 1;  // a window covers at most that many
    const uint64_t first = tile * 16 * rb + (uint64_t)s0 * R::BS;     // row r's window starts at first + r * rb
    const uint64_t g0 = (tile * nsb + s0) * R::GB;                    // the chunk's groups in the T16 tensor
    // byte o .. of group piece `i`: its place in the LDS rows
    auto place = [&](int sb, int o) {
        int r, p;
        t16_src(TYPE, o, r, p);
        return row + r * R::STRIDE + (int)((first + r * rb) & 15) + sb * R::BS + p;
    };
    if constexpr (TO_T16) {
        // all of a thread's words are loaded before the first is stored; wave v takes rows v, v + 4, ...
        constexpr int NW = R::STRIDE / 16, PASSES = (NW + 63) / 64;
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        u4 v[4][PASSES];
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int c = 0; c < PASSES; c++) {
                const uint64_t a = first + (wave + 4 * q) * rb, at = (a & ~15ull) + 16 * (lane + 64 * c);
                if (at < a + len) v[q][c] = ld16(src + at);
            }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int c = 0; c < PASSES; c++) {
                const uint64_t a = first + (wave + 4 * q) * rb, at = (a & ~15ull) + 16 * (lane + 64 * c);
                if (at < a + len) *(u4*)(row + (wave + 4 * q) * R::STRIDE + 16 * (lane + 64 * c)) = v[q][c];
            }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < (s1 - s0) * R::PIECES; i += 256) {
        const int sb = i / R::PIECES, o = 16 * (i - sb * R::PIECES);
        u4 v;
        if constexpr (!TO_T16) v = ld16(src + g0 + 16 * (uint64_t)i);
        if (R::plane(o)) {
            uint8_t* p = place(sb, o);
            if constexpr (TO_T16) v = lds_get16<TYPE>(p);
            else lds_put16<TYPE>(p, v);
        } else {
            unit_t u[16 / R::UNIT];
            if constexpr (!TO_T16) __builtin_memcpy(u, &v, 16);
#pragma unroll
            for (int j = 0; j < 16 / R::UNIT; j++) {
                unit_t* p = (unit_t*)place(sb, o + j * R::UNIT);
                if constexpr (TO_T16) u[j] = *p;
                else *p = u[j];
            }
            if constexpr (TO_T16) __builtin_memcpy(&v, u, 16);
        }
        if constexpr (TO_T16) *(u4*)(dst + g0 + 16 * (uint64_t)i) = v;
    }
    if constexpr (!TO_T16) {
        __syncthreads();
        for (int i = threadIdx.x; i < 16 * words; i += 256) {
            const int r = i / words, w = i - r * words;
            const uint64_t a = first + r * rb, at = (a & ~15ull) + 16 * w;
            const uint8_t* p = row + r * R::STRIDE + 16 * w;
            if (at >= a && at + 16 <= a + len) {
                *(u4*)(dst + at) = *(const u4*)p;
            } else {  // the window's ends share their word with a neighbour's bytes
                for (int j = 0; j < 16; j += 2)
                    if (at + j >= a && at + j < a + len) *(uint16_t*)(dst + at + j) = *(const uint16_t*)(p + j);
            }
        }
    }
}

__device__ inline uint8_t wbyte(const uint8_t* w, int layout, int type, int nsb, uint64_t rb, int row, int sb, int p) {
    const int bs = sb_bytes(type);
    if (layout == LAYOUT_GGUF) return w[(uint64_t)row * rb + (uint64_t)sb * bs + p];
    const uint64_t g = ((uint64_t)(row >> 4) * nsb + sb) * (uint64_t)(16 * bs);
    return w[g + t16_dst(type, row & 15, p)];
}

__device__ inline uint32_t wu16(const uint8_t* w, int layout, int type, int nsb, uint64_t rb, int row, int sb, int p) {
    return (uint32_t)wbyte(w, layout, type, nsb, rb, row, sb, p) |
           ((uint32_t)wbyte(w, layout, type, nsb, rb, row, sb, p + 1) << 8);
}

// Element e of row `row`, with the reference's exact fp32 expression: Q8_0 q*d, Q4_K / Q5_K
// (d*sc)*q - dmin*m, Q6_K (d*sc)*(q-32).  All are single-rounding forms (products exact in fp32), so
// FMA contraction cannot change the bits.
__device__ inline float dq_elem(const uint8_t* __restrict__ w, int type, int layout, int nsb, uint64_t rb, int row,
                                int e) {
    const int sb = e >> 8, ee = e & 255;
    if (type == T_F32)  // rows as stored (qwen_cpu/quants.h:193-203); GGUF layout only
        return *(const float*)(w + (uint64_t)row * rb + 4 * (uint64_t)e);
    if (type == T_Q8_0) {  // qwen_cpu/quants.h:45-51
        const int j = ee >> 5;
        const float d = h2f_bits(wu16(w, layout, type, nsb, rb, row, sb, 34 * j));
        return (float)(int8_t)wbyte(w, layout, type, nsb, rb, row, sb, 34 * j + 2 + (ee & 31)) * d;
    }
    if (type == T_Q4_K || type == T_Q5_K) {  // qwen_cpu/quants.h:53-94
        const float d = h2f_bits(wu16(w, layout, type, nsb, rb, row, sb, 0));
        const float dmin = h2f_bits(wu16(w, layout, type, nsb, rb, row, sb, 2));
        uint8_t sc12[12];
        for (int i = 0; i < 12; i++) sc12[i] = wbyte(w, layout, type, nsb, rb, row, sb, 4 + i);
        const int g = ee >> 6, h = (ee >> 5) & 1, l = ee & 31;
        int sc, m;
        scale_min_k4(2 * g + h, sc12, sc, m);
        const int qs0 = type == T_Q5_K ? 48 : 16;
        int q = (wbyte(w, layout, type, nsb, rb, row, sb, qs0 + 32 * g + l) >> (4 * h)) & 0xF;
        if (type == T_Q5_K) q |= ((wbyte(w, layout, type, nsb, rb, row, sb, 16 + l) >> (2 * g + h)) & 1) << 4;
        const float d1 = d * (float)sc, m1 = dmin * (float)m;
        return d1 * (float)q - m1;
    }
    // Q6_K, qwen_cpu/quants.h:96-121
    const float d = h2f_bits(wu16(w, layout, type, nsb, rb, row, sb, 208));
    const int n = ee >> 7, s = (ee >> 5) & 3, l = ee & 31;
    const int lo = (wbyte(w, layout, type, nsb, rb, row, sb, 64 * n + 32 * (s & 1) + l) >> (s >= 2 ? 4 : 0)) & 0xF;
    const int hi = (wbyte(w, layout, type, nsb, rb, row, sb, 128 + 32 * n + l) >> (2 * s)) & 3;
    const int sc = (int8_t)wbyte(w, layout, type, nsb, rb, row, sb, 192 + (ee >> 4));
    return (d * (float)sc) * (float)((lo | (hi << 4)) - 32);
}

// One work-group per requested row, bit-exact with qwen_cpu/quants.h dequant_row.  A row index
// outside [0, n) writes a NaN row instead of reading outside the tensor.
__global__ __launch_bounds__(256) void k_dequant(const uint8_t* __restrict__ w, int type, int layout, int k, int n,
                                                 uint64_t rb, const int32_t* __restrict__ rows, float* __restrict__ out) {
    const int row = rows[blockIdx.x];
    const int nsb = k / 256;
    float* dst = out + (uint64_t)blockIdx.x * k;
    const bool ok = (unsigned)row < (unsigned)n;
    for (int e = threadIdx.x; e < k; e += blockDim.x) dst[e] = ok ? dq_elem(w, type, layout, nsb, rb, row, e) : __builtin_nanf("");
}

// Token embedding (the reference's k_embed_* , qwen_cuda/kernels.cu:375-389, 396, launched at
// qwen_cuda/qwen.cpp:265): x[t] = embd[t] where mask[t] is set (an embedding computed elsewhere, e.g.
// an image token), else row tokens[t] of the table, bit-exact; a token id outside [0, n) writes a NaN
// row instead of reading outside the table.  One wave per (256-column run sb, token t): the lanes
// gather the row's block of that run into LDS in GGUF byte order (every byte load independent of the
// others, so the run costs one memory round trip however the layout scatters it), then lane l
// decodes elements 4l .. 4l + 3 of the run, which share their scale (and for Q8_0 their block), with
// the expressions of dq_elem, and stores them as one 16-byte write.
__device__ inline f4 dq4_block(const uint8_t* blk, int type, int ee) {  // blk: LDS, GGUF block order
    f4 o;
    if (type == T_Q8_0) {  // qwen_cpu/quants.h:45-51
        const int j = ee >> 5;
        const float d = h2f_bits((uint32_t)blk[34 * j] | ((uint32_t)blk[34 * j + 1] << 8));
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = (float)(int8_t)blk[34 * j + 2 + (ee & 31) + i] * d;
    } else if (type == T_Q4_K || type == T_Q5_K) {  // qwen_cpu/quants.h:53-94
        const float d = h2f_bits((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
        const float dmin = h2f_bits((uint32_t)blk[2] | ((uint32_t)blk[3] << 8));
        const int g = ee >> 6, h = (ee >> 5) & 1, l = ee & 31;
        int sc, m;
        scale_min_k4(2 * g + h, blk + 4, sc, m);
        const int qs0 = type == T_Q5_K ? 48 : 16;
        const float d1 = d * (float)sc, m1 = dmin * (float)m;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int q = (blk[qs0 + 32 * g + l + i] >> (4 * h)) & 0xF;
            if (type == T_Q5_K) q |= ((blk[16 + l + i] >> (2 * g + h)) & 1) << 4;
            o[i] = d1 * (float)q - m1;
        }
    } else {  // Q6_K, qwen_cpu/quants.h:96-121
        const float d = h2f_bits((uint32_t)blk[208] | ((uint32_t)blk[209] << 8));
        const int n = ee >> 7, s = (ee >> 5) & 3, l = ee & 31;
        const int sc = (int8_t)blk[192 + (ee >> 4)];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int lo = (blk[64 * n + 32 * (s & 1) + l + i] >> (s >= 2 ? 4 : 0)) & 0xF;
            const int hi = (blk[128 + 32 * n + l + i] >> (2 * s)) & 3;
            o[i] = (d * (float)sc) * (float)((lo | (hi << 4)) - 32);
        }
    }
    return o;
}

__global__ __launch_bounds__(64) void k_embed(const uint8_t* __restrict__ w, int type, int layout, int k, int n,
                                              uint64_t rb, const int32_t* __restrict__ tokens,
                                              const uint8_t* __restrict__ mask, const float* __restrict__ embd,
                                              float* __restrict__ x) {
    __shared__ __align__(16) uint8_t blk[Q8_COL_BYTES];
    const int sb = blockIdx.x, t = blockIdx.y, lane = threadIdx.x, nsb = k / 256;
    const size_t e0 = (size_t)t * k + 256 * (size_t)sb + 4 * lane;  // this lane's four outputs
    if (mask && mask[t]) {
        *(f4*)(x + e0) = *(const f4*)(embd + e0);
        return;
    }
    const int row = tokens[t];
    if ((unsigned)row >= (unsigned)n) {
        const float q = __builtin_nanf("");
        *(f4*)(x + e0) = f4{q, q, q, q};
        return;
    }
    if (type == T_F32) {  // rows as stored (qwen_cpu/quants.h:193-203); GGUF layout only
        *(f4*)(x + e0) = *(const f4*)(w + (uint64_t)row * rb + 4 * (256 * (uint64_t)sb + 4 * lane));
        return;
    }
    const int bs = sb_bytes(type);
    const uint8_t* base = layout == LAYOUT_GGUF ? w + (uint64_t)row * rb + (uint64_t)sb * bs
                                                : w + ((uint64_t)(row >> 4) * nsb + sb) * (uint64_t)(16 * bs);
    uint8_t v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {  // bytes 4 lane + i and 256 + 4 lane + i - 4 of the block
        const int p = i < 4 ? 4 * lane + i : 256 + 4 * lane + i - 4;
        v[i] = p < bs ? base[layout == LAYOUT_GGUF ? p : t16_dst(type, row & 15, p)] : 0;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int p = i < 4 ? 4 * lane + i : 256 + 4 * lane + i - 4;
        if (p < bs) blk[p] = v[i];
    }
    __syncthreads();
    *(f4*)(x + e0) = dq4_block(blk, type, 4 * lane);
}

// ---------------------------------------------------------------- synthetic blocks
__device__ inline uint64_t mix64(uint64_t z) {  // splitmix64 finaliser, qwen_cpu/qwen.cpp:314-319
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}
__device__ inline uint64_t sm_at(uint64_t seed, uint64_t i) { return mix64(seed + (i + 1) * 0x9e3779b97f4a7c15ULL); }
// fp16 bits of 0 <= f < 65504, rounded to nearest even in integer arithmetic: the device's float ->
// half conversion was measured to round a few fp16-subnormal results (about 1 in 2000 of the
// generator's d values) to the other neighbour.  Normal results have unit 2^(e-10), subnormal ones
// 2^-24; a carry out of the mantissa moves to the next binade by itself.
__device__ inline uint16_t f16_bits(float f) {
    const uint32_t x = __builtin_bit_cast(uint32_t, f);
    const int e = (int)(x >> 23) - 127;
    if (e < -25) return 0;
    const uint32_t mant = (x & 0x7FFFFFu) | 0x800000u;
    const int shift = e >= -14 ? 13 : -e - 1;  // 13 .. 24
    uint32_t q = mant >> shift;
    const uint32_t rem = mant & ((1u << shift) - 1), half = 1u << (shift - 1);
    if (rem > half || (rem == half && (q & 1))) q++;
    return e >= -14 ? (uint16_t)(((uint32_t)(e + 15) << 10) + q - 1024) : (uint16_t)q;
}

// One thread per output byte of the GGUF block stream; byte i of the fill (counted from block0) is
// handled by the launch whose window [off, off + nb) contains it.
__global__ __launch_bounds__(256) void k_synth(uint8_t* __restrict__ dst, int type, uint64_t seed, uint64_t block0,
                                               uint64_t off, uint64_t nb) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nb) return;
    const uint64_t i = off + t;
    const int bs = sb_bytes(type);
    const uint64_t blk = block0 + i / bs;
    const int p = (int)(i % bs);
    uint8_t v;
    if (type == T_Q8_0) {  // per 34-byte block j of the run: d = fp16_rne(u24 * 0.01f), then qs[32]
        const int j = p / 34, pb = p - 34 * j;
        const uint64_t base = (blk * 8 + j) * 33;
        if (pb < 2) {
            const uint16_t h = f16_bits((float)(sm_at(seed, base) >> 40) * (1.0f / 16777216.0f) * 0.01f);
            v = (uint8_t)(h >> (8 * pb));
        } else {
            v = (uint8_t)(sm_at(seed, base + 1 + (pb - 2)) >> 56);
        }
    } else if (type == T_Q5_K) {  // d, dmin = fp16_rne(u24 * 0.01f), then scales, qh, qs bytes
        const uint64_t base = blk * 174;
        if (p < 4) {
            const uint64_t r = sm_at(seed, base + (p >> 1));
            const uint16_t h = f16_bits((float)(r >> 40) * (1.0f / 16777216.0f) * 0.01f);
            v = (uint8_t)(h >> (8 * (p & 1)));
        } else {
            v = (uint8_t)(sm_at(seed, base + 2 + (p - 4)) >> 56);
        }
    } else if (type == T_Q4_K) {
        const uint64_t base = blk * 142;
        if (p < 4) {
            const uint64_t r = sm_at(seed, base + (p >> 1));
            const uint16_t h = f16_bits((float)(r >> 40) * (1.0f / 16777216.0f) * 0.01f);
            v = (uint8_t)(h >> (8 * (p & 1)));
        } else {
            v = (uint8_t)(sm_at(seed, base + 2 + (p - 4)) >> 56);
        }
    } else {
        const uint64_t base = blk * 209;
        if (p < 192) {
            v = (uint8_t)(sm_at(seed, base + p) >> 56);
        } else if (p < 208) {
            v = (uint8_t)(int8_t)((int)(sm_at(seed, base + p) % 64) - 32);
        } else {
            const uint64_t r = sm_at(seed, base + 208);
            const uint16_t h = f16_bits((float)(r >> 40) * (1.0f / 16777216.0f) * 0.005f);
            v = (uint8_t)(h >> (8 * (p & 1)));
        }
    }
    dst[i] = v;
}

}  // namespace

template <int TYPE>
static void launch_repack_type(const uint8_t* src, uint8_t* dst, int nsb, int n, int dir, hipStream_t s) {
    int sbs = 1;  // super-blocks per chunk, see REPACK_SBS
    while (sbs < REPACK_SBS && (long long)nsb * (n / 16) > 1152ll * sbs) sbs *= 2;
    const dim3 grid((nsb + sbs - 1) / sbs, n / 16);
    if (dir == 0) hipLaunchKernelGGL((k_repack<TYPE, true>), grid, dim3(256), 0, s, src, dst, nsb);
    else hipLaunchKernelGGL((k_repack<TYPE, false>), grid, dim3(256), 0, s, src, dst, nsb);
}

int launch_repack(const uint8_t* src, uint8_t* dst, int type, int k, int n, int dir, hipStream_t s) {
    if (type == T_Q4_K) launch_repack_type<T_Q4_K>(src, dst, k / 256, n, dir, s);
    else if (type == T_Q5_K) launch_repack_type<T_Q5_K>(src, dst, k / 256, n, dir, s);
    else if (type == T_Q6_K) launch_repack_type<T_Q6_K>(src, dst, k / 256, n, dir, s);
    else if (type == T_Q8_0) launch_repack_type<T_Q8_0>(src, dst, k / 256, n, dir, s);
    else return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_dequant(const uint8_t* w, int type, int layout, int k, int n, uint64_t rb, const int32_t* rows, int nrows,
                   float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_dequant, dim3(nrows), dim3(256), 0, s, w, type, layout, k, n, rb, rows, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_embed(const uint8_t* w, int type, int layout, int k, int n, uint64_t rb, const int32_t* tokens,
                 const uint8_t* mask, const float* embd, int m, float* x, hipStream_t s) {
    constexpr int MAXY = 65535;  // tokens per launch (the grid's second dimension)
    for (int t0 = 0; t0 < m; t0 += MAXY) {
        const int mt = m - t0 < MAXY ? m - t0 : MAXY;
        hipLaunchKernelGGL(k_embed, dim3(k / 256, mt), dim3(64), 0, s, w, type, layout, k, n, rb, tokens + t0,
                           mask ? mask + t0 : nullptr, embd ? embd + (size_t)t0 * k : nullptr, x + (size_t)t0 * k);
        if (hipGetLastError() != hipSuccess) return -1;
    }
    return 0;
}

int launch_synth(uint8_t* dst, int type, uint64_t seed, uint64_t block0, uint64_t nblocks, hipStream_t s) {
    const uint64_t nbytes = nblocks * sb_bytes(type);
    const uint64_t chunk = 1ull << 30;  // bytes per launch: 4M work-groups of 256 threads
    for (uint64_t off = 0; off < nbytes; off += chunk) {
        const uint64_t nb = nbytes - off < chunk ? nbytes - off : chunk;
        hipLaunchKernelGGL(k_synth, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, dst, type, seed, block0,
                           off, nb);
        if (hipGetLastError() != hipSuccess) return -1;
    }
    return 0;
}

}  // namespace qk
