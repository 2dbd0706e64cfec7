// Quantized GEMM for many tokens (prefill) on gfx950:
//   y[t][m] = sum_k W[m][k] * x[t][k],  t < rows, m < M
// with W a K-quant GGML tensor. Reference: the same product is
// matmul_dispatch (src/cuda/matmul_q4.cu:140-167,185-207) called once per
// token; batched, it is a contraction for the matrix cores.
//
// Below 16 tokens all operands are fp32 (gemm_f32). From there on x enters as two
// fp16 parts: a prep kernel (gemm_few itself) scales each token row by a power of two,
// v = x * 2^e with max |v| in [2^14, 2^15), and splits it into two fp16 parts
// v = h + l (h = fp16(v), l = fp16(v - h)): |v - h - l| <= 2^-22 |v|, or 2^-25
// absolute below 2^-18 of the row's largest, so the sums below carry an fp32
// dot product's accuracy unless they come from such elements alone. The weights enter as exact small integers:
//   Q4_K: B = q * sc (q 0..15, sc 0..63: at most 945, exact in fp16), so the
//         MFMA accumulator sums a whole 256-element block across its eight
//         scale groups, and per block
//         y += d * P_block - dmin * sum_g m_g S_g        (P = sum (q sc) v)
//         with S_g the group sums of v; the min terms are one fp16 MFMA per
//         tile and block (v_mfma_f32_16x16x16_f16, k = 8 groups x 2 parts):
//         m_g exact, S_g 2^-5 split into two fp16 parts like x (22 bits).
//   Q6_K: (q - 32) * sc reaches 12 bits, so B = Bh + Bl (exact, |Bl| <= 1) and
//         three products per operand pair, h Bh + l Bh + h Bl (l Bl is below
//         2^-22 of h Bh).
// The result is scaled back by 2^-e (exact). Products of fp16 values are exact
// in the MFMA's fp32 accumulation, so the roundings are those of an fp32 sum.
//
// fp16 operands are built from bits: a byte b under 0x64 is the fp16 1024 + b,
// so one and-or places two quants and one packed fused multiply-add with sc
// and -1024 sc leaves q * sc (Q4_K; a shift more for every second pair). The
// pairs are bytes (0, 2) and (1, 3) of a word; x is stored in that order.
//
// Five kernels, by token count (gemm_path below has the lines and both sides'
// times): gemm_f32 below 16 tokens; gemm_few (16 tokens, up to 128 where 4 does not
// divide the blocks of a row, up to 160 from K = 4096) converts x itself and splits
// K over its waves; gemm_kquant splits K in 4, 2 or no slices over waves of a
// workgroup with the tile shape that fills the 256 CUs in the fewest rounds;
// gemm_q4k_wide and gemm_q6k_wide (128 x 256 tiles) take long prompts.
// Measured, us for the GDN layer's input projections (M = 8192, 4096, 32, 32 at
// K = 2048, one call) and output projection (M = 2048 at K = 4096), Q4_K:
//   tokens                            9        77        300       777      4096
//   one form for all (before)     103 / 30  71 / 131  77 / 134  146 / 136  510 / 175
//   these kernels                  16 / 10  31 /  21  56 /  42  132 /  62  410 / 152
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <utility>

#include "capi_common.hpp"
#include "device_common.hpp"
#include "ggml_common.hpp"
#include "launch_rules.hpp"

namespace qk {
namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kGemmMinRows = 16;   // fewer tokens need no workspace
constexpr int kGemmMaxRows = 65535 * 128;

// Matrices of one launch (all of one K-quant type, one x): workgroup column
// c in [start[j], start[j+1]) works on matrix j's rows from
// (column - start[j]) * the tile's rows.
constexpr int kGemmJobs = 8;
struct GemmJobs {
    const uint8_t* w[kGemmJobs];
    float* y[kGemmJobs];
    uint64_t ub0[kGemmJobs];   // first block of row 0
    int M[kGemmJobs];
    int start[kGemmJobs + 1];
    int n;
};

struct GemmJob {
    const uint8_t* w;
    float* y;
    uint64_t ub0;
    int M, mb;
};

__device__ __forceinline__ GemmJob gemm_job(const GemmJobs& jobs, int bx) {
    int j = 0;
    while (j + 1 < jobs.n && bx >= jobs.start[j + 1]) ++j;
    return GemmJob{jobs.w[j], jobs.y[j], jobs.ub0[j], jobs.M[j], bx - jobs.start[j]};
}

// Workspace: per token the exponent e, the group sums of v per 32 elements and
// the fp16 parts [T][K/32][2][32].
inline size_t ws_align(size_t b) { return (b + 255) & ~size_t{255}; }
inline size_t ws_exp_bytes(int T) { return ws_align(4 * static_cast<size_t>(T)); }
inline size_t ws_sum_bytes(int T, int K) { return ws_align(4 * static_cast<size_t>(T) * (K / 32)); }
inline size_t ws_bytes(int T, int K) { return ws_exp_bytes(T) + ws_sum_bytes(T, K) + 4 * static_cast<size_t>(T) * K; }

__device__ __forceinline__ float wave_max_abs(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ uint32_t half_bits_of(float v) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
}

// Exponent slot of a token row holding an infinity: the fp16 split cannot carry
// it (h = inf, l = inf - inf = NaN would turn the whole output row into NaN),
// so the GEMM evaluates that row's outputs per element instead.
constexpr int kRowNonFinite = 0x7fffffff;

// e for a row whose largest |x| is m (NaN is ignored by the max; a NaN row's
// outputs are NaN either way): zero rows unscaled, rows with an infinity marked.
__device__ __forceinline__ int prep_exponent(float m) {
    if (!(m <= FLT_MAX)) return kRowNonFinite;
    int e = 0;
    if (m > 0.f) {
        int em;
        frexpf(m, &em);   // m in [2^(em-1), 2^em)
        e = 15 - em;
    }
    return e;
}

// y for (token row x, weight row at element `base`) when x holds an infinity:
// the reference's per-element fp32 products and sum (src/cuda/matmul_q4.cu:
// 140-167), so inf * w, 0 * inf = NaN and +inf + -inf = NaN give the same
// pattern of infinities and NaNs as its GEMV.
__device__ float row_dot_per_element(const uint8_t* __restrict__ w, int type, uint64_t base,
                                     const float* __restrict__ x, int K) {
    float s = 0.f;
    for (int k = 0; k < K; ++k) s = __builtin_fmaf(dequant_elem(w, type, base + k), x[k], s);
    return s;
}

__device__ __forceinline__ float max_abs4(float m, const float4& v) {
    return fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
}

// ------------------------------------------------------------------ x in fragment order
// A token tile is 16 tokens (the last one of a call T % 16, r of them); a block's 256 elements are 8 MFMA
// depths of 32. Lane (lr, lk) = (token or weight row, k group) of depth s = 2 u + j takes the 8 elements
//   128 (lk / 2) + 32 u + 16 (lk % 2) + 8 j + (0, 2, 1, 3, 4, 6, 5, 7)
// of its row, for x and for the weights alike: a lane's share of a weight block is then whole 16-byte pieces
// (Q4_K 2, Q6_K 3), and the order within 8 is the one in which pairs of quants leave a word (below).
// The fp16 parts of a tile are stored fragment by fragment, [block][depth][part][lk][lr] x 16 bytes, so that a
// wave's load of one A operand is 1 KB in a row.
constexpr int kTile = 16;

__device__ __forceinline__ size_t tile_base(int tile, int K) { return static_cast<size_t>(tile) * kTile * K * 4; }

// The fp16 parts of 8 values times 2^e, in the operand's order (packed pairs), and the sum of the scaled values.
__device__ __forceinline__ float split8(const float4& a, const float4& b, int e, uint32_t (&hi)[4], uint32_t (&lo)[4]) {
    const float f[8] = {ldexpf(a.x, e), ldexpf(a.y, e), ldexpf(a.z, e), ldexpf(a.w, e),
                        ldexpf(b.x, e), ldexpf(b.y, e), ldexpf(b.z, e), ldexpf(b.w, e)};
    uint32_t h[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const _Float16 hh = static_cast<_Float16>(f[i]);
        h[i] = __builtin_bit_cast(uint16_t, hh);
        l[i] = half_bits_of(f[i] - static_cast<float>(hh));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = 4 * (i >> 1) + (i & 1);
        hi[i] = h[k] | (h[k + 2] << 16);
        lo[i] = l[k] | (l[k + 2] << 16);
    }
    return ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
}

// One workgroup of 16 waves per token tile, wave = token; 512 elements (a chunk of 8 per lane) per round. Each
// lane's two 16-byte pieces go to the round's LDS image of the fragments (slot lr ^ (chunk % 16) of its 16, so
// neither side conflicts) and the workgroup writes the image out in order.
// NIT > 0: K == 512 NIT, the row is held in registers (read once); NIT == 0: any K % 256 == 0, read twice.
// gridDim.y is 1 or the number of rounds: then each workgroup still takes its rows' maxima over all of K, but splits
// and writes round blockIdx.y alone. A short prompt's rounds are a serial chain on a few CUs (5 workgroups at 77
// tokens): prep and a 256-row product at 77 tokens 18.4 -> 16.5 us (K = 2048), at 300 46.1 -> 45.0, at 300 and K = 4096
// 40.3 -> 37.3. The lines of the launch say where it stops paying.
template <int NIT>
__global__ __launch_bounds__(1024) void gemm_prep_x(const float* __restrict__ x, int* __restrict__ ex,
                                                    float* __restrict__ sx, uint8_t* __restrict__ xp, int T, int K) {
    __shared__ __align__(16) uint4 img[2][2048];
    const int wv = wave_in_block(), lane = threadIdx.x & 63;
    const int t = blockIdx.x * kTile + wv;
    const int r = min(kTile, T - static_cast<int>(blockIdx.x) * kTile);   // tokens of this tile
    const bool live = wv < r;
    const float* row = x + static_cast<size_t>(live ? t : T - 1) * K;
    const int nst = K >> 5, nit = NIT ? NIT : (K + 511) >> 9;
    float m = 0.f;
    float4 v[NIT ? 2 * NIT : 2];
    auto load = [&](int it, float4* d) {   // the lane's 8 elements of round `it` (zero past K)
        const int k = 512 * it + 8 * lane;
        const bool in = NIT || k < K;
        d[0] = in ? ld4(row + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        d[1] = in ? ld4(row + k + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    if constexpr (NIT > 0) {
#pragma unroll
        for (int it = 0; it < NIT; ++it) load(it, v + 2 * it);
#pragma unroll
        for (int i = 0; i < 2 * NIT; ++i) m = max_abs4(m, v[i]);
    } else {
        for (int it = 0; it < nit; ++it) {
            load(it, v);
            m = max_abs4(max_abs4(m, v[0]), v[1]);
        }
    }
    const int e = prep_exponent(wave_max_abs(m));
    if (live && lane == 0 && blockIdx.y == 0) ex[t] = e;
    const int es = e == kRowNonFinite ? 0 : e;   // a marked row's parts are not used
    uint8_t* out = xp + tile_base(blockIdx.x, K);
    const int c16 = lane & 15;                                             // chunk % 16 = 4 u + 2 (lk % 2) + j
    const int frag = ((lane >> 5) * 8 + 2 * (c16 >> 2) + (c16 & 1)) * 2;   // of part 0: (block of the round, depth)
    const int lk = 2 * ((lane >> 4) & 1) + ((c16 >> 1) & 1);
    const int slot = (frag * 4 + lk) * 16 + (wv ^ c16);
    auto round = [&](int it, const float4* d) {
        uint32_t h[4], l[4];
        float s = split8(d[0], d[1], es, h, l);
        uint4* im = img[it & 1];
        im[slot] = make_uint4(h[0], h[1], h[2], h[3]);
        im[slot + 64] = make_uint4(l[0], l[1], l[2], l[3]);
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        const int k = 512 * it + 8 * lane;
        if (live && (lane & 3) == 0 && (NIT || k < K)) sx[static_cast<size_t>(t) * nst + (k >> 5)] = s;
        __syncthreads();
        // 2048 pieces of the image: piece p = (fragment p / 64, lane (lk, lr) = p % 64)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int p = threadIdx.x + 1024 * i;
            const int f2 = p >> 6, k4 = (p >> 4) & 3, lr = p & 15;
            const int dep = (f2 >> 1) & 7;   // 2 u + j
            const int cc = 4 * (dep >> 1) + 2 * (k4 & 1) + (dep & 1);
            if (lr < r && (NIT || 512 * it + 256 * (f2 >> 4) < K))
                st16(out + 16 * (static_cast<size_t>((32 * it + f2) * 4 + k4) * r + lr), im[(p & ~15) + (lr ^ cc)]);
        }
    };
    if constexpr (NIT > 0) {
#pragma unroll
        for (int it = 0; it < NIT; ++it)
            if (gridDim.y == 1 || it == static_cast<int>(blockIdx.y)) round(it, v + 2 * it);
    } else {
        for (int it = 0; it < nit; ++it) {
            if (gridDim.y != 1 && it != static_cast<int>(blockIdx.y)) continue;
            load(it, v);
            round(it, v);
        }
    }
}

// ------------------------------------------------------------------ the GEMM
__device__ __forceinline__ f16x2_t h2(uint32_t w) { return __builtin_bit_cast(f16x2_t, w); }
__device__ __forceinline__ uint32_t w2(f16x2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f16x2_t fma2(f16x2_t a, f16x2_t b, f16x2_t c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ f16x2_t dup2(float v) {
    const _Float16 h = static_cast<_Float16>(v);
    return f16x2_t{h, h};
}

// 16 bytes at a 2-byte aligned address (gfx950 global loads take any byte
// alignment; Q6_K blocks are 210 bytes).
__device__ __forceinline__ uint4 ldg16_a2(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 16);
    return v;
}
__device__ __forceinline__ uint2 ldg8_a2(const uint8_t* p) {
    uint2 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 8);
    return v;
}

// A lane's share of one block of its weight row (the mapping above). Q4_K, element i of a block
// (src/cuda/matmul_q4.cu:76-96): qs byte 16 + 32 (i / 64) + i % 32, low nibble if i % 64 < 32, scale i / 32:
// q[g] holds the bytes of depths u = 2 g, 2 g + 1 (both nibbles), hd the 16-byte header. Q6_K
// (src/cuda/matmul_q4.cu:105-126): ql byte 64 (i / 128) + 32 ((i % 128) / 32 & 1) + i % 32, low nibble in quarters
// 0, 1 of a half, qh byte 128 + 32 (i / 128) + i % 32 bits 2 quarter, scale byte 192 + i / 16, d at 208: q[0], q[1]
// the ql bytes of even and odd u, qh, the half's 8 scales and d.
template <int TYPE>
struct WBlock;
template <>
struct WBlock<kQ4_K> {
    uint4 q[2], hd;
    __device__ __forceinline__ void load(const uint8_t* base, uint32_t row, int lk) {
        const uint32_t o = row + 16u + 64u * (lk >> 1) + 16u * (lk & 1);
        hd = ld16(base + row);
        q[0] = ld16(base + o);
        q[1] = ld16(base + (o + 32u));
    }
};
template <>
struct WBlock<kQ6_K> {
    uint4 q[2], qh;
    uint2 sc;
    uint16_t d;
    __device__ __forceinline__ void load(const uint8_t* base, uint32_t row, int lk) {
        const uint32_t h = lk >> 1, l = lk & 1, o = row + 64u * h + 16u * l;
        q[0] = ldg16_a2(base + o);
        q[1] = ldg16_a2(base + (o + 32u));
        qh = ldg16_a2(base + (row + 128u + 32u * h + 16u * l));
        sc = ldg8_a2(base + (row + 192u + 8u * h));
        d = *reinterpret_cast<const uint16_t*>(base + (row + 208u));
    }
};

__device__ __forceinline__ uint32_t word_of(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Scale of depth u of the lane's half-block, as the fp16 operands need it.
template <int TYPE>
struct WScale;
template <>
struct WScale<kQ4_K> {
    f16x2_t s, c;   // q sc = fma(1024 + q, sc, -1024 sc); high nibbles fma(1024 + 16 q, sc / 16, -64 sc): exact
    template <int U>
    __device__ __forceinline__ void set(const WBlock<kQ4_K>& b, int lk) {
        // scale_min_k4 (src/cuda/matmul_q4.cu:18-26): group 4 (lk / 2) + U
        const uint32_t lo = (b.hd.y >> (8 * U)) & 63u;
        const uint32_t hi = ((b.hd.w >> (8 * U)) & 15u) | ((b.hd.y >> (8 * U + 2)) & 0x30u);
        from<U>((lk & 2) ? hi : lo);
    }
    // (q - 8) sc = fma(16 + q, sc, -24 sc), exact
    template <int U>
    __device__ __forceinline__ void set_centred(const WBlock<kQ4_K>& b, int lk) {
        const uint32_t lo = (b.hd.y >> (8 * U)) & 63u;
        const uint32_t hi = ((b.hd.w >> (8 * U)) & 15u) | ((b.hd.y >> (8 * U + 2)) & 0x30u);
        s = h2(((lk & 2) ? hi : lo) * 0x00010001u + 0x64006400u) - dup2(1024.f);
        c = s * dup2(-24.f);
    }
    template <int U>
    __device__ __forceinline__ void from(uint32_t v) {
        const f16x2_t sc = h2(v * 0x00010001u + 0x64006400u) - dup2(1024.f);   // exact
        s = (U & 1) ? sc * dup2(0.0625f) : sc;
        c = sc * ((U & 1) ? dup2(-64.f) : dup2(-1024.f));
    }
};
template <>
struct WScale<kQ6_K> {
    f16x2_t s;
    template <int U>
    __device__ __forceinline__ void set(const WBlock<kQ6_K>& b, int lk) {
        const uint32_t w = U < 2 ? b.sc.x : b.sc.y;   // scales 2 U, 2 U + 1 of the half
        s = from((w >> (16 * (U & 1) + 8 * (lk & 1))) & 0xffu);
    }
    static __device__ __forceinline__ f16x2_t from(uint32_t byte) {
        return h2((byte ^ 0x80u) * 0x00010001u + 0x64006400u) - dup2(1152.f);   // signed 8 bits, exact
    }
};

// B operand(s) of depth (U, J). Bits 0x64bb are the fp16 1024 + bb, so quants placed under 0x64 by one and-or
// become exact small integers by one packed add or fused multiply-add.
template <int U, int J>
__device__ __forceinline__ void decode_q4(const uint4& q, const WScale<kQ4_K>& sc, uint32_t k64, f16x8_t (&B)[1]) {
    constexpr uint32_t mask = (U & 1) ? 0x00f000f0u : 0x000f000fu;
    uint32_t e[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t w = word_of(q, 2 * J + i);
        e[2 * i] = w2(fma2(h2((w & mask) | k64), sc.s, sc.c));
        e[2 * i + 1] = w2(fma2(h2(((w >> 8) & mask) | k64), sc.s, sc.c));
    }
    __builtin_memcpy(&B[0], e, 16);
}

template <int U, int J>
__device__ __forceinline__ void decode(const WBlock<kQ4_K>& b, const WScale<kQ4_K>& sc, uint32_t k64, f16x8_t (&B)[1]) {
    decode_q4<U, J>(b.q[U >> 1], sc, k64, B);
}

// (q - 8) sc: a nibble in the top four mantissa bits under 0x4c00 is the fp16 16 + q.
template <int U, int J>
__device__ __forceinline__ void decode_centred(const WBlock<kQ4_K>& b, const WScale<kQ4_K>& sc, f16x8_t (&B)[1]) {
    constexpr int lo = (U & 1) ? 2 : 6, hi = (U & 1) ? 6 : 2;   // left shift of bytes 0, 2; right shift of bytes 1, 3
    uint32_t e[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t w = word_of(b.q[U >> 1], 2 * J + i);
        e[2 * i] = w2(fma2(h2(((w << lo) & 0x03c003c0u) | 0x4c004c00u), sc.s, sc.c));
        e[2 * i + 1] = w2(fma2(h2(((w >> hi) & 0x03c003c0u) | 0x4c004c00u), sc.s, sc.c));
    }
    __builtin_memcpy(&B[0], e, 16);
}

// (q - 32) sc in two fp16 parts, exactly: magnitudes up to 2048 fit the first one. wd, hd: the ql and qh words of the
// operand's quants.
template <int U>
__device__ __forceinline__ void decode_q6(const uint32_t (&wd)[2], const uint32_t (&hd)[2], f16x2_t s, uint32_t k64,
                                          uint32_t kf, uint32_t k30, f16x8_t (&B)[2]) {
    f16x2_t q[4], p[4];
    uint32_t e[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // bytes (0, 2), (1, 3) of both words
        const int o = i & 1;
        constexpr int up = 4 - 2 * U;   // bits 2 U of qh to bits 4, 5
        const int sh = up - 8 * o;
        const uint32_t h = hd[i >> 1];
        uint32_t t = ((sh >= 0 ? h << (sh & 31) : h >> (-sh & 31)) & k30) | k64;
        asm("" : "+v"(t));   // two v_and_or_b32 rather than two ands and an or3
        q[i] = h2(((wd[i >> 1] >> (8 * o + 4 * (U >> 1))) & kf) | t) - dup2(1056.f);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        p[i] = q[i] * s;
        e[i] = w2(p[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) l[i] = w2(fma2(q[i], s, -p[i]));
    __builtin_memcpy(&B[0], e, 16);
    __builtin_memcpy(&B[1], l, 16);
}

template <int U, int J>
__device__ __forceinline__ void decode(const WBlock<kQ6_K>& b, const WScale<kQ6_K>& sc, uint32_t k64, f16x8_t (&B)[2]) {
    const uint32_t wd[2] = {word_of(b.q[U & 1], 2 * J), word_of(b.q[U & 1], 2 * J + 1)};
    const uint32_t hd[2] = {word_of(b.qh, 2 * J), word_of(b.qh, 2 * J + 1)};
    decode_q6<U>(wd, hd, sc.s, k64, 0x000f000fu, 0x00300030u, B);
}

// Q4_K's min terms, sum_g m_g S_g of a block, as one v_mfma_f32_16x16x16_f16 per tile: k = 8 groups x the two fp16
// parts of S_g 2^-5 (|S_g| < 2^20) against m_g twice. Lane (lr, lk): groups 2 lk, 2 lk + 1 of token (row) lr.
__device__ __forceinline__ f16x4_t min_operand(const float2& v) {
    const float s0 = v.x * 0.03125f, s1 = v.y * 0.03125f;
    const _Float16 a0 = static_cast<_Float16>(s0), a1 = static_cast<_Float16>(s1);
    return f16x4_t{a0, static_cast<_Float16>(s0 - static_cast<float>(a0)), a1,
                   static_cast<_Float16>(s1 - static_cast<float>(a1))};
}
__device__ __forceinline__ f16x4_t min_weights(const uint4& h, int lk) {
    const uint32_t sh = 16u * (lk & 1);
    const uint32_t l = (h.z >> sh) & 0x3f3fu;
    const uint32_t g = ((h.w >> (sh + 4)) & 0x0f0fu) | ((h.z >> (sh + 2)) & 0x3030u);
    const uint32_t m = lk < 2 ? l : g;
    const f16x2_t p = h2(((m & 0xffu) | ((m >> 8) << 16)) + 0x64006400u) - dup2(1024.f);   // exact
    return f16x4_t{p[0], p[0], p[1], p[1]};
}

// The same form with the block's scales in the place of its minima.
__device__ __forceinline__ f16x4_t scale_weights(const uint4& h, int lk) {
    const uint32_t sh = 16u * (lk & 1);
    const uint32_t l = (h.y >> sh) & 0x3f3fu;
    const uint32_t g = ((h.w >> sh) & 0x0f0fu) | ((h.y >> (sh + 2)) & 0x3030u);
    const uint32_t m = lk < 2 ? l : g;
    const f16x2_t p = h2(((m & 0xffu) | ((m >> 8) << 16)) + 0x64006400u) - dup2(1024.f);   // exact
    return f16x4_t{p[0], p[0], p[1], p[1]};
}

// A workgroup of 8 waves: RW row groups x KW slices of K (RW = 8 / KW); a wave owns 16 WT tokens x 16 WR rows of
// its slice's blocks, as 16 x 16 tiles on v_mfma_f32_16x16x32_f16. A step is two depths (64 elements) of every
// slice. x goes global -> VGPR -> LDS, four step slots deep: step st writes st + 2's fragments (loaded two steps
// earlier), requests st + 4's and reads its own, the next two token tiles' A operands always requested ahead, so
// the one barrier per step finds the first operands of the next step in registers. Weights: a lane loads its share
// of the next block during the current one and decodes it in registers (9 VALU instructions per Q4_K operand of 8
// quants), so no weight passes through LDS and no wave waits for another's decode. A block's products sum into C
// from zero; its epilogue applies the block scales in fp32: Q4_K acc += d C - 32 dmin P_min (P_min above); Q6_K
// acc += d C, with three products per depth, h Bh + l Bh + h Bl (l Bl is below 2^-22 of h Bh).
//
// The sums are over SL slices of K, each in block order, added in slice order: a wave that holds two slices
// (SL = 2 KW) puts the first one's sums by in LDS. So the bits do not depend on KW, WT or WR, and the shape is free
// to follow the launch: at 77 tokens and M = 12352 the 48 x 128 tile (KW = 2, two token blocks, 194 workgroups)
// takes 26 us where 64 x 256 tiles (98 workgroups, the whole of K serially) take 44.
//
// What bounds it: issue. A SIMD's MFMAs, the VALU work of decode and epilogue, LDS reads and the CU's vector
// loads add up rather than overlap (each one's removal took off its own time: of 55 us at 64 x 256, weight loads
// 7, x 8, A operands 8, decode 13); a round of one workgroup per CU is 12-46 us whatever its MFMA work, so the
// rounds are what the shape has to save.
template <int TYPE, int WT, int WR, int KW, int SL>
struct GemmShape {
    static constexpr int RW = 8 / KW, FR = WT * KW * 4, XF = FR / 8, SPW = SL / KW;
    static constexpr int tokens = 16 * WT, rows = 16 * WR * RW;
    static constexpr size_t ring = size_t{4} * FR * 1024, fold = KW > 1 ? size_t{8} * SPW * WT * WR * 1024 : 0;
    static constexpr size_t kept = SPW == 2 ? size_t{8} * WT * WR * 1024 : 0;
    static constexpr size_t lds = ring + kept > fold ? ring + kept : fold;
    static_assert(rows <= kGemmTileRows && FR % 8 == 0 && SPW >= 1 && SPW <= 2 && (KW > 1 || SPW == SL), "shape");
};

// A value the compiler may not fold into its users (keeps v_fmac_f32 from
// becoming v_fma_mix_f32, which issues at half the rate).
__device__ __forceinline__ float opaque(float v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <int S>
using IC = std::integral_constant<int, S>;

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(IC<I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int TYPE, int WT, int WR, int KW, int SL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_kquant(
    const GemmJobs jobs, const int* __restrict__ ex, const float* __restrict__ sx, const uint8_t* __restrict__ xp,
    const float* __restrict__ x, int T, int K) {
    using G = GemmShape<TYPE, WT, WR, KW, SL>;
    constexpr int BB = TYPE == kQ4_K ? 144 : 210, NB = TYPE == kQ4_K ? 1 : 2;
    __shared__ __align__(16) uint8_t smem[G::lds];
    uint4* xs = reinterpret_cast<uint4*>(smem);
    const int cols = jobs.start[jobs.n];
    const int tb = static_cast<int>(blockIdx.x) / cols;
    const GemmJob job = gemm_job(jobs, static_cast<int>(blockIdx.x) - tb * cols);
    float* __restrict__ y = job.y;
    const int M = job.M;
    const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = wave_in_block();
    const int kw = wv / G::RW, rw = wv % G::RW;
    const int nb = K >> 8, nbk = nb / KW, steps = 4 * nbk, nst = K >> 5;
    const int tile0 = tb * WT, tiles = (T + kTile - 1) / kTile;
    const int rw0 = job.mb * G::rows, r0 = rw0 + 16 * WR * rw;
    const uint8_t* wbase = job.w + (job.ub0 + static_cast<uint64_t>(rw0) * nb + static_cast<uint64_t>(kw) * nbk) * BB;
    uint32_t wo[WR];   // the lane's row, from the workgroup's first
#pragma unroll
    for (int rt = 0; rt < WR; ++rt)
        wo[rt] = static_cast<uint32_t>(min(r0 + 16 * rt + lr, M - 1) - rw0) * static_cast<uint32_t>(nb) * BB;

    // this wave's fragments of a step: fragment id -> (slice, tile of the workgroup, (depth, part))
    const uint8_t* xb[G::XF];
    uint32_t xo[G::XF], xstep[G::XF];
#pragma unroll
    for (int i = 0; i < G::XF; ++i) {
        const int id = wv * G::XF + i;
        const int ti = min(tile0 + id / 4 % WT, tiles - 1), ks = id / (4 * WT);
        const int r = min(kTile, T - kTile * ti);
        xb[i] = xp + tile_base(ti, K);
        xo[i] = 16u * static_cast<uint32_t>((ks * nbk * 16 + id % 4) * 4 * r + lk * r + min(lr, r - 1));
        xstep[i] = 256u * r;
    }
    uint4 xr[2][G::XF];
    auto x_load = [&](uint4 (&d)[G::XF], int st) {
#pragma unroll
        for (int i = 0; i < G::XF; ++i) d[i] = ld16(xb[i] + (xo[i] + static_cast<uint32_t>(min(st, steps - 1)) * xstep[i]));
    };
    auto x_store = [&](const uint4 (&d)[G::XF], int slot) {
#pragma unroll
        for (int i = 0; i < G::XF; ++i) xs[(slot * G::FR + wv * G::XF + i) * 64 + lane] = d[i];
    };
    const uint4* as = xs + kw * WT * 4 * 64 + lane;   // this wave's first A fragment of slot 0
    constexpr int PT = WT < 2 ? WT : 2;   // token tiles whose A operands are requested at a time
    f16x8_t An[PT][2];
    auto a_load = [&](f16x8_t (&d)[PT][2], int slot, int j, int t0) {
#pragma unroll
        for (int i = 0; i < PT; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                d[i][p] = *reinterpret_cast<const f16x8_t*>(&as[(slot * G::FR + 4 * min(t0 + i, WT - 1) + 2 * j + p) * 64]);
    };
    auto barrier = []() {   // this wave's LDS stores are done, then the workgroup meets (loads stay in flight)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    f32x4_t acc[WT][WR], C[WT][WR];
#pragma unroll
    for (int tt = 0; tt < WT; ++tt)
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) acc[tt][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    uint32_t k64 = 0x64006400u;   // kept in a register: v_and_or_b32 takes one constant
    asm volatile("" : "+v"(k64));
    WBlock<TYPE> wc[WR], wn[WR];
    WScale<TYPE> sc[WR];
    f16x8_t B[2][WR][NB];
    auto w_load = [&](int b) {   // the lane's share of block b of its rows (the last block again past the end)
        const uint8_t* p = wbase + static_cast<size_t>(min(b, nbk - 1)) * BB;
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) wn[rt].load(p, wo[rt], lk);
    };
    auto w_take = [&]() {
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) wc[rt] = wn[rt];
    };
    auto b_make = [&](auto dI) {   // B operands of depth D of the block in wc
        constexpr int D = decltype(dI)::value;
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) {
            if constexpr ((D & 1) == 0) sc[rt].template set<(D >> 1)>(wc[rt], lk);
            decode<(D >> 1), (D & 1)>(wc[rt], sc[rt], k64, B[D & 1][rt]);
        }
    };
    w_load(0);
    x_load(xr[0], 0);
    x_load(xr[1], 1);
    w_take();
    w_load(1);
    x_store(xr[0], 0);
    x_load(xr[0], 2);
    x_store(xr[1], 1);
    x_load(xr[1], 3);
    b_make(IC<0>{});
    barrier();
    a_load(An, 0, 0, 0);

    f32x4_t* kept = reinterpret_cast<f32x4_t*>(smem + G::ring) + wv * WT * WR * 64 + lane;   // the first slice's sums
    for (int b = 0; b < nbk; ++b) {
        if (G::SPW == 2 && b == nbk / 2) {
#pragma unroll
            for (int tt = 0; tt < WT; ++tt)
#pragma unroll
                for (int rt = 0; rt < WR; ++rt) {
                    kept[(tt * WR + rt) * 64] = acc[tt][rt];
                    acc[tt][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                }
        }
        // the block's epilogue operands
        f16x4_t Bm[WR];
        float dsc[WR], dmn[WR];
        float2 sg[WT];
        if constexpr (TYPE == kQ4_K) {
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) {
                Bm[rt] = min_weights(wc[rt].hd, lk);
                dsc[rt] = opaque(half_bits(wc[rt].hd.x & 0xffffu));
                dmn[rt] = opaque(-32.0f * half_bits(wc[rt].hd.x >> 16));
            }
#pragma unroll
            for (int tt = 0; tt < WT; ++tt) {   // group sums 2 lk, 2 lk + 1 of token lr
                const int t = min((tile0 + tt) * kTile + lr, T - 1);
                sg[tt] = *reinterpret_cast<const float2*>(sx + static_cast<size_t>(t) * nst + 8 * (kw * nbk + b) + 2 * lk);
            }
        } else {
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) dsc[rt] = opaque(half_bits(wc[rt].d));
        }
        static_for<8>([&](auto dI) {
            constexpr int D = decltype(dI)::value, U = D >> 1, J = D & 1;
            const int st = 4 * b + U;
            if constexpr (D == 7) {
                w_take();
                w_load(b + 2);
            }
            if constexpr (J == 0) {
                x_store(xr[U & 1], (U + 2) & 3);
                x_load(xr[U & 1], st + 4);
            }
            __builtin_amdgcn_sched_barrier(0);
            b_make(IC<(D + 1) & 7>{});
            static_for<(WT + 1) / 2>([&](auto pI) {   // pairs of token tiles
                constexpr int P0 = 2 * decltype(pI)::value, PN = P0 + 2 <= WT ? 2 : 1;
                f16x8_t A[2][2];
#pragma unroll
                for (int i = 0; i < PN; ++i) {
#pragma unroll
                    for (int p = 0; p < 2; ++p) A[i][p] = An[i][p];
                }
                if constexpr (P0 + 2 < WT)
                    a_load(An, U, J, P0 + 2);
                else
                    a_load(An, J == 0 ? U : (U + 1) & 3, J ^ 1, 0);
#pragma unroll
                for (int i = 0; i < PN; ++i)
#pragma unroll
                    for (int rt = 0; rt < WR; ++rt)   // a block's first depth starts its sums from zero
                        C[P0 + i][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            A[i][0], B[J][rt][0], D == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : C[P0 + i][rt], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < PN; ++i)
#pragma unroll
                    for (int rt = 0; rt < WR; ++rt)
                        C[P0 + i][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i][1], B[J][rt][0], C[P0 + i][rt], 0, 0, 0);
                if constexpr (NB == 2) {
#pragma unroll
                    for (int i = 0; i < PN; ++i)
#pragma unroll
                        for (int rt = 0; rt < WR; ++rt)
                            C[P0 + i][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i][0], B[J][rt][NB - 1], C[P0 + i][rt], 0, 0, 0);
                }
#pragma unroll
                for (int tt = P0; D == 7 && tt < P0 + PN; ++tt) {
                    f16x4_t As;
                    if constexpr (TYPE == kQ4_K) As = min_operand(sg[tt]);
#pragma unroll
                    for (int rt = 0; rt < WR; ++rt) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[tt][rt][i] = __builtin_fmaf(dsc[rt], C[tt][rt][i], acc[tt][rt][i]);
                        if constexpr (TYPE == kQ4_K) {
                            const f32x4_t pm =
                                __builtin_amdgcn_mfma_f32_16x16x16f16(As, Bm[rt], f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[tt][rt][i] = __builtin_fmaf(dmn[rt], pm[i], acc[tt][rt][i]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (J == 1) barrier();
        });
    }

    // lane L holds elements [4 (L / 16) + i][L % 16] of tile (tt, rt): token 4 lk + i, row lr
    auto put = [&](int tt, int rt, const f32x4_t& v) {
        const int row = r0 + 16 * rt + lr;
        if (row >= M) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = (tile0 + tt) * kTile + 4 * lk + i;
            if (t >= T) continue;
            const int et = ex[t];
            y[static_cast<size_t>(t) * M + row] =
                et == kRowNonFinite ? row_dot_per_element(job.w, TYPE, (job.ub0 + static_cast<uint64_t>(row) * nb) * 256,
                                                          x + static_cast<size_t>(t) * K, K)
                                    : ldexpf(v[i], -et);
        }
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int tt = 0; tt < WT; ++tt)
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) put(tt, rt, G::SPW == 2 ? kept[(tt * WR + rt) * 64] + acc[tt][rt] : acc[tt][rt]);
    } else {   // every slice's sums to LDS; wave kw of a row group adds the tiles tt * WR + rt = kw (mod KW)
        f32x4_t* part = reinterpret_cast<f32x4_t*>(smem);   // the ring and the kept sums are done with
        constexpr int tiles_w = WT * WR;
        auto at = [&](int slice, int tile) { return ((slice * G::RW + rw) * tiles_w + tile) * 64 + lane; };
        f32x4_t first[G::SPW == 2 ? tiles_w : 1];
        if constexpr (G::SPW == 2) {
#pragma unroll
            for (int i = 0; i < tiles_w; ++i) first[i] = kept[i * 64];
            barrier();
        }
#pragma unroll
        for (int tt = 0; tt < WT; ++tt)
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) {
                if constexpr (G::SPW == 2) part[at(2 * kw, tt * WR + rt)] = first[tt * WR + rt];
                part[at(G::SPW * kw + G::SPW - 1, tt * WR + rt)] = acc[tt][rt];
            }
        barrier();
#pragma unroll
        for (int tt = 0; tt < WT; ++tt)
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) {
                if ((tt * WR + rt) % KW != kw) continue;
                f32x4_t v = part[at(0, tt * WR + rt)];
#pragma unroll
                for (int sl = 1; sl < SL; ++sl) v += part[at(sl, tt * WR + rt)];
                put(tt, rt, v);
            }
    }
}

// ------------------------------------------------------------------ fewer than 16 tokens
// In fp32 throughout: x enters as it is, the weights as the reference's dequantized values (d sc q - dmin m, or
// d sc (q - 32): exact products and at most one rounding, src/cuda/matmul_q4.cu:76-126), on v_mfma_f32_16x16x4_f32.
// These counts stand in for one fp32 GEMV per token, which keeps x's 24 bits at any magnitude; two fp16 parts with one
// exponent for a token's 2048 elements keep 22, and fewer from 2^-18 of the largest down. Error against 64 bits with
// one channel of weight zero at 1, 1e5 and 1e7 times the others: GEMV 1.0e-7, 1.1e-7, 1.2e-7, the fp16 parts 1.0e-7,
// 3.0e-7, 3.3e-5, this 1.0e-7, 1.1e-7, 1.2e-7 (Q4_K, K = 2048; Q6_K GEMV 1.6e-7, this 1.1e-7). Infinities and NaNs
// need no path of their own.
//
// A workgroup owns 16 WR weight rows; K is split in 8 slices, slice s the blocks s, s + 8, ..., NW waves taking 8 / NW
// slices each. x and weights go straight to the operand registers (no LDS, no barrier before the end); the next
// block's x is requested piece by piece as the current one's is used up. Sums of 16 products from zero, added per
// block, per slice and over the slices as a tree, so the bits do not depend on WR or NW.
//
// What bounds it: the fp32 MFMAs (64 x 32 cycles for 16 rows and a block, 5.2 us at M = 12352, K = 2048 over the whole
// chip) and their operands' decode (18-24 VALU instructions per 8 weights), after 4 us of launch and first loads.
// us at 3 / 9 / 15 tokens, Q4_K, against the fp16 parts (flat over those counts) and a GEMV per token (at 3):
//   M = 32, K = 2048       5.4 / 6.0 / 7.0      6.6    6.8
//   2048 x 4096            9.0 / 9.9 / 11.9     11.2   12.2
//   8192 + 512 + 512       11.8 / 13.6 / 16.1   11.9   14.0
//   12352 in four          14.5 / 15.8 / 17.0   12.1   17.3
// gfx950 has no faster unit that holds 24 bits: three bf16 parts of x (exact) take 6 products of the 16 x 16 x 32 form
// with Q4_K's weights in two parts, and the splitting, and come out equal.
template <int TYPE>
struct WFloat;   // a lane's weights of depth (U, J) as fp32, in element order
template <>
struct WFloat<kQ4_K> {
    uint32_t sc, mn;   // the half's four scales and minima (scale_min_k4, src/cuda/matmul_q4.cu:18-26)
    float d, dmin;
    __device__ __forceinline__ void block(const WBlock<kQ4_K>& b, int lk) {
        d = half_bits(b.hd.x & 0xffffu);
        dmin = half_bits(b.hd.x >> 16);
        sc = lk < 2 ? b.hd.y & 0x3f3f3f3fu : (b.hd.w & 0x0f0f0f0fu) | ((b.hd.y >> 2) & 0x30303030u);
        mn = lk < 2 ? b.hd.z & 0x3f3f3f3fu : ((b.hd.w >> 4) & 0x0f0f0f0fu) | ((b.hd.z >> 2) & 0x30303030u);
    }
    template <int U, int J>
    __device__ __forceinline__ void get(const WBlock<kQ4_K>& b, int, float (&w)[8]) const {
        const float s = d * static_cast<float>(byte_of(sc, U)), m = dmin * static_cast<float>(byte_of(mn, U));   // exact
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t q = (word_of(b.q[U >> 1], 2 * J + i) >> (4 * (U & 1))) & 0x0f0f0f0fu;
            asm("" : "+v"(q));   // four v_cvt_f32_ubyte
#pragma unroll
            for (int k = 0; k < 4; ++k) w[4 * i + k] = __builtin_fmaf(static_cast<float>(byte_of(q, k)), s, -m);
        }
    }
};
template <>
struct WFloat<kQ6_K> {
    float d;
    __device__ __forceinline__ void block(const WBlock<kQ6_K>& b, int) { d = half_bits(b.d); }
    template <int U, int J>
    __device__ __forceinline__ void get(const WBlock<kQ6_K>& b, int lk, float (&w)[8]) const {
        const uint32_t sw = (U < 2 ? b.sc.x : b.sc.y) >> (16 * (U & 1) + 8 * (lk & 1));
        const float s = d * static_cast<float>(static_cast<int8_t>(sw & 0xffu));   // exact
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t q = ((word_of(b.q[U & 1], 2 * J + i) >> (4 * (U >> 1))) & 0x0f0f0f0fu) |
                         (((word_of(b.qh, 2 * J + i) >> (2 * U)) & 0x03030303u) << 4);
            asm("" : "+v"(q));
#pragma unroll
            for (int k = 0; k < 4; ++k) w[4 * i + k] = __builtin_fmaf(static_cast<float>(byte_of(q, k)), s, -32.0f * s);
        }
    }
};

constexpr int kF32Slices = 8;

template <int TYPE, int WR, int NW>
__global__ __launch_bounds__(NW * kWave) void gemm_f32(const GemmJobs jobs, const float* __restrict__ x, int T, int K) {
    constexpr int BB = TYPE == kQ4_K ? 144 : 210, NS = kF32Slices;
    static_assert(NS % NW == 0 && WR <= NW, "shape");
    __shared__ f32x4_t part[NS * WR * kWave];
    const GemmJob job = gemm_job(jobs, static_cast<int>(blockIdx.x));
    float* __restrict__ y = job.y;
    const int M = job.M;
    const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = wave_in_block();
    const int nb = K >> 8;
    const int r0 = job.mb * 16 * WR;
    const uint8_t* wbase = job.w + (job.ub0 + static_cast<uint64_t>(r0) * nb) * BB;
    uint32_t wo[WR];   // the lane's row, from the workgroup's first (the matrix's last again past the end)
#pragma unroll
    for (int rt = 0; rt < WR; ++rt)
        wo[rt] = static_cast<uint32_t>(min(16 * rt + lr, M - 1 - r0)) * static_cast<uint32_t>(nb) * BB;
    WBlock<TYPE> wc[WR];
    auto w_load = [&](int b) {
        const uint8_t* p = wbase + static_cast<size_t>(b) * BB;
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) wc[rt].load(p, wo[rt], lk);
    };
    // token lr (the last one again past the end), the lane's 16 elements of depths 2 u and 2 u + 1
    const float* xl = x + static_cast<size_t>(min(lr, T - 1)) * K + 128 * (lk >> 1) + 16 * (lk & 1);
    float4 v[16];
    auto x_load = [&](int b, int u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * u + i] = ld4(xl + 256 * b + 32 * u + 4 * i);
    };
    if (wv < nb) {
        w_load(wv);
#pragma unroll
        for (int u = 0; u < 4; ++u) x_load(wv, u);
    }
#pragma unroll 1
    for (int sl = wv; sl < NS; sl += NW) {
        f32x4_t tot[WR];
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) tot[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int b = sl; b < nb; b += NS) {
            // the wave's next block: of this slice, or the first of its next one
            const bool same = b + NS < nb;
            const int next = same ? b + NS : sl + NW;
            const bool more = same || (next < NS && next < nb);
            f32x4_t C[2][WR][2], sum[WR];
            WFloat<TYPE> wf[WR];
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) wf[rt].block(wc[rt], lk);
            auto add = [&](int d) {
#pragma unroll
                for (int rt = 0; rt < WR; ++rt) {
                    const f32x4_t c = C[d & 1][rt][0] + C[d & 1][rt][1];
                    sum[rt] = d == 0 ? c : sum[rt] + c;
                }
            };
            static_for<8>([&](auto dI) {
                constexpr int D = decltype(dI)::value, U = D >> 1, J = D & 1;
                const float4 a0 = v[2 * D], a1 = v[2 * D + 1];
                const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
                for (int rt = 0; rt < WR; ++rt) {
                    float w[8];
                    wf[rt].template get<U, J>(wc[rt], lk, w);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        C[J][rt][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            a[i], w[i], i < 2 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : C[J][rt][i & 1], 0, 0, 0);
                }
                if constexpr (J == 1) {
                    if (more) x_load(next, U);
                }
                if constexpr (D > 0) add(D - 1);
            });
            add(7);
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) tot[rt] += sum[rt];
            if (more) w_load(next);
        }
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) part[(sl * WR + rt) * kWave + lane] = tot[rt];
    }
    __syncthreads();
    if (wv >= WR) return;
    auto at = [&](int sl) { return part[(sl * WR + wv) * kWave + lane]; };
    const f32x4_t s = ((at(0) + at(1)) + (at(2) + at(3))) + ((at(4) + at(5)) + (at(6) + at(7)));
    const int mrow = r0 + 16 * wv + lr;
    if (mrow >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * lk + i < T) y[static_cast<size_t>(4 * lk + i) * M + mrow] = s[i];
}

// ------------------------------------------------------------------ a few tokens
// 16 tokens per workgroup and no prep pass: the workgroup converts its tokens' rows itself,
// 2048 elements of K (a round: 8 blocks) at a time, into an LDS image of the fragments (slot lr ^ c of its 16,
// c = 4 u + 2 (lk % 2) + j, so that neither the stores nor the loads conflict), with one exponent per token and
// round. Wave w takes block w of every round for the workgroup's 16 WR rows; its first block's weights are
// requested before the conversion. A round's sums are unscaled (exactly) and added to the wave's totals, and the
// 8 waves' totals are added in wave order through LDS.
//
// The products of x's low parts, 2^-11 of the others, have an accumulator of their own, and Q4_K's quants enter as
// q - 8, so that a block's sum is no larger than its result; the 8 d sum_g sc_g S_g taken out joins the min terms in
// fp32.
template <int TYPE, int WR>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_few(
    const GemmJobs jobs, const float* __restrict__ x, int T, int K) {
    constexpr int BB = TYPE == kQ4_K ? 144 : 210, NB = TYPE == kQ4_K ? 1 : 2;
    __shared__ __align__(16) uint4 xs[8 * 8 * 2 * 64];
    __shared__ __align__(16) float sums[16][64];
    __shared__ int exps[16], bad[16];
    const int cols = jobs.start[jobs.n];
    const int tb = static_cast<int>(blockIdx.x) / cols;
    const GemmJob job = gemm_job(jobs, static_cast<int>(blockIdx.x) - tb * cols);
    float* __restrict__ y = job.y;
    const int M = job.M, t0 = tb * kTile;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = wave_in_block();
    const int nb = K >> 8, rounds = (nb + 7) >> 3;
    const int r0 = job.mb * 16 * WR;
    const uint8_t* wbase = job.w + (job.ub0 + static_cast<uint64_t>(r0) * nb) * BB;
    uint32_t wo[WR];
#pragma unroll
    for (int rt = 0; rt < WR; ++rt)
        wo[rt] = static_cast<uint32_t>(min(16 * rt + lr, M - 1 - r0)) * static_cast<uint32_t>(nb) * BB;
    [[maybe_unused]] uint32_t k64 = 0x64006400u;   // kept in a register: v_and_or_b32 takes one constant
    asm volatile("" : "+v"(k64));
    WBlock<TYPE> wc[WR];
    auto w_load = [&](int b) {
        const uint8_t* p = wbase + static_cast<size_t>(min(b, nb - 1)) * BB;
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) wc[rt].load(p, wo[rt], lk);
    };
    // conversion: 32 threads per token, 8 pieces of 8 elements each
    const int tok = tid >> 5, ch0 = tid & 31;
    const bool live = t0 + tok < T;
    const float* row = x + static_cast<size_t>(live ? t0 + tok : 0) * K;
    float4 v[16];
    auto x_load = [&](int c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = 2048 * c + 256 * i + 8 * ch0;
            const bool in = live && k < K;
            v[2 * i] = in ? ld4(row + k) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[2 * i + 1] = in ? ld4(row + k + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    x_load(0);
    w_load(wv);
    if (tid < 16) bad[tid] = 0;

    f32x4_t tot[WR];
#pragma unroll
    for (int rt = 0; rt < WR; ++rt) tot[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < rounds; ++c) {
        __syncthreads();   // the previous round's fragments have been read
        {
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) m = max_abs4(m, v[i]);
#pragma unroll
            for (int o = 16; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
            const int e = prep_exponent(m);
            if (ch0 == 0) {
                exps[tok] = e == kRowNonFinite ? 0 : e;
                if (e == kRowNonFinite) bad[tok] = 1;   // evaluated per element at the end
            }
            const int es = e == kRowNonFinite ? 0 : e;
            const int c16 = ch0 & 15;                                   // 4 u + 2 (lk % 2) + j
            const int dep = 2 * (c16 >> 2) + (c16 & 1), k4 = 2 * (ch0 >> 4) + ((c16 >> 1) & 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint32_t h[4], l[4];
                const float s0 = split8(v[2 * i], v[2 * i + 1], es, h, l);
                const int slot = ((i * 8 + dep) * 2 * 4 + k4) * 16 + (tok ^ c16);
                xs[slot] = make_uint4(h[0], h[1], h[2], h[3]);
                xs[slot + 64] = make_uint4(l[0], l[1], l[2], l[3]);
                float s = s0 + __shfl_xor(s0, 1);
                s += __shfl_xor(s, 2);
                if ((ch0 & 3) == 0) sums[tok][8 * i + (ch0 >> 2)] = s;
            }
        }
        if (c + 1 < rounds) x_load(c + 1);
        __syncthreads();
        if (8 * c + wv >= nb) continue;   // the whole wave; the next barrier is met at the loop's head
        f32x4_t C[WR], Cl[WR];
        WScale<TYPE> sc[WR];
        const uint4* xw = xs + wv * 8 * 2 * 64 + lk * 16;
        const int sw = lr ^ (2 * (lk & 1));
        f16x8_t A[2][2];
        auto a_load = [&](auto dI) {
            constexpr int D = decltype(dI)::value;
#pragma unroll
            for (int p = 0; p < 2; ++p)
                A[D & 1][p] = *reinterpret_cast<const f16x8_t*>(&xw[(2 * D + p) * 64 + (sw ^ (4 * (D >> 1) + (D & 1)))]);
        };
        a_load(IC<0>{});
        static_for<8>([&](auto dI) {
            constexpr int D = decltype(dI)::value, U = D >> 1, J = D & 1;
            if constexpr (D < 7) a_load(IC<D + 1>{});
#pragma unroll
            for (int rt = 0; rt < WR; ++rt) {
                if constexpr (J == 0) {
                    if constexpr (TYPE == kQ4_K)
                        sc[rt].template set_centred<U>(wc[rt], lk);
                    else
                        sc[rt].template set<U>(wc[rt], lk);
                }
                f16x8_t B[NB];
                if constexpr (TYPE == kQ4_K)
                    decode_centred<U, J>(wc[rt], sc[rt], B);
                else
                    decode<U, J>(wc[rt], sc[rt], k64, B);
                const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
                C[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][0], B[0], D == 0 ? zero : C[rt], 0, 0, 0);
                Cl[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][1], B[0], D == 0 ? zero : Cl[rt], 0, 0, 0);
                if constexpr (NB == 2) Cl[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][0], B[NB - 1], Cl[rt], 0, 0, 0);
            }
        });
        f16x4_t As;
        if constexpr (TYPE == kQ4_K) As = min_operand(*reinterpret_cast<const float2*>(&sums[lr][8 * wv + 2 * lk]));
        int et[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) et[i] = -exps[4 * lk + i];
#pragma unroll
        for (int rt = 0; rt < WR; ++rt) {
            float d, d8 = 0.f, dmn = 0.f;
            f32x4_t pm, ps;
            if constexpr (TYPE == kQ4_K) {
                d = half_bits(wc[rt].hd.x & 0xffffu);
                d8 = 256.0f * d;   // 8 d, and the 2^5 of S 2^-5
                dmn = -32.0f * half_bits(wc[rt].hd.x >> 16);
                const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
                pm = __builtin_amdgcn_mfma_f32_16x16x16f16(As, min_weights(wc[rt].hd, lk), zero, 0, 0, 0);
                ps = __builtin_amdgcn_mfma_f32_16x16x16f16(As, scale_weights(wc[rt].hd, lk), zero, 0, 0, 0);
            } else {
                d = half_bits(wc[rt].d);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float s = d * (C[rt][i] + Cl[rt][i]);
                if constexpr (TYPE == kQ4_K) s += __builtin_fmaf(d8, ps[i], dmn * pm[i]);
                tot[rt][i] += ldexpf(s, et[i]);
            }
        }
        if (c + 1 < rounds) w_load(8 * (c + 1) + wv);
    }
    __syncthreads();
    f32x4_t* part = reinterpret_cast<f32x4_t*>(xs);
#pragma unroll
    for (int rt = 0; rt < WR; ++rt) part[(wv * WR + rt) * 64 + lane] = tot[rt];
    __syncthreads();
    if (wv >= WR) return;
    f32x4_t s = part[wv * 64 + lane];
#pragma unroll
    for (int w = 1; w < 8; ++w) s += part[(w * WR + wv) * 64 + lane];
    const int mrow = r0 + 16 * wv + lr;
    if (mrow >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = t0 + 4 * lk + i;
        if (t >= T) continue;
        y[static_cast<size_t>(t) * M + mrow] =
            bad[4 * lk + i] ? row_dot_per_element(job.w, TYPE, (job.ub0 + static_cast<uint64_t>(mrow) * nb) * 256,
                                                  x + static_cast<size_t>(t) * K, K)
                            : s[i];
    }
}

// ------------------------------------------------------------------ Q4_K, many tokens
// A workgroup (8 waves, one per CU) owns 128 tokens x 256 weight rows; wave w owns rows 64 (w % 4) .. +63 for
// tokens 64 (w / 4) .. +63, as 4 x 4 tiles. Operands arrive through an LDS ring filled by global_load_lds_dwordx4
// (no VGPRs, no LDS store instructions) kQ4Dist depths ahead: x fragments per depth, the quant bytes per half
// block (the 16-byte pieces of depths u = 2 g, 2 g + 1, row by row, which is also the order of a wave's B reads:
// no bank conflicts), headers and group sums per block. Each wave decodes the B operands of its own 64 rows in
// registers, a depth ahead, 9 VALU instructions per operand, and requests the next token tile's A operands before
// the current one's products; each MFMA is followed by two VALU instructions of the decode (the scheduling groups),
// which issue while it runs. Measured at 4096 x 8192 x 2048 and the other three projections, six rounds of 256
// workgroups: 370 us, 230 of them the MFMAs' own time; with the decode shared by wave pairs through LDS (24 VALU instructions
// per operand then) and no A operands ahead 437 us. Without its decode, DMA, A reads or epilogue it takes 72, 54,
// 60 and 37 us less: the parts add up, so fewer instructions is what is left to gain.
constexpr int kQ4Waves = 8;
constexpr int kQ4Block = kQ4Waves * kWave;
constexpr int kQ4R = 256;                   // weight rows per workgroup (64 per wave)
constexpr int kQ4T = 128;                   // tokens per workgroup
constexpr int kQ4Dist = 3;                  // ring distance (depths)
constexpr int kQ4XSlots = 4;                // x slots (one depth each)
typedef uint4 Q4XSlot[kQ4T / kTile][2][kWave];   // one depth of x: [tile][fp16 part][lane]
typedef uint4 Q4QSlot[kQ4R][4];             // one half block's quant bytes: [row][lk]
typedef uint8_t Q4HSlot[kQ4R][16];          // one block's headers (d, dmin, scales)
typedef float Q4SSlot[kQ4T][8];             // one block's group sums

// 16 bytes per lane global -> LDS (m0 + 16 lane). As inline assembly the
// compiler neither counts these loads nor waits for them; the kernel waits on
// its own vmcnt (only stricter for the compiler's own loads, of which the main
// loop has none).
__device__ __forceinline__ void dma16(uint32_t voff, const void* sbase, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds) : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// This wave's loads in ring group j: 2 (x) + 2 (a half block's quant bytes, j % 4 == 0) +
// 2 (headers and group sums, a block's first depth).
__host__ __device__ constexpr int q4_group_loads(int j) {
    return 2 + ((j & 3) == 0 ? 2 : 0) + ((j & 7) == 0 ? 2 : 0);
}

__global__ __launch_bounds__(kQ4Block, 1) void gemm_q4k_wide(const GemmJobs jobs, const int* __restrict__ ex,
                                                              const float* __restrict__ sx, const uint8_t* __restrict__ xp,
                                                              const float* __restrict__ x, int T, int K) {
    __shared__ __align__(16) Q4XSlot xr[kQ4XSlots];
    __shared__ __align__(16) Q4QSlot qr[2];
    __shared__ __align__(16) Q4HSlot hr[2];
    __shared__ __align__(16) Q4SSlot sr[2];
    const int cols = jobs.start[jobs.n];
    const int tb = static_cast<int>(blockIdx.x) / cols;
    const GemmJob job = gemm_job(jobs, static_cast<int>(blockIdx.x) - tb * cols);
    const uint8_t* __restrict__ w = job.w;
    float* __restrict__ y = job.y;
    const int M = job.M;
    const uint64_t ub0 = job.ub0;
    const int lane = threadIdx.x & 63;
    const int wv = wave_in_block();
    const int rg = wv & 3, th = wv >> 2;                       // row group, token half
    const int t0w = tb * kQ4T;                                 // the workgroup's first token
    const int tw = t0w + 64 * th;                              // this wave's first token
    const int rw0 = job.mb * kQ4R;                             // the workgroup's first row
    const int r0 = rw0 + 64 * rg;                              // this wave's first row
    const int nb = K >> 8, nst = K >> 5;
    const int lr = lane & 15, lk = lane >> 4;
    const uint8_t* wbase = w + ub0 * 144;
    // Ring loads of a wave (byte offsets; depth and block offsets go into the scalar base). x: tile wv of the
    // workgroup (its last one again past the end), both parts. Quant bytes: rows 32 wv + 16 i + lane / 4, piece
    // lane % 4. Headers: rows 64 (wv % 4) + lane; group sums: tokens 32 (wv % 4) + lane / 2 (waves 4-7 repeat
    // 0-3: the same bytes to the same place).
    const int xt = min(tb * (kQ4T / kTile) + wv, (T + kTile - 1) / kTile - 1);
    const int xrn = min(kTile, T - kTile * xt);
    const uint8_t* xbase = xp + tile_base(xt, K);
    const uint32_t xo = 16u * static_cast<uint32_t>(lk * xrn + min(lr, xrn - 1));
    const uint32_t xpart = 64u * xrn;   // bytes of one part of one depth
    auto qo = [&](int i) {
        const int row = min(rw0 + 32 * wv + 16 * i + (lane >> 2), M - 1), pc = lane & 3;
        return static_cast<uint32_t>(row) * static_cast<uint32_t>(nb) * 144u + 16u + 64u * (pc >> 1) + 16u * (pc & 1);
    };
    const uint32_t qo0 = qo(0), qo1 = qo(1);
    const uint32_t ho = static_cast<uint32_t>(min(r0 + lane, M - 1)) * static_cast<uint32_t>(nb) * 144u;
    const uint32_t so = 4u * (static_cast<uint32_t>(min(t0w + 32 * rg + (lane >> 1), T - 1)) * static_cast<uint32_t>(nst) +
                              4u * (lane & 1));
    auto lds_addr = [](const void* l) {
        return __builtin_amdgcn_readfirstlane(
            static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const void __attribute__((address_space(3)))*)(l))));
    };
    const uint32_t xr_a = lds_addr(&xr[0][wv][0][0]), qr_a = lds_addr(&qr[0][32 * wv][0]), hr_a = lds_addr(&hr[0][64 * rg][0]),
                   sr_a = lds_addr(&sr[0][32 * rg][0]);
    // ring group gs, in 4 parts: x (2), the half block's quant bytes, the block's headers and group sums
    auto issue_part = [&](int gs, int part) {   // past the last depth: the last group again, into slots not read any more
        const int ge = min(gs, nst - 1), gb = min(gs >> 3, nb - 1);
        if (part < 2) {
            dma16(xo, xbase + static_cast<size_t>(2 * ge + part) * xpart,
                  xr_a + static_cast<uint32_t>(gs % kQ4XSlots) * sizeof(Q4XSlot) + 1024u * part);
        } else if (part == 2) {
            if ((gs & 3) == 0) {
                const uint8_t* b = wbase + static_cast<size_t>(gb) * 144 + 32 * ((gs >> 2) & 1);
                const uint32_t l = qr_a + static_cast<uint32_t>((gs >> 2) & 1) * sizeof(Q4QSlot);
                dma16(qo0, b, l);
                dma16(qo1, b, l + 1024u);
            }
        } else if ((gs & 7) == 0) {
            const uint32_t hb = (gs >> 3) & 1;
            dma16(ho, wbase + static_cast<size_t>(gb) * 144, hr_a + hb * sizeof(Q4HSlot));
            dma16(so, sx + 8 * gb, sr_a + hb * sizeof(Q4SSlot));
        }
    };
    auto barrier = []() {   // the ring's loads stay in flight
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    uint32_t k64 = 0x64006400u;   // kept in a register: v_and_or_b32 takes one constant
    asm volatile("" : "+v"(k64));
    // B operands of this wave's rows: q[rt] holds the lane's piece of the current half block, sc[rt] the scales of
    // the half-block's depths
    uint4 q[4];
    uint32_t scb[4];   // the lane's four scale bytes (u = 0..3)
    f16x8_t B[2][4];
    auto take_hdr = [&](int blk) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            const uint4 h = *reinterpret_cast<const uint4*>(&hr[blk & 1][64 * rg + 16 * rt + lr][0]);
            const uint32_t lo = h.y & 0x3f3f3f3fu, hi = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
            scb[rt] = lk < 2 ? lo : hi;   // scale_min_k4 (src/cuda/matmul_q4.cu:18-26): groups 4 (lk / 2) + u
        }
    };
    auto take_q = [&](int half) {   // half block index: block 2 * half
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) q[rt] = qr[half & 1][64 * rg + 16 * rt + lr][lk];
    };
    WScale<kQ4_K> sc[4];
    auto b_make = [&](auto dI, int rt) {   // B operand rt of depth D of the block
        constexpr int D = decltype(dI)::value, U = D >> 1, J = D & 1;
        if constexpr (J == 0) sc[rt].template from<U>((scb[rt] >> (8 * U)) & 0xffu);
        f16x8_t b1[1];
        decode_q4<U, J>(q[rt], sc[rt], k64, b1);
        B[J][rt] = b1[0];
    };

    f16x8_t An[2];
    f32x4_t acc[4][4], C[4][4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // groups 0 .. kQ4Dist - 1 (nst >= 8); groups 0 and 1 complete
    for (int gs = 0; gs < kQ4Dist; ++gs)
#pragma unroll
        for (int part = 0; part < 4; ++part) issue_part(gs, part);
    wait_vm<q4_group_loads(2)>();
    barrier();
    take_hdr(0);
    take_q(0);
#pragma unroll
    for (int p = 0; p < 2; ++p) An[p] = *reinterpret_cast<const f16x8_t*>(&xr[0][4 * th][p][lane]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) b_make(IC<0>{}, rt);

    for (int b = 0; b < nb; ++b) {
        const int g0 = 8 * b;
        static_for<8>([&](auto sI) {
            constexpr int S = decltype(sI)::value;
            const int g = g0 + S;
            // the block's epilogue operands (last depth): d, -32 dmin and m_g
            float dsc[4], dmn5[4];
            f16x4_t Bm[4];
            if constexpr (S == 7) {
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) {
                    const uint4 h = *reinterpret_cast<const uint4*>(&hr[b & 1][64 * rg + 16 * rt + lr][0]);
                    Bm[rt] = min_weights(h, lk);
                    dsc[rt] = opaque(half_bits(h.x & 0xffffu));
                    dmn5[rt] = opaque(-32.0f * half_bits(h.x >> 16));
                }
            }
            // pieces and scales of the next depth's half block / block (stale ones after the last: not used)
            if constexpr (S == 3) take_q(2 * b + 1);
            if constexpr (S == 7) {
                take_q(2 * b + 2);
                take_hdr(b + 1);
            }
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                issue_part(g + kQ4Dist, tt);
                __builtin_amdgcn_sched_barrier(0);
                f16x8_t A[2];
#pragma unroll
                for (int p = 0; p < 2; ++p) {   // this tile's parts; the next tile's are requested
                    A[p] = An[p];
                    An[p] = *reinterpret_cast<const f16x8_t*>(&xr[(g + (tt == 3)) % kQ4XSlots][4 * th + ((tt + 1) & 3)][p][lane]);
                }
                // a block's first depth starts its sums from zero
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
                    C[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0], B[S & 1][rt], S == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : C[tt][rt], 0, 0, 0);
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) C[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[1], B[S & 1][rt], C[tt][rt], 0, 0, 0);
                b_make(IC<(S + 1) & 7>{}, tt);
                if constexpr (S == 7) {
                    // token tile tt of the block is complete: acc += d P_block - 32 dmin P_min
                    const f16x4_t As = min_operand(*reinterpret_cast<const float2*>(&sr[b & 1][64 * th + 16 * tt + lr][2 * lk]));
#pragma unroll
                    for (int rt = 0; rt < 4; ++rt) {
                        const f32x4_t pm = __builtin_amdgcn_mfma_f32_16x16x16f16(As, Bm[rt], f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[tt][rt][r] = __builtin_fmaf(dsc[rt], C[tt][rt][r], acc[tt][rt][r]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[tt][rt][r] = __builtin_fmaf(dmn5[rt], pm[r], acc[tt][rt][r]);
                    }
                }
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
                for (int i = 0; i < (S == 7 ? 12 : 8); ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, S == 7 ? 4 : 2, 0);
                }
            }
            // group g + 2 complete; group g + 3 may stay in flight
            wait_vm<q4_group_loads((S + 3) & 7)>();
            barrier();
        });
    }
    wait_vm<0>();
    // lane L holds C[4 (L/16) + r][L % 16] of tile (tt, rt): token 16 tt + 4 lk + r, row 16 rt + lr
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = tw + 16 * tt + 4 * lk + r;
            if (t >= T) continue;
            const int et = ex[t];
            if (et == kRowNonFinite) {
                for (int rt = 0; rt < 4; ++rt) {
                    const int row = r0 + 16 * rt + lr;
                    if (row < M)
                        y[static_cast<size_t>(t) * M + row] = row_dot_per_element(
                            w, kQ4_K, (ub0 + static_cast<uint64_t>(row) * nb) * 256, x + static_cast<size_t>(t) * K, K);
                }
                continue;
            }
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                const int row = r0 + 16 * rt + lr;
                if (row < M) y[static_cast<size_t>(t) * M + row] = ldexpf(acc[tt][rt][r], -et);
            }
        }
}

// ------------------------------------------------------------------ Q6_K, many tokens
// A workgroup (8 waves, one per CU) owns 128 tokens x 256 weight rows; wave w owns rows 64 (w % 4) .. +63 for tokens
// 64 (w / 4) .. +63, as 4 x 4 tiles, with the products and sums of gemm_kquant<kQ6_K, 4, 2, 1, 1> in its order (the
// same bits). A block's rows are only 2-byte aligned, so weights and x go global -> VGPR -> LDS, the quant bytes and
// scales in the lane order that decodes them. Work goes by row tile: the 12 products of one tile of 16 rows with the
// wave's 4 token tiles run while the next row tile's operand is decoded (28 VALU instructions) and the one after it
// is read from LDS; the A operands (4 tiles x 2 parts) stay in registers for the depth and the last row tile's
// products release them to the next depth's. The barrier stands in the middle of a depth, where the LDS reads before
// it are old: x needs two slots, and the ql bytes one (those of odd u are replaced while even u run and the other way
// round). A round of 256 workgroups at K = 2048: 90 us, 49 of them the MFMAs' own time, two rounds of 64 x 256 tiles 134.
// Before, B = q - 32 with a product and an FMA per 16 elements took 115 (fewer MFMAs, but 128 FMAs a stage beside 16
// of 32 x 32): M = 8192, 4096, 32, 32 at 500, 1500 and 4096 tokens 123, 348, 702 us then, 92, 290, 588 now.
constexpr int kQ6Waves = 8;
constexpr int kQ6Block = kQ6Waves * kWave;
constexpr int kQ6R = 256;                    // weight rows per workgroup (64 per wave)
constexpr int kQ6T = 128;                    // tokens per workgroup
typedef uint4 Q6XSlot[kQ6T / kTile][2][kWave];   // one depth of x: [tile][fp16 part][lane]
typedef uint2 Q6QSlot[2][kQ6R / kTile][kWave];   // 16 bytes a lane: [half, the depth of its u][row tile][lane]

__global__ __launch_bounds__(kQ6Block) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_q6k_wide(
    const GemmJobs jobs, const int* __restrict__ ex, const uint8_t* __restrict__ xp, const float* __restrict__ x, int T,
    int K) {
    __shared__ __align__(16) Q6XSlot xs[2];
    __shared__ __align__(16) Q6QSlot ql[2];        // of even and odd u
    __shared__ __align__(16) Q6QSlot qh[2];        // by block
    __shared__ __align__(16) uint8_t scl[2][kQ6R][16];
    __shared__ uint16_t dl[2][kQ6R];
    const int cols = jobs.start[jobs.n];
    const int tb = static_cast<int>(blockIdx.x) / cols;
    const GemmJob job = gemm_job(jobs, static_cast<int>(blockIdx.x) - tb * cols);
    const uint8_t* __restrict__ w = job.w;
    float* __restrict__ y = job.y;
    const int M = job.M;
    const uint64_t ub0 = job.ub0;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = wave_in_block();
    const int rg = wv & 3, th = wv >> 2;                       // row group, token half
    const int t0w = tb * kQ6T;                                 // the workgroup's first token
    const int tw = t0w + 64 * th;                              // this wave's first token
    const int rw0 = job.mb * kQ6R;                             // the workgroup's first row
    const int r0 = rw0 + 64 * rg;                              // this wave's first row
    const int nb = K >> 8, nst = K >> 5;

    // x: wave wv brings tile wv of the workgroup (the last one again past the end), both parts
    const int xt = min(tb * (kQ6T / kTile) + wv, (T + kTile - 1) / kTile - 1);
    const int xrn = min(kTile, T - kTile * xt);
    const uint8_t* xbase = xp + tile_base(xt, K);
    const uint32_t xo = 16u * static_cast<uint32_t>(lk * xrn + min(lr, xrn - 1));
    const uint32_t xpart = 64u * xrn;   // bytes of one part of one depth
    uint4 xr[2][2];
    auto x_load = [&](uint4 (&d)[2], int g) {   // past the last depth: the last one again
#pragma unroll
        for (int p = 0; p < 2; ++p) d[p] = ld16(xbase + (xo + static_cast<uint32_t>(2 * min(g, nst - 1) + p) * xpart));
    };
    auto x_store = [&](const uint4 (&d)[2], int g) {
#pragma unroll
        for (int p = 0; p < 2; ++p) xs[g & 1][wv][p][lane] = d[p];
    };
    // weights: 16-byte piece tid % 4 (the bytes of lanes lk = tid % 4) of rows tid / 4 and 128 + tid / 4; scales and d
    // of row tid / 2
    const uint8_t* wb = w + (ub0 + static_cast<uint64_t>(rw0) * nb) * 210;
    const int rlast = M - 1 - rw0;
    const uint32_t rbytes = 210u * static_cast<uint32_t>(nb);
    const int pc = tid & 3, pr = tid >> 2;
    const uint32_t wl[2] = {static_cast<uint32_t>(min(pr, rlast)) * rbytes + 64u * (pc >> 1) + 16u * (pc & 1),
                            static_cast<uint32_t>(min(pr + 128, rlast)) * rbytes + 64u * (pc >> 1) + 16u * (pc & 1)};
    const uint32_t wh = 128u - 32u * (pc >> 1);   // from there to the qh piece
    const uint32_t so = static_cast<uint32_t>(min(tid >> 1, rlast)) * rbytes + 192u + 2u * (tid & 1);
    auto block_at = [&](int b) { return 210u * static_cast<uint32_t>(min(b, nb - 1)); };   // the last block again
    auto ql_load = [&](uint4 (&d)[2], int b, int odd) {
        const uint32_t o = block_at(b) + 32u * odd;
#pragma unroll
        for (int i = 0; i < 2; ++i) d[i] = ldg16_a2(wb + (wl[i] + o));
    };
    auto qh_load = [&](uint4 (&d)[2], int b) {
        const uint32_t o = block_at(b);
#pragma unroll
        for (int i = 0; i < 2; ++i) d[i] = ldg16_a2(wb + (wl[i] + (o + wh)));
    };
    auto sc_load = [&](int b) { return ldg16_a2(wb + (so + block_at(b))); };   // the scales, or d in the last two bytes
    auto q_store = [&](const uint4& v, Q6QSlot& d, int i) {
        const int t = (pr >> 4) + 8 * i, l = 16 * pc + (pr & 15);
        d[0][t][l] = uint2{v.x, v.y};
        d[1][t][l] = uint2{v.z, v.w};
    };
    auto sc_store = [&](const uint4& v, int b) {
        if (tid & 1)
            dl[b & 1][tid >> 1] = static_cast<uint16_t>(v.w >> 16);
        else
            *reinterpret_cast<uint4*>(&scl[b & 1][tid >> 1][0]) = v;
    };
    auto barrier = []() {   // this wave's LDS work is done, then the workgroup meets (loads stay in flight)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    uint32_t k64 = 0x64006400u;   // kept in a register: v_and_or_b32 takes one constant
    asm volatile("" : "+v"(k64));
    uint32_t kf = 0x000f000fu, k30 = 0x00300030u;
    asm volatile("" : "+s"(kf), "+s"(k30));

    // B operands: row tile rt's come from raw[rt & 1] into B[rt & 1]
    struct Raw {
        uint2 l, h;
        uint32_t s;
    } raw[2];
    f16x2_t sc[4];   // of the current u
    f16x8_t B[2][2], A[4][2];
    auto raw_read = [&](auto dI, int rt, int b) {   // depth D of block b
        constexpr int D = decltype(dI)::value, U = D >> 1, J = D & 1;
        Raw& r = raw[rt & 1];
        r.l = ql[U & 1][J][4 * rg + rt][lane];
        r.h = qh[b & 1][J][4 * rg + rt][lane];
        if constexpr (J == 0) r.s = scl[b & 1][64 * rg + 16 * rt + lr][8 * (lk >> 1) + 2 * U + (lk & 1)];
    };
    auto b_make = [&](auto dI, int rt) {
        constexpr int D = decltype(dI)::value;
        const Raw& r = raw[rt & 1];
        if constexpr ((D & 1) == 0) sc[rt] = WScale<kQ6_K>::from(r.s);
        const uint32_t wd[2] = {r.l.x, r.l.y}, hd[2] = {r.h.x, r.h.y};
        decode_q6<(D >> 1)>(wd, hd, sc[rt], k64, kf, k30, B[rt & 1]);
    };
    f32x4_t acc[4][4], C[4][4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // blocks 0 (ql of odd u kept for the loop) and x of depths 0 .. 3 (nst >= 8)
    uint4 st[2];   // the weights on their way
    auto ql_put = [&](int odd) {
        q_store(st[0], ql[odd], 0);
        q_store(st[1], ql[odd], 1);
    };
    auto qh_put = [&](int b) {
        q_store(st[0], qh[b & 1], 0);
        q_store(st[1], qh[b & 1], 1);
    };
    x_load(xr[0], 0);
    x_load(xr[1], 1);
    ql_load(st, 0, 0);
    ql_put(0);
    qh_load(st, 0);
    qh_put(0);
    sc_store(sc_load(0), 0);
    ql_load(st, 0, 1);
    x_store(xr[0], 0);
    x_load(xr[0], 2);
    x_store(xr[1], 1);
    x_load(xr[1], 3);
    barrier();
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int p = 0; p < 2; ++p) A[tt][p] = *reinterpret_cast<const f16x8_t*>(&xs[0][4 * th + tt][p][lane]);
    raw_read(IC<0>{}, 0, 0);
    raw_read(IC<0>{}, 1, 0);
    b_make(IC<0>{}, 0);

    for (int b = 0; b < nb; ++b) {
        float dsc[4];
        auto epilogue = [&](int rt) {   // the block's sums of row tile rt are complete: acc += d C
            const float d = opaque(dsc[rt]);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[tt][rt][r] = __builtin_fmaf(d, C[tt][rt][r], acc[tt][rt][r]);
        };
        static_for<8>([&](auto sI) {
            constexpr int D = decltype(sI)::value;
            const int g = 8 * b + D;
            // The LDS slots in use (the barrier of depth D: MD): ql of even u are read M7 .. M1 and M3 .. M5, of odd u
            // M1 .. M3 and M5 .. M7, a block's qh M7 .. M7, x of depth g M(g - 1) .. Mg; scales with qh, d in depth 7.
            if constexpr (D == 0) {
                ql_put(1);
                st[0] = sc_load(b + 1);
            }
            if constexpr (D == 2) {
                sc_store(st[0], b + 1);
                qh_load(st, b + 1);
            }
            if constexpr (D == 4) {
                qh_put(b + 1);
                ql_load(st, b + 1, 0);
            }
            if constexpr (D == 6) {
                ql_put(0);
                ql_load(st, b + 1, 1);
            }
            static_for<4>([&](auto rI) {
                constexpr int rt = decltype(rI)::value;
                if constexpr (rt == 2) {
                    barrier();
                    x_store(xr[D & 1], g + 2);
                    x_load(xr[D & 1], g + 4);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (rt < 2)
                    raw_read(IC<D>{}, rt + 2, b);
                else
                    raw_read(IC<(D + 1) & 7>{}, rt - 2, b + (D == 7));
                if constexpr (D == 7) dsc[rt] = half_bits(dl[b & 1][64 * rg + 16 * rt + lr]);
                if constexpr (rt < 3)
                    b_make(IC<D>{}, rt + 1);
                else
                    b_make(IC<(D + 1) & 7>{}, 0);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt)   // a block's first depth starts its sums from zero
                    C[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        A[tt][0], B[rt & 1][0], D == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : C[tt][rt], 0, 0, 0);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    C[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[tt][1], B[rt & 1][0], C[tt][rt], 0, 0, 0);
                    if constexpr (rt == 3) A[tt][1] = *reinterpret_cast<const f16x8_t*>(&xs[(D + 1) & 1][4 * th + tt][1][lane]);
                }
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    C[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[tt][0], B[rt & 1][1], C[tt][rt], 0, 0, 0);
                    if constexpr (rt == 3) A[tt][0] = *reinterpret_cast<const f16x8_t*>(&xs[(D + 1) & 1][4 * th + tt][0][lane]);
                }
                if constexpr (D == 7 && rt > 0) epilogue(rt - 1);
                __builtin_amdgcn_sched_group_barrier(0x100, 2 + ((rt < 2 ? D : D + 1) % 2 == 0) + (D == 7), 0);
#pragma unroll
                for (int i = 0; i < 12; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, D == 7 ? 4 : 3, 0);
                    if (rt == 3 && i >= 4) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (D == 7) epilogue(3);
        });
    }
    // lane L holds C[4 (L/16) + r][L % 16] of tile (tt, rt): token 16 tt + 4 lk + r, row 16 rt + lr
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = tw + 16 * tt + 4 * lk + r;
            if (t >= T) continue;
            const int et = ex[t];
            if (et == kRowNonFinite) {
                for (int rt = 0; rt < 4; ++rt) {
                    const int row = r0 + 16 * rt + lr;
                    if (row < M)
                        y[static_cast<size_t>(t) * M + row] = row_dot_per_element(
                            w, kQ6_K, (ub0 + static_cast<uint64_t>(row) * nb) * 256, x + static_cast<size_t>(t) * K, K);
                }
                continue;
            }
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                const int row = r0 + 16 * rt + lr;
                if (row < M) y[static_cast<size_t>(t) * M + row] = ldexpf(acc[tt][rt][r], -et);
            }
        }
}

// Token rows that the matrix-core paths take; x's fragments and a matrix's rows are addressed with 32-bit byte
// offsets (gemm_offsets_fit).
bool gemm_rows_ok(int rows, int K, const float* x) {
    return K % 256 == 0 && aligned16(x) && rows <= kGemmMaxRows &&
           4 * static_cast<uint64_t>(rows) * static_cast<uint64_t>(K) < (uint64_t{1} << 32);
}

// Below 16 tokens a call stands in for one GEMV per token, after which a token's x may be overwritten: an output that
// overlaps x takes them.
bool outputs_apart(int rows, int M, int K, const float* x, const float* y) {
    return rows >= kGemmMinRows || !floats_overlap(x, static_cast<size_t>(rows) * K, y, static_cast<size_t>(rows) * M);
}

bool gemm_job_ok(int type, uint64_t element_offset, int M, int K) {
    return element_offset % 256 == 0 &&
           (type == kQ4_K ? gemm_offsets_fit(true, 144, M, K) : type == kQ6_K && gemm_offsets_fit(false, 210, M, K));
}

// Workgroup columns of `rows` weight rows each, matrix after matrix.
unsigned columns(GemmJobs& jobs, int rows) {
    jobs.start[0] = 0;
    for (int j = 0; j < jobs.n; ++j) jobs.start[j + 1] = jobs.start[j] + static_cast<int>(blocks_for(jobs.M[j], rows));
    return static_cast<unsigned>(jobs.start[jobs.n]);
}

constexpr unsigned kPrepSpread = 256;

struct Prepared {
    const int* ex;
    const float* sx;
    const uint8_t* xp;
    const float* x;   // the token rows themselves (rows holding an infinity)
};

// Checks the workspace (wanted from 16 rows on, whichever path runs) and launches the prep kernel if a path needs it.
int prepare_x(bool prep, const float* x, int rows, int K, void* workspace, size_t workspace_bytes, hipStream_t s,
              Prepared& p) {
    const size_t need = ws_bytes(rows, K);
    if (rows >= kGemmMinRows) QK_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace),
               "matmul_rows: workspace of %zu bytes (16-byte aligned) needed, got %zu", need,
               workspace ? workspace_bytes : size_t{0});
    p = Prepared{nullptr, nullptr, nullptr, x};
    if (!prep) return ok();
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    int* ex = reinterpret_cast<int*>(ws);
    float* sx = reinterpret_cast<float*>(ws + ws_exp_bytes(rows));
    uint8_t* xp = ws + ws_exp_bytes(rows) + ws_sum_bytes(rows, K);
    // A workgroup per round while each has a CU: at 196 and 256 workgroups 0.0 and 1.1 us less, at 376 and 512 (two on
    // a CU, every row read once per round) 2.3 us more at K = 2048, at 392 6.1 more at K = 4096.
    const unsigned tiles = blocks_for(rows, kTile), rounds = blocks_for(K, 512);
    const dim3 grid(tiles, static_cast<uint64_t>(tiles) * rounds <= kPrepSpread ? rounds : 1);
    switch (K) {
        case 512: gemm_prep_x<1><<<grid, 1024, 0, s>>>(x, ex, sx, xp, rows, K); break;
        case 1024: gemm_prep_x<2><<<grid, 1024, 0, s>>>(x, ex, sx, xp, rows, K); break;
        case 2048: gemm_prep_x<4><<<grid, 1024, 0, s>>>(x, ex, sx, xp, rows, K); break;
        case 4096: gemm_prep_x<8><<<grid, 1024, 0, s>>>(x, ex, sx, xp, rows, K); break;
        default: gemm_prep_x<0><<<grid, 1024, 0, s>>>(x, ex, sx, xp, rows, K); break;
    }
    p = Prepared{ex, sx, xp, x};
    return check_launch("matmul_rows prep");
}

// How a matrix of a call is computed. A matrix alone and among others takes the same path and adds in the same
// order, so the rule looks at the token count, K and the matrix itself only; which tile shape a path then uses
// (the sums are the same bits in all of its shapes) depends on the whole launch.
enum class Path { gemv, f32, few, sliced4, sliced2, whole };

// Measured at K = 2048 (M = 12352 in four matrices) and K = 4096 (M = 2048), Q4_K, us including the prep pass:
//   f32 against one GEMV per token: above, GEMV 6 / 3.6 per token, so it starts at 3 tokens (4 from K = 2304: at
//     2048 x 6144, 3 tokens, Q6_K 14.0 against 11.7). At 3 tokens a GEMV's better use of the memory tells in large
//     matrices: M = 32768 28 against 32, 65536 51 against 45 (Q6_K 34 and 39, 66 and 57).
//   few against sliced4 at 17..32 tokens 22 / 12 and 18 / 26, at 128 tokens 74 / 19 and 44 / 26, against sliced2 at
//     300 tokens 50 and 42 at K = 4096: few at 16 tokens, up to 160 from K = 4096.
//   sliced4 against whole at K = 2048: 77 tokens 31 and 48, 128 tokens 44 and 49, 200 tokens 58 and 53.
//   sliced2 against whole at K = 4096: 777 tokens 58 and 82, 1500 tokens 86 and 109, 2100 tokens 160 and 113. With
//     many rows the chip is full without the slices.
//   A matrix of up to 64 rows would leave most of a 256-row tile idle, a tile column more in every token block of the
//     others' launch: up to 1024 tokens that is a fiftieth of it, above a round at worst (4096 tokens: 61 us against 20
//     by sliced2 on its own).
// Q6_K times are about 1.5x these; the same lines hold within 10%.
Path gemm_path(int rows, int K, int M) {
    const int nb = K / 256;
    if (rows < (nb > 8 ? 4 : 3) || (rows == 3 && M >= 49152)) return Path::gemv;
    if (rows < kGemmMinRows) return Path::f32;
    if (rows <= (nb >= 16 ? 160 : nb % 4 ? 128 : 16)) return Path::few;
    if (rows <= 128) return Path::sliced4;
    if (M <= 64 && rows > 1024 && nb % 2 == 0) return Path::sliced2;
    if (nb >= 16 && nb % 2 == 0 && M < 4096 && rows <= 2048) return Path::sliced2;
    return Path::whole;
}

constexpr int kWideRows = kGemmTileRows, kWideTokens = 128;   // tile of the wide kernels, the tallest
static_assert(kQ4R == kWideRows && kQ4T == kWideTokens && kQ6R == kWideRows && kQ6T == kWideTokens, "wide tiles");

unsigned wide_grid(GemmJobs& jobs, int rows) { return columns(jobs, kWideRows) * blocks_for(rows, kWideTokens); }

template <int TYPE, int WT, int WR, int KW, int SL>
struct Shape {
    using G = GemmShape<TYPE, WT, WR, KW, SL>;
    // Workgroups of the launch in rounds of 256 (one per CU) times a round's measured time (us at K = 2048, Q4_K).
    static float cost(GemmJobs& jobs, int rows, float round) {
        const unsigned wgs = columns(jobs, G::rows) * blocks_for(rows, G::tokens);
        return round * static_cast<float>(blocks_for(wgs, 256));
    }
    static void launch(GemmJobs& jobs, const Prepared& p, int rows, int K, hipStream_t s) {
        const unsigned grid = columns(jobs, G::rows) * blocks_for(rows, G::tokens);
        gemm_kquant<TYPE, WT, WR, KW, SL><<<grid, 512, 0, s>>>(jobs, p.ex, p.sx, p.xp, p.x, rows, K);
    }
};

template <int TYPE, int WR, int NW>
void launch_f32(GemmJobs& jobs, const Prepared& p, int rows, int K, hipStream_t s) {
    gemm_f32<TYPE, WR, NW><<<columns(jobs, 16 * WR), NW * kWave, 0, s>>>(jobs, p.x, rows, K);
}

template <int TYPE>
void launch_gemm(Path path, GemmJobs& jobs, const Prepared& p, int rows, int K, hipStream_t s) {
    if (path == Path::f32) {
        // A slice per wave while each workgroup of 16 rows has a CU (2048 x 4096, 9 tokens: 9.9 us, 10.5 with two
        // slices). Above, two slices, and 16 rows (less work in a part-full round) or 32 (x, read by every workgroup,
        // half as often: more with the tokens): us = 4 + workgroups per CU, rounded up, times a workgroup's time at
        // K = 2048, within 10% from M = 8192 to 248320. Q6_K's 32 rows in 4 waves are 5-10% behind 8 waves.
        constexpr bool q4 = TYPE == kQ4_K;
        const unsigned n1 = columns(jobs, 16);
        const float t = static_cast<float>(rows);
        const float c1 = ((q4 ? 2.4f : 3.5f) + 0.1f * t) * static_cast<float>(blocks_for(n1, 256)),
                    c2 = ((q4 ? 5.6f : 7.0f) + 0.08f * t) * static_cast<float>(blocks_for(columns(jobs, 32), 256));
        if (n1 <= 256)
            launch_f32<TYPE, 1, 8>(jobs, p, rows, K, s);
        else if (c1 <= c2)
            launch_f32<TYPE, 1, 4>(jobs, p, rows, K, s);
        else
            launch_f32<TYPE, 2, q4 ? 4 : 8>(jobs, p, rows, K, s);
    } else if (path == Path::few) {
        // rounds of 256 workgroups times a round's measured time, 16, 32 and 64 rows a workgroup
        const int64_t tb = blocks_for(rows, kTile);
        const float c1 = 8.5f * blocks_for(columns(jobs, 16) * tb, 256), c2 = 9.5f * blocks_for(columns(jobs, 32) * tb, 256),
                    c4 = 13.f * blocks_for(columns(jobs, 64) * tb, 256);
        if (c1 <= c2 && c1 <= c4)
            gemm_few<TYPE, 1><<<columns(jobs, 16) * tb, 512, 0, s>>>(jobs, p.x, rows, K);
        else if (c2 <= c4)
            gemm_few<TYPE, 2><<<columns(jobs, 32) * tb, 512, 0, s>>>(jobs, p.x, rows, K);
        else
            gemm_few<TYPE, 4><<<columns(jobs, 64) * tb, 512, 0, s>>>(jobs, p.x, rows, K);
    } else if (path == Path::sliced4) {
        using S1 = Shape<TYPE, 2, 2, 4, 4>;
        using S2 = Shape<TYPE, 2, 2, 2, 4>;
        using S3 = Shape<TYPE, 3, 2, 2, 4>;
        const float c1 = S1::cost(jobs, rows, 12.5f), c2 = S2::cost(jobs, rows, 20.f), c3 = S3::cost(jobs, rows, 25.f);
        if (c1 <= c2 && c1 <= c3)
            S1::launch(jobs, p, rows, K, s);
        else if (c2 <= c3)
            S2::launch(jobs, p, rows, K, s);
        else
            S3::launch(jobs, p, rows, K, s);
    } else if (path == Path::sliced2) {
        using S1 = Shape<TYPE, 2, 2, 2, 2>;
        using S2 = Shape<TYPE, 3, 2, 2, 2>;
        using S3 = Shape<TYPE, 4, 2, 2, 2>;
        const float c1 = S1::cost(jobs, rows, 20.f), c2 = S2::cost(jobs, rows, 25.f), c3 = S3::cost(jobs, rows, 31.f);
        if (c1 <= c2 && c1 <= c3)
            S1::launch(jobs, p, rows, K, s);
        else if (c2 <= c3)
            S2::launch(jobs, p, rows, K, s);
        else
            S3::launch(jobs, p, rows, K, s);
    } else {
        using S1 = Shape<TYPE, 4, 2, 1, 1>;
        // 64 x 256 tiles or 128 x 256, us a round
        constexpr float small = TYPE == kQ4_K ? 46.f : 67.f, wide = TYPE == kQ4_K ? 61.f : 90.f;
        const unsigned grid = wide_grid(jobs, rows);
        if (S1::cost(jobs, rows, small) <= wide * static_cast<float>(blocks_for(grid, 256)))
            S1::launch(jobs, p, rows, K, s);
        else if constexpr (TYPE == kQ4_K)
            gemm_q4k_wide<<<grid, kQ4Block, 0, s>>>(jobs, p.ex, p.sx, p.xp, p.x, rows, K);
        else
            gemm_q6k_wide<<<grid, kQ6Block, 0, s>>>(jobs, p.ex, p.xp, p.x, rows, K);
    }
}

void launch_gemm(Path path, int type, GemmJobs& jobs, const Prepared& p, int rows, int K, hipStream_t s) {
    if (type == kQ4_K)
        launch_gemm<kQ4_K>(path, jobs, p, rows, K, s);
    else
        launch_gemm<kQ6_K>(path, jobs, p, rows, K, s);
}

// One GEMV per token (the reference's own loop).
int per_token(const void* weight, int type, uint64_t num_elements, const float* x, float* y, int rows, int M, int K,
              uint64_t element_offset, void* stream) {
    for (int t = 0; t < rows; ++t) {
        const int rc = qwen_matmul_dispatch(weight, type, num_elements, x + static_cast<size_t>(t) * K,
                                            y + static_cast<size_t>(t) * M, M, K, element_offset, stream);
        if (rc) return rc;
    }
    return ok();
}

}  // namespace
}  // namespace qk

using namespace qk;

extern "C" {

size_t qwen_matmul_rows_workspace_bytes(int rows, int K) {
    if (rows < kGemmMinRows || K <= 0 || K % 256 != 0) return 0;
    return ws_bytes(rows, K);
}

int qwen_matmul_rows(const void* weight, int type, uint64_t num_elements, const float* x, float* y, int rows, int M,
                     int K, uint64_t element_offset, void* workspace, size_t workspace_bytes, void* stream) {
    if (!weight) return fail(QWEN_STATUS_INVALID_ARGUMENT, "tensor is not loaded");
    if (!type_supported(type)) return fail(QWEN_STATUS_UNSUPPORTED_TYPE, "unsupported GGML type %d", type);
    if (M <= 0 || K <= 0 || element_offset > num_elements ||
        static_cast<uint64_t>(M) * static_cast<uint64_t>(K) > num_elements - element_offset)
        return fail(QWEN_STATUS_OUT_OF_RANGE, "GEMV shape exceeds tensor (M=%d, K=%d)", M, K);
    QK_REQUIRE(rows >= 0, "matmul_rows: negative rows %d", rows);
    if (rows == 0) return ok();
    QK_REQUIRE(x && y, "matmul_rows: null pointer");
    const bool gemm = gemm_rows_ok(rows, K, x) && gemm_job_ok(type, element_offset, M, K) &&
                      outputs_apart(rows, M, K, x, y);
    const Path path = gemm ? gemm_path(rows, K, M) : Path::gemv;
    if (path == Path::gemv) return per_token(weight, type, num_elements, x, y, rows, M, K, element_offset, stream);
    const hipStream_t s = as_stream(stream);
    Prepared p;
    if (const int rc = prepare_x(path != Path::few && path != Path::f32, x, rows, K, workspace, workspace_bytes, s, p)) return rc;
    GemmJobs jobs{};
    jobs.w[0] = static_cast<const uint8_t*>(weight);
    jobs.y[0] = y;
    jobs.ub0[0] = element_offset / 256;
    jobs.M[0] = M;
    jobs.n = 1;
    launch_gemm(path, type, jobs, p, rows, K, s);
    return check_launch("matmul_rows");
}

int qwen_matmul_rows_multi(const qwen_gemv_desc* descs, int n, const float* x, int rows, int K, void* workspace,
                           size_t workspace_bytes, void* stream) {
    QK_REQUIRE(n >= 0 && n <= 64, "matmul_rows_multi: n = %d outside [0, 64]", n);
    if (n == 0) return ok();
    QK_REQUIRE(descs, "matmul_rows_multi: null descriptors");
    for (int j = 0; j < n; ++j) {
        const qwen_gemv_desc& e = descs[j];
        if (!e.weight) return fail(QWEN_STATUS_INVALID_ARGUMENT, "descriptor %d: tensor is not loaded", j);
        if (!type_supported(e.type))
            return fail(QWEN_STATUS_UNSUPPORTED_TYPE, "descriptor %d: unsupported GGML type %d", j, e.type);
        if (e.M <= 0 || K <= 0 || e.element_offset > e.num_elements ||
            static_cast<uint64_t>(e.M) * static_cast<uint64_t>(K) > e.num_elements - e.element_offset)
            return fail(QWEN_STATUS_OUT_OF_RANGE, "descriptor %d: GEMV shape exceeds tensor (M=%d, K=%d)", j, e.M, K);
        QK_REQUIRE(e.split == 0, "matmul_rows_multi: descriptor %d: split rows are not supported", j);
        QK_REQUIRE(e.y, "matmul_rows_multi: descriptor %d has a null output", j);
    }
    QK_REQUIRE(rows >= 0, "matmul_rows_multi: negative rows %d", rows);
    if (rows == 0) return ok();
    QK_REQUIRE(x, "matmul_rows_multi: null x");
    bool gemm = gemm_rows_ok(rows, K, x);
    for (int j = 0; j < n; ++j) gemm &= outputs_apart(rows, descs[j].M, K, x, descs[j].y);
    Path path[64];
    bool prep = false, all_gemv = true;
    for (int j = 0; j < n; ++j) {
        const qwen_gemv_desc& e = descs[j];
        path[j] = gemm && gemm_job_ok(e.type, e.element_offset, e.M, K) ? gemm_path(rows, K, e.M) : Path::gemv;
        prep |= path[j] != Path::gemv && path[j] != Path::f32 && path[j] != Path::few;
        all_gemv &= path[j] == Path::gemv;
    }
    if (all_gemv) {   // every matrix in one call per token (each output the bits of its own GEMV)
        qwen_gemv_desc d[64];
        for (int t = 0; t < rows; ++t) {
            for (int j = 0; j < n; ++j) {
                d[j] = descs[j];
                d[j].y = descs[j].y + static_cast<size_t>(t) * descs[j].M;
            }
            if (const int rc = qwen_matmul_dispatch_multi(d, n, x + static_cast<size_t>(t) * K, K, stream)) return rc;
        }
        return ok();
    }
    const hipStream_t s = as_stream(stream);
    Prepared p;
    if (const int rc = prepare_x(prep, x, rows, K, workspace, workspace_bytes, s, p)) return rc;
    for (const int type : {static_cast<int>(kQ4_K), static_cast<int>(kQ6_K)})
        for (const Path to : {Path::f32, Path::few, Path::sliced4, Path::sliced2, Path::whole}) {
            GemmJobs jobs{};
            for (int j = 0; j < n; ++j) {
                const qwen_gemv_desc& e = descs[j];
                if (e.type != type || path[j] != to) continue;
                const int k = jobs.n++;
                jobs.w[k] = static_cast<const uint8_t*>(e.weight);
                jobs.y[k] = e.y;
                jobs.ub0[k] = e.element_offset / 256;
                jobs.M[k] = e.M;
                if (jobs.n == kGemmJobs) {
                    launch_gemm(to, type, jobs, p, rows, K, s);
                    jobs.n = 0;
                }
            }
            if (jobs.n) launch_gemm(to, type, jobs, p, rows, K, s);
        }
    if (const int rc = check_launch("matmul_rows_multi")) return rc;
    for (int j = 0; j < n; ++j) {   // the rest: one GEMV per token
        const qwen_gemv_desc& e = descs[j];
        if (path[j] != Path::gemv) continue;
        if (const int rc = per_token(e.weight, e.type, e.num_elements, x, e.y, rows, e.M, K, e.element_offset, stream))
            return rc;
    }
    return ok();
}

}  // extern "C"
