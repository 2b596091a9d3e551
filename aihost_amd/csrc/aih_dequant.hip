// aih_dequant.hip -- standalone GGUF block dequantization, bit-exact to the
// reference decoders.
//
// Element order and arithmetic follow the code that actually runs in the
// reference: the inline GLSL shaders and their CPU twins
//   Q4_K  AIHost/AIHost/Compute/QuantizationFormats.cs:140-196, ComputeOps.cs:1629-1678
//   Q6_K  AIHost/AIHost/Compute/QuantizationFormats.cs:269-321, ComputeOps.cs:1735-1774
// and, for the two formats the reference rejects (ComputeOps.cs:743), the GGUF
// definitions of Q8_0 (y = q*d) and Q4_0 (y = (q-8)*d).
//
// Each lane produces 4 consecutive outputs per tile (one 16-byte store), so a
// wave writes 1 KiB contiguous: one K-quant super-block, or eight Q8_0/Q4_0
// blocks.
// The fp32 expressions are evaluated exactly as the C# source writes them,
// left to right with one rounding per operation (contraction is disabled for
// the whole file), which makes the result bit-identical to the CPU decoder.
#include "aih_internal.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace {

// QuantizationFormats.cs:147-152 (the reference GPU decoder): IEEE decoding
// with -0 -> +0 and every NaN -> 0x7FC00000.
__device__ __forceinline__ float f16_ieee_glsl(uint32_t h)
{
    uint32_t s = (h >> 15) & 1u, e = (h >> 10) & 31u, m = h & 1023u;
    if (e == 0u) {
        if (m == 0u) return 0.0f;
        float v = (float)m * 5.9604644775390625e-8f;   // m * 2^-24, exact
        return s ? -v : v;
    }
    if (e == 31u) return m ? __uint_as_float(0x7FC00000u) : __uint_as_float(s ? 0xFF800000u : 0x7F800000u);
    return __uint_as_float((s << 31) | ((e + 112u) << 23) | (m << 13));
}

// ComputeOps.cs:1497-1522 (the reference CPU decoder), reproduced bit for bit:
// for subnormals it normalises the mantissa but sets the exponent to
// 1 - shift + 127 (shift = index of the leading mantissa bit), NaN payloads
// and the sign of zero are kept.
__device__ __forceinline__ float f16_refcpu(uint32_t h)
{
    uint32_t sign = (h >> 15) & 1u, exp = (h >> 10) & 0x1Fu, mant = h & 0x3FFu;
    if (exp == 0u) {
        if (mant == 0u) return __uint_as_float(sign << 31);
        int shift = 31 - __clz((int)mant);            // leading bit position, 0..9
        exp = (uint32_t)(1 - shift + 127);
        mant = ((mant << (10 - shift)) & 0x3FFu) << 13;
    } else if (exp == 0x1Fu) {
        exp = 0xFFu;
        mant <<= 13;
    } else {
        exp = exp - 15u + 127u;
        mant <<= 13;
    }
    return __uint_as_float((sign << 31) | (exp << 23) | (mant & 0x7FFFFFu));
}

template <int MODE>
__device__ __forceinline__ float f16_decode(uint32_t h)
{
    return MODE == AIH_F16_REFCPU ? f16_refcpu(h) : f16_ieee_glsl(h);
}

__device__ __forceinline__ uint32_t ld_u8(const uint8_t *p) { return *p; }
__device__ __forceinline__ uint32_t ld_u16(const uint8_t *p)
{
    uint16_t v;
    __builtin_memcpy(&v, p, 2);
    return v;
}
__device__ __forceinline__ uint32_t ld_u32(const uint8_t *p)
{
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

typedef float f4 __attribute__((ext_vector_type(4)));

// Each format in two parts: load() reads the packed bytes of a lane's four
// outputs (raw, nothing computed from them, so that the loads of several
// blocks can be in flight together) and value() computes the outputs.

// Q4_K: 64 lanes per 144-byte block (QuantizationFormats.cs:167-195).  The
// whole 16-byte header (d, dmin, scales[12]) is one load, the same address in
// all lanes of the block.
struct DQ4K {
    static constexpr int QK = 256, BB = 144, kTiles = 2;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    struct Raw { u4 hdr; uint32_t qs; };
    __device__ static void load(const uint8_t *b, int lane, Raw &r)
    {
        __builtin_memcpy(&r.hdr, b, 16);
        r.qs = ld_u32(b + 16 + (lane >> 4) * 32 + (lane & 7) * 4);
    }
    template <int MODE>
    __device__ static f4 value(const Raw &w, int lane)
    {
        // sub-block j = 2 * group + is_upper of elements 32 j .. 32 j + 31
        const int j = lane >> 3, sh = 8 * (j & 3);
        const uint32_t a = w.hdr.y >> sh, b = w.hdr.z >> sh, c = w.hdr.w >> sh;
        const uint32_t sc8 = j < 4 ? (a & 63u) : ((c & 0xFu) | ((a >> 2) & 0x30u));
        const uint32_t mn8 = j < 4 ? (b & 63u) : (((c >> 4) & 0xFu) | ((b >> 2) & 0x30u));
        const float d = f16_decode<MODE>(w.hdr.x & 0xFFFFu), dmin = f16_decode<MODE>(w.hdr.x >> 16);
        const float sc = (float)sc8, mn = (float)mn8;
        const uint32_t q4 = w.qs >> ((j & 1) * 4);
        f4 r;
        // y = d * sc * q - dmin * mn, one rounding per operation
        r.x = d * sc * (float)(q4 & 15u) - dmin * mn;
        r.y = d * sc * (float)((q4 >> 8) & 15u) - dmin * mn;
        r.z = d * sc * (float)((q4 >> 16) & 15u) - dmin * mn;
        r.w = d * sc * (float)((q4 >> 24) & 15u) - dmin * mn;
        return r;
    }
};

// Q6_K: 64 lanes per 210-byte block (QuantizationFormats.cs:286-320).
struct DQ6K {
    static constexpr int QK = 256, BB = 210, kTiles = 4;
    struct Raw { uint32_t ql, qh, sc, d; };
    __device__ static void load(const uint8_t *b, int lane, Raw &r)
    {
        const int h = lane >> 5, quarter = (lane >> 3) & 3, wq = (lane & 7) * 4;
        r.ql = ld_u32(b + h * 64 + (quarter & 1) * 32 + wq);
        r.qh = ld_u32(b + 128 + h * 32 + wq);
        r.sc = ld_u8(b + 192 + (lane >> 2));
        r.d = ld_u16(b + 208);
    }
    template <int MODE>
    __device__ static f4 value(const Raw &w, int lane)
    {
        const int quarter = (lane >> 3) & 3;
        const uint32_t ql = w.ql >> ((quarter >> 1) * 4), qh = w.qh >> (quarter * 2);
        const int sc = (int)(int8_t)(uint8_t)w.sc;
        const float d = f16_decode<MODE>(w.d);
        f4 r;
        // y = d * sc * (q - 32)
        r.x = d * (float)sc * (float)((int)((ql & 15u) | ((qh & 3u) << 4)) - 32);
        r.y = d * (float)sc * (float)((int)(((ql >> 8) & 15u) | (((qh >> 8) & 3u) << 4)) - 32);
        r.z = d * (float)sc * (float)((int)(((ql >> 16) & 15u) | (((qh >> 16) & 3u) << 4)) - 32);
        r.w = d * (float)sc * (float)((int)(((ql >> 24) & 15u) | (((qh >> 24) & 3u) << 4)) - 32);
        return r;
    }
};

// Q8_0: 8 lanes per 34-byte block; y = q * d.
struct DQ80 {
    static constexpr int QK = 32, BB = 34, kTiles = 2;
    struct Raw { uint32_t q, d; };
    __device__ static void load(const uint8_t *b, int lane, Raw &r)
    {
        r.d = ld_u16(b);
        r.q = ld_u32(b + 2 + lane * 4);
    }
    template <int MODE>
    __device__ static f4 value(const Raw &w, int)
    {
        const float d = f16_decode<MODE>(w.d);
        f4 r;
        r.x = (float)(int8_t)(w.q & 0xFFu) * d;
        r.y = (float)(int8_t)((w.q >> 8) & 0xFFu) * d;
        r.z = (float)(int8_t)((w.q >> 16) & 0xFFu) * d;
        r.w = (float)(int8_t)(w.q >> 24) * d;
        return r;
    }
};

// Q4_0: 8 lanes per 18-byte block; low nibble -> j, high nibble -> j + 16,
// y = (q - 8) * d.
struct DQ40 {
    static constexpr int QK = 32, BB = 18, kTiles = 2;
    struct Raw { uint32_t q, d; };
    __device__ static void load(const uint8_t *b, int lane, Raw &r)
    {
        r.d = ld_u16(b);
        r.q = ld_u32(b + 2 + (lane & 3) * 4);
    }
    template <int MODE>
    __device__ static f4 value(const Raw &w, int lane)
    {
        const float d = f16_decode<MODE>(w.d);
        const uint32_t q = w.q >> ((lane >> 2) * 4);
        f4 r;
        r.x = (float)((int)(q & 15u) - 8) * d;
        r.y = (float)((int)((q >> 8) & 15u) - 8) * d;
        r.z = (float)((int)((q >> 16) & 15u) - 8) * d;
        r.w = (float)((int)((q >> 24) & 15u) - 8) * d;
        return r;
    }
};

template <bool STREAM>
__device__ __forceinline__ void store4(f4 v, f4 *to)
{
    if (STREAM) __builtin_nontemporal_store(v, to);
    else *to = v;
}

// Bound by HBM.  The loads of a thread's kTiles tiles are in flight together.
// On MI355X, 32000 x 4096 over rotating tensors, against one tile per
// grid-stride step with plain stores: Q4_K 225 -> 81 us (7.3 TB/s), Q6_K 128 ->
// 114, Q8_0 165 -> 107, Q4_0 154 -> 84.  Two and four tiles differ by 0-4%, but
// for Q6_K (122 against 114); Q4_K with eight 95-120, with plain stores 111-114.
// STREAM: non-temporal stores (launch_type).
// Step g writes the 4 KB * kTiles of outputs from element 1024 * kTiles * g:
// thread t's outputs 4 t .. 4 t + 3 of each of the kTiles tiles.
template <class F, int MODE, int kTiles, bool STREAM>
__global__ void __launch_bounds__(256)
dequant_kernel(const uint8_t *__restrict__ q, f4 *__restrict__ out, uint64_t n_blocks)
{
    constexpr int LPB = F::QK / 4;  // lanes per block
    constexpr int step = 256 / LPB * F::BB;   // packed bytes of a tile
    const uint64_t total = n_blocks * LPB;
    const uint64_t groups = (total + 256 * kTiles - 1) / (256 * kTiles);
    const int lane = (int)(threadIdx.x % LPB);
    for (uint64_t g = blockIdx.x; g < groups; g += gridDim.x) {
        const uint64_t t0 = g * (256 * kTiles) + threadIdx.x;
        const uint8_t *b = q + t0 / LPB * F::BB;
        typename F::Raw r[kTiles];
        if ((g + 1) * (256 * kTiles) <= total) {
#pragma unroll
            for (int u = 0; u < kTiles; ++u) F::load(b + u * step, lane, r[u]);
#pragma unroll
            for (int u = 0; u < kTiles; ++u) store4<STREAM>(F::template value<MODE>(r[u], lane), out + t0 + 256 * u);
        } else {
#pragma unroll
            for (int u = 0; u < kTiles; ++u)
                if (t0 + 256 * u < total) {
                    F::load(b + u * step, lane, r[u]);
                    store4<STREAM>(F::template value<MODE>(r[u], lane), out + t0 + 256 * u);
                }
        }
    }
}

// Row gather: out[i, :] = dequantized row ids[i] of a [vocab, dim] table,
// with the same per-lane decoders as dequant_kernel (bit-exact to it).  An
// id outside [0, vocab) yields a row of zeros.
template <class F>
__global__ void __launch_bounds__(256)
embed_kernel(const uint8_t *__restrict__ table, int64_t vocab, int64_t row_bytes, int64_t blocks_per_row,
             const int32_t *__restrict__ ids, int64_t n, f4 *__restrict__ out)
{
    constexpr int QK = F::QK, BB = F::BB;
    constexpr int LPB = QK / 4;
    const uint64_t per_row = (uint64_t)blocks_per_row * LPB;
    const uint64_t total = (uint64_t)n * per_row;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
        const uint64_t i = t / per_row, r = t % per_row;
        const int64_t id = ids[i];
        f4 v = {0.f, 0.f, 0.f, 0.f};
        if (id >= 0 && id < vocab) {
            const uint8_t *b = table + id * row_bytes + (r / LPB) * BB;
            const int lane = (int)(r % LPB);
            typename F::Raw w;
            F::load(b, lane, w);
            v = F::template value<AIH_F16_IEEE>(w, lane);
        }
        out[t] = v;
    }
}

template <class F>
int launch_embed(aih_ctx *ctx, const void *table, int64_t vocab, int64_t dim, const int32_t *ids, int64_t n,
                 float *out)
{
    constexpr int QK = F::QK, BB = F::BB;
    const int64_t bpr = dim / QK;
    const uint64_t threads = (uint64_t)n * bpr * (QK / 4);
    const uint64_t want = (threads + 255) / 256;
    const uint64_t cap = (uint64_t)(ctx->cu_count > 0 ? ctx->cu_count : 256) * 16;
    const unsigned grid = (unsigned)(want < cap ? want : cap);
    hipLaunchKernelGGL((embed_kernel<F>), dim3(grid), dim3(256), 0, ctx->stream,
                       static_cast<const uint8_t *>(table), vocab, bpr * BB, bpr, ids, n, reinterpret_cast<f4 *>(out));
    return aih_launch_status();
}

template <class F, int KT, bool STREAM>
int launch_tiles(aih_ctx *ctx, const void *q, float *out, uint64_t n_blocks, int mode)
{
    const uint64_t groups = (n_blocks * (F::QK / 4) + 256 * KT - 1) / (256 * KT);
    const unsigned grid = (unsigned)std::min<uint64_t>(groups, 1u << 22);
    const uint8_t *qb = static_cast<const uint8_t *>(q);
    f4 *o = reinterpret_cast<f4 *>(out);
    if (mode == AIH_F16_REFCPU)
        hipLaunchKernelGGL((dequant_kernel<F, AIH_F16_REFCPU, KT, STREAM>), dim3(grid), dim3(256), 0, ctx->stream, qb, o,
                           n_blocks);
    else
        hipLaunchKernelGGL((dequant_kernel<F, AIH_F16_IEEE, KT, STREAM>), dim3(grid), dim3(256), 0, ctx->stream, qb, o,
                           n_blocks);
    return aih_launch_status();
}

// An output is there to be read: one that the 256 MB memory-side cache can hold
// is stored plainly, so that its reader finds it there.  Larger ones gain from
// non-temporal stores.  us for the call alone, and for it and an aih_add that
// reads all of the output, at K = 4096, plain against non-temporal:
//   Q6_K   8 MB  3.6, 9.9   against 3.7, 11.2      Q8_0  16 MB  5.0, 16.0 against 4.1, 18.7
//   Q4_K  67 MB 13.1, 37.1  against 11.6, 41.1     Q6_K  67 MB 13.4, 36.8 against 12.9, 40.8
//   Q6_K 134 MB 25.3, 69.7  against 24.3, 79.7     Q6_K 197 MB 39.8, 124 against 34.8, 121
// Fewer than five workgroups per CU at F::kTiles tiles each: one tile per thread
// (Q6_K 8 MB and its reader 9.9 us against 10.7 with four).
constexpr uint64_t kStreamBytes = 160u << 20;

template <class F>
int launch_type(aih_ctx *ctx, const void *q, float *out, uint64_t n_blocks, int mode)
{
    const uint64_t bytes = n_blocks * F::QK * sizeof(float), cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    if (bytes > kStreamBytes) return launch_tiles<F, F::kTiles, true>(ctx, q, out, n_blocks, mode);
    if (bytes >= 5 * cus * (4096 * F::kTiles)) return launch_tiles<F, F::kTiles, false>(ctx, q, out, n_blocks, mode);
    return launch_tiles<F, 1, false>(ctx, q, out, n_blocks, mode);
}

}  // namespace

int aih_launch_embed(aih_ctx *ctx, int type, const void *table, int64_t vocab, int64_t dim,
                     const int32_t *ids, int64_t n, float *out)
{
    if (n == 0) return AIH_OK;
    if (reinterpret_cast<uintptr_t>(out) % 16 != 0) return AIH_E_INVALID;
    switch (type) {
    case AIH_TYPE_Q4_K: return launch_embed<DQ4K>(ctx, table, vocab, dim, ids, n, out);
    case AIH_TYPE_Q6_K: return launch_embed<DQ6K>(ctx, table, vocab, dim, ids, n, out);
    case AIH_TYPE_Q8_0: return launch_embed<DQ80>(ctx, table, vocab, dim, ids, n, out);
    case AIH_TYPE_Q4_0: return launch_embed<DQ40>(ctx, table, vocab, dim, ids, n, out);
    default: return AIH_E_UNSUPPORTED;
    }
}

int aih_launch_dequant(aih_ctx *ctx, int type, const void *q, float *out,
                       uint64_t n_blocks, int f16_mode)
{
    if (reinterpret_cast<uintptr_t>(out) % 16 != 0) return AIH_E_INVALID;
    switch (type) {
    case AIH_TYPE_Q4_K: return launch_type<DQ4K>(ctx, q, out, n_blocks, f16_mode);
    case AIH_TYPE_Q6_K: return launch_type<DQ6K>(ctx, q, out, n_blocks, f16_mode);
    case AIH_TYPE_Q8_0: return launch_type<DQ80>(ctx, q, out, n_blocks, f16_mode);
    case AIH_TYPE_Q4_0: return launch_type<DQ40>(ctx, q, out, n_blocks, f16_mode);
    default: return AIH_E_UNSUPPORTED;
    }
}
