// aih_qgemm.hip -- prefill GEMM with the GGUF block dequantization fused in.
//
//   Y[m*N + n] = sum_k X[m*K + k] * W[n, k]        (m < M, n < N)
//
// This replaces, for M > 8, the reference's TempF32 -> DequantizeInto ->
// MatMulWeights sequence (AIHost/AIHost/Compute/TransformerBase.cs:254-271,
// ComputeOps.cs:761-861, ComputeOps.cs:275-309, ComputeShaders.cs:93-129): the
// F32 SIMT matmul over a dequantized scratch copy becomes one kernel that
// dequantizes tiles of W into LDS as fp16 and contracts them on the matrix
// cores (v_mfma_f32_32x32x16_f16, fp32 accumulation).
//
// Tiling.  X is first converted to fp16 in the context's workspace, stored in
// MFMA fragment order with a power of two per row (aih_operand.h; the
// conversion is aih_decoder.hip's x_tile_pre_kernel, which also computes the
// element-wise step before the GEMM when there is one).  A
// workgroup then owns a 128 (M) x 64 (N) tile of Y and walks K in super-steps
// of 256 elements: producer waves dequantize W for the next super-step
// into LDS while four consumer waves multiply the current one, their A
// fragments loaded straight from the tiled X (see qgemm_kernel).  Large grids
// use 256 x 64, 512 x 64 or 512 x 128 tiles with every wave in both roles
// (qgemm256_kernel); products whose grid leaves CUs idle split K over
// workgroups and sum the partials in a second pass (plan_gemm,
// launch_split_sum).  The epilogue stores Y or adds into it (the residual add
// of a layer), or is one of the fused ones below.
//
// Precision.  Both operands are rounded to fp16 (11-bit significand) and the
// products accumulate in fp32: normwise error near 3e-4 against the fp32
// reference.  Each activation row carries a power of two that keeps its
// largest value inside fp16's range (aih_operand.h), undone exactly in the
// fp32 epilogue, so that rows above 65504 or far below 1 keep their 11 bits.
// bf16 operands (8-bit significand) would give about 2.4e-3, more than the
// 1e-3 the path is held to.  Weights are dequantized in fp32 with the
// reference's formulas (ComputeOps.cs:1629-1678 for Q4_K, :1735-1774 for Q6_K,
// the GGUF definitions for Q8_0 and Q4_0), computed as one fused fp32
// multiply-add per weight with fp16 output (aih_pieces.h).
#include "aih_pieces.h"
#include "aih_operand.h"

#include <type_traits>

namespace {

using namespace aih_pieces;
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int BM = 128;          // activation rows per workgroup
constexpr int BN = 64;           // weight rows per workgroup
constexpr int BK = 64;           // K granularity (one 64-element chunk)

// Workgroup barrier for LDS traffic only: waits for this wave's LDS
// operations, then for every wave.  __syncthreads() would also wait for the
// global loads in flight (its fences cover global memory), draining the
// prefetch at every step.  The "memory" clobber keeps the compiler from
// moving LDS accesses across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Epilogues: 0 store Y, 1 add into Y, 2 the SiLU-pairs operand (below).
constexpr int kEpiStore = 0, kEpiAccumulate = 1, kEpiSiluOperand = 2, kEpiRopeQKV = 3;

// SiLU(gate) * up of a wave's 32 x 64 output block whose column pairs
// (2j, 2j+1) are gate and up rows (W interleaved), written as the fp16
// operand image of a following GEMM with K = N / 2 (aih_operand.h).  The
// wave's block is one 32-column block of that operand, so each of its rows
// gets its own block exponent; the row exponents are 0, and the image's
// fixup pass (operand_fixup_kernel) brings every row to one exponent before
// that GEMM.  The 32 x 32 fp32 results pass through `lds` (32 rows x 36
// floats, private to the wave) so that every lane writes whole 16-byte
// fragment slots.  Rows at or past M are zero; m0w is the wave's first row,
// n0 the block's first column.  The arithmetic is silu_mul_pairs_kernel's,
// (g * (1 / (1 + e^-g))) * u in fp32, so a row within the unscaled window
// holds the bits the GEMM's own conversion of that kernel's output gives.
__device__ __forceinline__ void silu_pairs_operand(const f16v &acc0, const f16v &acc1, int lane, int64_t m0w,
                                                   int64_t n0, int64_t M, int64_t N, float *lds,
                                                   _Float16 *__restrict__ out)
{
    const int fr = lane & 31, hf = lane >> 5;
    constexpr int LS = 36;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        // the up value of this lane's column pair, from the odd neighbour
        const float u0 = __builtin_amdgcn_update_dpp(0.0f, acc0[r], 0xB1, 0xF, 0xF, false);
        const float u1 = __builtin_amdgcn_update_dpp(0.0f, acc1[r], 0xB1, 0xF, 0xF, false);
        if ((fr & 1) == 0) {
            const int i = 8 * (r >> 2) + 4 * hf + (r & 3);
            const float g0 = acc0[r], g1 = acc1[r];
            lds[i * LS + (fr >> 1)] = (g0 * (1.0f / (1.0f + expf(-g0)))) * u0;
            lds[i * LS + 16 + (fr >> 1)] = (g1 * (1.0f / (1.0f + expf(-g1)))) * u1;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // lane: row fr of the block, outputs 16 hf .. 16 hf + 15 (two slots)
    const int64_t m = m0w + fr;
    const int64_t mpad = aih_operand::mpad_of(M);
    if (m >= mpad) return;   // both lanes of a row (fr, fr + 32) alike
    f4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        v[q] = m < M ? *reinterpret_cast<const f4 *>(&lds[fr * LS + 16 * hf + 4 * q]) : f4{0.f, 0.f, 0.f, 0.f};
    float mx = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[q].x), fabsf(v[q].y)), fmaxf(fabsf(v[q].z), fabsf(v[q].w))));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const int eb = aih_operand::block_exp(mx), e = eb == aih_operand::kZeroBlock ? 0 : eb;
    const int64_t kd = N / 2;
    const int64_t k0 = n0 / 2 + 16 * hf;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        h8 h;
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = (_Float16)ldexpf(v[2 * q + j / 4][j % 4], e);
        *reinterpret_cast<h8 *>(out + aih_operand::slot_half(m, k0 + 8 * q, kd)) = h;
    }
    char *const img = reinterpret_cast<char *>(out);
    if (hf == 0) {
        reinterpret_cast<int8_t *>(img + aih_operand::block_exp_offset(mpad, kd))[m * (kd / 32) + n0 / 64] = (int8_t)eb;
        if (n0 == 0) reinterpret_cast<int32_t *>(img + aih_operand::row_exp_offset(mpad, kd))[m] = 0;
    }
}

// The row exponents of the operand (aih_operand.h) undone in a wave's 32 x 32
// accumulator: lane l holds rows 8 (r / 4) + 4 (l / 32) + r % 4 of the
// wave's 32 rows from row mrow0, whose exponents start at E + mrow0.  `ev`,
// loaded when the kernel started, is lane l's row l % 32 exponent: when all
// are zero (rows within the unscaled window) nothing is done.
typedef int32_t i4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void undo_row_exp(f16v &acc0, f16v &acc1, int32_t ev, const int32_t *E, int64_t mrow0,
                                             int lane)
{
    if (__builtin_amdgcn_ballot_w64(ev != 0) == 0) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const i4 e = *reinterpret_cast<const i4 *>(E + mrow0 + 8 * q + 4 * (lane >> 5));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc0[4 * q + j] = ldexpf(acc0[4 * q + j], -e[j]);
            acc1[4 * q + j] = ldexpf(acc1[4 * q + j], -e[j]);
        }
    }
}

// A wave's two 32 x 32 accumulators stored into Y (rows mrow0 .., columns
// n0 + lane % 32 and n0 + 32 + lane % 32), or added into it (Y + acc, the
// operand order of aih_add).  A block wholly inside Y is written without
// per-value guards, and for the add all 32 of its lane's Y values are loaded
// before the first add, so that they are in flight together rather than one
// round trip per register.  On MI355X, 4096 x 4096 x 512 per call: the
// accumulate epilogue 42.5 -> 33.5-34.4 us (the guarded form cost 3-5 us
// over a plain store).
__device__ __forceinline__ void store_tile(const f16v &acc0, const f16v &acc1, int lane, int64_t mrow0, int64_t n0,
                                           int64_t M, int64_t N, float *__restrict__ Y, bool accumulate)
{
    const int64_t na = n0 + (lane & 31), nb = na + 32;
    auto row = [&](int r) { return mrow0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); };
    if (mrow0 + 32 <= M && n0 + 64 <= N) {
        if (accumulate) {
            float ya[16], yb[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                ya[r] = Y[row(r) * N + na];
                yb[r] = Y[row(r) * N + nb];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                Y[row(r) * N + na] = ya[r] + acc0[r];
                Y[row(r) * N + nb] = yb[r] + acc1[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                Y[row(r) * N + na] = acc0[r];
                Y[row(r) * N + nb] = acc1[r];
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t m = row(r);
        if (m < M) {
            if (na < N) Y[m * N + na] = accumulate ? Y[m * N + na] + acc0[r] : acc0[r];
            if (nb < N) Y[m * N + nb] = accumulate ? Y[m * N + nb] + acc1[r] : acc1[r];
        }
    }
}

// The Q|K|V epilogue (aih_rope_qkv_args): a wave's two 32 x 32 blocks
// (rows mrow0 .., columns n0 + lane % 32 and + 32) rotated and stored as
// aih_rope_qkv would rotate and store the stored product: for query and key
// columns the pair (2i, 2i + 1) of a head (adjacent lanes) becomes
// (x0 c - x1 s, x0 s + x1 c) with (c, s) the table's row p, pair i; queries
// go to Y (unrotated when p is outside the table), keys and values to the
// caches' row p (nothing outside the table or past the cache).  The head
// boundaries fall on multiples of 32 columns, so a block is one kind.
__device__ __forceinline__ void rope_qkv_block(const f16v acc, int lane, int64_t mrow0, int64_t nb0, int64_t M,
                                               int64_t N, float *__restrict__ Y, const aih_rope_qkv_args ra)
{
#pragma clang fp contract(off)
    if (nb0 >= N) return;
    const int32_t p0 = ra.start + (ra.pos ? *ra.pos : 0);
    const int64_t n = nb0 + (lane & 31);
    // query, key or value: the same for the whole block (wave-uniform)
    const int kind = nb0 < ra.qd ? 0 : nb0 < (int64_t)ra.qd + ra.kvd ? 1 : 2;
    const int64_t cn = kind == 0 ? n : kind == 1 ? n - ra.qd : n - ra.qd - ra.kvd;
    auto row = [&](int r) { return mrow0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); };
    if (kind == 2) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t m = row(r), p = (int64_t)p0 + m;
            if (m < M && p >= 0 && p < ra.table_rows && p < ra.cache_rows) ra.Vc[p * ra.kvd + cn] = acc[r];
        }
        return;
    }
    // the rows' cos/sin, all loads issued before the first use (rows outside
    // the table read row 0 and are not rotated)
    const int half = ra.head_dim / 2;
    const int i = (int)(cn % ra.head_dim) / 2;
    float cv[16], sv[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t p = (int64_t)p0 + row(r);
        const int64_t pt = p >= 0 && p < ra.table_rows ? p : 0;
        const float2 t = *reinterpret_cast<const float2 *>(ra.table + 2 * (pt * half + i));
        cv[r] = t.x;
        sv[r] = t.y;
    }
    const bool odd = lane & 1;
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        // the pair's other element, from the neighbouring lane
        const float other = __builtin_amdgcn_update_dpp(0.0f, acc[r], 0xB1, 0xF, 0xF, false);
        const float x0 = odd ? other : acc[r], x1 = odd ? acc[r] : other;
        v[r] = odd ? x0 * sv[r] + x1 * cv[r] : x0 * cv[r] - x1 * sv[r];
    }
    if (kind == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t m = row(r), p = (int64_t)p0 + m;
            if (m < M) Y[m * N + n] = p >= 0 && p < ra.table_rows ? v[r] : acc[r];
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t m = row(r), p = (int64_t)p0 + m;
            if (m < M && p >= 0 && p < ra.table_rows && p < ra.cache_rows) ra.Kc[p * ra.kvd + cn] = v[r];
        }
    }
}

__device__ __forceinline__ void rope_qkv_tile(const f16v &acc0, const f16v &acc1, int lane, int64_t mrow0, int64_t n0,
                                              int64_t M, int64_t N, float *__restrict__ Y,
                                              const aih_rope_qkv_args ra)
{
    rope_qkv_block(acc0, lane, mrow0, n0, M, N, Y, ra);
    rope_qkv_block(acc1, lane, mrow0, n0 + 32, M, N, Y, ra);
}

// Waves in two roles: eight producers (four for Q8_0) and four consumers, one
// consumer per SIMD; the workgroup owns a 128 (M) x 64 (N) tile of Y and walks
// K in super-steps of 256 (a Q4_K/Q6_K super-block, 8 blocks of Q8_0/Q4_0),
// with one LDS barrier per super-step and two tile buffers.
//   Producers (waves 4..) dequantize the next super-step of the 64 weight
//   rows into LDS: each owns RPW consecutive rows.  For Q4_K, Q4_0 and Q8_0
//   eight lanes per row take 32 weights each (the wide-tile kernel's pieces
//   and LDS positions); for Q6_K sixteen lanes per row take pieces 0..15 of
//   the row's 256-k span (each row read as one contiguous span), which
//   measured faster there.  Their packed loads run PR super-steps ahead in a
//   ring of register sets.  A single producer wave per SIMD issues its
//   dependent conversions at 5 to 7 cycles each; two fill each other's gaps
//   (4096 x 4096 x 512 per call, four against eight producers: 3% in all three
//   formats, Q4_K 32.8 -> 31.8 us; 4096 x 14336 x 33 unsplit, Q4_K 69.3 ->
//   59.4).  Twelve waves leave 168 registers a lane: the wave index is held in a
//   scalar register, or a few would be kept in private memory.  Q8_0, bound by its 34-byte blocks' unaligned loads,
//   gained nothing there and lost 1-3% where its weights fill the memory
//   (32000 x 14336 x 64: 198 against 203 us): it keeps four.
//   Consumers (waves 0..3): wave w owns rows 32w .. 32w+31 of the M tile and
//   all 64 columns (two 32x32 accumulators sharing each A fragment).  A
//   fragments come straight from the tiled fp16 copy of X, one super-step
//   ahead; B fragments from LDS.
// On MI355X the 4096 x 4096 x 512 Q4_K product takes 32-35 us per call (the
// kernel about 25 us, the X conversion 7.5 us).
constexpr int SK = 256;            // k per super-step (one barrier)
constexpr int SC = SK / 64;        // 64-k steps per super-step
constexpr int LD2 = SK + 8;        // LDS row stride in halves (16-byte pad against bank conflicts)
// producer waves, their ring depth in super-steps (Q6_K's larger raw sets: 2)
// and piece layout (P32: 32-weight pieces, else 16-weight)
template <class T> struct GRing { static constexpr int NP = 8, PR = 3; static constexpr bool P32 = true; };
template <> struct GRing<G6K> { static constexpr int NP = 8, PR = 2; static constexpr bool P32 = false; };
template <> struct GRing<G80> { static constexpr int NP = 4, PR = 3; static constexpr bool P32 = true; };

// LDS position (in 16-byte granules) of chunk granule g of a super-step (the
// k values 8g .. 8g+7): the 32-weight pieces' swizzle, or for 16-weight
// pieces s of chunk c (granules 8c + 2s, + 1) 4c + s and 16 + 4c + s, so that
// the 16 lanes of a row store 256 contiguous bytes
template <class T, bool P32 = GRing<T>::P32> struct BPos {
    __device__ static constexpr int pos(int g) { return Piece32<T>::type::swz(g); }
};
template <class T> struct BPos<T, false> {
    __device__ static constexpr int pos(int g) { return 16 * (g & 1) + 4 * (g >> 3) + ((g >> 1) & 3); }
};

template <class T>
__global__ void __launch_bounds__(64 * (4 + GRing<T>::NP))
qgemm_kernel(const uint8_t *W, int64_t N, int64_t K, int64_t row_bytes,
             const _Float16 *__restrict__ Xt, int64_t M, float *__restrict__ Y, int epi, float *__restrict__ P,
             int64_t zs, int ssper, aih_rope_qkv_args ra)
{
    constexpr int PR = GRing<T>::PR;
    constexpr bool P32 = GRing<T>::P32;
    typedef typename Piece32<T>::type Pc;
    typedef std::conditional_t<P32, typename Pc::Raw, typename T::Raw> Raw;
    constexpr int RPW = BN / GRing<T>::NP;   // weight rows per producer wave
    constexpr int NR = P32 ? RPW / 8 : RPW / 4;   // row groups per producer wave
    __shared__ __align__(16) _Float16 wsh[2][BN][LD2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;
    const int nch = (int)(K / 64);
    // split z of K (gridDim.z > 1: partial sums into P + z * zs): super-steps
    // ss0 .. ss0 + nss - 1; chunk indices below stay absolute
    const int ss0 = (int)blockIdx.z * ssper;
    const int nss = min(ssper, (nch + SC - 1) / SC - ss0);

    if (wave >= 4) {
        // rows RPW pw + (RPW / NR) i + rl; P32: chunk pc, half ps of it (32
        // weights); else chunk pc, piece ps (16 weights)
        const int pw = wave - 4;
        constexpr int LPR = 64 * NR / RPW;   // lanes per row
        const int rl = lane / LPR, p = lane % LPR, pc = p / (LPR / 4), ps = p % (LPR / 4);
        const uint8_t *wrow[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int64_t wn = n0 + RPW * pw + (RPW / NR) * i + rl;
            wrow[i] = W + (wn < N ? wn : N - 1) * row_bytes;
        }
        auto gload = [&](int ss, Raw *r) {
            int c = (ss0 + ss) * SC + pc;
            c = c < nch ? c : nch - 1;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                if constexpr (P32) Pc::load(wrow[i], c, ps, r[i]);
                else T::load(wrow[i], c, ps, r[i]);
            }
        };
        // chunks past K exist only in a last, partial super-step, staged as
        // zeros: only the stages after the main loop test for them
        auto stage = [&](auto tail, int ss, int buf, const Raw *r) {
            asm volatile("" : "+s"(ss));
            const int c = (ss0 + ss) * SC + pc;
            const bool zero = decltype(tail)::value && c >= nch;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                _Float16 *d = &wsh[buf][RPW * pw + (RPW / NR) * i + rl][0];
                if constexpr (P32) {
                    h8 o[4];
                    Pc::piece(r[i], c, ps, o);
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<h8 *>(d + 8 * Pc::swz(8 * pc + Pc::col(ps, q) / 8)) = zero ? h8{} : o[q];
                } else {
                    h8 lo, hi;
                    piece16h<T>(r[i], c, ps, lo, hi);
                    *reinterpret_cast<h8 *>(d + 8 * BPos<T>::pos(8 * pc + 2 * ps)) = zero ? h8{} : lo;
                    *reinterpret_cast<h8 *>(d + 8 * BPos<T>::pos(8 * pc + 2 * ps + 1)) = zero ? h8{} : hi;
                }
            }
        };
        Raw ring[PR][NR];
#pragma unroll
        for (int j = 0; j < PR; ++j) gload(j, ring[j]);
        __builtin_amdgcn_sched_barrier(0);
        int ss = 0;
        for (; ss + 2 * PR <= nss; ss += PR) {
#pragma unroll
            for (int j = 0; j < PR; ++j) {
                stage(std::false_type{}, ss + j, (ss + j) & 1, ring[j]);
                gload(ss + j + PR, ring[j]);
                __builtin_amdgcn_sched_barrier(0);
                lds_barrier();
            }
        }
#pragma unroll
        for (int j = 0; j < PR; ++j) {
            if (ss + j < nss) {
                stage(std::true_type{}, ss + j, (ss + j) & 1, ring[j]);
                if (ss + j + PR < nss) gload(ss + j + PR, ring[j]);
                lds_barrier();
            }
        }
#pragma unroll
        for (int j = 0; j < PR; ++j) {
            if (ss + PR + j < nss) {
                stage(std::true_type{}, ss + PR + j, (ss + PR + j) & 1, ring[j]);
                lds_barrier();
            }
        }
        return;
    }

    // consumer wave w: rows 32w .. 32w+31 of the M tile, all 64 columns
    const int fr = lane & 31, fk = 8 * (lane >> 5);
    const int64_t kc = K / 16, mblocks = (M + 31) / 32;
    int64_t mb = (m0 + 32 * wave) / 32;
    mb = mb < mblocks ? mb : mblocks - 1;
    const _Float16 *xa = Xt + (mb * kc * 64 + lane) * 8;
    // the row exponents of the operand, after its mblocks * 32 rows of values
    const int32_t *const E = reinterpret_cast<const int32_t *>(Xt + mblocks * 32 * K);
    const int32_t ev = E[mb * 32 + (lane & 31)];
    struct AF { h8 a[4]; };
    auto aload = [&](int kb, AF &f) {
        kb += SC * ss0;
        kb = kb < nch ? kb : nch - 1;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) f.a[kk] = ldg<h8>(xa + ((int64_t)kb * 4 + kk) * 512);
    };
    f16v acc0 = {}, acc1 = {};
    // B fragments of one 64-k step (both 32-column halves, four k16 slices),
    // read from LDS one step ahead of their MFMAs so that the reads' latency
    // is covered by the previous step's matrix work
    struct BF { h8 b0[4], b1[4]; };
    auto bload = [&](int buf, int t, BF &b) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            b.b0[kk] = *reinterpret_cast<const h8 *>(&wsh[buf][fr][8 * BPos<T>::pos(8 * t + 2 * kk + fk / 8)]);
            b.b1[kk] = *reinterpret_cast<const h8 *>(&wsh[buf][32 + fr][8 * BPos<T>::pos(8 * t + 2 * kk + fk / 8)]);
        }
    };
    auto mm = [&](const AF &f, const BF &b) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            acc0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[kk], b.b0[kk], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[kk], b.b1[kk], acc1, 0, 0, 0);
        }
    };
    // A ring of one super-step: slot t holds 64-k step SC*ss + t
    AF f[SC];
#pragma unroll
    for (int t = 0; t < SC; ++t) aload(t, f[t]);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    BF bb[2];
    int ss = 0;
    for (; ss + 2 <= nss; ++ss) {
        const int buf = ss & 1;
        bload(buf, 0, bb[0]);
#pragma unroll
        for (int t = 0; t < SC; ++t) {
            if (t + 1 < SC) bload(buf, t + 1, bb[(t + 1) & 1]);
            mm(f[t], bb[t & 1]);
            aload(SC * (ss + 1) + t, f[t]);
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();
    }
    {
        const int buf = ss & 1;
        bload(buf, 0, bb[0]);
#pragma unroll
        for (int t = 0; t < SC; ++t) {
            if (t + 1 < SC && SC * (ss0 + ss) + t + 1 < nch) bload(buf, t + 1, bb[(t + 1) & 1]);
            if (SC * (ss0 + ss) + t < nch) mm(f[t], bb[t & 1]);
        }
    }

    if (P) {   // a split's partial sums (the summing pass undoes the exponents and applies the epilogue)
        store_tile(acc0, acc1, lane, m0 + 32 * wave, n0, M, N, P + (int64_t)blockIdx.z * zs, false);
        return;
    }
    undo_row_exp(acc0, acc1, ev, E, mb * 32, lane);
    if (epi == kEpiSiluOperand) {
        // the tile buffer of super-step nss: nothing reads or writes it any more
        silu_pairs_operand(acc0, acc1, lane, m0 + 32 * wave, n0, M, N,
                           reinterpret_cast<float *>(&wsh[nss & 1][0][0]) + wave * 32 * 36,
                           reinterpret_cast<_Float16 *>(Y));
        return;
    }
    if (epi == kEpiRopeQKV) {
        rope_qkv_tile(acc0, acc1, lane, m0 + 32 * wave, n0, M, N, Y, ra);
        return;
    }
    store_tile(acc0, acc1, lane, m0 + 32 * wave, n0, M, N, Y, epi == kEpiAccumulate);
}

// Wide tiles for large products: a workgroup of eight waves owns a 256 MB (M)
// x 64 NB (N) tile (MB, NB = 1 or 2), so each dequantized weight feeds 2 MB
// times as many outputs as in qgemm_kernel.  Every wave takes both roles in each
// super-step s:
//   - it dequantizes its 8 NB of the 64 NB weight rows (rows 64 i + 8w + lane / 8) for
//     super-step s+1 into the other LDS buffer, 32 weights per lane
//     (Piece32), from packed loads PR256 (NB = 2: one) super-steps ahead (Q6_K: see LATE);
//   - it multiplies super-step s: wave w owns rows 32 MB w .. +32 MB - 1 of
//     the M tile and all 64 NB columns (2 MB NB 32x32 accumulators: each A fragment
//     feeds 2 NB, each B fragment MB), A fragments from the tiled X AD 64-k
//     chunks ahead, B fragments from LDS.
// The two waves of a SIMD (w and w + 4) run the two halves in opposite
// orders, so that one dequantizes while the other multiplies.  On MI355X a
// 256-row workgroup takes about 1.25 times as long as a 128-row one, for
// twice the outputs.
// With 64 columns every A fragment is loaded for two MFMAs, 64 bytes per clock
// and CU through the vector L1 at the full MFMA rate, which is all it gives.
// Counters of the 512 x 64 tile (14336 x 4096 x 512, its 224 CUs): 28 bytes per
// clock, the L1's return path busy 74% of the time, the MFMAs 42%.  The 512 x 128
// tile (NB = 2) halves those loads (x 2048: return path 70%, MFMAs 54% of all
// CUs, where the 256 x 64 tile has 80% and 43%); its 128 accumulator registers
// leave room for A one 64-k chunk and B one 16-k slice ahead.  Per call, Q4_K K =
// 4096: 14336 x 2048 301 -> 245 us, 28672 x 512 145 -> 123 us.  Left out one at a time (a copy, 237 us): the
// A loads -26 us, the dequantization -36 us, both -55 us: what remains is the
// MFMAs, and the last round of workgroups.
constexpr int BM2 = 256;
constexpr int PR256 = 2;

// This lane's index, computed again: the epilogue of the 512 x 128 tile would
// otherwise hold it, and what is derived from it, in registers that the loop
// then spills.
__device__ __forceinline__ int lane_id()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

template <class T, int MB, int NB, int AD>
__global__ void __launch_bounds__(512)
qgemm256_kernel(const uint8_t *W, int64_t N, int64_t K, int64_t row_bytes,
                const _Float16 *__restrict__ Xt, int64_t M, float *__restrict__ Y, int epi,
                float *__restrict__ P, int64_t zs, int ssper, aih_rope_qkv_args ra)
{
    static_assert(SC % AD == 0, "A ring depth divides a super-step");
    constexpr int PR = NB == 1 ? PR256 : 1;
    // Q6_K's 36 registers of packed weights do not fit beside the 512 x 128
    // accumulators all the way (spilled, they wait for their own loads): they
    // are loaded in the last chunk before their use, the others a super-step
    // ahead (Q8_0 loaded late: 3.5% slower).  With the wave index held in a
    // scalar register (A's addresses too), nothing is spilled in the loop;
    // 14336 x 4096 x 2048: Q6_K 283 -> 268 us, Q4_K 242 -> 236.
    constexpr bool LATE = NB > 1 && std::is_same<T, G6K>::value;
    typedef typename Piece32<T>::type Pc;
    typedef typename Pc::Raw Raw;
    __shared__ __align__(16) _Float16 wsh[2][BN * NB][LD2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t m0 = (int64_t)blockIdx.y * BM2 * MB, n0 = (int64_t)blockIdx.x * (BN * NB);
    const int nch = (int)(K / 64);
    // split z of K (gridDim.z > 1: partial sums into P + z * zs): super-steps
    // ss0 .. ss0 + nss - 1; chunk indices below stay absolute
    const int ss0 = (int)blockIdx.z * ssper;
    const int nss = min(ssper, (nch + SC - 1) / SC - ss0);

    // dequantization share: rows 64 i + 8 wave + rl, 32 weights per lane (chunk pc, half ph)
    const int rl = lane >> 3, p = lane & 7, pc = p >> 1, ph = p & 1;
    const uint8_t *wrow[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int64_t wn = n0 + 64 * i + 8 * wave + rl;
        wrow[i] = W + (wn < N ? wn : N - 1) * row_bytes;
    }
    auto gload = [&](int ss, Raw *r) {
        int c = (ss0 + ss) * SC + pc;
        c = c < nch ? c : nch - 1;
#pragma unroll
        for (int i = 0; i < NB; ++i) Pc::load(wrow[i], c, ph, r[i]);
    };
    // LDS positions of this lane in one index each (swz permutes the bits of a
    // granule's index and leaves bit 0 in place): where it stores piece 0, and
    // where it reads granule 2u + (lane / 32)
    const int wat = (8 * wave + rl) * LD2 + 8 * Pc::swz(8 * pc + Pc::col(ph, 0) / 8);
    const int rat = (lane & 31) * LD2 + 8 * (lane >> 5);
    // chunks past K exist only in a last, partial super-step, staged as zeros
    auto stage = [&](auto tail, int ss, int buf, const Raw *r) {
        const int c = (ss0 + ss) * SC + pc;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            h8 o[4];
            Pc::piece(r[i], c, ph, o);
            _Float16 *d = &wsh[buf][64 * i][0] + wat;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<h8 *>(d + 8 * Pc::swz(Pc::col(0, q) / 8)) =
                    decltype(tail)::value && c >= nch ? h8{} : o[q];
            if (NB > 1) __builtin_amdgcn_sched_barrier(0);   // one row's temporaries at a time
        }
    };

    // multiplication share: rows 32 MB wave .. +32 MB - 1 of the M tile, all columns
    const int fr = lane & 31, fk = 8 * (lane >> 5);
    const int64_t kc = K / 16, mblocks = (M + 31) / 32;
    const _Float16 *xa[MB];
    const int32_t *const E = reinterpret_cast<const int32_t *>(Xt + mblocks * 32 * K);
    int32_t ev[MB];   // the row exponents of the operand (lane: row lane % 32 of fragment j)
#pragma unroll
    for (int j = 0; j < MB; ++j) {
        int64_t mb = (m0 + 32 * (MB * wave + j)) / 32;
        mb = mb < mblocks ? mb : mblocks - 1;
        xa[j] = Xt + (mb * kc * 64 + lane) * 8;
        if (NB == 1) ev[j] = E[mb * 32 + (lane & 31)];
    }
    struct AF { h8 a[MB][4]; };
    auto aload = [&](int kb, AF &f) {
        kb += SC * ss0;
        kb = kb < nch ? kb : nch - 1;
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) f.a[j][kk] = ldg<h8>(xa[j] + ((int64_t)kb * 4 + kk) * 512);
    };
    f16v acc[MB][2 * NB] = {};
    struct BF { h8 b0[4], b1[4]; };
    auto bload = [&](int buf, int t, BF &b) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            b.b0[kk] = *reinterpret_cast<const h8 *>(&wsh[buf][fr][8 * Pc::swz(8 * t + 2 * kk + fk / 8)]);
            b.b1[kk] = *reinterpret_cast<const h8 *>(&wsh[buf][32 + fr][8 * Pc::swz(8 * t + 2 * kk + fk / 8)]);
        }
    };
    auto mm = [&](const AF &f, const BF &b) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int j = 0; j < MB; ++j) {
                acc[j][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[j][kk], b.b0[kk], acc[j][0], 0, 0, 0);
                acc[j][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[j][kk], b.b1[kk], acc[j][1], 0, 0, 0);
            }
    };

    // NB = 2: the B fragments of one k16 slice u of a super-step (all 128
    // columns), one slice ahead of their MFMAs
    struct BS { h8 b[2 * NB]; };
    auto bslice = [&](int buf, int u, BS &b) {
#pragma unroll
        for (int i = 0; i < 2 * NB; ++i)
            b.b[i] = *reinterpret_cast<const h8 *>(&wsh[buf][32 * i][8 * Pc::swz(2 * u)] + rat);
    };

    // Iteration it: products of super-step it from buffer it & 1, and, if
    // `more`, the dequantization of super-step it + 1 into the other buffer
    // from ring slot r, whose loads are then reissued for super-step
    // it + 1 + PR when `reload`.
    Raw ring[PR][NB];
    AF f[AD];   // chunk g of the A operand in f[g % AD]
    constexpr int BD = MB == 1 ? 2 : 1;   // B chunks in registers (the next one loaded early when 2)
    BF bb[BD];
    BS bs[2];
    // The two waves of a SIMD (w and w + 4) take the two halves in opposite
    // orders, so that one dequantizes while the other multiplies.
    const bool valu_first = wave < 4;
    auto body = [&](auto tail, int it, Raw *r, bool more, bool reload) {
        const int buf = it & 1;
        auto deq = [&] {
            if (more) {
                stage(tail, it + 1, buf ^ 1, r);
                if (reload && !LATE) gload(it + 1 + PR, r);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (NB == 1 && BD == 2) bload(buf, 0, bb[0]);
        if (valu_first) deq();
        // the multiplying half at raised wave priority, so that the SIMD
        // issues its MFMAs ahead of the other wave's dequantization when both
        // are ready (6144 x 4096 and 28672 x 4096 at M = 512: 2% faster)
        __builtin_amdgcn_s_setprio(1);
        if constexpr (NB > 1) {
            bslice(buf, 0, bs[0]);
#pragma unroll
            for (int u = 0; u < 4 * SC; ++u) {
                if (u + 1 < 4 * SC) bslice(buf, u + 1, bs[(u + 1) & 1]);
                if (LATE && u == 4 * (SC - 1)) gload(it + (valu_first ? 2 : 1), r);
                __builtin_amdgcn_sched_barrier(0);
                AF &a = f[(u >> 2) % AD];
#pragma unroll
                for (int i = 0; i < 2 * NB; ++i)
#pragma unroll
                    for (int j = 0; j < MB; ++j)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.a[j][u & 3], bs[u & 1].b[i], acc[j][i], 0, 0, 0);
                // this slice's A fragments, AD chunks ahead
                int kb = SC * (ss0 + it) + (u >> 2) + AD;
                kb = kb < nch ? kb : nch - 1;
#pragma unroll
                for (int j = 0; j < MB; ++j) a.a[j][u & 3] = ldg<h8>(xa[j] + ((int64_t)kb * 4 + (u & 3)) * 512);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else
#pragma unroll
        for (int t = 0; t < SC; ++t) {
            if (BD == 1)
                bload(buf, t, bb[0]);
            else if (t + 1 < SC)
                bload(buf, t + 1, bb[(t + 1) % BD]);
            __builtin_amdgcn_sched_barrier(0);
            mm(f[t % AD], bb[t % BD]);
            aload(SC * it + t + AD, f[t % AD]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        if (!valu_first) deq();
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
    };

#pragma unroll
    for (int j = 0; j < PR; ++j) gload(j, ring[j]);
#pragma unroll
    for (int t = 0; t < AD; ++t) aload(t, f[t]);
    stage(std::true_type{}, 0, 0, ring[0]);
    gload(PR, ring[0]);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    // iteration it stages super-step it + 1 from ring slot (it + 1) % PR; the
    // main loop's stages are all full super-steps before the last
    int ss = 0;
    for (; ss + PR + 1 < nss; ss += PR) {
#pragma unroll
        for (int j = 0; j < PR; ++j) body(std::false_type{}, ss + j, ring[(j + 1) % PR], true, true);
    }
#pragma unroll
    for (int j = 0; j <= PR; ++j) {
        const int it = ss + j;
        if (it < nss) body(std::true_type{}, it, ring[(j + 1) % PR], it + 1 < nss, it + 1 + PR < nss);
    }

    const int el = lane_id();
    if (!P) {   // the summing pass undoes a split's
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            int64_t mb = (m0 + 32 * (MB * wave + j)) / 32;
            mb = mb < mblocks ? mb : mblocks - 1;
            if (NB > 1) ev[j] = E[mb * 32 + (el & 31)];
#pragma unroll
            for (int i = 0; i < NB; ++i) undo_row_exp(acc[j][2 * i], acc[j][2 * i + 1], ev[j], E, mb * 32, el);
        }
    }
    // every 32 x 64 block b = j NB + i (row fragment j, column pair i) of the
    // wave, unrolled by hand: the epilogues are too large for the pragma
    auto each = [&](auto f) {
        f(std::integral_constant<int, 0>{});
        if constexpr (MB * NB > 1) f(std::integral_constant<int, 1>{});
        if constexpr (MB * NB > 2) {
            f(std::integral_constant<int, 2>{});
            f(std::integral_constant<int, 3>{});
        }
    };
    if (epi == kEpiSiluOperand) {
        // after the last barrier the tile buffers are free (N is a multiple of 64)
        each([&](auto bc) {
            constexpr int b = decltype(bc)::value;
            if (NB == 1 || n0 + 64 * (b % NB) < N)
                silu_pairs_operand(acc[b / NB][2 * (b % NB)], acc[b / NB][2 * (b % NB) + 1], el,
                                   m0 + 32 * (MB * wave + b / NB), n0 + 64 * (b % NB), M, N,
                                   reinterpret_cast<float *>(&wsh[0][0][0]) + wave * 32 * 36,
                                   reinterpret_cast<_Float16 *>(Y));
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the block is read before it is rewritten
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        });
        return;
    }
    if (epi == kEpiRopeQKV) {   // never split here (the plan splits this epilogue over 128-row tiles only)
        each([&](auto bc) {
            constexpr int j = decltype(bc)::value / NB, i = decltype(bc)::value % NB;
            rope_qkv_tile(acc[j][2 * i], acc[j][2 * i + 1], el, m0 + 32 * (MB * wave + j), n0 + 64 * i, M, N, Y, ra);
        });
        return;
    }
    // a split's partial sums are stored (the summing pass adds them into Y)
    float *const Pz = P ? P + (int64_t)blockIdx.z * zs : nullptr;
    each([&](auto bc) {
        constexpr int j = decltype(bc)::value / NB, i = decltype(bc)::value % NB;
        store_tile(acc[j][2 * i], acc[j][2 * i + 1], el, m0 + 32 * (MB * wave + j), n0 + 64 * i, M, N, Pz ? Pz : Y,
                   !Pz && epi == kEpiAccumulate);
    });
}

// Partial sums keep their row's power of two (aih_operand.h): those of a row of
// large values may exceed fp32 where their sum does not.  The summing passes
// undo it, row m's being E[m].
__device__ __forceinline__ f4 undo_row_exp4(f4 s, int e)
{
    return e == 0 ? s : f4{ldexpf(s.x, -e), ldexpf(s.y, -e), ldexpf(s.z, -e), ldexpf(s.w, -e)};
}

// The sum of the splits' partial sums p[0], p[zs], ... (in that order).
__device__ __forceinline__ f4 split_sum4(const float *__restrict__ p, int S, int64_t zs)
{
    f4 s = *reinterpret_cast<const f4 *>(p);
    int z = 1;
    for (; z + 4 <= S; z += 4) {   // four splits' loads in flight
        f4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const f4 *>(p + (int64_t)(z + j) * zs);
#pragma unroll
        for (int j = 0; j < 4; ++j) s += v[j];
    }
    for (; z < S; ++z) s += *reinterpret_cast<const f4 *>(p + (int64_t)z * zs);
    return s;
}

// The splits of a GEMM split over K: Y = P_0 + P_1 + ... (in that order),
// added into Y (Y + sum, the order of the accumulate epilogue) when
// `accumulate`.  Splits are zs floats apart (a multiple of 4, at least MN).
// Four elements per thread (16-byte accesses of Y when it is 16-byte aligned);
// ROWS4: N >= 4.  MN fits 32 bits: a split product has fewer tiles than the device has CUs.
template <bool VEC, bool ROWS4>
__global__ void __launch_bounds__(256)
split_k_sum_kernel(const float *__restrict__ P, int S, int64_t MN, uint32_t M, uint32_t N, int64_t zs,
                   const int32_t *__restrict__ E, float *__restrict__ Y, int accumulate)
{
    for (int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < MN; i += 4 * (int64_t)gridDim.x * 256) {
        // Four elements lie in the row of element i and the next one (N >= 4), or
        // past the end; their exponents are in flight beside the partials.
        const uint32_t m = (uint32_t)i / N, in_row = (m + 1) * N - (uint32_t)i;   // elements left in row m
        const int e0 = E[m], e1 = E[min(m + 1, M - 1)];
        f4 s = split_sum4(P + i, S, zs);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (ROWS4) s[j] = ldexpf(s[j], j < in_row ? -e0 : -e1);
            else s[j] = ldexpf(s[j], -E[min((uint32_t)i + j, (uint32_t)MN - 1) / N]);
        }
        if (VEC && i + 4 <= MN) {
            f4 *y = reinterpret_cast<f4 *>(Y + i);
            *y = accumulate ? *y + s : s;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i + j < MN) Y[i + j] = accumulate ? Y[i + j] + s[j] : s[j];
        }
    }
}

// The same sum with the Q|K|V epilogue: what rope_qkv_block stores, two pairs
// (four columns) per thread, one row (of at most 256) per blockIdx.y.  N and the
// head boundaries are multiples of 32.
__global__ void __launch_bounds__(256)
split_k_rope_kernel(const float *__restrict__ P, int S, int64_t N, int64_t zs,
                    const int32_t *__restrict__ E, float *__restrict__ Y, const aih_rope_qkv_args ra)
{
#pragma clang fp contract(off)
    const int64_t m = blockIdx.y, n = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x), t = m * N + n;
    if (n >= N) return;
    const int e = E[m];
    const f4 x = undo_row_exp4(split_sum4(P + t, S, zs), e);
    const int64_t p = (int64_t)ra.start + (ra.pos ? *ra.pos : 0) + m;
    const bool in_table = p >= 0 && p < ra.table_rows, in_cache = in_table && p < ra.cache_rows;
    const int kind = n < ra.qd ? 0 : n < (int64_t)ra.qd + ra.kvd ? 1 : 2;
    f4 v = x;
    if (kind < 2 && in_table) {
        const int64_t cn = kind == 0 ? n : n - ra.qd;
        const float *c = ra.table + 2 * (p * (ra.head_dim / 2) + cn % ra.head_dim / 2);
        v = f4{x.x * c[0] - x.y * c[1], x.x * c[1] + x.y * c[0], x.z * c[2] - x.w * c[3], x.z * c[3] + x.w * c[2]};
    }
    float *to;
    if (kind == 0) to = Y + t;
    else if (!in_cache) return;
    else if (kind == 1) to = ra.Kc + p * ra.kvd + (n - ra.qd);
    else to = ra.Vc + p * ra.kvd + (n - ra.qd - ra.kvd);
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = v[j];
}

// The same sum with the SiLU-pairs operand epilogue: what silu_pairs_operand
// writes.  Thread t of a row holds 16 columns (8 outputs, one 16-byte slot of
// the image); the four threads of a 32-output block share its exponent.
// N is a multiple of 64; rows M .. mpad - 1 are zero.
__global__ void __launch_bounds__(256)
split_k_silu_kernel(const float *__restrict__ P, int S, int64_t M, int64_t N, int64_t zs,
                    const int32_t *__restrict__ E, _Float16 *__restrict__ out)
{
    const int64_t mpad = aih_operand::mpad_of(M), kd = N / 2, per_row = N / 16;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t m = t / per_row, c = t % per_row;
    const bool live = m < M;   // whole groups of four threads alike (per_row is a multiple of 4)
    float v[8] = {};
    if (live) {
        const int e = E[m];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f4 x = undo_row_exp4(split_sum4(P + m * N + 16 * c + 4 * q, S, zs), e);
            v[2 * q] = (x.x * (1.0f / (1.0f + expf(-x.x)))) * x.y;
            v[2 * q + 1] = (x.z * (1.0f / (1.0f + expf(-x.z)))) * x.w;
        }
    }
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(v[j]));
    mx = fmaxf(mx, __shfl_xor(mx, 1));
    mx = fmaxf(mx, __shfl_xor(mx, 2));
    if (m >= mpad) return;
    const int eb = aih_operand::block_exp(mx), e = eb == aih_operand::kZeroBlock ? 0 : eb;
    h8 h;
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = (_Float16)ldexpf(v[j], e);
    *reinterpret_cast<h8 *>(out + aih_operand::slot_half(m, 8 * c, kd)) = h;
    char *const img = reinterpret_cast<char *>(out);
    if (c % 4 == 0) reinterpret_cast<int8_t *>(img + aih_operand::block_exp_offset(mpad, kd))[m * (kd / 32) + c / 4] = (int8_t)eb;
    if (c == 0) reinterpret_cast<int32_t *>(img + aih_operand::row_exp_offset(mpad, kd))[m] = 0;
}

// Before a GEMM reads an image written one 32-column block at a time
// (aih_operand.h), every row is brought to one exponent: one wave per row.
// A row whose block exponents are all 0 (or mark all-zero blocks) -- its
// values within the unscaled window -- is left as it is.  Otherwise each
// block of exponent d is scaled to the row's smallest exponent D (the block
// of its largest values): every half multiplied by 2^(D - d) <= 1 in fp32
// (exact) and rounded to fp16 once; then E[m] += D and the block exponents
// become 0, so a second pass changes nothing.
__global__ void __launch_bounds__(256)
operand_fixup_kernel(_Float16 *__restrict__ Xt, int64_t mpad, int64_t K)
{
    const int lane = threadIdx.x & 63;
    const int64_t m = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= mpad) return;
    const int64_t nb = K / 32;   // a multiple of 2 (K % 64 == 0)
    char *const img = reinterpret_cast<char *>(Xt);
    int8_t *const d = reinterpret_cast<int8_t *>(img + aih_operand::block_exp_offset(mpad, K)) + m * nb;
    int mn = 127;
    bool odd = false;
    // the row's exponents two at a time (rows start 2-byte aligned), the loads
    // of four passes issued together (K up to 16384 in one round trip)
#pragma unroll 4
    for (int64_t b = 2 * lane; b < nb; b += 128) {
        const uint16_t w2 = *reinterpret_cast<const uint16_t *>(d + b);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int v = (int8_t)(w2 >> (8 * j));
            if (v != aih_operand::kZeroBlock) {
                mn = min(mn, v);
                odd = odd || v != 0;
            }
        }
    }
    if (__builtin_amdgcn_ballot_w64(odd) == 0) return;
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) mn = min(mn, __shfl_xor(mn, s));
    for (int64_t b = lane; b < nb; b += 64) {
        const int v = d[b];
        if (v != aih_operand::kZeroBlock && v != mn) {
            const float f = ldexpf(1.f, mn - v);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                h8 *const p = reinterpret_cast<h8 *>(Xt + aih_operand::slot_half(m, 32 * b + 8 * q, K));
                h8 h = *p;
#pragma unroll
                for (int j = 0; j < 8; ++j) h[j] = (_Float16)((float)h[j] * f);
                *p = h;
            }
        }
        d[b] = 0;
    }
    if (lane == 0) reinterpret_cast<int32_t *>(img + aih_operand::row_exp_offset(mpad, K))[m] += mn;
}

// The tiling of a GEMM: rows (128, 256 or 512) and columns (64; 128 for the
// widest, never split) per workgroup tile and, for
// 128- and 512-row tiles, the number of K splits (splits > 1: partial sums in
// the second workspace, then a summing pass) of ssper super-steps each.
struct GemmPlan {
    int tile = 128;
    int cols = BN;
    int splits = 1;
    int ssper = 0;
};

// 256-row tiles halve the dequantization per output and 512-row tiles halve
// it again; a workgroup of them takes about 1.25 and 2.35 times as long as
// one of 128 rows, one of 512 x 128 about 3.6 times (measured on MI355X;
// chip full, all four formats: 112-127 us a round of 4096 of K, against 68-76
// of 512 x 64; nearly empty 82 against 62: 3.6 lies between).  The units were
// fitted with four producer waves.  With eight, every tile forced in turn over
// 64 unsplit products (all formats, 257 to 2048 rows, N 1096 to 31832, K 1024 to
// 7936): the plan's is the fastest or within 2%, but for three Q4_0 products
// where 128 rows would be 6 to 10% faster than its 512 x 64.  The shape with
// the fewest such rounds of workgroups over the device's CUs wins (ties to the
// smaller tile).  Costs in units of 1/20 of a 128-row workgroup.  Products of more than 256
// rows whose 512-row tiles leave CUs idle split K over workgroups: S splits
// of at least two whole super-steps, partial sums in the second workspace,
// then a summing pass (estimated at 5 TB/s over the partials, Y and the
// output, plus 2 us of launch; a 128-row workgroup takes about 29 us per
// 4096 of K).  The plan depends only on the shape, the epilogue, the CU count
// and whether the call may split, never on what the context has allocated.
//
// Products of at most 256 rows split the 128-row tiles over K, at most 8 ways,
// when those leave CUs idle (a 4096-row weight has 64 tiles).  A workgroup
// takes about 3 us and 1.1 us per super-step, and the summing pass 4 us and
// its traffic at 2.5 TB/s.  Every entry point and epilogue splits a shape
// alike, so the operand image and the partial sums together stay within the
// allocation-free entry point's buffer.
// Measured per call (Q4_K / Q6_K, whole -> split): 4096 x 14336 x 33 70 -> 26
// / 83 -> 31 us, 4096 x 4096 x 33 23 -> 14 / 28 -> 16, x 256 26 -> 22 / 31 ->
// 25, 1024 x 14336 x 64 69 -> 19 / 82 -> 23, 8192 x 4096 x 9 24 -> 17 / 29 ->
// 21; over 216 sizes of N 1024-32000, K 1024-14336 and M 9-256 none slower
// than the runs differ.
int64_t split_stride(int64_t M, int64_t N) { return (M * N + 3) / 4 * 4; }

GemmPlan plan_gemm(int64_t cu_count, int64_t N, int64_t K, int64_t M, int epi, bool may_split)
{
    const int64_t gx = (N + BN - 1) / BN, gy = (M + BM - 1) / BM, gy2 = (M + BM2 - 1) / BM2;
    const int64_t gy4 = (M + 2 * BM2 - 1) / (2 * BM2);
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    auto rounds = [&](int64_t wgs) { return (double)((wgs + cus - 1) / cus); };
    const double c1 = 20 * rounds(gx * gy), c2 = 25 * rounds(gx * gy2), c4 = 47 * rounds(gx * gy4);
    const int nss = (int)((K / 64 + SC - 1) / SC);
    GemmPlan p;
    p.ssper = nss;
    if (M <= BM2) {
        const size_t image = (size_t)aih_operand::image_bytes(aih_operand::mpad_of(M), K, false);
        const size_t room = image < AIH_NOALLOC_SCRATCH_BYTES ? AIH_NOALLOC_SCRATCH_BYTES - image : 0;
        const double whole = 3.0 + 1.1 * nss;
        double best = std::min(c1, c2) / 20.0 * whole;
        for (int want = 2; want <= 8 && 2 * want <= nss; ++want) {
            const int ssper = (nss + want - 1) / want;
            const int S = (nss + ssper - 1) / ssper;
            const size_t bytes = (size_t)S * (size_t)split_stride(M, N) * sizeof(float);
            if (bytes > room) break;
            const double us = rounds(gx * gy * S) * (3.0 + 1.1 * ssper) + 4.0 + (double)bytes / 2.5e6;
            if (us < best) {
                best = us;
                p.splits = S;
                p.ssper = ssper;
            }
        }
        if (p.splits > 1) return p;
    }
    if (may_split && epi != kEpiSiluOperand && epi != kEpiRopeQKV && M > BM2 && gx * gy4 < cus && M * N % 4 == 0) {
        const int want = (int)std::min<int64_t>(std::min<int64_t>(cus / (gx * gy4), nss / 2), 8);
        if (want >= 2) {
            const int ssper = (nss + want - 1) / want;
            const int S = (nss + ssper - 1) / ssper;
            const double unit_us = 29.0 * (double)K / 4096.0 / 20.0;
            const double sum_us = (double)(S + 2) * (double)(M * N) * 4.0 / 5e12 * 1e6 + 2.0;
            const double cs = 47 * rounds(gx * gy4 * S) * (double)ssper / (double)nss + sum_us / unit_us;
            if (S > 1 && cs < c1 && cs < c2 && cs < c4) {
                p.tile = 512;
                p.splits = S;
                p.ssper = ssper;
                return p;
            }
        }
    }
    p.tile = c4 < c2 && c4 < c1 ? 512 : c2 < c1 ? 256 : 128;
    const double c8 = 72 * rounds((N + 2 * BN - 1) / (2 * BN) * gy4);
    if (c8 < std::min(c1, std::min(c2, c4))) {
        p.tile = 512;
        p.cols = 2 * BN;
    }
    return p;
}

// The summing pass of a split product, with its epilogue; E: the operand's row
// exponents.
int launch_split_sum(aih_ctx *ctx, const float *P, const GemmPlan &p, int64_t M, int64_t N, const int32_t *E, float *Y,
                     int epi, const aih_rope_qkv_args &ra)
{
    const int64_t zs = split_stride(M, N);
    if (epi == kEpiRopeQKV) {
        hipLaunchKernelGGL(split_k_rope_kernel, dim3((unsigned)((N / 4 + 255) / 256), (unsigned)M), dim3(256), 0, ctx->stream, P,
                           p.splits, N, zs, E, Y, ra);
        return aih_launch_status();
    }
    if (epi == kEpiSiluOperand) {
        const int64_t threads = aih_operand::mpad_of(M) * (N / 16);
        hipLaunchKernelGGL(split_k_silu_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, P,
                           p.splits, M, N, zs, E, reinterpret_cast<_Float16 *>(Y));
        return aih_launch_status();
    }
    const int64_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const int64_t groups = ((M * N + 3) / 4 + 255) / 256;
    const dim3 grid((unsigned)std::min<int64_t>(groups, 8 * cus));
    const int add = epi == kEpiAccumulate ? 1 : 0;
    if (N < 4)
        hipLaunchKernelGGL((split_k_sum_kernel<false, false>), grid, dim3(256), 0, ctx->stream, P, p.splits, M * N,
                           (uint32_t)M, (uint32_t)N, zs, E, Y, add);
    else if (reinterpret_cast<uintptr_t>(Y) % 16 == 0)
        hipLaunchKernelGGL((split_k_sum_kernel<true, true>), grid, dim3(256), 0, ctx->stream, P, p.splits, M * N, (uint32_t)M,
                           (uint32_t)N, zs, E, Y, add);
    else
        hipLaunchKernelGGL((split_k_sum_kernel<false, true>), grid, dim3(256), 0, ctx->stream, P, p.splits, M * N, (uint32_t)M,
                           (uint32_t)N, zs, E, Y, add);
    return aih_launch_status();
}

// room: staging memory for partial sums that the caller supplies (the
// allocation-free entry point), else the second workspace.
template <class T>
int launch(aih_ctx *ctx, const uint8_t *W, int64_t N, int64_t K, int64_t row_bytes, const _Float16 *Xh, int64_t M,
           float *Y, int epi, bool may_split, const aih_rope_qkv_args &ra, const aih_scratch *room)
{
    const int64_t gx = (N + BN - 1) / BN, gy = (M + BM - 1) / BM, gy2 = (M + BM2 - 1) / BM2;
    const int64_t gy4 = (M + 2 * BM2 - 1) / (2 * BM2);
    if (gy > 65535 || gx > 0x7FFFFFFF) return AIH_E_LIMIT;
    const GemmPlan p = plan_gemm(ctx->cu_count, N, K, M, epi, may_split);
    const int64_t zs = split_stride(M, N);
    void *ws = nullptr;
    if (p.splits > 1) {
        // a shape that splits always splits: a workspace that cannot grow here
        // (512-row tiles during a graph capture; 128-row tiles fit the one that
        // aih_init sets aside) is an error, not a change of the order of the sum
        const size_t bytes = (size_t)p.splits * (size_t)zs * sizeof(float);
        if (room) {
            if (bytes > room->bytes) return AIH_E_SCRATCH;
            ws = room->ptr;
        } else if (const int rc = aih_workspace2(ctx, bytes, &ws)) {
            return rc;
        }
    }
    float *const P = static_cast<float *>(ws);
    const unsigned gz = (unsigned)p.splits;
    if (p.tile == 512 && p.cols == 2 * BN)
        hipLaunchKernelGGL((qgemm256_kernel<T, 2, 2, 1>), dim3((unsigned)((N + 2 * BN - 1) / (2 * BN)), (unsigned)gy4),
                           dim3(512), 0, ctx->stream, W, N, K, row_bytes, Xh, M, Y, epi, P, zs, p.ssper, ra);
    else if (p.tile == 512)
        hipLaunchKernelGGL((qgemm256_kernel<T, 2, 1, 2>), dim3((unsigned)gx, (unsigned)gy4, gz), dim3(512), 0, ctx->stream,
                           W, N, K, row_bytes, Xh, M, Y, epi, P, zs, p.ssper, ra);
    else if (p.tile == 256)
        hipLaunchKernelGGL((qgemm256_kernel<T, 1, 1, SC>), dim3((unsigned)gx, (unsigned)gy2), dim3(512), 0, ctx->stream,
                           W, N, K, row_bytes, Xh, M, Y, epi, P, zs, p.ssper, ra);
    else
        hipLaunchKernelGGL((qgemm_kernel<T>), dim3((unsigned)gx, (unsigned)gy, gz), dim3(64 * (4 + GRing<T>::NP)), 0, ctx->stream,
                           W, N, K, row_bytes, Xh, M, Y, epi, P, zs, p.ssper, ra);
    const int rc = aih_launch_status();
    if (rc || p.splits == 1) return rc;
    const int32_t *const E = reinterpret_cast<const int32_t *>(
        reinterpret_cast<const char *>(Xh) + aih_operand::row_exp_offset(aih_operand::mpad_of(M), K));
    return launch_split_sum(ctx, P, p, M, N, E, Y, epi, ra);
}

}  // namespace

int aih_launch_qgemm_tiled(aih_ctx *ctx, int type, const void *W, int64_t N, int64_t K, const void *Xtv,
                           int64_t M, float *Y, int epi, bool may_split, const aih_rope_qkv_args *rope,
                           const aih_scratch *room)
{
    const aih_rope_qkv_args ra = rope ? *rope : aih_rope_qkv_args{};
    if (K % BK != 0) return AIH_E_LIMIT;
    const int64_t rb = aih_row_bytes(type, K);
    const uint8_t *w = static_cast<const uint8_t *>(W);
    const _Float16 *Xt = static_cast<const _Float16 *>(Xtv);
    switch (type) {
    case AIH_TYPE_Q4_K: return launch<G4K>(ctx, w, N, K, rb, Xt, M, Y, epi, may_split, ra, room);
    case AIH_TYPE_Q6_K: return launch<G6K>(ctx, w, N, K, rb, Xt, M, Y, epi, may_split, ra, room);
    case AIH_TYPE_Q8_0: return launch<G80>(ctx, w, N, K, rb, Xt, M, Y, epi, may_split, ra, room);
    case AIH_TYPE_Q4_0: return launch<G40>(ctx, w, N, K, rb, Xt, M, Y, epi, may_split, ra, room);
    default: return AIH_E_UNSUPPORTED;
    }
}

int aih_launch_x_tile(aih_ctx *ctx, const float *X, int64_t M, int64_t K, void *Xt)
{
    return aih_launch_x_tile_pre(ctx, AIH_PRE_NONE, X, nullptr, 0.f, M, K, Xt);
}

int aih_launch_operand_fixup(aih_ctx *ctx, void *Xt, int64_t M, int64_t K)
{
    const int64_t mpad = aih_operand::mpad_of(M);
    hipLaunchKernelGGL(operand_fixup_kernel, dim3((unsigned)((mpad + 3) / 4)), dim3(256), 0, ctx->stream,
                       static_cast<_Float16 *>(Xt), mpad, K);
    return aih_launch_status();
}

int aih_launch_qgemm(aih_ctx *ctx, int type, const void *W, int64_t N, int64_t K,
                     const float *X, int64_t M, float *Y, const aih_scratch *ext, bool may_split)
{
    // K advances in 64-element steps.
    if (K % BK != 0) return AIH_E_LIMIT;
    if ((reinterpret_cast<uintptr_t>(X) & 15) != 0) return AIH_E_INVALID;
    void *work = nullptr;
    int rc = aih_stage(ctx, ext, (size_t)aih_operand::image_bytes(aih_operand::mpad_of(M), K, false), &work);
    if (rc) return rc;
    rc = aih_launch_x_tile(ctx, X, M, K, work);
    if (rc) return rc;
    aih_scratch room = {};
    if (ext) {
        const size_t image = (size_t)aih_operand::image_bytes(aih_operand::mpad_of(M), K, false);   // a multiple of 128
        room = {static_cast<char *>(work) + image, ext->bytes - image};
    }
    return aih_launch_qgemm_tiled(ctx, type, W, N, K, work, M, Y, 0, may_split && ext == nullptr, nullptr,
                                  ext ? &room : nullptr);
}

extern "C" int aih_qgemm_plan(aih_ctx *ctx, int64_t N, int64_t K, int64_t M, int may_split, int32_t *tile_rows,
                              int32_t *splits)
{
    if (!ctx || !tile_rows || !splits || N <= 0 || M <= 0 || K <= 0 || K % BK) return AIH_E_INVALID;
    const GemmPlan p = plan_gemm(ctx->cu_count, N, K, M, kEpiStore, may_split != 0);
    *tile_rows = p.tile;
    *splits = p.splits;
    return AIH_OK;
}

extern "C" int aih_qgemm_tile_columns(aih_ctx *ctx, int64_t N, int64_t K, int64_t M, int may_split)
{
    if (!ctx || N <= 0 || M <= 0 || K <= 0 || K % BK) return AIH_E_INVALID;
    return plan_gemm(ctx->cu_count, N, K, M, kEpiStore, may_split != 0).cols;
}
