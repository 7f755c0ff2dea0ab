/*
 * g4s_lmhead.hip -- the Q4_0 LM head feeding the sampler, bit-exact with
 * CpuMatVecQ4 (src/Gemma4.Tensors.pas:546-598).
 *
 * Every logit is the reference's left-to-right sum over the row's blocks,
 * each term `LSum := LSum + (Single(q) * LScale) * x` in block order, low
 * nibble (x[2j]) before high nibble (x[2j+1]) of byte j (:581-593).  The
 * product q*s is exact in binary32 (a 4-bit integer times the 11-bit fp16
 * scale) and q*s*x has at most 39 significant bits, so under the reference's
 * Extended intermediates the step rounds the exact S + q*s*x to 64 bits and
 * then to binary32.  One binary32 fma(q*s, x, S) rounds it once, and the
 * two agree unless the 64-bit rounding lands on a binary32 midpoint: that
 * needs the exact sum to span more than 64 bits while sitting within 2^-64
 * of a midpoint, which happens only for 0 < |S| <= 2^-64 |q*s*x| with q*s*x
 * itself a binary32 midpoint -- never for this workload (|S| is then at
 * least 2^-60 unless it is 0).  So the kernel is one fma per term, in the
 * reference's order.
 *
 * Layout: one weight row per thread (the TQ4Block row, 18 bytes per 32
 * weights, read in place), batch tiles of 32 hidden vectors whose values are
 * staged in LDS two blocks at a time (double-buffered, the next group's
 * loads in flight during the current one) and read as broadcasts; 32
 * independent running sums per thread.
 * Compute-bound at B=32: 2*B*rows*cols flops against 377 MB of weights.
 */
#include "g4s_lmhead.h"

namespace g4s {

namespace {

constexpr int kLmBlock = 256;
constexpr int kLmTile = 32; /* hidden vectors per pass over the weights */
constexpr int kLmKb = 2;    /* weight blocks (of 32 terms) per staged group of hidden values */

/* TFloat16.ToSingle (src/Gemma4.Types.pas:438-481) as written, including its
 * handling of subnormal halves (the exponent is raised while normalising). */
__device__ __forceinline__ float f16_to_f32_ref(uint32_t v)
{
    const uint32_t sign = (v >> 15) & 1u;
    uint32_t expo = (v >> 10) & 0x1Fu;
    uint32_t mant = v & 0x3FFu;
    uint32_t bits;
    if (expo == 0u) {
        if (mant == 0u) {
            bits = sign << 31;
        } else {
            const uint32_t shift = (uint32_t)__builtin_clz(mant) - 21u; /* until bit 10 is set */
            mant = (mant << shift) & 0x3FFu;
            expo = shift + 1u;
            bits = (sign << 31) | ((expo + (127u - 15u)) << 23) | (mant << 13);
        }
    } else if (expo == 0x1Fu) {
        bits = (sign << 31) | (0xFFu << 23) | (mant << 13);
    } else {
        bits = (sign << 31) | ((expo + (127u - 15u)) << 23) | (mant << 13);
    }
    return __uint_as_float(bits);
}

__global__ __launch_bounds__(kLmBlock) void lmhead_q4_kernel(const uint8_t* __restrict__ w,
                                                             int32_t rows, int32_t nblk,
                                                             const float* __restrict__ h,
                                                             int32_t cols, int32_t batch,
                                                             float* __restrict__ out,
                                                             int64_t stride, int32_t h_vec4)
{
    /* the hidden values of kLmKb weight blocks for the tile's kLmTile
     * vectors, double-buffered: every lane reads the same entry (an LDS
     * broadcast), so the fma operands come from VGPRs */
    __shared__ __align__(16) float xs[2][kLmTile][kLmKb * 32];
    constexpr int kStage = kLmTile * kLmKb * 8 / kLmBlock; /* float4 per thread per stage */
    static_assert(kLmTile * kLmKb * 8 % kLmBlock == 0, "whole float4 stages");
    const int32_t r = blockIdx.x * kLmBlock + threadIdx.x;
    const bool active = r < rows;
    const int32_t rr = active ? r : rows - 1;
    const uint8_t* wrow = w + (int64_t)rr * nblk * 18;
    const int32_t ngroup = (nblk + kLmKb - 1) / kLmKb;
    for (int32_t b0 = 0; b0 < batch; b0 += kLmTile) {
        const int32_t nb = batch - b0 < kLmTile ? batch - b0 : kLmTile;
        /* hidden values of block group g (zeros past the batch or the row) */
        const auto fetch = [&](int32_t g, float4 (&v)[kStage]) {
#pragma unroll
            for (int q = 0; q < kStage; ++q) {
                const int i = threadIdx.x + q * kLmBlock;
                const int b = i / (kLmKb * 8), c4 = i % (kLmKb * 8);
                const int32_t col = g * kLmKb * 32 + c4 * 4;
                float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (b < nb && col < cols) {
                    const float* src = h + (int64_t)(b0 + b) * cols + col;
                    if (h_vec4)
                        x = *reinterpret_cast<const float4*>(src);
                    else
                        x = make_float4(src[0], src[1], src[2], src[3]);
                }
                v[q] = x;
            }
        };
        const auto stash = [&](int buf, const float4 (&v)[kStage]) {
#pragma unroll
            for (int q = 0; q < kStage; ++q) {
                const int i = threadIdx.x + q * kLmBlock;
                reinterpret_cast<float4*>(&xs[buf][i / (kLmKb * 8)][0])[i % (kLmKb * 8)] = v[q];
            }
        };
        float S[kLmTile];
#pragma unroll
        for (int b = 0; b < kLmTile; ++b) S[b] = 0.0f;
        float4 nx[kStage];
        fetch(0, nx);
        stash(0, nx);
        __syncthreads();
        for (int32_t g = 0; g < ngroup; ++g) {
            const int buf = g & 1;
            if (g + 1 < ngroup) fetch(g + 1, nx); /* in flight during this group */
            for (int kk = 0; kk < kLmKb; ++kk) {
                const int32_t k = g * kLmKb + kk;
                if (k >= nblk) break;
                const uint16_t* blk = reinterpret_cast<const uint16_t*>(wrow + (int64_t)k * 18);
                uint32_t half[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) half[i] = blk[i];
                const float sc = f16_to_f32_ref(half[0]);
                float qs[32];
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const uint32_t byte = (half[1 + (j >> 1)] >> ((j & 1) * 8)) & 0xFFu;
                    qs[2 * j] = (float)((int)(byte & 0x0Fu) - 8) * sc;     /* Tensors.pas:586 */
                    qs[2 * j + 1] = (float)((int)(byte >> 4) - 8) * sc;    /* Tensors.pas:590 */
                }
                /* term j of every vector before term j+4: the 32 running sums
                 * are independent chains, each still in the reference's order */
#pragma unroll
                for (int j4 = 0; j4 < 8; ++j4) {
#pragma unroll
                    for (int b = 0; b < kLmTile; ++b) {
                        const float4 x = reinterpret_cast<const float4*>(&xs[buf][b][kk * 32])[j4];
                        S[b] = __builtin_fmaf(qs[4 * j4], x.x, S[b]);
                        S[b] = __builtin_fmaf(qs[4 * j4 + 1], x.y, S[b]);
                        S[b] = __builtin_fmaf(qs[4 * j4 + 2], x.z, S[b]);
                        S[b] = __builtin_fmaf(qs[4 * j4 + 3], x.w, S[b]);
                    }
                }
            }
            if (g + 1 < ngroup) stash(buf ^ 1, nx); /* read last in group g - 1 */
            __syncthreads();
        }
        if (active) {
#pragma unroll
            for (int b = 0; b < kLmTile; ++b)
                if (b < nb) out[(int64_t)(b0 + b) * stride + r] = S[b];
        }
        __syncthreads(); /* the next tile restages both buffers */
    }
}

/* ------------------------------------------------------------------
 * The matrix-core sum of 64 weight rows (lane = row) for 4 * NG hidden
 * vectors.
 *
 * v_mfma_f32_4x4x1_16b multiplies a 4x1 by a 1x4 in each of 16 blocks: one
 * product per output, so one instruction is one binary32 fma of every chain
 * and a sequence of them keeps the reference's order (checked bit for bit
 * against fmaf: ties, denormals, infinities and NaN included).  The weights
 * are the B operand: block b, column j is lane 4b + j, that is the lane's own
 * row.  The hidden values are the A operand with CBSZ = 4: block ABID's four
 * rows (vectors) go to all 16 blocks, so one VGPR holds four vectors' values
 * of 16 columns and nothing passes through LDS.  D: register i of a lane is
 * vector i of the lane's row.
 *
 * It runs 32 fmas per clock and SIMD (135 TFLOP/s measured, against 66 for
 * v_fmac_f32 with a DPP broadcast).  The binary32 matrix instructions share
 * the VALU's issue (a wave of each takes the sum of the two times), so the
 * dequantisation adds to them: 262,144 rows x 2,560 columns take 38 us of
 * matrix instructions per four vectors and about 60 us for the rest.
 * ------------------------------------------------------------------ */

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

/* Eight weights of a row: nibble t of `w` is weight t.  A byte 0..15 read as
 * fp8 (e4m3) is n * 2^-9 (its denormals and first binade), so one
 * v_cvt_pk_f32_fp8 gives two nibbles, and fma(n * 2^-9, 512 s, -8 s) is
 * (n - 8) s exactly (at most 15 significant bits).  s512 = 512 s, m8 = -8 s. */
__device__ __forceinline__ void dequant8(uint32_t w, float s512, float m8, float (&q)[8])
{
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    const auto l0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false);
    const auto l1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
    const auto h0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false);
    const auto h1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
    q[0] = __builtin_fmaf(l0[0], s512, m8);
    q[1] = __builtin_fmaf(h0[0], s512, m8);
    q[2] = __builtin_fmaf(l0[1], s512, m8);
    q[3] = __builtin_fmaf(h0[1], s512, m8);
    q[4] = __builtin_fmaf(l1[0], s512, m8);
    q[5] = __builtin_fmaf(h1[0], s512, m8);
    q[6] = __builtin_fmaf(l1[1], s512, m8);
    q[7] = __builtin_fmaf(h1[1], s512, m8);
}

/* Terms 8W .. 8W+7 of a block.  x[g]: lane l holds columns 2 (l / 4) and
 * 2 (l / 4) + 1 of vector 4g + l % 4. */
template <int W, int NG>
__device__ __forceinline__ void mac8(f32x4 (&S)[NG], const float (&q)[8], const float2 (&x)[NG])
{
#define G4S_MAC(T, C, AB)                                                                       \
    _Pragma("unroll") for (int g = 0; g < NG; ++g)                                              \
        S[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[g].C, q[T], S[g], 4, AB, 0);
    G4S_MAC(0, x, 4 * W)
    G4S_MAC(1, y, 4 * W)
    G4S_MAC(2, x, 4 * W + 1)
    G4S_MAC(3, y, 4 * W + 1)
    G4S_MAC(4, x, 4 * W + 2)
    G4S_MAC(5, y, 4 * W + 2)
    G4S_MAC(6, x, 4 * W + 3)
    G4S_MAC(7, y, 4 * W + 3)
#undef G4S_MAC
}

/* The 32 terms of one block. */
template <int NG>
__device__ __forceinline__ void mac32(f32x4 (&S)[NG], const uint4 w, float sc, const float2 (&x)[NG])
{
    const float s512 = 512.0f * sc, m8 = -8.0f * sc;
    float q[8];
    dequant8(w.x, s512, m8, q);
    mac8<0, NG>(S, q, x);
    dequant8(w.y, s512, m8, q);
    mac8<1, NG>(S, q, x);
    dequant8(w.z, s512, m8, q);
    mac8<2, NG>(S, q, x);
    dequant8(w.w, s512, m8, q);
    mac8<3, NG>(S, q, x);
}

/* ------------------------------------------------------------------
 * TILED64 layout and the LM head over it.
 *
 * One wave per 64 weight rows and 4 * NG hidden vectors, waves independent
 * (no LDS, no barrier).  Per 32-column block a lane loads its row's binary32
 * scale and 16 nibble bytes from the tile (256 + 1024 contiguous bytes per
 * wave) and two columns of its vectors (L1/L2 hits), kept DEPTH blocks ahead
 * in registers.  262,144 x 2,560 (a plain read of the 419 MB of tiles takes
 * 69-73 us): B = 1 645 -> 75 us, B = 8 152 us, B = 32 649 -> 361 us.
 * ------------------------------------------------------------------ */

constexpr int kTileWaves = 4; /* waves (64-row groups) per workgroup */

__global__ __launch_bounds__(256) void q4_tile_kernel(const uint8_t* __restrict__ src, int32_t rows,
                                                      int32_t nblk, uint8_t* __restrict__ dst)
{
    const int32_t groups = (rows + kQ4TileRows - 1) / kQ4TileRows;
    const int64_t total = (int64_t)groups * kQ4TileRows * nblk;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        /* t = (g * nblk + k) * 64 + lane: the destination is written in order */
        const int32_t lane = (int32_t)(t % kQ4TileRows);
        const int64_t tile = t / kQ4TileRows;
        const int32_t k = (int32_t)(tile % nblk);
        const int32_t g = (int32_t)(tile / nblk);
        const int32_t r = g * kQ4TileRows + lane;
        uint8_t* tp = dst + tile * kQ4TileBytes;
        float sc = 0.0f;
        uint32_t q[4] = {0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u};
        if (r < rows) {
            const uint16_t* b = reinterpret_cast<const uint16_t*>(src + ((int64_t)r * nblk + k) * 18);
            sc = f16_to_f32_ref(b[0]);
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] = (uint32_t)b[1 + 2 * i] | ((uint32_t)b[2 + 2 * i] << 16);
        }
        reinterpret_cast<float*>(tp)[lane] = sc;
        reinterpret_cast<uint4*>(tp + kQ4TileRows * 4)[lane] = make_uint4(q[0], q[1], q[2], q[3]);
    }
}

/* The logit of row r = 64 g + lane for vector b: written where wanted, and
 * the group's summary (its largest key, the lowest row holding it, and the
 * largest key of the other rows). */
__device__ __forceinline__ void put_logit(float v, int32_t b, int32_t r, int32_t rows, int lane,
                                          int32_t g, int32_t ngroups, float* __restrict__ out,
                                          int64_t stride, uint64_t* __restrict__ gsum)
{
    const bool live = r < rows;
    if (out && live) out[(int64_t)b * stride + r] = v;
    if (gsum) {
        const uint32_t key = live ? cand_key(v) : 0u;
        const uint32_t kmax = wave_max_u32(key);
        const uint32_t r6 = (uint32_t)__builtin_ctzll(__ballot(key == kmax));
        const uint32_t k2 = wave_max_u32((uint32_t)lane == r6 ? 0u : key);
        if (lane == 0) gsum[(int64_t)b * ngroups + g] = gsum_pack(kmax, r6, k2);
    }
}

template <int NG, int DEPTH>
__global__ __launch_bounds__(64 * kTileWaves, 4) void lmhead_tiled_kernel(
    const uint8_t* __restrict__ tiles, int32_t rows, int32_t nblk, const float* __restrict__ h,
    int32_t cols, int32_t batch, float* __restrict__ out, int64_t stride, uint64_t* __restrict__ gsum,
    int32_t ngroups)
{
    const int lane = threadIdx.x & 63;
    const int32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x * kTileWaves + (threadIdx.x >> 6));
    if (g >= ngroups) return; /* whole waves: no barrier below */
    const int32_t b0 = blockIdx.y * (4 * NG);
    const int32_t r = g * kQ4TileRows + lane;
    const uint8_t* tp = tiles + (int64_t)g * nblk * kQ4TileBytes;
    /* byte offsets of the lane's vectors (the hidden matrix is below 2 GiB:
     * checked by the caller); vectors past the batch read vector batch - 1
     * (any valid row; their sums are discarded) */
    uint32_t xo[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int32_t v = b0 + 4 * i + (lane & 3);
        xo[i] = (uint32_t)((v < batch ? v : batch - 1) * cols + 2 * (lane >> 2)) * 4u;
    }
    float sc[DEPTH];
    uint4 w[DEPTH];
    float2 x[DEPTH][NG];
    const auto fetch = [&](int d, int32_t k) {
        const uint8_t* t = tp + (uint32_t)k * (uint32_t)kQ4TileBytes;
        sc[d] = reinterpret_cast<const float*>(t)[lane];
        w[d] = reinterpret_cast<const uint4*>(t + kQ4TileRows * 4)[lane];
        const char* hk = reinterpret_cast<const char*>(h) + (uint32_t)k * 128u;
#pragma unroll
        for (int i = 0; i < NG; ++i) x[d][i] = *reinterpret_cast<const float2*>(hk + xo[i]);
    };
    f32x4 S[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) S[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        fetch(d, d < nblk ? d : nblk - 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    int32_t k = 0;
    for (; k + DEPTH <= nblk; k += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            mac32<NG>(S, w[d], sc[d], x[d]);
            const int32_t kn = k + d + DEPTH;
            fetch(d, kn < nblk ? kn : nblk - 1);
            /* keeps each load where it is issued, DEPTH blocks before its use */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
        if (k + d < nblk) mac32<NG>(S, w[d], sc[d], x[d]);
#pragma unroll
    for (int i = 0; i < 4 * NG; ++i)
        if (b0 + i < batch)
            put_logit(S[i / 4][i % 4], b0 + i, r, rows, lane, g, ngroups, out, stride, gsum);
}

/* Terms 8W .. 8W+7 of a block for 32 vectors.  x: lane l holds columns
 * 8W + 4 (l / 32) .. + 3 of vector l % 32. */
__device__ __forceinline__ void mac8x32(f32x32& S, const float (&q)[8], const float4 x)
{
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.x, q[0], S, 1, 0, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.y, q[1], S, 1, 0, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.z, q[2], S, 1, 0, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.w, q[3], S, 1, 0, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.x, q[4], S, 1, 1, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.y, q[5], S, 1, 1, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.z, q[6], S, 1, 1, 0);
    S = __builtin_amdgcn_mfma_f32_32x32x1f32(x.w, q[7], S, 1, 1, 0);
}

/* 32 vectors per wave on v_mfma_f32_32x32x1_2b: also one product per output,
 * the weights' two blocks being rows 0-31 and 32-63 and CBSZ = 1 handing
 * either half of the A register to both.  It reads eight times fewer operands
 * per fma than the 4x4 form (262,144 x 2,560 x 32: 361 against 391 us). */
template <int DEPTH>
__global__ __launch_bounds__(64 * kTileWaves, 4) void lmhead_tiled32_kernel(
    const uint8_t* __restrict__ tiles, int32_t rows, int32_t nblk, const float* __restrict__ h,
    int32_t cols, int32_t batch, float* __restrict__ out, int64_t stride, uint64_t* __restrict__ gsum,
    int32_t ngroups)
{
    const int lane = threadIdx.x & 63;
    const int32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x * kTileWaves + (threadIdx.x >> 6));
    if (g >= ngroups) return; /* whole waves: no barrier below */
    const int32_t b0 = blockIdx.y * 32;
    const uint8_t* tp = tiles + (int64_t)g * nblk * kQ4TileBytes;
    /* vectors past the batch read vector batch - 1 (their sums are discarded) */
    const int32_t v = b0 + (lane & 31);
    const uint32_t xo = (uint32_t)((v < batch ? v : batch - 1) * cols + 4 * (lane >> 5)) * 4u;
    float sc[DEPTH];
    uint4 w[DEPTH];
    float4 x[DEPTH][4];
    const auto fetch = [&](int d, int32_t k) {
        const uint8_t* t = tp + (uint32_t)k * (uint32_t)kQ4TileBytes;
        sc[d] = reinterpret_cast<const float*>(t)[lane];
        w[d] = reinterpret_cast<const uint4*>(t + kQ4TileRows * 4)[lane];
        const char* hk = reinterpret_cast<const char*>(h) + (uint32_t)k * 128u;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[d][i] = *reinterpret_cast<const float4*>(hk + xo + 32 * i);
    };
    f32x32 S;
#pragma unroll
    for (int i = 0; i < 32; ++i) S[i] = 0.0f;
    const auto term32 = [&](int d) {
        const float s512 = 512.0f * sc[d], m8 = -8.0f * sc[d];
        float q[8];
        dequant8(w[d].x, s512, m8, q);
        mac8x32(S, q, x[d][0]);
        dequant8(w[d].y, s512, m8, q);
        mac8x32(S, q, x[d][1]);
        dequant8(w[d].z, s512, m8, q);
        mac8x32(S, q, x[d][2]);
        dequant8(w[d].w, s512, m8, q);
        mac8x32(S, q, x[d][3]);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        fetch(d, d < nblk ? d : nblk - 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    int32_t k = 0;
    for (; k + DEPTH <= nblk; k += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            term32(d);
            const int32_t kn = k + d + DEPTH;
            fetch(d, kn < nblk ? kn : nblk - 1);
            /* keeps each load where it is issued, DEPTH blocks before its use */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
        if (k + d < nblk) term32(d);
    const int32_t r = g * kQ4TileRows + lane;
    /* register i: row lane % 32 (i < 16) or 32 + lane % 32 of vector
     * 8 (i % 16 / 4) + 4 (lane / 32) + i % 4; swapping halves between i and
     * i + 16 leaves lane = row, vectors c and c + 4 */
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(S[i]),
                                                        __float_as_uint(S[i + 16]), false, false);
        const int32_t c = b0 + 8 * (i / 4) + i % 4;
        if (c < batch)
            put_logit(__uint_as_float(y[0]), c, r, rows, lane, g, ngroups, out, stride, gsum);
        if (c + 4 < batch)
            put_logit(__uint_as_float(y[1]), c + 4, r, rows, lane, g, ngroups, out, stride, gsum);
    }
}

/* Terms 8W .. 8W+7 of a block for one vector.  x: lane l holds columns
 * 2 (l % 16) and 2 (l % 16) + 1; row_newbcast hands lane n's value to its
 * 16-lane row, the same value in all four rows.  The s_nop covers the two
 * wait states between a VALU write of x (a copy by the compiler) and its DPP
 * read. */
#define G4S_FMAC8(N0, N1, N2, N3)                                                               \
    asm("s_nop 1\n\t"                                                                           \
        "v_fmac_f32_dpp %0, %1, %3 row_newbcast:" N0 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %2, %4 row_newbcast:" N0 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %1, %5 row_newbcast:" N1 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %2, %6 row_newbcast:" N1 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %1, %7 row_newbcast:" N2 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %2, %8 row_newbcast:" N2 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %1, %9 row_newbcast:" N3 " row_mask:0xf bank_mask:0xf\n\t"          \
        "v_fmac_f32_dpp %0, %2, %10 row_newbcast:" N3 " row_mask:0xf bank_mask:0xf"             \
        : "+v"(S)                                                                               \
        : "v"(x.x), "v"(x.y), "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]), "v"(q[4]), "v"(q[5]), \
          "v"(q[6]), "v"(q[7]))
template <int W>
__device__ __forceinline__ void fmac8(float& S, const float (&q)[8], const float2 x)
{
    if constexpr (W == 0) G4S_FMAC8("0", "1", "2", "3");
    if constexpr (W == 1) G4S_FMAC8("4", "5", "6", "7");
    if constexpr (W == 2) G4S_FMAC8("8", "9", "10", "11");
    if constexpr (W == 3) G4S_FMAC8("12", "13", "14", "15");
}
#undef G4S_FMAC8

/* One or two hidden vectors per wave: one v_fmac_f32 with a DPP broadcast a
 * term.  A matrix instruction would spend its four vectors' time on one. */
template <int NV, int DEPTH>
__global__ __launch_bounds__(64 * kTileWaves, 4) void lmhead_tiled_few_kernel(
    const uint8_t* __restrict__ tiles, int32_t rows, int32_t nblk, const float* __restrict__ h,
    int32_t cols, float* __restrict__ out, int64_t stride, uint64_t* __restrict__ gsum,
    int32_t ngroups)
{
    const int lane = threadIdx.x & 63;
    const int32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x * kTileWaves + (threadIdx.x >> 6));
    if (g >= ngroups) return; /* whole waves: no barrier below */
    const int32_t b0 = blockIdx.y * NV;
    const uint8_t* tp = tiles + (int64_t)g * nblk * kQ4TileBytes;
    h += (int64_t)b0 * cols;
    float sc[DEPTH];
    uint4 w[DEPTH];
    float2 x[DEPTH][NV];
    const auto fetch = [&](int d, int32_t k) {
        const uint8_t* t = tp + (uint32_t)k * (uint32_t)kQ4TileBytes;
        sc[d] = reinterpret_cast<const float*>(t)[lane];
        w[d] = reinterpret_cast<const uint4*>(t + kQ4TileRows * 4)[lane];
#pragma unroll
        for (int b = 0; b < NV; ++b)
            x[d][b] = reinterpret_cast<const float2*>(h + (int64_t)b * cols + k * 32)[lane & 15];
    };
    float S[NV];
#pragma unroll
    for (int b = 0; b < NV; ++b) S[b] = 0.0f;
    const auto term32 = [&](int d) {
        const float s512 = 512.0f * sc[d], m8 = -8.0f * sc[d];
        float q[8];
        dequant8(w[d].x, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<0>(S[b], q, x[d][b]);
        dequant8(w[d].y, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<1>(S[b], q, x[d][b]);
        dequant8(w[d].z, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<2>(S[b], q, x[d][b]);
        dequant8(w[d].w, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<3>(S[b], q, x[d][b]);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        fetch(d, d < nblk ? d : nblk - 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    int32_t k = 0;
    for (; k + DEPTH <= nblk; k += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            term32(d);
            const int32_t kn = k + d + DEPTH;
            fetch(d, kn < nblk ? kn : nblk - 1);
            /* keeps each load where it is issued, DEPTH blocks before its use */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
        if (k + d < nblk) term32(d);
    const int32_t r = g * kQ4TileRows + lane;
#pragma unroll
    for (int b = 0; b < NV; ++b)
        put_logit(S[b], b0 + b, r, rows, lane, g, ngroups, out, stride, gsum);
}

/* DoEmbeddingLookup for a Q4_0 table (src/Gemma4.Model.pas:2047-2080):
 * row `token` dequantised as DequantQ4Block does (Single(q) * LScale,
 * src/Gemma4.Quant.pas:209-239; exact) and multiplied by `scale`
 * (CpuScaleF32, src/Gemma4.Tensors.pas:626-636; one rounding).  One thread
 * per weight; tokens outside [0, rows) give a zero vector. */
__global__ __launch_bounds__(256) void embed_q4_kernel(const uint8_t* __restrict__ w, int32_t rows,
                                                       int32_t nblk, const int32_t* __restrict__ tokens,
                                                       int32_t batch, float scale,
                                                       float* __restrict__ out)
{
    const int32_t cols = nblk * 32;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)batch * cols) return;
    const int32_t b = (int32_t)(i / cols), c = (int32_t)(i % cols);
    const int32_t t = tokens[b];
    float v = 0.0f;
    if (t >= 0 && t < rows) {
        const uint8_t* blk = w + ((int64_t)t * nblk + c / 32) * 18;
        const float sc = f16_to_f32_ref((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
        const uint32_t byte = blk[2 + (c % 32) / 2];
        const int q = (int)((c & 1) ? (byte >> 4) : (byte & 0x0Fu)) - 8;
        v = ((float)q * sc) * scale;
    }
    out[i] = v;
}

}  // namespace

hipError_t embed_q4_0_launch(const uint8_t* w, int32_t rows, int32_t cols, const int32_t* tokens,
                             int32_t batch, float scale, float* hidden, hipStream_t s)
{
    const int64_t n = (int64_t)batch * cols;
    hipLaunchKernelGGL(embed_q4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w, rows,
                       cols / 32, tokens, batch, scale, hidden);
    return hipGetLastError();
}

hipError_t q4_tile_launch(const uint8_t* src, int32_t rows, int32_t nblk, uint8_t* dst, hipStream_t s)
{
    const int64_t total = (int64_t)((rows + kQ4TileRows - 1) / kQ4TileRows) * kQ4TileRows * nblk;
    const int64_t want = (total + 255) / 256;
    const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
    hipLaunchKernelGGL(q4_tile_kernel, dim3(grid), dim3(256), 0, s, src, rows, nblk, dst);
    return hipGetLastError();
}

/* The split of a tiled launch into waves of 64 rows and some vectors:
 *  - every (row group, vector) pair its own wave while that leaves at most
 *    one wave per SIMD, and up to two vectors otherwise: the plain fma kernel
 *    (2,560 columns: 20 us for 8,000 rows x 8 against 31 us with four vectors
 *    a wave; 262,144 rows: 74 us for one vector against 105, 81 for two);
 *  - else 4 * NG vectors a wave on the matrix cores, NG as large as needed
 *    (up to 8) to leave at most one wave per SIMD (32,768 rows x 32: NG = 4
 *    64 us, NG = 2 75, NG = 8 102; 262,144 rows x 32: NG = 8 391 us, NG = 4
 *    416), and the 32-vector form where a wave takes 29 to 32. */
constexpr int32_t kLmSimds = 1024;

hipError_t lmhead_tiled_launch(const uint8_t* tiles, int32_t rows, int32_t cols, const float* h,
                               int32_t batch, float* logits, int64_t stride, uint64_t* gsum,
                               hipStream_t s)
{
    const int32_t ngroups = (rows + kQ4TileRows - 1) / kQ4TileRows;
    const int32_t nblk = cols / 32;
    const unsigned gx = (unsigned)((ngroups + kTileWaves - 1) / kTileWaves);
    const dim3 block(64 * kTileWaves);
    if (batch <= 2 || (int64_t)batch * ngroups <= kLmSimds) {
        if ((int64_t)batch * ngroups <= kLmSimds || batch == 1)
            hipLaunchKernelGGL((lmhead_tiled_few_kernel<1, 4>), dim3(gx, (unsigned)batch), block, 0,
                               s, tiles, rows, nblk, h, cols, logits, stride, gsum, ngroups);
        else
            hipLaunchKernelGGL((lmhead_tiled_few_kernel<2, 4>), dim3(gx), block, 0, s, tiles, rows,
                               nblk, h, cols, logits, stride, gsum, ngroups);
        return hipGetLastError();
    }
    const int32_t quads = (batch + 3) / 4;
    const int32_t fill = kLmSimds / ngroups;
    int32_t passes = (quads + 7) / 8;
    if (passes < fill) passes = fill < quads ? fill : quads;
    const int32_t ng = (quads + passes - 1) / passes;
    passes = (quads + ng - 1) / ng;
    const dim3 grid(gx, (unsigned)passes);
#define G4S_LM(NG, DEPTH)                                                                        \
    hipLaunchKernelGGL((lmhead_tiled_kernel<NG, DEPTH>), grid, block, 0, s, tiles, rows, nblk, h,\
                       cols, batch, logits, stride, gsum, ngroups)
    switch (ng) {
        case 1: G4S_LM(1, 4); break;
        case 2: G4S_LM(2, 4); break;
        case 3: G4S_LM(3, 3); break;
        case 4: G4S_LM(4, 2); break;
        case 5: G4S_LM(5, 2); break;
        case 6: G4S_LM(6, 2); break;
        case 7: G4S_LM(7, 2); break;
        default:
            hipLaunchKernelGGL(lmhead_tiled32_kernel<2>, grid, block, 0, s, tiles, rows, nblk, h,
                               cols, batch, logits, stride, gsum, ngroups);
            break;
    }
#undef G4S_LM
    return hipGetLastError();
}

hipError_t lmhead_q4_0_launch(const uint8_t* w, int32_t rows, int32_t cols, const float* h,
                              int32_t batch, float* logits, int64_t stride, hipStream_t s)
{
    const int32_t nblk = cols / 32;
    const int32_t h_vec4 = (reinterpret_cast<uintptr_t>(h) & 15u) == 0 ? 1 : 0;
    hipLaunchKernelGGL(lmhead_q4_kernel, dim3((unsigned)((rows + kLmBlock - 1) / kLmBlock)),
                       dim3(kLmBlock), 0, s, w, rows, nblk, h, cols, batch, logits, stride, h_vec4);
    return hipGetLastError();
}

}  // namespace g4s
