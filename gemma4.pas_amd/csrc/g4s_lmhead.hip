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
 * reference's order.  A weight of zero counts as +0 where the reference may
 * have -0: that shows only in a running sum of -0, as the sign of a zero logit,
 * and such a sum takes a product that underflows to zero (a scale is 0 or at
 * least 2^-14, so a hidden value below 2^-135).
 *
 * Every wave owns 64 weight rows (lane = row) and some hidden vectors: one
 * accumulator form per number of vectors, over either layout of the weights.
 */
#include "g4s_lmhead.h"

namespace g4s {

namespace {

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

/* The same value by the hardware's conversion: the two differ for subnormal
 * halves only, whose exponent field the reference takes as 113 + shift where
 * the value's is 113 - shift. */
__device__ __forceinline__ float f16_to_f32_fast(uint32_t v)
{
    const _Float16 hv = __builtin_bit_cast(_Float16, (uint16_t)v);
    float t = (float)hv;
    const bool sub = __builtin_amdgcn_classh(hv, 0x90);
    if (__ballot(sub)) {
        const uint32_t u = __float_as_uint(t), e = (u >> 23) & 0xFFu;
        if (sub) t = __uint_as_float(u + ((226u - 2u * e) << 23));
    }
    return t;
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
/* hidden values and row bytes may start on any element */
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(1)));

/* Eight weights of a row: nibble t of `w` is weight t.  A byte 0..15 read as
 * fp8 (e4m3) is n * 2^-9 (its denormals and first binade), so one
 * v_cvt_pk_f32_fp8 gives two nibbles, and fma(n * 2^-9, 512 s, -8 s) is
 * (n - 8) s exactly (at most 15 significant bits), a zero being +0.  An infinite
 * s gives NaN (sum_infinite).  s512 = 512 s, m8 = -8 s. */
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
__device__ __forceinline__ void mac8(f32x4 (&S)[NG], const float (&q)[8], const float2u (&x)[NG])
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
__device__ __forceinline__ void mac32(f32x4 (&S)[NG], const uint4 w, float sc, const float2u (&x)[NG])
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
 * 69-73 us): B = 1 636 -> 74 us, B = 8 639 -> 147, B = 32 642 -> 361-368.
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

/* 4 * NG hidden vectors per wave.  Vectors past the batch read vector
 * batch - 1 (any valid row; their sums are discarded).  Byte offsets stay
 * within 32 bits: a launch's hidden matrix is below 2 GiB. */
template <int NG>
struct QuadAcc {
    static constexpr int kVecs = 4 * NG;
    struct X {
        float2u v[NG];
    };
    f32x4 S[NG];
    uint32_t xo[NG];
    const char* hb;

    __device__ __forceinline__ void init(const float* h, int32_t cols, int32_t b0, int32_t batch,
                                         int lane)
    {
        hb = reinterpret_cast<const char*>(h);
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int32_t v = b0 + 4 * i + (lane & 3);
            xo[i] = (uint32_t)((v < batch ? v : batch - 1) * cols + 2 * (lane >> 2)) * 4u;
            S[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    __device__ __forceinline__ void load(X& x, int32_t k) const
    {
        const char* hk = hb + (uint32_t)k * 128u;
#pragma unroll
        for (int i = 0; i < NG; ++i) x.v[i] = *reinterpret_cast<const float2u*>(hk + xo[i]);
    }
    __device__ __forceinline__ void mac(const uint4 w, float sc, const X& x)
    {
        mac32<NG>(S, w, sc, x.v);
    }
    template <typename F>
    __device__ __forceinline__ void emit(F put) const
    {
#pragma unroll
        for (int i = 0; i < 4 * NG; ++i) put(S[i / 4][i % 4], i);
    }
};

/* Terms 8W .. 8W+7 of a block for 32 vectors.  x: lane l holds columns
 * 8W + 4 (l / 32) .. + 3 of vector l % 32. */
__device__ __forceinline__ void mac8x32(f32x32& S, const float (&q)[8], const float4u x)
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
 * per fma than the 4x4 form (262,144 x 2,560 x 32: 364 against 396 us). */
struct WideAcc {
    static constexpr int kVecs = 32;
    struct X {
        float4u v[4];
    };
    f32x32 S;
    uint32_t xo;
    const char* hb;

    __device__ __forceinline__ void init(const float* h, int32_t cols, int32_t b0, int32_t batch,
                                         int lane)
    {
        hb = reinterpret_cast<const char*>(h);
        const int32_t v = b0 + (lane & 31);
        xo = (uint32_t)((v < batch ? v : batch - 1) * cols + 4 * (lane >> 5)) * 4u;
#pragma unroll
        for (int i = 0; i < 32; ++i) S[i] = 0.0f;
    }
    __device__ __forceinline__ void load(X& x, int32_t k) const
    {
        const char* hk = hb + (uint32_t)k * 128u;
#pragma unroll
        for (int i = 0; i < 4; ++i) x.v[i] = *reinterpret_cast<const float4u*>(hk + xo + 32 * i);
    }
    __device__ __forceinline__ void mac(const uint4 w, float sc, const X& x)
    {
        const float s512 = 512.0f * sc, m8 = -8.0f * sc;
        float q[8];
        dequant8(w.x, s512, m8, q);
        mac8x32(S, q, x.v[0]);
        dequant8(w.y, s512, m8, q);
        mac8x32(S, q, x.v[1]);
        dequant8(w.z, s512, m8, q);
        mac8x32(S, q, x.v[2]);
        dequant8(w.w, s512, m8, q);
        mac8x32(S, q, x.v[3]);
    }
    /* register i: row lane % 32 (i < 16) or 32 + lane % 32 of vector
     * 8 (i % 16 / 4) + 4 (lane / 32) + i % 4; swapping halves between i and
     * i + 16 leaves lane = row, vectors c and c + 4 */
    template <typename F>
    __device__ __forceinline__ void emit(F put) const
    {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const auto y = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(S[i]), __float_as_uint(S[i + 16]), false, false);
            const int32_t c = 8 * (i / 4) + i % 4;
            put(__uint_as_float(y[0]), c);
            put(__uint_as_float(y[1]), c + 4);
        }
    }
};

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
__device__ __forceinline__ void fmac8(float& S, const float (&q)[8], const float2u x)
{
    if constexpr (W == 0) G4S_FMAC8("0", "1", "2", "3");
    if constexpr (W == 1) G4S_FMAC8("4", "5", "6", "7");
    if constexpr (W == 2) G4S_FMAC8("8", "9", "10", "11");
    if constexpr (W == 3) G4S_FMAC8("12", "13", "14", "15");
}
#undef G4S_FMAC8

/* One or two hidden vectors per wave: one v_fmac_f32 with a DPP broadcast a
 * term.  A matrix instruction would spend its four vectors' time on one. */
template <int NV>
struct FewAcc {
    static constexpr int kVecs = NV;
    struct X {
        float2u v[NV];
    };
    float S[NV];
    const float* hb;
    int32_t cols, at;

    __device__ __forceinline__ void init(const float* h, int32_t c, int32_t b0, int32_t, int lane)
    {
        hb = h + (int64_t)b0 * c;
        cols = c;
        at = lane & 15;
#pragma unroll
        for (int b = 0; b < NV; ++b) S[b] = 0.0f;
    }
    __device__ __forceinline__ void load(X& x, int32_t k) const
    {
#pragma unroll
        for (int b = 0; b < NV; ++b)
            x.v[b] = reinterpret_cast<const float2u*>(hb + (int64_t)b * cols + k * 32)[at];
    }
    __device__ __forceinline__ void mac(const uint4 w, float sc, const X& x)
    {
        const float s512 = 512.0f * sc, m8 = -8.0f * sc;
        float q[8];
        dequant8(w.x, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<0>(S[b], q, x.v[b]);
        dequant8(w.y, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<1>(S[b], q, x.v[b]);
        dequant8(w.z, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<2>(S[b], q, x.v[b]);
        dequant8(w.w, s512, m8, q);
#pragma unroll
        for (int b = 0; b < NV; ++b) fmac8<3>(S[b], q, x.v[b]);
    }
    template <typename F>
    __device__ __forceinline__ void emit(F put) const
    {
#pragma unroll
        for (int b = 0; b < NV; ++b) put(S[b], b);
    }
};

/* smax: the largest scale of a lane's row.  (Of fmaxf the compiler makes one
 * v_max3_f32 for two blocks and waits for the second block's loads before the
 * first is summed: 76.5 us instead of 74.9 for one vector.) */
__device__ __forceinline__ void max_scale(float& smax, float s)
{
    asm("v_max_f32 %0, %0, |%1|" : "+v"(smax) : "v"(s));
}

/* The sums of the rows with an infinite scale, of which dequant8 makes NaN,
 * taken again with the reference's product.  Waves without such a row end at
 * the test (262,144 x 2,560: 74.9 us for one vector, 368 for 32; with
 * q4_dequant8 for every sum 76.8 and 371.6).  block(k, s, w): the lane's block
 * k; rows that are not live have sums that nobody reads. */
template <int VECS, typename Block, typename Put>
__device__ __forceinline__ void sum_infinite(float smax, bool live, const float* h, int32_t cols,
                                             int32_t nblk, int32_t b0, int32_t batch, Block block,
                                             Put put)
{
    if (__builtin_expect(__ballot(live && smax == __builtin_inff()) == 0, 1)) return;
    for (int32_t i = 0; i < VECS && b0 + i < batch; ++i) {
        const float* x = h + (int64_t)(b0 + i) * cols;
        float S = 0.0f;
        for (int32_t k = 0; k < nblk; ++k, x += 32) {
            float s;
            uint32_t w[4];
            block(k, s, w);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                float q[8];
                q4_dequant8(w[d], 16.0f * s, q);
#pragma unroll
                for (int j = 0; j < 8; ++j) S = __builtin_fmaf(q[j], x[8 * d + j], S);
            }
        }
        put(S, i);
    }
}

template <typename Acc, int DEPTH>
__global__ __launch_bounds__(64 * kTileWaves, 4) void lmhead_tiled_kernel(
    const uint8_t* __restrict__ tiles, int32_t rows, int32_t nblk, const float* __restrict__ h,
    int32_t cols, int32_t batch, float* __restrict__ out, int64_t stride, uint64_t* __restrict__ gsum,
    int32_t ngroups)
{
    const int lane = threadIdx.x & 63;
    const int32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x * kTileWaves + (threadIdx.x >> 6));
    if (g >= ngroups) return; /* whole waves: no barrier below */
    const int32_t b0 = blockIdx.y * Acc::kVecs;
    const uint8_t* tp = tiles + (int64_t)g * nblk * kQ4TileBytes;
    Acc acc;
    acc.init(h, cols, b0, batch, lane);
    float sc[DEPTH], smax = 0.0f;
    uint4 w[DEPTH];
    typename Acc::X x[DEPTH];
    const auto fetch = [&](int d, int32_t k) {
        const uint8_t* t = tp + (uint32_t)k * (uint32_t)kQ4TileBytes;
        sc[d] = reinterpret_cast<const float*>(t)[lane];
        w[d] = reinterpret_cast<const uint4*>(t + kQ4TileRows * 4)[lane];
        acc.load(x[d], k);
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
            max_scale(smax, sc[d]);
            acc.mac(w[d], sc[d], x[d]);
            const int32_t kn = k + d + DEPTH;
            fetch(d, kn < nblk ? kn : nblk - 1);
            /* keeps each load where it is issued, DEPTH blocks before its use */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) {
        if (k + d < nblk) {
            max_scale(smax, sc[d]);
            acc.mac(w[d], sc[d], x[d]);
        }
    }
    const int32_t r = g * kQ4TileRows + lane;
    const auto put = [&](float v, int i) {
        if (b0 + i < batch) put_logit(v, b0 + i, r, rows, lane, g, ngroups, out, stride, gsum);
    };
    acc.emit(put);
    const auto block = [&](int32_t kb, float& s, uint32_t (&q)[4]) {
        const uint8_t* t = tp + (uint32_t)kb * (uint32_t)kQ4TileBytes;
        s = reinterpret_cast<const float*>(t)[lane];
        const uint4 n = reinterpret_cast<const uint4*>(t + kQ4TileRows * 4)[lane];
        q[0] = n.x, q[1] = n.y, q[2] = n.z, q[3] = n.w;
    };
    sum_infinite<Acc::kVecs>(smax, r < rows, h, cols, nblk, b0, batch, block, put);
}

/* ------------------------------------------------------------------
 * The LM head on the engine's own rows (18-byte blocks).
 *
 * Read lane by lane, a wave's 64 rows are 64 cache lines per 18 bytes.  So a
 * wave copies kRowKb blocks of its rows at a time into its own LDS (9 lanes
 * read 144 bytes of a row, seven rows a load; held in registers while the
 * previous stage is summed) and each lane then reads its own row from there.
 * The LDS pitch is an odd number of dwords, so the reads have no bank conflicts
 * (the copies, 16 bytes a lane over rows of that pitch, have some: 3.1 M cycles
 * over 256 compute units).  At least three waves a SIMD (141 VGPRs with 32
 * vectors; one vector takes 95 and fills the LDS with 16 waves a compute unit).
 *
 * 262,144 x 2,560: B = 1 652 -> 102 us, B = 8 667 -> 177, B = 32 740 -> 380-390
 * (one row per thread before, 32 vectors' time for any batch).  B = 1 is
 * bound by the weights' reads, which a stage's ends make 1.7 times their size
 * (a line shared by two stages has left L2 in between: 4,096 waves keep 70 MB
 * in flight; without the sums 95 us).  16 blocks a stage at
 * two waves a SIMD take 105, 187 and 387 us, and 100,003 x 1,120 for two
 * vectors 36 us against 30; four waves a SIMD spill at 32 vectors (409 us).
 * ------------------------------------------------------------------ */

constexpr int kRowKb = 8;                                 /* blocks per stage */
constexpr int kRowBytes = kRowKb * 18;
constexpr int kRowChunks = kRowBytes / 16;                /* 16-byte loads per row and stage */
constexpr int kRowPitch = kRowBytes / 4 + 1;              /* dwords */
constexpr int kRowPer = 64 / kRowChunks;                  /* rows per load */
constexpr int kRowLoads = (kQ4TileRows + kRowPer - 1) / kRowPer;
constexpr int kRowEach = (kRowLoads + kRowKb / 2 - 1) / (kRowKb / 2); /* issued per block */
static_assert(kRowBytes % 16 == 0, "whole 16-byte loads");

/* 16 bytes at `a`, of which only those below `hi` are read (the others come back
 * as anything); at least 16 bytes lie below `hi`. */
__device__ __forceinline__ uint4 load16_within(const uint8_t* a, const uint8_t* hi)
{
    const uint8_t* at = a > hi - 16 ? hi - 16 : a;
    const uint4u q = *reinterpret_cast<const uint4u*>(at);
    const int64_t off = a - at; /* the wanted bytes are this much further up */
    const int up = off > 15 ? 120 : (int)off * 8;
    const uint64_t l = ((uint64_t)q.y << 32) | q.x, u = ((uint64_t)q.w << 32) | q.z;
    const unsigned __int128 v = (((unsigned __int128)u << 64) | l) >> up;
    const uint64_t vl = (uint64_t)v, vu = (uint64_t)(v >> 64);
    return make_uint4((uint32_t)vl, (uint32_t)(vl >> 32), (uint32_t)vu, (uint32_t)(vu >> 32));
}

template <typename Acc, int DEPTH>
__global__ __launch_bounds__(64, 3) void lmhead_rows_kernel(
    const uint8_t* __restrict__ wt, int32_t rows, int32_t nblk, const float* __restrict__ h,
    int32_t cols, int32_t batch, float* __restrict__ out, int64_t stride)
{
    static_assert(kRowKb % 2 == 0 && kRowKb % DEPTH == 0, "whole pairs, whole prefetch rounds");
    __shared__ uint32_t stage[kQ4TileRows * kRowPitch];
    const int lane = threadIdx.x;
    const int32_t b0 = blockIdx.y * Acc::kVecs;
    const int64_t pitch = (int64_t)nblk * 18;
    const uint8_t* const wend = wt + (int64_t)rows * pitch;
    const int32_t nstage = (nblk + kRowKb - 1) / kRowKb;
    /* the last wave takes the last 64 rows and writes those that are its own */
    const int32_t own = blockIdx.x * kQ4TileRows;
    const int32_t r0 = own + kQ4TileRows <= rows ? own : rows > kQ4TileRows ? rows - kQ4TileRows : 0;
    const uint8_t* const base = wt + (int64_t)r0 * pitch;
    const int sub = lane / kRowChunks, chunk = lane % kRowChunks;
    const uint32_t voff = (uint32_t)sub * (uint32_t)pitch + 16u * chunk;
    /* lane's copies of load j: row kRowPer * j + sub */
    const auto copies = [&](int j) { return sub < kRowPer && kRowPer * j + sub < kQ4TileRows; };
    /* a stage whose copies could leave the weights: past the end of the last
     * rows, or fewer than 64 rows at all */
    const auto edge = [&](int32_t s) {
        return base + (kQ4TileRows - 1) * pitch + (int64_t)(s + 1) * kRowBytes > wend;
    };
    uint4 st[kRowLoads];
    const auto fetch = [&](int j, int32_t s) {
        if (copies(j)) {
            const uint4u q = *reinterpret_cast<const uint4u*>(
                base + ((int64_t)s * kRowBytes + (int64_t)(kRowPer * j) * pitch) + voff);
            st[j] = make_uint4(q.x, q.y, q.z, q.w);
        }
    };
    uint32_t* const copy_to = stage + sub * kRowPitch + 4 * chunk;
    const auto put = [&](int j, const uint4 v) {
        if (copies(j)) {
            uint32_t* d = copy_to + kRowPer * j * kRowPitch;
            d[0] = v.x;
            d[1] = v.y;
            d[2] = v.z;
            d[3] = v.w;
        }
    };
    const uint32_t* const lrow = stage + lane * kRowPitch;
    Acc acc;
    acc.init(h, cols, b0, batch, lane);
    typename Acc::X x[DEPTH];
    float smax = 0.0f;
    if (!edge(0)) {
#pragma unroll
        for (int j = 0; j < kRowLoads; ++j) fetch(j, 0);
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) acc.load(x[d], d < nblk ? d : nblk - 1);
    __builtin_amdgcn_sched_barrier(0);
    for (int32_t s = 0; s < nstage; ++s) {
        if (edge(s)) {
#pragma unroll 6
            for (int j = 0; j < kRowLoads; ++j)
                put(j, load16_within(
                           base + ((int64_t)s * kRowBytes + (int64_t)(kRowPer * j) * pitch) + voff,
                           wend));
        } else {
#pragma unroll
            for (int j = 0; j < kRowLoads; ++j) put(j, st[j]);
        }
        /* one wave: its LDS operations run in order */
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const bool more = s + 1 < nstage && !edge(s + 1);
        uint32_t raw[2][9]; /* two blocks (36 bytes), read two blocks ahead */
        const auto pair = [&](int p) {
#pragma unroll
            for (int i = 0; i < 9; ++i) raw[p & 1][i] = lrow[9 * p + i];
        };
        pair(0);
#pragma unroll
        for (int i = 0; i < kRowKb; ++i) {
            const int32_t k = s * kRowKb + i;
            if (k >= nblk) break;
            if (more) {
#pragma unroll
                for (int j = kRowEach * i; j < kRowEach * (i + 1); ++j)
                    if (j < kRowLoads) fetch(j, s + 1);
            }
            const uint32_t* e = raw[(i / 2) & 1];
            uint32_t half;
            uint4 w;
            if (i % 2 == 0) {
                if (i + 2 < kRowKb) pair(i / 2 + 1);
                half = e[0] & 0xFFFFu;
                w = make_uint4(
                    __builtin_amdgcn_alignbit(e[1], e[0], 16), __builtin_amdgcn_alignbit(e[2], e[1], 16),
                    __builtin_amdgcn_alignbit(e[3], e[2], 16), __builtin_amdgcn_alignbit(e[4], e[3], 16));
            } else {
                half = e[4] >> 16;
                w = make_uint4(e[5], e[6], e[7], e[8]);
            }
            const float sc = f16_to_f32_fast(half);
            max_scale(smax, sc);
            acc.mac(w, sc, x[i % DEPTH]);
            const int32_t kn = k + DEPTH;
            acc.load(x[i % DEPTH], kn < nblk ? kn : nblk - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_wave_barrier(); /* the next stage is written after these reads */
    }
    const int32_t r = r0 + lane;
    const bool live = r >= own && r < rows;
    const auto write = [&](float v, int i) {
        if (b0 + i < batch && live) out[(int64_t)(b0 + i) * stride + r] = v;
    };
    acc.emit(write);
    const auto block = [&](int32_t kb, float& s, uint32_t (&q)[4]) {
        const uint8_t* b = wt + (int64_t)(live ? r : own) * pitch + kb * 18;
        s = f16_to_f32_ref((uint32_t)b[0] | ((uint32_t)b[1] << 8));
        const uint4u n = *reinterpret_cast<const uint4u*>(b + 2);
        q[0] = n.x, q[1] = n.y, q[2] = n.z, q[3] = n.w;
    };
    sum_infinite<Acc::kVecs>(smax, live, h, cols, nblk, b0, batch, block, write);
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

/* The split of a launch into waves of 64 rows and some vectors:
 *  - every (row group, vector) pair its own wave while that leaves at most
 *    one wave per SIMD, and up to two vectors otherwise: the plain fma kernel
 *    (2,560 columns: 20 us for 8,000 rows x 8 against 31 us with four vectors
 *    a wave; 262,144 rows: 74 us for one vector against 105, 85-91 for two);
 *  - else 4 * NG vectors a wave on the matrix cores, NG as large as needed
 *    (up to 8) to leave at most one wave per SIMD (32,768 rows x 32: NG = 4
 *    66 us, NG = 2 75, NG = 8 105; 262,144 rows x 32: NG = 8 396 us, NG = 4
 *    460), and the 32-vector form where a wave takes 29 to 32 (364 us; at 28 it
 *    takes 359 against 354 with NG = 7).
 * launch(accumulator, prefetch depth, slices of the batch) starts the kernel. */
constexpr int32_t kLmSimds = 1024;

template <int D>
struct Depth {
    static constexpr int value = D;
};

template <typename F>
void lmhead_split(int32_t ngroups, int32_t batch, F launch)
{
    if (batch <= 2 || (int64_t)batch * ngroups <= kLmSimds) {
        if ((int64_t)batch * ngroups <= kLmSimds || batch == 1)
            launch(FewAcc<1>{}, Depth<4>{}, batch);
        else
            launch(FewAcc<2>{}, Depth<4>{}, 1);
        return;
    }
    const int32_t quads = (batch + 3) / 4;
    const int32_t fill = kLmSimds / ngroups;
    int32_t passes = (quads + 7) / 8;
    if (passes < fill) passes = fill < quads ? fill : quads;
    const int32_t ng = (quads + passes - 1) / passes;
    passes = (quads + ng - 1) / ng;
    switch (ng) {
        case 1: launch(QuadAcc<1>{}, Depth<4>{}, passes); break;
        case 2: launch(QuadAcc<2>{}, Depth<4>{}, passes); break;
        case 3: launch(QuadAcc<3>{}, Depth<3>{}, passes); break;
        case 4: launch(QuadAcc<4>{}, Depth<2>{}, passes); break;
        case 5: launch(QuadAcc<5>{}, Depth<2>{}, passes); break;
        case 6: launch(QuadAcc<6>{}, Depth<2>{}, passes); break;
        case 7: launch(QuadAcc<7>{}, Depth<2>{}, passes); break;
        default: launch(WideAcc{}, Depth<2>{}, passes); break;
    }
}

/* Vectors of one launch: byte offsets into its hidden values stay within 31
 * bits, its slices within a grid's second dimension. */
int32_t lmhead_most(int32_t cols)
{
    const int64_t most = INT32_MAX / ((int64_t)cols * 4);
    return (int32_t)(most < 1 ? 1 : most > 65535 ? 65535 : most);
}

hipError_t lmhead_tiled_launch(const uint8_t* tiles, int32_t rows, int32_t cols, const float* h,
                               int32_t batch, float* logits, int64_t stride, uint64_t* gsum,
                               hipStream_t s)
{
    const int32_t ngroups = (rows + kQ4TileRows - 1) / kQ4TileRows;
    const int32_t nblk = cols / 32;
    const unsigned gx = (unsigned)((ngroups + kTileWaves - 1) / kTileWaves);
    const int32_t most = lmhead_most(cols);
    for (int32_t b0 = 0; b0 < batch; b0 += most) {
        const int32_t n = batch - b0 < most ? batch - b0 : most;
        const float* hb = h + (int64_t)b0 * cols;
        float* lb = logits ? logits + (int64_t)b0 * stride : nullptr;
        uint64_t* gb = gsum ? gsum + (int64_t)b0 * ngroups : nullptr;
        lmhead_split(ngroups, n, [&](auto acc, auto depth, int32_t passes) {
            hipLaunchKernelGGL((lmhead_tiled_kernel<decltype(acc), decltype(depth)::value>),
                               dim3(gx, (unsigned)passes), dim3(64 * kTileWaves), 0, s, tiles, rows,
                               nblk, hb, cols, n, lb, stride, gb, ngroups);
        });
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t lmhead_q4_0_launch(const uint8_t* w, int32_t rows, int32_t cols, const float* h,
                              int32_t batch, float* logits, int64_t stride, hipStream_t s)
{
    const int32_t ngroups = (rows + kQ4TileRows - 1) / kQ4TileRows;
    const int32_t nblk = cols / 32;
    const int32_t most = lmhead_most(cols);
    for (int32_t b0 = 0; b0 < batch; b0 += most) {
        const int32_t n = batch - b0 < most ? batch - b0 : most;
        const float* hb = h + (int64_t)b0 * cols;
        float* lb = logits + (int64_t)b0 * stride;
        lmhead_split(ngroups, n, [&](auto acc, auto depth, int32_t passes) {
            /* prefetch distance in a stage of kRowKb blocks: a power of two */
            constexpr int D = decltype(depth)::value == 3 ? 4 : decltype(depth)::value;
            const dim3 grid((unsigned)ngroups, (unsigned)passes);
            hipLaunchKernelGGL((lmhead_rows_kernel<decltype(acc), D>), grid, dim3(64), 0, s, w, rows,
                               nblk, hb, cols, n, lb, stride);
        });
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace g4s
