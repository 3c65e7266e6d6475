// INT8 linear layer for gfx950: out[t][n] = epilogue(sum_k a[t][k] * w[n][k]).
//
// The projections between the encoder plugins (QKV, attention output, the two feed-forward
// layers) are plain GEMMs whose operands are both contiguous along k, which is what the INT8 MFMA
// wants: a lane feeds 16 consecutive k-bytes of one row.  v_mfma_i32_32x32x32_i8 is used: it runs at
// the full INT8 rate of the matrix core (measured: 32768 MACs in 33 cycles per SIMD, as does
// v_mfma_i32_16x16x64_i8 with 16384 in 16.5) and needs half as many fragment reads per MAC as the
// 16 x 16 form.  The kernel computes the transposed
// product (output channels are the M dimension, tokens the N dimension) so that a lane ends up with
// groups of four consecutive channels of one token, which pack into the token-major INT8 output of
// either layout.
//
// Tiling: a workgroup owns BM channels x BN tokens, its waves a WM x WN grid of (MT*32) x (NT*32)
// sub-tiles kept in INT32 (FP16 operands: binary32) accumulators.  Global loads are 16 bytes per lane,
// and a swizzle keeps the 16-byte-per-lane fragment reads from LDS conflict-free.  Three ways to bring
// a tile's operands in:
//   operands of one layout, chip-filling or middling launches: rings of stages of 64 or, for linear rows
//     of whole lines, 128 bytes of k by direct-to-LDS loads (linear_tile_dma; persistent 256 x 256 tiles of
//     interleaved operands: linear_tile_run_dma);
//   operands of one layout, few tokens: pieces whose eight wavefronts split k (linear_piece_kernel,
//     linear_piece_dma_kernel, linear_piece64);
//   operands of two layouts, INT32 and FP16 outputs of INT8 operands, or TRTAMD_LINEAR_DIRECT=0: stages of
//     64 bytes, double-buffered in LDS, through two register sets that run two stages ahead (linear_tile,
//     linear_tile_run).
//
// Activations, weights and outputs may be in the linear layout [R][C] or in the 32-interleaved
// layout [C/32][R][32] that the interleaved encoder plugins use; the interleaved one makes every
// load unit 1 KB of contiguous memory.
#include "device_utils.hpp"
#include "host_utils.hpp"
#include "network_ops.hpp"
#include "trtamd_encoder_ops.h"
#include "trtamd_test_hooks.h"

#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

namespace trtamd
{
namespace
{

constexpr int kBigTile = 256; // channels and tokens of the large workgroup tile

enum Epilogue
{
    kAFFINE = TRTAMD_LINEAR_AFFINE,
    kGELU = TRTAMD_LINEAR_GELU,
    kRAW = TRTAMD_LINEAR_RAW_INT32,
    kHALF = TRTAMD_LINEAR_AFFINE_FP16,
    // FP16 operands (trtamd_fp16_linear): the same kernels with v_mfma_f32_32x32x16_f16 and binary32 accumulators
    kF16_AFFINE = 4,
    kF16_GELU = 5,
    kF16_RAW = 6 // the binary32 accumulators (partial sums of fp16_linear_partial)
};

// INT8 operands accumulate in INT32, FP16 operands in binary32.  Either way a lane feeds 16 bytes of a row per
// operand and MFMA step (16 INT8 or 8 FP16 values of k), a fragment is 32 rows x 32 bytes, and the result has the
// same 32 x 32 accumulator layout, so the tiling, the LDS layout and the load schedule are shared.
template <int EPI>
using AccT = std::conditional_t<(EPI >= kF16_AFFINE), f32x16, i32x16>;

template <int EPI>
__device__ __forceinline__ AccT<EPI> mma(i32x4 const a, i32x4 const b, AccT<EPI> const c)
{
    if constexpr (EPI >= kF16_AFFINE)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(bits_as<f16x8>(a), bits_as<f16x8>(b), c, 0, 0, 0);
    }
    else
    {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
}

struct LinearArgs
{
    int8_t const* a;
    int8_t const* w;
    float const* alpha;
    float const* beta;
    void* out;
    int T, K, N; // K: bytes of k per row (elements for INT8, twice the elements for FP16)
    float qOut;
    int mainTiles; // workgroups that own a 256 x 256 tile
    int tokMain;   // rows of 256 tokens they cover
    int panel;     // channel tiles per panel of the tile numbering (divides the number of channel tiles)
    int persist;   // persistent kernel: workgroups that loop over the 256 x 256 tiles
    int pieces;    // large tiles: the tokens behind them go in 64 x 64 pieces (see linear_piece64)
    int parts;     // pieces: workgroups that share the k range of a piece, each with an output of its own
    int perPart;   // pieces: 32-byte k-slabs (interleaved operands) or stages of 64 or 128 bytes of each
    FastDiv panelDiv, perPanelDiv; // tiles: by panel and tokMain * panel
    WeightPrefetch prefetch; // by the workgroups behind mainTiles of the interleaved tile and piece kernels
};

// gelu(y) = y * Phi(y) = max(y, 0) - |y| * Phi(-|y|).  log2(Phi(-a)) is smooth and nearly quadratic, so
// Phi(-a) = exp2(P(a)) with a cubic fitted to minimise the error of a * Phi(-a) on [0, 7]; the leading coefficient is
// negative, so the term vanishes for larger a as it should.  Measured against the binary64 erf form the absolute
// error of gelu is below 5.5e-5 for every binary32 |y| <= 40 (largest near |y| = 1.1): at the output scales of an
// INT8 feed-forward layer (20-40 steps per unit) that moves 0.04-0.1 % of the requantised values by one step, half
// of what the parity tests allow, and it is far inside the FP16 output's tolerance.  Three fma, one v_exp_f32, one
// max and one fma per value (a degree-5 fit, 6.4e-7 and two more fma, measured the same results to 0.001 %).
__device__ inline float gelu_erf(float y)
{
    float const a = fabsf(y);
    float p = fmaf(a, -2.488555945e-02f, -4.988203049e-01f);
    p = fmaf(p, a, -1.129245639e+00f);
    p = fmaf(p, a, -1.003531814e+00f);
    return fmaf(-a, __builtin_amdgcn_exp2f(p), fmaxf(y, 0.f));
}

// One operand fragment of v_mfma_i32_32x32x32_i8 is 32 rows x 32 k-bytes; lane l feeds row l%32,
// bytes 16*(l/32)..+15.  In LDS a fragment is 1 KB, row-major, with the two 16-byte halves of a row
// swapped for rows 8..15 and 24..31: a 16-lane group then reads 16 different 16-byte columns of the
// bank array, and so does a group that writes 8 whole rows.
__device__ inline int frag_offset(int row, int half)
{
    return row * 32 + ((half ^ ((row >> 3) & 1)) << 4);
}

// Epilogue of one 32 x 32 accumulator block whose first channel is c0 (sAlpha / sBeta point at that channel's
// entry) and first token tb.  Accumulator register v is token l%32, channel 8*(v/4) + 4*(l/32) + v%4: four groups
// of four consecutive channels.  For the INT8 outputs the two lanes that share a token trade two packed dwords
// (v_permlane32_swap), after which lane l holds the 16 consecutive channels 16*(l/32)..+15 and stores them with
// one 16-byte write.
// THROUGH: the store writes through the L2 (inline assembly, which the compiler's own vmcnt bookkeeping does not see:
// only for the kernel that places its waits itself, and only where a wavefront's store covers whole cache lines, the
// 32-interleaved INT8 output: 32 tokens x 32 bytes; narrower pieces are better merged in the L2 first).
template <bool THROUGH, typename V>
__device__ __forceinline__ void store_out(void* p, V const& v)
{
    if constexpr (THROUGH)
    {
        store_through_l2(p, v);
    }
    else
    {
        *static_cast<V*>(p) = v;
    }
}

// The 16 scale / offset pairs a lane needs for one 32-channel block (channels 8g + 4 (l/32) + e of the block), read
// from the tile's vectors in LDS.  For the affine INT8 epilogue the offsets already carry the 128 of the unsigned
// byte conversion.  A block's scales serve every token block of the same channels, so callers that walk several
// token blocks load them once.
struct BlockScales
{
    f32x4 al[4], be[4];
};

template <int EPI>
__device__ __forceinline__ BlockScales load_block_scales(float const* sAlpha, float const* sBeta)
{
    BlockScales s;
    if constexpr (EPI != kRAW)
    {
        int const hi = (threadIdx.x & 63) >> 5;
#pragma unroll
        for (int g = 0; g < 4; ++g)
        {
            s.al[g] = *reinterpret_cast<f32x4 const*>(sAlpha + 8 * g + 4 * hi);
            s.be[g] = *reinterpret_cast<f32x4 const*>(sBeta + 8 * g + 4 * hi);
            if constexpr (EPI == kAFFINE)
            {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    s.be[g][e] += 128.f;
                }
            }
        }
    }
    return s;
}

// The FP16 results of a 32 x 32 block: 16 consecutive channels, 16 (l/32) .. +15, of token l%32 per lane.
template <int EPI>
__device__ __forceinline__ void pack_half_block(AccT<EPI> const& acc, BlockScales const& sc, u32x4& first, u32x4& second)
{
    u32x2 w[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
    {
        f16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            float const y = fmaf((float) acc[4 * g + e], sc.al[g][e], sc.be[g][e]);
            h[e] = (f16) (EPI == kF16_GELU ? gelu_erf(y) : y);
        }
        w[g] = __builtin_bit_cast(u32x2, h);
    }
    // lanes l < 32 hold channels 8g..8g+3 of each group g, lanes l+32 the other four: after the swaps lane l has
    // groups 0 and 1 whole, lane l+32 groups 2 and 3
    auto const a0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[2][0], false, false);
    auto const a1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[2][1], false, false);
    auto const b0 = __builtin_amdgcn_permlane32_swap(w[1][0], w[3][0], false, false);
    auto const b1 = __builtin_amdgcn_permlane32_swap(w[1][1], w[3][1], false, false);
    first = u32x4{a0[0], a1[0], a0[1], a1[1]};
    second = u32x4{b0[0], b1[0], b0[1], b1[1]};
}

template <bool IL_OUT, int EPI, bool FULL = false, bool THROUGH = false>
__device__ __forceinline__ void store_block_scaled(
    LinearArgs const& p, AccT<EPI> const& acc, int const c0, int const tb, BlockScales const& sc)
{
    int const lane = threadIdx.x & 63;
    int const hi = lane >> 5;
    int const t = tb + (lane & 31);
    bool const live = FULL || t < p.T; // FULL: the block lies inside the problem and is stored unconditionally
    f32x4 const(&al)[4] = sc.al;
    f32x4 const(&be)[4] = sc.be;
    if constexpr (EPI == kRAW)
    {
        if (live)
        {
#pragma unroll
            for (int g = 0; g < 4; ++g)
            {
                i32x4 const v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
                store_out<THROUGH>(static_cast<int32_t*>(p.out) + (size_t) t * p.N + c0 + 8 * g + 4 * hi, v);
            }
        }
    }
    else if constexpr (EPI >= kF16_AFFINE || EPI == kHALF)
    {
        u32x4 first, second;
        pack_half_block<EPI>(acc, sc, first, second);
        if (live)
        {
            f16* dst = static_cast<f16*>(p.out) + (size_t) t * p.N + c0 + 16 * hi;
            store_out<THROUGH>(dst, first);
            store_out<THROUGH>(dst + 8, second);
        }
    }
    else
    {
        // Results are formed as unsigned bytes, x + 128: v_cvt_pk_u8_f32 rounds to nearest even, saturates to
        // [0, 255] and places the byte in one instruction; one XOR per dword returns to two's complement.
        int d[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
        {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                if constexpr (EPI == kGELU)
                {
                    float const y = fmaf((float) acc[4 * g + e], al[g][e], be[g][e]);
                    w = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(gelu_erf(y), p.qOut, 128.f), e, w);
                }
                else
                {
                    w = __builtin_amdgcn_cvt_pk_u8_f32(fmaf((float) acc[4 * g + e], al[g][e], be[g][e]), e, w);
                }
            }
            d[g] = (int) (w ^ 0x80808080u);
        }
        // lanes l < 32 hold channels [0-3][8-11][16-19][24-27], lanes l+32 the gaps
        auto const s02 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
        auto const s13 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
        i32x4 const packed = {(int) s02[0], (int) s02[1], (int) s13[0], (int) s13[1]};
        if (live)
        {
            int const c = c0 + 16 * hi;
            size_t const o = IL_OUT ? ((size_t) (c >> 5) * p.T + t) * 32 + (c & 31) : (size_t) t * p.N + c;
            store_out<THROUGH>(static_cast<int8_t*>(p.out) + o, packed);
        }
    }
}

template <bool IL_OUT, int EPI, bool FULL = false, bool THROUGH = false>
__device__ __forceinline__ void store_block(
    LinearArgs const& p, AccT<EPI> const& acc, int const c0, int const tb, float const* sAlpha, float const* sBeta)
{
    store_block_scaled<IL_OUT, EPI, FULL, THROUGH>(p, acc, c0, tb, load_block_scales<EPI>(sAlpha, sBeta));
}

// Epilogue of one workgroup tile.
template <int WM, int WN, int MT, int NT, bool IL_OUT, int EPI>
__device__ __forceinline__ void store_tile(LinearArgs const& p, AccT<EPI> const (&acc)[MT][NT], int const n0, int const t0,
    float const* sAlpha, float const* sBeta)
{
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const wm = wave / WN;
    int const wn = wave % WN;
#pragma unroll
    for (int i = 0; i < MT; ++i)
    {
        int const cl = (wm * MT + i) * 32; // wave-uniform, and so is the guard: N is a multiple of 32
        if (n0 + cl >= p.N)
        {
            break;
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
            store_block<IL_OUT, EPI>(p, acc[i][j], n0 + cl, t0 + (wn * NT + j) * 32, sAlpha + cl, sBeta + cl);
        }
    }
}

// One output tile of BM = WM*MT*32 channels x BN = WN*NT*32 tokens at (n0, t0), by the whole workgroup.
template <int WM, int WN, int MT, int NT, bool IL_W, bool IL_IN, bool IL_OUT, int EPI>
__device__ __forceinline__ void linear_tile(
    LinearArgs const& p, int const n0, int const t0, uint8_t* __restrict__ lds, float* sAlpha, float* sBeta)
{
    constexpr int NWAVES = WM * WN;
    constexpr int BM = WM * MT * 32;    // output channels per workgroup
    constexpr int BN = WN * NT * 32;    // tokens per workgroup
    constexpr int AF = (BM / 32) * 2;   // weight fragments per stage (64 bytes of k = two MFMA steps)
    constexpr int BF = (BN / 32) * 2;   // activation fragments per stage
    static_assert(AF % NWAVES == 0 && BF % NWAVES == 0, "load units divide evenly among the waves");
    constexpr int LA = AF / NWAVES;
    constexpr int LB = BF / NWAVES;
    constexpr int STAGE = (AF + BF) * 1024;

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const wm = wave / WN;
    int const wn = wave % WN;
    int const col32 = lane & 31;
    int const hi = lane >> 5;

    // A load unit is 1 KB that one wave fetches with one 16-byte load per lane, consecutive lanes
    // reading consecutive memory.  Interleaved operand [K/32][R][32]: unit (rb, ks) is the 32 rows of
    // row block rb in k-slab ks, contiguous in memory, and is exactly one fragment.  Linear operand
    // [R][K]: unit (rb, h) is rows 16h..16h+15 of the block, 64 bytes of k each, and lands in the two
    // fragments (rb, 0) and (rb, 1).
    auto unit_addressing = [&](bool interleaved, int unit, int row0, int R, uint32_t& gOff, int& lOff) {
        int const rb = unit >> 1, sel = unit & 1;
        if (interleaved)
        {
            int const r = lane >> 1, c = lane & 1;
            int const row = min(row0 + rb * 32 + r, R - 1);
            gOff = ((uint32_t) sel * (uint32_t) R + (uint32_t) row) * 32u + (uint32_t) c * 16u;
            lOff = (rb * 2 + sel) * 1024 + frag_offset(r, c);
        }
        else
        {
            int const r = sel * 16 + (lane >> 2), c = lane & 3;
            int const row = min(row0 + rb * 32 + r, R - 1);
            gOff = (uint32_t) row * (uint32_t) p.K + (uint32_t) c * 16u;
            lOff = (rb * 2 + (c >> 1)) * 1024 + frag_offset(r, c & 1);
        }
    };
    uint32_t offA[LA], offB[LB];
    int ldsA[LA], ldsB[LB];
#pragma unroll
    for (int q = 0; q < LA; ++q)
    {
        unit_addressing(IL_W, q * NWAVES + wave, n0, p.N, offA[q], ldsA[q]);
    }
#pragma unroll
    for (int q = 0; q < LB; ++q)
    {
        unit_addressing(IL_IN, q * NWAVES + wave, t0, p.T, offB[q], ldsB[q]);
        ldsB[q] += AF * 1024;
    }
    uint32_t const stepA = IL_W ? 2u * (uint32_t) p.N * 32u : 64u;
    uint32_t const stepB = IL_IN ? 2u * (uint32_t) p.T * 32u : 64u;

    // two register sets: the loads of stage s+2 are issued while stage s is multiplied, so a load has
    // two stages of MFMA work to hide behind before its data is moved to LDS
    i32x4 ga[2][LA], gb[2][LB];
    auto fetch = [&](auto set, int kt) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            ga[S][q] = *reinterpret_cast<i32x4 const*>(p.w + offA[q] + (uint32_t) kt * stepA);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            gb[S][q] = *reinterpret_cast<i32x4 const*>(p.a + offB[q] + (uint32_t) kt * stepB);
        }
    };
    auto stash = [&](auto set, int buf) {
        constexpr int S = decltype(set)::value;
        uint8_t* base = lds + buf * STAGE;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            *reinterpret_cast<i32x4*>(base + ldsA[q]) = ga[S][q];
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            *reinterpret_cast<i32x4*>(base + ldsB[q]) = gb[S][q];
        }
    };

    AccT<EPI> acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
    {
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                acc[i][j][v] = 0;
            }
        }
    }
    int const readOff = frag_offset(col32, hi);
    auto multiply = [&](int buf) {
        uint8_t const* base = lds + buf * STAGE + readOff;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
        {
            i32x4 fa[MT], fb[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                fa[i] = *reinterpret_cast<i32x4 const*>(base + ((wm * MT + i) * 2 + ks) * 1024);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
            {
                fb[j] = *reinterpret_cast<i32x4 const*>(base + (AF + (wn * NT + j) * 2 + ks) * 1024);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
#pragma unroll
                for (int j = 0; j < NT; ++j)
                {
                    acc[i][j] = mma<EPI>(fa[i], fb[j], acc[i][j]);
                }
            }
        }
    };
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;

    // per-channel scale and offset of the tile, staged once for the epilogue
    if constexpr (EPI != kRAW)
    {
        for (int c = threadIdx.x; c < BM; c += 64 * NWAVES)
        {
            int const n = min(n0 + c, p.N - 1);
            sAlpha[c] = p.alpha[n];
            sBeta[c] = p.beta[n];
        }
    }

    // Stage kt sits in LDS buffer kt&1 and arrived through register set kt&1.  The loop body has no
    // branches (loads past the last stage re-read the last stage and are never used), so the number of
    // loads in flight at every point is fixed and a stash waits for its own four loads only.
    int const nk = p.K / 64;
    fetch(Set0{}, 0);
    fetch(Set1{}, min(1, nk - 1));
    stash(Set0{}, 0);
    __syncthreads();
    int kt = 0;
    for (; kt + 1 < nk; kt += 2)
    {
        fetch(Set0{}, min(kt + 2, nk - 1));
        multiply(0);
        stash(Set1{}, 1);
        __syncthreads();
        fetch(Set1{}, min(kt + 3, nk - 1));
        multiply(1);
        stash(Set0{}, 0);
        __syncthreads();
    }
    if (kt < nk)
    {
        multiply(0);
    }

    store_tile<WM, WN, MT, NT, IL_OUT, EPI>(p, acc, n0, t0, sAlpha, sBeta);
}

// A run of `count` tiles by one persistent workgroup, K % 128 == 0.  The stage pipeline does not drain
// between tiles: the last two stages of a tile already fetch the first two stages of the next one, the
// epilogue runs while those loads are in flight, and the next tile's scale/offset vectors are picked up at
// the start of the current one.  `origin(j, n0, t0)` gives the j-th tile's corner.
template <int WM, int WN, int MT, int NT, bool IL_W, bool IL_IN, bool IL_OUT, int EPI, typename Origin>
__device__ __forceinline__ void linear_tile_run(
    LinearArgs const& p, int const count, Origin origin, uint8_t* __restrict__ lds, float* sScale)
{
    constexpr int NWAVES = WM * WN;
    constexpr int BM = WM * MT * 32;
    constexpr int BN = WN * NT * 32;
    constexpr int AF = (BM / 32) * 2;
    constexpr int BF = (BN / 32) * 2;
    static_assert(AF % NWAVES == 0 && BF % NWAVES == 0, "load units divide evenly among the waves");
    static_assert((BM & (BM - 1)) == 0 && BM <= kBigTile, "scale staging");
    constexpr int LA = AF / NWAVES;
    constexpr int LB = BF / NWAVES;
    constexpr int STAGE = (AF + BF) * 1024;

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const wm = wave / WN;
    int const wn = wave % WN;

    int ldsA[LA], ldsB[LB];
    auto address = [&](int n0, int t0, uint32_t(&oa)[LA], uint32_t(&ob)[LB]) {
        auto unit = [&](bool interleaved, int u, int row0, int R, uint32_t& gOff, int& lOff) {
            int const rb = u >> 1, sel = u & 1;
            if (interleaved)
            {
                int const r = lane >> 1, c = lane & 1;
                int const row = min(row0 + rb * 32 + r, R - 1);
                gOff = ((uint32_t) sel * (uint32_t) R + (uint32_t) row) * 32u + (uint32_t) c * 16u;
                lOff = (rb * 2 + sel) * 1024 + frag_offset(r, c);
            }
            else
            {
                int const r = sel * 16 + (lane >> 2), c = lane & 3;
                int const row = min(row0 + rb * 32 + r, R - 1);
                gOff = (uint32_t) row * (uint32_t) p.K + (uint32_t) c * 16u;
                lOff = (rb * 2 + (c >> 1)) * 1024 + frag_offset(r, c & 1);
            }
        };
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            unit(IL_W, q * NWAVES + wave, n0, p.N, oa[q], ldsA[q]);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            unit(IL_IN, q * NWAVES + wave, t0, p.T, ob[q], ldsB[q]);
            ldsB[q] += AF * 1024;
        }
    };
    uint32_t const stepA = IL_W ? 2u * (uint32_t) p.N * 32u : 64u;
    uint32_t const stepB = IL_IN ? 2u * (uint32_t) p.T * 32u : 64u;

    i32x4 ga[2][LA], gb[2][LB];
    auto fetch = [&](auto set, uint32_t const(&oa)[LA], uint32_t const(&ob)[LB], int kt) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            ga[S][q] = *reinterpret_cast<i32x4 const*>(p.w + oa[q] + (uint32_t) kt * stepA);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            gb[S][q] = *reinterpret_cast<i32x4 const*>(p.a + ob[q] + (uint32_t) kt * stepB);
        }
    };
    auto stash = [&](auto set, int buf) {
        constexpr int S = decltype(set)::value;
        uint8_t* base = lds + buf * STAGE;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            *reinterpret_cast<i32x4*>(base + ldsA[q]) = ga[S][q];
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            *reinterpret_cast<i32x4*>(base + ldsB[q]) = gb[S][q];
        }
    };

    AccT<EPI> acc[MT][NT];
    int const readOff = frag_offset(lane & 31, lane >> 5);
    auto multiply = [&](int buf) {
        uint8_t const* base = lds + buf * STAGE + readOff;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
        {
            i32x4 fa[MT], fb[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                fa[i] = *reinterpret_cast<i32x4 const*>(base + ((wm * MT + i) * 2 + ks) * 1024);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
            {
                fb[j] = *reinterpret_cast<i32x4 const*>(base + (AF + (wn * NT + j) * 2 + ks) * 1024);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
#pragma unroll
                for (int j = 0; j < NT; ++j)
                {
                    acc[i][j] = mma<EPI>(fa[i], fb[j], acc[i][j]);
                }
            }
        }
    };
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;

    // scale/offset vectors: sScale[parity][alpha|beta][channel]; every thread copies channel tid % BM
    int const ch = threadIdx.x & (BM - 1);
    auto scales = [&](int parity, int which) { return sScale + (parity * 2 + which) * kBigTile; };

    int n0, t0;
    origin(0, n0, t0);
    uint32_t oaC[LA], obC[LB], oaN[LA], obN[LB];
    address(n0, t0, oaC, obC);
    if constexpr (EPI != kRAW)
    {
        int const n = min(n0 + ch, p.N - 1);
        scales(0, 0)[ch] = p.alpha[n];
        scales(0, 1)[ch] = p.beta[n];
    }
    int const nk = p.K / 64; // even, >= 2
    fetch(Set0{}, oaC, obC, 0);
    fetch(Set1{}, oaC, obC, 1);
    stash(Set0{}, 0);
    __syncthreads();
    for (int j = 0; j < count; ++j)
    {
        int n1 = n0, t1 = t0;
        if (j + 1 < count)
        {
            origin(j + 1, n1, t1);
        }
        address(n1, t1, oaN, obN);
        float nextAlpha = 0.f, nextBeta = 0.f;
        if constexpr (EPI != kRAW)
        {
            int const n = min(n1 + ch, p.N - 1);
            nextAlpha = p.alpha[n];
            nextBeta = p.beta[n];
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
        {
#pragma unroll
            for (int jj = 0; jj < NT; ++jj)
            {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                {
                    acc[i][jj][v] = 0;
                }
            }
        }
        for (int kt = 0; kt + 2 < nk; kt += 2)
        {
            fetch(Set0{}, oaC, obC, kt + 2);
            multiply(0);
            stash(Set1{}, 1);
            __syncthreads();
            fetch(Set1{}, oaC, obC, kt + 3);
            multiply(1);
            stash(Set0{}, 0);
            __syncthreads();
        }
        // last two stages of this tile; the loads are the next tile's first two stages
        fetch(Set0{}, oaN, obN, 0);
        multiply(0);
        stash(Set1{}, 1);
        __syncthreads();
        fetch(Set1{}, oaN, obN, 1);
        multiply(1);
        if constexpr (EPI != kRAW)
        {
            scales((j + 1) & 1, 0)[ch] = nextAlpha;
            scales((j + 1) & 1, 1)[ch] = nextBeta;
        }
        store_tile<WM, WN, MT, NT, IL_OUT, EPI>(p, acc, n0, t0, scales(j & 1, 0), scales(j & 1, 1));
        stash(Set0{}, 0);
        __syncthreads();
        n0 = n1;
        t0 = t1;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            oaC[q] = oaN[q];
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            obC[q] = obN[q];
        }
    }
}

// The persistent run of 256 x 256 tiles with the stages brought in by direct-to-LDS loads: a ring of four LDS stage
// buffers, stage k+3 requested while stage k is multiplied, no staging registers, no LDS-write instructions and
// nothing for a wavefront to wait for before the barrier except loads issued two steps earlier.  N a multiple of 256
// and K of 256 bytes (the ring index is then the stage index modulo 4 in every tile).  One instruction fills 1 KB of
// LDS with lane i's 16 bytes at offset 16 i, so the LDS swizzle is applied on the source side: lane i fetches the
// 16 bytes that belong there.
// Both operands are 32-interleaved: a load unit is one fragment, 32 rows x 32 bytes, contiguous in memory.
template <bool IL_OUT, int EPI, typename Origin>
__device__ __forceinline__ void linear_tile_run_dma(
    LinearArgs const& p, int const count, Origin origin, uint8_t* __restrict__ lds, float* sScale)
{
    constexpr int KS = 2; // k-halves of 32 bytes per stage
    constexpr int WN = 4, MT = 4, NT = 2, NWAVES = 8;
    constexpr int AF = (kBigTile / 32) * KS;   // 1 KB fragments per operand and stage: KS k-halves of 32 bytes per row block
    constexpr int BF = (kBigTile / 32) * KS;
    constexpr int LA = AF / NWAVES;
    constexpr int LB = BF / NWAVES;
    constexpr int STAGE = (AF + BF) * 1024;
    constexpr int kLoads = LA + LB;           // direct loads per wavefront and stage
    // global stores per wavefront in a tile's epilogue: one 16-byte store per accumulator block
    constexpr int kStores = MT * NT;
    static_assert(EPI == kAFFINE || EPI == kGELU, "store count per block");

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const wm = wave / WN;
    int const wn = wave % WN;
    uint32_t const ldsBase = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) lds;
    uint32_t const scaleBase = (uint32_t) (size_t) (__attribute__((address_space(3))) float*) sScale;

    // Lane i of a unit's load supplies LDS offset 16 i of the unit.  Its address is a wave-uniform part (the unit's
    // first row, kept in scalar registers and advanced by scalar arithmetic) plus a lane part that is the same for
    // every unit, tile and stage: the loop spends no vector-ALU instruction on addresses.
    int const loadRow = lane >> 1; // row of the fragment; the half that the swizzle puts at this offset
    uint32_t const laneOff = (uint32_t) loadRow * 32u + (uint32_t) ((lane & 1) ^ ((loadRow >> 3) & 1)) * 16u;
    auto unit_base = [&](int u, int row0, int R) -> uint32_t {
        int const rb = u >> 1, sel = u & 1;
        uint32_t const b = ((uint32_t) sel * (uint32_t) R + (uint32_t) (row0 + rb * 32)) * 32u;
        return (uint32_t) __builtin_amdgcn_readfirstlane((int) b);
    };
    auto address = [&](int n0, int t0, uint32_t(&oa)[LA], uint32_t(&ob)[LB]) {
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            oa[q] = unit_base(q * NWAVES + wave, n0, p.N);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            ob[q] = unit_base(q * NWAVES + wave, t0, p.T);
        }
    };
    uint32_t const stepA = (uint32_t) KS * (uint32_t) p.N * 32u;
    uint32_t const stepB = (uint32_t) KS * (uint32_t) p.T * 32u;
    int const nk = p.K / (32 * KS); // a multiple of 4

    uint32_t oaC[LA], obC[LB], oaN[LA], obN[LB];
    // stage kt of the current tile (or stage kt - nk of the next one) into ring slot `slot`
    auto fetch = [&](int kt, int slot) {
        bool const next = kt >= nk;
        uint32_t const k = (uint32_t) (next ? kt - nk : kt);
        uint32_t const dst = ldsBase + (uint32_t) slot * STAGE;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            load_to_lds16_sbase(p.w + (uint64_t) (next ? oaN[q] : oaC[q]) + (uint64_t) k * stepA, laneOff,
                dst + (uint32_t) (q * NWAVES + wave) * 1024u);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            load_to_lds16_sbase(p.a + (uint64_t) (next ? obN[q] : obC[q]) + (uint64_t) k * stepB, laneOff,
                dst + (uint32_t) (AF + q * NWAVES + wave) * 1024u);
        }
    };

    AccT<EPI> acc[MT][NT];
    // byte offset, inside a 32-row block's 2 KB, of this lane's 16 bytes of fragment ks
    int readOff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
    {
        readOff[ks] = ks * 1024 + frag_offset(lane & 31, lane >> 5);
    }
    auto multiply = [&](int slot) {
        uint8_t const* base = lds + slot * STAGE;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
        {
            i32x4 fa[MT], fb[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                fa[i] = *reinterpret_cast<i32x4 const*>(base + (wm * MT + i) * (KS * 1024) + readOff[ks]);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
            {
                fb[j] = *reinterpret_cast<i32x4 const*>(base + AF * 1024 + (wn * NT + j) * (KS * 1024) + readOff[ks]);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
#pragma unroll
                for (int j = 0; j < NT; ++j)
                {
                    acc[i][j] = mma<EPI>(fa[i], fb[j], acc[i][j]);
                }
            }
        }
    };
    // scale / offset vectors of a tile, 256 binary32 values each: one direct load by wave 0 and one by wave 1
    auto fetch_scales = [&](int n0, int parity) {
        if (wave < 2)
        {
            float const* src = (wave == 0 ? p.alpha : p.beta) + n0 + lane * 4;
            load_to_lds16(src, scaleBase + (uint32_t) ((parity * 2 + wave) * kBigTile) * 4u);
        }
    };
    auto scales = [&](int parity, int which) { return sScale + (parity * 2 + which) * kBigTile; };
    // one step: request stage k+3, multiply stage k, make sure this wavefront's part of stage k+1 has landed, meet
    // the others.  vmcnt counts the kLoads of stages k+2 and k+3 behind it, and `extra` operations known to sit
    // between (epilogue stores), which must not be waited for.
    auto step = [&](int k, auto slotTag, auto extraTag) {
        constexpr int SLOT = decltype(slotTag)::value;
        constexpr int EXTRA = decltype(extraTag)::value;
        fetch(k + 3, (SLOT + 3) & 3);
        multiply(SLOT);
        wait_vmcnt<2 * kLoads + EXTRA>();
        __syncthreads();
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    using NoExtra = std::integral_constant<int, 0>;
    using Stores = std::integral_constant<int, kStores>;

    int n0, t0;
    origin(0, n0, t0);
    address(n0, t0, oaC, obC);
#pragma unroll
    for (int q = 0; q < LA; ++q)
    {
        oaN[q] = oaC[q];
    }
#pragma unroll
    for (int q = 0; q < LB; ++q)
    {
        obN[q] = obC[q];
    }
    fetch_scales(n0, 0);
    fetch(0, 0);
    fetch(1, 1);
    fetch(2, 2);
    wait_vmcnt<2 * kLoads>();
    __syncthreads();
    for (int j = 0; j < count; ++j)
    {
        int n1 = n0, t1 = t0;
        if (j + 1 < count)
        {
            origin(j + 1, n1, t1);
        }
        address(n1, t1, oaN, obN);
#pragma unroll
        for (int i = 0; i < MT; ++i)
        {
#pragma unroll
            for (int jj = 0; jj < NT; ++jj)
            {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                {
                    acc[i][jj][v] = 0;
                }
            }
        }
        // The first two steps after an epilogue have its stores between the stage they wait for and the newer loads.
        // The next tile's scale vectors go into the buffer the previous tile's epilogue read: only after the first
        // barrier of this tile has every wavefront left that epilogue.  (On the two wavefronts that fetch them the
        // waits below then count one operation too few, which only makes them wait for one more load.)
        if (j == 0)
        {
            step(0, S0{}, NoExtra{});
            fetch_scales(n1, (j + 1) & 1);
            step(1, S1{}, NoExtra{});
        }
        else
        {
            step(0, S0{}, Stores{});
            fetch_scales(n1, (j + 1) & 1);
            step(1, S1{}, Stores{});
        }
        step(2, S2{}, NoExtra{});
        step(3, S3{}, NoExtra{});
        for (int k = 4; k < nk; k += 4)
        {
            step(k, S0{}, NoExtra{});
            step(k + 1, S1{}, NoExtra{});
            step(k + 2, S2{}, NoExtra{});
            step(k + 3, S3{}, NoExtra{});
        }
        BlockScales blockScales;
#pragma unroll
        for (int i = 0; i < MT; ++i)
        {
#pragma unroll
            for (int jj = 0; jj < NT; ++jj)
            {
                int const cl = (wm * MT + i) * 32;
                if (jj == 0)
                {
                    blockScales = load_block_scales<EPI>(scales(j & 1, 0) + cl, scales(j & 1, 1) + cl);
                }
                store_block_scaled<IL_OUT, EPI, true, IL_OUT && (EPI == kAFFINE || EPI == kGELU)>(
                    p, acc[i][jj], n0 + cl, t0 + (wn * NT + jj) * 32, blockScales);
            }
        }
        n0 = n1;
        t0 = t1;
#pragma unroll
        for (int q = 0; q < LA; ++q)
        {
            oaC[q] = oaN[q];
        }
#pragma unroll
        for (int q = 0; q < LB; ++q)
        {
            obC[q] = obN[q];
        }
    }
    // the loads requested for a tile after the last one are still in flight: they must land before the LDS is released
    wait_vmcnt<0>();
}

// Tokens [0, 256*tokMain) are cut into 256 x 256 tiles (workgroups 0 .. mainTiles-1); what is left, which
// would otherwise be a last round of big tiles on a fraction of the CUs, is cut into 128 x 128 tiles that
// spread over all of them.
constexpr int kBig = kBigTile;
constexpr int kSmall = 128;

template <bool IL_W, bool IL_IN, bool IL_OUT, int EPI>
__global__ __launch_bounds__(512) void int8_linear_kernel(LinearArgs const p)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * 2 * (kBig / 32) * 2 * 1024];
    __shared__ __attribute__((aligned(16))) float sAlpha[kBig];
    __shared__ __attribute__((aligned(16))) float sBeta[kBig];
    if ((int) blockIdx.x < p.mainTiles)
    {
        // Each XCD (own 4 MB L2) works through a contiguous run of tile numbers.  Tiles are numbered
        // panel by panel, a panel being `panel` channel tiles wide: inside a panel the channel tile varies
        // fastest, then the token tile.  The 32 workgroups resident on an XCD then cover 32/panel token
        // tiles x panel channel tiles, and the next 32 reuse the same weights from L2.
        uint32_t const pw = (uint32_t) p.panel;
        uint32_t const perPanel = (uint32_t) p.tokMain * pw;
        uint32_t const tile = xcd_remap(blockIdx.x, (uint32_t) p.mainTiles);
        uint32_t const pan = tile / perPanel, rem = tile % perPanel;
        linear_tile<2, 4, 4, 2, IL_W, IL_IN, IL_OUT, EPI>(
            p, (int) (pan * pw + rem % pw) * kBig, (int) (rem / pw) * kBig, lds, sAlpha, sBeta);
    }
    else
    {
        uint32_t const nbm = (uint32_t) ((p.N + kSmall - 1) / kSmall);
        uint32_t const tile = blockIdx.x - (uint32_t) p.mainTiles;
        linear_tile<2, 4, 2, 1, IL_W, IL_IN, IL_OUT, EPI>(
            p, (int) (tile % nbm) * kSmall, p.tokMain * kBig + (int) (tile / nbm) * kSmall, lds, sAlpha, sBeta);
    }
}

// The same tile plan run by persistent workgroups (K % 128 == 0): workgroups 0 .. persist-1 take the
// 256 x 256 tiles b, b + persist, ... in the panel numbering, the workgroups after them one 128 x 128 tile each.
template <bool IL_W, bool IL_IN, bool IL_OUT, int EPI>
__global__ __launch_bounds__(512) void int8_linear_persistent_kernel(LinearArgs const p)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * 2 * (kBig / 32) * 2 * 1024];
    __shared__ __attribute__((aligned(16))) float sScale[2 * 2 * kBig];
    if ((int) blockIdx.x < p.persist)
    {
        uint32_t const pw = (uint32_t) p.panel;
        uint32_t const perPanel = (uint32_t) p.tokMain * pw;
        int const count = (p.mainTiles - (int) blockIdx.x + p.persist - 1) / p.persist;
        auto origin = [&](int j, int& n0, int& t0) {
            uint32_t const tile = xcd_remap(blockIdx.x + (uint32_t) j * (uint32_t) p.persist, (uint32_t) p.mainTiles);
            uint32_t const pan = tile / perPanel, rem = tile % perPanel;
            n0 = (int) (pan * pw + rem % pw) * kBig;
            t0 = (int) (rem / pw) * kBig;
        };
        linear_tile_run<2, 4, 4, 2, IL_W, IL_IN, IL_OUT, EPI>(p, count, origin, lds, sScale);
    }
    else
    {
        uint32_t const nbm = (uint32_t) ((p.N + kSmall - 1) / kSmall);
        uint32_t const tile = blockIdx.x - (uint32_t) p.persist;
        auto origin = [&](int, int& n0, int& t0) {
            n0 = (int) (tile % nbm) * kSmall;
            t0 = p.tokMain * kBig + (int) (tile / nbm) * kSmall;
        };
        linear_tile_run<2, 4, 2, 1, IL_W, IL_IN, IL_OUT, EPI>(p, 1, origin, lds, sScale);
    }
}

// A 64-channel x 64-token piece of the output for the tokens behind the large tiles, interleaved INT8 operands,
// when those tokens would make only a few 128 x 128 tiles (a long k loop on a few CUs while the others idle).
// The eight wavefronts split k, not the piece: wavefront w multiplies the k-slabs w, w + 8, ... of all four 32 x 32
// blocks.  In the interleaved layout a fragment (32 rows x 32 bytes of one k-slab) is 1 KB of consecutive memory in
// exactly the order the MFMA wants it from the lanes, so every fragment is one 16-byte load per lane straight into the
// operand registers: no LDS stage, no barrier in the loop, and no byte is fetched twice by the workgroup.  The eight
// partial accumulators meet in LDS (8 x 16 KB), four wavefronts add them up, one block each, and run the epilogue.
// Integer addition is exact, so the result is the bits of any other order.  K % 256 == 0, N % 64 == 0.
template <bool IL_OUT, int EPI>
__device__ __forceinline__ void linear_piece64(
    LinearArgs const& p, int const n0, int const t0, uint8_t* __restrict__ lds, float* sScale)
{
    static_assert(EPI == kAFFINE || EPI == kGELU, "INT8 outputs");
    constexpr int kDepth = 4; // k-slabs in flight per wavefront
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const row = lane & 31, half = lane >> 5;
    // channel and token rows of this lane in the two row blocks of each operand; tokens beyond T re-read the last one
    uint32_t offA[2], offB[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
    {
        offA[b] = (uint32_t) (n0 + 32 * b + row) * 32u + (uint32_t) half * 16u;
        offB[b] = (uint32_t) min(t0 + 32 * b + row, p.T - 1) * 32u + (uint32_t) half * 16u;
    }
    uint32_t const slabA = (uint32_t) p.N * 32u, slabB = (uint32_t) p.T * 32u;
    int const steps = p.K / 256; // k-slabs of this wavefront
    if (threadIdx.x < 64)
    {
        sScale[threadIdx.x] = p.alpha[n0 + threadIdx.x];
        sScale[kBigTile + threadIdx.x] = p.beta[n0 + threadIdx.x];
    }
    i32x4 fa[kDepth][2], fb[kDepth][2];
    auto fetch = [&](int slot, int step) {
        uint32_t const ks = (uint32_t) (min(step, steps - 1) * 8 + wave);
#pragma unroll
        for (int b = 0; b < 2; ++b)
        {
            fa[slot][b] = *reinterpret_cast<i32x4 const*>(p.w + (size_t) ks * slabA + offA[b]);
            fb[slot][b] = *reinterpret_cast<i32x4 const*>(p.a + (size_t) ks * slabB + offB[b]);
        }
    };
    AccT<EPI> acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
    {
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                acc[i][j][v] = 0;
            }
        }
    }
#pragma unroll
    for (int d = 0; d < kDepth; ++d)
    {
        fetch(d, d);
    }
    for (int s0 = 0; s0 < steps; s0 += kDepth)
    {
#pragma unroll
        for (int d = 0; d < kDepth; ++d)
        {
            if (s0 + d < steps)
            {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                {
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                    {
                        acc[i][j] = mma<EPI>(fa[d][i], fb[d][j], acc[i][j]);
                    }
                }
                fetch(d, s0 + d + kDepth); // loads behind the last slab re-read it and are never used
            }
        }
    }
    // partial accumulators: [wavefront][block][four registers][lane], 16 bytes per lane and access
    i32x4* const part = reinterpret_cast<i32x4*>(lds);
#pragma unroll
    for (int i = 0; i < 2; ++i)
    {
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                part[(((wave * 4) + (i * 2 + j)) * 4 + q) * 64 + lane]
                    = i32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
        }
    }
    __syncthreads();
    if (wave < 4)
    {
        AccT<EPI> sum;
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            i32x4 t = part[((wave) * 4 + q) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 8; ++w)
            {
                t += part[(((w * 4) + wave) * 4 + q) * 64 + lane];
            }
            sum[4 * q] = t[0];
            sum[4 * q + 1] = t[1];
            sum[4 * q + 2] = t[2];
            sum[4 * q + 3] = t[3];
        }
        int const cb = (wave >> 1) * 32, tb = (wave & 1) * 32;
        store_block<IL_OUT, EPI>(p, sum, n0 + cb, t0 + tb, sScale + cb, sScale + kBigTile + cb);
    }
}

// The scales and offsets of the four channels that a lane of a piece stores: requested with the operands, since a trip to
// memory behind the sums is as long as everything else behind the operands' (see linear_piece_kernel).
struct QuadScales
{
    f32x4 al, be;
};

template <int EPI>
__device__ __forceinline__ QuadScales load_quad_scales(LinearArgs const& p, int const c)
{
    QuadScales s{};
    if constexpr (EPI != kRAW && EPI != kF16_RAW)
    {
        int const at = min(c, p.N - 4);
        s.al = *reinterpret_cast<f32x4 const*>(p.alpha + at);
        s.be = *reinterpret_cast<f32x4 const*>(p.beta + at);
    }
    return s;
}

// The results of one lane for four consecutive channels (c .. c+3) of one token, packed and stored.
template <bool IL_OUT, int EPI, typename Acc4>
__device__ __forceinline__ void store_quad(
    LinearArgs const& p, Acc4 const& acc, QuadScales const& sc, int const c, int const t, int const part)
{
    if constexpr (EPI == kRAW || EPI == kF16_RAW)
    {
        if (t < p.T)
        {
            static_cast<Acc4*>(p.out)[(((size_t) part * p.T + t) * p.N + c) >> 2] = acc;
        }
        return;
    }
    f32x4 const& al = sc.al;
    f32x4 const& be = sc.be;
    if (t >= p.T)
    {
        return;
    }
    if constexpr (EPI >= kF16_AFFINE)
    {
        f16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            float const y = fmaf(acc[e], al[e], be[e]);
            h[e] = (f16) (EPI == kF16_GELU ? gelu_erf(y) : y);
        }
        *reinterpret_cast<f16x4*>(static_cast<f16*>(p.out) + (size_t) t * p.N + c) = h;
    }
    else
    {
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            if constexpr (EPI == kGELU)
            {
                float const y = fmaf((float) acc[e], al[e], be[e]);
                w = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(gelu_erf(y), p.qOut, 128.f), e, w);
            }
            else
            {
                w = __builtin_amdgcn_cvt_pk_u8_f32(fmaf((float) acc[e], al[e], be[e] + 128.f), e, w);
            }
        }
        size_t const o = IL_OUT ? ((size_t) (c >> 5) * p.T + t) * 32 + (c & 31) : (size_t) t * p.N + c;
        *reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.out) + o) = w ^ 0x80808080u;
    }
}

// The last `rest` stages of a ring, MOST + 1 of them at most: f is called for each with the number of stages requested
// behind it as a constant (what its wait may leave in flight).
template <int MOST, typename F>
__device__ __forceinline__ void for_each_behind(int const rest, F&& f)
{
    if (MOST < rest)
    {
        f(std::integral_constant<int, MOST>{});
    }
    if constexpr (MOST > 0)
    {
        for_each_behind<MOST - 1>(rest, f);
    }
}

// Whether a tile's scale vectors come at its end, into a slot of the ring, since a place of their own would cost the CU its
// second workgroup.
constexpr bool scales_late(int ringBytes)
{
    constexpr int kHalfOfLds = 80 * 1024;
    return ringBytes <= kHalfOfLds && ringBytes + 2 * kBigTile * 4 > kHalfOfLds;
}

// One tile of BM = WM*MT*32 channels x BN = WN*NT*32 tokens with the stages brought in by direct-to-LDS loads.  Rows behind
// the last one are read as the last one (their results are not stored), so any T and N are taken.  Operands both
// interleaved (IL) or both linear.
//
// Stages.  KS k-halves of 32 bytes.  Interleaved operands arrive in whole lines whatever the stage is.  Of a linear operand
// a row's share of a stage is 32 KS bytes: with 64 of them every line crosses from the L2 to the CU twice, half of it for
// nothing, so linear rows come in stages of 128 bytes (KS = 4; K a multiple of that, otherwise KS = 2).  A load unit is
// 8 rows x 128 bytes, and in LDS the 16-byte chunk c of row r sits at chunk c ^ (r / 2) % 8 (KS = 2: 16 rows x 64 bytes,
// chunk c ^ r / 4): 16 rows x one chunk, a quarter of a fragment read, then touch every bank once.
//
// Schedule.  All RING slots are requested ahead; a stage's slot is requested again as soon as everybody has read it.  What
// a wavefront does between two matrix instructions is written out: the fragments of the next k-half are read while
// this one's are multiplied, across the barrier too, and the loads of a stage are spread over the k-halves of the one
// before, for a burst of them stalls the wavefront that issues it while the CU's one path to the L2 takes them in.
//
// What it is bound by: with every CU busy, by the power the chip may draw (768 channels, 7765 tokens x 3072 -> 768: 43 us on
// normal operands, 35 us on zeros; 31 us with either the loads or the matrix instructions left out).
// 7765 tokens, FP16, QKV / projection / feed-forward 1 / 2 of 768 channels, graph replays, the best plan of each, us:
//   stages of 64 bytes, fragments read behind the barrier     39.8 / 16.9 / 52.4 / 50.4
//   the same in tiles of 192 channels or tokens too           37.3 / 16.6 / 49.1 / 49.2
//   stages of 128 bytes                                       39.8 / 16.0 / 47.8 / 44.5
//   fragments read ahead                                      38.7 / 15.8 / 46.5 / 43.0
//   loads spread out, order kept                              36.0 / 14.8 / 45.1 / 39.3
//   rows stored whole, through the L2 (see the end)           32.6 / 12.5 / 41.2 / 35.5
template <bool IL, bool IL_OUT, int EPI, int WM, int WN, int MT, int NT, int RING, int KS = 2>
__device__ __forceinline__ void linear_tile_dma(
    LinearArgs const& p, int const n0, int const t0, uint8_t* __restrict__ lds)
{
    constexpr int NWAVES = WM * WN;
    constexpr int BM = WM * MT * 32;
    constexpr int BN = WN * NT * 32;
    constexpr int AF = (BM / 32) * KS;
    constexpr int BF = (BN / 32) * KS;
    constexpr int kLoads = (AF + BF + NWAVES - 1) / NWAVES;
    constexpr int STAGE = (AF + BF) * 1024;
    static_assert(BM <= kBigTile && STAGE >= 2 * kBigTile * 4, "scale vectors");

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const wm = wave / WN;
    int const wn = wave % WN;
    uint32_t const ldsBase = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) lds;

    auto unit_offset = [&](int u, int row0, int R) -> uint32_t {
        int const rb = u / KS, sel = u % KS;
        if constexpr (IL)
        {
            int const r = lane >> 1;
            uint32_t const half = (uint32_t) ((lane & 1) ^ ((r >> 3) & 1));
            return ((uint32_t) sel * (uint32_t) R + (uint32_t) min(row0 + rb * 32 + r, R - 1)) * 32u + half * 16u;
        }
        else
        {
            int const rr = lane / (2 * KS), r = sel * (32 / KS) + rr;
            uint32_t const chunk = (uint32_t) ((lane & (2 * KS - 1)) ^ (KS == 2 ? rr >> 2 : (r >> 1) & 7));
            return (uint32_t) min(row0 + rb * 32 + r, R - 1) * (uint32_t) p.K + chunk * 16u;
        }
    };
    // Units 0 .. AF-1 are the weights', the ones behind them the tokens', dealt to the wavefronts in turn.  Where they do
    // not come out even, the wavefronts without a last unit fetch the one before it again, to the same place: every
    // wavefront then has the same number of loads in flight, which is what the waits below count.
    uint32_t off[kLoads], step[kLoads], dstOff[kLoads];
    int8_t const* src[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
    {
        int const own = q * NWAVES + wave;
        int const u = (q + 1) * NWAVES <= AF + BF || own < AF + BF ? own : own - NWAVES;
        bool const weights = (q + 1) * NWAVES <= AF || (q * NWAVES < AF && u < AF);
        off[q] = weights ? unit_offset(u, n0, p.N) : unit_offset(u - AF, t0, p.T);
        src[q] = weights ? p.w : p.a;
        step[q] = KS * 32u * (IL ? (uint32_t) (weights ? p.N : p.T) : 1u);
        dstOff[q] = (uint32_t) u * 1024u;
    }
    int const nk = p.K / (32 * KS);
    auto fetch = [&](int kt, int slot) {
        uint32_t const dst = ldsBase + (uint32_t) slot * STAGE;
#pragma unroll
        for (int q = 0; q < kLoads; ++q)
        {
            load_to_lds16_sbase(src[q] + (uint64_t) kt * step[q], off[q], dst + dstOff[q]);
        }
    };
    AccT<EPI> acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
    {
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                acc[i][j][v] = 0;
            }
        }
    }
    int readOff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
    {
        if constexpr (IL)
        {
            readOff[ks] = ks * 1024 + frag_offset(lane & 31, lane >> 5);
        }
        else
        {
            int const fr = lane & 31, rr = fr & 15, chunk = ks * 2 + (lane >> 5);
            readOff[ks] = KS == 2 ? (fr >> 4) * 1024 + rr * 64 + ((chunk ^ (rr >> 2)) << 4)
                                  : fr * 128 + ((chunk ^ ((fr >> 1) & 7)) << 4);
        }
    }
    i32x4 fa[2][MT], fb[2][NT];
    // fragment r of k-half ks of the stage in `slot`, in the order in which the matrix instructions ask for them
    auto read_fragment = [&](auto setTag, int slot, int ks, int r) {
        constexpr int S = decltype(setTag)::value;
        uint8_t const* base = lds + slot * STAGE + readOff[ks];
        if (r == 0 || r > NT)
        {
            int const i = r == 0 ? 0 : r - NT;
            fa[S][i] = *reinterpret_cast<i32x4 const*>(base + (wm * MT + i) * (KS * 1024));
        }
        else
        {
            fb[S][r - 1] = *reinterpret_cast<i32x4 const*>(base + AF * 1024 + (wn * NT + r - 1) * (KS * 1024));
        }
    };
    // One k-half: the matrix instructions on fragment set S, and between them the reads of the next k-half's fragments
    // (ks of `slot`, into the other set) and this k-half's share of the loads of stage kt.  The order is kept as it stands.
    auto phase = [&](auto setTag, auto readTag, int slot, int ks, auto loadTag, int kt, int ktSlot) {
        constexpr int S = decltype(setTag)::value;
        constexpr bool READ = decltype(readTag)::value;
        constexpr int PART = decltype(loadTag)::value; // -1: no loads
        constexpr int M = MT * NT, R = MT + NT, kReadsAtOnce = (2 * R + M - 1) / M;
        // two stages in the ring: the loads of a stage have to be on their way early in the one before it
        constexpr int P = RING == 2 ? 2 : KS;
        constexpr int L0 = PART < 0 || PART >= P ? 0 : PART * kLoads / P, L1 = PART < 0 || PART >= P ? 0 : (PART + 1) * kLoads / P;
        uint32_t const dst = ldsBase + (uint32_t) ktSlot * STAGE;
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            acc[m / NT][m % NT] = mma<EPI>(fa[S][m / NT], fb[S][m % NT], acc[m / NT][m % NT]);
            if constexpr (READ)
            {
#pragma unroll
                for (int r = m * kReadsAtOnce; r < (m + 1) * kReadsAtOnce && r < R; ++r)
                {
                    read_fragment(std::integral_constant<int, 1 - S>{}, slot, ks, r);
                }
            }
#pragma unroll
            for (int q = L0 + m * (L1 - L0) / M; q < L0 + (m + 1) * (L1 - L0) / M; ++q)
            {
                load_to_lds16_sbase(src[q] + (uint64_t) kt * step[q], off[q], dst + dstOff[q]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    using Yes = std::true_type;
    using No = std::false_type;
    using NoLoads = std::integral_constant<int, -1>;
    constexpr bool kLate = scales_late(RING * STAGE);
    auto fetch_scales = [&](int at) {
        if (wave < 2 && lane < BM / 4)
        {
            float const* from = (wave == 0 ? p.alpha : p.beta) + min(n0 + lane * 4, p.N - 4);
            load_to_lds16(from, ldsBase + (uint32_t) (at + wave * kBigTile * 4));
        }
    };
    if constexpr (!kLate)
    {
        fetch_scales(RING * STAGE); // requested first, so the wait for stage 0 covers them
    }
#pragma unroll
    for (int s = 0; s < RING; ++s)
    {
        if (s < nk)
        {
            fetch(s, s);
        }
    }
    if (nk >= RING)
    {
        wait_vmcnt<(RING - 1) * kLoads>();
    }
    else
    {
        wait_vmcnt<0>();
    }
    __syncthreads();
    int slot = 0, k = 0;
#pragma unroll
    for (int r = 0; r < MT + NT; ++r)
    {
        read_fragment(Even{}, 0, 0, r);
    }
    // the k-halves of stage k but its last; `loads`: with the rest of the loads of stage k + RING - 1, which go where
    // stage k - 1 was
    auto first_halves = [&](auto loads) {
        constexpr bool LOADS = decltype(loads)::value;
        int const before = slot == 0 ? RING - 1 : slot - 1;
        phase(Even{}, Yes{}, slot, 1, std::integral_constant<int, LOADS ? 1 : -1>{}, k + RING - 1, before);
        if constexpr (KS == 4)
        {
            phase(Odd{}, Yes{}, slot, 2, std::integral_constant<int, LOADS ? 2 : -1>{}, k + RING - 1, before);
            phase(Even{}, Yes{}, slot, 3, std::integral_constant<int, LOADS ? 3 : -1>{}, k + RING - 1, before);
        }
    };
    // stage k, with stage k + 1 landed before its last k-half; BEHIND: stages that may still be on their way then
    auto stage = [&](auto restTag, auto behindTag, auto nextTag) {
        first_halves(restTag);
        wait_vmcnt<decltype(behindTag)::value * kLoads>(); // this wavefront's part of stage k + 1 has landed
        __syncthreads();                                   // everybody's has, and everybody has read stage k
        int const own = slot;
        slot = slot == RING - 1 ? 0 : slot + 1;
        phase(Odd{}, Yes{}, slot, 0, std::integral_constant<int, decltype(nextTag)::value ? 0 : -1>{}, k + RING, own);
        ++k;
    };
    using Behind = std::integral_constant<int, RING - 2>;
    if (k + RING < nk)
    {
        stage(No{}, Behind{}, Yes{});
        while (k + RING < nk)
        {
            stage(Yes{}, Behind{}, Yes{});
        }
        stage(Yes{}, Behind{}, No{});
    }
    for_each_behind<RING - 2>(nk - 1 - k, [&](auto behind) { stage(No{}, behind, No{}); });
    int const scalesAt = kLate ? (slot == 0 ? RING - 1 : slot - 1) * STAGE : RING * STAGE;
    if constexpr (kLate)
    {
        fetch_scales(scalesAt); // a slot that no further stage needs
    }
    first_halves(No{});
    phase(Odd{}, No{}, 0, 0, NoLoads{}, 0, 0);
    constexpr int kRow = MT * 64 + 16; // bytes; 16 of padding spread the rows over the banks
    constexpr bool kStaged = EPI >= kF16_AFFINE && NWAVES * 32 * kRow <= STAGE;
    if constexpr (kLate || kStaged)
    {
        wait_vmcnt<0>();
        __syncthreads(); // the scales have come, and nobody reads the last stage any more
    }
    float const* const sScale = reinterpret_cast<float const*>(lds + scalesAt);

    // FP16 rows leave through LDS, 32 tokens of the wavefront's channels at a time, so that a store writes whole lines, and can
    // write through the L2: what is left in it at the kernel's end is written back while nothing else runs (up to 32 MB;
    // stores of 16-byte pieces need the L2 to put them together, and cost 5 to 9 of the 44 us of feed-forward 1).
    if constexpr (kStaged)
    {
        uint8_t* const own = lds + slot * STAGE + wave * (32 * kRow);
        int const nw = n0 + wm * MT * 32;
        BlockScales sc[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
        {
            sc[i] = load_block_scales<EPI>(sScale + (wm * MT + i) * 32, sScale + kBigTile + (wm * MT + i) * 32);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                u32x4 first, second;
                pack_half_block<EPI>(acc[i][j], sc[i], first, second);
                u32x4* dst = reinterpret_cast<u32x4*>(own + (lane & 31) * kRow + i * 64 + (lane >> 5) * 32);
                dst[0] = first;
                dst[1] = second;
            }
            constexpr int kChunks = MT * 4; // 16-byte pieces of a row
            int const tb = t0 + (wn * NT + j) * 32;
#pragma unroll
            for (int q = 0; q < kChunks / 2; ++q)
            {
                int const c = q * 64 + lane, r = c / kChunks, ch = c % kChunks;
                u32x4 const v = *reinterpret_cast<u32x4 const*>(own + r * kRow + ch * 16);
                if (tb + r < p.T && nw + ch * 8 < p.N)
                {
                    store_out<true>(static_cast<f16*>(p.out) + (size_t) (tb + r) * p.N + nw + ch * 8, v);
                }
            }
        }
        return;
    }
    bool const full = t0 + BN <= p.T; // uniform
#pragma unroll
    for (int i = 0; i < MT; ++i)
    {
        int const cl = (wm * MT + i) * 32;
        if (n0 + cl >= p.N)
        {
            break;
        }
        BlockScales const sc = load_block_scales<EPI>(sScale + cl, sScale + kBigTile + cl);
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
            int const tb = t0 + (wn * NT + j) * 32;
            constexpr bool through = IL_OUT && (EPI == kAFFINE || EPI == kGELU);
            if (full)
            {
                store_block_scaled<IL_OUT, EPI, true, through>(p, acc[i][j], n0 + cl, tb, sc);
            }
            else
            {
                store_block_scaled<IL_OUT, EPI, false, through>(p, acc[i][j], n0 + cl, tb, sc);
            }
        }
    }
}

// The persistent tile plan with direct-to-LDS loads for the 256 x 256 tiles.
template <bool IL_OUT, int EPI>
__global__ __launch_bounds__(512) void int8_linear_dma_kernel(LinearArgs const p)
{
    __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * 2 * (kBig / 32) * 2 * 1024];
    __shared__ __attribute__((aligned(16))) float sScale[2 * 2 * kBig];
    if ((int) blockIdx.x < p.persist)
    {
        uint32_t const pw = (uint32_t) p.panel;
        uint32_t const perPanel = (uint32_t) p.tokMain * pw;
        int const count = (p.mainTiles - (int) blockIdx.x + p.persist - 1) / p.persist;
        auto origin = [&](int j, int& n0, int& t0) {
            uint32_t const tile = xcd_remap(blockIdx.x + (uint32_t) j * (uint32_t) p.persist, (uint32_t) p.mainTiles);
            uint32_t const pan = tile / perPanel, rem = tile % perPanel;
            n0 = (int) (pan * pw + rem % pw) * kBig;
            t0 = (int) (rem / pw) * kBig;
        };
        linear_tile_run_dma<IL_OUT, EPI>(p, count, origin, lds, sScale);
    }
    else
    {
        uint32_t const tile = blockIdx.x - (uint32_t) p.persist;
        if (p.pieces)
        {
            uint32_t const nbm = (uint32_t) p.N / 64u;
            linear_piece64<IL_OUT, EPI>(p, (int) (tile % nbm) * 64, p.tokMain * kBig + (int) (tile / nbm) * 64, lds, sScale);
            return;
        }
        uint32_t const nbm = (uint32_t) ((p.N + kSmall - 1) / kSmall);
        linear_tile_dma<true, IL_OUT, EPI, 2, 4, 2, 1, 4>(p, (int) (tile % nbm) * kSmall,
            p.tokMain * kBig + (int) (tile / nbm) * kSmall, lds);
    }
}

// The workgroups behind the tiles of a launch: each wavefront requests 4 KB of the weights in p.prefetch, on the XCD
// whose L2 the launch that uses them will look in (ids are dealt to the 8 XCDs in turn), waits for them and drops them.
constexpr int kPrefetchLoads = 4; // per wavefront, 1 KB each

__device__ __forceinline__ void prefetch_weights(LinearArgs const& p, uint32_t id, uint32_t waves)
{
    int const lane = threadIdx.x & 63;
    uint32_t const xcd = id & 7u, rank = (id - (uint32_t) p.mainTiles) >> 3;
    uint32_t const perXcd = p.prefetch.units / 8u;
    uint32_t const first = (rank * waves + (threadIdx.x >> 6)) * kPrefetchLoads;
    if (first >= perXcd)
    {
        return;
    }
    i32x4 v[kPrefetchLoads];
#pragma unroll
    for (int i = 0; i < kPrefetchLoads; ++i)
    {
        uint32_t const u = min(first + (uint32_t) i, perXcd - 1u);
        uint64_t const unit = (uint64_t) u * 8u + xcd;
        v[i] = *reinterpret_cast<i32x4 const*>(static_cast<uint8_t const*>(p.prefetch.data) + unit * 1024u + (uint32_t) lane * 16u);
    }
#pragma unroll
    for (int i = 0; i < kPrefetchLoads; ++i)
    {
        asm volatile("" ::"v"(v[i]));
    }
}

template <bool IL, bool IL_OUT, int EPI, int WM, int WN, int MT, int NT, int RING, int PER_SIMD, int KS = 2>
__global__ __launch_bounds__(WM* WN * 64, PER_SIMD) void linear_tile_kernel(uint64_t const w, uint64_t const a, int const K, int const T,
    int const N, int const mainTiles, uint32_t const panel, uint32_t const panelMul, uint32_t const panelShifts,
    uint32_t const perPanel, uint32_t const perPanelMul, uint32_t const perPanelShifts, LinearArgs const rest)
{
    LinearArgs p = rest; // what a workgroup needs before its first request comes preloaded instead
    p.w = global_ptr<int8_t const>(w);
    p.a = global_ptr<int8_t const>(a);
    p.K = K;
    p.T = T;
    p.N = N;
    p.mainTiles = mainTiles;
    p.panelDiv = {panel, panelMul, panelShifts};
    p.perPanelDiv = {perPanel, perPanelMul, perPanelShifts};
    constexpr int kRing = RING * (WM * MT + WN * NT) * KS * 1024;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kRing + (scales_late(kRing) ? 0 : 2 * kBigTile * 4)];
    if constexpr (IL)
    {
        if ((int) blockIdx.x >= p.mainTiles)
        {
            prefetch_weights(p, blockIdx.x, WM * WN);
            return;
        }
    }
    // panel numbering as for the large tiles (see int8_linear_kernel)
    uint32_t const tile = xcd_remap(blockIdx.x, (uint32_t) p.mainTiles);
    uint32_t const pan = tile / p.perPanelDiv, rem = tile - pan * p.perPanelDiv.d;
    uint32_t const tokenTile = rem / p.panelDiv, inPanel = rem - tokenTile * p.panelDiv.d;
    linear_tile_dma<IL, IL_OUT, EPI, WM, WN, MT, NT, RING, KS>(
        p, (int) (pan * p.panelDiv.d + inPanel) * (WM * MT * 32), (int) tokenTile * (WN * NT * 32), lds);
}

// The arguments of the piece kernels: what a wavefront needs for its requests comes preloaded, as the leading scalars of the
// argument list.  Left to their first uses in the struct, they were up to five trips of scalar loads of 0.1 to 0.2 us, one
// behind the other, and the divisions that took a piece's number apart (it is a grid of three extents now) as much again: a
// pass of one request, INT8, 24 layers of 1024 channels, 632 -> 590 us; FP16, 12 layers of 768, 386 -> 379 us.
__device__ __forceinline__ LinearArgs piece_args(uint64_t w, uint64_t a, uint64_t alpha, uint64_t beta, int K,
    int T, int N, int parts, int perPart, LinearArgs const& rest)
{
    LinearArgs p = rest;
    p.w = global_ptr<int8_t const>(w);
    p.a = global_ptr<int8_t const>(a);
    p.alpha = global_ptr<float const>(alpha);
    p.beta = global_ptr<float const>(beta);
    p.K = K;
    p.T = T;
    p.N = N;
    p.parts = parts;
    p.perPart = perPart;
    return p;
}

// A piece of CB x TB blocks of 32 channels x 32 tokens by one workgroup whose eight wavefronts split k, for launches
// with too few tokens to fill the chip with tiles that walk k one stage after the other: bound by the latency of one trip
// to memory and by what one CU can read (64 bytes a clock), not by the matrix cores.  Interleaved operands, as in
// linear_piece64: a fragment is 1 KB of consecutive memory and goes straight into the operand registers, DEPTH k-slabs
// in flight per wavefront, no LDS stage and no barrier before the eight partial accumulators meet in LDS; every wavefront
// then adds up and stores quarters of blocks.  40 tokens x 4096 -> 1024: 19.1 us in 128 x 128 tiles, 4.7 us in 32 x 32
// pieces; K any multiple of 32 bytes, N and T any.  The grid is (channel pieces, token pieces, parts and what prefetches):
// neither a division nor a trip for an argument stands between a wavefront's start and its first request.
template <bool IL_OUT, int EPI, int CB, int TB, int DEPTH, int PER_SIMD>
__global__ __launch_bounds__(512, PER_SIMD) void linear_piece_kernel(uint64_t const w, uint64_t const a, uint64_t const alpha,
    uint64_t const beta, int const K, int const T, int const N, int const parts, int const perPart, LinearArgs const rest)
{
    constexpr int NW = 8;
    LinearArgs const p = piece_args(w, a, alpha, beta, K, T, N, parts, perPart, rest);
    __shared__ __attribute__((aligned(16))) uint8_t lds[NW * CB * TB * 4096];
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const row = lane & 31, half = lane >> 5;
    if ((int) blockIdx.z >= p.parts)
    {
        uint32_t const nbm = (uint32_t) ceil_div(p.N, 32 * CB);
        prefetch_weights(p, (blockIdx.z * (uint32_t) p.tokMain + blockIdx.y) * nbm + blockIdx.x, NW);
        return;
    }
    int const n0 = (int) blockIdx.x * (32 * CB), t0 = (int) blockIdx.y * (32 * TB), kpart = (int) blockIdx.z;
    uint32_t offA[CB], offB[TB];
#pragma unroll
    for (int b = 0; b < CB; ++b)
    {
        uint32_t const r = (uint32_t) min(n0 + 32 * b + row, p.N - 1);
        offA[b] = r * 32u + (uint32_t) half * 16u;
    }
#pragma unroll
    for (int b = 0; b < TB; ++b)
    {
        uint32_t const r = (uint32_t) min(t0 + 32 * b + row, p.T - 1);
        offB[b] = r * 32u + (uint32_t) half * 16u;
    }
    uint32_t const slabA = (uint32_t) p.N * 32u, slabB = (uint32_t) p.T * 32u;
    static_assert(CB * TB * 4 <= NW, "a quarter of a block for each wavefront at most");
    QuadScales const scales = load_quad_scales<EPI>(p, n0 + (wave / (4 * TB)) * 32 + 8 * (wave & 3) + 4 * half);
    // this workgroup's k-slabs, and the consecutive ones of this wavefront
    int const slabs = min(p.K / 32, (kpart + 1) * p.perPart);
    int const per = ceil_div(p.perPart, NW), first = kpart * p.perPart + wave * per;
    int const steps = max(0, min(per, slabs - first));
    i32x4 fa[DEPTH][CB], fb[DEPTH][TB];
    auto fetch = [&](int slot, int step) {
        uint32_t const ks = (uint32_t) min(first + step, slabs - 1);
#pragma unroll
        for (int b = 0; b < CB; ++b)
        {
            fa[slot][b] = *reinterpret_cast<i32x4 const*>(p.w + (size_t) ks * slabA + offA[b]);
        }
#pragma unroll
        for (int b = 0; b < TB; ++b)
        {
            fb[slot][b] = *reinterpret_cast<i32x4 const*>(p.a + (size_t) ks * slabB + offB[b]);
        }
    };
    AccT<EPI> acc[CB][TB];
#pragma unroll
    for (int i = 0; i < CB; ++i)
    {
#pragma unroll
        for (int j = 0; j < TB; ++j)
        {
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                acc[i][j][v] = 0;
            }
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
    {
        fetch(d, d);
    }
    for (int s0 = 0; s0 < steps; s0 += DEPTH)
    {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
        {
            if (s0 + d < steps)
            {
#pragma unroll
                for (int i = 0; i < CB; ++i)
                {
#pragma unroll
                    for (int j = 0; j < TB; ++j)
                    {
                        acc[i][j] = mma<EPI>(fa[d][i], fb[d][j], acc[i][j]);
                    }
                }
                if (s0 + d + DEPTH < steps)
                {
                    fetch(d, s0 + d + DEPTH);
                }
            }
        }
    }
    using Acc4 = std::conditional_t<(EPI >= kF16_AFFINE), f32x4, i32x4>;
    // partial accumulators: [wavefront][block][four registers][lane], 16 bytes per lane and access
    Acc4* const part = reinterpret_cast<Acc4*>(lds);
#pragma unroll
    for (int i = 0; i < CB; ++i)
    {
#pragma unroll
        for (int j = 0; j < TB; ++j)
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                part[((wave * CB * TB + (i * TB + j)) * 4 + q) * 64 + lane]
                    = Acc4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
        }
    }
    __syncthreads();
    if (int const u = wave; u < CB * TB * 4)
    {
        Acc4 t = part[u * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w)
        {
            t += part[(w * CB * TB * 4 + u) * 64 + lane];
        }
        int const b = u >> 2, q = u & 3, cb = n0 + (b / TB) * 32, tb = t0 + (b % TB) * 32;
        if (cb < p.N)
        {
            store_quad<IL_OUT, EPI>(p, t, scales, cb + 8 * q + 4 * half, tb + row, kpart);
        }
    }
}

// The same pieces for linear operands, where the 32 rows of a fragment are 32 separate lines (read straight into
// registers, 40 tokens x 3072 -> 768 in FP16 take 16 us): every wavefront brings its own k range in through a ring of
// direct-to-LDS loads of its own (units, swizzle and fragment reads of the linear tiles), so there is still no barrier before
// the partial accumulators meet.  K a multiple of 32 KS bytes.
//
// KS = 4, rows in whole lines of 128 bytes, wherever K comes in those: what bounds a piece is what its CU can read from the L2,
// and that is 65 bytes a clock in whole lines and 31 in halves of them (168 workgroups of 96 rows x 6144 bytes, loads alone:
// 5.8 against 9.9 us).  The stages are twice as long for it, so four wavefronts share k instead of eight, with the LDS of the
// other four for their rings: 448 tokens x 3072 -> 768, FP16, pieces of 32 x 64: 11.5 -> 9.2 us by itself.  Pieces of 32 x 32
// leave room for two workgroups on a CU; rings of four stages, or eight wavefronts with rings of two, are slower.
template <bool IL_OUT, int EPI, int CB, int TB, int RING, int NW, int KS, int PER_SIMD>
__global__ __launch_bounds__(NW * 64, PER_SIMD) void linear_piece_dma_kernel(uint64_t const w, uint64_t const a, uint64_t const alpha,
    uint64_t const beta, int const K, int const T, int const N, int const parts, int const perPart, LinearArgs const rest)
{
    LinearArgs const p = piece_args(w, a, alpha, beta, K, T, N, parts, perPart, rest);
    constexpr int kLoads = (CB + TB) * KS;
    constexpr int STAGE = kLoads * 1024;
    constexpr int kUnits = CB * TB * 4; // quarters of blocks: what a wavefront adds up and stores at a time
    constexpr int kOwn = kUnits / NW > 1 ? kUnits / NW : 1;
    static_assert(kUnits % NW == 0 || kUnits < NW, "the same number of them for each wavefront that has any");
    static_assert(CB * TB * 4096 <= RING * STAGE, "the partial accumulators go where the wavefront's stages were");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NW * RING * STAGE];
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const row = lane & 31, half = lane >> 5;
    int const n0 = (int) blockIdx.x * (32 * CB), t0 = (int) blockIdx.y * (32 * TB), kpart = (int) blockIdx.z;
    uint8_t* const own = lds + wave * (RING * STAGE);
    uint32_t const ownBase = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) own;
    uint32_t off[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u)
    {
        int const r = u * (32 / KS) + lane / (2 * KS); // row of the stage: weights, then tokens
        int const g = u < KS * CB ? min(n0 + r, p.N - 1) : min(t0 + r - 32 * CB, p.T - 1);
        uint32_t const chunk = (uint32_t) ((lane & (2 * KS - 1)) ^ (KS == 2 ? (r >> 2) & 3 : (r >> 1) & 7));
        off[u] = (uint32_t) g * (uint32_t) p.K + chunk * 16u;
    }
    QuadScales scales[kOwn];
#pragma unroll
    for (int v = 0; v < kOwn; ++v)
    {
        int const u = v * NW + wave;
        scales[v] = load_quad_scales<EPI>(p, n0 + (u / (4 * TB)) * 32 + 8 * (u & 3) + 4 * half);
    }
    int const nk = min(p.K / (32 * KS), (kpart + 1) * p.perPart); // stages up to the end of this workgroup's
    int const per = ceil_div(p.perPart, NW), first = kpart * p.perPart + wave * per;
    int const steps = max(0, min(per, nk - first));
    auto fetch = [&](int step, int slot) {
        uint64_t const k = (uint64_t) (first + step) * (32u * KS);
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
        {
            load_to_lds16_sbase((u < KS * CB ? p.w : p.a) + k, off[u], ownBase + (uint32_t) (slot * STAGE + u * 1024));
        }
    };
    AccT<EPI> acc[CB][TB];
#pragma unroll
    for (int i = 0; i < CB; ++i)
    {
#pragma unroll
        for (int j = 0; j < TB; ++j)
        {
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                acc[i][j][v] = 0;
            }
        }
    }
    auto multiply = [&](int slot) {
        uint8_t const* base = own + slot * STAGE;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
        {
            int const chunk = ks * 2 + half, fr = row & 15;
            int const o = KS == 2 ? (row >> 4) * 1024 + fr * 64 + ((chunk ^ (fr >> 2)) << 4)
                                  : row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4);
            i32x4 fa[CB], fb[TB];
#pragma unroll
            for (int i = 0; i < CB; ++i)
            {
                fa[i] = *reinterpret_cast<i32x4 const*>(base + i * (KS * 1024) + o);
            }
#pragma unroll
            for (int j = 0; j < TB; ++j)
            {
                fb[j] = *reinterpret_cast<i32x4 const*>(base + (CB + j) * (KS * 1024) + o);
            }
#pragma unroll
            for (int i = 0; i < CB; ++i)
            {
#pragma unroll
                for (int j = 0; j < TB; ++j)
                {
                    acc[i][j] = mma<EPI>(fa[i], fb[j], acc[i][j]);
                }
            }
        }
    };
#pragma unroll
    for (int s = 0; s < RING - 1; ++s)
    {
        if (s < steps)
        {
            fetch(s, s);
        }
    }
    int slot = 0, k = 0;
    for (; k + RING - 1 < steps; ++k)
    {
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): stage k - 1 has been read before its slot is requested again
        fetch(k + RING - 1, slot == 0 ? RING - 1 : slot - 1);
        wait_vmcnt<(RING - 1) * kLoads>();
        asm volatile("" ::: "memory");
        multiply(slot);
        slot = slot == RING - 1 ? 0 : slot + 1;
    }
    for_each_behind<RING - 2>(steps - k, [&](auto behind) {
        wait_vmcnt<decltype(behind)::value * kLoads>();
        asm volatile("" ::: "memory");
        multiply(slot);
        slot = slot == RING - 1 ? 0 : slot + 1;
    });
    using Acc4 = std::conditional_t<(EPI >= kF16_AFFINE), f32x4, i32x4>;
    __builtin_amdgcn_s_waitcnt(0xC07F);
#pragma unroll
    for (int i = 0; i < CB; ++i)
    {
#pragma unroll
        for (int j = 0; j < TB; ++j)
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                reinterpret_cast<Acc4*>(own)[((i * TB + j) * 4 + q) * 64 + lane]
                    = Acc4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kOwn; ++v)
    {
        int const u = v * NW + wave;
        if (u >= kUnits)
        {
            break;
        }
        Acc4 t = reinterpret_cast<Acc4 const*>(lds)[u * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w)
        {
            t += reinterpret_cast<Acc4 const*>(lds + w * (RING * STAGE))[u * 64 + lane];
        }
        int const b = u >> 2, q = u & 3, cb = n0 + (b / TB) * 32, tb = t0 + (b % TB) * 32;
        if (cb < p.N)
        {
            store_quad<IL_OUT, EPI>(p, t, scales[v], cb + 8 * q + 4 * half, tb + row, kpart);
        }
    }
}

// Which kernel a launch with operands of one layout takes: the one with the lowest estimate of
//
//   launch + units(x) * (tile + gelu + stage * (1 + busy * min(x, 1)) * K / 64)                    [us]
//
// where x is the number of tiles per CU.  Up to `resident` tiles run on a CU at once and share it, each behind the first
// costing `share` of a tile's time on its own; the ones beyond that wait their turn at `turn` each.  The CUs with the
// most tiles decide how long the launch takes as far as `whole` says (1: entirely, 0: an even spread).  `busy`: what a stage
// takes longer when every CU works than when few do.  `spill`: GPUs differ in how many CUs each shader engine has left, and
// workgroups are dealt to the engines evenly, so on some GPUs a launch of one workgroup per CU runs a second round from
// 3/4 of the CUs on (7765 tokens x 768 -> 768, 246 workgroups: 12.3 us on one GPU, 16.8 us on another).  Small tiles fill the
// chip where the problem has few of them, large ones move fewer bytes per multiplication where it has many, and the pieces
// cut the chain of stages by eight, or by four where they read whole lines, where neither fills it.
//
// The constants are fits.  Linear operands: to launches by themselves on the four layers of 768- and 1024-channel FP16
// encoders (graph replays, weights in the last-level cache), 16 to 33289 tokens, on two GPUs, one of them with the uneven
// engines.  The plan they choose takes 0.8 % more than the best of all in the mean (24 % at most, a launch at the edge
// of a second round); the kernels and the choice before took 13 % more (50 % at most).  The pieces' among them, which read whole
// lines, are fits to 30 layers of 64 to 4096 FP16 values or twice as many INT8 ones, 32 to 4096 channels, 1 to 4000 tokens, 1800
// launches, each piece's time multiplied by what the estimate of 64 x 64 tiles exceeds theirs by at the same sizes: tiles are
// estimated 1.0 times what they take at rows of 8 KB and 1.4 times at 128 bytes, and the choice is between the two; the wider pieces'
// tile a tenth more than fitted, since where the two pieces are even the small ones are (102 tokens x 768 -> 3072: 4.85 us, 4.93 in
// the wide ones).  0.6 % more than the best of ten plans in the mean; one launch takes 4 % more than with the pieces of half lines, no
// other more than 3 %.  (Fitted to the encoders' layers
// only, the pieces were taken for short rows where tiles are faster, us: 2100 tokens x 128 -> 512, FP16, 5.3 against 3.7 in tiles;
// 1700 x 384 -> 384 4.9 / 4.2; 600 x 384 -> 1152 5.0 / 4.4; 384 x 512 -> 2048 5.6 / 5.2.)
// Linear operands whose rows end within a line have kernels and constants of their own: stages of 64 bytes, tiles of up to 128 x
// 256, and constants fitted to launches by themselves before the other linear operands had stages of whole lines.  10 layers of
// 96 to 3104 channels, 40 to 33289 tokens, FP16 and INT8, 240 launches: 6.5 % less in the mean than when all linear operands
// had those kernels (launches of 3 us up to 8 % more, others up to 4 %), 0.4 % more than the best of the six plans.  With only 128 x 128 and
// 64 x 64 tiles and the constants of the whole lines it was 2.5 % more, 29 % at most (7765 tokens x 3104 -> 768, FP16: 50.2 us
// then, 64.4 so, 50.3 now).
// Interleaved operands: to launches by themselves on those of a
// 1024-channel INT8 encoder with weights from memory, and the ones that decide from 2500 tokens on (large tiles, 128 x 256,
// 128 x 128, 64 x 128, 128 x 128 deep) to whole passes of that encoder with the plans of one or two of its layers changed at a
// time: what a launch takes by itself does not say what it costs the ones around it.  At 9084 tokens 128 x 128 tiles are the
// faster ones for either feed-forward layer by itself, and the pass is 2.5 % faster with large tiles for both.  Over 142
// sizes of 2465 to 23000 tokens the pass takes 0.8 % less than with constants for launches by themselves, one of them more
// than 0.8 % more (7399 tokens, 1.9 %), and the best of the measured combinations would take another 0.9 % less (4 % at
// most).  32 sequences of up to 256 tokens: 2979 -> 2877 us.
// Interleaved tiles of 256 x 256, 256 x 192 and 128 x 192 fill the chip once where the ones above need a round and a bit
// of it (128 x 128 tiles for 5012 tokens x 4096 -> 1024: 1.25 rounds; 128 x 192: 0.84): fitted to whole passes as well, 70
// sizes on two GPUs with one layer's plan changed at a time, and only to launches of one round, where they were 1 to 5 % of
// the pass faster or slower by the size alone; what they take beyond that follows no such line, and they are not taken
// there.  0.4 us in `launch` is the margin by which they have to win (without it some passes are 2 % slower).  At these sizes
// the pass takes 1.3 % less in the mean, 8.8 % at most (8200 tokens), and more than 0.5 % more at two of 140.
// Deep rings: where one workgroup per CU is all there is, a tile is bound by the trips to memory of its own stages, and
// the LDS of the workgroups that do not come is better used for more of them (interleaved, weights from memory, 600 tokens
// x 4096 -> 1024 in 64 x 64 tiles: 12.9 us with three stages ahead, 9.5 us with seven; 128 x 128 tiles, 1900 tokens 20.8
// us with two, 17.4 us with three); with two and more per CU they are slower.  Sharing the k range of such a tile between
// groups of wavefronts instead (two or four groups, rings of their own) measured 9.9-10.4 us on the first of these and
// lost elsewhere.
struct TileCost
{
    int channels, tokens, resident;
    float launch, tile, stage, gelu, share, turn, whole, busy, spill;
};
enum LinearPlan
{
    kLargeTiles = 0, // interleaved: whole rounds of 256 x 256 tiles by persistent workgroups and smaller ones for the rest
    kTile128x256,
    kTile128x128,
    kTile64x128,
    kTile64x64,
    kTile128x128Deep, // the same tiles with a deeper ring of stages and fewer workgroups per CU
    kTile64x128Deep,
    kTile64x64Deep,
    kPiece32x64,
    kPiece32x32,
    kTile256x256,
    kTile256x192,
    kTile128x192,
    kTile128x192Deep,
    kTile128x64,
    kLinearPlans
};
constexpr float kOneRound = 1e3f; // of tiles that are taken only where a launch has no more of them than CUs
// [0]: linear operands, [1]: interleaved ones, [2]: linear ones whose rows end within a line of 128 bytes.  No channels: the
// layout has no such kernel.
constexpr TileCost kTileCosts[3][kLinearPlans] = {
    {{}, {}, {128, 128, 2, 4.64f, 0.00f, 0.231f, 0.60f, 0.61f, 1.02f, 0.40f, 0.25f}, {},
        {64, 64, 2, 3.82f, 0.29f, 0.082f, 0.23f, 0.70f, 0.89f, 0.63f, 0.34f},
        {128, 128, 1, 4.02f, 0.77f, 0.142f, 0.99f, 0.f, 1.30f, 0.77f, 0.51f, 0.10f}, {}, {},
        {32, 64, 1, 3.12f, 1.25f, 0.038f, 0.02f, 0.f, 1.08f, 0.89f, 0.56f},
        {32, 32, 2, 3.73f, 0.13f, 0.018f, 0.f, 1.78f, 1.72f, 0.61f, 0.54f},
        {256, 256, 1, 0.00f, 4.48f, 0.440f, 1.88f, 0.f, 1.02f, 0.54f, 0.97f, 0.11f},
        {256, 192, 1, 5.13f, 0.01f, 0.388f, 1.26f, 0.f, 1.35f, 0.67f, 0.56f, 0.15f},
        {128, 192, 2, 4.47f, 0.10f, 0.289f, 0.70f, 0.78f, 0.99f, 0.47f, 0.38f},
        {128, 192, 1, 4.87f, 0.02f, 0.194f, 1.21f, 0.f, 1.45f, 0.62f, 0.55f, 0.11f},
        {128, 64, 2, 3.91f, 0.15f, 0.116f, 0.37f, 0.90f, 1.02f, 0.61f, 0.38f}},
    {{256, 256, 1, 0.00f, 3.34f, 0.542f, 4.36f, 0.f, 0.f, 0.f}, {128, 256, 2, 2.72f, 0.81f, 0.391f, 1.69f, 1.03f, 1.39f, 0.63f},
        {128, 128, 3, 3.06f, 0.79f, 0.233f, 0.53f, 0.87f, 1.01f, 0.47f}, {64, 128, 3, 2.96f, 0.26f, 0.169f, 0.32f, 1.59f, 0.94f, 0.00f},
        {64, 64, 4, 3.19f, 0.04f, 0.141f, 0.24f, 0.60f, 0.66f, 0.00f}, {128, 128, 2, 3.04f, 0.62f, 0.221f, 0.66f, 1.62f, 1.38f, 0.61f},
        {64, 128, 2, 2.54f, 0.60f, 0.150f, 0.32f, 1.22f, 0.93f, 0.35f}, {64, 64, 2, 2.46f, 0.54f, 0.100f, 0.35f, 0.93f, 0.91f, 0.46f},
        {32, 64, 2, 3.19f, 0.17f, 0.068f, 0.04f, 0.90f, 1.19f, 0.67f}, {32, 32, 4, 2.69f, 1.21f, 0.042f, 0.16f, 0.67f, 1.19f, 0.64f},
        {256, 256, 1, 5.39f, 0.f, 0.406f, 4.88f, 0.f, kOneRound, 1.f, 0.41f}, {256, 192, 1, 5.31f, 0.f, 0.217f, 2.67f, 0.f, kOneRound, 1.f, 1.50f},
        {128, 192, 1, 4.55f, 0.f, 0.142f, 1.01f, 0.f, kOneRound, 1.f, 1.47f}, {}, {}},
    {{}, {128, 256, 2, 2.06f, 2.05f, 0.430f, 0.64f, 1.50f, 1.22f, 0.62f}, {128, 128, 2, 1.93f, 1.06f, 0.292f, 0.41f, 1.30f, 1.10f, 0.53f},
        {64, 128, 3, 2.49f, 0.32f, 0.188f, 0.21f, 1.27f, 1.14f, 0.52f}, {64, 64, 4, 2.29f, 0.30f, 0.138f, 0.13f, 0.94f, 0.89f, 0.47f},
        {}, {}, {}, {32, 64, 1, 2.88f, 0.30f, 0.071f, 0.05f, 0.57f, 1.91f, 0.80f}, {32, 32, 1, 2.38f, 0.34f, 0.053f, 0.13f, 1.48f, 1.49f, 0.68f}}};

// The costs of a launch's plans.
template <bool IL>
TileCost const* tile_costs(LinearArgs const& a)
{
    return kTileCosts[IL ? 1 : a.K % 128 == 0 ? 0 : 2];
}

inline float tile_time(TileCost const& c, LinearArgs const& a, bool gelu)
{
    float const x = (float) ceil_div(a.N, c.channels) * (float) ceil_div(a.T, c.tokens) / (float) num_cus();
    float units = 1.f + c.spill * std::max(0.f, 4.f * x - 3.f);
    if (x > 1.f)
    {
        float const y = c.whole * std::ceil(x) + (1.f - c.whole) * x, r = (float) c.resident;
        units = 1.f + c.share * (std::min(y, r) - 1.f) + c.turn * std::max(0.f, y - r);
    }
    float const stage = c.stage * (1.f + c.busy * std::min(x, 1.f));
    return c.launch + units * (c.tile + (gelu ? c.gelu : 0.f) + stage * (float) (a.K / 64));
}

// The same for the large tiles: whole rounds, and what is left behind them, as 64 x 64 pieces or as 128 x 128 tiles.
inline float large_tiles_time(TileCost const& c, LinearArgs const& a, int64_t smallTiles, bool gelu)
{
    float const stages = (float) (a.K / 64), cus = (float) num_cus();
    float const rounds = (float) ceil_div(a.mainTiles, num_cus());
    float rest = 0.f;
    if (a.pieces)
    {
        rest = (float) (a.N / 64) * (float) ceil_div(a.T - a.tokMain * kBig, 64) / cus * (6.63f + 0.175f * stages);
    }
    else if (smallTiles)
    {
        rest = std::ceil((float) smallTiles / cus) * (0.83f + (gelu ? 0.25f * c.gelu : 0.f) + 0.51f * stages);
    }
    return c.launch + rounds * (c.tile + (gelu ? c.gelu : 0.f) + c.stage * stages) + rest;
}

bool is_piece(int plan)
{
    return plan == kPiece32x64 || plan == kPiece32x32;
}

// The widest panel of at most `limit` channel tiles that divides their number.
int widest_panel(int tiles, int limit)
{
    int w = std::max(limit, 1);
    while (tiles % w != 0)
    {
        --w;
    }
    return w;
}

// What fetches a.prefetch behind the tiles, where the launch leaves CUs idle.
uint32_t prefetch_workgroups(LinearArgs const& a, int threads)
{
    return a.prefetch.data && a.mainTiles <= num_cus()
        ? 8u * ceil_div(a.prefetch.units / 8u, (uint32_t) (threads / 64 * kPrefetchLoads))
        : 0u;
}

// The workgroups of a.mainTiles tiles, with those behind them.
template <typename Kernel>
int launch_tiles(hipStream_t stream, LinearArgs const& a, Kernel kernel, int threads)
{
    hipLaunchKernelGGL(kernel, dim3((uint32_t) a.mainTiles + prefetch_workgroups(a, threads)), dim3(threads), 0, stream, address(a.w),
        address(a.a), a.K, a.T, a.N, a.mainTiles, a.panelDiv.d, a.panelDiv.mul, a.panelDiv.shifts, a.perPanelDiv.d, a.perPanelDiv.mul,
        a.perPanelDiv.shifts, a);
    return check_launch("int8_linear");
}

// The same for pieces of `channels` x `tokens` by `threads` threads, stages of `stage` bytes of k dealt to them, in as many parts
// as a.parts says.
template <bool IL, typename Kernel>
int launch_pieces(hipStream_t stream, LinearArgs a, Kernel kernel, int channels, int tokens, int threads, int stage)
{
    uint32_t const nbm = (uint32_t) ceil_div(a.N, channels);
    a.tokMain = ceil_div(a.T, tokens);
    a.mainTiles = (int) nbm * a.tokMain * a.parts;
    a.perPart = ceil_div(a.K / stage, a.parts);
    uint32_t const behind = IL ? prefetch_workgroups(a, threads) : 0u;
    hipLaunchKernelGGL(kernel, dim3(nbm, (uint32_t) a.tokMain, (uint32_t) a.parts + ceil_div(behind, nbm * (uint32_t) a.tokMain)),
        dim3(threads), 0, stream, address(a.w), address(a.a), address(a.alpha), address(a.beta), a.K, a.T, a.N, a.parts,
        a.perPart, a);
    return check_launch("int8_linear");
}

template <bool IL, bool IL_OUT, int EPI>
int launch_plan(hipStream_t stream, LinearArgs a, int plan)
{
    TileCost const& c = tile_costs<IL>(a)[plan];
    int64_t const nbm = ceil_div(a.N, c.channels), grid = nbm * ceil_div(a.T, c.tokens);
    if (grid >= (int64_t) 1 << 31)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "int8_linear: too many tiles");
    }
    a.parts = 1;
    if (!is_piece(plan))
    {
        // panels of at most 2 MB of weights: half of an XCD's L2
        a.tokMain = ceil_div(a.T, c.tokens);
        a.mainTiles = (int) grid;
        a.panel = widest_panel((int) nbm, (int) std::min<int64_t>(nbm, (2 << 20) / ((int64_t) c.channels * a.K)));
        a.panelDiv = fast_div((uint32_t) a.panel);
        a.perPanelDiv = fast_div((uint32_t) a.panel * (uint32_t) a.tokMain);
    }
    auto run = [&](auto kernel, int threads) { return launch_tiles(stream, a, kernel, threads); };
    if constexpr (IL)
    {
        switch (plan)
        {
        case kTile128x256: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 4, 2, 2, 3, 4>, 512);
        case kTile128x128: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 2, 3, 3>, 256);
        case kTile64x128: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 2, 4, 3>, 256);
        case kTile64x64: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 1, 4, 4>, 256);
        case kTile128x128Deep: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 2, 4, 2>, 256);
        case kTile64x128Deep: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 2, 6, 2>, 256);
        case kTile64x64Deep:
            // 128 bytes of k per stage where k comes in those: half the barriers
            return a.K % 128 == 0 ? run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 1, 4, 2, 4>, 256)
                                  : run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 1, 8, 2>, 256);
        case kTile256x256: return run(linear_tile_kernel<IL, IL_OUT, EPI, 4, 2, 2, 4, 4, 2>, 512);
        case kTile256x192: return run(linear_tile_kernel<IL, IL_OUT, EPI, 4, 2, 2, 3, 5, 2>, 512);
        case kTile128x192: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 3, 4, 2>, 256);
        case kPiece32x64: return launch_pieces<IL>(stream, a, linear_piece_kernel<IL_OUT, EPI, 1, 2, 4, 4>, 32, 64, 512, 32);
        case kPiece32x32: return launch_pieces<IL>(stream, a, linear_piece_kernel<IL_OUT, EPI, 1, 1, 8, 4>, 32, 32, 512, 32);
        default: break;
        }
    }
    else if (a.K % 128 != 0)
    {
        // rows that end within a line: stages of 64 bytes
        switch (plan)
        {
        case kTile128x256: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 4, 2, 2, 3, 4>, 512);
        case kTile128x128: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 4, 2, 1, 4, 4>, 512);
        case kTile64x128: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 2, 4, 3>, 256);
        case kTile64x64: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 1, 4, 4>, 256);
        case kPiece32x64: return launch_pieces<IL>(stream, a, linear_piece_dma_kernel<IL_OUT, EPI, 1, 2, 3, 8, 2, 2>, 32, 64, 512, 64);
        case kPiece32x32: return launch_pieces<IL>(stream, a, linear_piece_dma_kernel<IL_OUT, EPI, 1, 1, 4, 8, 2, 2>, 32, 32, 512, 64);
        default: break;
        }
    }
    else
    {
        switch (plan)
        {
        case kPiece32x64: return launch_pieces<IL>(stream, a, linear_piece_dma_kernel<IL_OUT, EPI, 1, 2, 3, 4, 4, 1>, 32, 64, 256, 128);
        case kPiece32x32: return launch_pieces<IL>(stream, a, linear_piece_dma_kernel<IL_OUT, EPI, 1, 1, 2, 4, 4, 2>, 32, 32, 256, 128);
        case kTile256x256: return run(linear_tile_kernel<IL, IL_OUT, EPI, 4, 2, 2, 4, 2, 2, 4>, 512);
        case kTile256x192: return run(linear_tile_kernel<IL, IL_OUT, EPI, 4, 2, 2, 3, 2, 2, 4>, 512);
        case kTile128x192: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 3, 2, 2, 4>, 256);
        case kTile128x192Deep: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 3, 3, 1, 4>, 256);
        case kTile128x128: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 2, 2, 2, 4>, 256);
        case kTile128x128Deep: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 2, 4, 1, 4>, 256);
        case kTile128x64: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 2, 1, 3, 2, 4>, 256);
        case kTile64x64: return run(linear_tile_kernel<IL, IL_OUT, EPI, 2, 2, 1, 1, 5, 2, 4>, 256);
        default: break;
        }
    }
    return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: no such plan for this layout: %d", plan);
}

// Partial sums of `parts` workgroups per piece, in pieces of 32 x 32.  Parts are no more than bring the workgroups to one per CU, so
// linear operands have the LDS of a second one for rings of four stages of whole lines (up to 128 tokens x 3072 -> 768, FP16: 4.29 us
// in traced passes, 4.40 with rings of two).
template <bool IL, int EPI>
int launch_partial(hipStream_t stream, LinearArgs a, int parts, void* partial, WeightPrefetch const& prefetch = {nullptr, 0})
{
    a.out = partial;
    a.parts = parts;
    a.prefetch = prefetch;
    if constexpr (IL)
    {
        return launch_pieces<IL>(stream, a, linear_piece_kernel<false, EPI, 1, 1, 8, 4>, 32, 32, 512, 32);
    }
    else
    {
        return a.K % 128 == 0 ? launch_pieces<IL>(stream, a, linear_piece_dma_kernel<false, EPI, 1, 1, 4, 4, 4, 1>, 32, 32, 256, 128)
                              : launch_pieces<IL>(stream, a, linear_piece_dma_kernel<false, EPI, 1, 1, 4, 8, 2, 2>, 32, 32, 512, 64);
    }
}

// The plan of a launch with operands of one layout and tokMain / mainTiles / pieces set up for the large tiles.
template <bool IL>
int cheapest_plan(LinearArgs const& a, int64_t smallTiles, bool gelu, int plan)
{
    bool const large = IL && a.N % kBig == 0 && a.K % 256 == 0 && a.mainTiles > 0;
    TileCost const* const costs = tile_costs<IL>(a);
    auto const exists = [&](int q) {
        if (q == kLargeTiles)
        {
            return large;
        }
        if (is_piece(q) && ceil_div(a.T, costs[q].tokens) > 65535)
        {
            return false; // the second extent of their grid
        }
        return costs[q].channels != 0;
    };
    if (plan >= 0 && plan < kLinearPlans && exists(plan))
    {
        return plan;
    }
    float best = std::numeric_limits<float>::max();
    for (int q = kLargeTiles; q < kLinearPlans; ++q)
    {
        if (!exists(q))
        {
            continue;
        }
        float const t = q == kLargeTiles ? large_tiles_time(costs[q], a, smallTiles, gelu) : tile_time(costs[q], a, gelu);
        if (t < best)
        {
            best = t;
            plan = q;
        }
    }
    return plan;
}

thread_local int64_t gLinearEstimates = 0; // plans worked out rather than remembered, for trtamd_test_linear_estimates

// The same, remembered by each thread for the sizes it asked for last: the layers of a pass ask for the same few plans over
// and over, and the estimates take 0.3 us where a short launch costs the host 3.  Four layers and two halves of a batch are
// eight sizes; any sixteen of them have a place each, the oldest making room for the next.
template <bool IL>
int choose_plan(LinearArgs const& a, int64_t smallTiles, bool gelu)
{
    struct Choice
    {
        int T, K, N, mainTiles, pieces, gelu, setting, plan;
        int64_t smallTiles;
    };
    constexpr int kChoices = 16;
    thread_local Choice choices[kChoices] = {};
    thread_local int oldest = 0;
    int const setting = tuning(Tuning::kLinearPlan);
    bool const large = IL && a.mainTiles > 0; // if not, there is nothing for the other tiles to stand behind
    int const mainTiles = large ? a.mainTiles : 0, pieces = large ? a.pieces : 0;
    int64_t const behind = large ? smallTiles : 0;
    for (Choice const& c : choices)
    {
        if (c.T == a.T && c.K == a.K && c.N == a.N && c.gelu == (int) gelu && c.mainTiles == mainTiles && c.pieces == pieces
            && c.smallTiles == behind && c.setting == setting)
        {
            return c.plan;
        }
    }
    ++gLinearEstimates;
    Choice& c = choices[oldest];
    oldest = (oldest + 1) % kChoices;
    c = {a.T, a.K, a.N, mainTiles, pieces, (int) gelu, setting, cheapest_plan<IL>(a, smallTiles, gelu, setting), behind};
    return c.plan;
}

// The plan of a launch too short for large tiles, for callers that want to know ahead (-1: one that may have them).
template <bool IL>
int small_plan(LinearArgs a, bool gelu)
{
    bool const large = IL && (int64_t) ceil_div(a.N, kBig) * (a.T / kBig) > 0;
    if (large || !tuning(Tuning::kLinearPersistent) || !tuning(Tuning::kLinearDirect))
    {
        return -1;
    }
    a.mainTiles = 0;
    return choose_plan<IL>(a, 0, gelu);
}

// Parts of a layer whose launch is `plan`: as many as bring its workgroups to one per CU, and no less than 1 KB of k for
// each (two stages for each wavefront of linear operands, eight with 64 bytes or four with 128; four slabs of 32 bytes of interleaved
// ones).  The wider pieces are chosen where the smaller ones no longer fit on the CUs at once, so
// there is nothing left to share them between.
int parts_of(int plan, LinearArgs const& a)
{
    if (plan != kPiece32x32 || a.T <= 0 || a.T > kLinearPartialTokens || a.K < kLinearPartialK)
    {
        return 1;
    }
    int const grid = ceil_div(a.N, 32) * ceil_div(a.T, 32);
    return std::max(1, std::min({kMaxLinearParts, num_cus() / grid, a.K / 1024}));
}

// Large tiles for as many whole rows of 256 tokens as fit in full rounds of one workgroup per CU, plus a last partial round when
// it would occupy more than `partial` per cent of the CUs: in 128 x 128 tiles that remainder needs three rounds or more, which
// take longer than one round of large tiles.  Returns the 128 x 128 tiles behind them.
int64_t place_large_tiles(LinearArgs& a)
{
    int const nbmBig = ceil_div(a.N, kBig);
    int64_t const bigTiles = (int64_t) nbmBig * (a.T / kBig);
    int const cus = num_cus();
    int const partial = tuning(Tuning::kLinearPartialRound);
    int64_t roundedTiles = (bigTiles / cus) * cus;
    if ((bigTiles - roundedTiles) * 100 > (int64_t) partial * cus)
    {
        roundedTiles = bigTiles;
    }
    a.tokMain = (int) (roundedTiles / nbmBig);
    a.mainTiles = a.tokMain * nbmBig;
    return (int64_t) ceil_div(a.N, kSmall) * ceil_div(a.T - a.tokMain * kBig, kSmall);
}

// The plan of a launch whose large tiles are placed.  Few 128 x 128 tiles behind them (no more than TRTAMD_LINEAR_PIECES per cent
// of the CUs busy with a long k loop each): the same tokens as 64 x 64 pieces whose wavefronts split k (linear_piece64).
template <bool IL>
int plan_behind_large_tiles(LinearArgs& a, int64_t smallTiles, bool gelu)
{
    a.pieces = IL && a.T > a.tokMain * kBig && smallTiles * 100 <= (int64_t) tuning(Tuning::kLinearPieces) * num_cus();
    return choose_plan<IL>(a, smallTiles, gelu);
}

template <bool IL_W, bool IL_IN, bool IL_OUT, int EPI>
int launch_shape(hipStream_t stream, LinearArgs a)
{
    int const nbmBig = ceil_div(a.N, kBig), cus = num_cus();
    int64_t const smallTiles = place_large_tiles(a), grid = a.mainTiles + smallTiles;
    if (grid >= (int64_t) 1 << 31)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "int8_linear: too many tiles");
    }
    int const persistent = tuning(Tuning::kLinearPersistent);
    int const direct = tuning(Tuning::kLinearDirect);
    constexpr int kMaxPanel = 8; // 8 x 256 channels x K = 1024 of weights is half of an XCD's 4 MB L2
    if constexpr (IL_W == IL_IN && (EPI == kAFFINE || EPI == kGELU || EPI == kF16_AFFINE || EPI == kF16_GELU))
    {
        if (persistent && direct)
        {
            int const plan = plan_behind_large_tiles<IL_W>(a, smallTiles, EPI == kGELU || EPI == kF16_GELU);
            if (plan != kLargeTiles) // numbers its tiles itself
            {
                return launch_plan<IL_W, IL_OUT, EPI>(stream, a, plan);
            }
            if constexpr (IL_W && (EPI == kAFFINE || EPI == kGELU))
            {
                a.panel = widest_panel(nbmBig, std::min(nbmBig, kMaxPanel));
                a.persist = a.mainTiles < cus ? a.mainTiles : cus;
                int64_t const behind = a.pieces ? (int64_t) (a.N / 64) * ceil_div(a.T - a.tokMain * kBig, 64) : smallTiles;
                hipLaunchKernelGGL((int8_linear_dma_kernel<IL_OUT, EPI>), dim3((uint32_t) (a.persist + behind)), dim3(512), 0,
                    stream, a);
                return check_launch("int8_linear_dma_kernel");
            }
        }
    }
    a.panel = widest_panel(nbmBig, std::min(nbmBig, kMaxPanel));
    if (persistent && a.K % 128 == 0)
    {
        a.persist = a.mainTiles < cus ? a.mainTiles : cus;
        hipLaunchKernelGGL((int8_linear_persistent_kernel<IL_W, IL_IN, IL_OUT, EPI>),
            dim3((uint32_t) (grid - a.mainTiles + a.persist)), dim3(512), 0, stream, a);
        return check_launch("int8_linear_persistent_kernel");
    }
    hipLaunchKernelGGL((int8_linear_kernel<IL_W, IL_IN, IL_OUT, EPI>), dim3((uint32_t) grid), dim3(512), 0, stream, a);
    return check_launch("int8_linear_kernel");
}

template <bool IL_W, bool IL_IN>
int launch_out(hipStream_t stream, LinearArgs const& a, int epilogue, bool ilOut)
{
    switch (epilogue)
    {
    case kAFFINE:
        return ilOut ? launch_shape<IL_W, IL_IN, true, kAFFINE>(stream, a)
                     : launch_shape<IL_W, IL_IN, false, kAFFINE>(stream, a);
    case kGELU:
        return ilOut ? launch_shape<IL_W, IL_IN, true, kGELU>(stream, a)
                     : launch_shape<IL_W, IL_IN, false, kGELU>(stream, a);
    case kRAW: return launch_shape<IL_W, IL_IN, false, kRAW>(stream, a);
    case kHALF: return launch_shape<IL_W, IL_IN, false, kHALF>(stream, a);
    default: return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: unknown epilogue %d", epilogue);
    }
}

} // namespace
} // namespace trtamd

namespace trtamd
{
namespace
{

LinearArgs args_of(trtamd_int8_linear_params const& p)
{
    LinearArgs a{};
    a.a = p.a;
    a.w = p.w;
    a.alpha = p.alpha;
    a.beta = p.beta;
    a.out = p.out;
    a.T = p.T;
    a.K = p.K;
    a.N = p.N;
    a.qOut = p.out_scale;
    a.panel = 1;
    return a;
}

LinearArgs args_of(trtamd_fp16_linear_params const& p)
{
    LinearArgs a{};
    a.a = reinterpret_cast<int8_t const*>(p.a);
    a.w = reinterpret_cast<int8_t const*>(p.w);
    a.alpha = p.alpha;
    a.beta = p.beta;
    a.out = p.out;
    a.T = p.T;
    a.K = 2 * p.K;
    a.N = p.N;
    a.qOut = 1.f;
    a.panel = 1;
    return a;
}

int check_int8(trtamd_int8_linear_params const* p)
{
    if (p == nullptr || p->a == nullptr || p->w == nullptr || p->out == nullptr)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: null pointer");
    }
    if (p->T < 0 || p->K <= 0 || p->N <= 0 || p->K % 64 != 0 || p->N % 32 != 0)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: T=%d K=%d N=%d (K must be a multiple of 64, N of 32)",
            p->T, p->K, p->N);
    }
    if (p->epilogue != TRTAMD_LINEAR_RAW_INT32 && (p->alpha == nullptr || p->beta == nullptr))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: alpha and beta are required by this epilogue");
    }
    bool const wideOut = p->epilogue == TRTAMD_LINEAR_RAW_INT32 || p->epilogue == TRTAMD_LINEAR_AFFINE_FP16;
    if (wideOut && p->out_interleaved)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: INT32 and FP16 outputs are linear only");
    }
    if ((int64_t) p->T * p->K >= (int64_t) 1 << 31 || (int64_t) p->N * p->K >= (int64_t) 1 << 31)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "int8_linear: operand of 2 GiB or more");
    }
    if (!aligned16(p->a) || !aligned16(p->w) || !aligned16(p->out) || (p->alpha && !aligned16(p->alpha))
        || (p->beta && !aligned16(p->beta)))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "int8_linear: pointers must be 16-byte aligned");
    }
    return TRTAMD_STATUS_SUCCESS;
}

int run_int8(trtamd_stream_t stream, trtamd_int8_linear_params const* p, WeightPrefetch const& prefetch)
{
    int const checked = check_int8(p);
    if (checked != TRTAMD_STATUS_SUCCESS)
    {
        return checked;
    }
    if (p->T == 0)
    {
        return TRTAMD_STATUS_SUCCESS;
    }
    LinearArgs a = args_of(*p);
    a.prefetch = prefetch;
    bool const ilOut = p->out_interleaved != 0;
    hipStream_t const st = as_stream(stream);
    if (p->w_interleaved)
    {
        return p->a_interleaved ? launch_out<true, true>(st, a, p->epilogue, ilOut)
                                : launch_out<true, false>(st, a, p->epilogue, ilOut);
    }
    return p->a_interleaved ? launch_out<false, true>(st, a, p->epilogue, ilOut)
                            : launch_out<false, false>(st, a, p->epilogue, ilOut);
}

int check_fp16(trtamd_fp16_linear_params const* p)
{
    if (p == nullptr || p->a == nullptr || p->w == nullptr || p->out == nullptr || p->alpha == nullptr
        || p->beta == nullptr)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fp16_linear: null pointer");
    }
    if (p->T < 0 || p->K <= 0 || p->N <= 0 || p->K % 32 != 0 || p->N % 32 != 0)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fp16_linear: T=%d K=%d N=%d (K and N must be multiples of 32)", p->T,
            p->K, p->N);
    }
    if (p->epilogue != TRTAMD_LINEAR_AFFINE && p->epilogue != TRTAMD_LINEAR_GELU)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fp16_linear: unknown epilogue %d", p->epilogue);
    }
    if ((int64_t) p->T * p->K >= (int64_t) 1 << 30 || (int64_t) p->N * p->K >= (int64_t) 1 << 30)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fp16_linear: operand of 2 GiB or more");
    }
    if (!aligned16(p->a) || !aligned16(p->w) || !aligned16(p->out) || !aligned16(p->alpha) || !aligned16(p->beta))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fp16_linear: pointers must be 16-byte aligned");
    }
    return TRTAMD_STATUS_SUCCESS;
}

int run_fp16(trtamd_stream_t stream, trtamd_fp16_linear_params const* p)
{
    int const checked = check_fp16(p);
    if (checked != TRTAMD_STATUS_SUCCESS)
    {
        return checked;
    }
    if (p->T == 0)
    {
        return TRTAMD_STATUS_SUCCESS;
    }
    LinearArgs const a = args_of(*p);
    hipStream_t const st = as_stream(stream);
    return p->epilogue == TRTAMD_LINEAR_GELU ? launch_shape<false, false, false, kF16_GELU>(st, a)
                                             : launch_shape<false, false, false, kF16_AFFINE>(st, a);
}

// What the partial launches ask beyond that: the sums fit in linear_partial_bytes().
int check_partial(int32_t T, int32_t N, int parts, void const* partial)
{
    if (partial == nullptr || !aligned16(partial))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "linear layer: the buffer of partial sums must be 16-byte aligned");
    }
    if (T <= 0 || parts < 1 || parts > kMaxLinearParts || (int64_t) ceil_div(N, 32) * ceil_div(T, 32) * parts > num_cus())
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "linear layer: %d parts of T=%d N=%d do not fit the partial sums", parts, T, N);
    }
    return TRTAMD_STATUS_SUCCESS;
}

// Whether operands are what the partial launches take (the checks above see to the rest).
bool interleaved(trtamd_int8_linear_params const& p)
{
    return p.a_interleaved && p.w_interleaved && (p.epilogue == TRTAMD_LINEAR_AFFINE || p.epilogue == TRTAMD_LINEAR_GELU);
}

} // namespace

// Pieces, whose launches are as long as the trip of their weights; and layers with longer rows than they have of them, whose
// workgroups walk a chain of stages that each wait for weights from memory (a model of 24 layers does not stay in the last-level
// cache): a pass of 24 layers of 1024 channels without / with the second feed-forward layer's weights fetched by the projection, us,
// processes in turn: 464 tokens 737 / 730, 531 847 / 833, 795 916 / 903, 837 921 / 908, 1144 1074 / 1044, 1781 1253 / 1232, 3268
// 1758 / 1747, no difference where the projection leaves no CU idle.  The first feed-forward layer's weights ahead of their launch
// cost up to 1 %, the other two's bring nothing.
WeightPrefetch prefetch_of(trtamd_int8_linear_params const& next)
{
    // N: the channel blocks have to come round to the same XCD in every k-slab
    if (!interleaved(next) || next.N % 256 != 0
        || (next.K <= next.N && !is_piece(small_plan<true>(args_of(next), next.epilogue == TRTAMD_LINEAR_GELU))))
    {
        return {nullptr, 0};
    }
    return {next.w, (uint32_t) ((int64_t) next.N * next.K / 1024)};
}

int int8_linear(trtamd_stream_t stream, trtamd_int8_linear_params const& p, WeightPrefetch const& prefetch)
{
    return run_int8(stream, &p, prefetch);
}

int linear_parts(trtamd_int8_linear_params const& p)
{
    return interleaved(p) && p.epilogue == TRTAMD_LINEAR_AFFINE ? parts_of(small_plan<true>(args_of(p), false), args_of(p)) : 1;
}

int linear_parts(trtamd_fp16_linear_params const& p)
{
    return p.epilogue == TRTAMD_LINEAR_AFFINE ? parts_of(small_plan<false>(args_of(p), false), args_of(p)) : 1;
}

size_t linear_partial_bytes()
{
    return (size_t) num_cus() * 32 * 32 * sizeof(int32_t);
}

int int8_linear_partial(trtamd_stream_t stream, trtamd_int8_linear_params const& p, int parts, int32_t* partial,
    WeightPrefetch const& prefetch)
{
    int st = check_int8(&p);
    st = st ? st : check_partial(p.T, p.N, parts, partial);
    return st ? st : launch_partial<true, kRAW>(as_stream(stream), args_of(p), parts, partial, prefetch);
}

int fp16_linear_partial(trtamd_stream_t stream, trtamd_fp16_linear_params const& p, int parts, float* partial)
{
    int st = check_fp16(&p);
    st = st ? st : check_partial(p.T, p.N, parts, partial);
    return st ? st : launch_partial<false, kF16_RAW>(as_stream(stream), args_of(p), parts, partial);
}

int fp16_linear_check(trtamd_fp16_linear_params const& p)
{
    return check_fp16(&p);
}

} // namespace trtamd

extern "C" int trtamd_test_linear_plan(int32_t interleaved, int32_t T, int32_t row_bytes, int32_t N, int32_t gelu)
{
    using namespace trtamd;
    if (T <= 0 || row_bytes <= 0 || N <= 0 || row_bytes % 64 != 0 || N % 32 != 0)
    {
        return -1;
    }
    LinearArgs a{};
    a.T = T;
    a.K = row_bytes;
    a.N = N;
    int64_t const smallTiles = place_large_tiles(a);
    return interleaved ? plan_behind_large_tiles<true>(a, smallTiles, gelu != 0) : plan_behind_large_tiles<false>(a, smallTiles, gelu != 0);
}

extern "C" int64_t trtamd_test_linear_estimates(void)
{
    return trtamd::gLinearEstimates;
}

extern "C" int trtamd_int8_linear(trtamd_stream_t stream, trtamd_int8_linear_params const* p)
{
    return trtamd::run_int8(stream, p, {nullptr, 0});
}

extern "C" int trtamd_fp16_linear(trtamd_stream_t stream, trtamd_fp16_linear_params const* p)
{
    return trtamd::run_fp16(stream, p);
}
