// Fused multi-head attention for gfx950 (head size 64, sequence length <= 512), INT8 and FP16.
//
// Stands in for the precompiled fused_multihead_attention / fused_multihead_attention_v2 kernels
// the reference loads from cubins (plugin/bertQKVToContextPlugin/fused_multihead_attention*/):
// one launch computes softmax(Q K^T * scale) V for every (sequence, head).
//
// Work split: a workgroup stages K and V of one (sequence, head) in LDS once (both row-major, rows
// padded by 16 bytes so 16-byte reads of consecutive keys fall in different banks) and its
// wavefronts then walk the 16-row query tiles of that head round-robin; `qSplit` workgroups share
// one head when the batch is too small to fill the chip otherwise.  Per query tile a wave
//   1. computes S^T = K Q^T with v_mfma_i32_16x16x64_i8 (v_mfma_f32_16x16x32_f16 for FP16): the
//      accumulator layout gives every lane 4 keys x 1 query per 16-key tile, which is exactly the
//      B-operand layout of step 3, so probabilities never leave registers;
//   2. does the row softmax over the whole row (<= 512 keys) in registers: max/sum need only two
//      cross-lane steps (the 4 lane groups that share a query).  INT8 accumulators are seeded
//      with the bit pattern of 1.5*2^23 so the integer result reads directly as a binary32
//      number (no int->float conversion); probabilities are quantised with one fused
//      multiply-add against the same constant (round-to-nearest-even lands in the low byte);
//   3. computes O^T = V^T P^T with the same MFMA; the V^T operand (16 keys of one head-dim per
//      lane) is produced from row-major V by the LDS transpose reads ds_read_b64_tr_b8 /
//      ds_read_b64_tr_b16, so V is never transposed in memory;
//   4. requantises (INT8) or normalises (FP16) on store.
// Queries beyond the sequence length are neither computed nor written.
#include "device_utils.hpp"
#include "host_utils.hpp"
#include "trtamd_test_hooks.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

namespace trtamd
{
namespace
{

constexpr int kQPerWave = 16;
constexpr int kWavesI8 = 4;
constexpr int kWavesF16 = 8;  // FP16 K/V take twice the LDS, so one (larger) workgroup per CU
constexpr int kWavesF16T = 4; // where K and V take turns in LDS
constexpr int kHeadSize = 64;
constexpr int kMagicBits = 0x4B400000;         // bit pattern of 12582912.f = 1.5 * 2^23
constexpr float kMagic = 12582912.f;
constexpr float kLog2e = 1.4426950408889634f;

typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// a * b rounded to binary32 on its own: the caller's following add must not absorb it into an fma
__device__ inline float mul_rounded(float a, float b)
{
#pragma clang fp contract(off)
    return a * b;
}

// The MFMAs of the cu_seqlens kernels (fmha_i8_prefix_kernel, fmha_f16_turns_kernel, fmha_f16_stream_kernel) go through
// these wrappers.  A
// library built with -DTRTAMD_ABLATE_ATTENTION_MFMA (`python -m tensorrt_amd.build --ablation` writes it to
// lib/libtrtamd_ablation.so; `python -m tensorrt_amd.kernel_bench --ablation` times it; nothing else loads it) leaves
// the instruction out: the result registers keep what they held and every other instruction of the kernel stays, so
// the results are wrong and the launch takes what the kernel would take if its matrix work cost nothing.
__device__ __forceinline__ i32x4 attention_mfma_i8(i32x4 const a, i32x4 const b, i32x4 c)
{
#ifdef TRTAMD_ABLATE_ATTENTION_MFMA
    i32x4 d;
    asm volatile("; v_mfma_i32_16x16x64_i8 left out" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
#else
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
#endif
}

__device__ __forceinline__ f32x4 attention_mfma_f16(f16x8 const a, f16x8 const b, f32x4 c)
{
#ifdef TRTAMD_ABLATE_ATTENTION_MFMA
    f32x4 d;
    asm volatile("; v_mfma_f32_16x16x32_f16 left out" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
#else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
#endif
}

__device__ __forceinline__ f32x16 attention_mfma_f16_32(f16x8 const a, f16x8 const b, f32x16 c)
{
#ifdef TRTAMD_ABLATE_ATTENTION_MFMA
    f32x16 d;
    asm volatile("; v_mfma_f32_32x32x16_f16 left out" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
#else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
#endif
}

// x[dt] of the lane in 16-lane row g  ->  x[g'] = what row g' held in its x[g]: a 4 x 4 transpose over the four rows of
// a wavefront.  All 64 lanes must be active.  The attention kernels end with lane (g, query) holding a piece of each
// quarter dt of the query's output row; transposed, it holds the whole quarter dt = g and stores it in one piece.
__device__ inline void rows_transpose(uint32_t (&x)[4])
{
    // rows 0,1 keep x[0] / x[1] of their own and get the same from rows 2,3; rows 2,3 the other way round
    auto const s02 = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
    auto const s13 = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
    // even rows keep the first of a pair and get it from the odd row below them; odd rows the second
    auto const t01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    auto const t23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    x[0] = t01[0];
    x[1] = t01[1];
    x[2] = t23[0];
    x[3] = t23[1];
}

// The order in which a launch's workgroups take its units: bit 0 says the longest sequences first instead of the sequences as
// they come, the rest is the number of ids, a multiple of 512, of which every other round of 256 goes backwards.
constexpr uint32_t kRanked = 1;
constexpr uint32_t kTwoRounds = 512;

// Ids are dealt to the 8 XCDs in turn and there to the 32 CUs, so a round of 256 of them puts a workgroup on every CU, and the
// next round, in the same order, would give the CU of the longest unit the longest again, and the CU of a unit's first part,
// which is always full, a first part again: 32 is a multiple of 2 and of 4 parts, and the last part of a short sequence is
// empty.  Backwards, within each XCD, a round evens out what the one before it left uneven.  (What the hardware does beyond the
// first rounds, or with another number of CUs, only costs evenness: the ids of a whole round change places among themselves.)
__device__ __forceinline__ uint32_t id_of_workgroup(uint32_t bid, uint32_t order)
{
    uint32_t const odd = 0u - ((bid >> 8) & 1u);
    return bid ^ (odd & (bid < order ? 0xf8u : 0u)); // an id of an odd round is not a multiple of 512: bit 0 makes no difference
}

struct FmhaArgs
{
    void const* qkv;
    void* out;
    int32_t const* cuSeqlens;    // var-seqlen: [B+1]; nullptr = fixed layout
    uint32_t const* packedMask;  // fixed layout: packed key mask or nullptr (all keys valid)
    int64_t tokStrideIn;         // bytes between consecutive tokens of one sequence
    int64_t tokStrideOut;
    int64_t seqStrideIn;         // fixed layout: bytes between sequences (b -> b+1)
    int64_t seqStrideOut;
    int64_t maskStrideWords;
    int32_t B, N, S;
    int32_t qSplit;              // workgroups per (sequence, head)
    int32_t total;               // interleaved: total token count
    int32_t warpsM, warpsN;      // geometry of the packed mask
    uint32_t spanInverse;        // 2^20 / (16 warpsN) rounded up: key * this >> 20 is key / (16 warpsN) for keys below 512
    float c;                     // scale_bmm1 * log2(e)
    float scaleSoftmax;
    float scaleBmm2;
    int32_t clampP;              // scale_softmax may push p beyond 127
    int32_t* dbgAcc1;            // optional [B][N][S][S] int32 (INT8) / float bits (FP16)
    int8_t* dbgP8;               // optional [B][N][S][S]
    uint32_t order;              // see kRanked
    FastDiv partDiv, headDiv;    // by qSplit and N
};

// The arguments of the cu_seqlens kernels: what a workgroup needs to find its sequence comes preloaded, as the leading scalars
// of the argument list, ...
#define TRTAMD_FMHA_LEADING_PARAMS                                                                                     \
    uint64_t const qkv, uint64_t const cuSeqlens, uint32_t const qSplit, uint32_t const qSplitMul,                      \
        uint32_t const qSplitShifts, uint32_t const N, uint32_t const headMul, uint32_t const headShifts, int const B, \
        int const S, uint32_t const order, int const total
#define TRTAMD_FMHA_LEADING_ARGS(a)                                                                                    \
    address((a).qkv), address((a).cuSeqlens), (a).partDiv.d, (a).partDiv.mul, (a).partDiv.shifts, (a).headDiv.d,       \
        (a).headDiv.mul, (a).headDiv.shifts, (a).B, (a).S, (a).order, (a).total
#define TRTAMD_FMHA_ARGS_OF(rest)                                                                                      \
    fmha_args(qkv, cuSeqlens, {qSplit, qSplitMul, qSplitShifts}, {N, headMul, headShifts}, B, S, order, total, rest)
__device__ __forceinline__ FmhaArgs fmha_args(uint64_t qkv, uint64_t cuSeqlens, FastDiv const& partDiv,
    FastDiv const& headDiv, int B, int S, uint32_t order, int total, FmhaArgs const& rest)
{
    FmhaArgs a = rest;
    a.qkv = global_ptr<void const>(qkv);
    a.cuSeqlens = global_ptr<int32_t const>(cuSeqlens);
    a.partDiv = partDiv;
    a.headDiv = headDiv;
    a.qSplit = (int) partDiv.d;
    a.N = (int) headDiv.d;
    a.B = B;
    a.S = S;
    a.order = order;
    a.total = total;
    return a;
}

// ... and the others are requested together while the bounds of the sequence are on their way.
__device__ __forceinline__ void pin_args(FmhaArgs const& a)
{
    asm volatile("" ::"s"(a.out), "s"(a.packedMask), "s"(a.tokStrideIn), "s"(a.tokStrideOut), "s"(a.seqStrideIn),
                 "s"(a.seqStrideOut), "s"(a.c), "s"(a.scaleBmm2));
}

template <int ESIZE>
struct Lds
{
    // K and V rows of 64 elements, unpadded; the 16-byte chunks of a row are XOR-swizzled with
    // the row index (see swz) so that the 8 consecutive rows a 16-lane group reads fall in
    // different banks
    static constexpr int kRow = kHeadSize * ESIZE;
    static __host__ __device__ constexpr int matBytes(int kt)
    {
        return kt * 64 * kRow;
    }
    static __host__ __device__ constexpr int total(int kt)
    {
        return 2 * matBytes(kt) + 16 * 4;
    }
};

// LDS row, inside its 64-key block, at which V's key kk is stored.  The accumulator of S^T gives
// lane group g the keys 16u + 4g + j (u = 16-key tile, j = 0..3) and the P^T operand is built
// from it without moving data.  One INT8 transpose read returns 8 keys to each lane group, which
// must be 8 consecutive LDS rows: tiles (2h, 2h+1), keys 4g..4g+3 of each -> rows 32h + 8g + 4(u&1) + j.
// The FP16 transpose read returns 4 keys, already consecutive (16u + 4g + j): natural order.
template <int ESIZE>
__device__ inline int v_row(int kk)
{
    int const u = kk >> 4, g = (kk >> 2) & 3, j = kk & 3;
    return ESIZE == 1 ? 32 * (u >> 1) + 8 * g + 4 * (u & 1) + j : kk;
}

// Position of 16-byte chunk `chunk` inside LDS row `row`.  Rows are 64 (INT8) or 128 (FP16) bytes;
// consecutive rows advance by a quarter / a half of the 256-byte bank window, so rows 2 (INT8) or
// 1 (FP16) apart in the sense below would collide without the swizzle.
template <int ESIZE>
__device__ inline int swz(int row, int chunk)
{
    return ESIZE == 1 ? (chunk ^ ((row >> 1) & 3)) : (chunk ^ (row & 7));
}

// Byte address of the 16-byte chunk `chunk` of matrix `mat` (0 Q, 1 K, 2 V) for head n, token
// `tok` of the sequence described by (seqBase, firstTok).
template <int ESIZE, bool INTERLEAVED>
__device__ inline int64_t qkv_chunk_offset(
    FmhaArgs const& a, int64_t seqBase, int64_t firstTok, int tok, int n, int mat, int chunk)
{
    if (INTERLEAVED)
    {
        // [3][N][d/32][T][32] bytes; chunk = 16-byte unit of the 64-byte head row
        int64_t const grp = ((int64_t) mat * a.N + n) * 2 + (chunk >> 1);
        return (grp * a.total + firstTok + tok) * 32 + (chunk & 1) * 16;
    }
    return seqBase + (int64_t) tok * a.tokStrideIn + ((int64_t) n * 3 + mat) * kHeadSize * ESIZE + chunk * 16;
}

// Builds the 512-bit key-valid mask of sequence b in LDS (sMask[16]): every thread takes one key (and one word of the
// packed mask, if there is one), a wavefront's 64 answers become two words of the mask.
__device__ inline void build_key_mask(FmhaArgs const& a, int b, int nk, uint32_t* sMask)
{
    int const lane = threadIdx.x & (kWaveSize - 1);
    for (int key = threadIdx.x; key < 512; key += blockDim.x)
    {
        bool valid = key < nk;
        if (valid && a.packedMask != nullptr)
        {
            // bit layout of fillSBSMaskKernel (plugin/embLayerNormPlugin/embLayerNormKernel.cu:41-85)
            uint32_t const* pm = a.packedMask + (int64_t) b * a.maskStrideWords;
            int const span = 16 * a.warpsN;
            int const ni = key / span;
            int const r = key % span;
            int const warpN = r >> 4;
            int const r2 = r & 15;
            int const tidx = warpN * a.warpsM * 32 + ((r2 & 7) >> 1);
            int const bit = 8 * ni + (r2 & 1) + ((r2 & 8) ? 4 : 0);
            valid = ((pm[tidx] >> bit) & 1u) != 0;
        }
        uint64_t const m = __ballot(valid);
        if (lane == 0)
        {
            sMask[key >> 5] = (uint32_t) m;
            sMask[(key >> 5) + 1] = (uint32_t) (m >> 32);
        }
    }
}

// One past the last key of the mask that takes part (0: none does).  Keys behind it have probability zero whatever
// their scores, so the kernels treat the sequence as that much shorter: whole blocks of masked keys at the end are
// neither loaded nor multiplied.  sMask must be complete (barrier) before the call; the result is wave-uniform.
__device__ inline int used_keys(uint32_t const* sMask, int nk)
{
    int const lane = threadIdx.x & (kWaveSize - 1);
    uint32_t const w = lane < 16 ? sMask[lane] : 0u;
    int end = w ? lane * 32 + 32 - __builtin_clz(w) : 0;
#pragma unroll
    for (int d = 1; d < 16; d *= 2)
    {
        end = max(end, __shfl_xor(end, d));
    }
    return min(__builtin_amdgcn_readfirstlane(end), nk);
}

// Stage K and V of one (sequence, head) into LDS, 16 bytes per lane per access.  Rows at or
// beyond nk are zero, and so are the K rows of masked keys: a masked key's score is then exactly
// the accumulator's seed, which the caller sets to -infinity (see mask_seed).  ESIZE = bytes per
// element (1 INT8, 2 FP16).  sMask must be complete (barrier) before the call.
template <int ESIZE, int KT, bool INTERLEAVED, int WAVES>
__device__ inline void stage_kv(FmhaArgs const& a, int64_t seqBase, int64_t firstTok, int n, int nk, int nkb,
    uint32_t const* sMask, uint8_t* sK, uint8_t* sV)
{
    constexpr int kChunks = kHeadSize * ESIZE / 16;     // 16-byte chunks per head row: 4 or 8
    constexpr int kRowsPerPass = WAVES * kWaveSize / kChunks;
    constexpr int kPasses = 64 / kRowsPerPass;          // passes per 64-key block
    constexpr int kRow = Lds<ESIZE>::kRow;
    uint8_t const* src = static_cast<uint8_t const*>(a.qkv);
    int const chunk = threadIdx.x % kChunks;
    int const rowInPass = threadIdx.x / kChunks;
    // every global load of the workgroup is issued before the first LDS write, so the loads of
    // all key blocks are in flight together
    u32x4 kv[KT][kPasses], vv[KT][kPasses];
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
    {
#pragma unroll
        for (int p = 0; p < kPasses; ++p)
        {
            int const key = kb * 64 + p * kRowsPerPass + rowInPass;
            kv[kb][p] = u32x4{0, 0, 0, 0};
            vv[kb][p] = u32x4{0, 0, 0, 0};
            if (key < nk)
            {
                vv[kb][p] = *reinterpret_cast<u32x4 const*>(
                    src + qkv_chunk_offset<ESIZE, INTERLEAVED>(a, seqBase, firstTok, key, n, 2, chunk));
                if ((sMask[key >> 5] >> (key & 31)) & 1u)
                {
                    kv[kb][p] = *reinterpret_cast<u32x4 const*>(
                        src + qkv_chunk_offset<ESIZE, INTERLEAVED>(a, seqBase, firstTok, key, n, 1, chunk));
                }
            }
        }
    }
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
    {
        if (kb < nkb)
        {
#pragma unroll
            for (int p = 0; p < kPasses; ++p)
            {
                int const kk = p * kRowsPerPass + rowInPass;
                int const kr = kb * 64 + kk;
                int const vr = kb * 64 + v_row<ESIZE>(kk);
                *reinterpret_cast<u32x4*>(sK + kr * kRow + swz<ESIZE>(kr, chunk) * 16) = kv[kb][p];
                *reinterpret_cast<u32x4*>(sV + vr * kRow + swz<ESIZE>(vr, chunk) * 16) = vv[kb][p];
            }
        }
    }
}

// Accumulator seed of the four keys 16u + 4g + j of a 16-key tile: `valid` for keys that take
// part, the bit pattern of -infinity for masked ones (their K rows are zero, so the seed is their
// score): the integer/float row maximum ignores it and 2^(-inf) = 0 removes it from the softmax
// without any per-score instruction.
constexpr int kNegInfBits = (int) 0xFF800000u;
__device__ inline i32x4 mask_seed(uint32_t w0, uint32_t w1, int u, int g, int valid)
{
    uint32_t const bits = ((u < 2 ? w0 : w1) >> ((u & 1) * 16 + g * 4)) & 0xfu;
    i32x4 seed;
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        seed[j] = (bits >> j) & 1u ? valid : kNegInfBits;
    }
    return seed;
}

struct SeqInfo
{
    int64_t seqBaseIn, seqBaseOut, firstTok;
    int nq, nk;
};

__device__ inline SeqInfo seq_info(FmhaArgs const& a, int b, int capacity)
{
    SeqInfo s;
    if (a.cuSeqlens)
    {
        int const first = a.cuSeqlens[b], end = a.cuSeqlens[b + 1];
        pin_args(a);
        int const len = min(max(end - first, 0), capacity);
        s.firstTok = first;
        s.seqBaseIn = (int64_t) first * a.tokStrideIn;
        s.seqBaseOut = (int64_t) first * a.tokStrideOut;
        s.nq = len;
        s.nk = len;
    }
    else
    {
        s.firstTok = 0;
        s.seqBaseIn = (int64_t) b * a.seqStrideIn;
        s.seqBaseOut = (int64_t) b * a.seqStrideOut;
        s.nq = min(a.S, capacity);
        s.nk = min(a.S, capacity);
    }
    return s;
}

// Which sequence a workgroup serves.  Workgroups are dispatched in index order, so serving the
// longest sequences first (cost grows with the square of the length) lets the short ones fill the
// tail of the launch.  `rank` is the position in that order; every workgroup ranks the (at most
// kMaxRanked) sequence lengths itself with a counting sort in LDS: no state outside the launch.
constexpr int kMaxRanked = 1024;
template <int THREADS>
__device__ inline int pick_sequence(FmhaArgs const& a, int rank, int* sLens /* [kMaxRanked + 1] */)
{
    if (a.cuSeqlens == nullptr || a.B > kMaxRanked || a.B == 1)
    {
        return rank; // fixed layout (equal lengths) or too many sequences: natural order
    }
    for (int t = threadIdx.x; t < a.B; t += THREADS)
    {
        sLens[t] = a.cuSeqlens[t + 1] - a.cuSeqlens[t];
    }
    if (threadIdx.x == 0)
    {
        sLens[kMaxRanked] = rank;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < a.B; t += THREADS)
    {
        int const mine = sLens[t];
        int before = 0; // sequences served before t: longer ones, ties by index
        for (int o = 0; o < a.B; ++o)
        {
            int const other = sLens[o];
            before += (other > mine || (other == mine && o < t)) ? 1 : 0;
        }
        if (before == rank)
        {
            sLens[kMaxRanked] = t;
        }
    }
    __syncthreads();
    return sLens[kMaxRanked];
}

// ------------------------------------------------------------------------------------------
// INT8
// ------------------------------------------------------------------------------------------
template <int KT, bool INTERLEAVED, bool DEBUG>
__global__ __launch_bounds__(kWavesI8* kWaveSize) __attribute__((amdgpu_waves_per_eu(KT <= 6 ? 3 : 2))) void fmha_i8_kernel(FmhaArgs const a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* sK = smem;
    uint8_t* sV = smem + Lds<1>::matBytes(KT);
    uint32_t* sMask = reinterpret_cast<uint32_t*>(sV + Lds<1>::matBytes(KT));
    constexpr int kRow = Lds<1>::kRow;

    __shared__ int sLens[kMaxRanked + 1];
    UnitPart const up = unit_of_workgroup(blockIdx.x, gridDim.x, a.qSplit);
    int const part = up.part;
    int const n = up.unit % a.N;
    int const b = pick_sequence<kWavesI8 * kWaveSize>(a, up.unit / a.N, sLens);
    SeqInfo const sq = seq_info(a, b, KT * 64);
    int const nqt = (sq.nq + kQPerWave - 1) / kQPerWave;
    if (part * kWavesI8 >= nqt)
    {
        return; // no query tile for this workgroup
    }
    build_key_mask(a, b, sq.nk, sMask);
    __syncthreads();
    int const nkUsed = used_keys(sMask, sq.nk);
    int const nkb = (nkUsed + 63) >> 6;
    int const ntile = (nkUsed + 15) >> 4; // 16-key tiles that hold at least one key
    stage_kv<1, KT, INTERLEAVED, kWavesI8>(a, sq.seqBaseIn, sq.firstTok, n, nkUsed, nkb, sMask, sK, sV);
    __syncthreads();

    int const lane = threadIdx.x & (kWaveSize - 1);
    int const wave = threadIdx.x >> 6;
    int const lq = lane & 15; // query (column of S^T / O^T)
    int const g = lane >> 4;  // lane group: 16-byte k-chunk of the operands, 4 rows of the accumulators
    uint8_t const* src = static_cast<uint8_t const*>(a.qkv);

    // Q^T operand of a tile: 16 bytes d = 16g .. 16g+15 of query 16*qt + lq (zero beyond the
    // sequence).  The next tile's operand is requested while the current tile is computed.
    auto load_q = [&](int qt) -> i32x4 {
        int const qq = qt * kQPerWave + lq;
        i32x4 v = {0, 0, 0, 0};
        if (qq < sq.nq)
        {
            v = *reinterpret_cast<i32x4 const*>(
                src + qkv_chunk_offset<1, INTERLEAVED>(a, sq.seqBaseIn, sq.firstTok, qq, n, 0, g));
        }
        return v;
    };
    int const qtStep = a.qSplit * kWavesI8;
    i32x4 qnext = load_q(part * kWavesI8 + wave);
    for (int qt = part * kWavesI8 + wave; qt < nqt; qt += qtStep)
    {
        int const q = qt * kQPerWave + lq;
        bool const qValid = q < sq.nq;
        i32x4 const qreg = qnext;
        qnext = load_q(qt + qtStep);

        // ---- S^T = K Q^T, biased so that the int32 reads as binary32 12582912 + acc --------
        i32x4 acc[KT * 4];
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
                uint32_t const w0 = __builtin_amdgcn_readfirstlane(sMask[kb * 2]);
                uint32_t const w1 = __builtin_amdgcn_readfirstlane(sMask[kb * 2 + 1]);
                bool const full = (w0 & w1) == 0xffffffffu;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    if (kb * 4 + u >= ntile)
                    {
                        break; // tiles wholly beyond the sequence are never touched
                    }
                    int const key = kb * 64 + u * 16 + lq;
                    i32x4 const kreg = *reinterpret_cast<i32x4 const*>(sK + key * kRow + swz<1>(key, g) * 16);
                    i32x4 seed = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
                    if (!full)
                    {
                        asm volatile("" ::: "memory"); // scalar branch, taken for the ragged last block only
                        seed = mask_seed(w0, w1, u, g, kMagicBits);
                    }
                    acc[kb * 4 + u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kreg, qreg, seed, 0, 0, 0);
                }
            }
        }

        if (DEBUG && a.dbgAcc1 && qValid)
        {
#pragma unroll
            for (int kb = 0; kb < KT; ++kb)
            {
                if (kb < nkb)
                {
                    for (int u = 0; u < 4; ++u)
                    {
                        for (int j = 0; j < 4; ++j)
                        {
                            int const key = kb * 64 + u * 16 + g * 4 + j;
                            if (key < nkUsed)
                            {
                                a.dbgAcc1[(((int64_t) b * a.N + n) * a.S + q) * a.S + key]
                                    = acc[kb * 4 + u][j] - kMagicBits;
                            }
                        }
                    }
                }
            }
        }

        // ---- row max on the biased integers (the bias is monotone; masked keys hold the
        //      negative pattern of -infinity) ------------------------------------------------------
        int mx = kNegInfBits;
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    if (kb * 4 + u >= ntile)
                    {
                        break;
                    }
                    mx = max(mx, max(max(acc[kb * 4 + u][0], acc[kb * 4 + u][1]),
                                     max(acc[kb * 4 + u][2], acc[kb * 4 + u][3])));
                }
            }
        }
        mx = reduce_step<16>(mx, [](int x, int y) { return max(x, y); });
        mx = reduce_step<32>(mx, [](int x, int y) { return max(x, y); });

        // ---- e = 2^((acc - max) * c), row sum; a fully masked row has max = -inf -> all e = 0 --
        float const negK0 = mx == kNegInfBits ? 0.f : -__int_as_float(mx) * a.c;
        float sum = 0.f;
        // e overwrites the accumulators in place (as bit patterns) to keep one row in registers
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    if (kb * 4 + u >= ntile)
                    {
                        break;
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        float const ev
                            = __builtin_amdgcn_exp2f(fmaf(__int_as_float(acc[kb * 4 + u][j]), a.c, negK0));
                        acc[kb * 4 + u][j] = __float_as_int(ev);
                        sum += ev;
                    }
                }
            }
        }
        sum = reduce_step<16>(sum, [](float x, float y) { return x + y; });
        sum = reduce_step<32>(sum, [](float x, float y) { return x + y; });
        float const r = sum > 0.f ? a.scaleSoftmax / sum : 0.f;
        // e * r <= scale_softmax: only a scale above 127 can leave the INT8 range; the row is then
        // pre-clamped through e <= 127 / r (one extra op per score on that rare path only)
        if (a.clampP)
        {
            asm volatile("" ::: "memory"); // keep this a scalar branch: the clamp must not be speculated
            float const emax = r > 0.f ? 127.f / r : 0.f;
#pragma unroll
            for (int kb = 0; kb < KT; ++kb)
            {
                if (kb < nkb)
                {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        if (kb * 4 + u >= ntile)
                        {
                            break;
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                        {
                            acc[kb * 4 + u][j] = __float_as_int(fminf(__int_as_float(acc[kb * 4 + u][j]), emax));
                        }
                    }
                }
            }
        }

        // ---- p8 = rne(e * r) packed four keys to a dword; O^T = V^T P^T -----------------------
        i32x4 oacc[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
        {
            oacc[dt] = i32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
                i32x4 preg = {0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    if (kb * 4 + u >= ntile)
                    {
                        break;
                    }
                    uint32_t yb[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        yb[j] = __float_as_uint(fmaf(__int_as_float(acc[kb * 4 + u][j]), r, kMagic));
                    }
                    uint32_t const lo = __builtin_amdgcn_perm(yb[1], yb[0], 0x0c0c0400u);
                    uint32_t const hi = __builtin_amdgcn_perm(yb[3], yb[2], 0x0c0c0400u);
                    preg[u] = (int) __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                }
                if (DEBUG && a.dbgP8 && qValid)
                {
                    for (int u = 0; u < 4; ++u)
                    {
                        for (int j = 0; j < 4; ++j)
                        {
                            int const key = kb * 64 + u * 16 + g * 4 + j;
                            if (key < nkUsed)
                            {
                                a.dbgP8[(((int64_t) b * a.N + n) * a.S + q) * a.S + key]
                                    = (int8_t) ((uint32_t) preg[u] >> (8 * j));
                            }
                        }
                    }
                }
                // V^T operand for head dims 16dt .. 16dt+15: lane r of a group addresses LDS row
                // (8 keys per read: r/2) at byte 16dt + 8(r%2); the transpose read hands lane i
                // the 8 keys of head dim 16dt + i.
                int const vrow = kb * 64 + 8 * g + (lq >> 1);
                uint8_t const* vbase = sV + vrow * kRow + 8 * (lq & 1);
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
                {
                    // rows vrow and vrow + 32 share (row >> 1) & 3, hence the swizzled chunk
                    int const sc = swz<1>(vrow, dt) * 16;
                    i32x2 const v0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*) (vbase + sc));
                    i32x2 const v1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*) (vbase + 32 * kRow + sc));
                    i32x4 const vreg = {v0[0], v0[1], v1[0], v1[1]};
                    oacc[dt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vreg, preg, oacc[dt], 0, 0, 0);
                }
            }
        }

        // ---- out8 = sat8(rne(acc2 * scale_bmm2)); lane holds d = 16dt + 4g .. +3 of query q, after the transpose
        //      the whole quarter d = 16g .. 16g+15
        uint32_t pk[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
        {
            uint32_t yb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                float y = (float) oacc[dt][j] * a.scaleBmm2;
                y = __builtin_amdgcn_fmed3f(y, -128.f, 127.f);
                yb[j] = __float_as_uint(y + kMagic);
            }
            uint32_t const lo = __builtin_amdgcn_perm(yb[1], yb[0], 0x0c0c0400u);
            uint32_t const hi = __builtin_amdgcn_perm(yb[3], yb[2], 0x0c0c0400u);
            pk[dt] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        }
        rows_transpose(pk);
        if (qValid)
        {
            uint8_t* dst = static_cast<uint8_t*>(a.out);
            int const d0 = g * 16;
            int64_t off;
            if (INTERLEAVED)
            {
                // [N][d/32][T][32]
                off = (((int64_t) n * 2 + (d0 >> 5)) * a.total + sq.firstTok + q) * 32 + (d0 & 31);
            }
            else
            {
                off = sq.seqBaseOut + (int64_t) q * a.tokStrideOut + (int64_t) n * kHeadSize + d0;
            }
            u32x4 const quarter = {pk[0], pk[1], pk[2], pk[3]};
            *reinterpret_cast<u32x4*>(dst + off) = quarter;
        }
    }
}

// Sequence selection for the var-seqlen kernels with a single trip to global memory: all B+1
// cu_seqlens values go to LDS, sequences are ordered longest first by 16-token bucket (ties by
// index) with a histogram, and the workgroup looks up the sequence at its own position.  Every
// workgroup computes the same order, so no state outside the launch is needed.
constexpr int kLenBuckets = 34; // (length + 15) / 16 for lengths 0 .. 512, and one for longer
struct PickLds
{
    int cu[kMaxRanked + 1];
    int hist[kLenBuckets];
};

__device__ inline int len_bucket(int len)
{
    return min(max(len + 15, 0) >> 4, kLenBuckets - 1);
}

// The same for up to kPicksPerLane * 64 sequences without LDS or a barrier, by every wavefront for itself: a lane keeps the
// bounds of its sequences in registers, the bucket that holds position `rank` is found bit by bit from the number of
// sequences in it or above, one ballot each.  INT8, 12 heads, sequences of a third of the length to the length, us per
// launch: 128 x 128 keys 14.1 -> 13.0, 64 x 384 28.2 -> 27.2, 128 x 256 26.3 -> 25.4.
constexpr int kPicksPerLane = 2;

__device__ inline SeqInfo pick_sequence_in_registers(FmhaArgs const& a, int rank, int capacity, int& bOut)
{
    int const lane = threadIdx.x & (kWaveSize - 1);
    int first[kPicksPerLane], end[kPicksPerLane], bucket[kPicksPerLane];
#pragma unroll
    for (int i = 0; i < kPicksPerLane; ++i)
    {
        int const t = min(i * kWaveSize + lane, a.B - 1);
        first[i] = a.cuSeqlens[t];
        end[i] = a.cuSeqlens[t + 1];
    }
    pin_args(a);
#pragma unroll
    for (int i = 0; i < kPicksPerLane; ++i)
    {
        bucket[i] = i * kWaveSize + lane < a.B ? len_bucket(end[i] - first[i]) : -1;
    }
    auto from = [&](int k) { // sequences of bucket k or a longer one
        int c = 0;
#pragma unroll
        for (int i = 0; i < kPicksPerLane; ++i)
        {
            c += __popcll(__ballot(bucket[i] >= k));
        }
        return c;
    };
    int k = 0;
#pragma unroll
    for (int bit = 32; bit > 0; bit >>= 1)
    {
        k = from(k + bit) > rank ? k + bit : k;
    }
    int off = rank - from(k + 1); // among the sequences of bucket k, by index
    SeqInfo s{};
    int len = 0;
    bOut = 0;
#pragma unroll
    for (int i = 0; i < kPicksPerLane; ++i)
    {
        uint64_t const m = __ballot(bucket[i] == k);
        int const c = __popcll(m);
        if (off >= 0 && off < c)
        {
            int const before = __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
            int const at = (int) __builtin_ctzll(__ballot(bucket[i] == k && before == off));
            bOut = i * kWaveSize + at;
            s.firstTok = __builtin_amdgcn_readlane(first[i], at);
            len = __builtin_amdgcn_readlane(end[i], at) - (int) s.firstTok;
        }
        off -= c;
    }
    s.seqBaseIn = s.firstTok * a.tokStrideIn;
    s.seqBaseOut = s.firstTok * a.tokStrideOut;
    s.nq = s.nk = min(max(len, 0), capacity);
    return s;
}

template <int THREADS>
__device__ inline SeqInfo pick_sequence_info(FmhaArgs const& a, int rank, int capacity, PickLds& l, int& bOut)
{
    if (a.cuSeqlens == nullptr || a.B > kMaxRanked || !(a.order & kRanked))
    {
        bOut = rank; // fixed layout (equal lengths), too many sequences, or a launch of a single round: natural order
        return seq_info(a, rank, capacity);
    }
    if (a.B <= kPicksPerLane * kWaveSize)
    {
        return pick_sequence_in_registers(a, rank, capacity, bOut);
    }
    if (threadIdx.x < kLenBuckets)
    {
        l.hist[threadIdx.x] = 0;
    }
    for (int t = threadIdx.x; t <= a.B; t += THREADS)
    {
        l.cu[t] = a.cuSeqlens[t];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < a.B; t += THREADS)
    {
        atomicAdd(&l.hist[len_bucket(l.cu[t + 1] - l.cu[t])], 1);
    }
    __syncthreads();
    // bucket that holds position `rank` (longest bucket first) and the offset inside it: lane k of every wavefront
    // takes bucket k, a prefix sum over the lanes gives the number of sequences in longer buckets, and the bucket is
    // the first one with no more than `rank` sequences above it (one LDS read and a few cross-lane steps instead of
    // a chain of dependent reads, one per bucket)
    int k, off;
    {
        int const lane = threadIdx.x & (kWaveSize - 1);
        int const mine = lane < kLenBuckets ? l.hist[lane] : 0;
        int incl = mine;
#pragma unroll
        for (int d = 1; d < kWaveSize; d *= 2)
        {
            int const up = __shfl_up(incl, d);
            incl += lane >= d ? up : 0;
        }
        int const total = __builtin_amdgcn_readlane(incl, kWaveSize - 1);
        int const above = total - incl; // sequences in buckets longer than this lane's
        uint64_t const fits = __ballot(lane < kLenBuckets && above <= rank);
        k = fits ? (int) __builtin_ctzll(fits) : 0;
        off = rank - __builtin_amdgcn_readlane(above, k);
    }
    // the off-th sequence (by index) of bucket k: every wavefront scans on its own
    int b = a.B - 1;
    int const lane = threadIdx.x & (kWaveSize - 1);
    for (int t0 = 0; t0 < a.B; t0 += kWaveSize)
    {
        int const t = t0 + lane;
        bool const in = t < a.B && len_bucket(l.cu[t + 1] - l.cu[t]) == k;
        uint64_t const m = __ballot(in);
        int const c = __popcll(m);
        if (off < c)
        {
            int const before = __popcll(m & ((1ull << lane) - 1ull));
            uint64_t const hit = __ballot(in && before == off);
            b = t0 + (int) __builtin_ctzll(hit);
            break;
        }
        off -= c;
    }
    bOut = b;
    SeqInfo s;
    int const first = l.cu[b];
    int const len = min(max(l.cu[b + 1] - first, 0), capacity);
    s.firstTok = first;
    s.seqBaseIn = (int64_t) first * a.tokStrideIn;
    s.seqBaseOut = (int64_t) first * a.tokStrideOut;
    s.nq = len;
    s.nk = len;
    return s;
}

// ------------------------------------------------------------------------------------------
// INT8, the usual case (cu_seqlens, a packed mask with holes or without, or no mask; scales that keep probabilities within
// INT8): specialised on the exact number of 64-key blocks so that a query tile is one straight-line instruction stream.
// ------------------------------------------------------------------------------------------

// The keys that a packed mask leaves a sequence: 64 of them in each m, their number up to the last one in sq.nk; true where
// keys before that one are masked.  By every wavefront for itself, one key per lane and block, in one trip to memory: no
// LDS, no barrier (FP16, 16 x 12 x 128: 6.2 us with the mask built in LDS by the workgroup, 5.7 us).  Masks that are a
// prefix, which is what the embedding layer packs, then cost no more than lengths do.  us per launch with the general
// kernel / with this: FP16 16 x 12 x 128 6.3 / 5.7, 64 x 12 x 128 14.6 / 12.3, 32 x 12 x 384 40.6 / 25.0; INT8 64 x 12 x 128
// 12.3 / 11.5, 8 x 12 x 384 14.8 / 12.2, 64 x 16 x 384 68.6 / 50.2.
template <int KT>
__device__ inline bool packed_mask_keys(FmhaArgs const& a, int b, SeqInfo& sq, uint64_t (&m)[KT])
{
    int const lane = threadIdx.x & (kWaveSize - 1);
    uint32_t const* const pm = a.packedMask + (int64_t) b * a.maskStrideWords;
    uint32_t word[KT], bit[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i)
    {
        // the layout that build_key_mask reads
        int const key = 64 * i + lane, ni = (int) (((uint32_t) key * a.spanInverse) >> 20), r = key - ni * 16 * a.warpsN;
        int const r2 = r & 15;
        bit[i] = (uint32_t) (8 * ni + (r2 & 1) + ((r2 & 8) ? 4 : 0));
        word[i] = key < sq.nk ? pm[(r >> 4) * a.warpsM * 32 + ((r2 & 7) >> 1)] : 0u;
    }
    int used = 0;
#pragma unroll
    for (int i = 0; i < KT; ++i)
    {
        m[i] = __ballot(((word[i] >> (bit[i] & 31u)) & 1u) != 0);
        used = m[i] ? 64 * i + 64 - __builtin_clzll(m[i]) : used;
    }
    sq.nk = used;
    bool holes = false;
#pragma unroll
    for (int i = 0; i < KT; ++i)
    {
        int const here = used - 64 * i;
        uint64_t const all = here >= 64 ? ~0ull : here > 0 ? (1ull << here) - 1ull : 0ull;
        holes = holes || m[i] != all;
    }
    return holes;
}

// Rows q0 .. of a sequence that has no key at all are zeros: `queries` of them by the whole workgroup.
template <int ESIZE>
__device__ inline void store_zero_rows(FmhaArgs const& a, SeqInfo const& sq, int n, int q0, int queries)
{
    int const end = min(q0 + queries, sq.nq) - q0;
    for (int i = threadIdx.x; i < end * 4 * ESIZE; i += blockDim.x)
    {
        *reinterpret_cast<u32x4*>(static_cast<uint8_t*>(a.out) + sq.seqBaseOut + (int64_t) (q0 + i / (4 * ESIZE)) * a.tokStrideOut
            + (int64_t) n * Lds<ESIZE>::kRow + (i % (4 * ESIZE)) * 16)
            = u32x4{0, 0, 0, 0};
    }
}

// Stage K and V of one (sequence, head): rows < nk from memory, the rest of the last block zero.
template <int KT, bool INTERLEAVED>
__device__ inline void stage_kv_prefix_i8(FmhaArgs const& a, int64_t seqBase, int64_t firstTok, int n, int nk, int nkb,
    uint8_t* sK, uint8_t* sV)
{
    constexpr int kRowsPerPass = kWavesI8 * kWaveSize / 4;   // 4 chunks of 16 bytes per 64-byte row
    constexpr int kPasses = 64 / kRowsPerPass;
    constexpr int kRow = Lds<1>::kRow;
    uint8_t const* src = static_cast<uint8_t const*>(a.qkv);
    int const chunk = threadIdx.x & 3;
    int const rowInPass = threadIdx.x >> 2;
    // one address per matrix for this lane's first row; every further row of the lane is a whole number of tokens
    // further on (the address arithmetic of a layout is done once, not once per load)
    uint8_t const* kSrc = src + qkv_chunk_offset<1, INTERLEAVED>(a, seqBase, firstTok, rowInPass, n, 1, chunk);
    uint8_t const* vSrc = src + qkv_chunk_offset<1, INTERLEAVED>(a, seqBase, firstTok, rowInPass, n, 2, chunk);
    int64_t const tokBytes = INTERLEAVED ? 32 : a.tokStrideIn;
    u32x4 kv[KT][kPasses], vv[KT][kPasses];
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
    {
#pragma unroll
        for (int p = 0; p < kPasses; ++p)
        {
            int const key = kb * 64 + p * kRowsPerPass + rowInPass;
            kv[kb][p] = u32x4{0, 0, 0, 0};
            vv[kb][p] = u32x4{0, 0, 0, 0};
            if (key < nk)
            {
                int64_t const step = (int64_t) (kb * 64 + p * kRowsPerPass) * tokBytes;
                kv[kb][p] = *reinterpret_cast<u32x4 const*>(kSrc + step);
                vv[kb][p] = *reinterpret_cast<u32x4 const*>(vSrc + step);
            }
        }
    }
    // LDS positions: a block is 64 rows further on; the swizzle depends on the row inside the block only
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
    {
        if (kb < nkb)
        {
#pragma unroll
            for (int p = 0; p < kPasses; ++p)
            {
                int const kk = p * kRowsPerPass + rowInPass;
                int const vk = v_row<1>(kk);
                *reinterpret_cast<u32x4*>(sK + kb * 64 * kRow + kk * kRow + swz<1>(kk, chunk) * 16) = kv[kb][p];
                *reinterpret_cast<u32x4*>(sV + kb * 64 * kRow + vk * kRow + swz<1>(vk, chunk) * 16) = vv[kb][p];
            }
        }
    }
}

// One 16-query tile of a sequence of exactly NKB key blocks (the last one ragged): query tile qt of the sequence sq,
// head n; qreg = the tile's Q^T operand (16 bytes d = 16g .. 16g+15 of query 16 qt + lane % 16, zero beyond the
// sequence).  sK / sV: the head's keys and values in LDS as stage_kv_prefix_i8 lays them out.
template <int NKB, bool INTERLEAVED, bool DEBUG>
__device__ __forceinline__ void tile_i8(FmhaArgs const& a, SeqInfo const& sq, int const b, int const n, int const qt,
    uint8_t const* sK, uint8_t const* sV, i32x4 const qreg, uint64_t const* const masks, bool const holes)
{
    constexpr int kRow = Lds<1>::kRow;
    constexpr int NT = NKB * 4;
    int const lane = threadIdx.x & (kWaveSize - 1);
    int const lq = lane & 15;
    int const g = lane >> 4;

    // last block: keys 64(NKB-1) + 16u + 4g + j exist for (16u + 4g + j) < lastKeys
    int const lastKeys = sq.nk - (NKB - 1) * 64;
    int const lastTiles = (lastKeys + 15) >> 4;
    i32x4 const seedFull = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    int const lastRel = lastKeys - 4 * g; // key 16u + j of this lane group exists iff 16u + j < lastRel

    int const q = qt * kQPerWave + lq;
    bool const qValid = q < sq.nq;

    // ---- S^T = K Q^T; the int32 result reads as binary32 12582912 + acc, -inf for absent keys
    i32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
    {
        int const key = t * 16 + lq;
        i32x4 const kreg = *reinterpret_cast<i32x4 const*>(sK + key * kRow + swz<1>(key, g) * 16);
        i32x4 seed = seedFull;
        if (t >= NT - 4)
        {
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                seed[j] = (16 * (t & 3) + j) < lastRel ? kMagicBits : kNegInfBits;
            }
        }
        acc[t] = attention_mfma_i8(kreg, qreg, seed);
    }
    if (holes)
    {
#pragma unroll
        for (int t = 0; t < NT; ++t)
        {
            uint32_t const bits = (uint32_t) (masks[t >> 2] >> (32 * ((t >> 1) & 1))) >> (16 * (t & 1) + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                acc[t][j] = (bits >> j) & 1u ? acc[t][j] : kNegInfBits;
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    if (DEBUG && a.dbgAcc1 && qValid)
    {
        for (int t = 0; t < NT; ++t)
        {
            for (int j = 0; j < 4; ++j)
            {
                int const key = t * 16 + g * 4 + j;
                if (key < sq.nk)
                {
                    a.dbgAcc1[(((int64_t) b * a.N + n) * a.S + q) * a.S + key] = acc[t][j] - kMagicBits;
                }
            }
        }
    }

    // ---- row max on the biased integers (monotone in the score; -inf is a negative pattern)
    // two chains of three-input maxima (v_max3_i32): one instruction per two scores
    int mxA = kNegInfBits, mxB = kNegInfBits;
#pragma unroll
    for (int t = 0; t < NT; ++t)
    {
        mxA = max(max(mxA, acc[t][0]), acc[t][1]);
        mxB = max(max(mxB, acc[t][2]), acc[t][3]);
    }
    int mx = max(mxA, mxB);
    mx = reduce_step<16>(mx, [](int x, int y) { return max(x, y); });
    mx = reduce_step<32>(mx, [](int x, int y) { return max(x, y); });
    __builtin_amdgcn_sched_barrier(0);

    // ---- e = 2^((acc - max) * c) in place, row sum
    float const negK0 = -__int_as_float(mx) * a.c;
    float sum0 = 0.f, sum1 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t)
    {
        if ((t & 3) == 0)
        {
            __builtin_amdgcn_sched_barrier(0); // bound the live temporaries to one key block
        }
        if (t >= NT - 4 && (t & 3) >= lastTiles)
        {
            continue; // tile without keys: its accumulators keep the -inf pattern (p8 = 0 below)
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            float const ev = __builtin_amdgcn_exp2f(fmaf(__int_as_float(acc[t][j]), a.c, negK0));
            acc[t][j] = __float_as_int(ev);
            if (j & 1)
            {
                sum1 += ev;
            }
            else
            {
                sum0 += ev;
            }
        }
    }
    float sum = sum0 + sum1;
    sum = reduce_step<16>(sum, [](float x, float y) { return x + y; });
    sum = reduce_step<32>(sum, [](float x, float y) { return x + y; });
    float const r = a.scaleSoftmax / sum;   // sum >= 1: the row maximum contributes 2^0

    // ---- p8 = rne(e * r), four keys to a dword; O^T = V^T P^T
    i32x4 oacc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
    {
        oacc[dt] = i32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
    {
        __builtin_amdgcn_sched_barrier(0);
        i32x4 preg = {0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            if (kb == NKB - 1 && u >= lastTiles)
            {
                continue;
            }
            uint32_t yb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                yb[j] = __float_as_uint(fmaf(__int_as_float(acc[kb * 4 + u][j]), r, kMagic));
            }
            uint32_t const lo = __builtin_amdgcn_perm(yb[1], yb[0], 0x0c0c0400u);
            uint32_t const hi = __builtin_amdgcn_perm(yb[3], yb[2], 0x0c0c0400u);
            preg[u] = (int) __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        }
        if (DEBUG && a.dbgP8 && qValid)
        {
            for (int u = 0; u < 4; ++u)
            {
                for (int j = 0; j < 4; ++j)
                {
                    int const key = kb * 64 + u * 16 + g * 4 + j;
                    if (key < sq.nk)
                    {
                        a.dbgP8[(((int64_t) b * a.N + n) * a.S + q) * a.S + key]
                            = (int8_t) ((uint32_t) preg[u] >> (8 * j));
                    }
                }
            }
        }
        int const vrow = kb * 64 + 8 * g + (lq >> 1);
        uint8_t const* vbase = sV + vrow * kRow + 8 * (lq & 1);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
        {
            int const sc = swz<1>(vrow, dt) * 16;
            i32x2 const v0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*) (vbase + sc));
            i32x2 const v1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*) (vbase + 32 * kRow + sc));
            i32x4 const vreg = {v0[0], v0[1], v1[0], v1[1]};
            oacc[dt] = attention_mfma_i8(vreg, preg, oacc[dt]);
        }
    }

    // ---- out8 = sat8(rne(acc2 * scale_bmm2)): binary32 product (rounded on its own, not fused
    //      into the add), rounded to an integer through the magic constant, clamped on the bit
    //      patterns (monotone for the positive results; anything negative is below the range).
    //      Lane (g, query) then holds bytes 4g..4g+3 of each 16-byte quarter dt of the query's row; a 4 x 4
    //      transpose over the four rows of 16 lanes (v_permlane32_swap, v_permlane16_swap) leaves it with the
    //      whole quarter dt = g, which goes out as one 16-byte store.
    uint32_t pk[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
    {
        uint32_t yb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            int const bits = __float_as_int(mul_rounded((float) oacc[dt][j], a.scaleBmm2) + kMagic);
            yb[j] = (uint32_t) min(max(bits, kMagicBits - 128), kMagicBits + 127);
        }
        uint32_t const lo = __builtin_amdgcn_perm(yb[1], yb[0], 0x0c0c0400u);
        uint32_t const hi = __builtin_amdgcn_perm(yb[3], yb[2], 0x0c0c0400u);
        pk[dt] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
    rows_transpose(pk);
    if (qValid)
    {
        uint8_t* dst = static_cast<uint8_t*>(a.out);
        int const d0 = g * 16;
        int64_t off;
        if (INTERLEAVED)
        {
            off = (((int64_t) n * 2 + (d0 >> 5)) * a.total + sq.firstTok + q) * 32 + (d0 & 31);
        }
        else
        {
            off = sq.seqBaseOut + (int64_t) q * a.tokStrideOut + (int64_t) n * kHeadSize + d0;
        }
        u32x4 const quarter = {pk[0], pk[1], pk[2], pk[3]};
        *reinterpret_cast<u32x4*>(dst + off) = quarter;
    }
}

// Q^T operand of query tile qt (see tile_i8).
template <bool INTERLEAVED>
__device__ __forceinline__ i32x4 load_q_i8(FmhaArgs const& a, SeqInfo const& sq, int const n, int const qt)
{
    int const lane = threadIdx.x & (kWaveSize - 1);
    int const qq = qt * kQPerWave + (lane & 15);
    i32x4 v = {0, 0, 0, 0};
    if (qq < sq.nq)
    {
        v = *reinterpret_cast<i32x4 const*>(static_cast<uint8_t const*>(a.qkv)
            + qkv_chunk_offset<1, INTERLEAVED>(a, sq.seqBaseIn, sq.firstTok, qq, n, 0, lane >> 4));
    }
    return v;
}

// All query tiles of this wavefront for a sequence of exactly NKB key blocks.
template <int NKB, bool INTERLEAVED, bool DEBUG>
__device__ __forceinline__ void attend_i8(FmhaArgs const& a, SeqInfo const& sq, int const b, int const n,
    int const qtBegin, int const qtEnd, uint8_t const* sK, uint8_t const* sV, i32x4 const qFirst, uint64_t const* const masks,
    bool const holes)
{
    int const wave = threadIdx.x >> 6;
    constexpr int qtStep = kWavesI8;
    i32x4 qnext = qFirst; // requested by the caller together with K and V
    for (int qt = qtBegin + wave; qt < qtEnd; qt += qtStep)
    {
        i32x4 const qreg = qnext;
        qnext = load_q_i8<INTERLEAVED>(a, sq, n, qt + qtStep);
        tile_i8<NKB, INTERLEAVED, DEBUG>(a, sq, b, n, qt, sK, sV, qreg, masks, holes);
    }
}

// MASKED: the keys come from a packed mask (a kernel of its own: the other one keeps its registers).
template <int KT, bool INTERLEAVED, bool DEBUG, bool MASKED = false>
__global__ __launch_bounds__(kWavesI8* kWaveSize) __attribute__((amdgpu_waves_per_eu(KT <= 6 ? 3 : 2))) void fmha_i8_prefix_kernel(
    TRTAMD_FMHA_LEADING_PARAMS, FmhaArgs const rest)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* sK = smem;
    uint8_t* sV = smem + Lds<1>::matBytes(KT);
    __shared__ PickLds sPick;
    FmhaArgs const a = TRTAMD_FMHA_ARGS_OF(rest);
    uint32_t const bid = id_of_workgroup(blockIdx.x, order);
    UnitPart up = unit_of_workgroup(bid, B * N * qSplit, a.partDiv);
    if (!INTERLEAVED && a.qSplit == 1 && (a.N & 1) == 0)
    {
        // Linear layout ([token][head][Q K V][64 bytes]): V of head n and Q of head n + 1 lie in one 128-byte line, so
        // the two heads of a pair go to one XCD (18239 tokens x 16 heads: 36.2 -> 35.2 us)
        UnitPart const pair = unit_of_workgroup(bid, B * N * qSplit, 2);
        up.unit = pair.unit * 2u + (uint32_t) pair.part;
    }
    int const part = up.part;
    uint32_t const rank = up.unit / a.headDiv;
    int const n = (int) (up.unit - rank * a.headDiv.d);
    int b;
    SeqInfo sq = pick_sequence_info<kWavesI8 * kWaveSize>(a, (int) rank, KT * 64, sPick, b);
    // contiguous tile ranges, each a multiple of one round of the workgroup's wavefronts
    int const nqt = (sq.nq + kQPerWave - 1) / kQPerWave;
    int const per = kWavesI8 * (int) ((uint32_t) ((nqt + kWavesI8 * a.qSplit - 1) / kWavesI8) / a.partDiv);
    int const qtBegin = min(part * per, nqt);
    int const qtEnd = min(qtBegin + per, nqt);
    if (qtBegin >= qtEnd)
    {
        return; // no query tile for this workgroup (also: empty sequence)
    }
    uint64_t masks[KT] = {};
    bool holes = false;
    if constexpr (MASKED)
    {
        holes = packed_mask_keys<KT>(a, b, sq, masks);
        if (sq.nk == 0)
        {
            store_zero_rows<1>(a, sq, n, qtBegin * kQPerWave, (qtEnd - qtBegin) * kQPerWave);
            return;
        }
    }
    int const nkb = (sq.nk + 63) >> 6;
    // the first query tile of this wavefront travels with K and V
    i32x4 qFirst = {0, 0, 0, 0};
    {
        int const qq = (qtBegin + (int) (threadIdx.x >> 6)) * kQPerWave + (int) (threadIdx.x & 15);
        if (qq < sq.nq && qtBegin + (int) (threadIdx.x >> 6) < qtEnd)
        {
            qFirst = *reinterpret_cast<i32x4 const*>(static_cast<uint8_t const*>(a.qkv)
                + qkv_chunk_offset<1, INTERLEAVED>(a, sq.seqBaseIn, sq.firstTok, qq, n, 0, (threadIdx.x & 63) >> 4));
        }
    }
    stage_kv_prefix_i8<KT, INTERLEAVED>(a, sq.seqBaseIn, sq.firstTok, n, sq.nk, nkb, sK, sV);
    __syncthreads();
    switch (nkb)
    {
    case 1: attend_i8<1, INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes); break;
    case 2:
        if (KT >= 2) attend_i8<(KT >= 2 ? 2 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 3:
        if (KT >= 3) attend_i8<(KT >= 3 ? 3 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 4:
        if (KT >= 4) attend_i8<(KT >= 4 ? 4 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 5:
        if (KT >= 5) attend_i8<(KT >= 5 ? 5 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 6:
        if (KT >= 6) attend_i8<(KT >= 6 ? 6 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 7:
        if (KT >= 7) attend_i8<(KT >= 7 ? 7 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    case 8:
        if (KT >= 8) attend_i8<(KT >= 8 ? 8 : 1), INTERLEAVED, DEBUG>(a, sq, b, n, qtBegin, qtEnd, sK, sV, qFirst, masks, holes);
        break;
    default: break;
    }
}

// ------------------------------------------------------------------------------------------
// FP16
// ------------------------------------------------------------------------------------------
template <int KT, bool DEBUG>
__global__ __launch_bounds__(kWavesF16* kWaveSize) void fmha_f16_kernel(FmhaArgs const a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* sK = smem;
    uint8_t* sV = smem + Lds<2>::matBytes(KT);
    uint32_t* sMask = reinterpret_cast<uint32_t*>(sV + Lds<2>::matBytes(KT));
    constexpr int kRow = Lds<2>::kRow;

    __shared__ int sLens[kMaxRanked + 1];
    UnitPart const up = unit_of_workgroup(blockIdx.x, gridDim.x, a.qSplit);
    int const part = up.part;
    int const n = up.unit % a.N;
    int const b = pick_sequence<kWavesF16 * kWaveSize>(a, up.unit / a.N, sLens);
    SeqInfo const sq = seq_info(a, b, KT * 64);
    int const nqt = (sq.nq + kQPerWave - 1) / kQPerWave;
    if (part * kWavesF16 >= nqt)
    {
        return;
    }
    build_key_mask(a, b, sq.nk, sMask);
    __syncthreads();
    int const nkUsed = used_keys(sMask, sq.nk);
    int const nkb = (nkUsed + 63) >> 6;
    stage_kv<2, KT, false, kWavesF16>(a, sq.seqBaseIn, sq.firstTok, n, nkUsed, nkb, sMask, sK, sV);
    __syncthreads();

    int const lane = threadIdx.x & (kWaveSize - 1);
    int const wave = threadIdx.x >> 6;
    int const lq = lane & 15;
    int const g = lane >> 4;
    uint8_t const* src = static_cast<uint8_t const*>(a.qkv);
    f16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i)
    {
        ones[i] = (f16) 1.f;
    }

    // Q^T operands of a tile: MFMA h covers d = 32h + 8g .. +7 of query 16*qt + lq.  The next
    // tile's operands are requested while the current tile is computed.
    auto load_q = [&](int qt, int h) -> f16x8 {
        int const qq = qt * kQPerWave + lq;
        u32x4 raw = {0, 0, 0, 0};
        if (qq < sq.nq)
        {
            raw = *reinterpret_cast<u32x4 const*>(
                src + qkv_chunk_offset<2, false>(a, sq.seqBaseIn, sq.firstTok, qq, n, 0, h * 4 + g));
        }
        return __builtin_bit_cast(f16x8, raw);
    };
    int const qtStep = a.qSplit * kWavesF16;
    f16x8 qnext[2] = {load_q(part * kWavesF16 + wave, 0), load_q(part * kWavesF16 + wave, 1)};
    for (int qt = part * kWavesF16 + wave; qt < nqt; qt += qtStep)
    {
        int const q = qt * kQPerWave + lq;
        bool const qValid = q < sq.nq;
        f16x8 const qreg[2] = {qnext[0], qnext[1]};
        qnext[0] = load_q(qt + qtStep, 0);
        qnext[1] = load_q(qt + qtStep, 1);

        // ---- S^T = K Q^T (binary32 accumulation) -----------------------------------------------
        f32x4 acc[KT * 4];
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
                uint32_t const w0 = __builtin_amdgcn_readfirstlane(sMask[kb * 2]);
                uint32_t const w1 = __builtin_amdgcn_readfirstlane(sMask[kb * 2 + 1]);
                bool const full = (w0 & w1) == 0xffffffffu;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    int const key = kb * 64 + u * 16 + lq;
                    f32x4 s = {0.f, 0.f, 0.f, 0.f};
                    if (!full)
                    {
                        asm volatile("" ::: "memory"); // scalar branch, taken for the ragged last block only
                        s = __builtin_bit_cast(f32x4, mask_seed(w0, w1, u, g, 0));
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                    {
                        f16x8 const kreg
                            = *reinterpret_cast<f16x8 const*>(sK + key * kRow + swz<2>(key, h * 4 + g) * 16);
                        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kreg, qreg[h], s, 0, 0, 0);
                    }
                    acc[kb * 4 + u] = s;
                }
            }
        }

        if (DEBUG && a.dbgAcc1 && qValid)
        {
#pragma unroll
            for (int kb = 0; kb < KT; ++kb)
            {
                if (kb < nkb)
                {
                    for (int u = 0; u < 4; ++u)
                    {
                        for (int j = 0; j < 4; ++j)
                        {
                            int const key = kb * 64 + u * 16 + g * 4 + j;
                            if (key < nkUsed)
                            {
                                a.dbgAcc1[(((int64_t) b * a.N + n) * a.S + q) * a.S + key]
                                    = __float_as_int(acc[kb * 4 + u][j]);
                            }
                        }
                    }
                }
            }
        }

        // ---- row max (masked keys hold -infinity) ------------------------------------------------
        float mx = -__builtin_inff();
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    mx = fmaxf(mx, fmaxf(fmaxf(acc[kb * 4 + u][0], acc[kb * 4 + u][1]),
                                         fmaxf(acc[kb * 4 + u][2], acc[kb * 4 + u][3])));
                }
            }
        }
        mx = reduce_step<16>(mx, [](float x, float y) { return fmaxf(x, y); });
        mx = reduce_step<32>(mx, [](float x, float y) { return fmaxf(x, y); });

        // ---- p = 2^((s - max) * c) rounded to binary16; O^T = V^T P^T; the row sum is taken by
        //      the matrix unit as well (a tile of ones), so numerator and denominator see the
        //      same rounded probabilities ---------------------------------------------------------
        float const negK0 = mx == -__builtin_inff() ? 0.f : -mx * a.c; // fully masked row: every p = 0
        f32x4 oacc[4];
        f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
        {
            oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int kb = 0; kb < KT; ++kb)
        {
            if (kb < nkb)
            {
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) // 32-key half of the block
                {
                    f16x8 preg;
#pragma unroll
                    for (int w = 0; w < 2; ++w)
                    {
                        int const t = kb * 4 + hb * 2 + w;
                        float p[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                        {
                            p[j] = __builtin_amdgcn_exp2f(fmaf(acc[t][j], a.c, negK0));
                        }
                        f16x2 const p01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(p[0], p[1]));
                        f16x2 const p23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(p[2], p[3]));
                        preg[w * 4 + 0] = p01[0];
                        preg[w * 4 + 1] = p01[1];
                        preg[w * 4 + 2] = p23[0];
                        preg[w * 4 + 3] = p23[1];
                    }
                    // V^T operand: lane r of a group addresses LDS row (4 keys per read: r/4) at
                    // halfword 16dt + 4(r%4); the transpose read hands lane i the 4 keys of head
                    // dim 16dt + i.  Slots 0..3 = keys 16(2hb)+4g.., slots 4..7 = keys 16(2hb+1)+4g..
                    int const vrow = kb * 64 + hb * 32 + 4 * g + (lq >> 2);
                    uint8_t const* vbase = sV + vrow * kRow + 8 * (lq & 1);
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt)
                    {
                        // rows vrow and vrow + 16 share row & 7, hence the swizzled chunk
                        int const sc = swz<2>(vrow, 2 * dt + ((lq >> 1) & 1)) * 16;
                        i16x4 const v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) (vbase + sc));
                        i16x4 const v1
                            = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) (vbase + 16 * kRow + sc));
                        typedef short i16x8 __attribute__((ext_vector_type(8)));
                        i16x8 const both = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                        oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(f16x8, both), preg, oacc[dt], 0, 0, 0);
                    }
                    sacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, preg, sacc, 0, 0, 0);
                }
            }
        }

        {
            float const rinv = sacc[0] > 0.f ? 1.f / sacc[0] : 0.f;
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
            {
                f16x4 y;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    y[j] = (f16) (oacc[dt][j] * rinv);
                }
                u32x2 const w = __builtin_bit_cast(u32x2, y);
                lo[dt] = w[0];
                hi[dt] = w[1];
            }
            rows_transpose(lo);
            rows_transpose(hi);
            if (qValid)
            {
                uint8_t* dst = static_cast<uint8_t*>(a.out);
                int64_t const off
                    = sq.seqBaseOut + (int64_t) q * a.tokStrideOut + ((int64_t) n * kHeadSize + g * 16) * 2;
                u32x4 const first = {lo[0], hi[0], lo[1], hi[1]};
                u32x4 const second = {lo[2], hi[2], lo[3], hi[3]};
                *reinterpret_cast<u32x4*>(dst + off) = first;
                *reinterpret_cast<u32x4*>(dst + off + 16) = second;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// FP16, launches with too few workgroups for 128 queries each (route_of), and any with at most 64 keys, on cu_seqlens or a packed
// mask (with holes too): the same specialisation, but K and V take turns in LDS, one block of V in the place of each block of K as
// soon as every wavefront has multiplied it.  48 KB for 384 keys instead of 96 KB: three workgroups of four wavefronts share a CU, so
// that one computes while another waits for its sequence, its K or its V, and a unit's queries are shared out 64 at a time over as
// many workgroups.  What bounds either kernel is that wait; with one workgroup per CU nothing covered it.  All of Q, K and V come by
// direct-to-LDS loads, whose number in flight the waits below count; a wavefront requests 16 rows of every block.  12 heads, sequences
// of a third of the length to the length, that kernel / this one, us per plugin call: 32 x 128 keys 12.5 / 5.8, 128 x 256 41.7 / 37.5,
// 32 x 384 19.8 / 19.6, 128 x 384 71.7 / 64.6, 16 x 512 22.8 / 19.5.  What is left is the L2: K and V of a unit are read once for every
// 64 queries, 133 MB for the 35.8 MB of 32 x 384.
// WHOLE: launches so small that a CU has room for all of it (kWholeWorkgroups); K, V and Q of sequences of up to kWholeBlocks
// blocks are requested together then.
// ------------------------------------------------------------------------------------------
constexpr int kQueriesF16 = kWavesF16T * kQPerWave;
__device__ u32x4 const kZeroRow[8] = {}; // 64 binary16 zeros, in memory

template <int N, int I = 0, typename F>
__device__ __forceinline__ void for_each_block(F&& f)
{
    if constexpr (I < N)
    {
        f(std::integral_constant<int, I>{});
        for_each_block<N, I + 1>(f);
    }
}

// Launches of no more workgroups than CUs, each with a CU's LDS to itself, have K, V and 64 queries of a sequence there at once:
// nothing waits for a place, which takes one or two trips to the L2 out of the chain.  With five blocks of keys and more a CU takes
// longer to bring it all in than it waits otherwise, so longer sequences of such a launch go in turns.  In turns / so, graph
// replays, us, means over 1 to 250 sequences and 1 to 16 heads: all of 64 keys 3.75 / 3.59, of 128 4.23 / 4.24, of 192 4.78 / 4.74,
// of 256 5.24 / 5.23, of 320 5.93 / 6.00, of 384 6.55 / 6.76; up to 64 of the 384 keys that the kernel has room for 3.77 / 3.65.
// With more workgroups than CUs it would keep others off them: 8 x 180 5.08 / 5.25, 4 x 384 6.66 / 8.95.
constexpr int64_t kWholeWorkgroups = 256;
constexpr int kWholeBlocks = 4;
constexpr int kWholeCapacity = 6; // blocks that the kernels of such launches have room for at most

template <int NKB, bool DEBUG, bool WHOLE>
__device__ __forceinline__ void attend_f16_turns(
    FmhaArgs const& a, SeqInfo const& sq, int const b, int const n, int const q0, uint8_t* const lds,
    uint64_t const* const masks, bool const holes)
{
    constexpr int kRow = Lds<2>::kRow;
    constexpr int NT = NKB * 4;
    int const lane = threadIdx.x & (kWaveSize - 1);
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const lq = lane & 15;
    int const g = lane >> 4;
    uint32_t const ldsBase = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) lds;
    uint8_t const* const unit = static_cast<uint8_t const*>(a.qkv) + sq.seqBaseIn + (int64_t) n * 3 * kRow;
    uint32_t const stride = (uint32_t) a.tokStrideIn;

    // 16 rows of matrix `mat` from `row` on into the LDS rows from `to` on; unless complete, those at or behind `limit` as
    // the last one, or for V as zeros: 0, the weight of such a key, times an infinite V would not be 0
    int const r8 = lane >> 3;
    uint32_t const chunk = (uint32_t) (((lane & 7) ^ r8) * 16); // the swizzle of swz<2>, on the source side
    uint32_t const whole = (uint32_t) r8 * stride + chunk;
    auto request = [&](int mat, int row, int limit, int to, bool complete) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            int const first = complete ? row + 8 * i : min(row + 8 * i, limit - 1);
            uint8_t const* const src = unit + (int64_t) first * a.tokStrideIn + mat * kRow;
            uint32_t const dst = ldsBase + (to + 8 * i) * kRow;
            uint32_t off = whole;
            if (!complete && row + 8 * i + 8 > limit)
            {
                if (mat == 2)
                {
                    load_to_lds16(row + 8 * i + r8 < limit ? src + whole : reinterpret_cast<uint8_t const*>(kZeroRow) + chunk, dst);
                    continue;
                }
                off = (uint32_t) min(r8, limit - 1 - first) * stride + chunk;
            }
            load_to_lds16_sbase(src, off, dst);
        }
    };
    constexpr int kRowV = WHOLE ? NKB * 64 : 0; // V's first row in LDS
    auto request_block = [&](int mat, int kb) {
        request(mat, kb * 64 + wave * 16, sq.nk, (mat == 2 ? kRowV : 0) + kb * 64 + wave * 16, kb < NKB - 1);
    };

    int const qw = q0 + wave * kQPerWave; // this wavefront's first query
    bool const active = qw < sq.nq;       // if not, it only brings in its rows
    // Q passes through the place of this wavefront's rows of the last block; WHOLE: it has one of its own
    int const qRow = (WHOLE ? 2 * NKB : NKB - 1) * 64 + wave * 16;
    request(0, qw, sq.nq, qRow, false);
#pragma unroll
    for (int kb = 0; kb < (WHOLE ? NKB : NKB - 1); ++kb)
    {
        request_block(1, kb);
    }
    if constexpr (WHOLE)
    {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
        {
            request_block(2, kb);
        }
    }
    wait_vmcnt<WHOLE ? 4 * NKB : 2 * (NKB - 1)>();
    f16x8 qreg[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        qreg[h] = *reinterpret_cast<f16x8 const*>(lds + (qRow + lq) * kRow + swz<2>(lq, h * 4 + g) * 16);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(qreg[0]), "+v"(qreg[1])::"memory"); // read before it is overwritten
    if constexpr (!WHOLE)
    {
        request_block(1, NKB - 1);
    }

    int const lastKeys = sq.nk - (NKB - 1) * 64;
    int const lastHalves = (lastKeys + 31) >> 5;   // 32-key halves of the last block that hold keys
    int const lastRel = lastKeys - 4 * g;          // key 16u + j of this lane group exists iff 16u + j < lastRel

    // ---- S^T = K Q^T (binary32 accumulation); absent keys start from -infinity
    f32x4 acc[NT];
    auto scores = [&](auto block) {
        constexpr int kb = decltype(block)::value;
        // in flight behind block kb: the later blocks of K and V of the blocks before kb - 1; WHOLE: and all of V
        wait_vmcnt<2 * (NKB - 1 - kb + (WHOLE ? NKB : kb > 0 ? kb - 1 : 0))>();
        __syncthreads(); // everybody's rows of block kb have landed, and everybody has read block kb - 1
        if constexpr (kb > 0 && !WHOLE)
        {
            request_block(2, kb - 1);
        }
        if (active)
        {
#pragma unroll
            for (int t = kb * 4; t < kb * 4 + 4; ++t)
            {
                int const key = t * 16 + lq;
                f32x4 sd = {0.f, 0.f, 0.f, 0.f};
                if (kb == NKB - 1 && 16 * (t & 3) + 16 > lastKeys) // uniform: a tile that is not all there
                {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        sd[j] = (16 * (t & 3) + j) < lastRel ? 0.f : -__builtin_inff();
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
                {
                    f16x8 const kreg = *reinterpret_cast<f16x8 const*>(lds + key * kRow + swz<2>(key, h * 4 + g) * 16);
                    sd = attention_mfma_f16(kreg, qreg[h], sd);
                }
                acc[t] = sd;
            }
            if (holes)
            {
#pragma unroll
                for (int t = kb * 4; t < kb * 4 + 4; ++t)
                {
                    uint32_t const bits = (uint32_t) (masks[kb] >> (32 * ((t >> 1) & 1))) >> (16 * (t & 1) + 4 * g);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        acc[t][j] = (bits >> j) & 1u ? acc[t][j] : -__builtin_inff();
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for_each_block<NKB>(scores);
    if constexpr (!WHOLE)
    {
        __syncthreads();
        request_block(2, NKB - 1);
    }

    int const q = qw + lq;
    bool const qValid = q < sq.nq;
    if (DEBUG && a.dbgAcc1 && qValid)
    {
        for (int t = 0; t < NT; ++t)
        {
            for (int j = 0; j < 4; ++j)
            {
                int const key = t * 16 + g * 4 + j;
                if (key < sq.nk)
                {
                    a.dbgAcc1[(((int64_t) b * a.N + n) * a.S + q) * a.S + key] = __float_as_int(acc[t][j]);
                }
            }
        }
    }

    // ---- row max
    float negK0 = 0.f;
    __builtin_amdgcn_sched_barrier(0);
    if (active)
    {
        float mxA = -__builtin_inff(), mxB = -__builtin_inff();
#pragma unroll
        for (int t = 0; t < NT; ++t)
        {
            mxA = fmaxf(fmaxf(mxA, acc[t][0]), acc[t][1]);
            mxB = fmaxf(fmaxf(mxB, acc[t][2]), acc[t][3]);
        }
        float mx = fmaxf(mxA, mxB);
        mx = reduce_step<16>(mx, [](float x, float y) { return fmaxf(x, y); });
        mx = reduce_step<32>(mx, [](float x, float y) { return fmaxf(x, y); });
        negK0 = a.packedMask && mx == -__builtin_inff() ? 0.f : -mx * a.c; // a mask's row without a score is zeros
    }

    // ---- p = 2^((s - max) * c) rounded to binary16; O^T = V^T P^T; row sum by a tile of ones
    f16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i)
    {
        ones[i] = (f16) 1.f;
    }
    f32x4 oacc[4];
    f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
    {
        oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto weigh = [&](auto block) {
        constexpr int kb = decltype(block)::value;
        wait_vmcnt<DEBUG ? 0 : 2 * (NKB - 1 - kb)>();
        __syncthreads();
        if (!active)
        {
            return;
        }
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
        {
            if (kb == NKB - 1 && hb >= lastHalves)
            {
                continue; // no key in this half
            }
            __builtin_amdgcn_sched_barrier(0);
            f16x8 preg;
#pragma unroll
            for (int w = 0; w < 2; ++w)
            {
                int const t = kb * 4 + hb * 2 + w;
                float pr[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    pr[j] = __builtin_amdgcn_exp2f(fmaf(acc[t][j], a.c, negK0));
                }
                f16x2 const p01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(pr[0], pr[1]));
                f16x2 const p23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(pr[2], pr[3]));
                preg[w * 4 + 0] = p01[0];
                preg[w * 4 + 1] = p01[1];
                preg[w * 4 + 2] = p23[0];
                preg[w * 4 + 3] = p23[1];
            }
            int const vrow = kRowV + kb * 64 + hb * 32 + 4 * g + (lq >> 2);
            uint8_t const* vbase = lds + vrow * kRow + 8 * (lq & 1);
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
            {
                int const sc = swz<2>(vrow, 2 * dt + ((lq >> 1) & 1)) * 16;
                i16x4 const v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) (vbase + sc));
                i16x4 const v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) (vbase + 16 * kRow + sc));
                typedef short i16x8 __attribute__((ext_vector_type(8)));
                i16x8 const both = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                oacc[dt] = attention_mfma_f16(__builtin_bit_cast(f16x8, both), preg, oacc[dt]);
            }
            sacc = attention_mfma_f16(ones, preg, sacc);
        }
    };
    for_each_block<NKB>(weigh);

    // Lane (g, query) holds 8 bytes of each 32-byte quarter dt of the query's 128-byte row; a 4 x 4 transpose over
    // the four rows of 16 lanes (v_permlane32_swap, v_permlane16_swap, once for each dword) leaves it with the
    // whole quarter dt = g, which goes out as two 16-byte stores.
    if (active)
    {
        float const rinv = a.packedMask && !(sacc[0] > 0.f) ? 0.f : 1.f / sacc[0];
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
        {
            f16x4 y;
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                y[j] = (f16) (oacc[dt][j] * rinv);
            }
            u32x2 const w = __builtin_bit_cast(u32x2, y);
            lo[dt] = w[0];
            hi[dt] = w[1];
        }
        rows_transpose(lo);
        rows_transpose(hi);
        if (qValid)
        {
            uint8_t* dst = static_cast<uint8_t*>(a.out);
            int64_t const off = sq.seqBaseOut + (int64_t) q * a.tokStrideOut + ((int64_t) n * kHeadSize + g * 16) * 2;
            u32x4 const first = {lo[0], hi[0], lo[1], hi[1]};
            u32x4 const second = {lo[2], hi[2], lo[3], hi[3]};
            *reinterpret_cast<u32x4*>(dst + off) = first;
            *reinterpret_cast<u32x4*>(dst + off + 16) = second;
        }
    }
}

template <int KT, bool DEBUG, bool WHOLE>
__global__ __launch_bounds__(kWavesF16T* kWaveSize)
    __attribute__((amdgpu_waves_per_eu(KT <= 4 ? 4 : KT <= 6 ? 3 : 2))) void fmha_f16_turns_kernel(
    TRTAMD_FMHA_LEADING_PARAMS, FmhaArgs const rest)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ PickLds sPick;
    FmhaArgs const a = TRTAMD_FMHA_ARGS_OF(rest);
    uint32_t const bid = KT <= 2 ? blockIdx.x : id_of_workgroup(blockIdx.x, order);
    UnitPart const up = unit_of_workgroup(bid, B * N * qSplit, a.partDiv);
    uint32_t const rank = up.unit / a.headDiv;
    int const n = __builtin_amdgcn_readfirstlane((int) (up.unit - rank * a.headDiv.d));
    int const q0 = __builtin_amdgcn_readfirstlane(up.part) * kQueriesF16;
    int b;
    SeqInfo sq = pick_sequence_info<kWavesF16T * kWaveSize>(a, (int) rank, KT * 64, sPick, b);
    // the same in every lane, which the compiler cannot see where they come from LDS: scalars keep the addresses scalar
    b = __builtin_amdgcn_readfirstlane(b);
    sq.nq = __builtin_amdgcn_readfirstlane(sq.nq);
    sq.nk = __builtin_amdgcn_readfirstlane(sq.nk);
    sq.firstTok = __builtin_amdgcn_readfirstlane((int) sq.firstTok);
    if (a.cuSeqlens)
    {
        sq.seqBaseIn = sq.firstTok * a.tokStrideIn;
        sq.seqBaseOut = sq.firstTok * a.tokStrideOut;
    }
    else
    {
        sq.seqBaseIn = b * a.seqStrideIn;
        sq.seqBaseOut = b * a.seqStrideOut;
    }
    if (q0 >= sq.nq)
    {
        return;
    }
    uint64_t masks[KT] = {};
    bool holes = false;
    if (a.packedMask)
    {
        holes = packed_mask_keys<KT>(a, b, sq, masks);
        if (sq.nk == 0)
        {
            store_zero_rows<2>(a, sq, n, q0, kQueriesF16);
            return;
        }
    }
    switch ((sq.nk + 63) >> 6)
    {
#define TRTAMD_BLOCKS(NKB)                                                                                             \
    case NKB:                                                                                                          \
        if constexpr (KT >= NKB)                                                                                       \
            attend_f16_turns<NKB, DEBUG, WHOLE && NKB <= kWholeBlocks>(a, sq, b, n, q0, smem, masks, holes);           \
        break
        TRTAMD_BLOCKS(1);
        TRTAMD_BLOCKS(2);
        TRTAMD_BLOCKS(3);
        TRTAMD_BLOCKS(4);
        TRTAMD_BLOCKS(5);
        TRTAMD_BLOCKS(6);
        TRTAMD_BLOCKS(7);
        TRTAMD_BLOCKS(8);
#undef TRTAMD_BLOCKS
    default: break;
    }
}

// ------------------------------------------------------------------------------------------
// FP16, launches that fill the chip, on cu_seqlens or a packed mask (with holes too): 32 queries per wavefront, K and V in
// blocks of 64 keys through two slots of LDS, the softmax kept up from block to block.  A workgroup takes 128 queries, so K and
// V come from the L2 half as often as above (32 x 384: 78 MB read there with Q, where the kernel above reads 133), every
// fragment read from LDS serves twice the queries, and 36 KB let four workgroups share a CU.
// The weights are relative to a running maximum that is only moved when it would be passed by more than a factor of 2^8,
// which they and their binary32 sums hold without loss: a branch that is rarely taken after the first block.  What bounds it
// is issue, and what does not overlap of it: per wavefront and block 512 cycles of matrix instructions, as many of exponentials
// and 400 of other vector work, of 2180 that pass (32 x 384, counters: vector ALU 45 %, matrix pipe 23 % of the launch, its
// start and tail among the rest); with the matrix instructions left out launches take 15 to 23 % less.  12 heads, sequences of a third of the length to the length, the
// kernels it took the place of / this one, us: 32 x 256 keys 13.9 / 13.1, 32 x 384 21.6 / 19.0, 128 x 256 36.5 / 33.2,
// 64 x 384 35.8 / 32.8, 16 x 512 22.7 / 18.0, 16 heads x 128 x 384 98.5 / 82.4, 128 x 512 145 / 134.
// ------------------------------------------------------------------------------------------
constexpr int kWavesStream = 4;
constexpr int kStreamQueries = 32; // per wavefront
constexpr int kStreamBlock = 64 * Lds<2>::kRow;     // bytes of 64 rows of K or V
constexpr int kStreamStage = 2 * kStreamBlock;
constexpr int kStreamLds = 2 * kStreamStage;

template <bool DEBUG>
__global__ __launch_bounds__(kWavesStream* kWaveSize) __attribute__((amdgpu_waves_per_eu(4))) void fmha_f16_stream_kernel(
    TRTAMD_FMHA_LEADING_PARAMS, FmhaArgs const rest, int const capacity)
{
    constexpr int kRow = Lds<2>::kRow;
    constexpr int kLoads = 2 * 8 / kWavesStream; // direct loads per wavefront and block: 8 rows each, of K and of V
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ PickLds sPick;
    __shared__ uint64_t sMask[8];
    FmhaArgs const a = TRTAMD_FMHA_ARGS_OF(rest);
    uint32_t const bid = id_of_workgroup(blockIdx.x, order);
    UnitPart const up = unit_of_workgroup(bid, B * N * qSplit, a.partDiv);
    uint32_t const rank = up.unit / a.headDiv;
    int const n = __builtin_amdgcn_readfirstlane((int) (up.unit - rank * a.headDiv.d));
    int b;
    SeqInfo sq = pick_sequence_info<kWavesStream * kWaveSize>(a, (int) rank, capacity, sPick, b);
    // the same in every lane, which the compiler cannot see where they come from LDS: scalars keep the addresses scalar
    b = __builtin_amdgcn_readfirstlane(b);
    int const nq = __builtin_amdgcn_readfirstlane(sq.nq);
    int const firstTok = __builtin_amdgcn_readfirstlane((int) sq.firstTok);
    int64_t const baseIn = a.cuSeqlens ? firstTok * a.tokStrideIn : b * a.seqStrideIn;
    int64_t const baseOut = a.cuSeqlens ? firstTok * a.tokStrideOut : b * a.seqStrideOut;
    int const lane = threadIdx.x & (kWaveSize - 1);
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const q0 = __builtin_amdgcn_readfirstlane(up.part) * (kWavesStream * kStreamQueries);
    if (q0 >= nq)
    {
        return;
    }
    bool holes = false;
    if (a.packedMask)
    {
        uint64_t masks[8];
        holes = packed_mask_keys<8>(a, b, sq, masks);
        if (threadIdx.x == 0) // read behind the barrier before block 0
        {
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                sMask[i] = masks[i];
            }
        }
        if (sq.nk == 0)
        {
            store_zero_rows<2>(a, sq, n, q0, kWavesStream * kStreamQueries);
            return;
        }
    }
    int const nk = __builtin_amdgcn_readfirstlane(sq.nk);
    int const qw = q0 + wave * kStreamQueries; // this wavefront's first query
    bool const active = qw < nq;               // if not, it only brings in its rows
    int const lq = lane & 31, h = lane >> 5;
    uint32_t const ldsBase = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) lds;
    uint8_t const* const unit = static_cast<uint8_t const*>(a.qkv) + baseIn + (int64_t) n * 3 * kRow;
    uint32_t const stride = (uint32_t) a.tokStrideIn;

    // 8 rows of matrix `mat` from `row` on to LDS byte `to`; unless complete, those at or behind `limit` as the last one, or
    // for V as zeros: 0, the weight of such a key, times an infinite V would not be 0
    int const r8 = lane >> 3;
    uint32_t const chunk = (uint32_t) (((lane & 7) ^ r8) * 16); // the swizzle of swz<2>, on the source side
    uint32_t const whole = (uint32_t) r8 * stride + chunk;
    auto request = [&](int mat, int row, int limit, int to, bool complete) {
        int const first = complete ? row : min(row, limit - 1);
        uint8_t const* const src = unit + (int64_t) first * a.tokStrideIn + mat * kRow;
        uint32_t const dst = ldsBase + (uint32_t) to;
        uint32_t off = whole;
        if (!complete && row + 8 > limit)
        {
            if (mat == 2)
            {
                load_to_lds16(row + r8 < limit ? src + whole : reinterpret_cast<uint8_t const*>(kZeroRow) + chunk, dst);
                return;
            }
            off = (uint32_t) min(r8, limit - 1 - first) * stride + chunk;
        }
        load_to_lds16_sbase(src, off, dst);
    };
    int const nb = (nk + 63) >> 6;
    // A block that is all there: one address, advanced from block to block (a wavefront that waits for its own scalar
    // arithmetic here is late with the next block and everything behind it).
    uint64_t const step8 = (uint64_t) (8 * kWavesStream) * stride;
    uint64_t kNext = reinterpret_cast<uint64_t>(unit) + (uint64_t) (8 * wave) * stride + kRow;
    auto request_block = [&](int kb, int slot) {
        uint32_t const to = (uint32_t) (slot * kStreamStage + wave * 8 * kRow);
        if (kb * 64 + 64 <= nk)
        {
#pragma unroll
            for (int i = 0; i < kLoads / 2; ++i)
            {
                void const* const src = reinterpret_cast<void const*>(kNext + i * step8);
                load_to_lds16_sbase(src, whole, ldsBase + to + (uint32_t) (i * kWavesStream * 8 * kRow));
                load_to_lds16_sbase(src, whole + kRow, ldsBase + to + (uint32_t) (kStreamBlock + i * kWavesStream * 8 * kRow));
            }
            kNext += 64ull * stride;
            return;
        }
#pragma unroll
        for (int i = 0; i < kLoads / 2; ++i)
        {
            int const r = (i * kWavesStream + wave) * 8;
            request(1, kb * 64 + r, nk, slot * kStreamStage + r * kRow, false);
            request(2, kb * 64 + r, nk, slot * kStreamStage + kStreamBlock + r * kRow, false);
        }
    };

    // Q passes through the second slot
    static_assert(kWavesStream * kStreamQueries * kRow <= kStreamStage, "Q in a slot");
    int const qAt = kStreamStage + wave * kStreamQueries * kRow;
#pragma unroll
    for (int i = 0; i < kStreamQueries / 8; ++i)
    {
        request(0, qw + 8 * i, nq, qAt + 8 * i * kRow, false);
    }
    request_block(0, 0);
    wait_vmcnt<kLoads>();
    asm volatile("" ::: "memory");
    f16x8 qreg[4]; // B operand: query lq, elements 16 s + 8 h .. + 7
#pragma unroll
    for (int s = 0; s < 4; ++s)
    {
        qreg[s] = *reinterpret_cast<f16x8 const*>(lds + qAt + lq * kRow + swz<2>(lq, 2 * s + h) * 16);
    }

    f32x16 out[2]; // O^T: elements 32 d + 8 (v / 4) + 4 h + v % 4 of query lq
#pragma unroll
    for (int v = 0; v < 16; ++v)
    {
        out[0][v] = out[1][v] = 0.f;
    }
    float negMax = 0.f;  // -maximum * c of the scores that the weights are relative to
    float sum[2] = {0.f, 0.f}; // of this lane's keys, in two chains
    int const tr = (lane & 15) >> 2; // transposing reads: 16 lanes take 4 rows of 16 elements
    int const trBase = (4 * h + tr) * kRow + (lane & 1) * 8;
    int const trChunk = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);

    for (int kb = 0; kb < nb; ++kb)
    {
        wait_vmcnt<0>();
        __syncthreads(); // everybody's rows of block kb have landed, and everybody has read block kb - 1 (and Q)
        uint8_t const* const sK = lds + (kb & 1) * kStreamStage;
        uint8_t const* const sV = sK + kStreamBlock;
        auto request_next = [&] {
            if (kb + 1 < nb)
            {
                request_block(kb + 1, (kb + 1) & 1);
            }
        };
        if (!active)
        {
            request_next();
            continue;
        }
        int const keys = nk - kb * 64; // of this block, 64 and more: all
        // ---- S^T = K Q^T: keys 32 t + 8 (v / 4) + 4 h + v % 4 of query lq
        f32x16 acc[2];
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            acc[0][v] = acc[1][v] = 0.f;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
        {
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                int const key = 32 * t + lq;
                f16x8 const kreg = *reinterpret_cast<f16x8 const*>(sK + key * kRow + swz<2>(key, 2 * s + h) * 16);
                acc[t] = attention_mfma_f16_32(kreg, qreg[s], acc[t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        request_next(); // while the matrix instructions run
        __builtin_amdgcn_sched_barrier(0);
        if (DEBUG && a.dbgAcc1 && qw + lq < nq)
        {
            for (int v = 0; v < 32; ++v)
            {
                int const key = kb * 64 + 32 * (v >> 4) + 8 * ((v & 15) >> 2) + 4 * h + (v & 3);
                if (key < nk)
                {
                    a.dbgAcc1[(((int64_t) b * a.N + n) * a.S + qw + lq) * a.S + key] = __float_as_int(acc[v >> 4][v & 15]);
                }
            }
        }
        if (keys < 64) // uniform: absent keys weigh nothing
        {
#pragma unroll
            for (int v = 0; v < 32; ++v)
            {
                int const key = 32 * (v >> 4) + 8 * ((v & 15) >> 2) + (v & 3);
                acc[v >> 4][v & 15] = key < keys - 4 * h ? acc[v >> 4][v & 15] : -__builtin_inff();
            }
        }
        if (holes)
        {
#pragma unroll
            for (int v = 0; v < 32; v += 4)
            {
                uint32_t const bits = (uint32_t) (sMask[kb] >> (2 * v)) >> (4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    acc[v >> 4][(v & 15) + j] = (bits >> j) & 1u ? acc[v >> 4][(v & 15) + j] : -__builtin_inff();
                }
            }
        }
        float mxA = fmaxf(acc[0][0], acc[0][1]), mxB = fmaxf(acc[1][0], acc[1][1]);
#pragma unroll
        for (int v = 2; v < 16; v += 2)
        {
            mxA = fmaxf(fmaxf(mxA, acc[0][v]), acc[0][v + 1]);
            mxB = fmaxf(fmaxf(mxB, acc[1][v]), acc[1][v + 1]);
        }
        float const mx = reduce_step<32>(fmaxf(mxA, mxB), [](float x, float y) { return fmaxf(x, y); });
        // finite, whatever the scale is, so that a block whose scores are all -infinity weighs nothing
        float const negNew = fminf(-mx * a.c, 3.402823466e+38f);
        if (kb == 0)
        {
            negMax = negNew;
        }
        else if (__ballot(negNew < negMax - 8.f) != 0)
        {
            // Weights may grow to 2^8 before the sums so far are brought to the new maximum.
            float const to = fminf(negNew, negMax);
            float const f = __builtin_amdgcn_exp2f(to - negMax);
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                out[0][v] *= f;
                out[1][v] *= f;
            }
            sum[0] *= f;
            sum[1] *= f;
            negMax = to;
        }
        // ---- p = 2^(s * c - max * c) rounded to binary16; O^T = V^T P^T
#pragma unroll
        for (int t = 0; t < 2; ++t)
        {
            if (t == 1 && keys <= 32)
            {
                break; // no key in this half
            }
#pragma unroll
            for (int w = 0; w < 2; ++w)
            {
                f16x8 preg;
#pragma unroll
                for (int j = 0; j < 8; j += 2)
                {
                    float const p0 = __builtin_amdgcn_exp2f(fmaf(acc[t][8 * w + j], a.c, negMax));
                    float const p1 = __builtin_amdgcn_exp2f(fmaf(acc[t][8 * w + j + 1], a.c, negMax));
                    f16x2 const pp = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(p0, p1));
                    f16x2 const ones = {(f16) 1.f, (f16) 1.f};
                    sum[(j >> 1) & 1] = __builtin_amdgcn_fdot2(pp, ones, sum[(j >> 1) & 1], false);
                    preg[j] = pp[0];
                    preg[j + 1] = pp[1];
                }
#pragma unroll
                for (int d = 0; d < 2; ++d)
                {
                    int const row = 32 * t + 16 * w + 4 * h + tr;
                    uint8_t const* const v0 = sV + (32 * t + 16 * w) * kRow + trBase + swz<2>(row, 4 * d + trChunk) * 16;
                    i16x4 const lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) v0);
                    i16x4 const hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*) (v0 + 8 * kRow));
                    typedef short i16x8 __attribute__((ext_vector_type(8)));
                    i16x8 const both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    out[d] = attention_mfma_f16_32(__builtin_bit_cast(f16x8, both), preg, out[d]);
                }
            }
        }
    }

    // The two lanes of a query hold four consecutive elements in turn; after two swaps per 32 elements each has 16 of them.
    if (active)
    {
        float const total = reduce_step<32>(sum[0] + sum[1], [](float x, float y) { return x + y; });
        float const rinv = a.packedMask && !(total > 0.f) ? 0.f : 1.f / total; // a mask's row without a score is zeros
        uint8_t* const dst = static_cast<uint8_t*>(a.out) + baseOut + (int64_t) (qw + lq) * a.tokStrideOut + (int64_t) n * kRow;
#pragma unroll
        for (int d = 0; d < 2; ++d)
        {
            u32x2 w[4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
            {
                f16x4 y;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    y[j] = (f16) (out[d][4 * g + j] * rinv);
                }
                w[g] = __builtin_bit_cast(u32x2, y);
            }
            auto const a0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[2][0], false, false);
            auto const a1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[2][1], false, false);
            auto const b0 = __builtin_amdgcn_permlane32_swap(w[1][0], w[3][0], false, false);
            auto const b1 = __builtin_amdgcn_permlane32_swap(w[1][1], w[3][1], false, false);
            u32x4 const first = {a0[0], a1[0], a0[1], a1[1]};
            u32x4 const second = {b0[0], b1[0], b0[1], b1[1]};
            if (qw + lq < nq)
            {
                *reinterpret_cast<u32x4*>(dst + d * 64 + h * 32) = first;
                *reinterpret_cast<u32x4*>(dst + d * 64 + h * 32 + 16) = second;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------

// Raising the dynamic LDS limit is a per-function attribute, set once per process and kernel: at the first launch,
// or ahead of it by trtamd_fused_mha_prepare.
int ensure_lds(void const* key, char const* name, int ldsBytes)
{
    static std::mutex mtx;
    static std::vector<void const*> done;
    std::lock_guard<std::mutex> lock(mtx);
    for (void const* p : done)
    {
        if (p == key)
        {
            return TRTAMD_STATUS_SUCCESS;
        }
    }
    hipError_t const e = hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, ldsBytes);
    if (e != hipSuccess)
    {
        (void) hipGetLastError();
        return set_error(TRTAMD_STATUS_FAILURE, "%s: cannot reserve %d bytes of LDS: %s", name, ldsBytes,
            hipGetErrorString(e));
    }
    done.push_back(key);
    return TRTAMD_STATUS_SUCCESS;
}

template <auto KERNEL>
int launch_fmha(char const* name, hipStream_t stream, FmhaArgs const& args, int ldsBytes, int waves)
{
    static std::atomic<bool> reserved{false}; // known without the lock from the second launch on
    if (!reserved.load(std::memory_order_acquire))
    {
        int const st = ensure_lds(reinterpret_cast<void const*>(KERNEL), name, ldsBytes);
        if (st != TRTAMD_STATUS_SUCCESS)
        {
            return st;
        }
        reserved.store(true, std::memory_order_release);
    }
    unsigned const blocks = (unsigned) args.B * args.N * args.qSplit;
    if constexpr (std::is_invocable_v<decltype(KERNEL), FmhaArgs>)
    {
        hipLaunchKernelGGL(KERNEL, dim3(blocks), dim3(waves * kWaveSize), ldsBytes, stream, args);
    }
    else
    {
        hipLaunchKernelGGL(KERNEL, dim3(blocks), dim3(waves * kWaveSize), ldsBytes, stream, TRTAMD_FMHA_LEADING_ARGS(args), args);
    }
    return check_launch(name);
}

int pick_kt(int s)
{
    for (int kt : {1, 2, 3, 4, 6, 8})
    {
        if (s <= kt * 64)
        {
            return kt;
        }
    }
    return 0;
}

template <bool DEBUG>
int run_i8(hipStream_t stream, FmhaArgs const& a, bool interleaved)
{
    int const kt = pick_kt(a.S);
    // probabilities cannot leave the INT8 range: the kernel specialised on the number of key blocks serves the launch
    int const noFast = tuning(Tuning::kFmhaGeneric);
    if (!a.clampP && !noFast)
    {
#define TRTAMD_I8P(KT)                                                                                                 \
    case KT:                                                                                                           \
        return a.packedMask ? launch_fmha<fmha_i8_prefix_kernel<KT, false, DEBUG, true>>("fmha_i8_masked", stream, a,  \
                   Lds<1>::total(KT), kWavesI8)                                                                        \
            : interleaved ? launch_fmha<fmha_i8_prefix_kernel<KT, true, DEBUG>>("fmha_i8_prefix_interleaved", stream, \
                   a, Lds<1>::total(KT), kWavesI8)                                                                     \
                           : launch_fmha<fmha_i8_prefix_kernel<KT, false, DEBUG>>("fmha_i8_prefix", stream, a,         \
                               Lds<1>::total(KT), kWavesI8)
        switch (kt)
        {
            TRTAMD_I8P(1);
            TRTAMD_I8P(2);
            TRTAMD_I8P(3);
            TRTAMD_I8P(4);
            TRTAMD_I8P(6);
            TRTAMD_I8P(8);
        default: break;
        }
#undef TRTAMD_I8P
    }
#define TRTAMD_I8(KT)                                                                                                  \
    case KT:                                                                                                           \
        return interleaved ? launch_fmha<fmha_i8_kernel<KT, true, DEBUG>>("fmha_i8_interleaved", stream, a,           \
                   Lds<1>::total(KT), kWavesI8)                                                                        \
                           : launch_fmha<fmha_i8_kernel<KT, false, DEBUG>>("fmha_i8", stream, a, Lds<1>::total(KT),    \
                               kWavesI8)
    switch (kt)
    {
        TRTAMD_I8(1);
        TRTAMD_I8(2);
        TRTAMD_I8(3);
        TRTAMD_I8(4);
        TRTAMD_I8(6);
        TRTAMD_I8(8);
    default: break;
    }
#undef TRTAMD_I8
    return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: sequence length %d exceeds 512", a.S);
}

// Which of the FP16 kernels a launch takes.
enum class F16Kernel
{
    kGENERAL, // TRTAMD_FMHA_GENERIC, and strides beyond the 32-bit offsets of the direct-to-LDS loads
    kTURNS,
    kSTREAM
};

bool is_whole(int kt, int64_t workgroups)
{
    return kt <= kWholeCapacity && workgroups <= kWholeWorkgroups;
}
constexpr int whole_lds(int kt)
{
    int const whole = std::min(kt, kWholeBlocks);
    return std::max(Lds<2>::matBytes(kt), 2 * Lds<2>::matBytes(whole) + kQueriesF16 * Lds<2>::kRow);
}

template <int KT, bool DEBUG>
int launch_turns(hipStream_t stream, FmhaArgs const& a)
{
    if constexpr (KT <= kWholeCapacity)
    {
        if (is_whole(KT, (int64_t) a.B * a.N * a.qSplit))
        {
            return launch_fmha<fmha_f16_turns_kernel<KT, DEBUG, true>>("fmha_f16_whole", stream, a, whole_lds(KT), kWavesF16T);
        }
    }
    return launch_fmha<fmha_f16_turns_kernel<KT, DEBUG, false>>("fmha_f16_turns", stream, a, Lds<2>::matBytes(KT), kWavesF16T);
}

template <bool DEBUG>
int run_f16(hipStream_t stream, FmhaArgs const& a, F16Kernel which)
{
    int const kt = pick_kt(a.S);
    if (which == F16Kernel::kSTREAM)
    {
        int const st = ensure_lds(reinterpret_cast<void const*>(fmha_f16_stream_kernel<DEBUG>), "fmha_f16_stream", kStreamLds);
        if (st)
        {
            return st;
        }
        hipLaunchKernelGGL((fmha_f16_stream_kernel<DEBUG>), dim3((uint32_t) a.B * (uint32_t) a.N * (uint32_t) a.qSplit),
            dim3(kWavesStream * kWaveSize), kStreamLds, stream, TRTAMD_FMHA_LEADING_ARGS(a), a, kt * 64);
        return check_launch("fmha_f16_stream");
    }
    if (which == F16Kernel::kTURNS)
    {
#define TRTAMD_F16T(KT)                                                                                                \
    case KT: return launch_turns<KT, DEBUG>(stream, a)
        switch (kt)
        {
            TRTAMD_F16T(1);
            TRTAMD_F16T(2);
            TRTAMD_F16T(3);
            TRTAMD_F16T(4);
            TRTAMD_F16T(6);
            TRTAMD_F16T(8);
        default: break;
        }
#undef TRTAMD_F16T
    }
#define TRTAMD_F16(KT)                                                                                                 \
    case KT: return launch_fmha<fmha_f16_kernel<KT, DEBUG>>("fmha_f16", stream, a, Lds<2>::total(KT), kWavesF16)
    switch (kt)
    {
        TRTAMD_F16(1);
        TRTAMD_F16(2);
        TRTAMD_F16(3);
        TRTAMD_F16(4);
        TRTAMD_F16(6);
        TRTAMD_F16(8);
    default: break;
    }
#undef TRTAMD_F16
    return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: sequence length %d exceeds 512", a.S);
}

// Every shipped kernel's LDS reservation, so that no later launch has anything to set up.
template <int KT>
int prepare_kt()
{
    int st = ensure_lds(reinterpret_cast<void const*>(fmha_i8_prefix_kernel<KT, true, false>), "fmha_i8_prefix_interleaved",
        Lds<1>::total(KT));

    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_i8_prefix_kernel<KT, false, false>), "fmha_i8_prefix",
                      Lds<1>::total(KT));
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_i8_prefix_kernel<KT, false, false, true>), "fmha_i8_masked",
                      Lds<1>::total(KT));
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_i8_kernel<KT, true, false>), "fmha_i8_interleaved",
                      Lds<1>::total(KT));
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_i8_kernel<KT, false, false>), "fmha_i8", Lds<1>::total(KT));
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_f16_turns_kernel<KT, false, false>), "fmha_f16_turns",
                      Lds<2>::matBytes(KT));
    if constexpr (KT <= kWholeCapacity)
    {
        st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_f16_turns_kernel<KT, false, true>), "fmha_f16_whole", whole_lds(KT));
    }
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_f16_kernel<KT, false>), "fmha_f16", Lds<2>::total(KT));
    return st;
}

float bits_to_float(uint32_t u)
{
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// binary16 (low half of a half2 bit pattern) to binary32
float half_bits_to_float(uint16_t h)
{
    uint32_t const sign = (uint32_t) (h & 0x8000u) << 16;
    uint32_t const exp = (h >> 10) & 0x1fu;
    uint32_t const man = h & 0x3ffu;
    if (exp == 0)
    {
        float const v = (float) man * 5.9604644775390625e-08f;
        return sign ? -v : v;
    }
    uint32_t const bits = exp == 31 ? (sign | 0x7f800000u | (man << 13)) : (sign | ((exp + 112u) << 23) | (man << 13));
    return bits_to_float(bits);
}

// INT8 units that are alike: of the padded layout, where every query row is computed and units differ by their masks only, and of a
// packed batch that is as good as padded, which the interleaved layout's strides show, since they are its number of tokens.
bool alike(trtamd_fmha_params const& p)
{
    return !p.cu_seqlens || (p.interleaved && p.qkv_stride_in_bytes >= ceil_div<int64_t>((int64_t) p.b * p.s * 15, 16));
}

// INT8: from how many (sequence, head) units on each has a workgroup of its own, by blocks of keys (one block always has).  Three
// workgroups of up to six blocks have room on a CU, two of more; every extra workgroup of a unit stages K and V again.
// Packed sequences: once rounds that go forwards and backwards even out units of different lengths, from 640 units of one or two
// blocks (672 units: one 6.7, two 7.4 us; 600: 6.4 / 6.0), 768 of three or four (192 keys: 9.0 / 10.0; 720 units: 10.9 / 9.9), 640
// of five (752 units: 15.8 / 18.3), 896 of six, 720 of more (440 keys: 26.9 / 29.2).  (Six by themselves: 900 units 28.5 / 26.2,
// 1152 31.5 / 32.6; but such launches are also halves of a pass on two streams, whose other half fills the idle CUs: 1008 and 1040
// units side by side, 24 layers, 11.94 ms a pass with one workgroup per unit, 12.05 with two for 1008.)
// Units that are alike: those that do not come in even halves, an odd number of tiles of 64 queries or 96 queries, from 641 on: one
// round up to 768 units, and hardly worse than halves beyond (alone / in two, us: 700 units of 96 keys 6.9 / 7.9, of 192 14.9 /
// 15.7, of 320 28.4 / 30.6; 800 of 96 7.8 / 8.8, of 320 35.1 / 34.6).  128 keys are even halves, but masks leave some units shorter:
// alone with them (700 units 1.06 to 1.10 of the speed, 800 1.02 to 1.10), in two without (800 units 10.3 / 9.9).  Even halves stay
// together up to 895 units (800 of 256 keys: alone 0.82 to 0.86 of the speed, of 384 0.87, of 512 0.88), beyond which the line is
// not at its best: halves are still 1.07 to 1.14 times as fast at 1152 units.
int64_t int8_alone_from(trtamd_fmha_params const& p, int blocks)
{
    if (!alike(p))
    {
        constexpr int kUnlike[] = {640, 640, 768, 768, 640, 896, 720, 720};
        return kUnlike[blocks - 1];
    }
    bool const uneven = blocks % 2 == 1 || p.s <= 96 || (blocks == 2 && p.packed_mask_ptr && !p.cu_seqlens);
    return uneven ? 641 : 896;
}

// INT8: workgroups per unit.  Below that line as many as fill a round of 768, two to four, but for five and six blocks of keys and
// more, whose workgroups are longer.
// Alike, padded, us: three from 193 units on (240 units, in three / in four: 320 keys 1.29 of the speed, 384 15.5 / 18.4; of 256 keys,
// padded, 0.95 to 0.98, packed 8.8 / 9.5; of 512 27.2 / 24.9), of six blocks two from 342 on, where three would be more than four
// workgroups per CU (300 units, in two / in three, 20.6 / 19.1, 352 21.1 / 22.0).
// Others, geometric means over lengths of a third of s to s, of less than a sixth of s, from one on and between: of five blocks three
// from 193 units on (226 units 1.09 times as fast as in four; of 256 keys 0.99), of more from 171 (206 units of 384 keys 1.10 times
// as fast, of 448 1.15, of 512 1.11).  Two of six blocks from 288 on (268 units 0.95 times as fast as in three, 288 0.99, 316 1.00,
// 356 1.06), of more from 320 (288 units of 448 keys 0.93, of 512 0.99; 316 0.98 and 0.99, 356 1.00 and 0.98; where lengths spread
// from a third of s, 288 and 316 units 1.06).
int int8_parts(trtamd_fmha_params const& p, int blocks)
{
    int64_t const units = (int64_t) p.b * p.h;
    if (units >= int8_alone_from(p, blocks))
    {
        return 1;
    }
    int three = 256, two = 384;
    if (alike(p))
    {
        three = blocks == 5 || blocks == 6 || (blocks == 4 && p.cu_seqlens) ? 193 : three;
        two = blocks == 6 ? 342 : two;
    }
    else if (blocks >= 5)
    {
        three = blocks == 5 ? 193 : 171;
        two = blocks == 5 ? two : blocks == 6 ? 288 : 320;
    }
    return units >= two ? 2 : units >= three ? 3 : 4;
}

// What a launch runs.
struct FmhaRoute
{
    F16Kernel f16;
    int parts;      // workgroups per (sequence, head) unit
    uint32_t order; // FmhaArgs.order
};

FmhaRoute route_of(int32_t dataType, trtamd_fmha_params const& p)
{
    int const kt = pick_kt(p.s);
    int const blocks = ceil_div(p.s, 64);
    // FP16: 128 queries per workgroup from so many of these workgroups on, by blocks of 64 keys; 64 of them and the scores of all
    // their keys in registers below.  The latter run in one round up to four, three or two of them per CU, as their LDS leaves
    // room (longer sequences need more of it each), and a second round costs more than the wider workgroups that leave some CUs
    // with two of them, others with three: the lines lie in or behind that second round, where means over lengths alike, of a third
    // of s to s, of less than a sixth of s, from one on and between turn over.  12 or 16 heads, sequences of a third of the length to
    // the length, us with 64 / with 128 queries: 64 x 128 keys 8.1 / 7.7, 48 x 128 7.8 / 8.1; 27 x 180 in the capacity of 256 8.0 /
    // 7.1, 21 x 180 6.7 / 6.9; 27 x 230 10.1 / 7.9, 21 x 230 7.8 / 7.9; 16 x 384 12.0 / 9.8, 13 x 345 9.4 / 9.8, 10 x 384 8.2 / 9.1;
    // 8 x 448 12.4 / 10.0, of one length 14.8 / 12.8, of up to 74 keys 4.6 / 5.0, from one on, 6 x 448, 16 heads, 7.9 / 9.4;
    // 10 x 512 14.3 / 10.8 (16 heads), 6 x 512 7.5 / 9.5.  Three blocks: 28 x 192, all of them, 9.9 / 11.0; up to 32 keys 4.3 / 4.7.
    // With one or two blocks of keys a second round of the wide ones is no better: 110 x 128 13.0 / 14.4, 225 x 128 24.8 / 29.9 (only
    // sequences of up to 21 of 128 keys are slower so, 126 x 128 8.8 / 7.8);
    // and a row of at most 64 keys leaves half of them idle: 64 x 64 4.5 / 5.3, 600 x 64 25.6 / 28.3.
    // Padded sequences, whose workgroups are alike but for masks, with 64 / with 128 queries: 20 x 192, 16 heads, 9.6 / 10.6; 20 x 256
    // 13.5 / 13.9, 28 x 256, 12 heads, 14.5 / 14.1; 9 x 384, 16 heads, 14.3 / 12.5, 10 x 384 11.0 / 11.6; 8 x 448 14.9 / 12.2; 8 x 512
    // 15.6 / 13.7.
    constexpr int kStreamFrom[2][8] = {{INT32_MAX, 768, 768, 544, 540, 504, 384, 360}, // packed
        {INT32_MAX, 768, 768, 768, 540, 432, 384, 360}};
    constexpr int kStreamTile = kWavesStream * kStreamQueries;
    int const streamParts = ceil_div(kt * 64, kStreamTile);
    FmhaRoute r{F16Kernel::kGENERAL, 1, 0};
    F16Kernel& f16 = r.f16;
    if (dataType == 1 && !tuning(Tuning::kFmhaGeneric)
        && p.qkv_stride_in_bytes < (1LL << 29)) // eight tokens within a 32-bit offset
    {
        int64_t const wide = (int64_t) p.b * p.h * streamParts;
        f16 = wide >= kStreamFrom[p.cu_seqlens ? 0 : 1][blocks - 1] && (blocks > 2 || wide <= 1024) ? F16Kernel::kSTREAM : F16Kernel::kTURNS;
    }
    // Workgroups per (sequence, head).  The general FP16 kernel (its K and V take most of a CU's LDS, one workgroup per CU, and
    // staging them is 40 % of a workgroup's time) shares a unit only below 160 of them (192 units of 192-384 keys: 15.3 us alone,
    // 17.5 us shared by two; 144 units: 14.9 against 12.9 us).  The other FP16 kernels take 64 or 128 queries each, of as many as
    // the kernel has room for: a sequence longer than s that still fits is served whole, as by the kernels that walk the queries.
    int const waves = dataType == 2 ? kWavesI8 : kWavesF16;
    int const maxSplit = std::max(1, ceil_div(ceil_div(p.s, kQPerWave), waves));
    int64_t const heads = (int64_t) p.b * p.h;
    int split = 1;
    if (dataType == 2)
    {
        split = int8_parts(p, blocks);
    }
    else if (f16 != F16Kernel::kGENERAL)
    {
        split = f16 == F16Kernel::kTURNS ? kt : streamParts;
    }
    else
    {
        while (split < maxSplit && heads * split < 160)
        {
            split *= 2;
        }
    }
    r.parts = f16 != F16Kernel::kGENERAL ? split : std::min(split, maxSplit);
    // tuning override: TRTAMD_FMHA_QSPLIT=<n> forces the number of workgroups per head
    int const forced = tuning(Tuning::kFmhaQsplit);
    if (forced > 0 && f16 == F16Kernel::kGENERAL)
    {
        r.parts = std::min(forced, maxSplit);
    }
    // The order in which sequences are served: the longest first costs a workgroup the ranking (0.25 us: a trip to LDS or a
    // few across the lanes before its loads) and evens out the CUs, or fills the tail of a launch of several rounds with
    // short ones.  Every other round backwards (id_of_workgroup) costs nothing.  12 or 16 heads, sequences of a third of
    // the length to the length:
    // - FP16, 128 queries per workgroup: all resident at once up to four per CU; longest first below 3072 of them
    //   (16 x 512 18.0 us against 21.2 in natural order, 32 x 384 19.0 / 20.4; 128 x 384, 16 heads, 85.6 / 82.4).  Every other
    //   round backwards where a unit has an even number of parts (32 x 180 9.3 -> 8.2, 96 x 180 19.2 -> 17.0, and in natural order
    //   128 x 180 31.9 -> 27.0, 128 x 256 40.0 -> 37.2, 16 heads).  Three parts are spread by themselves, but for launches of up
    //   to three workgroups per CU (13 x 384, 16 heads, 12.5 -> 12.1) or beyond one round (32 x 384 15.3 -> 14.8); between 768 and
    //   1024 of them lengths of up to 276 of 384 keys lose up to 9 % (19 x 276, 16 heads, 11.9 -> 13.0), short ones 7 %, and in
    //   natural order any lose 1 to 3 %.
    // - FP16, 64 queries: short enough to even out by themselves, natural order.  Rounds backwards with four blocks of keys
    //   (lengths from one on, 10 x 256, 16 heads, 6.8 -> 6.4) and with more than six (8 x 448, 12.4 -> 10.6), not with three or
    //   five (23 x 192 of up to 140 keys 6.5 -> 7.0; 10 x 320 of up to 230 6.7 -> 7.4).  Six blocks: longest first and backwards up
    //   to 767 workgroups, three per CU, all resident (8 x 384 9.8 -> 8.9, of one length 10.25 -> 10.54); beyond, a second round of
    //   long ones waits for the first (11 x 384 of 256 keys and more 12.1 -> 13.6, of less than 64 4.36 -> 4.64).
    // - INT8, two or three workgroups per CU at a time: longest first beyond one round of all CUs' places, and before that
    //   where the units are long enough for the ranking to pay, from 768 of them with three and four blocks of keys
    //   (32 x 180 7.3 -> 6.9), beyond 512 with five and more (14 x 310 9.5 -> 8.7, 16 x 384 12.2 -> 9.9).  Rounds go backwards
    //   where a unit has an even number of parts (32 x 384 16.4 -> 11.7, longest first alone 12.7; 24 x 512, 16 heads,
    //   25.4 -> 23.0) or one, up to four of them per CU or with one or two blocks of keys (70 x 100 6.1 -> 5.7, 64 x 160
    //   8.6 -> 8.0; beyond, 86 x 256 17.5 -> 18.8); three parts are spread by themselves (24 x 180 5.6 -> 6.1).  Beyond
    //   768, four parts of four blocks, a tile of queries each, are short enough without the ranking (13 x 256, 16 heads, 8.0 ->
    //   7.2), and units that are alike have nothing to rank, but parts of different lengths (34 x 192 of one length, 16 heads,
    //   1.06 times as fast backwards).
    int64_t const workgroups = (int64_t) p.b * p.h * r.parts;
    bool ranked, back;
    if (f16 == F16Kernel::kSTREAM)
    {
        ranked = workgroups < 3072;
        back = r.parts % 2 == 0 || workgroups < 768 || (ranked && workgroups > 1024);
    }
    else if (f16 == F16Kernel::kTURNS)
    {
        ranked = blocks == 6 && workgroups >= 512 && workgroups < 768;
        back = ranked || blocks == 4 || blocks > 6;
    }
    else
    {
        int64_t const lds = dataType == 2 ? Lds<1>::total(kt) : Lds<2>::total(kt);
        int64_t const perCu
            = std::max<int64_t>(1, std::min<int64_t>(dataType == 2 ? 3 : 2, (160 * 1024) / std::max<int64_t>(lds, 1)));
        int64_t const without = dataType != 2 || blocks <= 2 ? perCu * 256 : blocks >= 5 ? 512 : 767;
        bool const beyond = workgroups > without;
        bool const level = dataType == 2 && (alike(p) || (blocks == 4 && r.parts == 4 && workgroups > 768));
        ranked = beyond && !level;
        back = dataType == 2 && beyond && (r.parts == 1 ? !level && (blocks <= 2 || workgroups <= 1024) : r.parts % 2 == 0);
    }
    // tuning override: TRTAMD_FMHA_RANKED=0 forces natural order with every round forwards, 1 the longest-first order
    int const forcedRank = tuning(Tuning::kFmhaRanked);
    if (forcedRank >= 0)
    {
        ranked = forcedRank != 0;
        back = back && ranked;
    }
    // Padded sequences go in their own order, every round forwards: of one length they have nothing to even out (32 x 384 24.0 us
    // forwards, 24.1 backwards); masks of different lengths were not tried backwards.
    uint32_t const paired = back && p.cu_seqlens ? (uint32_t) std::min<int64_t>(workgroups, INT32_MAX) / kTwoRounds * kTwoRounds : 0;
    r.order = paired | (ranked ? kRanked : 0);
    return r;
}

int fused_mha_run(hipStream_t stream, int32_t dataType, trtamd_fmha_params const* p, int32_t* dbgAcc1, int8_t* dbgP8)
{
    if (!p)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: null parameter block");
    }
    if (dataType != 1 && dataType != 2)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: data type %d (only FP16=1 and INT8=2)", dataType);
    }
    if (p->d != kHeadSize)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: head size %d (only 64)", p->d);
    }
    if (p->b < 0 || p->h <= 0 || p->s <= 0)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: bad dimensions b=%d h=%d s=%d", p->b, p->h, p->s);
    }
    if (p->s > 512)
    {
        return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: sequence length %d exceeds 512", p->s);
    }
    if (p->b == 0)
    {
        return TRTAMD_STATUS_SUCCESS;
    }
    if (!p->qkv_ptr || !p->o_ptr)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: null tensor pointer");
    }
    if (!aligned16(p->qkv_ptr) || (reinterpret_cast<uintptr_t>(p->o_ptr) & 7u) != 0)
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: qkv must be 16-byte and output 8-byte aligned");
    }
    bool const interleaved = p->interleaved != 0;
    if (interleaved && (dataType != 2 || !p->cu_seqlens))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: interleaved layout needs INT8 and cu_seqlens");
    }
    int const esize = dataType == 2 ? 1 : 2;
    FmhaArgs a{};
    a.qkv = p->qkv_ptr;
    a.out = p->o_ptr;
    a.cuSeqlens = p->cu_seqlens;
    a.B = p->b;
    a.N = p->h;
    a.S = p->s;
    FmhaRoute const route = route_of(dataType, *p);
    a.qSplit = route.parts;
    a.order = route.order;
    a.partDiv = fast_div((uint32_t) a.qSplit);
    a.headDiv = fast_div((uint32_t) a.N);
    a.dbgAcc1 = dbgAcc1;
    a.dbgP8 = dbgP8;
    if (interleaved)
    {
        // strides carry the total token count (qkvToContextInt8InterleavedPlugin.cpp:280-281)
        if (p->qkv_stride_in_bytes <= 0 || p->qkv_stride_in_bytes != p->o_stride_in_bytes
            || p->qkv_stride_in_bytes > 0x7fffffffLL)
        {
            return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: interleaved strides must both equal the token count");
        }
        a.total = (int32_t) p->qkv_stride_in_bytes;
    }
    else
    {
        int64_t const rowIn = (int64_t) 3 * p->h * kHeadSize * esize;
        int64_t const rowOut = (int64_t) p->h * kHeadSize * esize;
        a.tokStrideIn = p->qkv_stride_in_bytes;
        a.tokStrideOut = p->o_stride_in_bytes;
        if (a.tokStrideIn < rowIn || a.tokStrideOut < rowOut || (a.tokStrideIn & 15) != 0 || (a.tokStrideOut & 7) != 0)
        {
            return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: strides %lld/%lld too small or misaligned",
                (long long) a.tokStrideIn, (long long) a.tokStrideOut);
        }
        if (!p->cu_seqlens)
        {
            // fixed [S,B,N,3,d]: the token stride spans B sequences (MHARunner::setup, mhaRunner.h:62-83)
            a.seqStrideIn = rowIn;
            a.seqStrideOut = rowOut;
            if (a.tokStrideIn < rowIn * p->b || a.tokStrideOut < rowOut * p->b)
            {
                return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: fixed layout strides do not span the batch");
            }
        }
    }
    if (!p->cu_seqlens && p->packed_mask_ptr)
    {
        int wm = p->warps_m, wn = p->warps_n;
        if (wm == 0 || wn == 0)
        {
            // FusedMHARunner{FP16,Int8}::mhaImpl::setup, mhaRunner.cu:676-692, 805-821
            if (p->s == 64 || p->s == 96 || p->s == 128)
            {
                wm = 2;
                wn = 2;
            }
            else if (p->s == 384)
            {
                wm = 1;
                wn = 8;
            }
            else
            {
                return set_error(TRTAMD_STATUS_NOT_SUPPORTED, "fused MHA: no packed-mask geometry for s=%d", p->s);
            }
        }
        a.packedMask = static_cast<uint32_t const*>(p->packed_mask_ptr);
        a.warpsM = wm;
        a.warpsN = wn;
        a.spanInverse = ((1u << 20) + 16u * (uint32_t) wn - 1u) / (16u * (uint32_t) wn);
        a.maskStrideWords = p->packed_mask_stride_in_bytes / 4;
        int const xn = ceil_div(p->s, 16 * wn);
        if (xn > 4 || a.maskStrideWords < (int64_t) wm * wn * 32)
        {
            return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA: packed mask geometry/stride inconsistent with s");
        }
    }
    if (dataType == 2)
    {
        float const s1 = bits_to_float(p->scale_bmm1);
        float const ss = bits_to_float(p->scale_softmax);
        float const s2 = bits_to_float(p->scale_bmm2);
        if (!(s1 > 0.f) || !(ss > 0.f) || !(s2 > 0.f))
        {
            return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA INT8: scales must be positive (%g, %g, %g)", s1, ss, s2);
        }
        a.c = s1 * kLog2e;
        a.scaleSoftmax = ss;
        a.scaleBmm2 = s2;
        a.clampP = ss > 127.f ? 1 : 0;
        return (dbgAcc1 || dbgP8) ? run_i8<true>(stream, a, interleaved) : run_i8<false>(stream, a, interleaved);
    }
    // FP16: scale_bmm1 is a half2 holding 1/sqrt(d) twice; softmax/bmm2 scales are 1 (mhaRunner.cu:694-701)
    float const s1 = half_bits_to_float((uint16_t) (p->scale_bmm1 & 0xffffu));
    if (!(s1 > 0.f))
    {
        return set_error(TRTAMD_STATUS_BAD_PARAM, "fused MHA FP16: scale_bmm1 must be positive (%g)", s1);
    }
    a.c = s1 * kLog2e;
    a.scaleSoftmax = 1.f;
    a.scaleBmm2 = 1.f;
    return dbgAcc1 ? run_f16<true>(stream, a, route.f16) : run_f16<false>(stream, a, route.f16);
}

} // namespace
} // namespace trtamd

using namespace trtamd;

extern "C" int trtamd_fused_mha_run(trtamd_stream_t stream, int32_t data_type, trtamd_fmha_params const* params)
{
    return fused_mha_run(as_stream(stream), data_type, params, nullptr, nullptr);
}

// Test hook (include/trtamd_test_hooks.h): same launch, additionally dumping the first GEMM's accumulators
// ([b][h][s][s], int32 for INT8, binary32 bit patterns for FP16) and, for INT8, the quantised probabilities.
extern "C" int trtamd_fused_mha_run_debug(trtamd_stream_t stream, int32_t data_type,
    trtamd_fmha_params const* params, int32_t* acc1, int8_t* p8)
{
    return fused_mha_run(as_stream(stream), data_type, params, acc1, p8);
}

extern "C" int64_t trtamd_test_fmha_route(int32_t data_type, trtamd_fmha_params const* p)
{
    if (!p || (data_type != 1 && data_type != 2) || p->b <= 0 || p->h <= 0 || !trtamd_fused_mha_is_valid(data_type, p->d, p->s))
    {
        return -1;
    }
    FmhaRoute const r = route_of(data_type, *p);
    bool const whole = r.f16 == F16Kernel::kTURNS && is_whole(pick_kt(p->s), (int64_t) p->b * p->h * r.parts);
    return (int64_t) (whole ? 3 : (int) r.f16) | r.parts << 4 | (int64_t) r.order << 8;
}

extern "C" int trtamd_fused_mha_prepare(void)
{
    int st = prepare_kt<1>();
    st = st ? st : prepare_kt<2>();
    st = st ? st : prepare_kt<3>();
    st = st ? st : prepare_kt<4>();
    st = st ? st : prepare_kt<6>();
    st = st ? st : prepare_kt<8>();
    st = st ? st : ensure_lds(reinterpret_cast<void const*>(fmha_f16_stream_kernel<false>), "fmha_f16_stream", kStreamLds);
    return st;
}

extern "C" int trtamd_fused_mha_is_valid(int32_t data_type, int32_t d, int32_t s)
{
    return (data_type == 1 || data_type == 2) && d == kHeadSize && s > 0 && s <= 512;
}
