// Binary32 attention in one launch with the keys of a query split between the wavefronts of a workgroup: the shapes of
// the unfused path (unfused_mha.hip) that attention_split_keys_takes names.
#include "device_utils.hpp"
#include "host_utils.hpp"
#include "unfused_mha.hpp"

#include <cmath>

namespace trtamd
{
namespace
{

// ------------------------------------------------------------------------------------------
// A workgroup owns 16 queries of one (batch, head).  Its four wavefronts take every fourth tile of 16 keys each, go
// through K and then V of those tiles, and keep a maximum, a sum of exponentials and an output of their own; these meet
// once, at the end, in LDS.  Bound by the binary32 matrix pipe (16 queries x 16 keys x 64 dimensions: 512 cycles of one
// SIMD for either product), so what counts is that every SIMD has work and that nothing waits between the products:
//   - work in tiles of 16 x 16: nothing is multiplied for queries beyond S or for whole tiles beyond the valid length,
//     and many short workgroups even out over the chip (64 queries per workgroup with all their keys in each
//     wavefront: 384 workgroups at S=197, B=8, N=12, a quarter of them with 5 queries in 64);
//   - the tiles left over by a division by four go to another SIMD in every workgroup;
//   - no barrier before the last one: a wavefront shares no stage with the others.  K (and Q) pass through its own part
//     of LDS, because 16-byte reads of fragments straight from memory take 16 rows at a time and a cache line for every
//     lane (S=197: 16.0 -> 13.5 us); V needs no transposition, see below;
//   - no address arithmetic in vector registers beside the products: offsets of the lanes are constant, those of the
//     tiles scalar (13.5 -> 10.7 us; 64-bit products for every row took as many cycles as half of the matrix work).
// Which dimension or key a step of a product takes is free as long as both operands agree:
//   Q K^T  step (t, i): dimension 16 t + 4 g + i;
//   P V    step i of a tile: key 4 g + i of it, where the scores of the first product lie.  In a whole block of 64
//          dimensions lane n reads 16 bytes of the row, dimensions 64 b + 4 n .. + 3, and element dt of them is row n
//          of output tile 4 b + dt: an output tile is every fourth dimension of the block, and its four neighbours make
//          16 bytes again on the way out.  The dimensions behind the last block come in tiles of 16 consecutive ones.
// d = 64, against 64 queries per workgroup: S=197 B=8 N=12 19.0 -> 10.7 us, S=300 B=8 N=12 27.5 -> 18.2, S=384 B=20 N=12
// 90 -> 65, S=1000 B=8 N=12 221 -> 127 (two passes before), S=1024 B=32 N=16 1853 -> 1098 us (125 TFLOP/s of the 145
// that a loop of nothing but these instructions reaches).  Two tiles of queries per workgroup (half the reads of K and
// V) are slower nearly everywhere, S=197: 12.9 us; more than two tiles in flight give nothing.
// ------------------------------------------------------------------------------------------
constexpr int kBlock = 256;
constexpr int kInFlight = 2; // tiles of K, then V, on their way to a wavefront
// The weights of up to 1024 keys, each at most 1, on their way to the division by their sum: smaller by a power of two, so
// that no value is rounded and a weighted sum of V does not overflow where the result is finite.
constexpr float kDown = 1.f / 1024.f;

// Wavefronts per SIMD that the registers are to leave room for, without spills.
constexpr int split_waves(int const KD, int const NT)
{
    return KD <= 4 || KD * NT <= 40 ? 4 : KD * NT <= 80 ? 3 : 2;
}

template <int KD, int NT>
__global__ __launch_bounds__(kBlock, split_waves(KD, NT)) void attention_split_keys_kernel(int const S, int const heads,
    int const strips, float const wl2, float const* __restrict__ qkv, uint32_t const rowBytes,
    int32_t const* __restrict__ maskIdx, float* __restrict__ out, int64_t const ldOut)
{
    constexpr int d = 16 * KD;
    constexpr int kBlocks = KD / 4;     // whole blocks of 64 dimensions
    constexpr int kPitch = d + 4;       // floats per row in LDS: the 16-byte reads down a column are free of conflicts
    constexpr int kQueries = 16;
    constexpr int D = kInFlight;
    // a wavefront's own rows: its tile of Q or K on the way from whole rows to fragments, and its output at the end
    __shared__ __attribute__((aligned(16))) float lds[4][kQueries * kPitch];
    __shared__ float rowMax[4][kQueries], rowSum[4][kQueries];

    UnitPart const up = unit_of_workgroup(blockIdx.x, gridDim.x, strips); // parts of a unit share an XCD's L2
    int const z = (int) up.unit;        // batch * heads + head
    int const lane = threadIdx.x & (kWaveSize - 1);
    int const n = lane & 15, g = lane >> 4;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const own = lds[wave];
    int valid = S;
    if (maskIdx)
    {
        valid = max(0, min(S, maskIdx[z / heads]));
    }
    int const tiles = (valid + 15) / 16;
    int const turn = (wave + up.part + z) & 3; // this wavefront's tiles: turn, turn + 4, ...
    int const mine = (tiles - turn + 3) / 4;
    auto exists = [&](int const u) { return u < 2 * NT && (u < NT ? u : u - NT) < mine; };

    // The unit's rows of Q, K and V, d elements each side by side, rowBytes apart.  Offsets are 32 bits: the part that
    // depends on the lane never changes, the part that depends on the tile is the same for all lanes.  A tile that
    // would reach beyond the last row starts 16 rows before the end instead.
    auto const rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(qkv + (int64_t) z * 3 * d), 0, (int) 0xffffffffu, 0x00027000);
    auto first_row = [&](int const tile) { return min(16 * tile, S - 16); };
    // 16 rows as they lie in memory, 16 bytes per lane: consecutive lanes take consecutive pieces of a row
    constexpr int kPieces = 4 * KD; // per row
    constexpr bool kWholeRows = kWaveSize % kPieces == 0;
    uint32_t rowOffset[kWholeRows ? 1 : KD];
#pragma unroll
    for (int j = 0; j < (kWholeRows ? 1 : KD); ++j)
    {
        int const p = lane + kWaveSize * j;
        rowOffset[j] = p / kPieces * rowBytes + p % kPieces * 16;
    }
    auto fetch_rows = [&](f32x4(&dst)[KD], int const part, int const row0)
    {
#pragma unroll
        for (int j = 0; j < KD; ++j)
        {
            uint32_t const row = row0 + (kWholeRows ? kWaveSize / kPieces * j : 0);
            dst[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                rows, rowOffset[kWholeRows ? 0 : j] + part * d * 4, row * rowBytes, 0));
        }
    };
    // those rows in fragment order, through this wavefront's part of LDS: dst[t] = dimensions 16 t + 4 g .. of row n
    auto fragments = [&](f32x4(&dst)[KD], f32x4 const(&src)[KD])
    {
#pragma unroll
        for (int j = 0; j < KD; ++j)
        {
            int const p = lane + kWaveSize * j;
            *reinterpret_cast<f32x4*>(own + p / kPieces * kPitch + p % kPieces * 4) = src[j];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < KD; ++t)
        {
            dst[t] = *reinterpret_cast<f32x4 const*>(own + n * kPitch + 16 * t + 4 * g);
        }
        __builtin_amdgcn_wave_barrier();
    };
    f32x4 ring[D][KD];
    uint32_t const blockOffset = 4 * g * rowBytes + 16 * n, tileOffset = 4 * g * rowBytes + 4 * n;
    // item u of this wavefront: K of its tile u, behind those V of its tile u - NT
    auto fetch = [&](f32x4(&dst)[KD], int const u)
    {
        if (u < NT)
        {
            fetch_rows(dst, 1, first_row(4 * u + turn));
        }
        else
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                uint32_t const row = first_row(4 * (u - NT) + turn) + i;
#pragma unroll
                for (int b = 0; b < kBlocks; ++b)
                {
                    dst[4 * b + i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                        rows, blockOffset + (2 * d + 64 * b) * 4, row * rowBytes, 0));
                }
#pragma unroll
                for (int dt = 4 * kBlocks; dt < KD; ++dt)
                {
                    dst[dt][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        rows, tileOffset + (2 * d + 16 * dt) * 4, row * rowBytes, 0));
                }
            }
        }
    };

    f32x4 qf[KD];
    fetch_rows(qf, 0, first_row(up.part));
#pragma unroll
    for (int u = 0; u < D; ++u)
    {
        if (exists(u))
        {
            fetch(ring[u], u);
        }
    }
    fragments(qf, qf);

    // ---- S^T = K Q^T: element i of tile u's accumulator is key 16 (4 u + turn) + 4 g + i of query n -------------
    f32x4 acc[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u)
    {
        if (exists(u))
        {
            f32x4 kf[KD];
            fragments(kf, ring[u % D]);
            acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < KD; ++t)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][i], qf[t][i], acc[u], 0, 0, 0);
                }
            }
        }
        if (exists(u + D))
        {
            fetch(ring[u % D], u + D);
        }
    }

    // ---- softmax over this wavefront's keys: exp((x - max) w) as one fma per score, the way the reference's kernel
    // forms it; a masked key gets minus infinity, whose exponential is 0 whatever the maximum (which stays finite, so that
    // the fma does not subtract infinities where every valid score is one) -----------------------------------------
    float mx = -3.402823466e38f;
#pragma unroll
    for (int u = 0; u < NT; ++u)
    {
        if (exists(u))
        {
            f32x4 x = acc[u];
            int const tile = 4 * u + turn;
            if (16 * tile + 16 > valid) // the ragged tile (uniform branch)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    int const key = first_row(tile) + 4 * g + i;
                    x[i] = key >= 16 * tile && key < valid ? x[i] : -__builtin_inff();
                }
                acc[u] = x;
            }
            mx = fmaxf(fmaxf(mx, fmaxf(x[0], x[1])), fmaxf(x[2], x[3]));
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    float const nmx = -mx * wl2;
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < NT; ++u)
    {
        if (exists(u))
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                float const e = __builtin_amdgcn_exp2f(fmaf(acc[u][i], wl2, nmx));
                acc[u][i] = e * kDown;
                sum += e;
            }
        }
    }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (g == 0)
    {
        rowMax[wave][n] = mx;
        rowSum[wave][n] = sum;
    }

    // ---- O^T = V^T P^T over this wavefront's keys ---------------------------------------------------------------
    f32x4 o[KD];
#pragma unroll
    for (int dt = 0; dt < KD; ++dt)
    {
        o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = NT; u < 2 * NT; ++u)
    {
        if (exists(u))
        {
            int const before = 16 * (4 * (u - NT) + turn) - first_row(4 * (u - NT) + turn);
            if (before > 0) // uniform: rows of the tile in front of this one, which count there; 0 times infinity is no 0
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    bool const own = 4 * g + i >= before;
#pragma unroll
                    for (int b = 0; b < kBlocks; ++b)
                    {
                        ring[u % D][4 * b + i] = own ? ring[u % D][4 * b + i] : f32x4{0.f, 0.f, 0.f, 0.f};
                    }
#pragma unroll
                    for (int dt = 4 * kBlocks; dt < KD; ++dt)
                    {
                        ring[u % D][dt][i] = own ? ring[u % D][dt][i] : 0.f;
                    }
                }
            }
#pragma unroll
            for (int dt = 0; dt < KD; ++dt)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    float const v = dt < 4 * kBlocks ? ring[u % D][dt / 4 * 4 + i][dt % 4] : ring[u % D][dt][i];
                    o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, acc[u - NT][i], o[dt], 0, 0, 0);
                }
            }
        }
        if (exists(u + D))
        {
            fetch(ring[u % D], u + D);
        }
    }

    // ---- the four partial outputs of a query meet in LDS --------------------------------------------------------
    float* const row = own + n * kPitch;
#pragma unroll
    for (int dt = 0; dt < KD; ++dt)
    {
        // row m = 4 g + i of an output tile: dimension 64 b + 4 m + dt % 4 in a block, 16 dt + m behind the blocks
        if (dt < 4 * kBlocks)
        {
            int const b = dt / 4, i = dt % 4;
            *reinterpret_cast<f32x4*>(row + 64 * b + 16 * g + 4 * i)
                = f32x4{o[4 * b][i], o[4 * b + 1][i], o[4 * b + 2][i], o[4 * b + 3][i]};
        }
        else
        {
            *reinterpret_cast<f32x4*>(row + 16 * dt + 4 * g) = o[dt];
        }
    }
    __syncthreads();
    for (int p = threadIdx.x; p < kQueries * kPieces; p += kBlock)
    {
        int const q = p / kPieces, d0 = p % kPieces * 4;
        float const mx = fmaxf(fmaxf(rowMax[0][q], rowMax[1][q]), fmaxf(rowMax[2][q], rowMax[3][q]));
        float sum = 0.f;
        f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
            float const c = __builtin_amdgcn_exp2f((rowMax[v][q] - mx) * wl2); // 0 for a wavefront without keys
            sum += rowSum[v][q] * c;
            r += *reinterpret_cast<f32x4 const*>(lds[v] + q * kPitch + d0) * c;
        }
        r *= valid > 0 ? 1.f / (sum * kDown) : 0.f;
        int const query = first_row(up.part) + q;
        if (query >= 16 * up.part)
        {
            *reinterpret_cast<f32x4*>(out + (int64_t) query * ldOut + (int64_t) z * d + d0) = r;
        }
    }
}

template <int KD>
int launch(hipStream_t stream, int32_t S, int32_t B, int32_t N, float const* qkv, int32_t const* maskIdx, float* output)
{
    int64_t const ldOut = (int64_t) B * N * 16 * KD;
    int const strips = ceil_div(S, 16);
    int64_t const groups = (int64_t) strips * B * N;
    if (groups * kBlock > 0xffffffffll) // a launch holds fewer than 2^32 threads
    {
        return set_error(
            TRTAMD_STATUS_NOT_SUPPORTED, "unfused MHA: %lld workgroups exceed the grid", (long long) groups);
    }
    float const wl2 = 1.f / sqrtf((float) (16 * KD)) * 1.4426950408889634f; // exponentials as powers of two
    // tiles of scores per wavefront: as few registers as the sequence length asks for
    auto const kernel = S <= 256 ? attention_split_keys_kernel<KD, 4>
        : S <= 512               ? attention_split_keys_kernel<KD, 8>
                                 : attention_split_keys_kernel<KD, 16>;
    hipLaunchKernelGGL(kernel, dim3((unsigned) groups), dim3(kBlock), 0, stream, S, N, strips, wl2, qkv,
        (uint32_t) (12 * ldOut), maskIdx, output, ldOut);
    return check_launch("attention_split_keys_kernel");
}

} // namespace

bool attention_split_keys_takes(int32_t S, int32_t B, int32_t N, int32_t d, float const* qkv, float const* output)
{
    bool const aligned = ((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(output)) & 15u) == 0;
    return S >= 16 && S <= 1024 && d % 16 == 0 && d >= 32 && d <= 128 && aligned
        && (int64_t) S * 3 * B * N * d * 4 <= 0xffffffffll;
}

int attention_split_keys(hipStream_t stream, int32_t S, int32_t B, int32_t N, int32_t d, float const* qkv,
    int32_t const* maskIdx, float* output)
{
    switch (d / 16)
    {
    case 2: return launch<2>(stream, S, B, N, qkv, maskIdx, output);
    case 3: return launch<3>(stream, S, B, N, qkv, maskIdx, output);
    case 4: return launch<4>(stream, S, B, N, qkv, maskIdx, output);
    case 5: return launch<5>(stream, S, B, N, qkv, maskIdx, output);
    case 6: return launch<6>(stream, S, B, N, qkv, maskIdx, output);
    case 7: return launch<7>(stream, S, B, N, qkv, maskIdx, output);
    default: return launch<8>(stream, S, B, N, qkv, maskIdx, output);
    }
}

} // namespace trtamd
