// gq8_gemm.hip -- the multi-row Int8Blocks product on int8 MFMA (prefill).
//
// y[m, n] (+)= sum over 32-element blocks b of
//                  dot_i8(x[m, b], w[n, b]) * (scale_w[n, b] * scale_x[m, b])
//
// the reference's product (Linear.h:10-34, 284-298; the prefill's
// SimdTiledMatMul.h / TiledMatMul.h) with both operands in Int8Blocks: the
// activation rows quantized by the reference's own weight rule.  One
// v_mfma_i32_16x16x32_i8 covers exactly one block of a 16 x 16 tile, so every
// block's integer dot is exact; it is then scaled and accumulated in double.
// The 128 x 64 tile adds a row's blocks in order, as the oracle does.  The
// others' waves take the blocks of a chunk apart (KS) and add their sums at
// the end, so the order of a row's sum depends on the tile, and with it on how
// many rows share the step: equal to the row computed alone but for a few
// 2^-53 before the result is rounded to fp32, which is rarely seen in it.
//
// Tiling (TileShape): a workgroup of eight waves owns a TM x TN tile of y
// (rows x outputs), a wave RM x RN MFMA tiles of it over 1 / KS of every
// chunk's blocks.  A chunk of both operands and its fp16 scales (as doubles)
// is staged in LDS with 16-byte loads, so two workgroups share a CU and one's
// loads overlap the other's arithmetic; with KS > 1 the waves' sums are added
// in LDS at the end.  The double epilogue (a conversion, a product with the
// weight scale and a fused multiply-add with the activation scale per element
// and block) bounds the large tiles, not the MFMA.  The activation scales of
// a 16-lane row's four rows reach its lanes by DPP broadcast inside that
// multiply-add, so a chunk reads them from LDS once (four blocks a load)
// rather than per element.
//
// MFMA operand layout (checked on gfx950): for A 16 x 32 and B given as
// B[j][k] 16 x 32, lane l supplies A[l % 16][8 (l / 16) .. + 8) and
// B[l % 16][8 (l / 16) .. + 8); D[i][j] lands in lane 16 (i / 4) + j,
// element i % 4.
#include "gq8_kernels.hpp"
#include "gq8_lanes.hpp"
#include "gq8_numerics.hpp"

#include <algorithm>

namespace gq8 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kGemmThreads = 512;

// WM x WN wave tiles of RM x RN MFMA tiles, KS waves a wave tile, each taking
// CH of a chunk's KS * CH blocks.
template <int WM_, int WN_, int RM_, int RN_, int KS_, int CH_>
struct TileShape {
    static constexpr int WM = WM_, WN = WN_, RM = RM_, RN = RN_, KS = KS_, CH = CH_;
    static constexpr int TM = WM * RM * 16, TN = WN * RN * 16;
    static constexpr int chunk = KS * CH;               // blocks a chunk
    static constexpr int rowBytes = chunk * kBlock + 16; // padded LDS row: conflict-free fragment reads
    static constexpr int stageRows = TM + TN;           // operand rows a chunk
    static constexpr int rowPieces = chunk * 2;         // 16-byte pieces of a staged row
    static constexpr int vectors = stageRows * rowPieces / kGemmThreads; // a thread
    static constexpr int vectorsA = TM * rowPieces / kGemmThreads;       // of those, activation rows
    static constexpr int scales = (stageRows * chunk + kGemmThreads - 1) / kGemmThreads;
    static constexpr int stageBytes = stageRows * rowBytes + stageRows * (chunk + 1) * 8;
    static constexpr int mergeBytes = (KS - 1) * TM * TN * 8;
    static constexpr int ldsBytes = stageBytes > mergeBytes ? stageBytes : mergeBytes;
    static_assert(WM * WN * KS * 64 == kGemmThreads, "eight waves");
    static_assert(CH % 4 == 0, "a wave takes its activation scales four blocks a load");
    static_assert(vectors * kGemmThreads == stageRows * rowPieces
                      && vectorsA * kGemmThreads == TM * rowPieces,
                  "whole pieces a thread, a piece of one operand");
};

// acc[j][r] += part[j][r] * s', r = 0..3, where s' is the s held by lane
// 4 Q + r of this lane's 16-lane row (a DPP broadcast inside the
// multiply-add).  It rounds acc + part * s' once, as acc + d * (sw * sx)
// does: both products are exact in double.
template <int Q, int RN>
__device__ inline void fmac_row_scales(double (&acc)[RN][4], double s, const double (&part)[RN][4])
{
#pragma unroll
    for (int j = 0; j < RN; ++j)
        fmac_row_bcast4<4 * Q, 4 * Q + 1, 4 * Q + 2, 4 * Q + 3>(acc[j], s, part[j]);
}

// kGeglu: the gate|up product of a fused [2 F, inner] weight (gate rows
// first) with GeGLU and its Q8 folded in.  Tile column block bx stages gate
// rows [32 bx, 32 bx + 32) as B rows 0..31 and the matching up rows as B rows
// 32..63, so a tile holds both halves of 32 GeGLU outputs of its rows: the
// epilogue rounds both to fp32 (the stores the unfused product makes), takes
// the GeGLU of each pair and quantizes each row's 32 outputs as one block into
// q8_out ([rows, F] Q8 row buffer), with the fp32 outputs to debug_out if set.
//
// kTail: any block count.  The last chunk then starts early enough to end at
// the last block (a row shorter than a chunk repeats its last block), and the
// blocks it takes again get a zero weight scale.  Without it the block count
// is a multiple of the chunk.
template <typename S, bool kGeglu, bool kTail>
__global__ __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(4)))
void q8_gemm_kernel(
    const uint8_t *__restrict__ x8, int64_t xElements, int xRow0, int rows,
    const uint8_t *__restrict__ w8, int inner, int outputs, float *__restrict__ y, int yStride,
    int residual, uint8_t *__restrict__ q8_out, float *__restrict__ debug_out)
{
    constexpr int TM = S::TM, TN = S::TN, RM = S::RM, RN = S::RN, KS = S::KS, CH = S::CH;
    constexpr int kChunk = S::chunk, kRowBytes = S::rowBytes, kRowPieces = S::rowPieces;
    static_assert(!kGeglu || TN == 64, "GeGLU: 32 gate and 32 up rows a tile");
    // rows [0, TM) of the stage are A (activation rows), [TM, TM + TN) B (weight rows)
    __shared__ __attribute__((aligned(16))) uint8_t sStage[S::ldsBytes];
    uint8_t *sOps = sStage;
    double (*sScales)[kChunk + 1] =
        reinterpret_cast<double (*)[kChunk + 1]>(sStage + S::stageRows * kRowBytes);

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int ks = wave / (S::WM * S::WN), tileWave = wave % (S::WM * S::WN);
    const int wm = (tileWave / S::WN) * RM * 16, wn = (tileWave % S::WN) * RN * 16;
    const int nb = inner / kBlock;

    // the global source of the staged pieces this thread moves: row r of the
    // stage (clamped into range; rows past the end are computed, never
    // stored).  32-bit offsets from the two operands' tile bases: the first
    // S::vectorsA pieces of every thread are A rows, the rest B rows.
    const int F = outputs / 2;
    const int64_t wRow0 = kGeglu ? (int64_t) blockIdx.x * 32 : (int64_t) n0;
    const uint8_t *aBase = x8 + (int64_t) (xRow0 + m0) * inner;
    const uint8_t *wBase = w8 + wRow0 * inner;
    const uint16_t *aScales = reinterpret_cast<const uint16_t *>(x8 + xElements) + (int64_t) (xRow0 + m0) * nb;
    const uint16_t *wScales = reinterpret_cast<const uint16_t *>(w8 + (int64_t) outputs * inner) + wRow0 * nb;
    auto stage_row = [&](int r) -> uint32_t { // the row, from its operand's tile base
        if (r < TM)
            return (uint32_t) min(r, rows - 1 - m0);
        const int j = r - TM;
        if constexpr (kGeglu)
            return (uint32_t) ((j < 32 ? 0 : F) + min(j & 31, F - 1 - (int) blockIdx.x * 32));
        else
            return (uint32_t) min(j, outputs - 1 - n0);
    };
    uint32_t srcOff[S::vectors];
#pragma unroll
    for (int i = 0; i < S::vectors; ++i) {
        const int piece = t + i * kGemmThreads; // 16-byte pieces, kRowPieces a row
        const int p = piece % kRowPieces;
        const int block = kTail ? min(p >> 1, nb - 1) : p >> 1;
        srcOff[i] = stage_row(piece / kRowPieces) * (uint32_t) inner + block * kBlock + (p & 1) * 16;
    }
    uint32_t scaleOff[S::scales];
    bool scaleA[S::scales];
#pragma unroll
    for (int i = 0; i < S::scales; ++i) {
        const int e = min(t + i * kGemmThreads, S::stageRows * kChunk - 1);
        const int r = e / kChunk, b = kTail ? min(e % kChunk, nb - 1) : e % kChunk;
        scaleA[i] = r < TM;
        scaleOff[i] = stage_row(r) * (uint32_t) nb + b;
    }
    constexpr int kScalesA = TM * kChunk; // the first ones are the A rows'
    double acc[RM][RN][4];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[i][j][r] = 0.0;

    // this lane's fragment offsets in a stage
    const int kg = (lane >> 4) * 8 + ks * CH * kBlock;
    int aOff[RM], bOff[RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
        aOff[i] = (wm + i * 16 + (lane & 15)) * kRowBytes + kg;
#pragma unroll
    for (int j = 0; j < RN; ++j)
        bOff[j] = (TM + wn + j * 16 + (lane & 15)) * kRowBytes + kg;

    const int chunks = (nb + kChunk - 1) / kChunk;
    // the first block of chunk c
    auto chunk_block = [&](int c) { return kTail ? max(min(c * kChunk, nb - kChunk), 0) : c * kChunk; };
    // a chunk's pieces go global -> registers one chunk ahead, so their loads
    // are in flight while the previous chunk is computed
    // (native vectors in plain unrolled loops: HIP's int4 carried across the
    // loop, or arrays captured by a lambda, are left in scratch memory)
    v4i v[S::vectors];
    uint16_t sc[S::scales];
#define GQ8_SCALE_BASE(i, a, w)                                                                \
    (((i) + 1) * kGemmThreads <= kScalesA ? (a)                                                \
     : (i) * kGemmThreads >= kScalesA     ? (w)                                                \
                                          : (scaleA[i] ? (a) : (w)))
#pragma unroll
    for (int i = 0; i < S::vectors; ++i)
        v[i] = *reinterpret_cast<const v4i *>((i < S::vectorsA ? aBase : wBase) + srcOff[i]);
#pragma unroll
    for (int i = 0; i < S::scales; ++i)
        sc[i] = GQ8_SCALE_BASE(i, aScales, wScales)[scaleOff[i]];
    for (int c = 0; c < chunks; ++c) {
        __syncthreads(); // the previous chunk has been read
        {
#pragma unroll
            for (int i = 0; i < S::vectors; ++i) {
                const int piece = t + i * kGemmThreads;
                *reinterpret_cast<v4i *>(&sOps[(piece / kRowPieces) * kRowBytes + (piece % kRowPieces) * 16]) = v[i];
            }
            // blocks [first, last) of the chunk are new
            const int first = c * kChunk - chunk_block(c), last = nb - chunk_block(c);
#pragma unroll
            for (int i = 0; i < S::scales; ++i) {
                const int e = t + i * kGemmThreads;
                if (S::scales * kGemmThreads == S::stageRows * kChunk || e < S::stageRows * kChunk) {
                    const int b = e % kChunk;
                    sScales[e / kChunk][b] =
                        (!kTail || (b >= first && b < last)) ? (double) half_value(sc[i]) : 0.0;
                }
            }
        }
        __syncthreads();
        {
            // the next chunk (the last is a repeat, never stored); its offset
            // joins the uniform bases, so each piece's address is a 32-bit
            // offset from a scalar base.  The chunk index and the offsets pass
            // through empty asm statements: otherwise the loop keeps a stepped
            // 64-bit address a piece (twelve registers) or the offsets'
            // 64-bit extensions.
            int next = chunk_block(min(c + 1, chunks - 1));
            asm volatile("" : "+s"(next));
            const int64_t c0 = (int64_t) next;
            const uint8_t *aChunk = aBase + c0 * kBlock, *wChunk = wBase + c0 * kBlock;
            const uint16_t *aScaleChunk = aScales + c0, *wScaleChunk = wScales + c0;
#pragma unroll
            for (int i = 0; i < S::vectors; ++i) {
                uint32_t off = srcOff[i];
                asm volatile("" : "+v"(off));
                v[i] = *reinterpret_cast<const v4i *>((i < S::vectorsA ? aChunk : wChunk) + off);
            }
#pragma unroll
            for (int i = 0; i < S::scales; ++i) {
                uint32_t off = scaleOff[i];
                asm volatile("" : "+v"(off));
                sc[i] = GQ8_SCALE_BASE(i, aScaleChunk, wScaleChunk)[off];
            }
        }
        // the activation scales of the wave's rows, four blocks a load: lane
        // (g, j) holds row 4 g + (j & 3)'s scale of block 4 h + (j >> 2) (the
        // rows of MFMA tile i), and every lane of the 16-lane row g takes the
        // one it needs by DPP
        double sxRow[RM][CH / 4];
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int h = 0; h < CH / 4; ++h)
                sxRow[i][h] = sScales[wm + i * 16 + (lane >> 4) * 4 + (lane & 3)]
                                     [ks * CH + h * 4 + ((lane >> 2) & 3)];
        // a block's MFMAs go out together, then their double epilogue, so
        // the later MFMAs run while the first one's results are scaled; the
        // blocks are unrolled (LDS offsets as immediates).  The large tile has
        // a scheduling barrier between them, so no block's loads are hoisted
        // into another's registers
#pragma unroll
        for (int kb = 0; kb < CH; ++kb) {
            long af[RM], bf[RN];
#pragma unroll
            for (int i = 0; i < RM; ++i)
                af[i] = *reinterpret_cast<const long *>(sOps + aOff[i] + kb * kBlock);
#pragma unroll
            for (int j = 0; j < RN; ++j)
                bf[j] = *reinterpret_cast<const long *>(sOps + bOff[j] + kb * kBlock);
            double sw[RN];
#pragma unroll
            for (int j = 0; j < RN; ++j)
                sw[j] = sScales[TM + wn + j * 16 + (lane & 15)][ks * CH + kb];
            v4i d[RM][RN];
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < RN; ++j) {
                    const v4i zero = {0, 0, 0, 0};
                    d[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(af[i], bf[j], zero, 0, 0, 0);
                }
#pragma unroll
            for (int i = 0; i < RM; ++i) {
                double part[RN][4]; // d * sw: exact (a 20-bit integer times an fp16 value)
#pragma unroll
                for (int j = 0; j < RN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        part[j][r] = (double) d[i][j][r] * sw[j];
                switch (kb & 3) {
                case 0: fmac_row_scales<0, RN>(acc[i], sxRow[i][kb >> 2], part); break;
                case 1: fmac_row_scales<1, RN>(acc[i], sxRow[i][kb >> 2], part); break;
                case 2: fmac_row_scales<2, RN>(acc[i], sxRow[i][kb >> 2], part); break;
                default: fmac_row_scales<3, RN>(acc[i], sxRow[i][kb >> 2], part); break;
                }
            }
            if constexpr (CH == 8)
                __builtin_amdgcn_sched_barrier(0);
        }
    }
#undef GQ8_SCALE_BASE

    if constexpr (KS > 1) {
        // the waves' sums of a wave tile, added in the order of their blocks'
        // places in a chunk, over the staging buffer
        double *sMerge = reinterpret_cast<double *>(sStage);
        __syncthreads(); // every wave is past its last read
        auto slot = [&](int k, int i, int j, int r) {
            return ((((k * S::WM * S::WN + tileWave) * RM + i) * RN + j) * 4 + r) * 64 + lane;
        };
        if (ks > 0) {
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < RN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        sMerge[slot(ks - 1, i, j, r)] = acc[i][j][r];
        }
        __syncthreads();
        if (ks == 0) {
#pragma nounroll
            for (int k = 0; k < KS - 1; ++k) // not unrolled: one wave's sums in registers at a time
#pragma unroll
                for (int i = 0; i < RM; ++i)
#pragma unroll
                    for (int j = 0; j < RN; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[i][j][r] += sMerge[slot(k, i, j, r)];
        }
    }

    if constexpr (!kGeglu) {
        if (ks > 0)
            return;
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j) {
                const int n = n0 + wn + j * 16 + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + wm + i * 16 + (lane >> 4) * 4 + r;
                    if (m < rows && n < outputs) {
                        float *out = y + (int64_t) m * yStride + n;
                        const double old = residual ? (double) *out : 0.0;
                        *out = (float) (acc[i][j][r] + old);
                    }
                }
            }
    } else {
        // the fp32 gate (columns 0..31) and up (32..63) values of the tile in
        // LDS, over the staging buffer (every wave is past its last read)
        __syncthreads();
        float *sOut = reinterpret_cast<float *>(sStage); // [TM][65]
        if (ks == 0) {
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < RN; ++j) {
                    const int c = wn + j * 16 + (lane & 15);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        sOut[(wm + i * 16 + (lane >> 4) * 4 + r) * 65 + c] = (float) acc[i][j][r];
                }
        }
        __syncthreads();
        // thread t: row t / 4, outputs 8 (t % 4) .. + 8 (four lanes a 32-block)
        const int row = t >> 2, c0 = (t & 3) * 8;
        if (row >= TM) // whole waves
            return;
        const int m = m0 + row;
        float v[8];
        float amax = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            v[k] = geglu(sOut[row * 65 + c0 + k], sOut[row * 65 + 32 + c0 + k]);
            amax = fmaxf(amax, fabsf(v[k]));
        }
        amax = fmaxf(amax, __shfl_xor(amax, 1));
        amax = fmaxf(amax, __shfl_xor(amax, 2));
        const int o0 = blockIdx.x * 32 + c0;
        if (m < rows && o0 < F) {
            const uint16_t bits = scale_bits_from_amax(amax);
            const float sc = half_value(bits);
            const float inv = bits ? quantize_hint(sc) : 0.f;
            uint32_t packed[2] = {0u, 0u};
#pragma unroll
            for (int k = 0; k < 8; ++k)
                packed[k / 4] |= (uint32_t) (uint8_t) (int8_t) quantize_in_block(v[k], bits, sc, inv)
                                 << (8 * (k % 4));
            *reinterpret_cast<uint2 *>(q8_out + (int64_t) m * F + o0) = make_uint2(packed[0], packed[1]);
            if ((t & 3) == 0)
                reinterpret_cast<uint16_t *>(q8_out + (int64_t) rows * F)[(int64_t) m * (F / kBlock) + blockIdx.x] = bits;
            if (debug_out)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    debug_out[(int64_t) m * F + o0 + k] = v[k];
        }
    }
}

// The tiles.  Few rows or few outputs leave a large tile's grid short of the
// chip's 256 compute units, and a short row count leaves its rows unused, so
// smaller tiles take those products with more waves over the blocks of each
// (a wave's chain of chunks is then shorter too).
using Tile128x64 = TileShape<4, 2, 2, 2, 1, 8>; // whole chunks of 8 blocks only
using Tile64x64 = TileShape<2, 2, 2, 2, 2, 4>;
using Tile64x32 = TileShape<2, 1, 2, 2, 4, 4>;
using Tile32x64 = TileShape<1, 2, 2, 2, 4, 4>;
using Tile16x64 = TileShape<1, 2, 1, 2, 4, 4>;
using Tile16x32 = TileShape<1, 2, 1, 1, 4, 4>;
using Tile32x16 = TileShape<1, 1, 2, 1, 8, 4>;
using Tile16x16 = TileShape<1, 1, 1, 1, 8, 4>;

struct TileArgs {
    const uint8_t *x8;
    int64_t x_elements;
    int x_row0, rows;
    const uint8_t *w8;
    int inner, outputs;
    float *y;
    int y_stride, residual;
    uint8_t *q8_out;
    float *debug_out;
};

template <typename S, bool kGeglu, bool kTail>
hipError_t launch_tile(const TileArgs &a, hipStream_t stream)
{
    const int columns = kGeglu ? a.outputs / 2 / kBlock : (a.outputs + S::TN - 1) / S::TN;
    const dim3 grid(columns, (a.rows + S::TM - 1) / S::TM);
    hipLaunchKernelGGL((q8_gemm_kernel<S, kGeglu, kTail>), grid, dim3(kGemmThreads), 0, stream,
                       a.x8, a.x_elements, a.x_row0, a.rows, a.w8, a.inner, a.outputs, a.y,
                       a.y_stride, a.residual, a.q8_out, a.debug_out);
    return hipGetLastError();
}

// The choice among the tiles: the least estimated time.  A product whose grid
// is at most one workgroup a compute unit takes `alone` microseconds per 2048
// of the inner size (a workgroup's chain of chunks); n workgroups a compute
// unit take n times `packed` (n rounded up: the fullest unit ends last).
// Below an inner size of kShortInner a workgroup's staging, merge and store
// weigh as much as its chain, and `start` microseconds a round come on top of
// it (256 -> 1024 at 1500 rows: 10.3 us by the chains alone, 6.5 so; 77 of the
// 126 points at 256 and 512 gained, by 1.2 us, and none lost).
// All were fitted to sweeps on one MI355X over rows 2 .. 2048, inner sizes 256
// .. 16384 and 256 .. 256000 outputs, weights from HBM.  The estimate ranks the
// tiles and is no time: what every launch costs (2.5 to 5 us) is left out, so
// it is within 10 % at 35 of 59 points at an inner size of 16384 and 0.64 of
// the time in the median at 2048.  The choice is within 10 % of the fastest
// tile at nine points of ten and within 15 % at 421 of 434; the worst is
// 16384 -> 8192 at 17 rows, 51 against 38 us.  Microseconds, the 128 x 64 tile
// (the only one before) -> the chosen one: 16384 -> 2048 at 64 rows 165 -> 25,
// at 512 169 -> 90, at 1024 171 -> 154; 2048 -> 2048 at 64 rows 22.9 -> 5.8, at
// 512 24.5 -> 15.9; 2048 -> 32768 at 32 rows 39 -> 19.5, at 64 40 -> 25 (at 128
// and more it stays).  Below 32 rows, where the products had run in
// q8_product_kernel: 2048 -> 32768 at 16 rows 80 -> 15.4 (4.7 TB/s of weights),
// 16384 -> 2048 70 -> 19.5, 2048 -> 256000 at 5 rows 324 -> 92 (6.1 TB/s).
struct TileCost {
    int rows, outputs; // the tile
    double alone, packed;
    hipError_t (*launch)(const TileArgs &, hipStream_t);
    double start; // below kShortInner
};

constexpr int kShortInner = 1024;
constexpr int kComputeUnits = 256;
constexpr int kMaxTileRows = 65535; // the grid's y extent

const TileCost kProductTiles[] = {
    {128, 64, 20.2, 18.2, launch_tile<Tile128x64, false, false>, 0.2},
    {64, 64, 11.3, 10.0, launch_tile<Tile64x64, false, true>, 0.5},
    {64, 32, 6.6, 5.6, launch_tile<Tile64x32, false, true>, 0.4},
    {32, 64, 6.8, 6.4, launch_tile<Tile32x64, false, true>, 0.4},
    {16, 32, 3.6, 2.3, launch_tile<Tile16x32, false, true>, 0.2},
    {32, 16, 2.7, 2.7, launch_tile<Tile32x16, false, true>, 3.0},
    {16, 16, 2.1, 1.5, launch_tile<Tile16x16, false, true>, 0.4},
};
const TileCost kGegluTiles[] = { // 64 staged weight rows: 32 outputs
    {128, 64, 20.2, 18.2, launch_tile<Tile128x64, true, false>, 0.0},
    {64, 64, 11.3, 10.0, launch_tile<Tile64x64, true, true>, 0.0},
    {32, 64, 6.8, 6.4, launch_tile<Tile32x64, true, true>, 0.0},
    {16, 64, 5.4, 4.7, launch_tile<Tile16x64, true, true>, 0.0},
};

template <size_t N>
const TileCost &best_tile(const TileCost (&tiles)[N], int rows, int inner, int outputs)
{
    const TileCost *best = nullptr;
    double least = 0.0;
    for (const TileCost &c : tiles) {
        if (c.rows == 128 && inner % (Tile128x64::chunk * kBlock) != 0)
            continue; // the large tile takes whole chunks
        const int64_t tileRows = (rows + (int64_t) c.rows - 1) / c.rows;
        if (tileRows > kMaxTileRows && c.rows < 64)
            continue;
        const int64_t workgroups = tileRows * ((outputs + (int64_t) c.outputs - 1) / c.outputs);
        const int64_t rounds = (workgroups + kComputeUnits - 1) / kComputeUnits;
        const double chain = inner / 2048.0 * std::max(c.alone, (double) rounds * c.packed);
        const double cost = chain + (inner < kShortInner ? (double) rounds * c.start : 0.0);
        if (!best || cost < least) {
            best = &c;
            least = cost;
        }
    }
    return *best;
}

template <size_t N>
hipError_t launch_best(const TileCost (&tiles)[N], const TileArgs &a, hipStream_t stream)
{
    return best_tile(tiles, a.rows, a.inner, a.outputs).launch(a, stream);
}

} // namespace

ProductTile q8_gemm_tile(int rows, int inner, int outputs)
{
    const TileCost &c = best_tile(kProductTiles, rows, inner, outputs);
    return {c.rows, c.outputs};
}

hipError_t launch_q8_gemm(const uint8_t *x8, int64_t x_elements, int x_row0, int rows,
                          const uint8_t *w8, int inner, int outputs, float *y, int y_stride,
                          int residual, hipStream_t stream)
{
    if (rows <= 0 || outputs <= 0 || inner <= 0 || inner % kBlock != 0 || y_stride < outputs)
        return hipErrorInvalidValue;
    constexpr int kSlab = kMaxTileRows * 64; // rows a launch
    for (int r0 = 0; r0 < rows; r0 += std::min(kSlab, rows - r0)) {
        const hipError_t status = launch_best(
            kProductTiles,
            {x8, x_elements, x_row0 + r0, std::min(kSlab, rows - r0), w8, inner, outputs,
             y + (int64_t) r0 * y_stride, y_stride, residual, nullptr, nullptr},
            stream);
        if (status != hipSuccess)
            return status;
    }
    return hipSuccess;
}

bool q8_gemm_geglu_supported(int rows, int inner, int intermediate)
{
    // (a tile's up rows lie intermediate rows past its gate rows: a 32-bit offset)
    return rows > 1 && inner % kBlock == 0 && intermediate % kBlock == 0
           && ((int64_t) intermediate + 64) * inner < (int64_t(1) << 32);
}

hipError_t launch_q8_gemm_geglu(const uint8_t *x8, int64_t x_elements, int x_row0, int rows,
                                const uint8_t *w8, int inner, int intermediate, uint8_t *q8_out,
                                float *debug_out, hipStream_t stream)
{
    if (inner <= 0 || intermediate <= 0 || !q8_gemm_geglu_supported(rows, inner, intermediate)
        || !q8_out)
        return hipErrorInvalidValue;
    return launch_best(kGegluTiles,
                       {x8, x_elements, x_row0, rows, w8, inner, 2 * intermediate, nullptr, 0, 0,
                        q8_out, debug_out},
                       stream);
}

} // namespace gq8
