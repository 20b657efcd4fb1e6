// gq8_prefill_attention.hip -- causal multi-query attention of a prompt block
// (MultiQueryAttention.h:275-308, MultiQueryPrefillAttention) on fp64 MFMA.
//
// Row r of the block sits at position base + r and attends keys [0, base + r]
// of its KV head (query head h reads KV head h / (heads / kv_heads)).  Scores
// scale * q.k, the softmax and the value sums are double, as in the decode
// kernel and the oracle; the block's rows leave as fp32 and as the Q8 row of
// the o product.
//
// Work split: the query heads of one KV head and position share their keys, so
// a workgroup owns 16 (row, head) pairs of one KV head: block_rows consecutive
// rows with all of the KV head's query heads (two rows at eight heads a KV
// head).  Fewer than 16 rows take one row a block, so no row's arithmetic
// meets another row's keys.  The block's key tiles (16 keys) are split over
// several workgroups where the blocks alone would leave the chip idle or end
// unevenly (attention_split); a workgroup's four waves take its tiles round robin,
// each keeping an online softmax state (row maximum, sum and the 16 x head_dim
// sums), and the states are merged in LDS at the end.  A block in one
// workgroup finishes its rows there; the splits of one leave their scaled sums,
// maxima and totals in the workspace for the merge launch.  The grid starts the
// longest blocks first, so the short ones fill in behind them.  A wave
// requests a tile's values (16-byte loads) before its scores and the next
// tile's keys right after them, so no tile's operands wait in registers a
// whole tile ahead; the kernel is held to two waves a SIMD (256 registers a
// wave), and one wave's MFMAs run while the other waits on its loads or works
// on its softmax.
//
// Per tile a wave computes S^T = K Q^T with v_mfma_f64_16x16x4f64, so the
// result holds row j of the block on lanes j, j + 16, j + 32, j + 48 and is
// already the P operand of O += P V (no transpose through LDS).  The online
// softmax is lazy: a row's reference maximum moves (and its sums are
// rescaled) only when a tile's maximum exceeds it by more than kLazyMargin,
// so most tiles need no rescaling; the weights exp(s - m) stay below
// e^kLazyMargin and every sum stays double.
//
// fp64 MFMA operand layout (checked on gfx950): A 16 x 4 with lane l holding
// A[l % 16][l / 16]; B 4 x 16 with lane l holding B[l / 16][l % 16]; D 16 x 16
// with lane l holding D[l / 16 + 4 r][l % 16], r = 0..3.  With g = l / 16 and
// j = l % 16:
//  - S^T (keys x rows, reduced over channels): lane (g, j) supplies key j's
//    and query row j's channels [g E, g E + E) (E = head_dim / 4), read
//    contiguously, and receives the scores of row j against keys g + 4 r.
//  - O (rows x channels, reduced over 4 keys a step): step st takes keys
//    g + 4 st, so lane (g, j) supplies its own weight p[st]; output tile n
//    holds channels j T + n (T = head_dim / 16), so a lane's value operands
//    are T contiguous channels of one key row and its outputs T contiguous
//    channels of rows g + 4 r.
#include "gq8_kernels.hpp"
#include "gq8_numerics.hpp"

#include <algorithm>
#include <cmath>

namespace gq8 {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kPaRows = 16;   // (row, head) pairs a workgroup
constexpr int kPaWaves = 4;
constexpr int kPaThreads = kPaWaves * 64;
constexpr int kPaKeys = 16;   // keys a tile
constexpr double kLazyMargin = 8.0;

struct PrefillArgs {
    const float *queries;
    int q_stride;
    const uint16_t *key_cache, *value_cache;
    int heads, kv_heads, head_dim;
    int rows;
    const int *pos_ptr;
    int pos_value;
    float scale;
    float *out;   // optional [rows, heads * head_dim]
    uint8_t *q8;  // optional Q8 row buffer of rows x heads * head_dim
    AttentionSplit split;
    double *ws_o, *ws_ml; // the splits' sums and (maximum, total)s (mqa_merge_kernel's layout)
};

__device__ inline v4d mfma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// N consecutive fp16 values (N a multiple of 4), as N / 2 words
template <int N>
__device__ inline void load_halves(const uint16_t *p, uint32_t (&w)[N / 2])
{
    if constexpr (N % 8 == 0) {
#pragma unroll
        for (int i = 0; i < N / 8; ++i) {
            const uint4 v = reinterpret_cast<const uint4 *>(p)[i];
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
    } else {
        static_assert(N == 4, "4, 8, 16, ... halves");
        const uint2 v = *reinterpret_cast<const uint2 *>(p);
        w[0] = v.x; w[1] = v.y;
    }
}

template <int N>
__device__ inline double half_at(const uint32_t (&w)[N], int i)
{
    return (double) half_value((uint16_t) (w[i >> 1] >> (16 * (i & 1))));
}

// E channels a lane group, T = head_dim / 16 output column tiles.  kOneRow:
// blocks of one query row, whose every attended key is its own (a step of few
// rows): the copies of the last key in the last tile are zeroed there, since a
// zero weight times an infinity would not be zero.  Blocks of several rows
// read later rows' keys under a zero weight in any case, and do without the
// selects (2-3 % of the kernel).
template <int E, bool kOneRow>
__global__ __launch_bounds__(kPaThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_attention_kernel(PrefillArgs a)
{
    constexpr int HD = 4 * E, T = HD / 16;
    constexpr int KW = E / 2, VW = T / 2; // words of a lane's key channels / value channels
    constexpr int kBlockLanes = kBlock / T;  // lanes holding one 32-channel block of an output row
    constexpr int kMergeTiles = T < 4 ? T : 4;
    // the merge: every wave's maxima and scaled sums of the rows g + 4 r, and
    // kMergeTiles column tiles of every wave's output sums at a time (over
    // the query rows, which no wave reads once all are past their tiles)
    __shared__ double sMax[kPaWaves][4][64], sSum[kPaWaves][4][64];
    constexpr int kQBytes = kPaRows * (HD + 4) * (int) sizeof(float);
    constexpr int kPartBytes = kPaWaves * kMergeTiles * 4 * 64 * (int) sizeof(double);
    __shared__ __align__(16) unsigned char sQPart[kQBytes > kPartBytes ? kQBytes : kPartBytes];
    // padded: a 16-lane group's rows on distinct banks
    float (*sQ)[HD + 4] = reinterpret_cast<float (*)[HD + 4]>(sQPart);
    double (*sPart)[kMergeTiles][4][64] = reinterpret_cast<double (*)[kMergeTiles][4][64]>(sQPart);

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int g = lane >> 4, j = lane & 15;
    const int perKv = a.heads / a.kv_heads, blockRows = a.split.block_rows;
    const int blocks = (a.rows + blockRows - 1) / blockRows;
    const int rb = blocks - 1 - (int) blockIdx.x / a.kv_heads; // the longest blocks first
    const int kvh = (int) blockIdx.x % a.kv_heads;
    const int r0 = rb * blockRows;
    const int qWidth = a.heads * HD, kvWidth = a.kv_heads * HD;
    const int base = (a.pos_ptr ? *a.pos_ptr : 0) + a.pos_value;
    const int rowsHere = min(blockRows, a.rows - r0);
    const int pairs = rowsHere * perKv;            // pair p: row r0 + p / perKv, head p % perKv of the KV head
    const int lastKey = base + r0 + rowsHere - 1;  // the block's last row attends [0, lastKey]
    const TileSplit span = tile_split(lastKey / kPaKeys + 1, a.split);
    if ((int) blockIdx.y >= span.splits)
        return;
    const int firstTile = (int) blockIdx.y * span.per;
    const int tiles = min(firstTile + span.per, lastKey / kPaKeys + 1); // this split's end
    const int rowPos = base + r0 + min(j, pairs - 1) / perKv; // pairs past the block repeat its last

    // the block's query rows in LDS (pairs past the block repeat its last);
    // lane (g, j) reads pair j's channels [g E, g E + E), the B operand of S^T
#pragma unroll
    for (int i = t; i < kPaRows * HD / 4; i += kPaThreads) {
        const int pair = min(i / (HD / 4), pairs - 1), c = (i % (HD / 4)) * 4;
        const float *src = a.queries + (int64_t) (r0 + pair / perKv) * a.q_stride
                           + (kvh * perKv + pair % perKv) * HD + c;
        *reinterpret_cast<float4 *>(&sQ[i / (HD / 4)][c]) = *reinterpret_cast<const float4 *>(src);
    }
    __syncthreads();
    const int qAt = j * (HD + 4) + g * E; // lane (g, j)'s first query channel in sQ
    const uint16_t *keys = a.key_cache + kvh * HD + g * E;
    const uint16_t *values = a.value_cache + kvh * HD + j * T;
    // a tile's operands: key k0 + j's channels, and keys k0 + g + 4 st's value channels
    // (keys past the block's last are clamped to it and masked)
    auto load_keys = [&](int tile, uint32_t (&kw)[KW]) {
        const int k0 = tile * kPaKeys;
        load_halves<E>(keys + (int64_t) min(k0 + j, lastKey) * kvWidth, kw);
    };
    auto load_values = [&](int tile, uint32_t (&vw)[4][VW]) {
        const int k0 = tile * kPaKeys;
#pragma unroll
        for (int st = 0; st < 4; ++st)
            load_halves<T>(values + (int64_t) min(k0 + g + 4 * st, lastKey) * kvWidth, vw[st]);
    };

    double m = -INFINITY, l = 0.0; // row j's reference maximum and sum (alike on its 4 lanes)
    v4d o[T];
#pragma unroll
    for (int n = 0; n < T; ++n)
        o[n] = v4d{0.0, 0.0, 0.0, 0.0};

    uint32_t kw[KW], vw[4][VW];
    if (firstTile + wave < tiles)
        load_keys(firstTile + wave, kw);
    for (int tile = firstTile + wave; tile < tiles; tile += kPaWaves) {
        load_values(tile, vw); // arrive while the scores are computed
        const int k0 = tile * kPaKeys;

        // the query is read from LDS every tile: an opaque offset keeps the
        // compiler from holding all E channels as doubles across the loop
        int qOff = qAt;
        asm volatile("" : "+v"(qOff));
        const float *qRow = &sQ[0][0] + qOff;
        v4d s = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < E; c += 4) {
            const float4 qv = *reinterpret_cast<const float4 *>(qRow + c);
            s = mfma(half_at(kw, c), (double) qv.x, s);
            s = mfma(half_at(kw, c + 1), (double) qv.y, s);
            s = mfma(half_at(kw, c + 2), (double) qv.z, s);
            s = mfma(half_at(kw, c + 3), (double) qv.w, s);
        }

        // the next tile's keys: they arrive during the softmax and O += P V
        load_keys(min(tile + kPaWaves, tiles - 1), kw);

        // row j against keys k0 + g + 4 r
        double sv[4];
        bool live[4];
        double tileMax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            live[r] = k0 + g + 4 * r <= rowPos;
            sv[r] = live[r] ? (double) a.scale * s[r] : -INFINITY;
            tileMax = fmax(tileMax, sv[r]);
        }
        tileMax = fmax(tileMax, __shfl_xor(tileMax, 16));
        tileMax = fmax(tileMax, __shfl_xor(tileMax, 32));
        const bool raise = tileMax > m + kLazyMargin; // false while the tile is all masked
        const bool rescale = raise && m != -INFINITY;
        if (__any(rescale)) {
            const double alpha = rescale ? exp(m - tileMax) : 1.0;
            double alphaO[4]; // the factors of output rows g + 4 r
#pragma unroll
            for (int r = 0; r < 4; ++r)
                alphaO[r] = __shfl(alpha, g + 4 * r);
#pragma unroll
            for (int n = 0; n < T; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o[n][r] *= alphaO[r];
            l *= alpha;
        }
        if (raise)
            m = tileMax;
        double p[4], sum = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = live[r] ? exp(sv[r] - m) : 0.0;
            sum += p[r];
        }
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        l += sum;

        if (kOneRow && k0 + kPaKeys - 1 > lastKey) {
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int w = 0; w < VW; ++w)
                    vw[st][w] = k0 + g + 4 * st <= lastKey ? vw[st][w] : 0u;
        }

        // O += P V, four keys a step
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int n = 0; n < T; ++n)
                o[n] = mfma(p[st], half_at(vw[st], n), o[n]);

    }

    // the maximum and sum of output rows g + 4 r
    double mO[4], lO[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        mO[r] = __shfl(m, g + 4 * r);
        lO[r] = __shfl(l, g + 4 * r);
    }

    // merge the waves' states.  Every wave scales its sums to the rows'
    // common maximum (a wave whose keys a row never reached has m = -inf and
    // weighs nothing; in a split past a row's last key every wave has); then the waves exchange their sums kMergeTiles
    // column tiles at a time, and wave w adds the four waves' sums of its
    // rows g + 4 w in wave order and finishes those rows.
#pragma unroll
    for (int r = 0; r < 4; ++r)
        sMax[wave][r][lane] = mO[r];
    __syncthreads(); // (also: every wave is past its tiles, so sQ is free)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        double common = sMax[0][r][lane];
#pragma unroll
        for (int w = 1; w < kPaWaves; ++w)
            common = fmax(common, sMax[w][r][lane]);
        const double f = mO[r] == -INFINITY ? 0.0 : exp(mO[r] - common);
        lO[r] *= f;
#pragma unroll
        for (int n = 0; n < T; ++n)
            o[n][r] *= f;
        sSum[wave][r][lane] = lO[r];
    }
    double mine[T]; // the four waves' sums of row g + 4 wave, column tile n
#pragma unroll
    for (int n0 = 0; n0 < T; n0 += kMergeTiles) {
        if (n0 > 0)
            __syncthreads(); // the previous tiles have been read
#pragma unroll
        for (int n = 0; n < kMergeTiles; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sPart[wave][n][r][lane] = o[n0 + n][r];
        __syncthreads();
#pragma unroll
        for (int n = 0; n < kMergeTiles; ++n) {
            double v = sPart[0][n][wave][lane];
#pragma unroll
            for (int w = 1; w < kPaWaves; ++w)
                v += sPart[w][n][wave][lane];
            mine[n0 + n] = v;
        }
    }
    double total = sSum[0][wave][lane];
#pragma unroll
    for (int w = 1; w < kPaWaves; ++w)
        total += sSum[w][wave][lane];

    // pair g + 4 wave, channels [j T, j T + T)
    {
        const int pair = g + 4 * wave;
        const bool live = pair < pairs;
        const int row = r0 + min(pair, pairs - 1) / perKv;
        const int head = kvh * perKv + min(pair, pairs - 1) % perKv;
        const int64_t at = (int64_t) row * qWidth + head * HD + j * T;
        if (span.splits > 1) { // one of several: its sums, maximum and total for the merge
            if (!live)
                return;
            double common = sMax[0][wave][lane];
#pragma unroll
            for (int w = 1; w < kPaWaves; ++w)
                common = fmax(common, sMax[w][wave][lane]);
            const int64_t slot = (int64_t) row * kAttentionSplits + blockIdx.y;
            double *o = a.ws_o + slot * qWidth + head * HD + j * T;
#pragma unroll
            for (int n = 0; n < T; ++n)
                o[n] = mine[n];
            if (j == 0) {
                a.ws_ml[(slot * a.heads + head) * 2] = common;
                a.ws_ml[(slot * a.heads + head) * 2 + 1] = total;
            }
            return;
        }
        // the whole row: fp32, then Q8 per 32-block (kBlockLanes neighbouring
        // lanes a block)
        float v[T];
        float amax = 0.f;
#pragma unroll
        for (int n = 0; n < T; ++n) {
            v[n] = (float) (mine[n] / total);
            amax = fmaxf(amax, fabsf(v[n]));
        }
        if (a.out && live) {
#pragma unroll
            for (int n = 0; n < T; n += 4)
                *reinterpret_cast<float4 *>(a.out + at + n) = float4{v[n], v[n + 1], v[n + 2], v[n + 3]};
        }
        if (a.q8) {
#pragma unroll
            for (int mask = 1; mask < kBlockLanes; mask <<= 1)
                amax = fmaxf(amax, __shfl_xor(amax, mask));
            const uint16_t bits = scale_bits_from_amax(amax);
            const float sc = half_value(bits);
            const float inv = bits ? quantize_hint(sc) : 0.f;
            uint32_t packed[T / 4];
#pragma unroll
            for (int i = 0; i < T / 4; ++i) {
                uint32_t word = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int qv = quantize_in_block(v[4 * i + b], bits, sc, inv);
                    word |= (uint32_t) (uint8_t) (int8_t) qv << (8 * b);
                }
                packed[i] = word;
            }
            if (live) {
                if constexpr (T == 16)
                    *reinterpret_cast<uint4 *>(a.q8 + at) = uint4{packed[0], packed[1], packed[2], packed[3]};
                else if constexpr (T == 8)
                    *reinterpret_cast<uint2 *>(a.q8 + at) = uint2{packed[0], packed[1]};
                else
                    *reinterpret_cast<uint32_t *>(a.q8 + at) = packed[0];
                if (j % kBlockLanes == 0)
                    reinterpret_cast<uint16_t *>(a.q8 + (int64_t) a.rows * qWidth)[at / kBlock] = bits;
            }
        }
    }
}

} // namespace

bool tiled_attention_supported(int head_dim, const float *queries, int q_stride,
                                 const uint16_t *key_cache, const uint16_t *value_cache,
                                 const float *out, const uint8_t *q8)
{
    auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    return (head_dim == 64 || head_dim == 128 || head_dim == 256) && q_stride % 4 == 0
           && aligned(queries) && aligned(key_cache) && aligned(value_cache) && aligned(out)
           && aligned(q8);
}

// The split with the least estimated time.  A workgroup keeps a compute
// unit's matrix cores about as busy as two do (5.3 us a round of four tiles
// alone, 10.6 each beside another), so a unit is taken to run its workgroups
// one after another, the fullest unit ending last; the merge launch and the
// partials cost some microseconds and more with the rows.  Within 10 % of most
// of a sweep at eight heads of 256 over one KV head (rows 1 .. 2048, 0 .. 8000
// keys before them).  Microseconds there, one workgroup a block -> split: 333
// rows behind 700 keys 99 -> 77, 128 behind 4000 352 -> 105, 16 behind 8000
// 672 -> 42, one row of 8000 keys 680 -> 27 (110 in mqa_partial_kernel and its
// former merge); 512 rows behind 512 keys and 2048 alone stay whole (94, 330).
// The same constants serve narrower heads, whose rounds are shorter but whose
// workgroups do overlap on a unit: 2 to 4 times faster than whole blocks over
// long caches (512 rows behind 4000 keys at 4 heads of 64 131 -> 67), and up
// to 17 % slower where some 100 keys are split after all (64 rows behind 100
// keys at 16 heads of 64 9.4 -> 11.0).  Rounds scaled by the head width keep
// those whole, but lose 5 to 30 % at thirty other points of the sweep.
AttentionSplit attention_split(int rows, int heads, int kv_heads, int keys)
{
    constexpr int kUnits = 256, kSamples = 32;
    constexpr double kRound = 5.3, kStart = 5.0, kMerge = 4.0, kMergeRow = 0.012;
    constexpr double kWorth = 0.92; // a split's estimate against the whole blocks'
    AttentionSplit s{rows < kPaRows ? 1 : std::max(1, kPaRows / (heads / kv_heads)), 8,
                     kAttentionSplits};
    if (keys <= 0)
        return s;
    if (rows > 65535) { // past the merge's grid
        s.max_splits = 1;
        return s;
    }
    const int blocks = (rows + s.block_rows - 1) / s.block_rows;
    auto block_tiles = [&](int b) { // key tiles of block b
        return (keys - rows + std::min((b + 1) * s.block_rows, rows) - 1) / kAttentionTileKeys + 1;
    };
    const int longest = block_tiles(blocks - 1);
    const int stride = (blocks + kSamples - 1) / kSamples, samples = (blocks + stride - 1) / stride;
    double least = 0.0;
    int chosen = 0;
    for (int step = 1, last = 0; step < 2 * kAttentionSplits; step += 1 + step / 4) {
        const int splits = std::min(step, kAttentionSplits);
        const int per = ((longest + splits - 1) / splits + 3) / 4 * 4;
        if (per == last)
            continue;
        last = per;
        // the sampled blocks' workgroups and rounds of four tiles
        int64_t count = 0, rounds = 0;
        int smallest = per;
        for (int b = blocks - 1; b >= 0; b -= stride) {
            const int tiles = block_tiles(b), whole = tiles / per, rest = tiles % per;
            count += whole + (rest ? 1 : 0);
            rounds += whole * (per / 4) + (rest + 3) / 4;
            smallest = std::min(smallest, whole ? per : rest);
        }
        const double each = (double) blocks * kv_heads / samples / kUnits; // a unit's share of a sample
        const double mine = count * each;
        // the fullest unit: the longest workgroup, or its share of all rounds
        // and what whole workgroups leave uneven (the short ones go last)
        const double longestOne = (std::min(per, longest) + 3) / 4;
        const double busy = std::max(longestOne, rounds * each + (std::ceil(mine) - mine) * (smallest + 3) / 4);
        const double cost = busy * kRound + std::ceil(mine) * kStart
                            + (longest > per ? kMerge + rows * kMergeRow : 0.0);
        if (chosen == 0 || cost < least) {
            least = chosen == 0 ? kWorth * cost : cost;
            chosen = per;
        }
    }
    s.tiles = chosen;
    return s;
}

hipError_t launch_tiled_attention(const float *queries, int q_stride, const uint16_t *key_cache,
                                  const uint16_t *value_cache, int heads, int kv_heads,
                                  int head_dim, int rows, const int *pos_ptr, int pos_value,
                                  float scale, float *out, uint8_t *q8, const AttentionSplit &split,
                                  double *ws_o, double *ws_ml, hipStream_t stream)
{
    if (rows <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0
        || heads / kv_heads > kPaRows
        || !tiled_attention_supported(head_dim, queries, q_stride, key_cache, value_cache, out, q8)
        || q_stride < heads * head_dim || split.block_rows <= 0
        || split.block_rows * (heads / kv_heads) > kPaRows || split.max_splits <= 0
        || split.max_splits > kAttentionSplits || split.tiles <= 0 || split.tiles % kPaWaves != 0
        || (split.max_splits > 1 && (!ws_o || !ws_ml)))
        return hipErrorInvalidValue;
    PrefillArgs a{queries, q_stride, key_cache, value_cache, heads, kv_heads, head_dim, rows,
                  pos_ptr, pos_value, scale, out, q8, split, ws_o, ws_ml};
    const int blocks = (rows + split.block_rows - 1) / split.block_rows;
    // the splits of the longest block, where its keys are known here and every
    // block's workgroups take the same tiles
    const TileSplit longest = tile_split((pos_value + rows - 1) / kPaKeys + 1, split);
    const int splits = pos_ptr || longest.per != split.tiles ? split.max_splits : longest.splits;
    const dim3 grid((unsigned) (blocks * kv_heads), splits);
#define GQ8_TILED_ATTENTION(E)                                                                  \
    do {                                                                                       \
        if (split.block_rows == 1)                                                             \
            hipLaunchKernelGGL((prefill_attention_kernel<E, true>), grid, dim3(kPaThreads), 0,   \
                               stream, a);                                                     \
        else                                                                                   \
            hipLaunchKernelGGL((prefill_attention_kernel<E, false>), grid, dim3(kPaThreads), 0,  \
                               stream, a);                                                     \
    } while (0)
    switch (head_dim) {
    case 256: GQ8_TILED_ATTENTION(64); break;
    case 128: GQ8_TILED_ATTENTION(32); break;
    default: GQ8_TILED_ATTENTION(16); break;
    }
#undef GQ8_TILED_ATTENTION
    return hipGetLastError();
}

} // namespace gq8
