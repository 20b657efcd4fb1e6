// gq8_sample.hip -- one token drawn from one row of logits on the device:
// Sampler::sample (Sampler.cpp:78-213) in place of the reference's logits
// readback (Gemma.cpp:545-595).
//
// Candidates are the unmasked tokens, scored logit * (1 / temperature) in
// double and weighing exp(score - largest score).  With a cut set they are
// ranked (score descending, token ascending): the first k are kept, of those
// the shortest prefix whose mass reaches p of theirs, and the draw takes the
// first candidate whose running mass passes uniform of what is left.  With
// no cut the draw walks the row in token order, as the reference's does.
//
// Nothing sorts the row.  Each step needs one place in the ranking (the k-th
// candidate, the one that reaches a mass), so the row is spread over 2048
// bins (BinRule) whose order is the ranking's; a scan of the bins' counts and
// masses gives the bin that holds the place, and that bin's candidates alone
// are ranked.  The bins' width follows the row's spread, so a flat row or one
// of equal logits fills them too.  A bin past kRankCap candidates (a crowd of
// near ties below an outlier) is spread over 2048 bins again, of the range its
// (score, token) keys cover, until few enough are left: some passes of one
// workgroup over its candidates.  Four launches:
//   sample_max_kernel      each chunk's largest score, unmasked count and last
//                          unmasked token; the bins cleared
//   sample_bins_kernel     the chunks' masses; the bins' counts and masses
//   sample_gather_kernel   the candidates of the bins that a cut can reach,
//                          bin after bin
//   sample_draw_kernel     one workgroup: the cuts and the draw; where the
//                          gathered candidates are few enough to rank at once,
//                          from their running masses alone (28 -> 5 us there)
// A bin's mass is summed as integers of 2^-32 and 2^-64, so it does not depend
// on the order the atomics land in (and is within 2^-65 a candidate of exact);
// the sums along the ranking are doubles, so only their rounding differs from
// the reference's sequential loop.  The uniform draws come from the caller
// (the top 53 bits of std::mt19937_64 outputs).
//
// The launches are bound by their chains (a read of the chunk's 16 KB, the
// atomics, the scans), not by the row's 1 MB.  A row of 256 000 normal logits
// (sigma 3) at temperature 0.8, top-k 40, top-p 0.95: 46.6 us (4, 14, 12
// and 5 in the kernels; 1 of them for the row's spread); an eight-pass radix
// sort of the row, its one-workgroup scans and the draw over the ranked row
// had taken 811.  256 000 equal logits at temperature 1: 56 us (the sort 724;
// with bins of one width for all rows, all candidates in one of them, 2300).
// 255 999 logits within 1e-5 of each other below an outlier, temperature 4,
// top-k 1000: 717 (the sort 728).
#include "gq8_device.hpp"
#include "gq8_kernels.hpp"
#include "gq8_numerics.hpp"

#include <cfloat>
#include <climits>

namespace gq8 {
namespace {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / 64;
constexpr int kChunkRounds = 4;                                // tokens a thread
constexpr int kChunkTokens = kSampleThreads * kChunkRounds;    // 4096 a workgroup
constexpr int kBins = 2 * kSampleThreads;                      // two a thread in the scans
constexpr int kRankCap = 512;                                  // candidates ranked by counting

struct ChunkState {
    float largest, smallest; // of the chunk's unmasked row_logits but NaNs (-inf, inf where there is none)
    double mass;    // of its weights, in a fixed order
    int count;      // unmasked tokens
    int last;       // the last of them, -1 where there is none
    int bad;        // one that ranks before every number (a +infinity, a NaN of clear sign): no
                    // sum along the ranking is a number
    int nans;       // NaNs with the sign set, which rank after every number
};

// The bins of a row.  A score lies `distance` = top - score below the largest:
// 64 bins a unit up to 16, then 64 an octave (the top bits of the distance as
// a float), the last one for all that lie past 2^20.  Where all scores lie
// within 8 of the largest, distances are scaled by a power of two to fill the
// even bins, and where they tie, the bins go by token (`tokens` each): a flat
// row's candidates do not crowd a few bins.
struct BinRule {
    double top, scale; // bins a unit of distance
    int tokens;        // 0: by distance
};

// The whole row: its chunks together, and its bins.
struct RowState {
    ChunkState all;
    BinRule rule;
};

// What the gather leaves for the draw.
struct Gathered {
    double total; // the row's mass
    uint32_t count;
    uint32_t unused;
};

struct SampleWorkspace {
    ChunkState *chunks;
    RowState *row;
    Gathered *summary;
    uint32_t *counts;   // of the bins
    uint32_t *cursors;  // candidates of a bin gathered so far
    uint64_t *massHi;   // multiples of 2^-32
    uint64_t *massLo;   // multiples of 2^-64
    uint64_t *gathered; // (ranking key, token), bin after bin
    int chunkCount;
};

int sample_chunks(int vocab)
{
    return (vocab + kChunkTokens - 1) / kChunkTokens;
}

size_t align256(size_t n)
{
    return (n + 255) & ~size_t(255);
}

// +0 for a zero (the reference compares scores by value, so -0 and +0 tie)
__device__ inline double candidate_score(float logit, double inverse)
{
    const double s = (double) logit * inverse;
    return s == 0.0 ? 0.0 : s;
}

// A token's logit.  At an infinite temperature the scores are logit * 0, so
// the logits are taken as that: they tie (an infinity is then a NaN).
__device__ inline float row_logit(const SampleArgs &a, int64_t token)
{
    const float logit = a.logits[token];
    return a.temperature < INFINITY ? logit : logit * 0.f;
}

// The ranking key of a candidate: descending in row_logit (the score is
// strictly increasing in it), then ascending in the token.
__device__ inline uint64_t ranking_key(float logit, uint32_t token)
{
    uint32_t u = __float_as_uint(logit == 0.f ? 0.f : logit);
    u = (u >> 31) ? ~u : (u | (1u << 31));
    return ((uint64_t) ~u << 32) | token;
}

__device__ inline float logit_of_key(uint64_t key)
{
    uint32_t u = ~(uint32_t) (key >> 32);
    u = (u >> 31) ? (u & ~(1u << 31)) : ~u;
    return __uint_as_float(u);
}

// The row's largest score, which weighs 1 (the lowest double where all are
// -infinite).
__device__ inline double top_score(const ChunkState &row, double inverse)
{
    return fmax(-DBL_MAX, candidate_score(row.largest, inverse));
}

__device__ inline double candidate_weight(float logit, double inverse, double top)
{
    return exp(candidate_score(logit, inverse) - top);
}

// A NaN with the sign set: ranked after every number.
__device__ inline bool nan_behind(float logit)
{
    return logit != logit && (__float_as_uint(logit) >> 31);
}

__device__ inline BinRule bin_rule(const ChunkState &row, double inverse, int vocab)
{
    BinRule rule{top_score(row, inverse), 64.0, 0};
    const double range = rule.top - candidate_score(row.smallest, inverse);
    if (range == 0.0)
        rule.tokens = (vocab + kBins - 1) / kBins;
    else if (range > 0.0 && range < 8.0)
        rule.scale = ldexp(64.0, min(3 - ilogb(range), 1000));
    return rule;
}

// Never decreasing along the ranking.  A NaN: before every number with the
// sign clear, after with it set, as the ranking key has it (an infinity's
// distance to itself is a NaN of clear sign).
__device__ inline int candidate_bin(float logit, int token, double inverse, const BinRule &rule)
{
    const double steps = (rule.top - candidate_score(logit, inverse)) * rule.scale;
    if (!(steps >= 0.0))
        return nan_behind(logit) ? kBins - 1 : 0;
    if (rule.tokens)
        return token / rule.tokens;
    if (steps < kBins / 2)
        return (int) steps;
    const float f = (float) fmin(steps, 1e30);
    const int octaves = (int) (__float_as_uint(f) >> 17) - (int) (__float_as_uint(kBins / 2) >> 17);
    return min(kBins / 2 + octaves, kBins - 1);
}

// A NaN counts as nothing: it ranks after every number whose sum is used.
__device__ inline void split_mass(double w, uint64_t &hi, uint64_t &lo)
{
    const double scaled = fmax(w, 0.0) * 4294967296.0;
    const double whole = floor(scaled);
    hi = (uint64_t) whole;
    lo = (uint64_t) rint((scaled - whole) * 4294967296.0);
}

__device__ inline double joined_mass(uint64_t hi, uint64_t lo)
{
    return (double) hi * 0x1p-32 + (double) lo * 0x1p-64;
}

struct ScanShared {
    double mass[kSampleWaves];
    uint32_t count[kSampleWaves];
};

// Exclusive prefixes of every thread's (count, mass) over the workgroup, and
// their totals; the order of the sums is fixed.
__device__ inline void workgroup_scan(uint32_t count, double mass, uint32_t &countBefore,
                                      double &massBefore, uint32_t &countTotal, double &massTotal,
                                      ScanShared &sh)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t c = count;
    double m = mass;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t pc = __shfl_up(c, d);
        const double pm = __shfl_up(m, d);
        if (lane >= d) {
            c += pc;
            m = pm + m;
        }
    }
    __syncthreads(); // the previous scan's totals have been read
    if (lane == 63) {
        sh.count[wave] = c;
        sh.mass[wave] = m;
    }
    __syncthreads();
    uint32_t cb = 0, ct = 0;
    double mb = 0.0, mt = 0.0;
#pragma unroll
    for (int w = 0; w < kSampleWaves; ++w) {
        if (w == wave) {
            cb = ct;
            mb = mt;
        }
        ct += sh.count[w];
        mt += sh.mass[w];
    }
    const uint32_t pc = __shfl_up(c, 1);
    const double pm = __shfl_up(m, 1);
    countBefore = cb + (lane > 0 ? pc : 0u);
    massBefore = lane > 0 ? mb + pm : mb;
    countTotal = ct;
    massTotal = mt;
}

// A place in the ranking: the candidate of rank `rank`, or the first whose
// running mass reaches (kReaches) or passes (kPasses) `mass`.
enum PlaceKind { kRank, kReaches, kPasses };
struct Place {
    PlaceKind kind;
    uint32_t rank;
    double mass;
    __device__ bool here(uint32_t countThrough, double massThrough) const
    {
        return kind == kRank ? countThrough > rank
                             : (kind == kReaches ? massThrough >= mass : massThrough > mass);
    }
};

// Candidates before a set and in it.
struct Span {
    uint32_t before, count;
    double massBefore, mass;
    int bin;
};

struct BinShared {
    uint32_t counts[kBins];
    double masses[kBins];
    ScanShared scan;
    int first, last;
    Span span;
};

// The first bin of sh.counts / sh.masses (behind `before` candidates of
// `massBefore`) that holds the place; the last that holds anything where none
// does (the place lies within the sums' rounding of the end).
__device__ inline Span find_bin(BinShared &sh, const Place &place, uint32_t before, double massBefore)
{
    const int t = threadIdx.x;
    const uint32_t c0 = sh.counts[2 * t], c1 = sh.counts[2 * t + 1];
    const double m0 = sh.masses[2 * t], m1 = sh.masses[2 * t + 1];
    uint32_t cb, ct;
    double mb, mt;
    workgroup_scan(c0 + c1, m0 + m1, cb, mb, ct, mt, sh.scan);
    cb += before;
    mb += massBefore;
    if (t == 0) {
        sh.first = INT_MAX;
        sh.last = 0;
    }
    __syncthreads();
    if (c0 && place.here(cb + c0, mb + m0))
        atomicMin(&sh.first, 2 * t);
    else if (c1 && place.here(cb + c0 + c1, mb + m0 + m1))
        atomicMin(&sh.first, 2 * t + 1);
    if (c0 | c1)
        atomicMax(&sh.last, c1 ? 2 * t + 1 : 2 * t);
    __syncthreads();
    const int bin = sh.first == INT_MAX ? sh.last : sh.first;
    if (bin >> 1 == t)
        sh.span = bin & 1 ? Span{cb + c0, c1, mb + m0, m1, bin} : Span{cb, c0, mb, m0, bin};
    __syncthreads();
    const Span s = sh.span;
    __syncthreads(); // sh is rewritten by the next search
    return s;
}

struct RankShared {
    uint64_t massLo[kBins]; // `locate`: multiples of 2^-64 in a bin
    uint64_t keys[kRankCap], sorted[kRankCap];
    double masses[kRankCap];
    ScanShared scan;
    uint64_t low, high;
    uint32_t found, gathered;
    uint32_t rank;
    double mass;
    uint32_t token;
};

struct Candidate {
    uint32_t rank, token;
    double massThrough;
};

// Ranks the candidates of rs.keys[0, n), n <= kRankCap, into rs.sorted (each
// thread's takes its place among the others).
__device__ inline void rank_candidates(RankShared &rs, uint32_t n)
{
    const uint32_t t = threadIdx.x;
    if (t < n) {
        const uint64_t mine = rs.keys[t];
        uint32_t rank = 0;
        for (uint32_t i = 0; i < n; ++i)
            rank += rs.keys[i] < mine ? 1u : 0u;
        rs.sorted[rank] = mine;
    }
    __syncthreads();
}

// use(key) for each of keys[0, size), eight loads a thread in flight.
// kStretches: a thread takes a stretch of its own in place of every 1024th key.
// The loads then touch a line a lane, but the gather leaves a bin's keys
// about in token order, and where scores tie, neighbours share a bin of the
// search, whose LDS atomics a whole wave would make one after another.
template <bool kStretches, typename Use>
__device__ inline void each_key(const uint64_t *keys, uint32_t size, Use use)
{
    constexpr uint32_t kLoads = 8;
    constexpr uint32_t kStep = kStretches ? 1u : (uint32_t) kSampleThreads;
    const uint32_t batches = (size + kLoads * kSampleThreads - 1) / (kLoads * kSampleThreads);
    const uint32_t first = threadIdx.x * (kStretches ? kLoads * batches : 1u);
    for (uint32_t n = 0; n < batches; ++n) {
        const uint32_t i0 = first + n * kLoads * kStep;
        uint64_t k[kLoads];
#pragma unroll
        for (uint32_t r = 0; r < kLoads; ++r)
            k[r] = keys[min(i0 + r * kStep, size - 1)];
#pragma unroll
        for (uint32_t r = 0; r < kLoads; ++r)
            if (i0 + r * kStep < size)
                use(k[r]);
    }
}

// The place's candidate among those of `span` (contiguous in `keys`).  Keys
// are distinct, so every pass of the search leaves fewer of them; it ends on
// any content (the key range at least halves a pass) and ranks no more than
// rs.keys holds.
__device__ inline Candidate locate(const uint64_t *keys, Span span, const Place &place,
                                   double inverse, double top, BinShared &bs, RankShared &rs)
{
    const int t = threadIdx.x;
    const uint32_t size = span.count; // of `keys`
    uint64_t low = 0, high = ~0ull;   // the set: keys in [low, high]
    while (span.count > (uint32_t) kRankCap) {
        // the range the set's keys cover, in 2048 bins of a power of two
        if (t == 0) {
            rs.low = ~0ull;
            rs.high = 0ull;
        }
        for (int b = t; b < kBins; b += kSampleThreads) {
            bs.counts[b] = 0u;
            bs.masses[b] = 0.0; // all bits clear
            rs.massLo[b] = 0ull;
        }
        __syncthreads();
        uint64_t lo = ~0ull, hi = 0ull;
        each_key<false>(keys, size, [&](uint64_t k) {
            if (k >= low && k <= high) {
                lo = k < lo ? k : lo;
                hi = k > hi ? k : hi;
            }
        });
        atomicMin((unsigned long long *) &rs.low, (unsigned long long) lo);
        atomicMax((unsigned long long *) &rs.high, (unsigned long long) hi);
        __syncthreads();
        low = rs.low;
        high = rs.high;
        if (low >= high)
            break;
        int shift = 0;
        while (((high - low) >> shift) >= (uint64_t) kBins)
            ++shift;
        // a candidate's mass as integers, so the sums' order does not matter
        uint64_t *massHi = reinterpret_cast<uint64_t *>(bs.masses);
        each_key<true>(keys, size, [&](uint64_t k) {
            if (k < low || k > high)
                return;
            const int b = (int) ((k - low) >> shift);
            uint64_t mh, ml;
            split_mass(candidate_weight(logit_of_key(k), inverse, top), mh, ml);
            atomicAdd(&bs.counts[b], 1u);
            if (mh)
                atomicAdd((unsigned long long *) &massHi[b], (unsigned long long) mh);
            if (ml)
                atomicAdd((unsigned long long *) &rs.massLo[b], (unsigned long long) ml);
        });
        __syncthreads();
        for (int b = t; b < kBins; b += kSampleThreads)
            bs.masses[b] = joined_mass(massHi[b], rs.massLo[b]);
        __syncthreads();
        span = find_bin(bs, place, span.before, span.massBefore);
        low += (uint64_t) span.bin << shift;
        const uint64_t reach = (1ull << shift) - 1; // low + reach may pass 2^64
        high = high - low < reach ? high : low + reach;
    }
    // few enough: each thread's candidate takes its place among the others
    if (t == 0) {
        rs.gathered = 0u;
        rs.found = UINT_MAX;
    }
    __syncthreads();
    each_key<false>(keys, size, [&](uint64_t k) {
        if (k >= low && k <= high) {
            const uint32_t at = atomicAdd(&rs.gathered, 1u);
            if (at < (uint32_t) kRankCap)
                rs.keys[at] = k;
        }
    });
    __syncthreads();
    const uint32_t n = min(rs.gathered, (uint32_t) kRankCap);
    rank_candidates(rs, n);
    double weight = 0.0;
    if (t < (int) n)
        weight = candidate_weight(logit_of_key(rs.sorted[t]), inverse, top);
    uint32_t cb, ct;
    double mb, mt;
    workgroup_scan(t < (int) n ? 1u : 0u, weight, cb, mb, ct, mt, rs.scan);
    const uint32_t through = span.before + cb + 1;
    const double massThrough = span.massBefore + (mb + weight);
    if (t < (int) n && (place.here(through, massThrough) || t == (int) n - 1))
        atomicMin(&rs.found, (uint32_t) t); // the last where none holds it: within rounding
    __syncthreads();
    if (t == (int) rs.found) {
        rs.rank = through - 1;
        rs.mass = massThrough;
        rs.token = (uint32_t) rs.sorted[t];
    }
    __syncthreads();
    const Candidate c{rs.rank, rs.token, rs.mass};
    __syncthreads(); // rs is rewritten by the next search
    return c;
}

// The whole row's state from its chunks' (every thread takes part).
__device__ inline ChunkState row_state(const ChunkState *chunks, int count)
{
    __shared__ float sLargest[kSampleWaves], sSmallest[kSampleWaves];
    __shared__ int sCount, sLast, sBad, sNans;
    const int t = threadIdx.x;
    if (t == 0) {
        sCount = 0;
        sLast = -1;
        sBad = 0;
        sNans = 0;
    }
    __syncthreads();
    float largest = -INFINITY, smallest = INFINITY;
    for (int i = t; i < count; i += kSampleThreads) {
        const ChunkState c = chunks[i];
        largest = fmaxf(largest, c.largest);
        smallest = fminf(smallest, c.smallest);
        atomicAdd(&sCount, c.count);
        atomicMax(&sLast, c.last);
        if (c.bad)
            atomicOr(&sBad, 1);
        if (c.nans)
            atomicAdd(&sNans, c.nans);
    }
    largest = max_lanes<32>(largest);
    smallest = -max_lanes<32>(-smallest);
    if ((t & 63) == 0) {
        sLargest[t >> 6] = largest;
        sSmallest[t >> 6] = smallest;
    }
    __syncthreads();
    ChunkState s{};
    s.largest = -INFINITY;
    s.smallest = INFINITY;
    for (int w = 0; w < kSampleWaves; ++w) {
        s.largest = fmaxf(s.largest, sLargest[w]);
        s.smallest = fminf(s.smallest, sSmallest[w]);
    }
    s.count = sCount;
    s.last = sLast;
    s.bad = sBad;
    s.nans = sNans;
    return s;
}

__device__ inline bool masked(const SampleArgs &a, int token)
{
    return a.mask && a.mask[token] != 0.f;
}

__global__ __launch_bounds__(kSampleThreads) void sample_max_kernel(SampleArgs a, SampleWorkspace w)
{
    __shared__ float sLargest[kSampleWaves], sSmallest[kSampleWaves];
    __shared__ int sCount, sLast, sBad, sNans;
    const int t = threadIdx.x;
    for (int b = blockIdx.x * kSampleThreads + t; b < kBins; b += gridDim.x * kSampleThreads) {
        w.counts[b] = 0u;
        w.cursors[b] = 0u;
        w.massHi[b] = 0ull;
        w.massLo[b] = 0ull;
    }
    if (t == 0) {
        sCount = 0;
        sLast = -1;
        sBad = 0;
        sNans = 0;
    }
    __syncthreads();
    const int64_t first = (int64_t) blockIdx.x * kChunkTokens + t;
    float logit[kChunkRounds];
    bool live[kChunkRounds];
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        const int64_t e = first + r * kSampleThreads;
        live[r] = e < a.vocab && !masked(a, (int) e);
        logit[r] = row_logit(a, e < a.vocab ? e : 0);
    }
    float largest = -INFINITY, smallest = INFINITY;
    int count = 0, last = -1, bad = 0, nans = 0;
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r)
        if (live[r]) {
            largest = fmaxf(largest, logit[r]);
            smallest = fminf(smallest, logit[r]);
            ++count;
            last = (int) (first + r * kSampleThreads);
            const bool behind = nan_behind(logit[r]);
            nans += behind;
            bad |= !(logit[r] < INFINITY) && !behind;
        }
    largest = max_lanes<32>(largest);
    smallest = -max_lanes<32>(-smallest);
    const double deepest = wave_max_d((double) last); // exact: below 2^31
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        count += __shfl_xor(count, d);
    const bool anyBad = __any(bad) != 0;
    if (nans)
        atomicAdd(&sNans, nans);
    if ((t & 63) == 0) { // one atomic a wave
        sLargest[t >> 6] = largest;
        sSmallest[t >> 6] = smallest;
        atomicAdd(&sCount, count);
        atomicMax(&sLast, (int) deepest);
        if (anyBad)
            atomicOr(&sBad, 1);
    }
    __syncthreads();
    if (t == 0) {
        for (int i = 1; i < kSampleWaves; ++i) {
            largest = fmaxf(largest, sLargest[i]);
            smallest = fminf(smallest, sSmallest[i]);
        }
        w.chunks[blockIdx.x] = ChunkState{largest, smallest, 0.0, sCount, sLast, sBad, sNans};
    }
}

__global__ __launch_bounds__(kSampleThreads) void sample_bins_kernel(SampleArgs a, SampleWorkspace w,
                                                                     int ranked)
{
    __shared__ uint32_t sCounts[kBins];
    __shared__ unsigned long long sHi[kBins], sLo[kBins];
    __shared__ ScanShared sScan;
    const int t = threadIdx.x;
    const int64_t first = (int64_t) blockIdx.x * kChunkTokens + t;
    float logit[kChunkRounds];
    bool live[kChunkRounds];
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        const int64_t e = first + r * kSampleThreads;
        live[r] = e < a.vocab && !masked(a, (int) e);
        logit[r] = row_logit(a, e < a.vocab ? e : 0);
    }
    if (ranked)
        for (int b = t; b < kBins; b += kSampleThreads) {
            sCounts[b] = 0u;
            sHi[b] = 0ull;
            sLo[b] = 0ull;
        }
    const ChunkState row = row_state(w.chunks, w.chunkCount); // (syncs)
    const double inverse = 1.0 / (double) a.temperature;
    const BinRule rule = bin_rule(row, inverse, a.vocab);
    double mass = 0.0;
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        if (!live[r])
            continue;
        const double weight = candidate_weight(logit[r], inverse, rule.top);
        mass += weight;
        if (ranked) {
            const int b = candidate_bin(logit[r], (int) (first + r * kSampleThreads), inverse, rule);
            uint64_t hi = 0, lo = 0;
            if (!row.bad) // else no mass is a number, and none is used
                split_mass(weight, hi, lo);
            atomicAdd(&sCounts[b], 1u);
            if (hi)
                atomicAdd(&sHi[b], (unsigned long long) hi);
            if (lo)
                atomicAdd(&sLo[b], (unsigned long long) lo);
        }
    }
    uint32_t cb, ct;
    double mb, mt;
    workgroup_scan(0u, mass, cb, mb, ct, mt, sScan); // (syncs)
    if (t == 0) {
        w.chunks[blockIdx.x].mass = mt;
        if (blockIdx.x == 0)
            *w.row = RowState{row, rule};
    }
    if (ranked)
        for (int b = t; b < kBins; b += kSampleThreads)
            if (sCounts[b]) {
                atomicAdd(&w.counts[b], sCounts[b]);
                atomicAdd((unsigned long long *) &w.massHi[b], sHi[b]);
                atomicAdd((unsigned long long *) &w.massLo[b], sLo[b]);
            }
}

__device__ inline void load_bins(const SampleWorkspace &w, BinShared &sh)
{
    for (int b = threadIdx.x; b < kBins; b += kSampleThreads) {
        sh.counts[b] = w.counts[b];
        sh.masses[b] = joined_mass(w.massHi[b], w.massLo[b]);
    }
    __syncthreads();
}

// Whether any cut applies to a row of n candidates, and how many the first
// keeps.
__device__ inline bool cut(const SampleArgs &a, int n)
{
    return (a.top_k > 0 && a.top_k < n) || a.top_p < 1.f;
}

__device__ inline int first_kept(const SampleArgs &a, int n)
{
    return a.top_k > 0 && a.top_k < n ? a.top_k : n;
}

// Whether the weights of the first `kept` ranked candidates are numbers.
__device__ inline bool weights_are_numbers(const ChunkState &row, int kept)
{
    return !row.bad && kept <= row.count - row.nans;
}

__global__ __launch_bounds__(kSampleThreads) void sample_gather_kernel(SampleArgs a, SampleWorkspace w)
{
    __shared__ BinShared sh;
    __shared__ uint32_t sOffset[kBins], sMine[kBins], sBase[kBins];
    const int t = threadIdx.x;
    const int64_t first = (int64_t) blockIdx.x * kChunkTokens + t;
    float logit[kChunkRounds];
    bool live[kChunkRounds];
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        const int64_t e = first + r * kSampleThreads;
        live[r] = e < a.vocab && !masked(a, (int) e);
        logit[r] = row_logit(a, e < a.vocab ? e : 0);
    }
    const ChunkState row = w.row->all;
    const BinRule rule = w.row->rule;
    const int n = row.count;
    if (n == 0 || !cut(a, n))
        return;
    const double inverse = 1.0 / (double) a.temperature;
    load_bins(w, sh);
    // the bins' places, and the last bin that the draw reads: the k-th
    // candidate's (whose mass the other searches need), else the one where the
    // row's mass reaches p, else the last candidate's
    uint32_t cb, ct;
    double mb, mt;
    workgroup_scan(sh.counts[2 * t] + sh.counts[2 * t + 1], sh.masses[2 * t] + sh.masses[2 * t + 1], cb,
                   mb, ct, mt, sh.scan);
    sOffset[2 * t] = cb;
    sOffset[2 * t + 1] = cb + sh.counts[2 * t];
    sMine[2 * t] = 0u;
    sMine[2 * t + 1] = 0u;
    const int kept = first_kept(a, n);
    const bool byMass = kept == n && weights_are_numbers(row, n) && mt > 0.0;
    const Place end{byMass ? kReaches : kRank, (uint32_t) kept - 1u,
                    (double) a.top_p * mt * (1.0 + 1e-9)};
    const Span lastSpan = find_bin(sh, end, 0u, 0.0);
    const int lastBin = lastSpan.bin;
    if (blockIdx.x == 0 && t == 0)
        *w.summary = Gathered{mt, lastSpan.before + lastSpan.count, 0u};
    int bin[kChunkRounds];
    uint32_t place[kChunkRounds];
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        bin[r] = live[r] ? candidate_bin(logit[r], (int) (first + r * kSampleThreads), inverse, rule)
                         : kBins;
        if (bin[r] <= lastBin)
            place[r] = atomicAdd(&sMine[bin[r]], 1u);
    }
    __syncthreads();
    for (int b = t; b <= lastBin; b += kSampleThreads)
        if (sMine[b])
            sBase[b] = sOffset[b] + atomicAdd(&w.cursors[b], sMine[b]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r)
        if (bin[r] <= lastBin)
            w.gathered[sBase[bin[r]] + place[r]] =
                ranking_key(logit[r], (uint32_t) (first + r * kSampleThreads));
}

// The first token, in token order, whose running mass passes `target` (the
// chunks' masses, then the chunk's own weights); -1 where none does.
__device__ inline int token_order_draw(const SampleArgs &a, const SampleWorkspace &w, double uniform,
                                       double inverse, double top, ScanShared &scan)
{
    __shared__ int sFirst;
    __shared__ double sBefore;
    const int t = threadIdx.x;
    const int per = (w.chunkCount + kSampleThreads - 1) / kSampleThreads;
    const int c0 = min(t * per, w.chunkCount), c1 = min(c0 + per, w.chunkCount);
    double mass = 0.0;
    for (int i = c0; i < c1; ++i)
        mass += w.chunks[i].mass;
    uint32_t cb, ct;
    double before, total;
    workgroup_scan(0u, mass, cb, before, ct, total, scan);
    if (t == 0)
        sFirst = INT_MAX;
    __syncthreads();
    const double target = uniform * total;
    double through = before;
    for (int i = c0; i < c1; ++i) {
        through += w.chunks[i].mass;
        if (through > target) {
            atomicMin(&sFirst, i);
            break;
        }
    }
    __syncthreads();
    const int chunk = sFirst;
    __syncthreads();
    if (chunk == INT_MAX)
        return -1;
    if (chunk >= c0 && chunk < c1) {
        double b = before;
        for (int i = c0; i < chunk; ++i)
            b += w.chunks[i].mass;
        sBefore = b;
    }
    if (t == 0)
        sFirst = INT_MAX;
    __syncthreads();
    // kChunkRounds consecutive tokens a thread
    double weight[kChunkRounds], sum = 0.0;
    int last = -1;
    const int64_t first = (int64_t) chunk * kChunkTokens + t * kChunkRounds;
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        const int64_t e = first + r;
        const bool live = e < a.vocab && !masked(a, (int) e);
        weight[r] = live ? candidate_weight(row_logit(a, e), inverse, top) : 0.0;
        sum += weight[r];
        last = weight[r] > 0.0 ? (int) e : last;
    }
    double mine, all;
    workgroup_scan(0u, sum, cb, mine, ct, all, scan);
    __shared__ int sLast;
    if (t == 0)
        sLast = -1;
    __syncthreads();
    atomicMax(&sLast, last);
    double running = sBefore + mine;
#pragma unroll
    for (int r = 0; r < kChunkRounds; ++r) {
        running += weight[r];
        if (weight[r] > 0.0 && running > target) {
            atomicMin(&sFirst, (int) (first + r));
            break;
        }
    }
    __syncthreads();
    // the chunk's sum in this order may round below the target it passed
    return sFirst == INT_MAX ? sLast : sFirst;
}

// The cuts and the draw where every gathered candidate fits one ranking (a
// top-k of some hundred, a peaked row): their running masses once, then each
// place by a comparison a candidate.
__device__ inline uint32_t few_candidates_draw(const SampleArgs &a, const SampleWorkspace &w, int n,
                                               double uniform, double inverse, double top,
                                               RankShared &rs)
{
    const uint32_t t = threadIdx.x, count = w.summary->count;
    if (t < count)
        rs.keys[t] = w.gathered[t];
    __syncthreads();
    rank_candidates(rs, count);
    const double weight = t < count ? candidate_weight(logit_of_key(rs.sorted[t]), inverse, top) : 0.0;
    uint32_t cb, ct;
    double before, all;
    workgroup_scan(0u, weight, cb, before, ct, all, rs.scan);
    const double through = before + weight;
    if (t < count)
        rs.masses[t] = through;
    // the first candidate that holds a place, `count` where none does
    auto first = [&](const Place &place) {
        __syncthreads(); // (also: the masses are in)
        if (t == 0)
            rs.found = count;
        __syncthreads();
        if (t < count && place.here(t + 1, through))
            atomicMin(&rs.found, t);
        __syncthreads();
        return rs.found;
    };
    __syncthreads();
    uint32_t kept = (uint32_t) first_kept(a, n);
    double mass = kept < (uint32_t) n ? rs.masses[kept - 1] : w.summary->total;
    if (a.top_p < 1.f) {
        const uint32_t at = first(Place{kReaches, 0u, (double) a.top_p * mass});
        if (at + 1 < kept) {
            kept = min(at + 1, count); // the last gathered where rounding leaves none
            mass = rs.masses[kept - 1];
        }
    }
    kept = min(kept, count);
    const uint32_t at = first(Place{kPasses, 0u, uniform * mass});
    return (uint32_t) rs.sorted[at < kept ? at : kept - 1];
}

__global__ __launch_bounds__(kSampleThreads) void sample_draw_kernel(SampleArgs a, SampleWorkspace w)
{
    __shared__ BinShared bins;
    __shared__ RankShared ranks;
    const int t = threadIdx.x;
    const double uniform = a.draws ? a.draws[min(*a.draw_index, a.draw_count - 1)] : a.uniform;
    const ChunkState row = w.row->all;
    const double inverse = 1.0 / (double) a.temperature, top = w.row->rule.top;
    const int n = row.count;
    uint32_t chosen = 0;
    if (n > 0 && !cut(a, n)) {
        const int at = !weights_are_numbers(row, n) ? -1 : token_order_draw(a, w, uniform, inverse, top, bins.scan);
        chosen = (uint32_t) (at >= 0 ? at : row.last);
    } else if (n > 0 && weights_are_numbers(row, first_kept(a, n)) && w.summary->total > 0.0
               && w.summary->count <= (uint32_t) kRankCap) {
        chosen = few_candidates_draw(a, w, n, uniform, inverse, top, ranks);
    } else if (n > 0) {
        load_bins(w, bins);
        uint32_t cb, ct;
        double mb, all;
        workgroup_scan(0u, bins.masses[2 * t] + bins.masses[2 * t + 1], cb, mb, ct, all, bins.scan);
        int kept = first_kept(a, n);
        const bool sums = weights_are_numbers(row, kept) && all > 0.0; // else no running mass is a number
        double mass = all;
        Candidate end{}, drawn{};
        bool known = false; // `end` is the last kept candidate
        bool found = false;
        // the places one after another, in a loop so that the search is there once
        enum { kTopK, kTopP, kDraw, kEnd };
        for (int step = kTopK; step <= kEnd; ++step) {
            const bool wanted = step == kTopK   ? kept < n
                                : step == kTopP ? sums && a.top_p < 1.f
                                : step == kDraw ? sums
                                                : !found && !known;
            if (!wanted)
                continue;
            const Place place = step == kTopP   ? Place{kReaches, 0u, (double) a.top_p * mass}
                                : step == kDraw ? Place{kPasses, 0u, uniform * mass}
                                                : Place{kRank, (uint32_t) kept - 1u, 0.0};
            // its bin, and the candidate among the bin's gathered ones.  The
            // bins' running masses and `mass` are different sums of the same
            // weights: the largest draws may lie past the last kept
            // candidate's bin, where nothing is kept (or gathered)
            const Span span = find_bin(bins, place, 0u, 0.0);
            if (step == kDraw && (int) span.before >= kept)
                continue;
            const Candidate c = locate(w.gathered + span.before, span, place, inverse, top, bins, ranks);
            if (span.count > (uint32_t) kRankCap) // `locate` has used the bins' space
                load_bins(w, bins);
            if (step == kDraw) {
                drawn = c;
                found = (int) c.rank < kept;
            } else if (step != kTopP || (int) c.rank < kept - 1 || !known) {
                end = c;
                known = true;
                kept = (int) c.rank + 1;
                mass = c.massThrough;
            }
        }
        chosen = found ? drawn.token : end.token;
    }
    if (t == 0) {
        if (a.sequence)
            a.sequence[*a.position + a.offset] = chosen;
        if (a.token_out)
            *a.token_out = chosen;
        if (a.draws)
            *a.draw_index += 1;
    }
}

SampleWorkspace carve(void *workspace, int vocab)
{
    SampleWorkspace w{};
    w.chunkCount = sample_chunks(vocab);
    uint8_t *p = reinterpret_cast<uint8_t *>(align256(reinterpret_cast<uintptr_t>(workspace)));
    auto take = [&](size_t bytes) {
        uint8_t *at = p;
        p += align256(bytes);
        return at;
    };
    w.row = reinterpret_cast<RowState *>(take(sizeof(RowState)));
    w.summary = reinterpret_cast<Gathered *>(take(sizeof(Gathered)));
    w.chunks = reinterpret_cast<ChunkState *>(take(w.chunkCount * sizeof(ChunkState)));
    w.counts = reinterpret_cast<uint32_t *>(take(kBins * sizeof(uint32_t)));
    w.cursors = reinterpret_cast<uint32_t *>(take(kBins * sizeof(uint32_t)));
    w.massHi = reinterpret_cast<uint64_t *>(take(kBins * sizeof(uint64_t)));
    w.massLo = reinterpret_cast<uint64_t *>(take(kBins * sizeof(uint64_t)));
    w.gathered = reinterpret_cast<uint64_t *>(p);
    return w;
}

} // namespace

size_t sample_workspace_bytes(int vocab)
{
    if (vocab <= 0)
        return 0;
    return align256(sizeof(RowState)) + align256(sizeof(Gathered)) + align256(sample_chunks(vocab) * sizeof(ChunkState))
           + 2 * align256(kBins * sizeof(uint32_t)) + 2 * align256(kBins * sizeof(uint64_t))
           + align256((size_t) vocab * sizeof(uint64_t)) + 256; // and its alignment
}

bool sampling_options_valid(float temperature, int top_k, float top_p)
{
    // Sampler.cpp:28-41, spelled so that a NaN is refused
    return temperature >= 0.f && top_k >= 0 && top_p > 0.f && top_p <= 1.f;
}

hipError_t launch_sample(const SampleArgs &a, void *workspace, size_t workspace_bytes,
                         hipStream_t stream)
{
    if (!a.logits || a.vocab <= 0 || (a.draws && (a.draw_count <= 0 || !a.draw_index))
        || !(a.temperature > 0.f)
        || !sampling_options_valid(a.temperature, a.top_k, a.top_p)
        || (!a.sequence && !a.token_out) || (a.sequence && !a.position) || !workspace
        || workspace_bytes < sample_workspace_bytes(a.vocab))
        return hipErrorInvalidValue;
    const SampleWorkspace w = carve(workspace, a.vocab);
    const bool ranked = a.top_k > 0 || a.top_p < 1.f;
    const dim3 grid(w.chunkCount), block(kSampleThreads);
    hipLaunchKernelGGL(sample_max_kernel, grid, block, 0, stream, a, w);
    hipLaunchKernelGGL(sample_bins_kernel, grid, block, 0, stream, a, w, ranked ? 1 : 0);
    if (ranked)
        hipLaunchKernelGGL(sample_gather_kernel, grid, block, 0, stream, a, w);
    hipLaunchKernelGGL(sample_draw_kernel, dim3(1), block, 0, stream, a, w);
    return hipGetLastError();
}

} // namespace gq8
