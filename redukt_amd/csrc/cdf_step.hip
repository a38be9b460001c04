// Logits -> u32 CDF on the GPU, bit for bit the host coding path's cdf_from_logits
// (src/application/codec.rs:785-798 with Cdf::from_probs, src/domain/coder.rs:43-81, and
// the table-driven f64 exp of src/domain/fmath.rs:340-430).
//
// Every frequency depends on the last bit of every f64 operation, so the arithmetic is
// the host's operation for operation (contraction off below): the same exp (integer bit
// manipulation plus IEEE double adds and multiplies, one rounding each), the same
// products and conversions.  Three things are order-dependent and are kept in order:
//   * the two f64 sums (sum of exp, then sum of the f32 probabilities): each is one
//     sequential chain of adds in index order, formed exactly by one workgroup per row in
//     integer rounds on the running sum's grid (k_cdf_sums);
//   * the argmax of the fix-up takes the last of equal maxima, a reduction whose result
//     does not depend on the order it is combined in;
//   * `used` and the cumulative frequencies are integer sums (exact in any order).
// Everything else is element-wise and runs on every lane.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "host/exp_table.h"
#include "step.h"

#pragma clang fp contract(off)

namespace rdk {
namespace {

constexpr uint32_t kCdfTotal = 1u << 24;   // REDUKT_CDF_TOTAL
constexpr int kCdfBlock = 256;

__device__ __forceinline__ double as_f64(uint64_t b) { return __longlong_as_double((long long)b); }
__device__ __forceinline__ uint64_t as_u64(double d) { return (uint64_t)__double_as_longlong(d); }

// The host's 2^(k/128) table (generated from decimal arithmetic), copied into constant
// memory at compile time.
template <size_t... I>
struct ExpTable {
    uint64_t v[sizeof...(I)];
};
template <size_t... I>
constexpr ExpTable<I...> exp_table(std::index_sequence<I...>) {
    return ExpTable<I...>{{redukt_exp::kTable[I]...}};
}
__constant__ const auto c_exp = exp_table(std::make_index_sequence<256>{});

// exp(x) in f64, the host's redukt_exp_f64 (fmath.rs:383-430): x = k ln2/128 + r,
// e^x = 2^(k/128) e^r with the 128-entry table, a degree-5 polynomial for e^r - 1 - r,
// and the host's paths for tiny, huge and subnormal results.
__device__ double exp_out_of_range(double x, uint32_t abstop) {
    if (as_u64(x) == 0xfff0000000000000ULL) return 0.0;   // -inf
    if (abstop >= 0x7ff) return 1.0 + x;                  // +inf stays +inf, NaN propagates
    return (as_u64(x) >> 63) ? 0.0 : __longlong_as_double(0x7ff0000000000000LL);
}

__device__ double exp_rescale(double tmp, uint64_t sbits, uint64_t ki) {
    if ((ki & 0x80000000ULL) == 0) {
        const double scale = as_f64(sbits - (1009ULL << 52));
        return as_f64(uint64_t(1009 + 1023) << 52) * (scale + scale * tmp);
    }
    const double scale = as_f64(sbits + (1022ULL << 52));
    double y = scale + scale * tmp;
    if (y < 1.0) {
        double lo = scale - y + scale * tmp;
        const double hi = 1.0 + y;
        lo = 1.0 - hi + y + lo;
        y = (hi + lo) - 1.0;
        if (y == 0.0) y = 0.0;
    }
    return as_f64(1ULL << 52) * y;
}

__device__ double exp_f64(double x, const uint64_t* __restrict__ table) {
    constexpr uint64_t kPoly[4] = {0x3fdffffffffffdbdULL, 0x3fc555555555543cULL, 0x3fa55555cf172b91ULL,
                                   0x3f81111167a4d017ULL};
    constexpr uint64_t kShiftBits = 0x4338000000000000ULL;
    uint32_t abstop = uint32_t(as_u64(x) >> 52) & 0x7ff;
    bool rescale = false;
    if (abstop - 0x3c9u >= 0x408u - 0x3c9u) {
        if (abstop - 0x3c9u >= 0x80000000u) return 1.0 + x;
        if (abstop >= 0x409u) return exp_out_of_range(x, abstop);
        rescale = true;
    }
    const double z = as_f64(redukt_exp::kInvLn2N) * x;
    double kd = z + as_f64(kShiftBits);
    const uint64_t ki = as_u64(kd);
    kd -= as_f64(kShiftBits);
    const double r = x + kd * as_f64(redukt_exp::kNegLn2HiN) + kd * as_f64(redukt_exp::kNegLn2LoN);
    const uint64_t idx = 2 * (ki & 127);
    const uint64_t top = ki << 45;
    const double tail = as_f64(table[idx]);
    const uint64_t sbits = table[idx + 1] + top;
    const double r2 = r * r;
    const double tmp = tail + r + r2 * (as_f64(kPoly[0]) + r * as_f64(kPoly[1])) +
                       r2 * r2 * (as_f64(kPoly[2]) + r * as_f64(kPoly[3]));
    if (rescale) return exp_rescale(tmp, sbits, ki);
    const double scale = as_f64(sbits);
    return scale + scale * tmp;
}

// One row's f32 probability, the host's p[i] = float(e[i] * inv_sum).
__device__ __forceinline__ float prob_of(double e, double inv_sum) { return (float)(e * inv_sum); }

constexpr uint32_t kSpan = 16;                      // consecutive elements per thread in a chunk
constexpr uint32_t kChunk = kSpan * kCdfBlock;      // elements per chunk workgroup
constexpr uint32_t kTerms = 4;                      // consecutive elements per lane of a segment
constexpr uint32_t kSegTerms = 64 * kTerms;         // elements of a segment of the sums: one wave's
__host__ __device__ constexpr uint32_t segments(uint32_t n) { return (n + kSegTerms - 1) / kSegTerms; }

struct ChunkPart {
    double max;        // the chunk's max (NaN loses; -inf if none)
    uint64_t used;     // sum of the chunk's extra frequencies
    uint64_t best;     // (largest frequency << 32) | its last index
};

struct CdfArgs {
    const float* logits;   // [rows][n]
    uint32_t rows, n, chunks;
    double* e;             // [rows][n] scratch: exp(logit - max)
    double* sums;          // [rows] scratch: the sum of the probabilities
    double* seg;           // [rows][segments] scratch: sum of each kSegTerms elements of e, in any order
    ChunkPart* part;       // [rows][chunks] scratch
    uint32_t* cdf;         // [rows][n + 1]; k_cdf_sums leaves probability i's bits in element i + 1
};

// Block-wide reductions over kCdfBlock threads (four waves of 64).
template <class T, class F>
__device__ T block_reduce(T v, F op, T* sh) {
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const T u = __shfl_xor(v, o);
        v = op(v, u);
    }
    if (lane == 0) sh[w] = v;
    __syncthreads();
    T r = sh[0];
#pragma unroll
    for (int i = 1; i < kCdfBlock / 64; i++) r = op(r, sh[i]);
    __syncthreads();
    return r;
}

// A 64-bit value moved across lanes by DPP (each 32-bit half; lanes without a source
// read 0): a few cycles, against an LDS round trip for a lane permute.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = as_u64(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
    return as_f64(((uint64_t)hi << 32) | lo);
}

// Inclusive prefix sum over the wave's 64 lanes: shifts by 1, 2, 4, 8 within each row of
// 16 lanes, then the last lane of row 0 / 2 into rows 1 / 3 and lane 31 into rows 2 and 3.
__device__ __forceinline__ double wave_incl_sum(double v) {
    v += dpp_f64<0x111>(v);          // row_shr:1
    v += dpp_f64<0x112>(v);          // row_shr:2
    v += dpp_f64<0x114>(v);          // row_shr:4
    v += dpp_f64<0x118>(v);          // row_shr:8
    v += dpp_f64<0x142, 0xa>(v);     // row_bcast:15 into rows 1 and 3
    v += dpp_f64<0x143, 0xc>(v);     // row_bcast:31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ double max_nan_loses(double m, double v) { return (!isnan(v) && !(v <= m)) ? v : m; }

// A row whose logits start on 16 bytes: its chunks are read four elements a lane.
__device__ __forceinline__ bool vec_row(const float* l) { return ((uintptr_t)l & 15) == 0; }

// Phase 1a (chunk c of row r): the chunk's max (f64::max folding, NaN loses).
__global__ __launch_bounds__(kCdfBlock) void k_cdf_max(CdfArgs a) {
    __shared__ double sh[kCdfBlock / 64];
    const uint32_t c = blockIdx.x, row = blockIdx.y, n = a.n;
    const float* l = a.logits + (size_t)row * n;
    double m = -__longlong_as_double(0x7ff0000000000000LL);
    const uint32_t i0 = c * kChunk, i1 = min(n, (c + 1) * kChunk);
    if (vec_row(l)) {
        // four consecutive elements a lane (chunks start at multiples of 4)
        for (uint32_t i = i0 + 4 * threadIdx.x; i < i1; i += 4 * kCdfBlock) {
            if (i + 4 <= i1) {
                const float4 v = *(const float4*)(l + i);
                m = max_nan_loses(max_nan_loses(m, (double)v.x), (double)v.y);
                m = max_nan_loses(max_nan_loses(m, (double)v.z), (double)v.w);
            } else {
                for (uint32_t k = i; k < i1; k++) m = max_nan_loses(m, (double)l[k]);
            }
        }
    } else {
        for (uint32_t i = i0 + threadIdx.x; i < i1; i += kCdfBlock) m = max_nan_loses(m, (double)l[i]);
    }
    // every partial is -inf or a number, so the combination order does not matter
    m = block_reduce<double>(m, [](double x, double y) { return (y <= x) ? x : y; }, sh);
    if (threadIdx.x == 0) a.part[(size_t)row * a.chunks + c].max = m;
}

// Phase 1b (chunk c of row r): the row's max from the chunk maxima, then e = exp(logit - max),
// and each segment's sum of e (a wave's elements of one iteration), which only guides
// k_cdf_sums.
__global__ __launch_bounds__(kCdfBlock) void k_cdf_exp(CdfArgs a) {
    const uint32_t c = blockIdx.x, row = blockIdx.y, n = a.n;
    const ChunkPart* pr = a.part + (size_t)row * a.chunks;
    double m = pr[0].max;
    for (uint32_t i = 1; i < a.chunks; i++) m = (pr[i].max <= m) ? m : pr[i].max;
    const float* l = a.logits + (size_t)row * n;
    double* e = a.e + (size_t)row * n;
    double* seg = a.seg + (size_t)row * segments(n);
    const uint32_t lane = threadIdx.x % 64;
    const bool vec = vec_row(l) && ((uintptr_t)e & 15) == 0;
    for (uint32_t s0 = c * kChunk + threadIdx.x / 64 * kSegTerms; s0 < min(n, (c + 1) * kChunk);
         s0 += kCdfBlock / 64 * kSegTerms) {
        double sum = 0.0;
        const uint32_t i = s0 + kTerms * lane;
        if (vec && i + 4 <= n) {
            const float4 v = *(const float4*)(l + i);
            const double2 p = make_double2(exp_f64((double)v.x - m, c_exp.v), exp_f64((double)v.y - m, c_exp.v));
            const double2 q = make_double2(exp_f64((double)v.z - m, c_exp.v), exp_f64((double)v.w - m, c_exp.v));
            *(double2*)(e + i) = p;
            *(double2*)(e + i + 2) = q;
            sum = (p.x + p.y) + (q.x + q.y);
        } else {
            // a row that starts off 16 bytes (element s0 + lane + 64 k), or the row's last elements
            const uint32_t first = vec ? i : s0 + lane, step = vec ? 1 : 64;
            for (uint32_t k = 0; k < kTerms && first + k * step < n; k++) {
                const double x = exp_f64((double)l[first + k * step] - m, c_exp.v);
                e[first + k * step] = x;
                sum += x;
            }
        }
        sum = wave_incl_sum(sum);
        if (lane == 63) seg[s0 / kSegTerms] = sum;
    }
}

// Phase 2 (one workgroup per row): the two sequential f64 sums, in index order:
// sum = 0.0 + e[0] + e[1] + ... (codec.rs:791-794), then sum_p = -0.0 + p[0] + p[1] + ...
// (coder.rs:45-46) with p[i] = float(e[i] * (1 / sum)).  Every term is >= +0 or NaN.
//
// A sequential sum of non-negative terms can be computed exactly in parallel between binade
// changes of the running sum s.  While s stays in [2^E, 2^(E+1)), every double there is a
// multiple of u = 2^(E-52), s = T u with T < 2^53, and fl(s + x) = (T + a) u with
// a = round(x / u), half to the side that makes T + a even, as long as T + a < 2^53 (else
// the result leaves the binade and rounds on a coarser grid).  Halves (ties) need the parity
// of T, a prefix of one bit and a reset (a tie leaves T even), formed beside the counts'.
// They are not rare: an f32 probability 2^-29 of the sum or less has its last bit at or below
// half the sum's grid, and most of a trained model's vocabulary lies there.  The grid counts
// are integer-valued f64 (no integer conversion is a single instruction for 64 bits): a sum
// of non-negative integers is exact whenever its result is below 2^53, and rounding is
// monotone, so a sum that reaches 2^53 still reads as >= 2^53 - the crossing test needs no
// more.  Prefixes are formed by adding, never by subtracting, so that this holds for each of
// them.  Below 2^-1022 the grid is the subnormal spacing 2^-1074 with the same rule.
//
// So the row is cut into segments of 256 terms, a wave's.  k_cdf_exp's segment sums (any
// order, a relative error of a few 2^-53) tell which binade s is in at each segment's two
// ends; where it is the same one with 2^-30 to spare, the segment's whole count on that
// binade's grid, with its ties' parity, is formed by any wave at any time (grid_count).  The
// few segments where s may change binade, about one per doubling of s, are put into LDS
// instead.  One wave then goes through the row (chain): it adds runs of counted segments as
// one prefix sum of up to 64 counts, and takes the others in rounds (exact_segment): a prefix
// sum of the terms' counts up to the first event (a NaN, or a term that takes T to 2^53 or
// beyond), the event with one real f64 add, and the next round on the new s's grid.  A
// counted segment is used only if s really is in its binade and its count keeps T below 2^53;
// else it goes through the rounds too, so the result is the sequential sum bit for bit
// whatever the segment sums say.  The first segment, where s doubles most often, is added term
// by term.  The running sum of these rows is NaN or stays below 2^24 (each term <= 1, n < 2^24),
// so the grid is always finer than 1.
//
// Bound by latency.  128 rows of 50,280 normal logits of standard deviations 1 to 4: 65 us, about
// 7 of them the shares after the sums, where 4,096 terms of the whole workgroup a round in order
// (two barriers, 1.7 us each, about 46 rounds a row) took 120 without the shares; the whole call
// 171 -> 102 us.  Of a row, each sum: 1.8 us to classify, 7 to count (51 MB of e over all rows at
// 7 TB/s; the second sum 8 to 17, by how many of its terms are ties), 10 to 14 in the chain, whose
// lone wave issues at a third of the vector rate: about 1.3 us for each uncounted segment with
// the run before it.

// The same value in every lane, made visibly uniform (scalar registers): the round loop's
// control values come from LDS, and without this the compiler treats the loop as divergent
// (exec masking, and copies of the prefetched terms that wait for their loads every round).
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ double uni(double v) {
    const uint64_t b = as_u64(v);
    const uint32_t lo = uni((uint32_t)b), hi = uni((uint32_t)(b >> 32));
    return as_f64(((uint64_t)hi << 32) | lo);
}

// Lane L's copy of v, in every lane (a constant lane: two scalar reads).
__device__ __forceinline__ double lane_f64(double v, int L) {
    const uint64_t b = as_u64(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, L);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), L);
    return as_f64(((uint64_t)hi << 32) | lo);
}

// Lane L's copy of v for a wave-uniform L.
__device__ __forceinline__ double lane_f64_at(double v, int L) { return lane_f64(v, (int)uni((uint32_t)L)); }

// The members of a sequence of up to 64 (bit i: member i) that starts at an even T: members H
// hold a tie and then leave the parity that P has for them, the others flip the parity by
// their bit of P.  Bit i of the result: T is odd before member i.  All of it is scalar
// arithmetic on one mask for the wave.
__device__ __forceinline__ uint64_t odd_before(uint64_t H, uint64_t P) {
    uint64_t x = P << 1;   // the flips of all members before, ties or not
    x ^= x << 1;
    x ^= x << 2;
    x ^= x << 4;
    x ^= x << 8;
    x ^= x << 16;
    x ^= x << 32;
    // behind a tie only the flips from it on count: x of the last tie before is taken out, a bit
    // that a carry spreads from the member behind that tie up to the next tie
    const uint64_t other = ~H;
    return x ^ ((((x & H) << 1) + other) ^ other);
}
// T's parity behind all of them.
__device__ __forceinline__ uint32_t odd_behind(uint64_t H, uint64_t P) {
    const uint64_t from = H != 0 ? ~0ull << (63 - __builtin_clzll(H)) : ~0ull;   // the last tie on
    return (uint32_t)__builtin_popcountll(P & from) & 1u;
}
// Mask bit of the lane.
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

constexpr uint32_t kSumBlock = 1024;                 // threads of a row's workgroup
constexpr uint32_t kSumWaves = kSumBlock / 64;
constexpr uint32_t kWinSegs = 256;                   // segments of a window (65,536 terms)
constexpr uint32_t kSlots = 24;                      // uncounted segments whose terms fit the LDS
constexpr uint32_t kInFlight = 4;                    // segments a wave has requested ahead
constexpr int kNoGrid = 0;                           // (every grid's scale is a positive power)
static_assert(kWinSegs == 64 * kTerms, "wave 0 classifies kTerms segments a lane");

struct SumShared {
    double terms[kSlots][kSegTerms];   // the first kSlots uncounted segments' terms, in order
    double count[kWinSegs];            // a counted segment's grid count (grid_count)
    int grid[kWinSegs];                // its grid 2^-grid, or kNoGrid
    int slot[kWinSegs];                // an uncounted segment's place in terms, or kSlots or more
    uint32_t tie[kWinSegs];            // its ties (grid_count)
    double s;                          // the running sum after the window
};

// A term's count on a grid: x / u to the nearest integer, halves to even, which is the
// count's own rounding from an even T.  q = x / u must be below 2^52 (a larger one takes T past
// the binade: T >= 2^52 before it, or 2^52 is the subnormal grid's end): q + 2^52 rounds to
// an integer and shows its parity.
struct GridTerm {
    double a;       // the count
    double d;       // q - a: a tie is +-1/2, and from an odd T its count is a + 2 d
    uint32_t odd;   // the count's parity (bit 0)
};
__device__ __forceinline__ GridTerm grid_term(double q) {
    GridTerm g;
    const double m = q + 0x1p52;
    g.a = m - 0x1p52;
    g.d = q - g.a;
    g.odd = (uint32_t)as_u64(m);
    return g;
}

// +1 or -1 by d's sign in the lanes of the mask, else 0.
__device__ __forceinline__ double unit_step(uint64_t mask, double d) {
    const uint32_t hi = ((uint32_t)(as_u64(d) >> 32) & 0x80000000u) | 0x3ff00000u;
    return as_f64((uint64_t)(lane_in(mask) ? hi : 0u) << 32);
}

// A wave's ties settled as far as they can be without the parity of T before the wave.  A tie
// leaves an even T behind, so the parity a lane passes on is its own once it holds a tie, else
// the incoming one flipped by its counts.  step[j]: the lanes whose term j is a tie from an odd
// T (its count is a + 2 d); the wave's first tie (lane `first`, one bit; none: no tie) is
// left as from an even T.
struct WaveTies {
    uint64_t step[kTerms], lead[kTerms];   // lead[j]: term j is its lane's first tie
    uint64_t first;
    uint64_t odd;    // T is odd before the lane's first tie if it is even before the wave
    uint32_t behind;  // the parity of T behind the wave (without a tie: the flip)
};
__device__ __forceinline__ WaveTies wave_ties(const GridTerm (&g)[kTerms]) {
    WaveTies w;
    uint64_t x = 0, seen = 0, first_x = 0;   // x: parity since the lane's start or last tie
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) {
        const uint64_t tie = __ballot(fabs(g[j].d) == 0.5);
        w.lead[j] = tie & ~seen;
        w.step[j] = tie & seen & x;
        first_x |= w.lead[j] & x;
        seen |= tie;
        x = (x ^ __ballot((g[j].odd & 1u) != 0)) & ~tie;
    }
    w.odd = odd_before(seen, x) ^ first_x;
    w.behind = odd_behind(seen, x);
    w.first = seen & (0 - seen);
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) w.step[j] |= w.lead[j] & w.odd & ~w.first;
    return w;
}

// Segment i's count on its grid, into sh.  Its bits in sh.tie: 1: it holds a tie; 2: T is odd
// before the first one if it is even before the segment; 4: the parity of T behind it (without
// a tie: the flip); 8: the first tie steps down from an odd T, not up.
__device__ __forceinline__ void grid_count(const double (&fx)[kTerms], int ks, uint32_t i, int lane, SumShared& sh) {
    const double scale = as_f64((uint64_t)(1023 + ks) << 52);
    GridTerm g[kTerms];
    bool any_tie = false;
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) {
        g[j] = grid_term(fx[j] * scale);   // exact, or inf
        any_tie |= fabs(g[j].d) == 0.5;
    }
    double mine = (g[0].a + g[1].a) + (g[2].a + g[3].a);
    uint32_t ties = 0;
    if (__ballot(any_tie) != 0) {
        const WaveTies w = wave_ties(g);
        uint64_t down = 0;
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) {
            mine += unit_step(w.step[j], g[j].d);
            down |= w.lead[j] & __ballot(g[j].d < 0.0);
        }
        ties = 1u | ((w.odd & w.first) != 0 ? 2u : 0u) | w.behind << 2 | ((down & w.first) != 0 ? 8u : 0u);
    }
    const double total = wave_incl_sum(mine);
    if (lane == 63) {
        sh.count[i] = total;   // (NaN or not below 2^52 where a term is no count of the binade)
        sh.tie[i] = ties != 0 ? ties : ((uint32_t)as_u64(total + 0x1p52) & 1u) << 2;
    }
}

// s after the wave's 256 terms (lane L: terms L kTerms ..), by rounds.  Terms that are in s are
// zeros from then on.
__device__ double exact_segment(double (&fx)[kTerms], double s, int lane) {
    for (;;) {
        // a NaN stays one (only NaN-ness is used downstream); every other sum of a row is below 2^24
        if (!(s < 0x1p52)) return s;
        // the grid of the current binade: terms scale by 2^ks into units of it
        const bool sub = s < 0x1p-1022;
        const int ks = sub ? 1074 : 1075 - (int)(as_u64(s) >> 52);
        const double top = sub ? 0x1p52 : 0x1p53;
        const double T0 = ldexp(s, ks);   // exact and integer-valued: s is on the grid
        GridTerm g[kTerms];
        bool bad[kTerms];   // NaN, inf or certainly past the binade: an event
        bool any_tie = false;
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) {
            const double q = ldexp(fx[j], ks);   // exact, or +inf past the double range
            bad[j] = !(q < 0x1p52);
            g[j] = grid_term(bad[j] ? 0.0 : q);
            any_tie |= fabs(g[j].d) == 0.5;
        }
        if (__ballot(any_tie) != 0) {
            const WaveTies w = wave_ties(g);
            const bool t_odd = ((uint32_t)as_u64(sub ? T0 + 0x1p52 : T0) & 1u) != 0;
            const uint64_t first = ((w.odd & w.first) != 0) != t_odd ? w.first : 0;   // if it steps
#pragma unroll
            for (uint32_t j = 0; j < kTerms; j++) g[j].a += unit_step(w.step[j] | (w.lead[j] & first), g[j].d);
        }
        const double incl = wave_incl_sum((g[0].a + g[1].a) + (g[2].a + g[3].a));
        const double end = T0 + lane_f64(incl, 63);
        if (__ballot(bad[0] || bad[1] || bad[2] || bad[3]) == 0 && end < top) return uni(ldexp(end, -ks));   // no event
        double c[kTerms];   // the lane's inclusive prefix
        double mine = 0.0;
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) {
            mine += g[j].a;
            c[j] = mine;
        }
        const double base = T0 + dpp_f64<0x138>(incl);   // wave_shr:1 (lane 0 reads 0)
        // the lane's first term that is bad or takes T to the top of the binade
        bool hit = false;
        uint32_t at = 0;
        double T_ev = 0.0, x_ev = 0.0;
#pragma unroll
        for (int j = (int)kTerms - 1; j >= 0; j--) {
            const bool h = bad[j] || base + c[j] >= top;
            hit |= h;
            at = h ? (uint32_t)j : at;
            T_ev = h ? (j > 0 ? base + c[j - 1] : base) : T_ev;
            x_ev = h ? fx[j] : x_ev;
        }
        const uint64_t has = __ballot(hit);   // some lane: T passes the top, or a term is bad
        const int src = (int)uni((uint32_t)__builtin_ctzll(has));
        s = uni(ldexp(lane_f64(T_ev, src), -ks) + lane_f64(x_ev, src));
        const uint32_t done = (uint32_t)src * kTerms + (uint32_t)__builtin_amdgcn_readlane((int)at, src);
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) fx[j] = (uint32_t)lane * kTerms + j <= done ? 0.0 : fx[j];
    }
}

// Terms kTerms lane .. of the segment that starts at k0; past the row's end 0, which no sum of
// the row tells from nothing (s is +0 or more once it holds a term).
template <class F>
__device__ __forceinline__ void seg_terms(uint32_t n, uint32_t k0, int lane, F f, const double (&raw)[kTerms],
                                          double (&fx)[kTerms]) {
    if (k0 + kSegTerms <= n) {
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) fx[j] = f(raw[j]);
        return;
    }
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) fx[j] = k0 + (uint32_t)lane * kTerms + j < n ? f(raw[j]) : 0.0;
}
__device__ __forceinline__ void seg_load(const double* __restrict__ e, uint32_t n, uint32_t k0, int lane,
                                         double (&raw)[kTerms]) {
    if (k0 + kSegTerms <= n && ((uintptr_t)(e + k0) & 15) == 0) {
        const double2* p = (const double2*)(e + k0 + (uint32_t)lane * kTerms);
        const double2 v = p[0], w = p[1];
        raw[0] = v.x, raw[1] = v.y, raw[2] = w.x, raw[3] = w.y;
        return;
    }
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) raw[j] = e[min(k0 + (uint32_t)lane * kTerms + j, n - 1)];
}

// Which of the window's m segments lie in one binade, and the others' slots in order (wave 0).
// The segment sums are scaled by `scale`; s is the running sum before the window.
__device__ void classify(const double* __restrict__ seg, uint32_t m, double scale, double s, int lane, SumShared& sh) {
    double v[kTerms];
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) v[j] = seg[min((uint32_t)lane * kTerms + j, m - 1)] * scale;
    const double incl = wave_incl_sum((v[0] + v[1]) + (v[2] + v[3]));
    double at = s + dpp_f64<0x138>(incl);
    int grid[kTerms];
    uint32_t place = 0;   // uncounted segments of the lanes before
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) {
        // (exponents from 2^-900 to 2^51: the grid's scale is a normal double; NaN and inf: 2047)
        const uint32_t lo = (uint32_t)(as_u64(at * (1.0 - 0x1p-30)) >> 52);
        at += v[j];
        const uint32_t hi = (uint32_t)(as_u64(at * (1.0 + 0x1p-30)) >> 52);
        grid[j] = lo == hi && lo >= 1023 - 900 && lo < 1023 + 52 ? 1075 - (int)lo : kNoGrid;
        const uint64_t un = __ballot((uint32_t)lane * kTerms + j < m && grid[j] == kNoGrid);
        place += (uint32_t)__builtin_popcountll(un & ((1ull << lane) - 1));
    }
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) {
        const uint32_t i = (uint32_t)lane * kTerms + j;
        if (i < m) {
            sh.grid[i] = grid[j];
            sh.slot[i] = (int)place;
            place += grid[j] == kNoGrid ? 1u : 0u;
        }
    }
}

// s after the window's m segments (wave 0).
template <class F>
__device__ double chain(const double* __restrict__ e, uint32_t n, uint32_t k0, uint32_t m, double s, int lane, F f,
                        const SumShared& sh) {
    uint32_t i = 0;
    uint32_t slots = 0;   // uncounted segments before segment i
    if (k0 == 0) {
        // the row's first segment in order (classify leaves s = 0 without a grid and gives it
        // the first slot): every lane reads the terms back as broadcasts into one chain of adds
#pragma unroll 2
        for (uint32_t t = 0; t < kSegTerms; t += 16) {
            double v[16];
#pragma unroll
            for (uint32_t k = 0; k < 16; k++) v[k] = sh.terms[0][t + k];
#pragma unroll
            for (uint32_t k = 0; k < 16; k++) s += v[k];
        }
        s = uni(s);
        i = 1;
        slots = 1;
    }
    while (i < m) {
        if (isnan(s)) return s;
        // the next uncounted segment's terms, requested before the counts are added up
        double fx[kTerms];
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) fx[j] = sh.terms[min(slots, kSlots - 1)][(uint32_t)lane * kTerms + j];
        const int ks = s < 0x1p-1022 || !(s < 0x1p52) ? kNoGrid - 1 : 1075 - (int)(as_u64(s) >> 52);
        // the counted segments of s's binade from here on, up to 64
        const uint32_t i0 = i, at = min(i + (uint32_t)lane, m - 1);
        const int grid = sh.grid[at];
        const double count = sh.count[at];
        const uint32_t ties = sh.tie[at];
        const uint64_t off = ~__ballot(i + (uint32_t)lane < m && grid == ks);
        const int run = off != 0 ? __builtin_ctzll(off) : 64;
        if (run > 0) {
            double c = lane < run ? count : 0.0;
            const uint32_t t = lane < run ? ties : 0u;
            const double T0 = ldexp(s, ks);
            const uint64_t H = __ballot((t & 1u) != 0);
            if (H != 0) {
                // each segment's first tie, from the parity of T before that segment
                const uint64_t t_odd = ((uint32_t)as_u64(T0) & 1u) != 0 ? ~0ull : 0ull;
                const uint64_t in = odd_before(H, __ballot((t & 4u) != 0)) ^ (t_odd & ((H & (0 - H)) | ((H & (0 - H)) - 1)));
                const uint64_t step = H & (in ^ __ballot((t & 2u) != 0));
                c += lane_in(step) ? ((t & 8u) != 0 ? -1.0 : 1.0) : 0.0;
            }
            const double T = T0 + wave_incl_sum(c);
            const uint64_t past = __ballot(lane < run && !(T < 0x1p53));
            const int take = past != 0 ? __builtin_ctzll(past) : run;
            if (take > 0) s = uni(ldexp(lane_f64_at(T, take - 1), -ks));
            i += (uint32_t)take;
            if (take == 64 || i >= m) continue;
        }
        // segment i: lane i - i0's, whose grid is not s's or whose count takes T to the top
        const bool counted = __builtin_amdgcn_readlane(grid, (int)uni(i - i0)) != kNoGrid;
        if (counted || slots >= kSlots) {
            double raw[kTerms];
            seg_load(e, n, k0 + i * kSegTerms, lane, raw);
            seg_terms(n, k0 + i * kSegTerms, lane, f, raw, fx);
        }
        slots += counted ? 0u : 1u;
        s = exact_segment(fx, s, lane);
        i++;
    }
    return s;
}

// f's terms as f32 bits to p (lane L: kTerms L ..).
__device__ __forceinline__ void seg_store(uint32_t* p, uint32_t n, uint32_t k0, int lane, const double (&fx)[kTerms]) {
    struct __attribute__((packed, aligned(4))) U4 {
        uint32_t v[kTerms];
    };
    U4 u;
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) u.v[j] = __float_as_uint((float)fx[j]);
    const uint32_t i = k0 + (uint32_t)lane * kTerms;
    if (k0 + kSegTerms <= n) {
        *(U4*)(p + i) = u;
        return;
    }
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++)
        if (i + j < n) p[i + j] = u.v[j];
}

// The sequential sum s + f(e[0]) + f(e[1]) + ... of the row; f(x) is about x * scale.  P: the
// terms, which are f32 values, also go to p.
template <bool P, class F>
__device__ double exact_seq_sum(const double* __restrict__ e, const double* __restrict__ seg, uint32_t n, double s,
                                double scale, F f, uint32_t* p, SumShared& sh) {
    const int lane = threadIdx.x % 64;
    const uint32_t w = uni(threadIdx.x / 64);
    for (uint32_t k0 = 0; k0 < n; k0 += kWinSegs * kSegTerms) {
        const uint32_t m = min(kWinSegs, segments(n - k0));
        // wave w: segments w, w + kSumWaves, ..., kInFlight requested ahead
        double nx[kInFlight][kTerms];
#pragma unroll
        for (uint32_t d = 0; d < kInFlight; d++) seg_load(e, n, k0 + (w + d * kSumWaves) * kSegTerms, lane, nx[d]);
        if (w == 0) classify(seg + k0 / kSegTerms, m, scale, s, lane, sh);
        __syncthreads();
        for (uint32_t i0 = w; i0 < m; i0 += kInFlight * kSumWaves) {
#pragma unroll
            for (uint32_t d = 0; d < kInFlight; d++) {
                const uint32_t i = i0 + d * kSumWaves;
                double fx[kTerms];
                seg_terms(n, k0 + i * kSegTerms, lane, f, nx[d], fx);
                if (i + kInFlight * kSumWaves < m) seg_load(e, n, k0 + (i + kInFlight * kSumWaves) * kSegTerms, lane, nx[d]);
                if (i >= m) continue;
                if (P) seg_store(p, n, k0 + i * kSegTerms, lane, fx);
                const int ks = __builtin_amdgcn_readfirstlane(sh.grid[i]);
                if (ks != kNoGrid) {
                    grid_count(fx, ks, i, lane, sh);
                    continue;
                }
                const int slot = __builtin_amdgcn_readfirstlane(sh.slot[i]);
                if (slot < (int)kSlots) {
#pragma unroll
                    for (uint32_t j = 0; j < kTerms; j++) sh.terms[slot][(uint32_t)lane * kTerms + j] = fx[j];
                }
            }
        }
        __syncthreads();
        if (w == 0) {
            s = chain(e, n, k0, m, s, lane, f, sh);
            if (lane == 0) sh.s = s;
        }
        __syncthreads();
        s = uni(sh.s);
        // (the next write to sh.s comes after the next window's or sum's barriers)
    }
    return s;
}

// Phase 3, Cdf::from_probs (coder.rs:43-81) from the two sums: extra[i] =
// (u64)(p[i] * inv * rem + 0.5) and freq[i] = 1 + extra[i]; the surplus or deficit goes to
// the last of the largest frequencies; then the cumulative frequencies.  The row's workgroup
// gathers each chunk's used sum and its largest (frequency, last index) right after the sums, a
// wave a chunk, 3b writes the chunk's cumulative frequencies from those.  Both read the f32
// probabilities that the second sum left where the cumulative frequencies go, half of e's
// bytes: k_cdf_freq_write 18.7 -> 15.0 us at 128 rows of 50,280, and the gathering, a kernel
// of its own before (12 us and a launch), adds 7 us to the sums.  Every combination here is an integer sum
// or a max, exact in any order.
struct FreqRow {
    double inv, rem;
    uint64_t remaining;
};
__device__ __forceinline__ FreqRow freq_row(double sum_p, uint32_t n) {
    FreqRow f;
    f.remaining = (uint64_t)kCdfTotal - n;
    f.inv = sum_p > 0.0 ? 1.0 / sum_p : 0.0;
    f.rem = (double)f.remaining;
    return f;
}
// (u64)(p inv rem + 0.5), truncated, NaN -> 0.  The sum of the probabilities is no smaller
// than any of them (non-negative terms, monotone rounding), so this is 2^24 at most.
__device__ __forceinline__ uint32_t extra_of(uint32_t p, const FreqRow& f) {
    const double v = (double)__uint_as_float(p) * f.inv * f.rem + 0.5;
    return v > 0.0 ? (uint32_t)v : 0u;
}

// A wave's used sum and largest (frequency, last index) from its lanes' sum, largest share and
// that one's index.
__device__ __forceinline__ void part_reduce(uint32_t mine, uint32_t most, uint32_t at, uint64_t& used, uint64_t& best) {
    used = mine;
    best = (uint64_t)(1u + most) << 32 | at;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        used += __shfl_xor(used, o);
        const uint64_t b = __shfl_xor(best, o);
        best = b > best ? b : best;
    }
}

// Chunk c's used sum and largest frequency (one wave).
__device__ void freq_part(const uint32_t* __restrict__ p, uint32_t n, uint32_t c, int lane, const FreqRow& f,
                          ChunkPart& part) {
    uint32_t mine = 0, most = 0, at = 0;   // (kChunk / 64 shares a lane: below 2^31)
    const uint32_t c0 = c * kChunk, c1 = min(n, c0 + kChunk);
    uint32_t v[kSpan];
#pragma unroll
    for (uint32_t j = 0; j < kSpan; j++) v[j] = p[min(c0 + 64 * j + (uint32_t)lane, n - 1)];
    for (uint32_t k = c0; k < c1; k += 64 * kSpan) {
        uint32_t nx[kSpan];
#pragma unroll
        for (uint32_t j = 0; j < kSpan; j++) nx[j] = p[min(k + 64 * (kSpan + j) + (uint32_t)lane, n - 1)];
#pragma unroll
        for (uint32_t j = 0; j < kSpan; j++) {
            const uint32_t i = k + 64 * j + (uint32_t)lane;
            const uint32_t x = i < c1 ? extra_of(v[j], f) : 0u;
            mine += x;
            const bool last = i < c1 && x >= most;   // the last of equal ones
            most = last ? x : most;
            at = last ? i : at;
            v[j] = nx[j];
        }
    }
    uint64_t used, best;
    part_reduce(mine, most, at, used, best);
    if (lane == 0) {
        part.used = used;
        part.best = best;
    }
}

// A row of one segment (a byte vocabulary): one wave adds its terms in order, both times from
// the same registers, and takes their shares from there.  Bound by the two chains of adds and the
// launches: the whole call for 128 / 512 rows of 256 takes 13.5 / 14.4 us, 19.6 / 28.5 through
// k_cdf_sums; two segments gain from it no more (its second one would be another chain of 256).
__global__ __launch_bounds__(64) void k_cdf_sums_short(CdfArgs a) {
    __shared__ double terms[kSegTerms];
    const uint32_t row = blockIdx.x, n = a.n;
    const int lane = threadIdx.x;
    double raw[kTerms], fx[kTerms];
    seg_load(a.e + (size_t)row * n, n, 0, lane, raw);
    auto sum = [&](double s) {
#pragma unroll
        for (uint32_t j = 0; j < kTerms; j++) terms[(uint32_t)lane * kTerms + j] = fx[j];
        __builtin_amdgcn_s_waitcnt(0xc07f);   // this wave's LDS stores done
        __builtin_amdgcn_wave_barrier();
        for (uint32_t t = 0; t < n; t += 16) {
            double v[16];
#pragma unroll
            for (uint32_t k = 0; k < 16; k++) v[k] = terms[t + k];
#pragma unroll
            for (uint32_t k = 0; k < 16; k++) s += v[k];
        }
        __builtin_amdgcn_wave_barrier();
        return uni(s);
    };
    seg_terms(n, 0, lane, [](double v) { return v; }, raw, fx);
    const double inv_sum = 1.0 / sum(0.0);
    seg_terms(n, 0, lane, [inv_sum](double v) { return (double)prob_of(v, inv_sum); }, raw, fx);
    seg_store(a.cdf + (size_t)row * (n + 1) + 1, n, 0, lane, fx);
    const double sp = sum(-0.0);
    const FreqRow f = freq_row(sp, n);
    uint32_t mine = 0, most = 0, at = 0;
#pragma unroll
    for (uint32_t j = 0; j < kTerms; j++) {
        const uint32_t i = (uint32_t)lane * kTerms + j;
        const uint32_t x = i < n ? extra_of(__float_as_uint((float)fx[j]), f) : 0u;
        const bool last = i < n && x >= most;   // the last of equal ones
        mine += x;
        most = last ? x : most;
        at = last ? i : at;
    }
    uint64_t used, best;
    part_reduce(mine, most, at, used, best);
    if (lane == 0) {
        a.sums[row] = sp;
        a.part[row].used = used;
        a.part[row].best = best;
    }
}

__global__ __launch_bounds__(kSumBlock) void k_cdf_sums(CdfArgs a) {
    __shared__ SumShared sh;
    const uint32_t row = blockIdx.x, n = a.n;
    const double* e = a.e + (size_t)row * n;
    const double* seg = a.seg + (size_t)row * segments(n);
    const double s = exact_seq_sum<false>(e, seg, n, 0.0, 1.0, [](double v) { return v; }, nullptr, sh);
    const double inv_sum = 1.0 / s;
    const double sp = exact_seq_sum<true>(e, seg, n, -0.0, inv_sum,
                                          [inv_sum](double v) { return (double)prob_of(v, inv_sum); },
                                          a.cdf + (size_t)row * (n + 1) + 1, sh);
    if (threadIdx.x == 0) a.sums[row] = sp;
    // (the probabilities were stored before the barriers of the sum)
    const FreqRow f = freq_row(sp, n);
    for (uint32_t c = uni(threadIdx.x / 64); c < a.chunks; c += kSumWaves)
        freq_part(a.cdf + (size_t)row * (n + 1) + 1, n, c, threadIdx.x % 64, f, a.part[(size_t)row * a.chunks + c]);
}

// LDS index of a chunk position: one pad word per 32, so that both the coalesced pass
// (thread t at t + 256 j) and the per-thread pass (thread t at 16 t + j) meet no bank
// conflicts.
__device__ __forceinline__ uint32_t pad_ix(uint32_t p) { return p + p / 32; }

// What a row's chunks add up to, in every thread.
struct RowFix {
    FreqRow f;
    int64_t diff;      // the fix-up
    uint32_t at;       // the element that takes it
    uint64_t most;     // that element's frequency before it
    uint32_t total;    // cdf[n]
};
__device__ __forceinline__ RowFix row_fix(const CdfArgs& a, uint32_t row) {
    RowFix x;
    x.f = freq_row(a.sums[row], a.n);
    const ChunkPart* pr = a.part + (size_t)row * a.chunks;
    uint64_t used = 0, best = 0;
    for (uint32_t i = 0; i < a.chunks; i++) {
        used += pr[i].used;
        best = pr[i].best > best ? pr[i].best : best;
    }
    x.diff = (int64_t)x.f.remaining - (int64_t)used;
    x.at = (uint32_t)best;
    x.most = best >> 32;
    x.total = (uint32_t)((int64_t)(a.n + used) + x.diff);
    return x;
}
// Chunk c's first cumulative frequency (u32, wrapping, as the host's sum; each frequency is 1
// and its share).
__device__ __forceinline__ uint32_t chunk_offset(const CdfArgs& a, uint32_t row, uint32_t c, const RowFix& x) {
    const ChunkPart* pr = a.part + (size_t)row * a.chunks;
    uint32_t offset = 0;
    for (uint32_t i = 0; i < c; i++) offset += (uint32_t)pr[i].used + kChunk;
    return x.at < c * kChunk ? (uint32_t)((int64_t)offset + x.diff) : offset;
}

struct ChunkShared {
    uint32_t wave[kCdfBlock / 64];
    uint32_t cum[kChunk + kChunk / 32];   // element c0 + r's cumulative frequency (its own included) at pad_ix(r)
};
// Chunk c's cumulative frequencies into sh.cum (every thread of the workgroup; it may be
// called again once all have read).
__device__ __forceinline__ void chunk_cum(const CdfArgs& a, uint32_t row, uint32_t c, const RowFix& x, uint32_t offset,
                                          ChunkShared& sh) {
    const uint32_t c0 = c * kChunk, n = a.n;
    const uint32_t* cdf = a.cdf + (size_t)row * (n + 1);
    // the chunk's frequencies, from the probabilities in the elements that its cumulative
    // frequencies take at the end (read coalesced: element c0 + t + 256 j)
    uint32_t prob[kSpan];
#pragma unroll
    for (uint32_t j = 0; j < kSpan; j++) prob[j] = cdf[1 + min(c0 + threadIdx.x + kCdfBlock * j, n - 1)];
#pragma unroll
    for (uint32_t j = 0; j < kSpan; j++) {
        const uint32_t p = threadIdx.x + kCdfBlock * j, i = c0 + p;
        uint32_t v = 0;
        if (i < n) {
            v = 1u + extra_of(prob[j], x.f);
            if (i == x.at) v = (uint32_t)((int64_t)v + x.diff);
        }
        sh.cum[pad_ix(p)] = v;
    }
    __syncthreads();
    // thread t: kSpan consecutive elements; exclusive scan of the thread totals
    uint32_t fq[kSpan];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < kSpan; j++) {
        fq[j] = sh.cum[pad_ix(threadIdx.x * kSpan + j)];
        mine += fq[j];
    }
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    uint32_t incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = __shfl_up(incl, o);
        if (lane >= o) incl += up;
    }
    if (lane == 63) sh.wave[w] = incl;
    __syncthreads();
    uint32_t cum = offset + incl - mine;
#pragma unroll
    for (int i = 0; i < kCdfBlock / 64; i++)
        if (i < w) cum += sh.wave[i];
#pragma unroll
    for (uint32_t j = 0; j < kSpan; j++) {
        cum += fq[j];
        sh.cum[pad_ix(threadIdx.x * kSpan + j)] = cum;   // each thread rewrites only its own positions
    }
    __syncthreads();
}

__global__ __launch_bounds__(kCdfBlock) void k_cdf_freq_write(CdfArgs a) {
    __shared__ ChunkShared sh;
    const uint32_t c = blockIdx.x, row = blockIdx.y, n = a.n, c0 = c * kChunk;
    const RowFix x = row_fix(a, row);
    chunk_cum(a, row, c, x, chunk_offset(a, row, c, x), sh);
    uint32_t* cdf = a.cdf + (size_t)row * (n + 1);
    if (c == 0 && threadIdx.x == 0) cdf[0] = 0;
    for (uint32_t r = threadIdx.x; r < kChunk && c0 + r < n; r += kCdfBlock) cdf[c0 + r + 1] = sh.cum[pad_ix(r)];
}

// What the range coder reads of a row, straight from the shares: one workgroup a row works
// out the one chunk it needs, so the rows' cumulative frequencies are not written (at 128 rows of
// 50,280 k_cdf_freq_write's 15 us and 5 more for a kernel that reads three of them back; now 8, with the search 10).
// FIND false: symbol key[r] is known (coder.rs:163-177 via encode_symbol): out[3r] = cdf[r][key],
// out[3r + 1] = cdf[r][key + 1], out[3r + 2] = cdf[r][n], the total.  (The host checked it
// against n; the clamp keeps every read inside the row whatever it holds.)
// FIND true: the symbol s that the decoder's binary search finds for its target key[r]
// (coder.rs:100-115): out[4r] = s, out[4r + 1] = cdf[r][s], out[4r + 2] = cdf[r][s + 1],
// out[4r + 3] = cdf[r][n]; s = n (both bounds cdf[r][n]) where the target is not below the
// total.  The frequencies are positive but for the one that takes a deficit of the shares.
// Where it stays non-negative the row rises and the search finds the first element above the
// target: first the chunk, then the element.  Else the search is done as it is, probe by probe.
template <bool FIND>
__global__ __launch_bounds__(kCdfBlock) void k_cdf_read(CdfArgs a, const uint32_t* __restrict__ key, uint32_t* __restrict__ out) {
    __shared__ ChunkShared sh;
    __shared__ uint32_t first;
    const uint32_t row = blockIdx.x, n = a.n;
    const RowFix x = row_fix(a, row);
    const uint32_t k = key[row];
    uint32_t s, chunk, offset;
    if (!FIND) {
        s = min(k, n - 1);
        chunk = s / kChunk;
        offset = chunk_offset(a, row, chunk, x);
        chunk_cum(a, row, chunk, x, offset, sh);
    } else if ((int64_t)x.most + x.diff >= 0) {
        if (k >= x.total) {
            if (threadIdx.x == 0) {
                uint32_t* o = out + 4 * (size_t)row;
                o[0] = n;
                o[1] = o[2] = o[3] = x.total;
            }
            return;
        }
        uint32_t end = 0;   // of the chunk, before the fix-up
        for (chunk = 0; chunk + 1 < a.chunks; chunk++) {
            end += (uint32_t)a.part[(size_t)row * a.chunks + chunk].used + kChunk;
            if ((x.at < (chunk + 1) * kChunk ? (uint32_t)((int64_t)end + x.diff) : end) > k) break;
        }
        offset = chunk_offset(a, row, chunk, x);
        if (threadIdx.x == 0) first = kChunk;
        chunk_cum(a, row, chunk, x, offset, sh);
        uint32_t mine = kChunk;
#pragma unroll
        for (int j = (int)kSpan - 1; j >= 0; j--) {
            const uint32_t r = threadIdx.x * kSpan + (uint32_t)j;
            if (chunk * kChunk + r < n && sh.cum[pad_ix(r)] > k) mine = r;
        }
        if (mine < kChunk) atomicMin(&first, mine);
        __syncthreads();
        s = chunk * kChunk + first;
    } else {
        uint32_t lo = 0, hi = n;
        chunk = 0xffffffffu;
        offset = 0;
        auto load = [&](uint32_t c) {
            if (c == chunk) return;
            __syncthreads();   // the chunk before has been read
            chunk = c;
            offset = chunk_offset(a, row, c, x);
            chunk_cum(a, row, c, x, offset, sh);
        };
        while (lo < hi) {
            const uint32_t m = lo + (hi - lo) / 2;
            load(m / kChunk);
            if (sh.cum[pad_ix(m % kChunk)] <= k)
                lo = m + 1;
            else
                hi = m;
        }
        s = lo;
        if (s < n) load(s / kChunk);
    }
    if (threadIdx.x != 0) return;
    const uint32_t r = s % kChunk;
    const uint32_t below = s == n ? x.total : r > 0 ? sh.cum[pad_ix(r - 1)] : offset;
    const uint32_t above = s == n ? x.total : sh.cum[pad_ix(r)];
    uint32_t* o = out + (FIND ? 4 : 3) * (size_t)row;
    if (FIND) *o++ = s;
    o[0] = below;
    o[1] = above;
    o[2] = x.total;
}

}  // namespace

namespace {
uint32_t cdf_chunks(uint32_t n) { return (n + kChunk - 1) / kChunk; }
}  // namespace

size_t cdf_scratch_bytes(uint32_t rows, uint32_t n) {
    return (size_t)rows * n * 8 + (size_t)rows * 8 + (size_t)rows * segments(n) * 8 +
           (size_t)rows * cdf_chunks(n) * sizeof(ChunkPart);
}

namespace {
// The probabilities of every row (in the CDF elements) and the chunks' shares.
CdfArgs cdf_shares(const float* logits, uint32_t rows, uint32_t n, void* scratch, uint32_t* cdf, hipStream_t st) {
    const uint32_t chunks = cdf_chunks(n);
    double* e = (double*)scratch;
    double* sums = e + (size_t)rows * n;
    double* seg = sums + rows;
    ChunkPart* part = (ChunkPart*)(seg + (size_t)rows * segments(n));
    const CdfArgs a{logits, rows, n, chunks, e, sums, seg, part, cdf};
    const dim3 grid(chunks, rows);
    k_cdf_max<<<grid, dim3(kCdfBlock), 0, st>>>(a);
    k_cdf_exp<<<grid, dim3(kCdfBlock), 0, st>>>(a);
    if (n <= kSegTerms)
        k_cdf_sums_short<<<dim3(rows), dim3(64), 0, st>>>(a);
    else
        k_cdf_sums<<<dim3(rows), dim3(kSumBlock), 0, st>>>(a);
    return a;
}
}  // namespace

hipError_t cdf_launch(const float* logits, uint32_t rows, uint32_t n, void* scratch, uint32_t* cdf, hipStream_t st) {
    if (rows == 0) return hipSuccess;
    const CdfArgs a = cdf_shares(logits, rows, n, scratch, cdf, st);
    k_cdf_freq_write<<<dim3(a.chunks, rows), dim3(kCdfBlock), 0, st>>>(a);
    return hipGetLastError();
}

hipError_t cdf_read_launch(const float* logits, uint32_t rows, uint32_t n, void* scratch, uint32_t* space, bool find,
                           const uint32_t* key, uint32_t* out, hipStream_t st) {
    if (rows == 0) return hipSuccess;
    const CdfArgs a = cdf_shares(logits, rows, n, scratch, space, st);
    if (find)
        k_cdf_read<true><<<dim3(rows), dim3(kCdfBlock), 0, st>>>(a, key, out);
    else
        k_cdf_read<false><<<dim3(rows), dim3(kCdfBlock), 0, st>>>(a, key, out);
    return hipGetLastError();
}

}  // namespace rdk
