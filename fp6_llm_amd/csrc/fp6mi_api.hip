// C ABI of the FPx x FP16 linear-layer engine (include/fp6mi.h), the choice of the launch shape, and the split-K reduction.
// The kernels live in fp6mi_gemm.hip, compiled once per weight format; this file reaches them through fp6mi::FormatOps.
//
// Roles taken over from the reference (usyd-fsalab/fp6_llm, paths relative to it):
//   splitk_reduce      <- SplitK_Reduction        fp6_llm/csrc/include/kernel_reduction.cuh:28-47
//   pick_cfg           <- the N bucketing of      fp6_llm/csrc/fp6_linear.cu:58-99
//   fp6mi_linear*      <- fpx_linear_kernel       fp6_llm/csrc/fp6_linear.cu:44-102
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include "fp6mi_internal.h"

namespace {

typedef _Float16 half_t;
typedef float    v4f __attribute__((ext_vector_type(4)));

using fp6mi::LaunchCfg;

// C[i] = fp16_rn(sum over splits, in split order, of ws[s][i] + bias) for the four outputs from index i.  bias: of the first of them
template <bool BIAS> __device__ __forceinline__ void reduce_four(half_t *__restrict__ C, const float *__restrict__ ws, size_t MN, int splitK, size_t i, const half_t *bias)
{
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    v4h b;
    if constexpr (BIAS) b = (v4h){ bias[0], bias[1], bias[2], bias[3] }; // (any 2-byte boundary)
    v4f sum = { 0.f, 0.f, 0.f, 0.f };
    // up to eight loads in flight instead of one round trip to memory per split; the order of the sum is unchanged.  The
    // remainder after the groups of eight is one group of its exact size (a 3 done as 2 + 1 would be two round trips).
    auto chunk = [&](auto count, int s0) {
        constexpr int C = decltype(count)::value;
        v4f           part[C];
#pragma unroll
        for (int k = 0; k < C; k++) part[k] = *reinterpret_cast<const v4f *>(ws + (size_t)(s0 + k) * MN + i);
#pragma unroll
        for (int k = 0; k < C; k++) sum += part[k];
    };
    int s = 0;
    for (; s + 8 <= splitK; s += 8) chunk(std::integral_constant<int, 8>{}, s);
    switch (splitK - s) {
    case 7: chunk(std::integral_constant<int, 7>{}, s); break;
    case 6: chunk(std::integral_constant<int, 6>{}, s); break;
    case 5: chunk(std::integral_constant<int, 5>{}, s); break;
    case 4: chunk(std::integral_constant<int, 4>{}, s); break;
    case 3: chunk(std::integral_constant<int, 3>{}, s); break;
    case 2: chunk(std::integral_constant<int, 2>{}, s); break;
    case 1: chunk(std::integral_constant<int, 1>{}, s); break;
    default: break;
    }
    if constexpr (BIAS) {
#pragma unroll
        for (int k = 0; k < 4; k++) sum[k] += (float)b[k];
    }
    v4h o = { (half_t)sum[0], (half_t)sum[1], (half_t)sum[2], (half_t)sum[3] };
    *reinterpret_cast<v4h *>(C + i) = o;
}

// four outputs per thread, in the order of the output
template <bool BIAS>
__global__ __launch_bounds__(256) void splitk_reduce(half_t *__restrict__ C, const float *__restrict__ ws, size_t MN, int splitK, const half_t *__restrict__ bias,
                                                     uint32_t M)
{
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i < MN) reduce_four<BIAS>(C, ws, MN, splitK, i, BIAS ? bias + i % M : nullptr);
}

// The same sums with the workgroups placed where the partial sums were written.  gemm_tile hands XCD x (workgroup ids
// congruent to x mod 8) the consecutive (row block, split, column block) triples from start(x) = x * q + min(x, r) on, where
// q = grid / 8 and r = grid mod 8, i.e. the row blocks from start(x) / per_block (per_block = splits x column blocks; a row block
// cut by the boundary counts for the later XCD).  Workgroup b of this kernel also runs on XCD b mod 8 and takes the rows that
// XCD produced, for every batch column: its loads hit the L2 that the partial sums were written through, where the
// output-order kernel above finds most of them behind another XCD's L2 (measured: 4 MB written by one kernel are read by
// the next in 0.7 us from the writer's XCD and in 2.6 us from another).
template <bool BIAS>
__global__ __launch_bounds__(256) void splitk_reduce_by_xcd(half_t *__restrict__ C, const float *__restrict__ ws, uint32_t M, uint32_t N, int splitK,
                                                             uint32_t tile_rows, uint32_t q, uint32_t r, uint32_t per_block, const half_t *__restrict__ bias)
{
    const uint32_t x = blockIdx.x & 7u, j = blockIdx.x >> 3;
    const uint32_t s0 = x * q + (x < r ? x : r), s1 = (x + 1) * q + (x + 1 < r ? x + 1 : r);
    const uint32_t lo = s0 / per_block * tile_rows, hi = s1 / per_block * tile_rows, quads = (hi - lo) / 4;
    const uint32_t g = j * 256 + threadIdx.x;
    if (g >= quads * N) return;
    const uint32_t n = g / quads, m = lo + (g - n * quads) * 4;
    reduce_four<BIAS>(C, ws, (size_t)M * N, splitK, (size_t)n * M + m, BIAS ? bias + m : nullptr);
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Compute units of the current device, asked of the runtime once per device (the launch-shape rules and the measured table
// are written for 256; another count takes the rules).
int current_device_cus()
{
    static std::atomic<int> cus[64];
    int                     dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Rule for batches above 16 where no measured neighbour exists: score the six tile shapes that exhaustive sweeps showed to
// cover every case (64x32 with four K wavefronts; 128x32 with one or two; 128x64 with two; 256x64; 256x128) and take the
// best.  The score is the product of
//   * how full the chip is: workgroups / slots (one workgroup per CU, two for four-wavefront workgroups), divided by the
//     number of rounds that takes when there are more workgroups than slots;
//   * the share of the tile's columns that are real batch columns;
//   * pipeline fill: chunks / (chunks + 2), a workgroup with few K chunks is mostly prologue and epilogue;
//   * 1 / (1 + 32 * bytes through the CU's L1 per multiply-accumulate), which favours large tiles.
// Against an exhaustive sweep (99 problems, all compiled shapes) the choice loses 0.6 % on average and 15 % at worst.
struct TileShape { int nt, rt, wr, wk; };
constexpr TileShape kRuleShapes[] = { { 2, 1, 4, 4 }, { 2, 2, 4, 1 }, { 2, 2, 4, 2 }, { 4, 2, 4, 2 }, { 4, 2, 8, 1 }, { 8, 2, 8, 1 } };

inline double tile_score(size_t M, size_t N, size_t K, int splitK, const TileShape &t, int cus)
{
    const size_t TM = (size_t)t.wr * t.rt * 16, TN = (size_t)t.nt * 16, units = (K + 255) / 256, per_split = (units + splitK - 1) / splitK;
    if (M % TM || (size_t)t.wk > per_split) return 0.0;
    const size_t nblocks = (N + TN - 1) / TN;
    const double wgs = (double)(M / TM) * nblocks * splitK, slots = (double)cus * (t.wr * t.wk <= 4 ? 2 : 1);
    const double fill = wgs / slots, eff = fill >= 1.0 ? fill / std::ceil(fill) : fill;
    const double cover = (double)N / (double)(nblocks * TN);
    const double chunks = (double)per_split / t.wk, pipe = chunks / (chunks + 2.0);
    const double traffic = (0.75 * TM + 2.0 * TN) / ((double)TM * TN);
    return eff * cover * pipe / (1.0 + 32.0 * traffic);
}

// Estimated time in ns of the best shape for a given splitK: weight bytes at 6 TB/s divided by the score, plus, for a split, a
// second launch (2 us) and the FP32 partial sums written and read back (8 bytes per output per split at 8 TB/s).
inline double tile_estimate_ns(size_t M, size_t N, size_t K, int splitK, int cus, const TileShape **best_shape)
{
    double best = 0.0;
    for (const TileShape &t : kRuleShapes) {
        double sc = tile_score(M, N, K, splitK, t, cus);
        if (sc > best) { best = sc; if (best_shape) *best_shape = &t; }
    }
    if (best <= 0.0) return 1e30;
    double ns = (double)M * K * 0.75 / 6000.0 / best;
    if (splitK > 1) ns += 2000.0 + (double)splitK * M * N * 8.0 / 8000.0;
    return ns;
}

// ---- measured launch shapes (generated by `python -m fp6_llm_amd.tune`, MI355X, 256 CUs) ----
struct TuneCfg { uint8_t kind, nt, rt, wr, wk; uint16_t t; };              // t in 0.02 us; kind 255 = not measured
constexpr int kSplits[] = { 1, 2, 3, 4, 6, 8 };                             // the splits the table knows
constexpr int kNumSplits = sizeof(kSplits) / sizeof(kSplits[0]);
inline int split_index(int splitK) { for (int i = 0; i < kNumSplits; i++) if (kSplits[i] == splitK) return i; return -1; }
struct TuneEntry { uint8_t xb; uint16_t m256, k64, n; TuneCfg sk[kNumSplits]; };    // sk[i]: best shape for splitK = kSplits[i]
const TuneEntry kTune[] = {
    { 0, 0, 0, 0, { { 255, 0, 0, 0, 0, 0 }, { 255, 0, 0, 0, 0, 0 }, { 255, 0, 0, 0, 0, 0 }, { 255, 0, 0, 0, 0, 0 }, { 255, 0, 0, 0, 0, 0 }, { 255, 0, 0, 0, 0, 0 } } }, // keeps the array non-empty
#include "fp6mi_tuning.inc"
};

// (the stream kernel takes any number of row tiles per workgroup for any M: its last workgroup may hold fewer)
inline bool cfg_fits(const TuneCfg &c, size_t M) { return c.kind != 255 && (c.kind == 0 || M % (16u * c.rt * c.wr) == 0); }

// What the table says about a problem that need not be in it: per splitK the shape expected to be fastest and its expected
// time.  The batch is rounded UP to a measured batch of the same kernel family (a shape's cost steps at column-tile
// boundaries).  A measured (M, K) answers for itself; otherwise the up to four nearest measured problems (in ratio, at most a
// factor 1.5 away in M and in K) each propose their best shape per splitK, and a proposal's time is carried over to the
// query: in proportion to K, and for M by the number of rounds the shape's workgroups need on the chip.  Two matrices with
// 16384 and 17920 rows differ by 9 % in size but by a whole round of 64-row workgroups; sweeps off the grid showed that
// this, not the distance, decides which neighbour's shape is right.  Farther neighbours pay 15 % per octave of distance.
struct TuneGroup { int xb; size_t n, begin, end; }; // entries [begin, end) of kTune share format and batch (the table is sorted by them)
struct TuneAnswer { bool valid, measured, exact; size_t n; LaunchCfg cfg[kNumSplits]; float t[kNumSplits], by_k[kNumSplits]; }; // index i: splitK = kSplits[i]; t in 0.02 us, 0 = no proposal; by_k: t in proportion to K as a whole; measured: this very (M, K) at this or the next larger measured batch; exact: at this batch; n: the measured batch that answers

const std::vector<TuneGroup> &tune_groups()
{
    static const std::vector<TuneGroup> groups = [] {
        std::vector<TuneGroup> g;
        const size_t           count = sizeof(kTune) / sizeof(kTune[0]);
        for (size_t i = 1; i < count; i++) {
            if (g.empty() || g.back().xb != kTune[i].xb || g.back().n != kTune[i].n) g.push_back(TuneGroup{ kTune[i].xb, kTune[i].n, i, i });
            g.back().end = i + 1;
        }
        return g;
    }();
    return groups;
}

inline double rounds_on_chip(const TuneCfg &c, size_t M, size_t N, int splitK)
{
    const size_t TM = (size_t)(c.kind >= 1 ? c.wr : 1) * c.rt * 16, TN = (size_t)c.nt * 16;
    const double wgs = (double)((M + TM - 1) / TM) * (double)((N + TN - 1) / TN) * splitK;
    // tile kernel: one workgroup per CU, two for four-wavefront workgroups.  Stream kernel: several workgroups share a CU, but
    // they share its memory pipeline too, so what counts is the largest number of workgroups any CU is given.
    const double slots = 256.0 * (c.kind == 1 && c.wr * c.wk <= 4 ? 2 : 1);
    return std::ceil(wgs / slots);
}

// What a launch takes however short K is, in 0.02 us: 2 us, and with a split 2 us for the reduction's launch and the partial sums at 8 TB/s, as
// in tile_estimate_ns.  (Twice a time less the time at twice the K, over the table from 2048 columns on: 3-4 us unsplit, 5-8 us and the partial
// sums with a split.)  Up to 320 columns the splits are compared with this part carried over as it is and the rest in proportion; the shapes of one split
// are not.  In proportion to K as a whole, a split's time shrank with the part that does not, and matrices of little K were cut that none of their
// neighbours gains by: FP4 1280x2304 N 113 in eight (8.5 us, 5.5 unsplit), FP6 2048x3456 N 231 in four (11.0, 8.8), FP5 1536x1408 N 47 in three (5.9, 4.1).
// Time of the choice / time of the best proposal on 324 matrices off the table, every proposal measured: N 33-80 1.07 before, 1.02 now, N 81-160 1.02 and
// 1.01, N 161-320 1.03 and 1.02.  So it is up to 16 columns, and 17 to 32 with K up to 3072 or M up to 2560.  Time / time by proportion of what changes by it: an uncut launch in the place
// of a cut one, which in a stream saves the host 2.6 us besides, 0.87 in a graph (0.56-1.16) and 0.78 in a stream (0.64-1.05) on 891 problems up to 16 columns, 0.85 (0.61-1.17) and
// 0.82 (0.65-1.14) on 343 beyond (e3m2 2304x2176 N 13 in three 5.8 and 10.8 us, uncut 4.2 and 4.4; 2560x2688 N 5 in three 5.5 and 9.1, uncut 3.8 and 4.7); a graph alone is the slower by it
// where few rows meet a long K (M up to 1536 and K from 9216 1.05 and 0.85 in a stream: e2m1 1536x12480 N 3 in four 6.3 and 7.9, uncut 7.4 and 7.4).  Another cut is 0.99 and 1.00 on 216
// up to 16 columns, one of them 1.12.  From 17 on the stream kernel in three or four pieces, which the times above prefer to the tile kernel in six or eight, is behind it: 1.09 (0.94-1.27) on 62
// problems (e2m2 2048x14144 N 21 12.1 us, in eight 10.0), so that best_narrow leaves those as proportion has them.  Left as they were: the other 17 to 32 columns (1.04-1.22 on ten problems
// whose tiles in six or eight gave way to the stream kernel uncut), and beyond 320, where the few splits measured are for long K (11520x12800 N 456: 152 us in two pieces, 172 uncut).
inline double fixed_part(size_t M, size_t N, int splitK)
{
    return splitK == 1 ? 100.0 : 200.0 + (double)splitK * M * N * 8.0 / 8e6 / 0.02;
}

const TuneAnswer *tune_lookup(int xbits, size_t M, size_t N, size_t K)
{
    // a serving loop asks for the same few layer shapes at whatever batch size the scheduler formed: remember answers
    struct Memo { int xb; size_t M, N, K; TuneAnswer a; };
    static thread_local Memo memo[256];
    Memo &slot = memo[(M * 0x9E3779B97F4A7C15ull + N * 0xC2B2AE3D27D4EB4Full + K * 0x165667B19E3779F9ull + (size_t)xbits) >> 56];
    if (slot.xb == xbits && slot.M == M && slot.N == N && slot.K == K) return slot.a.valid ? &slot.a : nullptr;
    const TuneGroup *group = nullptr, *widest = nullptr;
    for (const TuneGroup &g : tune_groups()) {
        if (g.xb != xbits || (g.n <= 16) != (N <= 16)) continue;
        if (g.n >= N && (!group || g.n < group->n)) group = &g;
        if (!widest || g.n > widest->n) widest = &g;
    }
    if (!group) group = widest; // batches beyond the largest measured one behave like it, only with more column blocks
    constexpr int    kNear = 4;
    const TuneEntry *near[kNear] = {};
    float            dist[kNear] = {};
    int              count = 0;
    if (group) {
        const float lm = std::log2((float)M / 256.f), lk = std::log2((float)K / 64.f);
        for (size_t i = group->begin; i < group->end; i++) {
            const TuneEntry &e = kTune[i];
            float dm = std::fabs(lm - std::log2((float)e.m256)), dk = std::fabs(lk - std::log2((float)e.k64));
            if (dm > 0.585f || dk > 0.585f) continue;
            int pos = count < kNear ? count : kNear - 1; // insertion into the sorted list of the nearest
            if (count == kNear && dm + dk >= dist[pos]) continue;
            while (pos > 0 && dist[pos - 1] > dm + dk) { near[pos] = near[pos - 1]; dist[pos] = dist[pos - 1]; pos--; }
            near[pos] = &e, dist[pos] = dm + dk;
            if (count < kNear) count++;
        }
    }
    TuneAnswer a = {};
    a.n = group ? group->n : 0;
    if (count > 0 && dist[0] == 0.f) count = 1, a.measured = true, a.exact = group->n == N; // measured: nothing to carry over
    const size_t units = (K + 255) / 256;
    for (int j = 0; j < count; j++) {
        const TuneEntry &e = *near[j];
        const size_t     Me = (size_t)e.m256 * 256, Ke = (size_t)e.k64 * 64, Nq = N > group->n ? N : group->n;
        for (int i = 0; i < kNumSplits; i++) {
            const TuneCfg &c = e.sk[i];
            if (!cfg_fits(c, M) || (size_t)kSplits[i] > units) continue;
            const double rounds = rounds_on_chip(c, M, Nq, kSplits[i]) / rounds_on_chip(c, Me, group->n, kSplits[i]);
            double       t = (double)c.t * (double)K / (double)Ke * (1.0 + 0.15 * dist[j]);
            t *= rounds;
            if (a.t[i] == 0.f || (float)t < a.by_k[i]) { // (the shapes of one split are compared in proportion)
                a.by_k[i] = a.t[i] = (float)t;
                a.cfg[i] = LaunchCfg{ c.kind, c.nt, c.rt, c.wr, c.wk };
                a.valid = true;
                if (!a.measured && N <= 320 && (N <= 16 || N > 32 || K <= 3072 || M <= 2560)) {
                    const double there = std::fmin(fixed_part(Me, group->n, kSplits[i]), 0.8 * c.t), here = std::fmin(fixed_part(M, Nq, kSplits[i]), 0.8 * c.t);
                    a.t[i] = (float)((here + (c.t - there) * (double)K / (double)Ke * rounds) * (1.0 + 0.15 * dist[j]));
                }
            }
        }
    }
    slot = Memo{ xbits, M, N, K, a };
    return a.valid ? &slot.a : nullptr;
}

// Whether gemm_prefill's 128 x 128 tile replaces the shape `c` of another large-batch kernel.  Its workgroups take a CU as long as half a
// 256 x 128 one does (7 ns per column of K, measured from 64 to 3600 workgroups) and as long as a 256 x 64 one of the same area, so what
// decides first is the number of rounds on the chip.  Time here / time of the other shape (no splits, launches in a captured graph; median and range).
// Where the rule takes it, on 873 problems (M 2304-56832, K 64-27584, N 150-3867, all formats), with row scales only and with group exponents:
//   * from 256 x 128, fewer half rounds and K of 320 at least: 0.82 (0.65-0.94) and 0.85 (0.65-0.99) up to N 1024, 0.84 (0.63-0.95) and 0.88 (0.64-0.99) up to
//     N 2048; beyond, an eighth fewer, 0.84 (0.77-0.98) and 0.86 (0.80-0.97);
//   * from 256 x 64, as many rounds and two at least: 0.91 (0.77-1.04) and 0.91 (0.78-1.00); above 1 in 21 problems with row scales only and K of 3840 at least.
// Since large tiles are counted in panels, on problems with M 1024-28672, K 1024-28672 (6, 5 and 4 bits; row scales, then group exponents):
//   * from 256 x 128 between N 512 and 3072 it takes over whatever the rounds: as many half rounds 0.94 (0.83-1.02) on 1160 problems and 0.97 (0.87-1.04) on 368, fewer
//     0.85 (0.73-0.91) on 249 and 0.88 (0.77-0.94) on 83; rows of a multiple of 8 KB are no exception any more (N above 2048: 0.88, 0.73-1.00, and 0.92, 0.77-1.03);
//   * from 256 x 64 between N 2048 and 3072: 0.97 (0.87-1.05) on 208 and 0.90 (0.83-0.96) on 73, above 1.02 on 8, all with row scales only; with K 64-960
//     0.80 (0.71-0.92) on 64 and 0.81 (0.72-0.94) on 26.
// Beyond N 3072 the lines are those of before the panels, and so they are up to N 512 and, from 256 x 128, for K below 1024.
// Where it did not win before the panels, on 217 problems and (*) on 687 of another sweep, row scales only:
//   * 256 x 128 with K below 320, prologue and epilogue being most of it: 0.99 (0.95-1.05) with fewer half rounds, with group exponents 1.03 (0.99-1.10);
//   * (*) N up to 144, the second column block nearly empty: 256 x 128 0.98 (0.96-1.01), 256 x 64 1.16 (1.01-1.50);
//   * as many half rounds of 256 x 128, N up to 1024 (since the panels the line is at 512): 1.00 (0.92-1.10), with group exponents, whose loads come twice as often per output, 1.05 (0.95-1.19);
//   * (*) from 256 x 64: a single round 1.19 (1.00-1.86), more rounds 1.29 (0.87-1.44) up to N 1024;
//   * (*) long prompts, where what the activations cost comes in: with K above 8192, N above 3072 and an eighth fewer half rounds 0.97-1.06 (a quarter fewer
//     0.79-0.98 up to N 3712), N above 4096 with K above 3072 1.00 (0.89-1.12, no line found between the two; up to K 3072 0.92, 0.85-0.96).
// (*) Faster there on the whole, but not taken over, beyond N 3072: as many half rounds of 256 x 128 (0.94, 0.87-1.11), less than an eighth gained
// (0.88, 0.81-1.02), 256 x 64 (0.90, 0.74-1.04; with K above 8192 1.08) and rows of a multiple of 8 KB (256 x 128 0.92, 0.77-1.11; 256 x 64 0.98, 0.91-1.21).
inline bool prefill_tile_wins(const LaunchCfg &c, size_t M, size_t N, size_t K, int splitK, int cus)
{
    if (splitK != 1 || N <= 144 || K > (size_t)1 << 20 || (N > 3072 && K % 4096 == 0)) return false;
    if ((N > 3712 && K > 8192) || (N > 4096 && K > 3072)) return false;
    auto         rounds = [&](size_t rows, size_t cols) { return (M / rows * ((N + cols - 1) / cols) + cus - 1) / cus; };
    const size_t here = rounds(128, 128);
    if (c.kind == 1 && c.nt == 8 && c.rt == 2 && c.wr == 8 && c.wk == 1) {
        const size_t half = 2 * rounds(256, 128); // never less than `here`
        if (N > 512 && N <= 3072 && K >= 1024) return true;
        return K >= 320 && (N <= 2048 ? here < half : 8 * here <= (N > 3072 && K > 8192 ? 6 : 7) * half);
    }
    if (c.nt == 4 && c.rt == 2 && c.wr == 8 && (c.kind == 2 || (c.kind == 1 && c.wk == 1))) return rounds(256, 64) >= 2 && here <= rounds(256, 64) && N <= 3072;
    return false;
}

// Whether it replaces the shape the table gives for kSplits[i] on 256 CUs.  A problem that was itself measured keeps its shape.
inline bool prefill_replaces(const TuneAnswer &a, int i, size_t M, size_t N, size_t K)
{
    return !a.exact && prefill_tile_wins(a.cfg[i], M, N, K, kSplits[i], 256);
}

// K up to which the rules, which answer where the table does not, never split: its launch and partial sums (3 us and more) against at most five and a half K blocks.  On 440
// problems out of the table's reach with K 64-1472 and N 17-500 the best split was 1 every time.  (The table, whose least K is 2048, reaches K 1408 for some M and N and answers
// there for itself, in up to three pieces; K up to 1344 is the rules' everywhere.)
constexpr size_t kLittleK = 1408;

// Launch shape for a given splitK.
//  N <= 16: stream kernel.  Row tiles per wavefront (rt) reuse the activation registers, so rt grows with M; wavefronts
//           per workgroup follow the K blocks of one split and the register budget (16 wavefronts leave 128 VGPRs each).
//  N > 16:  stream kernel where K and the outputs are few, else tile kernel, 128 rows x 32 or 64 columns, with the K parallelism that splitK leaves open given to the
//           wavefronts of the workgroup (at most what its LDS holds).
inline LaunchCfg pick_cfg(int xbits, size_t M, size_t N, size_t K, int splitK, int cus)
{
    LaunchCfg c;
    if (const int i = split_index(splitK); cus == 256 && i >= 0) {
        if (const TuneAnswer *a = tune_lookup(xbits, M, N, K)) {
            if (a->t[i] > 0.f) return prefill_replaces(*a, i, M, N, K) ? LaunchCfg{ 2, 8, 4, 2, 2 } : a->cfg[i];
        }
    }
    size_t    tiles = M / 16, units = (K + 255) / 256, per_split = (units + splitK - 1) / splitK;
    if (N <= 16) {
        c.kind = 0;
        c.nt = 1;
        c.wr = 1;
        // Fitted to a sweep of every compiled shape over M in 2048..28672, K in 4096..28672, N in 1..16, both formats, on
        // the MI355X.  What it encodes: about eight to eleven wavefronts per CU keep the memory system full; small
        // workgroups (four wavefronts) balance better than large ones once there are several per CU; sharing the
        // activation registers among row tiles (rt) pays in proportion to the batch, because every workgroup pulls the
        // whole activation matrix through its CU's L1.
        const double per_cu = (double)tiles * splitK / cus; // 16-row tiles per CU
        if (N <= 4) {
            if (per_cu < 1.5)        { c.rt = 1; c.wk = N <= 2 ? 16 : 8; }
            else if (per_cu < 2.5)   { c.rt = 2; c.wk = 8; }
            else if (per_cu < 3.125) { c.rt = 1; c.wk = 4; }
            else if (per_cu < 5.5)   { c.rt = 2; c.wk = 4; }
            else                     { c.rt = 2; c.wk = 8; }
        } else {
            // Batches 5..16: every row tile a workgroup adds re-uses its activation registers, and a CU is done when its last
            // workgroup is, so give each CU its share of the row tiles in as few workgroups as hold them (at most eight tiles):
            // cost of rt tiles per workgroup = rounds of the 256 CUs x rt.  10240, 11008 and 12288 rows take 3, 17920 and 19968
            // rows 5, 22016 rows 6, 28672 rows 7 (measured: 5-20 % better than the power of two next to them).  Ties go to the
            // larger workgroup (12288 rows: three tiles at once beat three workgroups of one by 7 %).
            int    best = 1;
            size_t best_cost = ~(size_t)0;
            for (int rt = 1; rt <= 8; rt++) {
                const size_t wgs = (tiles + rt - 1) / rt * splitK, cost = (wgs + cus - 1) / cus * rt;
                if (cost <= best_cost) best = rt, best_cost = cost;
            }
            c.rt = best;
            c.wk = best >= 5 || (best == 4 && N > 8) ? 4 : 8;
        }
        while ((c.rt == 2 || c.rt == 4 || c.rt == 8) && tiles % c.rt) c.rt /= 2; // (the other counts need not divide: the last workgroup holds the rest)
        const int cap = per_split > 8 ? 16 : per_split > 4 ? 8 : 4; // no more wavefronts than K blocks to hand out
        if (c.wk > cap) c.wk = cap;
        if (c.rt == 4 && c.wk == 16) c.wk = 8; // not compiled: 16 wavefronts leave too few registers for four row tiles
        (void)xbits;
        return c;
    }
    // Little K, few outputs: the stream kernel over several column blocks, whose workgroups are many and done when their few K blocks are.  Per CU w workgroups of 16 x 16
    // outputs; time here / the rules' tile unsplit / the best of all shapes, on 190 problems (M 256-28672, N 17-500): two and three K blocks up to w = 8 0.64 and 1.01 (up to
    // 1.17 of the tile's beyond); from five on w up to 3 0.53-0.70 and 1.00-1.03, up to 4 0.75-0.79 and 1.02, up to 6 0.90-0.97 and 1.00-1.06, and beyond it the tiles are level
    // or ahead.  On 1500 other problems that it changes (K 64-1472, N 17-500, group exponents on 30 %) 0.62 of the time before in a graph, 0.86 in a stream, 6 above 1.03 (up to
    // 1.09); N 33-96 at w 5 to 6 1.00 (0.92-1.11).  us, before -> here: e2m1 1280x1216 N 21 6.7 -> 3.2, e2m2 3584x1088 N 20 7.2 -> 3.8, 2304x1088 N 31 7.8 -> 3.9, e3m2 3328x1344
    // N 41 6.5 -> 4.9.  5 bits: two row tiles on eight wavefronts take 135-142 registers there, 122-128 with 6 and 4 bits, and a CU holds one such workgroup instead of two: beyond
    // 128 columns 1.04 (0.99-1.09) of the tile's time where it would need a second round (w 2 to 4; 512x1280 N 385 6.1 -> 6.6), level up to 128 columns.  (A single K block leaves
    // all wavefronts but one idle; four of them stay with the tiles of four K wavefronts, which take them in one chunk: 0.74 here.)
    const size_t columns = (N + 15) / 16, wgs = tiles * columns, some = (size_t)cus;
    if (splitK == 1 && K <= kLittleK && units > 1 && units != 4 && wgs <= (units < 4 ? 8 : 6) * some) {
        if (units < 4) return LaunchCfg{ 0, 1, wgs < 3 * some ? 1 : 2, 1, 4 };
        const bool three = wgs > 2 * some && (tiles + 2) / 3 * columns <= some, one_to_a_cu = xbits == 5 && wgs <= 4 * some;
        if (wgs <= 2 * some || three || !one_to_a_cu || N <= 128) return LaunchCfg{ 0, 1, wgs <= some ? 1 : three ? 3 : 2, 1, wgs <= 4 * some ? 8 : 4 };
    }
    c.kind = 1;
    const TileShape *t = nullptr;
    tile_estimate_ns(M, N, K, splitK, cus, &t);
    if (!t) t = &kRuleShapes[1]; // 128 x 32, one K wavefront: divides every legal M and needs a single K block
    c.nt = t->nt, c.rt = t->rt, c.wr = t->wr, c.wk = t->wk;
    return prefill_tile_wins(c, M, N, K, splitK, cus) ? LaunchCfg{ 2, 8, 4, 2, 2 } : c;
}
// ---- gemm_wide: which of its tiles a problem takes, and whether it takes the place of the shape of the table or the rules ----
// Every tile of gemm_wide is one sum of rounds: its workgroups take the same time, and a CU holds one of eight wavefronts or two of four (two of eight
// where a wavefront takes at most 128 registers).  So a time is (full rounds) x (fixed + K x rate) + (the last, partly filled round), and a split adds its
// launch and its partial sums.  The constants are least squares of the relative error over 1050 problems (M 1024-28672, K 1024-28672, N 65-4096, most of them
// up to 600; 6, 5 and 4 bits; group exponents on 30 %; weights and activations changed from launch to launch, splits 1, 2, 3, 4, 6 and 8): 4-7 % off a single
// time, the smallest tiles most.  The shape and split that come out smallest are 0.8 % behind the best of these shapes on average, with a constant term, rates
// and splits only 1.1 %.
// gemm_span's tiles (odd widths, and 256 x 96 with the halves of K side by side) were fitted later, to 252 problems of N 97-1500 on which all twelve were measured (4-5 %
// off; what group exponents cost was taken from their neighbours).  Where they are asked, and what they have to be ahead by: span_margin.
struct WideShape {
    int   nt, rt, wk, slots;              // column tiles, row tiles per wavefront, K halves; workgroups that 256 CUs hold
    float full, full_k, full_kg;          // a full round: us, us per column of K, the same with group exponents on top
    float part, part_k, part_kf, part_kg; // the last round, of at most half the slots where a CU holds two workgroups: us, per column of K, that times its fill, group exponents
    float k6, k5;                         // either round, per column of K: 6- and 5-bit weights on top of 4-bit ones
    float base, x_mb, w_mb, out;          // once per launch; per MB of activations, per MB of weights; per million outputs unsplit
    float split, split_out;               // a split's second launch, and its partial sums per million of them
};
constexpr WideShape kWide[] = {
    { 3, 2, 2, 512, 0.f, 0.00481f, 0.0004f, 0.419f, 0.00315f, 0.000117f, 0.00013f, 0.000505f, 0.000437f, 1.77f, 0.262f, 0.0942f, 0.879f, 2.29f, 1.69f },
    { 4, 2, 2, 512, 0.64f, 0.00565f, 0.000445f, 0.779f, 0.0034f, 0.00017f, 0.000127f, 0.000512f, 0.000543f, 1.26f, 0.353f, 0.0607f, 0.85f, 2.89f, 1.35f },
    { 5, 2, 2, 256, 0.818f, 0.00446f, 0.0003f, 1.59f, 0.00369f, 0.000268f, 0.0002f, 0.000214f, 0.000416f, 1.55f, 0.303f, 0.0898f, 0.462f, 1.89f, 1.59f },
    { 5, 4, 2, 256, 1.71f, 0.00656f, 0.000388f, 1.76f, 0.00553f, 0.000671f, 0.000812f, 0.000938f, 0.000901f, 2.78f, 0.074f, 0.0772f, 0.627f, 2.98f, 1.47f },
    { 6, 2, 2, 256, 2.3f, 0.00496f, 0.000302f, 1.35f, 0.004f, 0.000994f, 0.000294f, 0.000379f, 0.000471f, 1.46f, 0.346f, 0.0541f, 0.205f, 2.77f, 0.936f },
    { 6, 4, 1, 512, 0.f, 0.0145f, 0.000878f, 0.0154f, 0.00811f, 0.000511f, 0.00109f, 0.000564f, 0.000919f, 3.3f, 0.144f, 0.0501f, 0.475f, 3.8f, 1.12f },
    { 6, 4, 2, 256, 3.7f, 0.00801f, 0.000388f, 4.22f, 0.00596f, 0.00166f, 0.000812f, 0.000649f, 0.000689f, 1.73f, 0.0414f, 0.0428f, 0.288f, 2.95f, 1.19f },
    { 7, 2, 2, 256, 1.9f, 0.00514f, 0.000315f, 2.78f, 0.00393f, 0.000609f, 0.00034f, 0.000385f, 0.000465f, 1.09f, 0.374f, 0.0979f, 0.328f, 1.87f, 1.37f },
    { 7, 4, 2, 256, 3.24f, 0.00918f, 0.000388f, 4.28f, 0.00669f, 0.00179f, 0.000812f, 0.000591f, 0.000692f, 1.68f, 0.0537f, 0.0378f, 0.299f, 3.07f, 1.2f },
    { 8, 2, 2, 256, 3.11f, 0.00552f, 0.000329f, 1.13f, 0.00458f, 0.00138f, 0.000385f, 0.000557f, 0.000652f, 1.93f, 0.272f, 0.0636f, 0.0816f, 2.61f, 1.11f },
    { 8, 4, 1, 512, 0.f, 0.0187f, 0.000715f, 0.434f, 0.00994f, 0.000692f, 0.00107f, 0.0006f, 0.00103f, 3.6f, 0.119f, 0.0321f, 0.458f, 3.81f, 1.15f },
    { 8, 4, 2, 256, 3.85f, 0.0102f, 0.000388f, 2.21f, 0.00798f, 0.00154f, 0.000812f, 0.000575f, 0.000692f, 3.05f, 0.119f, 0.021f, 0.325f, 3.17f, 1.19f },
};

inline float wide_estimate(const WideShape &w, int xbits, size_t M, size_t N, size_t K, int splitK, bool groups)
{
    const size_t units = (K + 255) / 256, kc = (units + splitK - 1) / splitK * 256;
    const size_t wgs = M / (64u * w.rt) * ((N + 16 * w.nt - 1) / (16 * w.nt)) * splitK;
    size_t       full = wgs / w.slots, rest = wgs % w.slots;
    if (w.slots == 512 && rest > 256) full++, rest = 0;
    const float k = (float)kc, kf = k * (xbits == 6 ? w.k6 : xbits == 5 ? w.k5 : 0.f), out = (float)M * (float)N * 1e-6f;
    float       t = w.base + w.x_mb * (float)N * (float)K * 2e-6f + w.w_mb * (float)M * (float)K * (float)xbits * 0.125e-6f;
    t += (float)full * (w.full + k * (w.full_k + (groups ? w.full_kg : 0.f)) + kf);
    if (rest) t += w.part + k * (w.part_k + w.part_kf * (float)rest / 256.f + (groups ? w.part_kg : 0.f)) + kf;
    return t + (splitK > 1 ? w.split + w.split_out * (float)splitK * out : w.out * out);
}

// What gemm_span's tile has to be ahead of gemm_wide's by; 0: it is not asked.  2.5 %, with a split or K below 1536 4 %, and with a last round more than three quarters full 3 % more
// for a split and for 128 x 112, which take that much longer there than their rows say (e3m2 2048x2176 N 1635 18.2 us, with 128 x 128 17.0).  From K 1024 up to N 3072, what lies
// beyond not having been measured; 128 x 48 up to N 600 (beyond, shapes of the table whose place it took were up to 11 % ahead of it).
// The rows of the 128-row tiles, fitted to K of some thousand, expect too little of a long K: measured / expected on 1900 problems 1.02 up to K 4096 and 1.12 beyond for 128 x 80, 1.02 and
// 1.11 for 128 x 112, 1.05 and 1.13-1.19 (K of a piece from 8192 on) for 128 x 48; gemm_wide's tiles and the 256-row ones 0.99-1.05.  Against gemm_wide at the same split they hold all the same
// (128 x 80: 0.95 of its time on 213 problems, none above 1.00; 128 x 48 0.98), but not everywhere, and not across splits.  Time / time of what is launched instead:
//   * 128 x 112 uncut without group exponents, beyond N 1400: 1.03 of 128 x 128 (109 problems; 0.965 up to there); with a last round below seven eighths and K from 8192: 1.09 (1.07-1.14) of
//     128 x 96, and 1.06 of the table's shapes.  With group exponents it holds against all (0.87-0.99 on 372 problems) but 128 x 96, K from 8192: 1.08-1.11 where their rows are within 15 %;
//   * 256 x 80 uncut, more columns than rows, K from 4096: 1.09 (1.03-1.15) of 128 x 128 on 33 of 60 problems, which a margin of 8 % finds; it is ahead of the other span tiles all
//     the same (0.94 of 256 x 96, 0.91-0.96, on 103 problems);
//   * uncut tiles of 128 rows in the place of a cut one: 1.06 (0.94-1.22) of gemm_wide's, 1.08-1.12 of a 256-row one; 128 x 112 in pieces 1.02, uncut 256 x 80 beyond K 20480
//     1.025.  They leave the choice of a split to the others;
//   * 128 x 48 in the place of the table's shape, K of a piece from 4096 and a single round of up to 256 workgroups: 1.09 (0.86-1.32).  wide_replaces allows for it.
// All of it together, against the choice without gemm_span: 1200 problems of N 97-4096 that it changes 0.93, 24 above 1.03 (up to 1.10, one 1.25: e3m2 15616x6656 N 132 with group
// exponents); 900 unsplit 0.91, 14 (1.10); 900 of a given split 0.93, 17 (1.11).
// Without these lines, on half as many, 0.94 with 53 above 1.03 (1.23), 0.92 with 23 (1.30: e2m3 1536x16448 N 2161 122 -> 159 us) and 0.93 with 11 (1.08).
inline float span_margin(const WideShape &w, size_t M, size_t N, size_t K, int splitK, bool groups)
{
    const bool   span112 = w.rt == 2 && w.nt == 7;
    const size_t last = M / (64u * w.rt) * ((N + 16 * w.nt - 1) / (16 * w.nt)) * splitK % w.slots; // workgroups of the last round, 0 for a full one
    if (K < 1024 || N > (w.nt == 3 ? 600 : span112 && splitK == 1 && !groups ? 1400 : 3072)) return 0.f;
    if (span112 && splitK == 1 && !groups && K >= 8192 && last && 8 * last < 7 * (size_t)w.slots) return 0.f;
    if (w.nt == 5 && w.rt == 4 && splitK == 1 && N > M && K >= 4096) return 1.08f;
    return (splitK > 1 || K < 1536 ? 1.04f : 1.025f) + ((splitK > 1 || span112) && (last == 0 || 4 * last >= 3 * (size_t)w.slots) ? 0.03f : 0.f);
}

// Which of gemm_span's tiles are asked: none; those that take part in the choice of a split; all.
enum class Spans { kNone, kForSplit, kAll };
inline bool span_asked(const WideShape &w, Spans spans, size_t K, int splitK)
{
    if (spans != Spans::kForSplit) return spans == Spans::kAll;
    return w.rt == 2 ? splitK > 1 && w.nt != 7 : w.nt != 5 || splitK > 1 || K <= 20480;
}

// the fastest of the shapes for a given split, and its time in us; 0 where none fits
inline float wide_best(LaunchCfg &c, int xbits, size_t M, size_t N, size_t K, int splitK, bool groups, Spans spans)
{
    float best = 0.f, t96 = 0.f, t80 = 0.f; // t96: of gemm_wide's 128 x 96; t80: of 256 x 80, where it is held to more against gemm_wide
    if (N <= 96 || K > (size_t)1 << 20 || (size_t)splitK > (K + 255) / 256) return best;
    for (const WideShape &w : kWide) {
        float t = wide_estimate(w, xbits, M, N, K, splitK, groups);
        if (w.nt == 6 && w.rt == 2) t96 = t;
        if (w.nt % 2 || (w.nt == 6 && w.rt == 4 && w.wk == 2)) { // gemm_span's
            const float margin = span_asked(w, spans, K, splitK) ? span_margin(w, M, N, K, splitK, groups) : 0.f;
            if (margin == 0.f || (groups && w.nt == 7 && w.rt == 2 && splitK == 1 && K >= 8192 && t * 1.15f > t96)) continue;
            if (margin == 1.08f) t80 = t * 1.025f;
            t *= margin;
        }
        if (best == 0.f || t < best) best = t, c = LaunchCfg{ 2, w.nt, w.rt, 4, w.wk };
    }
    if (t80 > 0.f && t80 < best && c.rt == 4 && c.wk == 2 && c.nt < 8) c.nt = 5; // (another of gemm_span's is ahead of gemm_wide's, and this one of it)
    return best;
}

// us that the table expects of a split on 256 CUs; 0 for none.  A row's time is that of the measured batch, which the query rounds up to: what this batch
// saves in rounds of the chip is taken off the part of it that is not fixed.
inline float narrow_estimate(const TuneAnswer *a, size_t M, size_t N, int splitK)
{
    const int i = split_index(splitK);
    if (!a || i < 0 || a->t[i] <= 0.f) return 0.f;
    if (N <= 96) return a->t[i] * 0.02f; // (where nothing else is compared with it)
    const LaunchCfg &c = a->cfg[i];
    const TuneCfg    tc = { (uint8_t)c.kind, (uint8_t)c.nt, (uint8_t)c.rt, (uint8_t)c.wr, (uint8_t)c.wk, 0 };
    const float      t = a->t[i] * 0.02f, fixed = std::fmin((float)fixed_part(M, N, splitK) * 0.02f, 0.8f * t);
    return fixed + (t - fixed) * (float)(rounds_on_chip(tc, M, N, splitK) / rounds_on_chip(tc, M, a->n > N ? a->n : N, splitK));
}

// Whether gemm_wide, expected to take t us, takes the place of the table's shape, expected to take `narrow` (0: not in the table's reach, K below 1366 for
// the most part; there it is a matter of the outputs, of which the rules' smaller tiles serve few better: 1536x1216 N 258 5.4 us against 7.3,
// 3072x1024 N 2867 26.0 against 22.5).  Time after / before on 500 problems that no line was drawn on (M and K 1024-28672, group exponents on 30 %, the split chosen anew):
// N 97-160 0.99 (0.84-1.03), N 161-256 0.98 (0.81-1.07), N 257-400 0.91 (0.60-1.02), N 401-640 0.85 (0.50-1.01), beyond 0.84 (0.36-1.04), 5 of all over 1.02 (16640x2752
// N 186 with group exponents 1.07); N 65-96 1.00, not worth it.  The margins are what the two estimates are off where the kernels are close, and allow for the
// table's, which is low, where they are not: of 849 problems that they were drawn on 40 were over 1.02 without them, 5 with them.
// The tile of 64 columns has the smallest margin whatever N is: on 175 problems beyond N 640 it took with 1.15 (1024x6144 N 1848, 2560x19904 N 3224) it was 1.00
// (0.56-1.28), 71 of them over 1.02; with 0.9 it takes 44 of them at 0.91 and 4 are over 1.02 (9472x17024 N 1984 in FP4 1.28, the others up to 1.03); on 34 problems of N 401-640 as good as with 0.95, 1 over 1.02 for 5.
// Out of the table's reach K up to 512 takes 2^22 outputs: 23 problems below that took 1.02 of the time of the rules' tiles (0.90-1.22: 5632x256 N 325 4.9 us -> 5.9);
// of the 177 others, 0.87 (0.63-1.09), 8 are over 1.02.
// (128 x 48 with a long K in a single round takes longer than its row says: see span_margin.)
inline bool wide_replaces(const LaunchCfg &wide, float t, float narrow, size_t M, size_t N, size_t K, int splitK)
{
    if (t <= 0.f) return false;
    if (wide.nt == 3 && K / splitK >= 4096 && M / 128 * ((N + 47) / 48) * splitK <= 256) t *= 1.2f;
    if (narrow <= 0.f) return M * N >= (size_t)1 << (K <= 512 ? 22 : 20);
    return t < narrow * (N <= 400 || wide.nt <= 5 && wide.rt == 2 ? 0.9f : N <= 640 ? 0.95f : 1.15f);
}

// The fastest split of the table's (3 % hysteresis towards fewer pieces; 10 % towards a single launch against pieces expected to take less than 8 us, since two launches take
// that of the host alone) and its time
// in us; 0 where it holds none.  One that takes more than ws_bytes has to be
// the faster by the table's times as they stand too, which were what decided before narrow_estimate.
inline float best_narrow(int &split, const TuneAnswer *a, size_t M, size_t N, size_t ws_bytes)
{
    float best = 0.f;
    split = 0;
    for (int s : kSplits)
        if (const float t = narrow_estimate(a, M, N, s); t > 0.f && (split == 0 || t * (split == 1 && t < 8.f ? 1.1f : 1.03f) < best)) {
            if (split && fp6mi_workspace_bytes(M, N, s) > ws_bytes && a->t[split_index(s)] * 1.03f >= a->t[split_index(split)]) continue;
            split = s, best = t;
        }
    if (N > 16 && N <= 32 && split > 1 && a->cfg[split_index(split)].kind == 0) { // a tile kernel in more pieces where proportion says so: see fixed_part
        int   cut = 0;
        float least = 0.f;
        for (int i = 0; i < kNumSplits; i++)
            if (const float t = a->by_k[i]; t > 0.f && (least == 0.f || t * 1.03f < least)) cut = i, least = t;
        if (cut && a->cfg[cut].kind != 0) split = kSplits[cut], best = a->t[cut] * 0.02f;
    }
    return best;
}
// The launch shape of a call: gemm_wide's, or that of the table and the rules.  A split that the table does not hold for a problem it does hold (in other
// splits) is compared with the fastest of those, as the heuristic, which knows no group exponents, does before it answers with one: of what the rules would
// launch there neither has a time.  60 problems whose split the rules launched until then (1280x2624 N 525 in four, say), time / time before gemm_wide: 0.74 (0.39-1.03), 0.77
// (0.37-1.26) by the rules.
inline LaunchCfg final_cfg(int xbits, size_t M, size_t N, size_t K, int splitK, bool groups, int cus)
{
    if (cus == 256 && N > 96) {
        const TuneAnswer *a = tune_lookup(xbits, M, N, K);
        const float       here = narrow_estimate(a, M, N, splitK);
        LaunchCfg         wide = {};
        auto              replaces = [&](Spans spans) { // (sets `wide`)
            const float t = wide_best(wide, xbits, M, N, K, splitK, groups, spans);
            if (wide_replaces(wide, t, groups ? 1.06f * here : here, M, N, K, splitK)) return true; // (the table's rows are row scales only; group exponents cost those kernels 3-10 %)
            LaunchCfg ungrouped = wide;
            int       split;
            return here <= 0.f && t > 0.f &&
                   wide_replaces(ungrouped, groups ? wide_best(ungrouped, xbits, M, N, K, splitK, false, spans) : t, best_narrow(split, a, M, N, SIZE_MAX), M, N, K, splitK);
        };
        // (wide_replaces asks more of gemm_span's small tiles than of most others.  Where gemm_wide's fastest passes, a span tile that is faster still is launched, too.)
        if (replaces(Spans::kAll)) return wide;
        if (replaces(Spans::kNone)) return wide_best(wide, xbits, M, N, K, splitK, groups, Spans::kAll), wide;
    }
    return pick_cfg(xbits, M, N, K, splitK, cus);
}

int linear_native(const fp6mi::FormatOps &ops, hipStream_t st, const void *W, const void *sc, const void *gexp, const void *bias, const void *B, void *C, size_t M, size_t N, size_t K, float *ws,
                  int splitK, const LaunchCfg *forced)
{
    LaunchCfg c = forced ? *forced : final_cfg(ops.bits, M, N, K, splitK, gexp != nullptr, current_device_cus());
    if (c.kind == 0 && !(c.rt & (c.rt - 1)) && (M / 16) % c.rt) return FP6MI_ERR_SHAPE; // (3, 5, 6, 7 tiles per workgroup end in a workgroup with fewer)
    int rc = ops.gemm(c, st, W, sc, gexp, B, C, splitK > 1 ? ws : static_cast<float *>(const_cast<void *>(bias)), M, N, K, splitK); // (a workspace given without a split is no bias)
    if (rc != 0) return rc;
    if (splitK > 1) {
        size_t MN = M * N; // M % 256 == 0, so MN % 4 == 0
        const size_t tile_rows = (size_t)c.wr * c.rt * 16, nblocks = (N + (size_t)c.nt * 16 - 1) / ((size_t)c.nt * 16);
        const size_t grid = c.kind >= 1 && M % tile_rows == 0 ? M / tile_rows * nblocks * splitK : 0; // gemm_tile and gemm_ws share the tile order
        if (grid && MN / 4 < ((size_t)1 << 31)) {
            // gemm_tile gave every XCD a run of consecutive triples: reduce where the partial sums lie
            const uint32_t q = (uint32_t)(grid / 8), r = (uint32_t)(grid % 8), per_block = (uint32_t)(nblocks * splitK);
            size_t         most = 0;
            for (uint32_t x = 0; x < 8; x++) {
                const size_t s0 = (size_t)x * q + (x < r ? x : r), s1 = (size_t)(x + 1) * q + (x + 1 < r ? x + 1 : r);
                const size_t rows = (s1 / per_block - s0 / per_block) * tile_rows;
                most = rows > most ? rows : most;
            }
            const size_t per_xcd = (most / 4 * N + 255) / 256;
            hipLaunchKernelGGL(bias ? splitk_reduce_by_xcd<true> : splitk_reduce_by_xcd<false>, dim3((uint32_t)(per_xcd * 8)), dim3(256), 0, st, static_cast<half_t *>(C), ws, (uint32_t)M, (uint32_t)N,
                               splitK, (uint32_t)tile_rows, q, r, per_block, static_cast<const half_t *>(bias));
        } else {
            hipLaunchKernelGGL(bias ? splitk_reduce<true> : splitk_reduce<false>, dim3((uint32_t)((MN / 4 + 255) / 256)), dim3(256), 0, st, static_cast<half_t *>(C), ws, MN, splitK, static_cast<const half_t *>(bias), (uint32_t)M);
        }
        rc = (int)hipGetLastError();
    }
    return rc;
}

} // namespace

// ------------------------------------------------------------------------------------------------ C ABI

extern "C" {

const char *fp6mi_error_string(int code)
{
    switch (code) {
    case FP6MI_OK: return "success";
    case FP6MI_ERR_FORMAT: return "unsupported (E,M): only FP6_e3m2 (3,2), FP5_e2m2 (2,2), FP6_e2m3 (2,3) and FP4_e2m1 (2,1)";
    case FP6MI_ERR_SHAPE: return "unsupported shape: need M % 256 == 0 (64 for CPU packers, 16 for native packers), K % 64 == 0, N >= 1, distinct in/out";
    case FP6MI_ERR_NULL: return "a required pointer is NULL";
    case FP6MI_ERR_WORKSPACE: return "splitK > 1 needs a workspace of splitK*M*N floats";
    case FP6MI_ERR_SPLITK: return "splitK must be >= 1";
    case FP6MI_ERR_ALIGN: return "weights, activations, output and workspace must be 16-byte aligned (scales, group exponents, bias: 2-byte)";
    case FP6MI_ERR_TOO_LARGE: return "splitK*M*N floats exceed the library's static workspace (fp6mi_static_workspace_bytes)";
    case FP6MI_ERR_CAPTURE: return "the stream is being captured and this call would have to allocate: convert the weights first (fp6mi_relayout_ref_to_native_gpu) or make the first call outside the capture";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown fp6mi error";
    }
}

const char *fp6mi_tuning_info(void)
{
    return
#include "fp6mi_tuning_info.inc"
        ;
}

int fp6mi_version(void) { return 142; } // 142: where gemm_span, little K and the stream kernel in pieces are taken, the dequantizer's stores; 141: gemm_span (odd column tiles of the wide kernel), little K on the stream kernel, splits of small batches off the table, dequantizer and quantizer kernels; 140: where gemm_wide is taken and with which splits, instances of gemm_tile for a bias, the quantizer chooses its arithmetic before a block; 139: a bias in the epilogues of the GEMM kernels, the quantizer's arithmetic; 138: gemm_wide (launch kind 2 with four rows of one or two wavefronts) in the place of larger tiles from 97 columns on, the other kernels unchanged; 137: group exponents of 128 rows through LDS in the wave-specialized kernel, panels of 256-row tiles only for activations beyond L2; 136: tiles of 48, 80 and 96 columns, deeper rings in the wave-specialized kernel of 128 rows, panels; 135: prefill kernel (launch kind 2 with 2 x 2 wavefronts), relayout and quantizer kernels rewritten, the other GEMM kernels unchanged; 134: three row tiles per workgroup in the small-batch kernel (any M: the last workgroup takes what is left), no other kernel changed; 133: wave-specialized tile kernel (launch kind 2) for large batches; 132: split-K reduction runs on the XCD that wrote the partial sums, every grid size gets XCD-contiguous tiles; 131: tile kernel stores through LDS; 130: small-batch kernel loads activations as whole rows and turns them into operand order through LDS

int fp6mi_prepack_ref(int E, int Mb, void *packed, const void *raw, size_t M, size_t K) { return fp6mi::prepack_ref(E, Mb, packed, raw, M, K); }
int fp6mi_unpack_ref(int E, int Mb, void *raw, const void *packed, size_t M, size_t K) { return fp6mi::unpack_ref(E, Mb, raw, packed, M, K); }
int fp6mi_dequant(int E, int Mb, void *out, const void *raw, size_t M, size_t K, const void *sc) { return fp6mi::dequant(E, Mb, out, raw, M, K, sc); }
size_t fp6mi_native_bytes(int E, int Mb, size_t M, size_t K) { return fp6mi::native_bytes(E, Mb, M, K); }
int fp6mi_prepack_native(int E, int Mb, void *native, const void *raw, size_t M, size_t K) { return fp6mi::prepack_native(E, Mb, native, raw, M, K); }
int fp6mi_unpack_native(int E, int Mb, void *raw, const void *native, size_t M, size_t K) { return fp6mi::unpack_native(E, Mb, raw, native, M, K); }
int fp6mi_relayout_ref_to_native(int E, int Mb, void *native, const void *ref, size_t M, size_t K)
{
    return fp6mi::relayout_ref_to_native(E, Mb, native, ref, M, K);
}

size_t fp6mi_group_exps_bytes(size_t M, size_t K) { return fp6mi::group_exps_bytes(M, K); }
int fp6mi_pack_group_exps(void *native_exps, const void *exps, size_t M, size_t K) { return fp6mi::pack_group_exps(native_exps, exps, M, K); }
int fp6mi_dequant_grouped(int E, int Mb, void *out, const void *raw, size_t M, size_t K, const void *sc, const void *exps)
{
    return fp6mi::dequant_grouped(E, Mb, out, raw, M, K, sc, exps);
}

size_t fp6mi_workspace_bytes(size_t M, size_t N, int splitK) { return splitK > 1 ? (size_t)splitK * M * N * sizeof(float) : 0; }

// Split-K choice.  Batches up to 16 (stream kernel): a cost model in microseconds on a part with `num_cus` compute
// units -- workgroups run in rounds of one per CU, a workgroup streams its weights at what one CU sustains, the whole
// chip cannot beat HBM, and a split costs a second launch plus writing and re-reading the FP32 partial sums; K is
// already split inside the workgroup, so a split rarely pays.  Larger batches (tile kernel): as much of the wanted K
// parallelism as keeps the FP32 partial-sum traffic (8 bytes per output per split) under half of the weight bytes.
//
// ws_bytes: what a split chosen for gemm_wide may take.  Its model asked for up to 370 MB where the table's splits take up to 99 (M up to 28672), and for more than
// the static workspace on 3.3 % of sizes of 98 to 4096 columns where it had taken them before.  On 60 of those, time / time before gemm_wide: 0.83 with any workspace, 0.84 held to 32 MiB.
constexpr size_t kStaticWsFloats = (size_t)8 << 20; // the static workspace: 32 MiB per GPU, held from the first use of the library on that GPU until the process ends

static int heuristic_splitk(int xbits, size_t M, size_t N, size_t K, int num_cus, size_t ws_bytes);

int fp6mi_heuristic_splitk(size_t M, size_t N, size_t K, int num_cus) { return heuristic_splitk(6, M, N, K, num_cus, kStaticWsFloats * sizeof(float)); }

int fp6mi_heuristic_splitk_format(int E, int Mb, size_t M, size_t N, size_t K, int num_cus)
{
    return fp6mi_heuristic_splitk_within(E, Mb, M, N, K, num_cus, kStaticWsFloats * sizeof(float));
}

int fp6mi_heuristic_splitk_within(int E, int Mb, size_t M, size_t N, size_t K, int num_cus, size_t ws_bytes)
{
    return heuristic_splitk(fp6mi::supported(E, Mb) ? 1 + E + Mb : 6, M, N, K, num_cus, ws_bytes);
}

static int heuristic_splitk(int xbits, size_t M, size_t N, size_t K, int num_cus, size_t ws_bytes)
{
    if (M == 0 || N == 0 || K == 0 || num_cus <= 0) return 1;
    size_t units = (K + 255) / 256;
    if (num_cus == 256) { // the fastest split by the times of measured neighbours, or of gemm_wide where it takes their place (3 % hysteresis towards fewer splits)
        int         best_s;
        const float best_t = best_narrow(best_s, tune_lookup(xbits, M, N, K), M, N, ws_bytes);
        auto wide_split = [&](Spans spans, float &t, LaunchCfg &wide) {
            int split = 0;
            for (int s : kSplits) {
                LaunchCfg c;
                if (fp6mi_workspace_bytes(M, N, s) > ws_bytes) break;
                if (const float ts = wide_best(c, xbits, M, N, K, s, false, spans); ts > 0.f && (split == 0 || ts * 1.03f < t)) split = s, t = ts, wide = c;
            }
            return split;
        };
        for (Spans spans : { Spans::kForSplit, Spans::kNone }) { // (as in final_cfg, which launches gemm_wide or gemm_span then)
            float     t = 0.f;
            LaunchCfg wide = {};
            if (const int split = wide_split(spans, t, wide); wide_replaces(wide, t, best_t, M, N, K, split)) return split;
        }
        if (best_s) return best_s;
    }
    if (N > 16) {
        int    best_s = 1;
        double best_ns = 1e30;
        if (K <= kLittleK) return 1;
        for (int sp = 1; sp <= 8 && (size_t)sp <= units; sp *= 2) {
            if (sp > 1 && (double)sp * 8.0 * (double)N > 0.75 * (double)K) break; // partial sums would outweigh the weights
            double ns = tile_estimate_ns(M, N, K, sp, num_cus, nullptr);
            if (ns < best_ns * 0.97) { best_ns = ns; best_s = sp; }
        }
        return best_s;
    }
    const double cu_gbps = 60.0, hbm_gbps = 6000.0, launch_us = 3.0;
    const double block_bytes = (double)fp6mi::native_block_bytes(xbits); // one 16-row x 256-column block of the format
    size_t       wgs = M / 16 ? M / 16 : 1;
    double       best = 1e30;
    int          best_s = 1;
    for (int s = 1; s <= 64 && (size_t)s <= units; s++) {
        double per_wg_bytes = (double)((units + s - 1) / s) * block_bytes;
        double rounds = std::ceil((double)(wgs * (size_t)s) / (double)num_cus);
        double t_cu = rounds * per_wg_bytes / (cu_gbps * 1e3);
        double t_hbm = (double)wgs * (double)units * block_bytes / (hbm_gbps * 1e3);
        double t = launch_us + (t_cu > t_hbm ? t_cu : t_hbm);
        if (s > 1) t += launch_us + 2.0 * (double)s * (double)M * (double)N * 4.0 / (hbm_gbps * 1e3);
        if (t < best * 0.97) { best = t; best_s = s; }
    }
    return best_s;
}

static int check_gemm_args(int E, int Mb, const void *W, const void *sc, const void *B, const void *C, size_t M, size_t N, size_t K,
                           const float *ws, int splitK)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!W || !sc || !B || !C) return FP6MI_ERR_NULL;
    if (M == 0 || M % 256 || K == 0 || K % 64 || N == 0) return FP6MI_ERR_SHAPE;
    if (M > 0x7fffffffu || N > 0x7fffffffu || K > 0x7fffffffu || (N + 15) / 16 > 65535) return FP6MI_ERR_SHAPE;
    if (splitK < 1 || splitK > 65535) return FP6MI_ERR_SPLITK;
    if (splitK > 1 && !ws) return FP6MI_ERR_WORKSPACE;
    if (!aligned16(W) || !aligned16(B) || !aligned16(C) || (ws && !aligned16(ws))) return FP6MI_ERR_ALIGN;
    if (reinterpret_cast<uintptr_t>(sc) & 1u) return FP6MI_ERR_ALIGN; // halfs; the tile kernel uses 8-byte loads where the pointer allows them
    return FP6MI_OK;
}

int fp6mi_linear_native(int E, int Mb, void *stream, const void *W, const void *sc, const void *B, void *C, size_t M, size_t N, size_t K,
                        float *ws, int splitK)
{
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return linear_native(*fp6mi::ops_for(E, Mb), st, W, sc, nullptr, nullptr, B, C, M, N, K, ws, splitK, nullptr);
}

int fp6mi_linear_native_grouped(int E, int Mb, void *stream, const void *W, const void *sc, const void *group_exps, const void *B, void *C, size_t M,
                                size_t N, size_t K, float *ws, int splitK)
{
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    if (!group_exps) return FP6MI_ERR_NULL;
    if (reinterpret_cast<uintptr_t>(group_exps) & 1u) return FP6MI_ERR_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return linear_native(*fp6mi::ops_for(E, Mb), st, W, sc, group_exps, nullptr, B, C, M, N, K, ws, splitK, nullptr);
}

int fp6mi_linear_native_bias(int E, int Mb, void *stream, const void *W, const void *sc, const void *group_exps, const void *bias, const void *B, void *C, size_t M,
                             size_t N, size_t K, float *ws, int splitK)
{
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    if (!bias) return FP6MI_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(group_exps) & 1u) || (reinterpret_cast<uintptr_t>(bias) & 1u)) return FP6MI_ERR_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return linear_native(*fp6mi::ops_for(E, Mb), st, W, sc, group_exps, bias, B, C, M, N, K, ws, splitK, nullptr);
}

int fp6mi_linear_native_cfg(int E, int Mb, void *stream, const void *W, const void *sc, const void *B, void *C, size_t M, size_t N, size_t K,
                            float *ws, int splitK, int kind, int n_tiles, int row_tiles, int row_waves, int k_waves)
{
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    LaunchCfg   c = { kind, n_tiles, row_tiles, row_waves, k_waves };
    hipStream_t st = static_cast<hipStream_t>(stream);
    return linear_native(*fp6mi::ops_for(E, Mb), st, W, sc, nullptr, nullptr, B, C, M, N, K, ws, splitK, &c);
}

int fp6mi_linear_native_grouped_cfg(int E, int Mb, void *stream, const void *W, const void *sc, const void *group_exps, const void *B, void *C, size_t M,
                                    size_t N, size_t K, float *ws, int splitK, int kind, int n_tiles, int row_tiles, int row_waves, int k_waves)
{
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    if (!group_exps) return FP6MI_ERR_NULL;
    if (reinterpret_cast<uintptr_t>(group_exps) & 1u) return FP6MI_ERR_ALIGN;
    LaunchCfg   c = { kind, n_tiles, row_tiles, row_waves, k_waves };
    hipStream_t st = static_cast<hipStream_t>(stream);
    return linear_native(*fp6mi::ops_for(E, Mb), st, W, sc, group_exps, nullptr, B, C, M, N, K, ws, splitK, &c);
}

static int query_args(int E, int Mb, size_t M, size_t N, size_t K, int splitK)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (M == 0 || M % 256 || K == 0 || K % 64 || N == 0) return FP6MI_ERR_SHAPE;
    return splitK < 1 ? FP6MI_ERR_SPLITK : FP6MI_OK;
}
static void write_shape(int *shape, const LaunchCfg &c) { shape[0] = c.kind, shape[1] = c.nt, shape[2] = c.rt, shape[3] = c.wr, shape[4] = c.wk; }

int fp6mi_query_table(int E, int Mb, size_t M, size_t N, size_t K, int splitK, int *shape)
{
    if (int rc = query_args(E, Mb, M, N, K, splitK); rc != FP6MI_OK) return rc;
    if (shape) write_shape(shape, pick_cfg(1 + E + Mb, M, N, K, splitK, current_device_cus())); // the count the launch path uses (256 where no device answers)
    const int i = split_index(splitK);
    if (i >= 0)
        if (const TuneAnswer *a = tune_lookup(1 + E + Mb, M, N, K))
            if (a->t[i] > 0.f) return prefill_replaces(*a, i, M, N, K) ? 2 : a->measured ? 0 : 1;
    return 2;
}

int fp6mi_query_kernel(int E, int Mb, size_t M, size_t N, size_t K, int splitK, int grouped, int *shape)
{
    if (int rc = query_args(E, Mb, M, N, K, splitK); rc != FP6MI_OK) return rc;
    if (!shape) return FP6MI_ERR_NULL;
    write_shape(shape, final_cfg(1 + E + Mb, M, N, K, splitK, grouped != 0, current_device_cus()));
    return FP6MI_OK;
}

int fp6mi_query_launch(int E, int Mb, size_t M, size_t N, size_t K, int splitK, int *shape) { return fp6mi_query_kernel(E, Mb, M, N, K, splitK, 0, shape); }

int fp6mi_launch_source(int E, int Mb, size_t M, size_t N, size_t K, int splitK)
{
    int        shape[5];
    const int  rc = fp6mi_query_launch(E, Mb, M, N, K, splitK, shape);
    const bool wide = rc == FP6MI_OK && shape[0] == 2 && shape[3] == 4 && shape[4] <= 2; // gemm_wide
    return rc != FP6MI_OK ? rc : wide ? 2 : fp6mi_query_table(E, Mb, M, N, K, splitK, nullptr);
}

// ---- allocation-free variant of fp6mi_linear_native: the split-K workspace is a static device array of the library ----
namespace {
__device__ __align__(256) float g_static_ws[kStaticWsFloats];

// Device address of g_static_ws on the current device (every GPU holds its own copy of the array at its own address); asked
// of the runtime once per device.  The array's name is only a host-side handle: kernels get this pointer as an argument.
int static_ws_ptr(float **out)
{
    static std::mutex mu;
    static float     *ptrs[64];
    int               dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= 64) return FP6MI_ERR_SHAPE;
    std::lock_guard<std::mutex> lock(mu);
    if (!ptrs[dev]) {
        void *p = nullptr;
        if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_static_ws)); e != hipSuccess) return (int)e;
        ptrs[dev] = static_cast<float *>(p);
    }
    *out = ptrs[dev];
    return FP6MI_OK;
}
} // namespace

size_t fp6mi_static_workspace_bytes(void) { return kStaticWsFloats * sizeof(float); }

int fp6mi_init(void)
{
    float *p = nullptr;
    (void)current_device_cus();
    return static_ws_ptr(&p);
}

int fp6mi_linear_native_static(int E, int Mb, void *stream, const void *W, const void *sc, const void *B, void *C, size_t M, size_t N, size_t K,
                               int splitK)
{
    float *ws = nullptr;
    if (splitK > 1) {
        // checked before the multiplication can overflow: M, N <= 2^31 and splitK <= 65535 are enforced by check_gemm_args below
        if (M > 0x7fffffffu || N > 0x7fffffffu || splitK > 65535) return FP6MI_ERR_SHAPE;
        if ((size_t)splitK * M > kStaticWsFloats || (size_t)splitK * M * N > kStaticWsFloats) return FP6MI_ERR_TOO_LARGE;
        if (int rc = static_ws_ptr(&ws); rc != FP6MI_OK) return rc;
    }
    int rc = check_gemm_args(E, Mb, W, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    return linear_native(*fp6mi::ops_for(E, Mb), static_cast<hipStream_t>(stream), W, sc, nullptr, nullptr, B, C, M, N, K, ws, splitK, nullptr);
}

// ---- drop-in entry on REFERENCE-layout weights: native twins are made on first sight of a weight pointer and kept ----
namespace {
struct Twin { void *native; int E, Mb; size_t M, K; int device; };
std::mutex                              g_twin_mutex;
std::unordered_map<const void *, Twin>  g_twins;
} // namespace

int fp6mi_linear(int E, int Mb, void *stream, const void *W_ref, const void *sc, const void *B, void *C, size_t M, size_t N, size_t K,
                 float *ws, int splitK)
{
    int rc = check_gemm_args(E, Mb, W_ref, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    int device = 0;
    if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return (int)e;
    void *native = nullptr, *stale = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_twin_mutex);
        auto it = g_twins.find(W_ref);
        if (it != g_twins.end()) {
            const Twin &t = it->second;
            if (t.E == E && t.Mb == Mb && t.M == M && t.K == K && t.device == device) {
                native = t.native;
            } else { // the address now holds a different matrix
                stale = t.native;
                g_twins.erase(it);
            }
        }
    }
    // Everything slow happens outside the lock (allocation, the relayout kernel, the wait for it, freeing a stale twin), so
    // that other threads' calls, cache hits on other weights above all, never queue behind one caller's stream.
    if (stale) (void)hipFree(stale);
    if (!native) {
        // A twin has to be allocated and filled: not possible while the stream is being captured (the allocation would end
        // the capture with an error, and a replay would not repeat it).
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipError_t e = hipStreamIsCapturing(static_cast<hipStream_t>(stream), &cap); e != hipSuccess) return (int)e;
        if (cap != hipStreamCaptureStatusNone) return FP6MI_ERR_CAPTURE;
        size_t bytes = fp6mi::native_bytes(E, Mb, M, K);
        if (hipError_t e = hipMalloc(&native, bytes); e != hipSuccess) return (int)e;
        rc = fp6mi_relayout_ref_to_native_gpu(E, Mb, stream, native, W_ref, M, K);
        // The twin becomes visible to other callers (and other streams) only once it is completely written: this
        // one-time path waits for the relayout kernel before it publishes the pointer.
        if (rc == 0) rc = (int)hipStreamSynchronize(static_cast<hipStream_t>(stream));
        if (rc != 0) {
            (void)hipFree(native);
            return rc;
        }
        void *duplicate = nullptr;
        {
            std::lock_guard<std::mutex> lock(g_twin_mutex);
            auto ins = g_twins.emplace(W_ref, Twin{ native, E, Mb, M, K, device });
            if (!ins.second) { // another thread converted the same weights meanwhile
                const Twin &t = ins.first->second;
                if (t.E == E && t.Mb == Mb && t.M == M && t.K == K && t.device == device) {
                    duplicate = native;   // keep theirs, which may already be in use
                    native = t.native;
                } else {                  // theirs describes another matrix at this address: ours is the newer truth
                    duplicate = t.native;
                    ins.first->second = Twin{ native, E, Mb, M, K, device };
                }
            }
        }
        if (duplicate) (void)hipFree(duplicate);
    }
    return fp6mi_linear_native(E, Mb, stream, native, sc, B, C, M, N, K, ws, splitK);
}

int fp6mi_linear_stateless(int E, int Mb, void *stream, const void *W_ref, const void *sc, const void *B, void *C, size_t M, size_t N, size_t K,
                           float *ws, int splitK, void *native_scratch)
{
    if (!native_scratch) return FP6MI_ERR_NULL;
    if (!aligned16(native_scratch) || native_scratch == W_ref) return native_scratch == W_ref ? FP6MI_ERR_SHAPE : FP6MI_ERR_ALIGN;
    int rc = check_gemm_args(E, Mb, W_ref, sc, B, C, M, N, K, ws, splitK);
    if (rc != FP6MI_OK) return rc;
    rc = fp6mi_relayout_ref_to_native_gpu(E, Mb, stream, native_scratch, W_ref, M, K);
    if (rc != FP6MI_OK) return rc;
    return fp6mi_linear_native(E, Mb, stream, native_scratch, sc, B, C, M, N, K, ws, splitK);
}

int fp6mi_twin_evict(const void *W_ref)
{
    std::lock_guard<std::mutex> lock(g_twin_mutex);
    auto it = g_twins.find(W_ref);
    if (it == g_twins.end()) return FP6MI_OK;
    hipError_t e = hipFree(it->second.native); // hipFree waits for work that may still read the buffer
    g_twins.erase(it);
    return (int)e;
}

int fp6mi_twin_clear(void)
{
    std::lock_guard<std::mutex> lock(g_twin_mutex);
    int rc = 0;
    for (auto &kv : g_twins) {
        hipError_t e = hipFree(kv.second.native);
        if (e != hipSuccess) rc = (int)e;
    }
    g_twins.clear();
    return rc;
}

int fp6mi_relayout_ref_to_native_gpu(int E, int Mb, void *stream, void *native, const void *ref, size_t M, size_t K)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!native || !ref) return FP6MI_ERR_NULL;
    if (M == 0 || M % 64 || K == 0 || K % 64 || M > 0x7fffffffu || K > 0x7fffffffu || native == ref) return FP6MI_ERR_SHAPE;
    if (!aligned16(native) || !aligned16(ref)) return FP6MI_ERR_ALIGN;
    return fp6mi::ops_for(E, Mb)->relayout(stream, native, ref, M, K);
}

int fp6mi_dequant_native_gpu(int E, int Mb, void *stream, void *out, const void *W, const void *sc, size_t M, size_t K)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!out || !W || !sc) return FP6MI_ERR_NULL;
    if (M == 0 || M % 16 || K == 0 || K % 64 || M > 0x7fffffffu || K > 0x7fffffffu) return FP6MI_ERR_SHAPE;
    if (!aligned16(out) || !aligned16(W)) return FP6MI_ERR_ALIGN;
    return fp6mi::ops_for(E, Mb)->dequant(stream, out, W, sc, nullptr, M, K);
}

int fp6mi_dequant_native_grouped_gpu(int E, int Mb, void *stream, void *out, const void *W, const void *sc, const void *group_exps, size_t M, size_t K)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!out || !W || !sc || !group_exps) return FP6MI_ERR_NULL;
    if (M == 0 || M % 16 || K == 0 || K % 64 || M > 0x7fffffffu || K > 0x7fffffffu) return FP6MI_ERR_SHAPE;
    if (!aligned16(out) || !aligned16(W) || (reinterpret_cast<uintptr_t>(group_exps) & 1u)) return FP6MI_ERR_ALIGN;
    return fp6mi::ops_for(E, Mb)->dequant(stream, out, W, sc, group_exps, M, K);
}

int fp6mi_quantize_native_gpu(int E, int Mb, void *stream, void *native, void *scales, const void *weights, int dtype, size_t M, size_t K)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!native || !scales || !weights) return FP6MI_ERR_NULL;
    if (dtype < 0 || dtype > 2) return FP6MI_ERR_FORMAT;
    if (M == 0 || M % 16 || K == 0 || K % 64 || M > 0x7fffffffu || K > 0x7fffffffu) return FP6MI_ERR_SHAPE;
    if (!aligned16(native) || !aligned16(weights)) return FP6MI_ERR_ALIGN;
    return fp6mi::ops_for(E, Mb)->quantize(stream, native, scales, nullptr, weights, dtype, M, K);
}

int fp6mi_quantize_native_grouped_gpu(int E, int Mb, void *stream, void *native, void *scales, void *group_exps, const void *weights, int dtype,
                                      size_t M, size_t K)
{
    if (!fp6mi::supported(E, Mb)) return FP6MI_ERR_FORMAT;
    if (!native || !scales || !weights || !group_exps) return FP6MI_ERR_NULL;
    if (dtype < 0 || dtype > 2) return FP6MI_ERR_FORMAT;
    if (M == 0 || M % 16 || K == 0 || K % 64 || M > 0x7fffffffu || K > 0x7fffffffu) return FP6MI_ERR_SHAPE;
    if (!aligned16(native) || !aligned16(weights)) return FP6MI_ERR_ALIGN;
    return fp6mi::ops_for(E, Mb)->quantize(stream, native, scales, group_exps, weights, dtype, M, K);
}

} // extern "C"
