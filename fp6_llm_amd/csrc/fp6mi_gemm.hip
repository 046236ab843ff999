// gfx950 (MI355X) kernels of the FPx x FP16 linear layer and their launchers, for ONE weight format per translation unit:
// the build compiles this file once per format with -DFP6MI_FORMAT=<10*E+M> (32, 22, 23, 21), in parallel, and each object
// exports one table of entry functions (fp6mi::FormatOps) that the C ABI in fp6mi_api.hip dispatches to.
//
// Roles taken over from the reference (usyd-fsalab/fp6_llm, paths relative to it):
//   gemm_stream, gemm_tile, gemm_ws, gemm_prefill, gemm_wide, gemm_span <- QUANT_GEMM_Kernel   fp6_llm/csrc/include/kernel_matmul.cuh:29-191
//                    (small batches / batches above 16 / large batches, the last four: five organisations of the same GEMM)
//   splitk_reduce <- SplitK_Reduction         fp6_llm/csrc/include/kernel_reduction.cuh:28-47   (in fp6mi_api.hip)
//   launchers     <- fpx_linear_kernel        fp6_llm/csrc/fp6_linear.cu:44-102
// The design is not a translation: weights use the native layout described in fp6mi_host.cpp, go from HBM straight
// to VGPRs with 128-bit non-temporal loads, FP6 codes are converted by the CDNA4 instruction
// v_cvt_scalef32_pk32_f16_bf6 (BF6 = e3m2, bias 3, no inf/nan: the very format of the reference), FP5 codes by the same
// instruction after a zero bit is slipped in above their exponent (an e2m2 code read as e3m2 is a quarter of its value),
// FP6_e2m3 codes by v_cvt_scalef32_pk32_f16_fp6 and FP4_e2m1 codes by that instruction after two zero bits are appended
// to their mantissa, and v_mfma_f32_16x16x32_f16 accumulates in FP32.  The per-row scale (and the factor 4 of FP5) is
// applied once to the FP32 sums instead of to every weight.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "fp6mi_internal.h"

#ifndef FP6MI_FORMAT
#error "compile with -DFP6MI_FORMAT=32, 22, 23 or 21 (10*E + M of the weight format)"
#endif

namespace {

using fp6mi::LaunchCfg;

typedef _Float16 half_t;
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v32h __attribute__((ext_vector_type(32)));
typedef float    v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v6u __attribute__((ext_vector_type(6)));

constexpr int kWave = 64;

// Formats are named by the tag FM = 10*E + M.  `hw_e3m2` says which conversion instruction reads the 6-bit fields that the
// native layout holds (BF6 = e3m2 or FP6 = e2m3); post_scale is the factor the epilogue owes the sums.
template <int FM> struct Fmt;
template <> struct Fmt<32> { static constexpr int bits = 6, man = 2, bias = 3, block_bytes = 3072; static constexpr bool hw_e3m2 = true;
                             static constexpr float post_scale = 1.0f; static constexpr double max_value = 28.0; };
template <> struct Fmt<22> { static constexpr int bits = 5, man = 2, bias = 1, block_bytes = 2560; static constexpr bool hw_e3m2 = true;
                             static constexpr float post_scale = 4.0f; static constexpr double max_value = 7.0; };
template <> struct Fmt<23> { static constexpr int bits = 6, man = 3, bias = 1, block_bytes = 3072; static constexpr bool hw_e3m2 = false;
                             static constexpr float post_scale = 1.0f; static constexpr double max_value = 7.5; };
template <> struct Fmt<21> { static constexpr int bits = 4, man = 1, bias = 1, block_bytes = 2048; static constexpr bool hw_e3m2 = false;
                             static constexpr float post_scale = 1.0f; static constexpr double max_value = 6.0; };

// The weights of one lane for one 16x256 block, as loaded from memory.
template <int FM> struct WFrag;
template <> struct WFrag<32> { v4u a, b, c; };
template <> struct WFrag<23> { v4u a, b, c; };
template <> struct WFrag<22> { v4u a, b; v2u s; };
template <> struct WFrag<21> { v4u a, b; };

template <int FM> __device__ __forceinline__ WFrag<FM> load_wfrag(const uint8_t *block, int lane)
{
    const v4u *p = reinterpret_cast<const v4u *>(block) + lane;
    WFrag<FM>  f;
    f.a = __builtin_nontemporal_load(p);
    f.b = __builtin_nontemporal_load(p + 64);
    if constexpr (Fmt<FM>::bits == 6) f.c = __builtin_nontemporal_load(p + 128);
    if constexpr (Fmt<FM>::bits == 5) f.s = __builtin_nontemporal_load(reinterpret_cast<const v2u *>(block + 2048) + lane);
    return f;
}

// One of the two or three loads of load_wfrag, for a kernel that spreads them over its compute.
template <int FM> __device__ __forceinline__ void load_wfrag_part(WFrag<FM> &f, const uint8_t *block, int lane, int part)
{
    const v4u *p = reinterpret_cast<const v4u *>(block) + lane;
    if (part == 0) f.a = __builtin_nontemporal_load(p);
    if (part == 1) f.b = __builtin_nontemporal_load(p + 64);
    if constexpr (Fmt<FM>::bits == 6) { if (part == 2) f.c = __builtin_nontemporal_load(p + 128); }
    if constexpr (Fmt<FM>::bits == 5) { if (part == 2) f.s = __builtin_nontemporal_load(reinterpret_cast<const v2u *>(block + 2048) + lane); }
}

// A operands (8 halfs = k 8q..8q+7 of this lane's row) of the eight MFMA steps of a block.
// FP5: a quarter of the values (exact; the epilogue multiplies the sums by 4).  The other formats: exact values.
template <int FM> struct AOps { v8h s[8]; };

__device__ __forceinline__ v8h slice8(const v32h &v, int i)
{
    switch (i) {
    case 0: return __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, 6, 7);
    case 1: return __builtin_shufflevector(v, v, 8, 9, 10, 11, 12, 13, 14, 15);
    case 2: return __builtin_shufflevector(v, v, 16, 17, 18, 19, 20, 21, 22, 23);
    default: return __builtin_shufflevector(v, v, 24, 25, 26, 27, 28, 29, 30, 31);
    }
}

// FP5: 32 codes are stored in five dwords; the sixth dword of the 6-bit string the conversion instruction reads is parked
// in the fixed-zero bits ("holes", bit 4 of every 6-bit field) of the other five and is put back here (layout: fp6mi_host.cpp).
__device__ __forceinline__ v6u fp5_expand(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3, uint32_t s4)
{
    constexpr uint32_t A = 0x10410410u, B = 0x04104104u, C = 0x41041041u;
    uint32_t lo = (s0 & A) | (s1 & B), hi = (s2 & C) | (s3 & A) | (s4 & B);
    return (v6u){ s0 & ~A, s1 & ~B, s2 & ~C, s3 & ~A, s4 & ~B, (hi << 1) | lo };
}

// FP4: 32 codes are stored in four dwords; the fifth and sixth dword of the 6-bit string sit in the fixed-zero bit pairs (the
// two bits appended below every mantissa) of the other four, at their own bit positions (layout: fp6mi_host.cpp).
__device__ __forceinline__ v6u fp4_expand(v4u s)
{
    constexpr uint32_t P = 0xC30C30C3u, Q = 0x30C30C30u, R = 0x0C30C30Cu;
    return (v6u){ s[0] & ~P, s[1] & ~Q, s[2] & ~R, s[3] & ~P, (s[0] & P) | (s[2] & R), (s[1] & Q) | (s[3] & P) };
}

// The 192-bit string of 6-bit fields of MFMA steps 4h..4h+3 (half of a K block) of one lane, and its conversion.
template <int FM> __device__ __forceinline__ v6u field_string(const WFrag<FM> &f, int h)
{
    if constexpr (Fmt<FM>::bits == 6)
        return h == 0 ? (v6u){ f.a[0], f.a[1], f.a[2], f.a[3], f.b[0], f.b[1] } : (v6u){ f.b[2], f.b[3], f.c[0], f.c[1], f.c[2], f.c[3] };
    else if constexpr (Fmt<FM>::bits == 5)
        return h == 0 ? fp5_expand(f.a[0], f.a[1], f.a[2], f.a[3], f.s[0]) : fp5_expand(f.b[0], f.b[1], f.b[2], f.b[3], f.s[1]);
    else
        return fp4_expand(h == 0 ? f.a : f.b);
}

// The conversion instruction multiplies its 32 values by the power of two in the exponent field of `scale` at no cost.
template <int FM> __device__ __forceinline__ v32h fields_to_halfs(v6u src, float scale)
{
    if constexpr (Fmt<FM>::hw_e3m2)
        return __builtin_amdgcn_cvt_scalef32_pk32_f16_bf6(src, scale);
    else
        return __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(src, scale);
}

// Group exponents: one byte b per (row, 128 columns), meaning the factor 2^(b-127) on those weights (the E8M0 scale type of
// the OCP MX formats).  A lane's 32-code string is exactly its row's share of one 128-column group, so the factor rides on
// the conversion instruction.  Native layout of the bytes: [row tile][K block][row in tile][half of the block], 32 bytes per
// block; `g` below is the lane's pair of bytes (half 0 in the low byte).  GS = false: no group exponents, factor 1.
template <bool GS> __device__ __forceinline__ float group_factor(uint32_t g, int h)
{
    if constexpr (GS)
        return __builtin_bit_cast(float, (h == 0 ? (g & 0xffu) : (g >> 8)) << 23);
    else
        return 1.0f;
}
// block = index of the 16x256 block counted from `gexp` (32 bytes each); nothing is computed or read without group exponents
template <bool GS> __device__ __forceinline__ uint32_t load_group_exps(const uint8_t *gexp, size_t block, int lane)
{
    if constexpr (GS)
        return *reinterpret_cast<const uint16_t *>(gexp + block * 32 + 2 * (lane & 15));
    else
        return 0;
}

template <int FM, bool GS> __device__ __forceinline__ void convert(const WFrag<FM> &f, AOps<FM> &o, uint32_t g)
{
    v32h h0 = fields_to_halfs<FM>(field_string<FM>(f, 0), group_factor<GS>(g, 0));
    v32h h1 = fields_to_halfs<FM>(field_string<FM>(f, 1), group_factor<GS>(g, 1));
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o.s[i]     = slice8(h0, i);
        o.s[4 + i] = slice8(h1, i);
    }
}

// `ws` of the GEMM kernels: the partial sums where K is split (splitk_reduce adds a bias then), else an fp16 bias [M] on any 2-byte boundary or null, which
// the epilogue adds to the float32 sums.  gemm_stream and gemm_tile have instances of their own for it: a branch in the epilogue that no launch took cost the one 0.04-0.1 us (1 % of
// 4096x4096 N 8), the other a register or two, in some instances spilled, and 0.2-0.5 % of calls of 5 us.  The kernels of larger tiles branch (gemm_ws +0.0-0.6 % on calls of
// 9-20 us, as much as two builds of the same instructions differ by).  Instead of an addition behind the GEMM, us, e3m2, replayed: 4096x4096 N 1 6.1 -> 4.4, N 8 7.6 -> 5.0; 8192x8192 N 16 15.7 -> 12.9,
// N 72 25.9 -> 22.1; 28672x8192 N 2048 680 -> 657.
template <typename P> __device__ __forceinline__ const half_t *bias_of(P ws) { return reinterpret_cast<const half_t *>(ws); }

// ---------------------------------------------------------------------------------------------------------------
// gemm_stream: weight-bandwidth-bound GEMM for small batches.
//   grid  = (M/(16*RT) row groups, splitK, ceil(N / (16*NT)))      block = WAVES wavefronts
// A workgroup owns 16*RT output rows and 16*NT batch columns over the K blocks of its split; its wavefronts take the
// blocks round-robin (K is split inside the workgroup), each streaming its weights HBM -> VGPR and its slice of the
// activations L2 -> VGPR -> LDS -> VGPR (reused for the RT row tiles); the partial accumulators are summed through LDS.
//
// Why the activations take the detour through LDS.  The MFMA wants lane (col, q) to hold 16 bytes of batch row `col`, so a
// load in operand order makes the 16 lanes of every quarter-wavefront touch 16 different 128-byte lines, 16 bytes of each.
// The vector memory pipeline looks up one line per cycle: measured on the MI355X with nothing else in the kernel, the
// operand-order loads of a 4096-wide K for batch 16 on all 256 CUs take 3.1 us, the same bytes loaded as whole rows
// (32 consecutive lanes = 512 consecutive bytes) 0.9 us; batch 8 with two MFMA steps per load 1.4 us against 0.25 us.
// So from batch 5 up every wavefront loads its slice as whole rows, writes it to an LDS area of its own (no barrier: nobody
// else reads it) and reads it back in operand order; LDS rows are padded to 544 bytes, the stride at which that read is
// conflict-free.  Batches of 5 to 8 stage 8 rows (B columns 8..15 re-read rows 0..7 and feed outputs that are never stored).
// Batches up to 4 keep operand-order loads: a quarter-wavefront then touches at most 4 lines, and the trip through LDS
// would only add latency (measured: 1-4 % slower there).
// ---------------------------------------------------------------------------------------------------------------
constexpr int kXsRowBytes = 544;

template <int FM, int RT> struct StageW {
    WFrag<FM> w[RT];
    uint32_t  g[RT]; // group exponents of the block (unused without them)
};

// LDS bytes per wavefront: the activation rows of one K block, or the RT*NT partial tiles of the epilogue (they share it)
__host__ __device__ constexpr uint32_t stream_wave_bytes(int rows, int RT, int NT)
{
    return (uint32_t)(rows * kXsRowBytes > RT * NT * 1024 ? rows * kXsRowBytes : RT * NT * 1024);
}

template <int FM, bool GS, int NT, int RT, int WAVES, bool SPLIT, bool BIAS>
__global__ __launch_bounds__(WAVES *kWave) void gemm_stream(const uint8_t *__restrict__ W, const half_t *__restrict__ scales,
                                                            const uint8_t *__restrict__ gexp, const half_t *__restrict__ X, half_t *__restrict__ C,
                                                            float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                            uint32_t units, uint32_t splitK)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    // every kernel argument is fetched by one batch of scalar loads at the top (left alone, the compiler fetches them in
    // three batches, each a round trip to memory, as the code reaches their first use)
    asm volatile("" ::"s"(W), "s"(scales), "s"(gexp), "s"(X), "s"(C), "s"(ws), "s"(M), "s"(N), "s"(K), "s"(units), "s"(splitK));
    // the wavefront's index as a scalar: the K-block loop, its bounds and its branches then run on the scalar unit
    const int      lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int      col = lane & 15, q = lane >> 4;
    const uint32_t R0 = blockIdx.x * RT, split = blockIdx.y, nbase = blockIdx.z * (16 * NT);

    // SPLIT = false is the launch with splitK == 1: its range is the whole of K and its epilogue writes fp16
    uint32_t u0 = 0, u1 = units;
    if constexpr (SPLIT) {
        const uint32_t avg = units / splitK, extra = units % splitK;
        u0 = split * avg + (split < extra ? split : extra);
        u1 = u0 + avg + (split < extra ? 1u : 0u);
    }

    const size_t   tile_stride = (size_t)units * Fmt<FM>::block_bytes;
    const uint8_t *wgroup = W + (size_t)R0 * tile_stride;
    const uint8_t *ggroup = GS ? gexp + (size_t)R0 * units * 32 : nullptr;
    // M is a multiple of 256, so 1, 2, 4 and 8 row tiles per workgroup divide its M/16 row tiles; 3, 5, 6 and 7 need not, and
    // the last workgroup then holds fewer.  Its missing tiles stand in as copies of its last real one (same loads, same arithmetic,
    // nothing stored): rlast is the largest r that names a real tile.
    constexpr bool kRagged = (RT & (RT - 1)) != 0;
    const uint32_t rlast = kRagged && R0 + RT > (M >> 4) ? (M >> 4) - 1 - R0 : RT - 1;
    auto           real = [&](int r) -> uint32_t { return kRagged && (uint32_t)r > rlast ? rlast : (uint32_t)r; };

    v4f acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = (v4f){ 0.f, 0.f, 0.f, 0.f };

    // The epilogue gives thread e the output (row tile e/(256*NT), column tile, batch column, row e%16); its row scale is
    // fetched now so that no global load sits on the tail of the kernel.
    constexpr int kOutPerThread = (RT * NT * 256 + WAVES * kWave - 1) / (WAVES * kWave);
    half_t        my_scale[kOutPerThread]; // kept as loaded: converting here would wait for the load before the weight loads issue
#pragma unroll
    for (int j = 0; j < kOutPerThread; j++) {
        int e = threadIdx.x + j * WAVES * kWave;
        my_scale[j] = scales[(R0 + real(e < RT * NT * 256 ? (e >> 8) / NT : 0)) * 16 + (e & 15)];
    }

    const uint32_t ncols = N - nbase;              // batch columns of this column block that exist (the launcher made sure of >= 1)
    const bool     small = NT == 1 && ncols <= 8;  // 8 rows are staged instead of 16
    const uint32_t wave_bytes = small ? stream_wave_bytes(8, RT, NT) : stream_wave_bytes(16 * NT, RT, NT);
    uint8_t       *mine = lds + wave * wave_bytes;  // this wavefront's LDS area

    // One K block at a time and no register double-buffering: the other wavefronts of the workgroup keep the memory system
    // busy while this one converts, and a second stage in registers measured slower at every size.
    // workgroups that share an L2 (ids congruent mod 8) start on different K blocks, so that the chip does not ask
    // the same activation lines of the same L2 channel at the same moment
    const uint32_t ufull = K / 256 < u1 ? K / 256 : u1; // the blocks before this one lie wholly inside K
    uint32_t       u = u0 + ((wave + (blockIdx.x >> 3)) % WAVES);
    // MODE 0: batches up to 4 load in operand order (a quarter-wavefront then touches at most 4 lines, and the detour through
    // LDS would only add latency); MODE 1: 8 rows through LDS; MODE 2: 16*NT rows through LDS.  TAIL: the block is cut by K
    // (only the last block of a K that is no multiple of 256).  The kernel chooses outside its K loop: a choice made per
    // block inside the loop cost 0.2 us of a 4.9 us launch.
    auto run = [&](auto mode_c, auto tail_c, uint32_t end) {
        constexpr int  MODE = decltype(mode_c)::value, ROWS = MODE == 2 ? 16 * NT : 8, LOADS = MODE == 0 ? 4 : ROWS / 2;
        constexpr bool TAIL = decltype(tail_c)::value;
        static_assert(!(MODE == 0 && (TAIL || NT != 1)), "operand-order loads serve whole blocks of one column tile");
        // MODE 0: lane (col, q) reads batch row col % 8 at MFMA step offset col / 8
        const uint32_t prow = (uint32_t)(col & 7) < ncols ? col & 7 : ncols - 1;
        const half_t  *xpaired = X + (size_t)(nbase + prow) * K + 8 * q + 32 * (col >> 3);
        // MODE 1, 2: load i of a block brings rows 2i and 2i+1, lane l takes bytes 16*(l%32).. of row 2i + l/32: a scalar base per
        // load plus one per-lane offset for the whole kernel.  Rows beyond the batch repeat its last row (an MFMA output column
        // depends only on its own B column, and those columns are never stored).
        const uint8_t *xbase = reinterpret_cast<const uint8_t *>(X + (size_t)nbase * K);
        const uint32_t off_one = (lane & 31) * 16, off_pair = (lane >> 5) * (K * 2) + off_one; // K < 2^31
        uint8_t       *xw = mine + (lane >> 5) * kXsRowBytes + (lane & 31) * 16;
        const uint8_t *xr = mine + (ROWS == 8 ? col & 7 : col) * kXsRowBytes + q * 16;
        constexpr int  kWParts = Fmt<FM>::bits == 4 ? 2 : 3;
        // Through LDS, the activation loads are issued BEFORE the weight loads: the memory pipeline returns loads in order, so
        // activations asked for first are back (from L2) long before the weights (from HBM), and their trip through LDS
        // is over when the weights arrive.  Issued after the weights they cost 5-10 % at batch 16.  In operand order they go
        // between the second and the third weight load of the first row tile.
        constexpr int kWBeforeX = MODE == 0 ? 2 : 0;
        for (; u < end; u += WAVES) {
            StageW<FM, RT> cur;
            v4u            xv[LOADS];
            auto           wpart = [&](int i) {
                const int r = i / kWParts, part = i % kWParts;
                load_wfrag_part<FM>(cur.w[r], wgroup + real(r) * tile_stride + (size_t)u * Fmt<FM>::block_bytes, lane, part);
            };
#pragma unroll
            for (int i = 0; i < kWBeforeX; i++) wpart(i);
            // K positions beyond K count as zero activations against the zero weights the native layout holds there (0 x 0,
            // whatever the row holds elsewhere: an infinite activation must not meet a padding weight): such a piece is read
            // at the row's start (a valid address) and replaced by zeros
            const bool beyond = TAIL && u * 256 + 8 * (lane & 31) >= K;
#pragma unroll
            for (int i = 0; i < LOADS; i++) {
                if constexpr (MODE == 0) {
                    xv[i] = *reinterpret_cast<const v4u *>(xpaired + (size_t)u * 256 + 64 * i);
                } else {
                    const uint32_t r0 = (uint32_t)(2 * i) < ncols ? 2 * i : ncols - 1;
                    const uint8_t *sb = xbase + ((size_t)r0 * K + (size_t)u * 256) * 2;
                    uint32_t       vo = (uint32_t)(2 * i + 1) < ncols ? off_pair : off_one;
                    if (beyond) vo -= off_one;
                    const v4u v = *reinterpret_cast<const v4u *>(sb + vo);
                    xv[i] = beyond ? (v4u){ 0u, 0u, 0u, 0u } : v;
                }
            }
#pragma unroll
            for (int i = kWBeforeX; i < RT * kWParts; i++) wpart(i);
#pragma unroll
            for (int r = 0; r < RT; r++) cur.g[r] = load_group_exps<GS>(ggroup, (size_t)real(r) * units + u, lane);
            __builtin_amdgcn_sched_barrier(0); // keep every load of the block issued before anything waits
            v8h x[8][NT];
            if constexpr (MODE == 0) {
                // one load brought two MFMA steps: a DPP rotation of each 16-lane row by 8 moves the second step's data down to
                // columns 0..7 (columns 8..15 then hold the other step's real, finite data and feed outputs never stored)
#pragma unroll
                for (int sl = 0; sl < 4; sl++) {
                    v4u w;
#pragma unroll
                    for (int i = 0; i < 4; i++) w[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)xv[sl][i], 0x128, 0xf, 0xf, false); // row_ror:8
                    x[2 * sl][0]     = __builtin_bit_cast(v8h, xv[sl]);
                    x[2 * sl + 1][0] = __builtin_bit_cast(v8h, w);
                }
            } else {
#pragma unroll
                for (int i = 0; i < LOADS; i++) *reinterpret_cast<v4u *>(xw + 2 * i * kXsRowBytes) = xv[i];
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int t = 0; t < NT; t++) x[s][t] = *reinterpret_cast<const v8h *>(xr + t * 16 * kXsRowBytes + 64 * s);
                // the trip through LDS is issued before anything that waits for weights (left alone, the compiler moves register
                // copies that feed the conversion above the LDS writes, and with them the wait for the weight loads)
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int r = 0; r < RT; r++) {
                AOps<FM> a;
                convert<FM, GS>(cur.w[r], a, cur.g[r]);
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int t = 0; t < NT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.s[s], x[s][t], acc[r][t], 0, 0, 0);
            }
        }
    };
    typedef std::integral_constant<int, 0> Direct;
    typedef std::integral_constant<int, 1> Staged8;
    typedef std::integral_constant<int, 2> StagedAll;
    auto staged = [&](auto mode_c, bool whole_blocks) {
        if (whole_blocks) run(mode_c, std::false_type{}, ufull);
        run(mode_c, std::true_type{}, u1); // at most one block, and only when K is not a multiple of 256
    };
    if (small) {
        if constexpr (NT == 1) {
            if (ncols <= 4) {
                run(Direct{}, std::false_type{}, ufull);
                staged(Staged8{}, false);
            } else {
                staged(Staged8{}, true);
            }
        }
    } else {
        staged(StagedAll{}, true);
    }

    // acc[r][t][i] = sum for output row 16r + 4q+i, batch column 16t+col.  Each wavefront parks its tiles in its own LDS
    // area (its activation rows are dead by now; nobody else ever touched them), then the workgroup sums them.
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) *reinterpret_cast<v4f *>(mine + (r * NT + t) * 1024 + lane * 16) = acc[r][t];
    half_t my_bias[BIAS ? kOutPerThread : 1];
    if constexpr (BIAS) { // (under the wait for the other wavefronts)
#pragma unroll
        for (int j = 0; j < kOutPerThread; j++) {
            const int e = threadIdx.x + j * WAVES * kWave;
            my_bias[j] = bias_of(ws)[(R0 + real(e < RT * NT * 256 ? (e >> 8) / NT : 0)) * 16 + (e & 15)];
        }
    }
    __syncthreads();

#pragma unroll
    for (int j = 0; j < kOutPerThread; j++) {
        const int e = threadIdx.x + j * WAVES * kWave;
        if (e >= RT * NT * 256) break;
        int   rt = e >> 8, i8 = e & 255, n = i8 >> 4, mm = i8 & 15;
        int   r = rt / NT, t = rt % NT;
        int   idx = (((mm >> 2) * 16 + n) << 2) | (mm & 3);
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) sum += *reinterpret_cast<const float *>(lds + w * wave_bytes + rt * 1024 + idx * 4);
        uint32_t ng = nbase + 16 * t + n, mg = (R0 + r) * 16 + mm;
        if (ng < N && (!kRagged || (uint32_t)r <= rlast)) {
            float v = sum * ((float)my_scale[j] * Fmt<FM>::post_scale);
            if constexpr (BIAS) v += (float)my_bias[j];
            if constexpr (!SPLIT)
                C[(size_t)ng * M + mg] = (half_t)v;
            else
                ws[((size_t)split * N + ng) * M + mg] = v;
        }
    }
}

// A operands of MFMA steps 4h..4h+3 (half of a K block) of one lane.
template <int FM, bool GS> __device__ __forceinline__ void convert_half(const WFrag<FM> &f, int h, v8h (&o)[4], uint32_t g)
{
    v32h v = fields_to_halfs<FM>(field_string<FM>(f, h), group_factor<GS>(g, h));
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = slice8(v, i);
}

// ---------------------------------------------------------------------------------------------------------------
// gemm_tile: GEMM for batches above 16, where every weight must meet many activation columns.
//   workgroup = WR x WK wavefronts; tile = (WR*RT*16) rows x (NT*16) columns
//   grid.x enumerates (row block, column block, split), neighbours on one XCD: tile_of
// The K blocks of a split are walked in chunks of WK blocks.  Per chunk the workgroup stages the activation chunk
// [WK][NT*16][256] in LDS (double-buffered, filled by fully coalesced 16-byte loads); wavefront (wr, wk) streams the
// weights of its RT row tiles for K block wk straight from HBM into VGPRs (prefetched one chunk ahead), converts them
// half a block at a time and runs RT*NT MFMAs per step against B operands read once per step from LDS.  The LDS row
// stride is 256+16 halfs (544 bytes): measured on the MI355X, the 16-column x 4-k-group operand read (ds_read_b128) then runs at
// the conflict-free rate of 7 cycles per wavefront, against 8.8 cycles at 528 bytes and 32 cycles without padding.
// The WK partial accumulators are summed through LDS at the end (WK > 1), then scaled and stored.
// Up to about 200 columns the bound is what passes through a CU's vector L1: about 256 lines in flight, an HBM latency of 1 us for the weights and
// 0.4 us from L2 for the activations, so a column block more costs the weights' way once more, all of them at the latency of the memory that the first asks.
// Tiles of 48, 80 and 96 columns exist for the batches that the powers of two miss (FP6 e3m2, us, the best of 32, 64 and 128 columns -> 256 x 80 and
// 256 x 96 here): 28672x8192 N 72 67.3 -> 48.0, N 160 117 -> 81; 8192x28672 N 72 69 -> 49, N 96 68.9 -> 57.9.
// ---------------------------------------------------------------------------------------------------------------

// One segment of a tile's K range: K blocks [u0, u1) of row block `mb` against the batch columns from `nbase`, accumulated
// into acc.  On return the wavefronts with wk == 0 hold the sums of all WK K-wavefronts; the LDS buffers are free again
// once every wavefront of the workgroup has passed a barrier.
template <int FM, bool GS, int NT, int RT, int WR, int WK>
__device__ __forceinline__ void tile_segment(v4f (&acc)[RT][NT], const uint8_t *__restrict__ W, const uint8_t *__restrict__ gexp,
                                             const half_t *__restrict__ X, uint32_t N, uint32_t K, uint32_t units, uint32_t mb, uint32_t nbase,
                                             uint32_t u0, uint32_t u1, uint8_t *lds, int tid, int lane, int wr, int wk, int col, int q)
{
    constexpr int  TN = NT * 16, NTHREADS = WR * WK * kWave;
    constexpr int  kBufBytes = WK * TN * kXsRowBytes;
    constexpr int  kPieces = WK * TN * 32, kPerThread = (kPieces + NTHREADS - 1) / NTHREADS;
    const uint32_t R0 = (mb * WR + wr) * RT; // first row tile of this wavefront
    const size_t   tile_stride = (size_t)units * Fmt<FM>::block_bytes;
    const uint8_t *wgroup = W + (size_t)R0 * tile_stride;
    const uint8_t *ggroup = GS ? gexp + (size_t)R0 * units * 32 : nullptr;

#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = (v4f){ 0.f, 0.f, 0.f, 0.f };

    WFrag<FM> wcur[RT], wnxt[RT];
    uint32_t  gcur[RT], gnxt[RT]; // group exponents travel with the weights (unused without them)
    v4u       xr[kPerThread];

    auto load_w = [&](WFrag<FM>(&dst)[RT], uint32_t(&gdst)[RT], uint32_t c0) {
        const uint32_t u = c0 + wk;
        if (u < u1) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                dst[r]  = load_wfrag<FM>(wgroup + r * tile_stride + (size_t)u * Fmt<FM>::block_bytes, lane);
                gdst[r] = load_group_exps<GS>(ggroup, (size_t)r * units + u, lane);
            }
        }
    };
    // Per-thread pieces of the activation chunk: piece p = tid + NTHREADS*j is 16 bytes, (K block p / (TN*32) of the chunk,
    // batch column (p/32) % TN, halfs 8*(p%32)..+7).  Row pointers and LDS offsets are fixed for the whole kernel.
    // Columns beyond N read the last real row (their outputs are never stored); positions beyond K or beyond the split are
    // read at position 0 of the row (a valid address) and staged as zeros (zero weights meet them, or no wavefront does).
    const half_t *xrow[kPerThread];
    uint32_t      xlds[kPerThread];
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {
        const uint32_t p = tid + NTHREADS * j, n = nbase + (p >> 5) % TN;
        xrow[j] = X + (size_t)(n < N ? n : N - 1) * K + (p & 31) * 8 + (size_t)(p / (TN * 32)) * 256;
        xlds[j] = (p >> 5) * kXsRowBytes + (p & 31) * 16;
    }
    // `full` (a compile-time flag): the whole chunk lies inside K and inside the segment, so every piece is a plain load.  The
    // K loop below is written out per case: one choice per chunk inside the loop costs a wait for the activation loads before
    // the weight loads can be issued.
    auto load_x = [&](auto full, uint32_t c0) {
        if constexpr (decltype(full)::value) {
#pragma unroll
            for (int j = 0; j < kPerThread; j++)
                if (kPieces % NTHREADS == 0 || tid + NTHREADS * j < kPieces) xr[j] = *reinterpret_cast<const v4u *>(xrow[j] + (size_t)c0 * 256);
        } else {
#pragma unroll
            for (int j = 0; j < kPerThread; j++) {
                const uint32_t p = tid + NTHREADS * j;
                if (kPieces % NTHREADS == 0 || p < (uint32_t)kPieces) {
                    const uint32_t u = c0 + p / (TN * 32), k = u * 256 + (p & 31) * 8;
                    const bool     ok = k < K && u < u1;
                    const v4u      v = *reinterpret_cast<const v4u *>(ok ? xrow[j] + (size_t)c0 * 256 : xrow[j] - ((p & 31) * 8 + (size_t)(p / (TN * 32)) * 256));
                    xr[j] = ok ? v : (v4u){ 0u, 0u, 0u, 0u };
                }
            }
        }
    };
    // The same loads one at a time (i = 0 .. kLoads-1: weights first, then activation pieces).  The 256 x 128 tile spreads them
    // over its MFMA steps instead of issuing them in one burst: measured 10-12 % faster for batches from 1024 up (the burst keeps
    // a wavefront, which issues in order, from starting its MFMAs until the CU has accepted its last load); for the smaller
    // tiles, with fewer MFMAs between two loads, spreading measured 0-8 % slower and they keep the burst.
    constexpr bool kSpreadLoads = NT >= 8 && WR * WK >= 8;
    constexpr int  kWParts = Fmt<FM>::bits == 4 ? 2 : 3, kWLoads = RT * kWParts, kLoads = kWLoads + kPerThread, kPerStep = (kLoads + 7) / 8;
    auto load_one = [&](auto full, int i, uint32_t c0) {
        if (i < kWLoads) {
            const int      r = i / kWParts, part = i % kWParts;
            const uint32_t u = c0 + wk;
            if (u < u1) {
                load_wfrag_part<FM>(wnxt[r], wgroup + r * tile_stride + (size_t)u * Fmt<FM>::block_bytes, lane, part);
                if (part == 0) gnxt[r] = load_group_exps<GS>(ggroup, (size_t)r * units + u, lane);
            }
        } else if (i < kLoads) {
            const int      j = i - kWLoads;
            const uint32_t p = tid + NTHREADS * j;
            if (kPieces % NTHREADS == 0 || p < (uint32_t)kPieces) {
                if constexpr (decltype(full)::value) {
                    xr[j] = *reinterpret_cast<const v4u *>(xrow[j] + (size_t)c0 * 256);
                } else {
                    const uint32_t u = c0 + p / (TN * 32), k = u * 256 + (p & 31) * 8;
                    const bool     ok = k < K && u < u1;
                    const v4u      v = *reinterpret_cast<const v4u *>(ok ? xrow[j] + (size_t)c0 * 256 : xrow[j] - ((p & 31) * 8 + (size_t)(p / (TN * 32)) * 256));
                    xr[j] = ok ? v : (v4u){ 0u, 0u, 0u, 0u };
                }
            }
        }
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int j = 0; j < kPerThread; j++)
            if (kPieces % NTHREADS == 0 || tid + NTHREADS * j < kPieces) *reinterpret_cast<v4u *>(lds + buf * kBufBytes + xlds[j]) = xr[j];
    };
    typedef std::integral_constant<int, 0> NoNext;       // the last chunk: nothing to fetch
    typedef std::integral_constant<int, 1> FullNext;     // the next chunk is a full one
    typedef std::integral_constant<int, 2> PartialNext;  // the next chunk is cut by K or by the end of the segment
    typedef std::integral_constant<bool, true> Full;
    typedef std::integral_constant<bool, false> Partial;

    if (u0 < u1) {
        const uint32_t ufull = K / 256 < u1 ? K / 256 : u1; // chunks that end at or before this block are full
        if (u0 + WK <= ufull)
            load_x(Full{}, u0);
        else
            load_x(Partial{}, u0);
        load_w(wcur, gcur, u0);
        store_x(0);
        __syncthreads();
        int      buf = 0;
        uint32_t c0 = u0;
        // one chunk: fetch the next one (if any), compute this one, stage the next one's activations, barrier
        auto chunk = [&](auto next) {
            constexpr int  kNext = decltype(next)::value;
            constexpr bool more = kNext != 0;
            typedef std::integral_constant<bool, kNext == 1> NextIsFull;
            if (more && (!kSpreadLoads || c0 + wk >= u1)) { // (a wavefront without a K block in this chunk has no MFMAs to spread over)
                load_x(NextIsFull{}, c0 + WK);
                load_w(wnxt, gnxt, c0 + WK);
            }
            if (c0 + wk < u1) {
                const uint8_t *xs = lds + buf * kBufBytes + (wk * TN + col) * kXsRowBytes + q * 16;
                v8h            a0[RT][4], a1[RT][4];
#pragma unroll
                for (int r = 0; r < RT; r++) convert_half<FM, GS>(wcur[r], 0, a0[r], gcur[r]);
                // second half converted ahead of the first half's MFMAs: the VALU work then runs under the matrix pipe
#pragma unroll
                for (int r = 0; r < RT; r++) convert_half<FM, GS>(wcur[r], 1, a1[r], gcur[r]);
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        v8h b[NT];
#pragma unroll
                        for (int t = 0; t < NT; t++) b[t] = *reinterpret_cast<const v8h *>(xs + t * 16 * kXsRowBytes + (4 * h + s) * 64);
#pragma unroll
                        for (int r = 0; r < RT; r++)
#pragma unroll
                            for (int t = 0; t < NT; t++)
                                acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h == 0 ? a0[r][s] : a1[r][s], b[t], acc[r][t], 0, 0, 0);
                        if constexpr (kSpreadLoads && more) {
#pragma unroll
                            for (int i = (4 * h + s) * kPerStep; i < (4 * h + s + 1) * kPerStep; i++) load_one(NextIsFull{}, i, c0 + WK);
                        }
                    }
                }
            }
            if (more) {
                store_x(buf ^ 1); // that buffer was last read before the barrier that ended the previous iteration
#pragma unroll
                for (int r = 0; r < RT; r++) wcur[r] = wnxt[r], gcur[r] = gnxt[r];
            }
            __syncthreads();
            c0 += WK, buf ^= 1;
        };
        while (c0 + 2 * WK <= ufull) chunk(FullNext{});
        while (c0 + WK < u1) chunk(PartialNext{});
        chunk(NoNext{});
    }

    // acc[r][t][i]: output row (R0+r)*16 + 4q+i, batch column nbase + 16t + col
    if (WK > 1) {
        float *red = reinterpret_cast<float *>(lds); // [WK][WR][RT*NT][256]; the last barrier above freed the buffers
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < NT; t++) *reinterpret_cast<v4f *>(&red[(((wk * WR + wr) * RT + r) * NT + t) * 256 + lane * 4]) = acc[r][t];
        __syncthreads();
        if (wk == 0) {
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int k2 = 1; k2 < WK; k2++)
                        acc[r][t] += *reinterpret_cast<const v4f *>(&red[(((k2 * WR + wr) * RT + r) * NT + t) * 256 + lane * 4]);
        }
    }
}

// The tile kernel's output goes through LDS.  An MFMA accumulator holds four consecutive rows of ONE batch column per lane, so
// a store straight from the accumulators makes the 16 lanes of a quarter-wavefront write 8 or 16 bytes into each of 16
// different lines (C and the partial sums are [N][M], rows contiguous); the memory pipeline takes a line at a time, and with
// every workgroup finishing at the same moment nothing hides it: measured, those stores were 10-16 % of the GEMMs that split K
// at batches 32-128 and 4-5 % at batch 512.  So the wavefronts that hold results scale them and park them in LDS as a
// [column][row] tile (fp16 for the final output, fp32 for partial sums), and after a barrier every thread of the workgroup
// stores 16 consecutive bytes of one column: a wavefront writes whole lines.
//   stage: TN columns of TM rows, column stride TM * (2 or 4) + 16 bytes
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
template <int NT, int RT, int WR> constexpr size_t tile_stage_bytes(bool partial) { return (size_t)NT * 16 * (WR * RT * 16 * (partial ? 4 : 2) + 16); }

// first half: a wavefront that holds results scales them and parks them in the stage
// (column tiles T0 .. T1-1 of it).  bias: of the tile's first row, or null; added before the one rounding to fp16
template <int FM, int NT, int RT, int WR, typename OutT, int T0 = 0, int T1 = NT>
__device__ __forceinline__ void tile_park(const v4f (&acc)[RT][NT], const v4h (&sc4)[RT], uint8_t *stage, int wr, int col, int q, const half_t *bias = nullptr)
{
    constexpr int TM = WR * RT * 16, kStride = TM * (int)sizeof(OutT) + 16;
    v4h           b4[RT] = {};
    if (sizeof(OutT) == 2 && bias) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const half_t *p = bias + (wr * RT + r) * 16 + 4 * q;
            b4[r] = (v4h){ p[0], p[1], p[2], p[3] };
        }
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = T0; t < T1; t++) {
            v4f v;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[i] = acc[r][t][i] * ((float)sc4[r][i] * Fmt<FM>::post_scale);
                if constexpr (sizeof(OutT) == 2) v[i] += (float)b4[r][i]; // (one instruction with the scaling)
            }
            uint8_t *dst = stage + (16 * (t - T0) + col) * kStride + ((wr * RT + r) * 16 + 4 * q) * (int)sizeof(OutT);
            if constexpr (sizeof(OutT) == 2)
                *reinterpret_cast<v4h *>(dst) = (v4h){ (half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3] };
            else
                *reinterpret_cast<v4f *>(dst) = v;
        }
}
// second half, after a barrier: every thread of the workgroup stores 16-byte pieces of the stage's columns
template <int NT, int RT, int WR, int NTHREADS, typename OutT>
__device__ __forceinline__ void tile_flush(OutT *__restrict__ out, const uint8_t *stage, uint32_t M, uint32_t N, uint32_t mb, uint32_t nbase, int tid)
{
    constexpr int TM = WR * RT * 16, TN = NT * 16, kStride = TM * (int)sizeof(OutT) + 16, kPer16 = 16 / (int)sizeof(OutT); // outputs per 16 bytes
    constexpr int kPiecesPerCol = TM / kPer16, kPieces = TN * kPiecesPerCol;
#pragma unroll
    for (int p = tid; p < kPieces; p += NTHREADS) {
        const int      c = p / kPiecesPerCol, piece = p % kPiecesPerCol;
        const uint32_t ng = nbase + c;
        if (ng < N) {
            const v4u d = *reinterpret_cast<const v4u *>(stage + c * kStride + piece * 16);
            *reinterpret_cast<v4u *>(out + (size_t)ng * M + (size_t)mb * TM + piece * kPer16) = d;
        }
    }
}

template <int FM, int NT, int RT, int WR, int NTHREADS, typename OutT>
__device__ __forceinline__ void tile_store(const v4f (&acc)[RT][NT], const v4h (&sc4)[RT], OutT *__restrict__ out, uint8_t *stage, bool holds_results,
                                           uint32_t M, uint32_t N, uint32_t mb, uint32_t nbase, int tid, int wr, int col, int q, const half_t *bias)
{
    if (holds_results) tile_park<FM, NT, RT, WR, OutT>(acc, sc4, stage, wr, col, q, bias);
    __syncthreads();
    tile_flush<NT, RT, WR, NTHREADS, OutT>(out, stage, M, N, mb, nbase, tid);
}

// Workgroup id -> (row block, split, column block).  Ids that are congruent mod 8 run on one XCD and share its L2, so XCD x is given a
// run of consecutive triples (the column blocks of a row block read the same weights, its splits write partial sums that one
// reduction workgroup reads): the first (grid mod 8) XCDs take one triple more than the others.
// Without a split the triples of the large tiles are counted in panels of 1024 rows, down the rows of a panel before the next column block:
// the 32 or 64 workgroups that an XCD holds then cover about 1024 rows x 512-1024 columns, and what its L2 fetches for them is about
// as small as it gets (with all the column blocks of one row block first, a long prompt's activations pass by once for every 256 or 512 rows).
// Measured at FP6 e3m2, us, rows first -> panels: gemm_prefill 8192x8192 N 4096 582 -> 444, 14336x4096 N 3000 334 -> 306, 28672x8192 N 2048 832 -> 787;
// gemm_ws 28672x8192 N 2048 914 -> 831, 8192x8192 N 4096 503 -> 472; gemm_tile 256 x 128 8192x8192 N 4096 488 -> 460
// (forced: the dispatch gives some of these another shape).  What is fetched falls from 2267 to 784 MB (gemm_tile) and 4101 to 1629 (gemm_prefill 28672x8192).  Panels of 512, 2048 and 4096
// rows: within 2 %, and up to 6 % behind.  128 x 32 tiles lose by 6 % and keep the rows.
// In panels every XCD reads all the weights of a panel, by rows few XCDs read the same ones: activations that stay in an L2 of 4 MB anyway are no
// reason for it (single rounds of 256-row tiles, K up to 1536: 0.8 us longer in panels with weights that come from memory, though less is fetched, 10.3 MB against
// 14.6 at 1280x768 N 1658; level with weights that the caches hold).  Tiles of 256 rows are counted in panels where the activations take more than 2 MB, in a single round of the 256 CUs more than 4 MB and
// with 128 workgroups at least (a few leave the order no part).  Time in panels / by rows on 440 problems (K 256 to 28288; activations kept and changed from
// launch to launch), always -> by this rule: gemm_tile 256 x 64 1.02 (0.90-1.19) -> 0.99 (0.90-1.05), 256 x 128 0.99 (0.84-1.10) -> 0.98 (0.84-1.01),
// gemm_ws 256 x 64 1.00 (0.87-1.11) -> 0.99 (0.87-1.04).  What it leaves to the rows was at most 4 % faster in panels, 1024x256 N 2537 1.18.  gemm_prefill
// 0.98 (0.64-1.03) always.
struct TileId { uint32_t mb, split, nb; };
template <int TM, int TN> __device__ __forceinline__ TileId tile_of(uint32_t splitK, uint32_t nblocks, uint32_t N, uint32_t K)
{
    constexpr uint32_t kPanel = TM * TN >= 128 * 128 ? 1024 / TM : 1; // row blocks per panel
    const uint32_t     q = gridDim.x >> 3, r = gridDim.x & 7u, x = blockIdx.x & 7u, id = x * q + (x < r ? x : r) + (blockIdx.x >> 3);
    const uint64_t     X = (uint64_t)N * K * 2; // bytes of the activations
    const bool         panels = kPanel > 1 && splitK == 1 && (TM < 256 || (gridDim.x > 256 ? X > 2u << 20 : gridDim.x >= 128 && X > 4u << 20));
    if (panels) {
        const uint32_t mblocks = gridDim.x / nblocks, first = id / (kPanel * nblocks) * kPanel, in = id - first * nblocks;
        const uint32_t high = mblocks - first < kPanel ? mblocks - first : kPanel; // the last panel may be lower
        return TileId{ first + in % high, 0, in / high };
    }
    const uint32_t rest = id / nblocks;
    return TileId{ rest / splitK, rest % splitK, id % nblocks };
}

template <int FM, bool GS, int NT, int RT, int WR, int WK, bool BIAS>
__global__ __launch_bounds__(WR *WK *kWave) void gemm_tile(const uint8_t *__restrict__ W, const half_t *__restrict__ scales,
                                                           const uint8_t *__restrict__ gexp, const half_t *__restrict__ X, half_t *__restrict__ C,
                                                           float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                           uint32_t units, uint32_t splitK, uint32_t nblocks)
{
    constexpr int  TN = NT * 16, NTHREADS = WR * WK * kWave;
    constexpr int  kBufBytes = WK * TN * kXsRowBytes;
    constexpr int  kPieces = WK * TN * 32, kPerThread = (kPieces + NTHREADS - 1) / NTHREADS;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    asm volatile("" ::"s"(W), "s"(scales), "s"(gexp), "s"(X), "s"(C), "s"(ws), "s"(M), "s"(N), "s"(K), "s"(units), "s"(splitK), "s"(nblocks)); // one batch of argument loads
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6); // a scalar, like all that follows from it
    const int wr = wave % WR, wk = wave / WR;
    const int col = lane & 15, q = lane >> 4;

    const TileId   id = tile_of<WR * RT * 16, TN>(splitK, nblocks, N, K);
    const uint32_t mb = id.mb, split = id.split, nb = id.nb;
    const uint32_t nbase = nb * TN, R0 = (mb * WR + wr) * RT; // first row tile of this wavefront

    uint32_t u0 = 0, u1 = units;
    if (splitK > 1) {
        const uint32_t avg = units / splitK, extra = units % splitK;
        u0 = split * avg + (split < extra ? split : extra);
        u1 = u0 + avg + (split < extra ? 1u : 0u);
    }

    v4f acc[RT][NT];
    // row scales of this lane's outputs (rows 4q..4q+3 of each of its row tiles), fetched before the main loop so that no
    // global load sits on the tail of the kernel
    v4h sc4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const half_t *p = scales + (R0 + r) * 16 + 4 * q;
        if ((reinterpret_cast<uintptr_t>(scales) & 7u) == 0) // uniform: one 8-byte load where the caller's pointer allows it
            sc4[r] = *reinterpret_cast<const v4h *>(p);
        else
            sc4[r] = (v4h){ p[0], p[1], p[2], p[3] };
    }

    tile_segment<FM, GS, NT, RT, WR, WK>(acc, W, gexp, X, N, K, units, mb, nbase, u0, u1, lds, tid, lane, wr, wk, col, q);

    // the output tile is parked where the partial sums of the K wavefronts met: everybody has read those first
    if (WK > 1) __syncthreads();
    uint8_t *stage = lds;
    if (BIAS || splitK == 1) // (a split's bias is added by the reduction)
        tile_store<FM, NT, RT, WR, NTHREADS>(acc, sc4, C, stage, wk == 0, M, N, mb, nbase, tid, wr, col, q, BIAS ? bias_of(ws) + mb * (WR * RT * 16) : nullptr);
    else
        tile_store<FM, NT, RT, WR, NTHREADS>(acc, sc4, ws + (size_t)split * N * M, stage, wk == 0, M, N, mb, nbase, tid, wr, col, q, nullptr);
}

// ---------------------------------------------------------------------------------------------------------------
// gemm_ws: the tile GEMM with the wavefronts of a workgroup divided into two kinds.
//   workgroup = WR arithmetic wavefronts + PW loading wavefronts; tile = (WR*RT*16) rows x (NT*16) columns; same grid as gemm_tile
// The loading wavefronts move K blocks from memory into LDS without passing through registers (global_load_lds_dwordx4):
// the tile's weight blocks exactly as they lie in memory (native blocks of raw codes, 16-byte pieces in lane order) and the
// activation rows of the block.  The arithmetic wavefronts never touch global memory inside the K loop (with 256 rows for group exponents only): they read their
// weight pieces and their B operands from LDS, convert and run the MFMAs.  In gemm_tile every wavefront does both, a
// wavefront issues its instructions in order, and the CU's memory pipeline accepts a chunk's loads at its own pace: there
// the second wavefront of every SIMD starts its MFMAs a third of a K step late, and a block has to arrive within the one
// step before it is used.  Here the weights travel SW-1 blocks ahead of the arithmetic and the activations SX-1 blocks
// (SW >= SX >= 2: the weights come from HBM, the activations from L2), during the whole of those steps.
// LDS: a ring of SW weight stages [WR*RT tiles x block bytes] and a ring of SX activation stages [NT*16 rows x 512 bytes].
// The activation rows are not padded (256 x 64 with FP6 weights and two stages each fills the 160 KB to the byte): piece p
// of row n (16 bytes) lies at slot p ^ (n & 15) of its row, which makes the operand read of eight batch columns at one K
// position touch eight different slots.  One barrier per K block: before it the loading wavefronts wait until the NEXT
// block has landed (s_waitcnt with the number of transfers issued after it: they complete in order).
// ---------------------------------------------------------------------------------------------------------------
template <int FM, int NT, int RT, int WR, int SW, int SX> constexpr size_t ws_ring_bytes()
{
    return (size_t)SW * WR * RT * Fmt<FM>::block_bytes + (size_t)SX * NT * 16 * 512;
}
// Group exponents of 128 rows travel with the weights, in a ring of SW stages behind the activations', 4 bytes a row.  Loaded by the arithmetic
// wavefronts, one block ahead, they were waited for at the barrier of every block, and the blocks that a ring of three has under way did not help: the
// shapes that had won without exponents lost up to 28 % with them to those they had replaced.  us, shape before the ring of three / loads in registers /
// through LDS: e2m1 8704x16192 N 53 29.5 / 38.1 / 29.1; e2m2 5632x10432 N 236 48.7 / 61.8 / 44.6; e2m1 1792x25984 N 672 133.8 / 144.7 / 101.0; over 167
// problems of N 33 to 946 LDS / registers 0.89 (0.70-1.00).  With 256 rows LDS is full and SW is 2, one block ahead as in registers.
template <bool GS, int WR> constexpr bool ws_exps_in_lds() { return GS && WR == 4; }
template <bool GS, int RT, int WR, int SW> constexpr size_t ws_exps_ring_bytes() { return ws_exps_in_lds<GS, WR>() ? (size_t)SW * WR * RT * 64 : 0; }

template <int N> __device__ __forceinline__ void wait_transfers_and_barrier()
{
    static_assert(N >= 0 && N <= 63, "s_waitcnt vmcnt holds six bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int FM, bool GS, int NT, int RT, int WR, int PW, int SW, int SX>
__global__ __launch_bounds__((WR + PW) * kWave) void gemm_ws(const uint8_t *__restrict__ W, const half_t *__restrict__ scales,
                                                             const uint8_t *__restrict__ gexp, const half_t *__restrict__ X, half_t *__restrict__ C,
                                                             float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                             uint32_t units, uint32_t splitK, uint32_t nblocks)
{
    static_assert(SW >= SX && SX >= 2, "weights run at least as far ahead as activations; a stage is filled while another is read");
    constexpr int TN = NT * 16, TILES = WR * RT, NTHREADS = (WR + PW) * kWave;
    constexpr int kBlock = Fmt<FM>::block_bytes, kWStage = TILES * kBlock, kXStage = TN * 512, kXRing = SW * kWStage; // the activation ring follows the weight ring
    constexpr bool kGLds = ws_exps_in_lds<GS, WR>();
    constexpr int  kGStage = TILES * 64, kGRing = kXRing + SX * kXStage;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    asm volatile("" ::"s"(W), "s"(scales), "s"(gexp), "s"(X), "s"(C), "s"(ws), "s"(M), "s"(N), "s"(K), "s"(units), "s"(splitK), "s"(nblocks)); // one batch of argument loads
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, q = lane >> 4;

    const TileId   id = tile_of<WR * RT * 16, NT * 16>(splitK, nblocks, N, K);
    const uint32_t mb = id.mb, split = id.split, nb = id.nb;
    const uint32_t nbase = nb * TN;
    uint32_t       u0 = 0, u1 = units;
    if (splitK > 1) {
        const uint32_t avg = units / splitK, extra = units % splitK;
        u0 = split * avg + (split < extra ? split : extra);
        u1 = u0 + avg + (split < extra ? 1u : 0u);
    }
    const int nk = (int)(u1 - u0); // K blocks of this workgroup, numbered 0 .. nk-1 below

    v4f acc[RT][NT];
    v4h sc4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = (v4f){ 0.f, 0.f, 0.f, 0.f };

    if (wave >= WR) {
        // ---------------------------------------------------------------- loading wavefronts
        // One instruction moves 64 x 16 bytes from memory straight into 1 KB of LDS, lane l to byte 16*l of the destination;
        // each lane chooses its source address.  Instruction i of a weight (activation) stage fills its pieces 64*i .. 64*i+63;
        // this wavefront issues the instructions pw, pw + PW, ...
        typedef __attribute__((address_space(1))) void gvoid;
        typedef __attribute__((address_space(3))) void lvoid;
        const int     pw = wave - WR;
        constexpr int PB = kBlock / 16, kWPieces = TILES * PB, kXPieces = TN * 32;
        static_assert(kWPieces % 64 == 0 && kXPieces % 64 == 0, "a stage is a whole number of 1 KB instructions");
        constexpr int kWInst = kWPieces / 64, kXInst = kXPieces / 64;
        static_assert(kWInst % PW == 0 && kXInst % PW == 0, "every loading wavefront issues the same number of transfers (the waits count them)");
        static_assert(!kGLds || TILES * 16 % PW == 0 && TILES * 16 / PW <= 64, "a stage of exponents is one transfer of every loading wavefront");
        constexpr int kWPer = kWInst / PW, kXPer = kXInst / PW, kGRows = TILES * 16 / PW, kWSteps = kWPer + (kGLds ? 1 : 0);
        // transfers issued after those of block j+1 when step j ends: the later of its two transfers is the activation one, issued
        // SX-2 steps ago and followed there by that step's weight transfers when the weight ring is the deeper one
        constexpr int kAhead = (SW > SX ? kWSteps : 0) + (SX - 2) * (kWSteps + kXPer);
        // weight piece P (16 bytes) of a stage = piece P % PB of the block of tile P / PB: a straight copy
        const uint8_t *wsrc[kWPer];
#pragma unroll
        for (int j = 0; j < kWPer; j++) {
            const uint32_t P = (pw + PW * j) * 64 + lane, tile = P / PB, within = P % PB;
            wsrc[j] = W + ((size_t)(mb * TILES + tile) * units + u0) * kBlock + within * 16;
        }
        const uint32_t grow = pw * kGRows + (kGLds ? lane % kGRows : 0);
        const uint8_t *gsrc = kGLds ? gexp + ((size_t)(mb * TILES + grow / 16) * units + u0) * 32 + grow % 16 * 2 : nullptr;
        // activation piece P of a stage = slot P % 32 of row P / 32, which holds piece slot ^ (row & 15) of that batch column's
        // 256 halfs (columns beyond N repeat the last real one: their outputs are never stored)
        const uint8_t *xsrc[kXPer];
        uint32_t       xpiece[kXPer];
#pragma unroll
        for (int j = 0; j < kXPer; j++) {
            const uint32_t P = (pw + PW * j) * 64 + lane, n = P >> 5, piece = (P & 31) ^ (n & 15);
            const uint32_t row = nbase + n < N ? nbase + n : N - 1;
            xsrc[j] = reinterpret_cast<const uint8_t *>(X + (size_t)row * K + (size_t)u0 * 256) + piece * 16;
            xpiece[j] = piece;
        }
        auto fetch_w = [&](int k, int slot) { // weights of block k -> stage `slot` of the weight ring
            uint8_t *st = lds + slot * kWStage;
#pragma unroll
            for (int j = 0; j < kWPer; j++)
                __builtin_amdgcn_global_load_lds((gvoid *)(wsrc[j] + (size_t)k * kBlock), (lvoid *)(st + (pw + PW * j) * 1024), 16, 0, 0);
            if constexpr (kGLds) // and their exponents: lane l takes the two of row pw * kGRows + l, which LDS receives as 32 bits
                if (lane < kGRows)
                    __builtin_amdgcn_global_load_lds((gvoid *)(gsrc + (size_t)k * 32), (lvoid *)(lds + kGRing + slot * kGStage + pw * kGRows * 4), 2, 0, 0);
        };
        auto fetch_x = [&](int k, int slot) { // activations of block k -> stage `slot` of the activation ring
            uint8_t *st = lds + kXRing + slot * kXStage;
            if ((u0 + k + 1) * 256 <= K) {
#pragma unroll
                for (int j = 0; j < kXPer; j++)
                    __builtin_amdgcn_global_load_lds((gvoid *)(xsrc[j] + (size_t)k * 512), (lvoid *)(st + (pw + PW * j) * 1024), 16, 0, 0);
            } else { // the block that K cuts goes through registers: positions beyond K are read at the block's start (a valid address) and stored as zeros
#pragma unroll
                for (int j = 0; j < kXPer; j++) {
                    const bool ok = (u0 + k) * 256 + xpiece[j] * 8 < K;
                    const v4u  v = *reinterpret_cast<const v4u *>(xsrc[j] + (size_t)k * 512 - (ok ? 0u : xpiece[j] * 16));
                    *reinterpret_cast<v4u *>(st + (pw + PW * j) * 1024 + lane * 16) = ok ? v : (v4u){ 0u, 0u, 0u, 0u };
                }
            }
        };
        if (nk > 0) {
            // step j (j = -(SW-1) .. nk-1; the negative ones fill the rings) issues the activations of block j+SX-1 and then the
            // weights of block j+SW-1; it ends with a barrier before which block j+1 must have landed
            int wslot = 0, xslot = 0; // ring positions the next transfers go to
            for (int j = 1 - SW; j < nk; j++) {
                const int kx = j + SX - 1, kw = j + SW - 1;
                if (kx >= 0 && kx < nk) {
                    fetch_x(kx, xslot);
                    xslot = xslot + 1 == SX ? 0 : xslot + 1;
                }
                if (kw < nk) {
                    fetch_w(kw, wslot);
                    wslot = wslot + 1 == SW ? 0 : wslot + 1;
                }
                if (j >= -1) {
                    // the count is exact only while every transfer it assumes was issued; at the end of K wait for everything
                    // (block j+1's last transfer is followed by exactly kAhead others as long as this step still had weights to fetch)
                    if (kw < nk)
                        wait_transfers_and_barrier<kAhead>();
                    else
                        wait_transfers_and_barrier<0>();
                }
            }
        }
    } else {
        // ---------------------------------------------------------------- arithmetic wavefronts
        const int      wr = wave;
        const uint32_t R0 = (mb * WR + wr) * RT; // first row tile of this wavefront
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const half_t *p = scales + (R0 + r) * 16 + 4 * q;
            if ((reinterpret_cast<uintptr_t>(scales) & 7u) == 0)
                sc4[r] = *reinterpret_cast<const v4h *>(p);
            else
                sc4[r] = (v4h){ p[0], p[1], p[2], p[3] };
        }
        const uint8_t *ggroup = GS ? gexp + ((size_t)R0 * units + u0) * 32 : nullptr;
        uint32_t       xoff[8]; // B operand of MFMA step s: row col, piece 4s+q, at its swizzled slot
#pragma unroll
        for (int s8 = 0; s8 < 8; s8++) xoff[s8] = kXRing + col * 512 + 16 * ((4 * s8 + q) ^ col);
        const uint32_t woff = wr * RT * kBlock + lane * 16;
        if (nk > 0) {
            uint32_t gnext[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) gnext[r] = load_group_exps<GS && !kGLds>(ggroup, (size_t)r * units, lane);
            __syncthreads(); // block 0 has landed
            int wslot = 0, xslot = 0;
            for (int k = 0; k < nk; k++) {
                const uint8_t *wst = lds + wslot * kWStage, *xst = lds + xslot * kXStage, *gst = lds + kGRing + wslot * kGStage;
                wslot = wslot + 1 == SW ? 0 : wslot + 1;
                xslot = xslot + 1 == SX ? 0 : xslot + 1;
                WFrag<FM> wf[RT];
                uint32_t  g[RT];
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const uint8_t *b = wst + woff + r * kBlock;
                    wf[r].a = *reinterpret_cast<const v4u *>(b);
                    wf[r].b = *reinterpret_cast<const v4u *>(b + 1024);
                    if constexpr (Fmt<FM>::bits == 6) wf[r].c = *reinterpret_cast<const v4u *>(b + 2048);
                    if constexpr (Fmt<FM>::bits == 5) wf[r].s = *reinterpret_cast<const v2u *>(wst + (wr * RT + r) * kBlock + 2048 + lane * 8);
                    g[r] = kGLds ? *reinterpret_cast<const uint32_t *>(gst + (wr * RT + r) * 64 + col * 4) : gnext[r];
                    if (GS && !kGLds && k + 1 < nk) gnext[r] = load_group_exps<GS>(ggroup, (size_t)r * units + k + 1, lane);
                }
                v8h a0[RT][4], a1[RT][4];
#pragma unroll
                for (int r = 0; r < RT; r++) convert_half<FM, GS>(wf[r], 0, a0[r], g[r]);
#pragma unroll
                for (int r = 0; r < RT; r++) convert_half<FM, GS>(wf[r], 1, a1[r], g[r]);
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        v8h b[NT];
#pragma unroll
                        for (int t = 0; t < NT; t++) b[t] = *reinterpret_cast<const v8h *>(xst + xoff[4 * h + s] + t * 16 * 512);
#pragma unroll
                        for (int r = 0; r < RT; r++)
#pragma unroll
                            for (int t = 0; t < NT; t++)
                                acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h == 0 ? a0[r][s] : a1[r][s], b[t], acc[r][t], 0, 0, 0);
                    }
                }
                __syncthreads();
            }
        }
    }
    // every wavefront has passed the last barrier of the K loop: the rings are free, the output tile is parked there
    uint8_t *stage = lds;
    if (splitK == 1) {
        if (wave < WR) tile_park<FM, NT, RT, WR, half_t>(acc, sc4, stage, wave, col, q, ws ? bias_of(ws) + mb * (WR * RT * 16) : nullptr);
        __syncthreads();
        tile_flush<NT, RT, WR, NTHREADS, half_t>(C, stage, M, N, mb, nbase, tid);
    } else {
        if (wave < WR) tile_park<FM, NT, RT, WR, float>(acc, sc4, stage, wave, col, q);
        __syncthreads();
        tile_flush<NT, RT, WR, NTHREADS, float>(ws + (size_t)split * N * M, stage, M, N, mb, nbase, tid);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// gemm_prefill: the tile GEMM for long prompts, where the matrix cores are the bound.
//   workgroup = 2 x 2 wavefronts; tile = (2*RT*16) rows x (2*NT*16) columns, (RT*16) x (NT*16) of it per wavefront; grid as gemm_tile
// What bounds such a GEMM on this chip is that the conversions do not run in the MFMAs' shadow (70-90 cycles against 17 per MFMA) and,
// in gemm_tile and gemm_ws, the LDS operand reads: there a wavefront owns 32 rows, one read for every two MFMAs.  Here it owns
// 64 x 64 outputs: a read feeds four MFMAs, a converted fragment sixteen, on a tile half as large as the 256 x 128 one that takes as
// many cycles per output, so that the last round of workgroups leaves half as much of the chip idle.
// K is walked in chunks of 128 (half a native block).  The chunk's B operands live in registers, all 4 steps x NT of them;
// the row tiles pass by one after the other: section r runs 4 * NT MFMAs on row tile r while tile r+1 is converted and the raw
// codes of tile r+1 of the NEXT chunk are asked for (memory -> registers, a whole chunk ahead).  The activations of the next chunk go
// memory -> LDS without registers in the first sections, and the last section, behind the only barrier of a chunk, replaces the B
// operands step by step as its own MFMAs release them.
// LDS: two stages of [2*NT*16 rows x 256 bytes], piece p of row n (16 bytes) at slot p ^ (n & 15): eight neighbouring columns at one
// K position then lie in eight different bank groups.
// 128 x 128 (RT = NT = 4) takes 197-227 registers and 64 KB, two workgroups per CU.  Measured on problems that the dispatch gives it (us, in turn
// in captured graphs, the shape it replaces -> this): FP6 4608x4544 N 777: 62.5 -> 40.4, 9984x3328 N 312: 41.4 -> 31.5, 28672x8192 N 384: 222 -> 185,
// N 1000: 473 -> 401, 18944x2432 N 1305: 154 -> 131; FP5 3584x4928 N 3435: 151 -> 125; FP4 6912x4416 N 2563: 199 -> 160.  With tiles counted in panels
// also where the rounds come out even (FP6 8192x7168 N 1676: 198 -> 184, 16384x13824 N 858: 366 -> 346, 16384x6656 N 2482: 474 -> 437).  Left to the other shapes: up to N 512 with even
// rounds, where it is level (8192x8192 N 512: 62.7 both), and a single round of 256 x 64 tiles, where it is behind
// (FP5 with group exponents 4608x4544 N 777: 39.5 against 42.8).  Tiles of 256 x 128 (RT 8, 400+ registers, one wavefront per SIMD: 3-15 % slower than
// gemm_tile's) and 256 x 256 (RT = NT = 8: spills) were left out.
// ---------------------------------------------------------------------------------------------------------------
// f(0), ..., f(RT - 1) with the index as a compile-time constant (a body this long is past what `#pragma unroll` takes)
template <int RT, int R = 0, typename F> __device__ __forceinline__ void sections(const F &f)
{
    f(std::integral_constant<int, R>{});
    if constexpr (R + 1 < RT) sections<RT, R + 1>(f);
}

struct RawHalf { v4u p; v2u s; uint32_t g; }; // one lane's codes of half a block of one row tile, as loaded (s, g: where the format has them)

// raw codes of half H of a native block (and its group exponent): what field_string(., H) needs
template <int FM, bool GS, int H> __device__ __forceinline__ void load_raw_half(RawHalf &f, const uint8_t *block, const uint8_t *gexp32, int lane)
{
    constexpr int kPiece = Fmt<FM>::bits == 6 ? 2048 : 1024; // the second half's 16-byte piece (6 bits: pieces a | b | c, b shared)
    f.p = *reinterpret_cast<const v4u *>(block + H * kPiece + lane * 16);
    if constexpr (Fmt<FM>::bits == 6) f.s = *reinterpret_cast<const v2u *>(block + 1024 + lane * 16 + 8 * H);
    if constexpr (Fmt<FM>::bits == 5) f.s[0] = *reinterpret_cast<const uint32_t *>(block + 2048 + lane * 8 + 4 * H);
    if constexpr (GS) f.g = gexp32[2 * (lane & 15) + H];
}
template <int FM, bool GS, int H> __device__ __forceinline__ v32h convert_raw_half(const RawHalf &f)
{
    v6u src;
    if constexpr (Fmt<FM>::bits == 6)
        src = H == 0 ? (v6u){ f.p[0], f.p[1], f.p[2], f.p[3], f.s[0], f.s[1] } : (v6u){ f.s[0], f.s[1], f.p[0], f.p[1], f.p[2], f.p[3] };
    else if constexpr (Fmt<FM>::bits == 5)
        src = fp5_expand(f.p[0], f.p[1], f.p[2], f.p[3], f.s[0]);
    else
        src = fp4_expand(f.p);
    return fields_to_halfs<FM>(src, GS ? __builtin_bit_cast(float, f.g << 23) : 1.0f);
}

// (no __restrict__ on what the K loop reads: its loads must stay where the waits count them, on their side of the barriers)
template <int FM, bool GS, int NT, int RT>
__global__ __launch_bounds__(4 * kWave, 2) void gemm_prefill(const uint8_t *W, const half_t *__restrict__ scales, const uint8_t *gexp, const half_t *X,
                                                          half_t *__restrict__ C, float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                          uint32_t units, uint32_t splitK, uint32_t nblocks)
{
    static_assert(RT >= 4 && RT % 2 == 0, "the activation transfers take the first half of the sections");
    constexpr int TN = 2 * NT * 16, kStage = TN * 256;
    constexpr int kDma = TN / 16;          // transfers of 1 KB (four rows) per wavefront and chunk
    constexpr int kDmaSections = RT / 2, kDmaPer = kDma / kDmaSections;
    static_assert(kDma % kDmaSections == 0, "every section issues the same number of transfers");
    // loads a wavefront issues for certain after its last transfer of a chunk and before the chunk's barrier
    constexpr int kRawLoads = (Fmt<FM>::bits == 4 ? 1 : 2) + (GS ? 1 : 0), kAfterDma = (RT - kDmaSections) * kRawLoads;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, q = lane >> 4, wr = wave & 1, wc = wave >> 1;

    const TileId   id = tile_of<2 * RT * 16, TN>(splitK, nblocks, N, K);
    const uint32_t mb = id.mb, split = id.split, nb = id.nb;
    const uint32_t nbase = nb * TN, R0 = (mb * 2 + wr) * RT;
    uint32_t       u0 = 0, u1 = units;
    if (splitK > 1) {
        const uint32_t avg = units / splitK, extra = units % splitK;
        u0 = split * avg + (split < extra ? split : extra);
        u1 = u0 + avg + (split < extra ? 1u : 0u);
    }

    v4f acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = (v4f){ 0.f, 0.f, 0.f, 0.f };

    const size_t   tile_stride = (size_t)units * Fmt<FM>::block_bytes;
    const uint8_t *wgroup = W + (size_t)R0 * tile_stride;
    const uint8_t *ggroup = GS ? gexp + (size_t)R0 * units * 32 : nullptr;
    RawHalf        raw[RT];
    auto           load_raw = [&](auto half_c, int r, uint32_t u) __attribute__((always_inline)) {
        load_raw_half<FM, GS, decltype(half_c)::value>(raw[r], wgroup + r * tile_stride + (size_t)u * Fmt<FM>::block_bytes,
                                                       GS ? ggroup + ((size_t)r * units + u) * 32 : nullptr, lane);
    };

    // transfer j of this wavefront fills rows 4*wave + 16*j .. +3 of a stage: lane l is slot l%16 of row 4*wave + 16*j + l/16, which
    // holds the piece slot ^ (row & 15), the same piece for every j.  Rows beyond N repeat the last real one (never stored).
    typedef __attribute__((address_space(3))) void lvoid;
    // Offsets are formed anew at every use (two instructions): kept, they would take two registers per transfer.
    const uint32_t xrow0 = 4 * wave + q, xpiece = (lane & 15) ^ xrow0; // xrow0 < 16
    const uint32_t xoff0 = xrow0 * K * 2, xlast = (N - nbase < (uint32_t)TN ? N - 1 - nbase : TN - 1) * K * 2; // 32 bits: the launcher bounds K
    auto           row_offset = [&](int j) __attribute__((always_inline)) {
        uint32_t o = xoff0;
        asm volatile("" : "+v"(o));
        o += (uint32_t)j * 32u * K;
        return o < xlast ? o : xlast;
    };
    // Positions beyond K (the last block of a K that is no multiple of 256) are given an offset outside the buffer, which reads as
    // zero: no branch, and the same number of transfers to wait for in every chunk.  (The buffer form of the instruction also lets the
    // compiler count the raw codes' loads; behind global_load_lds, which it takes for a flat access, it waits for all of them.)
    // The whole offset is in the vector operand, which the range check compares with the size as it is.  A scalar offset would be taken
    // off the size first, and with one row in the buffer and K % 256 == 64 the last half block's lies beyond the size.
    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(X + (size_t)nbase * K), 0, (int)(xlast + K * 2), 0x00027000);
    auto       transfer = [&](int j, uint32_t h, uint32_t stage) __attribute__((always_inline)) {
        const uint32_t pos = h * 128 + xpiece * 8, off = row_offset(j) + (pos < K ? pos * 2 : 0xc0000000u); // (row offset + 2K < 2^29)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xbuf, (lvoid *)(lds + stage * kStage + (wave + 4 * j) * 1024), 16, off, 0, 0, 0);
    };

    v8h            b[4][NT];
    const uint8_t *xread = lds + (wc * NT * 16 + col) * 256;
    auto           read_b = [&](int s, uint32_t stage) __attribute__((always_inline)) {
        const uint8_t *p = xread + stage * kStage + (((4 * s + q) ^ col) * 16);
#pragma unroll
        for (int t = 0; t < NT; t++) b[s][t] = *reinterpret_cast<const v8h *>(p + t * 16 * 256);
    };

    typedef std::integral_constant<int, 0> Half0;
    typedef std::integral_constant<int, 1> Half1;

    // Chunk h: its B operands are in b, its row tile 0 in a, its other raw codes in (or on the way to) raw[1..]; raw[0] is the next
    // chunk's.  There is no special last chunk: after it a chunk is fetched once more and not used.  One copy of the code per half
    // keeps the accumulators in place (copies for the ends of K made the compiler move them between the halves of the register file).
    v32h a;
    auto chunk = [&](auto half_c, uint32_t h) __attribute__((always_inline)) {
        constexpr int H = decltype(half_c)::value;
        typedef std::integral_constant<int, 1 - H> Other;
        const uint32_t hx = h + 1 < 2 * u1 ? h + 1 : h, u_next = hx >> 1, u_after = h + 2 < 2 * u1 ? (h + 2) >> 1 : h >> 1;
        sections<RT>([&](auto r_c) __attribute__((always_inline)) {
            constexpr int r = decltype(r_c)::value;
            if constexpr (r < kDmaSections) {
#pragma unroll
                for (int j = r * kDmaPer; j < (r + 1) * kDmaPer; j++) transfer(j, hx, (h + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (r == RT - 1) { // the next chunk's activations have landed, for every wavefront
                wait_transfers_and_barrier<kAfterDma>();
                __builtin_amdgcn_sched_barrier(0);
            }
            v32h a_next;
            if constexpr (r + 1 < RT) {
                a_next = convert_raw_half<FM, GS, H>(raw[r + 1]);
                load_raw(Other{}, r + 1, u_next);
            } else {
                a_next = convert_raw_half<FM, GS, 1 - H>(raw[0]);
                load_raw(half_c, 0, u_after);
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
#pragma unroll
                for (int t = 0; t < NT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(slice8(a, s), b[s][t], acc[r][t], 0, 0, 0);
                if constexpr (r == RT - 1) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_b(s, (h + 1) & 1);
                }
            }
            a = a_next;
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    if (u0 < u1) { // (more splits than K blocks leave some empty: their partial sums are zeros)
#pragma unroll
        for (int j = 0; j < kDma; j++) transfer(j, 2 * u0, 0);
#pragma unroll
        for (int r = 0; r < RT; r++) load_raw(Half0{}, r, u0);
        wait_transfers_and_barrier<0>();
#pragma unroll
        for (int s = 0; s < 4; s++) read_b(s, 0);
        a = convert_raw_half<FM, GS, 0>(raw[0]);
        load_raw(Half1{}, 0, u0);
        for (uint32_t u = u0; u < u1; u++) {
            chunk(Half0{}, 2 * u);
            chunk(Half1{}, 2 * u + 1);
        }
    }
    wait_transfers_and_barrier<0>(); // nothing is on its way to LDS any more, and nobody reads operands

    // output: as in the other tile kernels, through LDS; the row scales are asked for here, one round trip at the end of a long K loop
    v4h sc4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const half_t *p = scales + (R0 + r) * 16 + 4 * q;
        sc4[r] = (v4h){ p[0], p[1], p[2], p[3] };
    }
    if (splitK == 1) {
        tile_park<FM, NT, RT, 2, half_t>(acc, sc4, lds + (size_t)wc * NT * 16 * (2 * RT * 16 * 2 + 16), wr, col, q, ws ? bias_of(ws) + mb * (2 * RT * 16) : nullptr);
        __syncthreads();
        tile_flush<2 * NT, RT, 2, 4 * kWave, half_t>(C, lds, M, N, mb, nbase, tid);
    } else {
        // fp32 partial sums in two turns, one half of the columns each: both at once would not fit LDS
        float *out = ws + (size_t)split * N * M;
#pragma unroll
        for (int part = 0; part < 2; part++) {
            if (wc == part) tile_park<FM, NT, RT, 2, float>(acc, sc4, lds, wr, col, q);
            __syncthreads();
            tile_flush<NT, RT, 2, 4 * kWave, float>(out, lds, M, N, mb, nbase + part * NT * 16, tid);
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// gemm_wide: the tile GEMM of large batches, wavefronts one below the other across the whole width of the tile.
//   workgroup = 4 x WK wavefronts; tile = (4*RT*16) rows x (NT*16) columns, (RT*16) x (NT*16) of it per wavefront; grid as gemm_tile
// A chip full of MFMAs is held by its power, not by its clock: registers only, 16x16x32 MFMAs of zeros run at 2.39 GHz = 2.47 PFLOP/s, of random halfs at 1.78-1.93 GHz =
// 1.73-1.96, with one conversion for every 32 of them 1.79 PFLOP/s, for every 16 1.65, for every 8 1.38 (32x32x16 ones of random halfs at 1.56-1.73 GHz); and in 28672x8192
// N 2048 gemm_tile keeps the MFMAs busy for 0.57 of its cycles at 2.0 GHz, gemm_prefill 0.64 at 1.75, this kernel 0.75 at 1.57.  What a GEMM gets is then a matter of what
// it does beside them: conversions (64 cycles each, in which the SIMD starts no MFMA), operand reads from LDS, bytes from L2.  Here
//   * a converted fragment meets all NT column tiles: NT = 8 has one conversion per 32 MFMAs, where gemm_prefill, gemm_ws and 256 x 64 tiles have one per 16;
//   * a B operand read feeds RT row tiles: 4 in the 256-row tiles, where gemm_tile and gemm_ws have 2;
//   * no wavefront loads weights that another one loads, and 256 x 128 outputs share each byte of both operands.
// Weights go memory -> registers, activations memory -> LDS as in gemm_prefill.  K is walked in chunks of 128 columns (half a block), two stages in LDS,
// one barrier a chunk.  A chunk is eight half steps of RT * NT / 2 MFMAs, the B operands of the next half step being read meanwhile (across the barrier
// too).  All RT row tiles are converted at the top of a chunk; 256 x 128 then fills the register file (254-256), and the next raw codes are asked for when
// half of the converted fragments are used up.  With fewer outputs a second set of raw codes is a chunk and a half ahead.
// WK = 2 is for problems that do not fill the chip with two workgroups of four wavefronts to a CU: the second four take the other half of every K block (its
// odd chunks), with stages of their own, and hand their sums over through LDS at the end.
// Measured, us (FP6 e3m2, the best of gemm_tile 256 x 128, gemm_prefill and gemm_ws 256 x 64 -> here): 28672x8192 N 2048 759 -> 645 (1.49 PFLOP/s),
// 8192x8192 N 4096 453 -> 381, N 1024 116 -> 109, N 512 60.3 -> 57.9 (WK 2); 11008x4096 N 1500 132 -> 110 (256 x 96), 4096x4096 N 1024 30.5 -> 28.9; FP5 with
// group exponents 4608x4544 N 777 38.3 -> 33.1, 8192x8192 N 1024 114 -> 103.  One card to another differs by 4 %.
// Tried and left out (28672x8192 N 2048 / 8192x8192 N 512): s_setprio around the MFMAs (+ 0.5 %), no scheduling fence between half steps (+ 0.5 %, spills with
// group exponents), non-temporal weights (+ 5 %), panels of 2048 rows (level), conversions of two row tiles' quarters at once (level; with group exponents + 10 %),
// WK 2 there (+ 4 %); a ring of four stages of 64 columns (level / + 1 %: what is in flight is not the bound, a kernel that only transfers the second one's
// bytes takes 36 us).
// ---------------------------------------------------------------------------------------------------------------
template <int FM, bool GS, int NT, int RT, int WK>
__global__ __launch_bounds__(4 * WK *kWave, RT *NT <= 8 ? 4 : 2) void gemm_wide(const uint8_t *W, const half_t *__restrict__ scales, const uint8_t *gexp, const half_t *X,
                                                            half_t *__restrict__ C, float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                            uint32_t units, uint32_t splitK, uint32_t nblocks)
{
#include "fp6mi_wide_tile.inc"
}

// gemm_span: the same organisation with the tile widths between gemm_wide's: 128 x 48, 128 x 80, 128 x 112, 256 x 80 and 256 x 112, and 256 x 96 with the halves of K
// side by side, all of eight wavefronts.  What bounds a GEMM of some hundred columns is the same as there, and on top of it what the tile grid adds: columns that no tile
// is full of (777 columns are 7 tiles of 128 or of 112), a last round of few workgroups, and CUs with a single workgroup of four wavefronts.  A half step holds (NT + 1) / 2
// column tiles, the other one NT / 2.  Measured, us, what is launched without it -> here: e2m2 with group exponents 4608x4544 N 777 34.0 -> 31.3 (128 x 112), e2m1 20736x4992 N 142
// 39.9 -> 33.6 (128 x 48), e2m2 3584x3200 N 1293 37.2 -> 31.2 and e3m2 17408x7168 N 196 70.7 -> 62.8 (256 x 80), 8192x4992 N 445 40.8 -> 39.4 (128 x 112), e2m2 4864x5632
// N 1067 60.3 -> 53.8 (256 x 96).  256 x 112 takes all 256 registers with 6-bit weights and spills one, with group exponents eleven: written once a launch, of which one, four or seven
// are read back every two K blocks, between a barrier and the chunk's transfers (no counted wait sees them).  Left out: 256 x 48, 256 x 64, 256 x 80 and 256 x 112 of four wavefronts and 256 x 48, 256 x 64 of eight (0.4 % over all problems
// measured), and the same tiles for 33 to 96 columns (88 problems, the best of them with what there is: 0.990).
template <int FM, bool GS, int NT, int RT, int WK>
__global__ __launch_bounds__(4 * WK *kWave, RT == 2 && NT <= 4 ? 4 : 2) void gemm_span(const uint8_t *W, const half_t *__restrict__ scales, const uint8_t *gexp, const half_t *X,
                                                            half_t *__restrict__ C, float *__restrict__ ws, uint32_t M, uint32_t N, uint32_t K,
                                                            uint32_t units, uint32_t splitK, uint32_t nblocks)
{
#include "fp6mi_wide_tile.inc"
}

// Native layout -> fp16 [M,K], with the GEMM's own conversion code.  One lane per (row tile, K block, lane) triple.
// Bound by its writes, two thirds to four fifths of the bytes.  A lane holds eight columns of a row: stored as they are, a wavefront writes 64 bytes into each of 16 rows, half
// lines that meet their other half in L2.  So its block passes through LDS (its own part, no barrier) and leaves two whole rows of 512 bytes at a time.
// How they leave: what was written is read next, by a GEMM as a rule.  Up to 224 MiB (kDequantKept) the stores are written through L2 and stay in the 256 MiB of the memory-side
// cache; larger outputs go past the caches.  us, e3m2, alone and with the F.linear over N rows right behind: half lines / plain stores of rows / past the caches / written through:
//   4096x4096  9.9 / 8.8 / 8.5 / 8.4, N 512 36.8 / 36.5 / 40.9 / 37.0        3584x8128 19.1 / 16.1 / 14.8 / 15.2, N 1024 84.4 / 81.5 / 95.1 / 80.9
//   8192x8192  35.0 / 30.8 / 32.8 / 28.9, N 512 102.6 / 99.4 / 108.4 / 96.8  14336x8192 (224 MiB) 56.0 / 50.1 / 54.3 / 47.9, N 256 129 / 124 / 145 / 121, N 512 177 / 176 / 163 / 174
//   16384x8192 62.6 / 56.2 / 61.2 / 53.8, N 512 203 / 204 / 181 / 201        28672x8192 124 / 111 / 105 / 104, N 512 308 / 299 / 285 / 299
constexpr size_t kDequantKept = (size_t)224 << 20;
template <int FM, bool GS>
__global__ __launch_bounds__(256) void dequant_native(half_t *__restrict__ out, const uint8_t *__restrict__ W, const half_t *__restrict__ scales,
                                                     const uint8_t *__restrict__ gexp, uint32_t M, uint32_t K, uint32_t units, uint32_t kept)
{
    constexpr int  kRow = 528; // 16 bytes of padding: the reads of the 16 rows of a column start in different banks
    __shared__ __attribute__((aligned(16))) uint8_t stage[4][16 * kRow];
    const int      lane = threadIdx.x & 63;
    const uint32_t blk = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= (M / 16) * units) return;
    const uint32_t R = blk / units, U = blk % units;
    const int      m = lane & 15, q = lane >> 4;
    WFrag<FM>      wf = load_wfrag<FM>(W + (size_t)blk * Fmt<FM>::block_bytes, lane);
    AOps<FM>       a;
    convert<FM, GS>(wf, a, load_group_exps<GS>(gexp, blk, lane));
    const half_t sc = scales[R * 16 + m], post = (half_t)Fmt<FM>::post_scale;
    uint8_t *mine = stage[threadIdx.x >> 6];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        v8h v = a.s[s];
        if (Fmt<FM>::post_scale != 1.0f) v = v * post; // exact: a power of two, results are at most 7
        v = v * sc;                                    // one round-to-nearest-even, like fp16_rn(value * scale)
        *reinterpret_cast<v8h *>(mine + m * kRow + 64 * s + 16 * q) = v;
    }
    // The reads below are of other lanes' writes.  The LDS unit serves a wavefront in order, so no instruction is needed, but the compiler has to leave them in this order.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t k = U * 256 + 8 * (lane & 31);
    auto           row = [&](int r) { return *reinterpret_cast<const v4u *>(mine + r * kRow + 16 * (lane & 31)); };
    if (kept) {
        constexpr int kWriteThrough = 16; // sc1: the scope is the device
        const auto    obuf = __builtin_amdgcn_make_buffer_rsrc(out, 0, (int)(M * K * 2), 0x00027000);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t r = 2 * i + (lane >> 5);
            const v4u      v = row(r);
            if (k < K) __builtin_amdgcn_raw_buffer_store_b128(v, obuf, ((R * 16 + r) * K + k) * 2, 0, kWriteThrough);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int r = 2 * i + (lane >> 5);
            const v4u v = row(r);
            if (k < K) __builtin_nontemporal_store(v, reinterpret_cast<v4u *>(out + (size_t)(R * 16 + r) * K + k));
        }
    }
}

// Writes one lane's two 192-bit strings of 6-bit fields (MFMA steps 0..3 and 4..7 of a K block, in the order the conversion
// instruction reads them) into a native block: 12 (6-bit formats), 10 (FP5) or 8 (FP4) dwords at the places of lane `slot`.
// FP5 and FP4 park the payload bits of the last one or two dwords of a string in the fixed-zero bits of the others.  The stores
// leave the caches to what the quantizer reads twice (5-12 % off it at 4096x4096 and 8192x28672).
template <int FM> __device__ __forceinline__ void store_native_strings(v6u s0, v6u s1, uint8_t *dst, int slot)
{
    v4u *d4 = reinterpret_cast<v4u *>(dst) + slot;
    if constexpr (Fmt<FM>::bits == 6) {
        __builtin_nontemporal_store((v4u){ s0[0], s0[1], s0[2], s0[3] }, d4);
        __builtin_nontemporal_store((v4u){ s0[4], s0[5], s1[0], s1[1] }, d4 + 64);
        __builtin_nontemporal_store((v4u){ s1[2], s1[3], s1[4], s1[5] }, d4 + 128);
    } else if constexpr (Fmt<FM>::bits == 5) {
        constexpr uint32_t A = 0x10410410u, B = 0x04104104u, C = 0x41041041u;
        auto fold = [&](v6u D) { return (v4u){ D[0] | (D[5] & A), D[1] | (D[5] & B), D[2] | ((D[5] >> 1) & C), D[3] | ((D[5] >> 1) & A) }; };
        __builtin_nontemporal_store(fold(s0), d4);
        __builtin_nontemporal_store(fold(s1), d4 + 64);
        __builtin_nontemporal_store((v2u){ s0[4] | ((s0[5] >> 1) & B), s1[4] | ((s1[5] >> 1) & B) }, reinterpret_cast<v2u *>(dst + 2048) + slot);
    } else {
        constexpr uint32_t P = 0xC30C30C3u, Q = 0x30C30C30u, R = 0x0C30C30Cu;
        auto fold = [&](v6u D) { return (v4u){ D[0] | (D[4] & P), D[1] | (D[5] & Q), D[2] | (D[4] & R), D[3] | (D[5] & P) }; };
        __builtin_nontemporal_store(fold(s0), d4);
        __builtin_nontemporal_store(fold(s1), d4 + 64);
    }
}

// Reference layout -> native layout on the device, HBM-bound (reads and writes the weight bytes once).  One workgroup per 64-row
// tile of the reference and K block of 256 columns, one wavefront per 16-row block of the tile; lane = (m = l%16, q = l/16) as in
// the GEMM.  The segment words of a (16 rows x 16 columns) piece are 32 consecutive ones, word 4*(m%8) + t holding columns 2t,
// 2t+1, 2t+8, 2t+9 of rows m%8 and m%8 + 8.  So the eight columns 8q'..8q'+7 that a lane needs of a piece for one MFMA step are
// the four words from 4*(m%8) on, one 16-byte load per segment array (a quarter-wavefront reads one 128-byte line), and in each word its two
// codes sit 16 bits apart at a position that depends on the lane alone: a shift and a mask bring both out at once.  The whole block
// is in flight before the first use.  11008x4096 FP6: 12.0 us = 5.6 TB/s read + written, where one bit piece per load, a byte array per
// lane in scratch memory and a loop over its 64 codes took 266 us.
template <int FM>
__global__ __launch_bounds__(256) void relayout_ref_to_native(uint8_t *__restrict__ native, const uint8_t *__restrict__ ref,
                                                             uint32_t M, uint32_t K, uint32_t units)
{
    // segment arrays: 6 bits = [2-bit | 4-bit], 5 bits = [1-bit | 4-bit], 4 bits = [4-bit]
    constexpr int  bits = Fmt<FM>::bits, kHiWords = bits == 6 ? 64 : 32; // words of the high segment per 64-row tile and 16 columns
    const int      lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
    const uint32_t block = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x / units, U = blockIdx.x % units, g = m & 7, rowhalf = m >> 3;
    const uint32_t slices = K >> 4;
    const uint32_t *seg_hi = reinterpret_cast<const uint32_t *>(ref) + (size_t)tile * slices * kHiWords + (bits == 6 ? (block >> 1) * 32 : 0) + 4 * g;
    const uint32_t *seg4   = reinterpret_cast<const uint32_t *>(ref + (size_t)M * K * (bits - 4) / 8) + (size_t)tile * slices * 128 + block * 32 + 4 * g;

    v4u lo[8], hi[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const uint32_t slice = U * 16 + 2 * s + (q >> 1); // K is a multiple of 64: a 16-column piece lies inside K or beyond it
        const bool     in = slice < slices;
        lo[s] = in ? *reinterpret_cast<const v4u *>(seg4 + (size_t)slice * 128) : (v4u){ 0u, 0u, 0u, 0u };
        if constexpr (bits != 4) hi[s] = in ? *reinterpret_cast<const v4u *>(seg_hi + (size_t)slice * kHiWords) : (v4u){ 0u, 0u, 0u, 0u };
    }
    // positions inside a word of the code at the even column (the odd column's is 16 bits above); e = index of the pair among the
    // four pairs (row half, column half) of a word
    const uint32_t e = rowhalf + 2 * (q & 1);
    const uint32_t sh4 = (0x048Cu >> (4 * ((e & 1) * 2 + (e >> 1)))) & 15u; // e = 0, 1, 2, 3: 12, 4, 8, 0
    uint32_t       sh_hi = 0;
    if constexpr (bits == 6) { // 2-bit fields from the top of the word: field 8, 12, 9, 13, 10, 14, 11, 15 for pair 4*(block%2) + e
        const uint32_t pair = (block & 1) * 4 + e;
        sh_hi = 30 - 2 * (8 + (pair >> 1) + 4 * (pair & 1));
    }
    if constexpr (bits == 5) // bits from the top of the word: bit 16 or 24, plus 2*block + column half
        sh_hi = 31 - (16 + 8 * rowhalf + 2 * block + (q & 1));

    v6u str[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        uint32_t p[16]; // pairs of 6-bit fields
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                uint32_t c = (lo[4 * h + s][t] >> sh4) & 0x000F000Fu; // two codes (their low four bits), 16 bits apart
                if constexpr (bits == 6) c |= ((hi[4 * h + s][t] >> sh_hi) & 0x00030003u) << 4;
                if constexpr (bits == 5) c |= ((hi[4 * h + s][t] >> sh_hi) & 0x00010001u) << 5; // the fixed-zero bit goes in above the exponent
                if constexpr (bits == 4) c <<= 2;                                               // and here two below the mantissa
                p[4 * s + t] = (c | (c >> 10)) & 0xFFFu;
            }
#pragma unroll
        for (int k = 0; k < 2; k++) { // eight pairs = three dwords
            const uint32_t *v = p + 8 * k;
            str[h][3 * k]     = v[0] | v[1] << 12 | v[2] << 24;
            str[h][3 * k + 1] = v[2] >> 8 | v[3] << 4 | v[4] << 16 | v[5] << 28;
            str[h][3 * k + 2] = v[5] >> 4 | v[6] << 8 | v[7] << 20;
        }
    }
    store_native_strings<FM>(str[0], str[1], native + ((size_t)(tile * 4 + block) * units + U) * Fmt<FM>::block_bytes, lane);
}

// ---------------------------------------------------------------------------------------------------------------
// Quantizer on the device: float weights [M,K] (fp16, bf16 or fp32) -> per-row fp16 scales + native-layout FPx codes.
// Gives the bits of the host quantizer of this package, which computes in double precision:
//   scale[row] = fp16_rn(absmax(row) / max_value) (1.0 where that rounds to zero), computed from a double quotient;
//   code       = nearest representable magnitude to |w / scale| (clamped at max_value), ties to the even code, with the sign
//                bit of w.  NaN weights become +0, +-Inf saturates, and neither takes part in absmax.
// (The reference's only quantizer truncates and is not wired to any API: fp6_llm/csrc/utils/weight_quant.h:9-105.)
//
// The codes come from single precision and the packing conversion instruction (v_cvt_scalef32_2xpk16_bf6/fp6_f32: 32 floats to
// 32 fields, round to nearest even, saturating), and are exact all the same.  A code changes where |w| = t * scale, t a
// midpoint of at most 5 significant bits; t * scale has at most 16 bits.  A quotient computed as q = |w| * (1/scale)
// followed by one residual step q += fma(-q, scale, |w|) * (1/scale) is within a hair over half an ulp of the true one, and exact where
// the quotient is a midpoint.  A 16-bit w that is not on a boundary is at least 2^-16 away from it (relative), so q stays on
// its side.  A 24-bit w can be as near as 2^-24, where q might round onto the midpoint: for fp32 weights the sign of a second
// residual turns q into the quotient rounded to odd (truncated, last bit set if inexact), which never sits on a midpoint.
//
// HBM-bound but for its arithmetic, which does not hide: a chip's worth of workgroups loads, finds its maxima and converts in step.  Clamps, NaN tests and
// sign handling made that 10 operations a weight (17 us of 46 at 8192x8192); they are left to the wavefronts that have met an Inf, a NaN or a
// scale that is no normal number, the others take 5 (quantize_string's PLAIN).  us, e3m2, before -> now, row scales and group exponents: bf16 8192x8192
// 45.9 -> 41.9, 49.6 -> 44.0; 3072x8192 23.5 -> 18.9, 26.1 -> 20.7; 28672x8192 141 -> 136, 142 -> 137; 8192x28672 176 -> 165, 183 -> 176; fp16 8192x8192
// 47.1 -> 43.1, 51.6 -> 45.2; fp32 8192x8192, then with two blocks kept, 95.2 -> 87.6, 98.7 -> 91.9 (another card than below).
//
// Two organisations of the same arithmetic.  quant_fused: one workgroup of eight wavefronts per 16-row tile reads
// its rows, finds the scales, and converts; the last two blocks of every wavefront (three of 32-bit weights) are still in its registers then, with 16-bit
// weights the one before them in LDS, and the others are read again, latest first (8192x8192: a quarter of the weights twice).
// quant_row_scales + quant_blocks: a workgroup takes a row, then a wavefront a block, and all weights are read twice.
// Measured, us, e3m2, fused / two kernels (replayed from a graph, through more memory than the caches hold; the fp32 columns, both sides of them, on another card than the bf16 ones):
//               bf16            bf16 groups     fp32            fp32 groups
//   1024x3072     6.4 /   7.9     7.4 /   8.2     8.5 /  10.2     9.7 /  10.4
//   1024x4096     7.6 /   8.3     9.2 /   8.6    10.6 /  11.2    11.7 /  11.4
//   1536x4096     8.0 /   9.9     9.6 /  10.4    12.8 /  14.1    14.0 /  14.3
//   2048x4096     8.9 /  11.0    10.2 /  11.5    14.7 /  17.0    15.7 /  17.1
//   2048x6144    12.3 /  13.5    13.9 /  14.1    19.2 /  22.5    19.8 /  22.6
//   2048x8192    15.6 /  16.2    18.9 /  16.6    25.7 /  26.9    27.5 /  27.3
//   2560x8192    16.8 /  19.3    19.6 /  19.7    28.8 /  33.1    31.2 /  33.1
//   2816x16384   36.0 /  37.3    40.0 /  37.9    61.7 /  68.1    64.0 /  66.1
//   4096x8192    23.1 /  28.7    24.8 /  29.5    43.8 /  49.9    45.3 /  48.3
//   8192x8192    42.9 /  52.7    45.0 /  52.7    85.3 /  93.7    87.5 /  90.1
//   4096x28672   85.8 /  89.4    89.9 /  89.6   158 / 174       157 / 173
//  16384x4096    37.2 /  53.6    38.8 /  53.7    71.4 /  93.5    75.8 /  91.6
// Few workgroups do not pull enough from memory to pay for a second pass over a long row: fused from 160 tiles on, and below that up to K = 3072 or three
// times the rows.  On the wrong side of that line bf16 of 1024x4096 (9 %) and 2048x8192 (4 %), 16-bit weights with group exponents of 2816x16384 (6 %) and fp32 of 1024x4096 (6 %) and 2048x8192 (5 %).
// (16-bit weights: a block of every wavefront in LDS and two in registers leave room for two workgroups to a CU.  Three in registers and one in LDS, nothing
// read twice at 8192 columns, were slower with one workgroup to a CU, and held to 128 registers they spill.
// 32-bit weights, of which two blocks take 202 registers: a CU holds one workgroup either way, so a third block, 64 registers, takes the other 54 and spills eight, which are
// written once and read back once a row tile, around the search for its maxima (36 bytes of scratch a lane; the loops over blocks touch none).  us, e3m2, two blocks -> three:
// 4096x6144 29.8 -> 25.2, 14336x6144 99.8 -> 88.6, 8192x8192 95.6 -> 85.3, 8192x11008 114 -> 108, 8192x28672 316 -> 306; up to 4096 columns, where no
// wavefront has a third, within 1 %.  A block of 16 KB in LDS beside two gives the same, beside three it costs 10 % but at 8192 columns.)
// A conversion in double precision, code by code through a byte array in scratch memory, took 532 us at 8192x8192.
// ---------------------------------------------------------------------------------------------------------------
struct bf16_t { uint16_t bits; };
typedef short v2s __attribute__((ext_vector_type(2)));

// Eight consecutive weights as loaded, their widening, and a running maximum of their magnitudes: magnitude bits order like the values, with Inf and NaN above
// all others.  A wavefront that has met one of these (`special`) goes over its weights once more with `add_finite`, which lets them pass by.
template <typename T> struct WeightPiece {
    v4u x;
    __device__ __forceinline__ void load(const T *p) { x = *reinterpret_cast<const v4u *>(p); }
    __device__ __forceinline__ void zero() { x = (v4u){ 0u, 0u, 0u, 0u }; }
    __device__ __forceinline__ float value(int j) const
    {
        const uint32_t w = x[j >> 1];
        if constexpr (std::is_same<T, bf16_t>::value)
            return __builtin_bit_cast(float, j & 1 ? w & 0xFFFF0000u : w << 16);
        else
            return (float)__builtin_bit_cast(half_t, (uint16_t)(j & 1 ? w >> 16 : w));
    }
};
template <> struct WeightPiece<float> {
    v4u x, y;
    __device__ __forceinline__ void load(const float *p) { x = *reinterpret_cast<const v4u *>(p), y = *reinterpret_cast<const v4u *>(p + 4); }
    __device__ __forceinline__ void zero() { x = y = (v4u){ 0u, 0u, 0u, 0u }; }
    __device__ __forceinline__ float value(int j) const { return __builtin_bit_cast(float, j < 4 ? x[j] : y[j - 4]); }
};
template <typename T> struct MaxMagnitude {
    typedef unsigned short v2us __attribute__((ext_vector_type(2)));
    static constexpr uint16_t kInf = std::is_same<T, bf16_t>::value ? 0x7F80 : 0x7C00;
    v2us                      m = { 0, 0 };
    __device__ __forceinline__ void add(const WeightPiece<T> &p)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) m = __builtin_elementwise_max(m, __builtin_bit_cast(v2us, p.x[i] & 0x7FFF7FFFu));
    }
    __device__ __forceinline__ void add_finite(const WeightPiece<T> &p)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const v2us a = __builtin_bit_cast(v2us, p.x[i] & 0x7FFF7FFFu);
            m = __builtin_elementwise_max(m, (v2us){ a[0] < kInf ? a[0] : (uint16_t)0, a[1] < kInf ? a[1] : (uint16_t)0 });
        }
    }
    __device__ __forceinline__ uint16_t top() const { return m[0] > m[1] ? m[0] : m[1]; }
    __device__ __forceinline__ bool     special() const { return top() >= kInf; }
    __device__ __forceinline__ float    value() const
    {
        if constexpr (std::is_same<T, bf16_t>::value)
            return __builtin_bit_cast(float, (uint32_t)top() << 16);
        else
            return (float)__builtin_bit_cast(half_t, top());
    }
};
template <> struct MaxMagnitude<float> {
    static constexpr uint32_t kInf = 0x7F800000u;
    uint32_t                  m = 0;
    __device__ __forceinline__ void add(const WeightPiece<float> &p)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) m = max(m, max(p.x[i] & 0x7FFFFFFFu, p.y[i] & 0x7FFFFFFFu));
    }
    __device__ __forceinline__ void add_finite(const WeightPiece<float> &p)
    {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t a = (i < 4 ? p.x[i & 3] : p.y[i & 3]) & 0x7FFFFFFFu;
            m = max(m, a < kInf ? a : 0u);
        }
    }
    __device__ __forceinline__ bool  special() const { return m >= kInf; }
    __device__ __forceinline__ float value() const { return __builtin_bit_cast(float, m); }
};

// round-to-nearest-even of a non-negative double to fp16 without passing through float (no double rounding)
__device__ __forceinline__ half_t half_rn_from_double(double q)
{
    if (!(q > 0.0)) return (half_t)0.0f;
    int e = ilogb(q);                               // q = 1.xxx * 2^e
    int ulp_exp = (e < -14 ? -14 : e) - 10;          // fp16 spacing at q (subnormals share the spacing 2^-24)
    double r = rint(scalbn(q, -ulp_exp));            // exact scaling, then round to nearest even integer
    double v = scalbn(r, ulp_exp);                   // representable in fp16 unless it overflows
    return v >= 65520.0 ? (half_t)__builtin_inff() : (half_t)(float)v;
}
template <int FM> __device__ __forceinline__ half_t row_scale(float amax)
{
    const half_t sc = half_rn_from_double((double)amax / Fmt<FM>::max_value);
    return (float)sc == 0.f ? (half_t)1.0f : sc;
}

// FP4's coarser grid (steps of 1/2 below 2, 1 below 4, 2 above), on which values are exact in the fields
__device__ __forceinline__ float fp4_grid(float q)
{
    const float magic = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, __builtin_fmaxf(__builtin_fabsf(q), 1.f)) & 0x7F800000u) * 6291456.f; // 1.5 * 2^23 steps
    return (q + magic) - magic;
}

// The 32 weights of one field string (four pieces of eight) against the scale f -> their 6-bit fields.
// PLAIN: the weights are finite and the row's scale is a normal fp16 number, so that no quotient is beyond the largest code by more than the rounding of the
// scale (2^-11, which rounds to that code), and the arithmetic carries signs by itself: the residual is taken as q * f - w, whose exact zero leaves a
// quotient of -0 alone.  Three operations a 16-bit weight instead of eight.
template <int FM, typename T, bool PLAIN> __device__ __forceinline__ v6u quantize_string(const WeightPiece<T> *p, float f)
{
    typedef float v16f __attribute__((ext_vector_type(16)));
    // the fields of FP5 hold a quarter of the value (its grid up to 7 is the e3m2 grid up to 1.75, times 4)
    constexpr float top = (float)Fmt<FM>::max_value / Fmt<FM>::post_scale, kInf = __builtin_inff();
    f *= Fmt<FM>::post_scale;
    const bool  overflown = !PLAIN && f == kInf; // a row whose scale left fp16: finite weights become zeros
    const float rf = overflown ? 0.f : 1.0f / f, fd = overflown ? 0.f : f, limit = overflown ? 3.4028234663852886e38f : kInf;
    v16f        even, odd;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        const float w = p[i >> 3].value(i & 7);
        float       q;
        if constexpr (PLAIN) {
            q = w * rf;
            q = __builtin_fmaf(-__builtin_fmaf(q, fd, -w), rf, q);
            if constexpr (std::is_same<T, float>::value) {
                const float r = __builtin_fmaf(-q, fd, w);
                uint32_t    u = __builtin_bit_cast(uint32_t, q);
                if ((int)(__builtin_bit_cast(uint32_t, r) ^ u) < 0) u -= 1;
                q = r != 0.f ? __builtin_bit_cast(float, u | 1u) : q;
            }
            if constexpr (Fmt<FM>::bits == 4) q = __builtin_copysignf(fp4_grid(q), w);
        } else {
            const float a = __builtin_fabsf(w);
            q = __builtin_fminf(a * rf, 2.f * top);
            q = __builtin_fminf(__builtin_fmaf(__builtin_fmaf(-q, fd, a), rf, q), top);
            if constexpr (std::is_same<T, float>::value) {
                const float r = __builtin_fmaf(-q, fd, a);
                uint32_t    u = __builtin_bit_cast(uint32_t, q);
                if (r < 0.f) u -= 1;
                if (r != 0.f) u |= 1;
                q = __builtin_bit_cast(float, u);
            }
            if constexpr (Fmt<FM>::bits == 4) q = fp4_grid(q);
            q = a <= limit ? __builtin_copysignf(q, w) : 0.f; // NaN: +0
        }
        if (i & 1)
            odd[i >> 1] = q;
        else
            even[i >> 1] = q;
    }
    if constexpr (Fmt<FM>::hw_e3m2)
        return __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(even, odd, 1.0f);
    else
        return __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, 1.0f);
}
// (wave-uniform) whether every row of a wavefront's block has a scale of the PLAIN kind
__device__ __forceinline__ bool plain_scales(float sc) { return __all(sc >= 6.103515625e-5f && sc < __builtin_inff()); }

// A lane of the quantizer is (m = l/4, p = l%4): the four lanes of a row read 64 or 128 consecutive bytes, and its codes go to the places
// of lane (m, q = p) of the native block.  w points at the tile's first row.
template <typename T> __device__ __forceinline__ void load_quant_block(WeightPiece<T> (&x)[8], const T *w, uint32_t K, uint32_t U, int lane)
{
    const T *p = w + (size_t)(lane >> 2) * K + (size_t)U * 256 + 8 * (lane & 3);
#pragma unroll
    for (int s = 0; s < 8; s++) x[s].zero();
    if (U * 256 + 256 <= K) { // (uniform) one branch for all but the block that K cuts
#pragma unroll
        for (int s = 0; s < 8; s++) x[s].load(p + 32 * s);
    } else {
#pragma unroll
        for (int s = 0; s < 6; s += 2) // K is a multiple of 64
            if (U * 256 + 32 * s < K) x[s].load(p + 32 * s), x[s + 1].load(p + 32 * s + 32);
    }
}
// GROUPS: every group of 128 columns of a row also gets the smallest factor 2^k, -15 <= k <= 0, that still holds its largest
// magnitude, stored as the byte 127 + k, and its codes are chosen against scale * 2^k.  max_value * scale has at most 14 significant bits, so
// comparing amax with it (by exponent, then by mantissa) decides like the double quotient amax / scale against max_value * 2^k.
template <int FM, typename T, bool GROUPS, bool PLAIN>
__device__ __forceinline__ void quantize_block(const WeightPiece<T> (&x)[8], float sc, uint8_t *native, uint8_t *gexp, size_t blk, uint32_t K, uint32_t U, int lane)
{
    v6u str[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float f = sc;
        if constexpr (GROUPS) {
            MaxMagnitude<T> mm;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if constexpr (PLAIN)
                    mm.add(x[4 * h + s]);
                else
                    mm.add_finite(x[4 * h + s]);
            }
            float amax = mm.value();
            amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
            amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
            const float t = (float)Fmt<FM>::max_value * sc;
            int         k = __builtin_amdgcn_frexp_expf(amax) - __builtin_amdgcn_frexp_expf(t) + (__builtin_amdgcn_frexp_mantf(amax) > __builtin_amdgcn_frexp_mantf(t) ? 1 : 0);
            if (amax == 0.f || t == __builtin_inff()) k = -15;
            k = k < -15 ? -15 : k > 0 ? 0 : k;
            if (U * 256 + 128 * h >= K) k = 0; // a half block beyond K: factor 1 by convention
            f = ldexpf(sc, k);
            if ((lane & 3) == 0) gexp[(blk * 16 + (lane >> 2)) * 2 + h] = (uint8_t)(127 + k);
        }
        str[h] = quantize_string<FM, T, PLAIN>(x + 4 * h, f);
        __builtin_amdgcn_sched_barrier(0); // one string's 32 quotients at a time
    }
    store_native_strings<FM>(str[0], str[1], native + blk * Fmt<FM>::block_bytes, (lane >> 2) + 16 * (lane & 3));
}

// One block more of every wavefront waits in LDS, where a row has more than KEEP of them a wavefront and the weights 16 bits (64 KB; for the
// 128 KB of 32-bit ones see above).  It goes there straight from memory, lane l to byte 16 * l of its piece.
template <typename T, int WAVES> constexpr uint32_t quant_stash_bytes() { return sizeof(T) == 2 ? WAVES * 8 * 1024 : 0; }

template <int FM, typename T, bool GROUPS, int WAVES, int KEEP>
__global__ __launch_bounds__(WAVES *kWave, sizeof(T) == 2 ? WAVES / 2 : 1) void quant_fused(uint8_t *__restrict__ native, half_t *__restrict__ scales, uint8_t *__restrict__ gexp,
                                                            const T *__restrict__ Wf, uint32_t K, uint32_t units)
{
    __shared__ float  wave_max[WAVES][16];
    __shared__ half_t tile_scale[16];
    const int         lane = threadIdx.x & 63;
    const uint32_t    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), R = blockIdx.x;
    const T          *w = Wf + (size_t)R * 16 * K;

    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef __attribute__((address_space(1))) void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;

    // blocks wave, wave + WAVES, ...; the last KEEP of them stay in registers (kept[0] is the very last), the one before them in LDS
    const uint32_t  mine = wave < units ? (units - wave + WAVES - 1) / WAVES : 0;
    MaxMagnitude<T> mm;
    WeightPiece<T>  kept[KEEP][8];
    constexpr bool  kStash = quant_stash_bytes<T, WAVES>() != 0;
    const bool      stash = kStash && mine > KEEP;
    const uint32_t  held = KEEP + (stash ? 1 : 0);
    uint8_t *const  area = lds + wave * (8 * 1024);
    if (stash) { // (never the block that K cuts: that is the last one of the row, and the last of its wavefront)
        const T *p = w + (size_t)(lane >> 2) * K + (size_t)(wave + (mine - 1 - KEEP) * WAVES) * 256 + 8 * (lane & 3);
#pragma unroll
        for (int s = 0; s < 8; s++) __builtin_amdgcn_global_load_lds((gvoid *)(p + 32 * s), (lvoid *)(area + s * 1024), 16, 0, 0);
    }
    for (uint32_t i = 0; i + held < mine; i++) {
        WeightPiece<T> x[8];
        load_quant_block<T>(x, w, K, wave + i * WAVES, lane);
#pragma unroll
        for (int s = 0; s < 8; s++) mm.add(x[s]);
    }
#pragma unroll
    for (int k = KEEP - 1; k >= 0; k--)
        if ((uint32_t)k < mine) load_quant_block<T>(kept[k], w, K, wave + (mine - 1 - k) * WAVES, lane);
#pragma unroll
    for (int k = KEEP - 1; k >= 0; k--)
        if ((uint32_t)k < mine) {
#pragma unroll
            for (int s = 0; s < 8; s++) mm.add(kept[k][s]);
        }
    auto stashed = [&](WeightPiece<T>(&x)[8]) {
        if constexpr (kStash)
#pragma unroll
            for (int s = 0; s < 8; s++) x[s].x = *reinterpret_cast<const v4u *>(area + s * 1024 + lane * 16);
    };
    if (stash) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the transfers into LDS; the loads above have been waited for
        WeightPiece<T> x[8];
        stashed(x);
#pragma unroll
        for (int s = 0; s < 8; s++) mm.add(x[s]);
    }
    const bool special = __any(mm.special());
    if (special) { // Inf or NaN among this wavefront's weights: once more, without them
        mm = MaxMagnitude<T>{};
#pragma unroll 1
        for (uint32_t i = 0; i < mine; i++) {
            WeightPiece<T> x[8];
            load_quant_block<T>(x, w, K, wave + i * WAVES, lane);
#pragma unroll
            for (int s = 0; s < 8; s++) mm.add_finite(x[s]);
        }
    }
    float amax = mm.value();
    amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
    if ((lane & 3) == 0) wave_max[wave][lane >> 2] = amax;
    __syncthreads();
    if (threadIdx.x < 16) {
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < WAVES; i++) a = fmaxf(a, wave_max[i][threadIdx.x]);
        const half_t sc = row_scale<FM>(a);
        tile_scale[threadIdx.x] = sc;
        scales[R * 16 + threadIdx.x] = sc;
    }
    __syncthreads();
    const float sc = (float)tile_scale[lane >> 2];
    // Both arithmetics at every block, chosen before it: a slow pass of its own over all blocks, behind the fast one, cost a wavefront a second reading of its weights
    // where one row of 16 has a scale below 2^-14.  us, e3m2, such a row in every tile, before the two arithmetics / with that pass / now: bf16 8192x8192
    // 45.8 / 65.4 / 45.4, 28672x4096 63.1 / 104 / 64.9; fp32 8192x8192 101 / 144 / 98.5; a NaN in every tile, bf16 8192x8192 45.9 / 51.4 / 46.5.
    const bool plain = !special && plain_scales(sc); // (uniform)
    auto       convert = [&](const WeightPiece<T>(&x)[8], uint32_t U) __attribute__((always_inline)) {
        if (plain) {
            quantize_block<FM, T, GROUPS, true>(x, sc, native, gexp, (size_t)R * units + U, K, U, lane);
        } else if constexpr (GROUPS || sizeof(T) != 2) {
            quantize_block<FM, T, GROUPS, false>(x, sc, native, gexp, (size_t)R * units + U, K, U, lane);
        } else { // (opaque copies: what both would widen alike is kept from being widened ahead of the branch, into registers that the held blocks need)
            WeightPiece<T> y[8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                y[s] = x[s];
                asm volatile("" : "+v"(y[s].x));
            }
            quantize_block<FM, T, GROUPS, false>(y, sc, native, gexp, (size_t)R * units + U, K, U, lane);
        }
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++)
        if ((uint32_t)k < mine) convert(kept[k], wave + (mine - 1 - k) * WAVES);
    if (stash) {
        WeightPiece<T> x[8];
        stashed(x);
        convert(x, wave + (mine - 1 - KEEP) * WAVES);
    }
    for (uint32_t i = mine > held ? mine - held : 0; i-- > 0;) {
        WeightPiece<T> x[8];
        load_quant_block<T>(x, w, K, wave + i * WAVES, lane);
        convert(x, wave + i * WAVES);
    }
}

template <int FM, typename T>
__global__ __launch_bounds__(256) void quant_row_scales(half_t *__restrict__ scales, const T *__restrict__ Wf, uint32_t K)
{
    __shared__ float wave_max[4];
    const T         *p = Wf + (size_t)blockIdx.x * K;
    MaxMagnitude<T>  mm;
#pragma unroll 4
    for (uint32_t k = threadIdx.x * 8; k < K; k += 2048) {
        WeightPiece<T> x;
        x.load(p + k);
        mm.add(x);
    }
    if (__any(mm.special())) { // Inf or NaN: once more, without them
        mm = MaxMagnitude<T>{};
        for (uint32_t k = threadIdx.x * 8; k < K; k += 2048) {
            WeightPiece<T> x;
            x.load(p + k);
            mm.add_finite(x);
        }
    }
    float amax = mm.value();
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) scales[blockIdx.x] = row_scale<FM>(fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3])));
}

template <int FM, typename T, bool GROUPS>
__global__ __launch_bounds__(256) void quant_blocks(uint8_t *__restrict__ native, const half_t *__restrict__ scales, uint8_t *__restrict__ gexp,
                                                   const T *__restrict__ Wf, uint32_t M, uint32_t K, uint32_t units)
{
    const int      lane = threadIdx.x & 63;
    const uint32_t blk = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blk >= (M / 16) * units) return;
    const uint32_t R = blk / units, U = blk % units;
    WeightPiece<T> x[8];
    load_quant_block<T>(x, Wf + (size_t)R * 16 * K, K, U, lane);
    const float     sc = (float)scales[R * 16 + (lane >> 2)];
    MaxMagnitude<T> mm;
#pragma unroll
    for (int s = 0; s < 8; s++) mm.add(x[s]);
    if (!__any(mm.special()) && plain_scales(sc))
        quantize_block<FM, T, GROUPS, true>(x, sc, native, gexp, blk, K, U, lane);
    else
        quantize_block<FM, T, GROUPS, false>(x, sc, native, gexp, blk, K, U, lane);
}
// ------------------------------------------------------------------------------------------------ launch helpers

// Lets `Kernel` use up to `bytes` of dynamic LDS.  The attribute belongs to the device's copy of the kernel: set once per device.
template <auto Kernel> int allow_dynamic_lds(size_t bytes)
{
    static std::atomic<uint64_t> attr_set{ 0 }; // bit d: done on device d; setting it twice is harmless, so no lock
    int                          dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
    const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;
    if (!(attr_set.load(std::memory_order_relaxed) & bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return (int)e;
        attr_set.fetch_or(bit, std::memory_order_relaxed);
    }
    return 0;
}

template <int FM, bool GS, int NT, int RT, int WAVES>
int launch_stream(hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M, size_t N, size_t K,
                  int splitK)
{
    constexpr size_t kMaxLds = (size_t)WAVES * stream_wave_bytes(16 * NT, RT, NT);
    static_assert(kMaxLds <= 160 * 1024, "the wavefronts' activation rows do not fit in LDS");
    uint32_t     units = (uint32_t)((K + 255) / 256);
    dim3         grid((uint32_t)((M / 16 + RT - 1) / RT), (uint32_t)splitK, (uint32_t)((N + 16 * NT - 1) / (16 * NT)));
    const size_t lds_bytes = NT == 1 && N <= 8 ? (size_t)WAVES * stream_wave_bytes(8, RT, NT) : kMaxLds;
    auto         go = [&](auto kernel_c) -> int {
        constexpr auto kernel = decltype(kernel_c)::value;
        if (kMaxLds > 48 * 1024)
            if (int rc = allow_dynamic_lds<kernel>(kMaxLds)) return rc;
        hipLaunchKernelGGL(kernel, grid, dim3(WAVES * kWave), lds_bytes, st, static_cast<const uint8_t *>(W), static_cast<const half_t *>(sc),
                           static_cast<const uint8_t *>(gexp), static_cast<const half_t *>(B), static_cast<half_t *>(C), ws, (uint32_t)M, (uint32_t)N,
                           (uint32_t)K, units, (uint32_t)splitK);
        return (int)hipGetLastError();
    };
    typedef decltype(&gemm_stream<FM, GS, NT, RT, WAVES, false, false>) Kernel;
    if (splitK > 1) return go(std::integral_constant<Kernel, &gemm_stream<FM, GS, NT, RT, WAVES, true, false>>{});
    if (ws) return go(std::integral_constant<Kernel, &gemm_stream<FM, GS, NT, RT, WAVES, false, true>>{});
    return go(std::integral_constant<Kernel, &gemm_stream<FM, GS, NT, RT, WAVES, false, false>>{});
}

template <int FM, bool GS, int NT, int RT, int WR, int WK>
int launch_tile(hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M, size_t N, size_t K,
                int splitK)
{
    constexpr int TN = NT * 16, TM = WR * RT * 16;
    constexpr size_t x_bytes = 2 * (size_t)WK * TN * kXsRowBytes, red_bytes = WK > 1 ? (size_t)WK * WR * RT * NT * 1024 : 0;
    constexpr size_t kLoopLds = x_bytes > red_bytes ? x_bytes : red_bytes, out_max = tile_stage_bytes<NT, RT, WR>(true);
    constexpr size_t kMaxLds = kLoopLds > out_max ? kLoopLds : out_max;
    static_assert(kMaxLds <= 160 * 1024, "tile does not fit in LDS");
    const size_t out_bytes = tile_stage_bytes<NT, RT, WR>(splitK > 1), lds_bytes = kLoopLds > out_bytes ? kLoopLds : out_bytes;
    if (M % TM) return FP6MI_ERR_SHAPE;
    uint32_t units = (uint32_t)((K + 255) / 256), nblocks = (uint32_t)((N + TN - 1) / TN);
    size_t   wgs = (M / TM) * (size_t)splitK * nblocks;
    if (wgs > 0x7fffffffu) return FP6MI_ERR_SHAPE;
    auto go = [&](auto kernel_c) -> int {
        constexpr auto kernel = decltype(kernel_c)::value;
        if (kMaxLds > 48 * 1024)
            if (int rc = allow_dynamic_lds<kernel>(kMaxLds)) return rc;
        hipLaunchKernelGGL(kernel, dim3((uint32_t)wgs), dim3(WR * WK * kWave), lds_bytes, st, static_cast<const uint8_t *>(W), static_cast<const half_t *>(sc),
                           static_cast<const uint8_t *>(gexp), static_cast<const half_t *>(B), static_cast<half_t *>(C), ws, (uint32_t)M, (uint32_t)N, (uint32_t)K,
                           units, (uint32_t)splitK, nblocks);
        return (int)hipGetLastError();
    };
    typedef decltype(&gemm_tile<FM, GS, NT, RT, WR, WK, false>) Kernel;
    if (ws && splitK == 1) return go(std::integral_constant<Kernel, &gemm_tile<FM, GS, NT, RT, WR, WK, true>>{});
    return go(std::integral_constant<Kernel, &gemm_tile<FM, GS, NT, RT, WR, WK, false>>{});
}
template <int FM, bool GS, int NT, int RT, int WR, int PW, int SW, int SX>
int launch_ws(hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M, size_t N, size_t K,
              int splitK)
{
    constexpr int    TN = NT * 16, TM = WR * RT * 16;
    constexpr size_t kLoopLds = ws_ring_bytes<FM, NT, RT, WR, SW, SX>() + ws_exps_ring_bytes<GS, RT, WR, SW>(), out_max = tile_stage_bytes<NT, RT, WR>(true);
    constexpr size_t kMaxLds = kLoopLds > out_max ? kLoopLds : out_max;
    static_assert(kMaxLds <= 160 * 1024, "the rings do not fit in LDS");
    static_assert((WR + PW) * kWave <= 1024, "too many wavefronts");
    // a weight stage must be a whole number of 1 KB transfers per loading wavefront (FP5 blocks are 2.5 KB: 64-row tiles are out)
    constexpr bool kDivides = (WR * RT * Fmt<FM>::block_bytes) % (1024 * PW) == 0 && (TN * 512) % (1024 * PW) == 0;
    if constexpr (!kDivides) {
        return FP6MI_ERR_SHAPE;
    } else {
        const size_t out_bytes = tile_stage_bytes<NT, RT, WR>(splitK > 1), lds_bytes = kLoopLds > out_bytes ? kLoopLds : out_bytes;
        if (M % TM) return FP6MI_ERR_SHAPE;
        if (kMaxLds > 48 * 1024)
            if (int rc = allow_dynamic_lds<&gemm_ws<FM, GS, NT, RT, WR, PW, SW, SX>>(kMaxLds)) return rc;
        uint32_t units = (uint32_t)((K + 255) / 256), nblocks = (uint32_t)((N + TN - 1) / TN);
        size_t   wgs = (M / TM) * (size_t)splitK * nblocks;
        if (wgs > 0x7fffffffu) return FP6MI_ERR_SHAPE;
        hipLaunchKernelGGL((gemm_ws<FM, GS, NT, RT, WR, PW, SW, SX>), dim3((uint32_t)wgs), dim3((WR + PW) * kWave), lds_bytes, st,
                           static_cast<const uint8_t *>(W), static_cast<const half_t *>(sc), static_cast<const uint8_t *>(gexp), static_cast<const half_t *>(B),
                           static_cast<half_t *>(C), ws, (uint32_t)M, (uint32_t)N, (uint32_t)K, units, (uint32_t)splitK, nblocks);
        return (int)hipGetLastError();
    }
}
template <int FM, bool GS, int NT, int RT>
int launch_prefill(hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M, size_t N, size_t K,
                   int splitK)
{
    constexpr int    TN = 2 * NT * 16, TM = 2 * RT * 16;
    constexpr size_t kLoopLds = 2 * (size_t)TN * 256, out_full = tile_stage_bytes<2 * NT, RT, 2>(false), out_part = tile_stage_bytes<NT, RT, 2>(true);
    constexpr size_t kOut = out_full > out_part ? out_full : out_part, kLds = kLoopLds > kOut ? kLoopLds : kOut;
    static_assert(kLds <= 160 * 1024, "tile does not fit in LDS");
    if (M % TM) return FP6MI_ERR_SHAPE;
    if (kLds > 48 * 1024)
        if (int rc = allow_dynamic_lds<&gemm_prefill<FM, GS, NT, RT>>(kLds)) return rc;
    uint32_t units = (uint32_t)((K + 255) / 256), nblocks = (uint32_t)((N + TN - 1) / TN);
    size_t   wgs = (M / TM) * (size_t)splitK * nblocks;
    if (wgs > 0x7fffffffu || K > (size_t)1 << 20) return FP6MI_ERR_SHAPE; // (K: 32-bit offsets over TN rows)
    hipLaunchKernelGGL((gemm_prefill<FM, GS, NT, RT>), dim3((uint32_t)wgs), dim3(4 * kWave), kLds, st, static_cast<const uint8_t *>(W),
                       static_cast<const half_t *>(sc), static_cast<const uint8_t *>(gexp), static_cast<const half_t *>(B), static_cast<half_t *>(C), ws,
                       (uint32_t)M, (uint32_t)N, (uint32_t)K, units, (uint32_t)splitK, nblocks);
    return (int)hipGetLastError();
}
template <int FM, bool GS, int NT, int RT, int WK>
int launch_wide(hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M, size_t N, size_t K,
                int splitK)
{
    constexpr int    TN = NT * 16, TM = 4 * RT * 16;
    constexpr size_t kLoopLds = WK * 2 * (size_t)TN * 256, out_full = tile_stage_bytes<NT, RT, 4>(false), out_part = tile_stage_bytes<(NT + 1) / 2, RT, 4>(true);
    constexpr size_t kSums = WK == 2 ? (size_t)TM * ((NT + 1) / 2) * 128 : 0, kOut = out_full > out_part ? out_full : out_part, kMore = kOut > kSums ? kOut : kSums;
    constexpr size_t kLds = kLoopLds > kMore ? kLoopLds : kMore;
    static_assert(kLds <= 160 * 1024 / (3 - WK), "two workgroups of four wavefronts or one of eight do not fit in LDS");
    if (M % TM) return FP6MI_ERR_SHAPE;
    constexpr bool kSpan = NT % 2 == 1 || (NT == 6 && RT == 4 && WK == 2);
    constexpr auto kernel = [] {
        if constexpr (kSpan)
            return &gemm_span<FM, GS, NT, RT, WK>;
        else
            return &gemm_wide<FM, GS, NT, RT, WK>;
    }();
    if (kLds > 48 * 1024)
        if (int rc = allow_dynamic_lds<kernel>(kLds)) return rc;
    uint32_t units = (uint32_t)((K + 255) / 256), nblocks = (uint32_t)((N + TN - 1) / TN);
    size_t   wgs = (M / TM) * (size_t)splitK * nblocks;
    if (wgs > 0x7fffffffu || K > (size_t)1 << 20) return FP6MI_ERR_SHAPE; // (K: 32-bit offsets over TN rows)
    hipLaunchKernelGGL(kernel, dim3((uint32_t)wgs), dim3(4 * WK * kWave), kLds, st, static_cast<const uint8_t *>(W),
                       static_cast<const half_t *>(sc), static_cast<const uint8_t *>(gexp), static_cast<const half_t *>(B), static_cast<half_t *>(C), ws,
                       (uint32_t)M, (uint32_t)N, (uint32_t)K, units, (uint32_t)splitK, nblocks);
    return (int)hipGetLastError();
}
// kind 0: gemm_stream (wr == 1, wk = wavefronts per workgroup);  kind 1: gemm_tile (wr x wk wavefronts);  kind 2: gemm_ws (wr arithmetic + wk loading wavefronts),
// with wr = wk = 2 gemm_prefill (2 x 2 wavefronts; nt = column tiles of the whole workgroup, rt = row tiles per wavefront), with wr = 4 and wk = 1 or 2 gemm_wide or gemm_span (wk: parts of K)
template <int FM, bool GS>
int launch_cfg(const LaunchCfg &c, hipStream_t st, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M,
               size_t N, size_t K, int splitK)
{
    if (c.kind == 0) {
#define FP6MI_CASE(NT, RT, WV) \
    if (c.nt == NT && c.rt == RT && c.wk == WV && c.wr == 1) return launch_stream<FM, GS, NT, RT, WV>(st, W, sc, gexp, B, C, ws, M, N, K, splitK);
        FP6MI_CASE(1, 1, 4) FP6MI_CASE(1, 1, 8) FP6MI_CASE(1, 1, 16)
        FP6MI_CASE(1, 2, 4) FP6MI_CASE(1, 2, 8) FP6MI_CASE(1, 2, 16)
        FP6MI_CASE(1, 3, 4) FP6MI_CASE(1, 3, 8)
        FP6MI_CASE(1, 4, 4) FP6MI_CASE(1, 4, 8)
        FP6MI_CASE(1, 5, 4) FP6MI_CASE(1, 5, 8) FP6MI_CASE(1, 6, 4) FP6MI_CASE(1, 6, 8) FP6MI_CASE(1, 7, 4) FP6MI_CASE(1, 8, 4)
        FP6MI_CASE(2, 1, 4) FP6MI_CASE(2, 1, 8)
        FP6MI_CASE(2, 2, 4) FP6MI_CASE(2, 2, 8)
        FP6MI_CASE(2, 3, 4) FP6MI_CASE(2, 3, 8)
        FP6MI_CASE(2, 4, 4) FP6MI_CASE(2, 4, 8)
        FP6MI_CASE(2, 5, 4) FP6MI_CASE(2, 5, 8) FP6MI_CASE(2, 6, 4) FP6MI_CASE(2, 7, 4) FP6MI_CASE(2, 8, 4)
#undef FP6MI_CASE
    } else if (c.kind == 1) {
#define FP6MI_CASE(NT, RT, WR, WK) \
    if (c.nt == NT && c.rt == RT && c.wr == WR && c.wk == WK) return launch_tile<FM, GS, NT, RT, WR, WK>(st, W, sc, gexp, B, C, ws, M, N, K, splitK);
        FP6MI_CASE(2, 1, 4, 4) FP6MI_CASE(2, 2, 4, 4) FP6MI_CASE(2, 2, 4, 2) FP6MI_CASE(2, 2, 4, 1) FP6MI_CASE(2, 4, 4, 1) FP6MI_CASE(2, 4, 4, 2)
        FP6MI_CASE(4, 2, 4, 2) FP6MI_CASE(4, 2, 4, 1) FP6MI_CASE(4, 4, 4, 1) FP6MI_CASE(4, 4, 2, 1) FP6MI_CASE(4, 4, 2, 2)
        FP6MI_CASE(8, 2, 4, 1) FP6MI_CASE(8, 2, 2, 1) FP6MI_CASE(4, 2, 8, 1) FP6MI_CASE(4, 2, 8, 2) FP6MI_CASE(2, 2, 8, 1) FP6MI_CASE(2, 2, 8, 2) FP6MI_CASE(8, 2, 8, 1) FP6MI_CASE(4, 1, 8, 2) FP6MI_CASE(4, 1, 8, 1) FP6MI_CASE(4, 1, 4, 2) FP6MI_CASE(2, 1, 2, 4)
        FP6MI_CASE(3, 2, 4, 2) FP6MI_CASE(3, 2, 8, 1) FP6MI_CASE(5, 2, 8, 1) FP6MI_CASE(6, 2, 8, 1)
#undef FP6MI_CASE
    } else if (c.kind == 2) {
        // ring depths (weights, activations) that LDS holds: 256 rows (2, 2); 128 rows x 48 columns (3, 3), x 64 and x 80 (3, 2), x 96 (2, 2).  With two stages
        // the memory pipeline runs empty at every barrier: FP6 e3m2, us, (2, 2) -> these: 10240x8192 N 72 in 3 splits 28.1 -> 25.3, 28672x8192 N 72 54.4 -> 48.7,
        // N 40 46.5 -> 35.2, 8192x28672 N 72 in 4 splits 54.9 -> 49.4.  What they replace there (tiles of 32, 64 and 128 columns of gemm_tile): 28, 67, 46 and 69.
        // ((3, 3): the block that K cuts comes through registers; its loads are waited for, and with them every transfer before.)
#define FP6MI_CASE(NT, RT, WR, PW) \
    if (c.nt == NT && c.rt == RT && c.wr == WR && c.wk == PW) { \
        if constexpr (WR == 2) return launch_prefill<FM, GS, NT / 2, RT>(st, W, sc, gexp, B, C, ws, M, N, K, splitK); \
        else if constexpr (PW <= 2) return launch_wide<FM, GS, NT, RT, PW>(st, W, sc, gexp, B, C, ws, M, N, K, splitK); \
        else return launch_ws<FM, GS, NT, RT, WR, PW, WR == 4 && NT < 6 ? 3 : 2, WR == 4 && NT == 3 ? 3 : 2>(st, W, sc, gexp, B, C, ws, M, N, K, splitK); \
    }
        FP6MI_CASE(4, 2, 8, 4) FP6MI_CASE(4, 2, 4, 4) FP6MI_CASE(2, 2, 8, 4) FP6MI_CASE(8, 4, 2, 2) FP6MI_CASE(3, 2, 4, 4) FP6MI_CASE(5, 2, 4, 4) FP6MI_CASE(6, 2, 4, 4) FP6MI_CASE(8, 4, 4, 1) FP6MI_CASE(8, 4, 4, 2) FP6MI_CASE(6, 4, 4, 1) FP6MI_CASE(8, 2, 4, 2) FP6MI_CASE(6, 2, 4, 2) FP6MI_CASE(4, 2, 4, 2)
        FP6MI_CASE(3, 2, 4, 2) FP6MI_CASE(5, 2, 4, 2) FP6MI_CASE(7, 2, 4, 2) FP6MI_CASE(5, 4, 4, 2) FP6MI_CASE(6, 4, 4, 2) FP6MI_CASE(7, 4, 4, 2)
#undef FP6MI_CASE
    }
    return FP6MI_ERR_SHAPE;
}

// ------------------------------------------------------------------------------------------------ entry functions of this format
// (arguments are checked by the C ABI before it comes here)
// gexp: group exponents in their native layout, or null for none; ws: see bias_of
template <int FM>
int op_gemm(const LaunchCfg &c, void *stream, const void *W, const void *sc, const void *gexp, const void *B, void *C, float *ws, size_t M,
            size_t N, size_t K, int splitK)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    return gexp ? launch_cfg<FM, true>(c, st, W, sc, gexp, B, C, ws, M, N, K, splitK) : launch_cfg<FM, false>(c, st, W, sc, nullptr, B, C, ws, M, N, K, splitK);
}

template <int FM> int op_relayout(void *stream, void *native, const void *ref, size_t M, size_t K)
{
    uint32_t units = (uint32_t)((K + 255) / 256);
    hipLaunchKernelGGL(relayout_ref_to_native<FM>, dim3((uint32_t)((M / 64) * units)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<uint8_t *>(native), static_cast<const uint8_t *>(ref), (uint32_t)M, (uint32_t)K, units);
    return (int)hipGetLastError();
}

template <int FM> int op_dequant(void *stream, void *out, const void *W, const void *sc, const void *gexp, size_t M, size_t K)
{
    uint32_t    units = (uint32_t)((K + 255) / 256);
    size_t      blocks = (M / 16) * units;
    dim3        grid((uint32_t)((blocks + 3) / 4));
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t kept = M * K <= kDequantKept / 2; // (and every offset below 2^28)
    if (gexp)
        hipLaunchKernelGGL((dequant_native<FM, true>), grid, dim3(256), 0, st, static_cast<half_t *>(out), static_cast<const uint8_t *>(W),
                           static_cast<const half_t *>(sc), static_cast<const uint8_t *>(gexp), (uint32_t)M, (uint32_t)K, units, kept);
    else
        hipLaunchKernelGGL((dequant_native<FM, false>), grid, dim3(256), 0, st, static_cast<half_t *>(out), static_cast<const uint8_t *>(W),
                           static_cast<const half_t *>(sc), static_cast<const uint8_t *>(nullptr), (uint32_t)M, (uint32_t)K, units, kept);
    return (int)hipGetLastError();
}

// dtype: 0 = fp16, 1 = bf16, 2 = fp32
template <int FM> int op_quantize(void *stream, void *native, void *scales, void *gexp, const void *weights, int dtype, size_t M, size_t K)
{
    const uint32_t units = (uint32_t)((K + 255) / 256);
    const size_t   blocks = (M / 16) * units;
    hipStream_t    st = static_cast<hipStream_t>(stream);
    uint8_t       *nat = static_cast<uint8_t *>(native), *ge = static_cast<uint8_t *>(gexp);
    half_t        *sc = static_cast<half_t *>(scales);
    auto           run = [&](auto *typed, auto groups_c) {
        typedef std::remove_cv_t<std::remove_pointer_t<decltype(typed)>> T;
        constexpr bool GROUPS = decltype(groups_c)::value;
        if (M / 16 >= 160 || K <= 3072 || K <= M * 3) { // (where the two organisations cross: see quant_fused)
            constexpr int WAVES = 8, KEEP = sizeof(T) == 2 ? 2 : 3;
            const uint32_t stash = units > WAVES * KEEP ? quant_stash_bytes<T, WAVES>() : 0; // what some wavefront needs
            if (stash)
                if (int rc = allow_dynamic_lds<quant_fused<FM, T, GROUPS, WAVES, KEEP>>(stash)) return rc;
            hipLaunchKernelGGL((quant_fused<FM, T, GROUPS, WAVES, KEEP>), dim3((uint32_t)(M / 16)), dim3(WAVES * kWave), stash, st, nat, sc, ge, typed,
                               (uint32_t)K, units);
        } else {
            hipLaunchKernelGGL((quant_row_scales<FM, T>), dim3((uint32_t)M), dim3(256), 0, st, sc, typed, (uint32_t)K);
            hipLaunchKernelGGL((quant_blocks<FM, T, GROUPS>), dim3((uint32_t)((blocks + 3) / 4)), dim3(256), 0, st, nat, sc, ge, typed, (uint32_t)M,
                               (uint32_t)K, units);
        }
        return (int)hipGetLastError();
    };
    auto typed = [&](auto groups_c) {
        if (dtype == 0) return run(static_cast<const half_t *>(weights), groups_c);
        if (dtype == 1) return run(static_cast<const bf16_t *>(weights), groups_c);
        return run(static_cast<const float *>(weights), groups_c);
    };
    return gexp ? typed(std::true_type{}) : typed(std::false_type{});
}

} // namespace

namespace fp6mi {
#define FP6MI_OPS_NAME_(f) format_ops_##f
#define FP6MI_OPS_NAME(f) FP6MI_OPS_NAME_(f)
const FormatOps &FP6MI_OPS_NAME(FP6MI_FORMAT)() // a host function, so that the table of host pointers stays out of the device code
{
    static const FormatOps ops = { Fmt<FP6MI_FORMAT>::bits, &op_gemm<FP6MI_FORMAT>, &op_relayout<FP6MI_FORMAT>, &op_dequant<FP6MI_FORMAT>,
                                   &op_quantize<FP6MI_FORMAT> };
    return ops;
}
} // namespace fp6mi
