// bf16 / fp16 matrix-core matmul for gfx950 (v_mfma_f32_16x16x32_bf16 and
// _f16), FP32 accumulation and output. Takes the place of the reference's
// tensor-core kernels (src/cuda/matmul_tensor_core.cu:96-297):
//   - fp32 inputs rounded to nearest-even into bf16 / fp16 as they are
//     staged into LDS (the reference's mode), or
//   - inputs already in bf16 / fp16 in device memory (the pre-cast mode).
// TF32 does not exist on gfx950 (no xf32 matrix instruction): those requests
// report hipErrorNotSupported.
//
// The kernels:
//   matmul_mfma16_staged   row-major operands, fp32 (rounded on the way into
//                          LDS) or 16-bit, any shape and alignment, split K;
//   matmul_mfma16_fast     16-bit operands, B row-major, 256x256 tiles
//                          (gemm_mfma16_fast.h);
//   matmul_mfma16_packed, matmul_mfma16_two_sums, matmul_mfma16_frag   both
//                          operands packed (gemm_mfma16_fast.h, _frag.h).
// Asked for one K range, the staged and fast kernels add each element's products
// in one order (32 k per MFMA, K ascending) and give the same bits, and so does
// the packed one; two_sums has the bits of two such ranges added. The others
// have orders of their own: the frag kernels (a block's waves and accumulators)
// and the staged kernel asked for several ranges (wave groups and accumulators,
// whatever number of ranges runs).
//
// v_mfma_f32_16x16x32_*: lane l supplies row (A) / column (B) l % 16 and
// eight k values from group l / 16; A and B use the same k assignment, so
// any assignment gives the same sum (here group g holds k = 8g .. 8g+7 of the
// 32-wide step). Issued with B first the result is transposed: value v of
// lane l is row l % 16, column 4 (l / 16) + v.

#include "matmul.h"

#include <hip/hip_runtime.h>

#include <atomic>

#include "gemm_mfma16_fast.h"
#include "gemm_mfma16_frag.h"

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

enum { kTensorCoreTf32 = 8, kTensorCoreBf16 = 9, kTensorCoreF16 = 10 };

// Round-to-nearest-even of a float to the upper 16 bits (bf16). NaN stays a
// quiet NaN; values that round past the largest finite bf16 become infinity.
__device__ __forceinline__ unsigned short to_bf16_bits(float x) {
    const unsigned u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<unsigned short>((u >> 16) | 0x0040u);
    const unsigned rounded = u + 0x7fffu + ((u >> 16) & 1u);
    return static_cast<unsigned short>(rounded >> 16);
}

// IEEE half, round to nearest even (the hardware conversion).
__device__ __forceinline__ unsigned short to_f16_bits(float x) {
    const _Float16 h = static_cast<_Float16>(x);
    return __builtin_bit_cast(unsigned short, h);
}

template <bool kBf16>
__device__ __forceinline__ unsigned short to_bits(float x) {
    if constexpr (kBf16) return to_bf16_bits(x);
    return to_f16_bits(x);
}

// Eight floats rounded to 16 bits (to nearest even), as the 16-byte chunk of
// an MFMA operand. bf16: the hardware's packed conversion, the same bits as
// to_bf16_bits (checked over all exponents, subnormals, infinities and NaNs).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned short u16x8u __attribute__((ext_vector_type(8), aligned(2)));
typedef unsigned short u16x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned short u16x2u __attribute__((ext_vector_type(2), aligned(2)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

template <bool kBf16>
__device__ __forceinline__ u16x8 round8(f32x8 v) {
    if constexpr (kBf16) return __builtin_bit_cast(u16x8, __builtin_convertvector(v, bf16x8));
    return __builtin_bit_cast(u16x8, __builtin_convertvector(v, f16x8));
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

template <bool kBf16>
__device__ __forceinline__ u16x4 round4(f32x4 v) {
    if constexpr (kBf16) return __builtin_bit_cast(u16x4, __builtin_convertvector(v, bf16x4));
    return __builtin_bit_cast(u16x4, __builtin_convertvector(v, f16x4));
}

// ---------------------------------------------------------------- staged
//
// Row-major A [m, k] and B [k, n] of fp32 or 16-bit elements at any element
// address. What bounds it is each K step's chain of load, rounding, LDS write and
// barrier, with one block per CU. Counters on an MI355X: 2048^3 from fp32 keeps
// the matrix units 21% busy and brings each CU 67 GB/s from its L2 (81% hits), the
// waves 29% waiting, 37% blocked at issue and 15% in vector ALU instructions;
// 1000^3 bf16 8% busy, 46% waiting. Bank conflicts take a fifth of the LDS pipe's
// active cycles, which are 9% (5%) of the waves'.
//
// Block tile kBM x kBN, K step 64, 256 lanes = 4 waves. A step's operands are
// loaded into registers one or two steps ahead, rounded there (fp32), and written to
// one of two LDS stages in the fragment order of the packed layouts: per 32 k,
// 1 KiB per 16 rows (columns), the 16-byte chunk of 8 k of row r, chunk c at
// 256 c + 16 (r % 16 ^ swizzle). So each MFMA operand is one linear
// ds_read_b128. A lane loads 8 k of a row of A per chunk; of B
// it loads 8 k rows of kCV neighbouring columns and transposes them in
// registers (the fp32 form by choosing which two floats each packed conversion
// takes), where the form before this one wrote B to LDS two bytes at a time.
// The swizzles (chunk of 64 k for A; column block for B) spread 8 consecutive
// lanes' 16-byte writes over all banks.
//
// The edges. Rows past m read row m - 1. A lane whose columns cross n reads
// the last kCV columns instead and writes them to those columns' places (a
// neighbour writes the same values there), so no load is guarded; what lies
// past n in LDS is never stored from. The last K step, when it is not whole,
// is loaded element by element with zeros past K, as is everything when
// n < kCV. Vector loads need element alignment only.
//
// On an MI355X, one launch after another on one set of operands, against the
// 128x128 kernel this one replaced: fp32 operands as bf16 2048^3 282 -> 39.0 us,
// 4096^3 971 -> 224, 1000^3 (4 splits allowed) 43.7 -> 14.8; bf16 operands 1000^3
// (likewise) 24.9 -> 9.8, 3000x3001x1023 346 -> 51.1, 16x4096x4096 27.7 -> 10.2.
// kWM x kWN waves of a group tile the block's C tile; kG groups take every
// kG-th K step each and are added at the end; kAhead: steps loaded ahead (in
// registers); kBlocks: blocks per CU the register budget is cut for; kAcc: 1,
// or 4 accumulators per element that take the 32-wide half steps in turn and
// are added at the end. Where a caller allows K ranges, the 128x128 kernel ran
// all of them, up to eight times what these smaller tiles need to fill the
// chip; ranges x groups x accumulators keep its number of partial sums, and so
// its rounding error (launch16 picks the forms).
template <int kBM_, int kBN_, int kWM_, int kWN_, int kG_, int kAhead_, int kBlocks_, int kAcc_ = 1>
struct Staged {
    static constexpr int kBM = kBM_, kBN = kBN_, kBK = 64;
    static constexpr int kG = kG_, kAhead = kAhead_, kBlocks = kBlocks_, kAcc = kAcc_;
    static_assert(kAhead == 1 || kAhead == 2, "the main loop's unrolling");
    static_assert(kAcc == 1 || (kAcc == 4 && kAhead == 2), "step parities known to the unrolled loop");
    static constexpr int kWavesN = kWN_, kWaves = kWM_ * kWN_;
    static constexpr int kLanes = 64 * kWaves, kThreads = kLanes * kG;
    static constexpr int kRows = kBM / kWM_, kCols = kBN / kWN_;  // of a wave
    static constexpr int kRowFrags = kRows / 16, kColFrags = kCols / 16;
    // 16-byte loads of A per lane and step: 8 16-bit or 4 fp32 elements.
    static constexpr int a_loads(bool f32) { return kBM * (f32 ? 16 : 8) / kLanes; }
    static constexpr int kCV = kBN * 8 / kLanes;       // columns of B per lane
    static constexpr int kASub = kBM * 64, kBSub = kBN * 64;  // bytes per 32 k
    static constexpr int kStage = 2 * (kASub + kBSub);
    static constexpr int kStagePitch = kStage + 1024;  // and 16 bytes per lane for columns before the tile
    static constexpr int kSums = kG > 1 ? kG * kBM * kBN * 4 : 0;
    static constexpr int kLds = kSums > 2 * kStagePitch * kG ? kSums : 2 * kStagePitch * kG;
};

// A K step's parity, as a type.
template <int kParity>
struct Parity {
    static constexpr int value = kParity;
};

// kCV consecutive elements as 16-byte aligned or unaligned vector loads.
template <bool kF32In, int kCV>
struct BVec;
template <>
struct BVec<true, 4> { typedef f32x4u type; };
template <>
struct BVec<true, 2> { typedef f32x2u type; };
template <>
struct BVec<false, 4> { typedef u16x4u type; };
template <>
struct BVec<false, 2> { typedef u16x2u type; };

template <bool kBf16, bool kF32In, class Cfg>
__global__ void __launch_bounds__(Cfg::kThreads, Cfg::kBlocks) matmul_mfma16_staged(const void* __restrict__ a_, const void* __restrict__ b_,
                                                               float* __restrict__ c, int m, int n, int k, int k_split,
                                                               float* __restrict__ partial) {
    typedef typename std::conditional<kF32In, float, unsigned short>::type T;
    typedef typename BVec<kF32In, Cfg::kCV>::type BV;
    constexpr int kCV = Cfg::kCV, kBK = Cfg::kBK;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[Cfg::kLds];
    const T* __restrict__ a = static_cast<const T*>(a_);
    const T* __restrict__ b = static_cast<const T*>(b_);

    const int grp = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / Cfg::kLanes);
    const int tid = static_cast<int>(threadIdx.x) % Cfg::kLanes;  // in the group
    const int wave = tid / 64, lane = tid % 64;
    unsigned char* const stages = smem + grp * 2 * Cfg::kStagePitch;
    // Tiles in column groups of 8, row by row within a group; block L runs on
    // XCD L % 8, which takes a contiguous eighth of the list when the count is
    // a multiple of 8, so an L2 serves a compact patch of tiles.
    const int tiles_n = (n + Cfg::kBN - 1) / Cfg::kBN, tiles_m = (m + Cfg::kBM - 1) / Cfg::kBM;
    const int total = static_cast<int>(gridDim.x), L = static_cast<int>(blockIdx.x);
    int q = total % 8 == 0 ? (L % 8) * (total / 8) + L / 8 : L;
    const int z = q / (tiles_m * tiles_n);
    q -= z * tiles_m * tiles_n;
    const int group = q / (8 * tiles_m), in_group = q % (8 * tiles_m);
    const int width = min(8, tiles_n - 8 * group);
    const int row0 = (in_group / width) * Cfg::kBM, col0 = (8 * group + in_group % width) * Cfg::kBN;
    const int kb = z * k_split, ke = min(k, kb + k_split);

    // This lane's loads of A, a row's 64 k over 8 (16) consecutive lanes:
    // row tid / 8 (16) + .., k kAK ac .. kAK ac + kAK - 1 of the step.
    constexpr int kALoads = Cfg::a_loads(kF32In), kAK = kF32In ? 4 : 8, kARow = kBK / kAK;
    const int ac = tid % kARow;
    const T* a_src[kALoads];
    int a_dst[kALoads];
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
        const int r = tid / kARow + Cfg::kLanes / kARow * i;
        const int ch = ac * kAK / 8;  // its chunk of 8 k
        a_src[i] = a + static_cast<std::ptrdiff_t>(min(row0 + r, m - 1)) * k + kAK * ac;
        a_dst[i] = (ch / 4) * Cfg::kASub + (r / 16) * 1024 + (ch % 4) * 256 + ((r % 16) ^ ch) * 16 +
                   (kF32In ? (ac % 2) * 8 : 0);
    }
    // This lane's columns of B: bcol .. bcol + kCV - 1, k 8 bk .. 8 bk + 7.
    const bool whole_cols = n >= kCV;
    constexpr int kQuads = Cfg::kBN / kCV;
    const int bk = tid / kQuads;
    const int bcol = whole_cols ? min(col0 + (tid % kQuads) * kCV, n - kCV) : (tid % kQuads) * kCV;
    const T* const b_src = b + static_cast<std::ptrdiff_t>(8 * bk) * n + bcol;
    int b_dst[kCV];
#pragma unroll
    for (int j = 0; j < kCV; ++j) {
        const int col = bcol - col0 + j;  // may be before the tile: written past the stage
        b_dst[j] = col < 0 ? Cfg::kStage + lane * 16
                           : 2 * Cfg::kASub + (bk / 4) * Cfg::kBSub + (col / 16) * 1024 + (bk % 4) * 256 +
                                 ((col % 16) ^ ((col / 16) & 3)) * 16;
    }

    typedef typename std::conditional<kF32In, f32x4u, u16x8u>::type AV;
    struct Regs {
        AV a[kALoads];
        BV b[8];
    };
    auto load_whole = [&](Regs& r, int k0) {
#pragma unroll
        for (int i = 0; i < kALoads; ++i) r.a[i] = *reinterpret_cast<const AV*>(a_src[i] + k0);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            r.b[e] = *reinterpret_cast<const BV*>(b_src + static_cast<std::ptrdiff_t>(k0 + e) * n);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Element by element, zeros past ke. The loads are clamped to the last k
    // and column instead of guarded (32 branches, each a live mask).
    auto load_part = [&](Regs& r, int k0) {
#pragma unroll
        for (int i = 0; i < kALoads; ++i)
#pragma unroll
            for (int e = 0; e < kAK; ++e) {
                const int kk = k0 + kAK * ac + e;
                const T v = a_src[i][min(kk, ke - 1) - kAK * ac];
                r.a[i][e] = kk < ke ? v : T(0);
            }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int kk = k0 + 8 * bk + e;
            const T* const src = b + static_cast<std::ptrdiff_t>(min(kk, ke - 1)) * n;
#pragma unroll
            for (int j = 0; j < kCV; ++j) {
                const T v = src[min(bcol + j, n - 1)];
                r.b[e][j] = kk < ke ? v : T(0);
            }
        }
    };
    auto store = [&](const Regs& r, int stage) {
        unsigned char* const s = stages + stage * Cfg::kStagePitch;
#pragma unroll
        for (int i = 0; i < kALoads; ++i) {
            if constexpr (kF32In) {
                *reinterpret_cast<u16x4*>(s + a_dst[i]) = round4<kBf16>(r.a[i]);
            } else {
                *reinterpret_cast<u16x8*>(s + a_dst[i]) = r.a[i];
            }
        }
#pragma unroll
        for (int j = 0; j < kCV; ++j) {
            u16x8 v;
            if constexpr (kF32In) {
                v = round8<kBf16>(f32x8{r.b[0][j], r.b[1][j], r.b[2][j], r.b[3][j], r.b[4][j], r.b[5][j], r.b[6][j], r.b[7][j]});
            } else {
                v = u16x8{r.b[0][j], r.b[1][j], r.b[2][j], r.b[3][j], r.b[4][j], r.b[5][j], r.b[6][j], r.b[7][j]};
            }
            *reinterpret_cast<u16x8*>(s + b_dst[j]) = v;
        }
    };

    const int wr = (wave / Cfg::kWavesN) * Cfg::kRows, wc = (wave % Cfg::kWavesN) * Cfg::kCols;
    const int lk = lane / 16, li = lane % 16;
    f32x4 sum[Cfg::kAcc][Cfg::kRowFrags][Cfg::kColFrags];
#pragma unroll
    for (int x = 0; x < Cfg::kAcc; ++x)
#pragma unroll
        for (int i = 0; i < Cfg::kRowFrags; ++i)
#pragma unroll
            for (int j = 0; j < Cfg::kColFrags; ++j) sum[x][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int stage, auto parity) {
        const unsigned char* const s = stages + stage * Cfg::kStagePitch;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u16x8 av[Cfg::kRowFrags], bv[Cfg::kColFrags];
#pragma unroll
            for (int i = 0; i < Cfg::kRowFrags; ++i)
                av[i] = *reinterpret_cast<const u16x8*>(s + h * Cfg::kASub + (wr / 16 + i) * 1024 + lk * 256 +
                                                        (li ^ (4 * h + lk)) * 16);
#pragma unroll
            for (int j = 0; j < Cfg::kColFrags; ++j)
                bv[j] = *reinterpret_cast<const u16x8*>(s + 2 * Cfg::kASub + h * Cfg::kBSub + (wc / 16 + j) * 1024 +
                                                        lk * 256 + (li ^ ((wc / 16 + j) & 3)) * 16);
#pragma unroll
            for (int i = 0; i < Cfg::kRowFrags; ++i)
#pragma unroll
                for (int j = 0; j < Cfg::kColFrags; ++j) {
                    f32x4& acc = sum[(2 * decltype(parity)::value + h) % Cfg::kAcc][i][j];
                    acc = mc_mfma16<kBf16>(bv[j], av[i], acc);
                }
        }
    };

    // The group's i-th whole step is step i kG + grp, for i < mine: the same
    // count for every group, so the barriers match. Register set i % kAhead
    // holds it, loaded kAhead steps before it is written to LDS. Every load
    // is unconditional (past the last it loads that one again): under a
    // condition, the compiler's wait for one set would wait for the sets
    // loaded after it too. What is left is at most one more step per group,
    // whole, partial or empty (zeros), loaded ahead as well where there are
    // registers for it; with n < kCV every step is of that kind. An empty one
    // loads nothing (from fp32 768x768x320, one group's third step empty, 9.0 us
    // with clamped loads, 7.6 without).
    constexpr int kAhead = Cfg::kAhead, kG = Cfg::kG;
    const int tiles = ke > kb ? (ke - kb + kBK - 1) / kBK : 0;
    const int full = whole_cols ? (ke - kb) / kBK : 0;
    const int mine = full / kG;
    const int rounds = (tiles + kG - 1) / kG;
    constexpr bool kRestAhead = kAhead > 1;
    auto k_of = [&](int i) { return kb + (i * kG + grp) * kBK; };
    auto load_rest = [&](Regs& r, int i) {
        if (i * kG + grp < full) {
            load_whole(r, k_of(i));
        } else if (kG == 1 || i * kG + grp < tiles) {
            load_part(r, k_of(i));
        } else {
            r = Regs{};
        }
    };
    Regs rest;
    if (mine > 0) {
        Regs set[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load_whole(set[u], k_of(min(u, mine - 1)));
        if (kRestAhead && mine < rounds) load_rest(rest, mine);
        store(set[0], 0);
        load_whole(set[0], k_of(min(kAhead, mine - 1)));
        __syncthreads();
        auto step = [&](int i, Regs& next, auto parity) {
            // The other stage was last read before the previous barrier.
            store(next, (i + 1) & 1);
            load_whole(next, k_of(min(i + 1 + kAhead, mine - 1)));
            multiply(i & 1, parity);
            __syncthreads();
        };
        int i = 0;
        for (; i + kAhead <= mine; i += kAhead) {
            step(i, set[1 % kAhead], Parity<0>{});
            if constexpr (kAhead == 2) step(i + 1, set[0], Parity<1>{});
        }
        if (i < mine) step(i, set[1 % kAhead], Parity<0>{});
    }
    for (int i = mine; i < rounds; ++i) {
        if (!kRestAhead || mine == 0 || i > mine) load_rest(rest, i);
        store(rest, i & 1);
        __syncthreads();
        multiply(i & 1, Parity<1>{});
        __syncthreads();
    }

    f32x4(&acc)[Cfg::kRowFrags][Cfg::kColFrags] = sum[0];
    if constexpr (Cfg::kAcc == 4) {
#pragma unroll
        for (int i = 0; i < Cfg::kRowFrags; ++i)
#pragma unroll
            for (int j = 0; j < Cfg::kColFrags; ++j) acc[i][j] = (sum[0][i][j] + sum[1][i][j]) + (sum[2][i][j] + sum[3][i][j]);
    }
    // Lane l holds row l % 16, columns 4 (l / 16) .. + 3 of each fragment.
    float* __restrict__ out = partial != nullptr ? partial + static_cast<std::ptrdiff_t>(z) * m * n : c;
    auto store_c = [&](int i, int j, f32x4 v) {
        const int row = row0 + wr + i * 16 + li, col = col0 + wc + j * 16 + 4 * lk;
        if (row >= m) return;
        float* const dst = out + static_cast<std::ptrdiff_t>(row) * n + col;
        if (col + 4 <= n) {
            *reinterpret_cast<f32x4u*>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (col + e < n) dst[e] = v[e];
        }
    };
    if constexpr (kG == 1) {
#pragma unroll
        for (int i = 0; i < Cfg::kRowFrags; ++i)
#pragma unroll
            for (int j = 0; j < Cfg::kColFrags; ++j) store_c(i, j, acc[i][j]);
    } else {
        // The groups' tiles through LDS (the stages are done with), added in
        // group order, every group a share of the fragments.
        constexpr int kFrags = Cfg::kRowFrags * Cfg::kColFrags;
        f32x4* const sums = reinterpret_cast<f32x4*>(smem);
        auto at = [&](int g, int f) { return ((g * Cfg::kWaves + wave) * kFrags + f) * 64 + lane; };
#pragma unroll
        for (int f = 0; f < kFrags; ++f) sums[at(grp, f)] = acc[f / Cfg::kColFrags][f % Cfg::kColFrags];
        __syncthreads();
#pragma unroll
        for (int f = 0; f < kFrags; ++f) {
            if (f % kG != grp) continue;
            f32x4 v = sums[at(0, f)];
#pragma unroll
            for (int g = 1; g < kG; ++g) v += sums[at(g, f)];
            store_c(f / Cfg::kColFrags, f % Cfg::kColFrags, v);
        }
    }
}

// ---------------------------------------------------------------- fast path
//
// The body lives in gemm_mfma16_fast.h (also compiled at run time with fused
// epilogues); here it is instantiated with the identity epilogue.

template <bool kBf16, bool kPackedA>
__global__ void __launch_bounds__(kFThreads, 1) matmul_mfma16_fast(const unsigned short* __restrict__ a,
                                                                   const unsigned short* __restrict__ b,
                                                                   float* __restrict__ c, int m, int n, int k) {
    mc_gemm16_fast<kBf16, kPackedA>(a, b, c, m, n, k, McGemm16Store{});
}

// Both operands packed (what compiled graphs run).
template <bool kBf16>
__global__ void __launch_bounds__(kFThreads, 1) matmul_mfma16_packed(const unsigned short* __restrict__ a,
                                                                     const unsigned short* __restrict__ b,
                                                                     float* __restrict__ c, int m, int n, int k) {
    mc_gemm16_packed<kBf16>(a, b, c, m, n, k, McGemm16Store{});
}

template <bool kBf16>
__global__ void __launch_bounds__(kFThreads, 1) matmul_mfma16_two_sums(const unsigned short* __restrict__ a,
                                                                       const unsigned short* __restrict__ b,
                                                                       float* __restrict__ c, int m, int n, int k) {
    mc_gemm16_two_sums<kBf16>(a, b, c, m, n, k, McGemm16Store{});
}

template <bool kBf16, class Cfg>
__global__ void __launch_bounds__(Cfg::kThreads) matmul_mfma16_frag(const unsigned short* __restrict__ a,
                                                                    const unsigned short* __restrict__ b,
                                                                    float* __restrict__ c, int m, int n, int k) {
    mc_gemm16_frag<kBf16, Cfg>(a, b, c, m, n, k, McGemm16Store{});
}

// CUs of the current device, asked once per device.
int device_cus() {
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < 64) {
        const int c = cache[dev].load(std::memory_order_relaxed);
        if (c > 0) return c;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < 64) cache[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// Whether the 256x256-tile kernel can run the product: 16-bit A and B with K
// a multiple of 64, N a multiple of 8 (every 16-byte B chunk wholly inside or
// outside a row), A, B and C 16-byte aligned.
bool fast_eligible(const void* a, const void* b, const float* c, int m, int n, int k) {
    const auto al = [](const void* p) { return reinterpret_cast<std::uintptr_t>(p) % 16 == 0; };
    return mchip_mfma16_fast_fits(m, n, k) && al(a) && al(b) && al(c);
}

// And whether it should, on row-major operands: with at most two 64x64 tiles
// per CU the staged kernel is faster (bf16, K = 2048, graph-timed on an
// MI355X: 512x1024 19.4 us against 30.8, 1024x2048 23.8 against 32.3, 1536x2048
// 32.6 against 33.0; 2048^2 on its 128x128 tiles 34.7 against 34.4).
bool fast_preferred(int m, int n) {
    return static_cast<long long>((m + 63) / 64) * ((n + 63) / 64) > 2LL * std::max(device_cus(), 1);
}

template <bool kBf16, bool kPackedA = false>
int launch_fast(const void* a, const void* b, float* c, int m, int n, int k, hipStream_t stream) {
    const long long tiles = static_cast<long long>((m + kFBM - 1) / kFBM) * ((n + kFBN - 1) / kFBN);
    if (tiles > 0x3fffffffLL) return hipErrorInvalidValue;
    const unsigned grid = mchip_mfma16_fast_grid(m, n, device_cus());
    hipLaunchKernelGGL((matmul_mfma16_fast<kBf16, kPackedA>), dim3(grid), dim3(kFThreads), 0, stream,
                       static_cast<const unsigned short*>(a), static_cast<const unsigned short*>(b), c, m, n, k);
    return hipGetLastError();
}

// ------------------------------------------------------------ packed A
//
// One lane per 16-byte chunk of the packed layout (gemm_mfma16_fast.h): 8
// consecutive k of one row. Consecutive lanes take consecutive chunks, so a
// wave writes 1 KiB of consecutive memory and reads 16 rows x 4 chunks
// (64 bytes of 16-bit A, 128 of fp32 A, per row). Rows past M are zeros.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

struct PackedChunk {
    int row, kk;
};

__device__ __forceinline__ PackedChunk packed_chunk(long long q, int steps) {
    const long long blk = q >> 10;
    const int w = static_cast<int>(q & 1023);
    const int band = static_cast<int>(blk / steps), step = static_cast<int>(blk % steps);
    return {band * kFBM + (w >> 6) * 16 + (w & 15), step * kFBK + ((w >> 4) & 3) * 8};
}

// kVec: `in` 16-byte aligned (one 16-byte load per chunk), else 8 loads of
// 2 bytes.
template <bool kVec>
__global__ void __launch_bounds__(256) pack_a16_kernel(const unsigned short* __restrict__ in, u32x4* __restrict__ out,
                                                       int m, int k, long long chunks) {
    const int steps = k / kFBK;
    const long long stride = static_cast<long long>(gridDim.x) * 256;
    for (long long q = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; q < chunks; q += stride) {
        const PackedChunk p = packed_chunk(q, steps);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (p.row < m) {
            const unsigned short* src = in + static_cast<long long>(p.row) * k + p.kk;
            if constexpr (kVec) {
                v = *reinterpret_cast<const u32x4*>(src);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = src[2 * j] | (static_cast<unsigned>(src[2 * j + 1]) << 16);
            }
        }
        out[q] = v;
    }
}

// fp32 A of any K and alignment rounded and packed, K padded with zeros to
// `kp`: a wave takes two K steps of a 16-row block, lane l the 8 k values of
// row l % 16 from 8 (l / 16): 16 rows x 128 bytes read, 1 KiB written per
// step. Memory bound, 6 B per element; two steps per wave keep four 16-byte
// loads in flight per lane, which is what it takes: on an MI355X 4096^2 in
// 15.8 us (6.4 TB/s) where a form that turned 256-row regions through LDS
// took 22.1, and 512x4096 in 3.2 us against 8.7 (its regions were too few).
// `blocks16` 16-row blocks are written, rows past m as zeros; a product reads
// only those that hold a row (mchip_pack16_a_f32 writes no others).
template <bool kBf16>
__global__ void __launch_bounds__(256) pack16_a_rows(const float* __restrict__ in, u32x4* __restrict__ out, int m,
                                                     int k, int kp, int pairs, long long units) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const long long waves = static_cast<long long>(gridDim.x) * 4;
    for (long long w = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6); w < units; w += waves) {
        const int rb = static_cast<int>(w / pairs), s0 = static_cast<int>(w % pairs) * 2;
        const int row = rb * 16 + (lane & 15);
        f32x8 v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int kk = (s0 + u) * kFBK + (lane >> 4) * 8;
            const float* src = in + static_cast<long long>(row) * k + kk;
            if (row < m && kk + 8 <= k) {
                const f32x4 lo = *reinterpret_cast<const f32x4u*>(src), hi = *reinterpret_cast<const f32x4u*>(src + 4);
                v[u] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[u][e] = row < m && kk + e < k ? src[e] : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const long long at = static_cast<long long>(rb / 16) * kp * 32 + (s0 + u) * 1024LL + (rb % 16) * 64 + lane;
            out[at] = __builtin_bit_cast(u32x4, round8<kBf16>(v[u]));
        }
    }
}

// fp32 row-major B [k, n] rounded and packed (256-column panels, K padded
// with zeros to `kp`): a block takes one K step of one panel, a lane one
// column: 32 loads, each 1 KiB of consecutive memory over the block, then
// four 16-byte chunks of 8 k (5.0 TB/s at 4096^2 on an MI355X). Once per
// constant; per run for a B that is computed or fed.
template <bool kBf16>
__global__ void __launch_bounds__(256) pack16_b(const float* __restrict__ in, u32x4* __restrict__ out, int k, int n,
                                                int kp, long long units) {
    const int steps = kp / kFBK;
    const int t = static_cast<int>(threadIdx.x);
    for (long long u = blockIdx.x; u < units; u += gridDim.x) {
        const int panel = static_cast<int>(u / steps), k0 = static_cast<int>(u % steps) * kFBK;
        const int col = panel * kFBN + t;
        const float* src = in + static_cast<long long>(k0) * n + (col < n ? col : n - 1);
        float v[kFBK];
#pragma unroll
        for (int i = 0; i < kFBK; ++i) v[i] = k0 + i < k ? src[static_cast<long long>(i) * n] : 0.0f;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            const f32x8 w = {v[ch * 8],     v[ch * 8 + 1], v[ch * 8 + 2], v[ch * 8 + 3],
                             v[ch * 8 + 4], v[ch * 8 + 5], v[ch * 8 + 6], v[ch * 8 + 7]};
            out[u * 1024 + (t >> 4) * 64 + ch * 16 + (t & 15)] = __builtin_bit_cast(u32x4, round8<kBf16>(w));
        }
    }
}

unsigned pack_blocks(long long chunks) {
    return static_cast<unsigned>(std::max<long long>(1, std::min<long long>((chunks + 255) / 256, 16384)));
}

bool aligned(const void* p, std::uintptr_t bytes) { return reinterpret_cast<std::uintptr_t>(p) % bytes == 0; }

int split_len(int k, int splits, int step) {
    if (splits <= 1) return std::max(k, 1);
    const int per = (k + splits - 1) / splits;
    return (per + step - 1) / step * step;
}

// The staged kernel's tile and K ranges for a product (at most `splits`
// ranges, what the caller sized its workspace for).
struct StagedPlan {
    int bm, bn, k_split, depth;
    long long tiles;
};

// 128x128 tiles where they give at least four in five CUs one (the line of
// split_k_splits, past which it asks for no ranges: a caller's own count runs
// as given), else 64x64, or 32x64 for at most 32 rows; those in K ranges only
// where they leave half the CUs idle (on an MI355X, bf16 operands: 512x1024x2048,
// 128 tiles of 64x64, 12.7 us in 2 ranges with their sum against 15.5 unsplit;
// 1000^3, 256 tiles, 9.8 us unsplit, where the 128x128 kernel in 4 ranges took
// 24.9).
StagedPlan staged_plan(int m, int n, int k, int splits) {
    const long long cus = std::max(device_cus(), 1);
    const auto tiles = [&](int bm, int bn) {
        return static_cast<long long>((m + bm - 1) / bm) * ((n + bn - 1) / bn);
    };
    StagedPlan p;
    if (5 * tiles(128, 128) >= 4 * cus) {
        p.bm = p.bn = 128;
    } else {
        p.bm = m <= 32 ? 32 : 64;
        p.bn = 64;
    }
    p.tiles = tiles(p.bm, p.bn);
    const long long most = p.bm == 128 ? splits : 2 * p.tiles <= cus ? cus / p.tiles : 1;
    const long long want = std::max<long long>(1, std::min<long long>(splits, most));
    p.k_split = split_len(k, static_cast<int>(want), 64);
    p.depth = std::max(1, (k + p.k_split - 1) / p.k_split);
    return p;
}

template <bool kBf16, bool kF32In>
int launch16(const void* a, const void* b, float* c, int m, int n, int k, hipStream_t stream, int splits,
             float* workspace) {
    // Several ranges asked for need a workspace, whatever number of them runs.
    const int asked = split_len(k, splits, 64);
    if ((k + asked - 1) / asked > 1 && workspace == nullptr) return hipErrorInvalidValue;
    const StagedPlan p = staged_plan(m, n, k, splits);
    const long long blocks = p.tiles * p.depth;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    float* ws = p.depth > 1 ? workspace : nullptr;
    const auto run = [&](auto cfg) {
        using Cfg = decltype(cfg);
        hipLaunchKernelGGL((matmul_mfma16_staged<kBf16, kF32In, Cfg>), grid, dim3(Cfg::kThreads), 0, stream, a, b, c,
                           m, n, k, p.k_split, ws);
    };
    // The form of a tile, by operand type (us on an MI355X, K = 2048 or 2040).
    // 128x128: with at most one per CU two steps are loaded ahead (2048^2 fp32
    // 39.0 against 45.4 with one; bf16 30.5 against 32.9), with more than one a
    // second block per CU does better than the deeper prefetch (3072^2 fp32
    // 89.3 against 101.3; bf16 73 against 82.4). Eight waves where the
    // registers allow (bf16: 2048^2 30.5 against 39.2 with four; fp32 4096^2
    // 114.4 on four waves against 150).
    // 64x64, where the caller's split count leaves the order of adds open: two
    // groups of waves, each taking every other K step, where there is one tile
    // per CU at most (bf16 1024^2 12.2 against 15.3). fp32 operands are bound by
    // the loads themselves and run one group, but where its four accumulators per
    // range are fewer sums than the ranges asked for, and the ranges long enough
    // for the error to show it. 2-norm error with one group and with two, of that
    // in the ranges asked for, and us:
    //   1 range, 768x768: bf16 K = 4096 1.26 and 0.89, 39.5 and 35.2; K = 576 0.99
    //     and 0.89, 8.5 and 9.3; fp16 K = 448 1.06 and 0.94, 7.4 and 8.0;
    //   2 ranges, 256x1400: bf16 K = 4095 1.06 and 0.82, 30.5 and 29.4; fp16 K =
    //     2048 1.03 and 0.82, 15.8 and 15.3; K = 1536 0.96 with one;
    //   3 ranges, 128x2176: fp16 K = 6144 1.00 and 0.78, 24.6 and 23.5; K = 4032
    //     0.96 with one; bf16 K = 2048 0.88 and 0.79, 13.0 and 13.4.
    const long long cus = std::max(device_cus(), 1);
    const int enough = p.depth == 1 ? (kBf16 ? 576 : 256) : p.depth == 2 ? 768 : 1344;
    const bool more_sums = p.depth <= 3 && splits > 4 * p.depth && p.k_split > enough;
    if (p.bm == 128) {
        if constexpr (kF32In) {
            if (p.tiles <= cus) {
                run(Staged<128, 128, 2, 2, 1, 2, 1>{});
            } else {
                run(Staged<128, 128, 2, 2, 1, 1, 2>{});
            }
        } else {
            if (p.tiles <= cus) {
                run(Staged<128, 128, 2, 4, 1, 2, 1>{});
            } else {
                run(Staged<128, 128, 2, 4, 1, 1, 1>{});
            }
        }
    } else if (p.bm == 64) {
        if (splits <= 1) {
            run(Staged<64, 64, 2, 2, 1, 2, 2>{});
        } else if (p.tiles > cus || (kF32In && !more_sums)) {
            run(Staged<64, 64, 2, 2, 1, 2, 2, 4>{});
        } else {
            run(Staged<64, 64, 2, 2, 2, 2, 1, 4>{});
        }
    } else if (splits <= 1) {
        run(Staged<32, 64, 1, 4, 1, 2, 2>{});
    } else {
        run(Staged<32, 64, 1, 4, 1, 2, 2, 4>{});
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.depth == 1) return e;
    return mchip_sum_split_partials(workspace, c, static_cast<std::size_t>(m) * n, p.depth, stream);
}

__global__ void __launch_bounds__(256) convert_kernel(const float* __restrict__ in, unsigned short* __restrict__ out,
                                                      std::size_t count, int bf16) {
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * 256;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x; i < count; i += stride) {
        out[i] = bf16 ? to_bf16_bits(in[i]) : to_f16_bits(in[i]);
    }
}

// The same rounding on 16-byte-aligned `in` and 8-byte-aligned `out`: a lane
// reads a float4 and writes its four 16-bit values as one 8-byte store, for
// kConvertItems float4s spaced one block apart (each wave instruction reads
// 1 KiB and writes 512 bytes of consecutive memory). Elements past the last
// whole float4 are done one by one by the first block.
constexpr int kConvertItems = 4;

template <bool kBf16>
__global__ void __launch_bounds__(256) convert_vec_kernel(const f32x4* __restrict__ in, u16x4* __restrict__ out,
                                                          std::size_t groups, const float* __restrict__ tail_in,
                                                          unsigned short* __restrict__ tail_out, int tail) {
    const std::size_t span = static_cast<std::size_t>(256) * kConvertItems;
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * span;
    for (std::size_t base = static_cast<std::size_t>(blockIdx.x) * span + threadIdx.x; base < groups; base += stride) {
        f32x4 v[kConvertItems];
#pragma unroll
        for (int j = 0; j < kConvertItems; ++j) {
            const std::size_t g = base + static_cast<std::size_t>(j) * 256;
            if (g < groups) v[j] = __builtin_nontemporal_load(in + g);
        }
#pragma unroll
        for (int j = 0; j < kConvertItems; ++j) {
            const std::size_t g = base + static_cast<std::size_t>(j) * 256;
            if (g < groups) {
                const u16x4 r = {to_bits<kBf16>(v[j][0]), to_bits<kBf16>(v[j][1]), to_bits<kBf16>(v[j][2]),
                                 to_bits<kBf16>(v[j][3])};
                out[g] = r;
            }
        }
    }
    if (blockIdx.x == 0 && static_cast<int>(threadIdx.x) < tail) {
        tail_out[threadIdx.x] = to_bits<kBf16>(tail_in[threadIdx.x]);
    }
}

}  // namespace

extern "C" int mchip_launch_tensor_core(int kernel, const float* a, const float* b, float* c, int m, int n, int k,
                                        void* stream, int splits, float* workspace) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (m < 1 || n < 1 || k < 1) return hipErrorInvalidValue;
    switch (kernel) {
        case kTensorCoreBf16: return launch16<true, true>(a, b, c, m, n, k, s, splits, workspace);
        case kTensorCoreF16: return launch16<false, true>(a, b, c, m, n, k, s, splits, workspace);
        case kTensorCoreTf32: return hipErrorNotSupported;
        default: return hipErrorInvalidValue;
    }
}

extern "C" int mchip_launch_matmul_lowp(int kernel, int dtype, const void* a, const void* b, float* c, int m, int n,
                                        int k, void* stream, int splits, float* workspace) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (m < 1 || n < 1 || k < 1) return hipErrorInvalidValue;
    if (kernel == kTensorCoreTf32) return hipErrorNotSupported;
    const int asked = split_len(k, splits, 64);
    if ((k + asked - 1) / asked > 1 && workspace == nullptr) return hipErrorInvalidValue;
    const bool fast = splits <= 1 && fast_eligible(a, b, c, m, n, k) && fast_preferred(m, n);
    if (kernel == kTensorCoreBf16 && dtype == MCHIP_DTYPE_BF16) {
        return fast ? launch_fast<true>(a, b, c, m, n, k, s) : launch16<true, false>(a, b, c, m, n, k, s, splits, workspace);
    }
    if (kernel == kTensorCoreF16 && dtype == MCHIP_DTYPE_F16) {
        return fast ? launch_fast<false>(a, b, c, m, n, k, s) : launch16<false, false>(a, b, c, m, n, k, s, splits, workspace);
    }
    return hipErrorInvalidValue;
}

extern "C" long long mchip_packed_a16_elements(int m, int k) {
    if (m < 1 || k < 1) return 0;
    return static_cast<long long>((m + kFBM - 1) / kFBM) * kFBM * k;
}

extern "C" int mchip_pack_a16(const void* a, void* packed, int m, int k, void* stream) {
    if (m < 1 || k < 1 || k % (2 * kFBK) != 0 || !aligned(a, 2) || !aligned(packed, 16)) return hipErrorInvalidValue;
    const long long chunks = mchip_packed_a16_elements(m, k) / 8;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const auto* in = static_cast<const unsigned short*>(a);
    if (aligned(a, 16)) {
        hipLaunchKernelGGL(pack_a16_kernel<true>, dim3(pack_blocks(chunks)), dim3(256), 0, s, in,
                           static_cast<u32x4*>(packed), m, k, chunks);
    } else {
        hipLaunchKernelGGL(pack_a16_kernel<false>, dim3(pack_blocks(chunks)), dim3(256), 0, s, in,
                           static_cast<u32x4*>(packed), m, k, chunks);
    }
    return hipGetLastError();
}

// Writes row blocks 0 .. blocks16 - 1 of packed A.
static int launch_pack_a(int dtype, const float* a, void* packed, int m, int k, int blocks16, void* stream) {
    const int kp = mchip_pack16_k(k), pairs = kp / (2 * kFBK);
    const long long units = static_cast<long long>(blocks16) * pairs;
    const dim3 grid(static_cast<unsigned>(std::min<long long>((units + 3) / 4, 1 << 20)));
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto* out = static_cast<u32x4*>(packed);
    if (dtype == MCHIP_DTYPE_BF16) {
        hipLaunchKernelGGL((pack16_a_rows<true>), grid, dim3(256), 0, s, a, out, m, k, kp, pairs, units);
    } else {
        hipLaunchKernelGGL((pack16_a_rows<false>), grid, dim3(256), 0, s, a, out, m, k, kp, pairs, units);
    }
    return hipGetLastError();
}

extern "C" int mchip_convert_pack_a_f32(int dtype, const float* a, void* packed, int m, int k, void* stream) {
    if (dtype != MCHIP_DTYPE_BF16 && dtype != MCHIP_DTYPE_F16) return hipErrorInvalidValue;
    if (m < 1 || k < 1 || k % (2 * kFBK) != 0 || !aligned(a, 4) || !aligned(packed, 16)) return hipErrorInvalidValue;
    return launch_pack_a(dtype, a, packed, m, k, (m + kFBM - 1) / kFBM * (kFBM / 16), stream);
}

extern "C" int mchip_launch_matmul_lowp_packed(int kernel, int dtype, const void* a_packed, const void* b, float* c,
                                               int m, int n, int k, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (m < 1 || n < 1 || k < 1) return hipErrorInvalidValue;
    if (kernel == kTensorCoreTf32) return hipErrorNotSupported;
    if (!fast_eligible(a_packed, b, c, m, n, k)) return hipErrorInvalidValue;
    if (kernel == kTensorCoreBf16 && dtype == MCHIP_DTYPE_BF16) return launch_fast<true, true>(a_packed, b, c, m, n, k, s);
    if (kernel == kTensorCoreF16 && dtype == MCHIP_DTYPE_F16) return launch_fast<false, true>(a_packed, b, c, m, n, k, s);
    return hipErrorInvalidValue;
}

extern "C" int mchip_pack16_k(int k) { return (k + 2 * kFBK - 1) / (2 * kFBK) * (2 * kFBK); }

extern "C" int mchip_pack16_fits(int m, int n, int k) {
    if (m < 1 || n < 1 || k < 1 || k > (1 << 21)) return 0;  // 512 bytes per k in a band: 31-bit step offsets
    return static_cast<long long>(m) + kFBM < (1LL << 31) && static_cast<long long>(n) + kFBN < (1LL << 31) ? 1 : 0;
}

extern "C" int mchip_pack16_a_f32(int dtype, const float* a, void* packed, int m, int k, void* stream) {
    if (dtype != MCHIP_DTYPE_BF16 && dtype != MCHIP_DTYPE_F16) return hipErrorInvalidValue;
    if (!mchip_pack16_fits(m, 1, k) || !aligned(a, 4) || !aligned(packed, 16)) return hipErrorInvalidValue;
    return launch_pack_a(dtype, a, packed, m, k, (m + 15) / 16, stream);
}

extern "C" int mchip_pack16_b_f32(int dtype, const float* b, void* packed, int k, int n, void* stream) {
    if (dtype != MCHIP_DTYPE_BF16 && dtype != MCHIP_DTYPE_F16) return hipErrorInvalidValue;
    if (!mchip_pack16_fits(1, n, k) || !aligned(b, 4) || !aligned(packed, 16)) return hipErrorInvalidValue;
    const int kp = mchip_pack16_k(k);
    const long long units = static_cast<long long>((n + kFBN - 1) / kFBN) * (kp / kFBK);
    const dim3 grid(static_cast<unsigned>(std::min<long long>(units, 1 << 20)));
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto* out = static_cast<u32x4*>(packed);
    if (dtype == MCHIP_DTYPE_BF16) {
        hipLaunchKernelGGL((pack16_b<true>), grid, dim3(256), 0, s, b, out, k, n, kp, units);
    } else {
        hipLaunchKernelGGL((pack16_b<false>), grid, dim3(256), 0, s, b, out, k, n, kp, units);
    }
    return hipGetLastError();
}

extern "C" int mchip_frag_rows(int shape) { return shape == MCHIP_TWO_SUMS ? kFBM / 2 : 16 << (shape / 3); }
extern "C" int mchip_frag_cols(int shape) { return shape == MCHIP_TWO_SUMS ? kFBN : 16 << (shape % 3); }
extern "C" int mchip_frag_threads(int shape) { return shape == MCHIP_FRAG_64X64 ? 256 : 512; }

extern "C" unsigned mchip_frag_grid(int shape, int m, int n) {
    const int rows = mchip_frag_rows(shape), cols = mchip_frag_cols(shape);
    return static_cast<unsigned>(static_cast<long long>((m + rows - 1) / rows) * ((n + cols - 1) / cols));
}

// The tiles of a product on packed operands. Small tiles split K over a
// block's waves, so the widest that still gives every CU one wins (graph-timed
// on an MI355X, K = N = 4096: 128 rows 12.2 us on 64x32 tiles, 15.1 on 64x64,
// 16.9 on 64x16; 256 rows 15.5 on 64x64, 21.1 on 64x32). 64x64 tiles load an
// operand byte four times as often as 256x256 ones: 512 rows (two rounds of
// them) 29.0 us against 47.9, 1024 rows (four rounds) 62.5 against 47.8, so
// the line lies at three rounds; with at most 64 rows the 256-row tiles would
// multiply mostly padding (64 rows: 44.2 us against 10.2).
extern "C" int mchip_mfma16_packed_plan(int m, int n, int cu_count) {
    if (m > 64 && mchip_frag_grid(MCHIP_FRAG_64X64, m, n) > 3u * static_cast<unsigned>(cu_count)) return MCHIP_FRAG_NONE;
    const int shape = m <= 16 ? MCHIP_FRAG_16X16 : m <= 32 ? MCHIP_FRAG_32X16 : MCHIP_FRAG_64X16;
    for (int wider = 2; wider > 0; --wider) {
        if (mchip_frag_grid(shape + wider, m, n) >= static_cast<unsigned>(cu_count)) return shape + wider;
    }
    return shape;
}

namespace {

template <bool kBf16, int kRG, int kCG>
int launch_frag(const unsigned short* a, const unsigned short* b, float* c, int m, int n, int kp, unsigned grid,
                hipStream_t s) {
    using Cfg = McFragCfg<kRG, kCG>;
    hipLaunchKernelGGL((matmul_mfma16_frag<kBf16, Cfg>), dim3(grid), dim3(Cfg::kThreads), 0, s, a, b, c, m, n, kp);
    return hipGetLastError();
}

template <bool kBf16>
int launch_packed(int shape, const unsigned short* a, const unsigned short* b, float* c, int m, int n, int kp,
                  hipStream_t s) {
    if (shape == MCHIP_FRAG_NONE) {
        const long long tiles = static_cast<long long>((m + kFBM - 1) / kFBM) * ((n + kFBN - 1) / kFBN);
        if (tiles > 0x3fffffffLL) return hipErrorInvalidValue;
        hipLaunchKernelGGL((matmul_mfma16_packed<kBf16>), dim3(mchip_mfma16_fast_grid(m, n, device_cus())),
                           dim3(kFThreads), 0, s, a, b, c, m, n, kp);
        return hipGetLastError();
    }
    if (shape < MCHIP_TWO_SUMS || shape > MCHIP_FRAG_64X64) return hipErrorInvalidValue;
    const unsigned grid = mchip_frag_grid(shape, m, n);
    switch (shape) {
        case MCHIP_TWO_SUMS:
            hipLaunchKernelGGL((matmul_mfma16_two_sums<kBf16>), dim3(grid), dim3(kFThreads), 0, s, a, b, c, m, n, kp);
            return hipGetLastError();
        case MCHIP_FRAG_16X16: return launch_frag<kBf16, 1, 1>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_16X32: return launch_frag<kBf16, 1, 2>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_16X64: return launch_frag<kBf16, 1, 4>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_32X16: return launch_frag<kBf16, 2, 1>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_32X32: return launch_frag<kBf16, 2, 2>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_32X64: return launch_frag<kBf16, 2, 4>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_64X16: return launch_frag<kBf16, 4, 1>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_64X32: return launch_frag<kBf16, 4, 2>(a, b, c, m, n, kp, grid, s);
        case MCHIP_FRAG_64X64: return launch_frag<kBf16, 4, 4>(a, b, c, m, n, kp, grid, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

extern "C" int mchip_launch_mfma16_packed(int dtype, int shape, const void* a_packed, const void* b_packed, float* c,
                                          int m, int n, int k, void* stream) {
    if (!mchip_pack16_fits(m, n, k) || !aligned(a_packed, 16) || !aligned(b_packed, 16) || !aligned(c, 4)) {
        return hipErrorInvalidValue;
    }
    const auto* a = static_cast<const unsigned short*>(a_packed);
    const auto* b = static_cast<const unsigned short*>(b_packed);
    const int kp = mchip_pack16_k(k);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == MCHIP_DTYPE_BF16) return launch_packed<true>(shape, a, b, c, m, n, kp, s);
    if (dtype == MCHIP_DTYPE_F16) return launch_packed<false>(shape, a, b, c, m, n, kp, s);
    return hipErrorInvalidValue;
}

extern "C" int mchip_tensor_core_k_ranges(int m, int n, int k, int splits) {
    if (m < 1 || n < 1 || k < 1) return 0;
    return staged_plan(m, n, k, splits).depth;
}

extern "C" int mchip_mfma16_fast_fits(int m, int n, int k) {
    if (m < 1 || n < 8 || k < 1 || k % (2 * kFBK) != 0 || n % 8 != 0) return 0;
    return 2LL * kFBM * k < (1LL << 31) && 2LL * (static_cast<long long>(k) + kFBK) * n < (1LL << 31);
}

extern "C" unsigned mchip_mfma16_fast_grid(int m, int n, int cu_count) {
    const long long tiles = static_cast<long long>((m + kFBM - 1) / kFBM) * ((n + kFBN - 1) / kFBN);
    const long long rest = cu_count > 0 ? tiles % cu_count : 0;
    const long long halves = rest != 0 && 2 * rest <= cu_count ? rest : 0;
    return static_cast<unsigned>(tiles + halves);
}

extern "C" int mchip_matmul_supported(int kernel) { return kernel != kTensorCoreTf32; }

extern "C" int mchip_matmul_blocks_per_cu(int kernel) {
    int blocks = 0;
    hipError_t e = hipErrorInvalidValue;
    switch (kernel) {
        case kTensorCoreBf16:
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, matmul_mfma16_staged<true, true, Staged<128, 128, 2, 2, 1, 1, 2>>,
                                                             256, 0);
            break;
        case kTensorCoreF16:
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, matmul_mfma16_staged<false, true, Staged<128, 128, 2, 2, 1, 1, 2>>,
                                                             256, 0);
            break;
        default: return 2;
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return std::max(blocks, 1);
}

extern "C" int mchip_convert_f32(int dtype, const float* in, void* out, size_t count, void* stream) {
    if (dtype != MCHIP_DTYPE_BF16 && dtype != MCHIP_DTYPE_F16) return hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (count == 0) return hipSuccess;
    if (reinterpret_cast<std::uintptr_t>(in) % 16 == 0 && reinterpret_cast<std::uintptr_t>(out) % 8 == 0) {
        const std::size_t groups = count / 4;
        const int tail = static_cast<int>(count % 4);
        const std::size_t per_block = static_cast<std::size_t>(256) * kConvertItems;
        const unsigned blocks =
            static_cast<unsigned>(std::max<std::size_t>(1, std::min<std::size_t>((groups + per_block - 1) / per_block, 8192)));
        const float* tail_in = in + groups * 4;
        unsigned short* tail_out = static_cast<unsigned short*>(out) + groups * 4;
        if (dtype == MCHIP_DTYPE_BF16) {
            hipLaunchKernelGGL(convert_vec_kernel<true>, dim3(blocks), dim3(256), 0, s,
                               reinterpret_cast<const f32x4*>(in), static_cast<u16x4*>(out), groups, tail_in, tail_out,
                               tail);
        } else {
            hipLaunchKernelGGL(convert_vec_kernel<false>, dim3(blocks), dim3(256), 0, s,
                               reinterpret_cast<const f32x4*>(in), static_cast<u16x4*>(out), groups, tail_in, tail_out,
                               tail);
        }
        return hipGetLastError();
    }
    const unsigned blocks = static_cast<unsigned>(std::max<std::size_t>(1, std::min<std::size_t>((count + 255) / 256, 8192)));
    hipLaunchKernelGGL(convert_kernel, dim3(blocks), dim3(256), 0, s, in, static_cast<unsigned short*>(out), count,
                       dtype == MCHIP_DTYPE_BF16 ? 1 : 0);
    return hipGetLastError();
}
