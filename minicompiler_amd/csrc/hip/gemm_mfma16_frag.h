// bf16 / fp16 matrix-core GEMM body for products too small to fill the chip
// with the 256x256 tiles of gemm_mfma16_fast.h: C tiles of 16 kRG rows x
// 16 kCG columns (16 to 64 each way) on v_mfma_f32_16x16x32, both operands
// packed (the layouts of gemm_mfma16_fast.h, which the includer puts before
// this file). Shared by the ahead-of-time kernels and the GEMMs compiled at
// run time with a fused epilogue. No headers, so hipRTC compiles it as is.
//
// What bounds these products: at few rows B's bytes (every block reads its
// columns of B once), else the latency of too few blocks. So K is not split
// over blocks (no partials, no second launch) but over the kW waves of a
// block, and no operand goes through LDS: in the packed layout a 16-row (or
// 16-column) by 32-k fragment is 1 KiB in lane order, so one buffer load per
// fragment, whole lines, brings a lane exactly its MFMA operand, and a wave
// keeps two batches of kU steps of loads in flight with no barrier in its
// loop. The waves' tiles are added through LDS in wave order (a fixed order).
//
// Measured on an MI355X, graph-timed, K = N = 4096, bf16, against the 256x256
// tiles on the same packed operands (16 blocks, 32 as halves): 1 row 7.5 us
// (16x16 tiles, 33.5 MB of B: 4.5 TB/s; 8.8 with B past the MALL) against
// 42.9; 32 rows 8.2 against 43.4; 256 rows 15.5 against 46.1; 512 rows 29.0
// against 47.9.
#pragma once

template <int kRG_, int kCG_>
struct McFragCfg {
    static constexpr int kRG = kRG_, kCG = kCG_;
    static constexpr int kRows = 16 * kRG, kCols = 16 * kCG;
    // Eight waves; four for the 64x64 tiles (16 KiB of LDS per wave, two
    // blocks per CU).
    static constexpr int kW = kRG * kCG == 16 ? 4 : 8;
    static constexpr int kThreads = 64 * kW;
    // Steps of 32 k per batch: 10 to 16 loads of 1 KiB.
    static constexpr int kU = kRG + kCG <= 2 ? 8 : kRG + kCG <= 4 ? 4 : 2;
    // Accumulators per element, taken by the steps in turn and added at the end.
    // The operator cuts K into up to 256 / t ranges for t tiles of 128x128, more
    // than the waves where t is small, which is where the one-fragment-wide tiles
    // run; with two accumulators their error is no larger for K up to 4096
    // (2-norm, fp16, 16x2048x4095: 1.28e-7 in 16 ranges, 1.55e-7 with the waves
    // alone, 1.21e-7 so). Four cost 32 and 64 rows the second block per CU (more
    // than 128 VGPRs; 32x4096x8000 16.4 us against 15.1). The wider tiles are
    // picked only for at most as many ranges as they have waves.
    static constexpr int kAcc = kCG == 1 ? 2 : 1;
};

// Which of the two register sets a batch is in, as a type.
template <int kSet>
struct McFragSet {
    static constexpr int value = kSet;
};

template <class Cfg>
struct McFragRegs {
    mc_u16x8_t a[Cfg::kU][Cfg::kRG];
    mc_u16x8_t b[Cfg::kU][Cfg::kCG];
};

// Plain loads: non-temporal ones for B gained 4% where the weights of a
// program do not fit the 256 MB MALL (8.4 against 8.8 us) and lost 10-25% where
// they do (8.3 against 7.5 us at one row, 10.8 against 8.3 at 32).
__device__ __forceinline__ mc_u16x8_t mc_frag_load(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
    return __builtin_bit_cast(mc_u16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, soffset, 0));
}

// The grid is one-dimensional, one block per tile; k is the padded one (a
// multiple of 64). The epilogue maps each value v of element i = row n + col
// to what is stored. Rows past m and columns past n of the last tiles are
// read (inside the operands' padding to 256) and not stored.
template <bool kBf16, class Cfg, typename Epilogue>
__device__ __forceinline__ void mc_gemm16_frag(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b,
                                               float* __restrict__ c, int m, int n, int k, const Epilogue& epilogue) {
    constexpr int kRG = Cfg::kRG, kCG = Cfg::kCG, kW = Cfg::kW, kU = Cfg::kU;
    __shared__ mc_f32x4_t red[kW][kRG * kCG][64];
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    // Block L runs on XCD L % 8; with the count a multiple of 8, XCD x takes
    // the x-th contiguous eighth of the tiles, row tiles fastest, so the
    // blocks that read the same columns of B share an L2.
    const int tiles_m = (m + Cfg::kRows - 1) / Cfg::kRows;
    const int total = static_cast<int>(gridDim.x), L = static_cast<int>(blockIdx.x);
    const int q = total % 8 == 0 ? (L % 8) * (total / 8) + L / 8 : L;
    const int row0 = (q % tiles_m) * Cfg::kRows, col0 = (q / tiles_m) * Cfg::kCols;

    // Fragment (row block r, step s) is 1 KiB at 1024 r + 16 KiB s from the
    // tile's origin in A's band; B likewise. The lane's 16 bytes of it sit in
    // the vector offset, the step in the scalar one.
    const long long a0 = static_cast<long long>(row0 / kFBM) * kFBM * k + (row0 % kFBM) * kFBK;
    const long long b0 = static_cast<long long>(col0 / kFBN) * kFBN * k + (col0 % kFBN) * kFBK;
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a) + a0, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(b) + b0, 0, 0x7fffffff, 0x00020000);
    const int voff = 16 * lane;
    constexpr int kStepBytes = kFBM * kFBK * 2;

    // This wave's steps of 32 k.
    const int steps = k / kFBK;
    const int per = (steps + kW - 1) / kW;
    const int s0 = mc_min16(wave * per, steps), s1 = mc_min16(s0 + per, steps);

    constexpr int kAcc = Cfg::kAcc;
    mc_f32x4_t part[kAcc][kRG][kCG];
#pragma unroll
    for (int x = 0; x < kAcc; ++x)
#pragma unroll
        for (int r = 0; r < kRG; ++r)
#pragma unroll
            for (int g = 0; g < kCG; ++g) part[x][r][g] = mc_f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // The loads of the batch from step s (steps past the wave's last load the
    // last again: a load under a condition would make the compiler wait for
    // every load in flight), then nothing else (a scheduling barrier).
    auto load = [&](McFragRegs<Cfg>& x, int s) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int at = mc_min16(s + u, s1 - 1) * kStepBytes;
#pragma unroll
            for (int g = 0; g < kCG; ++g) x.b[u][g] = mc_frag_load(b_rsrc, voff + 1024 * g, at);
#pragma unroll
            for (int r = 0; r < kRG; ++r) x.a[u][r] = mc_frag_load(a_rsrc, voff + 1024 * r, at);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // B as the first operand: C^T fragments, so a lane holds four
    // consecutive columns of one row.
    auto multiply = [&](const McFragRegs<Cfg>& x, int u, auto set) {
        const int to = (decltype(set)::value * kU + u) % kAcc;  // known once unrolled
#pragma unroll
        for (int r = 0; r < kRG; ++r)
#pragma unroll
            for (int g = 0; g < kCG; ++g) part[to][r][g] = mc_mfma16<kBf16>(x.b[u][g], x.a[u][r], part[to][r][g]);
    };
    auto whole = [&](const McFragRegs<Cfg>& x, auto set) {
#pragma unroll
        for (int u = 0; u < kU; ++u) multiply(x, u, set);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto last = [&](const McFragRegs<Cfg>& x, int s, auto set) {
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (s + u < s1) multiply(x, u, set);
    };
    // Two register sets: the loads of batch i + 1 are issued before the MFMAs
    // of batch i.
    McFragRegs<Cfg> x0, x1;
    if (s0 < s1) {
        int s = s0;
        load(x0, s);
        for (; s + 2 * kU < s1; s += 2 * kU) {
            load(x1, s + kU);
            whole(x0, McFragSet<0>{});
            load(x0, s + 2 * kU);
            whole(x1, McFragSet<1>{});
        }
        if (s + kU < s1) {
            load(x1, s + kU);
            whole(x0, McFragSet<0>{});
            last(x1, s + kU, McFragSet<1>{});
        } else {
            last(x0, s, McFragSet<0>{});
        }
    }

    mc_f32x4_t(&acc)[kRG][kCG] = part[0];
#pragma unroll
    for (int step = 1; step < kAcc; step *= 2)
#pragma unroll
        for (int x = 0; x < kAcc; x += 2 * step)
#pragma unroll
            for (int r = 0; r < kRG; ++r)
#pragma unroll
                for (int g = 0; g < kCG; ++g) part[x][r][g] += part[x + step][r][g];
#pragma unroll
    for (int r = 0; r < kRG; ++r)
#pragma unroll
        for (int g = 0; g < kCG; ++g) red[wave][r * kCG + g][lane] = acc[r][g];
    __syncthreads();
    // The tile's 16-byte chunks, summed over the waves in wave order: every
    // chunk of a lane summed and through the epilogue before the first store,
    // so the epilogue's operand loads are in flight together.
    constexpr int kAll = kRG * kCG * 64;
    constexpr int kChunks = (kAll + Cfg::kThreads - 1) / Cfg::kThreads;
    mc_f32x4_t sums[kChunks];
    auto row_of = [&](int t) { return row0 + 16 * ((t >> 6) / kCG) + (t & 15); };
    auto col_of = [&](int t) { return col0 + 16 * ((t >> 6) % kCG) + 4 * ((t >> 4) & 3); };
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int t = static_cast<int>(threadIdx.x) + i * Cfg::kThreads;
        if (t >= kAll) continue;
        mc_f32x4_t sum = red[0][t >> 6][t & 63];
#pragma unroll
        for (int w = 1; w < kW; ++w) sum += red[w][t >> 6][t & 63];
        const int row = row_of(t), col = col_of(t);
        if (row < m && col < n) {
            const unsigned at = static_cast<unsigned>(row) * static_cast<unsigned>(n) + static_cast<unsigned>(col);
            if (n % 4 == 0 || col + 4 <= n) {  // a condition per chunk, as in fast_store
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] = epilogue(sum[e], at + e);
            } else {
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (col + e < n) sum[e] = epilogue(sum[e], at + e);
            }
        }
        sums[i] = sum;
    }
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int t = static_cast<int>(threadIdx.x) + i * Cfg::kThreads;
        if (t >= kAll) continue;
        const int row = row_of(t), col = col_of(t);
        if (row >= m || col >= n) continue;
        float* dst = c + static_cast<long long>(row) * n + col;
        if (col + 4 <= n) {
            *reinterpret_cast<mc_f32x4u_t*>(dst) = sums[i];
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (col + e < n) dst[e] = sums[i][e];
        }
    }
}
