// FP32 GEMM body for narrow tiles: C tiles of 16 kRG rows x 16 kVec columns
// (64x64 down to 16x16) on v_mfma_f32_16x16x4f32, for products too small
// or too thin to fill the chip
// with the ring body's 128x128 and 256x256 tiles (M <= 16, where B is read
// once and HBM is the bound; and products of a few million outputs or
// fewer, where small tiles give every CU a share without deep K splits).
// Shared by the ahead-of-time kernels (identity epilogue) and the GEMMs
// compiled at run time with a fused elementwise epilogue. No headers, so
// hipRTC compiles it as is; it uses the split-K helpers
// of gemm_split_arrival.h, which the includer puts before it.
//
// No LDS staging of operands: each wave loads its A and B fragments straight
// from global memory (L2 for data other waves share) into registers, all the
// loads of a batch of K before the batch's MFMAs, so a wave keeps many loads
// in flight and each group's MFMAs start as soon as that group has landed.
//
// Decomposition: logical block (x, y, z) owns columns 16 V x .. 16 V x +
// 16 V - 1, rows 16 kRG z .., and the y-th of `depth` ranges of K (k_split
// each); the grid is one-dimensional, ceil(n / 16 V) ceil(m / 16 kRG) depth
// blocks (mapped to logical blocks XCD by XCD, below); its kW
// waves cut that range into consecutive pieces, one accumulator set each.
// Lane l of a wave has k slot s = l / 16 and index c = l % 16. For each group
// of 16 k from kg the lane loads (V = kVec, 4, 2 or 1 columns per lane)
//   A[16 r + c][kg + 4s .. kg + 4s + 3]              for row group r < kRG
//   B[kg + 4s + e][col0 + V c .. col0 + V c + V - 1] for e = 0..3
// and MFMA (r, e, j) takes A load r's element e and B load e's element j:
// its k slot s is k = kg + 4s + e and its column slot c is column
// col0 + V c + j, so accumulator (r, j) holds, in lane l, C[16 r + 4s + v]
// [col0 + V c + j] for v = 0..3. The waves' tiles are then added in wave
// order through LDS (a fixed order), and the block stores its tile to C
// through the epilogue, or, with several K ranges, to its range's partial:
// with `counters`, the last of the tile's blocks to finish then adds the
// ranges' partials in range order and stores C through the epilogue
// (mc_split_last_arrival); without, a separate launch adds them.
//
// Requirements (checked by the host): k and k_split multiples of 16, n a
// multiple of kVec (the host asks for 4), A and B 16-byte aligned (C and
// the partials may be at any float address; counters: one zeroed unsigned
// per tile, in tile order). Rows past m read row m - 1 and
// columns past n the last ones of the tile (every load in bounds and at or past
// the block's origin); what they produce is not stored.
//
// The ragged form (kRagged) takes any K of 16 or more (k_split still a
// multiple of 16), any N of 4 or more and any float-aligned operands, without
// counters. Its vector accesses go to 4-byte aligned addresses, which the
// memory path takes; a chunk of columns that straddles n reads on into the
// next row, except in the last rows of K: the last wave of the block that
// holds the end of K loads its last K % 16 rows (16 when N alone is ragged)
// float by float (past the last row of K or column of N the last one, so no
// load is guarded), with zeros past K, before its other groups.
#pragma once

typedef float mc_nw_f32x4 __attribute__((ext_vector_type(4)));
typedef float mc_nw_f32x2 __attribute__((ext_vector_type(2)));

template <int N>
struct McNarrowUnits {
    static constexpr int value = N;
};

// B loads of kVec floats per lane (a 16-lane row segment of 16 kVec floats).
template <int kVec>
struct McNarrowVec;
template <>
struct McNarrowVec<1> {
    typedef float type __attribute__((ext_vector_type(1)));
    typedef float any __attribute__((ext_vector_type(1)));
};
template <>
struct McNarrowVec<4> {
    typedef mc_nw_f32x4 type;
    typedef float any __attribute__((ext_vector_type(4), aligned(4)));  // at any float address
};
template <>
struct McNarrowVec<2> {
    typedef mc_nw_f32x2 type;
    typedef float any __attribute__((ext_vector_type(2), aligned(4)));
};

// A configuration: kRG row groups of 16, kVec columns per lane and load
// (tiles of 16 kVec columns), kW waves, up to kU groups of 16 k per batch of
// loads; kStreamB: B is read by one tile row only (M <= 16), so its loads
// are non-temporal (a read-only stream reached 7.1 TB/s with them against
// 6.3 TB/s without on an MI355X). kRedRows: rows of the LDS array the waves
// add their tiles through (at least kRows); more than kRows only to keep a
// second block off the CU (LDS is 160 KiB per CU); kAcc: accumulators per
// element (a power of two), MFMA e of a group adding to accumulator e % kAcc
// (8: the groups of every second batch to the other four), summed pairwise.
template <int kRG_, int kVec_, int kW_, int kU_, bool kStreamB_, int kRedRows_ = 16 * kRG_, int kAcc_ = 1>
struct McNarrowCfg {
    static constexpr int kAcc = kAcc_;
    static constexpr int kRG = kRG_, kVec = kVec_, kW = kW_, kU = kU_;
    static constexpr bool kStreamB = kStreamB_;
    static constexpr int kRows = 16 * kRG, kCols = 16 * kVec, kThreads = 64 * kW;
    static constexpr int kRedRows = kRedRows_;
    static_assert(kRedRows >= kRows, "the reduction holds a whole tile");
};

// The configurations the library runs, 4 waves each and batches of up to 2
// groups but for the last one: 16x64 tiles for M <= 16 (B streamed), 32x64 tiles, and for
// short-K products that these would leave with half the CUs idle, 16x64 and
// 16x32 tiles. At one K range each of the 4-wave configurations adds the
// same products in the same order (per element: the 4 waves' pieces of K in
// wave order, each a chain of 16x16x4 MFMAs), so they give the same bits.
using McNarrow16 = McNarrowCfg<1, 4, 4, 2, true>;
using McNarrow32 = McNarrowCfg<2, 4, 4, 2, false>;
using McNarrow16x64 = McNarrowCfg<1, 4, 4, 2, false>;
using McNarrow16x32 = McNarrowCfg<1, 2, 4, 2, false>;
// The ragged form's 16x32 tiles past K = kNarrowSumsK: they take over from up to
// 31 ranges of the two-stage body, whose sums are more than four accumulators
// from about K = 1750 on (2-norm error in ranges / with four / with eight:
// 231x262x1677 1.93e-7 / 1.91e-7 / 1.44e-7, 74x1193x1815 1.95e-7 / 2.00e-7 /
// 1.49e-7, 444x156x2047 1.96e-7 / 2.11e-7 / 1.57e-7; 157x693x334 1.75e-7 /
// 1.00e-7 / 0.88e-7). Eight cost 0.02 to 0.2 us of 3.3 to 5.9 up to K = 1000
// (0.2 to 0.4 under a fused epilogue) and 0.04 to 0.2 of 7.3 to 13.2 past 1536
// (0.03 to 0.3).
using McNarrow16x32Sums = McNarrowCfg<1, 2, 4, 2, false, 16, 8>;
// 64x64 tiles: each operand byte a wave loads feeds 64 MFMAs per 16 k
// where 32x64 tiles feed 32 per 6 loads (1024^3 as 256 unsplit tiles). One
// block per CU: its 96 KiB reduction array leaves no room for a second.
// With 512 tiles (two per CU, 1024x2048x512) two co-resident blocks took
// 31-36 us against 22.5 us for one block per CU in two rounds.
using McNarrow64 = McNarrowCfg<4, 4, 4, 2, false, 96>;
// 16x16 tiles, eight waves: for products that any other shape would have to
// split over K ranges, and K short enough that a block's way down all of K
// (16 rows of A and 16 columns of B: 128 bytes per k) costs less than the
// ranges' sum launch (mchip_f32_narrow_plan has the figures). Eight accumulators
// per element: a wave's chain of adds is as short as with the ranges, and the
// error no larger (relative in the 2-norm, ranges / four accumulators / eight:
// 16x4096x1024 1.55e-7 / 1.20e-7 / 1.00e-7). Batches of one group: 2, 4 and 8
// groups were no faster (1x2048x1024 on an MI355X, graph-timed, one matrix /
// matrices past the MALL: 3.7 / 6.6 us against 3.7 / 6.9, 4.1 / 6.9 and
// 4.4 / 7.6).
using McNarrow16x16 = McNarrowCfg<1, 1, 8, 1, false, 16, 8>;

// A 16-, 8- or 4-byte buffer load at (voffset + soffset) from the resource's
// base; kStream: non-temporal (the slc bit: a read-only stream reached 7.1
// TB/s with non-temporal loads against 6.3 TB/s without on an MI355X).
template <typename T, bool kStream>
__device__ __forceinline__ T mc_narrow_load(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
    constexpr int kAux = kStream ? 2 : 0;
    if constexpr (sizeof(T) == 16)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, soffset, kAux));
    else if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voffset, soffset, kAux));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voffset, soffset, kAux));
}

// One batch of a wave's operands: kU groups of 16 k.
template <class Cfg>
struct McNarrowRegs {
    typedef typename McNarrowVec<Cfg::kVec>::type BV;
    mc_nw_f32x4 a[Cfg::kU][Cfg::kRG];
    BV b[Cfg::kU][4];
};

// The tile of C at (row0, col0) and its K range [kb, ke), accumulated by
// this block; the epilogue maps each value v of flat element i to what is
// stored (out = C), or the raw sums go to `out` (a partial), added in the
// launch when `counters` is given (not null).
template <class Cfg, bool kRagged = false, typename Epilogue>
__device__ __forceinline__ void mc_gemm_f32_narrow(const float* __restrict__ a, const float* __restrict__ b,
                                                   float* __restrict__ c, int m, int n, int k, int k_split,
                                                   int depth, float* __restrict__ partial, unsigned* __restrict__ counters,
                                                   const Epilogue& epilogue) {
    constexpr int kRG = Cfg::kRG, kW = Cfg::kW, kVec = Cfg::kVec, kU = Cfg::kU;
    typedef typename McNarrowVec<kVec>::type BV;
    __shared__ BV red[kW][Cfg::kRedRows][16];  // [wave][row][column chunk]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int s = lane >> 4, cl = lane & 15;
    // The grid is one-dimensional: block L runs on XCD L % 8 (the hardware
    // hands consecutive workgroups to the 8 XCDs in turn). With the count a
    // multiple of 8, XCD x takes the x-th contiguous eighth of the blocks in
    // (column tile, row tile, K range) order, or with the row tiles first
    // where B is the larger operand, so the blocks sharing an L2 share K
    // ranges of A and B (one range per XCD when there are 8) and an L2 reads
    // all of the smaller operand and a share of the larger (4 MB: on
    // an MI355X 100x2048x512 7.0 us with the columns first, 5.7 so;
    // 128x2048x1024 12.2 and 8.3).
    const int tiles_n = (n + Cfg::kCols - 1) / Cfg::kCols;
    const int tiles_m = (m + Cfg::kRows - 1) / Cfg::kRows;
    const int total = static_cast<int>(gridDim.x);
    const int L = static_cast<int>(blockIdx.x);
    const int q = total % 8 == 0 ? (L % 8) * (total / 8) + L / 8 : L;
    const bool rows_first = m < n && tiles_m > 1;
    const int inner = rows_first ? tiles_m : tiles_n;
    const int outer = rows_first ? tiles_n : tiles_m;
    const int rest = q / inner, by = rest / outer;
    const int bx = rows_first ? rest - by * outer : q - rest * inner;
    const int bz = rows_first ? q - rest * inner : rest - by * outer;
    const int col0 = bx * Cfg::kCols;
    const int row0 = bz * Cfg::kRows;
    // A lane past the last column reads the last kVec columns, or the tile's first
    // where those would begin before the tile (N no multiple of 4) and the offset
    // below its origin. With the first always, 128x6x192 took 3.6 us for 3.2.
    const int last = n - kVec > col0 ? n - kVec : col0;
    const int colc = col0 + kVec * cl < n ? col0 + kVec * cl : last;  // ragged: may straddle n

    // This wave's K range: the block's range cut into kW pieces of whole
    // 16-k groups (the last pieces may be empty).
    const int kb = by * k_split;
    const int ke = kb + k_split < k ? kb + k_split : k;
    // Ragged: the rows of K loaded float by float (the last wave's).
    const int part = kRagged ? (ke - kb) % 16 : 0;
    const int tail = kRagged && ke == k && (part != 0 || n % 4 != 0) ? (part != 0 ? part : 16) : 0;
    const int groups = (ke - kb - tail) / 16;
    const int per = (groups + kW - 1) / kW;
    const int g0 = wave * per < groups ? wave * per : groups;
    const int g1 = g0 + per < groups ? g0 + per : groups;

    // Operands through buffer loads: bases at the block's origin in A (row
    // row0, column kb) and B (row kb, column col0) in scalar registers, the
    // lane's byte offset from them in a vector register, the group's offset
    // (64 g bytes in A, 64 g n in B) in a scalar one, so no vector
    // instruction computes a load address (the host keeps every offset below
    // 2^31: mchip_f32_narrow_plan).
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a) + static_cast<long long>(row0) * k + kb, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(b) + static_cast<long long>(kb) * n + col0, 0, 0x7fffffff, 0x00020000);
    int a_off[kRG];
#pragma unroll
    for (int r = 0; r < kRG; ++r) {
        const int row = row0 + 16 * r + cl < m ? row0 + 16 * r + cl : m - 1;
        a_off[r] = 4 * ((row - row0) * k + 4 * s);
    }
    const int b_off = 4 * (4 * s * n + colc - col0);
    const int b_row = 4 * n;  // bytes per row of B

    // The ragged form keeps several accumulators too: the two-stage body it
    // replaces split K into more ranges than these tiles need, and with as
    // many partial sums the rounding error is no larger. Relative error in
    // the 2-norm and time on an MI355X, the two-stage body / one accumulator
    // / these: 449x1263x1472 2.9e-7 39.1 us / 3.5e-7 29.0 us / 2.5e-7 30.6 us,
    // 64x2032x1327 1.9e-7 19.0 us / 3.3e-7 8.7 us / 1.7e-7 8.7 us. (16x32 tiles
    // with long K: McNarrow16x32Sums.)
    constexpr int kAcc = Cfg::kAcc > 1 || !kRagged ? Cfg::kAcc : kRG * kVec <= 8 ? 4 : 2;
    mc_nw_f32x4 part_acc[kAcc][kRG][kVec] = {};
    // Loads of `units` groups from group g into x, then (after a scheduling
    // barrier: left to itself the scheduler interleaves each load with the
    // MFMAs that use it and waits for it there) nothing else.
    auto load = [&](McNarrowRegs<Cfg>& x, int g, auto units) {
        constexpr int kN = decltype(units)::value;
#pragma unroll
        for (int u = 0; u < kN; ++u) {
#pragma unroll
            for (int r = 0; r < kRG; ++r) x.a[u][r] = mc_narrow_load<mc_nw_f32x4, false>(a_rsrc, a_off[r], 64 * (g + u));
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x.b[u][e] = mc_narrow_load<BV, Cfg::kStreamB>(b_rsrc, b_off, (16 * (g + u) + e) * b_row);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // The MFMAs of `units` groups held in x: MFMA (u, e, r, j) multiplies A
    // load (u, r)'s element e by B load (u, e)'s element j. `set`: 0 or 1, the
    // register set, for eight accumulators.
    auto compute = [&](const McNarrowRegs<Cfg>& x, auto units, auto set) {
        constexpr int kN = decltype(units)::value;
        constexpr int kFirst = 4 * decltype(set)::value;
#pragma unroll
        for (int u = 0; u < kN; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int r = 0; r < kRG; ++r)
#pragma unroll
                    for (int j = 0; j < kVec; ++j)
                        part_acc[(kFirst + e) % kAcc][r][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            x.a[u][r][e], x.b[u][e][j], part_acc[(kFirst + e) % kAcc][r][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Whole batches, software-pipelined over two register sets: the loads of
    // batch i + 1 are issued before the MFMAs of batch i, so the wave keeps
    // loads in flight while its matrix core works. Every load is issued
    // unconditionally where it is issued (the last batch is peeled off): a
    // load under a condition would make the compiler wait for all loads
    // before the next MFMA. A batch is kU groups when each wave has 32 groups
    // or more and the block has one of several K ranges or 16-row tiles,
    // else one group: a short piece gains more from MFMAs that start after
    // one group's loads than from more loads in flight. Measured on an MI355X
    // (batches of 1 / 2 / 4 groups): 256x2048x512 on 32x64 tiles 7.8 / 9.0 /
    // 10.5 us, 512^3 on 16x64 tiles 5.0 / 5.2 / 6.1 us, 16x4096x4096 streamed
    // in 4 K ranges 13.4 / 13.9 / 14.4 us; with 32 groups per wave:
    // 256x256x16384 on 32x64 tiles in 8 ranges 21.7 / 21.0 / 24.9 us,
    // 256x512x2048 on 16x32 tiles 10.2 / 9.8 / 10.1 us, but 1024x512x2048 on
    // 32x64 tiles unsplit 18.5 / 20.2 us. The batching does not change the
    // order of the adds.
    McNarrowRegs<Cfg> x0, x1;
    if constexpr (kRagged) {
        // Every wave runs it, all but the block's last one on zeros: under a
        // condition the compiler kept two copies of the accumulators.
        const int mine = wave == kW - 1 ? tail : 0;
        const int rows = mine > 0 ? mine : 1;
        auto at = [&](int i) { return k - rows + (i < rows ? i : rows - 1); };
#pragma unroll
        for (int r = 0; r < kRG; ++r) {
            const int row = row0 + 16 * r + cl < m ? row0 + 16 * r + cl : m - 1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = a[static_cast<long long>(row) * k + at(4 * s + e)];
                x0.a[0][r][e] = 4 * s + e < mine ? v : 0.0f;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float* src = b + static_cast<long long>(at(4 * s + e)) * n;
#pragma unroll
            for (int j = 0; j < kVec; ++j) {
                const float v = src[colc + j < n ? colc + j : n - 1];
                x0.b[0][e][j] = 4 * s + e < mine ? v : 0.0f;
            }
        }
        compute(x0, McNarrowUnits<1>{}, McNarrowUnits<0>{});
    }
    auto pipeline = [&](auto units) {
        constexpr int kN = decltype(units)::value;
        const int batches = (g1 - g0) / kN;
        if (batches > 0) {
            int i = 0;
            load(x0, g0, units);
            for (; i + 2 < batches; i += 2) {
                load(x1, g0 + (i + 1) * kN, units);
                compute(x0, units, McNarrowUnits<0>{});
                load(x0, g0 + (i + 2) * kN, units);
                compute(x1, units, McNarrowUnits<1>{});
            }
            if (batches - i == 2) {
                load(x1, g0 + (i + 1) * kN, units);
                compute(x0, units, McNarrowUnits<0>{});
                compute(x1, units, McNarrowUnits<1>{});
            } else {
                compute(x0, units, McNarrowUnits<0>{});
            }
        }
        for (int g = g0 + batches * kN; g < g1; ++g) {
            load(x0, g, McNarrowUnits<1>{});
            compute(x0, McNarrowUnits<1>{}, McNarrowUnits<0>{});
        }
    };
    if (kU > 1 && per >= 32 && (depth > 1 || kRG == 1)) {
        pipeline(McNarrowUnits<kU>{});
    } else {
        pipeline(McNarrowUnits<1>{});
    }

    mc_nw_f32x4(&acc)[kRG][kVec] = part_acc[0];
#pragma unroll
    for (int step = 1; step < kAcc; step *= 2)
#pragma unroll
        for (int i = 0; i < kAcc; i += 2 * step)
#pragma unroll
            for (int r = 0; r < kRG; ++r)
#pragma unroll
                for (int j = 0; j < kVec; ++j) part_acc[i][r][j] += part_acc[i + step][r][j];
    // Lane l holds rows 16 r + 4s + v of column chunk cl.
#pragma unroll
    for (int r = 0; r < kRG; ++r)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            BV o;
#pragma unroll
            for (int j = 0; j < kVec; ++j) o[j] = acc[r][j][v];
            red[wave][16 * r + 4 * s + v][cl] = o;
        }
    __syncthreads();
    // The tile's chunks, summed over the waves (one accumulator: in wave order).
    const bool raw = depth > 1;
    float* __restrict__ out = raw ? partial + static_cast<long long>(by) * m * n : c;
    // C or a partial may sit at any 4-byte address (a caller's workspace):
    // then a chunk is stored float by float, the same values. Partials that
    // this launch adds go out as device-scope stores (mc_split_store).
    const bool fold = raw && counters != nullptr;
    const bool vec_out = !kRagged && (reinterpret_cast<unsigned long long>(out) & (sizeof(BV) - 1)) == 0;
    // A lane's chunks (kRows 16 / kThreads of them, 1 to 4): all summed and
    // through the epilogue before the first store, so the epilogue's operand
    // loads of every chunk are in flight together, and a per-column operand
    // (a bias: every chunk of a lane is in the same columns) is loaded once;
    // chunk by chunk, the compiler loaded it again and waited for it in each
    // chunk, after the previous chunk's store.
    constexpr int kAll = Cfg::kRows * 16;
    constexpr int kChunks = (kAll + Cfg::kThreads - 1) / Cfg::kThreads;
    static_assert(kAll % Cfg::kThreads == 0 || kChunks == 1, "a whole number of chunks per lane, or one for some lanes");
    BV sums[kChunks];
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int t = static_cast<int>(threadIdx.x) + i * Cfg::kThreads;
        if (t >= kAll) continue;
        const int r = t >> 4, ch = t & 15;
        BV sum = red[0][r][ch];
        if constexpr (kAcc > 1) {  // sums of its own: pairwise over the waves too
            BV w[kW];
#pragma unroll
            for (int i2 = 0; i2 < kW; ++i2) w[i2] = red[i2][r][ch];
#pragma unroll
            for (int step = 1; step < kW; step *= 2)
#pragma unroll
                for (int i2 = 0; i2 + step < kW; i2 += 2 * step) w[i2] += w[i2 + step];
            sum = w[0];
        } else {
#pragma unroll
            for (int w = 1; w < kW; ++w) sum += red[w][r][ch];
        }
        const int row = row0 + r, col = col0 + kVec * ch;
        if (!raw && row < m && col < n) {
            const long long at = static_cast<long long>(row) * n + col;
#pragma unroll
            for (int j = 0; j < kVec; ++j)
                if (!kRagged || col + j < n) sum[j] = epilogue(sum[j], static_cast<unsigned>(at + j));
        }
        sums[i] = sum;
    }
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int t = static_cast<int>(threadIdx.x) + i * Cfg::kThreads;
        const int r = t >> 4, ch = t & 15;
        const int row = row0 + r, col = col0 + kVec * ch;
        if (t >= kAll || row >= m || col >= n) continue;
        const long long at = static_cast<long long>(row) * n + col;
        if (fold) {
#pragma unroll
            for (int j = 0; j < kVec; ++j) mc_split_store(out + at + j, sums[i][j]);
        } else if (vec_out) {
            *reinterpret_cast<BV*>(out + at) = sums[i];
        } else if (kRagged && col + kVec <= n) {
            *reinterpret_cast<typename McNarrowVec<kVec>::any*>(out + at) = sums[i];
        } else {
#pragma unroll
            for (int j = 0; j < kVec; ++j)
                if (!kRagged || col + j < n) out[at + j] = sums[i][j];
        }
    }
    if (!fold) return;

    // The last block of the tile adds the ranges' partials, range 0 first (a
    // lane issues its loads of 8 ranges before it adds them), and stores C.
    __shared__ int last_flag;
    if (!mc_split_last_arrival(counters + bz * tiles_n + bx, depth, &last_flag)) return;
    const long long plane = static_cast<long long>(m) * n;
    const bool vec_c = (reinterpret_cast<unsigned long long>(c) & (sizeof(BV) - 1)) == 0;
    constexpr int kChunk = 8;
    for (int t = threadIdx.x; t < Cfg::kRows * 16; t += Cfg::kThreads) {
        const int r = t >> 4, ch = t & 15;
        const int row = row0 + r, col = col0 + kVec * ch;
        if (row >= m || col >= n) continue;
        const long long at = static_cast<long long>(row) * n + col;
        auto load = [&](int z) {
            const float* p = partial + z * plane + at;
            BV x;
#pragma unroll
            for (int j = 0; j < kVec; ++j) x[j] = mc_split_load(p + j);
            return x;
        };
        BV sum = load(0);
        for (int z0 = 1; z0 < depth; z0 += kChunk) {
            BV x[kChunk];
#pragma unroll
            for (int i = 0; i < kChunk; ++i) x[i] = load(z0 + i < depth ? z0 + i : depth - 1);
#pragma unroll
            for (int i = 0; i < kChunk; ++i)
                if (z0 + i < depth) sum += x[i];
        }
#pragma unroll
        for (int j = 0; j < kVec; ++j) sum[j] = epilogue(sum[j], static_cast<unsigned>(at + j));
        if (vec_c) {
            *reinterpret_cast<BV*>(c + at) = sum;
        } else {
#pragma unroll
            for (int j = 0; j < kVec; ++j) c[at + j] = sum[j];
        }
    }
}
