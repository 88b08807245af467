// C = A W^T on the matrix cores for weights in bfloat16 (v_mfma_f32_32x32x16_bf16) or float
// (v_mfma_f32_32x32x2_f32: true 32-bit products and sums).
//
// A workgroup takes a BM x BN tile, each of its waves an equal part of it in 32 x 32 pieces.  K goes in steps of 128 bytes
// per row; a step's rows are copied global -> LDS by direct 16-byte loads into one of STAGES stages, later steps' copies in
// flight while one is multiplied.  A fragment is the same 16 bytes per lane for both types: lane l holds row l & 31,
// chunk 2 kk + (l >> 5).
//
// What bounds it: bytes per product.  A 128 x 128 tile asks the L2 for 64 bytes a clock and CU at the matrix cores' full rate,
// which is all the L2 gives, and reads LDS as fast as LDS goes; a 256 x 256 tile asks for half of the one and three quarters of
// the other.  4095 x 12288 x 2048 in bfloat16 with the gated epilogue: 340 us with 128 x 128 tiles whose copies the compiler
// waited for ahead of every step's first LDS read (see lds16), 215 us = 960 TFLOP/s with 256 x 256.  4095 x 2048 x 6144: 146 us and
// 115 us, 2048 x 2048 x 2048: 46 us and 27 us.
#include <type_traits>

#include "dense_common.h"

namespace a81w41 {
namespace {

__device__ __forceinline__ void mma(f32x16& acc, const lds16& a, const lds16& b, bf16*) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(&a), *reinterpret_cast<const bf16x8*>(&b), acc, 0, 0, 0);
}
__device__ __forceinline__ void mma(f32x16& acc, const lds16& a, const lds16& b, float*) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[0]), __uint_as_float(b[0]), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[1]), __uint_as_float(b[1]), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[2]), __uint_as_float(b[2]), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[3]), __uint_as_float(b[3]), acc, 0, 0, 0);
}

struct NoHeads {};

// Chunk c of row r sits at place c ^ this: sixteen rows read at one chunk column then cover the 256 bytes of all banks.
__device__ __forceinline__ int place_of_row(int r) { return (r >> 1) & 7; }

// the value of the lane whose number differs in the lowest bit
__device__ __forceinline__ float swap_neighbours(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
}
// At most PENDING of this wave's vector-memory operations are outstanding, and none of its LDS reads.
template <int PENDING>
__device__ __forceinline__ void wait_copies() {
    __builtin_amdgcn_s_waitcnt((PENDING & 15) | (PENDING >> 4) << 14 | 0x0070);
    asm volatile("" ::: "memory");
}
// The same of every wave of the workgroup.
template <int PENDING>
__device__ __forceinline__ void wait_copies_and_meet() {
    wait_copies<PENDING>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// NV registers of a 32 x 32 product: register v of lane l holds row 8 (v / 4) + 4 (l / 32) + v % 4 from row0 on, column l % 32 from
// col0 on; rows from `rows` on are not stored.
template <typename T, Epilogue EPI, int NV, typename V, typename X>
__device__ __forceinline__ void store_piece(const GemmArgs& g, const X& heads, const V& x, int m0, int rows, int row0, int col0, long long batch) {
    const int lane = threadIdx.x & 63, col = col0 + (lane & 31), r0 = row0 + 4 * (lane >> 5);
    if constexpr (EPI == Epilogue::kGatedPair) {
        // Lanes 16 .. 31 and 48 .. 63 hold the ups of the 16 lanes before them.  Of two rows v, v + 1 the gates of the second and the
        // ups of the first trade places: every lane then has both of one row, and no unit is formed twice.
        const int odd = (lane >> 4) & 1;
        T* dst = static_cast<T*>(g.C) + (col >> 5) * 16 + (col & 15);
#pragma unroll
        for (int v = 0; v < NV; v += 2) {
            const auto both = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[v]), __float_as_uint(x[v + 1]), false, false);
            const float unit = gated_unit(g.unit, __uint_as_float(both[0]), __uint_as_float(both[1]));
            const int r = r0 + 8 * (v >> 2) + (v & 3) + odd;
            if (r < rows && col < g.N) dst[(size_t)(m0 + r) * g.ldc] = (T)unit;
        }
        return;
    }
    if constexpr (EPI == Epilogue::kHeads) {
        // the column's place once, then the rows' angles all at a time
        const HeadColumn<T> to(heads, min(col, g.N - 1));
        const int pos = min(max(heads.pos_dev[0], 0), heads.max_seq - 1);
        float cs[NV], sn[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) to.angle(min(m0 + r0 + 8 * (v >> 2) + (v & 3), g.M - 1), pos, cs[v], sn[v]);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int r = r0 + 8 * (v >> 2) + (v & 3);
            const float other = swap_neighbours(x[v]);
            if (r < rows && col < g.N) to.store(m0 + r, pos, x[v], other, cs[v], sn[v]);
        }
        return;
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int r = r0 + 8 * (v >> 2) + (v & 3);
        const size_t row = m0 + r;
        if (r < rows && col < g.N) {
            if constexpr (EPI == Epilogue::kFloat) {
                (static_cast<float*>(g.C) + (g.tiles ? 0 : batch * g.c_step))[row * g.ldc + col] = x[v];
            } else {
                float f = x[v];
                if constexpr (EPI == Epilogue::kHeadGate) f *= sigmoid(g.head_gate[row * g.ld_gate + batch]);
                (static_cast<T*>(g.C) + (g.tiles ? 0 : batch * g.c_step))[row * g.ldc + col] = (T)f;
            }
        }
    }
}

// Rows of tiles that are walked together: an XCD's workgroups then share these rows and a few column panels in its L2.
constexpr int kBandRows = 2048;

// X: HeadRows<T> with the epilogue kHeads, NoHeads with the others.  STAGES: how many steps LDS holds; all but one are under way.
// PIPE: a step's operands are read one 16-byte column ahead of their products; without it the other workgroup of the CU
// fills the wait.
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool PIPE, Epilogue EPI, typename X>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void dense_gemm_kernel(GemmArgs g, X heads) {
    constexpr int kThreads = 64 * WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, FM = WM / 32, FN = WN / 32;
    constexpr int LA = BM * 8 / kThreads, LB = BN * 8 / kThreads;  // direct copies per thread and stage
    constexpr int kStage = (BM + BN) * 128;
    static_assert(STAGES >= 2 && (STAGES - 2) * (LA + LB) < 64, "copies a wait can leave outstanding");
    __shared__ __attribute__((aligned(128))) uint8_t lds[STAGES * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l31 = lane & 31, half = lane >> 5;
    // Tiles dealt to the XCDs in contiguous runs, in bands of kBandRows rows and inside one column panel after the other; a
    // grouped product's in the order (column panel, row tile): a panel's weights come into one L2.
    const int n_nt = (g.N + BN - 1) / BN, n_mt = gridDim.x / n_nt;
    const int q = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int t = xcd < r8 ? xcd * (q + 1) + idx : r8 * (q + 1) + (xcd - r8) * q + idx;
    const int band = g.tiles ? n_mt : kBandRows / BM, first = t / (band * n_nt) * band;
    const int high = min(band, n_mt - first), at = t - first * n_nt;
    const int mt = first + at % high, nt = at / high;
    int m0 = mt * BM, rows = g.M - m0;
    long long batch = blockIdx.y;
    if (g.tiles) {
        if (mt >= *g.n_tiles) return;
        const GroupTile gt = g.tiles[mt];
        m0 = gt.row0;
        rows = gt.rows;
        batch = gt.expert;
    }
    const int n0 = nt * BN;
    const uint8_t* A = reinterpret_cast<const uint8_t*>(static_cast<const T*>(g.A) + (g.tiles ? 0 : batch * g.a_step));
    const uint8_t* W = reinterpret_cast<const uint8_t*>(static_cast<const T*>(g.W) + batch * g.w_step);
    const uint8_t *a_src[LA], *b_src[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int c = i * kThreads + tid, r = c >> 3;
        int row = m0 + min(r, rows - 1);
        if (g.a_rows) row = g.a_rows[row];
        a_src[i] = A + (size_t)row * g.lda * sizeof(T) + (((c & 7) ^ place_of_row(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int c = i * kThreads + tid, r = c >> 3;
        b_src[i] = W + (size_t)min(n0 + r, g.N - 1) * g.ldw * sizeof(T) + (((c & 7) ^ place_of_row(r)) << 4);
    }
    auto copy_step = [&](int step, int stage) {
        uint8_t* base = lds + stage * kStage + wave * 1024;
#pragma unroll
        for (int i = 0; i < LA; i++) copy16_to_lds(a_src[i] + (size_t)step * 128, base + i * kThreads * 16);
#pragma unroll
        for (int i = 0; i < LB; i++) copy16_to_lds(b_src[i] + (size_t)step * 128, base + BM * 128 + i * kThreads * 16);
    };
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
    const int wm = (wave % WAVES_M) * WM, wn = (wave / WAVES_M) * WN;
    const int n_steps = g.K * (int)sizeof(T) / 128;
    for (int step = 0; step < STAGES - 1 && step < n_steps; step++) copy_step(step, step);
    int stage = 0;
    for (int step = 0; step < n_steps; step++) {
        // the copies of the step are in LDS, later ones may be under way; and nobody still reads the stage before it
        if (step + STAGES - 2 < n_steps)
            wait_copies_and_meet<(STAGES - 2) * (LA + LB)>();
        else
            wait_copies_and_meet<0>();
        if (step + STAGES - 1 < n_steps) copy_step(step + STAGES - 1, stage ? stage - 1 : STAGES - 1);
        const uint8_t* sa = lds + stage * kStage;
        const uint8_t* sb = sa + BM * 128;
        stage = stage + 1 < STAGES ? stage + 1 : 0;
        lds16 a[2][FM], b[2][FN];
        auto read = [&](int kk) {
#pragma unroll
            for (int i = 0; i < FM; i++) {
                const int r = wm + i * 32 + l31;
                a[kk & 1][i] = *reinterpret_cast<const lds16*>(sa + r * 128 + (((2 * kk + half) ^ place_of_row(r)) << 4));
            }
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int r = wn + j * 32 + l31;
                b[kk & 1][j] = *reinterpret_cast<const lds16*>(sb + r * 128 + (((2 * kk + half) ^ place_of_row(r)) << 4));
            }
        };
        if constexpr (PIPE) read(0);
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            if constexpr (PIPE) __builtin_amdgcn_sched_barrier(0);
            if (!PIPE) read(kk);
            if (PIPE && kk < 3) read(kk + 1);
            if constexpr (PIPE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) mma(acc[i][j], a[kk & 1][i], b[kk & 1][j], static_cast<T*>(nullptr));
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) store_piece<T, EPI, 16>(g, heads, acc[i][j], m0, rows, wm + i * 32, n0 + wn + j * 32, batch);
}

// Few rows, so few tiles that a CU has one at most: what counts is that the weights are under way and that a step is short.  64
// rows and 32 columns a workgroup of six waves: two multiply 32 rows each, reading a step's operands beside the products of the step
// before, two copy A nine steps ahead, two copy W 19 steps ahead.  A wave that copies and multiplies takes 0.3 us a step
// however much is under way, these 0.13 us (a trip to memory of 2.4 us in 19 steps, one to the L2 of 0.9 us in nine).  The sums go
// in the order of the other kernels.  33 rows, 784 x 2048: 28 us with 64 x 64 tiles and one step's copies waited for at once, 8.8 us
// here; 2048 x 6144: 81 us and 19 us.  Cutting K between waves is no faster (7.5 and 20 us) and sums in another order.
template <typename T, Epilogue EPI, typename X>
__global__ __launch_bounds__(384, 1) void dense_gemm_few_kernel(GemmArgs g, X heads) {
    constexpr int SA = 10, SW = 20, kStageA = 64 * 128, kStageW = 32 * 128;
    __shared__ __attribute__((aligned(128))) uint8_t lds[SA * kStageA + SW * kStageW];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l31 = lane & 31, half = lane >> 5;
    // row tiles of a column panel next to each other on one XCD
    const int n_mt = (g.M + 63) / 64;
    const int q = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int t = xcd < r8 ? xcd * (q + 1) + idx : r8 * (q + 1) + (xcd - r8) * q + idx;
    const int m0 = t % n_mt * 64, n0 = t / n_mt * 32, rows = g.M - m0, n_steps = g.K * (int)sizeof(T) / 128;
    const long long batch = blockIdx.y;
    const int copy_row = (wave & 1) * (wave < 4 ? 32 : 16) + (lane >> 3);  // of the wave's first copy
    auto swapped = [&](int i) { return ((lane & 7) ^ place_of_row(copy_row + 8 * i)) << 4; };
    uint8_t* const lds_w = lds + SA * kStageA;
    if (wave >= 2) {  // COPIES a step and wave, 8 rows each, into a ring of S stages
        auto run = [&](auto copies, auto stages, const uint8_t* (&src)[4], uint8_t* ring, int stage_bytes) {
            constexpr int COPIES = decltype(copies)::value, S = decltype(stages)::value;
            uint8_t* to = ring + (wave & 1) * COPIES * 1024;
            auto copy_step = [&](int slot) {
#pragma unroll
                for (int i = 0; i < COPIES; i++) {
                    copy16_to_lds(src[i], to + slot * stage_bytes + i * 1024);
                    src[i] += 128;
                }
            };
            for (int step = 0; step < S - 1 && step < n_steps; step++) copy_step(step);
            int slot = S - 1;
            for (int step = 0; step < n_steps; step++) {
                if (step + S - 2 < n_steps)
                    wait_copies_and_meet<(S - 2) * COPIES>();
                else
                    wait_copies_and_meet<0>();
                if (step + S - 1 < n_steps) copy_step(slot);
                slot = slot + 1 < S ? slot + 1 : 0;
            }
        };
        const uint8_t* src[4];
        if (wave < 4) {
            const uint8_t* A = reinterpret_cast<const uint8_t*>(static_cast<const T*>(g.A) + batch * g.a_step);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int row = m0 + min(copy_row + 8 * i, rows - 1);
                if (g.a_rows) row = g.a_rows[row];
                src[i] = A + (size_t)row * g.lda * sizeof(T) + swapped(i);
            }
            run(std::integral_constant<int, 4>{}, std::integral_constant<int, SA>{}, src, lds, kStageA);
        } else {
            const uint8_t* W = reinterpret_cast<const uint8_t*>(static_cast<const T*>(g.W) + batch * g.w_step);
#pragma unroll
            for (int i = 0; i < 2; i++) src[i] = W + (size_t)min(n0 + copy_row + 8 * i, g.N - 1) * g.ldw * sizeof(T) + swapped(i);
            run(std::integral_constant<int, 2>{}, std::integral_constant<int, SW>{}, src, lds_w, kStageW);
        }
        return;
    }
    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = 0.f;
    lds16 a[2][4], w[2][4];
    int slot_a = 0, slot_w = 0;
    auto read = [&](lds16 (&x)[4], lds16 (&y)[4]) {
        const uint8_t *pa = lds + slot_a * kStageA + wave * 4096 + l31 * 128, *pw = lds_w + slot_w * kStageW + l31 * 128;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int at = ((2 * kk + half) ^ place_of_row(l31)) << 4;
            x[kk] = *reinterpret_cast<const lds16*>(pa + at);
            y[kk] = *reinterpret_cast<const lds16*>(pw + at);
        }
        slot_a = slot_a + 1 < SA ? slot_a + 1 : 0;
        slot_w = slot_w + 1 < SW ? slot_w + 1 : 0;
    };
    auto multiply = [&](const lds16 (&x)[4], const lds16 (&y)[4]) {
#pragma unroll
        for (int kk = 0; kk < 4; kk++) mma(acc, x[kk], y[kk], static_cast<T*>(nullptr));
    };
    // meet: the step is in LDS; its reads then run beside the products of the step before
    wait_copies_and_meet<0>();
    read(a[0], w[0]);
    for (int step = 1; step < n_steps; step += 2) {
        wait_copies_and_meet<0>();
        read(a[1], w[1]);
        multiply(a[0], w[0]);
        if (step + 1 < n_steps) {
            wait_copies_and_meet<0>();
            read(a[0], w[0]);
        }
        multiply(a[1], w[1]);
    }
    if (n_steps & 1) multiply(a[0], w[0]);
    store_piece<T, EPI, 16>(g, heads, acc, m0, rows, wave * 32, n0, batch);
}

// 256 x 256 tiles, one workgroup per CU, or 128 x 128, two per CU.  At K = 2048 a round of 256 large tiles takes 65 us whether
// it is full or not, small tiles 44 us per 512 of them.  Over several rounds small ones overlap the end of one with the start of the
// next, which counts where rounds are short: with exactly 768 of them a round, us with small / large, 2047 rows, 12288 x 1024 66 / 69,
// x 2048 117 / 120, x 4096 227 / 224; 3000 rows, 8192 x 512 40.8 / 43.2, x 2048 118 / 122, x 6144 331 / 329.  With a few more they
// begin one more round (2048 rows, 12320 x 2048, 776 a round, 131 / 125); one round, 2047 rows, 6144 x 1024 39.8 / 36.4.
bool large_tiles_preferred(long long large, long long small, int K) {
    const long long rounds = (large + 255) / 256;
    return rounds * (rounds > 1 && K <= 2048 ? 769 : 750) <= small;
}

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool PIPE, Epilogue EPI, typename X>
hipError_t launch_kernel(const GemmArgs& g, const X& heads, hipStream_t s) {
    const int n_mt = g.tiles ? g.max_tiles : (g.M + BM - 1) / BM, n_nt = (g.N + BN - 1) / BN;
    hipLaunchKernelGGL((dense_gemm_kernel<T, BM, BN, WAVES_M, WAVES_N, STAGES, PIPE, EPI, X>), dim3(n_mt * n_nt, g.batches),
                       dim3(64 * WAVES_M * WAVES_N), 0, s, g, heads);
    return hipGetLastError();
}

template <typename T, Epilogue EPI, typename X>
hipError_t launch_few(const GemmArgs& g, const X& heads, hipStream_t s) {
    hipLaunchKernelGGL((dense_gemm_few_kernel<T, EPI, X>), dim3((g.M + 63) / 64 * ((g.N + 31) / 32), g.batches), dim3(384), 0, s, g, heads);
    return hipGetLastError();
}

template <typename T, Epilogue EPI, typename X>
hipError_t launch_by_size(const GemmArgs& g, const X& heads, hipStream_t s) {
    auto tiles = [&](int size) { return (long long)((g.M + size - 1) / size) * ((g.N + size - 1) / size) * g.batches; };
    // A product of 192 to 256 tiles of 128 x 128 has one for a CU: it takes twice the waves and four stages in LDS (2048^3: 29 us
    // against 36 us with two).  Fewer give too few CUs work.  A grouped product's row tiles are kGroupTileRows high.
    if constexpr (sizeof(T) == 2)
        if (!g.tiles && large_tiles_preferred(tiles(256), tiles(128), g.K)) return launch_kernel<T, 256, 256, 2, 4, 2, true, EPI>(g, heads, s);
    if (!g.tiles && g.M > 64 && tiles(128) > 256) return launch_kernel<T, 128, 128, 2, 2, 2, false, EPI>(g, heads, s);
    if (!g.tiles && g.M > 64 && tiles(128) >= 192) return launch_kernel<T, 128, 128, 2, 4, 4, true, EPI>(g, heads, s);
    if (g.tiles && g.N >= 1024) return launch_kernel<T, kGroupTileRows, 128, 2, 2, 2, false, EPI>(g, heads, s);
    // So few tiles of 64 x 32 that no CU gets a second one (us, against 64 x 64 tiles with four stages): 33 rows, 784 x 2048 7.7 /
    // 12.5, 2048 x 6144 19 / 31; 256 rows, 2048 x 2048 10.2 / 13.5; with a second one 300 rows, 2048 x 2048 17.2 / 13.8, and 33
    // rows, 12288 x 2048 20 / 16.
    const long long few = (long long)((g.N + 31) / 32) * ((g.M + 63) / 64) * g.batches;
    if (!g.tiles && few <= 256) return launch_few<T, EPI>(g, heads, s);
    // 64 x 64 tiles with four stages fit a CU twice, with two stages five times: more tiles than 512 would go in rounds.  bfloat16,
    // us with four / two: 1030 rows, 544 tiles, 2048 x 1024 15.9 / 12.2, 2048 x 6144 63 / 50; 1000 grouped tiles, 512 x 512 14.7 /
    // 11.6; in one round, 400 rows, 448 tiles, 4096 x 4096 27.5 / 34.  float, 1030 rows, 2048 x 1024: 60.5 / 56.9.
    const long long tiles64 = (long long)(g.tiles ? g.max_tiles : (g.M + 63) / 64) * ((g.N + 63) / 64) * g.batches;
    if (tiles64 > 512) return launch_kernel<T, 64, 64, 2, 2, 2, false, EPI>(g, heads, s);
    return launch_kernel<T, 64, 64, 2, 2, 4, false, EPI>(g, heads, s);
}

}  // namespace

template <typename T>
hipError_t launch_dense_gemm(const GemmArgs& g, Epilogue epi, hipStream_t s) {
    switch (epi) {
        case Epilogue::kFloat: return launch_by_size<T, Epilogue::kFloat>(g, NoHeads{}, s);
        case Epilogue::kElement: return launch_by_size<T, Epilogue::kElement>(g, NoHeads{}, s);
        case Epilogue::kGatedPair: return launch_by_size<T, Epilogue::kGatedPair>(g, NoHeads{}, s);
        case Epilogue::kHeadGate: return launch_by_size<T, Epilogue::kHeadGate>(g, NoHeads{}, s);
        case Epilogue::kHeads: break;  // has a launcher of its own
    }
    return hipErrorInvalidValue;
}
template <typename T>
hipError_t launch_dense_gemm_heads(const GemmArgs& g, const HeadRows<T>& heads, hipStream_t s) {
    return launch_by_size<T, Epilogue::kHeads>(g, heads, s);
}
#define INSTANTIATE(T)                                                              \
    template hipError_t launch_dense_gemm<T>(const GemmArgs&, Epilogue, hipStream_t); \
    template hipError_t launch_dense_gemm_heads<T>(const GemmArgs&, const HeadRows<T>&, hipStream_t);
INSTANTIATE(bf16)
INSTANTIATE(float)

}  // namespace a81w41
