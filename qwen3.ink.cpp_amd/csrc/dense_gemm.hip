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
// waited for ahead of every step's first LDS read (see lds16), 209 us = 0.99 PFLOP/s with 256 x 256.  4095 x 2048 x 6144: 146 us and
// 104 us, 2048 x 2048 x 2048: 46 us and 25 us.
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
    if constexpr (EPI == Epilogue::kHeads || EPI == Epilogue::kQueries) {
        // The column's place once, then, where the piece has columns that turn, the rows' angles all at a time; a piece without skips
        // them, and rows follow by adding.  2048 x 3104 x 2048 with kHeads, 64 of 128 columns of a head turning: 51.5 us with an address
        // for every element, 45.7 so.  4095 x 3072 x 768 with kQueries, 64 of 192: 38.7 us; in 32 bits first and turned by a launch of
        // its own 32.6 + 21.5 us, with an address for every element no less than that.
        const int pos = min(max(heads.pos_dev[0], 0), heads.max_seq - 1);
        const ColumnPlace to = column_place(heads, min(col, g.N - 1), m0 + r0, pos);
        const bool turns = __any(to.pair >= 0);
        float cs[NV], sn[NV];
        if (turns) {
            const AngleRows angles(pos, m0 + r0, heads.max_seq, turned_pairs(heads));
            const size_t first = angles.base + max(to.pair, 0);
            const float *cos_t = heads.cos_t + first, *sin_t = heads.sin_t + first;
#pragma unroll
            for (int v = 0; v < NV; v++) {
                const int i = angles.behind(8 * (v >> 2) + (v & 3));
                cs[v] = cos_t[i], sn[v] = sin_t[i];
            }
        }
        uint8_t* dst = to.dst;
        const int high = col < g.N ? min(rows - r0, to.rows) : 0;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            if (v) dst += (v & 3) ? to.step : 5 * to.step;
            float y = x[v];
            if (turns) {
                const float other = swap_neighbours(y), turned = to.second ? y * cs[v] + other * sn[v] : y * cs[v] - other * sn[v];
                y = to.pair >= 0 ? turned : y;
            }
            if (8 * (v >> 2) + (v & 3) < high) {
                if (to.as_float)
                    *reinterpret_cast<float*>(dst) = y;
                else
                    *reinterpret_cast<T*>(dst) = (T)y;
            }
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

// X: HeadRows<T> with the epilogue kHeads, LatentQueries<T> with kQueries, NoHeads with the others.  STAGES: how many steps LDS holds; all but one are under way.
// PIPE: a step's operands are read one 16-byte column ahead of their products, also into the next step: the waves meet before a step's
// last products, whose operands are in registers by then, so that its stage is free for new copies and the next step's first
// reads run beside those products.  4095 x 12288 x 2048 into floats: 211 us with the meeting between two steps, 204 so.  Without PIPE the other workgroup of the CU fills the wait.
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool PIPE, Epilogue EPI, typename X>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void dense_gemm_kernel(GemmArgs g, X heads) {
    constexpr int kThreads = 64 * WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, FM = WM / 32, FN = WN / 32;
    constexpr int LA = BM * 8 / kThreads, LB = BN * 8 / kThreads;  // direct copies per thread and stage
    constexpr int kStage = (BM + BN) * 128;
    static_assert(STAGES >= 2 && (STAGES - 1) * (LA + LB) < 64, "copies a wait can leave outstanding");
    __shared__ __attribute__((aligned(128))) uint8_t lds[STAGES * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l31 = lane & 31, half = lane >> 5;
    // Tiles dealt to the XCDs in contiguous runs, in bands of kBandRows rows and inside one column panel after the other.  A grouped
    // product's go expert by expert, column panel by column panel: an XCD then reads the rows of a few experts once and their weights
    // once.  With the rows of all experts for one panel after the other (8192 rows of 4 KB, 32 experts, 16 panels) the rows were read from
    // behind the L2 again for every panel, 512 MB beside 268 MB of weights: 133.6 us, so 127.4.
    const int n_nt = (g.N + BN - 1) / BN, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int all = g.tiles ? *g.n_tiles * n_nt : gridDim.x, q = all >> 3, r8 = all & 7;
    if (idx >= q + (xcd < r8 ? 1 : 0)) return;
    const int t = xcd * q + min(xcd, r8) + idx;
    int m0, rows, nt;
    long long batch = blockIdx.y;
    if (g.tiles) {
        const GroupTile gt = g.tiles[t / n_nt];
        const int count = (gt.rows + BM - 1) / BM, at = t - gt.first * n_nt, skip = at % count * BM;
        nt = at / count;
        m0 = gt.row0 + skip;
        rows = gt.rows - skip;
        batch = gt.expert;
    } else {
        const int n_mt = all / n_nt, band = kBandRows / BM, first = t / (band * n_nt) * band;
        const int high = min(band, n_mt - first), at = t - first * n_nt;
        m0 = (first + at % high) * BM;
        nt = at / high;
        rows = g.M - m0;
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
    lds16 a[2][FM], b[2][FN];
    auto read = [&](int kk, const uint8_t* sa) {
        const uint8_t* sb = sa + BM * 128;
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
    auto multiply = [&](int kk) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) mma(acc[i][j], a[kk & 1][i], b[kk & 1][j], static_cast<T*>(nullptr));
    };
    if constexpr (PIPE) {
        for (int step = 0; step < STAGES && step < n_steps; step++) copy_step(step, step);
        if (n_steps >= STAGES)
            wait_copies_and_meet<(STAGES - 1) * (LA + LB)>();
        else
            wait_copies_and_meet<0>();
        read(0, lds);
        int stage = 0;
        for (int step = 0; step < n_steps; step++) {
            const uint8_t* sa = lds + stage * kStage;
            const int next = stage + 1 < STAGES ? stage + 1 : 0;
#pragma unroll
            for (int kk = 0; kk < 3; kk++) {
                __builtin_amdgcn_sched_barrier(0);
                read(kk + 1, sa);
                __builtin_amdgcn_sched_barrier(0);
                multiply(kk);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (step + 1 < n_steps) {
                if (step + STAGES <= n_steps)
                    wait_copies_and_meet<(STAGES - 2) * (LA + LB)>();
                else
                    wait_copies_and_meet<0>();
                if (step + STAGES < n_steps) copy_step(step + STAGES, stage);
                read(0, lds + next * kStage);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(3);
            stage = next;
        }
    } else {
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
            stage = stage + 1 < STAGES ? stage + 1 : 0;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                read(kk, sa);
                multiply(kk);
            }
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
    const int t = xcd * q + min(xcd, r8) + idx;
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

// Grouped products: the row tiles' height is that of the list.
template <typename T, Epilogue EPI, typename X>
hipError_t launch_grouped(const GemmArgs& g, const X& heads, hipStream_t s) {
    auto panels = [&](int width) { return (long long)((g.N + width - 1) / width); };
    if (g.tile_rows == kGroupTileManyRows) {
        // One 128 x 256 tile on a CU where its rounds of 256 come out seven tenths full or more, half of the experts' last tiles being
        // there, otherwise two 128 x 128.  us of gate and up + down, the second / the first: 2048 tokens of 4 experts out of 32, 2048 x 2048
        // 128.7 + 70.5 / 128.5 + 68.7, 1536 x 1536 74.2 + 44.8 / 74.6 + 41.3; 0.63 of two rounds full, 1024 x 1024 45.4 + 27.4 / 47.6 + 28.2.
        const int whole = g.M / kGroupTileManyRows;
        const long long tiles = (whole + g.max_tiles) / 2 * panels(256), rounds = (tiles + 255) / 256;
        if (10 * tiles >= 7 * 256 * rounds) return launch_kernel<T, kGroupTileManyRows, 256, 2, 4, 3, true, EPI>(g, heads, s);
        return launch_kernel<T, kGroupTileManyRows, 128, 2, 2, 2, true, EPI>(g, heads, s);
    }
    // 64 x 128 tiles with two stages fit a CU three times, with three stages twice and have more of the weights under way, which counts where
    // there are few rounds.  us of gate and up with two / three: 600 tokens of 4 out of 32, 2048 x 2048 82.4 / 72.3, 64 tokens 62.5 / 60.0,
    // 16 tokens, 1024 x 1024 13.4 / 10.9.  Past the line prompts of 760 to 1020 tokens at width 2048 take 0.96 to 0.98 of the time with three as
    // well; where 512 to 768 tiles are there, one round with two stages and two with three, 830 to 1020 tokens at width 1024 take 1.01 to 1.02 of it.
    if (g.N >= 1024) {
        if (g.max_tiles * panels(128) <= 1200) return launch_kernel<T, kGroupTileRows, 128, 2, 4, 3, true, EPI>(g, heads, s);
        return launch_kernel<T, kGroupTileRows, 128, 2, 2, 2, true, EPI>(g, heads, s);
    }
    // see launch_by_size: 1000 tiles, 512 x 512 14.7 us with four stages, 11.6 with two
    if (g.max_tiles * panels(64) > 512) return launch_kernel<T, kGroupTileRows, 64, 2, 2, 2, false, EPI>(g, heads, s);
    return launch_kernel<T, kGroupTileRows, 64, 2, 2, 4, false, EPI>(g, heads, s);
}

template <typename T, Epilogue EPI, typename X>
hipError_t launch_by_size(const GemmArgs& g, const X& heads, hipStream_t s) {
    if (g.tiles) {
        if constexpr (EPI == Epilogue::kGatedPair || EPI == Epilogue::kFloat) return launch_grouped<T, EPI>(g, heads, s);
        return hipErrorInvalidValue;
    }
    auto tiles = [&](int rows, int cols) { return (long long)((g.M + rows - 1) / rows) * ((g.N + cols - 1) / cols) * g.batches; };
    // One round of a tile for each CU, three quarters full or more; a tile has the larger one's stages and waves, so that its rows and
    // weights are under way early.  That takes some steps of K to pay: before the last of them are under way nothing fills the CU.
    auto one_round = [&](int rows, int cols) { return g.M > 64 && tiles(rows, cols) >= 192 && tiles(rows, cols) <= 256; };
    const int steps = g.K * (int)sizeof(T) / 128;
    if constexpr (sizeof(T) == 2)
        if (large_tiles_preferred(tiles(256, 256), tiles(128, 128), g.K)) return launch_kernel<T, 256, 256, 2, 4, 2, true, EPI>(g, heads, s);
    // us, so / with 128 x 128 tiles: 4095 rows, 2048 x 2048 39.6 / 41.1, 2048 x 6144 106 / 109; 2048 rows, 3104 x 2048 36.3 / 40.4.
    // Over 45 drawn shapes a type, on average: bfloat16 up to 10 steps 1.02 of the time and up to 1.075 (1854 rows, 4203 x 640 21.4 /
    // 20.1), 11 and more 0.98; float up to 4 steps 1.05 (951 rows, 6073 x 64 16.4 / 15.2), 6 and more 0.98.
    if (steps >= (sizeof(T) == 2 ? 11 : 6) && one_round(128, 256)) return launch_kernel<T, 128, 256, 2, 4, 3, true, EPI>(g, heads, s);
    // 2048^3: 24.8 us with twice the waves and four stages, 33 us as two a CU
    if (one_round(128, 128)) return launch_kernel<T, 128, 128, 2, 4, 4, true, EPI>(g, heads, s);
    if (g.M > 64 && tiles(128, 128) > 256) {
        // 300 rows, 12288 x 2048 26.7 / 36.8
        if (one_round(64, 256)) return launch_kernel<T, 64, 256, 2, 4, 3, true, EPI>(g, heads, s);
        return launch_kernel<T, 128, 128, 2, 2, 2, false, EPI>(g, heads, s);
    }
    // us, so / with 64 x 64 tiles: 1024 rows, 2048 x 2048 15.2 / 16.0, x 6144 45.1 / 49.2; 600 rows, 3072 x 1536 12.2 / 13.4; 180 rows, 9216
    // x 1536 14.6 / 16.3; over 45 drawn shapes 0.98 on average, with one and two steps 1.03 (2674 rows, 553 x 128 5.8 / 5.5)
    if (steps > 2 && one_round(64, 128)) return launch_kernel<T, 64, 128, 2, 4, 3, true, EPI>(g, heads, s);
    // So few tiles of 64 x 32 that no CU gets a second one (us, against 64 x 64 tiles with four stages): 33 rows, 784 x 2048 7.7 /
    // 12.5, 2048 x 6144 19 / 31; 256 rows, 2048 x 2048 10.2 / 13.5; with a second one 300 rows, 2048 x 2048 17.2 / 13.8, and 33
    // rows, 12288 x 2048 20 / 16.
    if (tiles(64, 32) <= 256) return launch_few<T, EPI>(g, heads, s);
    // 64 x 64 tiles with four stages fit a CU twice, with two stages five times: more tiles than 512 would go in rounds.  bfloat16,
    // us with four / two: 1030 rows, 544 tiles, 2048 x 1024 15.9 / 12.2, 2048 x 6144 63 / 50; in one round, 400 rows, 448 tiles, 4096 x
    // 4096 27.5 / 34.  float, 1030 rows, 2048 x 1024: 60.5 / 56.9.
    if (tiles(64, 64) > 512) return launch_kernel<T, 64, 64, 2, 2, 2, false, EPI>(g, heads, s);
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
        case Epilogue::kHeads:
        case Epilogue::kQueries: break;  // have launchers of their own
    }
    return hipErrorInvalidValue;
}
template <typename T>
hipError_t launch_dense_gemm_heads(const GemmArgs& g, const HeadRows<T>& heads, hipStream_t s) {
    return launch_by_size<T, Epilogue::kHeads>(g, heads, s);
}
template <typename T>
hipError_t launch_dense_gemm_queries(const GemmArgs& g, const LatentQueries<T>& q, hipStream_t s) {
    return launch_by_size<T, Epilogue::kQueries>(g, q, s);
}
#define INSTANTIATE(T)                                                                                \
    template hipError_t launch_dense_gemm<T>(const GemmArgs&, Epilogue, hipStream_t);                   \
    template hipError_t launch_dense_gemm_heads<T>(const GemmArgs&, const HeadRows<T>&, hipStream_t); \
    template hipError_t launch_dense_gemm_queries<T>(const GemmArgs&, const LatentQueries<T>&, hipStream_t);
INSTANTIATE(bf16)
INSTANTIATE(float)

}  // namespace a81w41
