// C = A W^T on the matrix cores for weights in bfloat16 (v_mfma_f32_16x16x32_bf16) or float
// (v_mfma_f32_16x16x4_f32: true 32-bit products and sums).
//
// A workgroup takes a BM x BN tile, each of its waves an equal part of it in 16 x 16 pieces.  K goes in steps of 128 bytes
// per row; a step's rows are copied global -> LDS by direct 16-byte loads into one of several stages, later steps' copies in
// flight while one is multiplied.  A fragment is the same 16 bytes per lane for both types: lane l holds row l & 15,
// chunk 4 phase + (l >> 4).
//
// What bounds it: where tiles are large the card's power: 4095 x 12288 x 2048 on random data runs at 1.6 to 1.8 GHz, on zeros, whose products
// cost less of it, it takes three quarters of the time.  So what counts is that no clock goes by without a matrix op and that a product costs few reads.  A step of 256 x 256 x 64
// has 2048 clocks of matrix ops a SIMD and takes 2340; with reads and copies in bursts between them 3300, since 64 copies in a row occupy
// the CU's way to its caches for 1000 clocks; with branches around copies and 64-bit addresses 2530.  16 x 16 pieces take 3 to 5 % less than 32 x 32 at equal clocks.  Then
// the weights' first trip: tiles whose LDS has room take W a stage further ahead than A.  us, so / as bursts: 4095 x 12288 x 2048 in bfloat16
// 159 / 194, gated 168 / 203, 4095 x 2048 x 6144 82 / 105, x 2048 33 / 40, 2048^3 20.4 / 24.4, 8192^3 750 / 940 (1.47 PFLOP/s; the library 145, -, 83, 34, 21, 670).
#include <algorithm>
#include <type_traits>

#include "dense_common.h"

namespace a81w41 {
namespace {

// 16 x 16 pieces: a fragment is sixteen rows of 64 bytes, lane l holds row l & 15, chunk l >> 4.
__device__ __forceinline__ void mma(f32x4& acc, const lds16& a, const lds16& b, bf16*) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&a), *reinterpret_cast<const bf16x8*>(&b), acc, 0, 0, 0);
}
__device__ __forceinline__ void mma(f32x4& acc, const lds16& a, const lds16& b, float*) {
#pragma unroll
    for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[e]), __uint_as_float(b[e]), acc, 0, 0, 0);
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

// Lanes whose numbers differ in the given low bit trade: of a pair one gives x and takes y's place of the other.
template <int BIT>
__device__ __forceinline__ void trade(float& x, float& y) {
    const bool set = threadIdx.x & BIT;
    const float mine = set ? x : y;
    const float other = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mine), BIT == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true));
    x = set ? other : x;
    y = set ? y : other;
}
// Of G pieces side by side lane l holds column l % 16 of each; then columns 0 .. G - 1 of group l % 16 / G of piece l % G.
template <int G>
__device__ __forceinline__ void gather_columns(float (&x)[G]) {
    if constexpr (G == 4) {
        trade<1>(x[0], x[1]), trade<1>(x[2], x[3]);
        trade<2>(x[0], x[2]), trade<2>(x[1], x[3]);
    } else if constexpr (G == 2) {
        trade<1>(x[0], x[1]);
    }
}
template <int G>
__device__ __forceinline__ int gathered_column(int lane) {
    return 16 * (lane & (G - 1)) + (lane & 15 & ~(G - 1));
}
template <typename T, int G>
__device__ __forceinline__ void store_columns(void* dst, const float (&x)[G]) {  // aligned to all of them
    struct alignas(G * sizeof(T)) {
        T e[G];
    } all;
#pragma unroll
    for (int i = 0; i < G; i++) all.e[i] = (T)x[i];
    __builtin_memcpy(__builtin_assume_aligned(dst, G * sizeof(T)), &all, sizeof(all));
}

// A wave's part of a tile, FM x FN pieces of 16 x 16: register v of lane l holds row 4 (l / 16) + v, column l % 16 of a piece.  Rows from
// `rows` on are not stored.  Where the target's rows are aligned for it a lane stores G neighbouring columns at a time, sixteen lanes 16 G of a
// row: an instruction then writes whole lines, with single columns half a line of floats or a quarter of one of elements of 16 bits.
template <typename T, Epilogue EPI, int FM, int FN, typename X>
__device__ __forceinline__ void store_tile(const GemmArgs& g, const X& heads, const f32x4 (&acc)[FM][FN], int m0, int rows, int row0, int col0, long long batch) {
    const int lane = threadIdx.x & 63, l15 = lane & 15, r0 = row0 + 4 * (lane >> 4);
    if constexpr (EPI == Epilogue::kHeads || EPI == Epilogue::kQueries) {
        constexpr int G = FN < 4 ? FN : 4;
        const int pos = min(max(heads.pos_dev[0], 0), heads.max_seq - 1), pairs = turned_pairs(heads);
        if (columns_go_together(heads, g.N, G)) {
#pragma unroll
            for (int j = 0; j < FN; j += G) {
                const int col = col0 + 16 * j + gathered_column<G>(lane);
                const ColumnPlace to = column_place(heads, min(col, g.N - 1), m0 + r0, pos);
                const bool turns = __any(to.pair >= 0);
                const int high = col < g.N ? min(rows - r0, to.rows) : 0;
                float cs[2][4][G / 2], sn[2][4][G / 2];  // the rows' angles of this i and the next
                auto request = [&](int i, int to_set) {
                    if (!turns || i >= FM) return;
                    const AngleRows angles(pos, m0 + r0 + 16 * i, heads.max_seq, pairs);
                    const size_t first = angles.base + max(to.pair, 0);
#pragma unroll
                    for (int v = 0; v < 4; v++)
#pragma unroll
                        for (int p = 0; p < G / 2; p++) {
                            const size_t at = first + angles.behind(v) + (to.pair + p < pairs ? p : 0);
                            cs[to_set][v][p] = heads.cos_t[at], sn[to_set][v][p] = heads.sin_t[at];
                        }
                };
                request(0, 0);
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    if (row0 + 16 * i >= rows) break;
                    request(i + 1, (i + 1) & 1);
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        float x[G];
#pragma unroll
                        for (int e = 0; e < G; e++) x[e] = acc[i][j + e][v];
                        gather_columns<G>(x);
                        if (turns) {
#pragma unroll
                            for (int p = 0; p < G / 2; p++) {
                                const float c = cs[i & 1][v][p], n = sn[i & 1][v][p], u = x[2 * p], w = x[2 * p + 1];
                                const bool own = to.pair >= 0 && to.pair + p < pairs;
                                x[2 * p] = own ? u * c - w * n : u;
                                x[2 * p + 1] = own ? w * c + u * n : w;
                            }
                        }
                        uint8_t* dst = to.dst + (16 * i + v) * (long long)to.step;
                        if (16 * i + v < high) {
                            if (to.as_float)
                                store_columns<float, G>(dst, x);
                            else
                                store_columns<T, G>(dst, x);
                        }
                    }
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int col = col0 + 16 * j + l15;
            const ColumnPlace to = column_place(heads, min(col, g.N - 1), m0 + r0, pos);
            const int high = col < g.N ? min(rows - r0, to.rows) : 0;
#pragma unroll
            for (int i = 0; i < FM; i++) {
                if (row0 + 16 * i >= rows) break;
                const AngleRows angles(pos, m0 + r0 + 16 * i, heads.max_seq, pairs);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float x = acc[i][j][v], other = swap_neighbours(x);
                    float y = x;
                    if (to.pair >= 0) {
                        const size_t at = angles.base + angles.behind(v) + to.pair;
                        const float c = heads.cos_t[at], n = heads.sin_t[at];
                        y = to.second ? x * c + other * n : x * c - other * n;
                    }
                    uint8_t* dst = to.dst + (16 * i + v) * (long long)to.step;
                    if (16 * i + v < high) {
                        if (to.as_float)
                            *reinterpret_cast<float*>(dst) = y;
                        else
                            *reinterpret_cast<T*>(dst) = (T)y;
                    }
                }
            }
        }
        return;
    }
    // units have half as many columns as the product
    using E = std::conditional_t<EPI == Epilogue::kFloat, float, T>;
    constexpr bool kGated = EPI == Epilogue::kGatedPair;
    constexpr int kPieces = kGated ? FN / 2 : FN, G = kPieces < 4 ? kPieces : 4;
    const int N = kGated ? g.N / 2 : g.N, first = kGated ? col0 / 2 : col0;
    E* const C = static_cast<E*>(g.C) + (g.tiles ? 0 : batch * g.c_step);
    // Pieces without a row are passed by, and each way of storing is a straight run of code: few rows' launches are short, and fetch theirs anew.  us, so /
    // with every piece stored by branches for each of its rows: 1 row, 71 x 64 2.2 / 2.7, 300 x 64 2.25 / 2.8; 30 rows, 300 x 64 2.6 / 2.9.
    // Waves of more than two pieces of rows pass none by: experts' 128 x 128 tiles in float a little over one round of two a CU put three on the fullest
    // CU, with the branches often four.  A prompt of 1200 rows at width 1536, so / with them, 4650 / 5000; 2000 rows at 1024, 4300 / 4450; in bfloat16 level.
    auto store = [&](auto wide) {
#pragma unroll
        for (int i = 0; i < FM; i++) {
            if (FM <= 2 && row0 + 16 * i >= rows) break;
            float gate[4];
            if constexpr (EPI == Epilogue::kHeadGate) {
#pragma unroll
                for (int v = 0; v < 4; v++) gate[v] = sigmoid(g.head_gate[(size_t)(m0 + min(r0 + 16 * i + v, rows - 1)) * g.ld_gate + batch]);
            }
#pragma unroll
            for (int j = 0; j < kPieces; j += G) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int r = r0 + 16 * i + v;
                    float x[G];
#pragma unroll
                    for (int e = 0; e < G; e++) {
                        if constexpr (kGated)
                            x[e] = gated_unit(g.unit, acc[i][2 * (j + e)][v], acc[i][2 * (j + e) + 1][v]);
                        else if constexpr (EPI == Epilogue::kHeadGate)
                            x[e] = acc[i][j + e][v] * gate[v];
                        else
                            x[e] = acc[i][j + e][v];
                    }
                    E* const row = C + (size_t)(m0 + r) * g.ldc;
                    if constexpr (decltype(wide)::value) {
                        gather_columns<G>(x);
                        const int col = first + 16 * j + gathered_column<G>(lane);
                        if (r < rows && col < N) store_columns<E, G>(row + col, x);
                    } else {
#pragma unroll
                        for (int e = 0; e < G; e++) {
                            const int col = first + 16 * (j + e) + l15;
                            if (r < rows && col < N) row[col] = (E)x[e];
                        }
                    }
                }
            }
        }
    };
    if (((g.ldc | N) & (G - 1)) == 0 && (reinterpret_cast<uintptr_t>(C) & (G * sizeof(E) - 1)) == 0)
        store(std::true_type{});
    else
        store(std::false_type{});
}

// Rows of tiles that are walked together: an XCD's workgroups then share these rows and a few column panels in its L2.
constexpr int kBandRows = 2048;

// X: HeadRows<T> with the epilogue kHeads, LatentQueries<T> with kQueries, NoHeads with the others.  SA, SW: how many steps' rows and weights LDS holds.
// A step has two phases of 64 bytes a row.  A phase's operands are read while the phase before it is multiplied, also over the end of a step:
// the waves meet ahead of a step's second phase, whose operands are in registers by then, so that its stage is free for new copies.
// Reads and copies go one by one between the matrix ops, kFirst of a stage's copies in that second phase and the rest in the next step's
// first; requested in a row they kept every wave of the CU waiting for its turn at the caches while the matrix cores idled.  That holds where
// a CU has several workgroups as well: 64 x 64 tiles with a step's copies in a row took 1.2 to 1.3 times as long.
// WIDE: rows by 64-bit offsets, for strides with which a tile's rows reach past 4 GB.
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int SA, int SW, Epilogue EPI, typename X, bool WIDE>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void dense_gemm_kernel(GemmArgs g, X heads) {
    constexpr int kThreads = 64 * WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, FM = WM / 16, FN = WN / 16;
    constexpr int LA = BM * 8 / kThreads, LB = BN * 8 / kThreads, L = LA + LB;  // direct copies per thread and stage
    constexpr int kStageA = BM * 128, kStageW = BN * 128;
    static_assert(SA >= 2 && (SA == SW || SW == SA + 1) && SW * L < 64, "copies a wait can leave outstanding");
    __shared__ __attribute__((aligned(128))) uint8_t lds[SA * kStageA + SW * kStageW];
    uint8_t* const lds_w = lds + SA * kStageA;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l15 = lane & 15;
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
    // A tile's rows by offsets from the first, in 32 bits where tile_offsets_fit; gathered rows from the start of A
    using Offset = std::conditional_t<WIDE, size_t, unsigned>;
    const T* const A = static_cast<const T*>(g.A) + (g.tiles ? 0 : batch * g.a_step) + (g.a_rows ? 0 : (size_t)m0 * g.lda);
    const T* const W = static_cast<const T*>(g.W) + batch * g.w_step + (size_t)n0 * g.ldw;
    const CopySource from_a = copy_source(A), from_w = copy_source(W);
    Offset a_at[LA], w_at[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int c = i * kThreads + tid, r = c >> 3, row = min(r, rows - 1);
        a_at[i] = (Offset)(g.a_rows ? g.a_rows[m0 + row] : row) * (g.lda * (Offset)sizeof(T)) + (((c & 7) ^ place_of_row(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int c = i * kThreads + tid, r = c >> 3;
        w_at[i] = (Offset)min(r, g.N - 1 - n0) * (g.ldw * (Offset)sizeof(T)) + (((c & 7) ^ place_of_row(r)) << 4);
    }
    auto copy = [&](const T* base, CopySource from, uint8_t* to, Offset at, int step) {
        if constexpr (WIDE)
            copy16_to_lds(reinterpret_cast<const uint8_t*>(base) + at + (size_t)step * 128, to);
        else
            copy16_to_lds(from, to, at, step * 128);
    };
    auto copy_a = [&](int i, int step, int stage) {
        copy(A, from_a, lds + stage * kStageA + wave * 1024 + i * kThreads * 16, a_at[i], step);
    };
    auto copy_w = [&](int i, int step, int stage) {
        copy(W, from_w, lds_w + stage * kStageW + wave * 1024 + i * kThreads * 16, w_at[i], step);
    };
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wm = (wave % WAVES_M) * WM, wn = (wave / WAVES_M) * WN;
    const int n_steps = g.K * (int)sizeof(T) / 128;
    constexpr int kReads = FM + FN, kOps = FM * FN;
    lds16 a[2][FM], b[2][FN];
    const int own_row = l15 * 128, own_place[2] = {((lane >> 4) ^ place_of_row(l15)) << 4, ((4 + (lane >> 4)) ^ place_of_row(l15)) << 4};
    auto read_one = [&](int r, int phase, const uint8_t* sa, const uint8_t* sw) {  // fragment r of the phase, A's first
        if (r < FM)
            a[phase][r < FM ? r : 0] = *reinterpret_cast<const lds16*>(sa + wm * 128 + r * 2048 + own_row + own_place[phase]);
        else
            b[phase][r < FM ? 0 : r - FM] = *reinterpret_cast<const lds16*>(sw + wn * 128 + (r - FM) * 2048 + own_row + own_place[phase]);
    };
    // Of the copies that a step makes room for, A's before W's, this many go beside its second phase, the rest beside the next step's first;
    // with two stages of A all, which need the time.
    constexpr int kFirst = SA == 2 ? L : (2 * L + 2) / 3;
    // copies that a step leaves under way when it waits for the next one's
    constexpr int kAfter = (SA - 2) * L + (SW > SA ? LB : 0);
    auto copy_one = [&](int i, int step, int stage_a, int stage_w) {
        if (i < LA)
            copy_a(i < LA ? i : 0, step + SA, stage_a);
        else
            copy_w(i < LA ? 0 : i - LA, step + SW, stage_w);
    };
    // as if steps -SW .. -1 had made room: W's further stage first, and of the last of them kFirst copies
    if constexpr (SW > SA) {
#pragma unroll
        for (int i = 0; i < LB; i++) copy_w(i, 0, 0);
    }
    const bool whole = n_steps >= SW;
    for (int step = -SA; step < 0; step++)
#pragma unroll
        for (int i = 0; i < L; i++)
            if ((step < -1 || i < kFirst || !whole) && (i < LA ? step + SA : step + SW) < n_steps) copy_one(i, step, step + SA, step + SW);
    if (whole)
        wait_copies_and_meet<kAfter + kFirst>();
    else
        wait_copies_and_meet<0>();
#pragma unroll
    for (int r = 0; r < kReads; r++) read_one(r, 0, lds, lds_w);
    int step = 0, sa = 0, sw = 0;
    // REST: copies of what the step before made room for are left; A, W: this step's stages are filled again; AHEAD: copies stay under
    // way at the meeting
    auto one_step = [&](auto rest, auto fill_a, auto fill_w, auto ahead, bool more) {
        constexpr int kRest = decltype(rest)::value ? L - kFirst : 0;
        constexpr int kFillA = decltype(fill_a)::value ? kFirst : 0, kFillW = decltype(fill_w)::value ? kFirst : 0;
        const int next_a = sa + 1 < SA ? sa + 1 : 0, next_w = sw + 1 < SW ? sw + 1 : 0;
        const int before_a = sa ? sa - 1 : SA - 1, before_w = sw ? sw - 1 : SW - 1;
        auto phase = [&](auto which, int c0, int copies, int of_step, int stage_a, int stage_w, const uint8_t* from_sa, const uint8_t* from_sw) {
            constexpr int P = decltype(which)::value;
            const int all = kReads + copies;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int o = 0; o < kOps; o++) {
#pragma unroll
                for (int x = 0; x < all; x++) {
                    if ((all <= kOps ? x : x * kOps / all) != o) continue;
                    if (x < kReads)
                        read_one(x, 1 - P, from_sa, from_sw);
                    else if (P == 0 || (c0 + x - kReads < LA ? kFillA : kFillW))
                        copy_one(c0 + x - kReads, of_step, stage_a, stage_w);
                }
                mma(acc[o / FN][o % FN], a[P][o / FN], b[P][o % FN], static_cast<T*>(nullptr));
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        phase(std::integral_constant<int, 0>{}, kFirst, kRest, step - 1, before_a, before_w, lds + sa * kStageA, lds_w + sw * kStageW);
        if (more) {
            __builtin_amdgcn_sched_barrier(0);
            wait_copies_and_meet<decltype(ahead)::value ? kAfter : 0>();
        }
        phase(std::integral_constant<int, 1>{}, 0, kFillA > kFillW ? kFillA : kFillW, step, sa, sw, lds + next_a * kStageA, lds_w + next_w * kStageW);
        sa = next_a, sw = next_w;
        step++;
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    while (step < n_steps - SW) one_step(yes, yes, yes, yes, true);
    if constexpr (SW > SA) {  // the last rows of A are still to come, no more of W
        static_assert(kFirst == L, "nothing is left to the next step");
        if (whole) one_step(no, yes, no, yes, step + 1 < n_steps);
    } else {
        if (whole) one_step(yes, no, no, yes, step + 1 < n_steps);
    }
    while (step < n_steps) one_step(no, no, no, no, step + 1 < n_steps);
    store_tile<T, EPI, FM, FN>(g, heads, acc, m0, rows, wm, n0 + wn, batch);
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
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15;
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
    f32x4 acc[2][2];
#pragma unroll
    for (int o = 0; o < 4; o++) acc[o / 2][o % 2] = f32x4{0.f, 0.f, 0.f, 0.f};
    lds16 a[2][4], w[2][4];  // of a step: phase 0's two fragments, then phase 1's
    int slot_a = 0, slot_w = 0;
    auto read = [&](lds16 (&x)[4], lds16 (&y)[4]) {
        const uint8_t *pa = lds + slot_a * kStageA + wave * 4096 + l15 * 128, *pw = lds_w + slot_w * kStageW + l15 * 128;
#pragma unroll
        for (int n = 0; n < 4; n++) {
            const int at = n % 2 * 2048 + (((n / 2 * 4 + (lane >> 4)) ^ place_of_row(l15)) << 4);
            x[n] = *reinterpret_cast<const lds16*>(pa + at);
            y[n] = *reinterpret_cast<const lds16*>(pw + at);
        }
        slot_a = slot_a + 1 < SA ? slot_a + 1 : 0;
        slot_w = slot_w + 1 < SW ? slot_w + 1 : 0;
    };
    auto multiply = [&](const lds16 (&x)[4], const lds16 (&y)[4]) {
#pragma unroll
        for (int o = 0; o < 8; o++) mma(acc[o / 2 % 2][o % 2], x[o / 4 * 2 + o / 2 % 2], y[o / 4 * 2 + o % 2], static_cast<T*>(nullptr));
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
    store_tile<T, EPI, 2, 2>(g, heads, acc, m0, rows, wave * 32, n0, batch);
}

// Whether the rows of any tile, 256 x 256 at most, lie within the 32 bits of its copies' offsets.  Rows that a_rows gathers are among a pass's.
bool tile_offsets_fit(const GemmArgs& g, size_t element) {
    const size_t rows_a = g.a_rows ? kPassRows : std::min(g.M, 256), rows_w = std::min(g.N, 256);
    return std::max(rows_a * g.lda, rows_w * g.ldw) * element < (size_t)1 << 32;
}

// The kernels of a product without a list of tiles.  One is chosen by an estimate of its time, fitted to what each of them took.
using Form = GemmForm;
struct FormTime {
    Form form;
    int rows, cols, per_cu;  // the tile, and how many of them fit a CU
    // us: of a launch; of each tile of the CU that has most of them, and of each of the tile's steps of K; of each round of per_cu tiles a CU
    float launch, tile, step, round, round_step;
    // more of a step's time where one row of tiles streams weights whose rows are whole multiples of 4 KB apart and meet in the same channels of the
    // caches: 1 row, 32768 x 4096 61 us with 64 x 128 tiles, 53 with 64 x 64; 30241 x 6336 72 and 71
    float aligned;
};
// Fitted to what every form took on 3402 products of 1 to 4096 rows, 64 to 65536 columns and 64 to 12288 of K in bfloat16 and 2101 of 1 to 4096,
// 64 to 16384 and 32 to 8192 in float, the weights from memory as a pass finds them; about half of them drawn evenly in the logarithm of each size, the
// rest with the whole multiples of 256 and 512 that models have.  The form chosen takes 1.003 (bfloat16) and 1.001 (float) of the time of the best one
// for the product on average, 61 and 5 of them more than 1.05 of it; a fit to two thirds does as well on the other third.
constexpr FormTime kTimesBf16[] = {{Form::k256x256, 256, 256, 1, 0.372f, 9.751f, 0.889f, 0, 0, 0.7f},
                                   {Form::k128x256, 128, 256, 1, 0.116f, 5.816f, 0.599f, 0, 0, 1.04f},
                                   {Form::k128x128, 128, 128, 1, 0.729f, 4.659f, 0.397f, 0, 0, 0.64f},
                                   {Form::k64x128, 64, 128, 2, 2.947f, 1.193f, 0.261f, 0.064f, 0.076f, 1.1f},
                                   {Form::kFew, 64, 32, 1, 1.397f, 1.887f, 0.163f, 0, 0, 0.05f},
                                   {Form::k64x64FourStages, 64, 64, 2, 1.556f, 0.263f, 0.153f, 1.98f, 0.06f, 0.47f},
                                   {Form::k64x64TwoStages, 64, 64, 5, 3.121f, 0.194f, 0.155f, 0.352f, 0.122f, 1.03f}};
// The matrix ops of a step are 16 times as long in float and hide everything else: larger tiles gain nothing and round worse.
constexpr FormTime kTimesFloat[] = {{Form::kFew, 64, 32, 1, 0.322f, 2.436f, 0.504f, 0, 0, 0},
                                    {Form::k64x64FourStages, 64, 64, 2, 2.612f, 0.922f, 0.44f, 0.486f, 0.073f, 0},
                                    {Form::k64x64TwoStages, 64, 64, 5, 3.134f, 0.774f, 0.427f, 0.029f, 0.103f, 0}};

template <size_t N>
Form fastest_form(const FormTime (&times)[N], const GemmArgs& g, size_t element) {
    constexpr long long kCus = 256;
    const int steps = g.K * (int)element / 128;
    const bool aligned = g.M <= 64 && g.ldw * element % 4096 == 0;
    Form best{};
    float least = INFINITY;
    for (const FormTime& f : times) {
        const long long tiles = (long long)((g.M + f.rows - 1) / f.rows) * ((g.N + f.cols - 1) / f.cols) * g.batches;
        // What no term of it says: over long K five to sixteen rows of 64 x 128 tiles that leave three eighths of the CUs without one are slower than
        // 64 x 64.  13 such products, 64 x 64 / 64 x 128: 0.90 on average, from 0.78 to 1.06; 500 rows, 2112 x 4096 24.7 / 31.1 us, 800 rows, 1536 x 4608
        // 27.6 / 34.9.
        if (f.form == Form::k64x128 && tiles <= 160 && steps >= 32 && g.M > 256 && g.M <= 1024) continue;
        const float most = (tiles + kCus - 1) / kCus, rounds = (tiles + kCus * f.per_cu - 1) / (kCus * f.per_cu);
        const float of_steps = steps * (aligned ? 1 + f.aligned : 1);
        const float time = f.launch + most * (f.tile + f.step * of_steps) + rounds * (f.round + f.round_step * of_steps);
        if (time < least) least = time, best = f.form;
    }
    return best;
}

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int SA, int SW, Epilogue EPI, bool WIDE = false, typename X>
hipError_t launch_kernel(const GemmArgs& g, const X& heads, hipStream_t s) {
    const int n_mt = g.tiles ? g.max_tiles : (g.M + BM - 1) / BM, n_nt = (g.N + BN - 1) / BN;
    hipLaunchKernelGGL((dense_gemm_kernel<T, BM, BN, WAVES_M, WAVES_N, SA, SW, EPI, X, WIDE>), dim3(n_mt * n_nt, g.batches),
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
        if (10 * tiles >= 7 * 256 * rounds) return launch_kernel<T, kGroupTileManyRows, 256, 2, 4, 3, 3, EPI>(g, heads, s);
        return launch_kernel<T, kGroupTileManyRows, 128, 2, 2, 2, 2, EPI>(g, heads, s);
    }
    // 64 x 128 tiles with two stages fit a CU three times, with three stages twice and have more of the weights under way, which counts where
    // there are few rounds.  us of gate and up with two / three: 600 tokens of 4 out of 32, 2048 x 2048 82.4 / 72.3, 64 tokens 62.5 / 60.0,
    // 16 tokens, 1024 x 1024 13.4 / 10.9.  Past the line prompts of 760 to 1020 tokens at width 2048 take 0.96 to 0.98 of the time with three as
    // well; where 512 to 768 tiles are there, one round with two stages and two with three, 830 to 1020 tokens at width 1024 take 1.01 to 1.02 of it.
    if (g.N >= 1024) {
        if (g.max_tiles * panels(128) <= 1200) return launch_kernel<T, kGroupTileRows, 128, 2, 4, 3, 3, EPI>(g, heads, s);
        return launch_kernel<T, kGroupTileRows, 128, 2, 2, 2, 2, EPI>(g, heads, s);
    }
    // Four stages fit a CU twice, two stages five times: past 512 tiles the first go in rounds.  kTimesBf16 has 7.0 / 7.3 us for 512 tiles
    // of 8 steps, 10.9 / 8.8 for 513.
    if (g.max_tiles * panels(64) > 512) return launch_kernel<T, kGroupTileRows, 64, 2, 2, 2, 2, EPI>(g, heads, s);
    return launch_kernel<T, kGroupTileRows, 64, 2, 2, 4, 4, EPI>(g, heads, s);
}

template <typename T>
Form form_of(const GemmArgs& g) {
    if (!tile_offsets_fit(g, sizeof(T))) return Form::kWide;
    if constexpr (sizeof(T) == 2) return fastest_form(kTimesBf16, g, sizeof(T));
    else return fastest_form(kTimesFloat, g, sizeof(T));
}

template <typename T, Epilogue EPI, typename X>
hipError_t launch_by_size(const GemmArgs& g, const X& heads, hipStream_t s) {
    // strides of 16 MB and more; a list's tiles of 64 rows fit those of 128
    if (!tile_offsets_fit(g, sizeof(T))) return launch_kernel<T, 128, 128, 2, 2, 2, 2, EPI, true>(g, heads, s);
    if (g.tiles) {
        if constexpr (EPI == Epilogue::kGatedPair || EPI == Epilogue::kFloat) return launch_grouped<T, EPI>(g, heads, s);
        return hipErrorInvalidValue;
    }
    const Form form = form_of<T>(g);
    if constexpr (sizeof(T) == 2) {
        if (form == Form::k256x256) return launch_kernel<T, 256, 256, 2, 4, 2, 3, EPI>(g, heads, s);
        if (form == Form::k128x256) return launch_kernel<T, 128, 256, 2, 4, 3, 3, EPI>(g, heads, s);
        if (form == Form::k128x128) return launch_kernel<T, 128, 128, 2, 4, 4, 4, EPI>(g, heads, s);
        if (form == Form::k64x128) return launch_kernel<T, 64, 128, 2, 4, 3, 3, EPI>(g, heads, s);
    }
    if (form == Form::kFew) return launch_few<T, EPI>(g, heads, s);
    if (form == Form::k64x64TwoStages) return launch_kernel<T, 64, 64, 2, 2, 2, 2, EPI>(g, heads, s);
    return launch_kernel<T, 64, 64, 2, 2, 4, 4, EPI>(g, heads, s);
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

GemmForm dense_gemm_form(const GemmArgs& g, bool is_bf16) { return is_bf16 ? form_of<bf16>(g) : form_of<float>(g); }

}  // namespace a81w41
