// Attention on the matrix cores over key rows that hold the values too: the work of a workgroup, for the kernels of its own
// (attend_mfma.hip, which says how it goes) and beside another product (dense_gemv.hip).
#pragma once
#include "dense_common.h"

namespace a81w41 {
namespace attend {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLowest = -1e30f;

// DK, DV: capacities for all and for value columns of a tile row; the scores take its columns from KEY0 on (rows form: the
// key part, 0 otherwise).  KT keys per tile, NBUF tiles in LDS.
// COLS (few rows): all four waves take the same query rows; each scores its 16 keys of a tile, the scores meet in LDS,
// and each sums its quarter of the value columns.
// blocks: row groups, heads, shares; at: the workgroup's.  lds: attend_lds(DK, KT, NBUF) bytes, scores: attend_scores(QS, KT) floats for COLS.
__host__ __device__ constexpr int attend_lds(int dk, int kt, int nbuf) { return nbuf * kt * dk * 2; }
__host__ __device__ constexpr int attend_scores(int qs, int kt) { return kt * (16 * qs + 4); }
template <int DK, int DV, int KEY0, int WAVES, int QS, int KT, int NBUF, bool COLS>
__device__ __forceinline__ void attend_workgroup(const AttendArgs<bf16>& a, const dim3& blocks, const dim3& at, uint8_t* lds, float* scores) {
    constexpr int CK = DK / 8;                    // 16-byte chunks of a key row
    constexpr int kBuf = KT * DK * 2;
    constexpr int KS = (DK - KEY0) / 32, VF = DV / 16 / (COLS ? WAVES : 1), kRows = 16 * QS * (COLS ? 1 : WAVES);
    static_assert(DK % 64 == 0 && KEY0 % 32 == 0 && DV % (COLS ? 16 * WAVES : 16) == 0 && KT % 32 == 0, "tile sizes");
    constexpr int kScoreRow = 16 * QS + 4;  // floats of a key's scores in LDS: lane groups fall into different banks
    static_assert(!COLS || KT == 16 * WAVES, "a wave scores 16 keys of a tile");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l15 = lane & 15, g = lane >> 4;
    const int row_wave = COLS ? 0 : wave, f0 = COLS ? wave * VF : 0;  // first 16 value columns of this wave
    const int z = at.y;
    // the longest rows first
    const int row0 = ((int)blocks.x - 1 - (int)at.x) * kRows;
    const int pos = min(max(a.pos_dev[0], 0), a.max_seq - 1);
    const int last_row = min(row0 + kRows, a.rows) - 1;
    const int wg_keys = min(pos + last_row / a.rows_per_token, a.max_seq - 1) + 1;  // keys any row of the workgroup sees
    auto chunk_begin = [&](int key) { return a.chunk ? key - key % a.chunk : 0; };
    int key_begin = chunk_begin(min(pos + row0 / a.rows_per_token, a.max_seq - 1)), key_end = wg_keys;
    if (a.splits > 1) {
        const int from = chunk_begin(pos), all = min(pos + (a.rows - 1) / a.rows_per_token, a.max_seq - 1) + 1 - from;
        const int share = ((all + a.splits - 1) / a.splits + KT - 1) / KT * KT, begin = from + (int)at.z * share;
        key_end = min(begin + share, wg_keys);
        key_begin = min(max(begin, key_begin), key_end);
    }
    const bf16* k_own = a.k_own + z * a.k_own_head;
    const int own_chunks = a.k_own_width >> 3;
    auto copy_tile = [&](int key0, int buf) {
        uint8_t* base = lds + buf * kBuf;
        for (int n = wave; n < KT * CK / 64; n += WAVES) {
            const int q = n * 64 + lane, r = q / CK, c = (q % CK) ^ (r & 7);
            const size_t key = min(key0 + r, wg_keys - 1);
            const bf16* src = k_own + key * a.ld_k_own;
            if constexpr (KEY0 > 0) {
                if (c < KEY0 / 8)
                    src += c < (a.v_width >> 3) ? c * 8 : 0;
                else if (c - KEY0 / 8 < own_chunks)
                    src += a.v_width + (c - KEY0 / 8) * 8;
            } else if (c < own_chunks)
                src += c * 8;
            copy16_to_lds(src, base + n * 1024);
        }
    };
    // query operands
    bf16x8 qf[QS][KS];
    int limit[QS], first[QS];  // last and first visible key of this lane's query
#pragma unroll
    for (int s = 0; s < QS; s++) {
        const int r = row0 + (row_wave * QS + s) * 16 + l15, rc = min(r, a.rows - 1);
        const int token = rc / a.rows_per_token, last = min(pos + token, a.max_seq - 1);
        limit[s] = r < a.rows ? last : -1;
        first[s] = chunk_begin(last);
        const bf16* src = a.q + z * a.q_head + (size_t)token * a.q_token + (rc - token * a.rows_per_token) * a.ld_q;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            uint4 u = make_uint4(0, 0, 0, 0);
            const int c = k * 4 + g;
            if (c < own_chunks) u = *reinterpret_cast<const uint4*>(src + c * 8);
            qf[s][k] = *reinterpret_cast<const bf16x8*>(&u);
        }
    }
    f32x4 acc[QS][VF];
    float mx[QS], sum[QS];
#pragma unroll
    for (int s = 0; s < QS; s++) {
        const bool sink = a.sink && (a.splits == 1 || at.z == 0);  // one lane group of one share counts it
        mx[s] = sink ? 0.f : kLowest;
        sum[s] = sink && g == 0 ? 1.f : 0.f;
#pragma unroll
        for (int f = 0; f < VF; f++) acc[s][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // Values that are columns of the key rows come by transposing reads (ds_read_b64_tr_b16): in a group of 16 lanes lane
    // i names four columns of key 4 g + i / 4 and receives its own column of the four keys.  The exclusive or of the chunk
    // places touches the low three bits of 2 f + ..., so four offsets serve all f.
    int value_at[4];
#pragma unroll
    for (int f = 0; f < 4; f++) {
        const int r = 4 * g + (l15 >> 2);
        value_at[f] = r * (DK * 2) + (((2 * (f0 + f) + ((l15 >> 1) & 1)) ^ (r & 7)) << 4) + (l15 & 1) * 8;
    }
    const float scale = a.scale * kLog2e;
    const int n_tiles = (key_end - key_begin + KT - 1) / KT;
    if (NBUF > 1 && n_tiles > 0) copy_tile(key_begin, 0);
    for (int tile = 0; tile < n_tiles; tile++) {
        const int key0 = key_begin + tile * KT;
        if (NBUF == 1) {
            if (tile) __syncthreads();  // nobody still reads the tile
            copy_tile(key0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        if (NBUF > 1 && tile + 1 < n_tiles) copy_tile(key0 + KT, (tile + 1) % NBUF);
        const uint8_t* kb = lds + (tile % NBUF) * kBuf;
        f32x4 sc[QS][KT / 16];
        auto score = [&](int t) {
#pragma unroll
            for (int s = 0; s < QS; s++) sc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            const uint8_t* row = kb + ((COLS ? wave : t) * 16 + l15) * (DK * 2);
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const bf16x8 kf = *reinterpret_cast<const bf16x8*>(row + (((KEY0 / 8 + k * 4 + g) ^ (l15 & 7)) << 4));
#pragma unroll
                for (int s = 0; s < QS; s++) sc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s][k], sc[s][t], 0, 0, 0);
            }
        };
        if constexpr (COLS) {
            score(0);
#pragma unroll
            for (int s = 0; s < QS; s++)
#pragma unroll
                for (int i = 0; i < 4; i++) scores[(wave * 16 + 4 * g + i) * kScoreRow + s * 16 + l15] = sc[s][0][i];
            dense_lds_barrier();
#pragma unroll
            for (int s = 0; s < QS; s++)
#pragma unroll
                for (int t = 0; t < KT / 16; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) sc[s][t][i] = scores[(t * 16 + 4 * g + i) * kScoreRow + s * 16 + l15];
        } else {
#pragma unroll
            for (int t = 0; t < KT / 16; t++) score(t);
        }
        bf16x8 pf[QS][KT / 32];
#pragma unroll
        for (int s = 0; s < QS; s++) {
            float m = mx[s];
#pragma unroll
            for (int t = 0; t < KT / 16; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int key = key0 + t * 16 + 4 * g + i;
                    const float v = sc[s][t][i] * scale;
                    sc[s][t][i] = key <= limit[s] && key >= first[s] && key < key_end ? v : kLowest;
                    m = fmaxf(m, sc[s][t][i]);
                }
            m = fmaxf(m, __shfl_xor(m, 16, 64));
            m = fmaxf(m, __shfl_xor(m, 32, 64));
            const float keep = exp2f(mx[s] - m);
            float add = 0.f;
#pragma unroll
            for (int t = 0; t < KT / 16; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float p = sc[s][t][i] > kLowest ? exp2f(sc[s][t][i] - m) : 0.f;
                    add += p;
                    pf[s][t >> 1][(t & 1) * 4 + i] = (bf16)p;
                }
            sum[s] = sum[s] * keep + add;
            mx[s] = m;
            if (__any(keep != 1.f)) {
#pragma unroll
                for (int f = 0; f < VF; f++) acc[s][f] *= keep;
            }
        }
#pragma unroll
        for (int u = 0; u < KT / 32; u++)
#pragma unroll
            for (int f = 0; f < VF; f++) {
                const uint8_t* from = kb + value_at[f & 3] + (f >> 2) * 128 + u * 32 * (DK * 2);
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(from));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(from + 16 * (DK * 2)));
                const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                const bf16x8 vf = *reinterpret_cast<const bf16x8*>(&both);
#pragma unroll
                for (int s = 0; s < QS; s++) acc[s][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[s][u], acc[s][f], 0, 0, 0);
            }
    }
    // lane l holds value columns 16 f + 4 g + i of query l % 16
#pragma unroll
    for (int s = 0; s < QS; s++) {
        float all = sum[s];
        all += __shfl_xor(all, 16, 64);
        all += __shfl_xor(all, 32, 64);
        const int r = row0 + (row_wave * QS + s) * 16 + l15;
        if (r >= a.rows) continue;
        if (a.splits > 1) {
            const size_t place = ((size_t)at.z * blocks.y + z) * a.rows + r;
            if (g == 0 && f0 == 0) {
                a.part_stats[2 * place] = mx[s];
                a.part_stats[2 * place + 1] = all;
            }
            float* dst = a.part + place * a.ld_part;
#pragma unroll
            for (int f = 0; f < VF; f++)
                if ((f0 + f) * 16 + 4 * g < a.ld_part) *reinterpret_cast<f32x4*>(dst + (f0 + f) * 16 + 4 * g) = acc[s][f];
        } else {
            const float inv = 1.0f / all;
            const int token = r / a.rows_per_token;
            bf16* dst = a.out + z * a.out_head + (size_t)token * a.out_token + (r - token * a.rows_per_token) * a.ld_out;
#pragma unroll
            for (int f = 0; f < VF; f++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int d = (f0 + f) * 16 + 4 * g + i;
                    if (d < a.dv) dst[d] = (bf16)(acc[s][f][i] * inv);
                }
        }
    }
}

}  // namespace attend
}  // namespace a81w41
