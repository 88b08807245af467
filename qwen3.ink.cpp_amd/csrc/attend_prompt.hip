// Causal attention of a prompt's many rows on the matrix cores, bfloat16, in two of attend_mfma.hip's forms:
//   rows      the queries of a group of heads look at the rows of their key/value head, [value | key];
//   expanded  a key is [own part | part shared by all heads], values come transposed ([value column][key]).
//
// A workgroup of KG x QW waves takes 32 QW query rows.  A wave owns 32 of them; KG waves share them, each with every KG-th tile of 64
// keys (or 32), and meet at the end: a workgroup of several groups keeps two waves on every SIMD while its rows, and with them the
// rows past the diagonal, stay few.  Scores are formed transposed, S^T = K Q^T (v_mfma_f32_32x32x16_bf16 with the keys
// as rows), so that a lane holds scores of query l % 32 only.  Row r of a 32-key product is key r with bits 2 and 3
// exchanged: register v of lane half h is then key 16 (v / 8) + 8 h + v % 8, and eight registers are, as they stand, the
// B operand of a 16-key step of O^T = V^T P^T whose A operand is eight neighbouring keys.  Running maximum and sum are
// one value per lane.  Scores, softmax and sums are fp32; the maximum follows every larger score, so that the heaviest
// weight, 1, is exact in 16 bits (left behind by up to 2^8 it is not: 14 % more error for 8 % less time).
//
// A tile is copied global -> LDS by direct 16-byte loads, the next one while this one is worked on; in the rows form only while its
// scores and weights are formed, as the compiler waits for every copy under way ahead of the first transposing read of values.
// Chunk c of key k sits at place c ^ (4 (k % 4) + k / 4 % 4), or, where rows are an odd number of 128 bytes, c ^ k / 2 % 8; chunk c of a
// transposed value column d at c ^ d / 2 % 8, of half a row at c ^ d / 4 % 4: sixteen rows read at one chunk column, and four rows that a transposing read
// takes four chunks of, cover the 256 bytes of all banks.  With c ^ k % 16 those four rows met in eight places, and more than half of
// the cycles of LDS were conflicts: 2048 rows in chunks of 1024, 16 heads on 4 of 128 + 128 columns 28.8 us, so 26.7.
//
// What bounds it: matrix ops and softmax of a SIMD's two waves, one after the other; then LDS, which gives an operand of 1 KiB
// for every matrix op; of a short prompt's workgroup its start and end.  So queries, the row's gate and the first tile are one trip, and rows are
// stored sixteen bytes a lane.  4095 rows of 16 heads, 192 + 128 columns: 114 us = 750 TFLOP/s, 118 with queries awaited ahead of
// the first tile's copies, the gate behind the last and stores of eight bytes.
#include "dense_common.h"

namespace a81w41 {
namespace {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLowest = -1e30f;

template <int DK>
__device__ __forceinline__ int place_of_key(int k) {
    return DK % 128 ? (k >> 1) & 7 : (k & 3) << 2 | (k >> 2 & 3);
}
template <int CV>  // a row of CV chunks
__device__ __forceinline__ int place_of_value(int d) {
    return CV == 8 ? (d >> 1) & 7 : (d >> 2) & 3;
}
// the value of the lane 32 away
__device__ __forceinline__ float other_half(float v) {
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(threadIdx.x & 32 ? both[0] : both[1]);
}

// DK: columns of a tile row; the scores take those from KEY0 on (rows form: the key part, 0 otherwise).  DV: value columns.
// kTile: keys of a tile, 64 or 32.
template <int DK, int DV, int KEY0, int KG, int QW, int kTile, bool EXPANDED>
__global__ __launch_bounds__(64 * KG * QW, KG * QW / 4) void attend_prompt_kernel(AttendArgs<bf16> a) {
    constexpr int CK = DK / 8, CV = kTile / 8, KT = kTile / 32, KS = (DK - KEY0) / 16, VF = DV / 32, kRows = 32 * QW;
    constexpr int kKeyBytes = kTile * DK * 2, kBuf = kKeyBytes + (EXPANDED ? DV * kTile * 2 : 0);
    constexpr int NK = kTile * CK / 64 / QW, NV = EXPANDED ? DV * CV / 64 / QW : 0;  // copies of a wave and tile
    static_assert(DK % 64 == 0 && DV % 32 == 0 && KEY0 % 64 == 0 && kTile * CK % (64 * QW) == 0 && DV * CV % (64 * QW) == 0, "tile sizes");
    static_assert((KG - 1) * 64 * 4 * (16 * VF + 2) * QW <= 2 * KG * kBuf, "the groups meet in LDS");
    __shared__ __attribute__((aligned(128))) uint8_t lds[2 * KG * kBuf];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l31 = lane & 31, half = lane >> 5;
    const int qw = wave % QW, kg = wave / QW;
    // heads next to each other, the longest rows first: what is left over for a CU that is done is short
    const int z = blockIdx.x, row0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kRows;
    const int pos = min(max(a.pos_dev[0], 0), a.max_seq - 1);
    auto last_key = [&](int row) { return min(pos + row / a.rows_per_token, a.max_seq - 1); };
    auto chunk_begin = [&](int key) { return a.chunk ? key - key % a.chunk : 0; };
    const int wg_keys = last_key(min(row0 + kRows, a.rows) - 1) + 1;  // keys any row of the workgroup sees
    int key_begin = chunk_begin(last_key(row0)), key_end = wg_keys;
    if (a.splits > 1) {
        const int from = chunk_begin(pos), all = last_key(a.rows - 1) + 1 - from;
        const int share = ((all + a.splits - 1) / a.splits + kTile - 1) / kTile * kTile, begin = from + (int)blockIdx.z * share;
        key_end = min(begin + share, wg_keys);
        key_begin = min(max(begin, key_begin), key_end);
    }
    const int n_tiles = (key_end - key_begin + kTile - 1) / kTile, n_turns = (n_tiles + KG - 1) / KG;
    const int own_chunks = a.k_own_width >> 3, all_chunks = own_chunks + (EXPANDED ? a.k_shared_width >> 3 : 0);

    // This lane's 16 bytes of every copy, at the group's first tile; a turn moves them on by KG tiles.
    const uint8_t* key_src[NK];
    int key_step[NK];
    const bf16* value_src[NV ? NV : 1];
    uint8_t* const my_lds = lds + kg * 2 * kBuf;
    auto key_place = [&](int n, int key, int* step) -> const uint8_t* {  // source of copy n if its row is that key
        const int q = (n * QW + qw) * 64 + lane, r = q / CK, c = (q % CK) ^ place_of_key<DK>(r);
        const bf16* src = a.k_own + z * a.k_own_head + (size_t)key * a.ld_k_own;
        int ld = a.ld_k_own;
        if constexpr (KEY0 > 0) {
            if (c < KEY0 / 8)
                src += c < (a.v_width >> 3) ? c * 8 : 0;
            else if (c - KEY0 / 8 < own_chunks)
                src += a.v_width + (c - KEY0 / 8) * 8;
        } else if (c < own_chunks) {
            src += c * 8;
        } else if (EXPANDED && c < all_chunks) {
            src = a.k_shared + (size_t)key * a.ld_k_shared + (c - own_chunks) * 8;
            ld = a.ld_k_shared;
        }
        *step = ld * 2 * (KG * kTile);
        return reinterpret_cast<const uint8_t*>(src);
    };
    auto row_of_copy = [&](int n) { return ((n * QW + qw) * 64 + lane) / CK; };
#pragma unroll
    for (int n = 0; n < NK; n++) key_src[n] = key_place(n, key_begin + kg * kTile + row_of_copy(n), &key_step[n]);
    if constexpr (EXPANDED) {
#pragma unroll
        for (int n = 0; n < NV; n++) {
            const int q = (n * QW + qw) * 64 + lane, r = q / CV, c = (q % CV) ^ place_of_value<CV>(r);
            value_src[n] = a.v_t + ((size_t)z * a.dv + min(r, a.dv - 1)) * a.ld_v + key_begin + kg * kTile + c * 8;
        }
    }
    auto copy_tile = [&](int tile, int buf) {
        uint8_t* base = my_lds + buf * kBuf + qw * 1024;
        const int key0 = key_begin + tile * kTile;
        if (key0 + kTile <= wg_keys) {
#pragma unroll
            for (int n = 0; n < NK; n++) {
                copy16_to_lds(key_src[n], base + n * QW * 1024);
                key_src[n] += key_step[n];
            }
        } else {  // the last rows stand in for those past the end
#pragma unroll
            for (int n = 0; n < NK; n++) {
                int step;
                copy16_to_lds(key_place(n, min(key0 + row_of_copy(n), wg_keys - 1), &step), base + n * QW * 1024);
            }
        }
#pragma unroll
        for (int n = 0; n < NV; n++) {
            copy16_to_lds(value_src[n], base + kKeyBytes + n * QW * 1024);
            value_src[n] += KG * kTile;
        }
    };

    // Query operands; a negative scale is their sign, so that the largest score is the largest product.
    const int wave_row0 = row0 + qw * 32, my_row = min(wave_row0 + l31, a.rows - 1), my_token = my_row / a.rows_per_token;
    const int limit = last_key(my_row), first = chunk_begin(limit);
    const int lowest_limit = last_key(min(wave_row0, a.rows - 1)), highest_limit = last_key(min(wave_row0 + 31, a.rows - 1));
    const int highest_first = chunk_begin(highest_limit);
    const float scale = fabsf(a.scale) * kLog2e;
    // They, the row's gate and the first tile are one trip.
    bf16x8 qf[KS];
    const float gate = a.head_gate ? a.head_gate[(size_t)my_row * a.ld_gate + z] : 0.f;
    {
        const bf16* src = a.q + z * a.q_head + (size_t)my_token * a.q_token + (my_row - my_token * a.rows_per_token) * a.ld_q;
        const unsigned sign = a.scale < 0.f ? 0x80008000u : 0u;
        uint4 u[KS];
#pragma unroll
        for (int k = 0; k < KS; k++) u[k] = *reinterpret_cast<const uint4*>(src + min(2 * k + half, all_chunks - 1) * 8);
        if (kg < n_tiles) copy_tile(kg, 0);
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const unsigned keep = 2 * k + half < all_chunks ? ~0u : 0u;
            u[k] = make_uint4((u[k].x ^ sign) & keep, (u[k].y ^ sign) & keep, (u[k].z ^ sign) & keep, (u[k].w ^ sign) & keep);
            qf[k] = *reinterpret_cast<const bf16x8*>(&u[k]);
        }
    }
    f32x16 acc[VF];
#pragma unroll
    for (int f = 0; f < VF; f++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[f][v] = 0.f;
    const bool sink = a.sink && kg == 0 && (a.splits == 1 || blockIdx.z == 0);  // one lane half of one group of one share counts it
    float mx = sink || scale == 0.f ? 0.f : kLowest, sum = sink && half == 0 ? 1.f : 0.f;

    const int key_row = (l31 & 0x13) | (l31 & 4) << 1 | (l31 & 8) >> 1;  // bits 2 and 3 exchanged
    const int key_at = key_row * (DK * 2), key_swap = place_of_key<DK>(key_row);
    // Values that are columns of the key rows come by transposing reads (ds_read_b64_tr_b16): in a group of 16 lanes lane i
    // names four columns of key i / 4 and receives its own column of the four keys.
    constexpr int VA = VF < 4 ? VF : 4;
    int value_at[VA][2];  // by f % 4, and for the first and the second four keys
    if constexpr (!EXPANDED) {
#pragma unroll
        for (int f = 0; f < VA; f++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int i = lane & 15, k = 8 * half + 4 * j + (i >> 2), c = 4 * f + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
                value_at[f][j] = k * (DK * 2) + ((c ^ place_of_key<DK>(k)) << 4) + (i & 1) * 8;
            }
    }

    for (int turn = 0; turn < n_turns; turn++) {
        const int tile = turn * KG + kg, key0 = key_begin + tile * kTile;
        // the tile is in LDS, everybody's copies of it; and nobody still reads the other buffer
        __builtin_amdgcn_s_waitcnt(0x0070);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (tile + KG < n_tiles) copy_tile(tile + KG, (turn + 1) & 1);
        if (tile >= n_tiles || key0 > highest_limit) continue;
        const uint8_t* kb = my_lds + (turn & 1) * kBuf;
        const uint8_t* vb = kb + kKeyBytes;
        f32x16 sc[KT];
#pragma unroll
        for (int t = 0; t < KT; t++) {
#pragma unroll
            for (int v = 0; v < 16; v++) sc[t][v] = 0.f;
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kb + key_at + t * 32 * (DK * 2) + (((KEY0 / 8 + 2 * k + half) ^ key_swap) << 4));
                sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[k], sc[t], 0, 0, 0);
            }
        }
        if (key0 + kTile - 1 > lowest_limit || key0 < highest_first || key0 + kTile > key_end) {
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int key = key0 + 32 * t + 16 * (v >> 3) + 8 * half + (v & 7);
                    if (key > limit || key < first || key >= key_end) sc[t][v] = -__builtin_inff();
                }
        }
        float top = sc[0][0];
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) top = fmaxf(top, sc[t][v]);
        top = fmaxf(top, other_half(top)) * scale;
        if (__any(top > mx)) {
            const float m = fmaxf(mx, top), keep = __builtin_amdgcn_exp2f(mx - m);
            mx = m;
            sum *= keep;
#pragma unroll
            for (int f = 0; f < VF; f++) acc[f] *= keep;
        }
        auto weights_sum = [&]() {
            float add[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) add[v & 3] += sc[t][v];
            return (add[0] + add[1]) + (add[2] + add[3]);
        };
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) sc[t][v] = __builtin_amdgcn_exp2f(fmaf(sc[t][v], scale, -mx));
        float add = weights_sum();
        // A weight that is no number, of a score that is none or of a masked one under a scale of zero, is 0.  Its sum tells, so that the
        // other tiles go without a comparison for every weight: 1 to 2 % of the time, against 1 to 5 % with all of them (a clamp to 0 .. 1
        // in the exponential's instruction is free but moves the last bits of sums).
        if (__builtin_expect(__any(add != add), 0)) {
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) sc[t][v] = fmaxf(sc[t][v], 0.f);
            add = weights_sum();
        }
        sum += add;
        bf16x8 pf[2 * KT];
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) pf[2 * t + (v >> 3)][v & 7] = (bf16)sc[t][v];
#pragma unroll
        for (int u = 0; u < 2 * KT; u++)
#pragma unroll
            for (int f = 0; f < VF; f++) {
                bf16x8 vf;
                if constexpr (EXPANDED) {
                    vf = *reinterpret_cast<const bf16x8*>(vb + (f * 32 + l31) * (kTile * 2) + (((2 * u + half) ^ place_of_value<CV>(l31)) << 4));
                } else {
                    const uint8_t* at = kb + (f >> 2) * 256 + u * 16 * (DK * 2);
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + value_at[f & 3][0]));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + value_at[f & 3][1]));
                    const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    vf = *reinterpret_cast<const bf16x8*>(&both);
                }
                acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[u], acc[f], 0, 0, 0);
            }
    }

    sum += other_half(sum);
    if constexpr (KG > 1) {  // the other groups hand their shares of the keys over, the first adds them one by one; registers (f, v .. v + 3) at 4 f + v / 4
        constexpr int kPart = (16 * VF + 2) * 64, kStats = 16 * VF * 64;
        float* part = reinterpret_cast<float*>(lds) + (size_t)qw * kPart;
        __syncthreads();
        if (kg > 0) {
            float* own = part + (kg - 1) * QW * kPart;
            own[kStats + lane] = mx, own[kStats + 64 + lane] = sum;
#pragma unroll
            for (int f = 0; f < VF; f++)
#pragma unroll
                for (int v = 0; v < 16; v += 4)
                    reinterpret_cast<f32x4*>(own)[(4 * f + v / 4) * 64 + lane] = f32x4{acc[f][v], acc[f][v + 1], acc[f][v + 2], acc[f][v + 3]};
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int k = 1; k < KG; k++, part += QW * kPart) {
            const float other = part[kStats + lane], m = fmaxf(mx, other);
            const float mine = __builtin_amdgcn_exp2f(mx - m), theirs = __builtin_amdgcn_exp2f(other - m);
            sum = sum * mine + part[kStats + 64 + lane] * theirs;
            mx = m;
#pragma unroll
            for (int f = 0; f < VF; f++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    if (v % 4 == 0) {
                        const f32x4 add = reinterpret_cast<const f32x4*>(part)[(4 * f + v / 4) * 64 + lane];
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[f][v + i] = acc[f][v + i] * mine + add[i] * theirs;
                    }
                }
        }
    }
    // register (f, v) holds value column 32 f + 8 (v / 4) + 4 half + v % 4 of query l % 32
    if (a.splits > 1) {
        const int r = wave_row0 + l31;
        if (r >= a.rows) return;
        const size_t at = ((size_t)blockIdx.z * gridDim.x + z) * a.rows + r;
        if (half == 0) {
            a.part_stats[2 * at] = mx;
            a.part_stats[2 * at + 1] = sum;
        }
        float* dst = a.part + at * a.ld_part;
#pragma unroll
        for (int f = 0; f < VF; f++)
#pragma unroll
            for (int v = 0; v < 16; v += 4) {
                const int d = 32 * f + 2 * v + 4 * half;
                if (d < a.ld_part) *reinterpret_cast<f32x4*>(dst + d) = f32x4{acc[f][v], acc[f][v + 1], acc[f][v + 2], acc[f][v + 3]};
            }
        return;
    }
    // The lane's row, formed again: a register that holds any of it over the loop costs the widest expanded form its second set of value
    // operands, and a wait goes by with every product.  us of a call, so / held: 8 heads of 256 + 256 columns, 330 rows 50.6 / 52.0, 2000 rows
    // 173.6 / 180; 16 heads of 320 + 256, 4000 rows 354 / 367; the other forms are level.
    int out_lane = l31;
    asm volatile("" : "+v"(out_lane));
    const int out_row = min(wave_row0 + out_lane, a.rows - 1), out_token = out_row / a.rows_per_token;
    float inv = 1.0f / sum;
    if (a.head_gate) inv *= sigmoid(gate);
    bf16* dst = a.out + z * a.out_head + (size_t)out_token * a.out_token + (out_row - out_token * a.rows_per_token) * a.ld_out;
    const bool real = wave_row0 + out_lane < a.rows;
    // Eight neighbouring columns a lane, of two fours the halves of a row trade one; or fours, or single columns, as widths and the target
    // allow.  us of a call, fours / single columns: 16 heads of 192 + 124, 4095 rows 127 / 138; 16 heads on 4 of 128 + 124, 2048 rows 45 / 51.
    const auto starts = [&](int together) {
        return ((a.dv | a.ld_out | a.out_token) & (together - 1)) == 0 && (a.out_head & (together - 1)) == 0 &&
               (reinterpret_cast<uintptr_t>(a.out) & (together * sizeof(bf16) - 1)) == 0;
    };
    const bool eights = starts(8), fours = starts(4);
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
    for (int f = 0; f < VF; f++)
#pragma unroll
        for (int v = 0; v < 16; v += 8) {
            if (eights) {
                unsigned first[2], second[2];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const bf16x2 x = {(bf16)(acc[f][v + 2 * i] * inv), (bf16)(acc[f][v + 2 * i + 1] * inv)};
                    const bf16x2 y = {(bf16)(acc[f][v + 4 + 2 * i] * inv), (bf16)(acc[f][v + 5 + 2 * i] * inv)};
                    const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y), false, false);
                    first[i] = both[0], second[i] = both[1];
                }
                const int d = 32 * f + 2 * v + 8 * half;
                if (real && d < a.dv) *reinterpret_cast<lds16*>(dst + d) = lds16{first[0], first[1], second[0], second[1]};
            } else if (fours) {
#pragma unroll
                for (int i = 0; i < 8; i += 4) {
                    const int d = 32 * f + 2 * (v + i) + 4 * half;
                    const bf16x4 x = {(bf16)(acc[f][v + i] * inv), (bf16)(acc[f][v + i + 1] * inv), (bf16)(acc[f][v + i + 2] * inv), (bf16)(acc[f][v + i + 3] * inv)};
                    if (real && d < a.dv) *reinterpret_cast<bf16x4*>(dst + d) = x;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int d = 32 * f + 2 * v + (i & 4) * 2 + 4 * half + (i & 3);
                    if (real && d < a.dv) dst[d] = (bf16)(acc[f][v + i] * inv);
                }
            }
        }
}

template <int DK, int DV, int KEY0, int KG, int QW, int kTile, bool EXPANDED>
hipError_t launch_kernel(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    hipLaunchKernelGGL((attend_prompt_kernel<DK, DV, KEY0, KG, QW, kTile, EXPANDED>), dim3(heads, (a.rows + 32 * QW - 1) / (32 * QW), a.splits),
                       dim3(64 * KG * QW), 0, s, a);
    return hipGetLastError();
}

}  // namespace

constexpr int kQW = kAttendPromptRows / 32;

// Heads of more than 128 columns leave LDS and registers for one group only.  us against the 16 x 16 kernel that took these rows before:
// 8 heads on 2, 256 + 256 columns, 330 rows 29.1 / 29.7, 2000 rows 121 / 128.
hipError_t launch_attend_rows_prompt(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    const int widest = a.k_own_width > a.v_width ? a.k_own_width : a.v_width;
    if (widest <= 64) return launch_kernel<128, 64, 64, 2, kQW, 64, false>(a, heads, s);
    if (widest <= 128) return launch_kernel<256, 128, 128, 2, kQW, 64, false>(a, heads, s);
    return launch_kernel<512, 256, 256, 1, kQW, 64, false>(a, heads, s);
}

// The widest form takes all 512 registers and spills 45 of them, addresses of copies, whose reloads wait for the copies before.  It is
// the faster one all the same (us, against 16 x 16): 8 heads, 192 + 64 and 256 columns, 330 rows 36 / 51, 2000 rows 159 / 212.
hipError_t launch_attend_expanded(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    const int dk = a.k_own_width + a.k_shared_width;
    // Workgroups of 64 rows where there is no more than one for a CU, their keys in four groups of 32: a long prompt's last rows then have
    // half as many turns.  us, so / with 128 rows in two groups of 64: 8 heads, 500 rows 16.5 / 20, 900 rows 22 / 28; 12 heads, 180 rows 13 / 14.
    // More of them copy more, every workgroup having its keys to itself, and begin a second round: over 420 drawn calls, so / with 128 rows, up to 256 of them
    // 0.70 to 1.0 but for 64 rows and fewer without a context before them (up to 1.09); 257 to 512 of them up to 1024 rows 1.08 to 1.44, past 1024 rows
    // 0.72 to 0.87 up to 384 of them, 0.94 to 1.06 past that, and past 2048 rows 0.91: the last rows' turns count there.  8 heads, 2048 rows 37 / 49; 16
    // heads 50 / 52.
    const int most = a.rows <= 1024 ? 256 : a.rows < 2048 ? 384 : 512;
    const bool few = (long long)heads * ((a.rows + 63) / 64) <= most;
    if (dk <= 128 && a.dv <= 64)
        return few ? launch_kernel<128, 64, 0, 4, 2, 32, true>(a, heads, s) : launch_kernel<128, 64, 0, 2, kQW, 64, true>(a, heads, s);
    if (dk <= 192 && a.dv <= 128)
        return few ? launch_kernel<192, 128, 0, 4, 2, 32, true>(a, heads, s) : launch_kernel<192, 128, 0, 2, kQW, 64, true>(a, heads, s);
    return launch_kernel<320, 256, 0, 1, kQW, 64, true>(a, heads, s);
}

}  // namespace a81w41
