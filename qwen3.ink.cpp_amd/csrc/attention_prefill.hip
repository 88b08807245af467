// Causal GQA attention for many new tokens at once (the prompt pass) on the matrix cores:
// QK^T * scale, causal mask, softmax, PV (QwenAttention.cc:150-195) over the fp16 KV cache.
//
// One workgroup per (tile of 32 query tokens, G query heads of a KV head) with G x S waves: the heads
// share every staged key / value tile, and the key tiles of a head are dealt round-robin
// to S waves, which shortens the serial walk over the context S times.  Each wave keeps the
// running-maximum ("online") softmax of its share in fp32; the S shares are merged at the end.
//
// Both products are computed transposed, so that a lane owns one query token:
//   S^T = K Q^T      A = key tile (row = key, k = head dim), B = Q^T (column = query)
//   O^T = V^T P^T    A = V^T (row = head dim, k = key),     B = P^T (column = query)
// with v_mfma_f32_32x32x16_f16, whose result registers of lane (query q, half kh) hold rows
// 8g + 4kh + i (g, i = 0..3).  A row's maximum and sum are therefore in-lane reductions over 16
// registers plus one exchange with lane q of the other half, and the rescaling factor of the
// running output is a per-lane scalar.  The same registers feed the second product directly:
// its contraction index may run over the keys in any order as long as V^T uses the same one,
// and transposing LDS reads give V^T in exactly the order the P registers have.
//
// The cache holds fp16, which the matrix cores take as it is.  The fp32 queries and
// probabilities are split into two fp16 terms (x = hi + lo, |lo| <= 2^-11 |hi|) and multiplied
// in two instructions, which keeps about 22 significant bits: the result matches the fp32
// vector kernels of the short-prompt path to rounding noise.
//
// Output: fp32 rows, or (q_out) the rows' 80 B quantised blocks for the linear that follows
// (quantize_row_q8_1_repack_fp32, quantized_gemx_kernels.cc:803-911).  A lane holds 16 of the 32
// values of each of its row's four 32-blocks per head and the lane of the other half the other 16,
// so the block maximum and sum are in-lane reductions plus one exchange; the bits equal those of
// quantising the fp32 rows.
#include "a81w41_kernels.h"

#include <cstdlib>
#include "quantize_common.h"

#include <hip/hip_fp16.h>

namespace a81w41 {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kHeadDim = 128;
constexpr int kTile = 32;         // query tokens per workgroup, keys per step
constexpr int kRowBytes = 256;    // of a staged key or value
constexpr int kKeyBytes = kTile * kRowBytes, kTileBytes = 2 * kKeyBytes;  // 32 keys, then their values, as the cache has them
constexpr int kQueryBytes = kTile * kHeadDim * 4;                        // a head's 32 queries in fp32
constexpr int kBlockBytes = 64 * 16 * 4;                                 // 32 head dims of one wave's 128 x 32 fp32 output
constexpr float kLowest = -3.0e38f;

// Sixteen-byte chunk c of a staged row sits at place c ^ this.  Keys are read 32 rows at one chunk, values by transposing
// reads of four rows and four chunks: either way the places of a read cover the banks.
__device__ __forceinline__ int key_swap(int key) { return key & 15; }
__device__ __forceinline__ int value_swap(int key) { return (key & 3) << 2; }

__device__ __forceinline__ void copy16(const void* src, void* lds_base) {  // lane l's sixteen bytes land at lds_base + 16 l
    __builtin_amdgcn_global_load_lds(src, (lds_ptr_t)lds_base, 16, 0, 0);
}
// This wave's copies are in LDS and its LDS reads done, then every wave's.
__device__ __forceinline__ void wait_and_meet() {
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// A^T operands of 32 keys' values: two steps of 16 keys for the lane's head dim.  `at`: where the lane's four dims of key 4 (lane / 32) +
// lane % 16 / 4 sit.  Reads and their wait in one: ahead of the builtin the compiler would wait for the copies under way.
__device__ __forceinline__ void read_values(uint32_t at, v2u (&v)[4]) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4\n"
        "ds_read_b64_tr_b16 %1, %4 offset:2048\n"
        "ds_read_b64_tr_b16 %2, %4 offset:4096\n"
        "ds_read_b64_tr_b16 %3, %4 offset:6144\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
        : "v"(at)
        : "memory");
}

__device__ __forceinline__ void split_fp16(const float (&x)[8], v8h& hi, v8h& lo) {
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const _Float16 h = (_Float16)x[t];
        hi[t] = h;
        lo[t] = (_Float16)(x[t] - (float)h);
    }
}

// exp for the softmax weights: v_exp_f32 on x * log2(e), relative error about |x| * 2^-24.
__device__ __forceinline__ float fast_exp(float x) { return __expf(x); }

// G = query heads per KV head, S = key splits: wave (h, sp) = (wave % G, wave / G) owns query head
// kvh*G + h and every S-th key tile starting at sp.  The queries, and a round of S tiles ahead of the one that is worked on, are copied
// global -> LDS directly; at the end the S partial (maximum, sum, output) triples of a head meet through LDS, where
// each of its waves takes a share of the head dims, merges, quantises and stores it.
//
// What bounds it: the way of the workgroup with the most keys, a round's wait, matrix ops and softmax one after the other.
// us, so / with tiles that went through registers and were transposed on their way to LDS, two waits a round, queries read row by row and one
// wave a head merging and quantising: 180 tokens, 16 heads on 4, 9.0 / 14.8; 322 tokens, 32 on 8, 13.2 / 23.1; 900 tokens, 12 on 3, 24.5 / 39.4;
// 2048 tokens, 32 on 8, 152 / 205; the same bits.
template <int G, int S>
__global__ __launch_bounds__(64 * G * S, G * S / 4) void attention_prefill_kernel(const float* __restrict__ q, int q_row_stride,
                                                                                 const __half* __restrict__ k_cache,
                                                                                 const __half* __restrict__ v_cache,
                                                                                 const int* __restrict__ pos_dev, float* __restrict__ out,
                                                                                 int out_row_stride, uint8_t* __restrict__ q_out, int n_q,
                                                                                 int M, int max_seq, float scale) {
    constexpr int kBuf = S * kTileBytes;     // a round's tiles
    constexpr int kCopies = kTileBytes / 1024;  // of a tile, dealt to the G waves
    constexpr int kOwn = 4 / S;              // 32-blocks of head dims that a wave finishes
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 31, kh = lane >> 5;
    const int h = wave % G, sp = wave / G;
    // gridDim.z workgroups share a KV head when its group of query heads is larger than G
    const int kvh = blockIdx.y, head = kvh * (n_q / (int)gridDim.y) + (int)blockIdx.z * G + h;
    const int m0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * kTile;  // the longest rows first
    const int pos0 = pos_dev[0];
    const int m_last = min(m0 + kTile, M) - 1;                  // last real token of the tile
    const int n_keys = min(pos0 + m_last, max_seq - 1) + 1;     // keys the tile's last token sees
    const int n_tiles = (n_keys + kTile - 1) / kTile;
    const int n_rounds = (n_tiles + S - 1) / S;
    const int m = m0 + r;                                       // this lane's query token
    const int last_key = min(pos0 + min(m, m_last), n_keys - 1);  // it sees keys 0..last_key
    const int first_last_key = min(pos0 + m0, n_keys - 1);      // what every token of the tile sees

    const uint8_t* k_base = reinterpret_cast<const uint8_t*>(k_cache) + (size_t)kvh * max_seq * kRowBytes;
    const uint8_t* v_base = reinterpret_cast<const uint8_t*>(v_cache) + (size_t)kvh * max_seq * kRowBytes;
    auto copy_tile = [&](int round) {  // this wave's share of its tile; rows past the context repeat the last one (they are masked)
        const int tile = round * S + sp;
        if (tile >= n_tiles) return;
        uint8_t* to = lds + (round & 1) * kBuf + sp * kTileBytes;
#pragma unroll
        for (int i = 0; i < (kCopies + G - 1) / G; i++) {
            const int n = i * G + h, key = 4 * (n & 7) + (lane >> 4), place = lane & 15;
            const size_t row = (size_t)min(tile * kTile + key, n_keys - 1) * kRowBytes;
            if (n < 8)
                copy16(k_base + row + 16 * (place ^ key_swap(key)), to + n * 1024);
            else
                copy16(v_base + row + 16 * (place ^ value_swap(key)), to + n * 1024);
        }
    };
    copy_tile(0);
    // The queries pass where round 1 will be: chunk c of row i at place c ^ i.
    uint8_t* const q_lds = lds + kBuf + h * kQueryBytes;
#pragma unroll
    for (int i = 0; i < 16 / S; i++) {
        const int n = i * S + sp, row = 2 * n + kh;
        const float* src = q + (size_t)min(m0 + row, M - 1) * q_row_stride + (size_t)head * kHeadDim;
        copy16(src + 4 * (r ^ row), q_lds + n * 1024);
    }
    wait_and_meet();
    // this lane's query row as B operands: step d covers head dims 16d + 8kh .. + 7
    v8h q_hi[8], q_lo[8];
#pragma unroll
    for (int d = 0; d < 8; d++) {
        const v4f a = *reinterpret_cast<const v4f*>(q_lds + r * 512 + 16 * ((4 * d + 2 * kh) ^ r));
        const v4f b = *reinterpret_cast<const v4f*>(q_lds + r * 512 + 16 * ((4 * d + 2 * kh + 1) ^ r));
        const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        split_fp16(x, q_hi[d], q_lo[d]);
    }

    // where this lane's transposing reads of 32-block b of the head dims start in a tile of values
    uint32_t value_at[4];
    {
        const int i = lane & 15, key = 4 * kh + (i >> 2);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int c = 4 * b + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
            value_at[b] = kKeyBytes + key * kRowBytes + 16 * (c ^ value_swap(key)) + 8 * (i & 1);
        }
    }
    v16f o_acc[4];
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int v = 0; v < 16; v++) o_acc[b][v] = 0.f;
    float m_run = kLowest, l_run = 0.f;

    for (int round = 0; round < n_rounds; round++) {  // uniform over the workgroup
        wait_and_meet();  // the round's tiles are in LDS, and nobody still reads what the next ones replace
        copy_tile(round + 1);
        const int tile = round * S + sp;
        if (tile >= n_tiles) continue;  // uniform over the wave
        const uint8_t* k_lds = lds + (round & 1) * kBuf + sp * kTileBytes;

        v16f s_acc;
#pragma unroll
        for (int v = 0; v < 16; v++) s_acc[v] = 0.f;
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const v8h a = *reinterpret_cast<const v8h*>(k_lds + r * kRowBytes + 16 * ((2 * d + kh) ^ key_swap(r)));
            s_acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, q_hi[d], s_acc, 0, 0, 0);
            s_acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, q_lo[d], s_acc, 0, 0, 0);
        }

        float sc[16];
        float t_max = kLowest;
        if (tile * kTile + kTile - 1 <= first_last_key) {
#pragma unroll
            for (int v = 0; v < 16; v++) sc[v] = s_acc[v] * scale;
        } else {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = tile * kTile + 8 * (v >> 2) + 4 * kh + (v & 3);
                sc[v] = key <= last_key ? s_acc[v] * scale : kLowest;
            }
        }
#pragma unroll
        for (int v = 0; v < 16; v++) t_max = fmaxf(t_max, sc[v]);
        t_max = fmaxf(t_max, __shfl_xor(t_max, 32, 64));
        const float m_new = fmaxf(m_run, t_max);
        // a token that sees none of this tile's keys and none before it (only possible in a wave
        // whose first tile is not tile 0) keeps m_new = kLowest: its weights must still be 0
        const float alpha = fast_exp(m_run - m_new);
        float p[16];
        float p_sum = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            p[v] = sc[v] > kLowest ? fast_exp(sc[v] - m_new) : 0.f;
            p_sum += p[v];
        }
        p_sum += __shfl_xor(p_sum, 32, 64);
        l_run = l_run * alpha + p_sum;
        if (__any(m_new > m_run)) {
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int v = 0; v < 16; v++) o_acc[b][v] *= alpha;
        }
        m_run = m_new;

        v8h p_hi[2], p_lo[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float x[8] = {p[8 * c], p[8 * c + 1], p[8 * c + 2], p[8 * c + 3],
                                p[8 * c + 4], p[8 * c + 5], p[8 * c + 6], p[8 * c + 7]};
            split_fp16(x, p_hi[c], p_lo[c]);
        }
        const uint32_t v_at = (uint32_t)(uintptr_t)(lds_ptr_t)k_lds;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            v2u part[4];
            read_values(v_at + value_at[b], part);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const uint4 a4 = make_uint4(part[2 * c][0], part[2 * c][1], part[2 * c + 1][0], part[2 * c + 1][1]);
                const v8h a = __builtin_bit_cast(v8h, a4);
                o_acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, p_hi[c], o_acc[b], 0, 0, 0);
                o_acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, p_lo[c], o_acc[b], 0, 0, 0);
            }
        }
    }

    // ---- merge the S partial results of each head ------------------------------------------------
    // LDS now holds 32-block b of wave w's scaled output at (w 4 + b) kBlockBytes, then the running maxima and sums of all waves.
    float l_tot = l_run;
    if constexpr (S > 1) {
        float* stat = reinterpret_cast<float*>(lds + 4 * G * S * kBlockBytes);
        wait_and_meet();  // the staged tiles are dead
        if (kh == 0) {
            stat[(sp * G + h) * 32 + r] = m_run;
            stat[(S * G + sp * G + h) * 32 + r] = l_run;
        }
        wait_and_meet();
        float m_fin = kLowest;
#pragma unroll
        for (int j = 0; j < S; j++) m_fin = fmaxf(m_fin, stat[(j * G + h) * 32 + r]);  // finite: tile 0 holds key 0
        l_tot = 0.f;
#pragma unroll
        for (int j = 0; j < S; j++)
            l_tot += stat[(S * G + j * G + h) * 32 + r] * fast_exp(stat[(j * G + h) * 32 + r] - m_fin);
        const float f = fast_exp(m_run - m_fin);  // 0 for a wave that had no visible key
#pragma unroll
        for (int b = 0; b < 4; b++) {
            v4f* slot = reinterpret_cast<v4f*>(lds + ((sp * G + h) * 4 + b) * kBlockBytes);
#pragma unroll
            for (int g = 0; g < 4; g++)
                slot[g * 64 + lane] = v4f{o_acc[b][4 * g] * f, o_acc[b][4 * g + 1] * f, o_acc[b][4 * g + 2] * f, o_acc[b][4 * g + 3] * f};
        }
        wait_and_meet();
    }
    const float inv = 1.0f / l_tot;
    // 32-block b of this head: values 8g + 4kh + i (g, i = 0..3) here, the rest in lane ^ 32.  All lanes
    // take part in the exchanges; rows past the last token store nothing.
#pragma unroll
    for (int own = 0; own < kOwn; own++) {
        const int b = sp * kOwn + own;
        float val[16];
        if constexpr (S > 1) {
            auto slot = [&](int j) { return reinterpret_cast<const v4f*>(lds + ((j * G + h) * 4 + b) * kBlockBytes); };
#pragma unroll
            for (int g = 0; g < 4; g++) {
                v4f sum = slot(0)[g * 64 + lane];
                if constexpr (S == 2) {
                    sum += slot(1)[g * 64 + lane];
                } else {
                    static_assert(S == 4, "the order of the sums");
                    sum = (sum + slot(2)[g * 64 + lane]) + (slot(1)[g * 64 + lane] + slot(3)[g * 64 + lane]);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) val[4 * g + i] = sum[i] * inv;
            }
        } else {
#pragma unroll
            for (int v = 0; v < 16; v++) val[v] = o_acc[own][v] * inv;
        }
        if (q_out == nullptr) {
            if (m <= m_last) {
                float* dst = out + (size_t)m * out_row_stride + (size_t)head * kHeadDim + 4 * kh;
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *reinterpret_cast<float4*>(dst + 32 * b + 8 * g) = make_float4(val[4 * g], val[4 * g + 1], val[4 * g + 2], val[4 * g + 3]);
            }
            continue;
        }
        float amax = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) amax = fmaxf(amax, fabsf(val[v]));
        amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
        const float d = amax / 127.f;                           // the quantiser's arithmetic, step by step
        const float id = (amax != 0.0f) ? 127.f / amax : 0.0f;
        unsigned sum = 0;
        uint32_t word[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            word[g] = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r_ = rne_i32(val[4 * g + i] * id);
                sum += (unsigned)r_;
                word[g] |= (uint32_t)(sat8(r_) & 0xff) << (8 * i);
            }
        }
        sum += (unsigned)__shfl_xor((int)sum, 32, 64);
        if (m <= m_last) {
            uint8_t* blk = q_out + ((size_t)m * (2 * n_q) + 2 * head + (b >> 1)) * kABlock32;
            const int h2 = b & 1;
#pragma unroll
            for (int g = 0; g < 4; g++) *reinterpret_cast<uint32_t*>(blk + 16 + 32 * h2 + 8 * g + 4 * kh) = word[g];
            if (kh == 0) {
                float* par = reinterpret_cast<float*>(blk);
                par[h2] = d;
                par[2 + h2] = __fmul_rn(d, (float)(int)sum);
            }
        }
    }
}

// Two rounds of tiles; one and the queries; or the waves' outputs and statistics.
template <int G, int S>
constexpr size_t prefill_lds_bytes() {
    constexpr size_t round = (size_t)S * kTileBytes, rest = (size_t)G * kQueryBytes > round ? (size_t)G * kQueryBytes : round;
    constexpr size_t merge = S > 1 ? (size_t)4 * G * S * kBlockBytes + (size_t)2 * S * G * 32 * sizeof(float) : 0;
    return round + rest > merge ? round + rest : merge;
}

template <int G, int S>
hipError_t launch_prefill(dim3 grid, const float* q, int q_row_stride, const __half* kc, const __half* vc, const int* pos_dev,
                          float* out, int out_row_stride, uint8_t* q_out, int n_q, int M, int max_seq, float scale,
                          hipStream_t s) {
    constexpr size_t lds = prefill_lds_bytes<G, S>();
    static_assert(lds <= (size_t)kLdsLimitBytes, "attention tile buffers exceed the LDS of a CU");
    if (lds > 64 * 1024) {  // a kernel gets 64 KiB of dynamic LDS without asking
        const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_prefill_kernel<G, S>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (attr != hipSuccess) return attr;
    }
    hipLaunchKernelGGL((attention_prefill_kernel<G, S>), grid, dim3(64 * G * S), lds, s, q, q_row_stride, kc, vc, pos_dev, out,
                       out_row_stride, q_out, n_q, M, max_seq, scale);
    return hipGetLastError();
}

}  // namespace

bool attention_prefill_fits(int M, int n_q, int n_kv) {
    if (M <= 8 || n_kv < 1 || n_q % n_kv) return false;
    const int g = n_q / n_kv;
    return g == 1 || g == 2 || g == 4 || g == 8;
}

hipError_t launch_attention_prefill(const float* q, int q_row_stride, const void* k_cache, const void* v_cache,
                                    const int* pos_dev, float* out, int out_row_stride, int M, int n_q, int n_kv, int max_seq,
                                    float scale, hipStream_t s, void* q_out, int heads_per_workgroup) {
    const int tiles = (M + kTile - 1) / kTile, group = n_q / n_kv;
    uint8_t* qo = static_cast<uint8_t*>(q_out);
    const __half* kc = static_cast<const __half*>(k_cache);
    const __half* vc = static_cast<const __half*>(v_cache);
    // G heads x S key splits per workgroup, at most 8 waves: a wave needs about 200 registers per lane (64 for its query, 64 for
    // its output).  One head and four splits where every workgroup gets a CU; two heads, whose tiles two waves share, while the longest
    // workgroup counts; the whole group where there are many rounds.  us with 1 / 2 / 4 heads: 180 tokens, 16 heads on 4, 9.0 / 10.0 / 12.4;
    // 322 tokens, 8 on 2 10.8 / 11.9 / 16.6, 32 on 8 (352, 176, 88 workgroups) 18.5 / 13.2 / 17.4; 900 tokens, 12 on 3 31.9 / 24.5 / 35.8;
    // 2048 tokens, 8 on 2 76 / 45 / 72, 32 on 8 252 / 157 / 152; 3000 tokens - / 244 / 234.  With 64 heads and more, whose prompts have that many
    // workgroups sooner, no two heads past one workgroup a CU: 64 on 8, 295 tokens - / 20.2 / 17.9, 509 30.6 / 26.0, 990 82 / 72.5; 64 on 16, 339 22.4 / 19.8.
    // A81W41_ATTENTION_HEADS=<G> fixes the heads per workgroup (measurement aid, tuning builds only).
    static const int env_g = tuning_env_int("A81W41_ATTENTION_HEADS");
    int g = 1;
    while (g < group && (long long)tiles * n_kv * (group / g) > (g == 1 || (g == 2 && n_q >= 64) ? 256 : 1024)) g <<= 1;
    if (env_g > 0 && env_g <= group && group % env_g == 0) g = env_g;
    if (heads_per_workgroup > 0) {
        if (heads_per_workgroup > group || group % heads_per_workgroup) return hipErrorInvalidValue;
        g = heads_per_workgroup;
    }
    const dim3 grid(tiles, n_kv, group / g);
    switch (g) {
        case 1: return launch_prefill<1, 4>(grid, q, q_row_stride, kc, vc, pos_dev, out, out_row_stride, qo, n_q, M, max_seq, scale, s);
        case 2: return launch_prefill<2, 4>(grid, q, q_row_stride, kc, vc, pos_dev, out, out_row_stride, qo, n_q, M, max_seq, scale, s);
        case 4: return launch_prefill<4, 2>(grid, q, q_row_stride, kc, vc, pos_dev, out, out_row_stride, qo, n_q, M, max_seq, scale, s);
        case 8: return launch_prefill<8, 1>(grid, q, q_row_stride, kc, vc, pos_dev, out, out_row_stride, qo, n_q, M, max_seq, scale, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace a81w41
