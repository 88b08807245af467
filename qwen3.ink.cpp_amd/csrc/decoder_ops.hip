// Kernels of the loop around every decoder model: embedding rows, the first maximum of the logits, the position.
//   embed_rows      Embedding::forward                     src/ops/embedding.cc:13-26
//   argmax_token    sample_token_greedy (first maximum)    Pipeline.cc:54-62
// Every index that depends on device data is clamped into its array.
#include <hip/hip_fp16.h>

#include <algorithm>

#include "decoder_session.h"

namespace a81w41 {
namespace {

struct Bf16Bits {
    uint16_t bits;
};
__device__ __forceinline__ float to_float(__half h) { return __half2float(h); }
__device__ __forceinline__ float to_float(Bf16Bits b) { return __uint_as_float((unsigned)b.bits << 16); }
__device__ __forceinline__ float to_float(float f) { return f; }

// One embedding row by a whole workgroup.  Eight values per load where the rows allow it (hidden and the row stride multiples of 8, 16-byte
// aligned).
template <typename E>
__device__ __forceinline__ void embed_row(const TokenRow& r, int id) {
    const E* row = static_cast<const E*>(r.table) + (size_t)id * r.ld;
    if (sizeof(E) == 2 && ((r.hidden | r.ld) & 7) == 0) {
        for (int j = threadIdx.x; j < (r.hidden >> 3); j += blockDim.x) {
            const uint4 u = reinterpret_cast<const uint4*>(row)[j];
            const E* e = reinterpret_cast<const E*>(&u);
            float4* dst = reinterpret_cast<float4*>(r.out) + 2 * j;
            dst[0] = make_float4(to_float(e[0]), to_float(e[1]), to_float(e[2]), to_float(e[3]));
            dst[1] = make_float4(to_float(e[4]), to_float(e[5]), to_float(e[6]), to_float(e[7]));
        }
    } else {
        for (int j = threadIdx.x; j < r.hidden; j += blockDim.x) r.out[j] = to_float(row[j]);
    }
}
__device__ __forceinline__ void embed_token(const TokenRow& r, int id) {
    id = min(max(id, 0), r.vocab - 1);
    switch (r.type) {
        case TableType::kFp16: return embed_row<__half>(r, id);
        case TableType::kBf16: return embed_row<Bf16Bits>(r, id);
        case TableType::kFp32: return embed_row<float>(r, id);
    }
}
// rows: that of the first of the tokens
__global__ __launch_bounds__(256) void embed_rows_kernel(const int* __restrict__ ids, TokenRow rows) {
    rows.out += (size_t)blockIdx.x * rows.hidden;
    embed_token(rows, ids[blockIdx.x]);
}

// of two candidates the larger value, of equal values the lower index; a NaN is no candidate
__device__ __forceinline__ void take_better(float& v, int& i, float ov, int oi) {
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

// Between two tokens of the loop: first index of the maximum of logits[0..n), written to next_id[0] and to history[*step]; the step
// counter and the position advance (the token just consumed is now in the cache); the row of the next token, if the next pass takes
// it (row.out).  What bounds it is the chain: logits, which thread, the row.  A token of Qwen3, Takosun,
// Dimesun with launches of their own for the row and the position, and four float4s in flight: 222.7, 248.8, 192.7 us, so 216.1, 241.9, 186.0.
__global__ __launch_bounds__(1024) void next_token_kernel(const float* __restrict__ logits, int n, int* __restrict__ next_id,
                                                        int* __restrict__ history, int history_len, int* __restrict__ step_dev,
                                                        int* __restrict__ pos_dev, int by, TokenRow row) {
    __shared__ float best_v[16];
    __shared__ int best_i[16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    constexpr float kNone = -3.402823466e38f;
    float bv = kNone;
    int bi = 0x7fffffff;
    int st = 0;
    if (t == 0) st = step_dev[0];
    // logits are 16-byte aligned: scan float4s, eight in flight, then the up to three left over
    const float4* l4 = reinterpret_cast<const float4*>(logits);
    const int n4 = n >> 2;
    constexpr int U = 8;
    for (int j0 = t; j0 < n4; j0 += U * 1024) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = l4[min(j0 + u * 1024, n4 - 1)];  // past the end its last ones again, which change nothing
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = 4 * min(j0 + u * 1024, n4 - 1);  // indices rise within a thread, so '>' keeps the first maximum
            const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (e[k] > bv) {
                    bv = e[k];
                    bi = i + k;
                }
        }
    }
    if (t < (n & 3)) {
        const float e = logits[4 * n4 + t];
        if (e > bv) {
            bv = e;
            bi = 4 * n4 + t;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) take_better(bv, bi, __shfl_xor(bv, off, 64), __shfl_xor(bi, off, 64));
    if (lane == 0) best_v[wave] = bv, best_i[wave] = bi;
    __syncthreads();
    bv = best_v[lane & 15], bi = best_i[lane & 15];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) take_better(bv, bi, __shfl_xor(bv, off, 64), __shfl_xor(bi, off, 64));
    const int id = bi == 0x7fffffff ? 0 : bi;
    if (row.out) embed_token(row, id);
    if (t == 0) {
        next_id[0] = id;
        if (st >= 0 && st < history_len) history[st] = id;
        step_dev[0] = st + 1;
        if (by) pos_dev[0] += by;
    }
}

// What the host left in pinned memory, read over the bus: a launch in the stream's order, where a copy would make the host wait twice.
__global__ __launch_bounds__(256) void take_tokens_kernel(const int* host_ids, int n, int* __restrict__ ids, const int* host_want, int n_want,
                                                        int* __restrict__ want) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        ids[i] = host_ids[i];
    else if (i - n < n_want)
        want[i - n] = host_want[i - n];
}
// One token, and its embedding row for the pass; a wanted place of one token is 0.
__global__ __launch_bounds__(256) void take_token_kernel(const int* host_id, int* __restrict__ ids, int* __restrict__ want, TokenRow row) {
    const int id = host_id[0];
    embed_token(row, id);
    if (threadIdx.x == 0) ids[0] = id, want[0] = 0;
}
// Behind a pass's logits the position is free to advance.
__global__ __launch_bounds__(256) void give_floats_kernel(const float* __restrict__ x, float* host, size_t n, int* __restrict__ pos_dev, int by) {
    if (by && blockIdx.x == 0 && threadIdx.x == 0) pos_dev[0] += by;
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) host[i] = x[i];
}
__global__ __launch_bounds__(256) void zero_words_kernel(unsigned* __restrict__ p, size_t n) {
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0;
}
__global__ void advance_kernel(int* __restrict__ pos_dev, int by) {
    if (threadIdx.x == 0 && blockIdx.x == 0) pos_dev[0] += by;
}

}  // namespace

hipError_t launch_embed_rows(const int* ids, const void* table, TableType type, int ld, float* out, int M, int hidden, int vocab,
                             hipStream_t s) {
    hipLaunchKernelGGL(embed_rows_kernel, dim3(M), dim3(256), 0, s, ids, TokenRow{table, type, ld, out, hidden, vocab});
    return hipGetLastError();
}
static hipError_t next_token(const float* logits, int n, int* next_id, int* history, int history_len, int* step_dev, int* pos_dev, int by,
                             const TokenRow& row, hipStream_t s) {
    hipLaunchKernelGGL(next_token_kernel, dim3(1), dim3(1024), 0, s, logits, n, next_id, history, history_len, step_dev, pos_dev, by, row);
    return hipGetLastError();
}
hipError_t launch_argmax_token(const float* logits, int n, int* next_id, int* history, int history_len, int* step_dev, hipStream_t s) {
    return next_token(logits, n, next_id, history, history_len, step_dev, nullptr, 0, TokenRow{}, s);
}
static hipError_t take_token(const int* host_id, int* ids, int* want, const TokenRow& row, hipStream_t s) {
    hipLaunchKernelGGL(take_token_kernel, dim3(1), dim3(256), 0, s, host_id, ids, want, row);
    return hipGetLastError();
}
hipError_t launch_take_tokens(const int* host_ids, int n, int* ids, const int* host_want, int n_want, int* want, hipStream_t s) {
    hipLaunchKernelGGL(take_tokens_kernel, dim3((n + n_want + 255) / 256), dim3(256), 0, s, host_ids, n, ids, host_want, n_want, want);
    return hipGetLastError();
}
static hipError_t give_floats(const float* x, float* host, size_t n, int* pos_dev, int by, hipStream_t s) {
    hipLaunchKernelGGL(give_floats_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 256)), dim3(256), 0, s, x, host, n, pos_dev, by);
    return hipGetLastError();
}
hipError_t launch_give_floats(const float* x, float* host, size_t n, hipStream_t s) { return give_floats(x, host, n, nullptr, 0, s); }
const JoinedLaunches* all_joined_launches() {
    static const JoinedLaunches table = {take_token, next_token, give_floats};
    return &table;
}
hipError_t launch_zero_words(void* p, size_t words, hipStream_t s) {
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)std::min<size_t>((words + 255) / 256, 1024)), dim3(256), 0, s,
                       static_cast<unsigned*>(p), words);
    return hipGetLastError();
}
hipError_t launch_advance(int* pos_dev, int by, hipStream_t s) {
    hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(64), 0, s, pos_dev, by);
    return hipGetLastError();
}

}  // namespace a81w41
