// Matrix memory token by token: the work of a workgroup, for a kernel of its own (matrix_memory.hip) and beside another product
// (dense_gemv.hip).
#pragma once
#include "dense_common.h"

namespace a81w41 {
namespace memory {

constexpr int kThreads = 256;

__device__ __forceinline__ float soft_cap(float z, float cap) { return cap * tanhf(z / cap); }
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
struct Gates {
    float log_in, log_keep;
};
__device__ __forceinline__ Gates gates_of(const MemoryArgs& a, int m, int h) {
    const float* row = a.in + (size_t)m * a.ld_in;
    Gates g;
    g.log_in = soft_cap(row[a.sh.at_i + h] + a.bias_i[h], a.sh.cap);
    g.log_keep = log_sigmoid(soft_cap(row[a.sh.at_f + h] + a.bias_f[h], a.sh.cap));
    return g;
}

__device__ __forceinline__ float* state_nm(const MemoryArgs& a, int parity) {
    return a.state + a.sh.s_size() + (size_t)(parity & 1) * a.sh.heads * (a.sh.dim + 1);
}

// Token by token.  A workgroup has kSlice columns of one head's S; W columns and every (kThreads W / kSlice)-th row of them
// are a thread's, in registers only while a token uses them.  n and m are formed by every workgroup of the head; the first
// writes them to the copy of the parity behind the tokens, which nobody reads if their number is odd.  With an even number it is the copy
// that all of them start from, also those that start when the first has ended: n and m are then held back for the launch behind (memory_norm_kernel).
constexpr int kSlice = 32;
// smem: step_floats(dim, W)
__host__ __device__ inline int step_floats(int dim, int w) { return 3 * dim + kThreads * w + kThreads / 64; }
__host__ __device__ inline bool steps_held_back(const MemoryArgs& a) { return a.M % 2 == 0 && a.sh.vdim > kSlice; }
template <int W>
__device__ __forceinline__ void memory_steps(const MemoryArgs& a, float* __restrict__ o, int slice, int h, float* smem) {
    constexpr int kPer = kSlice / W, kRows = kThreads / kPer;  // threads of a row of the slice, rows worked on at a time
    const MemoryShape sh = a.sh;
    float *n = smem, *q = n + sh.dim, *k = q + sh.dim, *sums = k + sh.dim, *red = sums + kRows * kSlice;
    const int t = threadIdx.x, pos = max(a.pos_dev[0], 0);
    const int c = slice * kSlice + (t % kPer) * W, r0 = t / kPer;
    const bool mine = c < sh.vdim;  // W > 1: vdim is a multiple of W
    float* S = a.state + (size_t)h * sh.dim * sh.vdim;
    const float* nm = state_nm(a, pos) + (size_t)h * (sh.dim + 1);
    for (int d = t; d < sh.dim; d += kThreads) n[d] = nm[d];
    float m = nm[sh.dim];
    for (int token = 0; token < a.M; token++) {
        const float* row = a.in + (size_t)token * a.ld_in;
        const Gates g = gates_of(a, token, h);
        const float next = fmaxf(g.log_keep + m, g.log_in), keep = expf(g.log_keep + m - next), add = expf(g.log_in - next);
        m = next;
        float nq = 0.f;
        for (int d = t; d < sh.dim; d += kThreads) {
            q[d] = row[sh.at_q + h * sh.dim + d] * sh.q_scale;
            k[d] = add * row[sh.at_k + h * sh.dim + d];
            n[d] = fmaf(keep, n[d], k[d]);
            nq = fmaf(n[d], q[d], nq);
        }
        nq = dense_wave_sum(nq);
        if ((t & 63) == 0) red[t >> 6] = nq;
        __syncthreads();
        float acc[W], v[W];
#pragma unroll
        for (int w = 0; w < W; w++) {
            acc[w] = 0.f;
            v[w] = mine ? row[sh.at_v + h * sh.vdim + c + w] : 0.f;
        }
        if (mine) {
#pragma unroll 8
            for (int d = r0; d < sh.dim; d += kRows) {
                float* at = S + (size_t)d * sh.vdim + c;
                float s[W];
                if constexpr (W == 4)
                    *reinterpret_cast<float4*>(s) = load4(at);
                else
                    s[0] = at[0];
#pragma unroll
                for (int w = 0; w < W; w++) {
                    s[w] = fmaf(keep, s[w], k[d] * v[w]);
                    acc[w] = fmaf(s[w], q[d], acc[w]);
                }
                if constexpr (W == 4)
                    store4(at, *reinterpret_cast<const float4*>(s));
                else
                    at[0] = s[0];
            }
        }
#pragma unroll
        for (int w = 0; w < W; w++) sums[r0 * kSlice + (t % kPer) * W + w] = acc[w];
        __syncthreads();
        const int col = slice * kSlice + t;
        if (t < kSlice && col < sh.vdim) {
            float s = 0.f, den = 0.f;
            for (int r = 0; r < kRows; r++) s += sums[r * kSlice + t];
            for (int w = 0; w < kThreads / 64; w++) den += red[w];
            o[((size_t)token * sh.heads + h) * sh.vdim + col] = s / (fmaxf(fabsf(den), expf(-m)) + kMemoryFloor);
        }
        __syncthreads();
    }
    if (slice == 0) {
        float* out = (steps_held_back(a) ? a.held : state_nm(a, pos + a.M)) + (size_t)h * (sh.dim + 1);
        for (int d = t; d < sh.dim; d += kThreads) out[d] = n[d];
        if (t == 0) out[sh.dim] = m;
    }
}

}  // namespace memory
}  // namespace a81w41
