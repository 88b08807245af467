// Latent attention: per token the cache holds one normed latent and one rotated key part, shared by all heads.  A
// head's unrotated key is W_uk c, so q . (W_uk c) = (W_uk^T q) . c: with the up-projection moved into the query, a
// query row has the layout of a cache row and the score is one dot product; the value is W_uv sum_j p_j c_j.
// Positions come from device memory; every index that depends on them is clamped into its array.
#include "dense_common.h"

namespace a81w41 {
namespace {

constexpr int kThreads = 256;

// One workgroup per token.
template <typename T>
__global__ __launch_bounds__(kThreads) void latent_rows_kernel(LatentRows in, LatentShape sh, T* __restrict__ q_latent, int ld_q,
                                                              T* __restrict__ cache) {
    __shared__ float inv[2], red[kThreads / 64];
    const int m = blockIdx.x, t = threadIdx.x;
    const float* row = in.down + (size_t)m * in.ld_down;
    group_inverse_rms<kThreads>([&](int i) { return row[i]; }, sh.q_rank, 1, in.eps, inv, red);
    for (int i = t; i < sh.q_rank; i += kThreads) q_latent[(size_t)m * ld_q + i] = (T)(row[i] * inv[0] * in.q_norm[i]);
    if (!cache) return;
    const float* c = row + sh.q_rank;
    group_inverse_rms<kThreads>([&](int i) { return c[i]; }, sh.rank, 1, in.eps, inv + 1, red);
    const int p = min(max(in.pos_dev[0] + m, 0), in.max_seq - 1);
    T* dst = cache + (size_t)p * sh.ld_cache;
    for (int i = t; i < sh.rank; i += kThreads) dst[i] = (T)(c[i] * inv[1] * in.kv_norm[i]);
    const int half = sh.rot >> 1;
    const float* k = c + sh.rank;
    for (int i = t; i < half; i += kThreads) {
        const float cs = in.cos_t[(size_t)p * half + i], sn = in.sin_t[(size_t)p * half + i];
        dst[sh.rank + 2 * i] = (T)(k[2 * i] * cs - k[2 * i + 1] * sn);
        dst[sh.rank + 2 * i + 1] = (T)(k[2 * i + 1] * cs + k[2 * i] * sn);
    }
}

}  // namespace

template <typename T>
hipError_t launch_latent_rows(const LatentRows& in, const LatentShape& sh, int M, T* q_latent, int ld_q, T* cache, hipStream_t s) {
    hipLaunchKernelGGL(latent_rows_kernel<T>, dim3(M), dim3(kThreads), 0, s, in, sh, q_latent, ld_q, cache);
    return hipGetLastError();
}

template hipError_t launch_latent_rows<bf16>(const LatentRows&, const LatentShape&, int, bf16*, int, bf16*, hipStream_t);
template hipError_t launch_latent_rows<float>(const LatentRows&, const LatentShape&, int, float*, int, float*, hipStream_t);

}  // namespace a81w41
