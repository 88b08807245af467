// One-token products for dense weights, with the row work around them fused in: every workgroup forms the input row in
// LDS (fp32) in its prologue -- residual step and norm, the norm of a latent, the attention output -- and its waves
// then stream weight rows in pairs, 16 bytes per lane and load, the next eight loads in flight while eight are used; the
// first ones are requested before the prologue.  A row's sum is formed
// in an order that depends on the row's length only.
#include "attend_rows.h"
#include "memory_steps.h"

namespace a81w41 {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float dot16(const uint4& w, const float* x, bf16*) {
    const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
    float s = __uint_as_float(w.x << 16) * a.x;
    s = fmaf(__uint_as_float(w.x & 0xffff0000u), a.y, s);
    s = fmaf(__uint_as_float(w.y << 16), a.z, s);
    s = fmaf(__uint_as_float(w.y & 0xffff0000u), a.w, s);
    s = fmaf(__uint_as_float(w.z << 16), b.x, s);
    s = fmaf(__uint_as_float(w.z & 0xffff0000u), b.y, s);
    s = fmaf(__uint_as_float(w.w << 16), b.z, s);
    return fmaf(__uint_as_float(w.w & 0xffff0000u), b.w, s);
}
__device__ __forceinline__ float dot16(const uint4& w, const float* x, float*) {
    const float4 a = *reinterpret_cast<const float4*>(x);
    float s = __uint_as_float(w.x) * a.x;
    s = fmaf(__uint_as_float(w.y), a.y, s);
    s = fmaf(__uint_as_float(w.z), a.z, s);
    return fmaf(__uint_as_float(w.w), a.w, s);
}

constexpr int kAhead = 4;  // 16-byte chunks of a row that a lane requests at once
__host__ __device__ constexpr int lanes_of(int chunks) {
    int lanes = 1;
    while (lanes < 64 && lanes * kAhead < chunks) lanes <<= 1;
    return lanes;
}
// How rows are dealt: `lanes` lanes (a power of two) share a pair of rows; `group` counts the lane groups of the launch.
struct Deal {
    int lanes, group, groups, at;
};
template <typename T>
__device__ __forceinline__ Deal deal_rows(int chunks, int workgroups) {
    Deal d;
    d.lanes = lanes_of(chunks);
    const int per_wg = kThreads / d.lanes;
    d.group = blockIdx.x * per_wg + threadIdx.x / d.lanes;
    d.groups = workgroups * per_wg;
    d.at = threadIdx.x & (d.lanes - 1);
    return d;
}

// Up to kAhead chunks per lane of two weight rows.
struct Pair {
    uint4 a[kAhead], b[kAhead];
};
struct RowPair {
    const void *w0, *w1;
};
__device__ __forceinline__ void load_pair(Pair& p, const RowPair& r, int c, int lanes, int chunks) {
    const uint4 *p0 = static_cast<const uint4*>(r.w0), *p1 = static_cast<const uint4*>(r.w1);
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
        const int cc = min(c + u * lanes, chunks - 1);
        p.a[u] = p0[cc];
        p.b[u] = p1[cc];
    }
}
template <typename T>
__device__ __forceinline__ void use_pair(const Pair& p, const float* xs, int c, int lanes, int chunks, float& s0, float& s1) {
    constexpr int E = 16 / (int)sizeof(T);
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
        const int cc = c + u * lanes;
        if (cc < chunks) {
            s0 += dot16(p.a[u], xs + cc * E, static_cast<T*>(nullptr));
            s1 += dot16(p.b[u], xs + cc * E, static_cast<T*>(nullptr));
        }
    }
}

// The lane group's share of `pairs` row pairs: rows(n) names pair n, emit(n, s0, s1) gets the dot products with xs (LDS,
// zero-padded to whole chunks).  The loads run one step ahead; `ahead` holds the first one's, requested by
// request_first before the caller's prologue.
template <typename Rows>
__device__ __forceinline__ void request_first(Pair& ahead, Rows rows, int pairs, int chunks, const Deal& d) {
    if (d.group < pairs) load_pair(ahead, rows(d.group), d.at, d.lanes, chunks);
}
template <typename T, typename Rows, typename Emit>
__device__ __forceinline__ void stream_pairs(Pair& ahead, Rows rows, Emit emit, int pairs, const float* xs, int chunks, const Deal& d) {
    const int per_step = kAhead * d.lanes, steps = (chunks + per_step - 1) / per_step;
    for (int n = d.group; n < pairs; n += d.groups) {
        float s0 = 0.f, s1 = 0.f;
        for (int step = 0; step < steps; step++) {
            const int c = d.at + step * per_step;
            const Pair now = ahead;
            if (step + 1 < steps)
                load_pair(ahead, rows(n), c + per_step, d.lanes, chunks);
            else if (n + d.groups < pairs)
                load_pair(ahead, rows(n + d.groups), d.at, d.lanes, chunks);
            use_pair<T>(now, xs, c, d.lanes, chunks, s0, s1);
        }
        s0 = dense_wave_sum(s0, d.lanes);
        s1 = dense_wave_sum(s1, d.lanes);
        if (d.at == 0) emit(n, s0, s1);
    }
}
// Rows 2 n and 2 n + 1 of a plain matrix.
template <typename T>
struct PlainRows {
    const T* w;
    int ld, N;
    __device__ RowPair operator()(int n) const { return {w + (size_t)(2 * n) * ld, w + (size_t)min(2 * n + 1, N - 1) * ld}; }
};
struct PlainEmit {
    float* C;
    int N;
    float factor;
    __device__ void operator()(int n, float s0, float s1) const {
        C[2 * n] = s0 * factor;
        if (2 * n + 1 < N) C[2 * n + 1] = s1 * factor;
    }
};

// xs[0 .. padded) = f(i), zero from n on
template <typename F>
__device__ __forceinline__ void fill_row(float* xs, int n, int padded, F f) {
    for (int i = threadIdx.x; i < padded; i += kThreads) xs[i] = i < n ? f(i) : 0.f;
}

// xs[0 .. padded) = src[0 .. n), zero from n on; sixteen bytes per load where the row is made of whole float4s
__device__ __forceinline__ void copy_row(float* xs, const float* src, int n, int padded) {
    if (((n & 3) | (int)(reinterpret_cast<uintptr_t>(src) & 15)) == 0) {
#pragma unroll 4
        for (int i = 4 * threadIdx.x; i < n; i += 4 * kThreads) store4(xs + i, load4(src + i));
        for (int i = n + threadIdx.x; i < padded; i += kThreads) xs[i] = 0.f;
    } else {
        fill_row(xs, n, padded, [&](int i) { return src[i]; });
    }
}

// The residual step and the norm of RowStep into xs; workgroup 0 of the launch also writes the stream.  Rows whose parts
// are whole float4s and fit PARTS of them per thread are requested at once by load() and stay in registers (a part's
// threads are neighbours); other rows are read when they are needed.
template <int PARTS>
class StepRow {
   public:
    __device__ __forceinline__ explicit StepRow(const RowStep& p) : p_(p), parts_(p.width, p.norm_h.groups, threadIdx.x), fast_(parts_.fits()) {}
    __device__ __forceinline__ void load() {
        if (!fast_) return;
        if (p_.before && p_.coef) coef_ = *p_.coef;
        // Without a branch a load: a thread without a part takes the row's first one and drops it.  A Takosun token, 16 such rows of 2048:
        // 254.6 us with a branch each, 249.2 so.
        auto part = [&](const float* a, int i) { return load4(a + max(i, 0)); };
        auto kept = [](float4 v, int i) { return make_float4(i < 0 ? 0.f : v.x, i < 0 ? 0.f : v.y, i < 0 ? 0.f : v.z, i < 0 ? 0.f : v.w); };
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        int at[kParts];
#pragma unroll
        for (int k = 0; k < kParts; k++) at[k] = parts_.place(k), y_[k] = wy_[k] = before_[k] = zero;
#pragma unroll
        for (int k = 0; k < kParts; k++) x_[k] = part(p_.x, at[k]), wh_[k] = part(p_.norm_h.w, at[k]);
        if (p_.y)
#pragma unroll
            for (int k = 0; k < kParts; k++) y_[k] = part(p_.y, at[k]);
        if (p_.norm_y.w)
#pragma unroll
            for (int k = 0; k < kParts; k++) wy_[k] = part(p_.norm_y.w, at[k]);
        if (p_.before)
#pragma unroll
            for (int k = 0; k < kParts; k++) before_[k] = part(p_.before, at[k]);
#pragma unroll
        for (int k = 0; k < kParts; k++) {
            x_[k] = kept(x_[k], at[k]), y_[k] = kept(y_[k], at[k]);
            wy_[k] = kept(wy_[k], at[k]), before_[k] = kept(before_[k], at[k]);
        }
    }
    __device__ __forceinline__ void finish(float* xs, int padded, float* inv, float* red) {
        if (!fast_) return slow(xs, padded, inv, red);
        const bool writer = blockIdx.x == 0 && blockIdx.y == 0;
        const float coef = coef_;
        const bool normed = p_.y && p_.norm_y.w;
        const float inv_y = normed ? parts_.inverse_rms(y_, p_.norm_y.eps, red) : 0.f;
#pragma unroll
        for (int k = 0; k < kParts; k++) {
            const int i = parts_.place(k);
            float4 r = normed ? add4(x_[k], scale4(y_[k], inv_y, wy_[k])) : fma4(p_.norm_y.scale, y_[k], x_[k]);
            if (i >= 0 && writer && p_.state) store4(p_.state + i, r);
            if (p_.before) r = fma4(coef, r, before_[k]);
            if (i >= 0 && writer && p_.x_out) store4(p_.x_out + i, r);
            x_[k] = r;
        }
        const float inv_h = parts_.inverse_rms(x_, p_.norm_h.eps, red);
#pragma unroll
        for (int k = 0; k < kParts; k++) {
            const int i = parts_.place(k);
            if (i < 0) continue;
            const float4 h = scale4(x_[k], inv_h, wh_[k]);
            store4(xs + i, h);
            if (writer && p_.h_out) store4(p_.h_out + i, h);
        }
        for (int i = p_.width + threadIdx.x; i < padded; i += kThreads) xs[i] = 0.f;
        dense_lds_barrier();
    }

   private:
    static constexpr int kParts = PARTS;
    __device__ void slow(float* xs, int padded, float* inv, float* red) const {
        const RowStep& p = p_;
        const int t = threadIdx.x, W = p.width;
        const bool writer = blockIdx.x == 0 && blockIdx.y == 0;
        const bool normed = p.y && p.norm_y.w;
        if (normed) group_inverse_rms<kThreads>([&](int i) { return p.y[i]; }, W, p.norm_y.groups, p.norm_y.eps, inv, red);
        const float coef = p.before && p.coef ? *p.coef : 1.f;
        const int size_y = normed ? W / p.norm_y.groups : 1;
        for (int i = t; i < padded; i += kThreads) {
            float r = 0.f;
            if (i < W) {
                r = p.x[i];
                if (p.y) r = normed ? r + p.y[i] * inv[i / size_y] * p.norm_y.w[i] : fmaf(p.norm_y.scale, p.y[i], r);
                if (writer && p.state) p.state[i] = r;
                if (p.before) r = fmaf(coef, r, p.before[i]);
                if (writer && p.x_out) p.x_out[i] = r;
            }
            xs[i] = r;
        }
        __syncthreads();
        group_inverse_rms<kThreads>([&](int i) { return xs[i]; }, W, p.norm_h.groups, p.norm_h.eps, inv, red);
        const int size_h = W / p.norm_h.groups;
        for (int i = t; i < W; i += kThreads) {
            xs[i] = xs[i] * inv[i / size_h] * p.norm_h.w[i];
            if (writer && p.h_out) p.h_out[i] = xs[i];
        }
        __syncthreads();
    }
    const RowStep& p_;
    RowParts<kThreads, PARTS> parts_;
    bool fast_;
    float coef_ = 1.f;
    float4 x_[kParts], y_[kParts], wy_[kParts], before_[kParts], wh_[kParts];
};

template <typename T>
struct HeadsEmit {
    HeadRows<T> heads;
    int N;
    __device__ void operator()(int n, float s0, float s1) const {
        const int pos = min(max(heads.pos_dev[0], 0), heads.max_seq - 1);
        store(2 * n, pos, s0, s1);
        if (2 * n + 1 < N) store(2 * n + 1, pos, s1, s0);
    }
    // One column of one row, branch by branch; a place for many rows, as the products of more rows form it, is slower here (rows of 4096, 772
    // workgroups: 18.1 us, so 17.8).
    __device__ void store(int col, int pos, float own, float other) const {
        const HeadRows<T>& p = heads;
        const int nq = p.heads * p.dim, nk = p.kv_heads * p.dim, nv = p.kv_heads * p.vdim;
        if (col >= nq + nk + nv) {
            p.rest[col - nq - nk - nv] = own;
            return;
        }
        if (col >= nq + nk) {
            const int c = col - nq - nk, h = c / p.vdim;
            p.cache[(size_t)pos * p.ld_cache + h * (p.vdim + p.dim) + (c - h * p.vdim)] = (T)own;
            return;
        }
        const bool key = col >= nq;
        const int c = key ? col - nq : col, h = c / p.dim, d = c - h * p.dim;
        if ((d >> 1) < p.rot_pairs) {
            const size_t i = (size_t)pos * p.rot_pairs + (d >> 1);
            const float cs = p.cos_t[i], sn = p.sin_t[i];
            own = (d & 1) ? own * cs + other * sn : own * cs - other * sn;
        }
        if (key)
            p.cache[(size_t)pos * p.ld_cache + h * (p.vdim + p.dim) + p.vdim + d] = (T)own;
        else
            p.q[c] = (T)own;
    }
};

// What a workgroup's first requests are made of stands ahead of the structs in the kernels' arguments: 14 leading dwords of scalars come with
// the dispatch, the others with a load that the requests would wait for.  us a token behind a short prompt with the structs first / so:
// Takosun, four layers, width 2048 241.5 / 234.6, 4096 480 / 465; Dimesun, two layers run twice, width 1024 151 / 145.  A launch of 784 rows
// of 2048 behind a residual step 6.6 / 5.8 us, of which the mean's coefficient, asked for only behind the row, is a part.
__device__ __forceinline__ void with_leading(RowStep& p, const float* x, const float* norm_h, const float* y, const float* norm_y, int width, int groups) {
    p.x = x, p.norm_h.w = norm_h, p.y = y, p.norm_y.w = norm_y, p.width = width, p.norm_h.groups = groups;
}
#define LEADING_OF(p) (p).x, (p).norm_h.w, (p).y, (p).norm_y.w

// emit gets W[n] . row, in pairs of n
template <typename T, int PARTS, typename Emit>
__global__ __launch_bounds__(kThreads) void gemv_step_kernel(const float* __restrict__ x, const float* __restrict__ norm_h, const float* __restrict__ y,
                                                            const float* __restrict__ norm_y, const T* __restrict__ w, int width, int groups, int ld,
                                                            int N, RowStep p, Emit emit, WeightsAhead later) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    if (blockIdx.y) {  // behind the launch's own workgroups
        const int n = (blockIdx.y - 1) * gridDim.x + blockIdx.x;
        return read_ahead<kThreads>(later, (gridDim.y - 1) * gridDim.x, n, gridDim.x + n);
    }
    with_leading(p, x, norm_h, y, norm_y, width, groups);
    float *xs = smem, *red = xs + ld, *inv = red + kThreads / 64;
    StepRow<PARTS> row(p);
    row.load();
    const int chunks = ld * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    const PlainRows<T> rows{w, ld, N};
    Pair ahead;
    request_first(ahead, rows, pairs, chunks, d);
    row.finish(xs, ld, inv, red);
    stream_pairs<T>(ahead, rows, emit, pairs, xs, chunks, d);
}

// C[n] = W[n] . x
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_plain_kernel(const float* __restrict__ x, int K, const T* __restrict__ w, int ld, int N,
                                                             float* __restrict__ C) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int chunks = ld * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    const PlainRows<T> rows{w, ld, N};
    Pair ahead;
    request_first(ahead, rows, pairs, chunks, d);
    copy_row(smem, x, K, ld);
    dense_lds_barrier();
    stream_pairs<T>(ahead, rows, PlainEmit{C, N, 1.f}, pairs, smem, chunks, d);
}

// A latent made of whole float4s, and the weights of its norm: held by the workgroup's threads from one request on.  What the queries'
// launch waits for is trips to memory, and the norm's weights, the angles and every state of the mean over depth were one
// each behind the row's: with 3072 x 768 weights 6.5 us, so 5.0; a Takosun token of four layers, width 2048, 246.5 -> 241.0 us, 4096
// 478 -> 469 us.
class NormedLatent {
   public:
    static __device__ __forceinline__ bool fits(const float* x, const float* w, int n) {
        return n <= 4 * kQuads * kThreads && ((n & 3) | (int)((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15)) == 0;
    }
    __device__ __forceinline__ void load(const float* x, const float* w, int n) {
#pragma unroll
        for (int u = 0; u < kQuads; u++) x_[u] = load4(x + min(at(u), n - 4));
#pragma unroll
        for (int u = 0; u < kQuads; u++) w_[u] = load4(w + min(at(u), n - 4));
    }
    // store(i, v): elements i .. i + 3.  red: kThreads / 64 floats of LDS
    template <typename Store>
    __device__ __forceinline__ void finish(int n, float eps, float* red, Store store) {
        float sum = 0.f;
#pragma unroll
        for (int u = 0; u < kQuads; u++) {
            if (at(u) >= n) x_[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            sum = fmaf(x_[u].x, x_[u].x, sum), sum = fmaf(x_[u].y, x_[u].y, sum);
            sum = fmaf(x_[u].z, x_[u].z, sum), sum = fmaf(x_[u].w, x_[u].w, sum);
        }
        sum = dense_wave_sum(sum);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
        dense_lds_barrier();
        sum = 0.f;
        for (int k = 0; k < kThreads / 64; k++) sum += red[k];
        const float scale = 1.0f / sqrtf(sum / (float)n + eps);
#pragma unroll
        for (int u = 0; u < kQuads; u++)
            if (at(u) < n) store(at(u), scale4(x_[u], scale, w_[u]));
    }

   private:
    static constexpr int kQuads = 2;
    static __device__ __forceinline__ int at(int u) { return 4 * (u * kThreads + (int)threadIdx.x); }
    float4 x_[kQuads], w_[kQuads];
};

// Queries from their normed latent.  The last workgroups of the launch do other work of the same stage: one appends the
// token's cache row, the others sum the states of the layers so far for the mean over depth.
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_query_kernel(const float* __restrict__ down, const float* __restrict__ q_norm, const T* __restrict__ w,
                                                             int q_rank, int ld, int N, int main_groups, float* __restrict__ q,
                                                             T* __restrict__ cache, LatentRows in, LatentShape sh, DepthAverage depth, int width,
                                                             float* __restrict__ before) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    in.down = down, in.q_norm = q_norm, sh.q_rank = q_rank;
    float *xs = smem, *red = xs + ld, *inv = red + kThreads / 64;
    const int t = threadIdx.x;
    if ((int)blockIdx.x >= main_groups) {
        int extra = blockIdx.x - main_groups;
        if (cache && extra-- == 0) {
            const float* c = in.down + sh.q_rank;
            const int p = min(max(in.pos_dev[0], 0), in.max_seq - 1), half = sh.rot >> 1;
            T* dst = cache + (size_t)p * sh.ld_cache;
            const float* k = c + sh.rank;
            if (NormedLatent::fits(c, in.kv_norm, sh.rank) && half <= kThreads) {
                NormedLatent latent;
                latent.load(c, in.kv_norm, sh.rank);
                const int j = min(t, half - 1);
                float re = 0.f, im = 0.f, cs = 0.f, sn = 0.f;
                if (half) re = k[2 * j], im = k[2 * j + 1], cs = in.cos_t[(size_t)p * half + j], sn = in.sin_t[(size_t)p * half + j];
                latent.finish(sh.rank, in.eps, red, [&](int i, float4 v) { dst[i] = (T)v.x, dst[i + 1] = (T)v.y, dst[i + 2] = (T)v.z, dst[i + 3] = (T)v.w; });
                if (t < half) {
                    dst[sh.rank + 2 * t] = (T)(re * cs - im * sn);
                    dst[sh.rank + 2 * t + 1] = (T)(im * cs + re * sn);
                }
                return;
            }
            group_inverse_rms<kThreads>([&](int i) { return c[i]; }, sh.rank, 1, in.eps, inv, red);
            for (int i = t; i < sh.rank; i += kThreads) dst[i] = (T)(c[i] * inv[0] * in.kv_norm[i]);
            for (int i = t; i < half; i += kThreads) {
                const float cs = in.cos_t[(size_t)p * half + i], sn = in.sin_t[(size_t)p * half + i];
                dst[sh.rank + 2 * i] = (T)(k[2 * i] * cs - k[2 * i + 1] * sn);
                dst[sh.rank + 2 * i + 1] = (T)(k[2 * i + 1] * cs + k[2 * i] * sn);
            }
        } else {
            const int i = extra * kThreads + t;
            if (i < width) {
                constexpr int U = 8;  // states requested at a time
                float s = 0.f;
                for (int j0 = 0; j0 < depth.n; j0 += U) {
                    float state[U], coef[U];
#pragma unroll
                    for (int u = 0; u < U; u++) state[u] = depth.states[min(j0 + u, depth.n - 1) * depth.state_step + i];
#pragma unroll
                    for (int u = 0; u < U; u++) coef[u] = depth.coef[min(j0 + u, depth.n - 1)];
#pragma unroll
                    for (int u = 0; u < U; u++) s = j0 + u < depth.n ? fmaf(coef[u], state[u], s) : s;
                }
                before[i] = s;
            }
        }
        return;
    }
    const int chunks = ld * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    const Deal d = deal_rows<T>(chunks, main_groups);
    const PlainRows<T> rows{w, ld, N};
    Pair ahead;
    if (NormedLatent::fits(in.down, in.q_norm, sh.q_rank)) {
        NormedLatent latent;
        latent.load(in.down, in.q_norm, sh.q_rank);
        request_first(ahead, rows, pairs, chunks, d);
        latent.finish(sh.q_rank, in.eps, red, [&](int i, float4 v) { store4(xs + i, v); });
        for (int i = sh.q_rank + t; i < ld; i += kThreads) xs[i] = 0.f;
    } else {
        request_first(ahead, rows, pairs, chunks, d);
        fill_row(xs, sh.q_rank, ld, [&](int i) { return in.down[i]; });
        float sum = 0.f;  // of this thread's own elements
        for (int i = t; i < sh.q_rank; i += kThreads) sum = fmaf(xs[i], xs[i], sum);
        sum = dense_wave_sum(sum);
        if ((t & 63) == 0) red[t >> 6] = sum;
        dense_lds_barrier();
        sum = 0.f;
        for (int k = 0; k < kThreads / 64; k++) sum += red[k];
        const float scale = 1.0f / sqrtf(sum / (float)sh.q_rank + in.eps);
        for (int i = t; i < sh.q_rank; i += kThreads) xs[i] *= scale * in.q_norm[i];
    }
    dense_lds_barrier();
    stream_pairs<T>(ahead, rows, PlainEmit{q, N, 1.f}, pairs, xs, chunks, d);
}

// Query rows in latent space, one head per blockIdx.y: columns 0..rank from the unrotated part through the transposed key
// up-projection, then the rotated part (first workgroup of the head).
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_absorb_kernel(const float* __restrict__ q, const T* __restrict__ uk_t, int ld, int rank, int dim, int rot,
                                                              T* __restrict__ q_lat, const int* __restrict__ pos_dev, LatentRows in, LatentShape sh) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    in.pos_dev = pos_dev, sh.rank = rank, sh.dim = dim, sh.rot = rot;
    const int h = blockIdx.y, half = sh.rot >> 1;
    const float *src = q + (size_t)h * sh.query_width(), *turned = src + sh.turned_at();
    T* dst = q_lat + (size_t)h * sh.ld_cache;
    const int N = sh.rank, chunks = ld * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    const PlainRows<T> rows{uk_t + (size_t)h * N * ld, ld, N};
    Pair ahead;
    request_first(ahead, rows, pairs, chunks, d);
    copy_row(smem, src, sh.dim, ld);
    if (blockIdx.x == 0) {
        const int p = min(max(in.pos_dev[0], 0), in.max_seq - 1);
        for (int j = threadIdx.x; j < half; j += kThreads) {
            const float u = turned[2 * j], v = turned[2 * j + 1];
            const float cs = in.cos_t[(size_t)p * half + j], sn = in.sin_t[(size_t)p * half + j];
            dst[sh.rank + 2 * j] = (T)(u * cs - v * sn);
            dst[sh.rank + 2 * j + 1] = (T)(v * cs + u * sn);
        }
    }
    dense_lds_barrier();
    stream_pairs<T>(
        ahead, rows,
        [&](int n, float s0, float s1) {
            dst[2 * n] = (T)s0;
            if (2 * n + 1 < N) dst[2 * n + 1] = (T)s1;
        },
        pairs, smem, chunks, d);
}

// Values of a head (blockIdx.y) from its weighted latent, times the head's gate.  The latent is a row of o_lat, or is
// merged here from the shares of the attention: sum_k w_k share_k / sum_k w_k sum_k, w_k = 2^(maximum_k - largest).
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_values_kernel(const float* __restrict__ o_lat, int ld_o, LatentShares shares,
                                                              LatentShape sh, const T* __restrict__ uv, int ld,
                                                              const float* __restrict__ gates, float* __restrict__ attn) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ float weight[kAttendMaxSplits];
    const int h = blockIdx.y, t = threadIdx.x;
    const int N = sh.vdim, chunks = ld * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    const PlainRows<T> rows{uv + (size_t)h * N * ld, ld, N};
    const float gate = sigmoid(gates[h]);
    Pair ahead;
    if (shares.part) {
        // a thread takes four columns of every `teams`-th share; the teams' sums meet in LDS.  Requested in the order of use.
        constexpr int U = 16;
        const int n = shares.splits, quads = shares.ld >> 2, teams = max(1, kThreads / quads);
        const int l63 = min(t & 63, n - 1);
        const float maximum = shares.stats[2 * ((size_t)l63 * sh.heads + h)], total = shares.stats[2 * ((size_t)l63 * sh.heads + h) + 1];
        const float* part = shares.part + (size_t)h * shares.ld;
        const size_t step = (size_t)sh.heads * shares.ld;
        float4 v[U];
        auto request = [&](int q, int k) {
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = load4(part + min(k + u * teams, n - 1) * step + 4 * (q % quads));
        };
        if (t < quads * teams) request(t, t / quads);
        request_first(ahead, rows, pairs, chunks, d);
        {   // every wave forms the shares' weights
            const bool real = (t & 63) < n;
            const float largest = dense_wave_max(real ? maximum : -3.402823466e38f), w = real ? exp2f(maximum - largest) : 0.f;
            const float all = dense_wave_sum(w * total);
            if (t < 64) weight[t] = w / all;
        }
        dense_lds_barrier();
        float* sums = smem + ld;
        for (int q = t; q < quads * teams; q += kThreads) {
            const int team = q / quads;
            if (q != t) request(q, team);
            float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int k = team; k < n; k += U * teams) {
                if (k != team) request(q, k);
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (k + u * teams < n) s = fma4(weight[k + u * teams], v[u], s);
            }
            store4(sums + team * shares.ld + 4 * (q % quads), s);
        }
        dense_lds_barrier();
        fill_row(smem, sh.rank, ld, [&](int i) {
            float s = 0.f;
            for (int k = 0; k < teams; k++) s += sums[k * shares.ld + i];
            return s;
        });
    } else {
        request_first(ahead, rows, pairs, chunks, d);
        copy_row(smem, o_lat + (size_t)h * ld_o, sh.rank, ld);
    }
    dense_lds_barrier();
    stream_pairs<T>(ahead, rows, PlainEmit{attn + (size_t)h * N, N, gate}, pairs, smem, chunks, d);
}

__device__ __forceinline__ int expert_of(const ExpertRows& e, int slot) {
    const int id = min(max(e.ids[0], 0), e.vocab - 1);
    return min(max(e.table[(size_t)id * e.top + slot], 0), e.experts - 1);
}

// The router's choice for one token, formed by a whole workgroup from its logits (z, best: LDS): ids[0 .. top).  The first one writes it out.
__device__ __forceinline__ void choose_experts(const ExpertRows& e, float* z, int* ids, float* best, bool first) {
    for (int i = threadIdx.x; i < e.experts; i += kThreads) z[i] = e.logits[i] + e.bias[i];
    __syncthreads();
    for (int i = threadIdx.x; i < e.experts; i += kThreads) {
        const int rank = expert_rank(z, e.experts, i);
        if (rank < e.top) {
            ids[rank] = i;
            best[rank] = z[i];
        }
    }
    __syncthreads();
    if (first && threadIdx.x < 64) {
        const int k = threadIdx.x;
        const float w = k < e.top ? expf(best[k] - best[0]) : 0.f, sum = dense_wave_sum(w);
        if (k < e.top) {
            e.chosen[k] = ids[k];
            e.weights[k] = w / sum;
        }
    }
}

// act = unit(gate, up) for the token's experts (slot < top) and the dense or shared feed-forward (the last).
template <typename T, int PARTS>
__device__ __forceinline__ void gate_up(const RowStep& p, const float* __restrict__ h, const ExpertRows& e, const T* __restrict__ experts,
                                        const T* __restrict__ dense, int ld, float* __restrict__ act, int slot) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ int ids[kMaxTop];
    __shared__ float best[kMaxTop];
    float *xs = smem, *red = xs + ld, *inv = red + kThreads / 64;
    StepRow<PARTS> row(p);
    if (!h) row.load();
    if (e.logits) choose_experts(e, red, ids, best, blockIdx.x == 0 && slot == 0);  // the places of red and inv are free until the row is formed
    const T* w = slot < e.top ? experts + (size_t)(e.logits ? ids[slot] : expert_of(e, slot)) * e.pair_rows * ld : dense;
    const int ff = slot < e.top ? e.ff : e.dense_ff;
    const int chunks = ld * (int)sizeof(T) / 16;
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    auto rows = [&](int j) {  // the gate and the up row of column j
        const T* r = w + (size_t)((j >> 4) * 32 + (j & 15)) * ld;
        return RowPair{r, r + (size_t)16 * ld};
    };
    Pair ahead;
    request_first(ahead, rows, ff, chunks, d);
    if (h) {
        copy_row(xs, h, p.width, ld);
        dense_lds_barrier();
    } else {
        if (e.logits) __syncthreads();
        row.finish(xs, ld, inv, red);
    }
    float* dst = act + (size_t)slot * e.ld_act;
    stream_pairs<T>(ahead, rows, [&](int j, float gate, float up) { dst[j] = gated_unit(e.unit, gate, up); }, ff, xs, chunks, d);
}

// Behind a residual step, and on a row that is normed already.
template <typename T, int PARTS>
__global__ __launch_bounds__(kThreads) void gemv_gate_up_kernel(const float* __restrict__ x, const float* __restrict__ norm_h, const float* __restrict__ y,
                                                               const float* __restrict__ norm_y, const T* __restrict__ dense, int width, int groups,
                                                               int ld, int top, RowStep p, ExpertRows e, const T* __restrict__ experts,
                                                               float* __restrict__ act) {
    with_leading(p, x, norm_h, y, norm_y, width, groups);
    e.top = top;
    gate_up<T, PARTS>(p, nullptr, e, experts, dense, ld, act, blockIdx.y);
}
// What else is done beside a token's experts: its mixer where both look at the same row.  The launch's first rows of workgroups do it.
struct NothingBeside {
    int workgroups() const { return 0; }
    size_t lds() const { return 0; }
    __device__ __forceinline__ void operator()(int, float*) const {}
};
struct MemoryBeside {  // a matrix memory's step
    MemoryArgs a;
    float* o;
    __host__ __device__ int slices() const { return (a.sh.vdim + memory::kSlice - 1) / memory::kSlice; }
    int workgroups() const { return slices() * a.sh.heads; }
    size_t lds() const { return memory::step_floats(a.sh.dim, 4) * sizeof(float); }
    __device__ __forceinline__ void operator()(int n, float* smem) const {
        const int h = n / slices();
        if (h < a.sh.heads) memory::memory_steps<4>(a, o, n - h * slices(), h, smem);
    }
};
template <int D>
struct AttendBeside {  // attention of a few rows of a key head, key and value columns D at most each
    static constexpr int kTile = 64;
    AttendArgs<bf16> a;
    int heads;
    __host__ __device__ int groups() const { return (a.rows + 15) / 16; }
    int workgroups() const { return groups() * heads * a.splits; }
    size_t lds() const { return attend::attend_lds(2 * D, kTile, 1) + attend::attend_scores(1, kTile) * sizeof(float); }
    __device__ __forceinline__ void operator()(int n, float* smem) const {
        const int share = n / (groups() * heads), m = n - share * groups() * heads, z = m / groups();
        uint8_t* tile = reinterpret_cast<uint8_t*>(smem);
        if (share < a.splits)
            attend::attend_workgroup<2 * D, D, D, 4, 1, kTile, 1, true>(a, dim3(groups(), heads, a.splits), dim3(m - z * groups(), z, share), tile,
                                                                        reinterpret_cast<float*>(tile + attend::attend_lds(2 * D, kTile, 1)));
    }
};

// A row that is normed already.  What bounds it behind a router: the choice, then the experts' rows from memory at a rate that the trip to them
// limits; the token's mixer, a few workgroups of trips one behind the other, costs next to nothing beside it.  Dimesun, width 2048, behind 33 to
// 64 tokens: attention 5.0 us and experts 12.2 in two launches, 11.8 in one; a memory's step 6.4 and 12.2, 12.4 in one.  32 tokens 7180 -> 6430 us,
// width 1536 6200 -> 5400, 1024 4900 -> 4400, behind 1500 tokens 0.91 of the time.  Attention has one tile of keys in LDS here, where its own launch
// has two, so that three workgroups still fit a CU.  A share then waits for each of its tiles, and is still done earlier than behind a launch of its own, also where
// a chunk is long: chunks of 65536, two launches / one, us a token behind 1000, 4000 and 16000 tokens: 16 heads on 4 of 128 columns 167 / 135, 222 /
// 184, 442 / 402; 32 on 8 of 64 161 / 133, 204 / 170, 385 / 350; width 512, 8 heads of 64, one expert of 8 103 / 88, 150 / 135, 303 / 290.
template <typename T, typename Beside>
__global__ __launch_bounds__(kThreads) void gemv_gate_up_kernel(const float* __restrict__ logits, const float* __restrict__ bias, const float* __restrict__ h,
                                                               const T* __restrict__ experts, int routed, int top, int ld, int width, RowStep p,
                                                               ExpertRows e, const T* __restrict__ dense, float* __restrict__ act, int rows_beside,
                                                               Beside beside) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    if ((int)blockIdx.y < rows_beside) return beside(blockIdx.y * gridDim.x + blockIdx.x, smem);
    e.logits = logits, e.bias = bias, e.experts = routed, e.top = top, p.width = width;
    gate_up<T, 4>(p, h, e, experts, dense, ld, act, blockIdx.y - rows_beside);
}

// y[n] = mean over the token's experts of W_e[n] . act_e, plus the dense or shared feed-forward's.
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_ff_down_kernel(const float* __restrict__ act, const T* __restrict__ dense, const T* __restrict__ experts,
                                                               int dense_ff, int ld_dense, int top, int ld, int N, float* __restrict__ y, ExpertRows e) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    e.dense_ff = dense_ff, e.top = top;
    __shared__ int chosen[64];
    const int chunks = ld * (int)sizeof(T) / 16, chunks_dense = ld_dense * (int)sizeof(T) / 16, pairs = (N + 1) / 2;
    float* xs_dense = smem + e.top * ld;
    auto fill = [&]() {
        for (int k = 0; k < e.top; k++) copy_row(smem + k * ld, act + (size_t)k * e.ld_act, e.ff, ld);
        if (e.dense_ff) copy_row(xs_dense, act + (size_t)e.top * e.ld_act, e.dense_ff, ld_dense);
    };
    if (!e.top) {
        const Deal d = deal_rows<T>(chunks_dense, gridDim.x);
        const PlainRows<T> rows{dense, ld_dense, N};
        Pair ahead;
        request_first(ahead, rows, pairs, chunks_dense, d);
        fill();
        dense_lds_barrier();
        stream_pairs<T>(ahead, rows, PlainEmit{y, N, 1.f}, pairs, xs_dense, chunks_dense, d);
        return;
    }
    // a pair of rows of every expert in turn, then of the shared feed-forward; the loads run one step ahead
    const Deal d = deal_rows<T>(chunks, gridDim.x);
    if ((int)threadIdx.x < e.top) chosen[threadIdx.x] = expert_of(e, threadIdx.x);
    fill();
    __syncthreads();
    const int parts = e.top + (e.dense_ff ? 1 : 0), per_step = kAhead * d.lanes;
    const float share = 1.0f / (float)e.top;
    auto rows_of = [&](int n, int k) {
        return k < e.top ? PlainRows<T>{experts + (size_t)chosen[k] * N * ld, ld, N}(n) : PlainRows<T>{dense, ld_dense, N}(n);
    };
    Pair ahead;
    if (d.group < pairs) load_pair(ahead, rows_of(d.group, 0), d.at, d.lanes, chunks);
    for (int n = d.group; n < pairs; n += d.groups) {
        float a0 = 0.f, a1 = 0.f;
        for (int k = 0; k < parts; k++) {
            const bool expert = k < e.top;
            const int all = expert ? chunks : chunks_dense, steps = (all + per_step - 1) / per_step;
            const float* xs = expert ? smem + k * ld : xs_dense;
            float s0 = 0.f, s1 = 0.f;
            for (int step = 0; step < steps; step++) {
                const int c = d.at + step * per_step;
                const Pair now = ahead;
                if (step + 1 < steps)
                    load_pair(ahead, rows_of(n, k), c + per_step, d.lanes, all);
                else if (k + 1 < parts)
                    load_pair(ahead, rows_of(n, k + 1), d.at, d.lanes, k + 1 < e.top ? chunks : chunks_dense);
                else if (n + d.groups < pairs)
                    load_pair(ahead, rows_of(n + d.groups, 0), d.at, d.lanes, chunks);
                use_pair<T>(now, xs, c, d.lanes, all, s0, s1);
            }
            a0 = fmaf(expert ? share : 1.f, s0, a0);
            a1 = fmaf(expert ? share : 1.f, s1, a1);
        }
        a0 = dense_wave_sum(a0, d.lanes);
        a1 = dense_wave_sum(a1, d.lanes);
        if (d.at == 0) PlainEmit{y, N, 1.f}(n, a0, a1);
    }
}

// The mixer's row: load() requests what a thread will need of it, finish() puts it into xs (LDS, zero-padded; ends without
// a barrier).  inv: LDS, a float for every head, or for every head and share.
class MixerPrologue {
   public:
    __device__ __forceinline__ explicit MixerPrologue(const MixerRow& m)
        : m_(m), parts_(m.width, m.norm ? m.heads : 1, threadIdx.x), quads_(m.shares.part && m.vdim % 4 == 0), normed_(m.norm && parts_.fits()) {}
    __device__ __forceinline__ void load() {
        const int t = threadIdx.x;
        if (quads_) {
            if (t < m_.heads) {
#pragma unroll
                for (int k = 0; k < kShares; k++) stats_[k] = stat(min(k, m_.shares.splits - 1), t);
            }
            request_shares(0);
        } else if (normed_) {
#pragma unroll
            for (int k = 0; k < RowParts<kThreads>::kParts; k++) {
                const int i = parts_.place(k), at = max(i, 0);
                row_[k] = load4(m_.row + at);
                norm_[k] = load4(m_.norm + at);
                gate_[k] = load4(m_.gates + at);
                if (i < 0) row_[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }
    __device__ __forceinline__ void finish(float* xs, int padded, float* inv, float* red) {
        const int t = threadIdx.x, n = m_.shares.splits, H = m_.heads;
        if (m_.shares.part) {
            for (int h = t; h < H; h += kThreads) {  // weights w_k / sum_k w_k sum_k, w_k = 2^(maximum_k - largest)
                if (!quads_ || h != t) {
#pragma unroll
                    for (int k = 0; k < kShares; k++) stats_[k] = stat(min(k, n - 1), h);
                }
                float largest = stats_[0].x, all = 0.f, w[kShares];
#pragma unroll
                for (int k = 1; k < kShares; k++) largest = fmaxf(largest, stats_[k].x);
#pragma unroll
                for (int k = 0; k < kShares; k++) {
                    w[k] = k < n ? exp2f(stats_[k].x - largest) : 0.f;
                    all = fmaf(w[k], stats_[k].y, all);
                }
                const float share = 1.0f / all;
#pragma unroll
                for (int k = 0; k < kShares; k++) inv[h * kShares + k] = w[k] * share;
            }
            dense_lds_barrier();
            if (quads_) {
                for (int q0 = 0; 4 * q0 < m_.width; q0 += kQuads * kThreads) {
                    if (q0) request_shares(q0);
#pragma unroll
                    for (int u = 0; u < kQuads; u++) {
                        const int i = 4 * (q0 + u * kThreads + t), h = i / m_.vdim;
                        if (i >= m_.width) continue;
                        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                        for (int k = 0; k < kShares; k++) s = fma4(inv[h * kShares + k], shares_[u][k], s);
                        store4(xs + i, s);
                    }
                }
                for (int i = m_.width + t; i < padded; i += kThreads) xs[i] = 0.f;
            } else {
                fill_row(xs, m_.width, padded, [&](int i) {
                    const int h = i / m_.vdim, d = i - h * m_.vdim;
                    float s = 0.f;
                    for (int k = 0; k < n; k++) s = fmaf(inv[h * kShares + k], share_row(k, h)[d], s);
                    return s;
                });
            }
        } else if (normed_) {
            const float scale = parts_.inverse_rms(row_, m_.eps, red);
#pragma unroll
            for (int k = 0; k < RowParts<kThreads>::kParts; k++) {
                const int i = parts_.place(k);
                if (i < 0) continue;
                const float4 r = row_[k], w = norm_[k], g = gate_[k], v = scale4(r, scale, w);
                store4(xs + i, make_float4(v.x * sigmoid(g.x), v.y * sigmoid(g.y), v.z * sigmoid(g.z), v.w * sigmoid(g.w)));
            }
            for (int i = m_.width + t; i < padded; i += kThreads) xs[i] = 0.f;
        } else if (m_.norm) {
            group_inverse_rms<kThreads>([&](int i) { return m_.row[i]; }, m_.width, H, m_.eps, inv, red);
            fill_row(xs, m_.width, padded, [&](int i) { return m_.row[i] * inv[i / m_.vdim] * m_.norm[i] * sigmoid(m_.gates[i]); });
        } else {
            copy_row(xs, m_.row, m_.width, padded);
        }
    }

   private:
    static constexpr int kShares = kMixerShares, kQuads = 2;
    __device__ __forceinline__ float2 stat(int k, int h) const {
        return *reinterpret_cast<const float2*>(m_.shares.stats + 2 * ((size_t)k * m_.heads + h));
    }
    __device__ __forceinline__ const float* share_row(int k, int h) const {
        return m_.shares.part + ((size_t)k * m_.heads + h) * m_.shares.ld;
    }
    __device__ __forceinline__ void request_shares(int q0) {
#pragma unroll
        for (int u = 0; u < kQuads; u++) {
            const int i = min(4 * (q0 + u * kThreads + (int)threadIdx.x), m_.width - 4), h = i / m_.vdim;
#pragma unroll
            for (int k = 0; k < kShares; k++) shares_[u][k] = load4(share_row(min(k, m_.shares.splits - 1), h) + (i - h * m_.vdim));
        }
    }
    const MixerRow& m_;
    RowParts<kThreads> parts_;
    bool quads_, normed_;
    float2 stats_[kShares];
    float4 shares_[kQuads][kShares], row_[RowParts<kThreads>::kParts], norm_[RowParts<kThreads>::kParts], gate_[RowParts<kThreads>::kParts];
};

// y[n] = W_o[n] . mixer row + sum_k weights[k] W_e(k)[n] . act_k, as one row of W_o's and the chosen experts' chunks in turn;
// the experts' weights are in the activations.
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_mixer_down_kernel(const T* __restrict__ wo, const float* __restrict__ row_or_part,
                                                                  const float* __restrict__ stats, const T* __restrict__ experts,
                                                                  const int* __restrict__ picked, int ld_wo, int top, int ld, int N,
                                                                  const float* __restrict__ act, float* __restrict__ y, MixerRow m, ExpertRows e) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    if (stats)
        m.shares.part = row_or_part, m.shares.stats = stats;
    else
        m.row = row_or_part, m.shares.part = nullptr;
    e.chosen = const_cast<int*>(picked), e.top = top;
    __shared__ int chosen[kMaxTop];
    const int t = threadIdx.x;
    const int chunks = ld * (int)sizeof(T) / 16, chunks_wo = ld_wo * (int)sizeof(T) / 16, all = chunks_wo + e.top * chunks;
    const int pairs = (N + 1) / 2;
    float *xs = smem, *xs_experts = xs + ld_wo, *red = xs_experts + e.top * ld, *inv = red + kThreads / 64;
    const Deal d = deal_rows<T>(all, gridDim.x);
    const float per_chunk = 1.0f / (float)max(chunks, 1);
    auto load = [&](Pair& p, int n, int c) __attribute__((always_inline)) {
        const int second = 2 * n + 1 < N ? 1 : 0;
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            int at = min(c + u * d.lanes, all - 1);
            size_t row = 2 * (size_t)n;
            const T* w = wo;
            int stride = ld_wo;
            if (at >= chunks_wo) {
                at -= chunks_wo;
                const int k = (int)(((float)at + 0.5f) * per_chunk);
                at -= k * chunks;
                row += (size_t)chosen[k] * N;
                w = experts;
                stride = ld;
            }
            const uint4* src = reinterpret_cast<const uint4*>(w + row * stride) + at;
            p.a[u] = *src;
            p.b[u] = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(src) + (second ? stride : 0));
        }
    };
    Pair ahead;
    MixerPrologue row(m);
    row.load();
    const bool early = kAhead * d.lanes <= chunks_wo;  // the first step is W_o's alone
    if (early && d.group < pairs) load(ahead, d.group, d.at);
    if (t < e.top) chosen[t] = min(max(e.chosen[t], 0), e.experts - 1);
    if ((e.ff & 3) == 0) {
        for (int i = t; i < e.top * (e.ff >> 2); i += kThreads) {
            const int k = i / (e.ff >> 2), c = 4 * (i - k * (e.ff >> 2));
            const float w = e.weights[k];
            const float4 v = load4(act + (size_t)k * e.ld_act + c);
            store4(xs_experts + k * ld + c, make_float4(w * v.x, w * v.y, w * v.z, w * v.w));
        }
        for (int i = t; i < e.top * (ld - e.ff); i += kThreads) {
            const int k = i / (ld - e.ff);
            xs_experts[k * ld + e.ff + (i - k * (ld - e.ff))] = 0.f;
        }
    } else {
        for (int k = 0; k < e.top; k++) {
            const float w = e.weights[k];
            fill_row(xs_experts + k * ld, e.ff, ld, [&](int i) { return w * act[(size_t)k * e.ld_act + i]; });
        }
    }
    if (!early) {
        dense_lds_barrier();
        if (d.group < pairs) load(ahead, d.group, d.at);
    }
    row.finish(xs, ld_wo, inv, red);
    dense_lds_barrier();
    const int per_step = kAhead * d.lanes, steps = (all + per_step - 1) / per_step;
    for (int n = d.group; n < pairs; n += d.groups) {
        float s0 = 0.f, s1 = 0.f;
        for (int step = 0; step < steps; step++) {
            const int c = d.at + step * per_step;
            const Pair now = ahead;
            if (step + 1 < steps)
                load(ahead, n, c + per_step);
            else if (n + d.groups < pairs)
                load(ahead, n + d.groups, d.at);
            use_pair<T>(now, xs, c, d.lanes, all, s0, s1);
        }
        s0 = dense_wave_sum(s0, d.lanes);
        s1 = dense_wave_sum(s1, d.lanes);
        if (d.at == 0) PlainEmit{y, N, 1.f}(n, s0, s1);
    }
}

// Workgroups for N rows of `ld` elements: at most `limit`, and as many as give every lane group the same number of pairs.
template <typename T>
int workgroups(int N, int ld, int limit) {
    const int per_wg = kThreads / lanes_of(ld * (int)sizeof(T) / 16), pairs = (N + 1) / 2;
    const int rounds = (pairs + per_wg * limit - 1) / (per_wg * limit);
    return (pairs + per_wg * rounds - 1) / (per_wg * rounds);
}
constexpr int kMaxGrid = 1024;

// Units of a workgroup's lane groups, the first ones; as many as fit.
template <typename T>
int lane_groups(int ld) {
    return kThreads / lanes_of(ld * (int)sizeof(T) / 16);
}

size_t step_lds(int ld, const RowStep& p) {
    const int groups = p.norm_y.groups > p.norm_h.groups ? p.norm_y.groups : p.norm_h.groups;
    return (ld + kThreads / 64 + groups) * sizeof(float);
}

// A row that fits two float4s a thread (2048 elements in 8 groups, say) leaves registers for four workgroups on a CU, one that needs
// four for three.  32768 x 2048 (a head, 1024 workgroups): 32.7 us with three, 27.2 us = 4.9 TB/s with four; 6192 x 2048: 12.1 and
// 9.5 us.  Forcing the larger form into registers for four spills and is slower (gate and up 14.4 -> 19.6 us).
bool fits_two_parts(const RowStep& p) { return RowParts<kThreads, 2>(p.width, p.norm_h.groups, 0).fits(); }

constexpr int kReadAhead = 400;  // workgroups that read ahead beside a small product; multiples of its own

template <typename T, typename Emit>
hipError_t launch_step(const RowStep& p, const T* w, int ld, int N, const Emit& emit, const WeightsAhead& ahead, hipStream_t s) {
    const int own = workgroups<T>(N, ld, kMaxGrid);
    const dim3 grid(own, 1 + (ahead.parts ? (kReadAhead + own - 1) / own : 0)), threads(kThreads);
    if (fits_two_parts(p))
        hipLaunchKernelGGL((gemv_step_kernel<T, 2, Emit>), grid, threads, step_lds(ld, p), s, LEADING_OF(p), w, p.width, p.norm_h.groups, ld, N, p, emit, ahead);
    else
        hipLaunchKernelGGL((gemv_step_kernel<T, 4, Emit>), grid, threads, step_lds(ld, p), s, LEADING_OF(p), w, p.width, p.norm_h.groups, ld, N, p, emit, ahead);
    return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_gemv_step(const RowStep& p, const T* w, int ld, int N, float* C, hipStream_t s, const WeightsAhead& ahead) {
    return launch_step(p, w, ld, N, PlainEmit{C, N, 1.f}, ahead, s);
}
template <typename T>
hipError_t launch_gemv_step_heads(const RowStep& p, const T* w, int ld, int N, const HeadRows<T>& heads, hipStream_t s) {
    return launch_step(p, w, ld, N, HeadsEmit<T>{heads, N}, WeightsAhead{}, s);
}
template <typename T>
hipError_t launch_gemv_plain(const float* x, int K, const T* w, int ld, int N, float* C, hipStream_t s) {
    hipLaunchKernelGGL(gemv_plain_kernel<T>, dim3(workgroups<T>(N, ld, kMaxGrid)), dim3(kThreads), ld * sizeof(float), s, x, K, w, ld, N, C);
    return hipGetLastError();
}
template <typename T>
WeightsAhead::Part gemv_rows_ahead(const T* w, int ld, int N, size_t room) {
    const int rows = 2 * lane_groups<T>(ld);  // of a workgroup's round
    WeightsAhead::Part part;
    part.base = reinterpret_cast<const uint8_t*>(w);
    part.step = part.bytes = (unsigned)(rows * ld * sizeof(T));
    part.block_step = part.step;
    part.count = (int)std::min<size_t>(N / rows, room / part.bytes);
    return part;
}
template <typename T>
WeightsAhead::Part gemv_gate_up_ahead(const T* w, int ld, int ff, int slots, size_t slot_step, size_t room) {
    const int rows = std::min(lane_groups<T>(ld), 16);  // sixteen rows of gate and sixteen of up in turn
    WeightsAhead::Part part;
    part.base = reinterpret_cast<const uint8_t*>(w);
    part.step = part.bytes = (unsigned)(rows * ld * sizeof(T));
    part.block = 16 / rows, part.block_step = (size_t)32 * ld * sizeof(T), part.also = (size_t)16 * ld * sizeof(T);
    part.slots = slots, part.slot_step = slot_step * sizeof(T);
    part.count = (int)std::min<size_t>(ff / 16 * part.block, room / (2 * part.bytes * (size_t)std::max(slots, 1)));
    return part;
}
template <typename T>
hipError_t launch_gemv_query(const LatentRows& in, const LatentShape& sh, const T* w, int ld, float* q, T* cache, const DepthAverage& depth,
                             int width, float* before, hipStream_t s) {
    const int N = sh.heads * sh.query_width(), main_groups = workgroups<T>(N, ld, kMaxGrid);
    const int extra = (cache ? 1 : 0) + (width + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(gemv_query_kernel<T>, dim3(main_groups + extra), dim3(kThreads), (ld + kThreads / 64 + 1) * sizeof(float), s, in.down,
                       in.q_norm, w, sh.q_rank, ld, N, main_groups, q, cache, in, sh, depth, width, before);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_gemv_absorb(const float* q, const LatentRows& in, const LatentShape& sh, const T* uk_t, int ld, T* q_lat, hipStream_t s) {
    hipLaunchKernelGGL(gemv_absorb_kernel<T>, dim3(workgroups<T>(sh.rank, ld, 64), sh.heads), dim3(kThreads), ld * sizeof(float), s, q, uk_t,
                       ld, sh.rank, sh.dim, sh.rot, q_lat, in.pos_dev, in, sh);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_gemv_values(const float* o_lat, int ld_o, const LatentShares& shares, const LatentShape& sh, const T* uv, int ld,
                              const float* gates, float* attn, hipStream_t s) {
    // every workgroup of a head repeats the merge of its shares
    const int teams = shares.part ? (kThreads * 4 > shares.ld ? kThreads * 4 / shares.ld : 1) : 0;
    hipLaunchKernelGGL(gemv_values_kernel<T>, dim3(workgroups<T>(sh.vdim, ld, shares.part ? 4 : 64), sh.heads), dim3(kThreads),
                       (ld + teams * shares.ld) * sizeof(float), s, o_lat, ld_o, shares, sh, uv, ld, gates, attn);
    return hipGetLastError();
}
namespace {
template <typename T, typename Beside>
hipError_t launch_gate_up(const RowStep& p, const float* h, const ExpertRows& e, const T* experts, const T* dense, int ld, float* act,
                          const Beside& beside, hipStream_t s) {
    const int most = e.top && e.ff > e.dense_ff ? e.ff : e.dense_ff;
    const int slots = e.top + (e.dense_ff ? 1 : 0);
    const size_t router = e.logits ? (ld + e.experts) * sizeof(float) : 0, lds = step_lds(ld, p);
    // behind a router a workgroup first has to learn its expert: two rounds of rows for each of the 512 that fit the chip at once
    const int limit = e.logits && slots < 16 ? 512 / slots : e.logits ? 32 : kMaxGrid;
    const int columns = workgroups<T>(2 * most, ld, limit), rows_beside = (beside.workgroups() + columns - 1) / columns;
    const dim3 grid(columns, slots + rows_beside), threads(kThreads);
    const size_t bytes = std::max({lds, router, beside.lds()});
    // A row that is already normed is held in no parts: the workgroups that stream behind a router are two a CU, and the larger form
    // has the registers they want.  Dimesun, a token: rows of 4096 416 us with the smaller form and 413 with the larger, 2048 both 197,
    // 1536 167.0 and 166.3, 1024 133.5 and 133.1.
    if (h)
        hipLaunchKernelGGL((gemv_gate_up_kernel<T, Beside>), grid, threads, bytes, s, e.logits, e.bias, h, experts, e.experts, e.top, ld, p.width, p, e, dense,
                           act, rows_beside, beside);
    else if (rows_beside)
        return hipErrorInvalidValue;
    else if (fits_two_parts(p))
        hipLaunchKernelGGL((gemv_gate_up_kernel<T, 2>), grid, threads, bytes, s, LEADING_OF(p), dense, p.width, p.norm_h.groups, ld, e.top, p, e, experts, act);
    else
        hipLaunchKernelGGL((gemv_gate_up_kernel<T, 4>), grid, threads, bytes, s, LEADING_OF(p), dense, p.width, p.norm_h.groups, ld, e.top, p, e, experts, act);
    return hipGetLastError();
}
int widest_of(const AttendArgs<bf16>& a) { return std::max(a.k_own_width, a.v_width); }
}  // namespace
template <typename T>
hipError_t launch_gemv_gate_up(const RowStep& p, const float* h, const ExpertRows& e, const T* experts, const T* dense, int ld, float* act,
                               hipStream_t s) {
    return launch_gate_up(p, h, e, experts, dense, ld, act, NothingBeside{}, s);
}
bool memory_beside_fits(const MemoryArgs& a) {
    return a.M == 1 && a.sh.vdim % 4 == 0 && memory::step_floats(a.sh.dim, 4) * sizeof(float) <= 32 * 1024;
}
template <typename T>
hipError_t launch_gemv_experts_and_memory(const RowStep& p, const float* h, const ExpertRows& e, const T* experts, int ld, float* act, const MemoryArgs& a,
                                          float* o, hipStream_t s) {
    if (!h || !memory_beside_fits(a)) return hipErrorInvalidValue;
    return launch_gate_up<T>(p, h, e, experts, nullptr, ld, act, MemoryBeside{a, o}, s);
}
bool attend_beside_fits(const AttendArgs<bf16>& a) { return a.rows <= kAttendFewRows && attend_rows_fits(a.k_own_width, a.v_width) && widest_of(a) <= 128; }
hipError_t launch_gemv_experts_and_attend(const RowStep& p, const float* h, const ExpertRows& e, const bf16* experts, int ld, float* act,
                                          const AttendArgs<bf16>& a, int kv_heads, hipStream_t s) {
    if (!h || !attend_beside_fits(a)) return hipErrorInvalidValue;
    const bf16* none = nullptr;
    if (widest_of(a) <= 64) return launch_gate_up(p, h, e, experts, none, ld, act, AttendBeside<64>{a, kv_heads}, s);
    return launch_gate_up(p, h, e, experts, none, ld, act, AttendBeside<128>{a, kv_heads}, s);
}
template <typename T>
hipError_t launch_gemv_ff_down(const ExpertRows& e, const float* act, const T* experts, int ld, const T* dense, int ld_dense, int N,
                               float* y, hipStream_t s) {
    const size_t lds = ((size_t)e.top * ld + (e.dense_ff ? ld_dense : 0)) * sizeof(float);
    hipLaunchKernelGGL(gemv_ff_down_kernel<T>, dim3(workgroups<T>(N, e.dense_ff ? ld_dense : ld, kMaxGrid)), dim3(kThreads), lds, s, act,
                       dense, experts, e.dense_ff, ld_dense, e.top, ld, N, y, e);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_gemv_mixer_down(const MixerRow& m, const T* wo, int ld_wo, const ExpertRows& e, const float* act, const T* experts,
                                  int ld, int N, float* y, hipStream_t s) {
    const int row = ld_wo + e.top * ld, inv = m.shares.part ? m.heads * kMixerShares : m.heads;
    const size_t lds = (row + kThreads / 64 + inv) * sizeof(float);
    hipLaunchKernelGGL(gemv_mixer_down_kernel<T>, dim3(workgroups<T>(N, row, kMaxGrid)), dim3(kThreads), lds, s, wo,
                       m.shares.part ? m.shares.part : m.row, m.shares.part ? m.shares.stats : nullptr, experts, e.chosen, ld_wo, e.top, ld, N, act, y, m, e);
    return hipGetLastError();
}

#define INSTANTIATE(T)                                                                                                            \
    template hipError_t launch_gemv_step<T>(const RowStep&, const T*, int, int, float*, hipStream_t, const WeightsAhead&);         \
    template hipError_t launch_gemv_plain<T>(const float*, int, const T*, int, int, float*, hipStream_t);                          \
    template WeightsAhead::Part gemv_rows_ahead<T>(const T*, int, int, size_t);                                                    \
    template WeightsAhead::Part gemv_gate_up_ahead<T>(const T*, int, int, int, size_t, size_t);                                    \
    template hipError_t launch_gemv_query<T>(const LatentRows&, const LatentShape&, const T*, int, float*, T*, const DepthAverage&, \
                                             int, float*, hipStream_t);                                                           \
    template hipError_t launch_gemv_absorb<T>(const float*, const LatentRows&, const LatentShape&, const T*, int, T*, hipStream_t); \
    template hipError_t launch_gemv_values<T>(const float*, int, const LatentShares&, const LatentShape&, const T*, int,           \
                                              const float*, float*, hipStream_t);                                                                       \
    template hipError_t launch_gemv_gate_up<T>(const RowStep&, const float*, const ExpertRows&, const T*, const T*, int, float*,    \
                                               hipStream_t);                                                                       \
    template hipError_t launch_gemv_experts_and_memory<T>(const RowStep&, const float*, const ExpertRows&, const T*, int, float*,             \
                                                          const MemoryArgs&, float*, hipStream_t);                                 \
    template hipError_t launch_gemv_step_heads<T>(const RowStep&, const T*, int, int, const HeadRows<T>&, hipStream_t);             \
    template hipError_t launch_gemv_mixer_down<T>(const MixerRow&, const T*, int, const ExpertRows&, const float*, const T*, int,   \
                                                  int, float*, hipStream_t);                                                       \
    template hipError_t launch_gemv_ff_down<T>(const ExpertRows&, const float*, const T*, int, const T*, int, int, float*,         \
                                               hipStream_t);
INSTANTIATE(bf16)
INSTANTIATE(float)

}  // namespace a81w41
