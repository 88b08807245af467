// Device helpers of the dense-weight kernels.
#pragma once
#include "dense.h"

namespace a81w41 {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((address_space(3))) void* dense_lds_ptr;
// What a kernel reads out of LDS while direct copies into other parts of it are under way is read as vectors of this type: ahead
// of a read through HIP's uint4 the compiler waits for every copy (s_waitcnt vmcnt(0)).
typedef __attribute__((ext_vector_type(4))) unsigned lds16;

__device__ __forceinline__ float dense_wave_sum(float v, int width = 64) {
    for (int off = width >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float dense_wave_max(float v, int width = 64) {
    for (int off = width >> 1; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float gated_unit(const GatedUnit& p, float gate, float up) {
    const float g = fminf(gate, p.limit), u = fminf(fmaxf(up, -p.limit), p.limit);
    return g / (1.0f + expf(-p.slope * g)) * (u + p.shift);
}

// How many of z[0 .. n) come before z[e]: the larger ones, and the equal ones with lower numbers.
__device__ __forceinline__ int expert_rank(const float* z, int n, int e) {
    const float own = z[e];
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < n; j++) rank += (z[j] > own || (z[j] == own && j < e)) ? 1 : 0;
    return rank;
}

// Where one column of a HeadRows or LatentQueries product goes, from row m on: element d of the column at dst + d step (bytes), the
// first `rows` rows, float instead of the element type for what is not a head's.  Columns with a pair turn with their neighbour.
struct ColumnPlace {
    uint8_t* dst;
    int step, rows = 0x7fffffff, pair = -1;
    bool as_float = false, second = false;
};
template <typename T>
__device__ __forceinline__ ColumnPlace column_place(const HeadRows<T>& p, int col, int m, int pos) {
    const int nq = p.heads * p.dim, nk = p.kv_heads * p.dim, nv = p.kv_heads * p.vdim;
    ColumnPlace to;
    int at;
    if (col >= nq + nk + nv) {
        to.as_float = true, to.step = p.ld_rest * (int)sizeof(float);
        to.dst = reinterpret_cast<uint8_t*>(p.rest + (size_t)m * p.ld_rest + (col - nq - nk - nv));
        return to;
    }
    const bool cached = col >= nq;
    if (col >= nq + nk) {
        const int c = col - nq - nk, h = c / p.vdim;
        at = h * (p.vdim + p.dim) + (c - h * p.vdim);
    } else {
        const int c = cached ? col - nq : col, h = c / p.dim, d = c - h * p.dim;
        at = cached ? h * (p.vdim + p.dim) + p.vdim + d : c;
        if ((d >> 1) < p.rot_pairs) to.pair = d >> 1, to.second = d & 1;
    }
    const int width = cached ? p.ld_cache : nq;
    to.step = width * (int)sizeof(T);
    to.dst = reinterpret_cast<uint8_t*>((cached ? p.cache : p.q) + (size_t)(cached ? pos + m : m) * width + at);
    if (cached) to.rows = p.max_seq - pos - m;
    return to;
}
template <typename T>
__device__ __forceinline__ ColumnPlace column_place(const LatentQueries<T>& p, int col, int m, int) {
    const int at = p.dim + (p.dim & 1), width = at + p.rot, h = col / width, c = col - h * width;
    ColumnPlace to;
    const bool turned = c >= at;
    if (turned) to.pair = (c - at) >> 1, to.second = (c - at) & 1;
    const int ld = turned ? p.ld_rot : p.ld_nope;
    to.step = p.heads * ld * (int)sizeof(T);
    to.dst = reinterpret_cast<uint8_t*>((turned ? p.rotated : p.nope) + ((size_t)m * p.heads + h) * ld + (turned ? c - at : c));
    if (!turned && c >= p.dim) to.rows = 0;
    return to;
}
// whether `together` columns (2 or 4) from a multiple of them on are stored next to each other and aligned to all of them
template <typename T>
__device__ __forceinline__ bool columns_go_together(const HeadRows<T>& p, int n, int together) {
    const uintptr_t elements = reinterpret_cast<uintptr_t>(p.q) | reinterpret_cast<uintptr_t>(p.cache);
    const bool rest = n <= p.heads * p.dim + p.kv_heads * (p.dim + p.vdim) ||
                      ((p.ld_rest & (together - 1)) == 0 && (reinterpret_cast<uintptr_t>(p.rest) & (together * sizeof(float) - 1)) == 0);
    return rest && ((n | p.dim | p.vdim | p.ld_cache) & (together - 1)) == 0 && (elements & (together * sizeof(T) - 1)) == 0;
}
template <typename T>
__device__ __forceinline__ bool columns_go_together(const LatentQueries<T>& p, int n, int together) {
    const uintptr_t elements = reinterpret_cast<uintptr_t>(p.nope) | reinterpret_cast<uintptr_t>(p.rotated);
    return ((n | p.dim | p.rot | p.ld_nope | p.ld_rot) & (together - 1)) == 0 && (elements & (together * sizeof(T) - 1)) == 0;
}
template <typename T>
__device__ __forceinline__ int turned_pairs(const HeadRows<T>& p) {
    return p.rot_pairs;
}
template <typename T>
__device__ __forceinline__ int turned_pairs(const LatentQueries<T>& p) {
    return p.rot >> 1;
}

// One direct copy global -> LDS of 16 bytes per lane: lane l's bytes land at lds_base + 16 l (lds_base uniform).
__device__ __forceinline__ void copy16_to_lds(const void* global_src, void* lds_base) {
    __builtin_amdgcn_global_load_lds(global_src, (dense_lds_ptr)lds_base, 16, 0, 0);
}

// The same from a uniform base: lane l's source is `at` + `step` bytes (32 bits, step uniform) behind it, with no address of 64 bits
// to form.
typedef __amdgpu_buffer_rsrc_t CopySource;
__device__ __forceinline__ CopySource copy_source(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xffffffff, 0x00027000);
}
__device__ __forceinline__ void copy16_to_lds(CopySource from, void* lds_base, unsigned at, int step) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (dense_lds_ptr)lds_base, 16, at, step, 0, 0);
}

// A barrier that orders LDS only: requested global loads stay in flight.
__device__ __forceinline__ void dense_lds_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt = 0; vector-memory and export counters left alone
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// 1 / sqrt(mean of squares + eps) of `groups` equal consecutive parts of a row, into inv[0..groups) (LDS).
// x(i) is element i.  red: THREADS / 64 floats of LDS.  Ends with a barrier.
template <int THREADS, typename F>
__device__ __forceinline__ void group_inverse_rms(F x, int width, int groups, float eps, float* inv, float* red) {
    const int t = threadIdx.x, size = width / groups;
    int per = 1;  // groups worked on at a time
    while (per < groups && per < THREADS) per <<= 1;
    const int tpg = THREADS / per;  // threads per group, a power of two
    for (int g0 = 0; g0 < groups; g0 += per) {
        const int g = g0 + t / tpg, at = t % tpg;
        float sum = 0.f;
        if (g < groups)
            for (int i = at; i < size; i += tpg) {
                const float v = x(g * size + i);
                sum = fmaf(v, v, sum);
            }
        sum = dense_wave_sum(sum, tpg < 64 ? tpg : 64);
        if (tpg > 64) {
            if ((t & 63) == 0) red[t >> 6] = sum;
            __syncthreads();
            sum = 0.f;
            const int w0 = (t / tpg) * (tpg >> 6);
            for (int w = 0; w < (tpg >> 6); w++) sum += red[w0 + w];
        }
        if (g < groups && at == 0) inv[g] = 1.0f / sqrtf(sum / (float)size + eps);
        __syncthreads();
    }
}

// A row whose norm groups are whole float4s, dealt to a workgroup so that a group's threads are neighbours and a thread
// holds at most PARTS float4s, all of one group: the row stays in registers between its norms.
template <int THREADS, int PARTS = 4>
class RowParts {
   public:
    static constexpr int kParts = PARTS;
    __host__ __device__ __forceinline__ RowParts(int width, int groups, int thread) : groups_(groups), size_(width / groups) {
        int per = 1;
        while (per < groups && per < THREADS) per <<= 1;
        log_tpg_ = 31 - __builtin_clz((unsigned)(THREADS / per));
        group_ = thread >> log_tpg_;
        at_ = thread & ((1 << log_tpg_) - 1);
    }
    __host__ __device__ __forceinline__ bool fits() const {
        return groups_ <= THREADS && (size_ & 3) == 0 && (size_ >> 2) <= (kParts << log_tpg_);
    }
    // first element of this thread's k-th float4, -1 if it has none
    __device__ __forceinline__ int place(int k) const {
        const int c = at_ + (k << log_tpg_);
        return group_ < groups_ && 4 * c < size_ ? group_ * size_ + 4 * c : -1;
    }
    // of this thread's group; v: the thread's parts (absent ones zero), red: THREADS / 64 floats of LDS
    __device__ __forceinline__ float inverse_rms(const float4* v, float eps, float* red) const {
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < kParts; k++) {
            sum = fmaf(v[k].x, v[k].x, sum), sum = fmaf(v[k].y, v[k].y, sum);
            sum = fmaf(v[k].z, v[k].z, sum), sum = fmaf(v[k].w, v[k].w, sum);
        }
        sum = dense_wave_sum(sum, log_tpg_ < 6 ? 1 << log_tpg_ : 64);
        if (log_tpg_ > 6) {
            dense_lds_barrier();  // nobody still reads red
            if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
            dense_lds_barrier();
            sum = 0.f;
            const int waves = 1 << (log_tpg_ - 6);
            for (int w = 0; w < waves; w++) sum += red[group_ * waves + w];
        }
        return 1.0f / sqrtf(sum / (float)size_ + eps);
    }

   private:
    int groups_, size_, log_tpg_, group_, at_;
};
__device__ __forceinline__ float4 load4(const float* a) { return *reinterpret_cast<const float4*>(a); }
__device__ __forceinline__ void store4(float* a, float4 v) { *reinterpret_cast<float4*>(a) = v; }
__device__ __forceinline__ float4 fma4(float a, float4 b, float4 c) {
    return make_float4(fmaf(a, b.x, c.x), fmaf(a, b.y, c.y), fmaf(a, b.z, c.z), fmaf(a, b.w, c.w));
}
__device__ __forceinline__ float4 scale4(float4 v, float s, float4 w) {
    return make_float4(v.x * s * w.x, v.y * s * w.y, v.z * s * w.z, v.w * s * w.w);
}
__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

}  // namespace a81w41
