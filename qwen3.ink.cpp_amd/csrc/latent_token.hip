// Attention of one token in latent space over a short context, and the product with W_uv behind it, in one launch: 32 rows of a head's
// W_uv a workgroup, each of which repeats the head's attention for itself.  Further workgroups read weights ahead (weights_ahead.h).
//
// What bounds it: a chain of dependent steps (query, scores, weights, merge, product) and what one CU draws at a time.  As two
// launches (attention with two workgroups for all heads, then the product that merges their shares) the chain has another launch, two
// more trips to memory, and one CU copies 64 keys of 1152 bytes.  Here the keys, in registers of 16 waves, and the rows of
// W_uv are requested at the start, beside the query; a key's row is read once, a lane holding eight columns of it for the score and
// for the weighted sum.  Queries and weights are rounded to bfloat16, as the matrix ops' operands are.
//
// A Takosun token of width 2048 (four layers, 16 heads, latents of 512 + 64) behind 64 tokens: 290.9 us with the two launches, 255.4 us
// so; width 1024 (8 heads) 210.0 and 181.2 us.
#include "dense_common.h"

namespace a81w41 {
namespace {

constexpr int kWaves = 16, kThreads = 64 * kWaves, kTile = 8;  // keys of a wave at a time
constexpr int kRank = 512, kRot = 64;                          // at most: a lane holds eight columns
constexpr int kRows = 2 * kWaves;                              // of W_uv
constexpr float kLog2e = 1.4426950408889634f, kLowest = -1e30f;

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

__device__ __forceinline__ float dot2(unsigned a, unsigned b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
__device__ __forceinline__ float dot8(const lds16& a, const lds16& b) { return dot2(a[3], b[3], dot2(a[2], b[2], dot2(a[1], b[1], dot2(a[0], b[0], 0.f)))); }
template <int CONTROL>
__device__ __forceinline__ float moved(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CONTROL, 0xf, 0xf, true));
}
// Lanes 0 .. 31: a of both halves, lanes 32 .. 63: b of both; the same for even and odd rows of sixteen lanes, and for their halves.
__device__ __forceinline__ float fold32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold8(float a, float b) {
    const bool high = threadIdx.x & 8;
    return (high ? b : a) + moved<0x128>(high ? a : b);
}
__device__ __forceinline__ float sum8(float v) {
    v += moved<0xB1>(v);
    v += moved<0x4E>(v);
    return v + moved<0x141>(v);
}

__global__ __launch_bounds__(kThreads, 4) void latent_token_kernel(const bf16* __restrict__ q_lat, const bf16* __restrict__ cache, int ld,
                                                                  const int* __restrict__ pos_dev, int max_seq, int rank, int rot, int vdim,
                                                                  float scale, const bf16* __restrict__ uv, int ld_uv,
                                                                  const float* __restrict__ gates, float* __restrict__ attn, const WeightsAhead ahead) {
    if ((int)blockIdx.y * kRows >= vdim) {
        const int linear = blockIdx.y * gridDim.x + blockIdx.x;
        return read_ahead<kThreads>(ahead, WeightsAhead::kWorkgroups, linear - (vdim + kRows - 1) / kRows * gridDim.x, linear);
    }
    __shared__ __attribute__((aligned(16))) float shares[kWaves * kRank];
    __shared__ __attribute__((aligned(16))) float merged[kRank];
    __shared__ float2 stats[kWaves];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = blockIdx.x;
    // chunks of eight columns; a lane beyond the row takes its last one, against zeros of the query
    const int at = 8 * min(lane, (rank >> 3) - 1), at_rot = rank + 8 * min(lane & 7, max((rot + 7) / 8 - 1, 0));
    auto load = [&](const bf16* p) { return *reinterpret_cast<const lds16*>(p); };
    const int pos = min(max(pos_dev[0], 0), max_seq - 1);
    lds16 q = load(q_lat + (size_t)h * ld + at), q_rot = load(q_lat + (size_t)h * ld + at_rot);
    lds16 latent[kTile], turned;
    auto request = [&](int tile, int last) {
#pragma unroll
        for (int j = 0; j < kTile; j++) latent[j] = load(cache + (size_t)min(tile * kTile + j, last) * ld + at);
        turned = load(cache + (size_t)min(tile * kTile + (lane >> 3), last) * ld + at_rot);
    };
    request(wave, max_seq - 1);  // which of them the token sees is not known yet
    const int row = blockIdx.y * kRows + 2 * wave;
    const bf16* w = uv + ((size_t)h * vdim + min(row, vdim - 1)) * ld_uv + at;
    const lds16 w0 = load(w), w1 = load(w + (row + 1 < vdim ? ld_uv : 0));
    const float gate = gates[h];
    const lds16 none = {0, 0, 0, 0};
    if (8 * lane >= rank) q = none;
    if (8 * (lane & 7) >= rot) q_rot = none;
    float top = kLowest, sum = 0.f, acc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = 0.f;
    scale *= kLog2e;
    for (int tile = wave; tile * kTile <= pos; tile += kWaves) {
        if (tile * kTile + kTile - 1 > pos) {  // what lies behind the token is not a number to count on
#pragma unroll
            for (int j = 1; j < kTile; j++)
                if (tile * kTile + j > pos) latent[j] = none;
        }
        float s[kTile];
#pragma unroll
        for (int j = 0; j < kTile; j++) s[j] = dot8(q, latent[j]);
#pragma unroll
        for (int j = 0; j < 4; j++) s[j] = fold32(s[j], s[j + 4]);
        s[0] = fold16(s[0], s[2]), s[1] = fold16(s[1], s[3]);
        const bool seen = tile * kTile + (lane >> 3) <= pos;  // of the lane's key, lane / 8
        const float z = sum8(fold8(s[0], s[1]) + dot8(q_rot, turned)) * scale, score = seen ? z : kLowest;
        float most = fmaxf(top, score);
        most = fmaxf(most, moved<0x128>(most));
        most = fmaxf(most, __shfl_xor(most, 16, 64));
        most = fmaxf(most, __shfl_xor(most, 32, 64));
        const float keep = exp2f(top - most), p = score > kLowest ? exp2f(score - most) : 0.f;
        top = most;
        sum = fmaf(sum, keep, p);
        const int bits = __builtin_bit_cast(unsigned short, (bf16)p);
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] *= keep;
#pragma unroll
        for (int j = 0; j < kTile; j += 2) {
            const unsigned both = __builtin_amdgcn_readlane(bits, 8 * j) | __builtin_amdgcn_readlane(bits, 8 * j + 8) << 16;
            const lds16 a = latent[j], b = latent[j + 1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                acc[2 * i] = dot2(both, __builtin_amdgcn_perm(b[i], a[i], 0x05040100), acc[2 * i]);
                acc[2 * i + 1] = dot2(both, __builtin_amdgcn_perm(b[i], a[i], 0x07060302), acc[2 * i + 1]);
            }
        }
        if ((tile + kWaves) * kTile <= pos) request(tile + kWaves, pos);
    }
    sum += moved<0x128>(sum);
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lane == 0) stats[wave] = make_float2(top, sum);
    store4(shares + wave * kRank + 8 * lane, make_float4(acc[0], acc[1], acc[2], acc[3]));
    store4(shares + wave * kRank + 8 * lane + 4, make_float4(acc[4], acc[5], acc[6], acc[7]));
    dense_lds_barrier();
    if (t < kRank) {
        float largest = stats[0].x, all = 0.f, o = 0.f;
#pragma unroll
        for (int k = 1; k < kWaves; k++) largest = fmaxf(largest, stats[k].x);
#pragma unroll
        for (int k = 0; k < kWaves; k++) {
            const float part = exp2f(stats[k].x - largest);
            all = fmaf(part, stats[k].y, all);
            o = fmaf(part, shares[k * kRank + t], o);
        }
        merged[t] = t < rank ? o / all : 0.f;
    }
    dense_lds_barrier();
    const float4 m0 = load4(merged + 8 * lane), m1 = load4(merged + 8 * lane + 4);
    auto product = [&](const lds16& u) {
        float y = __uint_as_float(u[0] << 16) * m0.x;
        y = fmaf(__uint_as_float(u[0] & 0xffff0000u), m0.y, y);
        y = fmaf(__uint_as_float(u[1] << 16), m0.z, y);
        y = fmaf(__uint_as_float(u[1] & 0xffff0000u), m0.w, y);
        y = fmaf(__uint_as_float(u[2] << 16), m1.x, y);
        y = fmaf(__uint_as_float(u[2] & 0xffff0000u), m1.y, y);
        y = fmaf(__uint_as_float(u[3] << 16), m1.z, y);
        return fmaf(__uint_as_float(u[3] & 0xffff0000u), m1.w, y);
    };
    float y = fold32(product(w0), product(w1));
    y = sum8(y);
    y += moved<0x128>(y);
    y += __shfl_xor(y, 16, 64);
    const int mine = row + (lane >> 5);
    if ((lane & 31) == 0 && mine < vdim) attn[(size_t)h * vdim + mine] = y * sigmoid(gate);
}

}  // namespace

bool latent_token_fits(const LatentShape& sh) { return sh.rank % 8 == 0 && sh.rank <= kRank && sh.rot > 0 && sh.rot <= kRot; }

hipError_t launch_latent_token(const bf16* q_lat, const LatentRows& in, const LatentShape& sh, const bf16* cache, const bf16* uv, int ld_uv,
                               const float* gates, float* attn, const WeightsAhead& ahead, hipStream_t s) {
    const int more = (ahead.workgroups() + sh.heads - 1) / sh.heads;
    hipLaunchKernelGGL(latent_token_kernel, dim3(sh.heads, (sh.vdim + kRows - 1) / kRows + more), dim3(kThreads), 0, s, q_lat, cache, sh.ld_cache,
                       in.pos_dev, in.max_seq, sh.rank, sh.rot, sh.vdim, sh.scale, uv, ld_uv, gates, attn, ahead);
    return hipGetLastError();
}

}  // namespace a81w41
