// Matrix memory with exponential gates: a recurrence over tokens whose state per head is a matrix S, a vector n and a
// scale m (dense.h has the equations).  Everything here is fp32, gate sums fp64.
//
// A prompt goes in chunks of 64 tokens.  With f_t, i_t the gates' logarithms, b_t = f_1 + .. + f_t inside the chunk,
// a_s = i_s - b_s and m_0, S_0, n_0 the state before the chunk, the recurrence unrolls to
//   M_t = max(m_0, max_{s <= t} a_s),   m_t = b_t + M_t
//   S_t = e^(m_0 - M_t) S_0 + sum_{s <= t} e^(a_s - M_t) k_s v_s^T          (n_t likewise)
//   S_t^T q_t = e^(m_0 - M_t) S_0^T q_t + sum_{s <= t} e^(a_s - M_t) (q_t . k_s) v_s
// so that a chunk needs S only at its start.  Three launches: every chunk's own sum over s for t = its last token (outer
// products, all chunks at once); the chain over chunks, element by element; the outputs of all chunks.
#include "memory_steps.h"

namespace a81w41 {
namespace {

using namespace memory;
constexpr int C = kMemoryChunk;
static_assert(C == 64, "the lanes of a wave hold a chunk's gates");

__device__ __forceinline__ double shfl_up(double v, int by) {
    const long long u = __double_as_longlong(v);
    const int lo = __shfl_up((int)u, by, 64), hi = __shfl_up((int)(u >> 32), by, 64);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// One wave, lane t = token t of the chunk: b_t, a_t and max_{s <= t} a_s; tokens from `count` on change nothing.
struct ChunkGates {
    double b, a, most;
};
__device__ __forceinline__ ChunkGates chunk_gates(const MemoryArgs& p, int m0, int count, int h) {
    const int t = threadIdx.x & 63;
    const Gates g = gates_of(p, m0 + min(t, count - 1), h);
    ChunkGates c;
    c.b = t < count ? (double)g.log_keep : 0.0;
    for (int off = 1; off < 64; off <<= 1) {
        const double other = shfl_up(c.b, off);
        if (t >= off) c.b += other;
    }
    c.a = t < count ? (double)g.log_in - c.b : -1e300;
    c.most = c.a;
    for (int off = 1; off < 64; off <<= 1) {
        const double other = shfl_up(c.most, off);
        if (t >= off) c.most = fmax(c.most, other);
    }
    return c;
}

// Token by token (memory_steps.h).
template <int W>
__global__ __launch_bounds__(kThreads) void memory_steps_kernel(MemoryArgs a, float* __restrict__ o) {
    extern __shared__ float smem[];
    memory_steps<W>(a, o, blockIdx.x, blockIdx.y, smem);
}

// One workgroup per token.
template <typename T>
__global__ __launch_bounds__(kThreads) void memory_norm_kernel(MemoryArgs a, const float* __restrict__ o, T* __restrict__ out, int ld_out) {
    extern __shared__ float smem[];
    const int width = a.sh.heads * a.sh.vdim;
    float *inv = smem, *red = inv + a.sh.heads;
    const float *row = o + (size_t)blockIdx.x * width, *gate = a.in + (size_t)blockIdx.x * a.ld_in + a.sh.at_g;
    if (steps_held_back(a)) {
        float* to = state_nm(a, max(a.pos_dev[0], 0) + a.M);
        for (int i = blockIdx.x * kThreads + threadIdx.x; i < a.sh.heads * (a.sh.dim + 1); i += gridDim.x * kThreads) to[i] = a.held[i];
    }
    group_inverse_rms<kThreads>([&](int i) { return row[i]; }, width, a.sh.heads, a.sh.eps, inv, red);
    T* dst = out + (size_t)blockIdx.x * ld_out;
    for (int i = threadIdx.x; i < width; i += kThreads) dst[i] = (T)(row[i] * inv[i / a.sh.vdim] * a.norm[i] * sigmoid(gate[i]));
}

__device__ __forceinline__ f32x16 mfma32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// W floats (4: aligned to 16 bytes), zeros where there are none
template <int W>
__device__ __forceinline__ void read_part(float* part, const float* src, bool real) {
    if constexpr (W == 4) {
        const float4 v = real ? load4(src) : make_float4(0.f, 0.f, 0.f, 0.f);
        part[0] = v.x, part[1] = v.y, part[2] = v.z, part[3] = v.w;
    } else {
        part[0] = real ? src[0] : 0.f;
    }
}
template <int W>
__device__ __forceinline__ void write_part(float* dst, const float* part) {
    if constexpr (W == 4)
        store4(dst, make_float4(part[0], part[1], part[2], part[3]));
    else
        dst[0] = part[0];
}

// A chunk's own sums for its last token: sum_s w_s k_s v_s^T and sum_s w_s k_s with w_s = e^(a_s - max a).  A workgroup has
// a 128 x 128 tile of a head's S; its waves take the 32 x 32 pieces in turn.  K and V sit in LDS as [token][column], column
// c of token s at place c ^ 32 (s & 1): the two tokens a matrix operand takes at a time lie in different banks.
constexpr int kOuter = 128;
template <int W>
__global__ __launch_bounds__(kThreads) void memory_outer_kernel(MemoryArgs a) {
    constexpr int kPer = kOuter / W, kLoads = C * kPer / kThreads, kBatch = W == 4 ? kLoads : 8;
    __shared__ __attribute__((aligned(16))) float ks[C * kOuter], vs[C * kOuter], weight[C];
    const MemoryShape sh = a.sh;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l31 = lane & 31, half = lane >> 5;
    const int chunk = blockIdx.x, h = blockIdx.y, m0 = chunk * C, count = min(C, a.M - m0);
    const int v_tiles = (sh.vdim + kOuter - 1) / kOuter, d0 = blockIdx.z / v_tiles * kOuter, v0 = blockIdx.z % v_tiles * kOuter;
    const int nd = min(kOuter, sh.dim - d0), nv = min(kOuter, sh.vdim - v0);
    const int cols_k = (nd + 31) / 32 * 32, cols_v = (nv + 31) / 32 * 32;
    // the rows are requested before the gates are formed
    float k_part[kBatch][W], v_part[kBatch][W];
    auto request = [&](int first) {
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int i = t + (first + u) * kThreads, s = i / kPer, c = i % kPer * W;
            const float* row = a.in + (size_t)(m0 + min(s, count - 1)) * a.ld_in;
            read_part<W>(k_part[u], row + sh.at_k + h * sh.dim + d0 + c, s < count && c < nd);
            read_part<W>(v_part[u], row + sh.at_v + h * sh.vdim + v0 + c, s < count && c < nv);
        }
    };
    request(0);
    if (wave == 0) {
        const ChunkGates g = chunk_gates(a, m0, count, h);
        const double most = __shfl(g.most, 63, 64);
        weight[lane] = lane < count ? expf((float)(g.a - most)) : 0.f;
        if (lane == 63 && blockIdx.z == 0) {
            float* st = a.chunk_stats + 2 * ((size_t)chunk * sh.heads + h);
            st[0] = (float)most;
            st[1] = (float)g.b;
        }
        if (blockIdx.z == 0) {
            double* to = a.chunk_gates + ((size_t)chunk * sh.heads + h) * 3 * C + lane;
            to[0] = g.b, to[C] = g.a, to[2 * C] = g.most;
        }
    }
    dense_lds_barrier();
    for (int first = 0; first < kLoads; first += kBatch) {
        if (first) request(first);
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int i = t + (first + u) * kThreads, s = i / kPer, c = i % kPer * W, at = s * kOuter + (c ^ ((s & 1) << 5));
            const float w = weight[s];
#pragma unroll
            for (int e = 0; e < W; e++) k_part[u][e] *= w;
            write_part<W>(ks + at, k_part[u]);
            write_part<W>(vs + at, v_part[u]);
        }
    }
    __syncthreads();
    float* out = a.chunk_states + ((size_t)chunk * sh.heads + h) * sh.chunk_size();
    const int v_pieces = cols_v / 32, pieces = cols_k / 32 * v_pieces;
    for (int piece = wave; piece < pieces; piece += kThreads / 64) {
        const int pd = piece / v_pieces * 32, pv = piece % v_pieces * 32;
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = 0.f;
#pragma unroll 8
        for (int s = 0; s < C; s += 2) {
            const int row = (s + half) * kOuter, turn = half << 5;
            acc = mfma32(ks[row + ((pd + l31) ^ turn)], vs[row + ((pv + l31) ^ turn)], acc);
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int d = pd + 8 * (i >> 2) + 4 * half + (i & 3), v = pv + l31;
            if (d < nd && v < nv) out[(size_t)(d0 + d) * sh.vdim + v0 + v] = acc[i];
        }
    }
    if (v0 == 0 && t < nd) {
        float s = 0.f;
#pragma unroll 8
        for (int k = 0; k < C; k++) s += ks[k * kOuter + (t ^ ((k & 1) << 5))];
        out[(size_t)sh.dim * sh.vdim + d0 + t] = s;
    }
}

// The chain over chunks for W neighbouring elements of a head's S and n: chunk_states becomes the state before each chunk,
// the state itself the one after the last; chunk_m the scales.
//
// What bounds it: the trips of one element's chain.  kAhead chunks of it are under way, and what a chunk's sums are scaled by is formed
// ahead, a chunk a lane: read and formed by every thread inside the chain, 8 heads of 128 x 256 over 32 chunks took 18.7 us, now 16.4; 141
// chunks of 32 x 64 and 2 heads 49.9, now 25.8.
template <int W>
__global__ __launch_bounds__(kThreads) void memory_chain_kernel(MemoryArgs a, int chunks) {
    constexpr int kAhead = 8, kScales = 64;
    __shared__ float keep[kScales], add[kScales];
    const MemoryShape sh = a.sh;
    const int h = blockIdx.y, pos = max(a.pos_dev[0], 0), lane = threadIdx.x & 63;
    const size_t e = ((size_t)blockIdx.x * kThreads + threadIdx.x) * W, s_size = (size_t)sh.dim * sh.vdim, size = sh.chunk_size();
    const size_t nm = (size_t)h * (sh.dim + 1);
    const bool mine = e < size, in_s = e < s_size;  // W > 1: the parts are whole multiples of W
    const float* from = in_s ? a.state + h * s_size + e : state_nm(a, pos) + nm + (e - s_size);
    float* to = in_s ? a.state + h * s_size + e : state_nm(a, pos + a.M) + nm + (e - s_size);
    alignas(16) float cur[W], next[kAhead][W];
    const size_t step = (size_t)sh.heads * size;
    float* at = a.chunk_states + h * size + e;
    auto load = [&](float* dst, int c) {
        const float* src = at + (size_t)min(c, chunks - 1) * step;
        if constexpr (W == 4)
            *reinterpret_cast<float4*>(dst) = load4(src);
        else
            dst[0] = src[0];
    };
    if (mine) {
#pragma unroll
        for (int w = 0; w < W; w++) cur[w] = from[w];
#pragma unroll
        for (int u = 0; u < kAhead; u++) load(next[u], u);
    }
    float m = state_nm(a, pos)[nm + sh.dim];
    for (int first = 0; first < chunks; first += kScales) {
        const int n = min(kScales, chunks - first);
        if (first) dense_lds_barrier();  // nobody still reads the scales before
        if (threadIdx.x < 64) {
            const float* st = a.chunk_stats + 2 * ((size_t)(first + min(lane, n - 1)) * sh.heads + h);
            const float most_own = st[0], sum_own = st[1];
            float before = m;
            for (int c = 0; c < n; c++) {
                if (lane == c) before = m;
                const float most = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(most_own), c));
                m = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sum_own), c)) + fmaxf(m, most);
            }
            const float most = fmaxf(before, most_own);
            keep[lane] = expf(before - most);
            add[lane] = expf(most_own - most);
            if (blockIdx.x == 0 && lane < n) a.chunk_m[(size_t)(first + lane) * sh.heads + h] = before;
        }
        dense_lds_barrier();
        if (!mine) continue;
        for (int c0 = first; c0 < first + n; c0 += kAhead) {
            alignas(16) float now[kAhead][W];
#pragma unroll
            for (int u = 0; u < kAhead; u++)
#pragma unroll
                for (int w = 0; w < W; w++) now[u][w] = next[u][w];
            if (c0 + kAhead < chunks) {
#pragma unroll
                for (int u = 0; u < kAhead; u++) load(next[u], c0 + kAhead + u);
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int c = c0 + u;
                if (c >= chunks) break;
                if constexpr (W == 4)
                    store4(at + c * step, *reinterpret_cast<const float4*>(cur));
                else
                    at[c * step] = cur[0];
#pragma unroll
                for (int w = 0; w < W; w++) cur[w] = fmaf(keep[c - first], cur[w], add[c - first] * now[u][w]);
            }
        }
    }
    if (mine) {
#pragma unroll
        for (int w = 0; w < W; w++) to[w] = cur[w];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) a.chunk_m[(size_t)chunks * sh.heads + h] = m;
}

// Outputs of 32 tokens of a chunk for one head, 32 tokens x vdim columns in the accumulators: 32 x 32 VF per wave.  q and k come
// through LDS, 64 columns at a time; rows of S and v go from memory to the matrix operands, S kAhead x 32 columns of q ahead.
//
// What bounds it: where chunks are few one workgroup's way, products in 32 bits (two fifths) and what waits for them; where they are many also
// the single floats of S and v, an instruction for two rows.  So a workgroup has half a chunk, two of them fit a CU, the halves with
// all keys come first, rows of v follow those of S in one ring, scores are weighted by all waves, and gates are as memory_outer_kernel left them.
// us, so / with a chunk a workgroup, S and v requested just ahead of their use and gates formed again: 8 heads of 128 + 256
// columns, 1 chunk 18.9 / 36.2, 3 chunks 19.9 / 36.7, 13 chunks 22.1 / 41.2, 32 chunks 34.0 / 44.7; 64 + 128, 32 chunks 20.1 / 28.7; 4 heads
// of 256 + 512, 11 chunks 46.6 / 85.
constexpr int kStep = 64;          // columns of q and k in LDS at a time
constexpr int kLd = kStep + 4;     // floats of an LDS row: sixteen-byte reads of neighbouring rows spread over the banks
constexpr int kOut = 32;           // tokens of a workgroup
static_assert(2 * kOut == C, "a chunk has two halves");
template <typename T, int W, int WAVES, int VF>
__global__ __launch_bounds__(64 * WAVES, W == 4 && WAVES == 8 && VF == 1 ? 4 : 2) void memory_outputs_kernel(MemoryArgs a, int chunks, T* __restrict__ out, int ld_out) {
    constexpr int kT = 64 * WAVES, kPer = kStep / W, kLoadsQ = kOut * kPer / kT, kLoadsK = C * kPer / kT;
    constexpr int kTeam = kT / C;  // threads that share a token's sums
    __shared__ __attribute__((aligned(16))) float qs[kOut * kLd], ks[C * kLd];
    __shared__ __attribute__((aligned(16))) float scored[2][kOut * kLd];  // the scores' shares [token][key], then weighted in the first
    __shared__ double log_a[C], log_most[kOut];                         // a_s, M_t
    __shared__ float start[kOut], floor_t[kOut], den[kOut], inv[kOut], squares[kOut][WAVES], n_part[kStep];
    const MemoryShape sh = a.sh;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l31 = lane & 31, half = lane >> 5;
    const int late = 1 - (int)blockIdx.z, chunk = blockIdx.x, h = blockIdx.y, m0 = chunk * C, t0 = late * kOut;
    const int count = min(C, a.M - m0), rows = min(kOut, count - t0), keys = min(count, t0 + kOut);  // rows: of this half
    // the scale after the last chunk goes to the state only now: the chain's workgroups all read the old one
    if (!late && chunk == chunks - 1 && t == 0)
        state_nm(a, max(a.pos_dev[0], 0) + a.M)[(size_t)h * (sh.dim + 1) + sh.dim] = a.chunk_m[(size_t)chunks * sh.heads + h];
    if (rows <= 0) return;
    const float* S = a.chunk_states + ((size_t)chunk * sh.heads + h) * sh.chunk_size();
    const float* n = S + (size_t)sh.dim * sh.vdim;
    const int col0 = wave * 32 * VF + l31;
    float q_part[kLoadsQ][W], k_part[kLoadsK][W], n_own = 0.f;
    auto request = [&](int d0) {
#pragma unroll
        for (int u = 0; u < kLoadsQ; u++) {
            const int i = t + u * kT, s = i / kPer, d = d0 + i % kPer * W;
            read_part<W>(q_part[u], a.in + (size_t)(m0 + t0 + min(s, rows - 1)) * a.ld_in + h * sh.dim + d + sh.at_q, s < rows && d < sh.dim);
        }
#pragma unroll
        for (int u = 0; u < kLoadsK; u++) {
            const int i = t + u * kT, s = i / kPer, d = d0 + i % kPer * W;
            read_part<W>(k_part[u], a.in + (size_t)(m0 + min(s, keys - 1)) * a.ld_in + h * sh.dim + d + sh.at_k, s < keys && d < sh.dim);
        }
        if (t < kStep) n_own = d0 + t < sh.dim ? n[d0 + t] : 0.f;
    };
    // Parts of 32 rows, kHalf operand steps of eight: those of S, in pairs, and two of v.  kAhead parts are under way.
    constexpr int kHalf = kStep / 16, kAhead = VF == 1 ? 2 : 1;
    const int parts = (sh.dim + 31) / 32, first_v = (parts + 1) / 2 * 2;
    const float* v_rows = a.in + (size_t)m0 * a.ld_in + sh.at_v + h * sh.vdim;
    float b[kAhead][kHalf][VF][4];
    auto request_part = [&](float (&to)[kHalf][VF][4], int p) {
        const bool values = p >= first_v;
        if (p >= first_v + late + 1) return;  // keys that come later count nothing
        const float* src = values ? v_rows : S;
        const int ld = values ? a.ld_in : sh.vdim, row0 = 32 * (values ? p - first_v : p), last = values ? count - 1 : sh.dim - 1;
#pragma unroll
        for (int kk = 0; kk < kHalf; kk++)
#pragma unroll
            for (int f = 0; f < VF; f++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    to[kk][f][j] = src[(size_t)min(row0 + 4 * (2 * kk + half) + j, last) * ld + min(col0 + 32 * f, sh.vdim - 1)];
    };
    request(0);
    if (wave == WAVES - 1) {
        const double* g = a.chunk_gates + ((size_t)chunk * sh.heads + h) * 3 * C;
        const float m_start = a.chunk_m[(size_t)chunk * sh.heads + h];
        log_a[lane] = g[C + lane];
        if (lane < kOut) {
            const double most = fmax((double)m_start, g[2 * C + t0 + lane]);
            log_most[lane] = most;
            start[lane] = expf((float)((double)m_start - most));
            floor_t[lane] = expf(-(float)(g[t0 + lane] + most));
        }
    }
#pragma unroll
    for (int u = 0; u < kAhead; u++) request_part(b[u], u);
    f32x16 acc[VF], score;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        score[i] = 0.f;
#pragma unroll
        for (int f = 0; f < VF; f++) acc[f][i] = 0.f;
    }
    // The scores of 32 keys: of two waves each has every second operand step, or one wave has all.
    constexpr int kShares = WAVES == 4 ? 1 : 2;
    const int ss = (wave & 1) * 32, share = wave >> 1;
    const bool scores = wave < 2 * kShares && ss <= t0;
    float nq = 0.f;  // of token t / kTeam, a share of the columns
    const bool sums = t < kOut * kTeam;
    for (int d0 = 0; d0 < sh.dim; d0 += kStep) {
        if (d0) dense_lds_barrier();  // nobody still reads the columns before
#pragma unroll
        for (int u = 0; u < kLoadsQ; u++) {
            const int i = t + u * kT, at = i / kPer * kLd + i % kPer * W;
#pragma unroll
            for (int e = 0; e < W; e++) q_part[u][e] *= sh.q_scale;
            write_part<W>(qs + at, q_part[u]);
        }
#pragma unroll
        for (int u = 0; u < kLoadsK; u++) {
            const int i = t + u * kT;
            write_part<W>(ks + i / kPer * kLd + i % kPer * W, k_part[u]);
        }
        if (t < kStep) n_part[t] = n_own;
        dense_lds_barrier();
        if (d0 + kStep < sh.dim) request(d0 + kStep);
#pragma unroll
        for (int part = 0; part < 2; part++) {
            const int p = d0 / 32 + part;
            if (p < parts) {
#pragma unroll
                for (int kk = 0; kk < kHalf; kk++) {
                    const int step = part * kHalf + kk, at = 4 * (2 * step + half);
                    alignas(16) float q[4], k[4];
                    *reinterpret_cast<float4*>(q) = load4(qs + l31 * kLd + at);
#pragma unroll
                    for (int f = 0; f < VF; f++)
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[f] = mfma32(q[j], b[part % kAhead][kk][f][j], acc[f]);
                    if (scores && (kShares == 1 || (step & 1) == share)) {
                        *reinterpret_cast<float4*>(k) = load4(ks + (ss + l31) * kLd + at);
#pragma unroll
                        for (int j = 0; j < 4; j++) score = mfma32(q[j], k[j], score);
                    }
                }
            }
            request_part(b[part % kAhead], p + kAhead);
        }
        if (sums) {
#pragma unroll
            for (int c = 0; c < kStep / kTeam; c++) {
                const int d = t % kTeam + kTeam * c;
                nq = fmaf(qs[t / kTeam * kLd + d], n_part[d], nq);
            }
        }
    }
    float gate[VF][16];
#pragma unroll
    for (int f = 0; f < VF; f++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int token = min(8 * (r >> 2) + 4 * half + (r & 3), rows - 1);
            gate[f][r] = a.in[(size_t)(m0 + t0 + token) * a.ld_in + sh.at_g + h * sh.vdim + min(col0 + 32 * f, sh.vdim - 1)];
        }
    if (scores) {
#pragma unroll
        for (int i = 0; i < 16; i++) scored[share][(8 * (i >> 2) + 4 * half + (i & 3)) * kLd + ss + l31] = score[i];
    }
    dense_lds_barrier();
    float* const weighted = scored[0];
    for (int i = t; i < kOut * C / 4; i += kT) {
        const int token = i / (C / 4), key0 = i % (C / 4) * 4, at = token * kLd + key0;
        float w[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool seen = key0 + e <= t0 + token;
            const float decay = expf((float)(log_a[key0 + e] - log_most[token]));
            w[e] = seen ? scored[0][at + e] * decay : 0.f;
            if (kShares == 2) w[e] += seen ? scored[1][at + e] * decay : 0.f;
        }
        store4(weighted + at, make_float4(w[0], w[1], w[2], w[3]));
    }
    dense_lds_barrier();
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const float w = start[8 * (r >> 2) + 4 * half + (r & 3)];
#pragma unroll
        for (int f = 0; f < VF; f++) acc[f][r] *= w;
    }
    if (sums) {
        const int token = t / kTeam;
        float sum = nq * start[token];
#pragma unroll
        for (int c = 0; c < C / kTeam; c++) sum += weighted[token * kLd + t % kTeam + kTeam * c];
        sum = dense_wave_sum(sum, kTeam);
        if (t % kTeam == 0) den[token] = 1.0f / (fmaxf(fabsf(sum), floor_t[token]) + kMemoryFloor);
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (u > late) break;
#pragma unroll
        for (int kk = 0; kk < kHalf; kk++) {
            alignas(16) float p[4];
            *reinterpret_cast<float4*>(p) = load4(weighted + l31 * kLd + 32 * u + 4 * (2 * kk + half));
#pragma unroll
            for (int f = 0; f < VF; f++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[f] = mfma32(p[j], b[u % kAhead][kk][f][j], acc[f]);
        }
        if (u + kAhead < 2) request_part(b[u % kAhead], first_v + u + kAhead);
    }
    dense_lds_barrier();
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int token = 8 * (r >> 2) + 4 * half + (r & 3);
        const float d = den[token];
        float sum = 0.f;
#pragma unroll
        for (int f = 0; f < VF; f++) {
            acc[f][r] *= d;
            if (col0 + 32 * f < sh.vdim) sum = fmaf(acc[f][r], acc[f][r], sum);
        }
        sum = dense_wave_sum(sum, 32);
        if (l31 == 0) squares[token][wave] = sum;
    }
    dense_lds_barrier();
    if (t < kOut) {
        float sum = 0.f;
        for (int w = 0; w < WAVES; w++) sum += squares[t][w];
        inv[t] = 1.0f / sqrtf(sum / (float)sh.vdim + sh.eps);
    }
    dense_lds_barrier();
#pragma unroll
    for (int f = 0; f < VF; f++) {
        const int col = col0 + 32 * f;
        if (col >= sh.vdim) continue;
        const float w = a.norm[h * sh.vdim + col];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int token = 8 * (r >> 2) + 4 * half + (r & 3);
            if (token < rows)
                out[(size_t)(m0 + t0 + token) * ld_out + h * sh.vdim + col] = (T)(acc[f][r] * inv[token] * w * sigmoid(gate[f][r]));
        }
    }
}

// whether heads, rows and what is read of them are whole float4s
bool whole_quads(const MemoryArgs& a) {
    const MemoryShape& sh = a.sh;
    return (sh.dim | sh.vdim | a.ld_in | sh.at_q | sh.at_k | sh.at_v) % 4 == 0;
}

template <typename T, int W>
hipError_t launch_chunks(const MemoryArgs& a, T* out, int ld_out, hipStream_t s) {
    const MemoryShape& sh = a.sh;
    const int chunks = (a.M + C - 1) / C, tiles = ((sh.dim + kOuter - 1) / kOuter) * ((sh.vdim + kOuter - 1) / kOuter);
    const int parts = (int)(sh.chunk_size() / W);
    hipLaunchKernelGGL(memory_outer_kernel<W>, dim3(chunks, sh.heads, tiles), dim3(kThreads), 0, s, a);
    hipLaunchKernelGGL(memory_chain_kernel<W>, dim3((parts + kThreads - 1) / kThreads, sh.heads), dim3(kThreads), 0, s, a, chunks);
    const dim3 grid(chunks, sh.heads, 2);
    if (sh.vdim <= 128)
        hipLaunchKernelGGL((memory_outputs_kernel<T, W, 4, 1>), grid, dim3(256), 0, s, a, chunks, out, ld_out);
    else if (sh.vdim <= 256)
        hipLaunchKernelGGL((memory_outputs_kernel<T, W, 8, 1>), grid, dim3(512), 0, s, a, chunks, out, ld_out);
    else
        hipLaunchKernelGGL((memory_outputs_kernel<T, W, 8, 2>), grid, dim3(512), 0, s, a, chunks, out, ld_out);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_memory_steps(const MemoryArgs& a, float* o, hipStream_t s) {
    if (steps_held_back(a) && !a.held) return hipErrorInvalidValue;
    const dim3 grid((a.sh.vdim + kSlice - 1) / kSlice, a.sh.heads);
    auto lds = [&](int w) { return step_floats(a.sh.dim, w) * sizeof(float); };
    if (a.sh.vdim % 4 == 0)
        hipLaunchKernelGGL(memory_steps_kernel<4>, grid, dim3(kThreads), lds(4), s, a, o);
    else
        hipLaunchKernelGGL(memory_steps_kernel<1>, grid, dim3(kThreads), lds(1), s, a, o);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_memory_norm(const MemoryArgs& a, const float* o, T* out, int ld_out, hipStream_t s) {
    hipLaunchKernelGGL(memory_norm_kernel<T>, dim3(a.M), dim3(kThreads), (a.sh.heads + kThreads / 64) * sizeof(float), s, a, o, out, ld_out);
    return hipGetLastError();
}

bool memory_chunks_fit(const MemoryShape& sh) { return sh.vdim <= 512; }

template <typename T>
hipError_t launch_memory_chunks(const MemoryArgs& a, T* out, int ld_out, hipStream_t s) {
    return whole_quads(a) ? launch_chunks<T, 4>(a, out, ld_out, s) : launch_chunks<T, 1>(a, out, ld_out, s);
}

#define INSTANTIATE(T)                                                                                   \
    template hipError_t launch_memory_norm<T>(const MemoryArgs&, const float*, T*, int, hipStream_t);     \
    template hipError_t launch_memory_chunks<T>(const MemoryArgs&, T*, int, hipStream_t);
INSTANTIATE(bf16)
INSTANTIATE(float)

}  // namespace a81w41
