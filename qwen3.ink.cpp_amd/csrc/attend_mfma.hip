// Causal attention on the matrix cores for bfloat16 rows, in three forms:
//   shared    every query row looks at the same key rows, whose first columns are also the values (attention in
//             latent space: the key rows are the cache itself);
//   rows      the queries of a group of heads look at the rows of their key/value head, [value | key] (grouped attention);
//   expanded  keys and values of every head were formed beforehand: a key is [own part | part shared by all heads],
//             values come transposed ([value column][key]).
// The first, and the second up to kAttendShortRows rows, are here, the others in attend_prompt.hip.
//
// A wave owns 16 (or 2 x 16) query rows.  It forms the scores transposed, S^T = K Q^T (v_mfma_f32_16x16x32_bf16 with
// the keys as rows), so that lane l holds scores of query l % 16 only: keys 16 t + 4 (l / 16) + i.  These registers
// are, without any exchange, the B operand of O^T = V^T P^T if lane group l / 16 takes the keys
// {4 g + i, 16 + 4 g + i} of a 32-key step as its eight k places; V^T is read from LDS in that order.  Running maximum
// and sum are one value per lane.  Scores, softmax and sums are fp32.
//
// A tile of keys is copied global -> LDS by direct 16-byte loads.  Key rows: chunk c of row r at place c ^ (r & 7).
// Query columns beyond the real width are zero, so whatever finite values sit there in the key rows do not count.
#include "attend_rows.h"

namespace a81w41 {
namespace {

using namespace attend;

template <int DK, int DV, int KEY0, int WAVES, int QS, int KT, int NBUF, bool COLS>
__global__ __launch_bounds__(64 * WAVES, 1) void attend_kernel(AttendArgs<bf16> a) {
    __shared__ __attribute__((aligned(128))) uint8_t lds[attend_lds(DK, KT, NBUF)];
    __shared__ float scores[COLS ? attend_scores(QS, KT) : 1];
    attend_workgroup<DK, DV, KEY0, WAVES, QS, KT, NBUF, COLS>(a, gridDim, blockIdx, lds, scores);
}

// out row = sum_s w_s part_s / sum_s w_s sum_s with w_s = 2^(m_s - max m); one workgroup per head's row and 256 columns
__global__ __launch_bounds__(256) void merge_shares_kernel(AttendArgs<bf16> a, int heads) {
    __shared__ float w[kAttendMaxSplits];
    __shared__ float norm;
    const int all_rows = heads * a.rows, at = blockIdx.x, t = threadIdx.x;
    if (t < 64) {
        float m = t < a.splits ? a.part_stats[2 * ((size_t)t * all_rows + at)] : kLowest;
        const float l = t < a.splits ? a.part_stats[2 * ((size_t)t * all_rows + at) + 1] : 0.f;
        const float top = dense_wave_max(m);
        const float mine = exp2f(m - top);
        if (t < a.splits) w[t] = mine;
        const float total = dense_wave_sum(t < a.splits ? mine * l : 0.f);
        if (t == 0) norm = 1.0f / total;
    }
    __syncthreads();
    const int d = blockIdx.y * 256 + t;
    if (d >= a.dv) return;
    float s = 0.f;
    for (int k = 0; k < a.splits; k++) s = fmaf(w[k], a.part[((size_t)k * all_rows + at) * a.ld_part + d], s);
    const int z = at / a.rows, r = at - z * a.rows, token = r / a.rows_per_token;
    a.out[z * a.out_head + (size_t)token * a.out_token + (r - token * a.rows_per_token) * a.ld_out + d] = (bf16)(s * norm);
}
static_assert(kAttendMaxSplits <= 64, "the merge reads one share per lane");

template <int DK, int DV, int KEY0, int WAVES, int QS, int KT, int NBUF, bool COLS>
hipError_t launch_kernel(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    constexpr int rows = 16 * QS * (COLS ? 1 : WAVES);
    hipLaunchKernelGGL((attend_kernel<DK, DV, KEY0, WAVES, QS, KT, NBUF, COLS>), dim3((a.rows + rows - 1) / rows, heads, a.splits),
                       dim3(64 * WAVES), 0, s, a);
    return hipGetLastError();
}
template <int DK, int DV>
hipError_t launch_shared(const AttendArgs<bf16>& a, hipStream_t s) {
    return a.rows <= kAttendFewRows ? launch_kernel<DK, DV, 0, 4, 1, 64, 2, true>(a, 1, s)
                                    : launch_kernel<DK, DV, 0, 4, 1, 32, 1, false>(a, 1, s);
}
// key and value columns: D at most each; up to kAttendShortRows rows
template <int D, int QS>
hipError_t launch_rows(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    return a.rows <= kAttendFewRows ? launch_kernel<2 * D, D, D, 4, 1, 64, 2, true>(a, heads, s)
                                    : launch_kernel<2 * D, D, D, 4, QS, 64, 2, false>(a, heads, s);
}

}  // namespace

bool attend_shared_fits(int dk, int dv) { return dk <= 576 && dv <= 512; }
bool attend_rows_fits(int key, int value) { return key % 8 == 0 && value % 8 == 0 && key <= 256 && value <= 256; }
bool attend_expanded_fits(int own, int shared, int dv) { return own % 8 == 0 && shared % 8 == 0 && own + shared <= 320 && dv <= 256; }

hipError_t launch_attend_shared(const AttendArgs<bf16>& a, hipStream_t s) {
    const int dk = a.k_own_width;
    if (dk <= 192 && a.dv <= 128) return launch_shared<192, 128>(a, s);
    if (dk <= 320 && a.dv <= 256) return launch_shared<320, 256>(a, s);
    return launch_shared<576, 512>(a, s);
}

hipError_t launch_attend_rows(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    if (a.rows > kAttendShortRows) return launch_attend_rows_prompt(a, heads, s);
    const int widest = a.k_own_width > a.v_width ? a.k_own_width : a.v_width;
    if (widest <= 64) return launch_rows<64, 2>(a, heads, s);
    if (widest <= 128) return launch_rows<128, 2>(a, heads, s);
    return launch_rows<256, 1>(a, heads, s);
}

hipError_t launch_merge_shares(const AttendArgs<bf16>& a, int heads, hipStream_t s) {
    hipLaunchKernelGGL(merge_shares_kernel, dim3(heads * a.rows, (a.dv + 255) / 256), dim3(256), 0, s, a, heads);
    return hipGetLastError();
}

}  // namespace a81w41
