// Merge pass over the partials of rows cut into a few parts (head_dim 128, 16-bit output):
// shared by the prefill path (tiles cut into parts) and the decode path (requests cut across
// workgroups).
#pragma once

#include "kv_tile.h"

namespace dskv {

// `n` parts added up under their maximum m_all, w_i = exp2(m_i - max_j m_j): acc = sum_i w_i O_i, l_all =
// sum_i w_i l_i, kAtOnce parts at a time under a running maximum.  Offsets are
// those of the thread's four dims of one head within a slot.  kAll: n == kAtOnce.
template <int kAtOnce, bool kAll>
__device__ __forceinline__ f32x4 merge_run(const float *__restrict__ o_src, const float *__restrict__ ml_src, int n,
                                           long o_stride, long ml_stride, float &m_all, float &l_all)
{
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    m_all = kNegBig;
    l_all = 0.f;
    for (int i0 = 0; i0 < n; i0 += kAtOnce) {
        f32x4 o[kAtOnce];
        f32x2 ml[kAtOnce];   // (maximum, sum)
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const long at = kAll ? i : min(i0 + i, n - 1);   // past the last: it again, weight zero
            o[i] = *reinterpret_cast<const f32x4 *>(o_src + at * o_stride);
            ml[i] = *reinterpret_cast<const f32x2 *>(ml_src + at * ml_stride);
        }
        float m_new = m_all;
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) m_new = fmaxf(m_new, ml[i].x);
        const float keep = __builtin_amdgcn_exp2f(m_all - m_new);
        l_all *= keep;
        acc *= keep;
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const float w = kAll || i0 + i < n ? __builtin_amdgcn_exp2f(ml[i].x - m_new) : 0.f;
            l_all += w * ml[i].y;
            acc += w * o[i];
        }
        m_all = m_new;
        if (kAll) break;
    }
    return acc;
}
template <int DT>
__device__ __forceinline__ void put_merged(uint16_t *__restrict__ dst, f32x4 acc, float l_all)
{
    typedef Elt<DT> E;
    const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
    *reinterpret_cast<u32x2 *>(dst) = u32x2{E::pack2(acc[0] * inv, acc[1] * inv), E::pack2(acc[2] * inv, acc[3] * inv)};
}
template <int DT, int kAtOnce, bool kAll>
__device__ __forceinline__ void merge_dims(uint16_t *__restrict__ dst, const float *__restrict__ o_src,
                                           const float *__restrict__ ml_src, int n, long o_stride, long ml_stride)
{
    float m_all, l_all;
    const f32x4 acc = merge_run<kAtOnce, kAll>(o_src, ml_src, n, o_stride, ml_stride, m_all, l_all);
    put_merged<DT>(dst, acc, l_all);
}

// row_parts[2 r] = row r's first slot, row_parts[2 r + 1] = its number of parts (consecutive
// slots); 0: the row was written by the attention kernel itself and is left alone.  row_map
// (may be null) names the output row of r.
//
// A workgroup per (row, kMergeHeads heads); a thread owns four dims of one head.  What bounds it is
// the row with the most parts: one workgroup per row (a thread per 16 dims) took 16 us for 128 requests
// of 64 heads, the longest in 15-20 parts of 33 KB, and eight heads a workgroup 11; 64 requests of 32 heads in 4-5
// parts take 4.7.  Four or two heads per workgroup take the same time.
//
// kMany (a decode batch of fewer requests than shares: some may be in more than kMergeFewParts parts): such a row gets a workgroup
// for two heads, in which four groups of threads take a quarter of the parts each, requested in one trip up to
// 32 parts: those 128 requests 10.9 -> 6.9 us a launch, 2406 -> 2368 us a step of 10 layers; the other rows' surplus
// workgroups return at once (64 requests: 4.7 us either way).  A batch of many rows, none of which can have so many
// parts (tiles), is launched without them: 512 rows of a chunk 7.1 against 7.7 us.
constexpr int kMergeHeads = 8, kMergeHeadsMany = 2, kMergeFewParts = 8;
constexpr int kMergeThreads = kMergeHeads * (kHeadDim / 4);
template <int DT, bool kMany>
__global__ __launch_bounds__(kMergeThreads) void merge_parts_kernel(
    uint16_t *__restrict__ out, const float *__restrict__ part_o, const float *__restrict__ part_ml,
    const int32_t *__restrict__ row_parts, const int32_t *__restrict__ row_map, int max_slots,
    int n_qo_heads)
{
    const long r = blockIdx.x;
    const const_i32_ptr table = as_const(row_parts) + 2 * r;
    const int first = table[0], n = table[1];   // uniform over the workgroup
    if (n <= 0 || first < 0 || first + n > max_slots) return;
    const long row = row_map ? as_const(row_map)[r] : r;
    const int head = (int)threadIdx.x / (kHeadDim / 4), d0 = (int)threadIdx.x % (kHeadDim / 4) * 4;
    const long o_stride = (long)n_qo_heads * kHeadDim, ml_stride = (long)n_qo_heads * 2;
    if (kMany && n > kMergeFewParts) {
        constexpr int kRuns = kMergeHeads / kMergeHeadsMany;
        __shared__ f32x4 o_lds[kRuns][kMergeHeadsMany][kHeadDim / 4];
        __shared__ f32x2 ml_lds[kRuns][kMergeHeadsMany];
        const int run = head / kMergeHeadsMany, mine = head % kMergeHeadsMany;
        const int qh = blockIdx.y * kMergeHeadsMany + mine;
        const int at = first + n * run / kRuns, end = first + n * (run + 1) / kRuns;
        float m = kNegBig, l = 0.f;
        if (qh < n_qo_heads)
            o_lds[run][mine][d0 / 4] = merge_run<8, false>(part_o + at * o_stride + (long)qh * kHeadDim + d0,
                                                           part_ml + at * ml_stride + (long)qh * 2, end - at, o_stride,
                                                           ml_stride, m, l);
        if (d0 == 0) ml_lds[run][mine] = f32x2{m, l};
        __syncthreads();
        if (run > 0 || qh >= n_qo_heads) return;
        float m_all = kNegBig, l_all = 0.f;
#pragma unroll
        for (int i = 0; i < kRuns; i++) m_all = fmaxf(m_all, ml_lds[i][mine].x);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kRuns; i++) {
            const float w = __builtin_amdgcn_exp2f(ml_lds[i][mine].x - m_all);
            l_all += w * ml_lds[i][mine].y;
            sum += w * o_lds[i][mine][d0 / 4];
        }
        put_merged<DT>(out + (row * n_qo_heads + qh) * kHeadDim + d0, sum, l_all);
        return;
    }
    const int qh = blockIdx.y * kMergeHeads + head;
    if (qh >= n_qo_heads) return;
    uint16_t *dst = out + (row * n_qo_heads + qh) * kHeadDim + d0;
    const float *o = part_o + first * o_stride + (long)qh * kHeadDim + d0;
    const float *ml = part_ml + first * ml_stride + (long)qh * 2;
    // up to eight parts are requested at once, exactly as many as there are
    switch (n) {
    case 1: merge_dims<DT, 1, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 2: merge_dims<DT, 2, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 3: merge_dims<DT, 3, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 4: merge_dims<DT, 4, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 5: merge_dims<DT, 5, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 6: merge_dims<DT, 6, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 7: merge_dims<DT, 7, true>(dst, o, ml, n, o_stride, ml_stride); break;
    case 8: merge_dims<DT, 8, true>(dst, o, ml, n, o_stride, ml_stride); break;
    default: merge_dims<DT, 16, false>(dst, o, ml, n, o_stride, ml_stride); break;
    }
}

}  // namespace dskv
