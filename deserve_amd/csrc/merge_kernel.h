// Merge pass over the partials of rows cut into a few parts (head_dim 128, 16-bit output):
// shared by the prefill path (tiles cut into parts) and the decode path (requests cut across
// workgroups).
#pragma once

#include "kv_tile.h"

namespace dskv {

// The merge of `n` parts in slots first .. first + n - 1: output row = sum_i w_i O_i / sum_i w_i l_i,
// w_i = exp2(m_i - max_j m_j), kAtOnce parts at a time under a running maximum.  Offsets are
// those of the thread's four dims of one head within a slot.  kAll: n == kAtOnce.
template <int DT, int kAtOnce, bool kAll>
__device__ __forceinline__ void merge_dims(uint16_t *__restrict__ dst, const float *__restrict__ o_src,
                                           const float *__restrict__ ml_src, int n, long o_stride, long ml_stride)
{
    typedef Elt<DT> E;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float m_all = kNegBig, l_all = 0.f;
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
    const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
    *reinterpret_cast<u32x2 *>(dst) = u32x2{E::pack2(acc[0] * inv, acc[1] * inv), E::pack2(acc[2] * inv, acc[3] * inv)};
}

// row_parts[2 r] = row r's first slot, row_parts[2 r + 1] = its number of parts (consecutive
// slots); 0: the row was written by the attention kernel itself and is left alone.  row_map
// (may be null) names the output row of r.
//
// A workgroup per (row, kMergeHeads heads); a thread owns four dims of one head.  What bounds it is
// the memory path of a compute unit (~36 GB/s) on the row with the most parts: one workgroup
// per row (a thread per 16 dims) took 16 us for 128 requests of 64 heads, the longest in 15-20 parts
// of 33 KB, and now 11.7; 64 requests of 32 heads in 4-5 parts take 4.9.  Four or two heads per
// workgroup take the same time.
constexpr int kMergeHeads = 8;
constexpr int kMergeThreads = kMergeHeads * (kHeadDim / 4);
template <int DT>
__global__ __launch_bounds__(kMergeThreads) void merge_parts_kernel(
    uint16_t *__restrict__ out, const float *__restrict__ part_o, const float *__restrict__ part_ml,
    const int32_t *__restrict__ row_parts, const int32_t *__restrict__ row_map, int max_slots,
    int n_qo_heads)
{
    const long r = blockIdx.x;
    const const_i32_ptr table = as_const(row_parts) + 2 * r;
    const int first = table[0], n = table[1];   // uniform over the workgroup
    if (n <= 0 || first < 0 || first + n > max_slots) return;
    const int qh = blockIdx.y * kMergeHeads + (int)threadIdx.x / (kHeadDim / 4);
    if (qh >= n_qo_heads) return;
    const long row = row_map ? as_const(row_map)[r] : r;
    const int d0 = (int)threadIdx.x % (kHeadDim / 4) * 4;
    const long o_stride = (long)n_qo_heads * kHeadDim, ml_stride = (long)n_qo_heads * 2;
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
