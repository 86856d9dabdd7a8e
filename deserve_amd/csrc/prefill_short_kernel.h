// The 16-bit paged prefill attention (head_dim 128) for launches that last as long as one workgroup does: a few short
// prompts or chunks, whose tiles leave most of the chip idle and whose walks are a handful of blocks.
//
// What bounds it: latency - the chain plan -> request -> page -> rows, the blocks one after the other, and the
// instructions in between, which a wave that depends on itself issues every five to ten cycles.  The kernel of
// long walks (prefill_kernel.h) gives a tile of 256 columns to a workgroup, whose waves walk all blocks of its keys
// together.  Here a workgroup has a quarter of that tile, 64 columns (or half of it): two (four) waves a key group,
// four (two) key groups, so that a wave computes every fourth (second) block of its 32 columns' keys; up to
// 256 keys come into LDS at once, with one wait and one barrier, and the key groups' sums meet in LDS.
// Measured with the launch that appends the new rows (bf16, 8 kv heads, groups of 4, us a layer, in the kernel of long
// walks -> here): prompts of 20 tokens 12.0 -> 8.3, of 128 16.2 -> 11.0, of 256 18.9 -> 13.8; three of 17 to 203
// 17.7 -> 13.6; 64 tokens behind 190 18.6 -> 13.4, behind 450 24.4 -> 20.7; 8 prompts of 128 (halves) 19.5 -> 16.5.
// The append inside this launch (rows from k and v, K rotated on the way into LDS) was slower than in front of it: 18.7
// against 13.6 for three prompts, the walk's registers spilled.
#pragma once

#include "kv_tile.h"
#include "prefill_kernel.h"
#include "rope_math.h"

namespace dskv {

constexpr int kShortWaves = 8;
constexpr int kShortQRows = 64;                                // columns whose q rows are in LDS at a time
constexpr int kShortRoundBlocks = kShortWaves;                 // blocks in LDS at a time: a wave loads one
constexpr int kShortRoundTokens = kShortRoundBlocks * kBlock;
constexpr int kShortPartPitch = 132;                           // floats of a column's partial sums in LDS
struct ShortShared {
    union {
        struct {
            char k[kShortRoundBlocks * kStageBytes], v[kShortRoundBlocks * kStageBytes];
        };
        float part[kShortWaves][32][kShortPartPitch];
    };
    char q[kShortQRows * kRowPitch];
    float ml[kShortWaves][32][2];
};
static_assert(sizeof(ShortShared) <= 160 * 1024, "");

struct ShortArgs {
    const int32_t *tile_info, *qo_indptr, *kv_indptr, *kv_last;
    const int32_t *kv_indices;
    const char *pages;
    const uint16_t *q;
    const float *rope;   // cos | sin by query row (q is rotated as it is loaded), or null
    uint16_t *out;
    int n_qo_heads, n_kv_heads, group;
    int group_inverse;   // x / group = x * this >> 16 for x < 32
    int page_shift, causal;
    float scale_log2;
};

// kColWaves: waves side by side, 32 columns each, in every key group (2: four groups, a quarter of a plan's tile; 4: two
// groups, half of it).
// kUnitRows: rows of a block that lie in one page for sure (16 or 8: pages of 16 tokens and more, of 8).
template <int DT, int kColWaves, int kUnitRows>
__global__ __launch_bounds__(64 * kShortWaves) void prefill_short_kernel(const ShortArgs a)
{
    typedef Elt<DT> E;
    constexpr int kKeyGroups = kShortWaves / kColWaves, kPasses = 32 * kColWaves / kShortQRows;
    constexpr int kUnits = kBlock / kUnitRows, kLoads = kUnitRows / 4;   // units of a block, loads of a unit
    __shared__ __align__(16) ShortShared sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;   // roles in the transposing reads
    const int h = lane >> 5, r = lane & 31;   // MFMA roles
    const int kvh = (int)blockIdx.x, tile = (int)blockIdx.y, sub = (int)blockIdx.z;
    const const_i32_ptr entry = as_const(a.tile_info) + tile * kTileWords;
    const int b = entry[0], pos_per_wave = (32 * a.group_inverse) >> 16;
    const int q0 = entry[1] + sub * kColWaves * pos_per_wave;
    const const_i32_ptr qo_at = as_const(a.qo_indptr) + b, kv_at = as_const(a.kv_indptr) + b;
    const int q_begin = qo_at[0], q_next = qo_at[1], page_begin = kv_at[0], page_next = kv_at[1];
    const int last_page_len = as_const(a.kv_last)[b];
    asm volatile("" ::"s"(q_begin), "s"(q_next), "s"(page_begin), "s"(page_next), "s"(last_page_len));   // (in one trip)
    const int n_b = q_next - q_begin, n_pages = page_next - page_begin;
    if (q0 >= n_b) return;   // a quarter of the plan's tile that has no rows
    const int kv_len = n_pages > 0 ? ((n_pages - 1) << a.page_shift) + last_page_len : 0;
    const const_i32_ptr page_ids = as_const(a.kv_indices) + page_begin;
    const int row_bytes = a.n_kv_heads * kHeadDim * 2, half_bytes = row_bytes << a.page_shift;
    const int rows_wg = min(kColWaves * pos_per_wave, n_b - q0);
    // keys [0, t_end) are seen by some row of the workgroup
    const int t_end = min(max(a.causal ? kv_len - n_b + q0 + rows_wg : kv_len, 0), kv_len);

    // ---- requests, in the order in which they are needed: page ids, q and angles, K and V
    // Every wave brings one block of a round into LDS: rows straight from memory, a region of four by each load (the
    // layout and the descriptors that end after the last valid row are those of prefill_kernel.h).
    typedef __attribute__((address_space(3))) void *lds_ptr;
    int direct_off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) direct_off[i] = (4 * i + (lane & 3)) * row_bytes + kvh * (kHeadDim * 2) + (lane >> 2) * 16;
    const int last_entry = max(n_pages - 1, 0);
    int pg[kUnits];
    auto look_up = [&](int block) {
#pragma unroll
        for (int u = 0; u < kUnits; u++) pg[u] = page_ids[min((block * kBlock + u * kUnitRows) >> a.page_shift, last_entry)];
        __builtin_amdgcn_sched_barrier(0);   // all requested before the first is waited for
#pragma unroll
        for (int u = 0; u < kUnits; u++) asm volatile("" : "+s"(pg[u]));
    };
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    auto load_block = [&](int block) {
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
            const int tok0 = block * kBlock + u * kUnitRows;
            const int bytes = min(max(t_end - tok0, 0), kUnitRows) * row_bytes;
            const char *first = a.pages + (long)pg[u] * (2L * half_bytes) + (long)((tok0 & ((1 << a.page_shift) - 1)) * row_bytes);
#pragma unroll
            for (int kv = 0; kv < 2; kv++) {
                const uint64_t at = (uint64_t)(first + (kv ? half_bytes : 0));
                const u32x4 desc = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at),
                                    (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(at >> 32) & 0xFFFFu)),
                                    (uint32_t)__builtin_amdgcn_readfirstlane(bytes), (uint32_t)kBufferFlags};
#pragma unroll
                for (int i = 0; i < kLoads; i++) {
                    char *region = (kv ? sh.v : sh.k) + wave * kStageBytes + (u * kLoads + i) * kRegionBytes;
                    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                                 :
                                 : "s"((uint32_t)(uintptr_t)(lds_ptr)region), "v"(direct_off[i]), "s"(desc)
                                 : "memory", "m0");
                }
            }
        }
    };
#pragma clang diagnostic pop
    if (wave * kBlock < t_end) look_up(wave);
    // q: a lane has chunk c of columns tid / 16 and tid / 16 + 32; a column without a row takes the workgroup's first
    struct Column {
        int row, head;   // of the request (negative: none), of the group
    };
    auto column_of = [&](int col) {
        const int in_wave = col & 31, pos = (in_wave * a.group_inverse) >> 16;
        const int row = q0 + (col >> 5) * pos_per_wave + pos;
        return Column{pos < pos_per_wave && row < n_b ? row : -1, in_wave - pos * a.group};
    };
    u32x4 q[2 * kPasses];
    f32x4 cs[2 * kPasses], sn[2 * kPasses];
    const int q_chunk = (int)threadIdx.x & 15;
#pragma unroll
    for (int i = 0; i < 2 * kPasses; i++) {
        const Column col = column_of(((int)threadIdx.x >> 4) + 32 * i);
        const long row = q_begin + (col.row < 0 ? q0 : col.row);
        q[i] = *reinterpret_cast<const u32x4 *>(
            a.q + (row * a.n_qo_heads + kvh * a.group + (col.row < 0 ? 0 : col.head)) * kHeadDim + q_chunk * 8);
        if (a.rope) {
            const float *tab = a.rope + row * kHeadDim + q_chunk * 4;
            cs[i] = *reinterpret_cast<const f32x4 *>(tab);
            sn[i] = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2);
        }
    }
    if (wave * kBlock < t_end) load_block(wave);
    // q turned and on its way to the operand, 64 columns at a time
    const int col_wave = wave & (kColWaves - 1), key_group = wave / kColWaves;
    u32x4 qreg[8];
#pragma unroll
    for (int pass = 0; pass < kPasses; pass++) {
        if (pass > 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (bare barriers: the rows need not be there)
            __builtin_amdgcn_s_barrier();
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
            *reinterpret_cast<u32x4 *>(sh.q + (((int)threadIdx.x >> 4) + 32 * i) * kRowPitch + q_chunk * 16) =
                a.rope ? rotate_chunk<DT>(q[2 * pass + i], cs[2 * pass + i], sn[2 * pass + i]) : q[2 * pass + i];
        if (pass + 1 == kPasses) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // this wave's rows are in LDS
            __syncthreads();
        } else {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        if (col_wave / 2 == pass)
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
                qreg[ks] = *reinterpret_cast<const u32x4 *>(sh.q + ((col_wave & 1) * 32 + r) * kRowPitch + (2 * ks + h) * 16);
    }

    // ---- a wave: its 32 columns over every fourth block
    const Column mine = column_of(col_wave * 32 + r);
    const int limit = mine.row < 0 ? 0 : min(max(a.causal ? kv_len - n_b + mine.row + 1 : kv_len, 0), kv_len);
    const int wq0 = q0 + col_wave * pos_per_wave, rows_w = min(pos_per_wave, n_b - wq0);
    // blocks that some of its columns see; from token `all_see` on some do not
    auto end_of = [&](int rows) { return rows > 0 ? min(max(a.causal ? kv_len - n_b + wq0 + rows : kv_len, 0), kv_len) : 0; };
    const int n_blocks = (end_of(rows_w) + kBlock - 1) / kBlock, all_see = end_of(min(rows_w, 1));
    f32x16 acc[4];
    float m_run = 2.f * kNegBig, l_run = 0.f;
    const int v_lane_off = h * kRegionBytes + (2 * (g & 1) + ((c & 3) >> 1)) * 64 + (c >> 2) * 16 + (c & 1) * 8;
    for (int first = 0, block = key_group; first * kBlock < t_end; first += kShortRoundBlocks) {
        if (first > 0) {
            __syncthreads();   // the rows of the round before have been read
            if ((first + wave) * kBlock < t_end) {
                look_up(first + wave);
                load_block(first + wave);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        for (; block < min(n_blocks, first + kShortRoundBlocks); block += kKeyGroups) {
            const char *k_rows = sh.k + (block - first) * kStageBytes + (r >> 2) * kRegionBytes + h * 64 + (r & 3) * 16;
            const char *v_rows = sh.v + (block - first) * kStageBytes + v_lane_off;
            u32x4 ka[8], va[4][2];
#pragma unroll
            for (int ks = 0; ks < 8; ks++) ka[ks] = *reinterpret_cast<const u32x4 *>(k_rows + ks * 128);
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    const char *vp = v_rows + ks * 4 * kRegionBytes + dt * 256;
                    const u32x2 lo = read_transposed(vp), hi = read_transposed(vp + 2 * kRegionBytes);
                    va[dt][ks] = u32x4{lo.x, lo.y, hi.x, hi.y};
                }
            __builtin_amdgcn_sched_barrier(0);
            f32x16 s;
#pragma unroll
            for (int v = 0; v < 16; v++) s[v] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 8; ks++) s = E::mfma_32x32(ka[ks], qreg[ks], s);
            const int t = block * kBlock;
            if (t + kBlock > all_see) {
                const int seen = limit - 4 * h - t;   // tokens of the lane's half that the column sees
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (8 * (v >> 2) + (v & 3) >= seen) s[v] = kNegBig;
            }
            float m = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
            for (int v = 3; v < 15; v += 2) m = fmaxf(fmaxf(m, s[v]), s[v + 1]);
            m = fmaxf(m, s[15]);
            float other = m;
            swap_halves32(m, other);
            // (never below half of a masked score: those come out as zeros)
            const float m_new = fmaxf(fmaxf(m_run, 0.5f * kNegBig * a.scale_log2), fmaxf(m, other) * a.scale_log2);
            float p[16], sum = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                p[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], a.scale_log2, -m_new));
                sum += p[v];
            }
            u32x4 pb[2];
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
                pb[ks] = u32x4{E::pack2(p[8 * ks], p[8 * ks + 1]), E::pack2(p[8 * ks + 2], p[8 * ks + 3]),
                               E::pack2(p[8 * ks + 4], p[8 * ks + 5]), E::pack2(p[8 * ks + 6], p[8 * ks + 7])};
            if (block == key_group) {
                l_run = sum;
#pragma unroll
                for (int dt = 0; dt < 4; dt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[dt][v] = 0.f;
            } else {
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                l_run = l_run * alpha + sum;
#pragma unroll
                for (int dt = 0; dt < 4; dt++) acc[dt] *= alpha;
            }
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) acc[dt] = E::mfma_32x32(va[dt][ks], pb[ks], acc[dt]);
        }
    }
    __syncthreads();   // the rows have been read
    if (key_group < n_blocks) {
        float l_other = l_run;
        swap_halves32(l_run, l_other);
        float *const part = sh.part[wave][r];
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                *reinterpret_cast<f32x4 *>(part + dt * 32 + 8 * i + 4 * h) =
                    f32x4{acc[dt][4 * i], acc[dt][4 * i + 1], acc[dt][4 * i + 2], acc[dt][4 * i + 3]};
        if (h == 0) *reinterpret_cast<f32x2 *>(sh.ml[wave][r]) = f32x2{m_run, l_run + l_other};
    }
    __syncthreads();

    // ---- the key groups' sums: kLanes lanes a column, kDims dims each
    constexpr int kLanes = 64 * kShortWaves / (32 * kColWaves), kDims = kHeadDim / kLanes;
    const int col = (int)threadIdx.x / kLanes, dims = (int)threadIdx.x % kLanes * kDims;
    const Column to = column_of(col);
    if (to.row < 0) return;
    const int col_w = col >> 5, in_wave = col & 31;   // (a wave's columns are of one column wave)
    const int cq0 = q0 + col_w * pos_per_wave, rows_c = min(pos_per_wave, n_b - cq0);
    const int seen_c = min(max(a.causal ? kv_len - n_b + cq0 + rows_c : kv_len, 0), kv_len);
    const int groups = min((seen_c + kBlock - 1) / kBlock, kKeyGroups);   // key groups with blocks
    f32x2 ml[kKeyGroups];
    f32x4 o[kKeyGroups][kDims / 4];
#pragma unroll
    for (int kg = 0; kg < kKeyGroups; kg++) {
        const int w = min(kg, max(groups - 1, 0)) * kColWaves + col_w;
        ml[kg] = *reinterpret_cast<const f32x2 *>(sh.ml[w][in_wave]);
#pragma unroll
        for (int i = 0; i < kDims / 4; i++) o[kg][i] = *reinterpret_cast<const f32x4 *>(sh.part[w][in_wave] + dims + 4 * i);
    }
    float m_all = 2.f * kNegBig, l_all = 0.f;
    f32x4 sum[kDims / 4] = {};
#pragma unroll
    for (int kg = 0; kg < kKeyGroups; kg++) m_all = kg < groups ? fmaxf(m_all, ml[kg].x) : m_all;
#pragma unroll
    for (int kg = 0; kg < kKeyGroups; kg++)
        if (kg < groups) {
            const float weight = __builtin_amdgcn_exp2f(ml[kg].x - m_all);
            l_all += weight * ml[kg].y;
#pragma unroll
            for (int i = 0; i < kDims / 4; i++) sum[i] += weight * o[kg][i];
        }
    const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
    uint16_t *const dst = a.out + ((long)(q_begin + to.row) * a.n_qo_heads + kvh * a.group + to.head) * kHeadDim + dims;
#pragma unroll
    for (int i = 0; i < kDims / 8; i++)
        *reinterpret_cast<u32x4 *>(dst + 8 * i) =
            u32x4{E::pack2(sum[2 * i][0] * inv, sum[2 * i][1] * inv), E::pack2(sum[2 * i][2] * inv, sum[2 * i][3] * inv),
                  E::pack2(sum[2 * i + 1][0] * inv, sum[2 * i + 1][1] * inv), E::pack2(sum[2 * i + 1][2] * inv, sum[2 * i + 1][3] * inv)};
}

}  // namespace dskv
