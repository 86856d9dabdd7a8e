// The 16-bit paged prefill attention kernel (head_dim 128): see prefill_attn.hip for the
// decomposition.  Kept in a header because two launches use its body: the stand-alone one
// (workgroups of eight waves) and the mixed launch of prefill_attn.hip, whose four-wave
// workgroups share their compute units with decode workgroups.
#pragma once

#include "append_rows.h"
#include "kv_tile.h"
#include "rope_math.h"

namespace dskv {

#ifndef DSKV_PREFILL_COLTILES
#define DSKV_PREFILL_COLTILES 1
#endif
constexpr int kPrefillWaves = 8;                    // waves per workgroup of the stand-alone launch
constexpr int kPrefillWavesShared = 4;              // ... of the launch whose workgroups share a CU with decode workgroups
constexpr int kColTiles = DSKV_PREFILL_COLTILES;    // column tiles (of 32 columns) per wave
constexpr int kWaveCols = 32 * kColTiles;           // columns per wave
constexpr int kBlock = 32;                          // tokens per step (one MFMA tile)
constexpr int kTileWords = 6;                       // plan entry: request, first row, block range, part, first slot
// LDS layout of a 32-token block of K (or V) rows of one kv head: eight regions of four rows.
// A region is what one load instruction delivers: 64 lanes x 16 bytes, lane p at byte 16 p.
// Lane p = 4 c + rho fetches the 16-byte chunk c of row rho, so the region holds its rows
// interleaved chunk by chunk ((4 c + rho) * 16); regions are 1088 bytes apart (64 bytes of
// padding).  Operand reads are free of bank conflicts: the 16 lanes of a K-operand read (16
// token rows, one chunk) and the 32 lanes of a transposing V read (4 rows x 4 chunks of a
// region) fall on 16 different 16-byte bank groups each.
constexpr int kRegionBytes = 1088;
constexpr int kStageBytes = (kBlock / 4) * kRegionBytes;
// The running maximum of a column is only raised when a block's probabilities under it sum to more
// than this in a lane (half of the block's tokens): the accumulators are rescaled a handful of times per
// query instead of once per block, and blocks that need no raise (nearly all) need no maximum: with the
// board at its power cap every instruction costs time.  With a maximum per block (17 of 85 vector instructions) 16
// chunks of 512 tokens took 11245 us in 16 layers, now 10957; a chunk of 512 over 4096 946, now 933.
constexpr float kMostProbability = 256.f;
#ifndef DSKV_PREFILL_KPREFETCH
#define DSKV_PREFILL_KPREFETCH 1   // K operands of the next iteration read before its barrier (direct path)
#endif
#ifndef DSKV_PREFILL_KREADS_FIRST
#define DSKV_PREFILL_KREADS_FIRST 0
#endif

// Lane roles of the 32x32x16 MFMA, with h = lane / 32 and r = lane % 32:
//   A operand: row r, k = 8h .. 8h+7.   B operand: column r, k = 8h .. 8h+7.
//   C/D: column r, rows 8i + 4h + j in register 4i + j (i, j = 0..3).
// LDS of one workgroup: four stages of K rows, then four of V rows; at the start, 256 bytes of sixteen of each
// wave's columns from V's third stage on (beyond the stages where there are eight waves: such a
// workgroup has its compute unit to itself), at the end of all of them (16 bytes of padding between them).
constexpr int kRowPitch = 256 + 16;
constexpr int kQRowsBytes = 16 * kRowPitch, kRowsOutBytes = 32 * kRowPitch;
constexpr int prefill_lds_bytes(int waves)
{
    return 6 * kStageBytes + (waves * kQRowsBytes > 2 * kStageBytes ? waves * kQRowsBytes : 2 * kStageBytes);
}
struct LdsStages {
    char *base;
    __device__ __forceinline__ char *operator[](int i) const { return base + i * kStageBytes; }
};

// The kernel's body for workgroup `wg` of kWaves waves (a tile of kWaves * 32 / group query
// rows of one kv head); `lds`: prefill_lds_bytes(kWaves) of the workgroup's LDS.  A function, so that
// one launch can hold workgroups of this kind next to workgroups of another.
//   kStreamOut: the rows leave past the L2 (non-temporal stores), which is the launch's K/V's.  Beside
//     decode workgroups, whose own K/V stream past it, the partials of a chunk in two parts (14.5 MB)
//     pushed the chunk's K/V out of it: 75 decode rows and the chunk 2638 -> 2471 us a step (16
//     layers), 70B-shaped 1527 -> 1410.  A launch of tiles only loses (a chunk of 512 in four parts 938
//     -> 955): its merge pass then reads the partials from farther away.
//   kAppends: the launch appends the step's rows (append_rows.h); false is returned if others' did not come in
//     time, with no output stored and no block requested that holds one: append_for_tile, then again with rows_there.
struct PrefillArgs {
    AppendRows append;   // at the front: read through the kernel's argument segment
    uint16_t *out;
    const uint16_t *q;
    const int32_t *qo_indptr;
    const char *pages;
    const int32_t *kv_indices, *kv_indptr, *kv_last, *tile_info;
    int n_qo_heads, n_kv_heads, page_shift;
    float scale_log2;
    int causal;
    float *part_o, *part_ml;
    int max_slots;
    const float *rope;
};
typedef const __attribute__((address_space(4))) PrefillArgs *const_prefill_ptr;

template <int DT, bool kRowsSharePage, int kWaves, bool kStreamOut, bool kAppends = false>
__device__ __forceinline__ bool prefill_attn_body(
    char *lds_base, int wg, uint16_t *__restrict__ out, const uint16_t *__restrict__ q,
    const int32_t *__restrict__ qo_indptr, const char *__restrict__ pages,
    const int32_t *__restrict__ kv_indices, const int32_t *__restrict__ kv_indptr,
    const int32_t *__restrict__ kv_last, const int32_t *__restrict__ tile_info, int n_qo_heads,
    int n_kv_heads, int page_shift, float scale_log2, int causal,
    float *__restrict__ part_o, float *__restrict__ part_ml, int max_slots, const float *__restrict__ rope,
    int wave, bool rows_there = true)
{
    typedef Elt<DT> E;
    constexpr int kRowsPerWave = kBlock / kWaves;   // rows of a block one wave loads
    constexpr int kRowGroups = kRowsPerWave / 4;    // in groups of 4 rows (one load each)
    static_assert(kRowsPerWave % 4 == 0 && kRowGroups >= 1, "a wave loads whole groups of 4 rows");
    const LdsStages k_stage{lds_base}, v_stage{lds_base + 4 * kStageBytes};

    const int lane = kAppends ? lane_id() : threadIdx.x & 63;
    const int g = lane >> 4;     // row group / chunk roles of the K/V row movement
    const int c = lane & 15;
    const int h = lane >> 5;     // MFMA roles
    const int r = lane & 31;
    const int kvh = wg % n_kv_heads;
    const int tile = wg / n_kv_heads;
    const int group = n_qo_heads / n_kv_heads;
    const int pos_per_wave = kWaveCols / group;    // query positions per wave

    // plan entry: request, first query row of the tile within it, and the 32-token blocks
    // [blk_begin, blk_end) of the request's K/V that this workgroup walks.  Word 4 is -1 for a
    // tile that walks all of its blocks and writes its output rows itself; for a tile cut
    // into parts (blk_begin a multiple of four) it is part | parts << 8, and word 5 the
    // partial slot of the tile's first row, part 0: row r of the tile, part s, leaves
    // (maximum, sum, unnormalised O) in slot first + (r - q0) * parts + s.
    const const_i32_ptr entry = as_const(tile_info) + (long)tile * kTileWords;
    const int b = entry[0];
    const int q0 = entry[1];
    const int blk_begin = entry[2];
    const int kv_cap_blocks = entry[3];
    const int part_word = entry[4];
    const bool partial = part_word >= 0;
    const int split = part_word & 0xff, tile_parts = part_word >> 8;
    const int first_slot = entry[5];
    // (all requested before the first is looked at: the chain plan -> request -> pages -> rows is what a
    // workgroup's start lasts)
    const const_i32_ptr qo_at = as_const(qo_indptr) + b, kv_at = as_const(kv_indptr) + b;
    const int q_begin = qo_at[0], q_next = qo_at[1], page_begin = kv_at[0], page_next = kv_at[1];
    const int last_page_len = as_const(kv_last)[b];
    __builtin_amdgcn_sched_barrier(0);
    const int n_b = q_next - q_begin, n_pages = page_next - page_begin;
    const int kv_len = n_pages > 0 ? ((n_pages - 1) << page_shift) + last_page_len : 0;
    // tokens this workgroup may look at end here: the request's end, or the end of its part
    const int kv_cap = min(kv_len, kv_cap_blocks < (1 << 25) ? kv_cap_blocks * kBlock : kv_len);
    const_i32_ptr page_ids = as_const(kv_indices) + page_begin;
    const int row_bytes = n_kv_heads * kHeadDim * 2;
    const int half_bytes = row_bytes << page_shift;
    const long page_bytes = 2L * half_bytes;
    const int page_mask = (1 << page_shift) - 1;

    // column r of column tile ct: query row wq0 + (32 ct + r)/group, head (32 ct + r)%group
    const int wq0 = q0 + wave * pos_per_wave;
    int qrow[kColTiles], c_head[kColTiles], limit[kColTiles];   // limit: kv tokens the column may see
    bool live[kColTiles];
#pragma unroll
    for (int ct = 0; ct < kColTiles; ct++) {
        const int col = 32 * ct + r;
        const int c_pos = col / group;
        c_head[ct] = col - c_pos * group;
        qrow[ct] = wq0 + c_pos;
        live[ct] = c_pos < pos_per_wave && qrow[ct] < n_b;
        const int lim = causal ? kv_len - n_b + qrow[ct] + 1 : kv_len;
        limit[ct] = live[ct] ? min(max(lim, 0), kv_cap) : 0;
    }
    // The wave's q rows, whole: lane (g, c) holds chunk c of column 4 j + g, and (rope: cos | sin by query row)
    // the cosines and sines of its four dim pairs.  Loaded as the operand they become, an instruction took 32 bytes
    // of each of 32 rows, and the address path was busy with a workgroup's before it took the first K and V: three
    // short prompts 323 us in 16 layers, now 313, a chunk of 512 over 4096 918, now 908.
    // q is rotated here: a row is loaded by one workgroup per kv head and part, so this costs a workgroup 16 more
    // loads and the rotation at its start and saves the launch that read
    // and wrote all of q: for 8192 rows of 32 heads 39 us for rotating q and k and appending
    // against 15 us for the append that is left, 5.8 against 4.4 for 512 rows.
    struct QRows {
        u32x4 q[8];
        f32x4 cs[8], sn[8];
    };
    auto load_q = [&](int ct, QRows &rows) {
        // a column without a row takes the tile's first: it is not stored
        const int row = q_begin + (live[ct] ? qrow[ct] : q0), at = row * n_qo_heads + kvh * group + (live[ct] ? c_head[ct] : 0);
        int from[8], tab_row[8];
#pragma unroll
        for (int j = 0; j < 8; j++) from[j] = __shfl(at, 4 * j + g);
#pragma unroll
        for (int j = 0; j < 8; j++) rows.q[j] = *reinterpret_cast<const u32x4 *>(q + (long)from[j] * kHeadDim + c * 8);
        if (!rope) return;
#pragma unroll
        for (int j = 0; j < 8; j++) tab_row[j] = __shfl(row, 4 * j + g);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float *tab = rope + (long)tab_row[j] * kHeadDim + c * 4;
            rows.cs[j] = *reinterpret_cast<const f32x4 *>(tab);
            rows.sn[j] = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2);
        }
    };
    u32x4 qreg[kColTiles][8];     // the B operand: dims 16*ks + 8h .. +7 of the column's query
    // ... through LDS, sixteen columns at a time, in a stretch of the wave's own that is zero afterwards: V(-1) lies
    // there, which is multiplied by P(-1) = 0
    char *const q_lds = v_stage[2] + wave * kQRowsBytes;
    static_assert(prefill_lds_bytes(4) == 8 * kStageBytes && 4 * kQRowsBytes == 2 * kStageBytes, "four stretches fill two stages");
    auto finish_q = [&](int ct, QRows &rows) {
        if (rope)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const f32x4 c4 = rows.cs[j], s4 = rows.sn[j];
                const float cs[4] = {c4[0], c4[1], c4[2], c4[3]}, sn[4] = {s4[0], s4[1], s4[2], s4[3]};
                float f[8];
                Chunk<DT>::unpack(rows.q[j], f);
                rope_rotate<4>(f, cs, sn);
                rows.q[j] = Chunk<DT>::pack(f);
            }
#pragma unroll
        for (int p = 0; p < 2; p++) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<u32x4 *>(q_lds + (4 * j + g) * kRowPitch + c * 16) = rows.q[4 * p + j];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (r >> 4 == p)
#pragma unroll
                for (int ks = 0; ks < 8; ks++)
                    qreg[ct][ks] = *reinterpret_cast<const u32x4 *>(q_lds + c * kRowPitch + (2 * ks + h) * 16);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4 *>(q_lds + (i * 64 + lane) * 16) = u32x4{0, 0, 0, 0};
        static_assert(kQRowsBytes == (4 * 64 + 16) * 16, "");
        if (lane < 16) *reinterpret_cast<u32x4 *>(q_lds + (4 * 64 + lane) * 16) = u32x4{0, 0, 0, 0};
    };
    // Token ranges from scalars only: they steer loops, barriers and page lookups
    // and must be uniform for the compiler too.  The workgroup walks [0, t_end);
    // a wave computes on [0, w_end) and masks from w_mask_from on.
    const int rows_wg = min(kWaves * pos_per_wave, n_b - q0);          // >= 1 by construction
    const int t_first = blk_begin * kBlock;                                   // the walk starts here
    const int t_end = min(max(causal ? kv_len - n_b + q0 + rows_wg : kv_len, 0), kv_cap);
    const int rows_w = min(pos_per_wave, n_b - wq0);                          // <= 0: idle wave
    const int w_mask_from =
        rows_w > 0 ? min(max(causal ? kv_len - n_b + wq0 + 1 : kv_len, 0), kv_cap) : 0;
    int w_end = rows_w > 0 ? min(max(causal ? kv_len - n_b + wq0 + rows_w : kv_len, 0), kv_cap) : 0;
    if (w_end <= t_first) w_end = 0;   // nothing of this part is visible to the wave's rows: idle

    const int n_blocks = (t_end + kBlock - 1) / kBlock;
    // Start value of the running maximum: far below any scaled score, far above a
    // scaled masked score (kNegBig * scale_log2).
    float m_run[kColTiles];
    f32x16 acc[kColTiles][4];     // O^T: dims 32*dt + 8i + 4h + j of column r in acc[ct][dt][4i + j]
    float l_run[kColTiles];       // row sums of P, of the lane's half of the tokens
    u32x4 pb[2][kColTiles][2];    // packed probabilities of this block and the one before, per k-step
#pragma unroll
    for (int ct = 0; ct < kColTiles; ct++) {
        m_run[ct] = 0.5f * kNegBig * scale_log2;
        l_run[ct] = 0.f;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[ct][dt][v] = 0.f;
        pb[1][ct][0] = pb[1][ct][1] = u32x4{0, 0, 0, 0};   // P(-1)
    }

    // A tile cut into parts: every part leaves (max, sum, unnormalised O) of its rows in the
    // workspace (O blocks of all slots, then their (max, sum) pairs); a part that sees nothing
    // leaves zeros and a maximum below any real one.
    auto slot_of = [&](int ct) { return (long)first_slot + (long)(qrow[ct] - q0) * tile_parts + split; };
    auto store_max_sum = [&](int ct, float m, float l) {
        float *ml = part_ml + (slot_of(ct) * n_qo_heads + (long)kvh * group + c_head[ct]) * 2;
        ml[0] = m;
        ml[1] = l;
    };
    // The workgroup's share of the rows that the launch appends (rows_there: it has been written before).
    AppendShare<DT, kWaves> share;
    const const_append_ptr append = (const_append_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    auto append_request_share = [&]() {
        if (kAppends)
            share.request(append, tile, kvh, n_kv_heads, wave, qo_indptr, kv_indptr, kv_last, q_begin, n_b, page_begin,
                          kv_len, kv_indices, page_shift, rope);
    };
    auto append_look_up = [&]() {
        if (kAppends) share.look_up(append, wave, kv_indices, page_shift, rope);
    };
    auto append_store = [&]() {
        if (kAppends) share.store(append, pages, page_shift, row_bytes, kvh, rope != nullptr);
    };
    auto raise_flag = [&]() {   // when all waves' stores have been acknowledged
        const_append_ptr a = (const_append_ptr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(a));
        if (wave == 0 && tile < a->n_tiles && lane_id() == 0)
            __hip_atomic_store(a->flags + (long)tile * n_kv_heads + kvh, a->launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto raise_when_stored = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        raise_flag();
    };
    // No kv token of this part visible to any row of the tile: the output rows are zero
    // (or the part is empty).  Uniform over the workgroup, and before the first barrier.
    if (t_end <= t_first) {
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) {
            if (!live[ct]) continue;
            if (partial) {
                if (slot_of(ct) >= max_slots) continue;   // a slot beyond the workspace is never written
                float *o = part_o + (slot_of(ct) * n_qo_heads + (long)kvh * group + c_head[ct]) * kHeadDim + 4 * h;
#pragma unroll
                for (int i = 0; i < 16; i++) *reinterpret_cast<f32x4 *>(o + 8 * i) = f32x4{0.f, 0.f, 0.f, 0.f};
                if (h == 0) store_max_sum(ct, m_run[ct], 0.f);
                continue;
            }
            uint16_t *o = out + ((long)(q_begin + qrow[ct]) * n_qo_heads + (long)kvh * group + c_head[ct]) * kHeadDim +
                          4 * h;
#pragma unroll
            for (int i = 0; i < 16; i++) *reinterpret_cast<u32x2 *>(o + 8 * i) = u32x2{0, 0};
        }
        if (kAppends && !rows_there) {   // others may wait for its share
            append_request_share();
            append_look_up();
            append_store();
            raise_when_stored();
        }
        return true;
    }

    // A walk whose first requests would hold new rows: a plan with one is not launched this way
    // (kAppendAheadBlocks), but the lengths that count are the device's.
    if (kAppends && !rows_there && t_end > kv_len - n_b && (blk_begin + 8) * kBlock > kv_len - n_b) return false;

    // Blocks that end behind new_from hold rows that this launch appends: they are requested when the
    // flags of the workgroups that append them have been seen by every wave, and never before.
    int new_from = kAppends && !rows_there && t_end > kv_len - n_b ? kv_len - n_b : 0x7fffffff;
    int *const late = reinterpret_cast<int *>(lds_base + prefill_lds_bytes(kWaves));
    auto await_new_rows = [&]() {   // whether some wave looked in vain
        const_append_ptr a = (const_append_ptr)__builtin_amdgcn_kernarg_segment_ptr();
        const int tokens = a->tokens;
        const bool in_time = rows_are_there(a, tile, (q_begin + max(t_first - new_from, 0)) / tokens,
                                            (q_begin + min(t_end - new_from, n_b) - 1) / tokens, kvh, n_kv_heads);
        new_from = 0x7fffffff;
        if (!in_time) *late = 1;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (bare, as the loop's barriers)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        return __builtin_amdgcn_readfirstlane(*late) != 0;
    };
    if (kAppends && wave == 0) *late = 0;

    // This wave's share of the K (or V) rows of block blk: rows wave*kRowsPerWave .. +kRowsPerWave,
    // in groups of four (one region each).  Rows at or past t_end arrive as zeros (their
    // probabilities are zero, but 0 * garbage is not).
    //
    // Pages of at least four tokens (kRowsSharePage): the rows go from memory straight into
    // their LDS region (buffer_load ... lds: lane p's 16 bytes land at region + 16 p, lanes
    // beyond the descriptor's end write zeros), addressed through descriptors that end after
    // the group's last valid row.  Page ids are looked up with a vector load (every lane the
    // same entry; entries past the table read as page 0, whose descriptor is then empty).
    // Smaller pages: every lane resolves its own page, the rows pass through registers.
    typedef __attribute__((address_space(3))) void *lds_ptr;
    const int direct_off = (lane & 3) * row_bytes + kvh * (kHeadDim * 2) + (lane >> 2) * 16;
    const int lane_off = kvh * (kHeadDim * 2) + c * 16;
    // Page ids come through scalar loads (block-table entries past the table are clamped to
    // its last one; their descriptors are empty).  They are consumed at the end of an
    // iteration, when every LDS read of the iteration has been waited for anyway (scalar
    // loads and LDS reads share a counter).
    const int last_entry = max(n_pages - 1, 0);
    auto lookup_pages = [&](int blk, int(&pg)[kRowGroups]) {
        if (!kRowsSharePage) return;
#pragma unroll
        for (int i = 0; i < kRowGroups; i++) {
            const int tok0 = blk * kBlock + wave * kRowsPerWave + 4 * i;
            pg[i] = page_ids[min(tok0 >> page_shift, last_entry)];
        }
    };
    // The descriptors of the rows of block blk (scalar work: page id into an SGPR, base
    // address, valid bytes), prepared an iteration before the loads are issued so that it
    // runs in the shadow of that iteration's MFMAs.
    struct RowDesc {
        u32x4 k[kRowGroups], v[kRowGroups];   // raw buffer descriptors: base, base >> 32, bytes, flags
    };
    auto make_desc = [&](const char *base, int bytes) {
        const uint64_t a = (uint64_t)base;
        return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                     (uint32_t)__builtin_amdgcn_readfirstlane(bytes), (uint32_t)kBufferFlags};
    };
    auto prepare_rows = [&](int blk, const int(&pg)[kRowGroups], RowDesc &d) {
        if (!kRowsSharePage) return;
#pragma unroll
        for (int i = 0; i < kRowGroups; i++) {
            const int tok0 = blk * kBlock + wave * kRowsPerWave + 4 * i;
            // one page holds the 4 rows: descriptors that end after the last
            // valid row make the bounds check free and keep offsets constant
            // (the clamp is selected as a vector instruction: back to a scalar register, the
            // descriptor words must live in SGPRs)
            const int valid = __builtin_amdgcn_readfirstlane(min(max(t_end - tok0, 0), 4));
            const char *first_row = pages + (long)pg[i] * page_bytes + (long)(tok0 & page_mask) * row_bytes;
            d.k[i] = make_desc(first_row, valid * row_bytes);
            d.v[i] = make_desc(first_row + half_bytes, valid * row_bytes);
        }
    };
    auto region_of = [&](char *stage, int i) { return stage + (wave * kRowGroups + i) * kRegionBytes; };
    // Written out as instructions: through the compiler's builtin every later LDS read waits
    // for ALL of these loads (it cannot tell which region a read touches), which would undo
    // requesting them three iterations early.  What it does not know it does not wait for:
    // the waits for these loads are the explicit ones below.
    // with_new_rows: with device scope, past the XCD's L2 - whoever has read a new row's line too early, nobody here
    // meets that reading.
    // M0 is on the clobber list (the compiler reserves it, sets it itself before the few
    // instructions that read it, and must not assume that such a setting survives this one).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    auto load_direct = [&](const u32x4(&rows)[kRowGroups], char *stage, bool with_new_rows = false) {   // (a literal)
#pragma unroll
        for (int i = 0; i < kRowGroups; i++) {
            const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_ptr)region_of(stage, i);
            if (with_new_rows)
                asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen sc1 lds"
                             :
                             : "s"(lds_addr), "v"(direct_off), "s"(rows[i])
                             : "memory", "m0");
            else
                asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                             :
                             : "s"(lds_addr), "v"(direct_off), "s"(rows[i])
                             : "memory", "m0");
        }
    };
#pragma clang diagnostic pop
    auto load_rows = [&](int blk, u32x4(&k_rows)[kRowGroups], u32x4(&v_rows)[kRowGroups]) {
#pragma unroll
        for (int i = 0; i < kRowGroups; i++) {
            const int tok = blk * kBlock + wave * kRowsPerWave + 4 * i + g;
            const int tc = max(min(tok, t_end - 1), 0);
            const char *p = pages + page_ids[tc >> page_shift] * page_bytes +
                            (long)(tc & page_mask) * row_bytes + lane_off;
            const u32x4 z = {0, 0, 0, 0};
            const u32x4 got_k = *reinterpret_cast<const u32x4 *>(p);
            const u32x4 got_v = *reinterpret_cast<const u32x4 *>(p + half_bytes);
            k_rows[i] = tok < t_end ? got_k : z;
            v_rows[i] = tok < t_end ? got_v : z;
        }
    };
    auto store_rows = [&](char *stage, const u32x4(&rows)[kRowGroups]) {   // lane (g, c): chunk c of row g
#pragma unroll
        for (int i = 0; i < kRowGroups; i++)
            *reinterpret_cast<u32x4 *>(region_of(stage, i) + (c * 4 + g) * 16) = rows[i];
    };
    // Waits until at most n of this wave's vector-memory operations are outstanding (the
    // other counters of s_waitcnt left at "do not wait").
#define DSKV_WAIT_VMEM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | 0x70 | 0xF00 | (((n) >> 4) << 14))

    // Two score buffers that the iterations use in turn (S(m) is still being turned into
    // P(m) while S(m+1) is computed): the loop is unrolled with static phases, so which
    // buffer is which is known at compile time and no copy is needed.
    f32x16 xs[2][kColTiles];
    // K rows of a block as MFMA operands: token r, dims 16*ks + 8h .. +7.  With the prefetch
    // the operands of K(m+1) are read at the end of iteration m-1 (the block has been published
    // by barrier m-1 then), into the buffer that iteration m's scores use; without, all use [0].
    constexpr bool kKPrefetch = DSKV_PREFILL_KPREFETCH && kRowsSharePage;
    u32x4 ka[kKPrefetch ? 2 : 1][8];
    auto read_k_operands = [&](const char *kst, int kb = 0) {
        // token r = row r & 3 of region r >> 2; chunk 2 ks + h
        const char *k_rows = kst + (r >> 2) * kRegionBytes + h * 64 + (r & 3) * 16;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) ka[kb][ks] = *reinterpret_cast<const u32x4 *>(k_rows + ks * 128);
    };
    auto scores = [&](int buf, int kb = 0) {
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++)
#pragma unroll
            for (int v = 0; v < 16; v++) xs[buf][ct][v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
#pragma unroll
            for (int ct = 0; ct < kColTiles; ct++)
                xs[buf][ct] = E::mfma_32x32(ka[kb][ks], qreg[ct][ks], xs[buf][ct]);
    };
    // Masks block blk's scores (needed from w_mask_from on).  The empty volatile statement
    // keeps this a branch: the compiler otherwise turns it into selects that every block
    // pays for (48 vector instructions), and only the blocks on the diagonal need it.
    auto mask_scores = [&](int blk, int buf) {
        const int t = blk * kBlock;
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) {
            asm volatile("" : "+v"(xs[buf][ct]));   // (re)defined here: the selects cannot leave the branch
            int seen = limit[ct] - 4 * h - t;   // tokens of the lane's half that the column sees
            asm volatile("" : "+v"(seen));      // the sixteen comparisons hold no registers outside the branch
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (8 * (v >> 2) + (v & 3) >= seen) xs[buf][ct][v] = kNegBig;
        }
    };
    // P of k-step ks (the lane's 8 tokens of it) of the block in xs[buf] under the running maximum, packed, and
    // its sum.  A sum too large for that maximum - infinities are, too - asks for P to be taken again under a higher one.
    auto probabilities = [&](int buf, int ks, float(&p_sum)[kColTiles]) {
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) {
            float p[8];
#pragma unroll
            for (int v = 0; v < 8; v++) {
                p[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(xs[buf][ct][8 * ks + v], scale_log2, -m_run[ct]));
                p_sum[ct] = ks == 0 && v == 0 ? p[v] : p_sum[ct] + p[v];
            }
            pb[buf][ct][ks] = u32x4{E::pack2(p[0], p[1]), E::pack2(p[2], p[3]), E::pack2(p[4], p[5]), E::pack2(p[6], p[7])};
            // keeps them in their half (they are only consumed by the next iteration)
            asm volatile("" ::"v"(pb[buf][ct][ks]), "v"(p_sum[ct]));
        }
    };
    // Raises the running maximum to the block's in xs[buf] and brings what was computed under the old one
    // (accumulators, row sum) to the new scale.
    auto raise_maximum = [&](int buf) {
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) {
            const f32x16 &xc = xs[buf][ct];
            // scale_log2 > 0: the maximum can be taken before scaling
            float m = fmaxf(fmaxf(xc[0], xc[1]), xc[2]);
#pragma unroll
            for (int v = 3; v < 15; v += 2) m = fmaxf(fmaxf(m, xc[v]), xc[v + 1]);
            m = fmaxf(m, xc[15]);
            float other = m;
            swap_halves32(m, other);
            const float m_new = fmaxf(m_run[ct], fmaxf(m, other) * scale_log2);
            const float alpha = __builtin_amdgcn_exp2f(m_run[ct] - m_new);
            m_run[ct] = m_new;
            l_run[ct] *= alpha;
#pragma unroll
            for (int dt = 0; dt < 4; dt++) acc[ct][dt] *= alpha;
        }
    };

    // Iteration m of the main loop multiplies P(m-1) into V(m-1), turns S(m) into
    // P(m) and computes S(m+1), so that every MFMA of the iteration is independent
    // of its exponentials and the matrix and vector pipelines of a wave overlap.
    // Block j lives in K stage j % 4 and V stage j % 4.  Per iteration one barrier; every
    // wave runs every iteration (idle ones only move rows), so the barriers match.  The loop
    // is unrolled by four so that all stage indices are static.
    //   Direct path: iteration m requests K(m+4) and V(m+2) behind its barrier (K(m+4)
    //   replaces K(m), whose operands were read at the end of iteration m-2; V(m+2) replaces
    //   V(m-2), last read in iteration m-1).  The operands of K(m+1) are read at the END of
    //   iteration m-1, into the registers iteration m's score MFMAs use, so that those MFMAs
    //   start right behind the barrier instead of waiting for LDS (steady state +0.65 %); for
    //   that K(m+2) must have been published by barrier m: it went out two iterations
    //   earlier, and a wave makes sure that its own part of it has landed (at most 3 younger
    //   loads per row group outstanding: V(m), K(m+3), V(m+1)) before it joins that barrier.
    //   The page of block j is looked up in iteration j-6 and its descriptors are built in
    //   iteration j-5, behind that iteration's MFMAs.  (DSKV_PREFILL_KPREFETCH=0: the operands
    //   of K(m+1) are read at the start of iteration m, every request one block nearer.)
    //   Register path: the rows of block m+4 are requested in iteration m and written to
    //   LDS in iteration m+2 (one iteration is shorter than a trip to memory).
    RowDesc desc[4];              // descriptors of block j in desc[j % 4]
    int pg[4][kRowGroups];        // page ids of block j in pg[j % 4]
    struct RowSet {
        u32x4 k[kRowGroups], v[kRowGroups];   // rows on their way to LDS (register path)
    };
    RowSet even, odd;
    bool raise_later = false;
    {
        // the walk starts at block blk_begin, a multiple of four: block j still lives in stage j % 4
        QRows rows;
        if (kAppends && !rows_there) append_request_share();
        load_q(0, rows);
        auto finish_all_q = [&]() {
            finish_q(0, rows);
#pragma unroll
            for (int ct = 1; ct < kColTiles; ct++) {
                load_q(ct, rows);
                finish_q(ct, rows);
            }
        };
        if (kRowsSharePage) {
            int ahead[2][kRowGroups];   // pages of blocks 4 and 5
#pragma unroll
            for (int blk = 0; blk < 4; blk++) lookup_pages(blk_begin + blk, pg[blk]);
#pragma unroll
            for (int blk = 0; blk < 2; blk++) lookup_pages(blk_begin + 4 + blk, ahead[blk]);
            __builtin_amdgcn_sched_barrier(0);   // all six requested before the first is waited for
#pragma unroll
            for (int i = 0; i < kRowGroups; i++)   // (their sign extension otherwise waits for each of them above)
                asm volatile("" : "+s"(pg[0][i]), "+s"(pg[1][i]), "+s"(pg[2][i]), "+s"(pg[3][i]), "+s"(ahead[0][i]),
                             "+s"(ahead[1][i]));
#pragma unroll
            for (int blk = 0; blk < 4; blk++) prepare_rows(blk_begin + blk, pg[blk], desc[blk]);
#pragma unroll
            for (int blk = 0; blk < (kKPrefetch ? 4 : 3); blk++) load_direct(desc[blk].k, k_stage[blk]);
#pragma unroll
            for (int blk = 0; blk < 2; blk++) load_direct(desc[blk].v, v_stage[blk]);
            raise_later = kAppends && !rows_there;
            if (raise_later) append_look_up();
            finish_all_q();
            if (raise_later) append_store();
#pragma unroll
            for (int i = 0; i < kRowGroups; i++) {
                pg[0][i] = ahead[0][i];
                if (kKPrefetch) pg[1][i] = ahead[1][i];
            }
            if (kKPrefetch) prepare_rows(blk_begin + 4, pg[0], desc[0]);   // one block further ahead: block 4's descriptors now
            DSKV_WAIT_VMEM(2 * kRowGroups);   // everything but V(0) and V(1), which iterations 1 and 2 multiply
        } else {
            u32x4 first_k[2][kRowGroups], first_v[2][kRowGroups];
#pragma unroll
            for (int blk = 0; blk < 2; blk++) load_rows(blk_begin + blk, first_k[blk], first_v[blk]);
            finish_all_q();
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                store_rows(k_stage[blk], first_k[blk]);
                store_rows(v_stage[blk], first_v[blk]);
            }
            load_rows(blk_begin + 2, even.k, even.v);
            load_rows(blk_begin + 3, odd.k, odd.v);
        }
    }
    if (kRowsSharePage) {   // (a bare barrier: with the fences of __syncthreads V would be waited for, too)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    } else {
        __syncthreads();
    }
    if (w_end > 0) {
        read_k_operands(k_stage[0], kKPrefetch ? 1 : 0);
        scores(0, kKPrefetch ? 1 : 0);
        if ((blk_begin + 1) * kBlock > w_mask_from) mask_scores(blk_begin, 0);
        if (kKPrefetch) read_k_operands(k_stage[1], 0);   // K(blk_begin + 1) for the first iteration
    }
    // V operand: token 16 ks + 8 hi + 4 h + (c >> 2) = row c >> 2 of region 4 ks + 2 hi + h;
    // bytes 64 dt + 32 (g & 1) + 8 (c & 3) of its row = half (c & 1) of chunk 4 dt + 2 (g & 1) + ((c & 3) >> 1)
    const int v_lane_off = h * kRegionBytes + (2 * (g & 1) + ((c & 3) >> 1)) * 64 + (c >> 2) * 16 + (c & 1) * 8;
    auto iteration = [&](int m, int phase, RowSet &rows, bool with_new_rows) {   // the last and phase = m % 4 are literals at each call
        if (kRowsSharePage) {
            // this wave's rows of K(m+1) have landed; then the bare barrier: with the fences of
            // __syncthreads the compiler waits for EVERY load into LDS still on its way, which
            // is the whole point of requesting them early.  Nothing else needs the fences here:
            // the loop of this path writes LDS through these loads only, and the LDS reads of
            // the previous iteration have been consumed.
            // (the empty statements pin the compiler's order of ordinary LDS accesses around the
            // barrier, which the builtin by itself does not: the previous iteration's operand
            // reads stay above it, this iteration's below)
            DSKV_WAIT_VMEM(3 * kRowGroups);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else {
            __syncthreads();
        }
        if (kRowsSharePage && kKPrefetch) {
            lookup_pages(m + 6, pg[(phase + 2) & 3]);
            load_direct(desc[phase].k, k_stage[phase], with_new_rows);                       // K(m+4) over K(m), read in iteration m-2
            load_direct(desc[(phase + 2) & 3].v, v_stage[(phase + 2) & 3], with_new_rows);   // V(m+2)
        } else if (kRowsSharePage) {
            lookup_pages(m + 5, pg[(phase + 1) & 3]);
            load_direct(desc[(phase + 3) & 3].k, k_stage[(phase + 3) & 3]);   // K(m+3)
            load_direct(desc[(phase + 2) & 3].v, v_stage[(phase + 2) & 3]);   // V(m+2)
        } else {
            store_rows(k_stage[(phase + 2) & 3], rows.k);                     // K(m+2)
            store_rows(v_stage[(phase + 2) & 3], rows.v);                     // V(m+2)
            load_rows(m + 4, rows.k, rows.v);
        }
        if (!(w_end > 0 && (m - 1) * kBlock < w_end)) {
            if (kKPrefetch) prepare_rows(m + 5, pg[(phase + 1) & 3], desc[(phase + 1) & 3]);
            else prepare_rows(m + 4, pg[phase], desc[phase]);
            return;
        }
        // The rest of the iteration is two straight-line halves, each an MFMA
        // strand with independent vector and LDS work in its shadow:
        //   S(m+1) = K(m+1).Q^T     |  half of P(m) = exp2(S(m) * scale - max), packed; V(m-1) operands from LDS
        //   O += P(m-1).V(m-1)      |  the other half; row sum; K(m+2) operands from LDS
        // with, where needed, the masking of S(m+1) between them and the raise of the maximum behind them.  (The
        // waves of a unit go through the halves together: with all of P(m) in the first, that one was bound by the
        // exponentials and the other by the matrix pipeline.  Three short prompts 312 -> 307 us in 16 layers, a chunk of
        // 512 942 -> 933, 16 chunks 11579 -> 11431.)  A masked score
        // is kNegBig and the maximum never drops below its start value, so masked
        // probabilities come out as exp2(-huge) = 0 without a select.
        const int cur = phase & 1, nxt = cur ^ 1;   // xs[cur] = S(m), xs[nxt] receives S(m+1)
        // V operand: the transposing read hands each block of 16 lanes four tokens
        // of 16 consecutive dims, lane i of the block supplying the address of dims
        // 4*(i%4) .. +3 of the block's token i/4
        if (!kKPrefetch) read_k_operands(k_stage[(phase + 1) & 3]);      // K(m+1)
#if DSKV_PREFILL_KREADS_FIRST
        __builtin_amdgcn_sched_barrier(0);   // all eight K operands requested before anything else
#endif
        const char *v_rows = v_stage[(phase + 3) & 3] + v_lane_off;        // V(m-1)
        u32x4 va[4][2];
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const char *vp = v_rows + ks * 4 * kRegionBytes + dt * 256;
                const u32x2 a_lo = read_transposed(vp);
                const u32x2 a_hi = read_transposed(vp + 2 * kRegionBytes);
                va[dt][ks] = u32x4{a_lo.x, a_lo.y, a_hi.x, a_hi.y};
            }
        scores(nxt, kKPrefetch ? (phase & 1) : 0);
        float p_sum[kColTiles];
        probabilities(cur, 0, p_sum);
        if ((m + 2) * kBlock > w_mask_from) mask_scores(m + 1, nxt);   // wave-uniform

#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int ct = 0; ct < kColTiles; ct++)
                    acc[ct][dt] = E::mfma_32x32(va[dt][ks], pb[nxt][ct][ks], acc[ct][dt]);   // P(m-1): the other buffer
        if (kKPrefetch) read_k_operands(k_stage[(phase + 2) & 3], (phase + 1) & 1);   // K(m+2), published by this iteration's barrier
        probabilities(cur, 1, p_sum);
        if (kKPrefetch) prepare_rows(m + 5, pg[(phase + 1) & 3], desc[(phase + 1) & 3]);
        else prepare_rows(m + 4, pg[phase], desc[phase]);   // for the loads of the next iterations
        bool over = false;
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) over |= p_sum[ct] > kMostProbability;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(over) != 0, 0)) {   // rare
            raise_maximum(cur);
            __builtin_amdgcn_sched_barrier(0);   // one after the other: side by side they spill
            probabilities(cur, 0, p_sum);
            probabilities(cur, 1, p_sum);
        }
#pragma unroll
        for (int ct = 0; ct < kColTiles; ct++) l_run[ct] += p_sum[ct];
    };
    // The four iterations from m on request blocks up to m + 7.  The walk is cut where they would first meet a
    // new row, so that the loop itself has nothing to look at; what is behind the cut is a loop of its own, with
    // device scope (a chunk of 512 over 4096 takes the same 880 us either way; with a scalar branch at each load
    // of one loop 889).
    for (int m = blk_begin;;) {
        int end = n_blocks + 1;
        const bool raise_now = kAppends && raise_later, wait_now = kAppends && !raise_now && new_from < 0x7fffffff;
        // The share's stores are older than the loads that three waits of `iteration` leave on their way:
        // behind the barriers of the first four iterations they have been acknowledged for all waves.
        if (raise_now) end = min(end, m + 4);
        if (wait_now) end = min(end, m + max(new_from / kBlock - 8 - m + 4, 0) / 4 * 4);
        for (; m < end; m += 4) {
            iteration(m, 0, even, false);
            iteration(m + 1, 1, odd, false);
            iteration(m + 2, 2, even, false);
            iteration(m + 3, 3, odd, false);
        }
        if (!kAppends) break;
        if (raise_now) {
            raise_flag();
            raise_later = false;
        }
        if (m > n_blocks) break;
        if (wait_now) {
            if (await_new_rows()) break;
            for (; m <= n_blocks; m += 4) {
                iteration(m, 0, even, true);
                iteration(m + 1, 1, odd, true);
                iteration(m + 2, 2, even, true);
                iteration(m + 3, 3, odd, true);
            }
            break;
        }
    }
    if (kRowsSharePage) DSKV_WAIT_VMEM(0);   // nothing of this wave may still be on its way into LDS
#undef DSKV_WAIT_VMEM

    // The rows leave through LDS, a stretch of the stages per wave: a lane holds four dims here and
    // four there of one column, and stored from the registers every instruction touched 32 rows,
    // 16 bytes (of the 16-bit output) or 32 (of a partial) of each.  Laid out by column, 16 lanes
    // store 256 consecutive bytes: the launch of three short prompts 17.5 -> 15.3 us, the step of a
    // chunk of 512 tokens in four parts (16 layers) 944 -> 920.
    __syncthreads();   // the stages have been read by everybody
    if (kAppends && __builtin_amdgcn_readfirstlane(*late)) return false;
    char *const rows_lds = lds_base + wave * kRowsOutBytes;
    static_assert(kWaves * kRowsOutBytes <= prefill_lds_bytes(kWaves), "a stretch per wave");
    // 256 bytes of every column from rows_lds to base + row * row_bytes + at, `row` being the lane's own
    // column's row there (negative: none); any lane may hold any column's bytes
    auto store_columns = [&](char *base, int row, int row_bytes, int at) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int col = 4 * j + g, to = __shfl(row, col);
            const u32x4 w = *reinterpret_cast<const u32x4 *>(rows_lds + col * kRowPitch + c * 16);
            if (to < 0) continue;
            u32x4 *const dst = reinterpret_cast<u32x4 *>(base + (long)to * row_bytes + at + c * 16);
            if (kStreamOut) __builtin_nontemporal_store(w, dst);
            else *dst = w;
        }
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int ct = 0; ct < kColTiles; ct++) {
        float l_other = l_run[ct];
        swap_halves32(l_run[ct], l_other);
        const float l = l_run[ct] + l_other;
        char *const mine = rows_lds + r * kRowPitch;
        if (partial) {   // (max, sum, unnormalised O) of the row into its slot, 64 dims at a time
            const int slot = (qrow[ct] - q0) * tile_parts + split, qh = kvh * group + c_head[ct];   // from first_slot
            const bool held = live[ct] && first_slot + (long)slot < max_slots;   // never beyond the workspace
            char *const o = reinterpret_cast<char *>(part_o + (long)first_slot * n_qo_heads * kHeadDim);
#pragma unroll
            for (int half = 0; half < 2; half++) {
#pragma unroll
                for (int dt = 0; dt < 2; dt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const f32x16 &a = acc[ct][2 * half + dt];
                        *reinterpret_cast<f32x4 *>(mine + (dt * 32 + 8 * i + 4 * h) * 4) =
                            f32x4{a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]};
                    }
                store_columns(o, held ? slot * n_qo_heads + qh : -1, kHeadDim * 4, half * 256);
            }
            if (held && h == 0) store_max_sum(ct, m_run[ct], l);
            continue;
        }
        const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                *reinterpret_cast<u32x2 *>(mine + (dt * 32 + 8 * i + 4 * h) * 2) =
                    u32x2{E::pack2(acc[ct][dt][4 * i] * inv, acc[ct][dt][4 * i + 1] * inv),
                          E::pack2(acc[ct][dt][4 * i + 2] * inv, acc[ct][dt][4 * i + 3] * inv)};
        store_columns(reinterpret_cast<char *>(out + ((long)(q_begin + q0) * n_qo_heads + (long)kvh * group) * kHeadDim),
                      live[ct] ? (qrow[ct] - q0) * n_qo_heads + c_head[ct] : -1, kHeadDim * 2, 0);
    }
    return true;
}

// A walk that ended before a block with new rows: its workgroup leaves its share of the launch's rows, in case the
// walk had not come to that, and appends all of its request's of its kv head.
template <int DT, int kWaves>
__device__ __forceinline__ void append_for_tile(const_prefill_ptr a, int wg, int wave)
{
    asm volatile("" : "+s"(a));
    const const_append_ptr append = (const_append_ptr)a;
    const int n_kv_heads = a->n_kv_heads, page_shift = a->page_shift, tile = wg / n_kv_heads, kvh = wg % n_kv_heads;
    const int b = a->tile_info[(long)tile * kTileWords];
    const int q_begin = a->qo_indptr[b], n_b = a->qo_indptr[b + 1] - q_begin;
    const int page_begin = a->kv_indptr[b];   // it has pages: the tile sees tokens
    const int kv_len = ((a->kv_indptr[b + 1] - page_begin - 1) << page_shift) + a->kv_last[b];
    AppendShare<DT, kWaves> share;
    share.request(append, tile, kvh, n_kv_heads, wave, a->qo_indptr, a->kv_indptr, a->kv_last, q_begin, n_b, page_begin,
                  kv_len, a->kv_indices, page_shift, a->rope);
    share.look_up(append, wave, a->kv_indices, page_shift, a->rope);
    share.store(append, a->pages, page_shift, n_kv_heads * kHeadDim * 2, kvh, a->rope != nullptr);
    append_request<DT, kWaves>(a->append.k, a->append.v, a->append.num_pages, q_begin, n_b, kv_len, a->pages,
                               a->kv_indices + page_begin, kvh, n_kv_heads, page_shift, a->rope, wave);
    if (wave > 0 || lane_id() > 0) return;
    __hip_atomic_fetch_add(a->append.flags + kAppendFlags, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tile < a->append.n_tiles)
        __hip_atomic_store(a->append.flags + (long)tile * n_kv_heads + kvh, a->append.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#ifndef DSKV_PREFILL_MIN_WAVES
#define DSKV_PREFILL_MIN_WAVES 1
#endif
template <int DT, bool kRowsSharePage, bool kAppends>
__global__ __launch_bounds__(64 * kPrefillWaves, DSKV_PREFILL_MIN_WAVES) void prefill_attn_mfma_kernel(const PrefillArgs a)
{
    static_assert(kRowsSharePage || !kAppends, "the register path's rows are in their pages before");
    __shared__ __align__(16) char lds[prefill_lds_bytes(kPrefillWaves) + (kAppends ? 16 : 0)];
    int wg = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (!kAppends) {
        prefill_attn_body<DT, kRowsSharePage, kPrefillWaves, false>(
            lds, wg, a.out, a.q, a.qo_indptr, a.pages, a.kv_indices, a.kv_indptr, a.kv_last, a.tile_info, a.n_qo_heads,
            a.n_kv_heads, a.page_shift, a.scale_log2, a.causal, a.part_o, a.part_ml, a.max_slots, a.rope, wave);
        return;
    }
    // Every walk reads the arguments anew: nothing is kept in registers for a second one, which hardly ever comes.
    for (bool rows_there = false;; rows_there = true) {
        const_prefill_ptr p = (const_prefill_ptr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p), "+s"(wg));
        if (prefill_attn_body<DT, kRowsSharePage, kPrefillWaves, false, kAppends>(
                lds, wg, p->out, p->q, p->qo_indptr, p->pages, p->kv_indices, p->kv_indptr, p->kv_last, p->tile_info,
                p->n_qo_heads, p->n_kv_heads, p->page_shift, p->scale_log2, p->causal, p->part_o, p->part_ml, p->max_slots,
                p->rope, wave, rows_there))
            return;
        append_for_tile<DT, kPrefillWaves>(p, wg, wave);
    }
}

}  // namespace dskv
