// The 16-bit decode attention kernel (head_dim 128) for batches that cannot give every compute
// unit a share of the work: one workgroup per (share, kv head), whose eight waves split the
// share's tiles.  See decode_attn.hip for the rule that picks it.
//
// What bounds it: latency.  A step over 7 MB of K/V (one request of 1777 tokens) needs 1 us of
// HBM time; what lasts is the chain plan -> page id -> tile -> result and everything that hangs
// behind it.  With workgroups of one wave per kv head (decode_kernel.h) that request is cut into
// 28 parts of four tiles, walked one after the other, and merged by a second launch that takes
// nearly as long (14.5 + 11.3 us by rocprofv3; 20.5 us per layer in a replayed graph).  Here a wave
// walks one tile or two, eight waves meet in LDS, the request has 18 parts, and the part that
// finishes last merges them in the same launch: 13.1 us.  8 requests of 512 tokens: 19.3 -> 13.0 us,
// 8 of 300-1100: 24.3 -> 14.7, 24 of 64-2048: 35 -> 28.
//
// A wave owns a slice of the share's tile stream, which may cross requests: the pieces it
// computes are whole items (it writes them itself), or the two ends of items that reach into its
// neighbours' slices (they meet in LDS, behind the workgroup's only barrier).
#pragma once

#include "decode_kernel.h"

namespace dskv {

constexpr int kSplitWaves = 8;
// K by whole rows (TileRegs): all waves request their tiles at once, at the start, and the address path is
// through with the requests sooner: 8 requests of 300-1100, 16 layers replayed, 277.1 -> 270.4 us.
constexpr bool kSplitWholeRows = true;
constexpr int kSplitRing = 2;        // tiles in flight per wave: a wave rarely has more
// The planner's rule, measured there: tiles of a batch at most (one kv head: at least), tiles of a
// share at least, and parts of one request that make a batch lopsided.
constexpr int kSplitMaxTiles = 2560, kSplitMinTilesOneHead = 5000, kSplitTilesPerShare = 6, kLopsidedParts = 64;
constexpr int kSplitMaxGroup = 8;    // q heads per kv head, at most (LDS for the pieces that meet)
// LDS: the waves' V tiles; two meeting places per wave ([0] a piece that continues an item of an
// earlier wave, [1] one that a later wave continues) of O and (m, l) per q head; the new token's
// K and V row per wave; the owner of each [0] piece, and what to do with each item that meets.
constexpr int kSplitPieceFloats = kSplitMaxGroup * kHeadDim;
struct SplitShared {
    char tiles[kSplitWaves * tile_lds_bytes(kSplitWholeRows)];
    float o[kSplitWaves][2][kSplitPieceFloats];
    float ml[kSplitWaves][2][kSplitMaxGroup][2];
    uint32_t new_row[kSplitWaves][2][kHeadDim / 2];
    int owner[kSplitWaves];          // wave that holds the item's first piece (-1: no such piece)
    int meet_row[kSplitWaves], meet_slot[kSplitWaves];   // item whose first piece is wave w's (row -1: none)
    int last[2];                     // this part completed the set (the share's first, last item)
};

// ---- Partials that other compute units read in the same launch.
//
// The parts of a cut request are merged by whoever finishes last: every part stores its
// partial, waits until the stores are acknowledged and counts itself in; the one that completes
// the count reads all parts and writes the output row.  No fence is involved: partials are
// stored and read as relaxed atomics of device scope (written through, and read past the L2 of
// the XCD), so nothing else in the caches has to be written back or dropped - release / acquire
// fences write back the whole L2.  The counter is set back to zero by the last one, ready for
// the next launch.
__device__ __forceinline__ void put2(float *p, f32x2 v)
{
    __hip_atomic_store(reinterpret_cast<uint64_t *>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x2 get2(const float *p)
{
    return __builtin_bit_cast(f32x2, __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void put4(float *p, f32x4 v)
{
    put2(p, f32x2{v[0], v[1]});
    put2(p + 2, f32x2{v[2], v[3]});
}
__device__ __forceinline__ f32x4 get4(const float *p)
{
    const f32x2 a = get2(p), b = get2(p + 2);
    return f32x4{a.x, a.y, b.x, b.y};
}
// Counts one part in; to be called by one lane.  True for the part that completes the set.
__device__ __forceinline__ bool arrive_last(uint32_t *counter, int parts)
{
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = before + 1 == (uint32_t)parts;
    if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return last;
}
// Dims d0 .. d0 + 3 of q head qh merged over `parts` consecutive slots, kAtOnce of them requested
// per trip to memory under a running maximum: their sum under maximum m, l the sum of weights.
template <int kAtOnce>
__device__ __forceinline__ f32x4 merge_slots(float *part_o, float *part_ml, int first, int parts,
                                             int n_qo_heads, int qh, int d0, float &m, float &l)
{
    m = kNegBig;
    l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < parts; i0 += kAtOnce) {
        f32x4 o[kAtOnce];
        f32x2 ml[kAtOnce];   // (maximum, sum)
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const long slot = first + min(i0 + i, parts - 1);   // past the last: it again, weight zero
            ml[i] = get2(part_ml + (slot * n_qo_heads + qh) * 2);
            o[i] = get4(part_o + (slot * n_qo_heads + qh) * kHeadDim + d0);
        }
        float m_new = m;
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) m_new = fmaxf(m_new, ml[i].x);
        const float keep = __builtin_amdgcn_exp2f(m - m_new);
        l *= keep;
        acc *= keep;
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const float w = i0 + i < parts ? __builtin_amdgcn_exp2f(ml[i].x - m_new) : 0.f;
            l += w * ml[i].y;
            acc += w * o[i];
        }
        m = m_new;
    }
    return acc;
}

struct SplitArgs {
    uint16_t *out;
    const uint16_t *q;
    const char *pages;
    const int32_t *kv_indices;
    const Item *items;
    const int32_t *wg_ptr;
    float *part_o, *part_ml;
    int max_slots, n_qo_heads, n_kv_heads, page_shift;
    float scale_log2;
    const uint16_t *k_new, *v_new;   // null: the newest tokens are in the pages already
    const float *rope;               // null: q and k_new are not to be rotated
    uint32_t *counters;              // one zeroed word per (partial slot, kv head); null: a merge launch follows
    int n_counters, n_shares;
};

// A workgroup fills its compute unit's LDS, so what counts is that the workgroups spread evenly: ids go
// round the 8 XCDs, and without gaps in them no XCD gets more than its 32, whatever the number of
// heads.  (The heads of a share need not meet on an XCD: they read other bytes of the same pages.)
template <int DT, int kPagesPerTile>
__global__ __launch_bounds__(64 * kSplitWaves) void decode_attn_split_kernel(const SplitArgs a)
{
    typedef Elt<DT> E;
    constexpr bool kPageCoversTile = kPagesPerTile == 1, kWholeRows = kSplitWholeRows;
    __shared__ __align__(16) SplitShared sh;
    const int share = (int)blockIdx.x % a.n_shares, kvh = (int)blockIdx.x / a.n_shares;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int group = a.n_qo_heads / a.n_kv_heads;
    const const_i32_ptr item_words = as_const(reinterpret_cast<const int32_t *>(a.items));
    const const_i32_ptr indices_c = as_const(a.kv_indices);
    const int item_begin = as_const(a.wg_ptr)[share], item_end = as_const(a.wg_ptr)[share + 1];
    if (item_begin >= item_end) return;

    // ---- this wave's slice of the share's tiles, and the items it meets
    auto tiles_of = [](int begin, int end) { return (end - begin + kTile - 1) / kTile; };
    const const_i32_ptr last_words = item_words + (long)(item_end - 1) * kItemWords;
    const int total = last_words[7] + tiles_of(last_words[1], last_words[2]);
    const int lo = total * wave / kSplitWaves, hi = total * (wave + 1) / kSplitWaves;   // tiles of the share
    int first_item = item_end, end_item = item_begin;
    for (int idx = item_begin; idx < item_end; idx++) {
        const const_i32_ptr w = item_words + (long)idx * kItemWords;
        const int at = w[7], n = tiles_of(w[1], w[2]);
        if (n == 0) {
            // a request without tokens: a row of zeros
            if (wave == 0)
                for (int i = lane * 8; i < group * kHeadDim; i += 64 * 8)
                    *reinterpret_cast<u32x4 *>(a.out + ((long)w[0] * a.n_qo_heads + (long)kvh * group) * kHeadDim + i) =
                        u32x4{0, 0, 0, 0};
        } else if (at < hi && at + n > lo) {
            first_item = min(first_item, idx);
            end_item = idx + 1;
        }
    }
    struct Piece {
        int b, tok_begin, tok_end, slot, page_begin;
        bool tail;        // holds the request's newest token
        bool starts, ends;   // the item starts / ends in this wave's slice
        int at;           // the item's first tile within the share
    };
    auto load_piece = [&](int idx) {
        const const_i32_ptr w = item_words + (long)idx * kItemWords;
        const int begin = w[1], end = w[2], at = w[7];
        Piece p;
        p.b = w[0];
        p.tok_begin = max(begin, begin + (lo - at) * kTile);
        p.tok_end = min(end, begin + (hi - at) * kTile);
        p.slot = w[3];
        p.page_begin = w[4];
        p.starts = at >= lo;
        p.ends = p.tok_end == end;
        p.tail = w[5] && p.ends;
        if (p.tok_end <= p.tok_begin) {   // not this wave's, or without tokens
            p.tok_end = p.tok_begin;
            p.tail = false;
        }
        p.at = at;
        return p;
    };

    KvView kv;
    kv.pages = a.pages;
    kv.page_ids = indices_c;
    kv.page_shift = a.page_shift;
    kv.row_bytes = a.n_kv_heads * kHeadDim * 2;
    kv.half_bytes = kv.row_bytes << a.page_shift;
    kv.page_bytes = 2L * kv.half_bytes;
    kv.head_off = kvh * (kHeadDim * 2);
    char *tile_lds = sh.tiles + wave * tile_lds_bytes(kSplitWholeRows);
    uint32_t *new_k = sh.new_row[wave][0], *new_v = sh.new_row[wave][1];

    // ---- what a piece needs besides its tiles: the q rows as the B operand of the score MFMAs
    // (zero beyond the group), their cosines and sines, and the new token's rows (lanes 0-15: K,
    // 16-31: V; lanes 0-15 also the cosines and sines of their chunk).
    struct Raw {
        u32x4 q[4], fresh;
        f32x4 cs[4], sn[4], fresh_cs, fresh_sn;
    };
    auto request = [&](const Piece &p, Raw &r) {
        const uint16_t *qrow = a.q + ((long)p.b * a.n_qo_heads + (long)kvh * group + c) * kHeadDim + g * 8;
        const u32x4 z = {0, 0, 0, 0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) r.q[kk] = c < group ? *reinterpret_cast<const u32x4 *>(qrow + kk * 32) : z;
        const float *tab = a.rope + (long)p.b * kHeadDim;
        if (a.rope) {   // dims 32*kk + 8*g .. +7
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                r.cs[kk] = *reinterpret_cast<const f32x4 *>(tab + g * 4 + kk * 16);
                r.sn[kk] = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2 + g * 4 + kk * 16);
            }
        }
        r.fresh = z;
        if (a.k_new && p.tail && lane < 32) {
            const long src = ((long)p.b * a.n_kv_heads + kvh) * kHeadDim + c * 8;
            r.fresh = *reinterpret_cast<const u32x4 *>((lane < 16 ? a.k_new : a.v_new) + src);
            if (a.rope && lane < 16) {
                r.fresh_cs = *reinterpret_cast<const f32x4 *>(tab + c * 4);
                r.fresh_sn = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2 + c * 4);
            }
        }
    };
    auto rotate = [&](u32x4 chunk, const f32x4 &cs, const f32x4 &sn) {
        const float c4[4] = {cs[0], cs[1], cs[2], cs[3]}, s4[4] = {sn[0], sn[1], sn[2], sn[3]};
        float f[8];
        Chunk<DT>::unpack(chunk, f);
        rope_rotate<4>(f, c4, s4);
        return Chunk<DT>::pack(f);
    };
    // Writes the new token's rows into their page slot, and into LDS, from where the tile that
    // holds them takes them: nobody waits for the page to have them.
    auto place_new_row = [&](const Piece &p, const Raw &r) {
        const int tok = p.tok_end - 1;
        const long page = indices_c[p.page_begin + (tok >> a.page_shift)];
        char *row = const_cast<char *>(a.pages) + page * kv.page_bytes +
                    (long)(tok & ((1 << a.page_shift) - 1)) * kv.row_bytes + kv.head_off + c * 16;
        if (lane < 32) {
            u32x4 chunk = r.fresh;
            if (a.rope && lane < 16) chunk = rotate(chunk, r.fresh_cs, r.fresh_sn);
            *reinterpret_cast<u32x4 *>(row + (lane < 16 ? 0 : kv.half_bytes)) = chunk;
            *reinterpret_cast<u32x4 *>((lane < 16 ? new_k : new_v) + c * 4) = chunk;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    // ---- load side: runs ahead of the compute side through the wave's pieces
    int next_item = first_item, t = 0, t_end = 0, t_pad_end = 0;
    long page[2] = {0, 0};
    auto settle = [&]() {
        while (t >= t_pad_end && next_item < end_item) {
            const Piece p = load_piece(next_item++);
            t = p.tok_begin;
            t_end = p.tok_end;
            t_pad_end = t + (tiles_of(t, t_end) + kSplitRing - 1) / kSplitRing * kSplitRing * kTile;
            kv.page_ids = indices_c + p.page_begin;
        }
        if (t >= t_pad_end) t_end = 0;   // exhausted: every further tile is empty and reads no block table
        if (kPagesPerTile >= 1)
#pragma unroll
            for (int j = 0; j < kPagesPerTile; j++)
                page[j] = t_end > 0 ? kv.page_ids[page_slot_of(kv, t + (j << kv.page_shift), t_end)] : 0;
    };
    auto load_next = [&](TileRegs &r) {
        if (kPageCoversTile) {
            load_kv_tile_in_page<kLoadStreaming, kWholeRows>(kv, page[0], t, t_end, g, c, r);
        } else if (kPagesPerTile == 2) {
            load_kv_tile_small_pages<2, kLoadStreaming, kWholeRows>(kv, page, t, t_end, g, c, r);
        } else {
            load_kv_tile<false, kLoadStreaming, kWholeRows>(kv, t, t_end, g, c, r);
        }
        t += kTile;
        settle();
    };

    if (lane == 0) {
        sh.owner[wave] = -1;
        sh.meet_row[wave] = -1;
    }
    if (first_item < end_item) {
        Piece piece = load_piece(first_item);
        Raw raw;
        request(piece, raw);
        settle();
        TileRegs ring[kSplitRing];
#pragma unroll
        for (int s = 0; s < kSplitRing; s++) load_next(ring[s]);

        for (int idx = first_item; idx < end_item; idx++) {
            u32x4 qreg[4];
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                qreg[kk] = raw.q[kk];
                if (a.rope) qreg[kk] = rotate(raw.q[kk], raw.cs[kk], raw.sn[kk]);
            }
            const bool fresh = a.k_new && piece.tail;
            if (fresh) place_new_row(piece, raw);
            const Piece next = load_piece(min(idx + 1, end_item - 1));
            if (idx + 1 < end_item) request(next, raw);

            f32x4 acc[8];
#pragma unroll
            for (int dt = 0; dt < 8; dt++) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            float m_run = kNegBig, l_run = 0.f;
            auto compute_tile = [&](int t0, TileRegs &r) {
                const int end = piece.tok_end;
                if (fresh && t0 + kTile >= end) {
                    // the newest token is this tile's row nr, and the page may not have it yet
                    const int nr = end - 1 - t0;
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) {
                        if (kWholeRows && g + 4 * kk == nr) r.k[kk] = *reinterpret_cast<const u32x4 *>(new_k + c * 4);
                        if (!kWholeRows && c == nr) r.k[kk] = *reinterpret_cast<const u32x4 *>(new_k + kk * 16 + g * 4);
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (g + 4 * i == nr) r.v[i] = *reinterpret_cast<const u32x4 *>(new_v + c * 4);
                }
                if (kWholeRows) stage_k_tile(tile_lds, r, g, c);
                f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < 4; kk++)
                    s = E::mfma_k32(kWholeRows ? read_k_operand(tile_lds, kk, g, c) : r.k[kk], qreg[kk], s);
                const bool ragged = t0 + kTile > end;
                float x[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    x[j] = s[j] * a.scale_log2;
                    if (ragged && t0 + 4 * g + j >= end) x[j] = kNegBig;
                }
                stage_v_tile<kPageCoversTile>(tile_lds, r, t0, end, g, c);
                const float m_new = fmaxf(m_run, quad_rows_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                float p[4], p_sum = 0.f;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    p[j] = x[j] > kNegBig ? __builtin_amdgcn_exp2f(x[j] - m_new) : 0.f;
                    p_sum += p[j];
                }
                l_run = l_run * alpha + p_sum;
                const u32x2 pb = {E::pack2(p[0], p[1]), E::pack2(p[2], p[3])};
#pragma unroll
                for (int dt = 0; dt < 8; dt++)
                    acc[dt] = E::mfma_k16(read_v_operand(tile_lds, dt, g, c), pb, acc[dt] * alpha);
                __builtin_amdgcn_wave_barrier();
            };
            const int pad_end = piece.tok_begin +
                                (tiles_of(piece.tok_begin, piece.tok_end) + kSplitRing - 1) / kSplitRing * kSplitRing * kTile;
            for (int t0 = piece.tok_begin; t0 < pad_end; t0 += kSplitRing * kTile) {
#pragma unroll
                for (int s = 0; s < kSplitRing; s++) {
                    if (t0 + s * kTile < piece.tok_end) compute_tile(t0 + s * kTile, ring[s]);
                    __builtin_amdgcn_sched_barrier(0);
                    load_next(ring[s]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            l_run = quad_rows_sum(l_run);
            if (piece.tok_end > piece.tok_begin) {
                if (piece.starts && piece.ends) {   // a whole item
                    if (c < group) {
                        const int qh = kvh * group + c;
                        if (piece.slot < 0) {
                            const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
                            uint16_t *o = a.out + ((long)piece.b * a.n_qo_heads + qh) * kHeadDim + 4 * g;
#pragma unroll
                            for (int dt = 0; dt < 8; dt++)
                                *reinterpret_cast<u32x2 *>(o + dt * 16) =
                                    u32x2{E::pack2(acc[dt][0] * inv, acc[dt][1] * inv),
                                          E::pack2(acc[dt][2] * inv, acc[dt][3] * inv)};
                        } else if (piece.slot < a.max_slots) {   // a slot beyond the workspace is never written
                            const long at = (long)piece.slot * a.n_qo_heads + qh;
#pragma unroll
                            for (int dt = 0; dt < 8; dt++) put4(a.part_o + at * kHeadDim + dt * 16 + 4 * g, acc[dt]);
                            if (g == 0) put2(a.part_ml + at * 2, f32x2{m_run, l_run});
                        }
                    }
                } else {   // one end of an item that other waves share
                    const int place = piece.starts ? 1 : 0;
                    if (c < group) {
                        float *o = sh.o[wave][place] + c * kHeadDim + 4 * g;
#pragma unroll
                        for (int dt = 0; dt < 8; dt++) *reinterpret_cast<f32x4 *>(o + dt * 16) = acc[dt];
                        if (g == 0) {
                            sh.ml[wave][place][c][0] = m_run;
                            sh.ml[wave][place][c][1] = l_run;
                        }
                    }
                    if (lane == 0) {
                        if (piece.starts) {
                            sh.meet_row[wave] = piece.b;
                            sh.meet_slot[wave] = piece.slot;
                        } else {
                            // the wave whose slice holds the item's first tile
                            int o = wave - 1;
                            while (total * o / kSplitWaves > piece.at) o--;
                            sh.owner[wave] = o;
                        }
                    }
                }
            }
            piece = next;
        }
    }

    // ---- the items that meet: a thread owns four values
    __syncthreads();
    const int per_item = group * (kHeadDim / 4), side_by_side = 64 * kSplitWaves / per_item;
    const int mine = (int)threadIdx.x / per_item, idx4 = (int)threadIdx.x % per_item;
    const int head = idx4 / (kHeadDim / 4), qh = kvh * group + head, d0 = idx4 % (kHeadDim / 4) * 4;
    if (mine < side_by_side) {
        for (int e = mine; e < kSplitWaves; e += side_by_side) {
            const int row = sh.meet_row[e], slot = sh.meet_slot[e];
            if (row < 0) continue;
            float m_all = sh.ml[e][1][head][0];
            for (int w = e + 1; w < kSplitWaves; w++)
                if (sh.owner[w] == e) m_all = fmaxf(m_all, sh.ml[w][0][head][0]);
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
            float l_all = 0.f;
            for (int w = e; w < kSplitWaves; w++) {
                if (w > e && sh.owner[w] != e) continue;
                const int place = w == e ? 1 : 0;
                const float weight = __builtin_amdgcn_exp2f(sh.ml[w][place][head][0] - m_all);
                l_all += weight * sh.ml[w][place][head][1];
                sum += weight * *reinterpret_cast<const f32x4 *>(sh.o[w][place] + head * kHeadDim + d0);
            }
            if (slot < 0) {
                const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
                *reinterpret_cast<u32x2 *>(a.out + ((long)row * a.n_qo_heads + qh) * kHeadDim + d0) =
                    u32x2{E::pack2(sum[0] * inv, sum[1] * inv), E::pack2(sum[2] * inv, sum[3] * inv)};
            } else if (slot < a.max_slots) {
                const long at = (long)slot * a.n_qo_heads + qh;
                put4(a.part_o + at * kHeadDim + d0, sum);
                if (d0 == 0) put2(a.part_ml + at * 2, f32x2{m_all, l_all});
            }
        }
    }

    // ---- the parts of cut requests.  Only the first and the last item of a share can be parts
    // (the shares' boundaries cut); both are counted in, and merged, side by side.
    if (!a.counters) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the partials are where other XCDs see them
    int row[2], first[2], parts[2];
    bool cut[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const const_i32_ptr w = item_words + (long)(k ? item_end - 1 : item_begin) * kItemWords;
        row[k] = w[0];
        first[k] = w[6] >> kPartsBits;
        parts[k] = w[6] & ((1 << kPartsBits) - 1);
        cut[k] = w[3] >= 0 && parts[k] > 0 && first[k] + parts[k] <= a.max_slots &&
                 (long)first[k] * a.n_kv_heads + kvh < a.n_counters && !(k && item_end - 1 == item_begin);
    }
    if (!cut[0] && !cut[1]) return;
    __syncthreads();
    if (wave < 2 && lane == 0)
        sh.last[wave] = cut[wave] && arrive_last(a.counters + (long)first[wave] * a.n_kv_heads + kvh, parts[wave]);
    __syncthreads();
    const bool last[2] = {sh.last[0] != 0, sh.last[1] != 0};
    if (!last[0] && !last[1]) return;
    asm volatile("" ::: "memory");
    // A set's parts are merged in `runs`, one per group of per_item threads where there are enough
    // of those, and the runs in LDS.  How a set is cut into runs depends on its parts alone: the
    // sums are in the same order whoever comes last and whatever else it merges.
    const int each = last[0] && last[1] ? side_by_side / 2 : side_by_side;   // groups of threads per set
    const int k = last[0] && mine < each ? 0 : 1, me = last[0] && last[1] ? mine - k * each : mine;
    const int runs = min(side_by_side, (parts[k] + 3) / 4);
    const bool works = mine < side_by_side && me < each;
    float *o_lds = sh.o[0][0] + (long)k * side_by_side * per_item * 4, *ml_lds = sh.ml[k][0][0];
    static_assert(sizeof(sh.o) >= 2 * 64 * kSplitWaves * 16 && sizeof(sh.ml[0]) >= 16 * 8, "a place per thread and set");
    if (works)
        for (int r = me; r < runs; r += each) {
            const int p0 = parts[k] * r / runs, p1 = parts[k] * (r + 1) / runs;
            float m, l;
            const f32x4 o =
                p1 - p0 <= 4 ? merge_slots<4>(a.part_o, a.part_ml, first[k] + p0, p1 - p0, a.n_qo_heads, qh, d0, m, l)
                             : merge_slots<8>(a.part_o, a.part_ml, first[k] + p0, p1 - p0, a.n_qo_heads, qh, d0, m, l);
            *reinterpret_cast<f32x4 *>(o_lds + (r * per_item + idx4) * 4) = o;
            if (d0 == 0) {
                ml_lds[(r * group + head) * 2] = m;
                ml_lds[(r * group + head) * 2 + 1] = l;
            }
        }
    __syncthreads();
    if (works && me == 0) {
        float m_all = kNegBig, l_all = 0.f;
        for (int r = 0; r < runs; r++) m_all = fmaxf(m_all, ml_lds[(r * group + head) * 2]);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int r = 0; r < runs; r++) {
            const float weight = __builtin_amdgcn_exp2f(ml_lds[(r * group + head) * 2] - m_all);
            l_all += weight * ml_lds[(r * group + head) * 2 + 1];
            sum += weight * *reinterpret_cast<const f32x4 *>(o_lds + (r * per_item + idx4) * 4);
        }
        const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
        *reinterpret_cast<u32x2 *>(a.out + ((long)row[k] * a.n_qo_heads + qh) * kHeadDim + d0) =
            u32x2{E::pack2(sum[0] * inv, sum[1] * inv), E::pack2(sum[2] * inv, sum[3] * inv)};
    }
}

}  // namespace dskv
