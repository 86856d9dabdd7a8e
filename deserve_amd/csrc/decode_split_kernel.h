// The 16-bit decode attention kernel (head_dim 128) for batches that cannot give every compute
// unit a share of the work: one workgroup per (share, kv head), whose eight waves split the
// share's tiles.  See decode_attn.hip for the rule that picks it.
//
// What bounds it: latency.  A step over 7 MB of K/V (one request of 1777 tokens) needs 1 us of
// HBM time; what lasts is the chain plan -> page id -> tile -> result and everything that hangs
// behind it, and in that chain the instructions: a wave that depends on itself issues one every five to ten cycles
// and fetches most of them for the first time, so everything that is executed once counts.  With
// workgroups of one wave per kv head (decode_kernel.h) that request is cut into
// 28 parts of four tiles, walked one after the other, and merged by a second launch that takes
// nearly as long (14.5 + 11.3 us by rocprofv3; 20.5 us per layer in a replayed graph).  Here a wave
// walks one tile or two, eight waves meet in LDS, and the part that
// finishes last merges the request's parts in the same launch: 9.2 us a layer in a replayed graph, 8 requests
// of 512 tokens 9.2, 8 of 300-1100 11.3, 24 of 64-2048 23.0, 32 of 60-200 9.1 (13.1, 12.9, 15.1, 25.6 and 14.4 while
// the code in front of the first tile and behind the last one was three times as long and shares were cut
// without regard to the requests).
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
// The planner's rules, measured there: tiles of a batch at most (one kv head: at least; one request with three or four heads:
// at most), and parts of one request that make a batch lopsided.  Tiles of a share at least, for the generic kernel's
// plans (the 16-bit ones follow the requests).
constexpr int kSplitMaxTiles = 2560, kSplitMinTilesOneHead = 5000, kSplitMaxTilesOneRequest = 192, kLopsidedParts = 64;
constexpr int kSplitTilesPerShare = 6;
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
// stored and read with device scope (written through, and read past the L2 of the XCD), so nothing
// else in the caches has to be written back or dropped - release / acquire fences write back the whole
// L2.  The counter is set back to zero by the last one, ready for the next launch.
// (Counting in at the start instead, the last one to start waiting for words that are zero between launches to be
// written, saves the acknowledgement and the counter's trip, and costs the looking and the zeros: the request
// of 1777 tokens 9.92 against 10.03 us, two of 1000-3000 with 64 heads 14.4 against 13.1, and the code is longer.)
constexpr int kCoherent = 16;   // cache policy of the buffer instructions: device scope (sc1)
struct Partials {
    __amdgpu_buffer_rsrc_t o, ml;     // the slots' O rows, and their (maximum, sum)
    int o_bytes, ml_bytes;            // of a slot
    __device__ __forceinline__ Partials(const float *part_o, const float *part_ml, int slots, int n_qo_heads)
    {
        o_bytes = n_qo_heads * kHeadDim * 4;
        ml_bytes = n_qo_heads * 8;
        o = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(part_o), 0, slots * o_bytes, kBufferFlags);
        ml = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(part_ml), 0, slots * ml_bytes, kBufferFlags);
    }
    __device__ __forceinline__ void put_o(int slot, int at, f32x4 v) const
    {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), o, at * 4, slot * o_bytes, kCoherent);
    }
    __device__ __forceinline__ void put_ml(int slot, int qh, f32x2 v) const
    {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), ml, qh * 8, slot * ml_bytes, kCoherent);
    }
    __device__ __forceinline__ f32x4 get_o(int slot, int at) const
    {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(o, at * 4, slot * o_bytes, kCoherent));
    }
    __device__ __forceinline__ f32x2 get_ml(int slot, int qh) const
    {
        return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(ml, qh * 8, slot * ml_bytes, kCoherent));
    }
};
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
__device__ __forceinline__ f32x4 merge_slots(const Partials &at, int first, int parts, int qh, int d0, float &m, float &l)
{
    m = kNegBig;
    l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < parts; i0 += kAtOnce) {
        f32x4 o[kAtOnce];
        f32x2 ml[kAtOnce];   // (maximum, sum)
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const int slot = first + min(i0 + i, parts - 1);   // past the last: it again, weight zero
            ml[i] = at.get_ml(slot, qh);
            o[i] = at.get_o(slot, qh * kHeadDim + d0);
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

// Two cache lines, what the first loads need in front (they come by scalar loads, a line at a time).
struct SplitArgs {
    const char *pages;
    const int32_t *kv_indices;
    const Item *items;
    const int32_t *wg_ptr;
    const uint16_t *q;
    const float *rope;               // null: q and k_new are not to be rotated
    const uint16_t *k_new, *v_new;   // null: the newest tokens are in the pages already
    int n_qo_heads, n_kv_heads, group, page_shift;
    float scale_log2;
    int max_slots;
    float *part_o, *part_ml;
    uint32_t *counters;              // one zeroed word per (partial slot, kv head); null: a merge launch follows
    int n_counters;
    uint16_t *out;
};
static_assert(sizeof(SplitArgs) == 128, "");
typedef const __attribute__((address_space(4))) SplitArgs *const_args_ptr;
typedef int32_t i32x8 __attribute__((ext_vector_type(8), aligned(4)));
typedef const __attribute__((address_space(4))) i32x8 *const_i32x8_ptr;

// A workgroup fills its compute unit's LDS, so what counts is that the workgroups spread evenly: ids go
// round the 8 XCDs, and without gaps in them no XCD gets more than its 32, whatever the number of
// heads.  (The heads of a share need not meet on an XCD: they read other bytes of the same pages.)
//
// What keeps the path through it short: no division (a share and a head are grid coordinates; an item's heads are
// dealt to whole waves), an item's words in one load, both first pages in one trip, q turned by a lane per chunk instead of by
// every lane for its operand (45 instead of 180 instructions), operands of a tile requested from LDS together, nothing issued
// for tiles that are not there, arguments read anew behind the loop instead of spilled, pieces that meet
// requested together.  All that: the request of 1777 tokens, in 18 parts, 13.1 -> 10.9 us a layer, 4 of 60 tokens 9.6 -> 6.3.
template <int DT, int kPagesPerTile>
__global__ __launch_bounds__(64 * kSplitWaves) void decode_attn_split_kernel(const SplitArgs a)
{
    typedef Elt<DT> E;
    constexpr bool kPageCoversTile = kPagesPerTile == 1, kWholeRows = kSplitWholeRows;
    __shared__ __align__(16) SplitShared sh;
    const int share = (int)blockIdx.x, kvh = (int)blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int group = a.group;
    const const_i32_ptr item_words = as_const(reinterpret_cast<const int32_t *>(a.items));
    const int item_begin = as_const(a.wg_ptr)[share], item_end = as_const(a.wg_ptr)[share + 1];
    if (item_begin >= item_end) return;

    // ---- this wave's slice of the share's tiles, and the items it meets
    struct Words {
        int row, begin, end, slot, page_begin, tail, parts, at;
    };
    auto words_of = [&](int idx) {   // (one load of eight words, not a few of two when they are needed)
        const i32x8 w = *reinterpret_cast<const_i32x8_ptr>(item_words + (long)idx * kItemWords);
        return Words{w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7]};
    };
    auto tiles_of = [](int begin, int end) { return (int)((unsigned)(end - begin + kTile - 1) / kTile); };
    const Words head_item = words_of(item_begin), tail_item = words_of(item_end - 1);   // (requested together)
    const int total = tail_item.at + tiles_of(tail_item.begin, tail_item.end);
    const int lo = (int)((unsigned)(total * wave) / kSplitWaves), hi = (int)((unsigned)(total * (wave + 1)) / kSplitWaves);
    // the first item whose tiles end behind lo, if they begin before hi
    Words w0 = head_item;
    int first_item = item_begin;
    while (w0.at + tiles_of(w0.begin, w0.end) <= lo && first_item < item_end - 1) w0 = words_of(++first_item);
    struct Piece {
        int b, tok_begin, tok_end, slot, page_begin;
        bool tail;        // holds the request's newest token
        bool starts, ends;   // the item starts / ends in this wave's slice
        int at;           // the item's first tile within the share
    };
    auto piece_of = [&](const Words &w) {   // (of an item with tiles in the slice, or without tiles: without any then)
        Piece p;
        p.b = w.row;
        p.tok_begin = w.begin + max(lo - w.at, 0) * kTile;
        p.tok_end = min(w.end, w.begin + (hi - w.at) * kTile);
        p.slot = w.slot;
        p.page_begin = w.page_begin;
        p.starts = w.at >= lo;
        p.ends = p.tok_end == w.end;
        p.tail = w.tail && p.ends;
        p.at = w.at;
        return p;
    };

    KvView kv;
    kv.pages = a.pages;
    kv.page_ids = as_const(a.kv_indices);
    kv.page_shift = a.page_shift;
    kv.row_bytes = a.n_kv_heads * kHeadDim * 2;
    kv.half_bytes = kv.row_bytes << a.page_shift;
    kv.page_bytes = 2L * kv.half_bytes;
    kv.head_off = kvh * (kHeadDim * 2);
    char *tile_lds = sh.tiles + wave * tile_lds_bytes(kSplitWholeRows);
    uint32_t *new_k = sh.new_row[wave][0], *new_v = sh.new_row[wave][1];

    // ---- what a piece needs besides its tiles: lane i has chunk i % 16 (8 dims) of q rows i / 16 and i / 16 + 4 (past
    // the group: some chunk), the cosines and sines of the chunk, and of the new token's rows (K in lanes 0-15, V in
    // lanes 16-31) the same chunk.
    struct Raw {
        u32x4 q[2], fresh;
        f32x4 cs, sn;
        int page;         // of the new token
    };
    auto request = [&](const Piece &p, Raw &r) {
        const uint16_t *rows = a.q + ((long)p.b * a.n_qo_heads + kvh * group) * kHeadDim;
        r.q[0] = *reinterpret_cast<const u32x4 *>(rows + min(lane, group * 16 - 1) * 8);
        if (group > 4) r.q[1] = *reinterpret_cast<const u32x4 *>(rows + min(64 + lane, group * 16 - 1) * 8);
        if (a.rope) {
            const float *tab = a.rope + (long)p.b * kHeadDim + c * 4;
            r.cs = *reinterpret_cast<const f32x4 *>(tab);
            r.sn = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2);
        }
        if (a.k_new && p.tail) {
            r.page = as_const(a.kv_indices)[p.page_begin + ((p.tok_end - 1) >> a.page_shift)];
            const long src = ((long)p.b * a.n_kv_heads + kvh) * kHeadDim;
            r.fresh = *reinterpret_cast<const u32x4 *>((lane < 16 ? a.k_new + src : a.v_new + src) + c * 8);
        }
    };
    auto rotate = [&](u32x4 chunk, const Raw &r) {
        const float c4[4] = {r.cs[0], r.cs[1], r.cs[2], r.cs[3]}, s4[4] = {r.sn[0], r.sn[1], r.sn[2], r.sn[3]};
        float f[8];
        Chunk<DT>::unpack(chunk, f);
        rope_rotate<4>(f, c4, s4);
        return Chunk<DT>::pack(f);
    };
    // The q rows as the B operand of the score MFMAs, through the wave's V tile; columns past the group repeat
    // the last row (nobody reads their results).
    auto operand_of = [&](const Raw &r, u32x4 (&qreg)[4]) {
        char *rows = tile_lds;
        __builtin_amdgcn_wave_barrier();
        *reinterpret_cast<u32x4 *>(rows + g * kVPitch + c * 16) = a.rope ? rotate(r.q[0], r) : r.q[0];
        if (group > 4) *reinterpret_cast<u32x4 *>(rows + (4 + g) * kVPitch + c * 16) = a.rope ? rotate(r.q[1], r) : r.q[1];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const char *mine = rows + min(c, group - 1) * kVPitch + g * 16;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) qreg[kk] = *reinterpret_cast<const u32x4 *>(mine + kk * 64);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // Writes the new token's rows into their page slot, and into LDS, from where the tile that
    // holds them takes them: nobody waits for the page to have them.
    auto place_new_row = [&](const Piece &p, const Raw &r) {
        const int tok = p.tok_end - 1;
        char *row = const_cast<char *>(a.pages) + (long)r.page * kv.page_bytes +
                    (long)(tok & ((1 << a.page_shift) - 1)) * kv.row_bytes + kv.head_off + c * 16;
        if (lane < 32) {
            u32x4 chunk = r.fresh;
            if (a.rope && lane < 16) chunk = rotate(chunk, r);
            *reinterpret_cast<u32x4 *>(row + (lane < 16 ? 0 : kv.half_bytes)) = chunk;
            *reinterpret_cast<u32x4 *>((lane < 16 ? new_k : new_v) + c * 4) = chunk;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    if (lane == 0) {
        sh.owner[wave] = -1;
        sh.meet_row[wave] = -1;
    }
    if (lo < hi) {
        // ---- load side: runs ahead of the compute side through the wave's pieces
        Piece piece = piece_of(w0);
        int left = hi - lo, t, t_end, next_item = first_item + 1;   // tiles that are not requested yet; the next of them
        auto enter = [&](const Piece &p) {
            t = p.tok_begin;
            t_end = p.tok_end;
            kv.page_ids = as_const(a.kv_indices) + p.page_begin;
        };
        auto look_up = [&](int tok, long (&pg)[2]) {
#pragma unroll
            for (int j = 0; j < kPagesPerTile; j++) pg[j] = kv.page_ids[page_slot_of(kv, tok + (j << kv.page_shift), t_end)];
        };
        auto load_tile = [&](TileRegs &r, const long (&pg)[2]) {
            if (kPageCoversTile) {
                load_kv_tile_in_page<kLoadStreaming, kWholeRows>(kv, pg[0], t, t_end, g, c, r);
            } else if (kPagesPerTile == 2) {
                load_kv_tile_small_pages<2, kLoadStreaming, kWholeRows>(kv, pg, t, t_end, g, c, r);
            } else {
                load_kv_tile<false, kLoadStreaming, kWholeRows>(kv, t, t_end, g, c, r);
            }
            t += kTile;
            left--;
            while (left > 0 && t >= t_end) enter(piece_of(words_of(next_item++)));   // (items without tokens are stepped over)
        };
        // Two tiles are in flight; the second passes to the first's registers when that one is done with, so that
        // there is one copy of the code.
        enter(piece);
        long page[2] = {0, 0}, page_after[2] = {0, 0};
        look_up(t, page);
        const bool both = t + kTile < t_end;
        if (both) look_up(t + kTile, page_after);
        Raw raw;
        request(piece, raw);
        TileRegs now, after;
        load_tile(now, page);
        auto load_after = [&]() {
            if (left <= 0) return;
            load_tile(after, page_after);
            if (left > 0) look_up(t, page_after);
        };
        if (left > 0 && !both) look_up(t, page_after);
        load_after();

        int idx = first_item, computed_tiles = 0;
        while (true) {
            u32x4 qreg[4];
            operand_of(raw, qreg);
            const bool fresh = a.k_new && piece.tail;
            if (fresh) place_new_row(piece, raw);
            // the wave's next piece, if there is one
            computed_tiles += tiles_of(piece.tok_begin, piece.tok_end);
            const bool more = computed_tiles < hi - lo;
            Piece next = piece;
            if (more) {
                do next = piece_of(words_of(++idx));
                while (next.tok_end <= next.tok_begin);   // (without tokens)
                request(next, raw);
            }

            f32x4 acc[8];
#pragma unroll
            for (int dt = 0; dt < 8; dt++) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            float m_run = kNegBig, l_run = 0.f;
            const bool own_maximum = piece.slot < 0 && piece.tok_end - piece.tok_begin > kTile;
            auto compute_tile = [&](int t0, TileRegs &r) {
                const int end = piece.tok_end;
                if (fresh && t0 + kTile >= end) {
                    // the newest token is this tile's row nr, and the page may not have it yet
                    const int nr = end - 1 - t0;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                    {
                        if (kWholeRows && g + 4 * i == nr) r.k[i] = *reinterpret_cast<const u32x4 *>(new_k + c * 4);
                        if (!kWholeRows && c == nr) r.k[i] = *reinterpret_cast<const u32x4 *>(new_k + i * 16 + g * 4);
                        if (g + 4 * i == nr) r.v[i] = *reinterpret_cast<const u32x4 *>(new_v + c * 4);
                    }
                }
                // all twelve operands are requested before the first is waited for
                if (kWholeRows) stage_k_tile(tile_lds, r, g, c);
                stage_v_tile<kPageCoversTile>(tile_lds, r, t0, end, g, c);
                u32x4 ka[4];
                u32x2 va[8];
#pragma unroll
                for (int kk = 0; kk < 4; kk++) ka[kk] = kWholeRows ? read_k_operand(tile_lds, kk, g, c) : r.k[kk];
#pragma unroll
                for (int dt = 0; dt < 8; dt++) va[dt] = read_v_operand(tile_lds, dt, g, c);
                __builtin_amdgcn_sched_barrier(0);
                f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < 4; kk++) s = E::mfma_k32(ka[kk], qreg[kk], s);
                const bool ragged = t0 + kTile > end;
                float x[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    x[j] = s[j] * a.scale_log2;
                    if (ragged && t0 + 4 * g + j >= end) x[j] = kNegBig;
                }
                const float m_tile = quad_rows_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
                const float m_new = fmaxf(m_run, m_tile);
                const float m_of_p = own_maximum ? m_tile : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                float p[4], p_sum = 0.f;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    p[j] = x[j] > kNegBig ? __builtin_amdgcn_exp2f(x[j] - m_of_p) : 0.f;
                    p_sum += p[j];
                }
                m_run = m_new;
                const u32x2 pb = {E::pack2(p[0], p[1]), E::pack2(p[2], p[3])};
                if (own_maximum) {
                    // A request that lies whole in the share, where a wave may have more tiles than in shares that cut
                    // it: P under the tile's own maximum, brought to the common one in fp32.  The largest
                    // probability of every tile is then exactly 1 in 16 bits, however many a wave has (under the running
                    // maximum two tiles a wave instead of one put the error against 64 bits up by 1.5 to 3 %).
                    const float beta = __builtin_amdgcn_exp2f(m_tile - m_new);
                    l_run = l_run * alpha + p_sum * beta;
                    f32x4 o[8];
#pragma unroll
                    for (int dt = 0; dt < 8; dt++) o[dt] = E::mfma_k16(va[dt], pb, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int dt = 0; dt < 8; dt++) acc[dt] = acc[dt] * alpha + o[dt] * beta;
                } else {
                    l_run = l_run * alpha + p_sum;
#pragma unroll
                    for (int dt = 0; dt < 8; dt++) acc[dt] = E::mfma_k16(va[dt], pb, acc[dt] * alpha);
                }
                __builtin_amdgcn_wave_barrier();
            };
            for (int t0 = piece.tok_begin;;) {
                compute_tile(t0, now);
                t0 += kTile;
                now = after;
                load_after();
                if (t0 >= piece.tok_end) break;
            }
            l_run = quad_rows_sum(l_run);
            const bool whole = piece.starts && piece.ends;
            if (whole && piece.slot < 0) {
                if (c < group) {
                    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
                    uint16_t *o = a.out + ((long)piece.b * a.n_qo_heads + kvh * group + c) * kHeadDim + 4 * g;
#pragma unroll
                    for (int dt = 0; dt < 8; dt++)
                        *reinterpret_cast<u32x2 *>(o + dt * 16) =
                            u32x2{E::pack2(acc[dt][0] * inv, acc[dt][1] * inv), E::pack2(acc[dt][2] * inv, acc[dt][3] * inv)};
                }
            } else if (whole) {
                // a part of a cut request that no other wave of the share has tiles of; a slot beyond the workspace is
                // never written
                const Partials to(a.part_o, a.part_ml, a.max_slots, a.n_qo_heads);
                if (c < group && piece.slot < a.max_slots) {
                    const int qh = kvh * group + c;
#pragma unroll
                    for (int dt = 0; dt < 8; dt++) to.put_o(piece.slot, qh * kHeadDim + 4 * g + dt * 16, acc[dt]);
                    if (g == 0) to.put_ml(piece.slot, qh, f32x2{m_run, l_run});
                }
            } else {
                // one end of an item that other waves share
                const int place = piece.starts ? 1 : 0;
                if (c < group) {
                    float *o = sh.o[wave][place] + c * kHeadDim + 4 * g;
#pragma unroll
                    for (int dt = 0; dt < 8; dt++) *reinterpret_cast<f32x4 *>(o + dt * 16) = acc[dt];
                    if (g == 0) *reinterpret_cast<f32x2 *>(sh.ml[wave][place][c]) = f32x2{m_run, l_run};
                }
                // the wave whose slice holds the item's first tile: the last one to begin at it or before
                const int holder = __builtin_popcountll(__builtin_amdgcn_ballot_w64(
                                       lane < kSplitWaves && (int)((unsigned)(total * lane) / kSplitWaves) <= piece.at)) - 1;
                if (lane == 0) {
                    if (piece.starts) {
                        sh.meet_row[wave] = piece.b;
                        sh.meet_slot[wave] = piece.slot;
                    } else {
                        sh.owner[wave] = holder;
                    }
                }
            }
            if (!more) break;
            piece = next;
        }
    }
    // requests without tokens: rows of zeros
    if (wave == kSplitWaves - 1 && (item_end - item_begin > 1 || total == 0))
        for (int i = item_begin; i < item_end; i++) {
            const const_i32_ptr w = item_words + (long)i * kItemWords;
            if (w[1] < w[2]) continue;
            uint16_t *row = a.out + ((long)w[0] * a.n_qo_heads + kvh * group) * kHeadDim;
            for (int at = lane * 8; at < group * kHeadDim; at += 64 * 8) *reinterpret_cast<u32x4 *>(row + at) = u32x4{0, 0, 0, 0};
        }
    // ---- behind the barrier a thread owns four dims of a head, and an item's heads are dealt to whole waves, two
    // each: `side` items are worked on side by side.  (Arguments and items are read anew from here on: held through
    // the loop, they are spilled.)
    __syncthreads();
    const_args_ptr late = (const_args_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late));
    const int waves_per_item = (group + 1) / 2;
    const int side_shift = waves_per_item >= 3 ? 1 : 4 - waves_per_item, side = 1 << side_shift;
    const int mine = waves_per_item == 3 ? wave / 3 : wave >> (3 - side_shift);
    const int head = (wave - mine * waves_per_item) * 2 + (lane >> 5), d0 = (lane & 31) * 4;
    const bool works = mine < side && head < group;
    const int qh = kvh * group + head;
    const Partials parts_at(late->part_o, late->part_ml, late->max_slots, late->n_qo_heads);
    auto put_row = [&](int row, f32x4 sum, float l) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        *reinterpret_cast<u32x2 *>(late->out + ((long)row * late->n_qo_heads + qh) * kHeadDim + d0) =
            u32x2{E::pack2(sum[0] * inv, sum[1] * inv), E::pack2(sum[2] * inv, sum[3] * inv)};
    };

    // ---- the items that meet
    const int in_wave = lane & (kSplitWaves - 1);
    const int owner = sh.owner[in_wave];
    uint32_t meetings = (uint32_t)__builtin_amdgcn_ballot_w64(sh.meet_row[in_wave] >= 0) & ((1 << kSplitWaves) - 1);
    for (int n = 0; meetings; n++, meetings &= meetings - 1) {
        if ((n & (side - 1)) != mine) continue;
        const int e = __builtin_ctz(meetings);
        const uint32_t from = (uint32_t)__builtin_amdgcn_ballot_w64(owner == e) & ((1 << kSplitWaves) - 1);
        const int row = __builtin_amdgcn_readfirstlane(sh.meet_row[e]), slot = __builtin_amdgcn_readfirstlane(sh.meet_slot[e]);
        // all waves' pieces are requested at once; waves that hold no piece of the item have its first, weighing nothing
        f32x4 o[kSplitWaves];
        f32x2 ml[kSplitWaves];
        const int h = min(head, group - 1);
#pragma unroll
        for (int w = 0; w < kSplitWaves; w++) {
            const bool in = from >> w & 1;
            const int from_wave = in ? w : e, place = in ? 0 : 1;
            o[w] = *reinterpret_cast<const f32x4 *>(sh.o[from_wave][place] + h * kHeadDim + d0);
            ml[w] = *reinterpret_cast<const f32x2 *>(sh.ml[from_wave][place][h]);
            if (!in && w != e) ml[w].x = 2.f * kNegBig;
        }
        __builtin_amdgcn_sched_barrier(0);
        float m_all = ml[0].x;
#pragma unroll
        for (int w = 1; w < kSplitWaves; w++) m_all = fmaxf(m_all, ml[w].x);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        float l_all = 0.f;
#pragma unroll
        for (int w = 0; w < kSplitWaves; w++) {
            const float weight = __builtin_amdgcn_exp2f(ml[w].x - m_all);
            l_all += weight * ml[w].y;
            sum += weight * o[w];
        }
        if (!works) continue;
        if (slot < 0) {
            put_row(row, sum, l_all);
        } else if (slot < late->max_slots) {
            parts_at.put_o(slot, qh * kHeadDim + d0, sum);
            if (d0 == 0) parts_at.put_ml(slot, qh, f32x2{m_all, l_all});
        }
    }

    // ---- the parts of cut requests.  Only the first and the last item of a share can be parts
    // (the shares' boundaries cut); both are counted in, and merged, side by side.
    if (!late->counters) return;
    struct Set {
        int row, first, parts, counter;
        bool cut;
    };
    const const_i32_ptr late_words = as_const(reinterpret_cast<const int32_t *>(late->items));
    auto set_of = [&](int idx) {
        const i32x8 w = *reinterpret_cast<const_i32x8_ptr>(late_words + (long)idx * kItemWords);
        Set s;
        s.row = w[0];
        s.first = w[6] >> kPartsBits;
        s.parts = w[6] & ((1 << kPartsBits) - 1);
        s.counter = s.first * late->n_kv_heads + kvh;
        s.cut = (w[3] >= 0) & (s.parts > 0) & (s.first + s.parts <= late->max_slots) & (s.counter < late->n_counters);
        return s;
    };
    Set sets[2] = {set_of(item_begin), set_of(item_end - 1)};
    sets[1].cut &= item_end - 1 != item_begin;
    if (!sets[0].cut && !sets[1].cut) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the partials are where other XCDs see them
    __syncthreads();
    if (wave < 2 && lane == 0) {
        const Set &s = wave ? sets[1] : sets[0];
        sh.last[wave] = s.cut && arrive_last(late->counters + s.counter, s.parts);
    }
    __syncthreads();
    const bool last[2] = {__builtin_amdgcn_readfirstlane(sh.last[0]) != 0, __builtin_amdgcn_readfirstlane(sh.last[1]) != 0};
    if (!last[0] && !last[1]) return;
    asm volatile("" ::: "memory");
    // A set's parts are merged in `runs`, one per `mine` where there are enough, and the runs in LDS.  How a
    // set is cut into runs depends on its parts alone: the sums are in the same order whoever merges and
    // whatever else it merges.
    const int each = last[0] && last[1] ? side >> 1 : side;   // per set
    const int k = last[0] && mine < each ? 0 : 1, me = last[0] && last[1] ? mine - k * each : mine;
    const int set_parts = k ? sets[1].parts : sets[0].parts, set_first = k ? sets[1].first : sets[0].first;
    const int set_row = k ? sets[1].row : sets[0].row;
    const int per_run = max(4, (set_parts + side - 1) >> side_shift);
    const bool merges = works && me < each;
    float *o_lds = sh.o[0][0] + k * side * group * kHeadDim, *ml_lds = sh.ml[0][0][0] + k * side * group * 2;
    static_assert(sizeof(sh.o) >= 2 * 8 * 2 * kHeadDim * 4 && sizeof(sh.ml) >= 2 * 16 * 8, "a place per run and set");
    if (merges)
        for (int r = me; r * per_run < set_parts; r += each) {
            const int at = set_first + r * per_run, n = min(per_run, set_parts - r * per_run);
            float m, l;
            const f32x4 o = n <= 4 ? merge_slots<4>(parts_at, at, n, qh, d0, m, l) : merge_slots<8>(parts_at, at, n, qh, d0, m, l);
            *reinterpret_cast<f32x4 *>(o_lds + (r * group + head) * kHeadDim + d0) = o;
            if (d0 == 0) *reinterpret_cast<f32x2 *>(ml_lds + (r * group + head) * 2) = f32x2{m, l};
        }
    __syncthreads();
    if (merges && me == 0) {
        float m_all = kNegBig, l_all = 0.f;
        for (int r = 0; r * per_run < set_parts; r++) m_all = fmaxf(m_all, ml_lds[(r * group + head) * 2]);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int r = 0; r * per_run < set_parts; r++) {
            const float weight = __builtin_amdgcn_exp2f(ml_lds[(r * group + head) * 2] - m_all);
            l_all += weight * ml_lds[(r * group + head) * 2 + 1];
            sum += weight * *reinterpret_cast<const f32x4 *>(o_lds + (r * group + head) * kHeadDim + d0);
        }
        put_row(set_row, sum, l_all);
    }
}

}  // namespace dskv
