// Paged prefill (multi-query) attention with the end-aligned causal mask:
// query i of the n_b new tokens of request b sees kv positions j <= kv_len_b - n_b + i.
//
// Bound: MFMA for long chunks.  Work decomposition: one workgroup = one kv head x
// one tile of query rows; each of its waves owns 32 columns (kColTiles tiles of
// 32), a column being a (query position, q head of the GQA group) pair, so the
// MFMA N dimension is dense.  The workgroup walks the request's K/V in blocks of
// 32 tokens that its waves load together (each four rows) into LDS stages, so a
// K/V byte crosses the vector memory path once per workgroup instead of once per
// wave: with every wave streaming K/V on its own the kernel was bound by that
// path at a sixth of the MFMA rate.  The rows go from global memory straight into
// LDS (`buffer_load_dwordx4 ... lds`, three blocks ahead of their use), without a
// trip through vector registers; pages shorter than four tokens take the register
// path (load, then ds_write) instead.  The loads are inline assembly with hand-set
// `s_waitcnt vmcnt` and a bare `s_barrier`: through the compiler's builtin every
// barrier and LDS read waited for all loads in flight, which undid the prefetch.
//
// All products use the 32x32x16 MFMA (measured on MI355X at 2.2 PFLOP/s bf16,
// against 1.3 PFLOP/s for 16x16x32).  Per block a wave computes S^T = K.Q^T
// (tokens x columns, K rows from LDS as the A operand), keeps S^T's C layout as
// the B operand P^T, and reads V through the transposing LDS read as the A
// operand of O^T += V^T.P^T.
//
// Workgroup ids are laid out head-fastest: consecutive ids go to different XCDs,
// so (with 8 kv heads) all query tiles of one kv head share one XCD's L2.
//
// A batch of few tiles (one 512-token chunk: 8 tiles x 8 kv heads) would leave most
// of the chip idle.  The plan then cuts every tile's K/V range into parts; a part is
// a workgroup of its own that leaves (maximum, sum, unnormalised O) of its rows in a
// workspace, and a merge pass (one workgroup per query row) turns the parts into the output.
#include "kv_tile.h"
#include "decode_kernel.h"

#include <algorithm>
#include <atomic>
#include <new>
#include <numeric>
#include <vector>

#include "prefill_kernel.h"
#include "prefill_short_kernel.h"

namespace dskv {

// Generic path (fp32 pools, head_dim != 128, group > 16): one wavefront per
// (query row, q head), plain VALU, sequential over the visible tokens.
template <int DT>
__global__ __launch_bounds__(64) void prefill_attn_generic_kernel(
    void *__restrict__ out, const void *__restrict__ q, const int32_t *__restrict__ qo_indptr,
    const void *__restrict__ pages, const int32_t *__restrict__ kv_indices,
    const int32_t *__restrict__ kv_indptr, const int32_t *__restrict__ kv_last, int batch,
    int n_qo_heads, int n_kv_heads, int head_dim, int page_size, float scale_log2, int causal)
{
    typedef LoadElt<DT> L;
    const int lane = threadIdx.x;
    const int row = blockIdx.x;
    const int qh = blockIdx.y;
    const int kvh = qh / (n_qo_heads / n_kv_heads);
    int lo = 0, hi = batch;   // largest b with qo_indptr[b] <= row
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (qo_indptr[mid] <= row) lo = mid; else hi = mid;
    }
    const int b = lo;
    if (row >= qo_indptr[b + 1]) return;
    const int n_b = qo_indptr[b + 1] - qo_indptr[b];
    const int page_begin = kv_indptr[b];
    const int n_pages = kv_indptr[b + 1] - page_begin;
    const int kv_len = n_pages > 0 ? (n_pages - 1) * page_size + kv_last[b] : 0;
    int limit = causal ? kv_len - n_b + (row - qo_indptr[b]) + 1 : kv_len;
    limit = min(max(limit, 0), kv_len);
    const long tok_row = (long)n_kv_heads * head_dim;
    const long half = tok_row * page_size;

    float qv[4], acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        qv[i] = d < head_dim ? L::get(q, ((long)row * n_qo_heads + qh) * head_dim + d) : 0.f;
        acc[i] = 0.f;
    }
    float m_run = kNegBig, l_run = 0.f;
    // kGroup tokens at a time: page ids, K rows and V rows of the group are all requested
    // before the first is used (token by token, every token waited for memory twice)
    constexpr int kGroup = 8;
    for (int t0 = 0; t0 < limit; t0 += kGroup) {
        long base[kGroup];
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            const int t = min(t0 + j, limit - 1);   // past the limit: the last token again, weight zero
            const long page = kv_indices[page_begin + t / page_size];
            base[j] = page * 2 * half + (long)(t % page_size) * tok_row + (long)kvh * head_dim;
        }
        float kx[kGroup][4], vx[kGroup][4];
#pragma unroll
        for (int j = 0; j < kGroup; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = lane + 64 * i;
                kx[j][i] = d < head_dim ? L::get(pages, base[j] + d) : 0.f;
            }
#pragma unroll
        for (int j = 0; j < kGroup; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = lane + 64 * i;
                vx[j][i] = d < head_dim ? L::get(pages, base[j] + half + d) : 0.f;
            }
        float x[kGroup], m_new = m_run;
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) dot += qv[i] * kx[j][i];
            x[j] = t0 + j < limit ? wave_sum(dot) * scale_log2 : kNegBig;
            m_new = fmaxf(m_new, x[j]);
        }
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] *= alpha;
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            const float p = x[j] > kNegBig ? __builtin_amdgcn_exp2f(x[j] - m_new) : 0.f;
            l_run += p;
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] += p * vx[j][i];
        }
        m_run = m_new;
    }
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        if (d < head_dim) L::put(out, ((long)row * n_qo_heads + qh) * head_dim + d, acc[i] * inv);
    }
}

static int prefill_rows_per_tile(int n_qo_heads, int n_kv_heads, int waves)
{
    const int group = n_qo_heads / n_kv_heads;
    return group <= kWaveCols ? waves * (kWaveCols / group) : 1;
}

// ---------------------------------------------------------------------------
// The mixed launch: decode workgroups and query tiles side by side on every CU.
//
// A compute unit moves at most ~36 GB/s through its vector memory path (measured: one
// decode workgroup of eight, four or two waves per CU streams 37, 35 and 31 GB/s, whatever
// else is free), so the chip's 8 TB/s are only there when EVERY CU has loads in flight -
// and a CU that computes a chunk's query tiles (bound by its matrix pipeline) contributes
// none.  Run one after the other, the decode rows and the chunk of a mixed step (75 rows over
// U[256,4096] tokens + 437 tokens over 2506) take 118 + 47 us; as tiles of one launch, with
// one live row per 64-row tile and the longest rows walked by a single workgroup, 147 us
// (228 us when the chunk follows 8000 tokens).  Here both kinds of work are workgroups of
// FOUR waves (one per SIMD, at most 256 vector registers, half a CU's LDS each), so two fit
// on a CU, and the launch starts with one decode workgroup per CU: the dispatcher places the
// first #CU workgroups of a grid one per CU (measured on the box), so the decode workgroups -
// statically balanced shares that must all start at once - own one slot of every CU for the
// whole launch, while the query tiles pass through the other slot.  Measured: 150 us (175 us
// behind 8000 tokens): the tile workgroups finish within 66 us, the decode workgroups, which
// share the CU's memory path with them meanwhile, after 145 us instead of 113 us alone.
// ---------------------------------------------------------------------------
// Tiles in flight per decode wave of the mixed launch: with three, the step of 75 rows and a chunk takes
// 2370 us instead of 2364, 70B-shaped 1338 instead of 1327; with four 2383 and 1398.
constexpr int kSharedRing = 2;
constexpr bool kSharedWholeRows = true;
// Wave priority of the tile workgroups.  At equal priority the compute unit serves the older
// waves first, and the decode waves - launched first, never short of a load to issue - kept
// the tile waves' few loads waiting: a tile workgroup took 162 us beside them instead of 38 us
// alone.  With the tile waves ahead (any priority above 0) it takes 66 us.
constexpr int kSharedTilePriority = 3;
struct MixedArgs {
    uint16_t *out;
    const uint16_t *q;
    const char *pages;
    const int32_t *kv_indices;
    int n_qo_heads, n_kv_heads, page_shift;
    float scale_log2;
    // decode side: shares x head groups workgroups come first in the grid
    const Item *items;
    const int32_t *wg_ptr;
    float *dec_part_o, *dec_part_ml;
    int dec_max_slots, n_decode_wgs, head_groups;
    // tile side
    const int32_t *qo_indptr, *kv_indptr, *kv_last, *tile_info;
    float *tile_part_o, *tile_part_ml;
    int tile_max_slots, causal;
    const float *rope;   // cos | sin by query row (q is rotated as it is loaded), or null
};

template <int DT, int kPagesPerTile>
__global__ __launch_bounds__(64 * kSharedWaves, 2) void mixed_attn_kernel(const MixedArgs a)
{
    static_assert(kSharedWaves == kPrefillWavesShared, "both kinds of workgroup have the launch's size");
    static_assert(prefill_lds_bytes(kSharedWaves) >= kSharedWaves * tile_lds_bytes(kSharedWholeRows), "the LDS is shared by the two bodies");
    __shared__ __align__(16) char lds[prefill_lds_bytes(kSharedWaves)];
    const int wg = blockIdx.x;
    if (wg < a.n_decode_wgs)
        decode_attn_body<DT, kPagesPerTile, kSharedWaves, kSharedRing, kSharedWholeRows>(
            lds, wg / a.head_groups, wg % a.head_groups, a.out, a.q, a.pages, a.kv_indices, a.items, a.wg_ptr,
            a.dec_part_o, a.dec_part_ml, a.dec_max_slots, a.n_qo_heads, a.n_kv_heads, a.page_shift,
            a.scale_log2, nullptr, nullptr, a.rope);
    else {
        __builtin_amdgcn_s_setprio(kSharedTilePriority);
        prefill_attn_body<DT, true, kPrefillWavesShared, true>(
            lds, wg - a.n_decode_wgs, a.out, a.q, a.qo_indptr, a.pages, a.kv_indices, a.kv_indptr, a.kv_last,
            a.tile_info, a.n_qo_heads, a.n_kv_heads, a.page_shift, a.scale_log2, a.causal,
            a.tile_part_o, a.tile_part_ml, a.tile_max_slots, a.rope, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    }
}

}  // namespace dskv

namespace dskv {

constexpr int kMaxPrefillSplits = 8;         // parts a tile's K/V range is cut into at most
// a part holds at least this many tokens: with 256, a 512-token chunk without prior context
// took 37 us in two parts instead of 29 us whole; with 1024, chunks over 1-2 k tokens of prior
// context lost a fifth of what the parts buy
constexpr int kMinSplitTokens = 512;
constexpr int kMaxSplitTarget = 1024;        // workgroups a split plan aims at, at most
// a workgroup's start and end, in 32-token blocks of walking (for the fair share of a launch)
constexpr int kTileOverheadBlocks = 4;
constexpr int32_t kWholeRange = 0x7fffffff;  // blk_end of a tile that is not split
// One-row requests of a mixed batch get decode workgroups of their own beside the tiles when
// there are at least this many of them ...
constexpr int kMinSharedLaunchRows = 12;
// ... and when, run as tiles (one live row per tile), they would be most of the launch's work:
// a tile is priced at its 32-token blocks plus this much for its start and end.
constexpr int kTileFixedCostBlocks = 16;
// ... or if a launch of tiles had a walk longer than 3/2 of those of the shared one's tiles and this many blocks more.
constexpr int kLongWalkBlocks = 16;
// (a shared launch's tile counts this much more where there are many: four of 350 to 980 beside eight of 100 to 230,
// groups of 8, 31.8 as tiles and 36.9 shared)
constexpr int kSharedTileOverheadBlocks = 8;

static int compute_units()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    (void)hipGetLastError();
    return cus;
}

}  // namespace dskv

extern "C" int64_t dskv_prefill_plan_bound(int32_t batch, int64_t nnz)
{
    using namespace dskv;
    if (batch < 0 || nnz < 0) return 0;
    // entries: one per tile (at most batch + nnz of them), times the parts of those that are
    // cut: filling the chip adds at most 2 * kMaxSplitTarget entries, cutting long walks down
    // to the fair share at most 2 * kMaxSplitTarget more; then two words per query row
    return kTileWords * ((int64_t)batch + nnz + 4 * kMaxSplitTarget + kMaxPrefillSplits) + 2 * nnz;
}

namespace dskv {

// The tile planner.  skip (may be null): requests marked there get no tiles (their single
// row is computed by the decode kernel).  Plan: the tile entries (kTileWords each), then, if
// any tile is cut into parts, two words per query row of the batch (first partial slot,
// number of parts; 0 parts = the row needs no merge).
static bool prefill_mfma_path(int dtype, int head_dim, int n_qo_heads, int n_kv_heads, float scale_log2)
{
    // the MFMA kernel takes maxima before scaling: it needs a positive, sane scale
    return (dtype == DSKV_BF16 || dtype == DSKV_F16) && head_dim == kHeadDim && n_kv_heads > 0 &&
           n_qo_heads / n_kv_heads <= kWaveCols && scale_log2 > 1e-6f && scale_log2 < 1e6f;
}

// Tiles of few and short walks (prefill_short_kernel.h): in quarters or halves, or as they are.
// A quarter is for a launch whose quarters with rows have a compute unit each: 16 more would be a second turn of all
// (bf16, 8 kv heads, groups of 4, us a layer, as they are -> quarters -> halves: 8 prompts of 64, 256 quarters:
// 15.1 -> 10.2 -> 12.3; 8 of 128, 512 quarters: 19.5 -> 19.5 -> 16.5; 16 of 128, 512 halves: 24.9 -> 33.0 -> 29.7).
// A workgroup has 256 keys in LDS and waits for memory anew for the next ones, a tile's ring does not; with half the
// waves for the keys it has lost what it gained by the second time (a prompt of 256 tokens: 18.9 -> 13.8 -> 16.9; of
// 512: 24.8 -> 20.3 -> 25.0), and the other pays for more only where it has columns enough to use the matrix
// pipeline for (128 tokens behind 300: 22.3 -> 18.3, 32 behind 400: 21.4 -> 21.5, 16 behind 500: 19.4 -> 20.7), and up
// to the fourth time (64 tokens behind 450 24.4 -> 20.7, behind 900 33.8 -> 30.3; 181 behind 450 27.0 -> 23.0, behind 900, where
// the tiles would be in two parts, 38.0 -> 33.0; 512 behind 450 34.6 -> 32.1; 64 behind 1500, in three parts, 31.3 -> 43.9).
constexpr int64_t kShortKeys = kShortRoundTokens, kShortMostKeys = 4 * kShortRoundTokens;
static int short_walk_workgroups(const int32_t *qo_indptr_host, const int32_t *kv_len_host, const int32_t *plan_host,
                                 int32_t n_tiles, int32_t n_qo_heads, int32_t n_kv_heads)
{
    const int rows = prefill_rows_per_tile(n_qo_heads, n_kv_heads, kPrefillWaves), quarter = rows / 4;
    int64_t quarters = 0, halves = 0;
    bool once = true;
    if (n_tiles == 0 || n_tiles > compute_units()) return 0;
    for (int32_t i = 0; i < n_tiles; i++) {
        const int32_t *e = plan_host + (int64_t)i * kTileWords;
        if (e[2] != 0) continue;   // a tile's second part
        const int64_t n_b = (int64_t)qo_indptr_host[e[0] + 1] - qo_indptr_host[e[0]];
        const int64_t live = std::min<int64_t>(rows, n_b - e[1]), keys = kv_len_host[e[0]] - n_b + e[1] + live;
        if (keys > (n_b > rows / 2 ? kShortMostKeys : kShortKeys)) return 0;
        once = once && keys <= kShortKeys;
        quarters += (live + quarter - 1) / quarter;
        halves += (live + 2 * quarter - 1) / (2 * quarter);
    }
    if (quarters * n_kv_heads <= compute_units()) return 4;
    return once && halves * n_kv_heads <= compute_units() ? 2 : 0;
}

static int plan_tiles(const int32_t *qo_indptr_host, const int32_t *kv_len_host, const char *skip,
                      int32_t batch, int32_t n_qo_heads, int32_t n_kv_heads, int32_t head_dim,
                      int32_t target_workgroups, int32_t *plan_host, int64_t capacity_words,
                      int32_t *n_tiles_out, int32_t *n_splits_out, int64_t *plan_words_out,
                      int64_t *workspace_bytes_out, int waves = kPrefillWaves, bool cut_long_walks = true)
{
    const int rows = prefill_rows_per_tile(n_qo_heads, n_kv_heads, waves);
    // later query tiles of a request see more keys: they come first within a request
    struct Tile { int32_t b, row, n_rows, parts; int64_t keys, first_slot; };
    std::vector<Tile> tiles;
    int64_t nnz = 0;
    for (int b = 0; b < batch; b++) {
        const int64_t n_b = (int64_t)qo_indptr_host[b + 1] - qo_indptr_host[b];
        DSKV_REQUIRE(n_b >= 0, "prefill_plan: qo_indptr not monotone at %d", b);
        nnz += n_b;
        if (skip && skip[b]) continue;
        for (int64_t i = (n_b + rows - 1) / rows - 1; i >= 0; i--) {
            const int64_t last_row = std::min<int64_t>(i * rows + rows, n_b) - 1;
            const int64_t keys = kv_len_host ? std::max<int64_t>((int64_t)kv_len_host[b] - n_b + last_row + 1, 0) : 0;
            tiles.push_back({b, (int32_t)(i * rows), (int32_t)(last_row + 1 - i * rows), 1, keys, 0});
        }
    }
    DSKV_REQUIRE(tiles.size() < (size_t(1) << 26) && nnz < (int64_t(1) << 31), "prefill_plan: too many tiles");
    // Workgroups are dispatched in plan order and a tile's time grows with the keys its
    // last row sees: longest first, so the short ones fill the end of the launch
    // (request order left a fifth of the wave slots idle on mixed lengths).
    if (kv_len_host && tiles.size() > 1)
        std::stable_sort(tiles.begin(), tiles.end(),
                         [](const Tile &x, const Tile &y) { return x.keys > y.keys; });
    // Parts.  A tile's K/V range can be cut into parts that run as workgroups of their own and
    // leave partials, merged by a second pass - the decode path's way of keeping all compute
    // units busy.  Needs the kv lengths and the 16-bit kernel's head dim.  Two reasons to cut:
    //  * few tiles (a chunk of a few hundred tokens, as the reference's scheduler hands out:
    //    one 512-token chunk of an 8-kv-head model is 64 workgroups) leave most of the chip
    //    idle: every tile is cut into as many parts as fill it;
    //  * a tile whose walk is longer than the launch's fair share per compute unit ends the
    //    launch by itself (a chunk behind 8000 tokens in a step of decode rows: 232 us, with
    //    its tiles cut in two 197 us): it is cut down to that share.  Cutting further does
    //    not pay: with walks of at most half (a quarter of) the share a mixed step of 75
    //    decode rows and a chunk takes 159 (178) us instead of 149 us - the partials cost more
    //    than the shorter tail buys.  For the same reason only outliers are cut: when the
    //    tiles above the share hold more than a quarter of the launch's blocks (one long
    //    prompt of many tiles, the later ones longer), the launch is made of them, every cut
    //    tile would pay for partials, and the longest-first order is left to do its work.
    int max_parts = 1;
    if (kv_len_host && head_dim == kHeadDim && target_workgroups >= 0 && !tiles.empty()) {
        const int64_t target =
            target_workgroups > 0 ? std::min<int64_t>(target_workgroups, kMaxSplitTarget) : compute_units();
        const int64_t wgs = (int64_t)tiles.size() * n_kv_heads;
        int fill = 1;
        if (wgs * 2 <= target) fill = (int)std::min<int64_t>(kMaxPrefillSplits, target / wgs);
        int64_t total_blocks = 0;
        for (const Tile &t : tiles) total_blocks += (t.keys + kBlock - 1) / kBlock + kTileOverheadBlocks;
        // blocks one compute unit walks if the launch is shared out evenly, and the longest
        // walk a single workgroup may then have
        const int64_t share = (total_blocks * n_kv_heads + target - 1) / target;
        const int64_t cap = std::max<int64_t>(kMinSplitTokens / kBlock, share);
        int64_t above = 0;
        for (const Tile &t : tiles)
            if ((t.keys + kBlock - 1) / kBlock > cap) above += (t.keys + kBlock - 1) / kBlock;
        if (above * 4 > total_blocks) cut_long_walks = false;
        for (Tile &t : tiles) {
            const int64_t blocks = (t.keys + kBlock - 1) / kBlock;
            int64_t parts = std::max<int64_t>(fill, cut_long_walks ? (blocks + cap - 1) / cap : 1);
            parts = std::min<int64_t>(parts, kMaxPrefillSplits);
            parts = std::min<int64_t>(parts, std::max<int64_t>(1, t.keys / kMinSplitTokens));
            t.parts = (int32_t)parts;
            max_parts = std::max(max_parts, t.parts);
        }
    }
    int64_t n_entries = 0, n_slots = 0;
    for (Tile &t : tiles) {
        n_entries += t.parts;
        if (t.parts > 1) {
            t.first_slot = n_slots;
            n_slots += (int64_t)t.n_rows * t.parts;
        }
    }
    DSKV_REQUIRE(n_slots < (int64_t(1) << 31), "prefill_plan: too many partial slots");
    const int64_t words = n_entries * kTileWords + (max_parts > 1 ? 2 * nnz : 0);
    if (words > capacity_words) {
        set_error("prefill_plan: plan needs %lld words, buffer has %lld", (long long)words,
                  (long long)capacity_words);
        return DSKV_E_NOMEM;
    }
    int32_t *p = plan_host;
    int32_t *row_parts = plan_host + n_entries * kTileWords;
    if (max_parts > 1) std::fill(row_parts, row_parts + 2 * nnz, 0);
    for (const Tile &t : tiles) {
        // Parts of equal length, in units of four 32-token blocks (the kernel's loop is
        // unrolled by four), measured on the keys the tile sees under the causal mask; the
        // last part is open-ended.  The parts are disjoint and cover all blocks, so they are
        // also right without the mask (the last part then holds the rest of the request); a
        // part that starts past what the tile sees is empty.
        const int64_t blocks = (t.keys + kBlock - 1) / kBlock;
        const int64_t chunk = ((blocks + t.parts - 1) / t.parts + 3) / 4 * 4;
        for (int s = 0; s < t.parts; s++) {
            *p++ = t.b;
            *p++ = t.row;
            *p++ = (int32_t)(s * chunk);
            *p++ = s + 1 < t.parts ? (int32_t)((s + 1) * chunk) : kWholeRange;
            *p++ = t.parts > 1 ? (s | (t.parts << 8)) : -1;
            *p++ = (int32_t)t.first_slot;
        }
        if (t.parts > 1)
            for (int r = 0; r < t.n_rows; r++) {
                const int64_t row = (int64_t)qo_indptr_host[t.b] + t.row + r;
                row_parts[2 * row] = (int32_t)(t.first_slot + (int64_t)r * t.parts);
                row_parts[2 * row + 1] = t.parts;
            }
    }
    *n_tiles_out = (int32_t)n_entries;
    *n_splits_out = max_parts;
    *plan_words_out = words;
    *workspace_bytes_out = n_slots * (int64_t)n_qo_heads * (head_dim + 2) * (int64_t)sizeof(float);
    return 0;
}

}  // namespace dskv

extern "C" int dskv_prefill_plan(const int32_t *qo_indptr_host, const int32_t *kv_len_host,
                                 int32_t batch, int32_t n_qo_heads, int32_t n_kv_heads,
                                 int32_t head_dim, int32_t target_workgroups, int32_t *plan_host,
                                 int64_t capacity_words, int32_t *n_tiles_out,
                                 int32_t *n_splits_out, int64_t *plan_words_out,
                                 int64_t *workspace_bytes_out)
{
    using namespace dskv;
    DSKV_REQUIRE(batch >= 0 && n_tiles_out && n_splits_out && plan_words_out && workspace_bytes_out,
                 "prefill_plan: bad arguments");
    DSKV_REQUIRE(n_qo_heads > 0 && n_kv_heads > 0 && n_qo_heads % n_kv_heads == 0,
                 "prefill_plan: n_qo_heads %d not a multiple of n_kv_heads %d", n_qo_heads,
                 n_kv_heads);
    *n_tiles_out = 0;
    *n_splits_out = 1;
    *plan_words_out = 0;
    *workspace_bytes_out = 0;
    if (batch == 0) return 0;
    DSKV_REQUIRE(qo_indptr_host && plan_host, "prefill_plan: null pointer argument");
    return plan_tiles(qo_indptr_host, kv_len_host, nullptr, batch, n_qo_heads, n_kv_heads, head_dim,
                      target_workgroups, plan_host, capacity_words, n_tiles_out, n_splits_out,
                      plan_words_out, workspace_bytes_out);
}

// ---------------------------------------------------------------------------
// Mixed batches: one-row requests to the decode kernel, the others to query tiles
// ---------------------------------------------------------------------------
extern "C" int64_t dskv_mixed_plan_bound(int32_t batch, int64_t nnz, int64_t total_kv_tokens)
{
    if (batch < 0 || nnz < 0 || total_kv_tokens < 0) return 0;
    // tile entries, padding, the decode plan, the row map, the list of tiled rows and the
    // table of parts per row of a shared launch
    return dskv_prefill_plan_bound(batch, nnz) + 4 + dskv_decode_plan_bound(batch, total_kv_tokens) +
           (int64_t)batch + 3 * nnz + 8;
}

extern "C" int dskv_mixed_plan(const int32_t *qo_indptr_host, const int32_t *kv_page_indptr_host,
                               const int32_t *kv_last_page_len_host, int32_t batch,
                               int32_t page_size, int32_t n_qo_heads, int32_t n_kv_heads,
                               int32_t head_dim, int32_t target_workgroups,
                               int32_t route_one_row_requests, int32_t *plan_host,
                               int64_t capacity_words, dskv_mixed_plan_t *info)
{
    return dskv_mixed_plan_typed(qo_indptr_host, kv_page_indptr_host, kv_last_page_len_host, batch, page_size,
                                 n_qo_heads, n_kv_heads, head_dim, DSKV_BF16, target_workgroups,
                                 route_one_row_requests, plan_host, capacity_words, info);
}

extern "C" int dskv_mixed_plan_typed(const int32_t *qo_indptr_host, const int32_t *kv_page_indptr_host,
                                     const int32_t *kv_last_page_len_host, int32_t batch,
                                     int32_t page_size, int32_t n_qo_heads, int32_t n_kv_heads,
                                     int32_t head_dim, int32_t dtype, int32_t target_workgroups,
                                     int32_t route_one_row_requests, int32_t *plan_host,
                                     int64_t capacity_words, dskv_mixed_plan_t *info)
{
    using namespace dskv;
    DSKV_REQUIRE(info, "mixed_plan: null info pointer");
    *info = dskv_mixed_plan_t{};
    info->n_splits = 1;
    DSKV_REQUIRE(batch >= 0, "mixed_plan: negative batch");
    DSKV_REQUIRE(dtype == DSKV_F32 || dtype == DSKV_F16 || dtype == DSKV_BF16, "mixed_plan: unknown dtype %d", dtype);
    DSKV_REQUIRE(page_size > 0 && n_qo_heads > 0 && n_kv_heads > 0 && head_dim > 0 &&
                     n_qo_heads % n_kv_heads == 0,
                 "mixed_plan: bad shape (page %d, heads %d/%d, dim %d)", page_size, n_qo_heads,
                 n_kv_heads, head_dim);
    if (batch == 0) return 0;
    DSKV_REQUIRE(qo_indptr_host && kv_page_indptr_host && kv_last_page_len_host && plan_host,
                 "mixed_plan: null pointer argument");
    // One query row under the end-aligned mask sees every kv token of its request, with or
    // without the mask: exactly a decode row.  Routed only where the 16-bit decode kernel
    // takes the shape; a request without kv tokens stays with the tiles (a row of zeros).
    DSKV_REQUIRE(route_one_row_requests >= 0 && route_one_row_requests <= DSKV_ROUTE_SHARED_LAUNCH,
                 "mixed_plan: unknown routing mode %d", route_one_row_requests);
    const bool route = route_one_row_requests && decode_mfma_shape(head_dim, n_qo_heads, n_kv_heads, page_size);
    std::vector<int32_t> kv_len(batch);
    std::vector<char> routed(batch, 0);
    std::vector<DecodeRow> rows;
    int64_t n_tile_rows = 0;
    for (int b = 0; b < batch; b++) {
        const int64_t np = (int64_t)kv_page_indptr_host[b + 1] - kv_page_indptr_host[b];
        DSKV_REQUIRE(np >= 0, "mixed_plan: kv_page_indptr not monotone at %d", b);
        const int32_t last = kv_last_page_len_host[b];
        DSKV_REQUIRE(np == 0 || (last >= 1 && last <= page_size),
                     "mixed_plan: kv_last_page_len[%d] = %d outside [1, %d]", b, last, page_size);
        const int64_t len = np > 0 ? (np - 1) * page_size + last : 0;
        DSKV_REQUIRE(len < (int64_t(1) << 30), "mixed_plan: request %d too long", b);
        kv_len[b] = (int32_t)len;
        const int64_t n_b = (int64_t)qo_indptr_host[b + 1] - qo_indptr_host[b];
        DSKV_REQUIRE(n_b >= 0, "mixed_plan: qo_indptr not monotone at %d", b);
        if (route && n_b == 1 && len > 0) {
            routed[b] = 1;
            rows.push_back(DecodeRow{len, kv_page_indptr_host[b], qo_indptr_host[b]});
        } else {
            n_tile_rows += n_b;
        }
    }
    // How the routed rows run.  Without tiled rows: the decode kernel by itself (workgroups of
    // eight waves; 117 us where the same rows take 138 us as tiles).  With both kinds: one
    // launch of four-wave workgroups that share the CUs (pages of at least four tokens: the
    // tile side then loads straight into LDS) and one merge pass for both - if the decode rows
    // are worth it.  As a tile, a decode row is a workgroup with one live row of 64 that walks
    // all of the row's keys by itself; measured over steps of 8 to 75 decode rows beside one to
    // sixteen chunks (bf16, 8 kv heads, groups of 4 and 8), the shared launch wins by 3-40 %
    // where these one-row tiles would be at least half of the launch's tile work (blocks walked
    // plus a fixed cost per tile) and there are a dozen rows or more (75 rows + a 437-token
    // chunk behind 2506 tokens: 147 against 152 us, behind 8000: 171 against 188; 24 rows behind
    // 4096: 86 against 126; 75 rows of at most 300 tokens: 53 against 87), and loses 5-10 %
    // beside a large prefill batch (16 chunks of 512: its four-wave tiles move every K/V row
    // through the CU twice) or with a handful of rows.
    const int rows_per_tile = prefill_rows_per_tile(n_qo_heads, n_kv_heads, kPrefillWaves);
    int64_t decode_cost = 0, tile_cost = 0;
    for (const DecodeRow &r : rows) decode_cost += (r.len + kBlock - 1) / kBlock + kTileFixedCostBlocks;
    for (int b = 0; b < batch; b++) {
        const int64_t n_b = (int64_t)qo_indptr_host[b + 1] - qo_indptr_host[b];
        if (routed[b] || n_b == 0) continue;
        for (int64_t r0 = 0; r0 < n_b; r0 += rows_per_tile) {
            const int64_t keys = std::max<int64_t>(kv_len[b] - n_b + std::min<int64_t>(r0 + rows_per_tile, n_b), 0);
            tile_cost += (keys + kBlock - 1) / kBlock + kTileFixedCostBlocks;
        }
    }
    // How long a launch of tiles lasts that does not fill the chip: as long as its longest walk.  A few rows of long
    // context are such walks (of 343 blocks beside two prompts), cut into parts or not, where the shared launch spreads
    // them over all compute units; and as tiles they use up the parts that the chunks' tiles would be cut into.
    // Microseconds a layer, all as tiles -> shared (8 kv heads, groups of 4): one row of 900 tokens beside a prompt of 40
    // 25.7 -> 17.4, of 10000 beside three of 67 53.3 -> 22.7; four of 3000 beside two chunks of 512 behind 500 69 -> 42,
    // eleven of 150 beside a chunk of 512 behind 3000 88 -> 55; groups of 8, two of 10000 beside three of 67
    // 91 -> 29.  It loses where the walks are no longer than its own tiles' (two of 3000 beside a chunk of 512 behind 3000,
    // 44 blocks against 56: 54 -> 61; groups of 8, two of 3000 beside 200 behind 1000, 44 against 32: 40 -> 43; six of
    // 1100 to 1700 beside two of 47, 28 against 9: 26.7 -> 30.5), hence 3/2 of them and kLongWalkBlocks.
    // A dozen rows and more that are most of the work are tiles only where the kernel of short walks takes all of them whole
    // (twelve of 50 beside three prompts of 30: shared 14.9, tiles 9.2; sixteen of 55, groups of 8: 16.4 and 10.3; in two
    // parts, eleven of 150 beside 200 behind 1000: 29.6 and 33.5).  Errors against 64 bits are 0.99 of the shared launch's over
    // 260 such steps, 0.93 to 1.01 (of the rows alone 1.01, 1.03 at most; of the chunks 0.98).  The kernel of long walks would be faster for some
    // more (29 rows of 465 beside 78 tokens behind 253: 25.3 and 22.3), but raises its maximum more seldom: errors of the rows
    // 1.10 of the shared launch's, 1.15 at most.
    auto plan_all = [&](int layout, int64_t *words, bool in_parts = true) {
        const bool shared = layout == DSKV_LAYOUT_SHARED;
        return plan_tiles(qo_indptr_host, kv_len.data(), rows.empty() ? nullptr : routed.data(), batch, n_qo_heads, n_kv_heads,
                          head_dim, in_parts ? target_workgroups : -1, plan_host, capacity_words, &info->n_tiles, &info->n_splits, words,
                          &info->tile_workspace_bytes, shared ? kPrefillWavesShared : kPrefillWaves,
                          /* the tiles of a shared launch run beside decode workgroups for its whole length */ !shared);
    };
    // blocks of the plan's longest walk; spread: no less than what a compute unit gets of all of them
    auto walk_of_plan = [&](int waves, bool spread) {
        const int64_t tile_rows = prefill_rows_per_tile(n_qo_heads, n_kv_heads, waves);
        int64_t longest = 0, total = 0;
        for (int32_t i = 0; i < info->n_tiles; i++) {
            const int32_t *e = plan_host + (int64_t)i * kTileWords;
            const int64_t n_b = (int64_t)qo_indptr_host[e[0] + 1] - qo_indptr_host[e[0]];
            const int64_t keys = kv_len[e[0]] - n_b + std::min<int64_t>(e[1] + tile_rows, n_b);
            const int64_t blocks = std::max<int64_t>(std::min<int64_t>(e[3], (keys + kBlock - 1) / kBlock) - e[2], 0);
            longest = std::max(longest, blocks);
            total += blocks + kSharedTileOverheadBlocks;
        }
        return spread ? std::max(longest, total * n_kv_heads / compute_units()) : longest;
    };
    auto short_walks = [&] {
        if (target_workgroups != 0 || page_size < 8 || !is_pow2(page_size) ||
            !prefill_mfma_path(dtype, head_dim, n_qo_heads, n_kv_heads, 1.f))
            return 0;
        return short_walk_workgroups(qo_indptr_host, kv_len.data(), plan_host, info->n_tiles, n_qo_heads, n_kv_heads);
    };
    int layout = DSKV_LAYOUT_SEPARATE, rc = 0;
    int64_t tile_words = 0;
    bool planned = false;
    if (!rows.empty() && n_tile_rows > 0) {
        const bool can_share = page_size >= 4, choose = route_one_row_requests == DSKV_ROUTE_AUTO;
        const bool most = choose && (int64_t)rows.size() >= kMinSharedLaunchRows && decode_cost >= tile_cost;
        // (a caller with less room than any plan may need keeps the form that it has room for)
        const bool weighs = choose && target_workgroups == 0 && prefill_mfma_path(dtype, head_dim, n_qo_heads, n_kv_heads, 1.f) &&
                            capacity_words >= dskv_mixed_plan_bound(batch, qo_indptr_host[batch],
                                                                    std::accumulate(kv_len.begin(), kv_len.end(), int64_t(0)));
        // (only a launch that gives every tile a compute unit may be better than most rows shared)
        const bool may_fit = weighs &&
                             ((int64_t)rows.size() + (n_tile_rows + rows_per_tile - 1) / rows_per_tile) * n_kv_heads <= compute_units();
        if (route_one_row_requests == DSKV_ROUTE_SHARED_LAUNCH || (most && !may_fit))
            layout = can_share ? DSKV_LAYOUT_SHARED : DSKV_LAYOUT_SEPARATE;
        if (layout != DSKV_LAYOUT_SHARED && route_one_row_requests != DSKV_ROUTE_TWO_LAUNCHES) {
            // everything as tiles, and a look at whether that is the better form where sharing is possible
            const std::vector<DecodeRow> decode_rows = std::move(rows);
            const std::vector<char> decode_routed = routed;
            const int64_t chunk_rows = n_tile_rows;
            auto take_rows_out = [&](bool out) {
                if (out) rows = decode_rows, routed = decode_routed;
                else rows.clear(), std::fill(routed.begin(), routed.end(), 0);
            };
            take_rows_out(false);
            if ((rc = plan_all(layout, &tile_words))) return rc;
            planned = true;
            const int64_t walk = walk_of_plan(kPrefillWaves, false);
            const bool brief = info->n_splits == 1 && short_walks();
            bool shared = can_share && weighs && (most ? !brief : walk > kLongWalkBlocks);
            if (shared) {
                take_rows_out(true);
                if ((rc = plan_all(DSKV_LAYOUT_SHARED, &tile_words))) return rc;
                shared = most || 2 * (walk - kLongWalkBlocks) >= 3 * walk_of_plan(kPrefillWavesShared, true);
                if (!shared) {
                    take_rows_out(false);
                    if ((rc = plan_all(layout, &tile_words))) return rc;
                }
            }
            if (shared) layout = DSKV_LAYOUT_SHARED;
            n_tile_rows = shared ? chunk_rows : qo_indptr_host[batch];
        }
    }
    info->layout = layout;
    if (!planned && (rc = plan_all(layout, &tile_words))) return rc;
    const int tile_workgroups = rows.empty() ? short_walks() : 0;
    if (tile_workgroups && info->n_splits > 1 && (rc = plan_all(layout, &tile_words, false))) return rc;
    info->tile_workspace_bytes = (info->tile_workspace_bytes + 255) / 256 * 256;
    // whether every walk that meets new rows has kAppendAheadBlocks in front of them (tiles_append)
    info->tile_workgroups = tile_workgroups;
    info->new_rows_late = info->n_tiles > 0;
    for (int32_t i = 0; i < info->n_tiles && info->new_rows_late; i++) {
        const int32_t *e = plan_host + (int64_t)i * kTileWords;
        const int64_t prior = (int64_t)kv_len[e[0]] - (qo_indptr_host[e[0] + 1] - qo_indptr_host[e[0]]);
        const bool meets = e[3] == kWholeRange || (int64_t)e[3] * kBlock > prior;
        if (meets && ((int64_t)e[2] + kAppendAheadBlocks) * kBlock > prior) info->new_rows_late = 0;
    }
    info->n_tile_rows = (int32_t)n_tile_rows;
    int64_t at = (tile_words + 3) / 4 * 4;
    info->plan_words = tile_words;
    if (rows.empty()) return 0;
    info->decode_plan_at = at;
    int64_t decode_words = 0;
    if (at > capacity_words) at = capacity_words;   // the decode planner then reports the shortage
    std::fill(plan_host + tile_words, plan_host + std::max(at, tile_words), 0);   // (words of a plan made before)
    // shared launch: one decode workgroup (a share x a group of four kv heads) per compute unit
    int32_t decode_target = target_workgroups;
    if (layout == DSKV_LAYOUT_SHARED) {
        const int head_groups = (n_kv_heads + kSharedWaves - 1) / kSharedWaves;
        const int cus = target_workgroups > 0 ? std::min<int>(target_workgroups, kMaxWorkgroups) : compute_units();
        decode_target = std::max(1, cus / head_groups);
    }
    rc = plan_decode_rows(rows.data(), (int32_t)rows.size(), n_qo_heads, n_kv_heads, head_dim, dtype, false,
                          decode_target, plan_host + at, capacity_words - at, &info->n_decode_items,
                          &info->n_decode_workgroups, &decode_words, &info->decode_workspace_bytes);
    if (rc) return rc;
    info->n_decode_rows = (int32_t)rows.size();
    const int32_t *req_parts = plan_host + at + kPlanHeaderWords + info->n_decode_workgroups + 1;
    at += decode_words;
    // a shared launch merges the parts of both kinds of rows in one pass: behind the row map, a
    // table of (first slot, parts) for every row of the batch, the tile parts' slots first
    const int64_t nnz = qo_indptr_host[batch];
    const int64_t total = at + (int64_t)rows.size() + (layout == DSKV_LAYOUT_SHARED ? 2 * nnz : 0);
    if (total > capacity_words) {
        set_error("mixed_plan: plan needs %lld words, buffer has %lld", (long long)total,
                  (long long)capacity_words);
        return DSKV_E_NOMEM;
    }
    info->row_map_at = at;
    for (const DecodeRow &r : rows) plan_host[at++] = r.row;
    if (layout == DSKV_LAYOUT_SHARED) {
        int32_t *table = plan_host + at;
        if (info->n_splits > 1) std::copy_n(plan_host + (int64_t)info->n_tiles * kTileWords, 2 * nnz, table);
        else std::fill_n(table, 2 * nnz, 0);
        const int64_t slot_bytes = (int64_t)n_qo_heads * (head_dim + 2) * (int64_t)sizeof(float);
        const int64_t tile_slots = info->tile_workspace_bytes / slot_bytes;
        for (size_t i = 0; i < rows.size(); i++) {
            const int32_t first = req_parts[2 * i], n = req_parts[2 * i + 1];
            table[2 * (int64_t)rows[i].row] = n > 0 ? (int32_t)(tile_slots + first) : 0;
            table[2 * (int64_t)rows[i].row + 1] = n > 0 ? n : 0;
        }
    }
    info->plan_words = total;
    return 0;
}

namespace dskv {

static int launch_parts_merge(void *out, const float *part_o, const float *part_ml,
                              const int32_t *row_parts, int32_t nnz, int64_t max_slots,
                              int32_t n_qo_heads, int32_t dtype, hipStream_t s);

// some_rows_elsewhere: the tiles do not cover all nnz rows of the batch (the others are the
// decode kernel's); an MFMA-path call with n_tiles == 0 then has nothing to do.
static int prefill_attn_impl(void *out, const void *q, const int32_t *qo_indptr,
                             const void *pages_layer, const int32_t *kv_page_indices,
                             const int32_t *kv_page_indptr, const int32_t *kv_last_page_len,
                             const int32_t *plan_dev, int32_t n_tiles, int32_t n_splits,
                             void *workspace, int64_t workspace_bytes, int32_t batch, int32_t nnz,
                             int32_t n_qo_heads, int32_t n_kv_heads, int32_t head_dim,
                             int32_t page_size, float sm_scale, int32_t causal, int32_t dtype,
                             void *stream, bool some_rows_elsewhere, const float *rope_table = nullptr,
                             const AppendRows &append = AppendRows{}, int tile_workgroups = 0)
{
    DSKV_REQUIRE(batch >= 0 && nnz >= 0 && n_tiles >= 0, "prefill_attn: negative sizes");
    if (batch == 0 || nnz == 0) return 0;
    // kv_page_indices may be null when no request has a page (it is only read for requests that do)
    DSKV_REQUIRE(out && q && qo_indptr && pages_layer && kv_page_indptr && kv_last_page_len,
                 "prefill_attn: null pointer argument");
    DSKV_REQUIRE(dtype == DSKV_F32 || dtype == DSKV_F16 || dtype == DSKV_BF16,
                 "prefill_attn: unknown dtype %d", dtype);
    DSKV_REQUIRE(n_qo_heads > 0 && n_kv_heads > 0 && n_qo_heads % n_kv_heads == 0,
                 "prefill_attn: n_qo_heads %d not a multiple of n_kv_heads %d", n_qo_heads,
                 n_kv_heads);
    DSKV_REQUIRE(head_dim > 0 && head_dim <= 256, "prefill_attn: head_dim %d outside (0, 256]",
                 head_dim);
    DSKV_REQUIRE(page_size > 0, "prefill_attn: page_size must be positive");
    DSKV_REQUIRE(n_qo_heads <= 65535, "prefill_attn: too many heads");
    const float scale_log2 = sm_scale * 1.4426950408889634f;
    hipStream_t s = (hipStream_t)stream;
    const bool mfma = prefill_mfma_path(dtype, head_dim, n_qo_heads, n_kv_heads, scale_log2);
    if (mfma && some_rows_elsewhere && n_tiles == 0) return 0;   // every row went to the decode kernel
    if (mfma) {
        DSKV_REQUIRE(plan_dev && n_tiles > 0, "prefill_attn: missing plan");
        DSKV_REQUIRE(n_splits >= 1 && n_splits <= kMaxPrefillSplits,
                     "prefill_attn: tiles in up to %d parts", n_splits);
        float *part_o = nullptr, *part_ml = nullptr;
        int64_t max_slots = 0;
        if (n_splits > 1) {
            // the plan's partial slots are numbered from 0; the kernels never touch a slot at or
            // beyond max_slots, so a workspace smaller than the plan asked for loses rows, not memory
            const int64_t slot_bytes = (int64_t)n_qo_heads * (head_dim + 2) * (int64_t)sizeof(float);
            DSKV_REQUIRE(workspace && workspace_bytes >= slot_bytes && (uintptr_t)workspace % 16 == 0,
                         "prefill_attn: a plan with tiles in parts needs a 16-byte aligned workspace "
                         "(dskv_prefill_plan says how large), got %lld bytes", (long long)workspace_bytes);
            max_slots = std::min<int64_t>(workspace_bytes / slot_bytes, 1 << 30);
            part_o = reinterpret_cast<float *>(workspace);
            part_ml = part_o + max_slots * n_qo_heads * (int64_t)head_dim;
        }
        DSKV_REQUIRE(((uintptr_t)out | (uintptr_t)q | (uintptr_t)pages_layer) % 16 == 0,
                     "prefill_attn: out/q/pages must be 16-byte aligned");
        DSKV_REQUIRE(is_pow2(page_size),
                     "prefill_attn: 16-bit path needs a power-of-two page size, got %d", page_size);
        DSKV_REQUIRE((int64_t)n_tiles * n_kv_heads < (int64_t(1) << 31), "prefill_attn: too many tiles");
        dim3 grid((unsigned)n_tiles * (unsigned)n_kv_heads);
        dim3 block(64 * kPrefillWaves);
        const int shift = ilog2(page_size);
        // (the plan's choice; the rows are appended in front)
        if ((tile_workgroups == 2 || tile_workgroups == 4) && !append.k && n_splits == 1 && page_size >= 8 && n_tiles <= 65535) {
            const int group = n_qo_heads / n_kv_heads;
            const ShortArgs short_args = {plan_dev, qo_indptr, kv_page_indptr, kv_last_page_len, kv_page_indices,
                                          (const char *)pages_layer, (const uint16_t *)q, rope_table, (uint16_t *)out,
                                          n_qo_heads, n_kv_heads, group, 65536 / group + 1, shift, causal, scale_log2};
#define DSKV_LAUNCH_SHORT_W(DT, W, ROWS)                                                                         \
    hipLaunchKernelGGL((prefill_short_kernel<DT, W, ROWS>), dim3((unsigned)n_kv_heads, (unsigned)n_tiles, kPrefillWaves / W), \
                       dim3(64 * kShortWaves), 0, s, short_args)
#define DSKV_LAUNCH_SHORT(DT, ROWS)                                       \
    do {                                                                  \
        if (tile_workgroups == 4) DSKV_LAUNCH_SHORT_W(DT, 2, ROWS);       \
        else DSKV_LAUNCH_SHORT_W(DT, 4, ROWS);                            \
    } while (0)
            if (dtype == DSKV_BF16) {
                if (page_size >= 16) DSKV_LAUNCH_SHORT(DSKV_BF16, 16);
                else DSKV_LAUNCH_SHORT(DSKV_BF16, 8);
            } else {
                if (page_size >= 16) DSKV_LAUNCH_SHORT(DSKV_F16, 16);
                else DSKV_LAUNCH_SHORT(DSKV_F16, 8);
            }
#undef DSKV_LAUNCH_SHORT
#undef DSKV_LAUNCH_SHORT_W
            DSKV_LAUNCH_CHECK("prefill_short_kernel");
            return 0;
        }
        const PrefillArgs args = {append, (uint16_t *)out, (const uint16_t *)q, qo_indptr, (const char *)pages_layer,
                                  kv_page_indices, kv_page_indptr, kv_last_page_len, plan_dev, n_qo_heads, n_kv_heads,
                                  shift, scale_log2, causal, part_o, part_ml, (int)max_slots, rope_table};
#define DSKV_LAUNCH_PREFILL(DT, SHARE, APPENDS) \
    hipLaunchKernelGGL((prefill_attn_mfma_kernel<DT, SHARE, APPENDS>), grid, block, 0, s, args)
        if (dtype == DSKV_BF16) {
            if (append.k) DSKV_LAUNCH_PREFILL(DSKV_BF16, true, true);
            else if (page_size >= 4) DSKV_LAUNCH_PREFILL(DSKV_BF16, true, false);
            else DSKV_LAUNCH_PREFILL(DSKV_BF16, false, false);
        } else {
            if (append.k) DSKV_LAUNCH_PREFILL(DSKV_F16, true, true);
            else if (page_size >= 4) DSKV_LAUNCH_PREFILL(DSKV_F16, true, false);
            else DSKV_LAUNCH_PREFILL(DSKV_F16, false, false);
        }
#undef DSKV_LAUNCH_PREFILL
        DSKV_LAUNCH_CHECK("prefill_attn_mfma_kernel");
        if (n_splits > 1)   // the parts' partials become the output rows
            return launch_parts_merge(out, part_o, part_ml, plan_dev + (int64_t)n_tiles * kTileWords, nnz,
                                      max_slots, n_qo_heads, dtype, s);
    } else {
        DSKV_REQUIRE(!rope_table, "prefill_attn: only the 16-bit kernel rotates q");
        dim3 grid((unsigned)nnz, (unsigned)n_qo_heads);
#define DSKV_LAUNCH_GEN(DT)                                                                      \
    hipLaunchKernelGGL((prefill_attn_generic_kernel<DT>), grid, dim3(64), 0, s, out, q, qo_indptr, \
                       pages_layer, kv_page_indices, kv_page_indptr, kv_last_page_len, batch,    \
                       n_qo_heads, n_kv_heads, head_dim, page_size, scale_log2, causal)
        if (dtype == DSKV_F32) DSKV_LAUNCH_GEN(DSKV_F32);
        else if (dtype == DSKV_F16) DSKV_LAUNCH_GEN(DSKV_F16);
        else DSKV_LAUNCH_GEN(DSKV_BF16);
#undef DSKV_LAUNCH_GEN
        DSKV_LAUNCH_CHECK("prefill_attn_generic_kernel");
    }
    return 0;
}

// Merge pass of a tile plan with parts: one workgroup per query row of the batch (the decode
// path's merge kernel for rows in a few parts, see merge_kernel.h; one wave per (row, head)
// took 11.5 us for the 512 rows of a chunk, this about half); rows without parts return at once.
static int launch_parts_merge(void *out, const float *part_o, const float *part_ml,
                              const int32_t *row_parts, int32_t nnz, int64_t max_slots,
                              int32_t n_qo_heads, int32_t dtype, hipStream_t s)
{
    return launch_partials_merge(out, part_o, part_ml, row_parts, nullptr, (int)max_slots, nnz, n_qo_heads,
                                 kHeadDim, dtype, false, s);
}

// One launch for a batch of decode rows and chunks (layout DSKV_LAYOUT_SHARED), then the two
// merge passes.  The plan info comes from dskv_mixed_plan; everything in it that sizes a
// launch or an array is checked here.
static int mixed_shared_launch(void *out, const void *q, const int32_t *qo_indptr, const void *pages_layer,
                               const int32_t *kv_page_indices, const int32_t *kv_page_indptr,
                               const int32_t *kv_last_page_len, const int32_t *plan_dev,
                               const dskv_mixed_plan_t *info, void *workspace, int64_t workspace_bytes,
                               int32_t batch, int32_t nnz, int32_t n_qo_heads, int32_t n_kv_heads,
                               int32_t head_dim, int32_t page_size, float sm_scale, int32_t causal,
                               int32_t dtype, const float *rope_table, hipStream_t s)
{
    DSKV_REQUIRE(out && q && qo_indptr && pages_layer && kv_page_indices && kv_page_indptr && kv_last_page_len,
                 "mixed_attn: null pointer argument");
    DSKV_REQUIRE(decode_mfma_shape(head_dim, n_qo_heads, n_kv_heads, page_size) && page_size >= 4 &&
                     (dtype == DSKV_BF16 || dtype == DSKV_F16),
                 "mixed_attn: the shared launch takes 16-bit data, head_dim 128, groups up to 16 and "
                 "power-of-two pages of at least 4 tokens");
    DSKV_REQUIRE(((uintptr_t)out | (uintptr_t)q | (uintptr_t)pages_layer | (uintptr_t)workspace) % 16 == 0,
                 "mixed_attn: out/q/pages/workspace must be 16-byte aligned");
    DSKV_REQUIRE((int64_t)2 * page_size * n_kv_heads * head_dim * 2 < (int64_t(1) << 31),
                 "mixed_attn: a page must be smaller than 2 GiB");
    const int head_groups = (n_kv_heads + kSharedWaves - 1) / kSharedWaves;
    const int32_t n_rows = info->n_decode_rows, n_items = info->n_decode_items, shares = info->n_decode_workgroups;
    DSKV_REQUIRE(n_items >= n_rows && shares >= 1 && shares <= kMaxWorkgroups && info->n_tiles > 0 &&
                     info->n_splits >= 1 && info->n_splits <= kMaxPrefillSplits,
                 "mixed_attn: inconsistent plan (%d items of %d rows in %d shares, %d tile entries in up to %d parts)",
                 n_items, n_rows, shares, info->n_tiles, info->n_splits);
    const int64_t slot_bytes = (int64_t)n_qo_heads * (head_dim + 2) * (int64_t)sizeof(float);
    // workspace: the O partials of the tile parts' slots, then those of the cut decode rows'
    // slots, then the (maximum, sum) pairs in the same order - one numbering of slots, so that
    // one merge pass takes both kinds of rows
    MixedArgs a{};
    const int64_t tile_slots = info->tile_workspace_bytes / slot_bytes;
    const int64_t dec_slots = info->decode_workspace_bytes / slot_bytes;
    const int64_t all_slots = tile_slots + dec_slots;
    DSKV_REQUIRE(all_slots < (int64_t(1) << 30) && all_slots * slot_bytes <= workspace_bytes &&
                     (all_slots == 0 || workspace),
                 "mixed_attn: the plan's %lld partial slots need %lld bytes of workspace, got %lld",
                 (long long)all_slots, (long long)(all_slots * slot_bytes), (long long)workspace_bytes);
    DSKV_REQUIRE(info->n_splits == 1 || tile_slots >= 2, "mixed_attn: tiles in parts without partial slots");
    DSKV_REQUIRE(n_items == n_rows || dec_slots >= 2, "mixed_attn: cut decode rows without partial slots");
    float *const part_o = reinterpret_cast<float *>(workspace);
    float *const part_ml = part_o ? part_o + all_slots * n_qo_heads * (int64_t)head_dim : nullptr;
    a.tile_max_slots = (int)tile_slots;
    a.tile_part_o = part_o;
    a.tile_part_ml = part_ml;
    a.dec_max_slots = (int)dec_slots;
    a.dec_part_o = part_o ? part_o + tile_slots * n_qo_heads * (int64_t)head_dim : nullptr;
    a.dec_part_ml = part_ml ? part_ml + tile_slots * n_qo_heads * 2 : nullptr;
    const int32_t *dplan = plan_dev + info->decode_plan_at;
    a.wg_ptr = dplan + kPlanHeaderWords;
    const int32_t *req_parts = a.wg_ptr + shares + 1;
    a.items = reinterpret_cast<const Item *>(req_parts + 2 * (int64_t)n_rows);
    a.out = (uint16_t *)out;
    a.q = (const uint16_t *)q;
    a.pages = (const char *)pages_layer;
    a.kv_indices = kv_page_indices;
    a.n_qo_heads = n_qo_heads;
    a.n_kv_heads = n_kv_heads;
    a.page_shift = ilog2(page_size);
    a.scale_log2 = sm_scale * 1.4426950408889634f;
    DSKV_REQUIRE(a.scale_log2 > 1e-6f && a.scale_log2 < 1e6f, "mixed_attn: sm_scale out of range");
    a.n_decode_wgs = shares * head_groups;
    a.head_groups = head_groups;
    a.qo_indptr = qo_indptr;
    a.kv_indptr = kv_page_indptr;
    a.kv_last = kv_last_page_len;
    a.tile_info = plan_dev;
    a.causal = causal;
    a.rope = rope_table;
    const int64_t grid = (int64_t)a.n_decode_wgs + (int64_t)info->n_tiles * n_kv_heads;
    DSKV_REQUIRE(grid < (int64_t(1) << 31), "mixed_attn: too many workgroups");
    const dim3 g((unsigned)grid), b(64 * kSharedWaves);
#define DSKV_LAUNCH_MIXED(DT, PPT) hipLaunchKernelGGL((mixed_attn_kernel<DT, PPT>), g, b, 0, s, a)
    if (dtype == DSKV_BF16) {
        if (page_size >= kTile) DSKV_LAUNCH_MIXED(DSKV_BF16, 1);
        else if (page_size == 8) DSKV_LAUNCH_MIXED(DSKV_BF16, 2);
        else DSKV_LAUNCH_MIXED(DSKV_BF16, 0);
    } else {
        if (page_size >= kTile) DSKV_LAUNCH_MIXED(DSKV_F16, 1);
        else if (page_size == 8) DSKV_LAUNCH_MIXED(DSKV_F16, 2);
        else DSKV_LAUNCH_MIXED(DSKV_F16, 0);
    }
#undef DSKV_LAUNCH_MIXED
    DSKV_LAUNCH_CHECK("mixed_attn_kernel");
    // Rows cut into dozens of parts (a few very long decode rows): the decode path's wide merge
    // for them, then the tile parts' own pass.  Otherwise one pass over the table of all rows.
    const bool wide = (int64_t)n_items > 32 * (int64_t)n_rows;
    if (wide) {
        int rc = launch_partials_merge(out, a.dec_part_o, a.dec_part_ml, req_parts, plan_dev + info->row_map_at,
                                       a.dec_max_slots, n_rows, n_qo_heads, head_dim, dtype, true, s);
        if (rc) return rc;
        if (info->n_splits > 1)
            return launch_parts_merge(out, a.tile_part_o, a.tile_part_ml,
                                      plan_dev + (int64_t)info->n_tiles * kTileWords, nnz, a.tile_max_slots,
                                      n_qo_heads, dtype, s);
        return 0;
    }
    if (n_items > n_rows || info->n_splits > 1)
        return launch_parts_merge(out, part_o, part_ml, plan_dev + info->row_map_at + n_rows, nnz, all_slots,
                                  n_qo_heads, dtype, s);
    return 0;
}

}  // namespace dskv

extern "C" int dskv_prefill_attn(void *out, const void *q, const int32_t *qo_indptr,
                                 const void *pages_layer, const int32_t *kv_page_indices,
                                 const int32_t *kv_page_indptr, const int32_t *kv_last_page_len,
                                 const int32_t *plan_dev, int32_t n_tiles, int32_t n_splits,
                                 void *workspace, int64_t workspace_bytes, int32_t batch,
                                 int32_t nnz, int32_t n_qo_heads, int32_t n_kv_heads,
                                 int32_t head_dim, int32_t page_size, float sm_scale,
                                 int32_t causal, int32_t dtype, void *stream)
{
    return dskv::prefill_attn_impl(out, q, qo_indptr, pages_layer, kv_page_indices, kv_page_indptr,
                                   kv_last_page_len, plan_dev, n_tiles, n_splits, workspace,
                                   workspace_bytes, batch, nnz, n_qo_heads, n_kv_heads, head_dim,
                                   page_size, sm_scale, causal, dtype, stream, false);
}

namespace dskv {

static int mixed_attn_impl(void *out, const void *q, const int32_t *qo_indptr, const void *pages_layer,
                           const int32_t *kv_page_indices, const int32_t *kv_page_indptr,
                           const int32_t *kv_last_page_len, const int32_t *plan_dev,
                           const dskv_mixed_plan_t *info, void *workspace, int64_t workspace_bytes,
                           int32_t batch, int32_t nnz, int32_t n_qo_heads, int32_t n_kv_heads,
                           int32_t head_dim, int32_t page_size, float sm_scale, int32_t causal,
                           int32_t dtype, const float *rope_table, void *stream,
                           const AppendRows &append = AppendRows{})
{
    DSKV_REQUIRE(info, "mixed_attn: null plan info");
    DSKV_REQUIRE(info->n_decode_rows >= 0 && info->n_tile_rows >= 0 && info->n_tiles >= 0 &&
                     info->tile_workspace_bytes >= 0 && info->decode_workspace_bytes >= 0,
                 "mixed_attn: negative sizes in the plan info");
    const bool routed = info->n_decode_rows > 0;
    const float scale_log2 = sm_scale * 1.4426950408889634f;
    // Shapes and types outside the 16-bit kernels: the generic kernel computes every row
    // of the batch by itself, routed or not.
    const bool mfma = n_qo_heads > 0 && n_kv_heads > 0 && n_qo_heads % n_kv_heads == 0 &&
                      prefill_mfma_path(dtype, head_dim, n_qo_heads, n_kv_heads, scale_log2);
    if (!routed || !mfma)
        return prefill_attn_impl(out, q, qo_indptr, pages_layer, kv_page_indices, kv_page_indptr,
                                 kv_last_page_len, plan_dev, info->n_tiles, info->n_splits, workspace,
                                 workspace_bytes, batch, nnz, n_qo_heads, n_kv_heads, head_dim,
                                 page_size, sm_scale, causal, dtype, stream, false, rope_table, append,
                                 info->tile_workgroups);
    DSKV_REQUIRE(plan_dev, "mixed_attn: missing plan");
    DSKV_REQUIRE(info->n_decode_rows + info->n_tile_rows == nnz && info->n_decode_rows <= batch,
                 "mixed_attn: the plan covers %d + %d rows, the batch has %d", info->n_decode_rows,
                 info->n_tile_rows, nnz);
    DSKV_REQUIRE(workspace_bytes >= info->tile_workspace_bytes + info->decode_workspace_bytes &&
                     (workspace || info->tile_workspace_bytes + info->decode_workspace_bytes == 0),
                 "mixed_attn: the plan needs a workspace of %lld bytes, got %lld",
                 (long long)(info->tile_workspace_bytes + info->decode_workspace_bytes),
                 (long long)workspace_bytes);
    if (info->layout == DSKV_LAYOUT_SHARED)
        return mixed_shared_launch(out, q, qo_indptr, pages_layer, kv_page_indices, kv_page_indptr,
                                   kv_last_page_len, plan_dev, info, workspace, workspace_bytes, batch, nnz,
                                   n_qo_heads, n_kv_heads, head_dim, page_size, sm_scale, causal, dtype,
                                   rope_table, (hipStream_t)stream);
    // The one-row requests: the split-KV decode pass (each K/V byte read once, at the speed
    // of memory) and its merge; their partials lie behind those of the tile parts.
    int rc = decode_rows_attn(out, q, pages_layer, kv_page_indices, plan_dev + info->decode_plan_at,
                              info->n_decode_items, info->n_decode_workgroups,
                              workspace ? (char *)workspace + info->tile_workspace_bytes : nullptr,
                              workspace ? workspace_bytes - info->tile_workspace_bytes : 0,
                              info->n_decode_rows, plan_dev + info->row_map_at, n_qo_heads, n_kv_heads,
                              head_dim, page_size, sm_scale, dtype, rope_table, (hipStream_t)stream);
    if (rc) return rc;
    // The others: query tiles (and the merge of their parts, over the tiled rows only).
    return prefill_attn_impl(out, q, qo_indptr, pages_layer, kv_page_indices, kv_page_indptr,
                             kv_last_page_len, plan_dev, info->n_tiles, info->n_splits, workspace,
                             info->tile_workspace_bytes, batch, nnz, n_qo_heads, n_kv_heads, head_dim,
                             page_size, sm_scale, causal, dtype, stream, true, rope_table);
}

}  // namespace dskv

extern "C" int dskv_mixed_attn(void *out, const void *q, const int32_t *qo_indptr,
                               const void *pages_layer, const int32_t *kv_page_indices,
                               const int32_t *kv_page_indptr, const int32_t *kv_last_page_len,
                               const int32_t *plan_dev, const dskv_mixed_plan_t *info,
                               void *workspace, int64_t workspace_bytes, int32_t batch, int32_t nnz,
                               int32_t n_qo_heads, int32_t n_kv_heads, int32_t head_dim,
                               int32_t page_size, float sm_scale, int32_t causal, int32_t dtype,
                               void *stream)
{
    return dskv::mixed_attn_impl(out, q, qo_indptr, pages_layer, kv_page_indices, kv_page_indptr,
                                 kv_last_page_len, plan_dev, info, workspace, workspace_bytes, batch, nnz,
                                 n_qo_heads, n_kv_heads, head_dim, page_size, sm_scale, causal, dtype, nullptr,
                                 stream);
}

extern "C" int dskv_mixed_step_supported(int32_t n_qo_heads, int32_t n_kv_heads, int32_t head_dim,
                                         int32_t page_size, float sm_scale, int32_t dtype)
{
    using namespace dskv;
    return n_qo_heads > 0 && n_kv_heads > 0 && n_qo_heads % n_kv_heads == 0 && page_size > 0 &&
           is_pow2(page_size) &&
           prefill_mfma_path(dtype, head_dim, n_qo_heads, n_kv_heads, sm_scale * 1.4426950408889634f);
}

namespace dskv {

// Whether a step's attention launch appends the step's rows itself: tiles only (decode workgroups beside
// them, or a decode pass in front, would need theirs before), loaded straight into LDS, which meet new rows
// late, and few enough tokens for the first tiles' workgroups.  Rows have to be whole cache lines: see append_rows.h.
// Results and partials that lie where the new rows do are written when the rows have been read by a launch before.
static bool tiles_append(const dskv_mixed_step_t &s, const void *out, const void *k, const void *v, const void *pages_layer,
                         AppendRows &a)
{
    const uintptr_t out_bytes = (uintptr_t)s.nnz * s.n_qo_heads * s.head_dim * 2;
    const uintptr_t kv_bytes = (uintptr_t)s.nnz * s.n_kv_heads * s.head_dim * 2;
    for (const void *rows : {k, v}) {
        const uintptr_t at = (uintptr_t)rows, o = (uintptr_t)out, w = (uintptr_t)s.workspace;
        if ((at < o + out_bytes && o < at + kv_bytes) || (at < w + s.workspace_bytes && w < at + kv_bytes)) return false;
    }
    // (short walks are shared instead: 181 tokens behind 456 27.7 us a layer with the append in the launch, 22.9 shared, with
    // it in front; 512 behind 450 35.8 and 32.0)
    if (!s.info->new_rows_late || s.info->tile_workgroups || s.page_size < 4 || s.info->n_decode_rows > 0 || s.info->n_tiles <= 0 || s.batch > kAppendMaxBatch ||
        s.n_kv_heads > kAppendFlags || ((uintptr_t)pages_layer % 256) || (((uintptr_t)k | (uintptr_t)v) % 16))
        return false;
    a.n_tiles = std::min(s.info->n_tiles, kAppendFlags / s.n_kv_heads);
    a.tokens = (s.nnz + a.n_tiles - 1) / a.n_tiles;
    return a.tokens <= kAppendMaxTokens;
}

static int mixed_step(const dskv_mixed_step_t &s, void *out, const void *q, const void *k_new, const void *v_new,
                      void *pages_layer, uint64_t *flags, int32_t polls, void *stream)
{
    AppendRows append{};
    if (s.batch > 0 && s.nnz > 0) {
        DSKV_REQUIRE(pages_layer && k_new && v_new && s.qo_indptr && s.kv_page_indices && s.kv_page_indptr &&
                         s.kv_last_page_len, "append: null pointer argument");
        DSKV_REQUIRE(s.num_pages > 0, "append: num_pages must be positive, got %d", s.num_pages);
        if (flags && tiles_append(s, out, k_new, v_new, pages_layer, append)) {
            static std::atomic<uint64_t> launches{0};
            append.launch = launches.fetch_add(1, std::memory_order_relaxed) + 1;   // 0: a fresh buffer's
            append.k = (const uint16_t *)k_new;
            append.v = (const uint16_t *)v_new;
            append.flags = flags;
            append.nnz = s.nnz;
            append.batch = s.batch;
            append.num_pages = s.num_pages;
            append.polls[0] = polls & ~DSKV_APPEND_ODD_LATE;
            append.polls[1] = polls & DSKV_APPEND_ODD_LATE ? 0 : polls;
        }
    }
    if (!append.k) {
        const int rc = launch_append(pages_layer, s.num_pages, k_new, v_new, s.qo_indptr, s.kv_page_indices,
                                     s.kv_page_indptr, s.kv_last_page_len, s.batch, s.nnz, s.page_size, s.n_kv_heads,
                                     s.head_dim, 2, s.rope_table, s.dtype, (hipStream_t)stream);
        if (rc) return rc;
    }
    return mixed_attn_impl(out, q, s.qo_indptr, pages_layer, s.kv_page_indices, s.kv_page_indptr, s.kv_last_page_len,
                           s.plan_dev, s.info, s.workspace, s.workspace_bytes, s.batch, s.nnz, s.n_qo_heads,
                           s.n_kv_heads, s.head_dim, s.page_size, s.sm_scale, s.causal, s.dtype, s.rope_table, stream,
                           append);
}

}  // namespace dskv

// A batch's pages that take new rows are few; every other entry of the tables passes a filter of 8192 bits first.
extern "C" int dskv_new_rows_apart(const int32_t *qo_indptr_host, const int32_t *kv_page_indptr_host,
                                   const int32_t *kv_last_page_len_host, const int32_t *kv_page_indices_host,
                                   int32_t batch, int32_t page_size)
{
    using namespace dskv;
    if (batch <= 0) return 1;
    if (!qo_indptr_host || !kv_page_indptr_host || !kv_last_page_len_host || !kv_page_indices_host || page_size <= 0) return 0;
    // entries [first, end) of request b's table take its new rows
    auto first_new = [&](int32_t b, int64_t end) {
        const int64_t n_b = (int64_t)qo_indptr_host[b + 1] - qo_indptr_host[b];
        if (n_b <= 0) return end;
        const int64_t prior = (end - 1) * page_size + kv_last_page_len_host[b] - n_b;
        return std::min(end, std::max<int64_t>(prior, 0) / page_size);
    };
    try {
        std::vector<int32_t> taking;
        for (int pass = 0; pass < 2; pass++) {
            uint64_t filter[128] = {};
            for (const int32_t id : taking) filter[(uint32_t)id / 64 % 128] |= 1ull << ((uint32_t)id % 64);
            for (int32_t b = 0; b < batch; b++) {
                const int32_t *table = kv_page_indices_host + kv_page_indptr_host[b];
                const int64_t end = (int64_t)kv_page_indptr_host[b + 1] - kv_page_indptr_host[b];
                if (end <= 0) continue;
                const int64_t first = first_new(b, end);
                if (pass == 0) {
                    taking.insert(taking.end(), table + first, table + end);
                    continue;
                }
                for (int64_t i = 0; i < first; i++) {
                    const uint32_t id = (uint32_t)table[i];
                    if ((filter[id / 64 % 128] >> (id % 64) & 1) && std::binary_search(taking.begin(), taking.end(), table[i]))
                        return 0;
                }
            }
            if (pass == 0) {
                std::sort(taking.begin(), taking.end());
                if (std::adjacent_find(taking.begin(), taking.end()) != taking.end()) return 0;
            }
        }
    } catch (const std::bad_alloc &) {
        return 0;
    }
    return 1;
}

extern "C" int64_t dskv_append_flags(void) { return 2 * (dskv::kAppendFlags + 1); }

extern "C" int dskv_mixed_layers_flagged(const dskv_mixed_step_t *step, uint32_t *append_flags, int64_t n_append_flags,
                                         int32_t polls, int32_t n_layers, void *out, const void *q, const void *k_new,
                                         const void *v_new, void *pages, int64_t pages_layer_bytes, void *stream)
{
    using namespace dskv;
    DSKV_REQUIRE(step && n_layers >= 0 && step->nnz >= 0 && n_append_flags >= 0, "mixed_layers: bad arguments");
    if (n_layers == 0) return 0;
    const dskv_mixed_step_t &s = *step;
    DSKV_REQUIRE(dskv_mixed_step_supported(s.n_qo_heads, s.n_kv_heads, s.head_dim, s.page_size, s.sm_scale, s.dtype),
                 "mixed_step: shape, scale or type outside the 16-bit kernels (see dskv_mixed_step_supported)");
    DSKV_REQUIRE(s.info, "mixed_step: null plan info");
    DSKV_REQUIRE((uintptr_t)s.rope_table % 16 == 0, "mixed_step: the table must be 16-byte aligned");
    DSKV_REQUIRE(polls >= 0 && (uintptr_t)append_flags % 4 == 0, "mixed_layers: bad flags");
    // A captured launch would raise its flags with the same number in every replay, and find them raised
    if (append_flags) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (n_append_flags < dskv_append_flags() || (uintptr_t)append_flags % 8 || hipStreamIsCapturing((hipStream_t)stream, &capture) != hipSuccess ||
            capture != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            append_flags = nullptr;
        }
    }
    const int64_t q_bytes = (int64_t)s.nnz * s.n_qo_heads * s.head_dim * 2;
    const int64_t kv_bytes = (int64_t)s.nnz * s.n_kv_heads * s.head_dim * 2;
    auto at = [](const void *p, int64_t bytes) { return p ? (const char *)p + bytes : nullptr; };
    for (int64_t l = 0; l < n_layers; l++) {
        const int rc = mixed_step(s, (void *)at(out, l * q_bytes), at(q, l * q_bytes), at(k_new, l * kv_bytes),
                                  at(v_new, l * kv_bytes), (void *)at(pages, l * pages_layer_bytes), (uint64_t *)append_flags,
                                  polls & ~DSKV_APPEND_ODD_LATE ? polls : polls | kAppendPolls, stream);
        if (rc) return rc;
    }
    return 0;
}

extern "C" int dskv_mixed_layers(const dskv_mixed_step_t *step, int32_t n_layers, void *out, const void *q,
                                 const void *k_new, const void *v_new, void *pages, int64_t pages_layer_bytes,
                                 void *stream)
{
    return dskv_mixed_layers_flagged(step, nullptr, 0, 0, n_layers, out, q, k_new, v_new, pages, pages_layer_bytes, stream);
}

extern "C" int dskv_mixed_step(const dskv_mixed_step_t *step, void *out, const void *q, const void *k_new,
                               const void *v_new, void *pages_layer, void *stream)
{
    return dskv_mixed_layers(step, 1, out, q, k_new, v_new, pages_layer, 0, stream);
}
