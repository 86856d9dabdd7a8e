// The step's new K/V rows, appended by the launch that attends to them: the workgroups of its first tiles write
// the rows of their kv head into their page slots, a share each, beside their first loads, and raise a flag;
// a tile looks at the flags of the rows that it needs before it requests the first block that holds one.
//
// What it saves is a launch in front of the attention (4.8 us for 512 tokens, most of it the start, the chain
// token -> request -> page -> store and the end of a launch): a chunk of 512 over 4096 904 -> 880 us in 16 layers.
// Workgroups that do nothing but append were tried first: one of eight waves and 250 registers fills its compute
// unit, so they ran in front of tiles and not beside them, and gained nothing; in the launch that tiles share
// with decode workgroups the loop of the tiles lost more (2341 -> 2395 us).  With
// more than kAppendMaxTokens a workgroup (16 chunks of 512) the launch in front stays: it moves bytes then, 14.7 us
// of 700 a layer, and a tile would start that much later.
//
// Rows that another compute unit reads in the same launch: they are stored with device scope (written
// through the L2 of the XCD), a flag is raised when all its stores are acknowledged, and blocks that hold
// new rows are loaded with device scope, too, when the flags have been seen.  So no line that an L2 has held from before
// is met, whoever brought it there - another stream's kernel that copies whole pages, for one.
//
// No order in which workgroups start is relied on: a wait is bounded, and a tile that has looked `polls` times in
// vain ends its walk there, before it requests a block with a new row, writes the rows that it needs itself - the
// same bytes to the same place - and walks again, with ordinary loads: its own stores have gone through
// the L1 and L2 that it reads through (rows are whole lines, 256 bytes at a multiple of 256).
#pragma once

#include "kv_tile.h"
#include "rope_math.h"

namespace dskv {

constexpr int kAppendFlags = 256;        // flags, at most: one per appending workgroup; behind them the count of second walks
constexpr int kAppendMaxTokens = 32;     // tokens of such a workgroup, at most: two for each lane half of eight waves
constexpr int kAppendMaxBatch = 63;      // requests, at most: a token's is found with one load and a ballot
// 32-token blocks that every walk has in front of its first new row, at least: a flag is raised four blocks into
// the walk of its workgroup.  Walks that begin with new rows - prompts - only wait: three short prompts took 358 us in
// 16 layers, 305 with the launch in front.
constexpr int kAppendAheadBlocks = 12;
constexpr int kAppendPolls = 256;        // looks at a flag (about 0.4 us each) before a tile appends itself

struct AppendRows {
    const uint16_t *k, *v;     // (nnz, Hkv, D) new rows; null: they are in the pages already
    uint64_t *flags;           // flag tile * Hkv + kv head, raised by writing `launch` to it
    uint64_t launch;           // a number no earlier launch of the process had
    int n_tiles, tokens;       // plan entries that append; tokens of each
    int nnz, batch, num_pages;
    int polls[2];              // looks at a flag of plan entries of even and of odd number
};
typedef const __attribute__((address_space(4))) AppendRows *const_append_ptr;

// The lane by itself, for code that would otherwise hold threadIdx in a register through a tile's walk.
__device__ __forceinline__ int lane_id()
{
    int none = 0;
    asm volatile("" : "+s"(none));
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
}

// 16 bytes with device scope.  (The data registers of a store of more than 8 bytes must not be written in the
// next cycle; what an asm statement stores the compiler does not know.)
__device__ __forceinline__ void store_through(char *p, u32x4 v)
{
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// A new row's chunk (lanes 0-15 of a half hold a token's K, 16-31 its V), K's rotated by its four pairs' angles.
template <int DT>
__device__ __forceinline__ u32x4 rotate_chunk(u32x4 raw, f32x4 c4, f32x4 s4)
{
    const float cs[4] = {c4[0], c4[1], c4[2], c4[3]}, sn[4] = {s4[0], s4[1], s4[2], s4[3]};
    float f[8];
    Chunk<DT>::unpack(raw, f);
    rope_rotate<4>(f, cs, sn);
    return Chunk<DT>::pack(f);
}

// Plan entry `tile`'s share of the rows of kv head kvh, tokens tile * tokens .. of the ragged batch, by the
// workgroup of that entry and head.  In three steps between the loads its walk begins with, so that none of the
// chain (token -> request -> page -> store) is waited for by itself; the flag is raised when the stores,
// by then a few requests old, have been acknowledged.
template <int DT, int kWaves>
struct AppendShare {
    static constexpr int kRounds = kAppendMaxTokens / (2 * kWaves);
    u32x4 raw[kRounds];
    f32x4 cs[kRounds], sn[kRounds];
    int q_i, p_i, l_i;             // lane i: entry i of qo_indptr, kv_indptr, kv_last
    long pos[kRounds], page[kRounds];   // page -1: no row of this lane's
    int begin, end;
    bool mine, found;

    // the rows, and what tells their requests - or, where that is the tile's own (tokens q_begin .. + n_b of the batch,
    // n_pages of the table from page_begin on, kv_len tokens), the pages and the angles at once
    __device__ __forceinline__ void request(const_append_ptr a, int tile, int kvh, int n_kv_heads, int wave,
                                            const int32_t *qo_indptr, const int32_t *kv_indptr, const int32_t *kv_last,
                                            int q_begin, int n_b, int page_begin, int kv_len, const int32_t *kv_indices,
                                            int page_shift, const float *rope)
    {
        asm volatile("" : "+s"(a));
        mine = tile < a->n_tiles;
        if (!mine) return;
        const int lane = lane_id(), nnz = a->nnz, batch = a->batch;
        begin = tile * a->tokens;
        end = min(begin + a->tokens, nnz);
        found = begin >= q_begin && end <= q_begin + n_b;
        if (found) {
#pragma unroll
            for (int i = 0; i < kRounds; i++) {
                const int t = begin + (i * kWaves + wave) * 2 + (lane >> 5);
                find(i, t, q_begin, n_b, page_begin, kv_len, lane, kv_indices, page_shift, rope);
            }
        } else {
            q_i = qo_indptr[min(lane, batch)];
            p_i = kv_indptr[min(lane, batch)];
            l_i = kv_last[min(lane, batch - 1)];
        }
        const uint16_t *const from = lane & 16 ? a->v : a->k;
#pragma unroll
        for (int i = 0; i < kRounds; i++) {
            const long t = min(begin + (i * kWaves + wave) * 2 + (lane >> 5), nnz - 1);
            raw[i] = *reinterpret_cast<const u32x4 *>(from + (t * n_kv_heads + kvh) * kHeadDim + (lane & 15) * 8);
        }
    }
    // the pages and the angles
    __device__ __forceinline__ void look_up(const_append_ptr a, int wave, const int32_t *kv_indices, int page_shift,
                                            const float *rope)
    {
        if (!mine || found) return;
        asm volatile("" : "+s"(a));
        const int lane = lane_id(), batch = a->batch;
#pragma unroll
        for (int i = 0; i < kRounds; i++) {
            const int t0 = begin + (i * kWaves + wave) * 2, t = t0 + (lane >> 5);
            // the request that owns a token: the largest b with qo_indptr[b] <= t
            const int b0 = __popcll(__ballot(lane <= batch && q_i <= t0)) - 1;
            const int b1 = __popcll(__ballot(lane <= batch && q_i <= t0 + 1)) - 1;
            const int b = min(max(lane >> 5 ? b1 : b0, 0), batch - 1);
            const int first = __shfl(q_i, b), n_b = __shfl(q_i, b + 1) - first;
            const int page_begin = __shfl(p_i, b), n_pages = __shfl(p_i, b + 1) - page_begin, last = __shfl(l_i, b);
            const long kv_len = n_pages > 0 ? ((long)(n_pages - 1) << page_shift) + last : 0;
            find(i, t, first, n_b, page_begin, kv_len, lane, kv_indices, page_shift, rope);
        }
    }
    // the page and the angles of round i's token t, of the request of tokens first .. + n_b
    __device__ __forceinline__ void find(int i, int t, int first, int n_b, int page_begin, long kv_len, int lane,
                                         const int32_t *kv_indices, int page_shift, const float *rope)
    {
        pos[i] = kv_len - n_b + (t - first);
        page[i] = -1;   // metadata that does not cover the token: touched by nobody
        if (t < end && t >= first && pos[i] >= 0 && pos[i] < kv_len) {
            page[i] = kv_indices[page_begin + (pos[i] >> page_shift)];
            if (rope) {
                const float *tab = rope + (long)t * kHeadDim + (lane & 15) * 4;   // dims 8 * chunk .. + 7: 4 pairs
                cs[i] = *reinterpret_cast<const f32x4 *>(tab);
                sn[i] = *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2);
            }
        }
    }
    __device__ __forceinline__ void store(const_append_ptr a, const char *pages, int page_shift, int row_bytes, int kvh,
                                          bool rotate)
    {
        if (!mine) return;
        asm volatile("" : "+s"(a));
        const int lane = lane_id(), num_pages = a->num_pages;
        const long half_bytes = (long)row_bytes << page_shift;
#pragma unroll
        for (int i = 0; i < kRounds; i++) {
            if (page[i] < 0 || page[i] >= num_pages) continue;   // an id outside the pool: touch nothing
            const u32x4 chunk = rotate && !(lane & 16) ? rotate_chunk<DT>(raw[i], cs[i], sn[i]) : raw[i];
            store_through(const_cast<char *>(pages) + page[i] * 2 * half_bytes + (lane & 16 ? half_bytes : 0) +
                              (pos[i] & ((1 << page_shift) - 1)) * row_bytes + kvh * (kHeadDim * 2) + (lane & 15) * 16,
                          chunk);
        }
    }
};

// Whether entries first .. last have raised their flags for kv head kvh, after as many looks as plan entry `tile` has.
// Called with a tile's registers full: the arguments are read where they are needed.
__device__ __forceinline__ bool rows_are_there(const_append_ptr a, int tile, int first, int last, int kvh, int n_kv_heads)
{
    asm volatile("" : "+s"(a));
    uint64_t *const flags = a->flags;
    const uint64_t launch = a->launch;
    const int polls = a->polls[tile & 1];
    const int lane = lane_id();
    for (int f = first; f <= last; f += 64) {
        bool there = false;
        for (int i = 0; i < polls && !there; i++) {
            if (i) __builtin_amdgcn_s_sleep(4);
            there = __ballot(__hip_atomic_load(flags + min(f + lane, last) * n_kv_heads + kvh, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT) != launch) == 0;
        }
        if (!there) return false;
    }
    return true;
}

// All n_b new rows of a request (tokens q_begin .. of the ragged batch) of kv head kvh, by one workgroup.
template <int DT, int kWaves>
__device__ __forceinline__ void append_request(const uint16_t *k, const uint16_t *v, int num_pages, int q_begin, int n_b,
                                               long kv_len, const char *pages, const int32_t *page_ids, int kvh,
                                               int n_kv_heads, int page_shift, const float *rope, int wave)
{
    const int lane = lane_id(), row_bytes = n_kv_heads * kHeadDim * 2;
    const long half_bytes = (long)row_bytes << page_shift;
    for (int i = 2 * wave + (lane >> 5); i < n_b; i += 2 * kWaves) {
        const long pos = kv_len - n_b + i;
        if (pos < 0) continue;
        const long page = page_ids[pos >> page_shift];
        if (page < 0 || page >= num_pages) continue;
        const long t = q_begin + i;
        u32x4 chunk = *reinterpret_cast<const u32x4 *>((lane & 16 ? v : k) + (t * n_kv_heads + kvh) * kHeadDim + (lane & 15) * 8);
        if (rope && !(lane & 16)) {
            const float *tab = rope + t * kHeadDim + (lane & 15) * 4;
            chunk = rotate_chunk<DT>(chunk, *reinterpret_cast<const f32x4 *>(tab),
                                     *reinterpret_cast<const f32x4 *>(tab + kHeadDim / 2));
        }
        store_through(const_cast<char *>(pages) + page * 2 * half_bytes + (lane & 16 ? half_bytes : 0) +
                          (pos & ((1 << page_shift) - 1)) * row_bytes + kvh * (kHeadDim * 2) + (lane & 15) * 16,
                      chunk);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

}  // namespace dskv
