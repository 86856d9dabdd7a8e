// KV append: scatter the new K/V rows of a ragged batch into their page slots.
// Pure byte movement (bit-exact by construction); HBM-bound for prefill chunks,
// launch-bound at decode sizes.
//
// Mapping: one 64-lane wavefront per token.  A token's K row set
// (n_kv_heads * head_dim elements, 2 KiB in bf16) is contiguous both in the
// source and in the page slot, so every lane moves 16 bytes per instruction and
// a wavefront moves 1 KiB per load/store pair, fully coalesced.
//
// A chunk of 8192 tokens is one round of waves on the chip (32 per CU), so the
// kernel lasts as long as its chain of dependent loads plus the copy itself, and
// for a few hundred tokens as the chain and the instructions in it: half of its 4 us
// are a launch's start and end.
// The chain is kept at two links: the token's rows are requested with what tells its
// request (neither address needs the other): the owner is found from ONE
// vector load of qo_indptr (lane i holds entry i; the owner is the number of
// entries <= t, a ballot and a popcount) instead of a binary search of
// dependent loads, with kv_page_indptr and kv_last_page_len fetched by the same
// lanes at the same time; the page id is the second link.  Batches over 63
// requests take the binary search.
// A wave's token is one, so everything between the links is scalar, the page of a power of two a
// shift, and the common row sets have code without bounds: 104 vector instructions instead of 249 for 8 kv heads
// with rotation.  Steps of a few prompts lost 0.5 to 0.7 us a layer of their 8 to 14 (3 prompts of 17 to 203: 13.95 ->
// 13.35; 16 of 16 tokens: 9.3 -> 8.6).
// Launches of many rows are bound by memory and take another form (kMany), see there.
// Nontemporal stores: ordinary ones made a small step 0.1 us a layer faster (the next launch finds some rows in
// its L2) and a mixed step of 512 tokens 2 us a layer slower (2334 -> 2368 us over 16 layers).
#include "kv_tile.h"
#include "rope_math.h"

namespace dskv {

constexpr int kAppendWaves = 4;
constexpr int kAppendMaxChunks = 4;   // 16-byte chunks per lane and row set held in registers (row sets <= 4 KiB)

// kRotate: K rows are rotated on their way (16-bit elements DT, head_dim 128).  `table` holds the
// token's 64 cosines and 64 sines; a lane's chunks lie 64 apart, so all of them are chunk lane % 16
// of a head and need the same four pairs.  Evaluating the angles here instead, as the stand-alone
// RoPE kernel does, is work and a barrier in every layer for values that are the same in all.
constexpr int kAppendRotatePairs = 64;   // dim pairs of a head
struct AppendArgs {
    char *pages;
    const char *k, *v;
    const int32_t *qo_indptr, *kv_indices, *kv_indptr, *kv_last;
    const float *table;
    int batch, nnz, row_bytes, num_pages;
    int page_size, page_shift;   // page_shift: -1 where page_size is no power of two
};

// kChunks: 16-byte chunks of a row set that a lane has in registers, where that is all of them (row sets of
// 1, 2 or 4 KiB); 0: any row set, up to four in registers, more of them copied after the lookup.
// kMany: for launches that memory bounds, with more K than kAppendManyBytes (half the waves of a full chip at 2 KiB a row
// set).  The rows are requested first, then the metadata, and the position and with it the page id are the vector
// unit's.  That chain is longer (512 tokens 3.2 us instead of 2.8) and lets many waves through faster: 16 x 512
// tokens of 8 heads, us without / with rotation, 13.1 / 13.0 -> 11.3 / 11.4 (5.9 TB/s).  Launches in a replayed
// graph, scalar form -> this one: 2048 tokens 4.7 / 4.7 -> 4.4 / 4.5, 4096 7.6 / 7.7 -> 6.7 / 6.9, 16384 25.1 / 24.1 ->
// 24.5 / 23.6; 16 heads, 1024 tokens 5.1 / 4.7 -> 4.9 / 5.0, 4096 13.4 / 13.3 -> 11.7 / 12.0; 4 heads, 4096 5.1 / 5.2 ->
// 4.8 / 5.0; 100 requests of 81 tokens 13.8 / 12.7 -> 12.2 / 12.2.  The line lies above the last size at which it still
// loses somewhere (4 MiB, 16 heads).
constexpr int64_t kAppendManyBytes = 4 << 20;
template <int DT, bool kRotate, int kChunks, bool kMany>
__global__ __launch_bounds__(64 * kAppendWaves) void append_kernel(const AppendArgs a)
{
    constexpr int kHeld = kChunks ? kChunks : kAppendMaxChunks;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int t = blockIdx.x * kAppendWaves + (kMany ? wave : __builtin_amdgcn_readfirstlane(wave));
    // (all arguments in one trip)
    asm volatile("" ::"s"(a.pages), "s"(a.k), "s"(a.v), "s"(a.qo_indptr), "s"(a.kv_indices), "s"(a.kv_indptr), "s"(a.kv_last),
                 "s"(a.table), "s"(a.batch), "s"(a.nnz), "s"(a.num_pages), "s"(a.page_size), "s"(a.page_shift));
    if (t >= a.nnz) return;

    // link 0: the rows themselves, and what tells the request
    const int row_bytes = kChunks ? kChunks * 1024 : a.row_bytes;
    const char *src_k = a.k + (long)t * row_bytes, *src_v = a.v + (long)t * row_bytes;
    const int batch = a.batch;
    const bool by_ballot = batch < 64;
    int q_i = 0, p_i = 0, l_i = 0;
    auto request_metadata = [&] {
        if (by_ballot) {
            q_i = a.qo_indptr[min(lane, batch)];
            p_i = a.kv_indptr[min(lane, batch)];
            l_i = a.kv_last[min(lane, batch - 1)];
        }
    };
    if (!kMany) request_metadata();
    const bool in_regs = kChunks || row_bytes <= kAppendMaxChunks * 64 * 16;
    u32x4 rk[kHeld], rv[kHeld];
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < kHeld; i++) {
            const int off = (i * 64 + lane) * 16;
            if (kChunks || off < row_bytes) {
                rk[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src_k + off));
                rv[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src_v + off));
            }
        }
    }
    f32x4 c4, s4;
    if (kRotate) {
        const float *tab = a.table + (long)t * (2 * kAppendRotatePairs) + (lane & 15) * 4;
        c4 = *reinterpret_cast<const f32x4 *>(tab);
        s4 = *reinterpret_cast<const f32x4 *>(tab + kAppendRotatePairs);
    }
    if (kMany) request_metadata();
    else asm volatile("" ::: "memory");   // (requested here, not where the branches below have met)
    auto k_chunk = [&](const u32x4 &raw) {
        if (!kRotate) return raw;
        const float cs[4] = {c4[0], c4[1], c4[2], c4[3]}, sn[4] = {s4[0], s4[1], s4[2], s4[3]};
        float f[Chunk<DT>::kElems];
        Chunk<DT>::unpack(raw, f);
        rope_rotate<4>(f, cs, sn);
        return Chunk<DT>::pack(f);
    };

    // link 1: request that owns token t = largest b with qo_indptr[b] <= t; the same for the whole wave
    int first, n_b, page_begin, n_pages, last;
    if (by_ballot) {
        const int b = min((int)__popcll(__ballot(lane <= batch && q_i <= t)) - 1, batch - 1);
        if (b < 0) return;   // qo_indptr[0] > t: malformed
        first = __builtin_amdgcn_readlane(q_i, b);
        n_b = __builtin_amdgcn_readlane(q_i, b + 1) - first;
        page_begin = __builtin_amdgcn_readlane(p_i, b);
        n_pages = __builtin_amdgcn_readlane(p_i, b + 1) - page_begin;
        last = __builtin_amdgcn_readlane(l_i, b);
    } else {
        const const_i32_ptr qo = as_const(a.qo_indptr);
        int lo = 0, hi = batch;  // invariant: qo_indptr[lo] <= t < qo_indptr[hi]
        if (t < batch && qo[t] == t && qo[t + 1] == t + 1) {
            lo = t;  // decode: one token per request
        } else {
            while (hi - lo > 1) {
                int mid = (lo + hi) >> 1;
                if (qo[mid] <= t) lo = mid; else hi = mid;
            }
        }
        first = qo[lo];
        n_b = qo[lo + 1] - first;
        page_begin = as_const(a.kv_indptr)[lo];
        n_pages = as_const(a.kv_indptr)[lo + 1] - page_begin;
        last = as_const(a.kv_last)[lo];
    }
    const long kv_len = (long)(n_pages - 1) * a.page_size + last;
    const long pos = kv_len - n_b + (t - first);
    if (n_pages <= 0 || pos < 0 || pos >= kv_len) return;  // malformed metadata: touch nothing
    // link 2: the page
    const int nth = a.page_shift >= 0 ? (int)(pos >> a.page_shift) : (int)(pos / a.page_size);
    const int page = as_const(a.kv_indices)[page_begin + nth];
    if (page < 0 || page >= a.num_pages) return;           // an id outside the pool: touch nothing
    const int slot = (int)(pos - (long)nth * a.page_size);

    const long half_bytes = (long)a.page_size * row_bytes;
    char *dst_k = a.pages + (long)page * 2 * half_bytes + (long)slot * row_bytes;
    char *dst_v = dst_k + half_bytes;
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < kHeld; i++) {
            const int off = (i * 64 + lane) * 16;
            if (kChunks || off < row_bytes) {
                __builtin_nontemporal_store(k_chunk(rk[i]), reinterpret_cast<u32x4 *>(dst_k + off));
                __builtin_nontemporal_store(rv[i], reinterpret_cast<u32x4 *>(dst_v + off));
            }
        }
    } else {
        for (int off = lane * 16; off < row_bytes; off += 64 * 16) {
            u32x4 x = *reinterpret_cast<const u32x4 *>(src_k + off);
            u32x4 y = *reinterpret_cast<const u32x4 *>(src_v + off);
            *reinterpret_cast<u32x4 *>(dst_k + off) = k_chunk(x);
            *reinterpret_cast<u32x4 *>(dst_v + off) = y;
        }
    }
}

// rope_table null: the rows are copied as they are (elements of elt_bytes); else dtype is 16-bit.
int launch_append(void *pages_layer, int32_t num_pages, const void *k, const void *v,
                  const int32_t *qo_indptr, const int32_t *kv_page_indices, const int32_t *kv_page_indptr,
                  const int32_t *kv_last_page_len, int32_t batch, int32_t nnz, int32_t page_size,
                  int32_t n_kv_heads, int32_t head_dim, int32_t elt_bytes, const float *rope_table,
                  int32_t dtype, hipStream_t stream)
{
    DSKV_REQUIRE(batch >= 0 && nnz >= 0, "append: negative batch/nnz (%d, %d)", batch, nnz);
    if (batch == 0 || nnz == 0) return 0;
    DSKV_REQUIRE(pages_layer && k && v && qo_indptr && kv_page_indices && kv_page_indptr &&
                     kv_last_page_len, "append: null pointer argument");
    DSKV_REQUIRE(page_size > 0 && n_kv_heads > 0 && head_dim > 0, "append: bad shape");
    DSKV_REQUIRE(num_pages > 0, "append: num_pages must be positive, got %d", num_pages);
    DSKV_REQUIRE(elt_bytes == 2 || elt_bytes == 4, "append: elt_bytes must be 2 or 4, got %d",
                 elt_bytes);
    const int64_t row_bytes = (int64_t)n_kv_heads * head_dim * elt_bytes;
    DSKV_REQUIRE(row_bytes % 16 == 0 && row_bytes < (1 << 30),
                 "append: a token's row set (%lld bytes) must be a multiple of 16 bytes",
                 (long long)row_bytes);
    DSKV_REQUIRE(((uintptr_t)pages_layer | (uintptr_t)k | (uintptr_t)v | (uintptr_t)rope_table) % 16 == 0,
                 "append: pages/k/v/table must be 16-byte aligned");
    DSKV_REQUIRE(!rope_table || (elt_bytes == 2 && head_dim == 2 * kAppendRotatePairs &&
                                 (dtype == DSKV_BF16 || dtype == DSKV_F16)),
                 "append: rotation by a table takes 16-bit rows of head_dim %d", 2 * kAppendRotatePairs);
    const unsigned grid = (unsigned)((nnz + kAppendWaves - 1) / kAppendWaves);
    const bool many = nnz * row_bytes > kAppendManyBytes;
    const AppendArgs args = {(char *)pages_layer, (const char *)k, (const char *)v, qo_indptr, kv_page_indices, kv_page_indptr,
                             kv_last_page_len, rope_table, batch, nnz, (int)row_bytes, num_pages, page_size,
                             is_pow2(page_size) ? ilog2(page_size) : -1};
#define DSKV_LAUNCH_APPEND_FORM(DT, ROTATE, CHUNKS, MANY) \
    hipLaunchKernelGGL((append_kernel<DT, ROTATE, CHUNKS, MANY>), dim3(grid), dim3(64 * kAppendWaves), 0, stream, args)
#define DSKV_LAUNCH_APPEND_CHUNKS(DT, ROTATE, CHUNKS)                          \
    do {                                                                       \
        if (many) DSKV_LAUNCH_APPEND_FORM(DT, ROTATE, CHUNKS, true);           \
        else DSKV_LAUNCH_APPEND_FORM(DT, ROTATE, CHUNKS, false);               \
    } while (0)
#define DSKV_LAUNCH_APPEND(DT, ROTATE)                                         \
    do {                                                                       \
        if (row_bytes == 1024) DSKV_LAUNCH_APPEND_CHUNKS(DT, ROTATE, 1);       \
        else if (row_bytes == 2048) DSKV_LAUNCH_APPEND_CHUNKS(DT, ROTATE, 2);  \
        else if (row_bytes == 4096) DSKV_LAUNCH_APPEND_CHUNKS(DT, ROTATE, 4);  \
        else DSKV_LAUNCH_APPEND_CHUNKS(DT, ROTATE, 0);                         \
    } while (0)
    if (!rope_table) DSKV_LAUNCH_APPEND(DSKV_BF16, false);
    else if (dtype == DSKV_BF16) DSKV_LAUNCH_APPEND(DSKV_BF16, true);
    else DSKV_LAUNCH_APPEND(DSKV_F16, true);
#undef DSKV_LAUNCH_APPEND_CHUNKS
#undef DSKV_LAUNCH_APPEND_FORM
#undef DSKV_LAUNCH_APPEND
    DSKV_LAUNCH_CHECK("append_kernel");
    return 0;
}

}  // namespace dskv

extern "C" int dskv_append_paged_kv(void *pages_layer, int32_t num_pages, const void *k, const void *v,
                                    const int32_t *qo_indptr, const int32_t *kv_page_indices,
                                    const int32_t *kv_page_indptr, const int32_t *kv_last_page_len,
                                    int32_t batch, int32_t nnz, int32_t page_size,
                                    int32_t n_kv_heads, int32_t head_dim, int32_t elt_bytes,
                                    void *stream)
{
    return dskv::launch_append(pages_layer, num_pages, k, v, qo_indptr, kv_page_indices, kv_page_indptr,
                               kv_last_page_len, batch, nnz, page_size, n_kv_heads, head_dim, elt_bytes,
                               nullptr, DSKV_BF16, (hipStream_t)stream);
}
