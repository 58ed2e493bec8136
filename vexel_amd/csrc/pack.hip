// Continuous-batching step metadata built on the device (vx_pack_batch).
//
// Host restatement of what this replaces: the per-sequence loop of
// inference/runtime/decode.go:642-650 calling GPUBlockPool.StoreKV for every sequence
// (inference/runtime/gpu_block_pool.go:234-252: ensure blocks up to (endPos-1)/blockSize by
// popping the free list's tail, slot = (table[pos/bs], pos%bs)) and the length bookkeeping
// of gpu_block_pool.go:318-320,354-363. Because the host loop visits sequences in batch
// order and every layer's free list evolves identically, sequence i's new blocks are the
// entries free[F-1-rank_i-j], rank_i = exclusive prefix sum of the blocks needed by the
// sequences before it. Two prefix scans (blocks needed, new tokens) give every output.
#include <algorithm>

#include "common.h"
#include "rope_angle.h"

using namespace vx;

namespace {

constexpr int PK_THREADS = 1024;

// Exclusive scans over four values of each of blockDim.x threads; returns the exclusive prefixes and writes the totals to *total (the
// same in every thread). Each wave scans its 64 threads' by shuffles, all four values at every step (a shuffle is waited for, and one
// after the other they are most of a small step's launch), the first wave then the waves' sums (sm: at least PK_THREADS / 64).
__device__ int4 block_exclusive_scan4(const int4 v, int4 *sm, int4 *total) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_waves = blockDim.x >> 6;
    const auto inclusive = [&](int4 x, int most) {
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            if (off >= most) break;
            const int4 t = make_int4(__shfl_up(x.x, off, 64), __shfl_up(x.y, off, 64), __shfl_up(x.z, off, 64), __shfl_up(x.w, off, 64));
            if (lane >= off) x.x += t.x, x.y += t.y, x.z += t.z, x.w += t.w;
        }
        return x;
    };
    const auto minus = [](int4 a, int4 b) { return make_int4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w); };
    const int4 incl = inclusive(v, 64);
    if (n_waves == 1) {
        *total = make_int4(__shfl(incl.x, 63, 64), __shfl(incl.y, 63, 64), __shfl(incl.z, 63, 64), __shfl(incl.w, 63, 64));
        return minus(incl, v);
    }
    if (lane == 63) sm[wave] = incl;
    __syncthreads();
    if (wave == 0) {
        const int4 w = inclusive(lane < n_waves ? sm[lane] : make_int4(0, 0, 0, 0), PK_THREADS / 64);
        if (lane < n_waves) sm[lane] = w;          // inclusive sums of the waves
    }
    __syncthreads();
    *total = sm[n_waves - 1];
    const int4 e = minus(incl, v);
    if (wave == 0) return e;
    const int4 before = sm[wave - 1];
    return make_int4(before.x + e.x, before.y + e.y, before.z + e.z, before.w + e.w);
}

struct PackArgs {
    const int32_t *seq_slots, *positions, *q_lens;
    int batch, total_tokens;
    int32_t *block_tables;
    int max_blocks;
    int32_t *num_blocks, *free_list, *free_count;
    int block_size;
    int32_t *cu_seqlens, *token_pos, *slot_mapping, *kv_lens, *status, *items;
    int items_cap;
};
// By one workgroup of up to THREADS threads.
template <int THREADS>
__device__ __forceinline__ void pack_batch(const PackArgs &a) {
    const int32_t *seq_slots = a.seq_slots, *positions = a.positions, *q_lens = a.q_lens;
    const int batch = a.batch, total_tokens = a.total_tokens, max_blocks = a.max_blocks, block_size = a.block_size, items_cap = a.items_cap;
    int32_t *block_tables = a.block_tables, *num_blocks = a.num_blocks, *free_list = a.free_list, *free_count = a.free_count;
    int32_t *cu_seqlens = a.cu_seqlens, *token_pos = a.token_pos, *slot_mapping = a.slot_mapping, *kv_lens = a.kv_lens, *status = a.status;
    int32_t *items = a.items;
    __shared__ int4 sm[THREADS / 64];
    __shared__ int2 s_key[THREADS], s_partials[THREADS / 64];
    __shared__ int s_cu[THREADS + 1];
    __shared__ int4 s_seq[THREADS];  // position, slot, blocks it had, blocks taken by the sequences before it
    const int tid = threadIdx.x;
    const bool act = tid < batch;
    int slot = 0, pos = 0, ql = 0, have = 0, need = 0, block = 0;
    const int F = *free_count;
    if (act) {
        slot = seq_slots[tid];
        pos = positions[tid];
        ql = q_lens ? q_lens[tid] : 1;
        have = num_blocks[slot];
        block = block_tables[(size_t)slot * max_blocks + min(max(pos / block_size, 0), max_blocks - 1)];  // where the first new token goes, if it is there
        int end = pos + ql;
        int want = end > 0 ? (end - 1) / block_size + 1 : 0;
        need = want > have ? want - have : 0;
    }
    const int len = act ? pos + ql : 0;
    const int full[2] = {len / ATTN_TPW, len / (ATTN_TPW / 2)}, rest[2] = {len % ATTN_TPW, len % (ATTN_TPW / 2)};
    int4 totals;
    const int4 ahead = block_exclusive_scan4(make_int4(need, ql, full[0], full[1]), sm, &totals);
    const int rank = ahead.x, cu = ahead.y, off[2] = {ahead.z, ahead.w};
    const int total_need = totals.x, total_q = totals.y, total_full[2] = {totals.z, totals.w};
    bool fail = total_need > F || total_q != total_tokens;
    if (act && have + need > max_blocks) fail = true;
    // any thread's failure fails the step
    const bool any_fail = __syncthreads_or(fail ? 1 : 0) != 0;
    const bool ones = !q_lens || __syncthreads_and(!act || ql == 1) != 0;  // one new token each
    if (any_fail) {
        if (tid == 0) {
            *status = 1;
            if (items) {
                items[0] = 0;
                items[(items_cap + 1) * 4] = 0;
            }
        }
        return;
    }
    if (items) {
        // The attention work lists: one item per ATTN_TPW tokens of a sequence, and a second list in items of half
        // that for the kernels that take half as many tokens per workgroup (grouped queries). Equal (full) items
        // first, in batch order; then the partial last items from the longest down, so that the kernel's last
        // workgroups are its smallest. The second list sits behind the first one's capacity.
        // A partial item's key in each list: its tokens, then the earlier sequence (0: none). The items ahead of it are those of larger keys.
        int key[2], before[2] = {0, 0}, partials[2] = {0, 0};
#pragma unroll
        for (int which = 0; which < 2; which++) key[which] = rest[which] > 0 ? rest[which] * PK_THREADS + PK_THREADS - 1 - tid : 0;
        s_key[tid] = make_int2(key[0], key[1]);
        const int2 in_wave = make_int2(__popcll(__ballot(key[0] > 0)), __popcll(__ballot(key[1] > 0)));
        if ((tid & 63) == 0) s_partials[tid >> 6] = in_wave;
        __syncthreads();
        for (int w = 0; w < (int)blockDim.x >> 6; w++) partials[0] += s_partials[w].x, partials[1] += s_partials[w].y;
        if (act) {
#pragma unroll 8
            for (int j = 0; j < batch; j++) {
                const int2 other = s_key[j];
                before[0] += other.x > key[0];
                before[1] += other.y > key[1];
            }
        }
#pragma unroll
        for (int which = 0; which < 2; which++) {
            const int cap = which == 0 ? items_cap : 2 * items_cap;
            int32_t *list = which == 0 ? items : items + (items_cap + 1) * 4;
            const int n_items = total_full[which] + partials[which];
            if (act && n_items <= cap) {
                int4 *rec = (int4 *)(list + 4);  // one 16-byte record per item: everything a workgroup needs to start
                for (int s2 = 0; s2 < full[which]; s2++) rec[off[which] + s2] = make_int4(tid, s2, len, slot);
                if (rest[which] > 0) rec[total_full[which] + before[which]] = make_int4(tid, full[which], len, slot);
            }
            if (tid == 0) list[0] = n_items <= cap ? n_items : -1;  // -1: the list did not fit, not to be used
        }
    }
    if (act) {
        for (int j = 0; j < need; j++)
            block_tables[(size_t)slot * max_blocks + have + j] = free_list[F - 1 - (rank + j)];
        num_blocks[slot] = have + need;
        kv_lens[tid] = pos + ql;
        s_cu[tid] = cu;
        s_seq[tid] = make_int4(pos, slot, have, rank);
        cu_seqlens[tid] = cu;
    }
    if (tid == 0) {
        *free_count = F - total_need;
        *status = 0;
        s_cu[batch] = total_q;
        cu_seqlens[batch] = total_q;
    }
    if (ones) {  // (a new block's number from where the sequence takes it: not a trip behind the store of it)
        if (act) {
            const int j = pos / block_size - have;
            if (j >= 0 && pos >= 0) block = free_list[F - 1 - (rank + j)];
            token_pos[tid] = pos;
            slot_mapping[tid] = block * block_size + pos % block_size;
        }
        return;
    }
    __syncthreads();
    for (int t = tid; t < total_q; t += blockDim.x) {
        // binary search: largest i with s_cu[i] <= t
        int lo = 0, hi = batch - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (s_cu[mid] <= t)
                lo = mid;
            else
                hi = mid - 1;
        }
        const int4 seq = s_seq[lo];
        const int p = seq.x + (t - s_cu[lo]), j = p / block_size - seq.z;
        const int blk = j >= 0 && p >= 0 ? free_list[F - 1 - (seq.w + j)] : block_tables[(size_t)seq.y * max_blocks + p / block_size];
        token_pos[t] = p;
        slot_mapping[t] = blk * block_size + p % block_size;
    }
}

__global__ void __launch_bounds__(PK_THREADS) pack_batch_kernel(const PackArgs a) { pack_batch<PK_THREADS>(a); }

// The start of a step of one new token a sequence, in one launch: workgroup 0 packs the batch; the next ones take the uploaded words to where the
// step's other launches read them, the rows' angles, the rows' embeddings. What is uploaded is read where the host has put it, in pinned memory.
// Bound by what follows one another, in the host as on the device: the copy, the packing, the embedding and the angles were four
// launches of 2.4, 5.7, 3.3 and 3.5 us, this one takes 5.1 (32 rows of 2048 columns, no angles) to 7.4 (64 rows of 4096 with angles). A step of
// one row of a 7B model 2016 -> 2004 us, of eight of a 1.1B one 1197 -> 1178. 2048 columns a workgroup: every one waits for its token from
// pinned memory, and with 512 the 128 workgroups of 32 rows asked for so much of it that the launch took 9.3.
constexpr int BEGIN_THREADS = 64, BEGIN_WORDS = 1024, BEGIN_VECS = 8, BEGIN_COLS = BEGIN_VECS * 4 * BEGIN_THREADS;
struct BeginArgs {
    PackArgs pack;
    const int32_t *words;
    int32_t *words_to;
    int n_words, copies;     // workgroups of BEGIN_WORDS words
    int turns;               // workgroups of a row's angles: batch or 0
    float2 *turn_tab;
    int head_dim;
    float theta;
    const int32_t *ids;      // a row's embedding: `parts` workgroups of BEGIN_COLS columns each, or 0
    const float *table;
    float *out;
    int parts, vocab, dim;
};
__global__ void __launch_bounds__(BEGIN_THREADS) step_begin_kernel(const BeginArgs a) {
    const int tid = threadIdx.x;
    int i = blockIdx.x;
    if (i == 0) return pack_batch<BEGIN_THREADS>(a.pack);
    if (i -= 1; i < a.copies) {
#pragma unroll 4
        for (int w = i * BEGIN_WORDS + tid; w < min((i + 1) * BEGIN_WORDS, a.n_words); w += BEGIN_THREADS) a.words_to[w] = a.words[w];
        return;
    }
    if (i -= a.copies; i < a.turns) {
        const int position = a.pack.positions[i], half = a.head_dim / 2;
        for (int j = tid; j < half; j += BEGIN_THREADS) a.turn_tab[(size_t)i * half + j] = rope_angle(position, j, a.head_dim, a.theta);
        return;
    }
    i -= a.turns;
    const int row = i / a.parts, c0 = i % a.parts * BEGIN_COLS, id = a.ids[row];
    if (id < 0 || id >= a.vocab) return;  // row left untouched
    const float *src = a.table + (size_t)id * a.dim;
    float *dst = a.out + (size_t)row * a.dim;
    if (a.dim % 4 == 0 && ((uintptr_t)a.table | (uintptr_t)a.out) % 16 == 0) {
        float4 v[BEGIN_VECS];
#pragma unroll
        for (int e = 0; e < BEGIN_VECS; e++) {
            const int c = c0 + 4 * (tid + e * BEGIN_THREADS);
            v[e] = c < a.dim ? *(const float4 *)(src + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int e = 0; e < BEGIN_VECS; e++) {
            const int c = c0 + 4 * (tid + e * BEGIN_THREADS);
            if (c < a.dim) *(float4 *)(dst + c) = v[e];
        }
        return;
    }
    for (int c = c0 + tid; c < min(c0 + BEGIN_COLS, a.dim); c += BEGIN_THREADS) dst[c] = src[c];
}

// What both entry points require, and the attention's work list for a batch: items (null: no room for one) and its capacity.
int pack_check(vx_backend *be, PackArgs &a) {
    be->write_epoch++;  // positions and slots change
    VX_REQUIRE(a.seq_slots && a.positions && a.block_tables && a.num_blocks && a.free_list && a.free_count && a.cu_seqlens &&
                   a.token_pos && a.slot_mapping && a.kv_lens && a.status,
               "vx_pack_batch: null pointer");
    VX_REQUIRE(a.batch >= 1 && a.batch <= PK_THREADS, "vx_pack_batch: batch %d not in 1..%d", a.batch, PK_THREADS);
    VX_REQUIRE(a.block_size >= 1 && a.max_blocks >= 1 && a.total_tokens >= 0, "vx_pack_batch: bad sizes");
    // room for the attention work list: every sequence at the longest context its block table allows
    const size_t per_seq = ((size_t)a.max_blocks * a.block_size + ATTN_TPW - 1) / ATTN_TPW;
    const size_t cap = (size_t)a.batch * per_seq;
    be->items.valid = false;
    if (a.batch <= 32767 && per_seq <= 65535 &&
        ensure_ws(be, (void **)&be->items.buf, &be->items.bytes, (3 * cap + 2) * 4 * sizeof(int32_t), "attention work list") == VX_OK)
        a.items = be->items.buf;
    a.items_cap = (int)cap;
    return VX_OK;
}
void list_stands(vx_backend *be, const PackArgs &a, const int32_t *table_rows) {
    if (!a.items) return;
    be->items.kv_lens = a.kv_lens;
    be->items.table_rows = table_rows;
    be->items.batch = a.batch;
    be->items.cap = a.items_cap;
    be->items.valid = true;
}

}  // namespace

extern "C" int vx_pack_batch(vx_backend *be, const int32_t *seq_slots, const int32_t *positions,
                             const int32_t *q_lens, int batch, int total_tokens, int32_t *block_tables,
                             int max_blocks, int32_t *num_blocks, int32_t *free_list, int32_t *free_count,
                             int block_size, int32_t *cu_seqlens, int32_t *token_pos, int32_t *slot_mapping,
                             int32_t *kv_lens, int32_t *status) {
    int rc = enter(be);
    if (rc) return rc;
    PackArgs a{seq_slots, positions, q_lens, batch, total_tokens, block_tables, max_blocks, num_blocks, free_list, free_count, block_size,
               cu_seqlens, token_pos, slot_mapping, kv_lens, status, nullptr, 0};
    if (rc = pack_check(be, a); rc) return rc;
    // A wave for every 64 sequences or new tokens. Bound by what follows one another: trips to memory, shuffles, barriers. With 16 waves always,
    // four scans one behind the other, the ranks in two passes of eight instructions a sequence and each new token's block read back behind
    // the store of it 32 sequences of one token each took 12.0 us, now 5.7; one sequence 8.2, now 6.4.
    const int threads = std::min(PK_THREADS, ceil_div(std::max(batch, total_tokens), 64) * 64);
    pack_batch_kernel<<<1, threads, 0, be->stream>>>(a);
    VX_CHECK_LAUNCH();
    list_stands(be, a, seq_slots);
    return VX_OK;
}

extern "C" int vx_step_begin(vx_backend *be, const vx_step_begin_args *s) {
    int rc = enter(be);
    if (rc) return rc;
    VX_REQUIRE(s && s->dst && s->src_host && s->bytes > 0, "vx_step_begin: no upload");
    VX_REQUIRE(!be->capturing, "vx_step_begin during graph capture");
    VX_REQUIRE(!s->table || (s->ids && s->out && s->dim > 0), "vx_step_begin: bad embedding");
    VX_REQUIRE(s->rope_dim >= 0 && s->rope_dim % 2 == 0, "vx_step_begin: bad head size");
    const bool turns = s->rope_dim > 0;
    const auto at = [&](const int32_t *p) { return (uintptr_t)p - (uintptr_t)s->dst; };  // (of what is uploaded, where it is)
    const auto uploaded = [&](const int32_t *p) { return (uintptr_t)p >= (uintptr_t)s->dst && at(p) % 4 == 0 && at(p) + (size_t)s->batch * 4 <= s->bytes; };
    // A wave packs 64 sequences, and more rows' embeddings would ask for more pinned memory than their launch saves.
    const bool one_launch = s->batch >= 1 && s->batch <= BEGIN_THREADS && s->bytes % 4 == 0 && (uintptr_t)s->dst % 4 == 0 && s->bytes <= (64 << 10) &&
                            uploaded(s->seq_slots) && uploaded(s->positions) && (!s->table || uploaded(s->ids)) && device_memory(be, s->dst, s->bytes) &&
                            (!turns || (s->batch <= VX_ROPE_TAB_ROWS && s->rope_dim / 2 <= VX_ROPE_TAB_PAIRS));
    if (!one_launch) {
        if (rc = vx_to_device_staged(be, s->dst, s->src_host, s->bytes); rc) return rc;
        if (rc = vx_pack_batch(be, s->seq_slots, s->positions, nullptr, s->batch, s->batch, s->block_tables, s->max_blocks, s->num_blocks,
                               s->free_list, s->free_count, s->block_size, s->cu_seqlens, s->token_pos, s->slot_mapping, s->kv_lens, s->status);
            rc)
            return rc;
        if (s->table)
            if (rc = vx_embedding(be, s->ids, s->batch, s->table, s->out, s->vocab, s->dim); rc) return rc;
        return turns ? vx_rope_table_prepare(be, s->token_pos, s->batch, s->rope_dim, s->rope_theta) : (int)VX_OK;
    }
    PackArgs p{s->seq_slots, s->positions, nullptr, s->batch, s->batch, s->block_tables, s->max_blocks, s->num_blocks, s->free_list, s->free_count,
               s->block_size, s->cu_seqlens, s->token_pos, s->slot_mapping, s->kv_lens, s->status, nullptr, 0};
    items_written(be, s->dst, s->bytes);
    if (rc = pack_check(be, p); rc) return rc;
    std::lock_guard<std::mutex> g(be->stage_mu);
    const char *staged;
    if (rc = stage_upload(be, s->src_host, s->bytes, &staged); rc) return rc;
    p.seq_slots = (const int32_t *)(staged + at(s->seq_slots)), p.positions = (const int32_t *)(staged + at(s->positions));
    BeginArgs a;
    a.pack = p, a.words = (const int32_t *)staged, a.words_to = (int32_t *)s->dst, a.n_words = (int)(s->bytes / 4);
    a.copies = ceil_div(a.n_words, BEGIN_WORDS);
    a.turns = turns ? s->batch : 0, a.turn_tab = (float2 *)be->rope_tab, a.head_dim = s->rope_dim, a.theta = s->rope_theta;
    a.ids = s->table ? (const int32_t *)(staged + at(s->ids)) : nullptr, a.table = s->table, a.out = s->out, a.vocab = s->vocab, a.dim = s->dim;
    a.parts = s->table ? ceil_div(s->dim, BEGIN_COLS) : 0;
    step_begin_kernel<<<1 + a.copies + a.turns + s->batch * a.parts, BEGIN_THREADS, 0, be->stream>>>(a);
    VX_CHECK_LAUNCH();
    list_stands(be, p, s->seq_slots);
    be->rope_tab_pos = nullptr;
    if (turns) rope_table_stands(be, s->token_pos, s->batch, s->rope_dim, s->rope_theta);
    return VX_OK;
}

namespace {
__global__ void decode_advance_kernel(int32_t *tokens, int32_t *positions, const int32_t *next_tokens,
                                      int32_t *out_log, int32_t *step_counter, int batch) {
    const int i = threadIdx.x;
    const int step = *step_counter;
    __syncthreads();
    if (i < batch) {
        const int t = next_tokens[i];
        out_log[(size_t)step * batch + i] = t;
        tokens[i] = t;
        positions[i] += 1;
    }
    if (i == 0) *step_counter = step + 1;
}
}  // namespace

extern "C" int vx_decode_advance(vx_backend *be, int32_t *tokens, int32_t *positions, const int32_t *next_tokens,
                                 int32_t *out_log, int32_t *step_counter, int batch) {
    int rc = enter(be);
    if (rc) return rc;
    be->write_epoch++;  // positions move on
    VX_REQUIRE(tokens && positions && next_tokens && out_log && step_counter, "vx_decode_advance: null pointer");
    VX_REQUIRE(batch >= 1 && batch <= PK_THREADS, "vx_decode_advance: batch %d not in 1..%d", batch, PK_THREADS);
    decode_advance_kernel<<<1, PK_THREADS, 0, be->stream>>>(tokens, positions, next_tokens, out_log, step_counter,
                                                            batch);
    VX_CHECK_LAUNCH();
    return VX_OK;
}
