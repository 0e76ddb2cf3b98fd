// Paged grouped-query attention, plain variant: any head size up to 512, any page size, optional
// window; 32-bit or bfloat16 storage, all arithmetic in 32-bit on the vector units.  It is the
// 32-bit path of the engine and the fallback for head sizes that the matrix-core kernels do not take.
//
// Formula as in the reference: S = (q . k) * scale after the dot product, keys j <= position
// (inferrs-models/src/models/attention_utils.rs:61-85), softmax over keys, O = P v
// (inferrs-models/src/models/qwen3.rs:166-192); query head h reads key/value head
// h / (nq / nkv) (attention_utils.rs:38-49).
//
// A (token, query head) pair walks its keys in ascending order in tiles of 64 that are aligned to
// absolute position, with a running maximum and sum; a score is one chain of fused multiply-adds
// over the head's dimensions in ascending order, an output one chain over the tile's keys in
// ascending order.  Nothing in that order depends on how the tokens were cut into steps, on the other
// rows of the batch or on which pages hold the keys, so the result for a position is the same bit
// pattern under every cutting.  The keys are walked in segments of 512 (aligned to absolute position as well):
// a segment's maximum, sum and outputs are formed from nothing and then merged into the totals in ascending order.
// That merge is the same arithmetic whether one wave walks all segments of a token (steps of many tokens) or one
// wave a segment leaves them in memory for a merge kernel (steps of few tokens, which would otherwise keep a few
// waves busy for a long walk): both forms give the same bits.
//
// One wave a (token, key/value head, group of up to four of its query heads): the heads of a group share
// every key and value that is read.  A tile's keys come into shared memory 64 dimensions at a time in whole
// rows (a lane fetching a key's row for itself asks for 64 cache lines with every load), then lane j forms
// key j's scores with the queries broadcast from shared memory; the values come the same way, 64 dimensions
// x 64 keys as they lie in a page (dimension-major), and lane e adds up dimension e.  Keys outside the range
// of a token are staged as zeros and take the probability 0, so that what a page holds beyond a request's
// range never meets arithmetic.
#include "common.h"
#include "api.h"

#define AG_MAX_HEAD_DIM 512
#define AG_TILE 64                      // keys of a tile = lanes of a wave
#define AG_CHUNK 64                     // dimensions staged at a time
#define AG_PITCH 68                     // floats between staged rows: 16-byte aligned, no two of 16 lanes on a bank
#define AG_HEADS 4                      // query heads a wave takes together
#define AG_SEGMENT 512                  // keys of a segment
#define AG_SEG_TILES (AG_SEGMENT / AG_TILE)

__device__ __forceinline__ float4 ag_load4(const float* p) { return *(const float4*)p; }
__device__ __forceinline__ float4 ag_load4(const bf16_t* p) {
    const uint2 v = *(const uint2*)p;
    return make_float4(bf16_bits_to_f32((uint16_t)v.x), bf16_bits_to_f32((uint16_t)(v.x >> 16)),
                       bf16_bits_to_f32((uint16_t)v.y), bf16_bits_to_f32((uint16_t)(v.y >> 16)));
}

// Which keys a position sees and which tiles of them are walked: those below `keep` and those from `lo` on (keep < lo; keep
// 0: no first ones, or nothing between them and the rest is hidden).  The tiles hole_lo .. hole_hi - 1 hold none of them.
struct AgWalk {
    int lo, keep, hole_lo, hole_hi;
    __device__ __forceinline__ int from(int tile) const { return tile >= hole_lo && tile < hole_hi ? hole_hi : tile; }
    __device__ __forceinline__ int tile0() const { return from(0); }
    __device__ __forceinline__ bool skips(int seg) const { return seg * AG_SEG_TILES >= hole_lo && (seg + 1) * AG_SEG_TILES <= hole_hi; }
};
__device__ __forceinline__ AgWalk ag_walk(int pos, int window, int mask_chunk, int keep_first) {
    AgWalk w;
    w.lo = ia_key_floor(pos, window, mask_chunk);
    w.keep = keep_first;
    if (w.keep >= w.lo) { w.lo = 0; w.keep = 0; }
    w.hole_lo = (w.keep + AG_TILE - 1) / AG_TILE;
    w.hole_hi = w.lo / AG_TILE;
    return w;
}

// Totals (big_m, big_l, big_o) take in a segment (m, l, o): the one place where this is written down.
__device__ __forceinline__ void ag_merge_scales(float big_m, float m, float& m_out, float& a, float& b) {
    m_out = fmaxf(big_m, m);
    a = expf(big_m - m_out);
    b = expf(m - m_out);
}
// (written so that the compiler has no choice of which product to fuse: both forms must round alike)
__device__ __forceinline__ float ag_merge_value(float big, float a, float part, float b) { return fmaf(part, b, big * a); }

// VEC: the head size and the page size are multiples of four, so that four neighbouring dimensions of a key and
// four neighbouring keys of a value's dimension are fetched with one load.  HEADS: query heads of a group (1 to 4).
template <typename T, bool VEC, int HEADS, bool AHEAD>
__global__ __launch_bounds__(IA_WAVE) void attn_generic_kernel(
    T* __restrict__ out,                 // [n, nq, dv]
    const T* __restrict__ q,             // [n, nq, d]
    const T* __restrict__ k_cache,       // [pages, nkv, page_size, d]
    const T* __restrict__ v_cache,       // [pages, nkv, dv, page_size]  (transposed inside a page; dv: the values' width)
    const int* __restrict__ positions,   // [n]
    const int* __restrict__ token_seq,   // [n] row of block_table
    const int* __restrict__ block_table, // [seqs, max_pages]
    int max_pages, int nq, int nkv, int d, int dv, int page_size, int window, float scale,
    float* __restrict__ partial,         // null: a wave walks all segments; else [n, nq, segs, dpad + 2], a wave a segment
    int segs,
    int sink,                            // 1: the softmax's denominator holds one more term, exp(0): a key of score 0 without a value
    int mask_chunk,                      // > 0: a query sees the keys of its own chunk of this many positions only
    const float* __restrict__ sinks,     // with sink: null, or [nq] values s_h a query head; the term is exp(s_h), not scaled
    int keep_first,                      // the first so many positions are seen beside the window or chunk
    float softcap) {                     // > 0: a score becomes softcap * tanh(score / softcap)
    __shared__ __attribute__((aligned(16))) float stage[AG_TILE * AG_PITCH];     // keys: [key][dim]; values: [dim][key]
    __shared__ __attribute__((aligned(16))) float sp[HEADS][AG_TILE];
    extern __shared__ __attribute__((aligned(16))) float ag_rows[];       // queries, a segment's outputs, the totals: [HEADS][dpad] each
    const int lane = threadIdx.x;
    const int g = nq / nkv;
    const int groups = (g + HEADS - 1) / HEADS;
    const int unit = partial != nullptr ? blockIdx.x / segs : blockIdx.x;
    const int only_seg = partial != nullptr ? blockIdx.x - unit * segs : -1;
    const int tok = unit / (nkv * groups);
    const int rest = unit - tok * (nkv * groups);
    const int kvh = rest / groups;
    const int h0 = kvh * g + (rest - kvh * groups) * HEADS;            // first query head of the group
    const int heads = kvh * g + g - h0 < HEADS ? kvh * g + g - h0 : HEADS;
    const int pos = positions[tok];
    const int* bt = block_table + (size_t)token_seq[tok] * max_pages;
    const AgWalk wk = ag_walk(pos, window, mask_chunk, keep_first);
    const int lo = wk.lo, keep = wk.keep;
    auto seen = [&](int key) { return key <= pos && (key >= lo || key < keep); };
    const int chunks = (d + AG_CHUNK - 1) / AG_CHUNK;                  // of a key's dimensions
    const int vchunks = (dv + AG_CHUNK - 1) / AG_CHUNK;                // of a value's
    const int dpad = (chunks > vchunks ? chunks : vchunks) * AG_CHUNK;
    float* const sq = ag_rows;
    float* const so = ag_rows + HEADS * dpad;
    float* const st_ = ag_rows + 2 * HEADS * dpad;

    // the queries, zeros beyond the head size and for heads the group does not have
    for (int h = 0; h < HEADS; ++h)
        for (int e = lane; e < dpad; e += IA_WAVE)
            sq[h * dpad + e] = (h < heads && e < d) ? ld(q + ((size_t)tok * nq + h0 + h) * d + e) : 0.f;

    const int seg_first = wk.tile0() / AG_SEG_TILES, seg_last = pos / AG_SEGMENT;
    if (only_seg >= 0 && (only_seg < seg_first || only_seg > seg_last || wk.skips(only_seg))) return;       // (the whole wave)
    float big_m[HEADS], big_l[HEADS];
#pragma unroll
    for (int h = 0; h < HEADS; ++h) { big_m[h] = -INFINITY; big_l[h] = 0.f; }
    if (only_seg < 0)
        for (int h = 0; h < HEADS; ++h)
            for (int e = lane; e < dpad; e += IA_WAVE) st_[h * dpad + e] = 0.f;
    for (int seg = only_seg >= 0 ? only_seg : seg_first; seg <= (only_seg >= 0 ? only_seg : seg_last); ++seg) {
    if (wk.skips(seg)) continue;
    // the segment's outputs so far: lane e owns dimensions e, e + 64, ... of every head (nobody else touches them)
    for (int h = 0; h < HEADS; ++h)
        for (int e = lane; e < dpad; e += IA_WAVE) so[h * dpad + e] = 0.f;
    float m[HEADS], l[HEADS];
#pragma unroll
    for (int h = 0; h < HEADS; ++h) { m[h] = -INFINITY; l[h] = 0.f; }
    const int tile_first = wk.from(seg * AG_SEG_TILES);
    const int tile_last = seg * AG_SEG_TILES + AG_SEG_TILES - 1 < pos / AG_TILE ? seg * AG_SEG_TILES + AG_SEG_TILES - 1 : pos / AG_TILE;

    // ---- the pieces of a tile's work (the same arithmetic in the same order whoever stages the operands) -----------
    float s[HEADS], alpha[HEADS];
    // scores: lane j against key j, chunk c of the dimensions from the stage
    auto scores = [&](int c) {
        const float* mine = stage + lane * AG_PITCH;
#pragma unroll 4
        for (int e4 = 0; e4 < AG_CHUNK / 4; ++e4) {
            const float4 kv = *(const float4*)(mine + e4 * 4);
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                const float4 qv = *(const float4*)(sq + h * dpad + c * AG_CHUNK + e4 * 4);
                s[h] = fmaf(qv.x, kv.x, s[h]);
                s[h] = fmaf(qv.y, kv.y, s[h]);
                s[h] = fmaf(qv.z, kv.z, s[h]);
                s[h] = fmaf(qv.w, kv.w, s[h]);
            }
        }
    };
    // running maximum and sum; the tile's probabilities go to shared memory
    auto softmax = [&](bool valid) {
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            float sc = s[h] * scale;
            if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
            sc = valid ? sc : -INFINITY;
            const float m_new = fmaxf(m[h], wave_max(sc));
            const float p = valid ? expf(sc - m_new) : 0.f;
            alpha[h] = expf(m[h] - m_new);
            l[h] = l[h] * alpha[h] + wave_sum(p);
            sp[h][lane] = p;
            m[h] = m_new;
        }
    };
    // values: lane e adds up dimension c * 64 + e over the tile's keys from the stage
    auto values = [&](int c) {
        const float* mine = stage + lane * AG_PITCH;
        float o[HEADS];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) o[h] = so[h * dpad + c * AG_CHUNK + lane] * alpha[h];
#pragma unroll 4
        for (int k4 = 0; k4 < AG_TILE / 4; ++k4) {
            const float4 vv = *(const float4*)(mine + k4 * 4);
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                const float4 pv = *(const float4*)(&sp[h][k4 * 4]);
                o[h] = fmaf(pv.x, vv.x, o[h]);
                o[h] = fmaf(pv.y, vv.y, o[h]);
                o[h] = fmaf(pv.z, vv.z, o[h]);
                o[h] = fmaf(pv.w, vv.w, o[h]);
            }
        }
#pragma unroll
        for (int h = 0; h < HEADS; ++h) so[h * dpad + c * AG_CHUNK + lane] = o[h];
    };
    // key j's page of a tile, in lane j - j0: asked for once a tile, handed round
    auto tile_pages = [&](int tile) {
        const int j = tile * AG_TILE + lane;
        return seen(j) ? bt[j / page_size] : 0;
    };

    if constexpr (VEC && AHEAD) {
        // Steps of few tokens, a wave a segment.  A tile is 2 * chunks steps: the chunks of its keys, then the chunks of
        // its values.  A step's operands are asked for while the step before it is multiplied (a wave is alone in its
        // block and mostly alone on its SIMD: nobody else would hide the memory's latency), held in registers meanwhile
        // and put on the stage when it is free: a decode step of 8 requests at a context of 8,192 in 32-bit 220 -> 150 us
        // a layer.  (Steps of many tokens have waves enough on every SIMD, and the registers that hold a step's operands
        // would cost them a tenth of their speed.)
        constexpr int LOADS = AG_TILE / 4;
        static_assert(AG_TILE == AG_CHUNK, "a step of either kind is as many loads");
        const int steps = chunks + vchunks;
        float4 held[LOADS];
        // keys: a load instruction takes four keys' rows of the chunk, 16 lanes a row, four dimensions a lane;
        // values: four dimensions, 16 lanes a dimension, four neighbouring keys a lane (four keys never straddle a page)
        auto ask = [&](int tile, int step, int pages) {
            const int j0 = tile * AG_TILE;
            if (step < chunks) {
                const int e = step * AG_CHUNK + (lane & 15) * 4;
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    const int r = 4 * i + (lane >> 4);
                    const int key = j0 + r;
                    const int page = __shfl(pages, r);
                    held[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (seen(key) && e < d)
                        held[i] = ag_load4(k_cache + (((size_t)page * nkv + kvh) * page_size + key % page_size) * d + e);
                }
            } else {
                const int c = step - chunks;
                const int k4 = (lane & 15) * 4;
                const int key = j0 + k4;
                const int off = key % page_size;
                const bool any = (key + 3 >= lo && key <= pos) || key < keep;
                // the page of the four keys, from a lane whose key is in the range (a page that a window has passed is
                // not in the table any more; the keys of these four that are in the range share their page)
                const int first_in = key >= lo || key < keep ? k4 : (lo - j0 < AG_TILE ? lo - j0 : k4);
                const int page = __shfl(pages, first_in);
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    const int e = c * AG_CHUNK + 4 * i + (lane >> 4);
                    held[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (any && e < dv) held[i] = ag_load4(v_cache + (((size_t)page * nkv + kvh) * dv + e) * page_size + off);
                }
            }
        };
        // what was asked for goes on the stage; values of keys outside the token's range as zeros
        auto put = [&](int tile, int step) {
            if (step < chunks) {
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                    *(float4*)(stage + (4 * i + (lane >> 4)) * AG_PITCH + (lane & 15) * 4) = held[i];
            } else {
                const int k4 = (lane & 15) * 4;
                const int key = tile * AG_TILE + k4;
                const bool in0 = seen(key), in1 = seen(key + 1), in2 = seen(key + 2), in3 = seen(key + 3);
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    float4 v = held[i];
                    v.x = in0 ? v.x : 0.f;
                    v.y = in1 ? v.y : 0.f;
                    v.z = in2 ? v.z : 0.f;
                    v.w = in3 ? v.w : 0.f;
                    *(float4*)(stage + (4 * i + (lane >> 4)) * AG_PITCH + k4) = v;
                }
            }
        };
        int pages = tile_pages(tile_first);
        if (tile_first <= tile_last) ask(tile_first, 0, pages);
        for (int tile = tile_first, next; tile <= tile_last; tile = next) {
            next = wk.from(tile + 1);
            const int j = tile * AG_TILE + lane;
            const bool valid = seen(j);
            const int pages_next = next <= tile_last ? tile_pages(next) : 0;
#pragma unroll
            for (int h = 0; h < HEADS; ++h) s[h] = 0.f;
            for (int step = 0; step < steps; ++step) {
                if (step == chunks) softmax(valid);
                __syncthreads();                                      // the stage is free (and the probabilities are there)
                put(tile, step);
                if (step + 1 < steps) ask(tile, step + 1, pages);
                else if (next <= tile_last) ask(next, 0, pages_next);
                __syncthreads();
                if (step < chunks) scores(step);
                else values(step - chunks);
            }
            pages = pages_next;
        }
    } else {
    for (int tile = tile_first; tile <= tile_last; tile = wk.from(tile + 1)) {
        const int j0 = tile * AG_TILE;
        const int j = j0 + lane;
        const bool valid = seen(j);
        const int my_page = tile_pages(tile);
#pragma unroll
        for (int h = 0; h < HEADS; ++h) s[h] = 0.f;
        for (int c = 0; c < chunks; ++c) {
            __syncthreads();                                          // the stage is free
            if constexpr (VEC) {
                // a load instruction takes four keys' rows of this chunk: 16 lanes a row, four dimensions a lane
                const int e = c * AG_CHUNK + (lane & 15) * 4;
                float4 v[AG_TILE / 4];
#pragma unroll
                for (int i = 0; i < AG_TILE / 4; ++i) {
                    const int r = 4 * i + (lane >> 4);
                    const int key = j0 + r;
                    const int page = __shfl(my_page, r);
                    v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (seen(key) && e < d)
                        v[i] = ag_load4(k_cache + (((size_t)page * nkv + kvh) * page_size + key % page_size) * d + e);
                }
#pragma unroll
                for (int i = 0; i < AG_TILE / 4; ++i)
                    *(float4*)(stage + (4 * i + (lane >> 4)) * AG_PITCH + (lane & 15) * 4) = v[i];
            } else {
                for (int r = 0; r < AG_TILE; ++r) {
                    const int key = j0 + r, e = c * AG_CHUNK + lane;
                    float v = 0.f;
                    const int page = __shfl(my_page, r);
                    if (seen(key) && e < d)
                        v = ld(k_cache + (((size_t)page * nkv + kvh) * page_size + key % page_size) * d + e);
                    stage[r * AG_PITCH + lane] = v;
                }
            }
            __syncthreads();
            scores(c);
        }
        softmax(valid);
        for (int c = 0; c < vchunks; ++c) {
            __syncthreads();                                          // the stage is free, the probabilities are there
            if constexpr (VEC) {
                // a load instruction takes four dimensions: 16 lanes a dimension, four neighbouring keys a lane
                const int k4 = (lane & 15) * 4;
                const int key = j0 + k4;
                const int off = key % page_size;                      // (four keys never straddle a page)
                const bool any = (key + 3 >= lo && key <= pos) || key < keep;
                // the page of the four keys, from a lane whose key is in the range (a page that a window has passed is
                // not in the table any more; the keys of these four that are in the range share their page)
                const int first_in = key >= lo || key < keep ? k4 : (lo - j0 < AG_TILE ? lo - j0 : k4);
                const int page = __shfl(my_page, first_in);
                float4 v[AG_CHUNK / 4];
#pragma unroll
                for (int i = 0; i < AG_CHUNK / 4; ++i) {
                    const int e = c * AG_CHUNK + 4 * i + (lane >> 4);
                    v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (any && e < dv) {
                        v[i] = ag_load4(v_cache + (((size_t)page * nkv + kvh) * dv + e) * page_size + off);
                        v[i].x = seen(key) ? v[i].x : 0.f;
                        v[i].y = seen(key + 1) ? v[i].y : 0.f;
                        v[i].z = seen(key + 2) ? v[i].z : 0.f;
                        v[i].w = seen(key + 3) ? v[i].w : 0.f;
                    }
                }
#pragma unroll
                for (int i = 0; i < AG_CHUNK / 4; ++i)
                    *(float4*)(stage + (4 * i + (lane >> 4)) * AG_PITCH + k4) = v[i];
            } else {
                const int off = j % page_size;
                for (int r = 0; r < AG_CHUNK; ++r) {
                    const int e = c * AG_CHUNK + r;
                    stage[r * AG_PITCH + lane] =
                        (valid && e < dv) ? ld(v_cache + (((size_t)my_page * nkv + kvh) * dv + e) * page_size + off) : 0.f;
                }
            }
            __syncthreads();
            values(c);
        }
    }
    }
    // ---- the segment is done ---------------------------------------------------------------------------------------
    if (only_seg >= 0) {
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            if (h >= heads) break;
            float* row = partial + (((size_t)tok * nq + h0 + h) * segs + seg) * (dpad + 2);
            for (int e = lane; e < dpad; e += IA_WAVE) row[e] = so[h * dpad + e];
            if (lane == 0) { row[dpad] = m[h]; row[dpad + 1] = l[h]; }
        }
        return;
    }
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        float m_out, a, b;
        ag_merge_scales(big_m[h], m[h], m_out, a, b);
        big_l[h] = ag_merge_value(big_l[h], a, l[h], b);
        big_m[h] = m_out;
        for (int e = lane; e < dpad; e += IA_WAVE)
            st_[h * dpad + e] = ag_merge_value(st_[h * dpad + e], a, so[h * dpad + e], b);
    }
    }
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        if (h >= heads) break;
        T* orow = out + ((size_t)tok * nq + h0 + h) * dv;
        const float inv = 1.0f / (sink ? big_l[h] + expf((sinks != nullptr ? sinks[h0 + h] : 0.f) - big_m[h]) : big_l[h]);
        for (int e = lane; e < dv; e += IA_WAVE) st(orow + e, st_[h * dpad + e] * inv);
    }
}

// The segments of a (token, query head) that waves of their own have left in `partial`, merged in ascending order.
template <typename T>
__global__ __launch_bounds__(IA_WAVE) void attn_generic_merge_kernel(
    T* __restrict__ out, const float* __restrict__ partial, const int* __restrict__ positions, int nq, int d, int dpad,
    int window, int segs, int sink, int mask_chunk, const float* __restrict__ sinks, int keep_first) {
    const int lane = threadIdx.x;
    const int tok = blockIdx.x / nq, h = blockIdx.x - tok * nq;
    const int pos = positions[tok];
    const AgWalk wk = ag_walk(pos, window, mask_chunk, keep_first);
    float big_m = -INFINITY, big_l = 0.f;
    float big_o[AG_MAX_HEAD_DIM / IA_WAVE];
#pragma unroll
    for (int t = 0; t < AG_MAX_HEAD_DIM / IA_WAVE; ++t) big_o[t] = 0.f;
    // (a position beyond the caller's bound has segments that nobody wrote: they are left out rather than read)
    const int seg_last = pos / AG_SEGMENT < segs - 1 ? pos / AG_SEGMENT : segs - 1;
    for (int seg = wk.tile0() / AG_SEG_TILES; seg <= seg_last; ++seg) {
        if (wk.skips(seg)) continue;
        const float* row = partial + (((size_t)tok * nq + h) * segs + seg) * (dpad + 2);
        float m_out, a, b;
        ag_merge_scales(big_m, row[dpad], m_out, a, b);
        big_l = ag_merge_value(big_l, a, row[dpad + 1], b);
        big_m = m_out;
#pragma unroll
        for (int t = 0; t < AG_MAX_HEAD_DIM / IA_WAVE; ++t) {
            const int e = lane + t * IA_WAVE;
            if (e < dpad) big_o[t] = ag_merge_value(big_o[t], a, row[e], b);
        }
    }
    const float inv = 1.0f / (sink ? big_l + expf((sinks != nullptr ? sinks[h] : 0.f) - big_m) : big_l);
    T* orow = out + ((size_t)tok * nq + h) * d;
#pragma unroll
    for (int t = 0; t < AG_MAX_HEAD_DIM / IA_WAVE; ++t) {
        const int e = lane + t * IA_WAVE;
        if (e < d) st(orow + e, big_o[t] * inv);
    }
}

// Floats of the workspace that steps of few tokens need (0: the step has tokens enough for a wave each to walk
// all its segments).  `max_kv_len`: an upper bound of the positions + 1.
extern "C" long long ia_attention_generic_workspace(int n, int nq, int nkv, int d, int dv, int max_kv_len) {
    if (n <= 0 || nq <= 0 || nkv <= 0 || d <= 0 || dv <= 0 || max_kv_len <= AG_SEGMENT) return 0;
    const int g = nq / nkv;
    const int per_group = g < AG_HEADS ? g : AG_HEADS;
    const long long units = (long long)n * nkv * ((g + per_group - 1) / per_group);
    if (units >= 2048) return 0;
    const int segs = (max_kv_len + AG_SEGMENT - 1) / AG_SEGMENT;
    const int dpad = ((d > dv ? d : dv) + AG_CHUNK - 1) / AG_CHUNK * AG_CHUNK;
    return (long long)n * nq * segs * (dpad + 2);
}

extern "C" int ia_attention_generic(void* out, const void* q, const void* k_cache, const void* v_cache,
                                    const int* positions, const int* token_seq, const int* block_table,
                                    int n, int max_pages, int nq, int nkv, int d, int dv, int page_size,
                                    int window, float scale, int dtype, float* workspace, int max_kv_len,
                                    int sink, int mask_chunk, const float* sinks, int keep_first, float softcap,
                                    hipStream_t stream) {
    IA_CHECK(mask_chunk >= 0 && (sinks == nullptr || sink), "attention: mask_chunk %d must be >= 0 (0 = none), and sink values go with a sink", mask_chunk);
    IA_CHECK(keep_first >= 0 && softcap >= 0.f, "attention: keep_first %d and softcap %g must be >= 0 (0 = none)", keep_first, (double)softcap);
    IA_CHECK(n >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention: bad head counts nq=%d nkv=%d (n=%d)", nq, nkv, n);
    IA_CHECK(d > 0 && d <= AG_MAX_HEAD_DIM, "attention: head_dim %d is outside 1..%d", d, AG_MAX_HEAD_DIM);
    IA_CHECK(dv > 0 && dv <= AG_MAX_HEAD_DIM, "attention: the values' width %d is outside 1..%d", dv, AG_MAX_HEAD_DIM);
    IA_CHECK(page_size > 0 && max_pages > 0, "attention: bad page geometry page_size=%d max_pages=%d", page_size, max_pages);
    IA_CHECK(window >= 0, "attention: window %d must be >= 0 (0 = all keys)", window);
    if (n == 0) return 0;
    const int g = nq / nkv;
    const int per_group = g < AG_HEADS ? g : AG_HEADS;                 // query heads a wave takes together
    const int groups = (g + per_group - 1) / per_group;
    IA_CHECK((long long)n * nkv * groups < 2147483647LL, "attention: %d tokens x %d heads exceed the grid", n, nq);
    // a wave a segment when the workspace is given (ia_attention_generic_workspace says when it is needed)
    const int segs = workspace != nullptr ? (max_kv_len + AG_SEGMENT - 1) / AG_SEGMENT : 1;
    IA_CHECK(workspace == nullptr || (max_kv_len > 0 && ia_attention_generic_workspace(n, nq, nkv, d, dv, max_kv_len) > 0),
             "attention: a workspace goes with max_kv_len and a step of few tokens");
    IA_CHECK((long long)n * nkv * groups * segs < 2147483647LL, "attention: %d tokens x %d heads exceed the grid", n, nq);
    const unsigned grid = (unsigned)n * (unsigned)nkv * (unsigned)groups * (unsigned)segs;
    const int dpad = ((d > dv ? d : dv) + AG_CHUNK - 1) / AG_CHUNK * AG_CHUNK;
    const size_t rows_bytes = (size_t)3 * per_group * dpad * sizeof(float);
    const size_t elem = dtype == IA_F32 ? 4 : 2;
    // loads of four elements: rows of the caches start at multiples of four elements, on aligned arrays
    const bool vec = d % 4 == 0 && dv % 4 == 0 && page_size % 4 == 0 &&
                     (((uintptr_t)k_cache | (uintptr_t)v_cache) % (4 * elem)) == 0;
#define AG_ARGS(T) (T*)out, (const T*)q, (const T*)k_cache, (const T*)v_cache, positions, token_seq, block_table, max_pages, nq, nkv, \
        d, dv, page_size, window, scale, workspace, segs, sink, mask_chunk, sinks, keep_first, softcap
    // (a wave a segment, steps of few tokens: the operands are asked for a step ahead)
#define AG_LAUNCH(T, V, H) do { \
        if (V && workspace != nullptr) attn_generic_kernel<T, V, H, true><<<grid, IA_WAVE, rows_bytes, stream>>>(AG_ARGS(T)); \
        else attn_generic_kernel<T, V, H, false><<<grid, IA_WAVE, rows_bytes, stream>>>(AG_ARGS(T)); } while (0)
#define AG_HEADS_OF(T, V) do { \
        if (per_group == 1) AG_LAUNCH(T, V, 1); else if (per_group == 2) AG_LAUNCH(T, V, 2); \
        else if (per_group == 3) AG_LAUNCH(T, V, 3); else AG_LAUNCH(T, V, 4); } while (0)
    if (dtype == IA_F32) { if (vec) AG_HEADS_OF(float, true); else AG_HEADS_OF(float, false); }
    else if (dtype == IA_BF16) { if (vec) AG_HEADS_OF(bf16_t, true); else AG_HEADS_OF(bf16_t, false); }
    else IA_CHECK(false, "attention: unknown dtype %d", dtype);
#undef AG_HEADS_OF
#undef AG_LAUNCH
#undef AG_ARGS
    IA_LAUNCH_CHECK("attention_generic");
    if (workspace != nullptr) {
        if (dtype == IA_F32)
            attn_generic_merge_kernel<float><<<(unsigned)n * nq, IA_WAVE, 0, stream>>>((float*)out, workspace, positions, nq, dv, dpad, window, segs, sink, mask_chunk, sinks, keep_first);
        else
            attn_generic_merge_kernel<bf16_t><<<(unsigned)n * nq, IA_WAVE, 0, stream>>>((bf16_t*)out, workspace, positions, nq, dv, dpad, window, segs, sink, mask_chunk, sinks, keep_first);
        IA_LAUNCH_CHECK("attention_generic_merge");
    }
    return 0;
}

// ---- portions of prompts in 32 bits, on the matrix cores ---------------------------------------------------------
// What the kernel above does with a wave a token and key/value head, 16 (token, query head) columns a wave at a time:
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after the other, a fused multiply-add each, so that a
// score with its dimensions ascending and an output with its keys ascending are the chains of that kernel, and with the same
// running maxima, sums (the butterfly's tree of additions) and segments the results are the same bits (tested).
//
// What bounds it: at 555 tokens the longest walk, nine tiles one after the other; a tile costs a wave 8,192 cycles of matrix
// products.  The kernel above brings every key and value once a token: 8B shape, 555 tokens, 309 us a layer by it, 104
// by this one.  A block of four waves owns 64 columns of a key/value head and shares a tile of 64 keys and values in shared
// memory, two blocks a compute unit; blocks of the latest tokens, whose walks are longest, start first.
//
// Row i of a product's tile of 16 keys is key 4 (i % 4) + i / 4 of them: lane (column r, group G) then holds the probabilities of the
// keys 4 s + G, which is where the second product's operand of step s wants them.  Columns of one wave see different keys: a key
// that a column does not see has the probability 0 there, and that product leaves its sums as they are unless the value is
// no number or infinite.  A tile with such a value is added up on the vector units, each column with its own keys.
typedef float ag_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float ag_pair_sum(float x, bool half) {
    const uint32_t u = __float_as_uint(x);
    if (half) {
        auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn_portions_f32_kernel(
    float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int* __restrict__ positions, const int* __restrict__ token_seq, const int* __restrict__ block_table,
    int n, int max_pages, int nq, int nkv, int page_size, int window, float scale, int sink, int mask_chunk,
    const float* __restrict__ sinks, int keep_first, float softcap) {
    constexpr int KP = D + 4, VP = AG_TILE + 4, DT = D / 16;
    __shared__ __attribute__((aligned(16))) float sk[AG_TILE * KP];     // [key][dim]
    __shared__ __attribute__((aligned(16))) float sv[D * VP];           // [dim][key]
    __shared__ int s_bad;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, G = lane >> 4;
    const int g = nq / nkv, kvh = blockIdx.y;
    const int first_col = (gridDim.x - 1 - blockIdx.x) * 64;
    const int tok_first = first_col / g, tok_last = min((first_col + 63) / g, n - 1);
    const int col = first_col + 16 * wave + r;
    const int tok = min(col / g, n - 1), head = kvh * g + col % g;
    const bool col_in = col < n * g;
    const int pos = positions[tok];
    const AgWalk wk = ag_walk(pos, window, mask_chunk, keep_first);
    auto seen = [&](int key) __attribute__((always_inline)) { return key <= pos && (key >= wk.lo || key < wk.keep); };
    float qf[D / 4];
#pragma unroll
    for (int i = 0; i < D / 4; ++i) qf[i] = q[((size_t)tok * nq + head) * D + 4 * i + G];

    // Tokens of one request at a time (lane i: the block's i-th token).
    const int my_tok = min(tok_first + lane, tok_last);
    const int my_seq = token_seq[my_tok], my_pos = positions[my_tok];
    const AgWalk my_walk = ag_walk(my_pos, window, mask_chunk, keep_first);
    for (int run = tok_first, run_end; run <= tok_last; run = run_end) {
        const int seq = __shfl(my_seq, run - tok_first);
        const unsigned long long others = __ballot(my_seq != seq || tok_first + lane > tok_last) >> (run - tok_first);
        run_end = others ? run + __ffsll(others) - 1 : tok_last + 1;
        const bool mine = tok_first + lane >= run && tok_first + lane < run_end;
        const int max_pos = (int)wave_max(mine ? (float)my_pos : -1.f);             // (positions are exact in 32-bit floats)
        const int min_lo = -(int)wave_max(mine ? -(float)my_walk.lo : -16777216.f);
        const int max_keep = (int)wave_max(mine ? (float)my_walk.keep : 0.f);
        const int* bt = block_table + (size_t)seq * max_pages;
        auto key_in = [&](int key) __attribute__((always_inline)) { return key <= max_pos && (key >= min_lo || key < max_keep); };
        const bool in = col_in && tok >= run && tok < run_end;

        float m = -INFINITY, l = 0.f, big_m = -INFINITY, big_l = 0.f;
        bool any_in_seg = false;
        ag_f32x4 o[DT], big_o[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = big_o[t] = (ag_f32x4){0.f, 0.f, 0.f, 0.f};
        auto end_segment = [&]() __attribute__((always_inline)) {
            float m_out, a, b;
            ag_merge_scales(big_m, m, m_out, a, b);
            if (any_in_seg) {
                big_l = ag_merge_value(big_l, a, l, b);
                big_m = m_out;
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    big_o[t][i] = any_in_seg ? ag_merge_value(big_o[t][i], a, o[t][i], b) : big_o[t][i];
                    o[t][i] = 0.f;
                }
            m = -INFINITY;
            l = 0.f;
            any_in_seg = false;
        };
        const int tile_last = max_pos / AG_TILE;
        int seg = -1;
        for (int tile = max_keep > 0 ? 0 : min_lo / AG_TILE; tile <= tile_last; ++tile) {
            const int j0 = tile * AG_TILE;
            if (j0 + AG_TILE - 1 < min_lo && j0 >= max_keep) continue;
            if (seg >= 0 && tile / AG_SEG_TILES != seg) end_segment();
            seg = tile / AG_SEG_TILES;
            // ---- the tile into shared memory: keys and values that no column of this request sees as zeros ------------------
            const int j4 = (j0 + lane) & ~3;
            const bool near_in = key_in(j4) || key_in(j4 + 1) || key_in(j4 + 2) || key_in(j4 + 3);      // (four keys share a page)
            const int my_page = near_in ? bt[(j0 + lane) / page_size] : 0, my_off = (j0 + lane) % page_size;
            float4 piece[D / 16];
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
                const int p = tid + 256 * i, key = p / (D / 4), e = p % (D / 4) * 4;
                const int page = __shfl(my_page, key), off = __shfl(my_off, key);
                piece[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (key_in(j0 + key)) piece[i] = *(const float4*)(k_cache + (((size_t)page * nkv + kvh) * page_size + off) * D + e);
            }
            __syncthreads();                                                    // (the last tile has been read)
            if (tid == 0) s_bad = 0;
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
                const int p = tid + 256 * i;
                *(float4*)(sk + p / (D / 4) * KP + p % (D / 4) * 4) = piece[i];
            }
            bool bad = false;
            {
                const int k4 = tid % 16 * 4, page = __shfl(my_page, k4), off = __shfl(my_off, k4);
                const bool in0 = key_in(j0 + k4), in1 = key_in(j0 + k4 + 1), in2 = key_in(j0 + k4 + 2), in3 = key_in(j0 + k4 + 3);
#pragma unroll
                for (int i = 0; i < D / 16; ++i) {
                    const int e = tid / 16 + 16 * i;
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (in0 || in1 || in2 || in3) v = *(const float4*)(v_cache + (((size_t)page * nkv + kvh) * D + e) * page_size + off);
                    v.x = in0 ? v.x : 0.f; v.y = in1 ? v.y : 0.f; v.z = in2 ? v.z : 0.f; v.w = in3 ? v.w : 0.f;
                    piece[i] = v;
                }
#pragma unroll
                for (int i = 0; i < D / 16; ++i) {
                    const uint32_t top = 0x7f800000u;
                    bad |= (__float_as_uint(piece[i].x) & top) == top || (__float_as_uint(piece[i].y) & top) == top ||
                           (__float_as_uint(piece[i].z) & top) == top || (__float_as_uint(piece[i].w) & top) == top;
                    *(float4*)(sv + (tid / 16 + 16 * i) * VP + k4) = piece[i];
                }
            }
            __syncthreads();
            if (bad) s_bad = 1;
            __syncthreads();
            const bool active = in && j0 <= pos && (j0 + AG_TILE - 1 >= wk.lo || j0 < wk.keep);
            if (!__any(active)) continue;
            // ---- scores ----------------------------------------------------------------------------------------------------
            ag_f32x4 s[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) s[t] = (ag_f32x4){0.f, 0.f, 0.f, 0.f};
            const float* const ka = sk + (4 * (r & 3) + (r >> 2)) * KP + G;
#pragma unroll
            for (int e = 0; e < D / 4; ++e)
#pragma unroll
                for (int t = 0; t < 4; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[16 * t * KP + 4 * e], qf[e], s[t], 0, 0, 0);
            // ---- running maximum and sum: lane (r, G) has the keys 16 t + 4 i + G -----------------------------------------------
            float p[4][4], mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float sc = s[t][i] * scale;
                    if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
                    p[t][i] = active && seen(j0 + 16 * t + 4 * i + G) ? sc : -INFINITY;
                    mx = fmaxf(mx, p[t][i]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, IA_WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, IA_WAVE));
            const float m_new = fmaxf(m, mx);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    p[t][i] = active && seen(j0 + 16 * t + 4 * i + G) ? expf(p[t][i] - m_new) : 0.f;
            // the additions of a butterfly over the 64 keys, 32 apart first: the tiles, then i, then the lane groups
            float four[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) four[i] = (p[0][i] + p[2][i]) + (p[1][i] + p[3][i]);
            float sum = (four[0] + four[2]) + (four[1] + four[3]);
            sum = ag_pair_sum(sum, true);
            sum = ag_pair_sum(sum, false);
            float alpha = 1.f;
            if (active) {
                alpha = expf(m - m_new);
                l = fmaf(l, alpha, sum);
                m = m_new;
                any_in_seg = true;
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[t][i] *= alpha;
            // ---- outputs ---------------------------------------------------------------------------------------------------
            if (!s_bad) {
                const float* const va = sv + r * VP + G;
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int d = 0; d < DT; ++d)
                            o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[16 * d * VP + 16 * t + 4 * i], p[t][i], o[d], 0, 0, 0);
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        for (int b = 0; b < 4; ++b) {
                            const int key = 16 * t + 4 * i + b;
                            const float pk = __shfl(p[t][i], 16 * b + r);
                            const bool ok = active && seen(j0 + key);
#pragma unroll
                            for (int d = 0; d < DT; ++d)
#pragma unroll
                                for (int c = 0; c < 4; ++c)
                                    o[d][c] = ok ? fmaf(pk, sv[(16 * d + 4 * G + c) * VP + key], o[d][c]) : o[d][c];
                        }
            }
        }
        if (seg >= 0) end_segment();
        if (in) {
            const float inv = 1.0f / (sink ? big_l + expf((sinks != nullptr ? sinks[head] : 0.f) - big_m) : big_l);
#pragma unroll
            for (int d = 0; d < DT; ++d)
                *(ag_f32x4*)(out + ((size_t)tok * nq + head) * D + 16 * d + 4 * G) =
                    (ag_f32x4){big_o[d][0] * inv, big_o[d][1] * inv, big_o[d][2] * inv, big_o[d][3] * inv};
        }
    }
}

// Whether portions of prompts (requests of several tokens each, 32-bit) take attn_portions_f32_kernel: its sizes, and columns
// for a block.  Steps of few tokens at long contexts stay with a wave a segment (their walks would be long ones in few blocks).
extern "C" int ia_attention_portions_f32_fits(int n, int nq, int nkv, int d, int dv, int page_size, int max_kv_len) {
    return n > 0 && nkv > 0 && nq % nkv == 0 && (d == 64 || d == 128) && dv == d && page_size % 4 == 0 && nkv <= 65535 &&
           (long long)n * (nq / nkv) >= 64 && (long long)n * (nq / nkv) < (1LL << 30) && max_kv_len <= (1 << 24) &&
           ia_attention_generic_workspace(n, nq, nkv, d, dv, max_kv_len) == 0;
}

extern "C" int ia_attention_portions_f32(void* out, const void* q, const void* k_cache, const void* v_cache, const int* positions,
                                         const int* token_seq, const int* block_table, int n, int max_pages, int nq, int nkv, int d,
                                         int page_size, int window, float scale, int max_kv_len, int sink, int mask_chunk,
                                         const float* sinks, int keep_first, float softcap, hipStream_t stream) {
    IA_CHECK(ia_attention_portions_f32_fits(n, nq, nkv, d, d, page_size, max_kv_len), "attention: no kernel for portions of %d tokens, "
             "%d and %d heads of %d, pages of %d", n, nq, nkv, d, page_size);
    IA_CHECK((((uintptr_t)out | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0, "attention: arrays must be 16-byte aligned");
    IA_CHECK(max_pages > 0 && window >= 0 && mask_chunk >= 0 && keep_first >= 0 && softcap >= 0.f && (sinks == nullptr || sink),
             "attention: bad arguments max_pages=%d window=%d mask_chunk=%d keep_first=%d", max_pages, window, mask_chunk, keep_first);
    const dim3 grid((unsigned)(((long long)n * (nq / nkv) + 63) / 64), nkv);
#define AG_PORTIONS(D) attn_portions_f32_kernel<D><<<grid, 256, 0, stream>>>((float*)out, (const float*)q, (const float*)k_cache, \
        (const float*)v_cache, positions, token_seq, block_table, n, max_pages, nq, nkv, page_size, window, scale, sink, mask_chunk, \
        sinks, keep_first, softcap)
    if (d == 64) AG_PORTIONS(64);
    else AG_PORTIONS(128);
#undef AG_PORTIONS
    IA_LAUNCH_CHECK("attention_portions_f32");
    return 0;
}
