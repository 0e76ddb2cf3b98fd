// Paged grouped-query attention on the matrix cores, bfloat16, for one head size per build
// (IA_HEAD_DIM, a multiple of 16 up to 256).  One kernel serves prefill and decode: a wave
// owns up to 16 * NB columns, a column being one (query token, query head) pair of one
// request and one key/value head, and walks that request's keys 32 at a time straight from
// the cache pages into MFMA operands.  Where a step has few columns and long key ranges, the
// keys are split between waves and the partial results are merged by a second kernel.  Decode
// steps (one token a request) at head sizes in steps of 64 have a kernel of their own with the
// per-head norm, the rotation, the cache write and that merge inside (attn_decode_kernel).  At
// head size 128, steps with 128 columns or more of a request (portions of prompts) go to blocks
// of four waves that share keys and values through shared memory (attn_tile_kernel).
//
// Formula as in the reference: S = (q . k) * scale after the product, keys j <= position
// (inferrs-models/src/models/attention_utils.rs:61-85), softmax over keys, O = P v
// (inferrs-models/src/models/qwen3.rs:166-192); query head h reads key/value head
// h / (nq / nkv) (attention_utils.rs:38-49).  Scores, the running maximum and sum, and the
// output accumulators are 32-bit; probabilities are rounded to bfloat16 for the second product.
//
// Everything is computed transposed so that no operand needs a transpose in flight:
//   S^T[key][col] = K[key][:] . Q[col][:]      A = 16 keys x 32 dims (rows of the K page),
//                                              B = 32 dims x 16 columns (rows of Q)
//   O^T[dim][col] = V^T[dim][:] . P^T[:][col]  A = 16 dims x 32 keys (rows of the V^T page),
//                                              B = 32 keys x 16 columns (the S^T accumulators)
// The cache keeps keys as [page][kv head][slot][dim] and values transposed, as
// [page][kv head][dim][slot], so both A operands are 16-byte pieces of contiguous rows.
// v_mfma_f32_16x16x32_bf16: lane l supplies row l%16 of A and column l%16 of B with the eight
// k values 8*(l/16)..+8, and receives D[4*(l/16)+i][l%16], i = 0..3.  The two S^T tiles of a
// 32-key step assign key k0 + 8G + 4t + i to row 4G+i of tile t, so that lane (col, G) ends
// up holding the probabilities of keys k0+8G .. k0+8G+7 in order: exactly the B operand of the
// second product.
#include <type_traits>

#include "common.h"
#include "api.h"

#ifndef IA_HEAD_DIM
#error "compile with -DIA_HEAD_DIM=<multiple of 16 up to 256>"
#endif
static_assert(IA_HEAD_DIM % 16 == 0 && IA_HEAD_DIM >= 16 && IA_HEAD_DIM <= 256, "head size");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define HD IA_HEAD_DIM
// The values' width where it is not the keys' (IA_VALUE_DIM, a multiple of 16 up to 256): the kernel of single waves
// the merges of split keys and the decode kernel take any, the tile kernel the widths below.
#ifndef IA_VALUE_DIM
#define IA_VALUE_DIM IA_HEAD_DIM
#endif
static_assert(IA_VALUE_DIM % 16 == 0 && IA_VALUE_DIM >= 16 && IA_VALUE_DIM <= 256, "value size");
#define HDV IA_VALUE_DIM
#define HDMAX (HD > HDV ? HD : HDV)
#define DBV (HDV / 16)          // 16-dim blocks of the values
// The tile kernel (prompt portions, keys of 128) takes values of 32 to 128 in steps of 32: a load of 1 KiB brings 32 features
// of 16 keys, and the groups' exchange at its end fits the stages up to the keys' own width.
#define TILE_FITS (HD == 128 && HDV % 32 == 0 && HDV <= 128)
#define KS ((HD + 31) / 32)     // 32-dim steps of the first product

struct AttnParams {
    bf16_t* out;                // [n, nq, dv]
    float* part_o;              // [n, nq, splits, dv]  when splits > 1
    float* part_ml;             // [n, nq, splits, 2]   running maximum (log2 domain) and sum
    const bf16_t* q;            // [n, nq, d]
    const bf16_t* k_cache;      // [pages, nkv, page, d]
    const bf16_t* v_cache;      // [pages, nkv, dv, page]
    bf16_t* k_cache_w;          // the same arrays for the fused form's writes
    bf16_t* v_cache_w;
    const int* block_table;     // [seqs, max_pages]
    const int* cu_tokens;       // [seqs + 1]  request s owns tokens cu[s]..cu[s+1]
    const int* positions;       // [n]         absolute position of each token
    int max_pages, nq, nkv, page, window, splits, chunk, pair, seq_begin;   // pair: see the kernels
    int token_begin;            // decode kernel: request seq_begin + i owns token token_begin + i
    float scale_log2;           // scale * log2(e)
    // The decode kernel, with the per-head norm, the rotation and the cache write inside: q is not
    // read from `q` but formed from the projections' output, and the wave that walks a request's
    // newest key forms that key and value, uses them and writes them to the cache.
    const bf16_t* qkv;          // [n, row_ld]: q heads at q_off, k heads at k_off, v heads at v_off of a token's row
    int row_ld, q_off, k_off, v_off;
    int rot;                    // features of a head that rotate, halves paired (a multiple of 8)
    const bf16_t* gate;         // null, or where a token's gate values begin in its row: the output is times their sigmoid
    int gate_ld, gate_per_head; // pitch of the rows; 1: a value a query head, 0: a value a feature
    const float* q_norm_w;      // [d], or null: no norm
    const float* k_norm_w;
    const float* cos_t;         // [n, rot / 2], or null: no rotation
    const float* sin_t;
    const int* slots;           // [n] cache slot of each token, or null: this layer writes no cache
    float norm_eps;
    int norm_add_one;
    int sink;                   // 1: the softmax's denominator holds one more term, 2^(0 - m): a key of score 0 without a value
    const float* sinks;         // with sink: null, or [nq] values s_h a query head (natural logarithm, not scaled): the term is 2^(s_h log2 e - m)
    int mask_chunk;             // > 0: a query sees the keys of its own chunk of this many positions only, up to itself
    int keep_first;             // > 0: it sees the first so many positions besides (forms 1 and 2)
    uint32_t page_magic;        // decode kernel: pos / page is umulhi(2 (pos / 16), page_magic) >> page_shift
    int page_shift;
    int teams, col_blocks;      // decode kernel: blocks that share the keys of a (request, key/value head, block of 16 query heads), and those blocks of heads
    float cap_in;               // form 2: a raw score s stands for tanh(s * scale / cap); this is 2 log2(e) scale / cap, and scale_log2 is cap * log2(e)
};

// What the kernels of single waves and of tiles are compiled for beside a window, a chunk and a sink: nothing (0), first
// positions that every query sees (1), these and capped scores (2).
enum { FORM_PLAIN = 0, FORM_KEEP = 1, FORM_CAP = 2 };

// tanh from the exponential of twice its argument: `x` is 2 log2(e) times it.  (Within 2^-22 of the value in absolute terms;
// at both ends the exponential is 0 or infinite and the value -1 or 1.)
__device__ __forceinline__ float tanh_exp2(float x) {
    return __builtin_fmaf(-2.0f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.0f), 1.0f);
}

__device__ __forceinline__ uint4 zero4() { return make_uint4(0, 0, 0, 0); }

// The sink's term of a row's denominator, in the kernels' log-2 domain: 2^(s_h log2 e - m), s_h = 0 without values.
__device__ __forceinline__ float sink_term(const float* sinks, int head, float m) {
    return exp2f((sinks != nullptr ? sinks[head] * 1.4426950408889634f : 0.f) - m);
}

// One column block (16 * NB columns) of one request and key/value head, over one split of the keys.
template <int NB, int FORM>
__device__ __forceinline__ void attn_column_block(const AttnParams& p, int cb, int kvh, int split, int seq) {
    const int lane = threadIdx.x;
    const int r = lane & 15, G = lane >> 4;
    const int g = p.nq / p.nkv;
    const int t0 = p.cu_tokens[seq], q_len = p.cu_tokens[seq + 1] - t0;
    const int n_cols = q_len * g;
    const int col0 = cb * 16 * NB;
    if (col0 >= n_cols) return;
    const int kv_start = p.positions[t0];
    const int kv_total = kv_start + q_len;
    const int* bt = p.block_table + (size_t)seq * p.max_pages;

    // this lane's columns
    int tq[NB], head[NB], pos[NB];
    bool cvalid[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int c = col0 + nb * 16 + r;
        cvalid[nb] = c < n_cols;
        const int cc = cvalid[nb] ? c : n_cols - 1;
        tq[nb] = cc / g;
        head[nb] = kvh * g + (cc - tq[nb] * g);
        pos[nb] = kv_start + tq[nb];
    }
    const int last_col = (col0 + 16 * NB <= n_cols ? col0 + 16 * NB : n_cols) - 1;
    const int pmin = kv_start + col0 / g, pmax = kv_start + last_col / g;

    // Q^T operands stay in registers for the whole walk.
    uint4 qreg[NB][KS];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const bf16_t* qrow = p.q + ((size_t)(t0 + tq[nb]) * p.nq + head[nb]) * HD;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int dim = ks * 32 + G * 8;
            qreg[nb][ks] = (cvalid[nb] && dim < HD) ? *(const uint4*)(qrow + dim) : zero4();
        }
    }

    f32x4 acc[NB][DBV];
    float m[NB], l[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m[nb] = -INFINITY;
        l[nb] = 0.f;
#pragma unroll
        for (int db = 0; db < DBV; ++db) acc[nb][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    const int window_floor = ia_key_floor(pmin, p.window, p.mask_chunk);   // first key any column sees
    const int last_floor = ia_key_floor(pmax, p.window, p.mask_chunk);     // first key that the last column sees
    int lo = window_floor;
    int hi = pmax + 1;
    // The first positions that every query sees are a range of steps of their own, [pre_lo, pre_hi), ahead of the rest;
    // where no whole step lies between the two, the walk starts at 0.
    const int keep = FORM != FORM_PLAIN ? p.keep_first : 0;
    int pre_lo = 0, pre_hi = 0;
    if (FORM != FORM_PLAIN && keep > 0) {
        if (keep >= (window_floor & ~31)) lo = 0;
        else pre_hi = (keep + 31) & ~31;
    }
    if (p.splits > 1) {
        const int c_lo = split * p.chunk, c_hi = c_lo + p.chunk;
        lo = lo > c_lo ? lo : c_lo;
        hi = hi < c_hi ? hi : c_hi;
        pre_lo = c_lo;
        pre_hi = pre_hi < c_hi ? pre_hi : c_hi;
    }
    lo &= ~31;

    // ---- operands of a step: 32 keys = two 16-slot halves, each inside one page --------------
    struct Operands {
        uint4 k[2][KS];         // tile t, dim step ks: row r <-> key k0 + 8*(r/4) + 4t + r%4
        uint4 v[DBV];            // dim block db: row r <-> dim 16 db + r, keys k0 + 8G .. +7
    };
    // A step's 32 keys are two groups of 16 slots, each inside one page (page sizes are multiples of
    // 16): a Place says where a group lies, and moves on without a division.
    struct Place { int idx, off; };                  // page index in the block table, slot in that page
    auto advance = [&](Place& at, int slots) {
        at.off += slots;
        while (at.off >= p.page) { at.off -= p.page; ++at.idx; }
    };
    // This lane's part of the addresses does not change from step to step: its key rows' slots inside
    // their group, its piece of a row, and which of the two groups they belong to.
    const bool k_second = r >= 8, v_second = G >= 2;
    const uint32_t k_lane[2] = {(uint32_t)((((8 * (r >> 2) + (r & 3)) & 15) * HD + G * 8) * 2),
                                (uint32_t)((((8 * (r >> 2) + 4 + (r & 3)) & 15) * HD + G * 8) * 2)};
    const uint32_t v_lane = (uint32_t)((r * p.page + 8 * (G & 1)) * 2);
    const size_t v_stride = (size_t)16 * p.page * 2;
    auto load_step = [&](Operands& op, int k0, const Place& at) {
        if (k0 + 32 <= kv_total) {
            // every slot of the step is written: the pages' numbers and the groups' places are the same
            // for all lanes (they come through the scalar cache), a lane adds its constant part
            Place next = at;
            advance(next, 16);
            const int page_a = bt[at.idx], page_b = bt[next.idx];
            const char* ka = (const char*)(p.k_cache + (((size_t)page_a * p.nkv + kvh) * p.page + at.off) * HD);
            const char* kb = (const char*)(p.k_cache + (((size_t)page_b * p.nkv + kvh) * p.page + next.off) * HD);
            const char* va = (const char*)(p.v_cache + ((size_t)page_a * p.nkv + kvh) * HDV * p.page + at.off);
            const char* vb = (const char*)(p.v_cache + ((size_t)page_b * p.nkv + kvh) * HDV * p.page + next.off);
            const char* kbase = k_second ? kb : ka;
            const char* vbase = (v_second ? vb : va) + v_lane;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    op.k[t][ks] = (ks * 32 + G * 8 < HD) ? *(const uint4*)(kbase + k_lane[t] + ks * 64) : zero4();
#pragma unroll
            for (int db = 0; db < DBV; ++db) op.v[db] = *(const uint4*)(vbase + db * v_stride);
            return;
        }
        // The request's last step.  Rows past its length are read from its last written slot instead
        // (their scores are masked in the step): the pages behind them may not exist.
        const int last_idx = (kv_total - 1) / p.page;
        const int idx_a = k0 / p.page;
        const int idx_b = (k0 + 16) / p.page < last_idx ? (k0 + 16) / p.page : last_idx;
        const int page_a = bt[idx_a], page_b = bt[idx_b];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            int key = k0 + 8 * (r >> 2) + 4 * t + (r & 3);
            key = key < kv_total ? key : kv_total - 1;
            const int kpage = key / p.page == idx_a ? page_a : page_b;
            const bf16_t* krow = p.k_cache + (((size_t)kpage * p.nkv + kvh) * p.page + key % p.page) * HD + G * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                op.k[t][ks] = (ks * 32 + G * 8 < HD) ? *(const uint4*)(krow + ks * 32) : zero4();
        }
        int vkey = k0 + 8 * G;
        vkey = vkey < kv_total ? vkey : (kv_total - 1) & ~7;
        const int vpage = vkey / p.page == idx_a ? page_a : page_b;
        const bf16_t* vbase = p.v_cache + (((size_t)vpage * p.nkv + kvh) * HDV + r) * p.page + vkey % p.page;
#pragma unroll
        for (int db = 0; db < DBV; ++db) op.v[db] = *(const uint4*)(vbase + (size_t)db * 16 * p.page);
    };
    auto compute_step = [&](Operands& op, int k0) {
        const bool edge = k0 + 31 > pmin || k0 < last_floor;
        if (k0 + 32 > kv_total) {
            // slots beyond the request's length hold anything at all: zero those values so that
            // a probability of zero times their content stays zero
            const int first_bad = kv_total - (k0 + 8 * G);          // keys >= this index are unwritten
            if (first_bad < 8) {
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    uint32_t w[4] = {op.v[db].x, op.v[db].y, op.v[db].z, op.v[db].w};
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (j >= first_bad) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                    op.v[db] = make_uint4(w[0], w[1], w[2], w[3]);
                }
            }
        }
        if (k0 < window_floor) {
            // The walk starts at a multiple of 32 below the first key that any column sees: the keys in between
            // may lie in pages that the window has passed and the request has given back (the block table then
            // names some other page, which holds anything at all).  Their scores are masked below; their values
            // are zeroed here, for the same reason as the slots beyond the length.
            const int first_good = window_floor - (k0 + 8 * G);     // keys below this index are outside every window
            const int kept = keep - (k0 + 8 * G);                   // (those below this one are first positions: seen)
            if (first_good > 0) {
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    uint32_t w[4] = {op.v[db].x, op.v[db].y, op.v[db].z, op.v[db].w};
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (j < first_good && (FORM == FORM_PLAIN || j >= kept)) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                    op.v[db] = make_uint4(w[0], w[1], w[2], w[3]);
                }
            }
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            // ---- S^T for 32 keys x 16 columns ----------------------------------------------
            f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, op.k[t][ks]), __builtin_bit_cast(bf16x8, qreg[nb][ks]), s[t], 0, 0, 0);
            }
            // raw scores; the scale (> 0) and the change to base 2 are folded into the exponent below
            float sc[8];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[4 * t + i] = FORM == FORM_CAP ? tanh_exp2(s[t][i] * p.cap_in) : s[t][i];
            if (edge) {
                const int kbase_idx = k0 + 8 * G;
                const int floor_key = ia_key_floor(pos[nb], p.window, p.mask_chunk);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = kbase_idx + j;
                    if (key > pos[nb] || (key < floor_key && (FORM == FORM_PLAIN || key >= keep))) sc[j] = -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
            mx = fmaxf(mx, __shfl_xor(mx, 16, IA_WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, IA_WAVE));
            const float m_new = fmaxf(m[nb], mx * p.scale_log2);        // running maximum of scale * log2(e) * score
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m[nb] - m_use);  // m = -inf gives 0
            float pr[8], psum = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                pr[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j], p.scale_log2, -m_use));
                psum += pr[j];
            }
            l[nb] = l[nb] * alpha + psum;
            m[nb] = m_new;
            uint4 pb;
            pb.x = pack_bf16x2(pr[0], pr[1]);
            pb.y = pack_bf16x2(pr[2], pr[3]);
            pb.z = pack_bf16x2(pr[4], pr[5]);
            pb.w = pack_bf16x2(pr[6], pr[7]);
            // ---- O^T += V^T . P^T ----------------------------------------------------------
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    acc[nb][db][0] *= alpha; acc[nb][db][1] *= alpha;
                    acc[nb][db][2] *= alpha; acc[nb][db][3] *= alpha;
                }
            }
#pragma unroll
            for (int db = 0; db < DBV; ++db)
                acc[nb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, op.v[db]), __builtin_bit_cast(bf16x8, pb), acc[nb][db], 0, 0, 0);
        }
    };

    // What bounds the walk of a long prompt, and what was tried (each variant measured against this
    // one in the same run; prompts of 2,048 and 8,192 tokens, head size 128).  At 8,192 tokens a layer's
    // waves ask the L2 for 121 M lines (15 GB, 12 TB/s) and the matrix pipes are busy 18 % of the time;
    // with 16 columns a wave instead of 32 (twice the reads, the same arithmetic) the walk takes 1.9
    // times as long: it is the L2's bandwidth.
    // - Blocks of four waves that bring keys and values into shared memory once, through registers and
    //   in the cache's own layout (stages of 64 keys, the next stage on its way in registers, one barrier
    //   a stage), halved the L2's requests and were still 3 % slower: a third of the shared memory's busy
    //   cycles were bank conflicts, and the registers of the stage on its way cost occupancy.  With loads
    //   straight into shared memory and a swizzled layout it pays: attn_tile_kernel below, which takes the
    //   prompt portions of head size 128 from this kernel.
    // - Loading the next step's operands ahead of this step's products doubles the operand registers,
    //   which costs a wave per SIMD, and that wave hid more latency.  Asking for the next keys right
    //   after the scores and for the next values right after the second product (no register held
    //   twice): prompts 5 % slower.
    // - Moving the exponents' reference point only when the running maximum has risen by 2^8 (the
    //   accumulators are then rescaled a few times a walk, not at most steps), row maxima through
    //   v_permlane swaps instead of shared memory, late and early column blocks as separate waves
    //   instead of one after the other in a wave: within 1 % each.
    // - Addresses without a division in the step (above): 1 % at 2,048 tokens.
    if constexpr (FORM == FORM_PLAIN) {
        Place at = {lo / p.page, lo % p.page};
        for (int k0 = lo; k0 < hi; k0 += 32) {
            Operands op;
            load_step(op, k0, at);
            compute_step(op, k0);
            advance(at, 32);
        }
    } else {
        const bool two = pre_lo < pre_hi;               // (pre_hi <= hi: the first range lies below every window)
        int k0 = two ? pre_lo : lo;
        Place at = {k0 / p.page, k0 % p.page};
        while (k0 < hi) {
            Operands op;
            load_step(op, k0, at);
            compute_step(op, k0);
            k0 += 32;
            advance(at, 32);
            if (two && k0 == pre_hi) {
                k0 = lo;
                at.idx = lo / p.page;
                at.off = lo % p.page;
            }
        }
    }

    // ---- results: lane (col, G) holds dims 16 db + 4 G + i of its column ---------------------
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        float lt = l[nb];
        lt += __shfl_xor(lt, 16, IA_WAVE);
        lt += __shfl_xor(lt, 32, IA_WAVE);
        if (!cvalid[nb]) continue;
        const size_t row = (size_t)(t0 + tq[nb]) * p.nq + head[nb];
        if (p.splits == 1) {
            const float inv = 1.0f / (p.sink ? lt + sink_term(p.sinks, head[nb], m[nb]) : lt);
            bf16_t* o = p.out + row * HDV + 4 * G;
#pragma unroll
            for (int db = 0; db < DBV; ++db) {
                uint2 w;
                w.x = pack_bf16x2(acc[nb][db][0] * inv, acc[nb][db][1] * inv);
                w.y = pack_bf16x2(acc[nb][db][2] * inv, acc[nb][db][3] * inv);
                *(uint2*)(o + 16 * db) = w;
            }
        } else {
            float* o = p.part_o + (row * p.splits + split) * HDV + 4 * G;
#pragma unroll
            for (int db = 0; db < DBV; ++db) *(f32x4*)(o + 16 * db) = acc[nb][db];
            if (G == 0) {
                float* ml = p.part_ml + (row * p.splits + split) * 2;
                ml[0] = m[nb];
                ml[1] = lt;
            }
        }
    }
}

// With `pair` a wave takes column block i from the end of its request and then block i from the
// start: under a causal mask the late blocks walk many keys and the early ones few, and every
// pair walks about the same number, so all waves end together.  It pays when the step's queries
// span most of the context; a short portion late in a long context has equal blocks already.
template <int NB, int FORM>
__global__ __launch_bounds__(IA_WAVE) __attribute__((amdgpu_waves_per_eu(HDMAX <= 128 ? 2 : 1, HDMAX > 64 ? 2 : 8)))
void attn_mfma_kernel(const AttnParams p) {
    const int kvh = blockIdx.y / p.splits, split = blockIdx.y - kvh * p.splits;
    const int seq = p.seq_begin + blockIdx.z;
    const int n_cols = (p.cu_tokens[seq + 1] - p.cu_tokens[seq]) * (p.nq / p.nkv);
    const int n_blocks = (n_cols + 16 * NB - 1) / (16 * NB);
    if (!p.pair) {
        // heavy column blocks first
        if ((int)blockIdx.x < n_blocks) attn_column_block<NB, FORM>(p, n_blocks - 1 - (int)blockIdx.x, kvh, split, seq);
        return;
    }
    const int late = n_blocks - 1 - (int)blockIdx.x, early = (int)blockIdx.x;
    if (late < early) return;
    attn_column_block<NB, FORM>(p, late, kvh, split, seq);
    if (early != late) attn_column_block<NB, FORM>(p, early, kvh, split, seq);
}

// The maximum / the sum over the four lanes that hold a column's values (lanes l, l ^ 16, l ^ 32, l ^ 48), in all
// of them, by swaps between rows of 16 lanes and between the halves of the wave: no trip through shared memory.
__device__ __forceinline__ float column_max(float x) {
    const uint32_t u = __float_as_uint(x);
    auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const uint32_t w = __float_as_uint(x);
    auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float column_sum(float x) {
    const uint32_t u = __float_as_uint(x);
    auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const uint32_t w = __float_as_uint(x);
    auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// ---- decode steps: one token a request, with the norm, the rotation, the cache write and the merge inside ------
// A wave owns up to 16 query heads of one request and key/value head and one split of that request's keys, as
// in the kernel above, but a decode step is short and every microsecond of it is latency, so the walk is laid
// out for that:
//  * the first step's keys and values are asked for before anything else: the query row is normed and rotated,
//    and the request's new key and value are formed and written to the cache, while they are on their way;
//  * a step's operands are asked for one step ahead (two sets of registers: a decode wave holds 16 columns and
//    has the room), so a wave waits for the memory once, not once a step;
//  * the waves of a block (`team`: 1, 2 or 4 neighbouring splits) add their results up in shared memory and
//    leave one partial result a block; the block that finishes last for its (request, key/value head), known by
//    a counter in memory, merges the blocks' partial results and writes the output.  No second kernel, and no
//    wave reads another compute unit's results before they are there: every wave waits until the memory has taken
//    its stores (`s_waitcnt vmcnt(0)`) before the barrier that precedes the block's one atomic increment, and the
//    last block reads past the caches after it has seen the full count.  The counters are zero
//    between calls (the last block puts its counter back), so calls that share them must not overlap.
// The sum over the splits runs in the order of the splits whoever comes last: the result is the same every time.
// Rows of any layout come in: query, key and value heads at places of their own, values narrower or wider than keys, the first `rot`
// features of a head turned, a gate's values behind them (the output is times their sigmoid before it is rounded), no keys at all
// (a layer that reads another's cache; queries that a kernel before has formed).  16 query heads of 128 beside values of 64 and a gate,
// 8 requests at 2,000 keys, window 1,024: four kernels of 5.3, 7.8, 4.5 and 4.0 us (norm and rotation, attention, merge, gate), 10.2 in
// this one, a step of six such layers 644 -> 600 us; the single tokens of a step that also brings a portion, 40 query heads, 9 requests at 3,100
// keys: 28.6 + 4.8 us by the kernel of single waves and its merge, 27.1 here beside nothing else.
// A wave is mostly alone on its SIMD, so every instruction it executes is four cycles of the step (returning from the kernel early, 16 query
// and 8 key/value heads, 700 keys, 64 a wave: rows and first keys are there 1.0 us after the start, rows formed 2.0 later, two steps done
// 3.5 later, a team merged 0.9 later, the hand-over 2.5).  So rows are formed by all lanes, numbers of pages come without divisions,
// the edges of a walk are handled once, ahead of its first and last step, and not in every copy of a step, results that meet are
// asked for together, and lanes exchange sums without a trip through shared memory; and nothing is held that can be read again, so
// that (head sizes up to 128) two waves share a SIMD.  us a layer, before and now: 16 query heads, batch 1, 200 keys 10.6 -> 7.9,
// 1,000 11.6 -> 9.0, 8,000 16.8 -> 14.0; 32 query heads, batch 4 at 2,000 15.2 -> 12.6, batch 8 at 700 13.7 -> 11.3, at
// 8,192 52.9 -> 51.2, batch 64 at 1,500 73.9 -> 72.0; 64 query heads, batch 2 at 1,500 15.2 -> 11.9.  Of the context at 8,192, batch 8, the
// bytes alone take 42.  A fence of device scope in place of the write-through stores cost 100 us a layer at batch 8 (it writes
// back and empties the whole L2 of the die, once a block).
// Partial results that blocks on other compute units read within the same kernel: written through to memory and
// read past the caches that are not coherent between the chip's dies (32-bit accesses of device scope, no order
// of their own), so that no cache has to be written back or emptied as a whole.
__device__ __forceinline__ void put_across(float* at, float v) {
    __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float get_across(const float* at) {
    return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The sum over `LANES` neighbouring lanes (8, 16 or 32, aligned), in all of them, in the vector units' own lane exchanges.
template <int LANES>
__device__ __forceinline__ float row_sum(float x) {
#define ROW_STEP(CTRL) x += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), CTRL, 0xf, 0xf, true))
    ROW_STEP(0xb1);                                         // lane ^ 1
    ROW_STEP(0x4e);                                         // lane ^ 2
    ROW_STEP(0x141);                                        // the other four of eight
    if constexpr (LANES >= 16) ROW_STEP(0x140);             // the other eight of sixteen
#undef ROW_STEP
    if constexpr (LANES >= 32) {
        auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    return x;
}

// 32-bit words of shared memory of a wave with `cols` columns: its rows and the new key, and behind its walk its partial outputs in
// the same place (a wave may be at its outputs while another still reads its rows: the places of two waves have nothing in common).
__host__ __device__ constexpr int decode_wave_words(int cols) {
    return cols * HDV > (cols + 1) * HD / 2 ? cols * HDV : (cols + 1) * HD / 2;
}

struct DecodeOperands {
    uint4 k[2][KS];             // as Operands above
    uint4 v[DBV];
};

#define DECODE_TEAM 4           // waves of a block at most

template <bool ENABLED = (HD % 64 == 0)>
__global__ __launch_bounds__(DECODE_TEAM * IA_WAVE) __attribute__((amdgpu_waves_per_eu(HDMAX <= 128 ? 2 : 1))) void attn_decode_kernel(const AttnParams p, int* counters, int team) {
    if constexpr (ENABLED) {
        extern __shared__ __align__(16) float team_mem[];       // [team][words of a wave], then [team][columns][2]
        __shared__ int s_last;
        // (the wave's number through a scalar register: what follows from it, the split's range and the pages' numbers,
        // is then the same for all lanes by construction, and the block table is read through the scalar cache)
        const int lane = threadIdx.x & (IA_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / IA_WAVE);
        const int r = lane & 15, G = lane >> 4;
        const int g = p.nq / p.nkv;
        const int teams = p.teams;
        const int cb = p.col_blocks > 1 ? (int)blockIdx.x / teams : 0;
        const int kvh = blockIdx.y, tm = (int)blockIdx.x - cb * teams;
        const int split = tm * team + wave;
        const int seq = p.seq_begin + blockIdx.z;
        const int col0 = cb * 16;
        const int n_cols = g - col0 < 16 ? g - col0 : 16;       // this block's columns (the grid has no empty block)
        // (a division by a number known at run time only is some thirty instructions one after the other, and the walk's start
        // would wait for six of them)
        auto page_of = [&](int pos) __attribute__((always_inline)) {
            return (int)(__umulhi((uint32_t)pos >> 3 & ~1u, p.page_magic) >> p.page_shift);
        };
        // What a wave needs before it can ask for its first keys is a chain of small reads, each a trip to the
        // memory: the token's position, then the pages' numbers.  A decode step's token is known without a read
        // (request seq_begin + i owns token token_begin + i), and where no window moves the walk's start the first
        // two steps' pages are read from the block table at the same time as the position (entries past the
        // request's last page are read but not used).
        const int t0 = p.token_begin + (int)blockIdx.z;
        const int* bt = p.block_table + (size_t)seq * p.max_pages;
        const int c_lo = p.splits > 1 ? split * p.chunk : 0;
        int early[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = page_of(c_lo + 16 * i);
            early[i] = bt[idx < p.max_pages ? idx : p.max_pages - 1];
        }
        const int kv_start = p.positions[t0];
        const int kv_total = kv_start + 1;
        const bool cvalid = r < n_cols;
        const int head = kvh * g + col0 + (cvalid ? r : n_cols - 1);

        const int window_floor = ia_key_floor(kv_start, p.window, p.mask_chunk);
        int lo = window_floor > c_lo ? window_floor : c_lo, hi = kv_total;
        if (p.splits > 1 && hi > c_lo + p.chunk) hi = c_lo + p.chunk;
        lo &= ~31;

        // ---- loads, in the order in which their results are needed ------------------------------------
        // The rows of the projections' output that this wave norms and rotates (its query heads' rows, and behind them the new
        // key's), the norms' weights and the angles, then the first step's keys and values: the rows are formed while those are
        // on their way, and the second step's are asked for after that (a wave can have 63 loads outstanding: all at once
        // would stall the issue of the last ones until the first come back).
        // The rows are shared out over all lanes: a lane has four features of a row and the four that they are turned with, rot / 2
        // further on (behind the features that rotate: the next four), a pass takes ROWS rows, and they meet the matrix operand's layout in the wave's own shared memory.  (With a
        // column's features in the four lanes that need them, 32 a lane, two rows took 2 of the 7 us that a wave has.)
        const bf16_t* token_row = p.qkv + (size_t)t0 * p.row_ld;
        constexpr int ROW_LANES = HD <= 64 ? 8 : HD <= 128 ? 16 : 32, ROWS = IA_WAVE / ROW_LANES, ROW_USED = HD / 8;
        const int ri = lane % ROW_LANES < ROW_USED ? lane % ROW_LANES : ROW_USED - 1, rsub = lane / ROW_LANES;
        const bool rotates = 8 * ri < p.rot;
        const int fa = rotates ? 4 * ri : 8 * ri, fb = rotates ? 4 * ri + p.rot / 2 : 8 * ri + 4;       // (the first rot / 8 lanes hold the rotated part)
        struct RowPart { uint2 lo, hi; float4 wlo, whi; };
        auto ask_rows = [&](RowPart& part, int pass) __attribute__((always_inline)) {
            const int t = pass * ROWS + rsub;
            const bf16_t* from = token_row + (t < n_cols ? p.q_off + (kvh * g + col0 + t) * HD : p.k_off + kvh * HD);
            part.lo = *(const uint2*)(from + fa);
            part.hi = *(const uint2*)(from + fb);
            if (p.q_norm_w != nullptr) {
                const float* w = t < n_cols ? p.q_norm_w : p.k_norm_w;
                part.wlo = *(const float4*)(w + fa);
                part.whi = *(const float4*)(w + fb);
            }
        };
        RowPart rows0, rows1;
        ask_rows(rows0, 0);
        float4 cs = make_float4(1.f, 1.f, 1.f, 1.f), sn = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p.cos_t != nullptr && rotates) {
            cs = *(const float4*)(p.cos_t + (size_t)t0 * (p.rot / 2) + 4 * ri);
            sn = *(const float4*)(p.sin_t + (size_t)t0 * (p.rot / 2) + 4 * ri);
        }
        if (n_cols + 1 > ROWS) ask_rows(rows1, 1);

        // A step's 32 keys are two groups of 16 slots, each inside one page (page sizes are multiples of 16).
        // Slots past the request's length are read like any others as long as their page is the request's (their
        // scores are masked and their values zeroed in the step); pages past its last are not asked for.
        const int last_idx = page_of(kv_total - 1);
        const bool k_second = r >= 8, v_second = G >= 2;
        const uint32_t k_lane[2] = {(uint32_t)((((8 * (r >> 2) + (r & 3)) & 15) * HD + G * 8) * 2),
                                    (uint32_t)((((8 * (r >> 2) + 4 + (r & 3)) & 15) * HD + G * 8) * 2)};
        const uint32_t v_lane = (uint32_t)((r * p.page + 8 * (G & 1)) * 2);
        const size_t v_stride = (size_t)16 * p.page * 2;
        auto load_pages = [&](DecodeOperands& op, int k0, int page_a, int page_b) __attribute__((always_inline)) {
            const int off_a = k0 - page_of(k0) * p.page, off_b = k0 + 16 - page_of(k0 + 16) * p.page;
            const char* ka = (const char*)(p.k_cache + (((size_t)page_a * p.nkv + kvh) * p.page + off_a) * HD);
            const char* kb = (const char*)(p.k_cache + (((size_t)page_b * p.nkv + kvh) * p.page + off_b) * HD);
            const char* va = (const char*)(p.v_cache + ((size_t)page_a * p.nkv + kvh) * HDV * p.page + off_a);
            const char* vb = (const char*)(p.v_cache + ((size_t)page_b * p.nkv + kvh) * HDV * p.page + off_b);
            const char* kbase = k_second ? kb : ka;
            const char* vbase = (v_second ? vb : va) + v_lane;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) op.k[t][ks] = *(const uint4*)(kbase + k_lane[t] + ks * 64);
#pragma unroll
            for (int db = 0; db < DBV; ++db) op.v[db] = *(const uint4*)(vbase + db * v_stride);
        };
        auto load_step = [&](DecodeOperands& op, int k0) __attribute__((always_inline)) {
            int idx_a = page_of(k0), idx_b = page_of(k0 + 16);
            idx_a = idx_a < last_idx ? idx_a : last_idx;
            idx_b = idx_b < last_idx ? idx_b : last_idx;
            load_pages(op, k0, bt[idx_a], bt[idx_b]);
        };
        // the first two steps, with the pages read ahead where the walk starts at the split's own start
        auto load_early = [&](DecodeOperands& op, int k0, int i) __attribute__((always_inline)) {
            if (lo == c_lo && page_of(k0 + 16) <= last_idx) load_pages(op, k0, early[2 * i], early[2 * i + 1]);
            else load_step(op, k0);
        };
        const int n_steps = lo < hi ? (hi - lo + 31) / 32 : 0;
        DecodeOperands opa, opb;
        load_early(opa, lo, 0);

        const bool has_new = p.slots != nullptr && hi == kv_total && lo < hi;
        const int slot = has_new ? p.slots[t0] : 0;
        uint32_t vnew[DBV];
        if (has_new) {
#pragma unroll
            for (int db = 0; db < DBV; ++db) vnew[db] = token_row[p.v_off + kvh * HDV + db * 16 + r].bits;
        }
        if (n_steps >= 2) load_early(opb, lo + 32, 1);

        // Rows, normed and rotated as the separate kernel does it (32-bit throughout, one rounding at the end).  A row's 16-byte
        // pieces lie exchanged by its number, so that operand reads of several rows meet no bank twice.  They fit where the wave's
        // partial outputs will lie.
        char* const row_mem = (char*)(team_mem + (size_t)wave * decode_wave_words(n_cols));
        auto form_rows = [&](const RowPart& part, int pass) __attribute__((always_inline)) {
            const int t = pass * ROWS + rsub;
            float a[4] = {__uint_as_float(part.lo.x << 16), __uint_as_float(part.lo.x & 0xffff0000u),
                          __uint_as_float(part.lo.y << 16), __uint_as_float(part.lo.y & 0xffff0000u)};
            float b[4] = {__uint_as_float(part.hi.x << 16), __uint_as_float(part.hi.x & 0xffff0000u),
                          __uint_as_float(part.hi.y << 16), __uint_as_float(part.hi.y & 0xffff0000u)};
            if (p.q_norm_w != nullptr) {
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) ss += a[j] * a[j];
#pragma unroll
                for (int j = 0; j < 4; ++j) ss += b[j] * b[j];
                if (ROW_USED != ROW_LANES) ss = lane % ROW_LANES < ROW_USED ? ss : 0.f;
                ss = row_sum<ROW_LANES>(ss);
                const float scale = 1.0f / sqrtf(ss / (float)HD + p.norm_eps), one = p.norm_add_one ? 1.0f : 0.0f;
                const float wa[4] = {part.wlo.x, part.wlo.y, part.wlo.z, part.wlo.w}, wb[4] = {part.whi.x, part.whi.y, part.whi.z, part.whi.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) { a[j] = scale * a[j] * (wa[j] + one); b[j] = scale * b[j] * (wb[j] + one); }
            }
            if (p.cos_t != nullptr && rotates) {
                const float c[4] = {cs.x, cs.y, cs.z, cs.w}, sv[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float x = a[j], y = b[j];
                    a[j] = x * c[j] - y * sv[j];
                    b[j] = x * sv[j] + y * c[j];
                }
            }
            if (t <= n_cols && lane % ROW_LANES < ROW_USED) {
                char* const at = row_mem + t * (HD * 2);
                *(uint2*)(at + ((fa >> 3) ^ (t & 7)) * 16 + (fa & 4) * 2) = make_uint2(pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]));
                *(uint2*)(at + ((fb >> 3) ^ (t & 7)) * 16 + (fb & 4) * 2) = make_uint2(pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3]));
            }
        };
        const int passes = (n_cols + (has_new ? 1 : 0) + ROWS - 1) / ROWS;
        form_rows(rows0, 0);
        if (passes > 1) form_rows(rows1, 1);
        for (int pass = 2; pass < passes; ++pass) {
            ask_rows(rows0, pass);
            form_rows(rows0, pass);
        }
        // (the wave's own memory: its shared-memory operations run in program order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        uint4 qreg[KS];
        {
            const int t = cvalid ? r : n_cols - 1;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) qreg[ks] = *(const uint4*)(row_mem + t * (HD * 2) + ((ks * 4 + G) ^ (t & 7)) * 16);
        }
        // the new key's features ks * 32 + G * 8 .. + 8
        auto new_key = [&](int ks) __attribute__((always_inline)) {
            return *(const uint4*)(row_mem + n_cols * (HD * 2) + ((ks * 4 + G) ^ (n_cols & 7)) * 16);
        };

        f32x4 acc[DBV];
        float m = -INFINITY, l = 0.f;
#pragma unroll
        for (int db = 0; db < DBV; ++db) acc[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

        // What only the walk's first step needs: keys below the window.
        auto first_edge = [&](DecodeOperands& op, int k0) __attribute__((always_inline)) {
            if (k0 < window_floor) {
                // keys below the window may lie in pages that the request has given back: as above
                const int first_good = window_floor - (k0 + 8 * G);
                if (first_good > 0) {
#pragma unroll
                    for (int db = 0; db < DBV; ++db) {
                        uint32_t w[4] = {op.v[db].x, op.v[db].y, op.v[db].z, op.v[db].w};
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (j < first_good) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                        op.v[db] = make_uint4(w[0], w[1], w[2], w[3]);
                    }
                }
            }
        };
        // What only its last step needs: the end of the request's keys, and the new one.
        auto last_edge = [&](DecodeOperands& op, int k0) __attribute__((always_inline)) {
            if (k0 + 32 > kv_total) {
                // slots beyond the request's length hold anything at all: zero those values so that a probability
                // of zero times their content stays zero
                const int first_bad = kv_total - (k0 + 8 * G);
                if (first_bad < 8) {
#pragma unroll
                    for (int db = 0; db < DBV; ++db) {
                        uint32_t w[4] = {op.v[db].x, op.v[db].y, op.v[db].z, op.v[db].w};
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (j >= first_bad) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                        op.v[db] = make_uint4(w[0], w[1], w[2], w[3]);
                    }
                }
            }
            if (has_new && k0 + 32 >= kv_total) {
                // (values chosen, never addresses: the operands stay in registers)
                const int kk = kv_total - 1 - k0;
                const bool mine = r == (((kk >> 3) << 2) | (kk & 3));
                const bool first = mine && ((kk >> 2) & 1) == 0, second = mine && ((kk >> 2) & 1) == 1;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const uint4 key = new_key(ks);
                    op.k[0][ks].x = first ? key.x : op.k[0][ks].x; op.k[0][ks].y = first ? key.y : op.k[0][ks].y;
                    op.k[0][ks].z = first ? key.z : op.k[0][ks].z; op.k[0][ks].w = first ? key.w : op.k[0][ks].w;
                    op.k[1][ks].x = second ? key.x : op.k[1][ks].x; op.k[1][ks].y = second ? key.y : op.k[1][ks].y;
                    op.k[1][ks].z = second ? key.z : op.k[1][ks].z; op.k[1][ks].w = second ? key.w : op.k[1][ks].w;
                }
                const int j = kk & 7;
                const bool vmine = G == (kk >> 3);
                const uint32_t keep = (j & 1) ? 0x0000ffffu : 0xffff0000u;
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    const uint32_t put = (j & 1) ? vnew[db] << 16 : vnew[db];
                    op.v[db].x = vmine && (j >> 1) == 0 ? (op.v[db].x & keep) | put : op.v[db].x;
                    op.v[db].y = vmine && (j >> 1) == 1 ? (op.v[db].y & keep) | put : op.v[db].y;
                    op.v[db].z = vmine && (j >> 1) == 2 ? (op.v[db].z & keep) | put : op.v[db].z;
                    op.v[db].w = vmine && (j >> 1) == 3 ? (op.v[db].w & keep) | put : op.v[db].w;
                }
            }
        };
        auto compute_step = [&](DecodeOperands& op, int k0) __attribute__((always_inline)) {
            f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, op.k[t][ks]), __builtin_bit_cast(bf16x8, qreg[ks]), s[t], 0, 0, 0);
            }
            float sc[8];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[4 * t + i] = s[t][i];
            if (k0 + 31 > kv_start || (k0 < window_floor)) {
                const int kbase_idx = k0 + 8 * G;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = kbase_idx + j;
                    if (key > kv_start || key < window_floor) sc[j] = -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
            const float m_new = fmaxf(m, column_max(mx) * p.scale_log2);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m - m_use);
            float pr[8], psum = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                pr[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j], p.scale_log2, -m_use));
                psum += pr[j];
            }
            l = l * alpha + psum;
            m = m_new;
            uint4 pb;
            pb.x = pack_bf16x2(pr[0], pr[1]);
            pb.y = pack_bf16x2(pr[2], pr[3]);
            pb.z = pack_bf16x2(pr[4], pr[5]);
            pb.w = pack_bf16x2(pr[6], pr[7]);
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    acc[db][0] *= alpha; acc[db][1] *= alpha;
                    acc[db][2] *= alpha; acc[db][3] *= alpha;
                }
            }
#pragma unroll
            for (int db = 0; db < DBV; ++db)
                acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, op.v[db]), __builtin_bit_cast(bf16x8, pb), acc[db], 0, 0, 0);
        };

        // The walk: two steps' operands are under way at any time.  Inside the loop the loads are unconditional (the compiler counts
        // what is outstanding and waits for the older set only; behind the walk's last step they fetch the request's last page once
        // more, which is in a cache); the last one or two steps follow it.  opa holds step k0, opb step k0 + 32.
        int k0 = lo, left = n_steps;
        if (left > 0) first_edge(opa, k0);
        while (left > 2) {
            compute_step(opa, k0);
            load_step(opa, k0 + 64);
            compute_step(opb, k0 + 32);
            load_step(opb, k0 + 96);
            k0 += 64;
            left -= 2;
        }
        if (left == 2) {
            compute_step(opa, k0);
            last_edge(opb, k0 + 32);
            compute_step(opb, k0 + 32);
        } else if (left == 1) {
            last_edge(opa, k0);
            compute_step(opa, k0);
        }

        // The request's newest key (position kv_total - 1, this step's token) is in no page yet: the wave whose
        // keys end with it has put it and its value into its last step's operands in place of what the loads
        // brought, and now writes them to the cache for the steps to come.  (After the walk: with no store before
        // them, the block table's reads go through the scalar cache.)
        if (has_new) {
            const int page = slot / p.page, off = slot - page * p.page;
            const int kk = (kv_total - 1) & 31;
            if (r == (((kk >> 3) << 2) | (kk & 3))) {
                bf16_t* krow = p.k_cache_w + (((size_t)page * p.nkv + kvh) * p.page + off) * HD + G * 8;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) *(uint4*)(krow + ks * 32) = new_key(ks);
            }
            if (G == (kk >> 3)) {
                bf16_t* vdst = p.v_cache_w + (((size_t)page * p.nkv + kvh) * HDV + r) * p.page + off;
#pragma unroll
                for (int db = 0; db < DBV; ++db) vdst[(size_t)db * 16 * p.page].bits = (uint16_t)vnew[db];
            }
        }

        const float lt = column_sum(l);
        const size_t row0 = (size_t)t0 * p.nq + kvh * g + col0;        // the block's first (token, head) row
        // A piece of four features of the output: divided by the row's sum, times the sigmoid of the gate's values.
        auto ask_gate = [&](int col, int feature) __attribute__((always_inline)) {
            const bf16_t* from = p.gate + (size_t)t0 * p.gate_ld;
            const int at = kvh * g + col0 + col;
            if (p.gate_per_head) {
                const uint32_t one = from[at].bits * 0x10001u;
                return make_uint2(one, one);
            }
            return *(const uint2*)(from + (size_t)at * HDV + feature);
        };
        auto put_out = [&](int col, int feature, const f32x4& o, float inv, const uint2& gate) __attribute__((always_inline)) {
            float v[4] = {o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
            if (p.gate != nullptr) {
                const float z[4] = {__uint_as_float(gate.x << 16), __uint_as_float(gate.x & 0xffff0000u),
                                    __uint_as_float(gate.y << 16), __uint_as_float(gate.y & 0xffff0000u)};
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = v[j] / (1.0f + expf(-z[j]));
            }
            *(uint2*)(p.out + (row0 + col) * HDV + feature) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        };
        if (p.splits == 1) {
            if (!cvalid) return;
            const float inv = 1.0f / (p.sink ? lt + sink_term(p.sinks, head, m) : lt);
            uint2 gate[DBV];
            if (p.gate != nullptr) {
#pragma unroll
                for (int db = 0; db < DBV; ++db) gate[db] = ask_gate(r, 16 * db + 4 * G);
            }
#pragma unroll
            for (int db = 0; db < DBV; ++db) put_out(r, 16 * db + 4 * G, acc[db], inv, gate[db]);
            return;
        }

        // ---- the block's waves add up: lane (col, G) holds dims 16 db + 4 G + i of its column --------
        const int words = decode_wave_words(n_cols);
        float* team_o = team_mem;                                       // [team][words], of each [n_cols][HDV]
        float* team_ml = team_mem + (size_t)team * words;               // [team][n_cols][2]
        if (cvalid) {
            float* o = team_o + (size_t)wave * words + r * HDV + 4 * G;
#pragma unroll
            for (int db = 0; db < DBV; ++db) *(f32x4*)(o + 16 * db) = acc[db];
            if (G == 0) {
                team_ml[(wave * n_cols + r) * 2] = m;
                team_ml[(wave * n_cols + r) * 2 + 1] = lt;
            }
        }
        __syncthreads();
        const int pieces = n_cols * (HDV / 4);                           // 16-byte pieces of the block's result
        for (int e = threadIdx.x; e < pieces; e += blockDim.x) {
            const int col = e / (HDV / 4), piece = e - col * (HDV / 4);
            // (all of the team's results are asked for together)
            float mw[DECODE_TEAM], lw[DECODE_TEAM], mx = -INFINITY, total = 0.f;
            uint2 gate = make_uint2(0, 0);
            if (teams == 1 && p.gate != nullptr) gate = ask_gate(col, piece * 4);
            f32x4 v[DECODE_TEAM], o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < DECODE_TEAM; ++w) {
                const int of = w < team ? w : 0, at = of * n_cols + col;
                mw[w] = team_ml[at * 2];
                lw[w] = team_ml[at * 2 + 1];
                v[w] = *(const f32x4*)(team_o + (size_t)of * words + col * HDV + piece * 4);
                mx = fmaxf(mx, mw[w]);
            }
#pragma unroll
            for (int w = 0; w < DECODE_TEAM; ++w) {
                const float wt = w >= team || mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - mx);      // (a split that held no key of this row)
                o[0] = fmaf(v[w][0], wt, o[0]); o[1] = fmaf(v[w][1], wt, o[1]);
                o[2] = fmaf(v[w][2], wt, o[2]); o[3] = fmaf(v[w][3], wt, o[3]);
                total = fmaf(lw[w], wt, total);
            }
            if (teams == 1) {
                const float inv = 1.0f / (p.sink ? total + sink_term(p.sinks, (int)((row0 + col) % p.nq), mx) : total);
                put_out(col, piece * 4, o, inv, gate);
            } else {
                float* po = p.part_o + ((row0 + col) * teams + tm) * HDV + piece * 4;
                put_across(po, o[0]); put_across(po + 1, o[1]); put_across(po + 2, o[2]); put_across(po + 3, o[3]);
                if (piece == 0) {
                    float* ml = p.part_ml + ((row0 + col) * teams + tm) * 2;
                    put_across(ml, mx);
                    put_across(ml + 1, total);
                }
            }
        }
        if (teams == 1) return;

        // ---- the last block of this (request, key/value head, column block) merges the blocks' results --------
        int* counter = counters + ((size_t)blockIdx.z * p.nkv + kvh) * p.col_blocks + cb;
        // The hand-over.  Writer: a wave's vector-memory counter counts a store down when the memory has taken it
        // (the stores above are written through, so that is the point where every die reads it), and
        // `s_waitcnt vmcnt(0)` holds the wave until all of its stores are there; then the barrier, so that this
        // holds for every wave of the block; only then the count.  (A release fence of workgroup scope does not wait
        // for stores that leave the compute unit, and one of device scope writes the die's L2 back.)  The compiler
        // moves no store across the wait (the asm names memory).
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            s_last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == teams - 1 ? 1 : 0;
        __syncthreads();
        if (!s_last) return;
        // Reader: thread 0 has the counter's old value in a register before it can write s_last, so the increment
        // that made it teams - 1, and with it every other block's stores, is in memory before any thread passes the
        // barrier above; the loads below are issued after it, and they read past the caches (device scope), so they
        // cannot meet a line that was fetched before the stores arrived.
        // Every thread takes part: the block's threads form as many groups as there are 16-byte pieces of the result
        // in them, group i sums the blocks i, i + groups, ... in that order, and the groups' sums meet in shared
        // memory and are added in the groups' order.
        const int groups = pieces <= (int)blockDim.x ? (int)blockDim.x / pieces : 1;
        float* red = team_mem;                                          // [groups][pieces][6]: maximum, sum, four outputs
        for (int e0 = 0; e0 < pieces; e0 += blockDim.x) {
            const int grp = groups > 1 ? (int)threadIdx.x / pieces : 0;
            const int e = groups > 1 ? (int)threadIdx.x - grp * pieces : e0 + (int)threadIdx.x;
            const bool active = grp < groups && e < pieces;
            float mx = -INFINITY, total = 0.f;
            f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
            const int col = active ? e / (HDV / 4) : 0, piece = active ? e - col * (HDV / 4) : 0;
            uint2 gate = make_uint2(0, 0);
            if (active) {
                if (grp == 0 && p.gate != nullptr) gate = ask_gate(col, piece * 4);
                const float* ml = p.part_ml + (row0 + col) * teams * 2;
                const float* po = p.part_o + (row0 + col) * teams * HDV + piece * 4;
                // (eight blocks' results at a time, their loads under way together and one change of the maximum for all)
                constexpr int AT_ONCE = 8;
                for (int t1 = grp; t1 < teams; t1 += AT_ONCE * groups) {
                    float mt[AT_ONCE], lt_[AT_ONCE], m_new = mx;
                    f32x4 v[AT_ONCE];
#pragma unroll
                    for (int i = 0; i < AT_ONCE; ++i) {
                        const int t = t1 + i * groups;
                        mt[i] = -INFINITY;
                        lt_[i] = 0.f;
                        v[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
                        if (t < teams) {
                            const float* pv = po + (size_t)t * HDV;
                            mt[i] = get_across(ml + 2 * t);
                            lt_[i] = get_across(ml + 2 * t + 1);
                            v[i] = (f32x4){get_across(pv), get_across(pv + 1), get_across(pv + 2), get_across(pv + 3)};
                        }
                    }
#pragma unroll
                    for (int i = 0; i < AT_ONCE; ++i) m_new = fmaxf(m_new, mt[i]);
                    const float back = m_new == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - m_new);       // rescales what is summed so far
                    o[0] *= back; o[1] *= back; o[2] *= back; o[3] *= back;
                    total *= back;
#pragma unroll
                    for (int i = 0; i < AT_ONCE; ++i) {
                        const float wt = mt[i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mt[i] - m_new);
                        o[0] = fmaf(v[i][0], wt, o[0]); o[1] = fmaf(v[i][1], wt, o[1]);
                        o[2] = fmaf(v[i][2], wt, o[2]); o[3] = fmaf(v[i][3], wt, o[3]);
                        total = fmaf(lt_[i], wt, total);
                    }
                    mx = m_new;
                }
            }
            if (groups > 1) {
                if (active) {                                           // (the waves' results in this memory were read before the count)
                    float* mine = red + ((size_t)grp * pieces + e) * 6;
                    mine[0] = mx; mine[1] = total; mine[2] = o[0]; mine[3] = o[1]; mine[4] = o[2]; mine[5] = o[3];
                }
                __syncthreads();
                if (!active || grp != 0) continue;
                for (int gi = 1; gi < groups; ++gi) {
                    const float* other = red + ((size_t)gi * pieces + e) * 6;
                    const float m_new = fmaxf(mx, other[0]);
                    const float back = m_new == -INFINITY ? 0.f : exp2f(mx - m_new);
                    const float wt = other[0] == -INFINITY ? 0.f : exp2f(other[0] - m_new);
                    o[0] = fmaf(other[2], wt, o[0] * back); o[1] = fmaf(other[3], wt, o[1] * back);
                    o[2] = fmaf(other[4], wt, o[2] * back); o[3] = fmaf(other[5], wt, o[3] * back);
                    total = fmaf(other[1], wt, total * back);
                    mx = m_new;
                }
            } else if (!active) {
                continue;
            }
            const float inv = 1.0f / (p.sink ? total + sink_term(p.sinks, (int)((row0 + col) % p.nq), mx) : total);
            put_out(col, piece * 4, o, inv, gate);
        }
        if (threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // zero again for the next call
    }
}

// ---- prompt portions, head size 128: blocks of eight waves that share keys and values ----------
// A block owns 128 columns of one request and key/value head and walks the keys in stages of 64: four waves
// (32 columns each) share a stage, and the block has two such groups, one on the even stages and one on the odd
// ones, that add up at the end.  A stage's keys and values come from the cache pages straight into shared memory
// (global_load_lds, 16 bytes a lane: no register holds them on the way), a group's next stage while this
// one is multiplied, and every wave reads its MFMA operands from there: the L2 is asked for a key once
// a block instead of once a wave.  A load instruction fills 1 KiB of shared memory in lane order, so
// the lane picks the piece it fetches such that the layout comes out swizzled:
//   keys    row of 256 bytes a key, the 16-byte piece c of key k at place c ^ ((k & 3) | ((k >> 3) & 3) << 2)
//   values  by groups of 16 keys: row of 32 bytes a feature, as the cache page holds it
// The swizzle of the keys spreads the 16 rows that a read takes at the same place over the banks (rows of 256
// bytes would all begin in the same one).  The counters show no bank conflict for either array
// (SQ_LDS_BANK_CONFLICT = 0); values with their halves swapped in every other block of eight features, which
// looked as good on paper, cost two extra cycles a read.
// Measured (one request, 32 query and 8 key/value heads; the kernel of single waves, then blocks of four waves, two
// a compute unit, then these): a prompt of 2,048 tokens 118 -> 77 -> 68 us, of 4,096 tokens 257 -> 201 us, of 8,192
// tokens 1.20 -> 0.75 -> 0.77 ms; a portion of 512 tokens at 7,680 181 -> 99 -> 116 us (keys split between two
// blocks).  Time stamps inside the kernel, 2,048 tokens: with blocks of four waves a compute unit held a long walk
// and a short one, the short one was done at once and the long one ran alone, a wave a SIMD, so the prompt took as
// long as its longest walk alone; and the blocks were handed out head by head (x was the tile), the longest walks of
// the last heads starting when the first heads' were done: compute units were busy between 15 and 102 us.  With the
// order of the kernel's comment and these blocks every unit runs two blocks and is busy 57 to 63 us; a block's
// pass over two stages takes 2.9 us (29 % of the matrix pipes' time), its start 1.2 us, the groups' sum 0.6, its
// end 2.4.  Timing-only variants of the blocks of four waves showed no single bound: without the exponentials 6 %
// faster, without the barrier 7 %, without the column maxima 8 %, without the second product 11 %, without the loads
// into shared memory 16 %.  Measured on a SIMD by itself: a matrix product takes 16 cycles and holds the issue for
// about 8 of them, an exponential 8 to 10, a 16-byte read of shared memory 32 when all four SIMDs read (128 bytes a
// cycle a compute unit: at 32 columns a wave the reads take as long as the products).
// 16 bytes a lane from memory straight into shared memory, 1 KiB a wave in lane order from `lds_at` on (the same for
// all lanes).  Written out so that the compiler does not count it among the loads it waits for: whoever reads the
// shared memory it fills waits for it by hand (s_waitcnt vmcnt) and passes a barrier.
__device__ __forceinline__ void lds_load16(const char* from, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(lds_at) : "memory");     // (m0 holds nothing of the compiler's across statements)
}

#define TILE_WAVES 4              // waves that share a stage: each with its own columns
#define TILE_GROUPS 2             // groups of such waves in a block: each with its own stages (see the kernel)
#define TILE_STAGE 64
#define TILE_K_BYTES (TILE_STAGE * HD * 2)
#define TILE_V_CHUNKS (HDV / 32)  // loads of 1 KiB that bring a group of 16 keys' values: 32 features each
#define TILE_BUF_BYTES (TILE_K_BYTES + TILE_STAGE * HDV * 2)

// Two column tiles of 16 a wave, two blocks a compute unit, two waves a SIMD.  (Four tiles a wave, so that every key and
// value read out of shared memory serves twice as many products, take the registers of a whole SIMD; with the softmax of
// one tile laid beside the products of the others in the instruction stream that ran at 530 TFLOP/s on a prompt of
// 8,192 tokens where two waves a SIMD run at 730, and the rescaling of accumulators that live in the matrix cores' own
// registers cost as much again.)
#define TILE_NBW 2
// NBW_: column tiles of 16 a wave.  One instead of two halves a block's columns (64) and doubles the blocks: for steps
// whose blocks of 128 columns would leave compute units without one (short prompts, few heads).
template <bool ENABLED = TILE_FITS, int NBW_ = TILE_NBW, int FORM = FORM_PLAIN>
__global__ __launch_bounds__(TILE_GROUPS * TILE_WAVES * IA_WAVE) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_tile_kernel(const AttnParams p) {
    if constexpr (ENABLED) {
        constexpr int NBW = NBW_;
        constexpr int WAVE_COLS = 16 * NBW;
        constexpr int TILE_COLS = TILE_WAVES * WAVE_COLS;
        // Two stages for each group.  The loads that fill them are written as instructions of their own below
        // (lds_load16): the compiler then neither knows of them nor waits for them before it reads an operand of
        // the other stage (it would, not knowing which stage a pointer chosen at run time names); the waits that
        // are needed stand in the code, one at the start of a stage.
        __shared__ __align__(16) char stage_mem[TILE_GROUPS * 2 * TILE_BUF_BYTES];
        // Two groups of four waves walk the same 128 columns: group 0 takes the even stages of the keys, group 1
        // the odd ones, each through its own two stages of shared memory, and at the end group 1 hands its sums
        // to group 0 through that memory.  A compute unit holds one block, two waves a SIMD that walk equally
        // far, and takes the next block when it is done.  (Two blocks of four waves, a long walk and a short
        // one so that a unit's work came out even, left the long walk alone on its unit for most of its time, a
        // wave a SIMD: a prompt of 2,048 tokens took as long as its longest walk took alone.)
        const int lane = threadIdx.x & (IA_WAVE - 1), wave = (threadIdx.x / IA_WAVE) & (TILE_WAVES - 1);
        const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x / (IA_WAVE * TILE_WAVES));
        const int r = lane & 15, G = lane >> 4;
        // The blocks of a launch are handed out in the order of their numbers, x fastest, to the chip's eight dies in
        // turn: x holds the key/value head, the split and the request, y the tile, longest walk first.  So the
        // longest walks of all heads and requests start first and a compute unit that is done takes the longest
        // that is left, and a head's tiles, which read the same keys, meet on one die and its L2 (eight heads).
        const int heads_splits = p.nkv * p.splits;
        const int seq_local = blockIdx.x / heads_splits, head_split = blockIdx.x - seq_local * heads_splits;
        const int kvh = head_split / p.splits, split = head_split - kvh * p.splits;
        const int seq = p.seq_begin + seq_local;
        const int g = p.nq / p.nkv;
        const int t0 = p.cu_tokens[seq], q_len = p.cu_tokens[seq + 1] - t0;
        const int n_cols = q_len * g;
        const int n_tiles = (n_cols + TILE_COLS - 1) / TILE_COLS;
        if ((int)blockIdx.y >= n_tiles) return;
        const int bcol0 = (n_tiles - 1 - (int)blockIdx.y) * TILE_COLS;
        const int kv_start = p.positions[t0];
        const int kv_total = kv_start + q_len;
        const int* bt = p.block_table + (size_t)seq * p.max_pages;
        const int blast = (bcol0 + TILE_COLS <= n_cols ? bcol0 + TILE_COLS : n_cols) - 1;
        const int bpmin = kv_start + bcol0 / g, bpmax = kv_start + blast / g;
        const int bfloor = ia_key_floor(bpmin, p.window, p.mask_chunk);   // first key the block sees
        int lo = bfloor;
        lo &= ~(TILE_STAGE - 1);
        int hi = bpmax + 1;
        // the first positions that every query sees: stages of their own ahead of the rest, or, where no whole stage lies
        // between the two, a walk from 0
        const int keep = FORM != FORM_PLAIN ? p.keep_first : 0;
        int pre_lo = 0, pre_hi = 0;
        if (FORM != FORM_PLAIN && keep > 0) {
            if (keep >= lo) lo = 0;
            else pre_hi = (keep + TILE_STAGE - 1) & ~(TILE_STAGE - 1);
        }
        if (p.splits > 1) {             // this block's share of the keys (`chunk` is a multiple of a stage)
            const int c_lo = split * p.chunk, c_hi = c_lo + p.chunk;
            lo = lo > c_lo ? lo : c_lo;
            hi = hi < c_hi ? hi : c_hi;
            pre_lo = c_lo;
            pre_hi = pre_hi < c_hi ? pre_hi : c_hi;
        }
        const int pre_stages = FORM != FORM_PLAIN && pre_lo < pre_hi ? (pre_hi - pre_lo) / TILE_STAGE : 0;
        const int stages = pre_stages + (hi > lo ? (hi - lo + TILE_STAGE - 1) / TILE_STAGE : 0);
        auto stage_key = [&](int s) {   // the first key of stage s
            if (FORM == FORM_PLAIN) return lo + s * TILE_STAGE;
            return s < pre_stages ? pre_lo + s * TILE_STAGE : lo + (s - pre_stages) * TILE_STAGE;
        };

        // this wave's columns (a wave without any still brings its share of the stages)
        const int col0 = bcol0 + wave * WAVE_COLS;
        const bool has_cols = col0 < n_cols;
        int tq[NBW], head[NBW], pos[NBW];
        bool cvalid[NBW];
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) {
            const int c = col0 + nb * 16 + r;
            cvalid[nb] = c < n_cols;
            const int cc = cvalid[nb] ? c : n_cols - 1;
            tq[nb] = cc / g;
            head[nb] = kvh * g + (cc - tq[nb] * g);
            pos[nb] = kv_start + tq[nb];
        }
        const int wlast = (col0 + WAVE_COLS <= n_cols ? col0 + WAVE_COLS : n_cols) - 1;
        const int pmin = kv_start + (has_cols ? col0 : 0) / g, pmax = has_cols ? kv_start + wlast / g : -1;
        const int wlo = ia_key_floor(pmin, p.window, p.mask_chunk);
        const int wtop = ia_key_floor(pmax > 0 ? pmax : 0, p.window, p.mask_chunk);      // the first key that the wave's last column sees

        uint4 qreg[NBW][KS];
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) {
            const bf16_t* qrow = p.q + ((size_t)(t0 + tq[nb]) * p.nq + head[nb]) * HD;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) qreg[nb][ks] = cvalid[nb] ? *(const uint4*)(qrow + ks * 32 + G * 8) : zero4();
        }
        f32x4 acc[NBW][DBV];
        float m[NBW], l[NBW];
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) {
            m[nb] = -INFINITY;
            l[nb] = 0.f;
#pragma unroll
            for (int db = 0; db < DBV; ++db) acc[nb][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }

        // ---- a stage on its way: wave w brings keys 16 w .. + 16 and features 32 w .. + 32 ----------
        // Groups of 16 keys past the request's length are read from the group of its last key instead
        // (their scores are masked and their values zeroed below): the pages behind may not exist.
        // Wave w brings the stage's w-th group of 16 keys and their values: one place in one page, the same
        // for all its lanes.  The pages' numbers come 64 at a time into a register, lane i with the entry
        // pages_base + i of the block table, and a stage takes its number from there with a lane read: a read
        // of the block table in every stage, through the scalar cache, kept each wave waiting for a trip to the
        // memory before its first operand of the stage (the counter of those reads is the shared memory's too).
        // What a lane adds to that place does not change from stage to stage.
        const int wave_s = __builtin_amdgcn_readfirstlane(wave);
        const int last_idx = (kv_total - 1) / p.page;
        int pages_base = 0, pages_reg = 0;
        auto pages_load = [&](int base) {
            pages_base = base;
            const int idx = base + lane;
            pages_reg = bt[idx < last_idx ? idx : last_idx];
        };
        auto pages_for = [&](int s, int& page, int& off) {
            const int key0 = stage_key(s) + 16 * wave_s;
            const int k = key0 < kv_total ? key0 : (kv_total - 1) & ~15;
            const int idx = k / p.page;
            if (idx >= pages_base + IA_WAVE) pages_load(idx);
            page = __builtin_amdgcn_readlane(pages_reg, idx - pages_base);
            off = k - idx * p.page;
        };
        uint32_t k_from[4];             // keys: chunk c is rows 4 c .. + 4 of the group, a lane's piece swizzled
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int row = 4 * c + (lane >> 4), key = 16 * wave + row;
            const int piece = (lane & 15) ^ ((key & 3) | (((key >> 3) & 3) << 2));
            k_from[c] = (uint32_t)(row * (HD * 2) + piece * 16);
        }
        // values: chunk c is features 32 c .. + 32, two lanes a feature (its 16 keys)
        const int v_half = lane & 1;                                            // which eight keys the lane's piece holds
        const uint32_t v_from = (uint32_t)(((lane >> 1) * p.page + v_half * 8) * 2);
        auto issue = [&](char* buf, int page, int off) {
            const char* krows = (const char*)(p.k_cache + (((size_t)page * p.nkv + kvh) * p.page + off) * HD);
            const char* vrows = (const char*)(p.v_cache + ((size_t)page * p.nkv + kvh) * HDV * p.page + off);
            const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)buf;
#pragma unroll
            for (int c = 0; c < 4; ++c) lds_load16(krows + k_from[c], at + (16 * wave_s + 4 * c) * (HD * 2));
#pragma unroll
            for (int c = 0; c < TILE_V_CHUNKS; ++c)
                lds_load16(vrows + (size_t)c * 32 * p.page * 2 + v_from, at + TILE_K_BYTES + wave_s * (16 * HDV * 2) + c * 1024);
        };
        // values of keys past the request's length may hold anything at all: a lane zeroes them in the
        // pieces that it brought itself, once they have arrived
        // So may the values of keys below the block's window, between the stage's start and the first key that any
        // of its columns sees: the window has passed them, and their pages may have been given back.
        auto zero_tail = [&](int s, char* buf) {
            const int kb = stage_key(s);
            const int mine = kb + 16 * wave_s + 8 * v_half;          // the first of this lane's eight keys
            const int first_bad = kb + TILE_STAGE <= kv_total ? 8 : kv_total - mine;
            const int first_good = kb < bfloor ? bfloor - mine : 0;
            if (first_bad >= 8 && first_good <= 0) return;
            const int kept = keep - mine;                            // (keys below this index are first positions: seen)
#pragma unroll
            for (int c = 0; c < TILE_V_CHUNKS; ++c) {
                uint4* at = (uint4*)(buf + TILE_K_BYTES + wave_s * (16 * HDV * 2) + c * 1024 + lane * 16);
                const uint4 v = *at;
                uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j >= first_bad || (j < first_good && (FORM == FORM_PLAIN || j >= kept))) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                *at = make_uint4(w[0], w[1], w[2], w[3]);
            }
        };

        // this lane's places in a stage: they do not change from stage to stage
        uint32_t k_at[KS];              // keys: the lane's row of tile 0 of step 0 and its swizzled piece of dim step ks
        {
            const int kl = 8 * (r >> 2) + (r & 3);
            const uint32_t k_xor = (uint32_t)((kl & 3) | (((kl >> 3) & 3) << 2));
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) k_at[ks] = (uint32_t)(kl * (HD * 2)) + (((uint32_t)(ks * 4 + G) ^ k_xor) * 16);
        }
        // values: group of 16 keys (G >> 1 of the step's two), feature row of 32 bytes, half G & 1
        const uint32_t v_at = (uint32_t)((G >> 1) * (16 * HDV * 2) + r * 32 + (G & 1) * 16);
        int page_l, off_l;
        auto stage = [&](int s, char* buf, char* other) __attribute__((always_inline)) {
            if (s >= stages) {                             // the other group has a stage more: its barrier is kept
                __syncthreads();
                return;
            }
            __builtin_amdgcn_s_waitcnt(0);                 // this wave's part of stage s has arrived
            zero_tail(s, buf);
            __syncthreads();                               // everybody's has, and everybody is done with the stage before
            // The loads of the group's next stage: group 0 asks for them here, group 1 between its two steps.  A load
            // instruction holds its wave until the compute unit's one address unit takes it, 1 KiB in 16 cycles: with
            // all eight waves asking at once after the barrier (64 KiB a pass) each waited some 1,100 to 1,700 cycles
            // of a pass's 6,500, all at the same time (8,192 tokens 736 -> 655 us).
            const bool more = s + TILE_GROUPS < stages;
            if (more && kg == 0) issue(other, page_l, off_l);
            const int kb = stage_key(s);
            // Steps of 32 keys.  A wave's operands are asked for a phase ahead of their use: the values of a
            // step before its softmax is worked out, the keys of the next step before this step's second
            // product, so that the shared memory's latency passes behind arithmetic.
            bool live[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)        // something of the step is visible to this wave's columns
                live[u] = !(kb + 32 * u > pmax || (kb + 32 * u + 31 < wlo && (FORM == FORM_PLAIN || kb + 32 * u >= keep)));
            uint4 kop[2][KS];
            auto read_keys = [&](int u) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        kop[t][ks] = *(const uint4*)(buf + (32 * u + 4 * t) * (HD * 2) + k_at[ks]);
            };
            if (live[0]) read_keys(0);
            else if (live[1]) read_keys(1);
            // A step of 32 keys.  The wave's two column tiles take turns so that the softmax of one (vector
            // arithmetic) has matrix products of the other beside it in the same stretch of code: the scores of
            // tile 1 beside the softmax of tile 0, the second product of tile 0 beside the softmax of tile 1.  The
            // order of every sum is as before.  EDGE: some key of the step is masked for some column.
            auto scores = [&](int nb, f32x4 (&sacc)[2]) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    sacc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, kop[t][ks]), __builtin_bit_cast(bf16x8, qreg[nb][ks]), sacc[t], 0, 0, 0);
                }
            };
            auto softmax = [&](auto edge_c, int nb, int k0, const f32x4 (&sacc)[2], uint4& pb, float& alpha) {
                constexpr bool EDGE = decltype(edge_c)::value;
                float sc[8];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) sc[4 * t + i] = FORM == FORM_CAP ? tanh_exp2(sacc[t][i] * p.cap_in) : sacc[t][i];
                if constexpr (EDGE) {
                    const int kbase_idx = k0 + 8 * G;
                    const int floor_key = ia_key_floor(pos[nb], p.window, p.mask_chunk);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int key = kbase_idx + j;
                        if (key > pos[nb] || (key < floor_key && (FORM == FORM_PLAIN || key >= keep))) sc[j] = -INFINITY;
                    }
                }
                // (the compiler's own maximum: written out as v_max3 instructions, which the compiler does not check
                // against the matrix products that wrote the scores, the maxima could read a score's register before
                // its product had written it, and took a probability of the step before for a score; with the wait
                // that forbids that tied to the scores a prompt of 8,192 tokens took 823 us, so 728)
                float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
                mx = column_max(mx);
                // The exponents' reference point moves only when the step's maximum has passed it by 2^8
                // (probabilities then reach 2^8 at most, which 32-bit sums and bfloat16 operands hold as
                // well as 1): the accumulators are rescaled a few times a walk instead of at most steps.
                const float cand = mx * p.scale_log2;
                const bool rise = cand > m[nb] + 8.0f;              // also the first finite maximum after -inf
                const float m_new = rise ? cand : m[nb];
                const float m_use = m_new == -INFINITY ? 0.f : m_new;
                alpha = rise ? __builtin_amdgcn_exp2f(m[nb] - m_use) : 1.0f;
                float pr[8], psum = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    pr[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j], p.scale_log2, -m_use));
                    psum += pr[j];
                }
                l[nb] = l[nb] * alpha + psum;
                m[nb] = m_new;
                pb.x = pack_bf16x2(pr[0], pr[1]);
                pb.y = pack_bf16x2(pr[2], pr[3]);
                pb.z = pack_bf16x2(pr[4], pr[5]);
                pb.w = pack_bf16x2(pr[6], pr[7]);
            };
            auto rescale = [&](int nb, float alpha) {
                if (__any(alpha != 1.0f)) {
#pragma unroll
                    for (int db = 0; db < DBV; ++db) {
                        acc[nb][db][0] *= alpha; acc[nb][db][1] *= alpha;
                        acc[nb][db][2] *= alpha; acc[nb][db][3] *= alpha;
                    }
                }
            };
            auto weighted = [&](int nb, const uint4 (&vop)[DBV], const uint4& pb) {
#pragma unroll
                for (int db = 0; db < DBV; ++db)
                    acc[nb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, vop[db]), __builtin_bit_cast(bf16x8, pb), acc[nb][db], 0, 0, 0);
            };
            // eight matrix products with a share of the vector instructions after each
            auto beside = [&]() {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one matrix product
                    __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);      // nine vector instructions
                }
            };
            auto pin = [&](uint4& pb, float& alpha) {
                // (pins the probabilities to the stretch of code they are formed in: left alone, the compiler moves
                // their arithmetic behind the branch of the rescaling, next to the product that uses them)
                asm volatile("" : "+v"(pb.x), "+v"(pb.y), "+v"(pb.z), "+v"(pb.w), "+v"(alpha));
            };
            auto step = [&](auto edge_c, int u) {
                const int k0 = kb + 32 * u;
                uint4 vop[DBV];
                if constexpr (NBW == 1) {
                    // one column tile: nothing of its own to lay beside the softmax (the SIMD's other wave is)
                    f32x4 s0[2];
                    uint4 pb0;
                    float alpha0;
                    scores(0, s0);
#pragma unroll
                    for (int db = 0; db < DBV; ++db)
                        vop[db] = *(const uint4*)(buf + TILE_K_BYTES + u * (32 * HDV * 2) + db * 512 + v_at);
                    softmax(edge_c, 0, k0, s0, pb0, alpha0);
                    if (u == 0) read_keys(1);
                    rescale(0, alpha0);
                    weighted(0, vop, pb0);
                } else {
                f32x4 s0[2], s1[2];
                uint4 pb0, pb1;
                float alpha0, alpha1;
                scores(0, s0);
#pragma unroll
                for (int db = 0; db < DBV; ++db)
                    vop[db] = *(const uint4*)(buf + TILE_K_BYTES + u * (32 * HDV * 2) + db * 512 + v_at);
                __builtin_amdgcn_sched_barrier(0);
                scores(1, s1);
                softmax(edge_c, 0, k0, s0, pb0, alpha0);
                pin(pb0, alpha0);
                beside();
                __builtin_amdgcn_sched_barrier(0);
                if (u == 0) read_keys(1);               // (a step that this wave skips: read all the same, used by nobody)
                rescale(0, alpha0);
                __builtin_amdgcn_sched_barrier(0);
                weighted(0, vop, pb0);
                softmax(edge_c, 1, k0, s1, pb1, alpha1);
                pin(pb1, alpha1);
                beside();
                __builtin_amdgcn_sched_barrier(0);
                rescale(1, alpha1);
                weighted(1, vop, pb1);
                }
            };
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (u == 1 && more && kg != 0) issue(other, page_l, off_l);
                if (!live[u]) continue;
                const int k0 = kb + 32 * u;
                // (The form of this condition matters: without the test of window and chunk the compiler merges the two
                // copies of the step, spills 107 registers and a prompt of 2,048 tokens takes 150 us instead of 56.)
                const bool edge = k0 + 31 > pmin || ((p.window > 0 || p.mask_chunk > 0) && k0 < wtop);
                if (edge) step(std::true_type(), u);
                else step(std::false_type(), u);
            }
            if (s + 2 * TILE_GROUPS < stages) pages_for(s + 2 * TILE_GROUPS, page_l, off_l);
        };
        // A group's walk: its stages are kg, kg + 2, ...; both groups pass the same number of barriers.
        auto walk = [&](char* first, char* second) __attribute__((always_inline)) {
            if (kg < stages) {
                const int key0 = stage_key(kg) + 16 * wave_s;
                pages_load((key0 < kv_total ? key0 : (kv_total - 1) & ~15) / p.page);
                pages_for(kg, page_l, off_l);
                issue(first, page_l, off_l);
                if (kg + TILE_GROUPS < stages) pages_for(kg + TILE_GROUPS, page_l, off_l);
            }
            for (int s = kg; s - kg < stages; s += 2 * TILE_GROUPS) {
                stage(s, first, second);
                if (s - kg + TILE_GROUPS < stages) stage(s + TILE_GROUPS, second, first);
            }
        };
        walk(stage_mem + (2 * kg) * TILE_BUF_BYTES, stage_mem + (2 * kg + 1) * TILE_BUF_BYTES);

        // ---- group 1 hands its sums to group 0: accumulators through its own two stages, maxima and sums through
        // group 0's first ------------------------------------------------------------------------------------------
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        {
            f32x4* xacc = (f32x4*)(stage_mem + 2 * TILE_BUF_BYTES + wave_s * (TILE_BUF_BYTES / 2));      // [nb][db][lane]
            __shared__ float2 xml_mem[TILE_WAVES * NBW * IA_WAVE];
            float2* xml = xml_mem + wave_s * NBW * IA_WAVE;                                             // [nb][lane]
            if (kg == 1) {
#pragma unroll
                for (int nb = 0; nb < NBW; ++nb) {
#pragma unroll
                    for (int db = 0; db < DBV; ++db) xacc[(nb * DBV + db) * IA_WAVE + lane] = acc[nb][db];
                    xml[nb * IA_WAVE + lane] = make_float2(m[nb], l[nb]);
                }
            }
            __syncthreads();
            if (kg == 1) return;
#pragma unroll
            for (int nb = 0; nb < NBW; ++nb) {
                const float2 other = xml[nb * IA_WAVE + lane];
                const float top = fmaxf(m[nb], other.x);
                const float mine_w = m[nb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[nb] - top);
                const float other_w = other.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(other.x - top);
                l[nb] = l[nb] * mine_w + other.y * other_w;
                m[nb] = top;
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    const f32x4 o = xacc[(nb * DBV + db) * IA_WAVE + lane];
                    acc[nb][db][0] = acc[nb][db][0] * mine_w + o[0] * other_w;
                    acc[nb][db][1] = acc[nb][db][1] * mine_w + o[1] * other_w;
                    acc[nb][db][2] = acc[nb][db][2] * mine_w + o[2] * other_w;
                    acc[nb][db][3] = acc[nb][db][3] * mine_w + o[3] * other_w;
                }
            }
        }
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) {
            const float lt = column_sum(l[nb]);
            if (!cvalid[nb]) continue;
            const size_t row = (size_t)(t0 + tq[nb]) * p.nq + head[nb];
            if (p.splits == 1) {
                const float inv = 1.0f / (p.sink ? lt + sink_term(p.sinks, head[nb], m[nb]) : lt);
                bf16_t* o = p.out + row * HDV + 4 * G;
#pragma unroll
                for (int db = 0; db < DBV; ++db) {
                    uint2 w;
                    w.x = pack_bf16x2(acc[nb][db][0] * inv, acc[nb][db][1] * inv);
                    w.y = pack_bf16x2(acc[nb][db][2] * inv, acc[nb][db][3] * inv);
                    *(uint2*)(o + 16 * db) = w;
                }
            } else {
                // for the merge: sums and accumulators relative to the exponents' reference point m
                float* o = p.part_o + (row * p.splits + split) * HDV + 4 * G;
#pragma unroll
                for (int db = 0; db < DBV; ++db) *(f32x4*)(o + 16 * db) = acc[nb][db];
                if (G == 0) {
                    float* ml = p.part_ml + (row * p.splits + split) * 2;
                    ml[0] = m[nb];
                    ml[1] = lt;
                }
            }
        }
    }
}

static int g_tiles = 1;
// Measurement switch: 0 keeps prompt portions on the kernel of single waves; 2: blocks of 64 columns whatever the
// step's size; 3: of 128.
extern "C" void ia_attention_mfma_tiles(int on) { g_tiles = on; }

// Compute units of the current device (asked for once a device).
static int attn_cus() {
    static int cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int n = 0;
        cus[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    }
    return cus[dev];
}

// Merges the partial results of the key splits of one (token, head): one block a row.  The
// partial results were written by other compute units, so every read is a long way off: the
// block's waves share the splits between them (wave w takes splits w, w + waves, ...) and
// every lane has all its loads in flight at once; the waves' sums meet in shared memory and
// are added in wave order.
#define MERGE_WAVES 16
__global__ __launch_bounds__(MERGE_WAVES * IA_WAVE) void attn_merge_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ part_o, const float* __restrict__ part_ml, int splits,
    size_t first_row, int sink, const float* __restrict__ sinks, int nq) {
    constexpr int PER = (HDV + IA_WAVE - 1) / IA_WAVE;
    __shared__ float weight[256];
    __shared__ float red[MERGE_WAVES][PER * IA_WAVE];
    __shared__ float s_total;
    const size_t row = first_row + blockIdx.x;
    const int lane = threadIdx.x & (IA_WAVE - 1), wave = threadIdx.x / IA_WAVE;
    const float* ml = part_ml + row * splits * 2;
    const float* po = part_o + row * splits * HDV;
    // this wave's partial outputs, asked for before anything is waited for
    float v[256 / MERGE_WAVES][PER];
#pragma unroll
    for (int i = 0; i < 256 / MERGE_WAVES; ++i) {
        const int s = wave + i * MERGE_WAVES;
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int e = lane + t * IA_WAVE;
            v[i][t] = (s < splits && e < HDV) ? po[(size_t)s * HDV + e] : 0.f;
        }
    }
    if (wave == 0) {
        float mx = -INFINITY;
        for (int s = lane; s < splits; s += IA_WAVE) mx = fmaxf(mx, ml[2 * s]);
        mx = wave_max(mx);
        float total = 0.f;
        for (int s = lane; s < splits; s += IA_WAVE) {
            const float ms = ml[2 * s];
            const float w = ms == -INFINITY ? 0.f : exp2f(ms - mx);      // a split that held no key of this row
            weight[s] = w;
            total += ml[2 * s + 1] * w;
        }
        total = wave_sum(total);
        if (lane == 0) s_total = sink ? total + sink_term(sinks, (int)(row % nq), mx) : total;
    }
    __syncthreads();
    float o[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) o[t] = 0.f;
#pragma unroll
    for (int i = 0; i < 256 / MERGE_WAVES; ++i) {
        const int s = wave + i * MERGE_WAVES;
        if (s < splits) {
            const float w = weight[s];
#pragma unroll
            for (int t = 0; t < PER; ++t) o[t] = fmaf(v[i][t], w, o[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < PER; ++t) red[wave][lane + t * IA_WAVE] = o[t];
    __syncthreads();
    if (wave != 0) return;
    const float inv = 1.0f / s_total;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int e = lane + t * IA_WAVE;
        float sum = red[0][e];
        for (int w = 1; w < MERGE_WAVES; ++w) sum += red[w][e];
        if (e < HDV) out[row * HDV + e].bits = f32_to_bf16_bits(sum * inv);
    }
}

// The same merge for steps with many rows and few splits (portions of prompts, decode steps of many
// requests): a wave a row, every lane with the splits' maxima and sums of its row and HDV / 64 features.
// Kernel times at head size 128, context 8,192, 32 heads (the block-a-row kernel against this one):
// 512 rows of 8 splits 4.9 against 7.6 us, 1,024 rows of 4 splits 7.0 against 5.1, 2,048 rows of 4 splits
// 12.2 against 5.0.
#define MERGE_ROWS_WAVES 4
#define MERGE_ROWS_FROM 1024
__global__ __launch_bounds__(MERGE_ROWS_WAVES * IA_WAVE) void attn_merge_rows_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ part_o, const float* __restrict__ part_ml, int splits,
    size_t first_row, size_t n_rows, int sink, const float* __restrict__ sinks, int nq) {
    constexpr int PER = (HDV + IA_WAVE - 1) / IA_WAVE;
    const int lane = threadIdx.x & (IA_WAVE - 1), wave = threadIdx.x / IA_WAVE;
    const size_t local = (size_t)blockIdx.x * MERGE_ROWS_WAVES + wave;
    if (local >= n_rows) return;
    const size_t row = first_row + local;
    const float* ml = part_ml + row * splits * 2;
    const float* po = part_o + row * splits * HDV;
    float mx = -INFINITY;
    for (int s = 0; s < splits; ++s) mx = fmaxf(mx, ml[2 * s]);
    float total = 0.f, o[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) o[t] = 0.f;
    for (int s = 0; s < splits; ++s) {
        const float ms = ml[2 * s];
        const float w = ms == -INFINITY ? 0.f : exp2f(ms - mx);          // a split that held no key of this row
        total += ml[2 * s + 1] * w;
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int e = lane + t * IA_WAVE;
            if (e < HDV) o[t] = fmaf(po[(size_t)s * HDV + e], w, o[t]);
        }
    }
    const float inv = 1.0f / (sink ? total + sink_term(sinks, (int)(row % nq), mx) : total);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int e = lane + t * IA_WAVE;
        if (e < HDV) out[row * HDV + e].bits = f32_to_bf16_bits(o[t] * inv);
    }
}

extern "C" int ia_attention_mfma_head_dim(void) { return HD; }
extern "C" int ia_attention_mfma_value_dim(void) { return HDV; }

// Floats of workspace that `splits` > 1 needs: partial outputs, then maxima and sums.
extern "C" long long ia_attention_mfma_workspace(int n, int nq, int splits) {
    return splits > 1 ? (long long)n * nq * splits * (HDV + 2) : 0;
}

// The requests seq_begin .. seq_begin + n_seqs of the step, whose tokens are token_begin ..
// token_begin + n_tokens of its n.  max_q_len: the most tokens any of them has in this step;
// max_kv_len: their greatest length after it; `chunk`: keys per split (a multiple of 32,
// splits * chunk >= max_kv_len).  The workspace is sized for all n tokens.
struct FusedArgs {
    const void* qkv; const float* q_norm_w; const float* k_norm_w; const float* cos_t; const float* sin_t;
    const int* slots; float eps; int add_one;
    int row_ld, q_off, k_off, v_off, rot;
    const void* gate; int gate_ld, gate_per_head;
    int* counters; int n_counters;
};

// Neighbouring splits that one block of the decode kernel takes (a wave each): up to four, or two where the waves'
// results for g query heads of a key/value head would not fit 64 KiB of shared memory; every block takes as many.
static size_t decode_team_bytes(int team, int g) {
    const int cols = g < 16 ? g : 16;
    const size_t waves = (size_t)team * (decode_wave_words(cols) + 2 * cols), groups = (size_t)team * IA_WAVE * 6;   // (see the kernel's end)
    return (waves > groups ? waves : groups) * sizeof(float);
}
static int decode_team(int splits, int g) {
    const int team = decode_team_bytes(DECODE_TEAM, g) <= 65536 ? DECODE_TEAM : 2;
    int t = splits < team ? splits : team;
    while (splits % t) --t;
    return t;
}

// Floats of workspace that a decode step of `splits` key splits needs (one partial result a block), and the
// zeroed 32-bit counters (one for each request, key/value head and block of 16 query heads).
extern "C" long long ia_attention_decode_workspace(int n, int nq, int nkv, int splits) {
    if (n <= 0 || nq <= 0 || nkv <= 0 || splits <= 0) return 0;
    const int teams = splits / decode_team(splits, nq / nkv);
    return teams > 1 ? (long long)n * nq * teams * (HDV + 2) : 0;
}
extern "C" long long ia_attention_decode_counters(int n, int nq, int nkv, int splits) {
    if (n <= 0 || nq <= 0 || nkv <= 0 || splits <= 0) return 0;
    const int teams = splits / decode_team(splits, nq / nkv);
    return teams > 1 ? (long long)n * nkv * ((nq / nkv + 15) / 16) : 0;
}

static int attention_launch(void* out, float* workspace, const void* q, const void* k_cache,
                            const void* v_cache, const int* block_table, const int* cu_tokens,
                            const int* positions, int n, int seq_begin, int n_seqs, int token_begin,
                            int n_tokens, int max_q_len, int max_kv_len, int max_pages,
                            int nq, int nkv, int d, int page_size, int window, float scale,
                            int splits, int chunk, int sink, int mask_chunk, const float* sinks, int keep_first, float softcap,
                            const FusedArgs* fused, hipStream_t stream) {
    IA_CHECK(d == HD, "attention_mfma: built for head_dim %d, called with %d", HD, d);
    IA_CHECK(n >= 0 && n_seqs >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0,
             "attention_mfma: bad sizes n=%d seqs=%d nq=%d nkv=%d", n, n_seqs, nq, nkv);
    IA_CHECK(seq_begin >= 0 && token_begin >= 0 && n_tokens >= 0 && token_begin + n_tokens <= n,
             "attention_mfma: bad ranges seq_begin=%d tokens %d..+%d of %d", seq_begin, token_begin, n_tokens, n);
    IA_CHECK(page_size > 0 && page_size % 16 == 0, "attention_mfma: page size %d must be a multiple of 16", page_size);
    IA_CHECK(max_pages > 0 && window >= 0 && max_q_len >= 1, "attention_mfma: bad geometry max_pages=%d window=%d max_q_len=%d",
             max_pages, window, max_q_len);
    IA_CHECK(splits >= 1 && splits <= 256 &&
             (splits == 1 || ((workspace != nullptr || fused != nullptr) && chunk >= 32 && chunk % 32 == 0)),
             "attention_mfma: bad split of the keys (splits=%d chunk=%d)", splits, chunk);
    IA_CHECK((long long)nkv * splits <= 65535 && n_seqs <= 65535, "attention_mfma: grid too large (nkv*splits=%d seqs=%d)",
             nkv * splits, n_seqs);
    if (n_tokens == 0 || n_seqs == 0) return 0;
    const int g = nq / nkv;
    AttnParams p;
    p.out = (bf16_t*)out;
    p.part_o = workspace;
    p.part_ml = workspace ? workspace + (size_t)n * nq * splits * HDV : nullptr;
    p.q = (const bf16_t*)q;
    p.k_cache = (const bf16_t*)k_cache;
    p.v_cache = (const bf16_t*)v_cache;
    p.k_cache_w = (bf16_t*)k_cache;
    p.v_cache_w = (bf16_t*)v_cache;
    p.qkv = nullptr; p.q_norm_w = p.k_norm_w = p.cos_t = p.sin_t = nullptr; p.slots = nullptr;
    p.norm_eps = 0.f; p.norm_add_one = 0; p.row_ld = p.q_off = p.k_off = p.v_off = p.rot = 0;
    p.gate = nullptr; p.gate_ld = p.gate_per_head = 0;
    p.block_table = block_table;
    p.cu_tokens = cu_tokens;
    p.positions = positions;
    p.max_pages = max_pages; p.nq = nq; p.nkv = nkv; p.page = page_size; p.window = window;
    p.splits = splits; p.chunk = chunk; p.seq_begin = seq_begin; p.token_begin = token_begin;
    p.scale_log2 = scale * 1.4426950408889634f;
    p.sink = sink ? 1 : 0;
    IA_CHECK(mask_chunk >= 0 && (sinks == nullptr || sink), "attention_mfma: mask_chunk %d must be >= 0 (0 = none), and sink values go with a sink", mask_chunk);
    p.sinks = sinks; p.mask_chunk = mask_chunk;
    IA_CHECK(keep_first >= 0 && softcap >= 0.f, "attention_mfma: keep_first %d and softcap %g must be >= 0 (0 = none)", keep_first, (double)softcap);
    p.keep_first = keep_first; p.cap_in = 0.f; p.page_magic = 0; p.page_shift = 0; p.teams = p.col_blocks = 1;
    if (softcap > 0.f) {
        p.cap_in = scale / softcap * (2.0f * 1.4426950408889634f);
        p.scale_log2 = softcap * 1.4426950408889634f;
    }
    const int form = softcap > 0.f ? FORM_CAP : keep_first > 0 ? FORM_KEEP : FORM_PLAIN;
    const long long cols = (long long)max_q_len * g;
    // Columns a wave: 16 for decode, 32 for portions of prompts.  (64 keep every loaded key and
    // value in use for twice as many products but need the registers of a whole SIMD; with 32
    // two waves share a SIMD and one's matrix work overlaps the other's softmax, which is faster.)
    p.pair = (splits == 1 && cols > 16 && 2LL * max_q_len > max_kv_len) ? 1 : 0;
    const int nb = cols > 16 ? 2 : 1;
    const long long col_blocks = (cols + 16 * nb - 1) / (16 * nb);
    const dim3 grid((unsigned)(p.pair ? (col_blocks + 1) / 2 : col_blocks), nkv * splits, n_seqs);
    if (fused != nullptr) {
        IA_CHECK(form == FORM_PLAIN, "attention_mfma: the fused form takes no kept first positions and no capped scores");
        IA_CHECK(HD % 64 == 0 && max_q_len == 1, "attention_mfma: the fused form takes single tokens and head sizes in "
                 "steps of 64 (head size %d, %d tokens a request)", HD, max_q_len);
        p.qkv = (const bf16_t*)fused->qkv;
        p.q_norm_w = fused->q_norm_w; p.k_norm_w = fused->k_norm_w;
        p.cos_t = fused->cos_t; p.sin_t = fused->sin_t; p.slots = fused->slots;
        p.norm_eps = fused->eps; p.norm_add_one = fused->add_one;
        p.row_ld = fused->row_ld; p.q_off = fused->q_off; p.k_off = fused->k_off; p.v_off = fused->v_off; p.rot = fused->rot;
        p.gate = (const bf16_t*)fused->gate; p.gate_ld = fused->gate_ld; p.gate_per_head = fused->gate_per_head;
        // 16 columns a wave, whatever the number of query heads of a key/value head
        const int team = decode_team(splits, g), teams = splits / team;
        const int col_blocks = (g + 15) / 16;
        IA_CHECK(teams == 1 || workspace != nullptr, "attention_mfma: the decode kernel needs a workspace for %d blocks a request "
                 "and key/value head", teams);
        IA_CHECK(teams == 1 || (fused->counters != nullptr && (long long)n_seqs * nkv * col_blocks <= fused->n_counters),
                 "attention_mfma: the decode kernel needs %lld zeroed counters, got %d", (long long)n_seqs * nkv * col_blocks,
                 fused->counters ? fused->n_counters : 0);
        p.part_ml = workspace ? workspace + (size_t)n * nq * teams * HDV : nullptr;
        const dim3 fgrid((unsigned)(col_blocks * teams), nkv, n_seqs);
        const size_t shared = decode_team_bytes(team, g);
        p.teams = teams;
        p.col_blocks = col_blocks;
        // With d = page / 16 and 2^(s - 1) < d <= 2^s, M = 2^(31 + s) / d rounded up fits 32 bits and exceeds the quotient by less than
        // 2^s / d parts of 2^-(31 + s): q M >> (31 + s) is q / d for every q = pos / 16 below 2^27, hence for every position.
        const uint32_t d16 = (uint32_t)page_size / 16;
        p.page_shift = d16 > 1 ? 32 - __builtin_clz(d16 - 1) : 0;
        p.page_magic = (uint32_t)(((1ULL << (31 + p.page_shift)) + d16 - 1) / d16);
        attn_decode_kernel<><<<fgrid, team * IA_WAVE, shared, stream>>>(p, fused->counters, team);
        IA_LAUNCH_CHECK("attention_decode");
        return 0;
    } else if (TILE_FITS && g_tiles && (cols >= 16 * TILE_NBW * TILE_WAVES ? splits == 1 || chunk % TILE_STAGE == 0 :
                                        splits == 1 && cols > 16 && max_kv_len > 32 && (cols + 63) / 64 * nkv * n_seqs <= attn_cus())) {
        // portions of prompts: blocks of four waves that share the keys through shared memory.  Portions of fewer columns than such a
        // block has too, as long as every block has a compute unit of its own: a wave alone walks its keys a step a trip to the memory
        // (a prompt of 40 tokens, two query heads a key head, 9.1 -> 6.0 us a layer, of 20 tokens 8.3 -> 5.5, of 17 behind 100 8.7 -> 6.4; in
        // a second round of the units the other way round: 64 requests of 9 tokens 5.7 us by single waves, 11.1 by blocks; and up to 32 keys, a wave's one
        // step, there is nothing to share: 24 tokens of five query heads a key head 5.2 and 6.1).
        // Blocks of 128 columns; of 64 (twice as many, the same bits) where the keys are not split and the blocks of 128
        // would be half a compute unit's worth or less, or, under a causal mask over most of the context, where the
        // blocks' walks differ in length, one a compute unit or less.  Measured, 32 query and 8 key/value heads, whole
        // prompts: 512 tokens 17.8 -> 15.1 us, 1,024 tokens (256 blocks) 28.2 -> 24.5, 2,048 tokens (512 blocks) 55.8 -> 69.7
        // (not taken); 16 query heads: 1,024 tokens 25.8 -> 18.2, 2,048 tokens 44.4 -> 36.3; a portion of 512 tokens at a
        // context of 2,048: 42.3 -> 29.7 (36.8 with the keys split in two), with 40 query heads (160 blocks) 43.0 -> 47.9 (not taken).
        const long long tiles128 = (cols + 16 * TILE_NBW * TILE_WAVES - 1) / (16 * TILE_NBW * TILE_WAVES);
        const long long blocks128 = tiles128 * nkv * n_seqs;
        const bool causal_most = 2LL * max_q_len > max_kv_len;
        const bool narrow = g_tiles == 2 || (g_tiles == 1 && splits == 1 &&
                                             blocks128 <= (causal_most ? attn_cus() : attn_cus() / 2));
        const int tile_cols = 16 * (narrow ? 1 : TILE_NBW) * TILE_WAVES;
        const long long tiles = (cols + tile_cols - 1) / tile_cols;
        IA_CHECK(tiles <= 65535, "attention_mfma: %lld tiles of columns in a request (at most 65535)", tiles);
        const dim3 tgrid((unsigned)(nkv * splits * n_seqs), (unsigned)tiles, 1);
        p.pair = 0;
#define ATTN_TILE(FORM)                                                                                                        \
        do {                                                                                                                   \
            if (narrow) attn_tile_kernel<TILE_FITS, 1, FORM><<<tgrid, TILE_GROUPS * TILE_WAVES * IA_WAVE, 0, stream>>>(p);       \
            else attn_tile_kernel<TILE_FITS, TILE_NBW, FORM><<<tgrid, TILE_GROUPS * TILE_WAVES * IA_WAVE, 0, stream>>>(p);       \
        } while (0)
        if (form == FORM_PLAIN) ATTN_TILE(FORM_PLAIN);
        else if (form == FORM_KEEP) ATTN_TILE(FORM_KEEP);
        else ATTN_TILE(FORM_CAP);
#undef ATTN_TILE
    } else {
#define ATTN_WAVES(FORM)                                                       \
        do {                                                                   \
            if (nb == 1) attn_mfma_kernel<1, FORM><<<grid, IA_WAVE, 0, stream>>>(p); \
            else attn_mfma_kernel<2, FORM><<<grid, IA_WAVE, 0, stream>>>(p);   \
        } while (0)
        if (form == FORM_PLAIN) ATTN_WAVES(FORM_PLAIN);
        else if (form == FORM_KEEP) ATTN_WAVES(FORM_KEEP);
        else ATTN_WAVES(FORM_CAP);
#undef ATTN_WAVES
    }
    IA_LAUNCH_CHECK("attention_mfma");
    if (splits > 1) {
        const long long rows = (long long)n_tokens * nq;
        if (rows >= MERGE_ROWS_FROM && splits <= 16)
            attn_merge_rows_kernel<<<(unsigned)((rows + MERGE_ROWS_WAVES - 1) / MERGE_ROWS_WAVES), MERGE_ROWS_WAVES * IA_WAVE,
                                     0, stream>>>((bf16_t*)out, p.part_o, p.part_ml, splits, (size_t)token_begin * nq,
                                                  (size_t)rows, p.sink, p.sinks, nq);
        else
            attn_merge_kernel<<<(unsigned)rows, MERGE_WAVES * IA_WAVE, 0, stream>>>(
                (bf16_t*)out, p.part_o, p.part_ml, splits, (size_t)token_begin * nq, p.sink, p.sinks, nq);
        IA_LAUNCH_CHECK("attention_merge");
    }
    return 0;
}

extern "C" int ia_attention_mfma(void* out, float* workspace, const void* q, const void* k_cache,
                                 const void* v_cache, const int* block_table, const int* cu_tokens,
                                 const int* positions, int n, int seq_begin, int n_seqs, int token_begin,
                                 int n_tokens, int max_q_len, int max_kv_len, int max_pages,
                                 int nq, int nkv, int d, int page_size, int window, float scale,
                                 int splits, int chunk, int sink, int mask_chunk, const float* sinks,
                                 int keep_first, float softcap, hipStream_t stream) {
    return attention_launch(out, workspace, q, k_cache, v_cache, block_table, cu_tokens, positions, n, seq_begin,
                            n_seqs, token_begin, n_tokens, max_q_len, max_kv_len, max_pages, nq, nkv, d, page_size,
                            window, scale, splits, chunk, sink, mask_chunk, sinks, keep_first, softcap, nullptr, stream);
}

// Whether this head size has the fused decode form.
extern "C" int ia_attention_mfma_has_fused(void) { return HD % 64 == 0 ? 1 : 0; }

// Decode steps, one token a request: the per-head norm of q and k (weights may be null: none), the rotation
// by each token's angles (cos, sin [n, rot / 2], the first `rot` features of a head, halves paired; may be null: none) and the
// write of the new key and value at `slots` (may be null: nothing is written and the cache is only read) happen
// inside the attention kernel.  `qkv` [n, row_ld] is the projections' output: query heads at q_off of a row, key heads at k_off,
// value heads at v_off (without `slots` the last two are not used).  `gate` (may be null) points at the first token's gate values,
// rows gate_ld apart, a value a feature of the joined heads or (gate_per_head) a head: the output is times their sigmoid.
extern "C" int ia_attention_mfma_decode_fused(void* out, float* workspace, const void* qkv, void* k_cache,
                                              void* v_cache, const int* block_table, const int* cu_tokens,
                                              const int* positions, const int* slots, const float* q_norm_w,
                                              const float* k_norm_w, const float* cos_t, const float* sin_t,
                                              float eps, int add_one, int row_ld, int q_off, int k_off, int v_off, int rot,
                                              const void* gate, int gate_ld, int gate_per_head, int n, int seq_begin, int n_seqs,
                                              int token_begin, int n_tokens, int max_kv_len, int max_pages,
                                              int nq, int nkv, int d, int page_size, int window, float scale,
                                              int splits, int chunk, int sink, int mask_chunk, int* counters, int n_counters,
                                              hipStream_t stream) {
    IA_CHECK(qkv != nullptr && (cos_t == nullptr) == (sin_t == nullptr) && (k_norm_w == nullptr || q_norm_w != nullptr) &&
             (slots == nullptr || (q_norm_w == nullptr) == (k_norm_w == nullptr)),
             "attention_mfma_decode_fused: qkv is needed; norm weights (where keys are written) and angle tables come in pairs");
    IA_CHECK((((uintptr_t)qkv | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w | (uintptr_t)cos_t | (uintptr_t)sin_t) & 15) == 0,
             "attention_mfma_decode_fused: arrays must be 16-byte aligned");
    IA_CHECK(n_seqs == n_tokens, "attention_mfma_decode_fused: one token a request (%d requests, %d tokens)", n_seqs, n_tokens);
    IA_CHECK(rot >= 0 && rot <= HD && rot % 8 == 0 && (cos_t == nullptr || rot > 0), "attention_mfma_decode_fused: rotation of %d features of "
             "%d (steps of 8)", rot, HD);
    IA_CHECK(row_ld % 4 == 0 && q_off % 4 == 0 && q_off >= 0 && nkv > 0 && q_off + (long long)nq * HD <= row_ld,
             "attention_mfma_decode_fused: %d query heads at %d of rows of %d", nq, q_off, row_ld);
    if (slots == nullptr) {                                  // (the row of a new key is asked for and not used: any row will do)
        k_off = q_off; v_off = 0;
        k_norm_w = q_norm_w;
    }
    IA_CHECK(k_off % 4 == 0 && k_off >= 0 && v_off >= 0 && k_off + (long long)nkv * HD <= row_ld &&
             (slots == nullptr || v_off + (long long)nkv * HDV <= row_ld),
             "attention_mfma_decode_fused: %d key heads at %d and value heads at %d of rows of %d", nkv, k_off, v_off, row_ld);
    IA_CHECK(gate == nullptr || (gate_ld >= (gate_per_head ? nq : nq * HDV) && (gate_per_head || (gate_ld % 4 == 0 && ((uintptr_t)gate & 7) == 0))),
             "attention_mfma_decode_fused: gate values of %d heads in rows %d apart (pieces of four are read at once)", nq, gate_ld);
    const FusedArgs fused = {qkv, q_norm_w, k_norm_w, cos_t, sin_t, slots, eps, add_one, row_ld, q_off, k_off, v_off, rot,
                             gate, gate_ld, gate_per_head, counters, n_counters};
    return attention_launch(out, workspace, nullptr, k_cache, v_cache, block_table, cu_tokens, positions, n, seq_begin,
                            n_seqs, token_begin, n_tokens, 1, max_kv_len, max_pages, nq, nkv, d, page_size,
                            window, scale, splits, chunk, sink, mask_chunk, nullptr, 0, 0.f, &fused, stream);
}
