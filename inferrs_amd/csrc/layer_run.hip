// Decode steps of one to eight rows: a run of whole decoder layers in one kernel, bfloat16, heads of 128.
//
// At one request a layer is five dependent products and attentions whose bytes take a few microseconds and whose launches, first
// bytes and last sums take most of the time.  Here every block of the kernel is one piece of one phase of one layer (q|k|v, attention,
// merge of split keys, output projection, gate|up, down), it asks for its weights or keys as soon as it starts, and only then waits for
// the rows that the phase before leaves: blocks of the phases to come hold their weights in registers while the phases before them
// run, so that the memory streams ahead and a phase costs a hand-over and little else.  us a step at 700 keys, five kernels a layer / this one:
// 28 layers of the 0.6B shape 1 row 910 / 455, 4 rows 939 / 550, 8 rows 999 / 715; 20 of the 1.7B shape 1 row 964 / 594; 16 of the 4B shape
// 1,155 / 860; 10 of the 8B shape 1,108 / 936.  What bounds a small layer (0.6B shape, 14 us): five hand-overs of 1.2 to 1.5 us (a word's way to the
// memory, the watching lane's read of it, the block's reads of its words), 0.7 us for a phase's products and 0.3 for its outputs, 3.5 us for the
// attention; a large one streams its weights at 5.7 TB/s.
//
// Hand-over.  Rows travel between blocks as 64-bit words, 32 bits of data (two bfloat16 values, or one 32-bit one) beside a
// 32-bit tag, written and read as one relaxed 64-bit access of device scope: a word that shows the tag has its data with it, so no
// flag follows the data and no fence is needed.  The tag counts layers over all launches that share the words; a region of words
// is written again a layer later, by blocks that cannot start to write before every reader of the layer before has published
// (each phase needs all of the one before it).  A word would be taken for another's only if it were left by exactly the layer 2^32
// before.  A block that waits lets one lane watch one of its words, another word for every block, and only when that is there do all
// threads ask for theirs: with all threads waiting at the memory a hand-over of 64 blocks took 3.0 us, with one lane 2.0, and
// copies of the words for groups of readers changed nothing.
//
// Order.  A block's piece is not its place in the grid but the number it draws from a counter when it starts: whatever it waits for
// belongs to lower numbers, which blocks that already run have drawn, so the kernel ends however few of its blocks are
// resident and whatever else runs on the GPU.  The counter's upper half holds the tags' base; the block that draws the last number
// sets both for the next launch.  Launches that share a workspace follow each other on one stream.  A draw costs the counter
// 14 ns, which is why blocks have 16 waves.
#include "common.h"
#include "api.h"

#define RUN_HD 128            // head size
#define RUN_WAVES 16
#define RUN_THREADS (RUN_WAVES * IA_WAVE)
#define RUN_LAYERS 32         // layers of a launch at most (their pointers travel as kernel arguments)
#define RUN_PAGE 16           // slots of a cache page
#define RUN_UNIT 512          // inner features that a wave takes with one load a weight row
#define RUN_ROWS 8
#define RUN_HEAD_WORDS 32     // words ahead of the regions: the counter, and the mark of a wait that was given up
#define RUN_PAD 16            // words behind a row in shared memory: the four rows that lanes read side by side begin in other banks
#define RUN_NAN 0x7fc07fc0u

typedef __bf16 run_bf2 __attribute__((ext_vector_type(2)));
typedef short run_s4 __attribute__((ext_vector_type(4)));
typedef __bf16 run_bf8 __attribute__((ext_vector_type(8)));
typedef float run_f4 __attribute__((ext_vector_type(4)));

struct RunLayer {
    const bf16_t *w_qkv, *w_o, *w_gate_up, *w_down;
    const float *norm1, *norm2, *q_norm, *k_norm;
    bf16_t *k_cache, *v_cache;      // [pages, nkv, page, 128] and [pages, nkv, 128, page]
};

struct RunArgs {
    RunLayer layer[RUN_LAYERS];
    bf16_t* x;                      // [rows, width]: the stream, read by the first layer and written by the last
    uint64_t* head;
    uint64_t *qkv, *part, *attn, *mid, *act, *next;     // regions of words, in the order of a layer's phases
    const int *positions, *slots, *block_table;
    const float *cos_t, *sin_t;     // [rows, 64]
    int n_layers, per_layer;
    int b_qkv, b_attn, b_merge, b_o, b_gate_up, b_down;  // blocks of a phase (b_merge 0: keys are not split)
    int s_qkv, s_o, s_gate_up, s_down;                   // log2 of the waves that share a group of weight rows along k
    int width, ff, nq, nkv, max_pages, splits, chunk, max_kv;
    float eps1, eps2, eps_qk, scale_log2;
    int one1, one2, one_qk;         // norms weigh with 1 + w
    int polls;                      // reads of a word after which a wait is given up
    int* given_up;                  // host memory: set where one is
};

__device__ __forceinline__ uint64_t word_load(const uint64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void word_store(uint64_t* p, uint32_t tag, uint32_t data) {
    __hip_atomic_store(p, (uint64_t)tag << 32 | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t word_tag(uint64_t v) { return (uint32_t)(v >> 32); }

// What a block waits for its layer's words with: their tag, and the limit of a wait, which the block reads once, beside its draw (read from the
// arguments at every wait it cost a step of 28 layers 2 us).
struct RunWait { uint32_t tag; int polls; };

// Whether a wait goes on that has `left` reads, the one just made among them: not beyond these, and not once another has been given up.  What is
// waited for in vain counts as no number, so that the launch ends, and the host is told: it reads its word where it has waited for the device
// anyway.
__device__ __forceinline__ bool wait_on(const RunArgs& a, int& left) {
    if (--left <= 0) {
        word_store(a.head + 16, 1, 0);
        __hip_atomic_store(a.given_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return (left & 1023) != 0 || word_load(a.head + 16) == 0;     // (at 0 the mark just set; no way out of its own: the waits' ends stay short)
}

// The data of the words at(0) .. at(N - 1), waited for: asked for together until all are there.  (A thread with fewer words names one of
// them again: loads behind a condition would each be waited for in turn.)
template <int N, typename AT>
__device__ __forceinline__ void words_wait(const RunArgs& a, RunWait wait, AT at, uint32_t (&data)[N]) {
    for (int left = wait.polls;;) {
        uint64_t v[N];
        bool there = true;
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = word_load(at(i));
#pragma unroll
        for (int i = 0; i < N; ++i) {
            there = there && word_tag(v[i]) == wait.tag;
            data[i] = (uint32_t)v[i];
        }
        if (there) return;
        __builtin_amdgcn_s_sleep(1);
        if (!wait_on(a, left)) break;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) data[i] = RUN_NAN;
}

// Held until `at`, one of the words that this block needs, shows the tag: one lane watches, and the others ask once.
__device__ __forceinline__ void watch(const RunArgs& a, const uint64_t* at, RunWait wait) {
    if (threadIdx.x == 0) {
        int left = wait.polls;
        while (word_tag(word_load(at)) != wait.tag) {
            __builtin_amdgcn_s_sleep(2);
            if (!wait_on(a, left)) break;
        }
    }
    __syncthreads();
}

__device__ __forceinline__ float lo_f32(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float hi_f32(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(run_bf2, a), __builtin_bit_cast(run_bf2, b), c, false);
}

// Sums over the wave of 4 R values a lane: row q of 16 lanes ends with those of v[q R] .. v[q R + R - 1], in v[0] .. v[R - 1].
template <int R>
__device__ __forceinline__ void sum_lanes(float* v) {
#pragma unroll
    for (int i = 0; i < 2 * R; ++i) {
        auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 2 * R]), false, false);
        v[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
        auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + R]), false, false);
        v[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
        v[i] += wave_lane<0xb1>(v[i]);                      // lane ^ 1
        v[i] += wave_lane<0x4e>(v[i]);                      // lane ^ 2
        v[i] += wave_lane<0x141>(v[i]);                     // the other four of eight
        v[i] += wave_lane<0x140>(v[i]);                     // the other eight of sixteen
    }
}

// The position of a row's newest token, which is the count of its cached keys, inside the bound that the launch is laid out for: beyond it a row
// would wait for shares of its keys that no block forms, and read pages behind its table's row.
__device__ __forceinline__ int run_last(const RunArgs& a, int row) { return min(max(a.positions[row], 0), a.max_kv - 1); }

// Features 2 i and 2 i + 1 of the attention of `head` (counted over all rows), from the shares of its row's keys.
__device__ __forceinline__ uint32_t run_merged(const RunArgs& a, int head, int i, int shares, RunWait wait) {
    constexpr int HD = RUN_HD, AT_ONCE = 2;
    const uint64_t* from = a.part + (size_t)head * a.splits * (HD + 2);
    float top = -INFINITY, total = 0.f, o0 = 0.f, o1 = 0.f;
    for (int s0 = 0; s0 < shares; s0 += AT_ONCE) {
        uint32_t d[AT_ONCE * 4];
        words_wait<AT_ONCE * 4>(a, wait, [&](int n) __attribute__((always_inline)) {
            const int q = n & 3;
            return from + (s0 + (n >> 2) < shares ? s0 + (n >> 2) : shares - 1) * (HD + 2) + (q < 2 ? HD + q : 2 * i + q - 2);
        }, d);
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            if (s0 + j < shares) {
                const float mj = __uint_as_float(d[4 * j]), lj = __uint_as_float(d[4 * j + 1]), x0 = __uint_as_float(d[4 * j + 2]), x1 = __uint_as_float(d[4 * j + 3]);
                const float m_new = fmaxf(top, mj);
                const float back = top == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(top - m_new), wt = mj == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mj - m_new);
                o0 = fmaf(x0, wt, o0 * back);
                o1 = fmaf(x1, wt, o1 * back);
                total = fmaf(lj, wt, total * back);
                top = m_new;
            }
        }
    }
    const float inv = 1.0f / total;
    return pack_bf16x2(o0 * inv, o1 * inv);
}

// Rows r0 .. r0 + R - 1 of the stream into shared memory, times the norm's weights and rounded, and every wave's sums of their squares;
// Q words a thread and row.
template <int R, int Q>
__device__ __forceinline__ void run_normed_rows(const RunArgs& a, int r0, uint32_t* xs, float* squares, const float* norm, float one, const uint64_t* in, const uint64_t* first, RunWait wait, bool plain) {
    const int tid = threadIdx.x, pairs = a.width >> 1;
    float2 weight[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int j = tid + q * RUN_THREADS;
        weight[q] = *(const float2*)(norm + 2 * (j < pairs ? j : pairs - 1));
    }
    auto place = [&](int i) __attribute__((always_inline)) {
        const int j = tid + i % Q * RUN_THREADS;
        return (r0 + i / Q) * pairs + (j < pairs ? j : pairs - 1);
    };
    uint32_t d[R * Q];
    if (plain) {
#pragma unroll
        for (int i = 0; i < R * Q; ++i) d[i] = ((const uint32_t*)a.x)[place(i)];
    } else {
        if (first != nullptr) watch(a, first, wait);    // (behind the loads of the weights)
        words_wait<R * Q>(a, wait, [&](int i) __attribute__((always_inline)) { return in + place(i); }, d);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int j = tid + q * RUN_THREADS;
            if (j < pairs) {
                const float x0 = lo_f32(d[r * Q + q]), x1 = hi_f32(d[r * Q + q]);
                ss += x0 * x0 + x1 * x1;
                xs[(r0 + r) * (pairs + RUN_PAD) + j] = pack_bf16x2(x0 * (weight[q].x + one), x1 * (weight[q].y + one));
            }
        }
        ss = wave_sum(ss);
        if ((tid & (IA_WAVE - 1)) == 0) squares[(r0 + r) * RUN_WAVES + tid / IA_WAVE] = ss;
    }
}

template <int R>
__device__ __forceinline__ void run_normed_rows(const RunArgs& a, int r0, uint32_t* xs, float* squares, const float* norm, float one, const uint64_t* in, const uint64_t* first, RunWait wait, bool plain) {
    if (a.width <= 2 * RUN_THREADS) run_normed_rows<R, 1>(a, r0, xs, squares, norm, one, in, first, wait, plain);
    else if (a.width <= 4 * RUN_THREADS) run_normed_rows<R, 2>(a, r0, xs, squares, norm, one, in, first, wait, plain);
    else run_normed_rows<R, 3>(a, r0, xs, squares, norm, one, in, first, wait, plain);
}

enum { RUN_QKV, RUN_O, RUN_GATE_UP, RUN_DOWN };

// A product's piece: 16 >> ksl groups of four weight rows (gate|up: two gate rows and the two up rows beside them), a group's inner
// features shared out among 1 << ksl waves, 512 a step of four loads; two chunks of two steps a wave are asked for before the wait for
// the step's rows.  Two forms, by how a lane's 16 bytes are multiplied.  DOT: a load brings 1 KiB of one weight row, and pairs go through the vector
// unit's dot products, for every row of the step anew.  Otherwise a load brings 256 bytes of each of the four weight rows, and a lane's 16 bytes
// are two operands of v_mfma_f32_4x4x4_16b_bf16: sixteen blocks of four weight rows, four of the step's rows and four inner features, the blocks
// summed at the end; up to four rows cost what one costs, but neighbouring lanes read four rows of memory.  (us a layer, DOT / not, 700
// keys: 0.6B shape 1 row 14.0 / 14.4, 2 rows 17.2 / 15.8, 4 rows 22.5 / 17.3; 8B shape 1 row 68 / 75, 2 rows 73 / 77.)
template <int R, bool DOT>
__device__ __forceinline__ void run_product(const RunArgs& a, const RunLayer& L, char* mem, int kind, int item, int layer, RunWait wait) {
    constexpr int C = (R + 3) / 4;                          // groups of four rows
    const int tid = threadIdx.x, lane = tid & (IA_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / IA_WAVE);
    const int heads_width = a.nq * RUN_HD;
    const bf16_t* w = kind == RUN_QKV ? L.w_qkv : kind == RUN_O ? L.w_o : kind == RUN_GATE_UP ? L.w_gate_up : L.w_down;
    const int K = kind == RUN_O ? heads_width : kind == RUN_DOWN ? a.ff : a.width;
    const int ksl = kind == RUN_QKV ? a.s_qkv : kind == RUN_O ? a.s_o : kind == RUN_GATE_UP ? a.s_gate_up : a.s_down;
    const int groups = RUN_WAVES >> ksl, g = wave >> ksl, s = wave & ((1 << ksl) - 1);
    const int f = lane & 3;                                 // the lane's weight row of the group, and its row of the step
    const int row0 = (item * groups + g) * (kind == RUN_GATE_UP ? 2 : 4);     // the group's rows are row0, row0 + 1, row0 + skip and row0 + skip + 1
    const int skip = kind == RUN_GATE_UP ? a.ff : 2;
    const size_t row_bytes = (size_t)K * 2;
    const char* w_lane = (const char*)w + (size_t)row0 * row_bytes + s * (RUN_UNIT * 2)
                         + (DOT ? (size_t)lane * 16 : ((f & 1) + (size_t)(f >> 1) * skip) * row_bytes + (lane >> 2) * 16);
    const int steps = ((K / RUN_UNIT - s - 1) >> ksl) + 1, chunks = (steps + 1) >> 1;
    uint4 wa[2][4], wb[2][4];
    auto load = [&](uint4 (&to)[2][4], int c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (2 * c + j < steps) {
                const char* from = w_lane + ((size_t)(2 * c + j) << ksl) * (RUN_UNIT * 2);
                if constexpr (DOT) {
                    to[j][0] = *(const uint4*)from;
                    to[j][1] = *(const uint4*)(from + row_bytes);
                    to[j][2] = *(const uint4*)(from + skip * row_bytes);
                    to[j][3] = *(const uint4*)(from + (skip + 1) * row_bytes);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) to[j][i] = *(const uint4*)(from + i * 256);
                }
            }
        }
    };
    load(wa, 0);
    if (chunks > 1) load(wb, 1);

    // ---- the rows ---------------------------------------------------------------------------------------
    const int pairs = K >> 1, row_words = pairs + RUN_PAD;
    uint32_t* xs = (uint32_t*)mem;                          // [R][row_words]: pairs
    float* sums = (float*)(xs + R * row_words);             // [waves][4][R]
    float* squares = sums + RUN_WAVES * 4 * R;            // [R][waves]
    const bool normed = kind == RUN_QKV || kind == RUN_GATE_UP;
    const bool plain = kind == RUN_QKV && layer == 0;     // the stream as the kernel before this one left it
    if (normed) {
        const float* norm = kind == RUN_QKV ? L.norm1 : L.norm2;
        const float one = (kind == RUN_QKV ? a.one1 : a.one2) ? 1.0f : 0.0f;
        const uint64_t* in = kind == RUN_QKV ? a.next : a.mid;
        run_normed_rows<(R < 4 ? R : 4)>(a, 0, xs, squares, norm, one, in, in + (item * 37) % (R * pairs), wait, plain);
        if constexpr (R > 4) run_normed_rows<R - 4>(a, 4, xs, squares, norm, one, in, nullptr, wait, plain);
    } else {
        const uint64_t* in = kind == RUN_O ? a.attn : a.act;
        const int n = R * pairs;
        const uint32_t per_row = 0xffffffffu / (uint32_t)pairs + 1;      // (j / pairs by a product: exact for j * pairs below 2^32)
        auto put = [&](int j, uint32_t d) __attribute__((always_inline)) { xs[R == 1 ? j : j + RUN_PAD * (int)__umulhi((uint32_t)j, per_row)] = d; };
        const bool merges = kind == RUN_O && a.splits > 1 && a.b_merge == 0;
        int shares[R];                                      // of the rows' keys
#pragma unroll
        for (int r = 0; r < R; ++r) shares[r] = merges ? run_last(a, r) / a.chunk + 1 : 0;
        watch(a, merges ? a.part + (size_t)(item % (R * a.nq)) * a.splits * (RUN_HD + 2) : in + (item * 37) % n, wait);
        if (merges) {
            // the shares of every head's keys come together here: few of them, and few blocks that would read them all
            for (int j = tid; j < n; j += RUN_THREADS) {
                int of = shares[0];
#pragma unroll
                for (int r = 1; r < R; ++r) of = j >= r * pairs ? shares[r] : of;
                put(j, run_merged(a, j >> 6, j & 63, of, wait));
            }
        } else {
            constexpr int Q = 4;
            for (int j0 = tid; j0 < n; j0 += Q * RUN_THREADS) {
                uint32_t d[Q];
                words_wait<Q>(a, wait, [&](int q) __attribute__((always_inline)) { return in + (j0 + q * RUN_THREADS < n ? j0 + q * RUN_THREADS : j0); }, d);
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    if (j0 + q * RUN_THREADS < n) put(j0 + q * RUN_THREADS, d[q]);
            }
        }
    }
    // What the outputs' threads need beside the sums comes while the products are formed: the stream's old values (there before this block's rows
    // were) and the norm's factor.
    const int out_log = (kind == RUN_GATE_UP ? 4 : 5) - ksl;                  // log2 of the block's pairs of outputs a row
    const int r = tid >> out_log, p = tid & ((1 << out_log) - 1);
    const int pair = (item << out_log) + p;                                     // of the row's outputs
    const int at = r * (a.width >> 1) + pair;                                   // (o and down: the outputs are the stream's)
    const uint64_t* old_at = kind == RUN_O ? a.next + at : a.mid + at;
    uint32_t was[1] = {0};
    if (!normed && r < R) {
        if (kind == RUN_O && layer == 0) was[0] = ((const uint32_t*)a.x)[at];
        else words_wait<1>(a, wait, [&](int) { return old_at; }, was);
    }
    __syncthreads();
    float scale = 1.f;
    if (normed && r < R) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < RUN_WAVES; ++i) ss += squares[r * RUN_WAVES + i];
        scale = 1.0f / sqrtf(ss / (float)K + (kind == RUN_QKV ? a.eps1 : a.eps2));
    }

    // ---- the products -----------------------------------------------------------------------------------
    run_f4 acc[C][2] = {};                                // (two sums of alternating operands: the next product need not wait for the last)
    float dots[4 * R] = {};
    const char* x_lane[C];
#pragma unroll
    for (int cg = 0; cg < C; ++cg)
        x_lane[cg] = mem + s * (RUN_UNIT * 2) + (DOT ? lane * 16 : (4 * cg + f < R ? 4 * cg + f : 0) * row_words * 4 + (lane >> 2) * 16);
    auto multiply = [&](const uint4 (&of)[2][4], int c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (2 * c + j < steps) {
                const int at = ((2 * c + j) << ksl) * (RUN_UNIT * 2);
                if constexpr (DOT) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const uint4 x = *(const uint4*)(x_lane[0] + at + r * row_words * 4);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float t = dots[i * R + r];
                            t = dot2(of[j][i].x, x.x, t);
                            t = dot2(of[j][i].y, x.y, t);
                            t = dot2(of[j][i].z, x.z, t);
                            dots[i * R + r] = dot2(of[j][i].w, x.w, t);
                        }
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint4 wi = of[j][i];
#pragma unroll
                        for (int cg = 0; cg < C; ++cg) {
                            const uint4 xi = *(const uint4*)(x_lane[cg] + at + i * 256);
                            acc[cg][0] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(run_s4, make_uint2(wi.x, wi.y)), __builtin_bit_cast(run_s4, make_uint2(xi.x, xi.y)), acc[cg][0], 0, 0, 0);
                            acc[cg][1] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(run_s4, make_uint2(wi.z, wi.w)), __builtin_bit_cast(run_s4, make_uint2(xi.z, xi.w)), acc[cg][1], 0, 0, 0);
                        }
                    }
                }
            }
        }
    };
    for (int c = 0; c < chunks; c += 2) {
        multiply(wa, c);
        if (c + 2 < chunks) load(wa, c + 2);
        if (c + 1 < chunks) {
            multiply(wb, c + 1);
            if (c + 3 < chunks) load(wb, c + 3);
        }
    }
    if constexpr (DOT) {
        sum_lanes<R>(dots);
        if ((lane & 15) == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) sums[(wave * 4 + (lane >> 4)) * R + r] = dots[r];
        }
    } else {
        // Lane 4 b + j holds block b's sums of weight rows 0 .. 3 with row j of the step: over the blocks, row q of 16 lanes ends with weight row q.
#pragma unroll
        for (int cg = 0; cg < C; ++cg) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = acc[cg][0][i] + acc[cg][1][i];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 2]), false, false);
                v[i] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
            }
            auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
            float u = __uint_as_float(t[0]) + __uint_as_float(t[1]);
            u += wave_lane<0x128>(u);                           // turned by 8
            u += wave_lane<0x124>(u);                           // turned by 4
            if ((lane & 15) < 4 && 4 * cg + f < R) sums[(wave * 4 + (lane >> 4)) * R + 4 * cg + f] = u;
        }
    }
    __syncthreads();

    // ---- a thread a pair of outputs: the waves that shared a group, the norm, the activation or the stream ----------
    if (r >= R) return;
    auto total = [&](int group, int f) __attribute__((always_inline)) {
        float t = 0.f;
        for (int i = 0; i < 1 << ksl; ++i) t += sums[(((group << ksl) + i) * 4 + f) * R + r];
        return t;
    };
    if (kind == RUN_GATE_UP) {
        const float g0 = total(p, 0) * scale, g1 = total(p, 1) * scale, u0 = total(p, 2) * scale, u1 = total(p, 3) * scale;
        word_store(a.act + r * (a.ff >> 1) + pair, wait.tag, pack_bf16x2(gate_act(g0, IA_ACT_SILU) * u0, gate_act(g1, IA_ACT_SILU) * u1));
        return;
    }
    const float v0 = total(p >> 1, (p & 1) * 2) * scale, v1 = total(p >> 1, (p & 1) * 2 + 1) * scale;
    if (kind == RUN_QKV) {
        word_store(a.qkv + r * ((a.nq + 2 * a.nkv) * (RUN_HD / 2)) + pair, wait.tag, pack_bf16x2(v0, v1));
        return;
    }
    const uint32_t sum = pack_bf16x2(lo_f32(was[0]) + v0, hi_f32(was[0]) + v1);
    if (kind == RUN_O) word_store(a.mid + at, wait.tag, sum);
    else if (layer + 1 < a.n_layers) word_store(a.next + at, wait.tag + 1, sum);
    else ((uint32_t*)a.x)[at] = sum;
}

// Attention of one row's query heads of a key/value head over one share of its keys: steps of 32 cached keys, a wave every sixteenth.  The
// operands' layouts are those of the decode kernel in attention_mfma.hip: S^T = K Q^T and O^T = V^T P^T, key k0 + 8 G + 4 t + i in
// row 4 G + i of tile t.  The first step's keys and values are asked for before the wait; the row's heads are normed and turned by a
// wave each, once for the block; the new key, which is in no page yet, is a step of its own, of a wave that has none where there is one.
__device__ __forceinline__ void run_attention(const RunArgs& a, const RunLayer& L, char* mem, int item, RunWait wait) {
    constexpr int HD = RUN_HD, KS = HD / 32, DB = HD / 16;
    const int tid = threadIdx.x, lane = tid & (IA_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / IA_WAVE);
    const int r = lane & 15, G = lane >> 4;
    const int g = a.nq / a.nkv;
    const int split = item % a.splits, of = item / a.splits, kvh = of % a.nkv, row = of / a.nkv;
    const int last = run_last(a, row);
    const int lo = split * a.chunk;
    if (lo > last) return;
    const bool has_new = last < lo + a.chunk;
    const int hi = has_new ? last : lo + a.chunk;
    const int steps = (hi - lo + 31) >> 5;
    const int* bt = a.block_table + (size_t)row * a.max_pages;
    constexpr int page = RUN_PAGE;
    const int last_page = last / page;
    const bool k_second = r >= 8, v_second = G >= 2;
    const uint32_t k_lane = (uint32_t)((((8 * (r >> 2) + (r & 3)) & 15) * HD + G * 8) * 2);
    const uint32_t v_lane = (uint32_t)((r * page + 8 * (G & 1)) * 2);
    uint4 k[2][KS], v[DB];
    auto pages = [&](int k0, bool second) __attribute__((always_inline)) {
        int ia = k0 / page, ib = ia + 1;
        ia = ia < last_page ? ia : last_page;               // (slots past the request's length are read like others as long as their page is its own)
        ib = ib < last_page ? ib : last_page;
        return ((second ? (size_t)bt[ib] : (size_t)bt[ia]) * a.nkv + kvh) * (page * HD * 2);
    };
    auto load_keys = [&](int k0) __attribute__((always_inline)) {
        const char* from = (const char*)L.k_cache + pages(k0, k_second) + k_lane;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) k[t][ks] = *(const uint4*)(from + t * (4 * HD * 2) + ks * 64);
    };
    auto load_values = [&](int k0) __attribute__((always_inline)) {
        const char* from = (const char*)L.v_cache + pages(k0, v_second) + v_lane;
#pragma unroll
        for (int db = 0; db < DB; ++db) v[db] = *(const uint4*)(from + db * 32 * page);
    };
    if (wave < steps) {
        load_keys(lo + wave * 32);
        load_values(lo + wave * 32);
    }
    // what the rows need: query heads are waves 0 .. g - 1, the new key wave g, its value wave g + 1
    const int used = g + (has_new ? 2 : 0);
    char* rows = mem;                                       // [g + 2][128], 16-byte pieces exchanged by the row's number
    {
        float2 cs = make_float2(1.f, 1.f), sn = make_float2(0.f, 0.f), nw = make_float2(1.f, 1.f);
        if (wave <= g) {
            cs = *(const float2*)(a.cos_t + (size_t)row * (HD / 2) + 2 * (lane & 31));
            sn = *(const float2*)(a.sin_t + (size_t)row * (HD / 2) + 2 * (lane & 31));
            nw = *(const float2*)((wave < g ? L.q_norm : L.k_norm) + 2 * lane);
            if (a.one_qk) { nw.x += 1.0f; nw.y += 1.0f; }
        }
        watch(a, a.qkv + ((size_t)row * (a.nq + 2 * a.nkv) + kvh * g) * (HD / 2), wait);
        if (wave < used) {
            const int head = wave < g ? kvh * g + wave : wave == g ? a.nq + kvh : a.nq + a.nkv + kvh;
            const uint64_t* at = a.qkv + ((size_t)row * (a.nq + 2 * a.nkv) + head) * (HD / 2) + lane;
            uint32_t one[1];
            words_wait<1>(a, wait, [&](int) { return at; }, one);
            uint32_t d = one[0];
            if (wave <= g) {                                // (features 2 lane and 2 lane + 1; what they are turned with is 32 lanes away)
                float x = lo_f32(d), y = hi_f32(d);
                const float scale = 1.0f / sqrtf(wave_sum(x * x + y * y) / (float)HD + a.eps_qk);
                x = scale * x * nw.x;
                y = scale * y * nw.y;
                auto sx = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
                auto sy = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
                const float x_lo = __uint_as_float(sx[0]), x_hi = __uint_as_float(sx[1]), y_lo = __uint_as_float(sy[0]), y_hi = __uint_as_float(sy[1]);
                x = lane < 32 ? x_lo * cs.x - x_hi * sn.x : x_lo * sn.x + x_hi * cs.x;
                y = lane < 32 ? y_lo * cs.y - y_hi * sn.y : y_lo * sn.y + y_hi * cs.y;
                d = pack_bf16x2(x, y);
            }
            *(uint32_t*)(rows + wave * (HD * 2) + ((lane >> 2) ^ (wave & 7)) * 16 + (lane & 3) * 4) = d;
        }
    }
    __syncthreads();
    auto piece = [&](int t, int i) __attribute__((always_inline)) { return *(const uint4*)(rows + t * (HD * 2) + (i ^ (t & 7)) * 16); };
    const int column = r < g ? r : g - 1;

    run_f4 acc[DB];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = (run_f4){0.f, 0.f, 0.f, 0.f};
    auto step = [&](int k0, bool first) __attribute__((always_inline)) {
        run_f4 s4[2] = {};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const uint4 q = piece(column, ks * 4 + G);
#pragma unroll
            for (int t = 0; t < 2; ++t)
                s4[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(run_bf8, k[t][ks]), __builtin_bit_cast(run_bf8, q), s4[t], 0, 0, 0);
        }
        if (!first) load_values(k0);                        // (not beside its keys: the registers of a wave are 128)
        if (k0 + 32 > hi) {                                 // slots behind the cached keys hold anything at all: their values count as zeros
            const int first_bad = hi - k0 - 8 * G;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                uint32_t w[4] = {v[db].x, v[db].y, v[db].z, v[db].w};
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j >= first_bad) w[j >> 1] &= (j & 1) ? 0x0000ffffu : 0xffff0000u;
                v[db] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
        float sc[8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[4 * t + i] = k0 + 8 * G + 4 * t + i < hi ? s4[t][i] : -INFINITY;
        float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
        {   // over the four lanes of a column
            auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
            auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
        }
        const float m_new = fmaxf(m, mx * a.scale_log2);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);
        float pr[8], psum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            pr[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j], a.scale_log2, -m_use));
            psum += pr[j];
        }
        l = first ? psum : l * alpha + psum;
        m = m_new;
        uint4 pb;
        pb.x = pack_bf16x2(pr[0], pr[1]);
        pb.y = pack_bf16x2(pr[2], pr[3]);
        pb.z = pack_bf16x2(pr[4], pr[5]);
        pb.w = pack_bf16x2(pr[6], pr[7]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (!first) acc[db] *= alpha;
            acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(run_bf8, v[db]), __builtin_bit_cast(run_bf8, pb), acc[db], 0, 0, 0);
        }
    };
    if (wave < steps) step(lo + wave * 32, true);
    for (int st = wave + RUN_WAVES; st < steps; st += RUN_WAVES) {
        load_keys(lo + st * 32);
        step(lo + st * 32, false);
    }
    const int newest = steps < RUN_WAVES ? steps : RUN_WAVES - 1;       // the wave that takes the new key
    if (has_new && wave == newest) {
        run_f4 s4 = {};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)                     // (the same key in all rows of the operand: every lane gets its column's score)
            s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(run_bf8, piece(g, ks * 4 + G)), __builtin_bit_cast(run_bf8, piece(column, ks * 4 + G)), s4, 0, 0, 0);
        const float s = s4[0] * a.scale_log2;
        const float m_new = fmaxf(m, s);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use), p = __builtin_amdgcn_exp2f(s - m_use);
        l = l * alpha + (G == 0 ? p : 0.f);
        m = m_new;
#pragma unroll
        for (int db = 0; db < DB; ++db) {                   // features 16 db + 4 G + i
            const int f = 16 * db + 4 * G;
            const uint2 d = *(const uint2*)(rows + (g + 1) * (HD * 2) + ((f >> 3) ^ ((g + 1) & 7)) * 16 + (f & 4) * 2);
            acc[db][0] = fmaf(lo_f32(d.x), p, acc[db][0] * alpha);
            acc[db][1] = fmaf(hi_f32(d.x), p, acc[db][1] * alpha);
            acc[db][2] = fmaf(lo_f32(d.y), p, acc[db][2] * alpha);
            acc[db][3] = fmaf(hi_f32(d.y), p, acc[db][3] * alpha);
        }
    }
    {
        auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(l), __float_as_uint(l), false, false);
        l = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
        auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
        l = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
    }

    // ---- the waves add up: a wave a column, a lane a pair of features; lane w first weighs wave w's results ----------
    constexpr int LD = HD + 4;                              // (floats of a column: neighbours begin in other banks)
    const int waves = steps + (has_new ? 1 : 0) < RUN_WAVES ? steps + (has_new ? 1 : 0) : RUN_WAVES;
    float2* tops = (float2*)(mem + (g + 2) * (HD * 2));     // [16 columns][waves]: maximum and sum
    float* outs = (float*)(tops + 16 * RUN_WAVES);        // [waves][8 columns][LD]
    if (G == 0) tops[r * RUN_WAVES + wave] = make_float2(m, l);
    if (wave < waves && r < g) {
        float* o = outs + (wave * 8 + r) * LD + 4 * G;
#pragma unroll
        for (int db = 0; db < DB; ++db) *(run_f4*)(o + 16 * db) = acc[db];
    }
    __syncthreads();
    if (wave < g) {
        const int col = wave, i = lane;
        const float2 ml = tops[col * RUN_WAVES + r];
        float2 o[RUN_WAVES];                              // (all asked for together)
#pragma unroll
        for (int w = 0; w < RUN_WAVES; ++w) o[w] = *(const float2*)(outs + (w * 8 + col) * LD + 2 * i);
        float top = ml.x;
        top = fmaxf(top, wave_lane<0xb1>(top));
        top = fmaxf(top, wave_lane<0x4e>(top));
        top = fmaxf(top, wave_lane<0x141>(top));
        top = fmaxf(top, wave_lane<0x140>(top));
        const float weight = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - top);
        float total = ml.y * weight;
        total += wave_lane<0xb1>(total);
        total += wave_lane<0x4e>(total);
        total += wave_lane<0x141>(total);
        total += wave_lane<0x140>(total);
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int w = 0; w < RUN_WAVES; ++w) {
            if (w < waves) {                                // (behind the last wave's results lies anything at all)
                const float of_w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), w));
                o0 = fmaf(o[w].x, of_w, o0);
                o1 = fmaf(o[w].y, of_w, o1);
            }
        }
        const size_t head = (size_t)row * a.nq + kvh * g + col;
        if (a.splits == 1) {
            const float inv = 1.0f / total;
            word_store(a.attn + head * (HD / 2) + i, wait.tag, pack_bf16x2(o0 * inv, o1 * inv));
        } else {
            uint64_t* to = a.part + (head * a.splits + split) * (HD + 2);
            word_store(to + 2 * i, wait.tag, __float_as_uint(o0));
            word_store(to + 2 * i + 1, wait.tag, __float_as_uint(o1));
            if (i < 2) word_store(to + HD + i, wait.tag, __float_as_uint(i == 0 ? top : total));
        }
    }
    // the new key and value, for the steps to come
    if (has_new && (wave == g || wave == g + 1)) {
        const int slot = a.slots[row], in_page = slot & (RUN_PAGE - 1);
        const size_t at = (size_t)(slot / RUN_PAGE) * a.nkv + kvh;
        const uint32_t d = *(const uint32_t*)(rows + wave * (HD * 2) + ((lane >> 2) ^ (wave & 7)) * 16 + (lane & 3) * 4);
        if (wave == g) {
            ((uint32_t*)(L.k_cache + (at * page + in_page) * HD))[lane] = d;
        } else {
            bf16_t* to = L.v_cache + (at * HD + 2 * lane) * page + in_page;
            to[0].bits = (uint16_t)d;
            to[page].bits = (uint16_t)(d >> 16);
        }
    }
}

// The shares of a row's keys come together: one key/value head's query heads a block, a thread a pair of features.
__device__ __forceinline__ void run_merge(const RunArgs& a, int item, RunWait wait) {
    const int tid = threadIdx.x, g = a.nq / a.nkv;
    const int shares = run_last(a, item / a.nkv) / a.chunk + 1;
    watch(a, a.part + ((size_t)(item / a.nkv) * a.nq + (item % a.nkv) * g) * a.splits * (RUN_HD + 2), wait);
    if (tid >= g * (RUN_HD / 2)) return;
    const int head = (item / a.nkv) * a.nq + (item % a.nkv) * g + tid / (RUN_HD / 2), i = tid & (RUN_HD / 2 - 1);
    word_store(a.attn + (size_t)head * (RUN_HD / 2) + i, wait.tag, run_merged(a, head, i, shares, wait));
}

template <int R, bool DOT>
__global__ __launch_bounds__(RUN_THREADS) void layer_run_kernel(const RunArgs a) {
    extern __shared__ __align__(16) char run_mem[];
    __shared__ uint64_t s_draw;
    if (threadIdx.x == 0) s_draw = __hip_atomic_fetch_add(a.head, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int polls = a.polls;
    asm volatile("" : "+s"(polls));                         // (here, and not where it is used)
    __syncthreads();
    const uint64_t drawn = s_draw;
    const uint32_t number = __builtin_amdgcn_readfirstlane((uint32_t)drawn), base = __builtin_amdgcn_readfirstlane((uint32_t)(drawn >> 32));
    if (number == (uint32_t)a.per_layer * a.n_layers - 1 && threadIdx.x == 0)
        __hip_atomic_store(a.head, (uint64_t)(base + a.n_layers) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (number == 0 && threadIdx.x == 0) __hip_atomic_store(a.head + 16, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int layer = number / (uint32_t)a.per_layer;
    int item = number - layer * a.per_layer;
    const RunWait wait = {base + layer + 1, polls};
    const RunLayer& L = a.layer[layer];
    int kind;
    if (item < a.b_qkv) kind = RUN_QKV;
    else if ((item -= a.b_qkv) < a.b_attn) { run_attention(a, L, run_mem, item, wait); return; }
    else if ((item -= a.b_attn) < a.b_merge) { run_merge(a, item, wait); return; }
    else if ((item -= a.b_merge) < a.b_o) kind = RUN_O;
    else if ((item -= a.b_o) < a.b_gate_up) kind = RUN_GATE_UP;
    else { item -= a.b_gate_up; kind = RUN_DOWN; }
    run_product<R, DOT>(a, L, run_mem, kind, item, layer, wait);
}

// ---- host -----------------------------------------------------------------------------------------------

// log2 of the waves that share a group of weight rows: as many as leave a wave `least` loads a weight row.
static int run_waves_log2(int inner, int least) {
    int s = 0;
    while (s < 4 && inner / RUN_UNIT >> (s + 1) >= least) ++s;
    return s;
}

extern "C" long long ia_layer_run_words(int rows, int width, int ff, int nq, int nkv, int splits) {
    return RUN_HEAD_WORDS + (long long)rows * ((nq + 2 * nkv) * (RUN_HD / 2) + (splits > 1 ? (long long)nq * splits * (RUN_HD + 2) : 0)
                                                 + nq * (RUN_HD / 2) + width + ff / 2);
}

extern "C" int ia_layer_run_layers(void) { return RUN_LAYERS; }

extern "C" int ia_layer_run(void* x, const void* layers, int n_layers, long long* words, long long n_words, int* given_up, int polls,
                            const int* positions, const int* slots, const int* block_table, const float* cos_t, const float* sin_t, int rows,
                            int width, int ff, int nq, int nkv, int page_size, int max_pages, int max_kv_len, int splits, int chunk, float eps1,
                            float eps2, float eps_qk, int one1, int one2, int one_qk, float scale, hipStream_t stream) {
    IA_CHECK(rows >= 1 && rows <= RUN_ROWS && n_layers >= 1 && n_layers <= RUN_LAYERS, "layer_run: %d rows, %d layers", rows, n_layers);
    IA_CHECK(width > 0 && width % RUN_UNIT == 0 && width <= 6144 && ff > 0 && ff % RUN_UNIT == 0 && nkv > 0 && nq % nkv == 0 && nq % 4 == 0
                 && nq / nkv <= 8 && (nq + 2 * nkv) % 2 == 0,
             "layer_run: width %d, feed-forward %d, %d and %d heads", width, ff, nq, nkv);
    IA_CHECK(page_size == RUN_PAGE && max_pages >= 1 && max_kv_len >= 1 && max_kv_len <= (long long)max_pages * RUN_PAGE,
             "layer_run: %d keys in %d pages of %d", max_kv_len, max_pages, page_size);
    IA_CHECK(splits >= 1 && chunk >= 32 && chunk % 32 == 0 && (long long)splits * chunk >= max_kv_len
                 && n_words >= ia_layer_run_words(rows, width, ff, nq, nkv, splits),
             "layer_run: %d shares of %d keys for %d keys, %lld words", splits, chunk, max_kv_len, n_words);
    IA_CHECK(given_up != nullptr && polls >= 1, "layer_run: a wait ends after %d reads, and says so in host memory", polls);
    RunArgs a = {};
    const void* const* from = (const void* const*)layers;
    for (int i = 0; i < n_layers; ++i, from += 10) {
        RunLayer& L = a.layer[i];
        L.w_qkv = (const bf16_t*)from[0]; L.w_o = (const bf16_t*)from[1]; L.w_gate_up = (const bf16_t*)from[2]; L.w_down = (const bf16_t*)from[3];
        L.norm1 = (const float*)from[4]; L.norm2 = (const float*)from[5]; L.q_norm = (const float*)from[6]; L.k_norm = (const float*)from[7];
        L.k_cache = (bf16_t*)from[8]; L.v_cache = (bf16_t*)from[9];
        uintptr_t wide = 0, pairs = 0;                      // what is read 16 bytes at a time, and what 8
        for (int j = 0; j < 10; ++j) (j >= 4 && j < 8 ? pairs : wide) |= (uintptr_t)from[j];
        IA_CHECK(wide % 16 == 0 && pairs % 8 == 0, "layer_run: layer %d: weights and caches must be 16-byte aligned, the norms' weights 8-byte", i);
    }
    IA_CHECK(((uintptr_t)x & 3) == 0 && (((uintptr_t)cos_t | (uintptr_t)sin_t | (uintptr_t)words) & 7) == 0,
             "layer_run: rows must be 4-byte aligned, angles and words 8-byte");
    a.x = (bf16_t*)x;
    a.head = (uint64_t*)words;
    a.given_up = given_up; a.polls = polls;
    a.qkv = a.head + RUN_HEAD_WORDS;
    a.part = a.qkv + (size_t)rows * (nq + 2 * nkv) * (RUN_HD / 2);
    a.attn = a.part + (splits > 1 ? (size_t)rows * nq * splits * (RUN_HD + 2) : 0);
    a.mid = a.attn + (size_t)rows * nq * (RUN_HD / 2);
    a.next = a.mid + (size_t)rows * (width / 2);
    a.act = a.next + (size_t)rows * (width / 2);
    a.positions = positions; a.slots = slots; a.block_table = block_table; a.cos_t = cos_t; a.sin_t = sin_t;
    a.n_layers = n_layers;
    const long long weights = 2ll * ((long long)(2 * nq + 2 * nkv) * RUN_HD * width + 3ll * width * ff);
    const int least = weights <= 64ll << 20 ? 2 : weights <= 128ll << 20 ? 3 : weights <= 512ll << 20 ? 4 : 5;
    a.s_qkv = a.s_gate_up = run_waves_log2(width, least);
    a.s_o = run_waves_log2(nq * RUN_HD, least);
    a.s_down = run_waves_log2(ff, least);
    a.b_qkv = (nq + 2 * nkv) * RUN_HD / (64 >> a.s_qkv);
    a.b_attn = rows * nkv * splits;
    a.b_o = width / (64 >> a.s_o);
    a.b_merge = splits > 1 && (long long)a.b_o * rows * nq * splits > 2048 ? rows * nkv : 0;
    a.b_gate_up = ff / (32 >> a.s_gate_up);
    a.b_down = width / (64 >> a.s_down);
    a.per_layer = a.b_qkv + a.b_attn + a.b_merge + a.b_o + a.b_gate_up + a.b_down;
    a.width = width; a.ff = ff; a.nq = nq; a.nkv = nkv; a.max_pages = max_pages; a.splits = splits; a.chunk = chunk; a.max_kv = max_kv_len;
    a.eps1 = eps1; a.eps2 = eps2; a.eps_qk = eps_qk; a.scale_log2 = scale * 1.4426950408889634f;
    a.one1 = one1; a.one2 = one2; a.one_qk = one_qk;
    const int g = nq / nkv, widest = ff > nq * RUN_HD ? (ff > width ? ff : width) : (nq * RUN_HD > width ? nq * RUN_HD : width);
    const size_t product = (size_t)rows * (widest * 2 + RUN_PAD * 4) + (RUN_WAVES * 4 + RUN_WAVES) * rows * sizeof(float);
    const size_t attention = (size_t)(g + 2) * RUN_HD * 2 + (2 * 16 * RUN_WAVES + (size_t)RUN_WAVES * 8 * (RUN_HD + 4)) * sizeof(float);
    const size_t mem = product > attention ? product : attention;
    IA_CHECK(mem <= 160 * 1024 - 64, "layer_run: %d rows of %d inner features need %zu bytes of shared memory", rows, widest, mem);
    const dim3 grid(a.per_layer * n_layers), block(RUN_THREADS);
#define RUN_LAUNCH(R, DOT)                                                                                                            \
    do {                                                                                                                                \
        (void)hipFuncSetAttribute((const void*)layer_run_kernel<R, DOT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mem);     \
        layer_run_kernel<R, DOT><<<grid, block, mem, stream>>>(a);                                                                  \
    } while (0)
    const bool dots = rows == 1 || (rows <= 3 && weights > 128ll << 20);
    switch (rows) {
        case 1: RUN_LAUNCH(1, true); break;
        case 2: if (dots) RUN_LAUNCH(2, true); else RUN_LAUNCH(2, false); break;
        case 3: if (dots) RUN_LAUNCH(3, true); else RUN_LAUNCH(3, false); break;
        case 4: RUN_LAUNCH(4, false); break;
        case 5: RUN_LAUNCH(5, false); break;
        case 6: RUN_LAUNCH(6, false); break;
        case 7: RUN_LAUNCH(7, false); break;
        default: RUN_LAUNCH(8, false);
    }
#undef RUN_LAUNCH
    IA_LAUNCH_CHECK("layer_run");
    return 0;
}
