// Token selection on the device.
//
// ia_argmax: greedy choice, the lowest index among equal maxima (the reference's CPU argmax
// keeps the first maximum, candle-core/src/cpu_backend/mod.rs:150-157; its CUDA reduction
// leaves ties unspecified, inferrs-kernels/candle-kernels/src/reduce.cu:500-520).
//
// ia_penalize: logit bias, repetition penalty (z >= 0 ? z / p : z * p, once per distinct token
// of the window), frequency and presence penalties (z -= f * count + p), in the reference's
// order (inferrs/src/sampler.rs:186-229), in place on 32-bit logits.
//
// ia_sample: the rest of the reference's sampler (sampler.rs:232-335) for a row of logits:
// divide by the temperature, softmax, order by probability (descending, equal values by
// index), keep the first top_k, cut where the running sum reaches top_p, drop what is below
// min_p times the largest probability, renormalise, and walk the kept list until the running
// sum exceeds the row's random number u.  Every one of these filters keeps a prefix of the
// ordered list, so no sort is needed: a prefix is named by a threshold key K and a count m of
// the tokens equal to K (taken by ascending index), and the threshold for "the shortest
// prefix whose weight reaches a target" is found by bisection over the 32 bits of the key,
// one block-wide sum per bit.  Sums are tree sums in a fixed order; they differ from the
// reference's sequential sums by rounding only.  Rows with a top_k of up to 1,024 take a
// shorter way (sample_top_k): their first top_k tokens are picked out and sorted, and the
// reference's steps run on that list as it runs them.  Rows without a top_k try that way with
// the first 1,024 tokens of their list and take the long one when the list does not end there.
// Probabilities, keys and each stretch's candidates for that list are the work of many blocks
// a row (two kernels); one block a row then makes the choice.
#include <mutex>

#include "common.h"
#include "api.h"

// ---- greedy ---------------------------------------------------------------------------------
// every thread's best (value, index; 0x7fffffff: none) -> the block's, the lowest index among equal maxima, in *out
__device__ __forceinline__ void argmax_block(float best, int idx, float* sv, int* si, int* out) {
#pragma unroll
    for (int o = IA_WAVE / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, IA_WAVE);
        const int oi = __shfl_xor(idx, o, IA_WAVE);
        if (ov > best || (ov == best && oi < idx)) { best = ov; idx = oi; }
    }
    const int lane = threadIdx.x & (IA_WAVE - 1), wave = threadIdx.x / IA_WAVE;
    __syncthreads();
    if (lane == 0) { sv[wave] = best; si[wave] = idx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + IA_WAVE - 1) / IA_WAVE;
        for (int w = 1; w < nw; ++w)
            if (sv[w] > best || (sv[w] == best && si[w] < idx)) { best = sv[w]; idx = si[w]; }
        *out = idx == 0x7fffffff ? 0 : idx;       // a row of NaN or -inf
    }
}

__device__ __forceinline__ void argmax_row(const float* __restrict__ row, int vocab, float* sv, int* si, int* out) {
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int c = threadIdx.x; c < vocab; c += blockDim.x) {
        const float v = row[c];
        if (v > best || (v == best && c < idx)) { best = v; idx = c; }
    }
    argmax_block(best, idx, sv, si, out);
}

__global__ __launch_bounds__(1024) void argmax_kernel(int* __restrict__ out, const float* __restrict__ logits, int vocab) {
    __shared__ float sv[16];
    __shared__ int si[16];
    argmax_row(logits + (size_t)blockIdx.x * vocab, vocab, sv, si, out + blockIdx.x);
}

// Long rows in two steps: blocks of a row take a stretch each, then one block a row picks among
// their candidates (lowest index among equal maxima in both steps).
#define ARGMAX_STRETCH 8192
__global__ __launch_bounds__(256) void argmax_stretch_kernel(float* __restrict__ cand_v, int* __restrict__ cand_i,
                                                             const float* __restrict__ logits, int vocab) {
    __shared__ float sv[16];
    __shared__ int si[16];
    const int row = blockIdx.y, stretch = blockIdx.x;
    const int lo = stretch * ARGMAX_STRETCH;
    const int len = vocab - lo < ARGMAX_STRETCH ? vocab - lo : ARGMAX_STRETCH;
    int idx;
    if ((vocab & 3) == 0 && ((uintptr_t)logits & 15) == 0) {
        // four neighbours a load and all of a thread's loads under way together (one after the other, each waiting for
        // its own, a stretch took 16 us)
        constexpr int PER = ARGMAX_STRETCH / 4 / 256;
        const float4* src = (const float4*)(logits + (size_t)row * vocab + lo);
        float4 v[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = (j * 256 + (int)threadIdx.x) * 4;
            v[j] = c < len ? src[c / 4] : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        }
        float best = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = (j * 256 + (int)threadIdx.x) * 4;
            const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (c + i < len && (e[i] > best || (e[i] == best && c + i < at))) { best = e[i]; at = c + i; }
        }
        argmax_block(best, at, sv, si, &idx);
    } else {
        argmax_row(logits + (size_t)row * vocab + lo, len, sv, si, &idx);
    }
    if (threadIdx.x == 0) {
        cand_i[(size_t)row * gridDim.x + stretch] = lo + idx;
        cand_v[(size_t)row * gridDim.x + stretch] = logits[(size_t)row * vocab + lo + idx];
    }
}

__global__ __launch_bounds__(IA_WAVE) void argmax_pick_kernel(int* __restrict__ out, const float* __restrict__ cand_v,
                                                              const int* __restrict__ cand_i, int stretches) {
    const int row = blockIdx.x;
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int c = threadIdx.x; c < stretches; c += IA_WAVE) {
        float v = cand_v[(size_t)row * stretches + c];
        v = v != v ? -INFINITY : v;                      // a stretch of NaN never wins over a number
        const int i = cand_i[(size_t)row * stretches + c];
        if (v > best || (v == best && i < idx) || idx == 0x7fffffff) { best = v; idx = i; }
    }
#pragma unroll
    for (int o = IA_WAVE / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, IA_WAVE);
        const int oi = __shfl_xor(idx, o, IA_WAVE);
        if (oi != 0x7fffffff && (idx == 0x7fffffff || ov > best || (ov == best && oi < idx))) { best = ov; idx = oi; }
    }
    if (threadIdx.x == 0) out[row] = idx == 0x7fffffff ? 0 : idx;
}

extern "C" long long ia_argmax_workspace(int rows, int vocab) {
    return vocab > 2 * ARGMAX_STRETCH ? 2LL * rows * ((vocab + ARGMAX_STRETCH - 1) / ARGMAX_STRETCH) : 0;
}

// `workspace`: ia_argmax_workspace(rows, vocab) words, or null for the one-block-a-row kernel.
extern "C" int ia_argmax(int* out, const float* logits, void* workspace, int rows, int vocab, hipStream_t stream) {
    IA_CHECK(rows >= 0 && vocab > 0, "argmax: bad sizes rows=%d vocab=%d", rows, vocab);
    if (rows == 0) return 0;
    if (workspace != nullptr && vocab > 2 * ARGMAX_STRETCH) {
        const int stretches = (vocab + ARGMAX_STRETCH - 1) / ARGMAX_STRETCH;
        IA_CHECK(rows <= 65535, "argmax: %d rows exceed the grid", rows);
        float* cand_v = (float*)workspace;
        int* cand_i = (int*)workspace + (size_t)rows * stretches;
        argmax_stretch_kernel<<<dim3(stretches, rows), 256, 0, stream>>>(cand_v, cand_i, logits, vocab);
        IA_LAUNCH_CHECK("argmax");
        argmax_pick_kernel<<<rows, IA_WAVE, 0, stream>>>(out, cand_v, cand_i, stretches);
        IA_LAUNCH_CHECK("argmax");
        return 0;
    }
    argmax_kernel<<<rows, 1024, 0, stream>>>(out, logits, vocab);
    IA_LAUNCH_CHECK("argmax");
    return 0;
}

// ---- greedy, for callers that cannot allocate -----------------------------------------------
// The two-step arg max needs a place for the stretches' candidates.  ia_argmax takes it from the caller; this
// entry point keeps one of a fixed size in the library's own device memory instead, so that nothing is
// allocated on the way (declared in api.h with the reasons).  Each GPU holds its own copy of the array at its
// own address: the address is asked for once per device, with that device current, and only that pointer
// (never the array's name, which on the host is a stand-in and no device address) goes to the kernels.
#define ARGMAX_STATIC_WORDS 16384                  // 64 KiB a GPU, held until the process ends
#define ARGMAX_STATIC_DEVICES 64
static __device__ __align__(256) int argmax_scratch[ARGMAX_STATIC_WORDS];
static void* g_argmax_scratch_ptr[ARGMAX_STATIC_DEVICES];    // per device; written once, under the lock
static std::mutex g_argmax_scratch_lock;

extern "C" long long ia_argmax_static_capacity(void) { return ARGMAX_STATIC_WORDS; }

extern "C" int ia_argmax_static(int* out, const float* logits, int rows, int vocab, hipStream_t stream) {
    IA_CHECK(rows >= 0 && vocab > 0, "argmax_static: bad sizes rows=%d vocab=%d", rows, vocab);
    IA_CHECK(out != nullptr && logits != nullptr, "argmax_static: null operand");
    if (rows == 0) return 0;
    const long long words = ia_argmax_workspace(rows, vocab);
    IA_CHECK(words <= ARGMAX_STATIC_WORDS, "argmax_static: %d rows of %d logits need %lld words of scratch, the "
             "library's array holds %d (use ia_argmax with a workspace of your own)", rows, vocab, words, ARGMAX_STATIC_WORDS);
    if (words == 0) {                              // short rows: one block a row, no scratch at all
        argmax_kernel<<<rows, 1024, 0, stream>>>(out, logits, vocab);
        IA_LAUNCH_CHECK("argmax_static");
        return 0;
    }
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    IA_CHECK(e == hipSuccess && device >= 0 && device < ARGMAX_STATIC_DEVICES,
             "argmax_static: cannot tell the current device (%s, device %d)", hipGetErrorString(e), device);
    void* scratch = nullptr;
    {
        std::lock_guard<std::mutex> hold(g_argmax_scratch_lock);
        if (g_argmax_scratch_ptr[device] == nullptr) {
            void* ptr = nullptr;
            e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(argmax_scratch));
            IA_CHECK(e == hipSuccess && ptr != nullptr, "argmax_static: no address for the scratch array on device %d: %s",
                     device, hipGetErrorString(e));
            g_argmax_scratch_ptr[device] = ptr;
        }
        scratch = g_argmax_scratch_ptr[device];
    }
    IA_CHECK(rows <= 65535, "argmax_static: %d rows exceed the grid", rows);
    const int stretches = (vocab + ARGMAX_STRETCH - 1) / ARGMAX_STRETCH;
    // (every candidate that the second kernel reads is written by the first in this call: nothing has to start at zero)
    float* cand_v = (float*)scratch;
    int* cand_i = (int*)scratch + (size_t)rows * stretches;
    argmax_stretch_kernel<<<dim3(stretches, rows), 256, 0, stream>>>(cand_v, cand_i, logits, vocab);
    IA_LAUNCH_CHECK("argmax_static");
    argmax_pick_kernel<<<rows, IA_WAVE, 0, stream>>>(out, cand_v, cand_i, stretches);
    IA_LAUNCH_CHECK("argmax_static");
    return 0;
}

// ---- penalties ------------------------------------------------------------------------------
// window [rows, w]: the last tokens of prompt and output, -1 where a row has fewer.
// bias_ids / bias_vals [rows, nb]: -1 ends a row's list.
struct Penalties {
    const int* window;
    int w;
    const float *rep, *freq, *pres;
    const int* bias_ids;
    const float* bias_vals;
    int nb;
    __host__ __device__ bool any() const { return w > 0 || nb > 0; }
};

#define PENALTY_STAGED 1024                         // entries of a window that a block keeps in shared memory
#define SAMPLE_STRETCH 4096                         // tokens of a row that a block draws among (see RowLayout)

// one thread per distinct token of the window: the one holding its first occurrence
__device__ __forceinline__ void penalize_window(float* z, int lo, int n, const int* held, int w, float rp, float fp, float pp) {
    for (int j = threadIdx.x; j < w; j += blockDim.x) {
        const int id = held[j];
        if (id < lo || id - lo >= n) continue;
        int before = 0, count = 0;
#pragma unroll 8
        for (int i = 0; i < w; ++i) {
            const int same = held[i] == id ? 1 : 0;
            before += i < j ? same : 0;
            count += same;
        }
        if (before > 0) continue;
        float v = z[id - lo];
        if (rp != 1.0f && rp != 0.0f) v = v >= 0.f ? v / rp : v * rp;
        if (fp != 0.0f || pp != 0.0f) {
            v -= fp * (float)count;
            v -= pp;
        }
        z[id - lo] = v;
    }
}

// A row's window into shared memory (PENALTY_STAGED words at `s_win`); a barrier has to follow.
__device__ __forceinline__ void stage_window(const Penalties& p, int rowi, int* s_win) {
    if (p.w <= PENALTY_STAGED)
        for (int j = threadIdx.x; j < p.w; j += blockDim.x) s_win[j] = p.window[(size_t)rowi * p.w + j];
}

// A row's bias and penalties on the logits of its tokens lo .. lo + n, which lie at z[0 .. n) (shared or global memory).
// All threads of the block call it, with every z and the staged window written behind a barrier; it ends with one.  `s_win`: see
// stage_window, PENALTY_STAGED words also where the window is longer.
__device__ __forceinline__ void penalize_range(float* z, int lo, int n, const Penalties& p, int rowi, int* s_win) {
    const int w = p.w;
    const float rp = w > 0 ? p.rep[rowi] : 1.f, fp = w > 0 ? p.freq[rowi] : 0.f, pp = w > 0 ? p.pres[rowi] : 0.f;
    if (p.nb > 0) {
        for (int j = threadIdx.x; j < p.nb; j += blockDim.x) {
            const int id = p.bias_ids[(size_t)rowi * p.nb + j];
            if (id >= lo && id - lo < n) atomicAdd(z + (id - lo), p.bias_vals[(size_t)rowi * p.nb + j]);
        }
        __syncthreads();
    }
    const int* held = s_win;
    int m = w;
    if (w > PENALTY_STAGED) {
        // A long window: its entries among the stretch's tokens, in any order, where these fit (each entry searched the whole window in
        // memory: whole draws with the last 4,000 tokens, us, 128 rows of 262,144 21,615 -> 7,932, 24 rows of 151,936 4,612 -> 1,557).  A
        // whole row's do not fit.
        __shared__ int s_held;
        const int* const all = p.window + (size_t)rowi * w;
        held = all;
        if (n <= SAMPLE_STRETCH) {
            if (threadIdx.x == 0) s_held = 0;
            __syncthreads();
            for (int j = threadIdx.x; j < w; j += blockDim.x) {
                const int id = all[j];
                if (id < lo || id - lo >= n) continue;
                const int slot = atomicAdd(&s_held, 1);
                if (slot < PENALTY_STAGED) s_win[slot] = id;
            }
            __syncthreads();
            if (s_held <= PENALTY_STAGED) {
                held = s_win;
                m = s_held;
            }
        }
    }
    penalize_window(z, lo, n, held, m, rp, fp, pp);
    __syncthreads();
}

__global__ __launch_bounds__(256) void penalize_kernel(float* __restrict__ logits, int vocab, const Penalties p) {
    __shared__ int s_win[PENALTY_STAGED];
    stage_window(p, blockIdx.x, s_win);
    __syncthreads();
    penalize_range(logits + (size_t)blockIdx.x * vocab, 0, vocab, p, blockIdx.x, s_win);
}

static int check_penalties(const char* who, const Penalties& p) {
    IA_CHECK(p.w >= 0 && p.nb >= 0, "%s: bad sizes window=%d bias=%d", who, p.w, p.nb);
    IA_CHECK(p.w == 0 || (p.window != nullptr && p.rep != nullptr && p.freq != nullptr && p.pres != nullptr),
             "%s: a window of %d tokens without its arrays", who, p.w);
    IA_CHECK(p.nb == 0 || (p.bias_ids != nullptr && p.bias_vals != nullptr), "%s: %d bias entries without their arrays", who, p.nb);
    return 0;
}

extern "C" int ia_penalize(float* logits, int rows, int vocab, const int* window, int w, const float* rep,
                           const float* freq, const float* pres, const int* bias_ids, const float* bias_vals,
                           int nb, hipStream_t stream) {
    IA_CHECK(rows >= 0 && vocab > 0, "penalize: bad sizes rows=%d vocab=%d", rows, vocab);
    const Penalties p = {window, w, rep, freq, pres, bias_ids, bias_vals, nb};
    if (const int bad = check_penalties("penalize", p)) return bad;
    if (rows == 0 || !p.any()) return 0;
    penalize_kernel<<<rows, 256, 0, stream>>>(logits, vocab, p);
    IA_LAUNCH_CHECK("penalize");
    return 0;
}

// A row's window after it has drawn `tokens[row]`: the last `caps[row]` tokens of its prompt and output
// (entries from caps[row] on stay -1; caps[row] = 0: the row has no window).  For runs of decode steps that
// are queued without the host in between.
__global__ void window_push_kernel(int* __restrict__ window, int w, const int* __restrict__ caps,
                                   const int* __restrict__ tokens, int rows) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    int* win = window + (size_t)row * w;
    const int cap = caps[row] < w ? caps[row] : w;
    if (cap <= 0) return;
    int held = 0;
    while (held < cap && win[held] >= 0) ++held;
    if (held < cap) {
        win[held] = tokens[row];
        return;
    }
    for (int i = 0; i + 1 < cap; ++i) win[i] = win[i + 1];
    win[cap - 1] = tokens[row];
}

// The same for windows of up to 64 entries (the reference's default, `repeat_last_n`), a wave a row and a lane an
// entry: one thread that moves 64 entries one after the other took 17 us.
__global__ __launch_bounds__(IA_WAVE) void window_push_wave_kernel(int* __restrict__ window, int w, const int* __restrict__ caps,
                                                                   const int* __restrict__ tokens) {
    const int row = blockIdx.x, lane = threadIdx.x;
    int* win = window + (size_t)row * w;
    const int cap = caps[row] < w ? caps[row] : w;
    if (cap <= 0) return;
    const int mine = lane < cap ? win[lane] : -1;
    const unsigned long long empty = __ballot(lane < cap && mine < 0);
    const int held = empty ? __ffsll((long long)empty) - 1 : cap;
    const int next = __shfl_down(mine, 1, IA_WAVE);
    if (held < cap) {
        if (lane == held) win[lane] = tokens[row];
    } else if (lane < cap) {
        win[lane] = lane + 1 < cap ? next : tokens[row];
    }
}

extern "C" int ia_window_push(int* window, int rows, int w, const int* caps, const int* tokens, hipStream_t stream) {
    IA_CHECK(rows >= 0 && w > 0, "window_push: bad sizes rows=%d w=%d", rows, w);
    if (rows == 0) return 0;
    if (w <= IA_WAVE) window_push_wave_kernel<<<rows, IA_WAVE, 0, stream>>>(window, w, caps, tokens);
    else window_push_kernel<<<(rows + 63) / 64, 64, 0, stream>>>(window, w, caps, tokens, rows);
    IA_LAUNCH_CHECK("window_push");
    return 0;
}

// ---- sampling -------------------------------------------------------------------------------
#define SAMPLE_THREADS 1024

// Keys order like the values they come from; NaN sorts below everything.
__device__ __forceinline__ uint32_t order_key(float z) {
    if (z != z) return 0u;
    const uint32_t u = __float_as_uint(z);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct Sums { float w; float n; };

__device__ __forceinline__ Sums block_sums(float w, float n, float* scratch) {
    Sums s;
    s.w = block_sum(w, scratch);
    s.n = block_sum(n, scratch + 16);
    return s;
}

// Weight (probability, or 1 when `by_count`) and number of the tokens with key >= t.
__device__ __forceinline__ Sums at_least(const uint32_t* __restrict__ keys, const float* __restrict__ probs,
                                         int vocab, uint32_t t, bool by_count, float* scratch) {
    float w = 0.f, n = 0.f;
    for (int c = threadIdx.x; c < vocab; c += blockDim.x)
        if (keys[c] >= t) { w += by_count ? 1.0f : probs[c]; n += 1.0f; }
    return block_sums(w, n, scratch);
}

struct Prefix { uint32_t key; int above; int ties; int take; float w_above; float p_key; };

// The shortest prefix of the ordered list whose weight reaches `target` (strictly exceeds it
// when `strict`): every token with a key above `key` and the first `take` of the `ties` tokens
// equal to it.  When even the whole list does not reach the target, the whole list.
__device__ Prefix shortest_prefix(const uint32_t* __restrict__ keys, const float* __restrict__ probs, int vocab,
                                  float target, bool by_count, bool strict, float* scratch) {
    uint32_t k = 0u;
    for (int bit = 31; bit >= 0; --bit) {
        const uint32_t t = k | (1u << bit);
        const float w = at_least(keys, probs, vocab, t, by_count, scratch).w;
        if (strict ? w > target : w >= target) k = t;
    }
    // k is the largest key whose "at least" weight reaches the target (0 if none does).
    float wa = 0.f, na = 0.f, ne = 0.f, pk = 0.f;
    for (int c = threadIdx.x; c < vocab; c += blockDim.x) {
        const uint32_t key = keys[c];
        if (key > k) { wa += by_count ? 1.0f : probs[c]; na += 1.0f; }
        else if (key == k) { ne += 1.0f; pk = by_count ? 1.0f : probs[c]; }
    }
    Prefix r;
    r.key = k;
    r.w_above = block_sum(wa, scratch);
    r.above = (int)block_sum(na, scratch + 16);
    r.ties = (int)block_sum(ne, scratch);
    // every token with this key has the same probability: take it from any thread that saw one
    __shared__ float s_pk;
    if (threadIdx.x == 0) s_pk = 0.f;
    __syncthreads();
    if (ne > 0.f) s_pk = pk;
    __syncthreads();
    r.p_key = s_pk;
    int take = r.ties;
    if (r.ties > 0 && r.p_key > 0.f) {
        float run = r.w_above;
        take = 0;
        while (take < r.ties) {
            run += r.p_key;
            ++take;
            if (strict ? run > target : run >= target) break;
        }
    }
    r.take = take < 1 ? (r.ties > 0 ? 1 : 0) : take;
    return r;
}

// Index of the `rank`-th (1-based, ascending index) token whose key equals `key` (-1: there are fewer).  A thread
// counts a run of neighbouring tokens; the counts are scanned in the wave and over the waves, and the thread in
// whose run the rank falls walks it.  `s_counts`: an entry a wave.
__device__ int nth_with_key(const uint32_t* __restrict__ keys, int vocab, uint32_t key, int rank, int* s_counts) {
    const int per = (vocab + blockDim.x - 1) / blockDim.x;
    const int lo = threadIdx.x * per, hi = lo + per < vocab ? lo + per : vocab;
    int mine = 0;
    for (int c = lo; c < hi; ++c) mine += keys[c] == key;
    const int lane = threadIdx.x & (IA_WAVE - 1), wave = threadIdx.x / IA_WAVE;
    int upto = mine;
#pragma unroll
    for (int o = 1; o < IA_WAVE; o <<= 1) {
        const int other = __shfl_up(upto, o, IA_WAVE);
        if (lane >= o) upto += other;
    }
    __shared__ int s_index;
    __syncthreads();
    if (lane == IA_WAVE - 1) s_counts[wave] = upto;
    if (threadIdx.x == 0) s_index = -1;
    __syncthreads();
    int before = upto - mine;
    for (int w = 0; w < wave; ++w) before += s_counts[w];
    if (before < rank && rank <= before + mine) {
        int seen = before;
        for (int c = lo; c < hi; ++c)
            if (keys[c] == key && ++seen == rank) { s_index = c; break; }
    }
    __syncthreads();
    return s_index;
}

// The first token after (prev_key, prev_idx) in the order of the reference's sorted list: keys
// descending, equal keys by ascending index (its sort is stable).  Returns the index, or -1.
__device__ int next_in_order(const uint32_t* __restrict__ keys, int vocab, uint32_t prev_key, int prev_idx,
                             uint32_t* s_key, int* s_idx) {
    uint32_t bk = 0u;
    int bi = -1;
    for (int c = threadIdx.x; c < vocab; c += blockDim.x) {
        const uint32_t k = keys[c];
        if (!(k < prev_key || (k == prev_key && c > prev_idx))) continue;
        if (bi < 0 || k > bk || (k == bk && c < bi)) { bk = k; bi = c; }
    }
#pragma unroll
    for (int o = IA_WAVE / 2; o > 0; o >>= 1) {
        const uint32_t ok = (uint32_t)__shfl_xor((int)bk, o, IA_WAVE);
        const int oi = __shfl_xor(bi, o, IA_WAVE);
        if (oi >= 0 && (bi < 0 || ok > bk || (ok == bk && oi < bi))) { bk = ok; bi = oi; }
    }
    __syncthreads();
    if ((threadIdx.x & (IA_WAVE - 1)) == 0) { s_key[threadIdx.x / IA_WAVE] = bk; s_idx[threadIdx.x / IA_WAVE] = bi; }
    __syncthreads();
    bk = 0u; bi = -1;
    for (int w = 0; w < (int)(blockDim.x / IA_WAVE); ++w) {
        const uint32_t ok = s_key[w];
        const int oi = s_idx[w];
        if (oi >= 0 && (bi < 0 || ok > bk || (ok == bk && oi < bi))) { bk = ok; bi = oi; }
    }
    __syncthreads();
    return bi;
}

#define SAMPLE_MAX_TOP 20

// With a top_k of up to SAMPLE_FAST_K every filter works on the first top_k entries of the ordered list, so
// the row's top_k tokens are picked out first (three histograms over the key's bits find the k-th largest
// key; equal keys are taken by ascending index), sorted in shared memory, and one thread then does what the
// reference does with its sorted list, in its order and with its sums (sampler.rs:256-335): six passes over
// the row instead of the hundred of the bisections below (16 rows of 152 k: 2.5 ms -> 0.16 ms).
#define SAMPLE_FAST_K 1024
// f(index, key) for all keys of a row, this thread's share, four loads under way at a time.
template <typename F>
__device__ __forceinline__ void for_each_key(const uint32_t* __restrict__ keys, int vocab, F f) {
    for (int c0 = threadIdx.x; c0 < vocab; c0 += 4 * blockDim.x) {
        uint32_t k[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + j * (int)blockDim.x;
            k[j] = c < vocab ? keys[c] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + j * (int)blockDim.x;
            if (c < vocab) f(c, k[j]);
        }
    }
}
// The first k entries of the ordered list of `n` keys (keys descending, equal keys by ascending place): every
// key above `kth`, and the keys equal to it up to place `last_tie`.  0 < k < n.  Three histograms over the
// key's bits, 11 + 11 + 10 at a time, find the k-th largest key.
struct Cut { uint32_t kth; int last_tie; };
__device__ Cut top_k_cut(const uint32_t* __restrict__ keys, int n, int k, int* s_counts) {
    __shared__ int hist[2048];
    __shared__ int s_bin, s_above;
    uint32_t prefix = 0u;
    int prefix_bits = 0, need = k;
    for (int level = 0; level < 3; ++level) {
        const int bits = level < 2 ? 11 : 10;
        const int shift = 32 - prefix_bits - bits;
        for (int i = threadIdx.x; i < 2048; i += blockDim.x) hist[i] = 0;
        __syncthreads();
        for_each_key(keys, n, [&](int, uint32_t key) {
            if (prefix_bits == 0 || (key >> (32 - prefix_bits)) == prefix)
                atomicAdd(&hist[(key >> shift) & ((1u << bits) - 1u)], 1);
        });
        __syncthreads();
        // the highest bin at which the count from the top reaches `need`: lane l of the first wave adds up
        // bins top - 32 l - 31 .. top - 32 l, the lanes' sums are scanned, and the lane where the count is
        // reached walks its own bins
        if (threadIdx.x < IA_WAVE) {
            const int n_bins = 1 << bits, per = n_bins / IA_WAVE;
            const int top = n_bins - 1 - (int)threadIdx.x * per;
            int mine = 0;
            for (int i = 0; i < per; ++i) mine += hist[top - i];
            int upto = mine;                                   // inclusive scan over the lanes
#pragma unroll
            for (int o = 1; o < IA_WAVE; o <<= 1) {
                const int other = __shfl_up(upto, o, IA_WAVE);
                if ((int)threadIdx.x >= o) upto += other;
            }
            const unsigned long long reached = __ballot(upto >= need);
            const int first = reached ? __ffsll((long long)reached) - 1 : IA_WAVE - 1;
            if ((int)threadIdx.x == first) {
                int cum = upto - mine, b = top;
                for (; b > top - per + 1; --b) {
                    if (cum + hist[b] >= need) break;
                    cum += hist[b];
                }
                s_bin = b;
                s_above = cum;
            }
        }
        __syncthreads();
        need -= s_above;
        prefix = (prefix << bits) | (uint32_t)s_bin;
        prefix_bits += bits;
        __syncthreads();
    }
    Cut cut;
    cut.kth = prefix;                                       // `need` (>= 1) of the tokens with this key belong to the list
    const int ties = hist[cut.kth & 1023u];
    __syncthreads();
    cut.last_tie = n;                                       // ties up to this place are taken
    if (ties > need) cut.last_tie = nth_with_key(keys, n, cut.kth, need, s_counts);
    return cut;
}

// The reference's steps on the first k entries of a row's ordered list.  `keys` [n] holds the row's candidates in
// the order of their tokens' indices (every stretch of the row has left its own first k there, so the row's first
// k are among them), `token_of` [n] their tokens (null: a candidate's place is its token), `probs` the whole row's
// probabilities by token.
// `open`: the row has no top_k; k tokens are only the beginning of its list, whose weight is `total`.  The steps
// then succeed if top_p or min_p end the list within these k, or else the walk ends there; if not, nothing is
// written and false comes back (the caller goes the long way).
__device__ bool sample_top_k(int* __restrict__ out, const uint32_t* __restrict__ keys, const int* __restrict__ token_of,
                             const float* __restrict__ probs, int n_keys, int rowi, int k, bool open, float total,
                             float tp, float mp, float u, int want_top, float* __restrict__ lp_out,
                             int* __restrict__ lp_ids, int* s_counts) {
    __shared__ unsigned long long cand[SAMPLE_FAST_K];      // (key, ~place): larger is earlier in the list
    __shared__ int s_n, s_done;
    Cut cut;
    if (k < n_keys) cut = top_k_cut(keys, n_keys, k, s_counts);
    else { cut.kth = 0u; cut.last_tie = n_keys; }
    const uint32_t kth = cut.kth;
    const int last_tie = cut.last_tie;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for_each_key(keys, n_keys, [&](int c, uint32_t key) {
        if (key > kth || (key == kth && c <= last_tie)) {
            const int slot = atomicAdd(&s_n, 1);
            if (slot < SAMPLE_FAST_K) cand[slot] = ((unsigned long long)key << 32) | (uint32_t)~(uint32_t)c;
        }
    });
    __syncthreads();
    const int n = s_n < k ? s_n : k;                        // = k
    int padded = 2;
    while (padded < n) padded <<= 1;
    for (int i = n + threadIdx.x; i < padded; i += blockDim.x) cand[i] = 0ull;
    // ---- bitonic sort, descending
    for (int size = 2; size <= padded; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (int t = threadIdx.x; t < padded / 2; t += blockDim.x) {
                const int i = 2 * t - (t & (stride - 1)), j = i + stride;
                const bool down = (i & size) == 0;
                const unsigned long long a = cand[i], b = cand[j];
                if ((a < b) == down) { cand[i] = b; cand[j] = a; }
            }
        }
    __syncthreads();
    __shared__ float cprob[SAMPLE_FAST_K];
    auto index_of = [&](int i) {
        const int place = (int)~(uint32_t)(cand[i] & 0xffffffffull);
        return token_of != nullptr ? token_of[place] : place;
    };
    for (int i = threadIdx.x; i < n; i += blockDim.x) cprob[i] = probs[index_of(i)];
    __syncthreads();
    if (threadIdx.x == 0) {
        // ---- the reference's steps 7 to 12 on its sorted list
        bool ended = !open, done = true;                    // ended: the list's end lies within these n tokens
        int len = n;
        if (tp < 1.0f) {
            float cumsum = 0.f;
            bool found = false;
            for (int i = 0; i < len; ++i) {
                cumsum += cprob[i];
                if (cumsum >= tp) { len = i + 1; found = true; break; }
            }
            if (found) ended = true;
            else if (open) done = false;                    // the nucleus is longer than what was picked out
        }
        if (done && mp > 0.0f && len > 0) {
            const float threshold = cprob[0] * mp;
            int cut = 0;
            while (cut < len && cprob[cut] >= threshold) ++cut;
            if (cut < len) { if (cut > 0) len = cut; ended = true; }
            else if (!ended) done = false;                  // every picked token passes: the cut lies further on
        }
        float filtered = total;
        if (done && ended) {
            filtered = 0.f;
            for (int i = 0; i < len; ++i) filtered += cprob[i];
        }
        int at = -1;
        if (done && filtered > 0.f) {
            float rng = u;
            for (int i = 0; i < len; ++i) {
                const float norm = cprob[i] / filtered;
                if (rng < norm) { at = i; break; }
                rng -= norm;
            }
            if (at < 0) {
                if (ended) at = len - 1;
                else done = false;                          // the walk goes on beyond what was picked out
            }
        }
        if (done) {
            const float denom = filtered > 0.f ? filtered : 1.0f;
            if (want_top >= 0)
                for (int i = 0; i < want_top && i < SAMPLE_MAX_TOP && i < len; ++i) {
                    const float pi = cprob[i];
                    lp_ids[(size_t)rowi * SAMPLE_MAX_TOP + i] = index_of(i);
                    lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP) + 1 + i] = pi > 0.f ? logf(pi / denom) : -INFINITY;
                }
            if (!(filtered > 0.f)) {
                out[rowi] = len > 0 ? index_of(0) : 0;
                if (want_top >= 0) lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP)] = -INFINITY;
            } else {
                out[rowi] = index_of(at);
                if (want_top >= 0) {
                    const float pt = cprob[at] / filtered;
                    lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP)] = pt > 0.f ? logf(pt) : -INFINITY;
                }
            }
        }
        s_done = done ? 1 : 0;
    }
    __syncthreads();
    return s_done != 0;
}

// ---- a row's workspace and the two passes that fill it --------------------------------------
// Temperature, softmax and the ordering keys of a row are the work of many blocks (a row of 152 k logits kept one
// block busy for 150 us, whatever the batch): the row is cut into stretches of up to SAMPLE_STRETCH tokens, a block each
// (a stretch's keys fit the block's shared memory).
//   pass 1 (sample_partials_kernel): the stretch's maximum of z / temperature and its sum of exp(. - that maximum);
//   pass 2 (sample_stretch_kernel): the row's maximum and sum from the stretches' (every block adds them up in the
//     same order), probabilities and keys of the stretch, the sum of its probabilities, and the stretch's own
//     first k entries of the ordered list (k: the row's top_k, or SAMPLE_FAST_K for a row without one), written
//     in the order of their tokens at a place that follows from k and the stretches' lengths alone;
//   then one block a row (sample_kernel) picks the row's first k among those candidates and walks them.
// Rows with a top_k of up to SAMPLE_NARROW_K ("narrow" ones, see is_narrow; the reference's default is 50) need no second pass: the
// first leaves those of its stretch's logits that can be among the row's first k (see NARROW_MARGIN), the last
// block works out their probabilities alone.  24 rows of 151,936 logits with the default parameters: 86 us of kernels,
// of them the second pass 36 (16 bytes written a logit, three histograms of keys that mostly fall into one bin) and the
// last 28 (three more of them and one thread's walk through shared memory), before; 30 now, 16 and 13.
// Bias and penalties are applied where a stretch's logits are read; the caller's logits stay as they are.
// A row's words: keys [vocab], probabilities [vocab], the candidates' keys (narrow rows: their logits over the
// temperature) and tokens [stretches * SAMPLE_FAST_K] each, and the stretches' maxima, sums and sums of probabilities
// (narrow rows: numbers of candidates) [stretches] each.
#define SAMPLE_STAGED 8192              // candidates of a row that its last block keeps in shared memory
#define SAMPLE_MAX_STRETCHES 1024       // 4 M tokens a row
#define SAMPLE_NARROW_K 64
struct RowLayout {
    int vocab, stretches, stretch;      // stretch: tokens a stretch (the last one may be shorter), a multiple of 4
    long long words;                    // of a row
    __host__ __device__ int length(int b) const { const int left = vocab - b * stretch; return left < stretch ? left : stretch; }
    // candidates that the stretches before b leave when every stretch leaves its first k (or all it has)
    __host__ __device__ int candidates_before(int b, int k) const {
        const int each = k < stretch ? k : stretch;     // every stretch before the last is a whole one
        return b * each;
    }
    __host__ __device__ int candidates(int k) const {
        const int last = length(stretches - 1);
        return candidates_before(stretches - 1, k) + (k < last ? k : last);
    }
    __device__ uint32_t* keys(uint32_t* ws, int row) const { return ws + (size_t)row * words; }
    __device__ float* probs(uint32_t* ws, int row) const { return (float*)(keys(ws, row) + vocab); }
    __device__ uint32_t* cand_keys(uint32_t* ws, int row) const { return keys(ws, row) + 2 * (size_t)vocab; }
    __device__ int* cand_tokens(uint32_t* ws, int row) const { return (int*)(cand_keys(ws, row) + (size_t)stretches * SAMPLE_FAST_K); }
    __device__ float* part_max(uint32_t* ws, int row) const { return (float*)(cand_tokens(ws, row) + (size_t)stretches * SAMPLE_FAST_K); }
    __device__ float* part_sum(uint32_t* ws, int row) const { return part_max(ws, row) + stretches; }
    __device__ float* part_total(uint32_t* ws, int row) const { return part_sum(ws, row) + stretches; }
    __device__ int* part_count(uint32_t* ws, int row) const { return (int*)part_total(ws, row); }
};

static RowLayout row_layout(int vocab) {
    RowLayout l;
    l.vocab = vocab;
    l.stretches = (vocab + SAMPLE_STRETCH - 1) / SAMPLE_STRETCH;
    l.stretch = ((vocab + l.stretches - 1) / l.stretches + 3) & ~3;
    const long long words = 2LL * vocab + 2LL * l.stretches * SAMPLE_FAST_K + 3LL * l.stretches;
    l.words = (words + 3) & ~3LL;
    return l;
}

// The temperature a row is sampled at; false: the row is a greedy one and has no use for probabilities.
__device__ __forceinline__ bool row_temperature(const float* temperature, const int* n_top, int rowi, float& temp) {
    temp = temperature[rowi];
    if (temp < 1e-5f) {
        if (n_top == nullptr || n_top[rowi] < 0) return false;
        temp = 1e-5f;           // with log-probabilities the reference takes no shortcut (sampler.rs:176, :232-239)
    }
    return true;
}

// Lane i's value, i the same for all lanes: no trip through shared memory.
__device__ __forceinline__ float lane_value(float v, int i) { return __uint_as_float((uint32_t)__builtin_amdgcn_readlane(__float_as_int(v), i)); }

// The row's maximum, the sum of exp(z / temperature - maximum) and (with `with_total`) the sum of the probabilities
// from the stretches' (a stretch of nothing but -inf adds nothing to the sum); every block that asks gets the same bits.
// All threads of the block call it; the first wave does the work, a stretch a lane, and adds up in order through scalar
// registers (every thread adding them up out of shared memory kept its reads busy for 2 us of the last block's time).
struct RowSums { float mx, sum, total; };
__device__ RowSums row_sums(const RowLayout& l, uint32_t* ws, int rowi, bool with_total) {
    __shared__ RowSums s_sums;
    if (threadIdx.x < IA_WAVE) {
        const float *maxima = l.part_max(ws, rowi), *sums = l.part_sum(ws, rowi), *totals = l.part_total(ws, rowi);
        const int lane = threadIdx.x;
        RowSums r;
        r.mx = -INFINITY;
        float first_m = -INFINITY, first_s = 0.f, first_t = 0.f;      // (the first 64 stretches' are read once)
        if (lane < l.stretches) {
            first_m = maxima[lane];
            first_s = sums[lane];
            if (with_total) first_t = totals[lane];
        }
        for (int b = lane; b < l.stretches; b += IA_WAVE) r.mx = fmaxf(r.mx, b == lane ? first_m : maxima[b]);
        r.mx = wave_max(r.mx);
        r.sum = r.total = 0.f;
        for (int b0 = 0; b0 < l.stretches; b0 += IA_WAVE) {
            const int b = b0 + lane;
            float m = first_m, a = first_s, t = first_t;
            if (b0 > 0) {
                m = b < l.stretches ? maxima[b] : -INFINITY;
                a = b < l.stretches ? sums[b] : 0.f;
                t = with_total && b < l.stretches ? totals[b] : 0.f;
            }
            const float e = m > -INFINITY ? expf(m - r.mx) : 0.f;
            const unsigned long long counts = __ballot(m > -INFINITY);
            const int here = l.stretches - b0 < IA_WAVE ? l.stretches - b0 : IA_WAVE;
            for (int i = 0; i < here; ++i) {
                if ((counts >> i) & 1) r.sum = fmaf(lane_value(a, i), lane_value(e, i), r.sum);
                if (with_total) r.total += lane_value(t, i);
            }
        }
        if (lane == 0) s_sums = r;
    }
    __syncthreads();
    return s_sums;
}

// A stretch's logits into shared memory, with the row's bias and penalties.  All threads of the block call it; it ends with a barrier.
__device__ __forceinline__ void load_stretch(float* s_z, const float* __restrict__ logits, const RowLayout& l, int rowi, int b,
                                             const Penalties& pen, int* s_win) {
    const int lo = b * l.stretch, n = l.length(b);
    const float* row = logits + (size_t)rowi * l.vocab + lo;
    stage_window(pen, rowi, s_win);
    if (((uintptr_t)row & 15) == 0) {
        // all of a thread's pieces of four under way together
        constexpr int PER = SAMPLE_STRETCH / 4 / 256;
        float4 v[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = (j * 256 + (int)threadIdx.x) * 4;
            v[j] = c + 4 <= n ? *(const float4*)(row + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = (j * 256 + (int)threadIdx.x) * 4;
            if (c + 4 <= n) *(float4*)(s_z + c) = v[j];
        }
        const int rest = (n & ~3) + (int)threadIdx.x;
        if (rest < n) s_z[rest] = row[rest];
    } else {
        constexpr int PER = SAMPLE_STRETCH / 256;
        float v[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = j * 256 + (int)threadIdx.x;
            v[j] = c < n ? row[c] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int c = j * 256 + (int)threadIdx.x;
            if (c < n) s_z[c] = v[j];
        }
    }
    __syncthreads();
    if (pen.any()) penalize_range(s_z, lo, n, pen, rowi, s_win);
}

// What decides whether a row is a narrow one: a top_k of up to SAMPLE_NARROW_K, and candidates that hold what it reports.  A row that
// reports entries (two and more; the first is always a candidate) of a list that neither top_p nor min_p ends reports tokens far
// under its maximum, down to those whose probability is 0 (by index then), and the candidates end at NARROW_FLOOR, 83 under it.
// At NARROW_COOL these are 20 between the logits, more than a model's first entries are apart; below it, and where a bias may set
// a token apart from all others, such rows stay with the second pass.  Whole draws of 24 rows of 151,936 with entries and no
// top_p, us, candidates and one block a row for what they do not settle / second pass: temperature 0 877 / 356, a bias of 100
// 887 / 362; temperature 0.1 with logits close enough to be settled 243 / 310.
#define NARROW_COOL 0.25f
__host__ __device__ __forceinline__ bool is_narrow(int k, int vocab, float temp, float tp, float mp, int want_top, bool biased) {
    const bool open = want_top > 1 && !(tp < 1.0f) && !(mp > 0.0f);
    return k > 0 && k < vocab && k <= SAMPLE_NARROW_K && !(open && (biased || temp < NARROW_COOL));
}

// A row's parameters as the passes read them.
struct RowParams {
    const float* temperature;
    const int* top_k;
    const float *top_p, *min_p;
    const int* n_top;
};
// (a row's list of biases starts with its first token or holds none)
__device__ __forceinline__ bool row_is_narrow(const RowParams& r, const Penalties& p, int rowi, int vocab, int fast) {
    return fast == 1 && is_narrow(r.top_k[rowi], vocab, r.temperature[rowi], r.top_p[rowi], r.min_p[rowi], r.n_top != nullptr ? r.n_top[rowi] : -1,
                                  p.nb > 0 && p.bias_ids[(size_t)rowi * p.nb] >= 0);
}

// Those of a stretch's logits that can be among the row's first k tokens, k <= SAMPLE_NARROW_K, ordered by their
// rounded probabilities p = exp(y - the row's maximum) / the row's sum and by index where these are equal; y, the logits over the
// temperature.  Of the 128 pairs of threads k hold a maximum of at least Y, the k-th largest of these
// maxima.  A y under Y by NARROW_MARGIN has k tokens of its stretch strictly before it as long as its p is no denormal: the
// difference y - maximum is off by 4e-6 at most (up to 128 away; p vanishes beyond 104), the exponential by two units in
// the last place and the quotient by half of one, 3e-7 of p together, so that p's of tokens 2e-5 apart cannot meet.  (The
// margin is twice that, for the rounding of Y - margin; where y is so large that the margin is below its spacing, tokens under Y
// are a whole unit in the last place of y below it.)  A y of NARROW_DEPTH under the stretch's maximum has a p under
// NARROW_FLOOR.  The last block takes no token whose p is under the floor from these candidates (sample_narrow), so
// both may be left out.  SAMPLE_FAST_K places; a stretch with more candidates (equal logits in great number) says so by its count.
#define NARROW_MARGIN 4e-5f
#define NARROW_DEPTH 88.0f              // exp(-88) = 6e-39, under a hundredth of the floor
#define NARROW_FLOOR 1e-36f

// Bound by the trip to the memory, a logit's division and exponential, and the barriers between its phases; several blocks a
// compute unit hide each other's.
__global__ __launch_bounds__(256) void sample_partials_kernel(const float* __restrict__ logits, uint32_t* __restrict__ workspace,
                                                              const RowLayout l, const RowParams params, const Penalties pen,
                                                              int fast) {
    __shared__ __attribute__((aligned(16))) float s_z[SAMPLE_STRETCH];
    __shared__ int s_win[PENALTY_STAGED];
    __shared__ __attribute__((aligned(16))) uint32_t s_group[128];
    __shared__ float s_max[256 / IA_WAVE], s_sum[256 / IA_WAVE];
    __shared__ uint32_t s_kth;
    __shared__ int s_n;
    constexpr int PER = SAMPLE_STRETCH / 256;
    const int rowi = blockIdx.y, b = blockIdx.x, t = threadIdx.x, wave = t / IA_WAVE;
    const int k = params.top_k[rowi];
    const bool narrow = row_is_narrow(params, pen, rowi, l.vocab, fast);
    float temp;
    if (!row_temperature(params.temperature, params.n_top, rowi, temp)) return;
    const int n = l.length(b);
    if (t == 0) { s_kth = 0u; s_n = 0; }
    load_stretch(s_z, logits, l, rowi, b, pen, s_win);
    // temperature, and the softmax's two sums (sampler.rs:232-249)
    float y[PER], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int c = t + j * 256;
        y[j] = c < n ? s_z[c] / temp : -INFINITY;
        mx = fmaxf(mx, y[j]);
    }
    // (the keys of the pairs' maxima; a NaN is no maximum, and a row that holds one is not settled by candidates)
    const uint32_t mine = order_key(fmaxf(mx, __shfl_xor(mx, 1, IA_WAVE)));
    if ((t & 1) == 0) s_group[t >> 1] = mine;
    mx = wave_max(mx);
    if ((t & (IA_WAVE - 1)) == 0) s_max[wave] = mx;
    __syncthreads();
    for (int w = 0; w < 256 / IA_WAVE; ++w) mx = fmaxf(mx, s_max[w]);
    float sum = 0.f;
    if (mx > -INFINITY) {
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (t + j * 256 < n) sum += expf(y[j] - mx);
    }
    sum = wave_sum(sum);
    if ((t & (IA_WAVE - 1)) == 0) s_sum[wave] = sum;
    if (narrow) {
        // a pair's rank among the pairs, half of the comparisons each
        int before = 0;
#pragma unroll
        for (int i = 0; i < 64; i += 4) {
            const int at = (t & 1) * 64 + i;
            const uint4 g = *(const uint4*)(s_group + at);
            const uint32_t e[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) before += (e[q] > mine || (e[q] == mine && at + q < (t >> 1))) ? 1 : 0;
        }
        before += __shfl_xor(before, 1, IA_WAVE);
        if (before == k - 1 && (t & 1) == 0) s_kth = mine;
    }
    __syncthreads();
    if (t == 0) {
        float total = 0.f;
        for (int w = 0; w < 256 / IA_WAVE; ++w) total += s_sum[w];
        l.part_max(workspace, rowi)[b] = mx;
        l.part_sum(workspace, rowi)[b] = total;
    }
    if (!narrow) return;
    uint32_t* cand_y = l.cand_keys(workspace, rowi) + (size_t)b * SAMPLE_FAST_K;
    int* cand_token = l.cand_tokens(workspace, rowi) + (size_t)b * SAMPLE_FAST_K;
    const uint32_t kth = s_kth;
    const float least = fmaxf(__uint_as_float((kth & 0x80000000u) ? kth & 0x7fffffffu : ~kth) - NARROW_MARGIN, mx - NARROW_DEPTH);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int c = t + j * 256;
        if (c < n && y[j] >= least && y[j] > -INFINITY) {
            const int slot = atomicAdd(&s_n, 1);
            if (slot < SAMPLE_FAST_K) {
                cand_y[slot] = __float_as_uint(y[j]);
                cand_token[slot] = b * l.stretch + c;
            }
        }
    }
    __syncthreads();
    if (t == 0) l.part_count(workspace, rowi)[b] = s_n;
}

// How many entries of a row's ordered list are picked out before the reference's steps run on them: the row's
// top_k, SAMPLE_FAST_K for a row without one, 0 for a row that goes the long way (a top_k beyond SAMPLE_FAST_K, a
// vocabulary within it, or the switch off).
__device__ __forceinline__ int picked_out(int k, int vocab, int fast_top_k) {
    if (!fast_top_k) return 0;
    if (k > 0 && k < vocab) return k <= SAMPLE_FAST_K ? k : 0;
    return vocab > SAMPLE_FAST_K ? SAMPLE_FAST_K : 0;
}

#define STRETCH_THREADS 256
__global__ __launch_bounds__(STRETCH_THREADS) void sample_stretch_kernel(
    const float* __restrict__ logits, uint32_t* __restrict__ workspace, const RowLayout l, const RowParams params, const Penalties pen,
    int fast_top_k) {
    __shared__ float scratch[32];
    __shared__ int s_counts[STRETCH_THREADS];
    __shared__ int s_waves[STRETCH_THREADS / IA_WAVE];
    __shared__ __attribute__((aligned(16))) uint32_t s_keys[SAMPLE_STRETCH];   // the stretch's logits, then its keys: the choice below reads them several times
    __shared__ int s_win[PENALTY_STAGED];
    const int rowi = blockIdx.y, b = blockIdx.x;
    float temp;
    if (!row_temperature(params.temperature, params.n_top, rowi, temp)) return;
    if (row_is_narrow(params, pen, rowi, l.vocab, fast_top_k)) return;
    const int lo = b * l.stretch, n = l.length(b);
    load_stretch((float*)s_keys, logits, l, rowi, b, pen, s_win);
    uint32_t* keys = l.keys(workspace, rowi) + lo;
    float* probs = l.probs(workspace, rowi) + lo;
    const RowSums rs = row_sums(l, workspace, rowi, false);
    // The list is ordered by the probabilities themselves, as the reference sorts them: logits whose
    // probabilities round to the same number (or vanish together) are ties, taken in index order.
    float t = 0.f;
    for (int c0 = threadIdx.x; c0 < n; c0 += 4 * blockDim.x) {
        float z[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + j * (int)blockDim.x;
            z[j] = c < n ? __uint_as_float(s_keys[c]) : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + j * (int)blockDim.x;
            if (c < n) {
                const float e = expf(z[j] / temp - rs.mx);
                const float pr = rs.sum > 0.f ? e / rs.sum : e;
                const uint32_t key = order_key(pr);
                probs[c] = pr;
                keys[c] = key;
                s_keys[c] = key;
                t += pr;
            }
        }
    }
    t = block_sum(t, scratch);
    if (threadIdx.x == 0) l.part_total(workspace, rowi)[b] = t;
    const int k = picked_out(params.top_k[rowi], l.vocab, fast_top_k);
    if (k == 0) return;
    __syncthreads();
    // ---- the stretch's own first k, in the order of their tokens
    uint32_t* ck = l.cand_keys(workspace, rowi) + l.candidates_before(b, k);
    int* ct = l.cand_tokens(workspace, rowi) + l.candidates_before(b, k);
    if (k >= n) {
        for (int c = threadIdx.x; c < n; c += blockDim.x) { ck[c] = s_keys[c]; ct[c] = lo + c; }
        return;
    }
    const Cut cut = top_k_cut(s_keys, n, k, s_counts);
    // a thread takes a run of neighbouring tokens, counts those of the list, and writes them behind what the
    // threads before it have counted
    const int per = (n + blockDim.x - 1) / blockDim.x;
    const int first = threadIdx.x * per, last = first + per < n ? first + per : n;
    int mine = 0;
    for (int c = first; c < last; ++c) {
        const uint32_t key = s_keys[c];
        mine += (key > cut.kth || (key == cut.kth && c <= cut.last_tie)) ? 1 : 0;
    }
    int upto = mine;                                        // inclusive scan over the wave's lanes
    const int lane = threadIdx.x & (IA_WAVE - 1), wave = threadIdx.x / IA_WAVE;
#pragma unroll
    for (int o = 1; o < IA_WAVE; o <<= 1) {
        const int other = __shfl_up(upto, o, IA_WAVE);
        if (lane >= o) upto += other;
    }
    if (lane == IA_WAVE - 1) s_waves[wave] = upto;
    __syncthreads();
    int at = upto - mine;
    for (int w = 0; w < wave; ++w) at += s_waves[w];
    for (int c = first; c < last; ++c) {
        const uint32_t key = s_keys[c];
        if (key > cut.kth || (key == cut.kth && c <= cut.last_tie)) {
            if (at < k) { ck[at] = key; ct[at] = lo + c; }
            ++at;
        }
    }
}

// The reference's steps (sampler.rs:251-335) on a narrow row: the candidates' probabilities, the first k of them in order
// and the walk, with the sums in the reference's order.  False, and nothing that counts is written, where the candidates
// do not settle the row: a stretch had more than its places, there is a NaN or no number to start from, or the draw (or
// an entry that is reported) lies among probabilities under the floor, whose order and ties the candidates do not hold.  (A list
// that top_p or min_p ends before that holds none of these, however few candidates there are: at temperature 0 it is mostly one.)
// A block of 1,024 threads; all of them call it.
// One block a row, so the time is a chain: one trip to the memory (a wave takes the stretches wave, wave + 16, ...; the first
// 128 candidates of three of them are asked for before their number is known, the places exist), five barriers, and the
// reference's running sums over up to 64 values, which go lane by lane through a scalar register (through shared memory a step
// took 100 cycles).
__device__ bool sample_narrow(int* __restrict__ out, const RowLayout& l, uint32_t* __restrict__ ws, int rowi, int k,
                              float tp, float mp, float u, int want_top, float* __restrict__ lp_out, int* __restrict__ lp_ids) {
    __shared__ unsigned long long s_list[SAMPLE_FAST_K];    // (key, ~token): larger is earlier in the list
    __shared__ unsigned long long s_first[SAMPLE_NARROW_K];
    __shared__ __attribute__((aligned(16))) uint32_t s_group[128];
    __shared__ uint32_t s_kth;
    __shared__ int s_n, s_over, s_settled;
    const int t = threadIdx.x, lane = t & (IA_WAVE - 1), wave = t / IA_WAVE;
    const uint32_t* cand_y = l.cand_keys(ws, rowi);
    const int* cand_token = l.cand_tokens(ws, rowi);
    const int* counts = l.part_count(ws, rowi);
    if (t == 0) { s_n = 0; s_over = 0; s_kth = 0u; s_settled = 0; }
    constexpr int KEEP = 3, WAVES = SAMPLE_THREADS / IA_WAVE;
    uint32_t key[KEEP][2];
    int token[KEEP][2], held[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int b = wave + i * WAVES;
        const int from = b < l.stretches ? b : 0;
        held[i] = b < l.stretches ? counts[from] : 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            key[i][h] = cand_y[(size_t)from * SAMPLE_FAST_K + h * IA_WAVE + lane];
            token[i][h] = cand_token[(size_t)from * SAMPLE_FAST_K + h * IA_WAVE + lane];
        }
    }
    const RowSums rs = row_sums(l, ws, rowi, false);
    // A candidate's key; 0 for one under the floor, which settles nothing (a token far above all others leaves thousands of
    // those behind, more than there are places: 50 of each stretch whose probabilities are all 0).
    auto key_of = [&](uint32_t y) {
        const float e = expf(__uint_as_float(y) - rs.mx);
        const float p = rs.sum > 0.f ? e / rs.sum : e;
        return p >= NARROW_FLOOR ? order_key(p) : 0u;
    };
    uint32_t mine = 0u;
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            key[i][h] = h * IA_WAVE + lane < held[i] ? key_of(key[i][h]) : 0u;
            mine = key[i][h] > mine ? key[i][h] : mine;
        }
    // the k-th largest of 128 groups' maxima: at least k candidates are no smaller
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)mine, o, IA_WAVE);
        mine = other > mine ? other : mine;
    }
    if ((t & 7) == 0) s_group[t >> 3] = mine;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
        const int at = (t & 7) * 16 + i;
        const uint4 g = *(const uint4*)(s_group + at);
        const uint32_t e[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) before += (e[q] > mine || (e[q] == mine && at + q < (t >> 3))) ? 1 : 0;
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) before += __shfl_xor(before, o, IA_WAVE);
    if (before == k - 1 && (t & 7) == 0) s_kth = mine;
    __syncthreads();
    const uint32_t kth = s_kth;
    auto take = [&](uint32_t ky, int tok) {
        if (ky == 0u || ky < kth) return;
        const int slot = atomicAdd(&s_n, 1);
        if (slot < SAMPLE_FAST_K) s_list[slot] = ((unsigned long long)ky << 32) | (uint32_t)~(uint32_t)tok;
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) take(key[i][h], token[i][h]);
    // what the registers did not hold: candidates beyond 128 of a stretch, stretches beyond 48
    for (int b = wave, i = 0; b < l.stretches; b += WAVES, ++i) {
        const int all = counts[b], end = all < SAMPLE_FAST_K ? all : SAMPLE_FAST_K;
        if (all > SAMPLE_FAST_K && lane == 0) s_over = 1;
        for (int at = (i < KEEP ? 2 * IA_WAVE : 0) + lane; at < end; at += IA_WAVE)
            take(key_of(cand_y[(size_t)b * SAMPLE_FAST_K + at]), cand_token[(size_t)b * SAMPLE_FAST_K + at]);
    }
    __syncthreads();
    const int found = s_n;
    if (s_over || found > SAMPLE_FAST_K || found == 0 || !(rs.mx > -INFINITY && rs.mx < INFINITY) || !(rs.sum > 0.f && rs.sum < INFINITY))
        return false;
    // an entry's place is the number of larger ones (no two are equal: a token has one entry)
    if (t < found) {
        const unsigned long long e = s_list[t];
        int place = 0;
#pragma unroll 8
        for (int i = 0; i < found; ++i) place += s_list[i] > e ? 1 : 0;
        if (place < k) s_first[place] = e;
    }
    __syncthreads();
    if (wave == 0) {
        const int n = found < k ? found : k;
        const unsigned long long e = lane < n ? s_first[lane] : 0ull;
        const float p = lane < n ? __uint_as_float((uint32_t)(e >> 32) & 0x7fffffffu) : 0.f;     // (a probability's sign bit is 0)
        const int id = (int)~(uint32_t)(e & 0xffffffffull);
        int len = n;
        bool ended = n == k;                                // the list ends within the candidates
        float filtered = 0.f;
        for (int i = 0; i < n; ++i) {
            filtered += lane_value(p, i);
            if (tp < 1.0f && filtered >= tp) { len = i + 1; ended = true; break; }
        }
        if (mp > 0.0f) {
            const float least = lane_value(p, 0) * mp;
            const unsigned long long under = __ballot(lane < len && !(p >= least));
            const int cut = under ? __ffsll((long long)under) - 1 : len;
            // (tokens that are no candidates are under the floor: a threshold above it leaves them out)
            if (cut > 0) ended = ended || cut < len || least >= NARROW_FLOOR;
            if (cut > 0 && cut < len) {
                len = cut;
                filtered = 0.f;
                for (int i = 0; i < len; ++i) filtered += lane_value(p, i);
            }
        }
        const float norm = p / filtered;
        float rng = u;
        int at = -1;
        for (int i = 0; i < len; ++i) {
            const float step = lane_value(norm, i);
            if (rng < step) { at = i; break; }
            rng -= step;
        }
        // (a list that ends before its k-th token only for want of candidates goes on in tokens under the floor)
        bool settled = filtered > 0.f && (at >= 0 || ended);
        if (at < 0) at = len - 1;
        const int shown = want_top < SAMPLE_MAX_TOP ? want_top : SAMPLE_MAX_TOP;
        settled = settled && lane_value(p, at) >= NARROW_FLOOR;
        if (shown > 0) settled = settled && (len >= shown || ended) && lane_value(p, (shown < len ? shown : len) - 1) >= NARROW_FLOOR;
        if (settled) {
            if (want_top >= 0) {
                if (lane < shown && lane < len) {
                    lp_ids[(size_t)rowi * SAMPLE_MAX_TOP + lane] = id;
                    lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP) + 1 + lane] = p > 0.f ? logf(norm) : -INFINITY;
                }
                if (lane == at) lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP)] = p > 0.f ? logf(norm) : -INFINITY;
            }
            if (lane == at) out[rowi] = id;
            if (lane == 0) s_settled = 1;
        }
    }
    __syncthreads();
    return s_settled != 0;
}

// n_top (may be null): per row -1 = no log-probabilities, else how many of the list's first entries are
// reported besides the drawn token's (sampler.rs:285-352).  lp_out [rows, 1 + SAMPLE_MAX_TOP]: the drawn
// token's log-probability within the kept list, then the entries'; lp_ids [rows, SAMPLE_MAX_TOP]: their ids (-1: none).
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    int* __restrict__ out, const float* __restrict__ logits, uint32_t* __restrict__ workspace, const RowLayout l,
    const RowParams params, const float* __restrict__ u, float* __restrict__ lp_out, int* __restrict__ lp_ids, const Penalties pen,
    int fast_top_k, int narrow_only) {
    __shared__ float scratch[32];
    __shared__ int s_counts[SAMPLE_THREADS];
    __shared__ float sv[16];
    __shared__ int si[16];
    const int rowi = blockIdx.x;
    const int vocab = l.vocab;
    const float* row = logits + (size_t)rowi * vocab;
    const int want_top = params.n_top != nullptr ? params.n_top[rowi] : -1;
    if (want_top >= 0 && threadIdx.x < SAMPLE_MAX_TOP) {
        lp_ids[(size_t)rowi * SAMPLE_MAX_TOP + threadIdx.x] = -1;
        lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP) + 1 + threadIdx.x] = -INFINITY;
    }
    uint32_t* keys = l.keys(workspace, rowi);
    float* probs = l.probs(workspace, rowi);
    __shared__ int s_win[PENALTY_STAGED];
    // The row's logits with its bias and penalties, in the keys' place.
    auto touched_row = [&]() {
        float* z = (float*)keys;
        stage_window(pen, rowi, s_win);
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) z[c] = row[c];
        __syncthreads();
        if (pen.any()) penalize_range(z, 0, vocab, pen, rowi, s_win);
        return z;
    };
    // (all of a row's parameters are asked for at once: one after the other each is a trip to the memory)
    const int k = params.top_k[rowi];
    const float tp = params.top_p[rowi], mp = params.min_p[rowi], draw = u[rowi];
    const bool narrow = row_is_narrow(params, pen, rowi, vocab, fast_top_k);
    float temp;
    if (!row_temperature(params.temperature, params.n_top, rowi, temp)) {
        int touched = 0;
        for (int i = threadIdx.x; i < pen.w; i += blockDim.x) touched |= pen.window[(size_t)rowi * pen.w + i] >= 0;
        for (int i = threadIdx.x; i < pen.nb; i += blockDim.x) touched |= pen.bias_ids[(size_t)rowi * pen.nb + i] >= 0;
        argmax_row(__syncthreads_or(touched) ? touched_row() : row, vocab, sv, si, out + rowi);
        return;
    }
    if (narrow && sample_narrow(out, l, workspace, rowi, k, tp, mp, draw, want_top, lp_out, lp_ids)) return;
    const bool listed = !narrow && !narrow_only;            // the second pass has been over the row
    __syncthreads();
    const RowSums rs = row_sums(l, workspace, rowi, listed);
    const float sum = rs.sum;
    float total = rs.total;                                 // the weight of the whole list
    if (!listed) {
        // what the second pass leaves, by this block alone
        const float* z = touched_row();
        total = 0.f;
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) {
            const float e = expf(z[c] / temp - rs.mx);
            const float pr = sum > 0.f ? e / sum : e;
            probs[c] = pr;
            keys[c] = order_key(pr);
            total += pr;
        }
        total = block_sum(total, scratch);
        __syncthreads();
    }

    const int picked = picked_out(k, vocab, fast_top_k);
    if (picked > 0) {
        // the list's first entries: the row's top_k, or, without one, 1,024 tokens, which hold the nucleus, the min_p
        // cut or the walk's end for all but flat distributions
        const bool open = !(k > 0 && k < vocab);
        // (few candidates are read from shared memory: the choice among them reads them several times)
        __shared__ uint32_t s_cand[SAMPLE_STAGED];
        const int n_cand = listed ? l.candidates(picked) : vocab;
        const uint32_t* cand_keys = listed ? l.cand_keys(workspace, rowi) : keys;
        if (n_cand <= SAMPLE_STAGED) {
            for (int i = threadIdx.x; i < n_cand; i += blockDim.x) s_cand[i] = cand_keys[i];
            __syncthreads();
            cand_keys = s_cand;
        }
        if (sample_top_k(out, cand_keys, listed ? l.cand_tokens(workspace, rowi) : nullptr, probs, n_cand, rowi,
                         picked, open, total, tp, mp, draw, want_top, lp_out, lp_ids, s_counts))
            return;
    }
    // how long the kept prefix is (sampler.rs:256-283)
    int keep = vocab;
    if (k > 0 && k < keep) keep = k;
    if (tp < 1.0f) {
        const Prefix p = shortest_prefix(keys, probs, vocab, tp, false, false, scratch);
        const int n = p.above + p.take;
        if (n < keep) keep = n;
    }
    if (mp > 0.0f) {
        const float thr = (sum > 0.f ? 1.0f / sum : 1.0f) * mp;       // the largest probability is exp(0) / sum
        float n = 0.f;
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) n += probs[c] >= thr ? 1.0f : 0.0f;
        const int cnt = (int)block_sum(n, scratch);
        if (cnt > 0 && cnt < keep) keep = cnt;
    }

    // the kept prefix by key and tie count, and its weight (sampler.rs:286-292)
    Prefix kept;
    float filtered;
    if (keep < vocab) {
        kept = shortest_prefix(keys, probs, vocab, (float)keep, true, false, scratch);
        float wa = 0.f;
        float pk = 0.f, seen = 0.f;
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) {
            if (keys[c] > kept.key) wa += probs[c];
            else if (keys[c] == kept.key) { pk = probs[c]; seen = 1.f; }
        }
        wa = block_sum(wa, scratch);
        __shared__ float s_pk2;
        if (threadIdx.x == 0) s_pk2 = 0.f;
        __syncthreads();
        if (seen > 0.f) s_pk2 = pk;
        __syncthreads();
        filtered = wa + (float)kept.take * s_pk2;
    } else {
        kept.key = 0u; kept.above = 0; kept.ties = 0; kept.take = 0;
        filtered = total;
    }

    // the walk (sampler.rs:323-335): the first place where the running sum of p / filtered exceeds u
    int token;
    if (!(filtered > 0.f)) {
        argmax_row(pen.any() ? touched_row() : row, vocab, sv, si, out + rowi);
        if (want_top >= 0 && threadIdx.x == 0) lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP)] = -INFINITY;
        return;
    }
    const Prefix hit = shortest_prefix(keys, probs, vocab, draw * filtered, false, true, scratch);
    if (keep < vocab && (hit.ties == 0 || hit.above + hit.take > keep)) {
        token = nth_with_key(keys, vocab, kept.key, kept.take, s_counts);          // the last kept token
    } else if (hit.ties == 0) {
        // u * filtered is not exceeded even by the whole list (rounding): the last of the list,
        // that is the last token with the smallest key
        uint32_t lowest = 0xffffffffu;
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) lowest = keys[c] < lowest ? keys[c] : lowest;
#pragma unroll
        for (int o = IA_WAVE / 2; o > 0; o >>= 1) {
            const uint32_t other = (uint32_t)__shfl_xor((int)lowest, o, IA_WAVE);
            lowest = other < lowest ? other : lowest;
        }
        __syncthreads();
        if ((threadIdx.x & (IA_WAVE - 1)) == 0) si[threadIdx.x / IA_WAVE] = (int)lowest;
        __syncthreads();
        for (int w = 0; w < SAMPLE_THREADS / IA_WAVE; ++w) lowest = (uint32_t)si[w] < lowest ? (uint32_t)si[w] : lowest;
        float n = 0.f;
        for (int c = threadIdx.x; c < vocab; c += blockDim.x) n += keys[c] == lowest ? 1.0f : 0.0f;
        token = nth_with_key(keys, vocab, lowest, (int)block_sum(n, scratch), s_counts);
    } else {
        token = nth_with_key(keys, vocab, hit.key, hit.take, s_counts);
    }
    if (threadIdx.x == 0) out[rowi] = token;
    if (want_top < 0) return;
    // log-probabilities within the kept list: the drawn token's, then the list's first entries
    if (threadIdx.x == 0) {
        const float pt = probs[token];
        lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP)] = pt > 0.f ? logf(pt / filtered) : -INFINITY;
    }
    const int n_list = keep < vocab ? keep : vocab;
    uint32_t prev_key = 0xffffffffu;
    int prev_idx = -1;
    uint32_t* s_key = (uint32_t*)scratch;
    for (int i = 0; i < want_top && i < SAMPLE_MAX_TOP && i < n_list; ++i) {
        const int idx = next_in_order(keys, vocab, prev_key, prev_idx, s_key, si);
        if (idx < 0) break;
        if (threadIdx.x == 0) {
            const float pi = probs[idx];
            lp_ids[(size_t)rowi * SAMPLE_MAX_TOP + i] = idx;
            lp_out[(size_t)rowi * (1 + SAMPLE_MAX_TOP) + 1 + i] = pi > 0.f ? logf(pi / filtered) : -INFINITY;
        }
        prev_key = keys[idx];
        prev_idx = idx;
    }
}

// Words of workspace for `rows` rows (see the layout of a row above).
extern "C" long long ia_sample_workspace(int rows, int vocab) {
    return vocab > 0 && rows > 0 ? (long long)rows * row_layout(vocab).words : 0;
}

static int g_sample_fast = 1;
// Measurement and test switch: 0 sends rows with a top_k through the bisections as well, 2 narrow ones the way of other rows
// with a top_k.
extern "C" void ia_sample_tune(int fast_top_k) { g_sample_fast = fast_top_k; }

extern "C" int ia_sample_max_top(void) { return SAMPLE_MAX_TOP; }
extern "C" int ia_sample_narrow_top(void) { return SAMPLE_NARROW_K; }
// Whether a row with these parameters needs no second pass (n_top: as in ia_sample; biased: it has a logit bias).
extern "C" int ia_sample_is_narrow(int top_k, int vocab, float temperature, float top_p, float min_p, int n_top, int biased) {
    return is_narrow(top_k, vocab, temperature, top_p, min_p, n_top, biased != 0);
}

// n_top, lp_out, lp_ids: all null, or all given (see sample_kernel).  window .. nb: bias and penalties as in ia_penalize
// (w = nb = 0: none), on the way; the logits stay as they are.  `narrow_only`: the caller knows that every row is a narrow one
// (ia_sample_is_narrow) or a greedy one, so that the second pass has nothing to do (a row of another kind is still drawn rightly, by
// one block).
extern "C" int ia_sample(int* out, const float* logits, void* workspace, int rows, int vocab,
                         const float* temperature, const int* top_k, const float* top_p, const float* min_p,
                         const float* u, const int* n_top, float* lp_out, int* lp_ids, const int* window, int w,
                         const float* rep, const float* freq, const float* pres, const int* bias_ids, const float* bias_vals,
                         int nb, int narrow_only, hipStream_t stream) {
    IA_CHECK(rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", rows, vocab);
    IA_CHECK(workspace != nullptr || rows == 0, "sample: needs a workspace of ia_sample_workspace(rows, vocab) words");
    IA_CHECK((n_top == nullptr) == (lp_out == nullptr) && (n_top == nullptr) == (lp_ids == nullptr),
             "sample: the arrays of the log-probabilities come together");
    IA_CHECK(rows <= 65535, "sample: at most 65535 rows a call, not %d", rows);
    IA_CHECK(vocab <= SAMPLE_STRETCH * SAMPLE_MAX_STRETCHES, "sample: at most %d tokens a row, not %d", SAMPLE_STRETCH * SAMPLE_MAX_STRETCHES, vocab);
    const Penalties pen = {window, w, rep, freq, pres, bias_ids, bias_vals, nb};
    if (const int bad = check_penalties("sample", pen)) return bad;
    if (rows == 0) return 0;
    const RowLayout l = row_layout(vocab);
    const dim3 grid((unsigned)l.stretches, (unsigned)rows);
    const int fast = g_sample_fast;
    const RowParams params = {temperature, top_k, top_p, min_p, n_top};
    sample_partials_kernel<<<grid, 256, 0, stream>>>(logits, (uint32_t*)workspace, l, params, pen, fast);
    if (fast != 1) narrow_only = 0;
    if (!narrow_only)
        sample_stretch_kernel<<<grid, STRETCH_THREADS, 0, stream>>>(logits, (uint32_t*)workspace, l, params, pen, fast);
    sample_kernel<<<rows, SAMPLE_THREADS, 0, stream>>>(out, logits, (uint32_t*)workspace, l, params, u, lp_out, lp_ids, pen, fast,
                                                       narrow_only);
    IA_LAUNCH_CHECK("sample");
    return 0;
}
