// bfloat16 products for steps of more rows than gemm_mid.hip takes (portions of prompts, several short prompts together):
// out[M, N] = x[M, K] . w[N, K]^T, or with an activation act(x . gate^T) * (x . up^T) for w = [gate; up].
//
// The reference hands these products to cuBLAS like all others (`candle-core/src/cuda_backend/mod.rs:2260-2305`).
//
// What bounds it: the matrix pipes, once every compute unit has a share.  A few hundred rows are a few tiles of rows only,
// and the weights of an output projection or of a feed-forward's second product a few tiles of features: k is split between
// blocks until there is one for every unit, and the splits' 32-bit sums, [splits][M][N], are added up in their order by
// whoever reads them (gemm_mid.hip's readers: the kernel that adds a product to the residual stream and norms it, or
// ia_sum_partials).  A block's rows of x come in steps of 16, so that 521 rows do not pay for 768 (gw_plan below).
//
// A block of four waves, one a SIMD, owns 16 MT rows of x by 256 rows of w (or 192: ia_gemm_wide_narrow_fits) and a range of k.  A wave multiplies 64 of the
// rows of w (four MFMA A-operands, v_mfma_f32_16x16x32_bf16) with all of the block's rows of x: MT + 4 operand reads from
// shared memory for 4 MT products.  Stages of 64 k (whole lines of 128 bytes a row: a load of 1 KiB takes the compute unit's
// address unit 18 cycles, in rows of 64 bytes 37) go from memory straight into shared memory (global_load_lds), two places
// for x, which the step has just written and comes from a cache, and three for w, which comes from memory: at 128 rows a
// stage is multiplied in 0.6 us when its operands lie in the die's L2, and in 0.85 when w comes from memory.  The walk is
// laid out so that the matrix pipe does not wait for an operand that was asked for just before:
//   * the operands of a step (32 k) are read while the step before it is multiplied, two reads beside each of its first
//     groups of four products, across stages too;
//   * the one barrier of a stage stands between its two steps: there every wave has read all of the stage (its places are
//     free from here on) and has seen its own loads of the next stage arrive;
//   * a stage's loads go out one beside a group: four waves that issue theirs in a row stand still until the address unit
//     has taken them.
// Shared memory: piece c (16 bytes) of row r lies at place c ^ ((r >> 1) & 7) of its row's 128 bytes, so that the rows which
// one operand read takes at the same k fall on different banks.
//
// Measured in captured graphs (us, the vendor's GEMM and the kernel behind it / this one and its reader; 8B and 14B shapes): down at
// 200 rows 54 / 42 and 230 / 64, at 456 88 / 59 and 173 / 87, at 521 109 / 66 and 184 / 93, at 1,024 132 / 103 and 257 / 160, at 2,048
// 196 / 184 and 301 / 300; output projection at 256 28 / 25 and 56 / 33, at 1,024 51 / 48 and 76 / 67; gate|up with the activation, 8B
// shape, at 320 81 / 77, at 700 165 / 135, 14B shape at 900 404 / 300.  A stage's rate over a long k is 1,270 to 1,340 TFLOP/s with
// 160 to 240 rows a block and 1,140 with 256, at the chip's power limit (with operands of zeros a stage takes a fifth less).
// Tiles that are shared along k between all compute units, each an equal share of the stages, were slower at every size (gate|up of the 14B
// shape at 521 rows 209 -> 289): the blocks of a die are then at different places of k and of w, and share nothing in its L2.
#include <type_traits>
#include <utility>

#include "common.h"
#include "api.h"
#include "activation.h"

typedef __bf16 gw_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gw_f32x4 __attribute__((ext_vector_type(4)));

#define GW_BN 256                            // rows of w of a block at most
#define GW_NARROW_MT 21                      // tiles of 16 rows of x of a block of 192 rows of w, at most (its stages fill the shared memory)
#define GW_STAGE_K 64                        // k of a stage: two steps of the matrix instruction
#define GW_ROW 128                           // bytes of a staged row

struct GemmWideParams {
    void* out;
    const bf16_t* x;
    const bf16_t* w;
    int M, N, K;                             // N: output features (with the activation inside, w has 2 N rows)
    int act;
    int tiles_m, tiles_n, stages;            // stages: of a split (the last split may have fewer)
};

// 16 bytes a lane from memory straight into shared memory, 1 KiB a wave in lane order from `lds_at` on (the same for all
// lanes), from `base` (the same for all lanes) + `off`.  Written out so that the compiler does not wait for it at every read
// of shared memory: the waits stand in the code (loads come back in the order they were asked for).
__device__ __forceinline__ void gw_load16(const char* base, uint32_t off, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds_at) : "memory");
}

// s_waitcnt with vmcnt(n) and lgkmcnt(0) (gfx9 encoding: vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8, expcnt left alone)
#define GW_WAIT(n) (((n) & 15) | ((((n) >> 4) & 3) << 14) | (7 << 4))

template <int... I, typename Fn>
__device__ __forceinline__ void gw_unrolled(std::integer_sequence<int, I...>, Fn fn) {
    (fn(std::integral_constant<int, I>()), ...);
}

enum { GW_BF16 = 0, GW_F32 = 1, GW_DUAL = 2 };          // what leaves the kernel; GW_F32: a split's sums

// NA: tiles of 16 rows of w that a wave owns, 4 or (with the activation inside) 3.
template <int MT, int OUT, int NA = 4>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_wide_kernel(const GemmWideParams p) {
    constexpr bool DUAL = OUT == GW_DUAL;
    constexpr int BM = 16 * MT;
    constexpr int BN = 64 * NA;                              // rows of w of a block
    constexpr int XL = (MT + 1) / 2, WL = 2 * NA;               // a wave's loads of 1 KiB (8 rows) for a stage's rows of x and of w
    constexpr int W1 = MT - XL < WL ? MT - XL : WL;          // (an odd MT: the last ones of x fetch a row again into a place nobody reads)
    constexpr uint32_t X_STAGE = XL * 4 * 1024, W_STAGE = WL * 4 * 1024, W_AT = 2 * X_STAGE;
    static_assert(2 * X_STAGE + 3 * W_STAGE <= 160 * 1024, "the stages fit a compute unit's shared memory");
    static_assert(WL - W1 <= MT, "a group has room for a load");
    static_assert(NA == 4 || (NA == 3 && DUAL), "blocks of 192 rows of w are those of the activation inside");
    constexpr int FEATS = DUAL ? BN / 2 : BN;                // output features of a block
    __shared__ __attribute__((aligned(1024))) char lds[2 * X_STAGE + 3 * W_STAGE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;

    // Blocks go round the eight dies in turn, and each die has an L2 of its own: a die takes a contiguous range of the
    // blocks of one range of k, rows of x fastest, so that the blocks which run together on a die share both operands.
    const int blocks = gridDim.x, die = blockIdx.x & 7;
    const int id = die * (blocks >> 3) + min(die, blocks & 7) + (blockIdx.x >> 3);
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = id / tiles, tile = id - split * tiles;
    const int m0 = (tile % p.tiles_m) * BM, n0 = (tile / p.tiles_m) * FEATS;
    const int k_first = split * p.stages * GW_STAGE_K;
    const int stages = min(p.stages, (p.K - k_first) / GW_STAGE_K);
    // (blocks of different features start at different places of their range of k: rows are a power of two apart, and blocks
    // that walk k in step ask the same memory channels at any moment)
    const int rot = (int)((unsigned)(tile / p.tiles_m) * 5u % (unsigned)stages);

    // ---- what this lane fetches: load i of the wave brings rows 8 (4 i + wave) .. + 8 of x, or of w
    const size_t pitch = (size_t)p.K * 2;
    const char* xbase = (const char*)p.x + (size_t)m0 * pitch + (size_t)k_first * 2;
    const char* wbase = (const char*)p.w + (size_t)n0 * pitch + (size_t)k_first * 2;
    uint32_t xoff[XL], woff[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int row = 8 * (4 * i + wave) + (lane >> 3);
        xoff[i] = (uint32_t)min(row, p.M - 1 - m0) * (uint32_t)pitch + ((lane & 7) ^ ((row >> 1) & 7)) * 16;     // (rows beyond the
    }                                                                                                   // matrices are never stored)
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int row = 8 * (4 * i + wave) + (lane >> 3);
        int at;
        if (DUAL) {
            // a tile's 16 rows: two of gate and the same two of up in turn, so that a lane's four sums are two pairs
            at = min((row >> 4) * 8 + ((row >> 2) & 3) * 2 + (row & 1), p.N - 1 - n0) + ((row >> 1) & 1) * p.N;
        } else {
            at = min(row, p.N - 1 - n0);
        }
        woff[i] = (uint32_t)at * (uint32_t)pitch + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
    // load i of stage kt of an operand into the place at `slot` (past the walk's end a stage is fetched again into a place that
    // nobody reads any more, so that the count of loads under way is the same at every stage)
    auto k_of = [&](int kt) __attribute__((always_inline)) {
        const int at = (kt < stages ? kt : stages - 1) + rot;
        return (size_t)(at < stages ? at : at - stages) * (GW_STAGE_K * 2);
    };
    auto fetch_x = [&](size_t k, uint32_t slot, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i >= 0 && i < XL) gw_load16(xbase + k, xoff[i], lds0 + slot + (uint32_t)(4 * i + wave) * 1024);
    };
    auto fetch_w = [&](size_t k, uint32_t slot, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i >= 0 && i < WL) gw_load16(wbase + k, woff[i], lds0 + W_AT + slot + (uint32_t)(4 * i + wave) * 1024);
    };

    gw_f32x4 acc[NA][MT];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = (gw_f32x4){0.f, 0.f, 0.f, 0.f};
    uint4 fw[2][NA], fx[2][MT];
    // the lane's place in a tile of 16 rows, for the two steps of a stage
    const uint32_t in_tile[2] = {(uint32_t)(r * GW_ROW + ((g ^ ((r >> 1) & 7)) * 16)),
                                 (uint32_t)(r * GW_ROW + (((4 + g) ^ ((r >> 1) & 7)) * 16))};
    const uint32_t w_rows = W_AT + (uint32_t)(16 * NA * wave) * GW_ROW;
    // read i of a step's MT + NA operands: the rows of w first
    auto read = [&](uint32_t xslot, uint32_t wslot, int step, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < NA) fw[step][i] = *(const uint4*)(lds + wslot + w_rows + in_tile[step] + i * 16 * GW_ROW);
        else if constexpr (i < MT + NA) fx[step][i - NA] = *(const uint4*)(lds + xslot + in_tile[step] + (i - NA) * 16 * GW_ROW);
    };
    // one step: `step`'s operands are multiplied, the other step's are read, two beside each of the first groups of NA
    // products, and `load(b)` asks for something beside group b
    auto multiply = [&](auto step_c, uint32_t xslot, uint32_t wslot, auto load) __attribute__((always_inline)) {
        constexpr int step = decltype(step_c)::value;
        gw_unrolled(std::make_integer_sequence<int, MT>(), [&](auto bc) __attribute__((always_inline)) {
            constexpr int b = decltype(bc)::value;
            read(xslot, wslot, 1 - step, std::integral_constant<int, 2 * b>());
            read(xslot, wslot, 1 - step, std::integral_constant<int, 2 * b + 1>());
            load(bc);
#pragma unroll
            for (int a = 0; a < NA; ++a)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gw_bf16x8, fw[step][a]),
                                                                    __builtin_bit_cast(gw_bf16x8, fx[step][b]), acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr auto all_x = std::make_integer_sequence<int, XL>();
    constexpr auto all_w = std::make_integer_sequence<int, WL>();
    // (in the order of the walk: x of a stage ahead of w of the stage behind it)
    gw_unrolled(all_w, [&](auto i) { fetch_w(k_of(0), 0, i); });
    gw_unrolled(all_x, [&](auto i) { fetch_x(k_of(0), 0, i); });
    gw_unrolled(all_w, [&](auto i) { fetch_w(k_of(1), W_STAGE, i); });
    gw_unrolled(all_x, [&](auto i) { fetch_x(k_of(1), X_STAGE, i); });
    {
        const size_t k = k_of(2);
        gw_unrolled(std::make_integer_sequence<int, W1>(), [&](auto i) { fetch_w(k, 2 * W_STAGE, i); });
    }
    __builtin_amdgcn_s_waitcnt(GW_WAIT(WL + XL + W1));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    uint32_t xs = 0, wh = 0, wn = W_STAGE, wl = 2 * W_STAGE;     // places: this stage's x; w of this stage, the next, the one behind it
    gw_unrolled(std::make_integer_sequence<int, MT + NA>(), [&](auto i) __attribute__((always_inline)) { read(0, 0, 0, i); });
    size_t k_w = k_of(2);
    for (int s = 0; s < stages; ++s) {
        // the stage's first step; the rest of w of stage s + 2 is asked for
        multiply(std::integral_constant<int, 0>(), xs, wh, [&](auto bc) __attribute__((always_inline)) {
            fetch_w(k_w, wl, std::integral_constant<int, decltype(bc)::value + W1>());
        });
        __builtin_amdgcn_s_waitcnt(GW_WAIT(WL));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        // its second step; x of stage s + 2 and then w of stage s + 3 go into this stage's places
        const size_t k_x = k_w;
        k_w = k_of(s + 3);
        multiply(std::integral_constant<int, 1>(), X_STAGE - xs, wn, [&](auto bc) __attribute__((always_inline)) {
            constexpr int b = decltype(bc)::value;
            if constexpr (b < XL) fetch_x(k_x, xs, bc);
            else if constexpr (b - XL < W1) fetch_w(k_w, wh, std::integral_constant<int, b - XL>());
        });
        xs = X_STAGE - xs;
        const uint32_t t = wh;
        wh = wn; wn = wl; wl = t;
    }
    // (without this the compiler carries half of the accumulators through copies, 3 moves for every two products)
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) asm volatile("" : "+a"(acc[a][b]));
    __builtin_amdgcn_s_waitcnt(GW_WAIT(0));                  // (nothing may still be on its way into shared memory at the end)

    // ---- results: the lane holds features 4 g .. + 4 of w tile a for row r of x tile b (N is a multiple of 4)
    if constexpr (OUT == GW_F32) {
        // A wave's 64 features, a share of its rows at a time, through shared memory of its own, so that a store writes 256 bytes to each of four
        // rows and not 64 to each of 16 (16 bytes behind each row, as below).  us a step, twelve layers of the 8B shape, 459 rows 3,033 -> 2,981; ten of
        // the 14B shape, 521 rows 4,918 -> 4,882.
        constexpr int PITCH = 64 * 4 + 16, ROUNDS = 4 * BM * PITCH <= (int)sizeof(lds) ? 1 : 2, EACH = (MT + ROUNDS - 1) / ROUNDS;
        static_assert(4 * EACH * 16 * PITCH <= (int)sizeof(lds), "the waves' rows fit the stages' places");
        char* const mine = lds + wave * (EACH * 16 * PITCH);
        const int n = n0 + wave * 64 + r * 4;
        float* const out = (float*)p.out + (size_t)split * p.M * p.N + n;
        __builtin_amdgcn_s_barrier();                        // (every wave has read its last operands, and no load is under way)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int round = 0; round < ROUNDS; ++round) {
#pragma unroll
            for (int b = round * EACH; b < (round + 1) * EACH && b < MT; ++b)
#pragma unroll
                for (int a = 0; a < 4; ++a) *(gw_f32x4*)(mine + ((b - round * EACH) * 16 + r) * PITCH + (a * 16 + 4 * g) * 4) = acc[a][b];
            // (the wave's own memory: its shared-memory operations run in program order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int first = m0 + round * EACH * 16, end = min(min(EACH * 16, BM - round * EACH * 16), p.M - first);
            if (n < p.N)
                for (int m = g; m < end; m += 4) *(gw_f32x4*)(out + (size_t)(first + m) * p.N) = *(const gw_f32x4*)(mine + m * PITCH + r * 16);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    } else {
        // The tile's rounded rows go through shared memory and out a row of the tile after the other, so that whole lines leave together: from
        // the accumulators a store writes 32 bytes to each of 16 rows (1,500 rows of 8,512 over k of 2,048 50.9 -> 47.4 us, 16,384 over 4,096
        // at 1,300 152 -> 147).  16 bytes behind each row, so that a lane's 16 rows fall on different banks.
        constexpr int PITCH = FEATS * 2 + 16;
        static_assert(BM * PITCH <= (int)sizeof(lds), "a tile's rows fit the stages' places");
        __builtin_amdgcn_s_barrier();                        // (every wave has read its last operands, and no load is under way)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int b = 0; b < MT; ++b) {
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                const gw_f32x4 v = acc[a][b];
                char* const at = lds + (b * 16 + r) * PITCH + (wave * (FEATS / 4) + (DUAL ? a * 8 + 2 * g : a * 16 + 4 * g)) * 2;
                if constexpr (DUAL) {
                    float z[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        // the products are rounded to the storage precision before the activation, as the two-kernel way rounds them
                        const uint32_t both = pack_bf16x2(v[i], v[2 + i]);
                        z[i] = gate_act(__uint_as_float(both << 16), p.act) * __uint_as_float(both & 0xffff0000u);
                    }
                    *(uint32_t*)at = pack_bf16x2(z[0], z[1]);
                } else {
                    *(uint2*)at = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                }
            }
        }
        __syncthreads();
        constexpr int LANES = FEATS / 4;                     // threads of a row, four features each
        const int at = threadIdx.x % LANES * 4, m_end = min(BM, p.M - m0);
        if (n0 + at >= p.N || threadIdx.x >= 256 / LANES * LANES) return;
        // an activation without a gate comes here, over the rounded values: unrolled over the accumulators the exact GELU would be 60 KB of code
        auto rows = [&](auto act_c) __attribute__((always_inline)) {
            constexpr int ACT = decltype(act_c)::value;
            for (int m = threadIdx.x / LANES; m < m_end; m += 256 / LANES) {
                uint2 q = *(const uint2*)(lds + m * PITCH + at * 2);
                if constexpr (ACT) {
                    q.x = pack_bf16x2(act_stored<bf16_t>(__uint_as_float(q.x << 16), ACT), act_stored<bf16_t>(__uint_as_float(q.x & 0xffff0000u), ACT));
                    q.y = pack_bf16x2(act_stored<bf16_t>(__uint_as_float(q.y << 16), ACT), act_stored<bf16_t>(__uint_as_float(q.y & 0xffff0000u), ACT));
                }
                *(uint2*)((bf16_t*)p.out + (size_t)(m0 + m) * p.N + n0 + at) = q;
            }
        };
        if (DUAL || p.act == 0) rows(std::integral_constant<int, 0>());
        else if constexpr (!DUAL) {
            if (p.act == 1) rows(std::integral_constant<int, 1>());
            else if (p.act == 2) rows(std::integral_constant<int, 2>());
            else rows(std::integral_constant<int, 3>());
        }
    }
}

// How a product is shared out: rows of x a block (16 mt), ways k is split, stages of a split.
struct WidePlan { int mt, splits, stages; double cost; int na; };
static WidePlan g_wide_forced = {0, 0, 0, 0.0, 4};
static int wide_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        cus = hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    }
    return cus;
}
// A stage of 64 k, measured with every compute unit at work, rows of 16 mt (us): the memory's latency up to 8, then the matrix
// pipes at the clock that the chip's power leaves them.
static const double gw_stage_us[11] = {0.83, 0.89, 0.93, 1.00, 1.05, 1.16, 1.20, 1.32, 1.41, 1.55, 1.89};
// Blocks of 192 rows of w: by what their stages took in products of one and two rounds, on the scale of the others.
static const double gw_narrow_us[16] = {0.75, 0.79, 0.82, 0.88, 0.95, 0.99, 1.08, 1.17, 1.24, 1.38, 1.43, 1.50, 1.57, 1.64, 1.76, 1.83};
static WidePlan gw_plan(int M, int N, int K, bool dual, bool may_split, bool may_narrow = true) {
    const int cus = wide_cus(), stages = K / GW_STAGE_K;
    WidePlan best = {0, 0, 0, 1e30, 4};
    for (int na = 4; na >= (dual && may_narrow ? 3 : 4); --na) {
        const int feats = 64 * na / (dual ? 2 : 1);
        const long long tiles_n = (N + feats - 1) / feats;
        for (int mt = 6; mt <= (na == 3 ? GW_NARROW_MT : 16); ++mt) {
            const long long tiles_m = (M + 16 * mt - 1) / (16 * mt);
            for (int splits = 1; splits <= (may_split && !dual ? 8 : 1); ++splits) {
                const int each = (stages + splits - 1) / splits;
                if (splits > 1 && each < 8) break;
                if ((splits - 1) * each >= stages) continue;
                const long long rounds = (tiles_m * tiles_n * splits + cus - 1) / cus;
                // in us: a block's stages, its start and its end, and the splits' sums on their way out and back in
                const double stage_us = na == 3 ? gw_narrow_us[mt - 6] : gw_stage_us[mt - 6];
                const double cost = (double)rounds * (each * stage_us + 3.0) + (splits > 1 ? 1.0 + 0.42e-6 * splits * M * N * 4.0 : 0.0);
                if (cost < best.cost) best = {mt, splits, each, cost, na};
            }
        }
    }
    return best;
}

// (a plan for measurements and tests: blocks of 16 mt rows, k split `splits` ways; mt + 32: those of 192 rows of w, for the activation
// inside; 0, 0: the plan's own)
extern "C" int ia_gemm_wide_plan(int mt, int splits) {
    const bool narrow = mt > 32;
    IA_CHECK((mt == 0 && splits == 0) || (mt >= 6 && mt <= 16 && splits >= 1 && splits <= 8) || (mt >= 38 && mt <= 32 + GW_NARROW_MT && splits == 1),
             "gemm_wide_plan: no blocks of %d rows with %d splits of k", 16 * mt, splits);
    g_wide_forced = {narrow ? mt - 32 : mt, splits, 0, 0.0, narrow ? 3 : 4};
    return 0;
}

static WidePlan wide_plan(int M, int N, int K, bool dual, bool may_split) {
    WidePlan p = gw_plan(M, N, K, dual, may_split);
    if (g_wide_forced.mt && (dual || g_wide_forced.na == 4)) {
        p.mt = g_wide_forced.mt;
        p.na = g_wide_forced.na;
        int splits = may_split && !dual ? g_wide_forced.splits : 1;
        const int stages = K / GW_STAGE_K;
        if (splits > stages) splits = stages;
        p.stages = (stages + splits - 1) / splits;
        p.splits = (stages + p.stages - 1) / p.stages;
    }
    return p;
}

// The ways k is split where the result may stay split (ia_gemm_wide_bf16 with out_mode 2).
extern "C" int ia_gemm_wide_splits(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4) return 0;
    return wide_plan(M, N, K, false, true).splits;
}

// The rules below say where this kernel goes ahead of the vendor's GEMM.  They were measured in whole steps: prompts of 130 to 2,048
// tokens of six dense shapes (width 1,024 to 5,120) replayed from graphs, with each product on either kernel, side by side in one
// process.  (A graph of the product and its reader alone is no measure: its operands lie in caches that a step's other kernels have
// turned over, and it put [gate; up] of the 8B shape at 176 to 360 rows on the wrong side by 2 to 3 % of the layer.)

// The share of full rounds of the compute units that blocks of 256 x 256, the vendor's largest, would make of a product.
static double vendor_fill(int M, int N) {
    const long long tiles = (long long)((M + 255) / 256) * ((N + 255) / 256), cus = wide_cus();
    return (double)tiles / (double)((tiles + cus - 1) / cus * cus);
}

// Whether a step of M rows of a stream of `width` features is one that the host bounds where it is met eagerly, as every length of a
// prompt is the first times: a call of the vendor's GEMM costs the host 14 us and one of this package's kernels 6.5, and these products
// take the GPU little more.  They stay here even where a replayed step would have the vendor's GEMM a little ahead.  us a layer, eager /
// replayed, the products by the rules for wide steps and by this one: 0.6B shape (width 1,024), 300 tokens 156 / 92 and 125 / 86,
// 512 tokens 155 / 97 and 105 / 100, 1.7B shape (2,048), 400 tokens 156 / 127 and 128 / 123, 640 tokens 158 / 149 and 149 / 146, 4B shape
// (2,560), 130 tokens 165 / 151 and 153 / 143.  Beyond it the GPU is the bound either way (1.7B shape, 1,024 tokens 191 / 186 and 197 /
// 195; 4B shape, 512 tokens 207 / 198 and 206 / 200).
static bool host_bound(int M, int width) { return width <= 2048 ? M < 1024 : width <= 3072 && (long long)M * width < (1LL << 20); }

// Whether a product whose result may stay split goes here instead of to the vendor's GEMM, for the reader that adds it to the
// residual stream and norms it.  The kernel gains by what the split gives, so it needs a long k and enough features; short products are
// a few microseconds of fixed costs and the sums' way out and back in on top (us a layer by the vendor's GEMM and by this one: 14B
// shape, down at 200 rows 534 / 366, at 521 625 / 541, o at 256 572 / 546; 1.7B shape, 1,024 rows, down 197 / 192, o 197 / 200).
// Unsplit: where the vendor's blocks leave a third of the chip empty (14B shape, down at 1,536 rows, 1,249 / 1,130).
extern "C" int ia_gemm_wide_norm_fits(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4) return 0;
    if (host_bound(M, N)) return 1;
    if (gw_plan(M, N, K, false, true).splits == 1) return K >= 8192 && vendor_fill(M, N) < 0.63;
    return K >= 4096 && N >= 1024 && (long long)K * (N < 3072 ? N : 3072) >= (M <= 192 ? 3072 : M <= 256 ? 2560 : 2048) * 4096LL;
}

// The same for the kernel that norms and turns queries and keys and writes the cache, up to 1,024 rows.  A product of q|k|v has many
// features, so that the split gives less than above: over a short k the vendor's GEMM is as fast or faster (us a layer: 4B shape, 456
// rows 241 / 244, 850 rows 332 / 336), over a long one this kernel, split or not (8B shape, 130 rows 251 / 236, 700 rows 436 / 420, 900
// 484 / 475; 14B shape, 521 rows 625 / 605; 32B shape, 900 rows 1,105 / 1,085; of 69 points three are slower, by up to 0.4 %).
extern "C" int ia_gemm_wide_rope_fits(int M, int N, int K) {
    if (M <= 0 || M > 1024 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4) return 0;
    return host_bound(M, K) || (K >= 4096 && (long long)N * K >= 4096LL * 5120);
}

// Whether a [gate; up] of N features each goes here instead of to the vendor's GEMM and the activation's kernel, up to 1,024 rows.  The
// product cannot be split.  This kernel's own time has to come within a tenth of 1.22 PFLOP/s (or of 4 TB/s over the operands) and what
// the second kernel takes; not where its blocks leave two fifths of their rounds empty (14B shape, 130 to 200 rows: 454 / 461, 468 / 474,
// 534 / 544 us a layer) nor where the vendor's are nearly all work (4B shape, 768 rows, 287 / 298).  Elsewhere 8B shape, 200 rows 250 /
// 243, 700 rows 436 / 412, 14B shape, 900 rows 934 / 831, 32B shape, 1,024 rows 1,222 / 1,167; of the 63 points of wide shapes where the
// rule says yes ten are slower by more than half a percent, 1.2 at most.  It still refuses some that would gain (14B shape, 580 rows
// 692 / 662, 32B shape, 400 rows 803 / 773).
// (Said of blocks of 256 rows of w; ia_gemm_wide_narrow_fits says where those of 192 do better than the vendor's.)
extern "C" int ia_gemm_wide_dual_fits(int M, int N, int K) {
    if (M <= 0 || M > 1024 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4 || ((long long)N + GW_BN) * K * 2 >= (1LL << 32)) return 0;
    const WidePlan plan = gw_plan(M, N, K, true, false, false);
    if (!host_bound(M, K)) {
        const long long cus = wide_cus(), tiles_m = (M + 16 * plan.mt - 1) / (16 * plan.mt), tiles_n = (N + GW_BN / 2 - 1) / (GW_BN / 2);
        const long long ours = (tiles_m * tiles_n + cus - 1) / cus * cus;                  // (blocks that this kernel's rounds have room for)
        const long long theirs = ((M + 255) / 256 * ((2LL * N + 255) / 256) + cus - 1) / cus * cus;
        if (N < 2048 || tiles_m * tiles_n < 0.6 * ours || 2.0 * M * N >= 0.85 * 65536.0 * theirs) return 0;
    }
    const double flops = 4.0 * M * N * K / 1.22e9, bytes = (2.0 * N + M) * K * 2.0 / 4.0e6;
    return plan.cost <= 1.1 * ((flops > bytes ? flops : bytes) + 8.0 + M * (double)N * 6.0 / 5.0e6);
}

// out_mode 0: out [M, N] bfloat16; 2: [splits][M][N] float with splits = ia_gemm_wide_splits(M, N, K).  dual (an activation,
// IA_ACT_*): w = [gate; up] of N rows each (mode 0 only).  K a multiple of 64, operands 16-byte aligned.
extern "C" int ia_gemm_wide_bf16(void* out, const void* x, const void* w, int M, int N, int K, int out_mode, int dual,
                                 hipStream_t stream) {
    IA_CHECK(M > 0 && N > 0 && K > 0 && K % GW_STAGE_K == 0 && N % 4 == 0, "gemm_wide: bad sizes M=%d N=%d K=%d (K a multiple of %d, N of 4)",
             M, N, K, GW_STAGE_K);
    IA_CHECK((out_mode == 0 || out_mode == 2) && (!dual || out_mode == 0), "gemm_wide: output mode %d%s", out_mode,
             dual ? " does not go with the activation inside" : " is unknown");
    IA_CHECK(dual >= 0 && dual <= IA_ACT_LAST, "gemm_wide: unknown activation %d", dual);
    IA_CHECK((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "gemm_wide: operands must be 16-byte aligned");
    // (a lane's offset from its block's first row is 32 bits wide)
    IA_CHECK(((dual ? (long long)N : 0) + GW_BN) * K * 2 < (1LL << 32), "gemm_wide: N=%d rows of K=%d are too far apart", N, K);
    const WidePlan plan = wide_plan(M, N, K, dual != 0, out_mode == 2);
    const int feats = 64 * plan.na / (dual ? 2 : 1);
    GemmWideParams p;
    p.out = out; p.x = (const bf16_t*)x; p.w = (const bf16_t*)w;
    p.M = M; p.N = N; p.K = K; p.act = dual;
    p.tiles_m = (M + 16 * plan.mt - 1) / (16 * plan.mt);
    p.tiles_n = (N + feats - 1) / feats;
    p.stages = plan.stages;
    const long long blocks = (long long)p.tiles_m * p.tiles_n * plan.splits;
    IA_CHECK(plan.mt >= 6 && plan.stages > 0 && blocks < (1LL << 31), "gemm_wide: %lld blocks", blocks);
    if (plan.na == 3) {
        switch (plan.mt) {
#define GW_CASE(MT) case MT: gemm_wide_kernel<MT, GW_DUAL, 3><<<(unsigned)blocks, 256, 0, stream>>>(p); break;
        GW_CASE(6) GW_CASE(7) GW_CASE(8) GW_CASE(9) GW_CASE(10) GW_CASE(11) GW_CASE(12) GW_CASE(13) GW_CASE(14) GW_CASE(15) GW_CASE(16)
        GW_CASE(17) GW_CASE(18) GW_CASE(19) GW_CASE(20) GW_CASE(21)
#undef GW_CASE
        }
        IA_LAUNCH_CHECK("gemm_wide");
        return 0;
    }
    switch (plan.mt) {
#define GW_CASE(MT) \
    case MT: if (dual) gemm_wide_kernel<MT, GW_DUAL><<<(unsigned)blocks, 256, 0, stream>>>(p); \
             else if (out_mode == 0) gemm_wide_kernel<MT, GW_BF16><<<(unsigned)blocks, 256, 0, stream>>>(p); \
             else gemm_wide_kernel<MT, GW_F32><<<(unsigned)blocks, 256, 0, stream>>>(p); break;
    GW_CASE(6) GW_CASE(7) GW_CASE(8) GW_CASE(9) GW_CASE(10) GW_CASE(11) GW_CASE(12) GW_CASE(13) GW_CASE(14) GW_CASE(15) GW_CASE(16)
#undef GW_CASE
    }
    IA_LAUNCH_CHECK("gemm_wide");
    return 0;
}

// out [M, N] = x . w^T in bfloat16 with an activation over the rounded result (1 SiLU, 2 GELU in its tanh form, 3 the exact GELU; 0 none),
// k never split.  K a multiple of 64, N of 4, operands 16-byte aligned.
extern "C" int ia_gemm_wide_rows_bf16(void* out, const void* x, const void* w, int M, int N, int K, int act, hipStream_t stream) {
    IA_CHECK(M > 0 && N > 0 && K > 0 && K % GW_STAGE_K == 0 && N % 4 == 0, "gemm_wide_rows: bad sizes M=%d N=%d K=%d (K a multiple of %d, N of 4)",
             M, N, K, GW_STAGE_K);
    IA_CHECK(act >= 0 && act <= 3, "gemm_wide_rows: unknown activation %d", act);
    IA_CHECK((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "gemm_wide_rows: operands must be 16-byte aligned");
    IA_CHECK((long long)GW_BN * K * 2 < (1LL << 32), "gemm_wide_rows: rows of K=%d are too far apart", K);
    const WidePlan plan = wide_plan(M, N, K, false, false);
    GemmWideParams p;
    p.out = out; p.x = (const bf16_t*)x; p.w = (const bf16_t*)w;
    p.M = M; p.N = N; p.K = K; p.act = act;
    p.tiles_m = (M + 16 * plan.mt - 1) / (16 * plan.mt);
    p.tiles_n = (N + GW_BN - 1) / GW_BN;
    p.stages = plan.stages;
    const long long blocks = (long long)p.tiles_m * p.tiles_n;
    IA_CHECK(plan.mt >= 6 && plan.stages > 0 && blocks < (1LL << 31), "gemm_wide_rows: %lld blocks", blocks);
    switch (plan.mt) {
#define GW_CASE(MT) case MT: gemm_wide_kernel<MT, GW_BF16><<<(unsigned)blocks, 256, 0, stream>>>(p); break;
    GW_CASE(6) GW_CASE(7) GW_CASE(8) GW_CASE(9) GW_CASE(10) GW_CASE(11) GW_CASE(12) GW_CASE(13) GW_CASE(14) GW_CASE(15) GW_CASE(16)
#undef GW_CASE
    }
    IA_LAUNCH_CHECK("gemm_wide_rows");
    return 0;
}

// What the vendor's GEMM takes for whole rows (us): a round of the chip with blocks of 256 x 256 at 1.49 us a stage where they fill it, less
// where smaller blocks share the work out, and at least 1.4 rounds beyond one.  Fitted to 150 sizes (150 to 2,048 rows, 2,064 to 16,928
// features, k 1,024 to 4,096, in graphs that walk more weights than the caches hold): within a tenth for the most part; with features that
// are no multiple of 256 the library is 1.0 to 1.7 times that slow.
static double vendor_rows_us(int M, int N, int K) {
    const double rounds = (double)((M + 255) / 256) * ((N + 255) / 256) / wide_cus();
    return (rounds <= 1.0 ? 0.38 + 0.6 * rounds : rounds > 1.4 ? rounds : 1.4) * (K / GW_STAGE_K * 1.49 + 3.0);
}

// Whether a product whose whole rows are wanted goes here instead of to the vendor's GEMM.  us, the vendor's / this: 8,512 features over 2,048,
// 600 rows 30.6 / 27.1, 1,500 54.3 / 47.4, 2,048 82 / 66; 4,304 over 1,024, 1,000 rows 18.3 / 13.5; 16,928 over 4,096, 1,300 rows 214 /
// 152; of features in whole blocks of 256 10,240 over 2,560, 800 rows 51.4 / 45.8.  Not where the library's blocks fill their
// rounds (8,192 over 2,048, 2,048 rows 50.9 / 61.3).  Features in whole blocks were measured again inside prompts of the six dense shapes, one product
// of a layer on either kernel (us a layer): above 1,024 rows 0.6B shape, 1,300 rows, q|k|v 133 / 127, 4B 1,400 rows 384 / 375, 8B 1,536 rows 628 / 617,
// 14B 1,800 rows 1,219 / 1,203; of 60 points 0.993 to 1.071, 1.010 in the mean.  Up to 1,024 rows a plan has to be ahead clearly, since both sides' times are
// known to a tenth (4B shape, q|k|v, 800 rows 255.4 / 260.5, 900 rows 289.7 / 293.3), and whole multiples of 1,024 rows, which the library's smaller blocks
// share out evenly, gain nothing (2,048 rows, o of the 8B shape 0.998 and 1.004, of the 4B shape 0.994 and 0.997).  (Two rounds of
// this kernel over a long k take 7 % longer than its stages add up to: 34,816 over 5,120 at 521 rows 187 / 205.)
extern "C" int ia_gemm_wide_rows_fits(int M, int N, int K) {
    if (M < 512 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4) return 0;
    if (N % 256 == 0 && M % 1024 == 0) return 0;
    const WidePlan plan = gw_plan(M, N, K, false, false);
    const bool one_round = (long long)((M + 16 * plan.mt - 1) / (16 * plan.mt)) * ((N + GW_BN - 1) / GW_BN) <= wide_cus();
    return plan.cost <= (N % 256 ? 1.2 : M <= 1024 ? 0.93 : one_round ? 1.02 : 0.95) * vendor_rows_us(M, N, K);
}

// The same with an activation, which costs this kernel a few microseconds at its end (four waves a unit form it: 8,192 features, 1,500 rows,
// exact GELU, 8) and the other way a kernel (11.4 there).  8,192 over 2,048, 1,500 rows 55.3 / 51.3, 1,000 43.7 / 38.3; 4,096 over 1,024,
// 2,048 rows 28.9 / 25.1; 16,384 over 4,096, 800 rows 106 / 91.
extern "C" int ia_gemm_wide_act_fits(int M, int N, int K) {
    if (M < 512 || N <= 0 || K <= 0 || K % GW_STAGE_K || N % 4) return 0;
    const double values = (double)M * N;
    return gw_plan(M, N, K, false, false).cost + 3.0 + values * 3.5e-7 <= vendor_rows_us(M, N, K) + 2.5 + values * 8e-7;
}

// Whether a [gate; up] of N features each goes here in blocks of 192 rows of w: widths of 3 x 2^i make whole rounds of them (12,288 features
// 128 tiles, so that two tiles of up to 336 rows of x are one block for every compute unit, where blocks of 256 x 256 leave a quarter of the chip idle or a
// second round nearly empty).  us with the activation, the vendor's / blocks of 256 / of 192: 12,288 over 4,096, 200 rows 66 / 65 / 57, 300 76 / 73 /
// 69, 459 95.6 / 101 / 97.9, 521 133 / 121 / 107, 600 133 / 127 / 117; 17,408 over 5,120, 150 rows 113 / 116 / 98.5, 260 159 / 165 / 122, 330 169 /
// 181 / 141; 6,144 over 2,048, 400 rows 36.6 / 32.2 / 30.3.
extern "C" int ia_gemm_wide_narrow_fits(int M, int N, int K) {
    if (M <= 0 || M > 1024 || N < 2048 || K <= 0 || K % GW_STAGE_K || N % 4 || ((long long)N + GW_BN) * K * 2 >= (1LL << 32)) return 0;
    const WidePlan plan = gw_plan(M, N, K, true, false);
    return plan.na == 3 && plan.cost <= 0.97 * (vendor_rows_us(M, 2 * N, K) + 2.5 + (double)M * N * 1.2e-6);
}
