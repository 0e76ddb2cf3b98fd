// Products of the true 32-bit path for more rows than a decode step has: out[M, N] = x[M, K] . w[N, K]^T on the matrix
// cores' 32-bit instruction (v_mfma_f32_16x16x4_f32: 32-bit operands, 32-bit sums).  The instruction adds its four
// products to the accumulator one after the other, a fused multiply-add each, so that with k ascending every output is
// the same chain of fused multiply-adds as in gemm.hip's kernels on the vector units, and has their bits: a row's result
// does not depend on how many rows a step has (tests/test_kernels_gpu.py compares the bits).
//
// What bounds it: the matrix pipes, 157 TFLOP/s, which is twice what the vector units give without packed instructions.
// Measured, us, the vector units' kernels of 128 x 128 tiles before: 555 rows and the products of an 8B shape, gate|up 1,567 ->
// 917 (122 TFLOP/s), down 1,400 -> 556, q|k|v 703 -> 262, output -> 188; a prompt of 555 tokens and four layers 22.6 ms -> 9.8.
// A block of four waves owns 16 MT rows of x by 64 NR rows of w, a wave 16 NR of them for all of the block's rows: each
// value that it reads from shared memory meets NR or MT instructions of 32 cycles.  Chunks of 32 k lie in shared memory
// twice, the next chunk on its way from memory through registers while this one is multiplied, one barrier a chunk.  Few rows
// and features make blocks that are alone on their compute units and multiply a chunk in less time than memory takes to
// answer: those walk k in chunks of 64 or 128.
// Rows are padded by 16 bytes: a read takes four neighbouring k of 16 rows, which then fall on different banks.
#include "common.h"
#include "api.h"

typedef float gf_f32x4 __attribute__((ext_vector_type(4)));

template <int MT, int NR, int GF_K>
__global__ __launch_bounds__(256) void gemm_f32_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                       const float* __restrict__ w, int M, int N, int K, int tiles_m) {
    constexpr int GF_PITCH = GF_K + 4;      // floats of a staged row
    constexpr int BM = 16 * MT, BN = 64 * NR, ROWS = BM + BN;
    constexpr int PIECES = (ROWS * (GF_K / 4) + 255) / 256;     // 16-byte pieces of a chunk that a thread brings
    __shared__ __attribute__((aligned(16))) float sh[2][ROWS * GF_PITCH];
    // Blocks go round the eight dies in turn and each die has an L2 of its own: a die takes a contiguous range of tiles,
    // rows of x fastest, so that the blocks which run together on a die share tiles of both operands.
    const int blocks = gridDim.x, die = blockIdx.x & 7;
    const int tile = die * (blocks >> 3) + min(die, blocks & 7) + (blockIdx.x >> 3);
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    const float* from[PIECES];
    int to[PIECES], kk[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int p = min(tid + 256 * i, ROWS * (GF_K / 4) - 1);        // (the last pieces may be brought twice)
        const int row = p / (GF_K / 4);
        kk[i] = p % (GF_K / 4) * 4;
        to[i] = row * GF_PITCH + kk[i];
        const float* base = row < BM ? x + (size_t)min(m0 + row, M - 1) * K             // (rows beyond the matrices are
                                     : w + (size_t)min(n0 + row - BM, N - 1) * K;       // never stored)
        from[i] = base + kk[i];
    }
    float4 piece[PIECES];
    auto fetch = [&](int k0) {
        if (k0 + GF_K <= K) {
#pragma unroll
            for (int i = 0; i < PIECES; ++i) piece[i] = *(const float4*)(from[i] + k0);
        } else {
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
                piece[i] = k0 + kk[i] < K ? *(const float4*)(from[i] + k0) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) *(float4*)(&sh[buf][to[i]]) = piece[i];
    };

    gf_f32x4 acc[NR][MT];
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = (gf_f32x4){0.f, 0.f, 0.f, 0.f};
    const int r = lane & 15, g = lane >> 4;
    const int x_at = r * GF_PITCH + g, w_at = (BM + wave * 16 * NR + r) * GF_PITCH + g;

    // Step j of a chunk is multiplied while the operands of step j + 1 are read.  The chunk after this one goes into the other
    // buffer behind step GF_K / 4 - 4, so that the writes are done when the barrier comes, ahead of the last step: all of
    // this buffer has been read by then (the last step's operands are in registers), and the first operands of the next
    // chunk come in while the last step is multiplied.
    constexpr int STEPS = GF_K / 4;
    float wf[2][NR], xf[2][MT];
    auto read = [&](const float* s, int j, int half) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < NR; ++a) wf[half][a] = s[w_at + a * 16 * GF_PITCH + 4 * j];
#pragma unroll
        for (int b = 0; b < MT; ++b) xf[half][b] = s[x_at + b * 16 * GF_PITCH + 4 * j];
    };
    auto multiply = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MT; ++b)
#pragma unroll
            for (int a = 0; a < NR; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[half][a], xf[half][b], acc[a][b], 0, 0, 0);
    };
    fetch(0);
    put(0);
    __syncthreads();
    read(sh[0], 0, 0);
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += GF_K, buf ^= 1) {
        fetch(k0 + GF_K < K ? k0 + GF_K : k0);          // (past the end: the last chunk again, which nobody multiplies)
        const float* s = sh[buf];
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            if (j + 1 < STEPS) read(s, j + 1, (j + 1) & 1);
            if (j == STEPS - 3) put(buf ^ 1);
            if (j + 1 == STEPS) {
                __syncthreads();
                read(sh[buf ^ 1], 0, 0);
            }
            // (the compiler sinks the reads behind the step's products to save registers; a step of one instruction in a wave
            // that is alone on its SIMD is then the reads' latency: 4,096 x 4,096, 64 rows 48.0 -> 37.2 us.  Larger tiles, and several
            // blocks a unit, lose 2 to 6 % by it, and by a second chunk on its way 5 to 15 %: there neither the shared memory's
            // latency nor the memory's sets the pace.)
            if constexpr (MT * NR == 1 && GF_K == 128) __builtin_amdgcn_sched_barrier(0);
            multiply(j & 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // a lane holds features 4 g .. + 4 of row r of every tile
    const bool vec = (N & 3) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
        const int m = m0 + 16 * b + r;
        if (m >= M) continue;
#pragma unroll
        for (int a = 0; a < NR; ++a) {
            const int n = n0 + (wave * NR + a) * 16 + 4 * g;
            float* o = out + (size_t)m * N + n;
            if (vec && n < N) *(gf_f32x4*)o = acc[a][b];
            else
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) o[i] = acc[a][b][i];
        }
    }
}

template <int MT, int NR>
static void gf_launch(float* out, const float* x, const float* w, int M, int N, int K, int cus, hipStream_t stream) {
    constexpr int LONG = MT * NR <= 3 ? 128 : MT * NR <= 6 ? 64 : 32;
    const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 64 * NR - 1) / (64 * NR), blocks = tiles_m * tiles_n;
    // (4,096 x 4,096 at 17 to 64 rows, chunks of 32 against 128: 69 -> 44 us; 24,576 features at 64 rows, where several blocks
    // share a compute unit and long chunks leave room for one only: 146 against 241)
    if (blocks <= cus) gemm_f32_kernel<MT, NR, LONG><<<blocks, 256, 0, stream>>>(out, x, w, M, N, K, tiles_m);
    else gemm_f32_kernel<MT, NR, 32><<<blocks, 256, 0, stream>>>(out, x, w, M, N, K, tiles_m);
}

static int g_f32_shape = 0;             // 0: by the rule below; else 10 * (16 rows of x) + (64 rows of w), forced (measurements and tests)
extern "C" int ia_gemm_f32_tune(int shape) {
    IA_CHECK(shape == 0 || (shape / 10 >= 1 && shape / 10 <= 10 && shape % 10 >= 1 && shape % 10 <= 2),
             "gemm_f32_tune: no kernel of %d x %d rows a block", shape / 10 * 16, shape % 10 * 64);
    g_f32_shape = shape;
    return 0;
}

// x and w 16-byte aligned, K a multiple of 4.
extern "C" int ia_gemm_f32(void* out, const void* x, const void* w, int M, int N, int K, hipStream_t stream) {
    IA_CHECK(M > 0 && N > 0 && K > 0 && K % 4 == 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
    IA_CHECK((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "gemm_f32: x and w must be 16-byte aligned");
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        cus = hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    }
    // A compute unit's time is what its blocks multiply one after the other or side by side: full turns of the compute units
    // times the instructions a block has for a step of four k, and a little a turn; a block that is alone on its unit waits for
    // memory besides (32 rows, 4,096 features: 1 x 1 tiles 36 us, 2 x 1 60, 3 x 1 77, 4 x 1 95; 100 rows: 1 x 1 tiles in two turns 73, 2 x 1 in one 63).  Measured at 555 rows and 4,096 features:
    // 9 x 1 tiles in one turn 192 us, 5 x 1 in two 191, 3 x 1 in three 188, 10 x 1 in one 204; at 24,576 features 9 x 2 in three
    // turns 918, 7 x 2 in four 942, 9 x 1 in six 969; 130 rows and 24,576 features: 5 x 1 in three turns 297, 3 x 2 in three 330.
    int best_m = 8, best_n = 2;
    double best = 1e30;
    for (int nr = 1; nr <= 2; ++nr)
        for (int mt = 10; mt >= 1; --mt) {
            const long long blocks = (long long)((M + 16 * mt - 1) / (16 * mt)) * ((N + 64 * nr - 1) / (64 * nr));
            const double work = mt * nr;
            // (two turns of the smallest blocks are no cheaper than two blocks alone)
            const long long turns = (blocks + cus - 1) / cus;
            const double alone = mt * nr == 1 ? 1.65 : 0.65 * work + 1.55 > 1.03 * work ? 0.65 * work + 1.55 : 1.03 * work;
            const double cost = turns == 1 ? alone : (double)turns * (work + (mt * nr == 1 && turns == 2 ? 0.5 : 0.3));
            if (cost < best && blocks < (1LL << 31)) best = cost, best_m = mt, best_n = nr;
        }
    if (g_f32_shape) best_m = g_f32_shape / 10, best_n = g_f32_shape % 10;
    const long long blocks = (long long)((M + 16LL * best_m - 1) / (16 * best_m)) * ((N + 64LL * best_n - 1) / (64 * best_n));
    IA_CHECK(blocks < (1LL << 31), "gemm_f32: %d rows by %d features are %lld blocks, too many for one launch", M, N, blocks);
    float* o = (float*)out;
    const float *xi = (const float*)x, *wi = (const float*)w;
    switch (best_m * 10 + best_n) {
#define GF_CASE(MT) \
    case MT * 10 + 1: gf_launch<MT, 1>(o, xi, wi, M, N, K, cus, stream); break; \
    case MT * 10 + 2: gf_launch<MT, 2>(o, xi, wi, M, N, K, cus, stream); break;
    GF_CASE(1) GF_CASE(2) GF_CASE(3) GF_CASE(4) GF_CASE(5) GF_CASE(6) GF_CASE(7) GF_CASE(8) GF_CASE(9) GF_CASE(10)
#undef GF_CASE
    }
    IA_LAUNCH_CHECK("gemm_f32");
    return 0;
}
