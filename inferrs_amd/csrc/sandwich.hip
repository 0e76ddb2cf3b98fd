// A residual stream kept in 32-bit whose sub-layers stand between two norms:
//     x <- x + rmsnorm(y) * w_post,      y = s1 * y1 (+ s2 * y2)      (the sub-layer's output, or two outputs side by side; eps_post)
//     x <- x + e_rows + e_vec                                         (optional: a row and a vector that enter the stream here)
//     h  = rmsnorm(x) * w_pre                                         (the next sub-layer's input, in its products' precision)
// ONE kernel does what stands between two sub-layers; every half may be absent.  A block owns a row; sums of squares,
// the stream and its sums are 32-bit.  With `rows` the kernel reads the named rows only and writes nothing back to the
// stream (the model's end: the wanted rows through the final norm).
#include "api.h"
#include "common.h"
#include "activation.h"

template <typename TY, typename TH>
__global__ __launch_bounds__(1024) void sandwich_step_kernel(
    float* __restrict__ x, const TY* __restrict__ y1, float s1, const TY* __restrict__ y2, float s2,
    const float* __restrict__ w_post, const TY* __restrict__ e_rows, const float* __restrict__ e_vec,
    const float* __restrict__ w_pre, float eps_post, float eps, TH* __restrict__ h, const int* __restrict__ rows, int W) {
    extern __shared__ float sw_row[];            // [W]
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const int row = rows != nullptr ? rows[r] : r;
    float* xr = x + (long long)row * W;
    float rs = 0.f;
    if (y1 != nullptr) {
        float sq = 0.f;
        for (int c = threadIdx.x; c < W; c += blockDim.x) {
            float v = s1 * ld(y1 + (long long)row * W + c);
            if (y2 != nullptr) v = fmaf(s2, ld(y2 + (long long)row * W + c), v);
            sw_row[c] = v;
            sq = fmaf(v, v, sq);
        }
        rs = 1.0f / sqrtf(block_sum(sq, scratch) / (float)W + eps_post);
    }
    float sq = 0.f;
    for (int c = threadIdx.x; c < W; c += blockDim.x) {
        float v = xr[c];
        if (y1 != nullptr) v += sw_row[c] * rs * w_post[c];
        if (e_rows != nullptr) v += ld(e_rows + (long long)row * W + c);
        if (e_vec != nullptr) v += e_vec[c];
        if (rows == nullptr && (y1 != nullptr || e_rows != nullptr || e_vec != nullptr)) xr[c] = v;
        sw_row[c] = v;
        sq = fmaf(v, v, sq);
    }
    if (h == nullptr) return;
    const float rs2 = 1.0f / sqrtf(block_sum(sq, scratch) / (float)W + eps);
    for (int c = threadIdx.x; c < W; c += blockDim.x)
        st(h + (long long)r * W + c, sw_row[c] * rs2 * (w_pre != nullptr ? w_pre[c] : 1.f));
}

// The same for widths of a multiple of eight: a thread owns eight neighbouring features, which stay in registers between the two
// norms, and moves them 16 bytes at a time.  Bound by the memory: 14 bytes a feature for a bfloat16 output and rows (1,500 rows of
// 2,048: 17.0 -> 9.8 us; one feature a thread asked for 2 and 4 bytes at a time and read the row back from shared memory twice).
__device__ __forceinline__ void sw_load8(const float* p, float (&v)[8]) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void sw_load8(const bf16_t* p, float (&v)[8]) {
    const uint4 q = *(const uint4*)p;
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = __uint_as_float(w[j] << 16);
        v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
}
__device__ __forceinline__ void sw_store8(float* p, const float (&v)[8]) {
    *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void sw_store8(bf16_t* p, const float (&v)[8]) {
    *(uint4*)p = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
}

template <typename TY, typename TH>
__global__ __launch_bounds__(1024) void sandwich_step8_kernel(
    float* __restrict__ x, const TY* __restrict__ y1, float s1, const TY* __restrict__ y2, float s2,
    const float* __restrict__ w_post, const TY* __restrict__ e_rows, const float* __restrict__ e_vec,
    const float* __restrict__ w_pre, float eps_post, float eps, TH* __restrict__ h, const int* __restrict__ rows, int W) {
    __shared__ float scratch[16];
    const int r = blockIdx.x, c = threadIdx.x * 8;
    const bool in = c < W;
    const int row = rows != nullptr ? rows[r] : r;
    const long long at = (long long)row * W + c;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, t[8];
    if (in) sw_load8(x + at, v);
    if (y1 != nullptr) {
        float sq = 0.f;
        if (in) {
            sw_load8(y1 + at, y);
            if (y2 != nullptr) sw_load8(y2 + at, t);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                y[j] *= s1;
                if (y2 != nullptr) y[j] = fmaf(s2, t[j], y[j]);
                sq = fmaf(y[j], y[j], sq);
            }
        }
        const float rs = 1.0f / sqrtf(block_sum(sq, scratch) / (float)W + eps_post);
        if (in) {
            sw_load8(w_post + c, t);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += y[j] * rs * t[j];
        }
    }
    float sq = 0.f;
    if (in) {
        if (e_rows != nullptr) {
            sw_load8(e_rows + at, t);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += t[j];
        }
        if (e_vec != nullptr) {
            sw_load8(e_vec + c, t);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += t[j];
        }
        if (rows == nullptr && (y1 != nullptr || e_rows != nullptr || e_vec != nullptr)) sw_store8(x + at, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) sq = fmaf(v[j], v[j], sq);
    }
    if (h == nullptr) return;
    const float rs2 = 1.0f / sqrtf(block_sum(sq, scratch) / (float)W + eps);
    if (!in) return;
    if (w_pre != nullptr) sw_load8(w_pre + c, t);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = v[j] * rs2 * (w_pre != nullptr ? t[j] : 1.f);
    sw_store8(h + (long long)r * W + c, v);
}

// y_dtype: precision of y1, y2 and e_rows; h_dtype: of h.  0 float32, 1 bfloat16.
extern "C" int ia_sandwich_step(float* x, const void* y1, float s1, const void* y2, float s2, const float* w_post,
                                const void* e_rows, const float* e_vec, const float* w_pre, float eps_post, float eps, void* h,
                                const int* rows, int n, int W, int y_dtype, int h_dtype, hipStream_t stream) {
    IA_CHECK(n >= 0 && W > 0, "sandwich_step: n=%d width=%d", n, W);
    IA_CHECK((size_t)W * sizeof(float) <= 60 * 1024, "sandwich_step: width %d does not fit shared memory", W);
    IA_CHECK(y1 != nullptr || y2 == nullptr, "sandwich_step: a second output goes with a first");
    IA_CHECK(y1 == nullptr || w_post != nullptr, "sandwich_step: an output to add needs the weight of the norm behind it");
    if (n == 0) return 0;
    if (W % 8 == 0 && W <= 8192 && (((uintptr_t)x | (uintptr_t)y1 | (uintptr_t)y2 | (uintptr_t)w_post | (uintptr_t)e_rows |
                                     (uintptr_t)e_vec | (uintptr_t)w_pre | (uintptr_t)h) & 15) == 0) {
        const int threads8 = (W / 8 + IA_WAVE - 1) / IA_WAVE * IA_WAVE;
#define IA_LAUNCH8(TY, TH)                                                                                        \
    sandwich_step8_kernel<TY, TH><<<n, threads8, 0, stream>>>(x, (const TY*)y1, s1, (const TY*)y2, s2, w_post,      \
                                                              (const TY*)e_rows, e_vec, w_pre, eps_post, eps, (TH*)h, rows, W)
        if (y_dtype == IA_F32 && h_dtype == IA_F32) { IA_LAUNCH8(float, float); }
        else if (y_dtype == IA_F32) { IA_LAUNCH8(float, bf16_t); }
        else if (h_dtype == IA_F32) { IA_LAUNCH8(bf16_t, float); }
        else { IA_LAUNCH8(bf16_t, bf16_t); }
#undef IA_LAUNCH8
        IA_LAUNCH_CHECK("sandwich_step");
        return 0;
    }
    const int threads = W >= 4096 ? 1024 : W >= 1024 ? 512 : 256;
    const size_t shm = (size_t)W * sizeof(float);
#define IA_LAUNCH(TY, TH)                                                                                         \
    sandwich_step_kernel<TY, TH><<<n, threads, shm, stream>>>(x, (const TY*)y1, s1, (const TY*)y2, s2, w_post,      \
                                                              (const TY*)e_rows, e_vec, w_pre, eps_post, eps, (TH*)h, rows, W)
    if (y_dtype == IA_F32 && h_dtype == IA_F32) { IA_LAUNCH(float, float); }
    else if (y_dtype == IA_F32) { IA_LAUNCH(float, bf16_t); }
    else if (h_dtype == IA_F32) { IA_LAUNCH(bf16_t, float); }
    else { IA_LAUNCH(bf16_t, bf16_t); }
#undef IA_LAUNCH
    IA_LAUNCH_CHECK("sandwich_step");
    return 0;
}

// An activation over every element, in place.  act: 1 SiLU, 2 GELU in its tanh form, 3 the exact GELU,
// z / 2 * (1 + erf(z / sqrt 2)).
template <typename T>
__global__ void activation_kernel(T* __restrict__ x, long long n, int act) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float z = ld(x + i);
    st(x + i, act_stored<T>(z, act));
}

// Eight neighbouring bfloat16 values a thread (16-byte accesses), for arrays of a multiple of eight elements.  GELU, 1,500 rows of 8,192: 14.2 -> 11.8 us (4.2 TB/s).
template <int ACT>
__global__ void activation8_kernel(bf16_t* __restrict__ x, long long n8) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    uint4 q = *reinterpret_cast<const uint4*>(x + 8 * i);
    uint32_t* w = reinterpret_cast<uint32_t*>(&q);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        w[e] = pack_bf16x2(act_stored<bf16_t>(__uint_as_float(w[e] << 16), ACT), act_stored<bf16_t>(__uint_as_float(w[e] & 0xffff0000u), ACT));
    *reinterpret_cast<uint4*>(x + 8 * i) = q;
}

extern "C" int ia_activation(void* x, long long n, int act, int dtype, hipStream_t stream) {
    IA_CHECK(n >= 0 && act >= 1 && act <= 3, "activation: n=%lld act=%d (1 SiLU, 2 GELU tanh, 3 GELU)", n, act);
    if (n == 0) return 0;
    if (dtype != IA_F32 && n % 8 == 0 && ((uintptr_t)x & 15) == 0) {
        const unsigned grid = (unsigned)((n / 8 + 255) / 256);
        if (act == 1) activation8_kernel<1><<<grid, 256, 0, stream>>>((bf16_t*)x, n / 8);
        else if (act == 2) activation8_kernel<2><<<grid, 256, 0, stream>>>((bf16_t*)x, n / 8);
        else activation8_kernel<3><<<grid, 256, 0, stream>>>((bf16_t*)x, n / 8);
        IA_LAUNCH_CHECK("activation");
        return 0;
    }
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (dtype == IA_F32) activation_kernel<float><<<blocks, 256, 0, stream>>>((float*)x, n, act);
    else activation_kernel<bf16_t><<<blocks, 256, 0, stream>>>((bf16_t*)x, n, act);
    IA_LAUNCH_CHECK("activation");
    return 0;
}
