// Standalone row / elementwise operators of the forward graph, as the
// reference dispatches them (its variants rmsnorm_*, rope_*, geglu,
// add_scaled).  Each is built for f16 activations (the reference's storage:
// read f16, compute in f32 as the shaders do, round the result to f16) and
// for fp32 activations (the model driver's type).  The decode driver fuses
// these into its row kernels instead; these serve the dispatch surface and
// the prefill driver (many rows per launch, latency-bound, one pass over HBM).
#include "sgq_internal.h"

namespace sgq {
namespace {

constexpr int kNormWG = 256;

// gelu_tanh as x·sigmoid(2u), u = sqrt(2/pi)·(x + 0.044715x³): the same
// function (tanh(u) = 2·sigmoid(2u) - 1) from one exp2 and one IEEE division,
// about a third of the library tanh's instructions, and without its
// cancellation at negative x.
__device__ __forceinline__ float gelu_tanh_f(float x) {
    const float k = 0.7978845608028654f;  // (2/pi)^0.5
    const float u = k * (x + 0.044715f * x * x * x);
    return x / (1.f + __builtin_amdgcn_exp2f(u * (-2.0f * 1.44269504088896341f)));
}

// 16 bytes of activations: 4 fp32 or 8 f16.
template <typename T>
constexpr int kVec = 16 / sizeof(T);
__device__ __forceinline__ void ldv(const float *p, uint64_t i, float (&v)[4]) {
    const float4 t = reinterpret_cast<const float4 *>(p)[i];
    v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
}
__device__ __forceinline__ void ldv(const uint16_t *p, uint64_t i, float (&v)[8]) {
    const uint4 t = reinterpret_cast<const uint4 *>(p)[i];
    const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int e = 0; e < 4; e++)
        v[2 * e] = f16_bits_to_f32(w[e] & 0xffffu), v[2 * e + 1] = f16_bits_to_f32(w[e] >> 16);
}
__device__ __forceinline__ void stv(float *p, uint64_t i, const float (&v)[4]) {
    reinterpret_cast<float4 *>(p)[i] = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void stv(uint16_t *p, uint64_t i, const float (&v)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        w[e] = (uint32_t)f32_to_f16_bits(v[2 * e]) | (uint32_t)f32_to_f16_bits(v[2 * e + 1]) << 16;
    reinterpret_cast<uint4 *>(p)[i] = make_uint4(w[0], w[1], w[2], w[3]);
}
__device__ __forceinline__ void st4(float *p, uint64_t j, float4 v) {
    reinterpret_cast<float4 *>(p)[j] = v;
}
__device__ __forceinline__ void st4(uint16_t *p, uint64_t j, float4 v) {
    reinterpret_cast<uint2 *>(p)[j] =
        make_uint2((uint32_t)f32_to_f16_bits(v.x) | (uint32_t)f32_to_f16_bits(v.y) << 16,
                   (uint32_t)f32_to_f16_bits(v.z) | (uint32_t)f32_to_f16_bits(v.w) << 16);
}

__device__ __forceinline__ float4 norm_weight4(const float *w, int j, int plus_one) {
    if (!w) return make_float4(1.f, 1.f, 1.f, 1.f);
    float4 t = reinterpret_cast<const float4 *>(w)[j];
    if (plus_one) t.x = 1.f + t.x, t.y = 1.f + t.y, t.z = 1.f + t.z, t.w = 1.f + t.w;
    return t;
}
// The vector norms sum in f64 (as fast as f32 on this chip), so that the
// factor is the f64 one rounded once, whatever the order of the sum.
__device__ __forceinline__ double sumsq(float4 a) {
    const double x = a.x, y = a.y, z = a.z, w = a.w;
    return x * x + y * y + (z * z + w * w);
}
__device__ __forceinline__ float norm_factor(double ss, int n, float eps) {
    return (float)(1.0 / sqrt(ss / (double)n + (double)eps));
}

// rmsnorm.wgsl:24-61: y = x·rsqrt(mean(x²)+eps)·w (or ·(1+w)); fixed-order
// reductions (deterministic).  Three forms by row length:
// * whole rows in registers, one workgroup per row (quads of 4, NV per
//   thread, loaded in one round trip with the weights behind them);
// * rows of at most 512: a wave (half a wave up to 128) per row, no LDS;
// * anything else (odd lengths, misaligned pointers, very long rows): strided
//   scalar loads, the row read twice.
template <typename T, int WG, int NV>
__global__ __launch_bounds__(WG) void rmsnorm_quads_kernel(const T *__restrict__ x,
                                                           const float *__restrict__ w,
                                                           T *__restrict__ y, int n4, int plus_one,
                                                           float eps) {
    __shared__ double red[WG / kWave];
    const int t = threadIdx.x;
    const T *xr = x + (size_t)blockIdx.x * n4 * 4;
    T *yr = y + (size_t)blockIdx.x * n4 * 4;
    float4 v[NV], wt[NV];
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * WG < n4) v[i] = act_ld4(xr, t + i * WG);
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * WG < n4) wt[i] = norm_weight4(w, t + i * WG, plus_one);
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * WG < n4) ss += sumsq(v[i]);
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int i = 0; i < WG / kWave; i++) tot += red[i];
    const float inv = norm_factor(tot, n4 * 4, eps);
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * WG < n4)
            st4(yr, t + i * WG,
                make_float4(v[i].x * inv * wt[i].x, v[i].y * inv * wt[i].y, v[i].z * inv * wt[i].z,
                            v[i].w * inv * wt[i].w));
}

// LPR lanes per row, NV quads per lane (row_len <= 4·LPR·NV).
template <typename T, int LPR, int NV>
__global__ __launch_bounds__(256) void rmsnorm_short_kernel(const T *__restrict__ x,
                                                            const float *__restrict__ w,
                                                            T *__restrict__ y, uint32_t rows, int n4,
                                                            int plus_one, float eps) {
    const uint32_t row = blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
    const int t = threadIdx.x % LPR;
    if (row >= rows) return;  // whole LPR groups
    const T *xr = x + (size_t)row * n4 * 4;
    T *yr = y + (size_t)row * n4 * 4;
    float4 v[NV];
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * LPR < n4) {
            v[i] = act_ld4(xr, t + i * LPR);
            ss += sumsq(v[i]);
        }
    for (int o = LPR / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
    const float inv = norm_factor(ss, n4 * 4, eps);
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (t + i * LPR < n4) {
            const float4 wt = norm_weight4(w, t + i * LPR, plus_one);
            st4(yr, t + i * LPR,
                make_float4(v[i].x * inv * wt.x, v[i].y * inv * wt.y, v[i].z * inv * wt.z,
                            v[i].w * inv * wt.w));
        }
}

template <typename T>
__global__ __launch_bounds__(kNormWG) void rmsnorm_rows_kernel(const T *__restrict__ x,
                                                               const float *__restrict__ w,
                                                               T *__restrict__ y, int row_len,
                                                               int plus_one, float eps) {
    __shared__ float red[kNormWG / kWave];
    const T *xr = x + (size_t)blockIdx.x * row_len;
    T *yr = y + (size_t)blockIdx.x * row_len;
    const int t = threadIdx.x;
    float ss = 0.f;
    for (int i = t; i < row_len; i += kNormWG) {
        const float v = act_ld(xr, i);
        ss += v * v;
    }
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < kNormWG / kWave; i++) tot += red[i];
    const float inv = 1.0f / sqrtf(tot / (float)row_len + eps);
    for (int i = t; i < row_len; i += kNormWG) {
        const float wt = w ? (plus_one ? 1.f + w[i] : w[i]) : 1.f;
        act_st(yr, i, act_ld(xr, i) * inv * wt);
    }
}

// rope.wgsl:35-52: NEOX pairing over the whole head (pair i couples dims
// i and i + head_dim/2); only the first rot_dims/2 pairs rotate; table
// cos_sin[token × rot_dims/2] of (cos, sin); rows [token × n_heads × head_dim].
// Four adjacent pairs per thread (rot_dims % 8 == 0, aligned rows): 777 x 32
// heads of 256, fp32, 12.0 -> 10.4 us.
template <typename T>
__global__ __launch_bounds__(256) void rope4_kernel(T *__restrict__ xs, const float4 *__restrict__ cs,
                                                    uint32_t head4, uint32_t rot4, uint32_t n_heads,
                                                    uint32_t items) {
    const uint32_t g = blockIdx.x * 256 + threadIdx.x;
    if (g >= items) return;
    const uint32_t row = g / rot4, p = g - row * rot4, token = row / n_heads;
    const float4 c0 = cs[((size_t)token * rot4 + p) * 2], c1 = cs[((size_t)token * rot4 + p) * 2 + 1];
    const size_t ia = (size_t)row * head4 + p, ib = ia + head4 / 2;
    const float4 a = act_ld4(xs, ia), b = act_ld4(xs, ib);
    st4(xs, ia, make_float4(a.x * c0.x - b.x * c0.y, a.y * c0.z - b.y * c0.w,
                            a.z * c1.x - b.z * c1.y, a.w * c1.z - b.w * c1.w));
    st4(xs, ib, make_float4(b.x * c0.x + a.x * c0.y, b.y * c0.z + a.y * c0.w,
                            b.z * c1.x + a.z * c1.y, b.w * c1.z + a.w * c1.w));
}

template <typename T>
__global__ __launch_bounds__(256) void rope_kernel(T *__restrict__ xs, const float2 *__restrict__ cs,
                                                   int head_dim, int half_rot, int n_heads,
                                                   uint64_t pairs) {
    const uint64_t g = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= pairs) return;
    const uint64_t row = g / half_rot;
    const int pair = (int)(g % half_rot);
    const uint64_t token = row / n_heads;
    const float2 c = cs[token * half_rot + pair];
    T *base = xs + row * head_dim;
    const float a = act_ld(base, pair), b = act_ld(base, pair + head_dim / 2);
    act_st(base, pair, a * c.x - b * c.y);
    act_st(base, pair + head_dim / 2, b * c.x + a * c.y);
}

// geglu.wgsl:14-24 / add_scaled.wgsl:21-27: elementwise streams, 16 bytes per
// thread and operand (777 x 21504 GeGLU, fp32: 55 -> 30 us, 6.6 TB/s; 777 x
// 5376 add 12.2 -> 9.4 us); VEC = false: one element per thread (misaligned
// operands).  The n % kVec elements of the end go to the last workgroup's
// first threads.
struct GegluOp {
    __device__ float operator()(float g, float u, float) const { return gelu_tanh_f(g) * u; }
};
struct AddScaledOp {
    __device__ float operator()(float a, float b, float s) const { return (a + b) * s; }
};
template <typename T, typename Op, bool VEC>
__global__ __launch_bounds__(256) void binary_kernel(const T *__restrict__ a, const T *__restrict__ b,
                                                     T *__restrict__ y, uint64_t n, float s) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const Op op;
    if (!VEC) {
        if (i < n) act_st(y, i, op(act_ld(a, i), act_ld(b, i), s));
        return;
    }
    constexpr int V = kVec<T>;
    const uint64_t nv = n / V;
    if (i < nv) {
        float va[V], vb[V];
        ldv(a, i, va);
        ldv(b, i, vb);
#pragma unroll
        for (int e = 0; e < V; e++) va[e] = op(va[e], vb[e], s);
        stv(y, i, va);
    }
    const uint64_t tail = nv * V + threadIdx.x;
    if (blockIdx.x + 1 == gridDim.x && tail < n)
        act_st(y, tail, op(act_ld(a, tail), act_ld(b, tail), s));
}

uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + 255) / 256); }

bool aligned_to(size_t bytes, const void *a, const void *b, const void *c = nullptr) {
    return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & (bytes - 1)) == 0;
}

// Which norm: rows of whole quads on quad-aligned pointers stay in registers.
// Up to 512 values a wave holds the row (24864 rows of 256, fp32: 23.2 -> 11.4
// us); longer ones take 1024 threads while the rows are few and a row's round
// trip is the time (1 row of 5376 and 32 of 256, f16: 11.1 -> 5.0 us together),
// 256 with more quads each once the rows fill the chip (777 rows of 5376: 23.2
// -> 7.7 us).
template <typename T>
int rmsnorm_t(hipStream_t st, const T *x, const float *w, T *y, uint32_t rows, uint32_t row_len,
              int plus_one, float eps) {
    SGQ_CHECK(rows > 0 && rows < (1u << 31) && row_len > 0, "rmsnorm: %u rows of %u", rows, row_len);
    const bool quads = row_len % 4 == 0 && aligned_to(4 * sizeof(T), x, y) && aligned_to(16, w, w);
    const int n4 = (int)(row_len / 4);
    if (quads && n4 <= 32)
        hipLaunchKernelGGL((rmsnorm_short_kernel<T, 32, 1>), dim3((rows + 7) / 8), dim3(256), 0, st,
                           x, w, y, rows, n4, plus_one, eps);
    else if (quads && n4 <= 64)
        hipLaunchKernelGGL((rmsnorm_short_kernel<T, 64, 1>), dim3((rows + 3) / 4), dim3(256), 0, st,
                           x, w, y, rows, n4, plus_one, eps);
    else if (quads && n4 <= 128)
        hipLaunchKernelGGL((rmsnorm_short_kernel<T, 64, 2>), dim3((rows + 3) / 4), dim3(256), 0, st,
                           x, w, y, rows, n4, plus_one, eps);
    else if (quads && rows <= 512 && n4 <= 2 * 1024)
        hipLaunchKernelGGL((rmsnorm_quads_kernel<T, 1024, 2>), dim3(rows), dim3(1024), 0, st, x, w,
                           y, n4, plus_one, eps);
    else if (quads && n4 <= 6 * 256)
        hipLaunchKernelGGL((rmsnorm_quads_kernel<T, 256, 6>), dim3(rows), dim3(256), 0, st, x, w, y,
                           n4, plus_one, eps);
    else
        hipLaunchKernelGGL(rmsnorm_rows_kernel<T>, dim3(rows), dim3(kNormWG), 0, st, x, w, y,
                           (int)row_len, plus_one, eps);
    SGQ_HIP(hipGetLastError());
    return SGQ_OK;
}

template <typename T>
int rope_t(hipStream_t st, T *xs, const float *cos_sin, uint64_t rows, uint32_t head_dim,
           uint32_t rot_dims, uint32_t n_heads) {
    SGQ_CHECK(head_dim > 0 && head_dim % 2 == 0 && rot_dims % 2 == 0 && rot_dims <= head_dim &&
                  rot_dims > 0 && n_heads > 0,
              "rope: head_dim %u, rot_dims %u, n_heads %u", head_dim, rot_dims, n_heads);
    const uint64_t pairs = rows * (rot_dims / 2);
    if (!pairs) return SGQ_OK;
    SGQ_CHECK(pairs / 256 < (1u << 31), "rope: too many rows");
    if (head_dim % 8 == 0 && rot_dims % 8 == 0 && pairs < (1ull << 32) &&
        aligned_to(4 * sizeof(T), xs, xs) && aligned_to(16, cos_sin, cos_sin))
        hipLaunchKernelGGL(rope4_kernel<T>, dim3(blocks_for(pairs / 4)), dim3(256), 0, st, xs,
                           reinterpret_cast<const float4 *>(cos_sin), head_dim / 4, rot_dims / 8,
                           n_heads, (uint32_t)(pairs / 4));
    else
        hipLaunchKernelGGL(rope_kernel<T>, dim3(blocks_for(pairs)), dim3(256), 0, st, xs,
                           reinterpret_cast<const float2 *>(cos_sin), (int)head_dim,
                           (int)(rot_dims / 2), (int)n_heads, pairs);
    SGQ_HIP(hipGetLastError());
    return SGQ_OK;
}

template <typename T, typename Op>
int binary_t(hipStream_t st, const T *a, const T *b, T *y, uint64_t n, float s) {
    if (aligned_to(16, a, b, y))
        hipLaunchKernelGGL((binary_kernel<T, Op, true>),
                           dim3(blocks_for(n < (uint64_t)kVec<T> ? 1 : n / kVec<T>)), dim3(256), 0,
                           st, a, b, y, n, s);
    else
        hipLaunchKernelGGL((binary_kernel<T, Op, false>), dim3(blocks_for(n)), dim3(256), 0, st, a,
                           b, y, n, s);
    SGQ_HIP(hipGetLastError());
    return SGQ_OK;
}

template <typename T>
int geglu_t(hipStream_t st, const T *g, const T *u, T *y, uint64_t n) {
    if (!n) return SGQ_OK;
    SGQ_CHECK(n / 256 < (1u << 31), "geglu: n too large");
    return binary_t<T, GegluOp>(st, g, u, y, n, 0.f);
}

template <typename T>
int add_scaled_t(hipStream_t st, const T *a, const T *b, T *y, uint64_t n, float s) {
    if (!n) return SGQ_OK;
    SGQ_CHECK(n / 256 < (1u << 31), "add_scaled: n too large");
    return binary_t<T, AddScaledOp>(st, a, b, y, n, s);
}

}  // namespace

int launch_rmsnorm(hipStream_t st, const float *x, const float *w, float *y, uint32_t rows,
                   uint32_t row_len, int plus_one, float eps) {
    return rmsnorm_t(st, x, w, y, rows, row_len, plus_one, eps);
}
int launch_rmsnorm(hipStream_t st, const uint16_t *x, const float *w, uint16_t *y, uint32_t rows,
                   uint32_t row_len, int plus_one, float eps) {
    return rmsnorm_t(st, x, w, y, rows, row_len, plus_one, eps);
}
int launch_rope(hipStream_t st, float *xs, const float *cos_sin, uint64_t rows, uint32_t head_dim,
                uint32_t rot_dims, uint32_t n_heads) {
    return rope_t(st, xs, cos_sin, rows, head_dim, rot_dims, n_heads);
}
int launch_rope(hipStream_t st, uint16_t *xs, const float *cos_sin, uint64_t rows,
                uint32_t head_dim, uint32_t rot_dims, uint32_t n_heads) {
    return rope_t(st, xs, cos_sin, rows, head_dim, rot_dims, n_heads);
}
int launch_geglu(hipStream_t st, const float *g, const float *u, float *y, uint64_t n) {
    return geglu_t(st, g, u, y, n);
}
int launch_geglu(hipStream_t st, const uint16_t *g, const uint16_t *u, uint16_t *y, uint64_t n) {
    return geglu_t(st, g, u, y, n);
}
int launch_add_scaled(hipStream_t st, const float *a, const float *b, float *y, uint64_t n,
                      float s) {
    return add_scaled_t(st, a, b, y, n, s);
}
int launch_add_scaled(hipStream_t st, const uint16_t *a, const uint16_t *b, uint16_t *y,
                      uint64_t n, float s) {
    return add_scaled_t(st, a, b, y, n, s);
}

}  // namespace sgq
