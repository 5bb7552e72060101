// Fourier-layer surrogate of the collision operator: forward, backward,
// loss, Adam and the AoSoA gather / conservation-check / scatter kernels.
//
// The network (N^3 grid with N = 16 or 32, width 32, 8^3 retained modes,
// L layers):
//   v_0      = P g + p0                                 (lift, per point)
//   X_l(k)   = (1/n) sum_x v_l(x) e^{-2 pi i k.x/N}    (k_sur_dft, per channel)
//   Y_l(o,k) = sum_i X_l(i,k) R_l(i,o,k)               (k_sur_mix_lds, per mode)
//   s_l(x)   = Re sum_k Y_l(k) e^{+2 pi i k.x/N}        (k_sur_idft, per channel)
//   z_l      = Wm_l v_l + b_l + s_l,  v_{l+1} = gelu(z_l) (last layer: z_l)
//   out      = Qw . v_L + q0                            (projection)
// This is the unfolded pass (training, one layer).  Inference with the lift and
// the projection folded in, and the gradients, run on the matrix cores with real
// 9-coefficient transforms (k_fno_*, k_fnt_*, further down).
//
// Layouts: activations are [batch][channel][x] FP32 with x = (I*N+J)*N+K
// ([batch][x][channel] in the inference pass, FP32 or 16 bit);
// mode arrays are [batch][channel][k] complex with k = (px*8+py)*8+pz and
// wavenumber index kidx(p) per axis; theta holds P, p0, per layer
// (R (i,o,k) complex interleaved, Wm (o,i), b), Qw, q0.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>
#include <type_traits>

#include "../../include/frfs_sur.h"

int fq_internal_fail(int code, const std::string &msg);   // fq_lib.hip

namespace {

constexpr int SW = 32, SM = 8, SM3 = SM * SM * SM;
constexpr int64_t SR = 2LL * SW * SW * SM3;          // floats of one layer's R
constexpr int64_t SLAYER = SR + SW * SW + SW;        // floats of one layer

// Grid constants of the N^3 grid (N = 16 or 32).
template <int N> struct SG {
    static_assert(N == 16 || N == 32, "grids of 16^3 and 32^3 points");
    static constexpr int N2 = N * N, N3 = N * N * N;
    static constexpr int LOG3 = N == 16 ? 12 : 15;  // log2(N^3)
};

template <int N> __device__ __forceinline__ int kidx(int p) { return p < SM / 2 ? p : p + N - SM; }

// cos(2 pi j / 32), j = 0..31.
__device__ constexpr float kCos32[32] = {
    1.0f, 0.9807852804032304f, 0.9238795325112867f, 0.8314696123025452f,
    0.7071067811865476f, 0.5555702330196023f, 0.38268343236508984f, 0.19509032201612833f,
    0.0f, -0.1950903220161282f, -0.3826834323650897f, -0.555570233019602f,
    -0.7071067811865475f, -0.8314696123025453f, -0.9238795325112867f, -0.9807852804032304f,
    -1.0f, -0.9807852804032304f, -0.9238795325112868f, -0.8314696123025455f,
    -0.7071067811865477f, -0.5555702330196022f, -0.38268343236509034f, -0.19509032201612866f,
    0.0f, 0.1950903220161283f, 0.38268343236509f, 0.5555702330196018f,
    0.7071067811865474f, 0.8314696123025452f, 0.9238795325112865f, 0.9807852804032303f};
// cos(2 pi j / N) and sin(2 pi j / N) = cos(2 pi (j - N/4) / N), N = 16 or
// 32: the table entry (j mod N) (32 / N).  Called with compile-time j
// (unrolled loops) the values fold into the instructions; otherwise they are
// uniform loads of the table.
template <int N> __device__ __forceinline__ float cosN(int j) { return kCos32[(j * (32 / N)) & 31]; }
template <int N> __device__ __forceinline__ float sinN(int j) { return cosN<N>(j - N / 4); }

// 1 + erf(z / sqrt 2) = 2 - E for z > 0, else E, with E = erfc(|z| / sqrt 2) =
// 2^{-q(|z|)} and q a degree-10 fit of -log2 erfc (weighted least squares for
// the error of gelu, |z| <= 6.2; positive and growing beyond).  About 20
// instructions without a branch (erff takes both of its ranges in most waves).
// The FP32 gelu from it is off by 7.0e-8 rms and 3.8e-7 at most on [-6, 6]
// (7.9e-8 and 4.5e-7 with a correctly rounded erf).
__device__ __forceinline__ float one_plus_erf(float z) {
    const float u = fabsf(z);
    float a = 1.756848888589957e-08f;
    a = __builtin_fmaf(a, u, -5.725348728446988e-07f);
    a = __builtin_fmaf(a, u, 7.934887435112614e-06f);
    a = __builtin_fmaf(a, u, -5.907857484999113e-05f);
    a = __builtin_fmaf(a, u, 0.00022106834512669593f);
    a = __builtin_fmaf(a, u, 0.00011856652417918667f);
    a = __builtin_fmaf(a, u, -0.007087948732078075f);
    a = __builtin_fmaf(a, u, 0.05253392457962036f);
    a = __builtin_fmaf(a, u, 0.4591914415359497f);
    a = __builtin_fmaf(a, u, 1.1511074304580688f);
    const float e = __builtin_amdgcn_exp2f(-(a * u));
    return z > 0.f ? 2.0f - e : e;
}
__device__ __forceinline__ float gelu_fit(float z) { return 0.5f * z * one_plus_erf(z); }
// Training keeps erff: gelu' needs 1 + erf itself, for which the fit (weighed by
// z) is less exact near zero.
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
// Activation storage: FP32, or FP16 / BF16 for inference (arithmetic stays
// FP32; conversions round to nearest even).
template <typename TA> __device__ __forceinline__ float ldA(const TA *p, int64_t i) { return float(p[i]); }
template <typename TA> __device__ __forceinline__ void stA(TA *p, int64_t i, float v) { p[i] = TA(v); }
// two neighbouring values (even index), one 4- or 8-byte access
template <typename TA> struct alignas(2 * sizeof(TA)) Pair { TA a, b; };
template <typename TA> __device__ __forceinline__ float2 ld2(const TA *p, int64_t i) {
    const Pair<TA> h = *reinterpret_cast<const Pair<TA> *>(p + i);
    return make_float2(float(h.a), float(h.b));
}
template <typename TA> __device__ __forceinline__ void st2(TA *p, int64_t i, float2 v) {
    Pair<TA> h;
    h.a = TA(v.x);
    h.b = TA(v.y);
    *reinterpret_cast<Pair<TA> *>(p + i) = h;
}
// eight 16-bit values, one 16-byte store
template <typename TA> struct alignas(16) Pack8 { TA v[8]; };

// gelu(z), gelu'(z)
__device__ __forceinline__ float2 gelu_both(float z) {
    const float h = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
    return make_float2(z * h, h + z * 0.39894228040143268f * __expf(-0.5f * z * z));
}

// X[slice] = scale * sum_x v[slice](x) e^{-i k.x} over the retained modes.
// 16^3 grid: one workgroup per (batch, channel) slice; separable z, y, x stages in LDS,
// each thread reading its inputs once and producing all the modes of its
// line with compile-time twiddles.
template <typename TA>
__global__ __launch_bounds__(256) void k_sur_dft16(const TA *__restrict__ v, float scale, float2 *__restrict__ X) {
    __shared__ float vin[SG<16>::N2 * 17];
    __shared__ float2 A[SG<16>::N2 * 9];            // [I][J][pz]
    __shared__ float2 Bs[16 * SM * SM];      // [I][py][pz]
    const int t = threadIdx.x;
    const int64_t slice = blockIdx.x;
    const TA *src = v + slice * SG<16>::N3;
#pragma unroll
    for (int r = 0; r < SG<16>::N3 / 256; ++r) {
        const int e = t + 256 * r;
        vin[(e >> 4) * 17 + (e & 15)] = ldA(src, e);
    }
    __syncthreads();
    {
        float a[16];
#pragma unroll
        for (int K = 0; K < 16; ++K) a[K] = vin[t * 17 + K];
#pragma unroll
        for (int p = 0; p < SM; ++p) {
            const int k = kidx<16>(p);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int K = 0; K < 16; ++K) {
                re += a[K] * cosN<16>(k * K);
                im -= a[K] * sinN<16>(k * K);
            }
            A[t * 9 + p] = make_float2(re, im);
        }
    }
    __syncthreads();
    // y: thread t < 128 owns (I, pz) = (t / 8, t % 8): its 16 values once, the
    // 8 y modes with compile-time twiddles
    if (t < 16 * SM) {
        const int I = t >> 3, pz = t & 7;
        float2 a[16];
#pragma unroll
        for (int J = 0; J < 16; ++J) a[J] = A[(I * 16 + J) * 9 + pz];
#pragma unroll
        for (int py = 0; py < SM; ++py) {
            const int k = kidx<16>(py);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int J = 0; J < 16; ++J) {
                const float c = cosN<16>(k * J), sn = sinN<16>(k * J);
                re += a[J].x * c + a[J].y * sn;
                im += a[J].y * c - a[J].x * sn;
            }
            Bs[(I * SM + py) * SM + pz] = make_float2(re, im);
        }
    }
    __syncthreads();
    // x: thread t < 64 owns (py, pz) = (t / 8, t % 8): 16 values, the 8 x modes
    if (t < SM * SM) {
        float2 a[16];
#pragma unroll
        for (int I = 0; I < 16; ++I) a[I] = Bs[I * SM * SM + t];
#pragma unroll
        for (int px = 0; px < SM; ++px) {
            const int k = kidx<16>(px);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int I = 0; I < 16; ++I) {
                const float c = cosN<16>(k * I), sn = sinN<16>(k * I);
                re += a[I].x * c + a[I].y * sn;
                im += a[I].y * c - a[I].x * sn;
            }
            X[slice * SM3 + px * SM * SM + t] = make_float2(scale * re, scale * im);
        }
    }
}

// out[slice](x) = Re sum_k Y[slice](k) e^{+i k.x}
// (16^3 grid).
template <typename TA>
__global__ __launch_bounds__(256) void k_sur_idft16(const float2 *__restrict__ Y, TA *__restrict__ out) {
    __shared__ float2 Ys[SM3];               // [px][py][pz]
    __shared__ float2 T1[16 * SM * SM];      // [I][py][pz]
    __shared__ float2 T2[SG<16>::N2 * 9];           // [I][J][pz]
    const int t = threadIdx.x;
    const int64_t slice = blockIdx.x;
    Ys[t] = Y[slice * SM3 + t];
    Ys[t + 256] = Y[slice * SM3 + t + 256];
    __syncthreads();
    // x: thread t < 64 owns (py, pz) = (t / 8, t % 8): its 8 modes once, the 16
    // grid values I with compile-time twiddles
    if (t < SM * SM) {
        float2 a[SM];
#pragma unroll
        for (int px = 0; px < SM; ++px) a[px] = Ys[px * SM * SM + t];
#pragma unroll
        for (int I = 0; I < 16; ++I) {
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int px = 0; px < SM; ++px) {
                const float c = cosN<16>(kidx<16>(px) * I), sn = sinN<16>(kidx<16>(px) * I);
                re += a[px].x * c - a[px].y * sn;
                im += a[px].x * sn + a[px].y * c;
            }
            T1[I * SM * SM + t] = make_float2(re, im);
        }
    }
    __syncthreads();
    // y: thread t < 128 owns (I, pz) = (t / 8, t % 8): 8 values, the 16 rows J
    if (t < 16 * SM) {
        const int I = t >> 3, pz = t & 7;
        float2 a[SM];
#pragma unroll
        for (int py = 0; py < SM; ++py) a[py] = T1[(I * SM + py) * SM + pz];
#pragma unroll
        for (int J = 0; J < 16; ++J) {
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int py = 0; py < SM; ++py) {
                const float c = cosN<16>(kidx<16>(py) * J), sn = sinN<16>(kidx<16>(py) * J);
                re += a[py].x * c - a[py].y * sn;
                im += a[py].x * sn + a[py].y * c;
            }
            T2[(I * 16 + J) * 9 + pz] = make_float2(re, im);
        }
    }
    __syncthreads();
    // z: thread t owns grid row (I, J) = t: its 8 modes from LDS once, the 16
    // outputs with compile-time twiddles, written as four 16-byte stores
    float2 a[SM];
#pragma unroll
    for (int pz = 0; pz < SM; ++pz) a[pz] = T2[t * 9 + pz];
    float o[16];
#pragma unroll
    for (int K = 0; K < 16; ++K) {
        float sum = 0.f;
#pragma unroll
        for (int pz = 0; pz < SM; ++pz) sum += a[pz].x * cosN<16>(kidx<16>(pz) * K) - a[pz].y * sinN<16>(kidx<16>(pz) * K);
        o[K] = sum;
    }
    if constexpr (std::is_same<TA, float>::value) {
        float4 *dst = reinterpret_cast<float4 *>(out + slice * SG<16>::N3 + t * 16);
#pragma unroll
        for (int q = 0; q < 16 / 4; ++q) {
            dst[q] = make_float4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
        }
    } else {                                  // 16-bit activations
        static_assert(sizeof(TA) == 2, "16-bit storage");
        Pack8<TA> *dst = reinterpret_cast<Pack8<TA> *>(out + slice * SG<16>::N3 + t * 16);
#pragma unroll
        for (int q = 0; q < 16 / 8; ++q) {
            Pack8<TA> w;
#pragma unroll
            for (int j = 0; j < 8; ++j) w.v[j] = TA(o[8 * q + j]);
            dst[q] = w;
        }
    }
}

// The same transform on the 32^3 grid.  One workgroup of 512 threads per
// slice.  The z stage runs in two passes of 512 grid rows: each pass loads
// its rows with coalesced 16-byte loads into LDS (vin), then thread t turns
// row t into its 8 modes (A, 76 KB).  The y and x stages then work from LDS
// as on the 16^3 grid (Bs reuses vin).  143 KB of LDS: one workgroup per CU.
constexpr int kDft32Threads = 512;
// four floats at a float's alignment (the caller's g has no more), one 16-byte load
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
// LDS index of the 8 modes of grid row r = I*32 + J in the 32^3 transforms:
// rows padded to 9 and the 32 rows of one I to 296 float2 values, so that
// both the per-row accesses (z stage) and the per-(I, pz) accesses (y stage)
// spread over the LDS banks.
constexpr int kRowsI = 296;
__device__ __forceinline__ int aidx32(int I, int J, int pz) { return I * kRowsI + J * 9 + pz; }
template <typename TA>
__global__ __launch_bounds__(kDft32Threads) void k_sur_dft32(const TA *__restrict__ v, float scale,
                                                           float2 *__restrict__ X) {
    constexpr int N = 32, N3 = SG<32>::N3, T = kDft32Threads, RS = N + 1;
    __shared__ float2 A[N * kRowsI];          // [I][J][pz], aidx32
    __shared__ float vin[T * RS];             // one pass of rows; then Bs [I][py][pz]
    float2 *Bs = reinterpret_cast<float2 *>(vin);
    const int t = threadIdx.x;
    const int64_t slice = blockIdx.x;
    const TA *src = v + slice * N3;
#pragma unroll 1
    for (int q = 0; q < N * N / T; ++q) {
        const TA *rows = src + int64_t(q) * T * N;
        if constexpr (std::is_same<TA, float>::value) {
#pragma unroll
            for (int w = 0; w < T * N / 4 / T; ++w) {
                const int e4 = t + T * w;                 // float4 index in the pass
                const f32x4_u x = reinterpret_cast<const f32x4_u *>(rows)[e4];
                float *d = vin + (e4 >> 3) * RS + (e4 & 7) * 4;
                d[0] = x.x; d[1] = x.y; d[2] = x.z; d[3] = x.w;
            }
        } else {
#pragma unroll
            for (int w = 0; w < T * N / 8 / T; ++w) {
                const int e8 = t + T * w;                 // 8-value pack index in the pass
                const Pack8<TA> x = reinterpret_cast<const Pack8<TA> *>(rows)[e8];
                float *d = vin + (e8 >> 2) * RS + (e8 & 3) * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) d[j] = float(x.v[j]);
            }
        }
        __syncthreads();
        float a[N];
#pragma unroll
        for (int K = 0; K < N; ++K) a[K] = vin[t * RS + K];
        const int r = q * T + t;
#pragma unroll
        for (int pz = 0; pz < SM; ++pz) {
            const int k = kidx<N>(pz);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int K = 0; K < N; ++K) {
                re += a[K] * cosN<N>(k * K);
                im -= a[K] * sinN<N>(k * K);
            }
            A[aidx32(r >> 5, r & 31, pz)] = make_float2(re, im);
        }
        __syncthreads();
    }
    // y: thread t < 256 owns (I, pz) = (t / 8, t % 8): 32 values, the 8 y modes
    if (t < N * SM) {
        const int I = t >> 3, pz = t & 7;
        float2 a[N];
#pragma unroll
        for (int J = 0; J < N; ++J) a[J] = A[aidx32(I, J, pz)];
#pragma unroll
        for (int py = 0; py < SM; ++py) {
            const int k = kidx<N>(py);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int J = 0; J < N; ++J) {
                const float c = cosN<N>(k * J), sn = sinN<N>(k * J);
                re += a[J].x * c + a[J].y * sn;
                im += a[J].y * c - a[J].x * sn;
            }
            Bs[(I * SM + py) * SM + pz] = make_float2(re, im);
        }
    }
    __syncthreads();
    // x: thread t < 64 owns (py, pz): 32 values, the 8 x modes
    if (t < SM * SM) {
        float2 a[N];
#pragma unroll
        for (int I = 0; I < N; ++I) a[I] = Bs[I * SM * SM + t];
#pragma unroll
        for (int px = 0; px < SM; ++px) {
            const int k = kidx<N>(px);
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int I = 0; I < N; ++I) {
                const float c = cosN<N>(k * I), sn = sinN<N>(k * I);
                re += a[I].x * c + a[I].y * sn;
                im += a[I].y * c - a[I].x * sn;
            }
            X[slice * SM3 + px * SM * SM + t] = make_float2(scale * re, scale * im);
        }
    }
}

// The inverse transform on the 32^3 grid, 512 threads per slice: x and y
// stages in LDS (the mode block Ys shares its space with the y-stage output
// T2, and T1 with the output staging), then two passes of 512 grid rows:
// thread t computes row t's 32 outputs into LDS (ob) and the workgroup writes
// the pass with coalesced 16-byte stores.
template <typename TA>
__global__ __launch_bounds__(kDft32Threads) void k_sur_idft32(const float2 *__restrict__ Y, TA *__restrict__ out) {
    constexpr int N = 32, N3 = SG<32>::N3, T = kDft32Threads, RS = N + 1;
    __shared__ float2 T2[N * kRowsI];         // [I][J][pz] (aidx32); first the modes [px][py][pz]
    __shared__ float ob[T * RS];              // T1 [I][py][pz], then one pass of output rows
    float2 *Ys = T2;
    float2 *T1 = reinterpret_cast<float2 *>(ob);
    const int t = threadIdx.x;
    const int64_t slice = blockIdx.x;
    Ys[t] = Y[slice * SM3 + t];
    __syncthreads();
    // x: thread t < 64 owns (py, pz): 8 modes, the 32 grid values I
    if (t < SM * SM) {
        float2 a[SM];
#pragma unroll
        for (int px = 0; px < SM; ++px) a[px] = Ys[px * SM * SM + t];
#pragma unroll
        for (int I = 0; I < N; ++I) {
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int px = 0; px < SM; ++px) {
                const float c = cosN<N>(kidx<N>(px) * I), sn = sinN<N>(kidx<N>(px) * I);
                re += a[px].x * c - a[px].y * sn;
                im += a[px].x * sn + a[px].y * c;
            }
            T1[I * SM * SM + t] = make_float2(re, im);
        }
    }
    __syncthreads();
    // y: thread t < 256 owns (I, pz) = (t / 8, t % 8): 8 values, the 32 rows J
    if (t < N * SM) {
        const int I = t >> 3, pz = t & 7;
        float2 a[SM];
#pragma unroll
        for (int py = 0; py < SM; ++py) a[py] = T1[(I * SM + py) * SM + pz];
#pragma unroll
        for (int J = 0; J < N; ++J) {
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int py = 0; py < SM; ++py) {
                const float c = cosN<N>(kidx<N>(py) * J), sn = sinN<N>(kidx<N>(py) * J);
                re += a[py].x * c - a[py].y * sn;
                im += a[py].x * sn + a[py].y * c;
            }
            T2[aidx32(I, J, pz)] = make_float2(re, im);
        }
    }
    __syncthreads();
    // z: two passes of 512 rows
#pragma unroll 1
    for (int q = 0; q < N * N / T; ++q) {
        const int r = q * T + t;
        float2 a[SM];
#pragma unroll
        for (int pz = 0; pz < SM; ++pz) a[pz] = T2[aidx32(r >> 5, r & 31, pz)];
#pragma unroll
        for (int K = 0; K < N; ++K) {
            float sum = 0.f;
#pragma unroll
            for (int pz = 0; pz < SM; ++pz)
                sum += a[pz].x * cosN<N>(kidx<N>(pz) * K) - a[pz].y * sinN<N>(kidx<N>(pz) * K);
            ob[t * RS + K] = sum;
        }
        __syncthreads();
        TA *rows = out + slice * N3 + int64_t(q) * T * N;
        if constexpr (std::is_same<TA, float>::value) {
#pragma unroll
            for (int w = 0; w < T * N / 4 / T; ++w) {
                const int e4 = t + T * w;
                const float *sp = ob + (e4 >> 3) * RS + (e4 & 7) * 4;
                reinterpret_cast<float4 *>(rows)[e4] = make_float4(sp[0], sp[1], sp[2], sp[3]);
            }
        } else {                              // 16-bit activations
#pragma unroll
            for (int w = 0; w < T * N / 8 / T; ++w) {
                const int e8 = t + T * w;
                const float *sp = ob + (e8 >> 2) * RS + (e8 & 3) * 8;
                Pack8<TA> x;
#pragma unroll
                for (int j = 0; j < 8; ++j) x.v[j] = TA(sp[j]);
                reinterpret_cast<Pack8<TA> *>(rows)[e8] = x;
            }
        }
        __syncthreads();
    }
}

// Launchers of the per-slice transforms on the N^3 grid.
template <int N, typename TA>
void launch_dft(const TA *v, float scale, float2 *X, unsigned slices, hipStream_t st) {
    if constexpr (N == 16) hipLaunchKernelGGL(k_sur_dft16<TA>, dim3(slices), dim3(256), 0, st, v, scale, X);
    else hipLaunchKernelGGL(k_sur_dft32<TA>, dim3(slices), dim3(kDft32Threads), 0, st, v, scale, X);
}
template <int N, typename TA>
void launch_idft(const float2 *Y, TA *out, unsigned slices, hipStream_t st) {
    if constexpr (N == 16) hipLaunchKernelGGL(k_sur_idft16<TA>, dim3(slices), dim3(256), 0, st, Y, out);
    else hipLaunchKernelGGL(k_sur_idft32<TA>, dim3(slices), dim3(kDft32Threads), 0, st, Y, out);
}

// The mode product of the unfolded forward pass, Y(b,o,k) = sum_i X(b,i,k) R(i,o,k).
// A workgroup takes 8 consecutive modes and 16 DOFs and stages the 8 modes'
// 32 x 32 weights in LDS (64 KB) once; thread (mode m = t % 8, DOF t / 8 % 16,
// half t / 128 of the outputs) keeps its 16 outputs in registers.  Within a
// wave the eight DOFs of a mode read the same LDS word (a broadcast), so the
// weight reads are conflict-free.  Bound by latency for a training batch: 64
// DOFs 40 us with 32 DOFs and 32 outputs per thread (128 workgroups, the
// weights loaded one LDS store at a time), 20 us now; the sums are the same.
__global__ __launch_bounds__(256) void k_sur_mix_lds(const float2 *__restrict__ a, const float2 *__restrict__ R,
                                                     float2 *__restrict__ c, int64_t batch) {
    __shared__ float2 Rl[SW * SW * 8];               // [(i*32 + o)*8 + m]
    const int t = threadIdx.x;
    const int k0 = blockIdx.x * 8;
    const int m = t & 7, h = (t >> 7) * (SW / 2);
    const int64_t b = int64_t(blockIdx.y) * 16 + ((t >> 3) & 15);
    const int k = k0 + m;
    // all 32 inputs in flight at once, before the weights: occupancy is set by
    // the LDS tile (two waves per SIMD), so the registers are free
    float2 xs[SW];
#pragma unroll
    for (int j = 0; j < SW; ++j) xs[j] = a[((b < batch ? b : batch - 1) * SW + j) * SM3 + k];
#pragma unroll 1
    for (int e = t; e < SW * SW * 8; e += 256 * 16) {
        float2 r[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) r[u] = R[int64_t((e + 256 * u) >> 3) * SM3 + k0 + (e & 7)];
#pragma unroll
        for (int u = 0; u < 16; ++u) Rl[e + 256 * u] = r[u];
    }
    __syncthreads();
    if (b >= batch) return;
    float2 acc[SW / 2];
#pragma unroll
    for (int j = 0; j < SW / 2; ++j) acc[j] = make_float2(0.f, 0.f);
#pragma unroll
    for (int j = 0; j < SW; ++j) {
        const float2 x = xs[j];
#pragma unroll
        for (int q = 0; q < SW / 2; ++q) {
            const float2 r = Rl[(j * SW + h + q) * 8 + m];
            acc[q].x += x.x * r.x - x.y * r.y;
            acc[q].y += x.x * r.y + x.y * r.x;
        }
    }
#pragma unroll
    for (int j = 0; j < SW / 2; ++j) c[(b * SW + h + j) * SM3 + k] = acc[j];
}

// v_0(b, c, x) = P_c g(b, x) + p0_c
template <int N, typename TA>
__global__ __launch_bounds__(256) void k_sur_lift(const float *__restrict__ g, const float *__restrict__ th,
                                                  TA *__restrict__ v, int64_t total) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int64_t b = idx >> SG<N>::LOG3;
    const int x = int(idx & (SG<N>::N3 - 1));
    const float gv = g[idx];
#pragma unroll 8
    for (int c = 0; c < SW; ++c) stA(v, (b * SW + c) * SG<N>::N3 + x, th[c] * gv + th[SW + c]);
}

// z = Wm v + b + s; vout = act ? gelu(z) : z (z stored when zout is set).
// One thread per two neighbouring grid points (total = points, even).
template <int N, typename TA>
__global__ __launch_bounds__(256) void k_sur_pw(const TA *__restrict__ v, const TA *__restrict__ s,
                                                const float *__restrict__ lw, int act, TA *__restrict__ zout,
                                                TA *__restrict__ vout, int64_t total) {
    // the weights are the same for every lane: read at uniform addresses, they
    // arrive through scalar loads instead of LDS
    const int64_t idx = 2 * (int64_t(blockIdx.x) * 256 + threadIdx.x);
    if (idx >= total) return;
    const int64_t b = idx >> SG<N>::LOG3;
    const int x = int(idx & (SG<N>::N3 - 1));
    float2 vi[SW];
#pragma unroll
    for (int i = 0; i < SW; ++i) vi[i] = ld2(v, (b * SW + i) * SG<N>::N3 + x);
#pragma unroll 4
    for (int o = 0; o < SW; ++o) {
        const int64_t at = (b * SW + o) * SG<N>::N3 + x;
        const float2 sv = ld2(s, at);
        float z0 = lw[SW * SW + o] + sv.x, z1 = lw[SW * SW + o] + sv.y;
#pragma unroll
        for (int i = 0; i < SW; ++i) {
            z0 += lw[o * SW + i] * vi[i].x;
            z1 += lw[o * SW + i] * vi[i].y;
        }
        if (zout) st2(zout, at, make_float2(z0, z1));
        st2(vout, at, act ? make_float2(gelu(z0), gelu(z1)) : make_float2(z0, z1));
    }
}

// out(b, x) = Qw . v_L(b, :, x) + q0
template <int N, typename TA>
__global__ __launch_bounds__(256) void k_sur_proj(const TA *__restrict__ v, const float *__restrict__ qw,
                                                  float *__restrict__ out, int64_t total) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int64_t b = idx >> SG<N>::LOG3;
    const int x = int(idx & (SG<N>::N3 - 1));
    float s = qw[SW];
#pragma unroll 8
    for (int c = 0; c < SW; ++c) s += qw[c] * ldA(v, (b * SW + c) * SG<N>::N3 + x);
    out[idx] = s;
}

// Per-DOF workgroups are dealt round-robin to the eight XCDs; workgroup w
// takes DOF (w % 8) * per + w / 8 so that each XCD works through a contiguous
// DOF range and neighbouring elements, which share AoSoA cache lines, meet in
// one L2.  Launch 8 * per workgroups; the result is count or more when idle.
__device__ __forceinline__ int64_t xcd_slot(int64_t count) {
    const int64_t per = (count + 7) / 8;
    return int64_t(blockIdx.x & 7) * per + int64_t(blockIdx.x >> 3);
}

inline unsigned xcd_grid(int64_t count) { return unsigned(8 * ((count + 7) / 8)); }

// Sum over the 256 threads, to all of them.
__device__ __forceinline__ double block_sum(double v, double *red) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const double r = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
    return r;
}

// gout = 2 (out - target) / count; sums[0] += sum (out - target)^2,
// sums[1] += sum target^2.  At most 256 workgroups: the FP64 atomics on the two
// sums are serial, 28 us for 2048 of them (262144 values), 8 us now.
__global__ __launch_bounds__(256) void k_sur_loss(const float *__restrict__ out, const float *__restrict__ tgt,
                                                  float *__restrict__ gout, double *__restrict__ sums, int64_t count) {
    __shared__ double red[4];
    double d2 = 0, t2 = 0;
    for (int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x; idx < count; idx += int64_t(gridDim.x) * 256) {
        const float d = out[idx] - tgt[idx];
        gout[idx] = float(2.0 / double(count)) * d;
        d2 += double(d) * d;
        t2 += double(tgt[idx]) * tgt[idx];
    }
    const double s0 = block_sum(d2, red);
    const double s1 = block_sum(t2, red);
    if (threadIdx.x == 0) {
        atomicAdd(&sums[0], s0);
        atomicAdd(&sums[1], s1);
    }
}

__global__ __launch_bounds__(256) void k_sur_adam(float *__restrict__ th, const float *__restrict__ g,
                                                  float *__restrict__ m, float *__restrict__ v, int64_t n, float lr,
                                                  float b1, float b2, float eps, float c1, float c2) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    th[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// dst(b, x) = src(dof, x) / (rho_b^power * scale), rho_b = rho_in[b] or
// sum_x src(dof, x) cw (written to rho_out).  One workgroup per DOF.
__global__ __launch_bounds__(256) void k_sur_gather(int n, double cw, double scale, int power,
                                                    const double *__restrict__ src, int nupts, int64_t ldim,
                                                    int64_t first, const double *__restrict__ rho_in,
                                                    double *__restrict__ rho_out, float *__restrict__ dst,
                                                    int64_t ndof) {
    __shared__ double red[4];
    const int64_t b = xcd_slot(ndof);
    if (b >= ndof) return;
    const int64_t dof = first + b;
    const int64_t e = dof / nupts;
    const int u = int(dof % nupts);
    const double *base = src + u * ldim + (e / 32) * int64_t(n) * 32 + e % 32;
    double rho;
    if (rho_in) {
        rho = rho_in[b];
    } else {
        double s = 0;
        for (int x = threadIdx.x; x < n; x += 256) s += base[int64_t(x) * 32];
        rho = block_sum(s, red) * cw;
        if (rho_out && threadIdx.x == 0) rho_out[b] = rho;
    }
    double den = scale;
    for (int k = 0; k < power; ++k) den *= rho;
    const double inv = den != 0.0 ? 1.0 / den : 0.0;
    for (int x = threadIdx.x; x < n; x += 256) dst[b * n + x] = float(base[int64_t(x) * 32] * inv);
}

struct SurGram {
    double ginv[25];
    double gdiag[5];
};

// Conservation check and scatter.  For DOF b: moments m_j = cw sum_x q phi_j
// of the collision invariants phi = (1, cx, cy, cz, |c|^2); defect = max_j
// |m_j| / sqrt(G_jj cw sum q^2); DOFs with defect > tol are flagged and not
// written; the rest get Q = rho_b^2 scale (q - sum_j lambda_j phi_j) with
// lambda = G^{-1} m (the least-squares conservation projection).
__global__ __launch_bounds__(256) void k_sur_finish(int N, double c0, double dc, double cw, double scale, double tol,
                                                    const float *__restrict__ q, const double *__restrict__ rho,
                                                    SurGram gm, double *__restrict__ dst, int nupts, int64_t ldim,
                                                    int64_t first, double *__restrict__ defect,
                                                    int32_t *__restrict__ flag, int64_t ndof) {
    __shared__ double red[4];
    const int n = N * N * N;
    const int64_t b = xcd_slot(ndof);
    if (b >= ndof) return;
    const float *qb = q + b * n;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int x = threadIdx.x; x < n; x += 256) {
        const double cx = c0 + dc * (x / (N * N)), cy = c0 + dc * ((x / N) % N), cz = c0 + dc * (x % N);
        const double v = qb[x];
        acc[0] += v;
        acc[1] += v * cx;
        acc[2] += v * cy;
        acc[3] += v * cz;
        acc[4] += v * (cx * cx + cy * cy + cz * cz);
        acc[5] += v * v;
    }
    double mom[5];
    for (int j = 0; j < 5; ++j) mom[j] = block_sum(acc[j], red) * cw;
    const double nq = sqrt(block_sum(acc[5], red) * cw);
    double d = 0;
    for (int j = 0; j < 5; ++j) {
        const double cj = nq > 0 ? fabs(mom[j]) / (sqrt(gm.gdiag[j]) * nq) : 0.0;
        d = cj > d ? cj : d;
    }
    const bool bad = !(d <= tol);
    if (threadIdx.x == 0) {
        defect[b] = d;
        flag[b] = bad ? 1 : 0;
    }
    if (bad) return;
    double lam[5];
    for (int j = 0; j < 5; ++j) {
        double s = 0;
        for (int k = 0; k < 5; ++k) s += gm.ginv[j * 5 + k] * mom[k];
        lam[j] = s;
    }
    const double r = rho[b];
    const double f = r * r * scale;
    const int64_t dof = first + b;
    const int64_t e = dof / nupts;
    const int u = int(dof % nupts);
    double *out = dst + u * ldim + (e / 32) * int64_t(n) * 32 + e % 32;
    for (int x = threadIdx.x; x < n; x += 256) {
        const double cx = c0 + dc * (x / (N * N)), cy = c0 + dc * ((x / N) % N), cz = c0 + dc * (x % N);
        const double p = lam[0] + lam[1] * cx + lam[2] * cy + lam[3] * cz + lam[4] * (cx * cx + cy * cy + cz * cz);
        out[int64_t(x) * 32] = f * (double(qb[x]) - p);
    }
}

// Conservation penalty of a training batch (one workgroup per DOF b): the
// invariant component u_b = Phi^T G^{-1} Phi out_b cw of the network output,
// the orthogonal projection of out_b onto span{1, cx, cy, cz, |c|^2} (G the
// Gram matrix Phi Phi^T cw); gout_b += (2 lambda / count) u_b and sums[2] +=
// |u_b|^2, the gradient and value of lambda |u|^2 / count added to the mean
// square loss.  The targets conserve (they are projected), so this weights
// the error in the invariant directions lambda + 1 times.
__global__ __launch_bounds__(256) void k_sur_cons(int N, double c0, double dc, double cw, SurGram gm, double coef,
                                                  const float *__restrict__ out, float *__restrict__ gout,
                                                  double *__restrict__ sums) {
    __shared__ double red[4];
    const int n = N * N * N;
    const int64_t b = blockIdx.x;
    const float *ob = out + b * n;
    float *gb = gout + b * n;
    double acc[5] = {0, 0, 0, 0, 0};
    for (int x = threadIdx.x; x < n; x += 256) {
        const double cx = c0 + dc * (x / (N * N)), cy = c0 + dc * ((x / N) % N), cz = c0 + dc * (x % N);
        const double v = ob[x];
        acc[0] += v;
        acc[1] += v * cx;
        acc[2] += v * cy;
        acc[3] += v * cz;
        acc[4] += v * (cx * cx + cy * cy + cz * cz);
    }
    double mom[5], lam[5];
    for (int j = 0; j < 5; ++j) mom[j] = block_sum(acc[j], red) * cw;
    for (int j = 0; j < 5; ++j) {
        double t = 0;
        for (int k = 0; k < 5; ++k) t += gm.ginv[j * 5 + k] * mom[k];
        lam[j] = t;
    }
    double uu = 0;
    for (int x = threadIdx.x; x < n; x += 256) {
        const double cx = c0 + dc * (x / (N * N)), cy = c0 + dc * ((x / N) % N), cz = c0 + dc * (x % N);
        const double u = lam[0] + lam[1] * cx + lam[2] * cy + lam[3] * cz + lam[4] * (cx * cx + cy * cy + cz * cz);
        gb[x] += float(coef * u);
        uu += u * u;
    }
    const double tot = block_sum(uu, red);
    if (threadIdx.x == 0) atomicAdd(&sums[2], tot);
}

// ---------------------------------------------------------------------------
// Inference with the lift folded into the first layer and the projection into
// the last (layers >= 2).  With Ghat = DFT(g)/n (one channel):
//   first layer: X_0(i,k) = P_i Ghat(k) + p0_i [k = 0], so
//     Y_0(o,k) = Ghat(k) Rp(o,k) + [k = 0] c0(o),  Rp = sum_i P_i R_0(i,o,.),
//     c0 = sum_i p0_i R_0(i,o,0);  z_0 = A g + a0 + s_0,  A = Wm_0 P,
//     a0 = Wm_0 p0 + b_0;
//   last layer: Qw.s = Re IDFT(sum_o Qw_o Y(o,.)) and sum_o Qw_o Y(o,k) =
//     sum_i X(i,k) Rq(i,k), Rq = sum_o Qw_o R(i,o,.), so
//     out = QW.v + qb + Re IDFT(Y1),  QW = Qw Wm,  qb = Qw.b + q0.
// The folded weights (k_sur_fuse) are laid out as Rp (SW x SM3 complex), c0
// (SW complex), Rq (SW x SM3 complex), A, a0, QW (SW each), qb.
// ---------------------------------------------------------------------------
constexpr int64_t FRC0 = 2LL * SW * SM3, FRQ = FRC0 + 2 * SW, FA = FRQ + 2LL * SW * SM3;
constexpr int64_t FA0 = FA + SW, FQW = FA0 + SW, FQB = FQW + SW, FTOT = FQB + 1;
static_assert(FTOT == FQ_SUR_FUSED_FLOATS, "folded weight layout");
static_assert(FA0 == FA + SW && FQB == FQW + SW, "k_fno_plane reads A, a0 and QW, qb side by side");

__global__ __launch_bounds__(256) void k_sur_fuse(const float *__restrict__ th, int L, float *__restrict__ fw) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const float *P = th, *p0 = th + SW;
    const float *l0 = th + 2 * SW, *ll = th + 2 * SW + int64_t(L - 1) * SLAYER;
    const float2 *R0 = reinterpret_cast<const float2 *>(l0), *RL = reinterpret_cast<const float2 *>(ll);
    const float *W0 = l0 + SR, *b0 = l0 + SR + SW * SW, *WL = ll + SR, *bL = ll + SR + SW * SW;
    const float *Qw = th + 2 * SW + int64_t(L) * SLAYER, q0 = Qw[SW];
    int64_t j = idx;
    if (j < SW * SM3) {                      // Rp(o, k)
        const int k = int(j % SM3), o = int(j / SM3);
        float2 a = make_float2(0.f, 0.f);
        for (int i = 0; i < SW; ++i) {
            const float2 r = R0[(int64_t(i) * SW + o) * SM3 + k];
            a.x += P[i] * r.x;
            a.y += P[i] * r.y;
        }
        reinterpret_cast<float2 *>(fw)[j] = a;
        return;
    }
    j -= SW * SM3;
    if (j < SW * SM3) {                      // Rq(i, k)
        const int k = int(j % SM3), i = int(j / SM3);
        float2 a = make_float2(0.f, 0.f);
        for (int o = 0; o < SW; ++o) {
            const float2 r = RL[(int64_t(i) * SW + o) * SM3 + k];
            a.x += Qw[o] * r.x;
            a.y += Qw[o] * r.y;
        }
        reinterpret_cast<float2 *>(fw + FRQ)[j] = a;
        return;
    }
    j -= SW * SM3;
    if (j < SW) {                            // c0(o), A(o), a0(o), QW(i = j)
        const int o = int(j);
        float2 c = make_float2(0.f, 0.f);
        float a = 0.f, a0 = b0[o], qw = 0.f;
        for (int i = 0; i < SW; ++i) {
            const float2 r = R0[(int64_t(i) * SW + o) * SM3];
            c.x += p0[i] * r.x;
            c.y += p0[i] * r.y;
            a += W0[o * SW + i] * P[i];
            a0 += W0[o * SW + i] * p0[i];
            qw += Qw[i] * WL[i * SW + o];     // QW at input channel o
        }
        reinterpret_cast<float2 *>(fw + FRC0)[o] = c;
        fw[FA + o] = a;
        fw[FA0 + o] = a0;
        fw[FQW + o] = qw;
        return;
    }
    if (j == SW) {                           // qb
        float q = q0;
        for (int o = 0; o < SW; ++o) q += Qw[o] * bL[o];
        fw[FQB] = q;
    }
}

// ---------------------------------------------------------------------------
// The inference pass on the matrix cores.
//
// The retained modes of one axis, wavenumbers -4..3, are the span of the nine
// real functions beta_r: 1; cos(q t), q = 1..3; sin(q t), q = 1..3; cos(4 t);
// sin(4 t) (t = 2 pi x / N).  For a real input the mode X(k) with signs
// s_d = sign k_d and q_d = |k_d| is a signed sum of the eight products of
// cos / sin coefficients of its class (q_x, q_y, q_z),
//   e^{-i k.x} = prod_d (cos - i s_d sin),
// and the real part of the inverse transform needs only the transposed sums,
// so both transforms are real and separable, 9 coefficients per axis:
//   P[xr][yr][zr] = sum_{I,J,K} beta_xr(I) beta_yr(J) beta_zr(K) v(I,J,K)
//   s(I,J,K) = sum_{xr,yr,zr} beta_xr(I) beta_yr(J) beta_zr(K) Q[xr][yr][zr],
// with Q the folded mode outputs Y(k) = sum_i X_i(k) R(i,o,k).  Every stage is
// a small dense product of FP32 values and runs as
// v_mfma_f32_16x16x4_f32 (FP32 operands, FP32 sums):
//   k_fno_plane   one plane I of one DOF: z = Wm v + b + s from the plane's
//                 T[yr][zr][c] (y stage, then the z stage fused into the
//                 channel product), gelu, the new v, and the z and y stages of
//                 its forward transform, U[yr][zr][c]
//   k_fno_x       the x stages: U -> P (forward) and Q -> T (inverse)
//   k_fno_mix     P -> Q, a workgroup per class and 64 DOFs
// so one layer reads and writes the activations once (the transforms' volume s
// and the second and third pass over v are gone), and the last layer's input is
// never stored.  Activations are kept as
// [b][x][channel], so a lane's operands are contiguous.
//
// What bounds it: the plane kernel's two streams of v (8.4 MB per DOF and
// layer on the 32^3 grid, 1 MB on 16^3; the texture data units are busy in 92-98%
// of the cycles) and, nearly as long, its 30 matrix instructions (34-52% of the
// cycles) and 8 gelu per lane for every 16 points.  Measured for L = 4: 8192 DOFs
// on 16^3 20.2 ms with one VALU pass over v per stage, 10.9 ms now; 700 DOFs on
// 32^3 10.97 -> 4.51 ms, of it the plane kernels 4.00 ms (first layer 1.06,
// writing 2.9 GB; middle 1.57, reading and writing them; last 1.36, reading), the
// mode product 0.12 and the x stages 0.39.  Error against 64 bits 2.4e-7 ->
// 1.8e-7 (other inputs: 1.4e-7 -> 5.3e-8).
// Channels of a column tile t: o = 2 * (lane % 16) + t, so that the two tiles
// of a lane are neighbours (8-byte accesses).
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int NR = 9, NR2 = NR * NR, NR3 = NR2 * NR;     // real coefficients per axis, plane, volume

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// beta_r(j); zero for the padding rows r >= 9.
template <int N> __device__ __forceinline__ float beta(int r, int j) {
    const bool sn = (r >= 4 && r <= 6) || r == 8;
    const int q = r < 4 ? r : (r < 7 ? r - 3 : 4);
    const float v = kCos32[(q * j * (32 / N) - (sn ? 8 : 0)) & 31];
    return r < NR ? v : 0.f;
}

// Eight consecutive activations as floats.
__device__ __forceinline__ void ld8(const float *p, float *v) {
    const f32x4 a = reinterpret_cast<const f32x4 *>(p)[0], b = reinterpret_cast<const f32x4 *>(p)[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
}
template <typename TA> __device__ __forceinline__ void ld8(const TA *p, float *v) {
    const Pack8<TA> a = *reinterpret_cast<const Pack8<TA> *>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = float(a.v[i]);
}

// Sum over the 16 lanes of a row (DPP rotations by 8, 4, 2, 1).
__device__ __forceinline__ float row_sum(float x) {
    auto ror = [](float y, auto c) {
        return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, y), decltype(c)::value, 0xF, 0xF, true));
    };
    x += ror(x, std::integral_constant<int, 0x128>{});
    x += ror(x, std::integral_constant<int, 0x124>{});
    x += ror(x, std::integral_constant<int, 0x122>{});
    x += ror(x, std::integral_constant<int, 0x121>{});
    return x;
}

// The y stages of a plane kernel's LDS array Fz[J][zr][c], four waves: from
// T[yr][zr][c] (a barrier has to follow), and into U[yr][zr][c] (after one).
template <int N> __device__ __forceinline__ void plane_y_in(const float *__restrict__ tp, float *Fz, int wave, int col, int q) {
    constexpr int KT = N / 16;
    for (int u = wave; u < NR * KT; u += 4) {                // Fz[J][zr] = sum_yr beta_yr(J) T[yr][zr]
        const int zr = u % NR, j0 = u / NR * 16;
        f32x4 d0 = {0, 0, 0, 0}, d1 = d0;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int yr = q + 4 * s;
            const float2 t = *reinterpret_cast<const float2 *>(tp + ((yr < NR ? yr : NR - 1) * NR + zr) * SW + 2 * col);
            const float a = beta<N>(yr, j0 + col);
            d0 = mfma4(a, t.x, d0);
            d1 = mfma4(a, t.y, d1);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float2 *>(Fz + ((j0 + 4 * q + i) * NR + zr) * SW + 2 * col) = make_float2(d0[i], d1[i]);
    }
}
template <int N> __device__ __forceinline__ void plane_y_out(const float *Fz, float *__restrict__ up, int wave, int col, int q) {
    for (int zr = wave; zr < NR; zr += 4) {                  // U[yr][zr] = sum_J beta_yr(J) Fz[J][zr]
        f32x4 d0 = {0, 0, 0, 0}, d1 = d0;
#pragma unroll
        for (int s = 0; s < N / 4; ++s) {
            const int J = q + 4 * s;
            const float2 t = *reinterpret_cast<const float2 *>(Fz + (J * NR + zr) * SW + 2 * col);
            const float a = beta<N>(col, J);
            d0 = mfma4(a, t.x, d0);
            d1 = mfma4(a, t.y, d1);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < NR)
                *reinterpret_cast<float2 *>(up + ((4 * q + i) * NR + zr) * SW + 2 * col) = make_float2(d0[i], d1[i]);
    }
}

// One plane I of DOF b per workgroup; FIRST: v_1 from g (lw: the folded first
// layer's A, a0), else v_{l+1} from v_l in place (lw: the layer's Wm, b).
// LAST: v_{L-1} is not stored; its part of the projection, QW . v + qb, goes
// to out (qw: QW, qb) and its modes to U.  out may be g: a wave reads its 16 points
// of g before it writes them.
template <int N, typename TA, bool FIRST, bool LAST>
__global__ __launch_bounds__(256) void k_fno_plane(const float *__restrict__ T, const float *g,
                                                   const float *__restrict__ lw, TA *__restrict__ v,
                                                   float *__restrict__ U, const float *__restrict__ qw, float *out) {
    constexpr int KT = N / 16;                               // 16-point tiles of a row, 16-row tiles of the plane
    __shared__ float Fz[N * NR * SW];                        // [J][zr][c]: the row's z coefficients, in then out
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int64_t plane = blockIdx.x;                        // b * N + I
    plane_y_in<N>(T + plane * (NR2 * SW), Fz, wave, col, q);
    // operands that stay: the channel matrix and bias of this lane's two outputs, the z tables
    float wm[2][FIRST ? 1 : 8], w0[2], b0[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int o = 2 * col + t;
        if constexpr (FIRST) {
            w0[t] = lw[o];                                   // A
            b0[t] = lw[SW + o];                              // a0
        } else {
            b0[t] = lw[SW * SW + o];
#pragma unroll
            for (int s = 0; s < 8; ++s) wm[t][s] = lw[o * SW + 8 * q + s];
        }
    }
    float qw0 = 0.f, qw1 = 0.f, qb = 0.f;
    if constexpr (LAST) { qw0 = qw[2 * col]; qw1 = qw[2 * col + 1]; qb = qw[SW]; }
    float ez[KT][3], ef[KT][4];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
#pragma unroll
        for (int s = 0; s < 3; ++s) ez[k][s] = beta<N>(q + 4 * s, 16 * k + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) ef[k][i] = beta<N>(col, 16 * k + 4 * q + i);
    }
    __syncthreads();
    for (int J = wave; J < N; J += 4) {
        TA *row = v + ((plane * N + J) * N) * SW;
        float2 f[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int zr = q + 4 * s;
            f[s] = *reinterpret_cast<const float2 *>(Fz + (J * NR + (zr < NR ? zr : NR - 1)) * SW + 2 * col);
        }
        f32x4 az0 = {0, 0, 0, 0}, az1 = az0;
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            f32x4 d0, d1;
            if constexpr (FIRST) {
                const float *gp = g + (plane * N + J) * N + 16 * k + 4 * q;
                const float gv[4] = {gp[0], gp[1], gp[2], gp[3]};       // the caller's g: no alignment beyond a float's
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    d0[i] = w0[0] * gv[i] + b0[0];
                    d1[i] = w0[1] * gv[i] + b0[1];
                }
            } else {
                float a[8];
                ld8(row + (16 * k + col) * SW + 8 * q, a);
                d0 = {b0[0], b0[0], b0[0], b0[0]};
                d1 = {b0[1], b0[1], b0[1], b0[1]};
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    d0 = mfma4(a[s], wm[0][s], d0);
                    d1 = mfma4(a[s], wm[1][s], d1);
                }
            }
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                d0 = mfma4(ez[k][s], f[s].x, d0);
                d1 = mfma4(ez[k][s], f[s].y, d1);
            }
            float pv = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // the transform and the projection take the value as stored
                const TA x0 = TA(gelu_fit(d0[i])), x1 = TA(gelu_fit(d1[i]));
                if constexpr (LAST) {
                    const float r = row_sum(__builtin_fmaf(qw0, float(x0), qw1 * float(x1)));
                    if (col == i) pv = r;                    // lane col < 4 keeps point 4 q + col
                } else {
                    Pair<TA> h;
                    h.a = x0;
                    h.b = x1;
                    *reinterpret_cast<Pair<TA> *>(row + (16 * k + 4 * q + i) * SW + 2 * col) = h;
                }
                az0 = mfma4(ef[k][i], float(x0), az0);
                az1 = mfma4(ef[k][i], float(x1), az1);
            }
            if (LAST && col < 4) out[(plane * N + J) * N + 16 * k + 4 * q + col] = pv + qb;
        }
        // the row's coefficients take the place of the ones just read (same wave, LDS in order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < NR)
                *reinterpret_cast<float2 *>(Fz + (J * NR + 4 * q + i) * SW + 2 * col) = make_float2(az0[i], az1[i]);
    }
    __syncthreads();
    plane_y_out<N>(Fz, U + plane * (NR2 * SW), wave, col, q);
}

// x stages, one wave per (b, yr, zr) and 32 channels, block blk of four.
// FWD: P[b][xr][yz][c] = scale sum_I beta_xr(I) U[b][I][yz][c];
// else T[b][I][yz][c] = scale sum_xr beta_xr(I) Q[b][xr][yz][c].
template <int N, bool FWD>
__device__ __forceinline__ void x_stage(int64_t blk, const float *__restrict__ in, float *__restrict__ out, float scale,
                                        int64_t units) {
    const int lane = threadIdx.x & 63, col = lane & 15, q = lane >> 4;
    const int64_t u = blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (u >= units) return;
    const int64_t b = u / NR2;
    const int yz = int(u % NR2);
    if constexpr (FWD) {
        const float *p = in + (b * N * NR2 + yz) * SW + 2 * col;
        f32x4 d0 = {0, 0, 0, 0}, d1 = d0;
#pragma unroll
        for (int s = 0; s < N / 4; ++s) {
            const int I = q + 4 * s;
            const float2 t = *reinterpret_cast<const float2 *>(p + I * NR2 * SW);
            const float a = beta<N>(col, I);
            d0 = mfma4(a, t.x, d0);
            d1 = mfma4(a, t.y, d1);
        }
        float *o = out + (b * NR3 + yz) * SW + 2 * col;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < NR)
                *reinterpret_cast<float2 *>(o + (4 * q + i) * NR2 * SW) = make_float2(scale * d0[i], scale * d1[i]);
    } else {
        const float *p = in + (b * NR3 + yz) * SW + 2 * col;
        float2 t[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int xr = q + 4 * s;
            t[s] = *reinterpret_cast<const float2 *>(p + (xr < NR ? xr : NR - 1) * NR2 * SW);
        }
        float *o = out + (b * N * NR2 + yz) * SW + 2 * col;
#pragma unroll
        for (int k = 0; k < N / 16; ++k) {
            f32x4 d0 = {0, 0, 0, 0}, d1 = d0;
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const float a = beta<N>(q + 4 * s, 16 * k + col);
                d0 = mfma4(a, t[s].x, d0);
                d1 = mfma4(a, t[s].y, d1);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float2 *>(o + (16 * k + 4 * q + i) * NR2 * SW) = make_float2(scale * d0[i], scale * d1[i]);
        }
    }
}

template <int N, bool FWD>
__global__ __launch_bounds__(256) void k_fno_x(const float *__restrict__ in, float *__restrict__ out, float scale,
                                               int64_t units) {
    x_stage<N, FWD>(blockIdx.x, in, out, scale, units);
}

// Class (q_x, q_y, q_z), q in 0..4, of the modes: class index cls = (q_x*5 + q_y)*5 + q_z.
// Real coefficient e (bits x, y, z: 0 cos, 1 sin) of the class in the 9^3
// layout, or -1 where a sine of q = 0 does not exist.
__device__ __forceinline__ int cls_coef(int cls, int e) {
    const int qd[3] = {cls / 25, cls / 5 % 5, cls % 5};
    int at = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int sn = (e >> (2 - d)) & 1, qq = qd[d];
        if (sn && qq == 0) return -1;
        at = at * NR + (qq == 4 ? 7 + sn : qq + (sn ? 3 : 0));
    }
    return at;
}
// Mode m (bits x, y, z: 1 the negative wavenumber) of the class: index in the
// 8^3 mode set and the signs, or -1 where the class has no such mode.
__device__ __forceinline__ int cls_mode(int cls, int m, float *sg) {
    const int qd[3] = {cls / 25, cls / 5 % 5, cls % 5};
    int at = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int neg = (m >> (2 - d)) & 1, qq = qd[d];
        if (qq == 0 && neg) return -1;                   // zero has one sign
        if (qq == 4 && !neg) return -1;                  // only -4 is retained
        at = at * SM + (neg ? SM - qq : qq);
        sg[d] = qq == 0 ? 0.f : (neg ? -1.f : 1.f);
    }
    return at;
}
// X(k) from the class's real coefficients p[e], signs s.
__device__ __forceinline__ float2 cls_x(const float *p, const float *s) {
    return make_float2(p[0] - s[1] * s[2] * p[3] - s[0] * s[2] * p[5] - s[0] * s[1] * p[6],
                       -(s[2] * p[1] + s[1] * p[2] + s[0] * p[4]) + s[0] * s[1] * s[2] * p[7]);
}
// Q += the folded Y(k).
__device__ __forceinline__ void cls_fold(float *Q, float yr, float yi, const float *s) {
    Q[0] += yr;
    Q[3] -= s[1] * s[2] * yr;
    Q[5] -= s[0] * s[2] * yr;
    Q[6] -= s[0] * s[1] * yr;
    Q[1] -= s[2] * yi;
    Q[2] -= s[1] * yi;
    Q[4] -= s[0] * yi;
    Q[7] += s[0] * s[1] * s[2] * yi;
}

// Packed weights: mode k's matrix as 1024 complex values in the order in which
// k_fno_mix stages it, a half of the output channels o after the other, row rho
// = 4 (i % 8) + i / 8 of input channel i (the four lane groups then read
// neighbouring rows, each 32 LDS banks).  In theta a mode's weights are 4096
// bytes apart, 8 of 64 or 128 bytes fetched are used.
constexpr int kPack = SW * SW * SM3;                     // complex values of a layer
constexpr int kHalf = SW * SW / 2;
__device__ __forceinline__ int stage_at(int i, int o) {
    const int rho = (i % 8) * 4 + i / 8;
    return o / 16 * kHalf + rho * 16 + o % 16;
}

// dst = packed R of a layer (ADJ: of conj(R)^T), rows row and row + 1 of the
// packed matrices (32 columns) of 64 modes through LDS.
template <bool ADJ>
__device__ __forceinline__ void pack_tile(const float2 *__restrict__ src, float2 *__restrict__ dst, int row, int k0,
                                          float2 (*tile)[65]) {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int e = (t >> 6) + 4 * j, i = ADJ ? e % SW : row + e / SW, o = ADJ ? row + e / SW : e % SW;
        tile[e][t & 63] = src[int64_t(i * SW + o) * SM3 + k0 + (t & 63)];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int e = t & 63, k = (t >> 6) + 4 * j;
        const float2 r = tile[e][k];
        dst[int64_t(k0 + k) * (SW * SW) + stage_at(row + e / SW, e % SW)] = make_float2(r.x, ADJ ? -r.y : r.y);
    }
}

__global__ __launch_bounds__(256) void k_fno_pack(const float2 *__restrict__ R, float2 *__restrict__ Rp) {
    __shared__ float2 tile[64][65];
    pack_tile<false>(R, Rp, 2 * blockIdx.x, blockIdx.y * 64, tile);
}

// Q = fold(X R) for the modes of class blockIdx.x, the output channels o = 16
// blockIdx.z + col and 64 DOFs at a time (blockIdx.y, then by gridDim.y), sixteen
// per wave.  The class's weights (up to 8 modes, 32 KB) are staged in LDS, from
// the packed ones or (PACKED false, where there is no room for those) from
// theta.  ADJ: conj(R)^T in place of R, the backward product (P = gQ, Q = gP).
// Bound by the matrix instructions of the classes with 8 modes, 32 of 32 cycles
// per mode, wave and tile: 64 DOFs 24 us with both halves in one workgroup (125
// of them), 14 us now; 8192 DOFs 773 -> 645.
template <bool ADJ, bool PACKED>
__global__ __launch_bounds__(256) void k_fno_mix(const float *__restrict__ P, const float2 *__restrict__ R,
                                                 float *__restrict__ Q, int batch) {
    __shared__ float2 Rl[8][kHalf];
    const int cls = blockIdx.x, half = blockIdx.z, tid = threadIdx.x, lane = tid & 63, col = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    {
        constexpr int E = kHalf / 256;
        float2 r[E][8];                                  // all loads in flight, then the LDS stores
#pragma unroll
        for (int j = 0; j < E; ++j)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                float sg[3];
                const int k = cls_mode(cls, m, sg), e = tid + 256 * j, rho = e / 16;
                r[j][m] = make_float2(0.f, 0.f);
                if (k < 0) continue;
                const int i = rho % 4 * 8 + rho / 4, o = 16 * half + e % 16;
                if constexpr (PACKED) r[j][m] = R[int64_t(k) * (SW * SW) + half * kHalf + e];
                else r[j][m] = R[int64_t(ADJ ? o * SW + i : i * SW + o) * SM3 + k];
            }
#pragma unroll
        for (int j = 0; j < E; ++j)
#pragma unroll
            for (int m = 0; m < 8; ++m)
                Rl[m][tid + 256 * j] = make_float2(r[j][m].x, ADJ && !PACKED ? -r[j][m].y : r[j][m].y);
    }
    __syncthreads();
    const int o = 16 * half + col, ro = q * 16 + col;
#pragma unroll 1
    for (int b0 = blockIdx.y * 64 + wave * 16; b0 < batch; b0 += gridDim.y * 64) {   // no barrier inside
        const int bl = b0 + col < batch ? b0 + col : batch - 1;
        float p[8][8];                                   // [coefficient][s], input channel 8 q + s
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int at = cls_coef(cls, e);
#pragma unroll
            for (int s = 0; s < 8; ++s) p[e][s] = 0.f;
            if (at >= 0) ld8(P + (int64_t(bl) * NR3 + at) * SW + 8 * q, p[e]);
        }
        float acc[4][8];                                 // [row][coefficient]
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[i][e] = 0.f;
#pragma unroll 1
        for (int m = 0; m < 8; ++m) {
            float sg[3];
            if (cls_mode(cls, m, sg) < 0) continue;
            f32x4 yr[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, yi[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const float pe[8] = {p[0][s], p[1][s], p[2][s], p[3][s], p[4][s], p[5][s], p[6][s], p[7][s]};
                const float2 x = cls_x(pe, sg);
                const float2 r = Rl[m][4 * s * 16 + ro];
                yr[0] = mfma4(x.x, r.x, yr[0]);
                yi[0] = mfma4(x.x, r.y, yi[0]);
                yr[1] = mfma4(-x.y, r.y, yr[1]);
                yi[1] = mfma4(x.y, r.x, yi[1]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) cls_fold(acc[i], yr[0][i] + yr[1][i], yi[0][i] + yi[1][i], sg);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = b0 + 4 * q + i;
            if (b >= batch) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int at = cls_coef(cls, e);
                if (at >= 0) Q[(int64_t(b) * NR3 + at) * SW + o] = acc[i][e];
            }
        }
    }
}

// First layer's Q from the one-channel modes Xg: Y(o,k) = Xg(k) Rp(o,k) +
// [k = 0] c0(o).  One thread per (b, class, o).
__global__ __launch_bounds__(256) void k_fno_first(const float2 *__restrict__ Xg, const float *__restrict__ fw,
                                                   float *__restrict__ Q, int64_t total) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int o = int(idx % SW), cls = int(idx / SW % 125);
    const int64_t b = idx / (SW * 125);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        float sg[3];
        const int k = cls_mode(cls, m, sg);
        if (k < 0) continue;
        const float2 x = Xg[b * SM3 + k], r = reinterpret_cast<const float2 *>(fw)[o * SM3 + k];
        float2 y = make_float2(x.x * r.x - x.y * r.y, x.x * r.y + x.y * r.x);
        if (k == 0) {
            const float2 c = reinterpret_cast<const float2 *>(fw + FRC0)[o];
            y.x += c.x;
            y.y += c.y;
        }
        cls_fold(acc, y.x, y.y, sg);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int at = cls_coef(cls, e);
        if (at >= 0) Q[(b * NR3 + at) * SW + o] = acc[e];
    }
}

// Last layer's one output channel: Y1(b,k) = sum_i X(b,i,k) Rq(i,k).  One
// half-wave per (b, class), a lane per input channel.
__global__ __launch_bounds__(256) void k_fno_last(const float *__restrict__ P, const float *__restrict__ fw,
                                                  float2 *__restrict__ Y1, int64_t units) {
    const int64_t u = int64_t(blockIdx.x) * 8 + threadIdx.x / 32;
    if (u >= units) return;
    const int i = threadIdx.x & 31, cls = int(u % 125);
    const int64_t b = u / 125;
    const float2 *Rq = reinterpret_cast<const float2 *>(fw + FRQ);
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int at = cls_coef(cls, e);
        p[e] = at >= 0 ? P[(b * NR3 + at) * SW + i] : 0.f;
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        float sg[3];
        const int k = cls_mode(cls, m, sg);
        if (k < 0) continue;
        const float2 x = cls_x(p, sg), r = Rq[i * SM3 + k];
        float yr = x.x * r.x - x.y * r.y, yi = x.x * r.y + x.y * r.x;
#pragma unroll
        for (int s = 16; s > 0; s >>= 1) {
            yr += __shfl_xor(yr, s);
            yi += __shfl_xor(yi, s);
        }
        if (i == 0) Y1[b * SM3 + k] = make_float2(yr, yi);
    }
}

// out += s1
__global__ __launch_bounds__(256) void k_fno_add(const float *__restrict__ s1, float *__restrict__ out, int64_t pts) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx < pts) out[idx] += s1[idx];
}

// ---------------------------------------------------------------------------
// The gradients on the same transforms.
//
// With V the (real) analysis of all three axes, s = V^T Q and P = V v, so the
// backward pass runs the forward transforms on gz_l = dLoss/dz_l: gQ = V gz_l,
// and gv_l gains V^T gP; in the modes gX = gY conj(R)^T and gR = sum_b conj(X)
// gY, with the 1/n of the analysis on X and on gX.  v_l is taken as
// gelu(z_{l-1}), or the lift of g, where it is needed.
//   k_fnt_top    coefficients of gz_{L-1} = Qw gout, and dQw
//   k_fnt_back   from gz_l and T: dWm, db, gv_l, then gz_{l-1} and its U, or
//                the lift's gradients; gz_{l-1} takes the place of gz_l
//   k_fnt_pre    the packed weights, the sums over the planes of the layer above
//                and the x stage of gQ, in one launch
//   k_fnt_sum    the last sums over the planes
// gz is [b][x][c]; z and X are the forward pass's, [b][c][x] and [b][c][k].
// A layer reads gz_l and z_{l-1} and writes gz_{l-1}, three streams of the
// activations (15 with a kernel per product and transform), and its matrix
// instructions, 46 for 16 points, and 8 gelu and gelu' per lane take about as
// long.  A plane's weight gradients stay in registers, and the sums over planes
// are taken from one partial per plane, not with an atomic per plane and weight.
// 64 rows on 16^3, 4 layers: forward and backward 1467 us, 720 us now; the
// backward kernels of one layer 226 -> 84 us (k_fnt_back 33, k_fnt_mix_grad 21,
// k_fno_mix 14, k_fnt_pre 10, k_fno_x 6).  Error of the gradient against
// 64 bits 1.7e-7..5.4e-7 -> 3.5e-8..1.3e-7 over inputs and orders of the sums.  The
// forward pass in training keeps its kernels and their rounding.
// ---------------------------------------------------------------------------
constexpr int kPart = SW * SW + 3 * SW;      // partials of a plane: dWm, db, dP, dp0
constexpr int kPart0 = 2 * SW;               // and of the start: dQw, dq0 (the rest unused)

// Sum of a lane's value over the four lane groups.
__device__ __forceinline__ float group_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

// z [b][c][x] at four neighbouring points, channels c and c + 1 (p: channel c).
template <int N, typename TA> __device__ __forceinline__ void ld4x2(const TA *p, float2 *v) {
    struct alignas(4 * sizeof(TA)) Four { TA v[4]; };
    const Four a = *reinterpret_cast<const Four *>(p), b = *reinterpret_cast<const Four *>(p + SG<N>::N3);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = make_float2(float(a.v[i]), float(b.v[i]));
}

// One plane of gz_{L-1} = Qw gout: its coefficients U, and the plane's sums of
// gout z_{L-1} (dQw) and gout (dq0).
template <int N, typename TA>
__global__ __launch_bounds__(256) void k_fnt_top(const float *__restrict__ gout, const float *__restrict__ qw,
                                                 const TA *__restrict__ z, float *__restrict__ U,
                                                 float *__restrict__ part) {
    constexpr int KT = N / 16;
    __shared__ float Fz[N * NR * SW];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t plane = blockIdx.x;
    const TA *zp = z + (plane / N * SW + 2 * col) * SG<N>::N3 + plane % N * SG<N>::N2;
    const float w0 = qw[2 * col], w1 = qw[2 * col + 1];
    float ef[KT][4];
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) ef[k][i] = beta<N>(col, 16 * k + 4 * q + i);
    float s0 = 0.f, s1 = 0.f, sg = 0.f;
    for (int J = wave; J < N; J += 4) {
        f32x4 az0 = {0, 0, 0, 0}, az1 = az0;
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const int at = J * N + 16 * k + 4 * q;
            float2 zz[4];
            ld4x2<N>(zp + at, zz);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = gout[plane * SG<N>::N2 + at + i];
                s0 += v * zz[i].x;
                s1 += v * zz[i].y;
                sg += v;
                az0 = mfma4(ef[k][i], w0 * v, az0);
                az1 = mfma4(ef[k][i], w1 * v, az1);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < NR)
                *reinterpret_cast<float2 *>(Fz + (J * NR + 4 * q + i) * SW + 2 * col) = make_float2(az0[i], az1[i]);
    }
    __syncthreads();
    plane_y_out<N>(Fz, U + plane * (NR2 * SW), wave, col, q);
    __syncthreads();
    s0 = group_sum(s0);
    s1 = group_sum(s1);
    sg = group_sum(sg);
    if (q == 0) {
        *reinterpret_cast<float2 *>(Fz + wave * kPart0 + 2 * col) = make_float2(s0, s1);
        if (col == 0) Fz[wave * kPart0 + SW] = sg;
    }
    __syncthreads();
    if (tid <= SW)
        part[plane * kPart0 + tid] = (Fz[tid] + Fz[kPart0 + tid]) + (Fz[2 * kPart0 + tid] + Fz[3 * kPart0 + tid]);
}

// One plane of layer l backward.  gz_l: Qw gout (TOP) or from gz; v_l: the lift
// of g (BOT) or gelu(z_{l-1}) (zin).  part: this plane's dWm = gz_l v_l^T and
// db = gz_l, and for BOT the lift's gradients.  Otherwise gz_{l-1} =
// (Wm^T gz_l + s) gelu'(z_{l-1}) is written to gz and its coefficients to U.
template <int N, typename TA, bool TOP, bool BOT>
__global__ __launch_bounds__(256) void k_fnt_back(const float *__restrict__ T, const float *__restrict__ g,
                                                  const float *__restrict__ gout, const float *__restrict__ th,
                                                  const float *__restrict__ lw, const float *__restrict__ qw,
                                                  const TA *__restrict__ zin, float *gz, float *__restrict__ U,
                                                  float *__restrict__ part) {
    constexpr int KT = N / 16;
    __shared__ float Fz[N * NR * SW];
    static_assert(N * NR * SW >= 4 * kPart, "the waves' partials fit");
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t plane = blockIdx.x;
    plane_y_in<N>(T + plane * (NR2 * SW), Fz, wave, col, q);
    const TA *zp = zin + (plane / N * SW + 2 * col) * SG<N>::N3 + plane % N * SG<N>::N2;
    float wm[2][8], qa[TOP ? 8 : 1];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        wm[0][s] = lw[(8 * q + s) * SW + 2 * col];
        wm[1][s] = lw[(8 * q + s) * SW + 2 * col + 1];
        if constexpr (TOP) qa[s] = qw[8 * q + s];
    }
    float qw0 = 0.f, qw1 = 0.f, p0 = 0.f, p1 = 0.f, c0 = 0.f, c1 = 0.f;
    if constexpr (TOP) { qw0 = qw[2 * col]; qw1 = qw[2 * col + 1]; }
    if constexpr (BOT) { p0 = th[2 * col]; p1 = th[2 * col + 1]; c0 = th[SW + 2 * col]; c1 = th[SW + 2 * col + 1]; }
    float ez[KT][3], ef[KT][4];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
#pragma unroll
        for (int s = 0; s < 3; ++s) ez[k][s] = beta<N>(q + 4 * s, 16 * k + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) ef[k][i] = beta<N>(col, 16 * k + 4 * q + i);
    }
    f32x4 dw[2][2] = {{{0, 0, 0, 0}, {0, 0, 0, 0}}, {{0, 0, 0, 0}, {0, 0, 0, 0}}};   // [o parity][i parity]
    float db0 = 0.f, db1 = 0.f, dp0 = 0.f, dp1 = 0.f, dc0 = 0.f, dc1 = 0.f;
    __syncthreads();
    for (int J = wave; J < N; J += 4) {
        const int64_t row = (plane * N + J) * N;
        float2 f[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int zr = q + 4 * s;
            f[s] = *reinterpret_cast<const float2 *>(Fz + (J * NR + (zr < NR ? zr : NR - 1)) * SW + 2 * col);
        }
        f32x4 az0 = {0, 0, 0, 0}, az1 = az0;
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const int64_t pt = row + 16 * k;
            float a[8], gv[4];
            float2 gd[4], zd[4];                             // gz_l and z_{l-1} of points 4 q + i, channels 2 col, + 1
            if constexpr (TOP) {
                const float go = gout[pt + col];
#pragma unroll
                for (int s = 0; s < 8; ++s) a[s] = qa[s] * go;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float gi = gout[pt + 4 * q + i];
                    gd[i] = make_float2(qw0 * gi, qw1 * gi);
                }
            } else {
                ld8(gz + (pt + col) * SW + 8 * q, a);
#pragma unroll
                for (int i = 0; i < 4; ++i) gd[i] = ld2(gz, (pt + 4 * q + i) * SW + 2 * col);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (BOT) gv[i] = g[pt + 4 * q + i];
            }
            if constexpr (!BOT) ld4x2<N>(zp + J * N + 16 * k + 4 * q, zd);
            f32x4 d0 = {0, 0, 0, 0}, d1 = d0;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                d0 = mfma4(a[s], wm[0][s], d0);
                d1 = mfma4(a[s], wm[1][s], d1);
            }
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                d0 = mfma4(ez[k][s], f[s].x, d0);
                d1 = mfma4(ez[k][s], f[s].y, d1);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v0, v1;
                if constexpr (BOT) {
                    v0 = p0 * gv[i] + c0;
                    v1 = p1 * gv[i] + c1;
                    dp0 += d0[i] * gv[i];
                    dp1 += d1[i] * gv[i];
                    dc0 += d0[i];
                    dc1 += d1[i];
                } else {
                    const float2 e0 = gelu_both(zd[i].x), e1 = gelu_both(zd[i].y);
                    v0 = e0.x;
                    v1 = e1.x;
                    const float x0 = d0[i] * e0.y, x1 = d1[i] * e1.y;
                    *reinterpret_cast<float2 *>(gz + (pt + 4 * q + i) * SW + 2 * col) = make_float2(x0, x1);
                    az0 = mfma4(ef[k][i], x0, az0);
                    az1 = mfma4(ef[k][i], x1, az1);
                }
                dw[0][0] = mfma4(gd[i].x, v0, dw[0][0]);
                dw[0][1] = mfma4(gd[i].x, v1, dw[0][1]);
                dw[1][0] = mfma4(gd[i].y, v0, dw[1][0]);
                dw[1][1] = mfma4(gd[i].y, v1, dw[1][1]);
                db0 += gd[i].x;
                db1 += gd[i].y;
            }
        }
        if constexpr (!BOT) {
            // the row's coefficients take the place of the ones just read (same wave, LDS in order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * q + i < NR)
                    *reinterpret_cast<float2 *>(Fz + (J * NR + 4 * q + i) * SW + 2 * col) = make_float2(az0[i], az1[i]);
        }
    }
    __syncthreads();
    if constexpr (!BOT) {
        plane_y_out<N>(Fz, U + plane * (NR2 * SW), wave, col, q);
        __syncthreads();
    }
    float *mine = Fz + wave * kPart;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<float2 *>(mine + (2 * (4 * q + r) + t) * SW + 2 * col) = make_float2(dw[t][0][r], dw[t][1][r]);
    float *tail = mine + SW * SW;
    db0 = group_sum(db0);
    db1 = group_sum(db1);
    if (q == 0) *reinterpret_cast<float2 *>(tail + 2 * col) = make_float2(db0, db1);
    if constexpr (BOT) {
        dp0 = group_sum(dp0);
        dp1 = group_sum(dp1);
        dc0 = group_sum(dc0);
        dc1 = group_sum(dc1);
        if (q == 0) {
            *reinterpret_cast<float2 *>(tail + SW + 2 * col) = make_float2(dp0, dp1);
            *reinterpret_cast<float2 *>(tail + 2 * SW + 2 * col) = make_float2(dc0, dc1);
        }
    }
    __syncthreads();
    for (int j = tid; j < (BOT ? kPart : SW * SW + SW); j += 256)
        part[plane * kPart + j] = (Fz[j] + Fz[kPart + j]) + (Fz[2 * kPart + j] + Fz[3 * kPart + j]);
}

// to[j] += sum over planes of from[plane][j], j < cols: 64 columns and 64 planes per workgroup.
struct Sum { const float *from; float *to; int stride, cols; };
__device__ __forceinline__ void sum_block(const Sum &sm, int cb, int64_t pb, int64_t planes, float *red) {
    const int t = threadIdx.x, j = cb * 64 + (t & 63);
    const int64_t r0 = pb * 64 + (t >> 6);
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int64_t r = r0 + 4 * k;
        if (j < sm.cols && r < planes) s += sm.from[r * sm.stride + j];
    }
    red[t] = s;
    __syncthreads();
    if (t < 64 && j < sm.cols) atomicAdd(&sm.to[j], (red[t] + red[t + 64]) + (red[t + 128] + red[t + 192]));
}

// The start of a layer, its parts side by side on the blocks of one launch (each
// alone is too short to fill the chip):
//   pk blocks    conj(R)^T packed into Rp (64 modes, two rows)
//   sm blocks    the sum sm over the planes, of what the kernel before left
//   then         gQ = x stage of U
struct Pre {
    const float2 *R;
    float2 *Rp;
    Sum sm;
    int64_t planes;
    const float *U;
    float *gQ;
    int64_t units;
    int pk, smb;
};
template <int N> __global__ __launch_bounds__(256) void k_fnt_pre(Pre a) {
    __shared__ float2 tile[64][65];
    int64_t b = blockIdx.x;                                  // every branch is uniform
    if (b < a.pk) return pack_tile<true>(a.R, a.Rp, 2 * int(b / 8), int(b % 8) * 64, tile);
    b -= a.pk;
    if (b < a.smb) {
        const int cb = (a.sm.cols + 63) / 64;
        return sum_block(a.sm, int(b % cb), b / cb, a.planes, &tile[0][0].x);
    }
    x_stage<N, true>(b - a.smb, a.U, a.gQ, 1.0f, a.units);
}

// The last sums of a pass: dWm and db of layer 0 (a) and the lift's gradients (b).
__global__ __launch_bounds__(256) void k_fnt_sum(Sum a, Sum b, int64_t planes) {
    __shared__ float red[256];
    const Sum &s = blockIdx.z ? b : a;
    if (int(blockIdx.x) * 64 < s.cols) sum_block(s, blockIdx.x, blockIdx.y, planes, red);
}

// gR(i,o,k) += sum_b conj X(b,i,k) gY(b,o,k), gY from the coefficients gQ of gz.
// A workgroup takes the eight modes (px, py) = blockIdx.x, a wave each, and the
// input channels i = 16 blockIdx.y + col; the DOFs are the inner dimension of the
// product.  The eight modes are 64 contiguous bytes of X and of the gradient, both
// taken through LDS.  Bound by latency (128 workgroups, a batch of loads per 16
// DOFs): 64 DOFs on 16^3 21 us; 22 with X read by each wave for itself, 37 with
// the output channels on two workgroups besides.  A class of modes per workgroup
// took 14, but 12 more to transpose X and to bring the result into place, in
// arrays that few DOFs have no room for.
__global__ __launch_bounds__(512) void k_fnt_mix_grad(const float2 *__restrict__ X, const float *__restrict__ gQ,
                                                      float2 *__restrict__ gR, int batch) {
    __shared__ float2 buf[16 * SW][SM + 1];                  // [i * 32 + o][pz]
    __shared__ float2 xs[16][16][SM + 1];                    // X of 16 DOFs [b][i][pz]
    const int lane = threadIdx.x & 63, col = lane & 15, q = lane >> 4;
    const int pz = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the mode's class and signs (cls_mode's inverse)
    const int pd[3] = {int(blockIdx.x) / SM, int(blockIdx.x) % SM, pz};
    int cls = 0;
    float sg[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const bool neg = pd[d] >= SM / 2;
        cls = cls * 5 + (neg ? SM - pd[d] : pd[d]);
        sg[d] = pd[d] == 0 ? 0.f : (neg ? -1.f : 1.f);
    }
    int at[8];
    float has[8];                                            // 0 where the class has no such coefficient
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int c = cls_coef(cls, e);
        at[e] = (c < 0 ? 0 : c) * SW + 2 * col;
        has[e] = c < 0 ? 0.f : 1.f;
    }
    // X of 16 DOFs at a time through LDS, eight lanes on a channel's eight modes:
    // element threadIdx.x + 512 j is DOF (threadIdx.x / 128) + 4 j
    const int xi = int(threadIdx.x) / SM % 16, xp = int(threadIdx.x) % SM, xb = int(threadIdx.x) / (16 * SM);
    const float2 *xk = X + (16 * blockIdx.y + xi) * SM3 + blockIdx.x * SM + xp;
    float2 nx[4];
    auto load = [&](int b0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = b0 + xb + 4 * j;
            nx[j] = xk[int64_t(b < batch ? b : batch - 1) * (SW * SM3)];
        }
    };
    f32x4 re[2][2], im[2][2];                                // [o parity][term]
#pragma unroll
    for (int t = 0; t < 4; ++t) re[t >> 1][t & 1] = im[t >> 1][t & 1] = {0, 0, 0, 0};
    load(0);
#pragma unroll 1
    for (int s0 = 0; s0 < batch; s0 += 16) {
        __syncthreads();                                         // xs is free
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[xb + 4 * j][xi][xp] = nx[j];
        __syncthreads();
        load(s0 + 16);
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int b = s0 + 4 * it + q, bl = b < batch ? b : batch - 1;
            const bool live = b < batch;
            float py[2][8];
            float2 x = xs[4 * it + q][col][pz];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float2 y = *reinterpret_cast<const float2 *>(gQ + int64_t(bl) * (NR3 * SW) + at[e]);
                py[0][e] = has[e] != 0.f ? y.x : 0.f;
                py[1][e] = has[e] != 0.f ? y.y : 0.f;
            }
            float2 Y[2] = {cls_x(py[0], sg), cls_x(py[1], sg)};
            if (!live) x = Y[0] = Y[1] = make_float2(0.f, 0.f);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                re[u][0] = mfma4(x.x, Y[u].x, re[u][0]);
                re[u][1] = mfma4(x.y, Y[u].y, re[u][1]);
                im[u][0] = mfma4(x.x, Y[u].y, im[u][0]);
                im[u][1] = mfma4(-x.y, Y[u].x, im[u][1]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < 2; ++u)
            buf[(4 * q + r) * SW + 2 * col + u][pz] = make_float2(re[u][0][r] + re[u][1][r], im[u][0][r] + im[u][1][r]);
    __syncthreads();
    constexpr int E = 16 * SW * SM / 512;
    float2 *g = gR + int64_t(16 * blockIdx.y) * SW * SM3 + blockIdx.x * SM;
    float2 old[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int e = threadIdx.x + 512 * j;
        old[j] = g[int64_t(e / SM) * SM3 + e % SM];
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int e = threadIdx.x + 512 * j;
        const float2 w = buf[e / SM][e % SM];
        g[int64_t(e / SM) * SM3 + e % SM] = make_float2(old[j].x + w.x, old[j].y + w.y);
    }
}

inline unsigned nblk(int64_t n) { return unsigned((n + 255) / 256); }

// Workgroups of k_fno_mix: 64 DOFs each, but more of them per staged class
// beyond 16 * 64 DOFs (the chip is full by then).
inline dim3 mix_grid(int64_t batch) {
    const int64_t t = (batch + 63) / 64;
    return dim3(125, unsigned(t < 16 ? t : 16), 2);
}

int check_shape(const fq_sur_shape *s, const char *who) {
    if (!s) return fq_internal_fail(FQ_ERR_INVALID, std::string(who) + ": null shape");
    if (s->abi_version != FQ_SUR_ABI_VERSION)
        return fq_internal_fail(FQ_ERR_INVALID, std::string(who) + ": ABI version mismatch");
    if ((s->Nv != 16 && s->Nv != 32) || s->width != SW || s->modes != SM || s->layers < 1 ||
        s->layers > FQ_SUR_MAX_LAYERS)
        return fq_internal_fail(FQ_ERR_UNSUPPORTED, std::string(who) +
                                ": supported shapes are Nv 16 or 32, width 32, modes 8, 1..8 layers");
    return FQ_SUCCESS;
}

int hip_status(const char *who) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? FQ_SUCCESS : fq_internal_fail(FQ_ERR_HIP, std::string(who) + ": " + hipGetErrorString(e));
}

struct ActPtrs {
    float *v[FQ_SUR_MAX_LAYERS + 1];
    float *z[FQ_SUR_MAX_LAYERS];
    float2 *X[FQ_SUR_MAX_LAYERS];
    float *s;
    float2 *Y;
};

// Activation layout (floats): training keeps v_0..v_L, z_0..z_{L-1} and
// X_0..X_{L-1}; inference keeps two v buffers and one X.  Both end with the
// s and Y scratch.
int64_t act_floats(int N3, int L, int64_t B, bool training) {
    const int64_t vol = B * SW * N3, md = 2 * B * SW * SM3;
    return training ? (L + 1) * vol + L * vol + L * md + vol + md : 2 * vol + md + vol + md;
}

ActPtrs act_ptrs(int N3, float *acts, int L, int64_t B, bool training) {
    const int64_t vol = B * SW * N3, md = 2 * B * SW * SM3;
    ActPtrs p{};
    float *q = acts;
    if (training) {
        for (int l = 0; l <= L; ++l) p.v[l] = q + l * vol;
        q += (L + 1) * vol;
        for (int l = 0; l < L; ++l) p.z[l] = q + l * vol;
        q += L * vol;
        for (int l = 0; l < L; ++l) p.X[l] = reinterpret_cast<float2 *>(q + l * md);
        q += L * md;
    } else {
        for (int l = 0; l <= L; ++l) p.v[l] = q + (l & 1) * vol;
        q += 2 * vol;
        for (int l = 0; l < L; ++l) p.X[l] = reinterpret_cast<float2 *>(q);
        q += md;
    }
    p.s = q;
    p.Y = reinterpret_cast<float2 *>(q + vol);
    return p;
}

// Room for a layer's packed weights between `from` and `end` (floats), 16-byte
// aligned as the arrays before them are, or null: few DOFs leave none and the
// weights are read from theta in place.
inline float2 *pack_room(float *from, float *end) {
    float *at = from + (-(reinterpret_cast<uintptr_t>(from) / sizeof(float)) & 3);
    return end - at >= 2LL * kPack ? reinterpret_cast<float2 *>(at) : nullptr;
}
template <bool ADJ> void mix(const float *P, const float *R, const float2 *Rp, float *Q, int64_t batch, hipStream_t st) {
    hipLaunchKernelGGL((Rp ? k_fno_mix<ADJ, true> : k_fno_mix<ADJ, false>), mix_grid(batch), dim3(256), 0, st, P,
                       Rp ? Rp : reinterpret_cast<const float2 *>(R), Q, int(batch));
}

// The folded inference pass with activations stored as A (FP32 or 16 bits),
// in the inference activation space: v [b][x][c], then T and U
// [b][I][yr][zr][c], P and Q [b][xr][yr][zr][c], the one-channel modes X and
// the one-channel volume s.
template <int N, typename A>
void forward_fused(int L, const float *theta, const float *fused, const float *g, int64_t batch, float *acts,
                   float *out, hipStream_t st) {
    constexpr int N3 = SG<N>::N3;
    const int64_t vol = batch * SW * N3, tp = batch * N * NR2 * SW, pq = batch * NR3 * SW;
    A *v = reinterpret_cast<A *>(acts);
    float *T = acts + vol, *U = T + tp, *P = U + tp, *Q = P + pq;
    float2 *X = reinterpret_cast<float2 *>(Q + pq);
    float *s1 = Q + pq + 2 * batch * SM3;
    static_assert(int64_t(SW) * N3 + 2 * N * NR2 * SW + 2 * NR3 * SW + 2 * SM3 + N3 <=
                  3LL * SW * N3 + 4 * SW * SM3, "fits the inference activation space");
    float2 *Rp = pack_room(s1 + batch * N3, acts + act_floats(N3, L, batch, false));
    const int64_t pts = batch * N3, xu = batch * NR2;
    const dim3 blk(256), pg(unsigned(batch * N)), xg(unsigned((xu + 3) / 4));
    // first layer from the one-channel transform of g
    launch_dft<N, float>(g, 1.0f / N3, X, unsigned(batch), st);
    hipLaunchKernelGGL(k_fno_first, dim3(nblk(batch * 125 * SW)), blk, 0, st, X, fused, Q, batch * 125 * SW);
    hipLaunchKernelGGL((k_fno_x<N, false>), xg, blk, 0, st, Q, T, 1.0f, xu);
    hipLaunchKernelGGL((L == 2 ? k_fno_plane<N, A, true, true> : k_fno_plane<N, A, true, false>), pg, blk, 0, st, T, g,
                       fused + FA, v, U, fused + FQW, out);
    for (int l = 1; l < L - 1; ++l) {
        const float *lay = theta + 2 * SW + l * SLAYER;
        hipLaunchKernelGGL((k_fno_x<N, true>), xg, blk, 0, st, U, P, 1.0f / N3, xu);
        if (Rp)
            hipLaunchKernelGGL(k_fno_pack, dim3(16, 8), blk, 0, st, reinterpret_cast<const float2 *>(lay), Rp);
        mix<false>(P, lay, Rp, Q, batch, st);
        hipLaunchKernelGGL((k_fno_x<N, false>), xg, blk, 0, st, Q, T, 1.0f, xu);
        hipLaunchKernelGGL((l == L - 2 ? k_fno_plane<N, A, false, true> : k_fno_plane<N, A, false, false>), pg, blk, 0,
                           st, T, g, lay + SR, v, U, fused + FQW, out);
    }
    // last layer and projection as one output channel
    hipLaunchKernelGGL((k_fno_x<N, true>), xg, blk, 0, st, U, P, 1.0f / N3, xu);
    hipLaunchKernelGGL(k_fno_last, dim3(unsigned((batch * 125 + 7) / 8)), blk, 0, st, P, fused, X, batch * 125);
    launch_idft<N, float>(X, s1, unsigned(batch), st);
    hipLaunchKernelGGL(k_fno_add, dim3(nblk(pts)), blk, 0, st, s1, out, pts);
}

// The unfolded pass (training keeps v_l, z_l and X_l) with activations
// stored as A in the FP32-sized regions of the activation layout.
template <int N, typename A>
void forward_impl(int L, const float *theta, const float *g, int64_t batch, bool tr, float *acts, float *out,
                  hipStream_t st) {
    const ActPtrs p = act_ptrs(SG<N>::N3, acts, L, batch, tr);
    const int64_t pts = batch * SG<N>::N3;
    const unsigned slices = unsigned(batch * SW);
    A *sa = reinterpret_cast<A *>(p.s);
    hipLaunchKernelGGL((k_sur_lift<N, A>), dim3(nblk(pts)), dim3(256), 0, st, g, theta, reinterpret_cast<A *>(p.v[0]), pts);
    for (int l = 0; l < L; ++l) {
        const float *lay = theta + 2 * SW + l * SLAYER;
        const float2 *R = reinterpret_cast<const float2 *>(lay);
        A *vl = reinterpret_cast<A *>(p.v[l]), *vn = reinterpret_cast<A *>(p.v[l + 1]);
        launch_dft<N, A>(vl, 1.0f / SG<N>::N3, p.X[l], slices, st);
        hipLaunchKernelGGL(k_sur_mix_lds, dim3(SM3 / 8, unsigned((batch + 15) / 16)), dim3(256), 0, st, p.X[l],
                           R, p.Y, batch);
        launch_idft<N, A>(p.Y, sa, slices, st);
        hipLaunchKernelGGL((k_sur_pw<N, A>), dim3(nblk(pts / 2)), dim3(256), 0, st, vl, sa, lay + SR, int(l < L - 1),
                           tr ? reinterpret_cast<A *>(p.z[l]) : nullptr, vn, pts);
    }
    hipLaunchKernelGGL((k_sur_proj<N, A>), dim3(nblk(pts)), dim3(256), 0, st, reinterpret_cast<const A *>(p.v[L]),
                       theta + 2 * SW + L * SLAYER, out, pts);
}

// Gradients from the activations of a training forward_impl<A>; the
// gradients themselves (gz, the coefficient arrays) stay FP32.  Everything is
// kept in work, so that calls with work arrays of their own can share one acts:
//   gz, gQ, gP, U, T; free space; the planes' partial sums of a layer and of the start.
// From a layer's gQ to its T the T array holds nothing: the packed weights stand
// there and in the free space behind it (16^3: from 12 DOFs on; fewer read the
// weights in place).  The bottom layer writes no U: its partial sums take that place.
template <int N, typename A>
void backward_impl(int L, const float *theta, const float *g, int64_t batch, float *acts, const float *gout,
                   float *grad, float *work, hipStream_t st) {
    constexpr int64_t V = int64_t(SW) * SG<N>::N3, TP = int64_t(N) * NR2 * SW, PQ = int64_t(NR3) * SW, MD = 2LL * SW * SM3;
    constexpr int64_t PP = int64_t(N) * kPart, P0 = int64_t(N) * kPart0;
    static_assert(V + 2 * PQ + 2 * TP + PP + P0 <= 2 * V + 2 * MD, "fits the work size");
    static_assert(PP <= TP, "the bottom layer's partial sums in place of U");
    const ActPtrs p = act_ptrs(SG<N>::N3, acts, L, batch, true);     // read only
    float *gz = work, *gQ = gz + batch * V, *gP = gQ + batch * PQ, *U = gP + batch * PQ, *T = U + batch * TP;
    float *part0 = work + batch * (2 * V + 2 * MD - P0), *part = part0 - batch * PP;
    float2 *Rp = pack_room(T, part);
    const int64_t xu = batch * NR2, planes = batch * N, qoff = 2 * SW + L * SLAYER;
    const int64_t xb = (xu + 3) / 4, pb = (planes + 63) / 64;
    const dim3 blk(256), pg = dim3(unsigned(planes));
    auto wsum = [&](const float *from, int l) { return Sum{from, grad + 2 * SW + l * SLAYER + SR, kPart, SW * SW + SW}; };
    hipLaunchKernelGGL((k_fnt_top<N, A>), pg, blk, 0, st, gout, theta + qoff, reinterpret_cast<const A *>(p.z[L - 1]), U,
                       part0);
    for (int l = L - 1; l >= 0; --l) {
        const int64_t lo = 2 * SW + l * SLAYER;
        const bool top = l == L - 1;
        Pre pre{reinterpret_cast<const float2 *>(theta + lo), Rp, top ? Sum{part0, grad + qoff, kPart0, SW + 1} : wsum(part, l + 1),
                planes, U, gQ, xu, Rp ? 16 * 8 : 0, 0};
        pre.smb = int(pb * ((pre.sm.cols + 63) / 64));
        hipLaunchKernelGGL(k_fnt_pre<N>, dim3(unsigned(pre.pk + pre.smb + xb)), blk, 0, st, pre);
        mix<true>(gQ, theta + lo, Rp, gP, batch, st);
        hipLaunchKernelGGL(k_fnt_mix_grad, dim3(SM * SM, 2), dim3(512), 0, st, p.X[l], gQ,
                           reinterpret_cast<float2 *>(grad + lo), int(batch));
        hipLaunchKernelGGL((k_fno_x<N, false>), dim3(unsigned(xb)), blk, 0, st, gP, T, 1.0f / SG<N>::N3, xu);
        auto *k = l == 0 ? (top ? k_fnt_back<N, A, true, true> : k_fnt_back<N, A, false, true>)
                         : (top ? k_fnt_back<N, A, true, false> : k_fnt_back<N, A, false, false>);
        hipLaunchKernelGGL(k, pg, blk, 0, st, T, g, gout, theta, theta + lo + SR, theta + qoff,
                           reinterpret_cast<const A *>(p.z[l ? l - 1 : 0]), gz, U, l ? part : U);
    }
    hipLaunchKernelGGL(k_fnt_sum, dim3((SW * SW + SW + 63) / 64, unsigned(pb), 2), blk, 0, st, wsum(U, 0),
                       Sum{U + SW * SW + SW, grad, kPart, 2 * SW}, planes);
}

// Dispatch on the activation storage type.
template <int N>
void forward_acts(int acts_type, int L, const float *theta, const float *g, int64_t batch, bool tr, float *acts,
                  float *out, hipStream_t st) {
    if (acts_type == FQ_SUR_ACTS_FP16) forward_impl<N, _Float16>(L, theta, g, batch, tr, acts, out, st);
    else if (acts_type == FQ_SUR_ACTS_BF16) forward_impl<N, __bf16>(L, theta, g, batch, tr, acts, out, st);
    else forward_impl<N, float>(L, theta, g, batch, tr, acts, out, st);
}
template <int N>
void fused_acts(int acts_type, int L, const float *theta, const float *fused, const float *g, int64_t batch,
                float *acts, float *out, hipStream_t st) {
    if (acts_type == FQ_SUR_ACTS_FP16) forward_fused<N, _Float16>(L, theta, fused, g, batch, acts, out, st);
    else if (acts_type == FQ_SUR_ACTS_BF16) forward_fused<N, __bf16>(L, theta, fused, g, batch, acts, out, st);
    else forward_fused<N, float>(L, theta, fused, g, batch, acts, out, st);
}
template <int N>
void backward_acts(int acts_type, int L, const float *theta, const float *g, int64_t batch, float *acts,
                   const float *gout, float *grad, float *work, hipStream_t st) {
    if (acts_type == FQ_SUR_ACTS_FP16) backward_impl<N, _Float16>(L, theta, g, batch, acts, gout, grad, work, st);
    else if (acts_type == FQ_SUR_ACTS_BF16) backward_impl<N, __bf16>(L, theta, g, batch, acts, gout, grad, work, st);
    else backward_impl<N, float>(L, theta, g, batch, acts, gout, grad, work, st);
}

}  // namespace

extern "C" {

int fq_sur_sizes(const fq_sur_shape *shape, int64_t batch, int32_t training, int64_t *nparams, int64_t *act_size,
                 int64_t *work_size) {
    if (int rc = check_shape(shape, "fq_sur_sizes")) return rc;
    if (batch < 0) return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_sizes: negative batch");
    const int L = shape->layers;
    if (nparams) *nparams = 2 * SW + L * SLAYER + SW + 1;
    const int N3 = shape->Nv * shape->Nv * shape->Nv;
    if (act_size) *act_size = act_floats(N3, L, batch, training != 0);
    if (work_size) *work_size = 2 * batch * SW * N3 + 4 * batch * SW * SM3;
    return FQ_SUCCESS;
}

int fq_sur_forward(const fq_sur_shape *shape, const float *theta, const float *g, int64_t batch, int32_t training,
                   int32_t acts_type, float *acts, float *out, void *stream) {
    if (int rc = check_shape(shape, "fq_sur_forward")) return rc;
    if (batch < 0 || batch > FQ_SUR_MAX_BATCH || !theta || !g || !acts || !out ||
        acts_type < FQ_SUR_ACTS_FP32 || acts_type > FQ_SUR_ACTS_BF16)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_forward: invalid arguments");
    if (batch == 0) return FQ_SUCCESS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool tr = training != 0;
    if (shape->Nv == 16) forward_acts<16>(acts_type, shape->layers, theta, g, batch, tr, acts, out, st);
    else forward_acts<32>(acts_type, shape->layers, theta, g, batch, tr, acts, out, st);
    return hip_status("fq_sur_forward");
}

int fq_sur_fuse(const fq_sur_shape *shape, const float *theta, float *fused, void *stream) {
    if (int rc = check_shape(shape, "fq_sur_fuse")) return rc;
    if (shape->layers < 2) return fq_internal_fail(FQ_ERR_UNSUPPORTED, "fq_sur_fuse: needs at least two layers");
    if (!theta || !fused) return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_fuse: invalid arguments");
    hipLaunchKernelGGL(k_sur_fuse, dim3(nblk(2LL * SW * SM3 + SW + 1)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), theta, shape->layers, fused);
    return hip_status("fq_sur_fuse");
}

int fq_sur_forward_fused(const fq_sur_shape *shape, const float *theta, const float *fused, const float *g,
                         int64_t batch, int32_t acts_type, float *acts, float *out, void *stream) {
    if (int rc = check_shape(shape, "fq_sur_forward_fused")) return rc;
    if (shape->layers < 2)
        return fq_internal_fail(FQ_ERR_UNSUPPORTED, "fq_sur_forward_fused: needs at least two layers");
    if (batch < 0 || batch > FQ_SUR_MAX_BATCH || !theta || !fused || !g || !acts || !out ||
        acts_type < FQ_SUR_ACTS_FP32 || acts_type > FQ_SUR_ACTS_BF16)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_forward_fused: invalid arguments");
    if (batch == 0) return FQ_SUCCESS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (shape->Nv == 16) fused_acts<16>(acts_type, shape->layers, theta, fused, g, batch, acts, out, st);
    else fused_acts<32>(acts_type, shape->layers, theta, fused, g, batch, acts, out, st);
    return hip_status("fq_sur_forward_fused");
}

int fq_sur_backward(const fq_sur_shape *shape, const float *theta, const float *g, int64_t batch, int32_t acts_type,
                    float *acts, const float *gout, float *grad, float *work, void *stream) {
    if (int rc = check_shape(shape, "fq_sur_backward")) return rc;
    if (batch < 0 || batch > FQ_SUR_MAX_BATCH || !theta || !g || !acts || !gout || !grad || !work ||
        acts_type < FQ_SUR_ACTS_FP32 || acts_type > FQ_SUR_ACTS_BF16)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_backward: invalid arguments");
    if (batch == 0) return FQ_SUCCESS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (shape->Nv == 16) backward_acts<16>(acts_type, shape->layers, theta, g, batch, acts, gout, grad, work, st);
    else backward_acts<32>(acts_type, shape->layers, theta, g, batch, acts, gout, grad, work, st);
    return hip_status("fq_sur_backward");
}

int fq_sur_loss(int64_t count, const float *out, const float *target, float *gout, double *sums, void *stream) {
    if (count < 0 || !out || !target || !gout || !sums)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_loss: invalid arguments");
    if (count == 0) return FQ_SUCCESS;
    hipLaunchKernelGGL(k_sur_loss, dim3(count > 65536 ? 256 : nblk(count)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), out,
                       target, gout, sums, count);
    return hip_status("fq_sur_loss");
}

int fq_sur_cons(int32_t Nv, double L, double cw, double lambda, int64_t batch, const float *out,
                const double *gram_inv, float *gout, double *sums, void *stream) {
    if ((Nv != 16 && Nv != 32) || !(L > 0) || !(cw > 0) || !(lambda >= 0) || batch < 0 || batch > FQ_SUR_MAX_BATCH ||
        !out || !gram_inv || !gout || !sums)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_cons: invalid arguments");
    if (batch == 0 || lambda == 0) return FQ_SUCCESS;
    SurGram gm;
    for (int j = 0; j < 25; ++j) gm.ginv[j] = gram_inv[j];
    for (int j = 0; j < 5; ++j) gm.gdiag[j] = 0;
    const double count = double(batch) * Nv * Nv * Nv;
    hipLaunchKernelGGL(k_sur_cons, dim3(unsigned(batch)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), Nv,
                       -L + L / Nv, 2 * L / Nv, cw, gm, 2.0 * lambda / count, out, gout, sums);
    return hip_status("fq_sur_cons");
}

int fq_sur_adam(int64_t nparams, float *theta, const float *grad, float *m, float *v, float lr, float beta1,
                float beta2, float eps, int32_t step, void *stream) {
    if (nparams < 0 || !theta || !grad || !m || !v || step < 1 || !(lr >= 0) || !(beta1 >= 0 && beta1 < 1) ||
        !(beta2 >= 0 && beta2 < 1) || !(eps > 0))
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_adam: invalid arguments");
    if (nparams == 0) return FQ_SUCCESS;
    const float c1 = float(1.0 / (1.0 - pow(double(beta1), step)));
    const float c2 = float(1.0 / (1.0 - pow(double(beta2), step)));
    hipLaunchKernelGGL(k_sur_adam, dim3(nblk(nparams)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), theta,
                       grad, m, v, nparams, lr, beta1, beta2, eps, c1, c2);
    return hip_status("fq_sur_adam");
}

int fq_sur_gather(int32_t Nv, double cw, double scale, int32_t power, const double *src, int32_t nupts, int64_t ldim,
                  int32_t neles, int64_t first_dof, int64_t ndof, const double *rho_in, double *rho_out, float *dst,
                  void *stream) {
    if (Nv <= 0 || !(cw > 0) || !(scale != 0) || power < 0 || power > 4 || !src || !dst || nupts <= 0 ||
        neles <= 0 || first_dof < 0 || ndof < 0 || first_dof + ndof > int64_t(nupts) * neles)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_gather: invalid arguments");
    const int64_t nparr = (int64_t(neles) + 31) / 32 * 32;
    if (ldim < int64_t(Nv) * Nv * Nv * nparr) return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_gather: ldim too small");
    if (ndof == 0) return FQ_SUCCESS;
    hipLaunchKernelGGL(k_sur_gather, dim3(xcd_grid(ndof)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                       Nv * Nv * Nv, cw, scale, power, src, nupts, ldim, first_dof, rho_in, rho_out, dst, ndof);
    return hip_status("fq_sur_gather");
}

int fq_sur_finish(int32_t Nv, double L, double cw, double scale, double tol, const float *q, const double *rho,
                  const double *gram_inv, const double *gram_diag, double *dst, int32_t nupts, int64_t ldim,
                  int32_t neles, int64_t first_dof, int64_t ndof, double *defect, int32_t *flag, void *stream) {
    if (Nv <= 0 || !(L > 0) || !(cw > 0) || !q || !rho || !gram_inv || !gram_diag || !dst || !defect || !flag ||
        nupts <= 0 || neles <= 0 || first_dof < 0 || ndof < 0 || first_dof + ndof > int64_t(nupts) * neles)
        return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_finish: invalid arguments");
    const int64_t nparr = (int64_t(neles) + 31) / 32 * 32;
    if (ldim < int64_t(Nv) * Nv * Nv * nparr) return fq_internal_fail(FQ_ERR_INVALID, "fq_sur_finish: ldim too small");
    if (ndof == 0) return FQ_SUCCESS;
    SurGram gm;
    for (int j = 0; j < 25; ++j) gm.ginv[j] = gram_inv[j];
    for (int j = 0; j < 5; ++j) gm.gdiag[j] = gram_diag[j];
    hipLaunchKernelGGL(k_sur_finish, dim3(xcd_grid(ndof)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), Nv,
                       -L + L / Nv, 2 * L / Nv, cw, scale, tol, q, rho, gm, dst, nupts, ldim, first_dof, defect, flag,
                       ndof);
    return hip_status("fq_sur_finish");
}

}  // extern "C"
