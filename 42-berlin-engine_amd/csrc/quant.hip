// quant.hip -- INT8 / FP8 E4M3 codecs of the reference, row-wise, on gfx950.
//
// quant_f32_to_int8  src/compute/ops_quant.c:229-270
// quant_f32_to_fp8   src/compute/ops_quant.c:103-136 (float_to_fp8 :68-98)
// g_fp8_lut          src/compute/ops_quant.c:18-63
//
// Codes and scales are bit-identical to the reference: the absmax is an exact
// max reduction, the divisions are IEEE divisions, roundf rounds half away
// from zero, and the FP8 exponent reproduces glibc's floorf(log2f(a)) through
// a per-binade threshold table measured on the host at init.
#include <cmath>
#include <cstring>

#include "be42_common.h"

namespace be42 {

__constant__ float c_fp8_thr[kFp8ThrN];

// Reference E4M3 encoder (ops_quant.c:68-98) on the device.
__device__ __forceinline__ uint8_t f32_to_fp8(float v)
{
    if (v == 0.0f)
        return 0;
    const uint32_t sign = v < 0.0f ? 0x80u : 0u;
    float a = fabsf(v);
    if (a > 448.0f)
        a = 448.0f;
    int ex = (int)((__float_as_uint(a) >> 23) & 0xFF) - 127;   // floor(log2 a), a normal
    if ((__float_as_uint(a) >> 23) == 0)
        ex = -127;                                            // subnormal: far below e = 0
    const int up = ex + 1;
    // a threshold lies at most 64 ulps below its power of two
    // (host_fp8_thresholds), so the table is read for such values only
    if ((__float_as_uint(a) & 0x7FFFFFu) >= 0x7FFFC0u && up >= kFp8ThrE0 && up < kFp8ThrE0 + kFp8ThrN &&
        a >= c_fp8_thr[up - kFp8ThrE0])
        ex = up;                                              // log2f rounded up to an integer
    int e = ex + 7;
    e = e < 0 ? 0 : (e > 15 ? 15 : e);
    const float frac = (e == 0) ? a * 64.0f
                                : a * __uint_as_float((uint32_t)(127 + 7 - e) << 23) - 1.0f;
    int m = (int)__fmaf_rn(frac, 8.0f, 0.5f);
    if (m > 7)
        m = 7;
    return (uint8_t)(sign | ((uint32_t)e << 3) | (uint32_t)m);
}


// quant_f32_to_int8's code of one element (ops_quant.c:262-267)
__device__ __forceinline__ int8_t f32_to_int8(float v, float inv)
{
    const int c = (int)roundf(v * inv);
    return (int8_t)(c > 127 ? 127 : (c < -127 ? -127 : c));
}

// block-wide absmax of one row (256 threads)
__device__ __forceinline__ float row_absmax(const float *x, int cols, float *red)
{
    float m = 0.0f;
    for (int i = threadIdx.x; i < cols; i += blockDim.x)
        m = fmaxf(m, fabsf(x[i]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = m;
    __syncthreads();
    float r = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++)
        r = fmaxf(r, red[w]);
    return r;
}

__global__ __launch_bounds__(256) void k_quant_rows_int8(int8_t *q, float *scales, const float *x,
                                                         int cols)
{
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const float *xr = x + row * cols;
    const float amax = row_absmax(xr, cols, red);
    float scale = 1.0f, inv = 1.0f;
    if (amax > 0.0f) {
        scale = amax / 127.0f;
        inv = 127.0f / amax;
    }
    if (threadIdx.x == 0)
        scales[row] = scale;
    for (int i = threadIdx.x; i < cols; i += blockDim.x)
        q[row * cols + i] = f32_to_int8(xr[i], inv);
}

__global__ __launch_bounds__(256) void k_quant_rows_fp8(uint8_t *q, float *scales, const float *x,
                                                        int cols)
{
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const float *xr = x + row * cols;
    const float amax = row_absmax(xr, cols, red);
    float scale = 1.0f, inv = 1.0f;
    if (amax > 0.0f) {
        scale = amax / 224.0f;
        inv = 1.0f / scale;
    }
    if (threadIdx.x == 0)
        scales[row] = scale;
    for (int i = threadIdx.x; i < cols; i += blockDim.x)
        q[row * cols + i] = f32_to_fp8(xr[i] * inv);
}

// Both codecs on rows whose elements come four to an aligned word.  HBM bound
// (4 bytes in, 1 out per element): a block keeps its row in registers between
// the absmax and the codes, so the row is read once, by NV 16-byte loads per
// thread that are all in flight together, and leaves as 4-byte stores; the
// one-element loops above read it twice, a round trip per element.  A pass of
// quantize + product: FP8 8192 x 4096 x 14336 616 -> 559 us, INT8 500 x 4096 x
// 4096 29.3 -> 24.3 us (the product alone 22).
template <bool FP8, int NV>
__global__ __launch_bounds__(256) void k_quant_rows_vec(uint8_t *__restrict__ q, float *__restrict__ scales,
                                                        const float *__restrict__ x, int cols)
{
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const float4 *xr = (const float4 *)(x + row * cols);
    const int n4 = cols / 4;
    float4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = threadIdx.x + 256 * j;
        v[j] = i < n4 ? xr[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++)
        m = fmaxf(fmaxf(fmaxf(m, fabsf(v[j].x)), fmaxf(fabsf(v[j].y), fabsf(v[j].z))), fabsf(v[j].w));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = m;
    __syncthreads();
    const float amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float scale = 1.0f, inv = 1.0f;
    if (amax > 0.0f) {
        scale = amax / (FP8 ? 224.0f : 127.0f);
        inv = FP8 ? 1.0f / scale : 127.0f / amax;
    }
    if (threadIdx.x == 0)
        scales[row] = scale;
    uint32_t *qr = (uint32_t *)(q + row * cols);
    auto code = [&](float e) {
        return FP8 ? (uint32_t)f32_to_fp8(e * inv) : (uint32_t)(uint8_t)f32_to_int8(e, inv);
    };
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = threadIdx.x + 256 * j;
        if (i < n4)
            qr[i] = code(v[j].x) | code(v[j].y) << 8 | code(v[j].z) << 16 | code(v[j].w) << 24;
    }
}

// Rows of up to 16384 elements (16 words per thread) in 16-byte words; longer,
// odd or unaligned ones take the one-element kernels.
template <bool FP8>
static bool launch_quant_vec(uint8_t *q, float *scales, const float *x, int rows, int cols, hipStream_t s)
{
    const int nv = (cols / 4 + 255) / 256;
    if (cols % 4 || nv > 16 || (uintptr_t)x % 16 || (uintptr_t)q % 4)
        return false;
    const dim3 g(rows), b(256);
    if (nv <= 1)
        hipLaunchKernelGGL((k_quant_rows_vec<FP8, 1>), g, b, 0, s, q, scales, x, cols);
    else if (nv <= 4)
        hipLaunchKernelGGL((k_quant_rows_vec<FP8, 4>), g, b, 0, s, q, scales, x, cols);
    else if (nv <= 8)
        hipLaunchKernelGGL((k_quant_rows_vec<FP8, 8>), g, b, 0, s, q, scales, x, cols);
    else
        hipLaunchKernelGGL((k_quant_rows_vec<FP8, 16>), g, b, 0, s, q, scales, x, cols);
    return true;
}

__global__ void k_dequant_rows_int8(float *out, const int8_t *q, const float *scales, int cols,
                                    size_t total)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (size_t)gridDim.x * blockDim.x)
        out[i] = (float)q[i] * scales[i / cols];
}

__global__ void k_fp8_decode(float *out, const uint8_t *q, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        out[i] = fp8_to_f32(q[i]);
}

// Threshold table of glibc's log2f: smallest float in [2^(E-1), 2^E) whose
// floorf(log2f()) is E (log2f rounds up within a few ulps of 2^E).
static void host_fp8_thresholds(float *thr)
{
    for (int i = 0; i < kFp8ThrN; i++) {
        const int E = kFp8ThrE0 + i;
        float a = ldexpf(1.0f, E);
        for (int step = 0; step < 64; step++) {
            const float b = nextafterf(a, 0.0f);
            if ((int)floorf(log2f(b)) != E)
                break;
            a = b;
        }
        thr[i] = a;
    }
}

static int g_thr_ready[64];

int upload_fp8_thresholds(int device)
{
    if (device < 0 || device >= 64)
        return BE42_EINVAL;
    if (g_thr_ready[device])
        return BE42_OK;
    float thr[kFp8ThrN];
    host_fp8_thresholds(thr);
    BE42_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_fp8_thr), thr, sizeof thr));
    g_thr_ready[device] = 1;
    return BE42_OK;
}

int fp8_thresholds_ready(int device) { return device >= 0 && device < 64 && g_thr_ready[device]; }

}  // namespace be42

using namespace be42;

static int ensure_thresholds()
{
    int dev = 0;
    BE42_HIP(hipGetDevice(&dev));
    if (!fp8_thresholds_ready(dev))
        return upload_fp8_thresholds(dev);
    return BE42_OK;
}

extern "C" int be42_quant_rows_int8(int8_t *q, float *scales, const float *x, int rows, int cols,
                                    void *stream)
{
    BE42_CHECK(q && scales && x, "be42_quant_rows_int8: null pointer");
    BE42_CHECK(rows >= 0 && cols > 0, "be42_quant_rows_int8: bad shape %d x %d", rows, cols);
    if (rows == 0)
        return BE42_OK;
    if (!launch_quant_vec<false>((uint8_t *)q, scales, x, rows, cols, as_stream(stream)))
        hipLaunchKernelGGL(k_quant_rows_int8, dim3(rows), dim3(256), 0, as_stream(stream), q, scales, x, cols);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

extern "C" int be42_quant_rows_fp8(uint8_t *q, float *scales, const float *x, int rows, int cols,
                                   void *stream)
{
    BE42_CHECK(q && scales && x, "be42_quant_rows_fp8: null pointer");
    BE42_CHECK(rows >= 0 && cols > 0, "be42_quant_rows_fp8: bad shape %d x %d", rows, cols);
    int rc = ensure_thresholds();
    if (rc)
        return rc;
    if (rows == 0)
        return BE42_OK;
    if (!launch_quant_vec<true>(q, scales, x, rows, cols, as_stream(stream)))
        hipLaunchKernelGGL(k_quant_rows_fp8, dim3(rows), dim3(256), 0, as_stream(stream), q, scales, x, cols);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

extern "C" int be42_dequant_rows_int8(float *out, const int8_t *q, const float *scales, int rows,
                                      int cols, void *stream)
{
    BE42_CHECK(out && q && scales, "be42_dequant_rows_int8: null pointer");
    BE42_CHECK(rows >= 0 && cols > 0, "be42_dequant_rows_int8: bad shape");
    size_t total = (size_t)rows * cols;
    if (total == 0)
        return BE42_OK;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 8192)
        blocks = 8192;
    hipLaunchKernelGGL(k_dequant_rows_int8, dim3(blocks), dim3(256), 0, as_stream(stream), out, q, scales,
                       cols, total);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

extern "C" int be42_fp8_decode(float *out, const uint8_t *q, size_t n, void *stream)
{
    BE42_CHECK(out && q, "be42_fp8_decode: null pointer");
    if (n == 0)
        return BE42_OK;
    int blocks = (int)((n + 255) / 256);
    if (blocks > 8192)
        blocks = 8192;
    hipLaunchKernelGGL(k_fp8_decode, dim3(blocks), dim3(256), 0, as_stream(stream), out, q, n);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}
