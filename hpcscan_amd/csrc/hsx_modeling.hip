// Modeling kernels: point sources and receivers (the reference's
// DataAcquisition, src/data_Acquisition.cpp:58-305), the imaging condition of
// the adjoint, and the low-precision checkpoint codec.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "hsx_internal.h"
#include "hsx_step_end.h"

namespace hsx {

// ---- sources / receivers ------------------------------------------------------------
// u[idx[i]] (+)= scale * val[i] * (w ? w[i] : 1); indices are distinct within one call;
// an index outside [0, npoint) is skipped (the host checks them where it builds them)
template <typename TS>
__global__ void __launch_bounds__(256) k_inject(TS *u, int64_t npoint, int64_t n, const int64_t *idx, const TS *val,
                                                const TS *w, double scale, int mode)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if ((uint64_t)idx[i] >= (uint64_t)npoint) continue;
        double v = scale * (double)val[i];
        if (w) v *= (double)w[i];
        TS *p = u + idx[i];
        *p = mode == HSX_INJECT_SET ? (TS)v : (TS)((double)*p + v);
    }
}

// out[i] = u[idx[i]]; 0 for an index outside [0, npoint)
template <typename TS>
__global__ void __launch_bounds__(256) k_gather(const TS *u, int64_t npoint, int64_t n, const int64_t *idx, TS *out)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = idx[i];
        out[i] = (uint64_t)j < (uint64_t)npoint ? u[j] : (TS)0;
    }
}

// ---- imaging condition -----------------------------------------------------------
// grad[ii] += scale * mu[ii] * (un[ii] - 2 u[ii] + up[ii] - f(ii)) in double over
// the box, f = src_val at src_idx (the source term of that step), 0 elsewhere.
template <typename TS>
__global__ void __launch_bounds__(256) k_imaging(double *grad, const TS *mu, const TS *un, const TS *u, const TS *up,
                                                 Box b, int64_t n1, int64_t n12, double scale, int64_t src_idx,
                                                 double src_val)
{
    const int64_t N1 = b.n1(), N2 = b.n2(), rows = N2 * b.n3();
    for (int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.y; row < rows; row += (int64_t)gridDim.x * 4) {
        const int64_t base = (b.s2 + row % N2) * n1 + (b.s3 + row / N2) * n12 + b.s1;
        for (int64_t k = threadIdx.x; k < N1; k += 64) {
            const int64_t ii = base + k;
            double d2 = ((double)un[ii] - 2.0 * (double)u[ii]) + (double)up[ii];
            if (ii == src_idx) d2 -= src_val;
            grad[ii] += scale * (double)mu[ii] * d2;
        }
    }
}

// ---- checkpoint codec ------------------------------------------------------------
// A snapshot of n values is stored as n 16-bit codes after a 256-byte header
// holding the scale (float) and the max |value| (float):
//   code = round_to_format(v / scale), v = code * scale,
//   scale = maxabs / FORMAT_TARGET (1 if the snapshot is zero).
// Pair snapshots hold u_n and d = u_n - u_{n-1} (each with its own scale), so
// that the small step-to-step difference keeps its relative precision.
constexpr size_t CKPT_HEADER = 256;

__device__ __forceinline__ float fmt_target(int fmt) { return fmt == HSX_CKPT_FP16 ? 16384.f : 1.f; }

__device__ __forceinline__ uint16_t enc16(float x, int fmt)
{
    if (fmt == HSX_CKPT_FP16) return __half_as_ushort(__float2half_rn(x));
    return __bfloat16_as_ushort(__float2bfloat16(x));     // round to nearest even
}

__device__ __forceinline__ float dec16(uint16_t c, int fmt)
{
    if (fmt == HSX_CKPT_FP16) return __half2float(__ushort_as_half(c));
    return __bfloat162float(__ushort_as_bfloat16(c));
}

// The kernels take 16 bytes of floats at a time, in grid-stride loops over the
// groups, the last n % 4 values one by one; VEC: every buffer 16-byte aligned.
// PAIR: the two snapshots of a pair in one launch, u_n into p0 and u_n - u_{n-1}
// into p1, so that each wavefield is read once for the two.  Bound by memory;
// 208^3 FP32, a pair, us: clear 4.0 (two snapshots one after the other: 8), max
// 17 (51), encode 16 (24), decode 19 (45).
struct alignas(8) Code4 {
    uint16_t c[4];
};
typedef float Float4 __attribute__((ext_vector_type(4)));

template <bool VEC, typename F4, typename F1>
__device__ __forceinline__ void ckpt_loop(int64_t n, F4 &&four, F1 &&one)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    const int64_t ng = VEC ? n / 4 : 0;
    for (int64_t i = t; i < ng; i += step) four(i);
    for (int64_t i = 4 * ng + t; i < n; i += step) one(i);
}

// max |a - (b ? b : 0)| of the block into hdr[1] (as float bits; values are >= 0
// so the unsigned order of the bits is the float order)
__device__ __forceinline__ void ckpt_max(float m, unsigned *hdr_bits)
{
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    __shared__ float wm[4];
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; k++) m = fmaxf(m, wm[k]);
        atomicMax(hdr_bits + 1, __float_as_uint(m));
    }
}

template <bool PAIR, bool VEC>
__global__ void __launch_bounds__(256) k_ckpt_maxabs(const float *a, const float *b, int64_t n, unsigned *h0,
                                                     unsigned *h1)
{
    float m = 0.f, d = 0.f;
    auto value = [&](float x, float y) {
        m = fmaxf(m, fabsf(PAIR || !b ? x : x - y));
        if (PAIR) d = fmaxf(d, fabsf(x - y));
    };
    ckpt_loop<VEC>(
        n,
        [&](int64_t i) {
            const Float4 x = reinterpret_cast<const Float4 *>(a)[i];
            Float4 y = {};
            if (b) y = reinterpret_cast<const Float4 *>(b)[i];
#pragma unroll
            for (int e = 0; e < 4; e++) value(x[e], y[e]);
        },
        [&](int64_t i) { value(a[i], b ? b[i] : 0.f); });
    ckpt_max(m, h0);
    if (PAIR) ckpt_max(d, h1);
}

__device__ __forceinline__ float ckpt_scale(const char *packed, int fmt)
{
    const float maxabs = reinterpret_cast<const float *>(packed)[1];
    return maxabs > 0.f ? maxabs / fmt_target(fmt) : 1.f;
}

template <bool PAIR, bool VEC>
__global__ void __launch_bounds__(256) k_ckpt_encode(const float *a, const float *b, int64_t n, char *p0, char *p1,
                                                     int fmt)
{
    const float s0 = ckpt_scale(p0, fmt), s1 = PAIR ? ckpt_scale(p1, fmt) : 1.f;
    const float i0 = 1.f / s0, i1 = 1.f / s1;
    uint16_t *c0 = reinterpret_cast<uint16_t *>(p0 + CKPT_HEADER), *c1 = reinterpret_cast<uint16_t *>(p1 + CKPT_HEADER);
    ckpt_loop<VEC>(
        n,
        [&](int64_t i) {
            const Float4 x = reinterpret_cast<const Float4 *>(a)[i];
            Float4 y = {};
            if (b) y = reinterpret_cast<const Float4 *>(b)[i];
            Code4 u, v;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                u.c[e] = enc16((PAIR || !b ? x[e] : x[e] - y[e]) * i0, fmt);
                if (PAIR) v.c[e] = enc16((x[e] - y[e]) * i1, fmt);
            }
            reinterpret_cast<Code4 *>(c0)[i] = u;
            if (PAIR) reinterpret_cast<Code4 *>(c1)[i] = v;
        },
        [&](int64_t i) {
            const float x = a[i], y = b ? b[i] : 0.f;
            c0[i] = enc16((PAIR || !b ? x : x - y) * i0, fmt);
            if (PAIR) c1[i] = enc16((x - y) * i1, fmt);
        });
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        reinterpret_cast<float *>(p0)[0] = s0;
        if (PAIR) reinterpret_cast<float *>(p1)[0] = s1;
    }
}

// out = decoded, or base - decoded; PAIR: cur from p0 and cur - decoded p1 into out
template <bool PAIR, bool VEC>
__global__ void __launch_bounds__(256) k_ckpt_decode(const char *p0, const char *p1, int64_t n, int fmt,
                                                     const float *base, float *cur, float *out)
{
    const float s0 = reinterpret_cast<const float *>(p0)[0], s1 = PAIR ? reinterpret_cast<const float *>(p1)[0] : 1.f;
    const uint16_t *c0 = reinterpret_cast<const uint16_t *>(p0 + CKPT_HEADER);
    const uint16_t *c1 = reinterpret_cast<const uint16_t *>(p1 + CKPT_HEADER);
    ckpt_loop<VEC>(
        n,
        [&](int64_t i) {
            const Code4 u = reinterpret_cast<const Code4 *>(c0)[i];
            Code4 v = {};
            Float4 y = {}, x, o;
            if (PAIR) v = reinterpret_cast<const Code4 *>(c1)[i];
            if (!PAIR && base) y = reinterpret_cast<const Float4 *>(base)[i];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[e] = dec16(u.c[e], fmt) * s0;
                o[e] = PAIR ? x[e] - dec16(v.c[e], fmt) * s1 : base ? y[e] - x[e] : x[e];
            }
            if (PAIR) reinterpret_cast<Float4 *>(cur)[i] = x;
            reinterpret_cast<Float4 *>(out)[i] = o;
        },
        [&](int64_t i) {
            const float x = dec16(c0[i], fmt) * s0;
            if (PAIR) {
                cur[i] = x;
                out[i] = x - dec16(c1[i], fmt) * s1;
            } else {
                out[i] = base ? base[i] - x : x;
            }
        });
}

__global__ void k_ckpt_clear(unsigned *h0, unsigned *h1)
{
    if (threadIdx.x < 2) (blockIdx.x ? h1 : h0)[threadIdx.x] = 0u;
}

static unsigned blocks_for(int64_t n)
{
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 8192));
}

// k_ckpt_maxabs ends each block with one atomic on the same word: 512 blocks
// keep those few (8192 of them took ~97 us on a 208^3 grid, the pass itself ~10)
static unsigned blocks_for_max(int64_t n)
{
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 512));
}

template <bool PAIR>
static int ckpt_encode(const float *u, const float *u_prev, int64_t n, char *p0, char *p1, int format, hipStream_t s)
{
    const bool vec = ((uintptr_t)u | (uintptr_t)u_prev) % 16 == 0;
    const int64_t items = vec ? (n + 3) / 4 : n;
    unsigned *h0 = reinterpret_cast<unsigned *>(p0), *h1 = reinterpret_cast<unsigned *>(p1);
    hipLaunchKernelGGL(k_ckpt_clear, dim3(PAIR ? 2 : 1), dim3(64), 0, s, h0, h1);
    HSX_LAUNCHED("k_ckpt_clear");
    auto go = [&](auto v) -> int {
        constexpr bool VEC = decltype(v)::value;
        hipLaunchKernelGGL((k_ckpt_maxabs<PAIR, VEC>), dim3(blocks_for_max(items)), dim3(256), 0, s, u, u_prev, n, h0, h1);
        HSX_LAUNCHED("k_ckpt_maxabs");
        hipLaunchKernelGGL((k_ckpt_encode<PAIR, VEC>), dim3(blocks_for(items)), dim3(256), 0, s, u, u_prev, n, p0, p1,
                           format);
        HSX_LAUNCHED("k_ckpt_encode");
        return HSX_OK;
    };
    return vec ? go(std::true_type()) : go(std::false_type());
}

template <bool PAIR>
static int ckpt_decode(const char *p0, const char *p1, int64_t n, int format, const float *base, float *cur, float *out,
                       hipStream_t s)
{
    const bool vec = ((uintptr_t)base | (uintptr_t)cur | (uintptr_t)out) % 16 == 0;
    const unsigned nb = blocks_for(vec ? (n + 3) / 4 : n);
    if (vec)
        hipLaunchKernelGGL((k_ckpt_decode<PAIR, true>), dim3(nb), dim3(256), 0, s, p0, p1, n, format, base, cur, out);
    else
        hipLaunchKernelGGL((k_ckpt_decode<PAIR, false>), dim3(nb), dim3(256), 0, s, p0, p1, n, format, base, cur, out);
    HSX_LAUNCHED("k_ckpt_decode");
    return HSX_OK;
}

int ckpt_encode_pair(const float *u, const float *u_prev, int64_t n, void *p0, void *p1, int format, hipStream_t s)
{
    return ckpt_encode<true>(u, u_prev, n, (char *)p0, (char *)p1, format, s);
}

int ckpt_decode_pair(const void *p0, const void *p1, int64_t n, int format, float *u, float *u_prev, hipStream_t s)
{
    return ckpt_decode<true>((const char *)p0, (const char *)p1, n, format, nullptr, u, u_prev, s);
}

} // namespace hsx

using namespace hsx;

extern "C" {

// header + codes, rounded up to whole 256-byte units: snapshots stored back to
// back keep every header 256-byte aligned (its max |value| is updated with a
// 32-bit atomic)
size_t hsx_ckpt_bytes(int64_t n) { return CKPT_HEADER + ((size_t)n * 2 + CKPT_HEADER - 1) / CKPT_HEADER * CKPT_HEADER; }

int hsx_inject(const hsx_grid *g, void *u, int64_t n, const int64_t *idx, const void *val, const void *w,
               double scale, int mode, void *stream)
{
    int rc = check_grid(g);
    if (rc) return rc;
    if ((rc = check_ptr(u, "u")) || (rc = check_ptr(idx, "idx")) || (rc = check_ptr(val, "val"))) return rc;
    if (n < 0) return fail(HSX_ERR_INVALID, "n = %lld", (long long)n);
    if (mode != HSX_INJECT_ADD && mode != HSX_INJECT_SET) return fail(HSX_ERR_INVALID, "inject mode %d", mode);
    if ((rc = ensure_init())) return rc;
    if (n == 0) return HSX_OK;
    hipStream_t s = stream_of(stream);
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        hipLaunchKernelGGL(k_inject<TS>, dim3(blocks_for(n)), dim3(256), 0, s, (TS *)u, g->n1 * g->n2 * g->n3, n, idx,
                           (const TS *)val,
                           (const TS *)w, scale, mode);
        HSX_LAUNCHED("k_inject");
        return HSX_OK;
    });
}

int hsx_gather(const hsx_grid *g, const void *u, int64_t n, const int64_t *idx, void *out, void *stream)
{
    int rc = check_grid(g);
    if (rc) return rc;
    if ((rc = check_ptr(u, "u")) || (rc = check_ptr(idx, "idx")) || (rc = check_ptr(out, "out"))) return rc;
    if (n < 0) return fail(HSX_ERR_INVALID, "n = %lld", (long long)n);
    if ((rc = ensure_init())) return rc;
    if (n == 0) return HSX_OK;
    hipStream_t s = stream_of(stream);
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        hipLaunchKernelGGL(k_gather<TS>, dim3(blocks_for(n)), dim3(256), 0, s, (const TS *)u, g->n1 * g->n2 * g->n3, n,
                           idx, (TS *)out);
        HSX_LAUNCHED("k_gather");
        return HSX_OK;
    });
}

int hsx_imaging(const hsx_grid *g, double *grad, const void *mu, const void *u_next, const void *u, const void *u_prev,
                const int64_t range[6], double scale, int64_t src_idx, double src_val, void *stream)
{
    int rc = check_grid(g);
    if (rc) return rc;
    if ((rc = check_range(g, range))) return rc;
    if ((rc = check_ptr(grad, "grad")) || (rc = check_ptr(mu, "mu")) || (rc = check_ptr(u_next, "u_next")) ||
        (rc = check_ptr(u, "u")) || (rc = check_ptr(u_prev, "u_prev")))
        return rc;
    if ((rc = ensure_init())) return rc;
    const Box b = box_of(range);
    hipStream_t s = stream_of(stream);
    const int64_t rows = b.n2() * b.n3();
    const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>((rows + 3) / 4, 1 << 20));
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        hipLaunchKernelGGL(k_imaging<TS>, dim3(nb), dim3(64, 4), 0, s, grad, (const TS *)mu, (const TS *)u_next,
                           (const TS *)u, (const TS *)u_prev, b, g->n1, g->n1 * g->n2, scale, src_idx, src_val);
        HSX_LAUNCHED("k_imaging");
        return HSX_OK;
    });
}

int hsx_ckpt_encode(const float *u, const float *u_prev, int64_t n, void *packed, int format, void *stream)
{
    int rc;
    if ((rc = check_ptr(u, "u")) || (rc = check_ptr(packed, "packed"))) return rc;
    if (format != HSX_CKPT_FP16 && format != HSX_CKPT_BF16) return fail(HSX_ERR_INVALID, "format %d", format);
    if (n <= 0) return fail(HSX_ERR_INVALID, "n = %lld", (long long)n);
    if ((uintptr_t)packed % 16) return fail(HSX_ERR_INVALID, "packed snapshot not 16-byte aligned");
    if ((rc = ensure_init())) return rc;
    hipStream_t s = stream_of(stream);
    return ckpt_encode<false>(u, u_prev, n, (char *)packed, (char *)packed, format, s);
}

int hsx_ckpt_decode(const void *packed, int64_t n, int format, const float *base, float *out, void *stream)
{
    int rc;
    if ((rc = check_ptr(packed, "packed")) || (rc = check_ptr(out, "out"))) return rc;
    if (format != HSX_CKPT_FP16 && format != HSX_CKPT_BF16) return fail(HSX_ERR_INVALID, "format %d", format);
    if (n <= 0) return fail(HSX_ERR_INVALID, "n = %lld", (long long)n);
    if ((uintptr_t)packed % 16) return fail(HSX_ERR_INVALID, "packed snapshot not 16-byte aligned");
    if ((rc = ensure_init())) return rc;
    hipStream_t s = stream_of(stream);
    return ckpt_decode<false>((const char *)packed, (const char *)packed, n, format, base, nullptr, out, s);
}

} // extern "C"
