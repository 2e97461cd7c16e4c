// Stencil entry points of the C ABI and the reference-order kernels.
//
// Reference kernels: one thread per inner point, block 64 x 4 over (i1, i2),
// grid z over i3.  The per-point arithmetic is the reference macro order
// (src/fdm.h:281-545) with no contraction (built with -ffp-contract=off):
//   O2 : ((A0*u0 + u[+1]) + u[-1]) * inv2
//   O2R: ((A0*u0 + A1*(u[+1]+u[-1])) + ... + AR*(u[+R]+u[-R])) * inv2
// where each pair sum is done in the storage type (both operands are Myfloat).
// hsx_ac2_step / hsx_laplacian / hsx_fd_d2 use the LDS-tiled kernels of
// hsx_stencil_tiled.hip when the grid fits them, else these.
#include "hsx_internal.h"
#include "hsx_route.h"
#include "hsx_stencil_point.h"

namespace hsx {

constexpr int RX = 64, RY = 4;

template <typename TS, typename TC, int R>
__global__ void __launch_bounds__(RX *RY) k_fd_d2_ref(const TS *__restrict__ u, TS *__restrict__ w, Box b,
                                                      int64_t n1, int64_t n12, int64_t stride, Coefs<TC> c,
                                                      TC inv2)
{
    const int64_t i1 = b.s1 + (int64_t)blockIdx.x * RX + threadIdx.x;
    const int64_t i2 = b.s2 + (int64_t)blockIdx.y * RY + threadIdx.y;
    const int64_t i3 = b.s3 + blockIdx.z;
    if (i1 > b.e1 || i2 > b.e2) return;
    const int64_t ii = i1 + i2 * n1 + i3 * n12;
    w[ii] = (TS)d2_point<TS, TC, R>(u, ii, stride, c.A, inv2);
}

template <typename TS, typename TC, int R>
__global__ void __launch_bounds__(RX *RY) k_fd_d1_ref(const TS *__restrict__ u, TS *__restrict__ w, Box b,
                                                      int64_t n1, int64_t n12, int64_t stride, Coefs<TC> c,
                                                      TC inv)
{
    const int64_t i1 = b.s1 + (int64_t)blockIdx.x * RX + threadIdx.x;
    const int64_t i2 = b.s2 + (int64_t)blockIdx.y * RY + threadIdx.y;
    const int64_t i3 = b.s3 + blockIdx.z;
    if (i1 > b.e1 || i2 > b.e2) return;
    const int64_t ii = i1 + i2 * n1 + i3 * n12;
    w[ii] = (TS)d1_point<TS, TC, R>(u, ii, stride, c.D1, inv);
}

template <typename TS, typename TC, int R, int DIM>
__global__ void __launch_bounds__(RX *RY) k_laplacian_ref(const TS *__restrict__ u, TS *__restrict__ w, Box b,
                                                          int64_t n1, int64_t n12, Coefs<TC> c)
{
    const int64_t i1 = b.s1 + (int64_t)blockIdx.x * RX + threadIdx.x;
    const int64_t i2 = b.s2 + (int64_t)blockIdx.y * RY + threadIdx.y;
    const int64_t i3 = b.s3 + blockIdx.z;
    if (i1 > b.e1 || i2 > b.e2) return;
    const int64_t ii = i1 + i2 * n1 + i3 * n12;
    w[ii] = (TS)laplacian_point<TS, TC, R, DIM>(u, ii, n1, n12, c);
}

// out = 2 prc - prn + coef * Lap(prc); out may be prn (the in-place step)
template <typename TS, typename TC, int R, int DIM>
__global__ void __launch_bounds__(RX *RY) k_ac2_ref(TS *out, const TS *prn, const TS *__restrict__ prc,
                                                    const TS *__restrict__ coef, Box b, int64_t n1, int64_t n12,
                                                    Coefs<TC> c)
{
    const int64_t i1 = b.s1 + (int64_t)blockIdx.x * RX + threadIdx.x;
    const int64_t i2 = b.s2 + (int64_t)blockIdx.y * RY + threadIdx.y;
    const int64_t i3 = b.s3 + blockIdx.z;
    if (i1 > b.e1 || i2 > b.e2) return;
    const int64_t ii = i1 + i2 * n1 + i3 * n12;
    const TC lap = laplacian_point<TS, TC, R, DIM>(prc, ii, n1, n12, c);
    out[ii] = leapfrog<TS, TC>(prc[ii], prn[ii], coef[ii], lap);
}

// ---- 2D grids: the fused step and the Laplacian in vectors -------------------------
// One lane computes VW = 16 bytes of points along n1 in RY consecutive rows: the
// RY + 2R rows it needs are loaded once each (16-byte loads, the n2 sums from
// registers), the n1 neighbours as the vectors beside the row's own, which the
// neighbouring lanes load too (L1).  That is (RY + 2R) / RY + 2 loads per 16
// bytes instead of 4R + 1 per value.  These grids lie in the caches, and what
// bounds them is the halo rows: dealt round robin, neighbouring rows go to
// different XCDs and each L2 fetches them again, so each XCD takes a contiguous
// run of rows (1501 x 2001 order 8 FP32 12.6 -> 8.3 us; one thread per point
// 12.9).  FP64 order 16 38 -> 20 us, 6000 x 6000 FP32 order 8 172 -> 116 us.
// Vectors count back from the row's end (t1s, down to -(VW - 1)), so that none
// reaches past it; one that starts before the row takes in the end of the row
// before, except in row 0, where its points inside the row are loaded one by one.
template <typename TS, typename TC, int R, int RY, bool AC2>
__global__ void __launch_bounds__(256) k_plane(TS *out, const TS *prn, const TS *__restrict__ u,
                                               const TS *__restrict__ coef, Box b, int64_t n1, int64_t t1s,
                                               uint32_t lanes, Coefs<TC> c)
{
    constexpr int VW = 16 / sizeof(TS), NHG = (R + VW - 1) / VW, HL = NHG * VW;
    struct V { TS v[VW]; };
    // each XCD takes a contiguous run of rows, whose halo rows then meet in its L2
    const uint32_t per_xcd = (gridDim.x + 7) / 8, blk = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;
    const uint32_t t = blk * 256u + threadIdx.x, band = t / lanes;
    const int64_t i1 = t1s + (int64_t)(t - band * lanes) * VW;
    const int64_t r0 = b.s2 + (int64_t)band * RY;
    if (r0 > b.e2) return;
    auto load = [&](const TS *p) {
        V x;
        __builtin_memcpy(&x, p, sizeof(x));
        return x;
    };
    // every load first (rows past the grid's need are read as its last one, so
    // that no branch holds a load back), then the sums
    V col[RY + 2 * R], side[RY][2 * NHG], pv[RY], cv[RY];
    if (i1 >= 0 || r0 > R) {
#pragma unroll
        for (int k = 0; k < RY + 2 * R; k++) col[k] = load(u + min(r0 - R + k, b.e2 + R) * n1 + i1);
    } else {
#pragma unroll
        for (int k = 0; k < RY + 2 * R; k++) {
            const int64_t ii = min(r0 - R + k, b.e2 + R) * n1 + i1;
#pragma unroll
            for (int v = 0; v < VW; v++) col[k].v[v] = ii + v >= 0 ? u[ii + v] : (TS)0;
        }
    }
#pragma unroll
    for (int y = 0; y < RY; y++) {
        const int64_t row = min(r0 + y, b.e2) * n1;            // >= n1: a vector may start before the row
#pragma unroll
        for (int g = 0; g < NHG; g++) {
            // groups that hold no point of the row hold no neighbour either
            const int64_t jl = max(i1 - (NHG - g) * VW, (int64_t)(1 - VW)), jr = min(i1 + (g + 1) * VW, n1 - VW);
            side[y][g] = load(u + row + jl);
            side[y][NHG + g] = load(u + row + jr);
        }
        if (AC2) {
            pv[y] = load(prn + row + i1);
            cv[y] = load(coef + row + i1);
        }
    }
    bool all = true;
#pragma unroll
    for (int v = 0; v < VW; v++) all &= i1 + v >= b.s1 && i1 + v <= b.e1;
#pragma unroll
    for (int y = 0; y < RY; y++) {
        TS xr[2 * HL + VW];
#pragma unroll
        for (int g = 0; g < NHG; g++)
#pragma unroll
            for (int v = 0; v < VW; v++) {
                xr[g * VW + v] = side[y][g].v[v];
                xr[HL + VW + g * VW + v] = side[y][NHG + g].v[v];
            }
#pragma unroll
        for (int v = 0; v < VW; v++) xr[HL + v] = col[y + R].v[v];
        V res;
#pragma unroll
        for (int v = 0; v < VW; v++) {
            TS pp[R], mm[R];
#pragma unroll
            for (int j = 1; j <= R; j++) {
                pp[j - 1] = xr[HL + v + j];
                mm[j - 1] = xr[HL + v - j];
            }
            const TS c0 = xr[HL + v];
            const TC d1 = d2_values<TS, TC, R>(c0, pp, mm, c.A, c.inv2[0]);
#pragma unroll
            for (int j = 1; j <= R; j++) {
                pp[j - 1] = col[y + R + j].v[v];
                mm[j - 1] = col[y + R - j].v[v];
            }
            const TC lap = d1 + d2_values<TS, TC, R>(c0, pp, mm, c.A, c.inv2[1]);
            res.v[v] = AC2 ? leapfrog<TS, TC>(c0, pv[y].v[v], cv[y].v[v], lap) : (TS)lap;
        }
        if (r0 + y > b.e2) break;
        TS *o = out + ((r0 + y) * n1 + i1);
        if (all) {
            __builtin_memcpy(o, &res, sizeof(res));
        } else {
#pragma unroll
            for (int v = 0; v < VW; v++)
                if (i1 + v >= b.s1 && i1 + v <= b.e1) o[v] = res.v[v];
        }
    }
}

// waves = 16-byte vectors of the inner points / 64.  Below 1500 of them one
// thread per point (4 times the waves) is as fast: 501 x 501 FP32 order 8 4.0
// us against 4.2; 701 x 701 (1927) 4.25 / 4.20, 1001 x 1001 (3915) 5.9 / 4.3.
// Four rows per lane from 8192 on, two below: 5000 x 300 order 12 (5859) 6.7 us
// with four, 5.9 with two; 1501 x 2001 order 8 (11725) 8.3 with four, 8.7 with
// two, 10.3 with one; 6000 x 6000 116 / 133 / 155, and 111 with eight, which
// are slower below (3000 x 3000 23.9 against 21.2).
template <bool AC2>
static int run_plane(const hsx_grid *g, void *out, const void *prn, const void *u, const void *coef, hipStream_t s)
{
    const Box b = box_of(g->inner);
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        constexpr int VW = 16 / sizeof(TS);
        const Coefs<TC> c = make_coefs<TC>(g);
        const int64_t t1s = b.s1 - (b.s1 + VW - g->n1 % VW) % VW;
        const int64_t lanes = (b.e1 - t1s) / VW + 1;
        const int64_t waves = lanes * b.n2() / 64;
        if (waves < 1500) return HSX_ERR_UNSUPPORTED;
        const int ry = waves >= 8192 ? 4 : 2;
        const int64_t threads = lanes * ((b.n2() + ry - 1) / ry);
        if (threads >= ((int64_t)1 << 31) || g->n1 < VW) return fail(HSX_ERR_UNSUPPORTED, "2D kernel: grid size");
        return dispatch_R(g->fd_order / 2, [&](auto rc_) -> int {
            constexpr int R = decltype(rc_)::value;
            const dim3 grid((unsigned)((threads + 2047) / 2048 * 8));     // whole XCD rounds
            auto go = [&](auto ryc) {
                hipLaunchKernelGGL((k_plane<TS, TC, R, decltype(ryc)::value, AC2>), grid, dim3(256), 0, s, (TS *)out,
                                   (const TS *)prn, (const TS *)u, (const TS *)coef, b, g->n1, t1s, (uint32_t)lanes, c);
            };
            if (ry == 4)
                go(IC<4>());
            else
                go(IC<2>());
            HSX_LAUNCHED("k_plane");
            return HSX_OK;
        });
    });
}

static int ref_grid(const Box &b, dim3 &grid)
{
    if (b.n3() > 65535) return fail(HSX_ERR_UNSUPPORTED, "n3 inner %lld > 65535", (long long)b.n3());
    grid = dim3((unsigned)((b.n1() + RX - 1) / RX), (unsigned)((b.n2() + RY - 1) / RY), (unsigned)b.n3());
    return HSX_OK;
}

int ac2_step_points(const hsx_grid *g, void *out, const void *prn, const void *prc, const void *coef, hipStream_t s)
{
    const Box b = box_of(g->inner);
    dim3 grid;
    const int rc = ref_grid(b, grid);
    if (rc) return rc;
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        const Coefs<TC> c = make_coefs<TC>(g);
        return dispatch_R(g->fd_order / 2, [&](auto rc_) -> int {
            constexpr int R = decltype(rc_)::value;
            return dispatch_dim(g->dim, [&](auto dc) -> int {
                constexpr int DIM = decltype(dc)::value;
                hipLaunchKernelGGL((k_ac2_ref<TS, TC, R, DIM>), grid, dim3(RX, RY), 0, s, (TS *)out,
                                   (const TS *)prn, (const TS *)prc, (const TS *)coef, b, g->n1, g->n1 * g->n2, c);
                HSX_LAUNCHED("k_ac2_ref");
                return HSX_OK;
            });
        });
    });
}

static int stencil_checks(const hsx_grid *g, std::initializer_list<std::pair<const void *, const char *>> ptrs)
{
    int rc = check_grid(g);
    for (auto &p : ptrs)
        if (!rc) rc = check_ptr(p.first, p.second);
    if (!rc) rc = ensure_init();
    return rc;
}

} // namespace hsx

using namespace hsx;

extern "C" {

int hsx_fd_d2(const hsx_grid *g, int axis, const void *u, void *w, void *stream)
{
    int rc = stencil_checks(g, {{u, "u"}, {w, "w"}});
    if (rc) return rc;
    if (axis < 0 || axis >= g->dim) return fail(HSX_ERR_INVALID, "axis %d with dim %d", axis, g->dim);
    hipStream_t s = stream_of(stream);
    if (kernel_family() != HSX_KERNEL_REF && tiled_pays(g)) {
        rc = tiled_fd_d2(g, axis, u, w, s);
        if (rc != HSX_ERR_UNSUPPORTED || kernel_family() == HSX_KERNEL_TILED) return rc;
    }
    const Box b = box_of(g->inner);
    dim3 grid;
    if ((rc = ref_grid(b, grid))) return rc;
    const int64_t stride = axis == 0 ? 1 : axis == 1 ? g->n1 : g->n1 * g->n2;
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        const Coefs<TC> c = make_coefs<TC>(g);
        return dispatch_R(g->fd_order / 2, [&](auto rc_) -> int {
            constexpr int R = decltype(rc_)::value;
            hipLaunchKernelGGL((k_fd_d2_ref<TS, TC, R>), grid, dim3(RX, RY), 0, s, (const TS *)u, (TS *)w, b,
                               g->n1, g->n1 * g->n2, stride, c, c.inv2[axis]);
            HSX_LAUNCHED("k_fd_d2_ref");
            return HSX_OK;
        });
    });
}

int hsx_fd_d1(const hsx_grid *g, int axis, const void *u, void *w, void *stream)
{
    int rc = stencil_checks(g, {{u, "u"}, {w, "w"}});
    if (rc) return rc;
    if (axis < 0 || axis >= g->dim) return fail(HSX_ERR_INVALID, "axis %d with dim %d", axis, g->dim);
    hipStream_t s = stream_of(stream);
    if (kernel_family() != HSX_KERNEL_REF && tiled_pays(g)) {
        rc = tiled_fd_d1(g, axis, u, w, s);
        if (rc != HSX_ERR_UNSUPPORTED || kernel_family() == HSX_KERNEL_TILED) return rc;
    }
    const Box b = box_of(g->inner);
    dim3 grid;
    if ((rc = ref_grid(b, grid))) return rc;
    const int64_t stride = axis == 0 ? 1 : axis == 1 ? g->n1 : g->n1 * g->n2;
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        const Coefs<TC> c = make_coefs<TC>(g);
        return dispatch_R(g->fd_order / 2, [&](auto rc_) -> int {
            constexpr int R = decltype(rc_)::value;
            hipLaunchKernelGGL((k_fd_d1_ref<TS, TC, R>), grid, dim3(RX, RY), 0, s, (const TS *)u, (TS *)w, b,
                               g->n1, g->n1 * g->n2, stride, c, c.inv[axis]);
            HSX_LAUNCHED("k_fd_d1_ref");
            return HSX_OK;
        });
    });
}

int hsx_laplacian(const hsx_grid *g, const void *u, void *w, void *stream)
{
    int rc = stencil_checks(g, {{u, "u"}, {w, "w"}});
    if (rc) return rc;
    hipStream_t s = stream_of(stream);
    if (kernel_family() != HSX_KERNEL_REF && tiled_pays(g)) {
        rc = tiled_laplacian(g, u, w, s);
        if (rc != HSX_ERR_UNSUPPORTED || kernel_family() == HSX_KERNEL_TILED) return rc;
    }
    const Box b = box_of(g->inner);
    dim3 grid;
    if (g->dim == 2 && kernel_family() != HSX_KERNEL_REF) {
        rc = run_plane<false>(g, w, nullptr, u, nullptr, s);
        if (rc != HSX_ERR_UNSUPPORTED) return rc;
    }
    if ((rc = ref_grid(b, grid))) return rc;
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        const Coefs<TC> c = make_coefs<TC>(g);
        return dispatch_R(g->fd_order / 2, [&](auto rc_) -> int {
            constexpr int R = decltype(rc_)::value;
            return dispatch_dim(g->dim, [&](auto dc) -> int {
                constexpr int DIM = decltype(dc)::value;
                hipLaunchKernelGGL((k_laplacian_ref<TS, TC, R, DIM>), grid, dim3(RX, RY), 0, s, (const TS *)u,
                                   (TS *)w, b, g->n1, g->n1 * g->n2, c);
                HSX_LAUNCHED("k_laplacian_ref");
                return HSX_OK;
            });
        });
    });
}

int hsx_ac2_step(const hsx_grid *g, void *prn, const void *prc, const void *coef, void *stream)
{
    return hsx_ac2_step_to(g, prn, prn, prc, coef, stream);
}

int hsx_ac2_step_to(const hsx_grid *g, void *out, const void *prn, const void *prc, const void *coef, void *stream)
{
    int rc = stencil_checks(g, {{out, "out"}, {prn, "prn"}, {prc, "prc"}, {coef, "coef"}});
    if (rc) return rc;
    if (prn == prc || out == prc) return fail(HSX_ERR_INVALID, "prn / out and prc must be different grids");
    hipStream_t s = stream_of(stream);
    if (kernel_family() != HSX_KERNEL_REF && step_tiled(g)) {
        rc = tiled_ac2_step(g, out, prn, prc, coef, s);
        if (rc != HSX_ERR_UNSUPPORTED || kernel_family() == HSX_KERNEL_TILED) return rc;
    }
    if (g->dim == 2 && kernel_family() != HSX_KERNEL_REF) {
        rc = run_plane<true>(g, out, prn, prc, coef, s);
        if (rc != HSX_ERR_UNSUPPORTED) return rc;
    }
    return ac2_step_points(g, out, prn, prc, coef, s);
}

int hsx_ac2_step_fs(const hsx_grid *g, void *prn, const void *prc, const void *coef, int face_mask, int fold,
                    void *stream)
{
    if (fold & ~(HSX_FOLD_PRC | HSX_FOLD_PRN | HSX_FOLD_HALO)) return fail(HSX_ERR_INVALID, "fold flags 0x%x", fold);
    if (fold == 0) return hsx_ac2_step(g, prn, prc, coef, stream);
    int rc = stencil_checks(g, {{prn, "prn"}, {prc, "prc"}, {coef, "coef"}});
    if (rc) return rc;
    if (prn == prc) return fail(HSX_ERR_INVALID, "prn and prc must be different grids");
    if (g->dim != 3 || kernel_family() == HSX_KERNEL_REF)
        return fail(HSX_ERR_UNSUPPORTED, "folded free surface: 3D grids on the tiled kernels only");
    FaceSet fs;
    bool closed = false;
    int64_t most = 0, most_plane = 0;
    if ((rc = make_faceset(g, face_mask, &fs, &closed, &most, &most_plane))) return rc;
    if (!closed) return fail(HSX_ERR_UNSUPPORTED, "folded free surface: fewer than R+2 inner points on an axis");
    int64_t fb[6];
    for (int k = 0; k < 6; k++) fb[k] = (fs.zmask >> k) & 1 ? fs.zidx[k / 2][k % 2] : -1;
    return tiled_ac2_step_fold(g, prn, prc, coef, fold, fb, stream_of(stream));
}

} // extern "C"
