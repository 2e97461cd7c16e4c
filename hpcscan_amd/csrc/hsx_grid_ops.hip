// Grid operations of the C ABI other than the stencils: fills, array
// operations, the free-surface boundary, the leapfrog update and the
// double-precision reductions.
//
// These are HBM-streaming passes: one thread per value, rows of the index box
// mapped to waves so that n1 (contiguous) runs across the 64 lanes.
#include <algorithm>
#include <cfloat>
#include <mutex>

#include "hsx_internal.h"
#include "hsx_step_end.h"

namespace hsx {

constexpr int ROW_THREADS = 64;   // one wave per row
constexpr int ROWS_PER_BLOCK = 4; // 256 threads

static dim3 row_grid(const Box &b)
{
    const int64_t rows = b.n2() * b.n3();
    int64_t nb = (rows + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    return dim3((unsigned)(nb > 65535 * 16 ? 65535 * 16 : nb));
}

// Visit every point of box b: f(flat index, i1, i2, i3)
template <typename F>
__device__ inline void for_box(const Box &b, int64_t n1, int64_t n12, F &&f)
{
    const int64_t N1 = b.n1(), N2 = b.n2(), rows = N2 * b.n3();
    for (int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.y; row < rows;
         row += (int64_t)gridDim.x * ROWS_PER_BLOCK) {
        const int64_t i2 = b.s2 + row % N2, i3 = b.s3 + row / N2;
        const int64_t base = i2 * n1 + i3 * n12;
        for (int64_t k = threadIdx.x; k < N1; k += ROW_THREADS) {
            const int64_t i1 = b.s1 + k;
            f(base + i1, i1, i2, i3);
        }
    }
}

// Visit box b row by row in 16-byte groups of VW points (flat indices aligned
// to VW, so the buffer must be 16-byte aligned): group(ii, i1, i2, i3) for each
// whole group inside the row's [s1, e1] span (points ii .. ii + VW - 1, i1 the
// first one's n1 index), point(ii, i1, i2, i3) for the unaligned head and tail
// points of the row.  One wave per row, as for_box.
template <int VW, typename FP, typename FG>
__device__ inline void for_box_groups(const Box &b, int64_t n1, int64_t n12, FP &&point, FG &&group)
{
    const int64_t N2 = b.n2(), rows = N2 * b.n3();
    const int lane = threadIdx.x;
    for (int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.y; row < rows;
         row += (int64_t)gridDim.x * ROWS_PER_BLOCK) {
        const int64_t i2 = b.s2 + row % N2, i3 = b.s3 + row / N2;
        const int64_t base = i2 * n1 + i3 * n12;
        const int64_t a0 = base + b.s1, a1 = base + b.e1 + 1;       // [a0, a1) flat
        const int64_t g0 = (a0 + VW - 1) / VW, g1 = a1 / VW;          // whole groups
        if (g0 >= g1) {
            for (int64_t i = a0 + lane; i < a1; i += ROW_THREADS) point(i, i - base, i2, i3);
            continue;
        }
        const int64_t h = g0 * VW - a0, t = a1 - g1 * VW;
        if (lane < h) point(a0 + lane, a0 + lane - base, i2, i3);
        if (lane < t) point(g1 * VW + lane, g1 * VW + lane - base, i2, i3);
        for (int64_t gi = g0 + lane; gi < g1; gi += ROW_THREADS) group(gi * VW, gi * VW - base, i2, i3);
    }
}

// ---- fills (src/grid.cpp:1650-1826) -----------------------------------------
// VEC: 16-byte stores (u 16-byte aligned)
template <typename TS, bool VEC>
__global__ void __launch_bounds__(256) k_fill_const(TS *u, Box b, int64_t n1, int64_t n12, TS val)
{
    if constexpr (!VEC) {
        for_box(b, n1, n12, [&](int64_t ii, int64_t, int64_t, int64_t) { u[ii] = val; });
    } else {
        constexpr int VW = 16 / sizeof(TS);
        using NV = TS __attribute__((ext_vector_type(VW)));
        const NV vv = (NV)val;
        for_box_groups<VW>(
            b, n1, n12, [&](int64_t ii, int64_t, int64_t, int64_t) { u[ii] = val; },
            [&](int64_t ii, int64_t, int64_t, int64_t) { *reinterpret_cast<NV *>(u + ii) = vv; });
    }
}

// amp * v1 * v2 * v3 left to right in double, then rounded to the storage type
template <typename TS, bool VEC>
__global__ void __launch_bounds__(256) k_fill_sep(TS *u, Box b, int64_t n1, int64_t n12, const double *t1,
                                                  const double *t2, const double *t3, double amp)
{
    auto one = [&](int64_t i1, int64_t i2, int64_t i3) -> TS {
        return (TS)(amp * t1[i1 - b.s1] * t2[i2 - b.s2] * t3[i3 - b.s3]);
    };
    if constexpr (!VEC) {
        for_box(b, n1, n12, [&](int64_t ii, int64_t i1, int64_t i2, int64_t i3) { u[ii] = one(i1, i2, i3); });
    } else {
        constexpr int VW = 16 / sizeof(TS);
        using NV = TS __attribute__((ext_vector_type(VW)));
        for_box_groups<VW>(
            b, n1, n12, [&](int64_t ii, int64_t i1, int64_t i2, int64_t i3) { u[ii] = one(i1, i2, i3); },
            [&](int64_t ii, int64_t i1, int64_t i2, int64_t i3) {
                NV r;
#pragma unroll
                for (int e = 0; e < VW; e++) r[e] = one(i1 + e, i2, i3);
                *reinterpret_cast<NV *>(u + ii) = r;
            });
    }
}

// ---- array operations (src/grid.cpp:1830-1920) --------------------------------
template <typename TS>
__device__ __forceinline__ void array_elem(int op, TS *w, const TS *u, const TS *v, TS val, int64_t i)
{
    switch (op) {
    case HSX_ARRAY_FILL: w[i] = val; break;
    case HSX_ARRAY_COPY: w[i] = u[i]; break;
    case HSX_ARRAY_ADD: w[i] = u[i] + v[i]; break;
    case HSX_ARRAY_MULTIPLY: w[i] = u[i] * v[i]; break;
    default: w[i] = w[i] + u[i]; break;
    }
}

// 16-byte vectors per lane when every pointer is 16-byte aligned (the usual
// case: whole grids from hsx_malloc), element loop for the tail
template <typename TS>
__global__ void __launch_bounds__(256) k_array16(int op, TS *w, const TS *u, const TS *v, TS val, int64_t n)
{
    constexpr int VW = 16 / sizeof(TS);
    struct alignas(16) V { TS x[VW]; };
    const int64_t nv = n / VW;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += (int64_t)gridDim.x * blockDim.x) {
        V r, a, b;
        if (op != HSX_ARRAY_FILL) a = reinterpret_cast<const V *>(u)[i];
        if (op == HSX_ARRAY_ADD || op == HSX_ARRAY_MULTIPLY) b = reinterpret_cast<const V *>(v)[i];
        if (op == HSX_ARRAY_ADDTO) r = reinterpret_cast<const V *>(w)[i];
#pragma unroll
        for (int k = 0; k < VW; k++) {
            switch (op) {
            case HSX_ARRAY_FILL: r.x[k] = val; break;
            case HSX_ARRAY_COPY: r.x[k] = a.x[k]; break;
            case HSX_ARRAY_ADD: r.x[k] = a.x[k] + b.x[k]; break;
            case HSX_ARRAY_MULTIPLY: r.x[k] = a.x[k] * b.x[k]; break;
            default: r.x[k] = r.x[k] + a.x[k]; break;
            }
        }
        reinterpret_cast<V *>(w)[i] = r;
    }
    for (int64_t i = nv * VW + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        array_elem(op, w, u, v, val, i);
}

template <typename TS>
__global__ void __launch_bounds__(256) k_array(int op, TS *w, const TS *u, const TS *v, TS val, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        array_elem(op, w, u, v, val, i);
}

// ---- free surface, one face (src/grid.cpp:3065-3230) ---------------------------
// For every row of the two other axes: u[inner] = 0 and u[i] = -u[2*inner - i]
// for i in the halo range.  Sources are inner points at distance >= 1 from the
// zeroed plane and no halo point is a source, so one face is a parallel map;
// faces run one after the other, in the reference order.
template <typename TS>
__global__ void __launch_bounds__(256) k_free_surface(TS *u, Face f)
{
    const int64_t H = f.he - f.hs + 2;           // zero + halo points per row
    const int64_t NB = f.be - f.bs + 1, NO = f.oe - f.os + 1;
    const int64_t total = H * NB * NO;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        int64_t k, ib, io;
        if (f.axis == 0) {                        // face axis contiguous: k fastest
            k = t % H;
            ib = (t / H) % NB;
            io = t / (H * NB);
        } else {                                  // i1 contiguous: i1 fastest
            ib = t % NB;
            k = (t / NB) % H;
            io = t / (NB * H);
        }
        const int64_t base = (f.os + io) * f.so + (f.bs + ib) * f.sb;
        if (k == 0) {
            u[base + f.inner * f.sa] = (TS)0.0;
        } else {
            const int64_t i = f.hs + k - 1;
            u[base + i * f.sa] = -u[base + (2 * f.inner - i) * f.sa];
        }
    }
}

// ---- free surface, all faces in two launches -------------------------------------
// The six sequential phases of the reference (I1HALO1, I1HALO2, I2HALO1, ... each
// zeroing its boundary plane then mirroring) have a closed form when every
// active axis has at least R+2 inner points, so that a mirror source never
// reaches the far boundary plane or a halo:
//  * halo point p of face (a, side), mirror m:  u[p] = -0 if some face of an
//    axis a' < a in the mask has its boundary plane through p (p and m share
//    that coordinate; the plane was zeroed before phase a), else -u_old[m];
//  * then every boundary plane of the mask is zero.
// A halo point is written once and mirrors read only inner points that the
// first launch does not write, so the first launch has no ordering inside it,
// and the second launch (the planes) only writes inner points.
// The face loops index with IT = uint32_t when the face fits (always, below
// 65536^2 points per face): the 64-bit divisions otherwise dominate these
// kernels, which move only a few bytes per index.
// bx / nbx: this block's index and the number of blocks sharing the face (a
// launch may give other blocks other work).
template <typename TS, typename IT>
__device__ __forceinline__ void bc_mirror_loop(TS *u, const FaceSet &fs, const Face &f, IT H, IT NB, IT total,
                                               uint32_t bx, uint32_t nbx)
{
    const int a = f.axis;
    const int oa = a == 2 ? 1 : 2, ob = a == 0 ? 1 : 0;
    for (IT t = (IT)bx * blockDim.x + threadIdx.x; t < total; t += (IT)nbx * blockDim.x) {
        IT k, ib, io;
        if (a == 0) {
            const IT r = t / H;
            k = t - r * H;
            io = r / NB;
            ib = r - io * NB;
        } else {
            const IT r = t / NB;
            ib = t - r * NB;
            io = r / H;
            k = r - io * H;
        }
        int64_t c[3];
        c[a] = f.hs + (int64_t)k;
        c[oa] = f.os + (int64_t)io;
        c[ob] = f.bs + (int64_t)ib;
        bool zero = false;
        for (int ap = 0; ap < a; ap++)
            for (int sp = 0; sp < 2; sp++)
                if ((fs.zmask >> (2 * ap + sp)) & 1) zero |= c[ap] == fs.zidx[ap][sp];
        const int64_t base = c[oa] * f.so + c[ob] * f.sb;
        const int64_t i = c[a];
        u[base + i * f.sa] = zero ? -(TS)0.0 : -u[base + (2 * f.inner - i) * f.sa];
    }
}

// n2 / n3 faces with 16-byte groups along n1 (fs.vec1): one thread per group of a
// halo row; the elements of an edge group outside the face's n1 range are left
// alone (scalar stores there), the -0 rule is applied per element for the n1
// boundary planes and per row for the n2 ones. 1000^3 FP32 order 8, mirror and
// zero: n2 faces 0.020 ms, n3 faces 0.020 ms, against 0.033 / 0.035 ms with one
// point per thread.
template <typename TS>
__device__ __forceinline__ void bc_mirror_vec(TS *u, const FaceSet &fs, const Face &f, uint32_t bx, uint32_t nbx)
{
    constexpr int VW = 16 / sizeof(TS);
    using NV = TS __attribute__((ext_vector_type(VW)));
    const int a = f.axis;                          // 1 or 2; n1 is the inner-other axis (stride 1)
    const int64_t g0 = f.bs / VW;
    const uint32_t NG = (uint32_t)(f.be / VW - g0 + 1), H = (uint32_t)(f.he - f.hs + 1);
    const uint32_t total = NG * H * (uint32_t)(f.oe - f.os + 1);
    const bool z1lo = fs.zmask & 1, z1hi = fs.zmask & 2;
    for (uint32_t t = bx * blockDim.x + threadIdx.x; t < total; t += nbx * blockDim.x) {
        const uint32_t r = t / NG, g = t - r * NG;
        const uint32_t io = r / H, k = r - io * H;
        const int64_t i = f.hs + (int64_t)k;       // halo index along the face axis
        const int64_t o = f.os + (int64_t)io;      // index along the outer axis
        // -0 for the whole row: its n2 coordinate on a folded n2 boundary plane (n3 faces)
        bool zrow = false;
        if (a == 2)
            for (int sp = 0; sp < 2; sp++)
                if ((fs.zmask >> (2 + sp)) & 1) zrow |= o == fs.zidx[1][sp];
        const int64_t i1 = (g0 + (int64_t)g) * VW;
        const int64_t row = o * f.so + i1;
        const NV m = *reinterpret_cast<const NV *>(u + row + (2 * f.inner - i) * f.sa);
        NV w;
#pragma unroll
        for (int e = 0; e < VW; e++) {
            const bool z = zrow || (z1lo && i1 + e == fs.zidx[0][0]) || (z1hi && i1 + e == fs.zidx[0][1]);
            w[e] = z ? -(TS)0.0 : -m[e];
        }
        TS *p = u + row + i * f.sa;
        if (i1 >= f.bs && i1 + VW - 1 <= f.be) {
            *reinterpret_cast<NV *>(p) = w;
        } else {
#pragma unroll
            for (int e = 0; e < VW; e++)
                if (i1 + e >= f.bs && i1 + e <= f.be) p[e] = w[e];
        }
    }
}

template <typename TS>
__device__ __forceinline__ void bc_mirror_face(TS *u, const FaceSet &fs, int face, uint32_t bx, uint32_t nbx)
{
    const Face &f = fs.f[face];
    if (fs.vec1 && f.axis != 0) {
        bc_mirror_vec(u, fs, f, bx, nbx);
        return;
    }
    const int64_t H = f.he - f.hs + 1;
    const int64_t NB = f.be - f.bs + 1, NO = f.oe - f.os + 1;
    const int64_t total = H * NB * NO;
    if (total <= (int64_t)UINT32_MAX - (int64_t)nbx * blockDim.x)
        bc_mirror_loop<TS, uint32_t>(u, fs, f, (uint32_t)H, (uint32_t)NB, (uint32_t)total, bx, nbx);
    else
        bc_mirror_loop<TS, uint64_t>(u, fs, f, (uint64_t)H, (uint64_t)NB, (uint64_t)total, bx, nbx);
}

template <typename TS, typename IT>
__device__ __forceinline__ void bc_zero_loop(TS *u, const Face &f, IT NB, IT total)
{
    for (IT t = (IT)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (IT)gridDim.x * blockDim.x) {
        const IT io = t / NB, ib = t - io * NB;
        u[(f.os + (int64_t)io) * f.so + (f.bs + (int64_t)ib) * f.sb + f.inner * f.sa] = (TS)0.0;
    }
}

template <typename TS>
__device__ __forceinline__ void bc_zero_face(TS *u, const FaceSet &fs, int face)
{
    const Face &f = fs.f[face];
    const int64_t NB = f.be - f.bs + 1, NO = f.oe - f.os + 1;
    const int64_t total = NB * NO;
    if (total <= (int64_t)UINT32_MAX - (int64_t)gridDim.x * blockDim.x)
        bc_zero_loop<TS, uint32_t>(u, f, (uint32_t)NB, (uint32_t)total);
    else
        bc_zero_loop<TS, uint64_t>(u, f, (uint64_t)NB, (uint64_t)total);
}

// The n1 faces with 16-byte accesses, one thread per row end, when R is a
// multiple of the vector width and the halo groups are aligned: the halo
// groups get -u of their mirrors and the boundary group its zero in the same
// pass. Closed form: an n1 halo point never lies on a boundary plane of an
// earlier axis, and no mirror of another face reads the n1 boundary plane
// (those halo points are -0 by the same rule), so the zero may be written
// here; the mirrors read old values of the other faces' boundary planes,
// which k_bc_zero clears after this launch. The rest of each written group
// is stored back as read. 1000^3 FP32 order 8: 0.075 ms for both n1 faces,
// against 0.111 ms through k_bc_mirror + k_bc_zero (a second pass over the
// same 64-byte sectors of 2 x 10^6 rows).
// skip(c2, c3): rows left out (the one-launch form).
struct NoRow {
    __device__ bool operator()(int, int) const { return false; }
};
template <typename TS, int NH, typename SKIP = NoRow>
__device__ __forceinline__ void bc_n1_rows(TS *u, const Face &lo, const Face &hi, int sides, uint32_t t,
                                           SKIP skip = SKIP())
{
    constexpr int VW = 16 / sizeof(TS), R = NH * VW;
    using NV = TS __attribute__((ext_vector_type(VW)));
    const Face &f = (sides & 1) ? lo : hi;           // both faces span the same rows
    const uint32_t NB = (uint32_t)(f.be - f.bs + 1), rows = NB * (uint32_t)(f.oe - f.os + 1);
    const uint32_t ns = (uint32_t)(sides & 1) + (uint32_t)(sides >> 1);
    if (t >= rows * ns) return;
    const uint32_t row = ns == 2 ? t >> 1 : t;
    const int side = ns == 2 ? (int)(t & 1) : ((sides & 1) ? 0 : 1);
    const uint32_t io = row / NB, ib = row - io * NB;
    if (skip((int)f.bs + (int)ib, (int)f.os + (int)io)) return;
    NV *r = reinterpret_cast<NV *>(u + (f.os + (int64_t)io) * f.so + (f.bs + (int64_t)ib) * f.sb);
    NV w[NH + 1];
    if (side == 0) {
        // boundary b = lo.inner (first of its group), halo b-R .. b-1, mirrors b+1 .. b+R
        const int64_t g = lo.inner / VW;
#pragma unroll
        for (int j = 0; j <= NH; j++) w[j] = r[g + j];
#pragma unroll
        for (int h = 0; h < NH; h++) {
            NV o;
#pragma unroll
            for (int e = 0; e < VW; e++) {
                const int k = R - h * VW - e;            // halo point b - k, mirror b + k
                o[e] = -w[k / VW][k % VW];
            }
            r[g - NH + h] = o;
        }
        w[0][0] = (TS)0.0;
        r[g] = w[0];
    } else {
        // boundary b = hi.inner (last of its group), halo b+1 .. b+R, mirrors b-1 .. b-R
        const int64_t g = hi.inner / VW;
#pragma unroll
        for (int j = 0; j <= NH; j++) w[j] = r[g - NH + j];
#pragma unroll
        for (int h = 0; h < NH; h++) {
            NV o;
#pragma unroll
            for (int e = 0; e < VW; e++) {
                const int k = 1 + h * VW + e;            // halo point b + k, mirror b - k
                const int p = (NH + 1) * VW - 1 - k;     // position of b - k in w
                o[e] = -w[p / VW][p % VW];
            }
            r[g + 1 + h] = o;
        }
        w[NH][VW - 1] = (TS)0.0;
        r[g] = w[NH];
    }
}

template <typename TS, int NH>
__global__ void __launch_bounds__(256) k_bc_n1(TS *u, Face lo, Face hi, int sides)
{
    bc_n1_rows<TS, NH>(u, lo, hi, sides, blockIdx.x * 256u + threadIdx.x);
}

// The n1 faces (bc_n1_rows) and the mirrors of the other faces in one launch:
// they write disjoint halo points and neither reads what the other writes
// (bc_n1_rows rewrites the n1 boundary group with its own values and a zero
// that the other faces' mirrors take as -0 without reading it), so the two
// need no order; blocks [0, nb_n1) take the n1 rows, the next nb1 * rest.n the
// mirrors (nb1 blocks per face).  The boundary planes follow in k_bc_zero.
template <typename TS, int NH>
__global__ void __launch_bounds__(256) k_bc_n1_mirror(TS *u, Face lo, Face hi, int sides, FaceSet rest,
                                                     uint32_t nb_n1, uint32_t nb1)
{
    if (blockIdx.x < nb_n1) {
        bc_n1_rows<TS, NH>(u, lo, hi, sides, blockIdx.x * 256u + threadIdx.x);
        return;
    }
    const uint32_t m = blockIdx.x - nb_n1;
    bc_mirror_face(u, rest, (int)(m / nb1), m % nb1, nb1);
}

// the same for many grids: blockIdx.y = grid; blocks past nb_n1 take the
// mirrors of faces (blockIdx.x - nb_n1) / nb1 < fs[grid].n
template <typename TS, int NH>
__global__ void __launch_bounds__(256) k_bc_n1_mirror_batch(TS *const *u, const N1Faces *nf, const FaceSet *fs,
                                                           uint32_t nb_n1, uint32_t nb1)
{
    const int s = blockIdx.y;
    if (blockIdx.x < nb_n1) {
        const N1Faces &x = nf[s];
        if (x.sides) bc_n1_rows<TS, NH>(u[s], x.lo, x.hi, x.sides, blockIdx.x * 256u + threadIdx.x);
        return;
    }
    const uint32_t m = blockIdx.x - nb_n1;
    const int face = (int)(m / nb1);
    if (face < fs[s].n) bc_mirror_face(u[s], fs[s], face, m % nb1, nb1);
}

// ---- free surface, all faces in one launch ----------------------------------------
// The closed form above needs its second launch only because the planes it
// zeroes hold mirror sources: a point on a boundary plane of axis a is the
// source of the halos of the axes before a (of those after a it gives -0,
// unread).  Here the thread that zeroes such a point first writes those halos
// itself, and the mirror threads leave them out, so that no thread reads a
// point that another one writes: one launch in any order.  A point on planes
// of two axes belongs to the lower one's plane.  The faces' boundary planes
// must be the first / last inner planes (fs_one_launch).
// Bound by launches on small grids, by the row ends of the n1 faces (a sector or
// two each) on large ones.  Two launches before, us: 61^3 FP32 order 8 6.4 ->
// 3.8, 200^3 7.0 -> 5.3, 403 x 307 x 255 order 4 15.2 -> 6.5, 601 x 600 x 580
// order 10 51 -> 33, FP64 500^3 order 12 46.5 -> 43.5, 1000^3 order 8 111 -> 109,
// 1501 x 2001 (2D) 5.6 -> 3.3.
// Geometry: inner ranges per axis (s, e: the boundary planes), halo widths of
// the masked faces (0: not masked), first block of each n2 / n3 face.
struct BcOne {
    int s[3], e[3];
    int h[3][2];
    int64_t n1, n12;
    uint32_t first[5];       // first block of faces n2 low, n2 high, n3 low, n3 high, and the end
    int sides;               // n1 faces by bc_n1_rows (bit 0 / 1), 0: by points
};

template <typename TS>
struct VecOf {
    static constexpr int W = 16 / sizeof(TS);
    using U = TS __attribute__((ext_vector_type(W), aligned(sizeof(TS))));       // any element address
};

// c lies on a masked boundary plane of the axis
__device__ __forceinline__ bool on_plane(const BcOne &b, int axis, int c)
{
    return (b.h[axis][0] && c == b.s[axis]) || (b.h[axis][1] && c == b.e[axis]);
}

// -v, or -0 on the masked n1 boundary planes / the whole row
template <typename TS, typename V>
__device__ __forceinline__ V mirror_of(const BcOne &b, const V &v, int i1, bool zrow)
{
    V w;
#pragma unroll
    for (int e = 0; e < VecOf<TS>::W; e++) w[e] = zrow || on_plane(b, 0, i1 + e) ? -(TS)0.0 : -v[e];
    return w;
}

// store the elements of w that lie in the inner n1 range, without those of skip (bits)
template <typename TS, typename V>
__device__ __forceinline__ void store_in(const BcOne &b, TS *p, const V &w, int i1, uint32_t skip = 0)
{
    constexpr int VW = VecOf<TS>::W;
    if (!skip && i1 >= b.s[0] && i1 + VW - 1 <= b.e[0]) {
        *reinterpret_cast<typename VecOf<TS>::U *>(p) = w;
    } else {
#pragma unroll
        for (int e = 0; e < VW; e++)
            if (i1 + e >= b.s[0] && i1 + e <= b.e[0] && !((skip >> e) & 1)) p[e] = w[e];
    }
}

// One n2 (A = 1) or n3 (A = 2) face in 16-byte groups along n1, item t: its
// boundary plane (k = 0) and its halo rows (k = 1 .. h).  The last group of a
// row may take in a few points past the inner range; they are read (inside the
// grid: these rows are inner rows) and not written.
template <typename TS, int A, typename X>
__device__ __forceinline__ void bc1_face(TS *u, const BcOne &b, int side, uint32_t t, const X &x)
{
    constexpr int VW = VecOf<TS>::W, O = 3 - A;           // O: the outer axis
    using U = typename VecOf<TS>::U;
    const int64_t so = A == 1 ? b.n12 : b.n1, sa = A == 1 ? b.n1 : b.n12;
    const int h = b.h[A][side], plane = side == 0 ? b.s[A] : b.e[A], g0 = b.s[0] / VW;
    const uint32_t NG = (uint32_t)(b.e[0] / VW - g0 + 1), H = (uint32_t)(h + 1);
    const uint32_t r = t / NG, io = r / H;
    const int k = (int)(r - io * H), i1 = (g0 + (int)(t - r * NG)) * VW, o = b.s[O] + (int)io;
    if (o > b.e[O]) return;
    // n2 faces: the halo rows on an n3 plane belong to that plane's threads; n3
    // faces: the plane's rows on an n2 plane to the n2 plane's threads
    const bool oz = on_plane(b, O, o);
    if (oz && (A == 1) == (k > 0)) return;
    const int d = side == 0 ? k : -k;
    TS *p = u + (o * so + (plane + d) * sa + i1);         // the mirror source, or the plane's own points
    const U v = *reinterpret_cast<const U *>(p);
    if (k > 0) {
        const int m = plane + d;
        store_in<TS, U>(b, p - 2 * d * sa, mirror_of<TS, U>(b, v, i1, A == 2 && oz), i1,
                        x.points(A == 1 ? m : o, A == 1 ? o : m, i1, VW));
        return;
    }
    const uint32_t skip = x.plane_points(A == 1 ? plane : o, A == 1 ? o : plane, i1, VW);
    if (A == 2) {
        // the n2 halos that mirror this row
        const int d0 = o - b.s[1], d1 = b.e[1] - o;
        if (d0 >= 1 && d0 <= b.h[1][0])
            store_in<TS, U>(b, p - 2 * d0 * b.n1, mirror_of<TS, U>(b, v, i1, false), i1, skip);
        if (d1 >= 1 && d1 <= b.h[1][1])
            store_in<TS, U>(b, p + 2 * d1 * b.n1, mirror_of<TS, U>(b, v, i1, false), i1, skip);
    }
    // the n1 halos that mirror points of this group
    if (i1 <= b.s[0] + b.h[0][0] || i1 + VW - 1 >= b.e[0] - b.h[0][1]) {
#pragma unroll
        for (int e = 0; e < VW; e++) {
            if ((skip >> e) & 1) continue;
            const int d0 = i1 + e - b.s[0], d1 = b.e[0] - (i1 + e);
            if (d0 >= 1 && d1 >= 0 && d0 <= b.h[0][0]) p[e - 2 * d0] = -v[e];
            if (d1 >= 1 && d0 >= 0 && d1 <= b.h[0][1]) p[e + 2 * d1] = -v[e];
        }
    }
    U z;
#pragma unroll
    for (int e = 0; e < VW; e++) z[e] = (TS)0.0;
    store_in<TS, U>(b, p, z, i1, skip);
}

// The n1 faces, one point per thread (R not a multiple of the vector, rows at
// any address), item t: the boundary point (k = 0) and the halo points of a row
template <typename TS, typename X>
__device__ __forceinline__ void bc1_n1_points(TS *u, const BcOne &b, uint32_t t, const X &x)
{
    const int h0 = b.h[0][0], h1 = b.h[0][1];
    const uint32_t H = (uint32_t)((h0 ? h0 + 1 : 0) + (h1 ? h1 + 1 : 0)), N2 = (uint32_t)(b.e[1] - b.s[1] + 1);
    const uint32_t r = t / H, i3 = r / N2;
    int k = (int)(t - r * H);
    const int c2 = b.s[1] + (int)(r - i3 * N2), c3 = b.s[2] + (int)i3;
    if (c3 > b.e[2] || on_plane(b, 1, c2) || on_plane(b, 2, c3) || x.row(c2, c3)) return;   // the planes' threads
    const bool lo = h0 && k <= h0;
    if (!lo && h0) k -= h0 + 1;
    TS *p = u + (c3 * b.n12 + c2 * b.n1 + (lo ? b.s[0] + k : b.e[0] - k));
    if (k == 0)
        *p = (TS)0.0;
    else
        p[lo ? -2 * k : 2 * k] = -*p;
}

// Work that shares the launch (X): blocks [0, nblk()) run it, and the points it
// changes are its own with their mirrors: x.points (inside, bits of a group),
// x.plane_points (on the n2 and n3 planes), x.row (the n1 halos of a whole row).
struct NoExtra {
    __host__ __device__ uint32_t nblk() const { return 0; }
    template <typename TS>
    __device__ void run(TS *, const BcOne &, uint32_t) const {}
    __device__ uint32_t points(int, int, int, int) const { return 0; }
    __device__ uint32_t plane_points(int, int, int, int) const { return 0; }
    __device__ bool row(int, int) const { return false; }
};

// Sources and receivers of a forward step, then the free surface.  Block 0 adds
// the sources, records the receivers that sit on one, and writes every halo
// point that mirrors a source and the n1 halos of the sources' rows from the
// new values; it records the receivers on the n2 and n3 planes, then zeroes
// these points and writes what mirrors them.  The other blocks record the
// other receivers.  All other sources and receivers lie strictly inside the
// boundary planes (step_end_check), so that no thread uses a point that another
// one changes.  Against sources and receivers in a launch of their own before
// the free surface's (4.6 + 6.0 us on 200^3 FP32 order 8): 6.9 us, the
// shot of 100 steps 4172 -> 3996 us.
template <typename TS>
struct ForwardEnd {
    int ns;
    const int64_t *src;
    const TS *w;
    const EndWork *work;
    int64_t nrec;
    const int64_t *rec;
    TS *tr;
    uint32_t nb_rec;

    __host__ __device__ uint32_t nblk() const { return 1 + nb_rec; }
    __device__ uint32_t points(int c2, int c3, int i1, int vw) const
    {
        uint32_t m = 0;
        for (int k = 0; k < ns; k++) {
            const int e = work->c[k][0] - i1;
            if (c2 == work->c[k][1] && c3 == work->c[k][2] && e >= 0 && e < vw) m |= 1u << e;
        }
        return m;
    }
    __device__ uint32_t plane_points(int c2, int c3, int i1, int vw) const
    {
        uint32_t m = 0;
        const int ne = work->ne;
        for (int k = 0; k < ne; k++) {
            const int e = work->e[k][0] - i1;
            if (c2 == work->e[k][1] && c3 == work->e[k][2] && e >= 0 && e < vw) m |= 1u << e;
        }
        return m;
    }
    __device__ bool row(int c2, int c3) const
    {
        bool r = false;
        for (int k = 0; k < ns; k++) r |= c2 == work->c[k][1] && c3 == work->c[k][2];
        return r;
    }
    __device__ void run(TS *u, const BcOne &b, uint32_t bx) const
    {
        const int t = (int)threadIdx.x;
        if (bx > 0) {
            for (int64_t i = (int64_t)(bx - 1) * blockDim.x + t; i < nrec; i += (int64_t)nb_rec * blockDim.x) {
                const int64_t j = rec[i];
                bool on = false;
                for (int k = 0; k < ns; k++) on |= src[k] == j;
                const int ne = work->ne;
                for (int k = 0; k < ne; k++) on |= work->ei[k] == i;
                if (!on) tr[i] = u[j];
            }
            return;
        }
        // receivers on the planes: the values now, the zeros after the barrier (an
        // index may be listed twice).  nrec = 0 (no traces): the planes' threads'
        // points all the same
        const bool edge = t < work->ne;
        const int e1 = edge ? work->e[t][0] : 0, e2 = edge ? work->e[t][1] : 0, e3 = edge ? work->e[t][2] : 0;
        TS *ep = u + (e3 * b.n12 + e2 * b.n1 + e1);
        const TS ev = edge ? *ep : (TS)0;
        __shared__ TS nv[END_SRC_MAX];
        if (t < ns) {
            const int64_t j = src[t];
            const TS x = (TS)((double)u[j] + 1.0 * (double)w[t]);
            nv[t] = x;
            u[j] = x;
        }
        __syncthreads();
        if (edge) {
            if (nrec > 0) tr[work->ei[t]] = ev;
            if (!on_plane(b, 1, e2)) {
                const int d0 = e2 - b.s[1], d1 = b.e[1] - e2;
                if (d0 >= 1 && d0 <= b.h[1][0]) ep[-2 * d0 * b.n1] = -ev;
                if (d1 >= 1 && d1 <= b.h[1][1]) ep[2 * d1 * b.n1] = -ev;
            }
            const int d0 = e1 - b.s[0], d1 = b.e[0] - e1;
            if (d0 >= 1 && d0 <= b.h[0][0]) ep[-2 * d0] = -ev;
            if (d1 >= 1 && d1 <= b.h[0][1]) ep[2 * d1] = -ev;
            *ep = (TS)0.0;
        }
        for (int64_t i = t; i < nrec; i += blockDim.x) {
            const int64_t j = rec[i];
            for (int k = 0; k < ns; k++)
                if (src[k] == j) tr[i] = nv[k];
        }
        // n1 ends of the sources' rows: boundary point (d = 0) and halo of each side
        constexpr int D = 9;                       // R + 1 at most
        const int s = t / (2 * D), r = t - s * 2 * D, side = r / D, d = r - side * D;
        if (s < ns && b.h[0][side] && d <= b.h[0][side]) {
            const int plane = side ? b.e[0] : b.s[0], in = side ? -d : d;
            TS *p = u + (work->c[s][2] * b.n12 + work->c[s][1] * b.n1 + plane);
            if (d == 0) {
                *p = (TS)0.0;
            } else {
                int at = -1;
                for (int k = 0; k < ns; k++)
                    if (work->c[k][0] == plane + in && work->c[k][1] == work->c[s][1] && work->c[k][2] == work->c[s][2])
                        at = k;
                p[-in] = -(at >= 0 ? nv[at] : p[in]);
            }
        }
        // the n2 and n3 halo points that mirror a source
        if (t < 4 * ns) {
            const int k = t >> 2, a = 1 + ((t >> 1) & 1), sd = t & 1;
            const int d2 = sd ? b.e[a] - work->c[k][a] : work->c[k][a] - b.s[a];
            if (d2 >= 1 && d2 <= b.h[a][sd]) {
                const int64_t sa = a == 1 ? b.n1 : b.n12;
                u[src[k] + (sd ? 2 * d2 : -2 * d2) * sa] = -nv[k];
            }
        }
    }
};

template <typename TS>
struct ReverseExtra {
    ReverseEnd<TS> r;
    __host__ __device__ uint32_t nblk() const { return r.nb_src + r.nb_rec; }
    __device__ void run(TS *, const BcOne &, uint32_t bx) const { r.block(bx); }
    __device__ uint32_t points(int, int, int, int) const { return 0; }
    __device__ uint32_t plane_points(int, int, int, int) const { return 0; }
    __device__ bool row(int, int) const { return false; }
};

// block bx of the free surface; NH > 0: the n1 faces by 16-byte row ends
// (bc_n1_rows), else by points
template <typename TS, int NH, typename X>
__device__ __forceinline__ void bc_one_block(TS *u, const BcOne &b, const Face &lo, const Face &hi, uint32_t bx, const X &x)
{
    if (bx < b.first[0]) {
        const uint32_t t = bx * 256u + threadIdx.x;
        if constexpr (NH > 0)
            bc_n1_rows<TS, NH>(u, lo, hi, b.sides, t,
                               [&](int c2, int c3) { return on_plane(b, 1, c2) || on_plane(b, 2, c3) || x.row(c2, c3); });
        else
            bc1_n1_points(u, b, t, x);
    } else if (bx < b.first[2]) {
        const int side = bx >= b.first[1];
        bc1_face<TS, 1>(u, b, side, (bx - b.first[side]) * 256u + threadIdx.x, x);
    } else {
        const int side = bx >= b.first[3];
        bc1_face<TS, 2>(u, b, side, (bx - b.first[2 + side]) * 256u + threadIdx.x, x);
    }
}

template <typename TS, int NH, typename X>
__global__ void __launch_bounds__(256) k_bc_one(TS *u, BcOne b, Face lo, Face hi, X x)
{
    if (blockIdx.x < x.nblk())
        x.run(u, b, blockIdx.x);
    else
        bc_one_block<TS, NH>(u, b, lo, hi, blockIdx.x - x.nblk(), x);
}

// the same for many grids: blockIdx.y = grid.  32 shots of 192^3-320^3 FP32 order
// 8: 282 us (two launches, mirrors and planes: 281 + 32 us).
struct BcOneGrid {
    BcOne b;
    Face lo, hi;
};
template <typename TS, int NH>
__global__ void __launch_bounds__(256) k_bc_one_batch(TS *const *u, const BcOneGrid *grids)
{
    const BcOneGrid &g = grids[blockIdx.y];
    if (blockIdx.x < g.b.first[4]) bc_one_block<TS, NH>(u[blockIdx.y], g.b, g.lo, g.hi, blockIdx.x, NoExtra());
}

// arguments of k_bc_one; false where it does not serve the faces (a boundary
// plane that is not the first / last inner plane, index spaces past 32 bits)
static bool fill_bc_one(const hsx_grid *g, const FaceSet &fs, int sides, BcOne *b)
{
    if (g->n1 >= INT32_MAX || g->n2 >= INT32_MAX || g->n3 >= INT32_MAX) return false;
    const int VW = g->storage == HSX_FP64 ? 2 : 4;
    b->n1 = g->n1;
    b->n12 = g->n1 * g->n2;
    b->sides = sides;
    int64_t n[3];
    for (int a = 0; a < 3; a++) {
        b->s[a] = (int)g->inner[2 * a];
        b->e[a] = (int)g->inner[2 * a + 1];
        b->h[a][0] = b->h[a][1] = 0;
        n[a] = b->e[a] - b->s[a] + 1;
    }
    for (int k = 0; k < fs.n; k++) {
        const Face &f = fs.f[k];
        const int side = f.inner > f.he ? 0 : 1;
        if (f.inner != g->inner[2 * f.axis + side] || f.he < f.hs) return false;
        b->h[f.axis][side] = (int)(f.he - f.hs + 1);
    }
    int64_t at = 0;
    const int64_t most = ((int64_t)1 << 31) - 256;
    auto take = [&](int64_t items) {
        at += (items + 255) / 256;
        return items < most && at < most;
    };
    const int64_t rows = n[1] * n[2];
    const int64_t per_row = sides ? (sides & 1) + (sides >> 1)
                                  : (b->h[0][0] ? b->h[0][0] + 1 : 0) + (b->h[0][1] ? b->h[0][1] + 1 : 0);
    if (!take(rows * per_row)) return false;
    const int64_t ng = b->e[0] / VW - b->s[0] / VW + 1;
    for (int f = 0; f < 4; f++) {
        const int a = 1 + f / 2, h = b->h[a][f % 2];
        b->first[f] = (uint32_t)at;
        if (!take(h ? ng * (h + 1) * n[3 - a] : 0)) return false;
    }
    b->first[4] = (uint32_t)at;
    return at > 0;
}

int n1_groups_ok(const hsx_grid *g, const void *u, const FaceSet &fs)
{
    const int VW = g->storage == HSX_FP64 ? 2 : 4;
    if (g->n1 % VW || (uintptr_t)u % 16) return 0;
    for (int k = 0; k < fs.n; k++) {
        const Face &f = fs.f[k];
        if (f.axis == 0) continue;
        const int64_t n = (f.be / VW - f.bs / VW + 1) * (f.he - f.hs + 1) * (f.oe - f.os + 1);
        if (n >= ((int64_t)1 << 31)) return 0;
    }
    return 1;
}

int n1_vector_sides(const hsx_grid *g, const void *u, const FaceSet &fs, Face *lo, Face *hi)
{
    const int VW = g->storage == HSX_FP64 ? 2 : 4;
    if (g->n1 % VW || (uintptr_t)u % 16) return 0;
    int sides = 0;
    for (int k = 0; k < fs.n; k++) {
        const Face &f = fs.f[k];
        if (f.axis != 0) continue;
        const int64_t R = f.he - f.hs + 1;
        if (R % VW || R / VW < 1 || R / VW > 4 || f.hs % VW) return 0;
        const int64_t rows = (f.be - f.bs + 1) * (f.oe - f.os + 1);
        if (rows <= 0 || 2 * rows >= ((int64_t)1 << 31)) return 0;
        if (f.inner > f.he) {
            *lo = f;
            sides |= 1;
        } else {
            *hi = f;
            sides |= 2;
        }
    }
    if (sides == 3 && lo->he - lo->hs != hi->he - hi->hs) return 0;
    return sides;
}

// the free surface in one launch with the work of x, or HSX_ERR_UNSUPPORTED
template <typename TS, typename X>
static int bc_one_launch(const hsx_grid *g, TS *u, const FaceSet &fs, const X &x, hipStream_t s)
{
    BcOne one;
    Face flo{}, fhi{};
    const int n1s = n1_vector_sides(g, u, fs, &flo, &fhi);
    if (!fill_bc_one(g, fs, n1s, &one)) return HSX_ERR_UNSUPPORTED;
    const dim3 grid(one.first[4] + x.nblk());
    auto go = [&](auto nh) {
        constexpr int NH = decltype(nh)::value;
        hipLaunchKernelGGL((k_bc_one<TS, NH, X>), grid, dim3(256), 0, s, u, one, flo, fhi, x);
    };
    const Face &f = (n1s & 1) ? flo : fhi;
    switch (n1s ? (int)((f.he - f.hs + 1) / (16 / (int64_t)sizeof(TS))) : 0) {
    case 0: go(IC<0>()); break;
    case 1: go(IC<1>()); break;
    case 2: go(IC<2>()); break;
    case 3: go(IC<3>()); break;
    default: go(IC<4>()); break;
    }
    HSX_LAUNCHED("k_bc_one");
    return HSX_OK;
}

__global__ void k_end_clear(EndWork *work)
{
    if (threadIdx.x == 0) work->outside = work->ne = 0;
}

__global__ void __launch_bounds__(256) k_end_check(Box box, Box in, int64_t n1, int64_t n12, int64_t npoint, int64_t nsrc,
                                                   const int64_t *src, int64_t nrec, const int64_t *rec, EndWork *work)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nsrc + nrec; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = i < nsrc ? src[i] : rec[i - nsrc];
        if (j < 0 || j >= npoint) {
            work->outside = 1;
            continue;
        }
        const int64_t i3 = j / n12, i2 = (j - i3 * n12) / n1, i1 = j - i3 * n12 - i2 * n1;
        const bool row_in = i1 >= in.s1 && i1 <= in.e1;
        const bool inside = row_in && i2 >= in.s2 && i2 <= in.e2 && i3 >= in.s3 && i3 <= in.e3;
        if (!inside) {
            const bool inner = i2 >= box.s2 && i2 <= box.e2 && i3 >= box.s3 && i3 <= box.e3;
            const int k = i >= nsrc && row_in && inner ? atomicAdd(&work->ne, 1) : END_EDGE_MAX;
            if (k < END_EDGE_MAX) {
                work->e[k][0] = (int)i1;
                work->e[k][1] = (int)i2;
                work->e[k][2] = (int)i3;
                work->ei[k] = i - nsrc;
            } else {
                work->outside = 1;
            }
        }
        if (i < nsrc) {
            work->c[i][0] = (int)i1;
            work->c[i][1] = (int)i2;
            work->c[i][2] = (int)i3;
        }
    }
}

// all six faces of g in one launch?
static bool end_faces(const hsx_grid *g, FaceSet *fs)
{
    bool closed;
    int64_t most, most_plane;
    BcOne one;
    return make_faceset(g, 0x3F, fs, &closed, &most, &most_plane) == HSX_OK && fs->n > 0 && closed &&
           fill_bc_one(g, *fs, 0, &one);
}

int step_end_check(const hsx_grid *g, int64_t nsrc, const int64_t *src, int64_t nrec, const int64_t *rec,
                   EndWork *work, bool *merge, hipStream_t s)
{
    *merge = false;
    FaceSet fs;
    if (nsrc < 1 || nsrc > END_SRC_MAX || !end_faces(g, &fs)) return HSX_OK;
    int64_t r[6];
    for (int a = 0; a < 3; a++) {
        r[2 * a] = g->inner[2 * a] + (a < g->dim ? 1 : 0);
        r[2 * a + 1] = g->inner[2 * a + 1] - (a < g->dim ? 1 : 0);
    }
    const unsigned nb = (unsigned)std::min<int64_t>((nsrc + nrec + 255) / 256, 1024);
    hipLaunchKernelGGL(k_end_clear, dim3(1), dim3(64), 0, s, work);
    HSX_LAUNCHED("k_end_clear");
    hipLaunchKernelGGL(k_end_check, dim3(nb), dim3(256), 0, s, box_of(g->inner), box_of(r), g->n1, g->n1 * g->n2,
                       g->n1 * g->n2 * g->n3, nsrc, src, nrec, rec, work);
    HSX_LAUNCHED("k_end_check");
    int outside = 1;
    HSX_HIP(hipMemcpyAsync(&outside, &work->outside, sizeof(int), hipMemcpyDeviceToHost, s));
    HSX_HIP(hipStreamSynchronize(s));
    *merge = !outside;
    return HSX_OK;
}

int step_end_forward(const hsx_grid *g, void *u, int64_t nsrc, const int64_t *src, const void *w, int64_t nrec,
                     const int64_t *rec, void *tr, const EndWork *work, hipStream_t s)
{
    FaceSet fs;
    if (!end_faces(g, &fs)) return fail(HSX_ERR_UNSUPPORTED, "step end: the free surface takes several launches");
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        const int64_t nr = tr ? nrec : 0;
        const ForwardEnd<TS> x = {(int)nsrc, src, (const TS *)w, work, nr, rec, (TS *)tr,
                                  (uint32_t)std::min<int64_t>((nr + 255) / 256, 1024)};
        return bc_one_launch(g, (TS *)u, fs, x, s);
    });
}

template <typename TS>
int step_end_reverse(const hsx_grid *g, void *u, const ReverseEnd<TS> &r, hipStream_t s)
{
    FaceSet fs;
    if (!end_faces(g, &fs)) return HSX_ERR_UNSUPPORTED;
    return bc_one_launch(g, (TS *)u, fs, ReverseExtra<TS>{r}, s);
}
template int step_end_reverse<float>(const hsx_grid *, void *, const ReverseEnd<float> &, hipStream_t);
template int step_end_reverse<double>(const hsx_grid *, void *, const ReverseEnd<double> &, hipStream_t);

// one grid: blockIdx.y = face
template <typename TS>
__global__ void __launch_bounds__(256) k_bc_mirror(TS *u, FaceSet fs)
{
    bc_mirror_face(u, fs, blockIdx.y, blockIdx.x, gridDim.x);
}

template <typename TS>
__global__ void __launch_bounds__(256) k_bc_zero(TS *u, FaceSet fs)
{
    bc_zero_face(u, fs, blockIdx.y);
}

// many grids: blockIdx.y = 6 * grid + face
template <typename TS>
__global__ void __launch_bounds__(256) k_bc_mirror_batch(TS *const *u, const FaceSet *fs)
{
    const int s = blockIdx.y / 6, face = blockIdx.y % 6;
    if (face < fs[s].n) bc_mirror_face(u[s], fs[s], face, blockIdx.x, gridDim.x);
}

template <typename TS>
__global__ void __launch_bounds__(256) k_bc_zero_batch(TS *const *u, const FaceSet *fs)
{
    const int s = blockIdx.y / 6, face = blockIdx.y % 6;
    if (face < fs[s].n) bc_zero_face(u[s], fs[s], face);
}

int make_faceset(const hsx_grid *g, int face_mask, FaceSet *fs, bool *closed_form, int64_t *most,
                 int64_t *most_plane)
{
    const int64_t st[3] = {1, g->n1, g->n1 * g->n2};
    fs->n = 0;
    fs->zmask = 0;
    fs->vec1 = 0;
    for (int a = 0; a < 3; a++) fs->zidx[a][0] = fs->zidx[a][1] = -1;
    *closed_form = true;
    *most = *most_plane = 0;
    for (int axis = 0; axis < g->dim; axis++) {
        for (int side = 0; side < 2; side++) {
            if (!(face_mask & (1 << (2 * axis + side)))) continue;
            const int64_t *hr = side == 0 ? g->halo1 : g->halo2;
            Face f;
            f.axis = axis;
            f.hs = hr[2 * axis];
            f.he = hr[2 * axis + 1];
            f.inner = side == 0 ? f.he + 1 : f.hs - 1;
            // other axes: outer = the higher one, inner-other = the lower one
            const int oa = axis == 2 ? 1 : 2, ob = axis == 0 ? 1 : 0;
            f.os = g->inner[2 * oa];
            f.oe = g->inner[2 * oa + 1];
            f.bs = g->inner[2 * ob];
            f.be = g->inner[2 * ob + 1];
            f.so = st[oa];
            f.sb = st[ob];
            f.sa = st[axis];
            // mirror sources must stay inside the allocation
            const int64_t n_ax = axis == 0 ? g->n1 : axis == 1 ? g->n2 : g->n3;
            if (2 * f.inner - f.hs >= n_ax || 2 * f.inner - f.he < 0 || f.inner < 0 || f.inner >= n_ax)
                return fail(HSX_ERR_INVALID, "free surface: mirror of axis %d face %d outside the grid", axis + 1,
                            side + 1);
            fs->f[fs->n++] = f;
            fs->zidx[axis][side] = f.inner;
            fs->zmask |= 1 << (2 * axis + side);
            const int64_t plane = (f.be - f.bs + 1) * (f.oe - f.os + 1);
            *most = std::max(*most, plane * (f.he - f.hs + 1));
            *most_plane = std::max(*most_plane, plane);
        }
        // closed form: the mirrors of each face stay strictly between the two
        // boundary planes of the axis (both computed as the sequential phases do);
        // an axis with no face in the mask adds no phase and no condition
        const int64_t z0 = g->halo1[2 * axis + 1] + 1, z1 = g->halo2[2 * axis] - 1;
        const int64_t h1 = g->halo1[2 * axis + 1] - g->halo1[2 * axis] + 1;
        const int64_t h2 = g->halo2[2 * axis + 1] - g->halo2[2 * axis] + 1;
        if (((fs->zmask >> (2 * axis)) & 3) && z1 - z0 <= (h1 > h2 ? h1 : h2)) *closed_form = false;
    }
    return HSX_OK;
}

size_t bc_one_batch_bytes(void) { return sizeof(BcOneGrid); }

bool bc_one_batch_fill(const hsx_grid *g, const void *u, const FaceSet &fs, void *out, int *nh, uint32_t *blocks)
{
    BcOneGrid *o = static_cast<BcOneGrid *>(out);
    o->lo = o->hi = Face{};
    const int sides = n1_vector_sides(g, u, fs, &o->lo, &o->hi);
    if (!fill_bc_one(g, fs, sides, &o->b)) return false;
    const Face &f = (sides & 1) ? o->lo : o->hi;
    *nh = sides ? (int)((f.he - f.hs + 1) / (g->storage == HSX_FP64 ? 2 : 4)) : 0;
    *blocks = o->b.first[4];
    return true;
}

int bc_one_batch_launch(int storage, int nshots, void *const *d_fields, const void *d_grids, int nh, uint32_t blocks,
                        hipStream_t s)
{
    auto launch = [&](auto ts, auto n) -> int {
        using TS = decltype(ts);
        hipLaunchKernelGGL((k_bc_one_batch<TS, decltype(n)::value>), dim3(blocks, (unsigned)nshots), dim3(256), 0, s,
                           (TS *const *)d_fields, (const BcOneGrid *)d_grids);
        HSX_LAUNCHED("k_bc_one_batch");
        return HSX_OK;
    };
    auto go = [&](auto ts) -> int {
        switch (nh) {
        case 0: return launch(ts, IC<0>());
        case 1: return launch(ts, IC<1>());
        case 2: return launch(ts, IC<2>());
        case 3: return launch(ts, IC<3>());
        default: return launch(ts, IC<4>());
        }
    };
    return storage == HSX_FP64 ? go(0.0) : go(0.0f);
}

int bc_batch_launch(int storage, int nshots, void *const *d_fields, const FaceSet *d_sets, int64_t most,
                    int64_t most_plane, hipStream_t s)
{
    const unsigned nb1 = (unsigned)std::max<int64_t>(1, std::min<int64_t>((most + 255) / 256, 4096));
    const unsigned nb2 = (unsigned)std::max<int64_t>(1, std::min<int64_t>((most_plane + 255) / 256, 4096));
    if (storage == HSX_FP64) {
        hipLaunchKernelGGL(k_bc_mirror_batch<double>, dim3(nb1, 6 * nshots), dim3(256), 0, s,
                           (double *const *)d_fields, d_sets);
        HSX_LAUNCHED("k_bc_mirror_batch");
        hipLaunchKernelGGL(k_bc_zero_batch<double>, dim3(nb2, 6 * nshots), dim3(256), 0, s,
                           (double *const *)d_fields, d_sets);
    } else {
        hipLaunchKernelGGL(k_bc_mirror_batch<float>, dim3(nb1, 6 * nshots), dim3(256), 0, s,
                           (float *const *)d_fields, d_sets);
        HSX_LAUNCHED("k_bc_mirror_batch");
        hipLaunchKernelGGL(k_bc_zero_batch<float>, dim3(nb2, 6 * nshots), dim3(256), 0, s,
                           (float *const *)d_fields, d_sets);
    }
    HSX_LAUNCHED("k_bc_zero_batch");
    return HSX_OK;
}

int bc_batch_fs_launch(int storage, int nshots, void *const *d_fields, const N1Faces *d_n1, int nh,
                       int64_t most_rows, const FaceSet *d_sets, int64_t most, int64_t most_plane, hipStream_t s)
{
    if (nh < 1 || nh > 4) return fail(HSX_ERR_INVALID, "batch free surface: %d n1 halo groups", nh);
    const uint32_t nbn = (uint32_t)std::max<int64_t>(1, (2 * most_rows + 255) / 256);
    const uint32_t nb1 = (uint32_t)std::max<int64_t>(1, std::min<int64_t>((most + 255) / 256, 4096));
    const uint32_t nb2 = (uint32_t)std::max<int64_t>(1, std::min<int64_t>((most_plane + 255) / 256, 4096));
    const dim3 both(nbn + 6 * nb1, (unsigned)nshots);
    auto launch = [&](auto ts) -> int {
        using TS = decltype(ts);
        TS *const *u = (TS *const *)d_fields;
        switch (nh) {
        case 1: hipLaunchKernelGGL((k_bc_n1_mirror_batch<TS, 1>), both, dim3(256), 0, s, u, d_n1, d_sets, nbn, nb1); break;
        case 2: hipLaunchKernelGGL((k_bc_n1_mirror_batch<TS, 2>), both, dim3(256), 0, s, u, d_n1, d_sets, nbn, nb1); break;
        case 3: hipLaunchKernelGGL((k_bc_n1_mirror_batch<TS, 3>), both, dim3(256), 0, s, u, d_n1, d_sets, nbn, nb1); break;
        default: hipLaunchKernelGGL((k_bc_n1_mirror_batch<TS, 4>), both, dim3(256), 0, s, u, d_n1, d_sets, nbn, nb1); break;
        }
        HSX_LAUNCHED("k_bc_n1_mirror_batch");
        hipLaunchKernelGGL(k_bc_zero_batch<TS>, dim3(nb2, 6 * nshots), dim3(256), 0, s, u, d_sets);
        HSX_LAUNCHED("k_bc_zero_batch");
        return HSX_OK;
    };
    return storage == HSX_FP64 ? launch(0.0) : launch(0.0f);
}

// ---- leapfrog update of the split propagator (src/grid.cpp:4579-4610) -----------
// prn = TWO*prc - prn + coef*lapla; coef*lapla is a product of two storage values
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_update_pressure(TS *prn, const TS *prc, const TS *coef, const TS *lapla,
                                                         Box b, int64_t n1, int64_t n12)
{
    const TC two = (TC)2.0;
    for_box(b, n1, n12, [&](int64_t ii, int64_t, int64_t, int64_t) {
        const TS cl = coef[ii] * lapla[ii];
        prn[ii] = (TS)(two * (TC)prc[ii] - (TC)prn[ii] + (TC)cl);
    });
}

// The same update with 16-byte lanes (n1 a multiple of the vector width, 16-byte
// aligned grids): one thread per aligned group of a row's [s1, e1] span, 256
// threads per block over the (row, group) space in address order; points of an
// edge group outside the box are written back with the prn value they were
// read with. Every grid is read once and prn written once, so the accesses are
// nontemporal. At 1000^3 FP32 this measured 3.64-3.70 ms against 3.95 ms for
// the row kernel above (wave-per-row 16-byte lanes: 3.86-3.91 ms cached,
// 4.16-4.20 ms nontemporal).
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_update_pressure16(TS *prn, const TS *prc, const TS *coef, const TS *lapla,
                                                           Box b, int64_t n1, int64_t n12, int64_t ng, int64_t total)
{
    constexpr int VW = 16 / sizeof(TS);
    using NV = TS __attribute__((ext_vector_type(VW)));
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int64_t row = t / ng, k = t - row * ng, N2 = b.n2();
    const int64_t i2 = b.s2 + row % N2, i3 = b.s3 + row / N2;
    const int64_t i1 = (b.s1 / VW + k) * VW, ii = i2 * n1 + i3 * n12 + i1;
    const TC two = (TC)2.0;
    const NV p = __builtin_nontemporal_load(reinterpret_cast<const NV *>(prn + ii));
    const NV c = __builtin_nontemporal_load(reinterpret_cast<const NV *>(prc + ii));
    const NV co = __builtin_nontemporal_load(reinterpret_cast<const NV *>(coef + ii));
    const NV la = __builtin_nontemporal_load(reinterpret_cast<const NV *>(lapla + ii));
    NV r;
#pragma unroll
    for (int v = 0; v < VW; v++) {
        const TS cl = co[v] * la[v];
        const TS nv = (TS)(two * (TC)c[v] - (TC)p[v] + (TC)cl);
        r[v] = (i1 + v >= b.s1 && i1 + v <= b.e1) ? nv : p[v];
    }
    __builtin_nontemporal_store(r, reinterpret_cast<NV *>(prn + ii));
}

// ---- reductions (src/grid.cpp:2006-2370) ----------------------------------------
enum RedOp { RED_SUM_ABS, RED_SUM_ABS_DIFF, RED_L1, RED_MAX_ERR, RED_MIN_MAX };

template <int OP>
struct RedInit {
    static __device__ double a() { return OP == RED_MAX_ERR ? -FLT_MAX : OP == RED_MIN_MAX ? FLT_MAX : 0.0; }
    static __device__ double b() { return OP == RED_MIN_MAX ? -FLT_MAX : 0.0; }
};

template <int OP>
__device__ inline void red_combine(double &a, double &b, double a2, double b2)
{
    if (OP == RED_MAX_ERR) {
        a = a2 > a ? a2 : a;
    } else if (OP == RED_MIN_MAX) {
        a = a2 < a ? a2 : a;
        b = b2 > b ? b2 : b;
    } else {
        a += a2;
        b += b2;
    }
}

template <int OP>
__device__ inline void block_reduce(double &a, double &b)
{
    __shared__ double sa[8], sb[8];
    for (int off = 32; off > 0; off >>= 1) {
        double a2 = __shfl_down(a, off, 64), b2 = __shfl_down(b, off, 64);
        red_combine<OP>(a, b, a2, b2);
    }
    const int lane = (threadIdx.y * blockDim.x + threadIdx.x) & 63;
    const int wave = (threadIdx.y * blockDim.x + threadIdx.x) >> 6;
    const int nwave = (blockDim.x * blockDim.y + 63) >> 6;
    if (lane == 0) {
        sa[wave] = a;
        sb[wave] = b;
    }
    __syncthreads();
    if (wave == 0) {
        a = lane < nwave ? sa[lane] : RedInit<OP>::a();
        b = lane < nwave ? sb[lane] : RedInit<OP>::b();
        for (int off = 4; off > 0; off >>= 1) {
            double a2 = __shfl_down(a, off, 64), b2 = __shfl_down(b, off, 64);
            red_combine<OP>(a, b, a2, b2);
        }
    }
}

// one point of a reduction: the sums in double, min / max in the storage type
// as the reference's Myfloat accumulator (src/grid.cpp:2006-2370)
template <typename TS, int OP>
__device__ __forceinline__ void red_point(TS x, TS y, double &a, double &c, TS &mn, TS &mx, float maxerr)
{
    if (OP == RED_SUM_ABS) {
        a += fabs((double)x);
    } else if (OP == RED_SUM_ABS_DIFF) {
        a += fabs((double)x - (double)y);
    } else if (OP == RED_L1) {
        a += fabs((double)x - (double)y);
        c += fabs((double)y);
    } else if (OP == RED_MAX_ERR) {
        const double d = fabs((double)x - (double)y);
        const double e = fabsf((float)y) < maxerr ? d : d / fabs((double)y);
        if (e > a) a = e;
    } else {
        if (x < mn) mn = x;
        if (x > mx) mx = x;
    }
}

// VEC: 16-byte loads over the aligned groups of each row (u and v 16-byte
// aligned), four loads in flight per operand, the unaligned head and tail of
// the row point by point; one wave per row either way.  1000^3 FP32 inner
// box: sum |u| 0.68 ms (1.86 ms point by point), sum |u - v| 1.40 ms (2.26 ms).
template <typename TS, int OP, bool VEC>
__global__ void __launch_bounds__(256) k_reduce(const TS *u, const TS *v, Box b, int64_t n1, int64_t n12,
                                                float maxerr, double *part)
{
    double a = RedInit<OP>::a(), c = RedInit<OP>::b();
    TS mn = (TS)FLT_MAX, mx = (TS)-FLT_MAX;
    constexpr bool TWO = OP != RED_SUM_ABS && OP != RED_MIN_MAX;
    if constexpr (!VEC) {
        for_box(b, n1, n12, [&](int64_t ii, int64_t, int64_t, int64_t) {
            red_point<TS, OP>(u[ii], TWO ? v[ii] : (TS)0, a, c, mn, mx, maxerr);
        });
    } else {
        constexpr int VW = 16 / sizeof(TS), UN = 4;                    // 4 loads in flight per operand
        using NV = TS __attribute__((ext_vector_type(VW)));
        const int64_t N2 = b.n2(), rows = N2 * b.n3();
        const int lane = threadIdx.x;
        for (int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.y; row < rows;
             row += (int64_t)gridDim.x * ROWS_PER_BLOCK) {
            const int64_t base = (b.s2 + row % N2) * n1 + (b.s3 + row / N2) * n12;
            const int64_t a0 = base + b.s1, a1 = base + b.e1 + 1;       // [a0, a1) flat
            const int64_t g0 = (a0 + VW - 1) / VW, g1 = a1 / VW;          // whole groups
            if (g0 >= g1) {                                               // short row
                for (int64_t i = a0 + lane; i < a1; i += ROW_THREADS)
                    red_point<TS, OP>(u[i], TWO ? v[i] : (TS)0, a, c, mn, mx, maxerr);
                continue;
            }
            const int64_t h = g0 * VW - a0, t = a1 - g1 * VW;             // head / tail points
            if (lane < h) red_point<TS, OP>(u[a0 + lane], TWO ? v[a0 + lane] : (TS)0, a, c, mn, mx, maxerr);
            if (lane < t) {
                const int64_t i = g1 * VW + lane;
                red_point<TS, OP>(u[i], TWO ? v[i] : (TS)0, a, c, mn, mx, maxerr);
            }
            for (int64_t gi = g0 + lane; gi < g1; gi += UN * ROW_THREADS) {
                NV x[UN], y[UN];
#pragma unroll
                for (int k = 0; k < UN; k++) {
                    const int64_t gk = gi + k * ROW_THREADS;
                    if (gk < g1) {
                        x[k] = *reinterpret_cast<const NV *>(u + gk * VW);
                        if constexpr (TWO) y[k] = *reinterpret_cast<const NV *>(v + gk * VW);
                    }
                }
#pragma unroll
                for (int k = 0; k < UN; k++) {
                    if (gi + k * ROW_THREADS >= g1) break;
#pragma unroll
                    for (int e = 0; e < VW; e++)
                        red_point<TS, OP>(x[k][e], TWO ? y[k][e] : (TS)0, a, c, mn, mx, maxerr);
                }
            }
        }
    }
    if (OP == RED_MIN_MAX) {
        a = (double)mn;
        c = (double)mx;
    }
    block_reduce<OP>(a, c);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        part[blockIdx.x] = a;
        part[gridDim.x + blockIdx.x] = c;
    }
}

// the 16-byte path where both operands are 16-byte aligned
static bool red_vec(const void *u, const void *v)
{
    return ((uintptr_t)u % 16) == 0 && ((uintptr_t)v % 16) == 0;
}

template <int OP>
__global__ void __launch_bounds__(256) k_reduce_final(const double *part, int nb, double *out)
{
    double a = RedInit<OP>::a(), c = RedInit<OP>::b();
    for (int i = threadIdx.x; i < nb; i += blockDim.x) red_combine<OP>(a, c, part[i], part[nb + i]);
    block_reduce<OP>(a, c);
    if (threadIdx.x == 0) {
        out[0] = a;
        out[1] = c;
    }
}

static std::mutex g_red_mu;   // the partial sums and the result are shared by all callers
// the result: 16 bytes of pinned host memory, allocated once for the process,
// which k_reduce_final writes (a copy from device memory took 3 us more).  The
// last block of k_reduce combining the partial sums itself was slower: the
// fences of its 1024 blocks took 35 us (300^3 sum |u| 60 us against 27 + 6).
static double *g_red_out;

// partial results per reduction: one block per ROWS_PER_BLOCK rows, at most
// RED_BLOCKS blocks (the rows of larger ranges are strided over them)
constexpr int RED_BLOCKS = 1024;
static int red_blocks(const Box &b)
{
    const int64_t rows = b.n2() * b.n3();
    const int64_t nb = (rows + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    return (int)(nb < RED_BLOCKS ? nb : RED_BLOCKS);
}

// Scratch of hsx_l1_sums_noalloc: the two partial sums of each of at most
// RED_BLOCKS blocks (16 KiB), one copy per device for the life of the process.
// Host code never uses this name as an address: it takes the device address
// of each device's copy from hipGetSymbolAddress (noalloc_scratch below).
static __device__ __align__(256) double scratch[2 * RED_BLOCKS];
constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_noalloc_mu;
static double *g_noalloc_ptr[NOALLOC_MAX_DEVICES];   // device address of scratch, per device

// the current device's copy of scratch, looked up once per device (with that
// device current)
static int noalloc_scratch(double **out)
{
    int dev = -1;
    HSX_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
        return fail(HSX_ERR_UNSUPPORTED, "device %d: the allocation-free entry points serve devices 0..%d", dev,
                    NOALLOC_MAX_DEVICES - 1);
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *p = nullptr;
        HSX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(HSX_ERR_HIP, "hipGetSymbolAddress(scratch) gave a null address");
        g_noalloc_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_noalloc_ptr[dev];
    return HSX_OK;
}

template <int OP>
static int run_reduce(const hsx_grid *g, const void *u, const void *v, const int64_t r[6], float maxerr,
                      double out[2], void *stream)
{
    int rc = check_grid(g);
    if (!rc) rc = check_range(g, r);
    if (!rc) rc = check_ptr(u, "u");
    if (!rc && OP != RED_SUM_ABS && OP != RED_MIN_MAX) rc = check_ptr(v, "v");
    if (!rc && !out) rc = fail(HSX_ERR_INVALID, "null out");
    if (!rc) rc = ensure_init();
    if (rc) return rc;
    std::lock_guard<std::mutex> lk(g_red_mu);
    const Box b = box_of(r);
    const int nb = red_blocks(b);
    double *part = nullptr;
    void *res = nullptr;
    if ((rc = scratch_get(SCRATCH_PARTIALS, sizeof(double) * 2 * nb, (void **)&part))) return rc;
    if (!g_red_out) HSX_HIP(hipHostMalloc((void **)&g_red_out, 2 * sizeof(double), hipHostMallocPortable));
    HSX_HIP(hipHostGetDevicePointer(&res, g_red_out, 0));
    hipStream_t s = stream_of(stream);
    rc = dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        if (red_vec(u, v))
            hipLaunchKernelGGL((k_reduce<TS, OP, true>), dim3(nb), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (const TS *)u, (const TS *)v, b, g->n1, g->n1 * g->n2, maxerr, part);
        else
            hipLaunchKernelGGL((k_reduce<TS, OP, false>), dim3(nb), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (const TS *)u, (const TS *)v, b, g->n1, g->n1 * g->n2, maxerr, part);
        HSX_LAUNCHED("k_reduce");
        return HSX_OK;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((k_reduce_final<OP>), dim3(1), dim3(256), 0, s, part, nb, (double *)res);
    HSX_LAUNCHED("k_reduce_final");
    HSX_HIP(hipStreamSynchronize(s));
    out[0] = g_red_out[0];
    out[1] = g_red_out[1];
    return HSX_OK;
}

static int common_checks(const hsx_grid *g, std::initializer_list<std::pair<const void *, const char *>> ptrs)
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

int hsx_fill_const(const hsx_grid *g, void *u, const int64_t range[6], double val, void *stream)
{
    int rc = common_checks(g, {{u, "u"}});
    if (!rc) rc = check_range(g, range);
    if (rc) return rc;
    const Box b = box_of(range);
    hipStream_t s = stream_of(stream);
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        if (((uintptr_t)u % 16) == 0)
            hipLaunchKernelGGL((k_fill_const<TS, true>), row_grid(b), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (TS *)u, b, g->n1, g->n1 * g->n2, (TS)val);
        else
            hipLaunchKernelGGL((k_fill_const<TS, false>), row_grid(b), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (TS *)u, b, g->n1, g->n1 * g->n2, (TS)val);
        HSX_LAUNCHED("k_fill_const");
        return HSX_OK;
    });
}

int hsx_fill_separable(const hsx_grid *g, void *u, const int64_t range[6], const double *t1,
                       const double *t2, const double *t3, double amp, void *stream)
{
    int rc = common_checks(g, {{u, "u"}, {t1, "t1"}, {t2, "t2"}, {t3, "t3"}});
    if (!rc) rc = check_range(g, range);
    if (rc) return rc;
    const Box b = box_of(range);
    const size_t l1 = b.n1(), l2 = b.n2(), l3 = b.n3();
    double *tab = nullptr;
    static std::mutex mu;   // the table staging buffer is shared
    std::lock_guard<std::mutex> lk(mu);
    if ((rc = scratch_get(SCRATCH_TABLES, sizeof(double) * (l1 + l2 + l3), (void **)&tab))) return rc;
    hipStream_t s = stream_of(stream);
    HSX_HIP(hipMemcpyAsync(tab, t1, sizeof(double) * l1, hipMemcpyHostToDevice, s));
    HSX_HIP(hipMemcpyAsync(tab + l1, t2, sizeof(double) * l2, hipMemcpyHostToDevice, s));
    HSX_HIP(hipMemcpyAsync(tab + l1 + l2, t3, sizeof(double) * l3, hipMemcpyHostToDevice, s));
    rc = dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        if (((uintptr_t)u % 16) == 0)
            hipLaunchKernelGGL((k_fill_sep<TS, true>), row_grid(b), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (TS *)u, b, g->n1, g->n1 * g->n2, tab, tab + l1, tab + l1 + l2, amp);
        else
            hipLaunchKernelGGL((k_fill_sep<TS, false>), row_grid(b), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (TS *)u, b, g->n1, g->n1 * g->n2, tab, tab + l1, tab + l1 + l2, amp);
        HSX_LAUNCHED("k_fill_sep");
        return HSX_OK;
    });
    if (rc) return rc;
    // the staging buffer is reused by the next call: finish with it here
    HSX_HIP(hipStreamSynchronize(s));
    return HSX_OK;
}

int hsx_array_op(const hsx_grid *g, int op, void *w, const void *u, const void *v, double val, void *stream)
{
    int rc = common_checks(g, {{w, "w"}});
    if (rc) return rc;
    if (op < HSX_ARRAY_FILL || op > HSX_ARRAY_ADDTO) return fail(HSX_ERR_INVALID, "array op %d", op);
    if (op != HSX_ARRAY_FILL && (rc = check_ptr(u, "u"))) return rc;
    if ((op == HSX_ARRAY_ADD || op == HSX_ARRAY_MULTIPLY) && (rc = check_ptr(v, "v"))) return rc;
    const int64_t n = g->n1 * g->n2 * g->n3;
    hipStream_t s = stream_of(stream);
    auto a16 = [](const void *p) { return p == nullptr || ((uintptr_t)p & 15) == 0; };
    const bool vec = a16(w) && a16(u) && a16(v);
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        const int64_t work = vec ? n / (16 / (int64_t)sizeof(TS)) + 1 : n;
        int64_t nb = (work + 255) / 256;
        if (nb > 8192) nb = 8192;
        if (vec)
            hipLaunchKernelGGL(k_array16<TS>, dim3((unsigned)nb), dim3(256), 0, s, op, (TS *)w, (const TS *)u,
                               (const TS *)v, (TS)val, n);
        else
            hipLaunchKernelGGL(k_array<TS>, dim3((unsigned)nb), dim3(256), 0, s, op, (TS *)w, (const TS *)u,
                               (const TS *)v, (TS)val, n);
        HSX_LAUNCHED("k_array");
        return HSX_OK;
    });
}

int hsx_free_surface(const hsx_grid *g, void *u, int face_mask, void *stream)
{
    int rc = common_checks(g, {{u, "u"}});
    if (rc) return rc;
    hipStream_t s = stream_of(stream);
    FaceSet fs;
    bool closed_form;
    int64_t most, most_plane;
    if ((rc = make_faceset(g, face_mask, &fs, &closed_form, &most, &most_plane))) return rc;
    if (fs.n == 0) return HSX_OK;
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        // n1 faces alone in 16-byte row ends are one launch anyway (k_bc_n1: no rows to
        // leave out; 500^3 FP32 order 8 19.4 us for both faces, in k_bc_one 21.4)
        Face nlo{}, nhi{};
        const bool n1_only = fs.zmask < 4 && n1_vector_sides(g, u, fs, &nlo, &nhi);
        if (closed_form && !n1_only) {
            const int r = bc_one_launch(g, (TS *)u, fs, NoExtra(), s);
            if (r != HSX_ERR_UNSUPPORTED) return r;
        }
        if (closed_form) {
            const unsigned nb1 = (unsigned)std::min<int64_t>((most + 255) / 256, 4096);
            const unsigned nb2 = (unsigned)std::min<int64_t>((most_plane + 255) / 256, 4096);
            FaceSet rest = fs;                   // the faces left to the two generic launches
            rest.vec1 = n1_groups_ok(g, u, fs);
            Face lo{}, hi{};
            const int sides = n1_vector_sides(g, u, fs, &lo, &hi);
            if (sides) {
                const Face &f = (sides & 1) ? lo : hi;
                const int64_t threads = (f.be - f.bs + 1) * (f.oe - f.os + 1) * (sides == 3 ? 2 : 1);
                const dim3 grid((unsigned)((threads + 255) / 256));
                rest.n = 0;
                for (int k = 0; k < fs.n; k++)
                    if (fs.f[k].axis != 0) rest.f[rest.n++] = fs.f[k];
                if (rest.n == 0) {
                    switch ((f.he - f.hs + 1) / (16 / (int64_t)sizeof(TS))) {
                    case 1: hipLaunchKernelGGL((k_bc_n1<TS, 1>), grid, dim3(256), 0, s, (TS *)u, lo, hi, sides); break;
                    case 2: hipLaunchKernelGGL((k_bc_n1<TS, 2>), grid, dim3(256), 0, s, (TS *)u, lo, hi, sides); break;
                    case 3: hipLaunchKernelGGL((k_bc_n1<TS, 3>), grid, dim3(256), 0, s, (TS *)u, lo, hi, sides); break;
                    default: hipLaunchKernelGGL((k_bc_n1<TS, 4>), grid, dim3(256), 0, s, (TS *)u, lo, hi, sides); break;
                    }
                    HSX_LAUNCHED("k_bc_n1");
                    return HSX_OK;
                }
                const uint32_t nbn = grid.x;
                const dim3 both(nbn + nb1 * (uint32_t)rest.n);
                switch ((f.he - f.hs + 1) / (16 / (int64_t)sizeof(TS))) {
                case 1: hipLaunchKernelGGL((k_bc_n1_mirror<TS, 1>), both, dim3(256), 0, s, (TS *)u, lo, hi, sides, rest, nbn, nb1); break;
                case 2: hipLaunchKernelGGL((k_bc_n1_mirror<TS, 2>), both, dim3(256), 0, s, (TS *)u, lo, hi, sides, rest, nbn, nb1); break;
                case 3: hipLaunchKernelGGL((k_bc_n1_mirror<TS, 3>), both, dim3(256), 0, s, (TS *)u, lo, hi, sides, rest, nbn, nb1); break;
                default: hipLaunchKernelGGL((k_bc_n1_mirror<TS, 4>), both, dim3(256), 0, s, (TS *)u, lo, hi, sides, rest, nbn, nb1); break;
                }
                HSX_LAUNCHED("k_bc_n1_mirror");
                hipLaunchKernelGGL(k_bc_zero<TS>, dim3(nb2, rest.n), dim3(256), 0, s, (TS *)u, rest);
                HSX_LAUNCHED("k_bc_zero");
                return HSX_OK;
            }
            hipLaunchKernelGGL(k_bc_mirror<TS>, dim3(nb1, rest.n), dim3(256), 0, s, (TS *)u, rest);
            HSX_LAUNCHED("k_bc_mirror");
            hipLaunchKernelGGL(k_bc_zero<TS>, dim3(nb2, rest.n), dim3(256), 0, s, (TS *)u, rest);
            HSX_LAUNCHED("k_bc_zero");
            return HSX_OK;
        }
        // small grids: the reference's six phases one after the other
        for (int k = 0; k < fs.n; k++) {
            const Face &f = fs.f[k];
            const int64_t total = (f.he - f.hs + 2) * (f.be - f.bs + 1) * (f.oe - f.os + 1);
            const unsigned nb = (unsigned)std::min<int64_t>((total + 255) / 256, 16384);
            hipLaunchKernelGGL(k_free_surface<TS>, dim3(nb), dim3(256), 0, s, (TS *)u, f);
            HSX_LAUNCHED("k_free_surface");
        }
        return HSX_OK;
    });
}

int hsx_update_pressure(const hsx_grid *g, void *prn, const void *prc, const void *coef, const void *lapla,
                        void *stream)
{
    int rc = common_checks(g, {{prn, "prn"}, {prc, "prc"}, {coef, "coef"}, {lapla, "lapla"}});
    if (rc) return rc;
    const Box b = box_of(g->inner);
    hipStream_t s = stream_of(stream);
    return dispatch_types(g, [&](auto ts, auto tc) -> int {
        using TS = decltype(ts);
        using TC = decltype(tc);
        constexpr int VW = 16 / sizeof(TS);
        const bool wide = g->n1 % VW == 0 &&
                          ((uintptr_t)prn | (uintptr_t)prc | (uintptr_t)coef | (uintptr_t)lapla) % 16 == 0;
        const int64_t ng = b.e1 / VW - b.s1 / VW + 1, total = ng * b.n2() * b.n3();
        if (wide && total > 0 && (total + 255) / 256 <= INT32_MAX) {
            hipLaunchKernelGGL((k_update_pressure16<TS, TC>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                               (TS *)prn, (const TS *)prc, (const TS *)coef, (const TS *)lapla, b, g->n1,
                               g->n1 * g->n2, ng, total);
            HSX_LAUNCHED("k_update_pressure16");
            return HSX_OK;
        }
        hipLaunchKernelGGL((k_update_pressure<TS, TC>), row_grid(b), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                           (TS *)prn, (const TS *)prc, (const TS *)coef, (const TS *)lapla, b, g->n1,
                           g->n1 * g->n2);
        HSX_LAUNCHED("k_update_pressure");
        return HSX_OK;
    });
}

int hsx_sum_abs(const hsx_grid *g, const void *u, const int64_t range[6], double *out, void *stream)
{
    double r[2];
    int rc = run_reduce<RED_SUM_ABS>(g, u, nullptr, range, 0.f, r, stream);
    if (!rc) *out = r[0];
    return rc;
}

int hsx_sum_abs_diff(const hsx_grid *g, const void *u, const void *v, const int64_t range[6], double *out,
                     void *stream)
{
    double r[2];
    int rc = run_reduce<RED_SUM_ABS_DIFF>(g, u, v, range, 0.f, r, stream);
    if (!rc) *out = r[0];
    return rc;
}

int hsx_l1_sums(const hsx_grid *g, const void *u, const void *v, const int64_t range[6], double out[2],
                void *stream)
{
    return run_reduce<RED_L1>(g, u, v, range, 0.f, out, stream);
}

int hsx_l1_sums_noalloc(const hsx_grid *g, const void *u, const void *v, const int64_t range[6], double *out,
                        void *stream)
{
    int rc = check_grid(g);
    if (!rc) rc = check_range(g, range);
    if (!rc) rc = check_ptr(u, "u");
    if (!rc) rc = check_ptr(v, "v");
    if (!rc) rc = check_ptr(out, "out");
    if (!rc) rc = ensure_init();
    if (rc) return rc;
    double *part = nullptr;
    if ((rc = noalloc_scratch(&part))) return rc;
    const Box b = box_of(range);
    const int nb = red_blocks(b);
    if (nb < 1 || nb > RED_BLOCKS)
        return fail(HSX_ERR_INVALID, "l1_sums_noalloc: %d partial blocks, the scratch holds %d", nb, RED_BLOCKS);
    hipStream_t s = stream_of(stream);
    // every block writes its own partials before k_reduce_final reads them:
    // nothing in scratch has to start at zero
    rc = dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        if (red_vec(u, v))
            hipLaunchKernelGGL((k_reduce<TS, RED_L1, true>), dim3(nb), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (const TS *)u, (const TS *)v, b, g->n1, g->n1 * g->n2, 0.f, part);
        else
            hipLaunchKernelGGL((k_reduce<TS, RED_L1, false>), dim3(nb), dim3(ROW_THREADS, ROWS_PER_BLOCK), 0, s,
                               (const TS *)u, (const TS *)v, b, g->n1, g->n1 * g->n2, 0.f, part);
        HSX_LAUNCHED("k_reduce");
        return HSX_OK;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((k_reduce_final<RED_L1>), dim3(1), dim3(256), 0, s, part, nb, out);
    HSX_LAUNCHED("k_reduce_final");
    return HSX_OK;
}

int hsx_max_err(const hsx_grid *g, const void *u, const void *v, const int64_t range[6], double max_err_float,
                double *out, void *stream)
{
    double r[2];
    int rc = run_reduce<RED_MAX_ERR>(g, u, v, range, (float)max_err_float, r, stream);
    if (!rc) *out = r[0];
    return rc;
}

int hsx_min_max(const hsx_grid *g, const void *u, const int64_t range[6], double out[2], void *stream)
{
    return run_reduce<RED_MIN_MAX>(g, u, nullptr, range, 0.f, out, stream);
}

} // extern "C"
