// What ends a time step of the shot loops (sources, receivers, the residual and
// source terms of a reverse step) in one launch with the free surface that the
// next step begins with.
#ifndef HSX_STEP_END_H
#define HSX_STEP_END_H

#include "hsx_internal.h"

namespace hsx {

// forward: the most sources that the merged launch takes (each thread of the
// free surface compares its points with them)
constexpr int END_SRC_MAX = 4;
// forward: the most receivers on the n2 and n3 boundary planes (the ends of a
// receiver line), which the merged launch records before it zeroes them
constexpr int END_EDGE_MAX = 16;
// device workspace of a shot: whether another source or receiver lies on a point
// that the free surface writes, the sources' coordinates, and the receivers on
// the planes, coordinates and numbers
struct EndWork {
    int outside;
    int c[END_SRC_MAX][3];
    int ne;
    int e[END_EDGE_MAX][3];
    int64_t ei[END_EDGE_MAX];
};

// The source term of reverse step k (the imaging condition's -F part:
// grad[src_i] -= scale * mu^k[src_i] * f_i, for the sources inside the imaging
// box b only) and the residual of step k-1 into
// mu^{k+1} (v[rec_i] += -1 * res_i * crec_i, in double, as k_inject): blocks
// [0, nb_src) take the sources, the next nb_rec the receivers; the two parts
// touch different buffers.
// side (imaging in pairs of steps, first of the pair: hold, then not): the pair's
// sum over the whole grid lacks the first step's source term between its two
// terms, so the points with a source are summed here in the order of single
// steps, through side[i], and overwrite the pair's.
template <typename TS>
struct ReverseEnd {
    double *grad;
    const TS *mu, *q0, *q1, *q2;
    double *side;
    int hold;
    int64_t nsrc;
    const int64_t *sidx;
    const TS *f;
    double scale;
    Box b;
    int64_t n1, n12;
    uint32_t nb_src, nb_rec;
    TS *v;
    int64_t npoint, nrec;
    const int64_t *ridx;
    const TS *res, *crec;

    __device__ __forceinline__ void block(uint32_t bx) const
    {
        if (bx < nb_src) {
            const int64_t i = (int64_t)bx * blockDim.x + threadIdx.x;
            if (i >= nsrc) return;
            const int64_t j = sidx[i];
            const int64_t i3 = j / n12, i2 = (j - i3 * n12) / n1, i1 = j - i3 * n12 - i2 * n1;
            if (i1 < b.s1 || i1 > b.e1 || i2 < b.s2 || i2 > b.e2 || i3 < b.s3 || i3 > b.e3) return;
            double x = side && !hold ? side[i] : grad[j];
            if (side) {
                const double d2 = ((double)q0[j] - 2.0 * (double)q1[j]) + (double)q2[j];
                x += scale * (double)mu[j] * d2;
            }
            x += -scale * (double)mu[j] * (double)f[i];
            (hold ? side + i : grad + j)[0] = x;
            return;
        }
        for (int64_t i = (int64_t)(bx - nb_src) * blockDim.x + threadIdx.x; i < nrec; i += (int64_t)nb_rec * blockDim.x) {
            if ((uint64_t)ridx[i] >= (uint64_t)npoint) continue;
            double x = -1.0 * (double)res[i];
            x *= (double)crec[i];
            TS *p = v + ridx[i];
            *p = (TS)((double)*p + x);
        }
    }
};

// Forward: *merge = whether step_end_forward serves the shot (few sources, every
// source and, but for a few on the n2 and n3 planes, every receiver strictly
// inside the boundary planes, a free surface in one launch); fills work and
// waits for the stream.
int step_end_check(const hsx_grid *g, int64_t nsrc, const int64_t *src, int64_t nrec, const int64_t *rec,
                   EndWork *work, bool *merge, hipStream_t s);
// u += the sources' samples, tr = u at the receivers (tr NULL: none), then the
// free surface of u
int step_end_forward(const hsx_grid *g, void *u, int64_t nsrc, const int64_t *src, const void *w, int64_t nrec,
                     const int64_t *rec, void *tr, const EndWork *work, hipStream_t s);
// r's blocks and the free surface of u (not r.v; a buffer that r reads inside
// the boundary planes only); HSX_ERR_UNSUPPORTED, nothing done, where the free
// surface takes several launches
template <typename TS>
int step_end_reverse(const hsx_grid *g, void *u, const ReverseEnd<TS> &r, hipStream_t s);

// the free surface of many grids in one launch: bytes of one grid's entry in the
// device table; the entry (false: this grid needs several launches), with its
// n1 halo groups and blocks; the launch over all entries, of one nh, with the
// largest number of blocks
size_t bc_one_batch_bytes(void);
bool bc_one_batch_fill(const hsx_grid *g, const void *u, const FaceSet &fs, void *out, int *nh, uint32_t *blocks);
int bc_one_batch_launch(int storage, int nshots, void *const *d_fields, const void *d_grids, int nh, uint32_t blocks,
                        hipStream_t s);

// both snapshots of a 16-bit checkpoint (u in p0, u - u_prev in p1; the codes of
// hsx_ckpt_encode, 16-byte aligned buffers), and back
int ckpt_encode_pair(const float *u, const float *u_prev, int64_t n, void *p0, void *p1, int format, hipStream_t s);
int ckpt_decode_pair(const void *p0, const void *p1, int64_t n, int format, float *u, float *u_prev, hipStream_t s);

} // namespace hsx

#endif
