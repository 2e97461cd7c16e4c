// Forward modeling of a shot and the gradient of the receiver misfit with
// respect to squared slowness (adjoint of the Ac2 propagator with
// checkpointing).  The reference has no adjoint (its ADJOINT mode is a stub,
// src/data_Acquisition.cpp:307-310); the forward step is the reference's
// Propagator_Ac2 step (src/propagator_Ac2.cpp:366-393) plus a point source.
//
// Discrete problem, with q^n the wavefield after the free surface B:
//   q^{n+1} = B( 2 q^n - q^{n-1} + c (L q^n) + F^n ),   c = dt^2 / m,
//   d^n_r = q^{n+1}(x_r),   J = 1/2 sum_{n,r} (d^n_r - dobs^n_r)^2,
// L the FD Laplacian with the antisymmetric halos of B, which is symmetric on
// the points B does not zero.  The adjoint field is carried as mu = c lambda:
//   mu^k = 2 mu^{k+1} - (mu^{k+2} - c e^k) + c (L mu^{k+1}),  e^k = residual at step k-1,
// i.e. the forward step itself (free surface + fused kernel) with the residual,
// scaled by c, taken off mu^{k+2} at the receivers first.  The imaging condition is
//   dJ/dm = -(1/dt^2) sum_k mu^k (q^k - 2 q^{k-1} + q^{k-2} - F^{k-1}),
// accumulated in double over the points B does not touch, by the adjoint
// step's own kernel where the tiled kernels take the grid.
#include <algorithm>
#include <vector>

#include "hsx_internal.h"
#include "hsx_route.h"
#include "hsx_step_end.h"

namespace hsx {

// res = d - dobs (d NULL: res = dobs, the residual given by the caller);
// partial[block] = sum of res^2 over the block (double)
template <typename TS>
__global__ void __launch_bounds__(256) k_residual(const TS *d, const TS *dobs, TS *res, int64_t n, double *partial)
{
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const TS r = d ? d[i] - dobs[i] : dobs[i];
        res[i] = r;
        acc += (double)r * (double)r;
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    __shared__ double wsum[4];
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
}

__global__ void k_sum_partials(const double *partial, int n, double *out)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        double s = 0.0;
        for (int i = 0; i < n; i++) s += partial[i];
        out[0] = s;
    }
}

// Sources then receivers of one forward step in one launch (k_inject + k_gather
// in order): block 0 adds the sources (out += 1.0 * w, in double), waits, then
// records the receivers that sit on a source point; the other blocks record
// every other receiver, whose points no source writes.  nsrc <= SRCREC_MAX
// (the membership test is a loop over the sources).
constexpr int64_t SRCREC_MAX = 64;

__device__ __forceinline__ bool on_source(int64_t j, int64_t nsrc, const int64_t *src)
{
    for (int64_t k = 0; k < nsrc; k++)
        if (src[k] == j) return true;
    return false;
}

// A step out of place writes the inner points of its output only; outside them a
// step in place leaves q^{n-1} as its free surface left it.  A receiver there
// records that (hsx_forward's traces, whose steps are in place), so the point is
// carried from prev, q^{n-1}, into the output, whose two next steps need it in
// turn.  prev NULL: a step in place, nothing to carry.
template <typename TS>
struct Carry {
    const TS *prev;
    Box in;
    int64_t n1, n12;

    __device__ __forceinline__ bool at(int64_t j) const
    {
        if (!prev) return false;
        const int64_t i3 = j / n12, i2 = (j - i3 * n12) / n1, i1 = j - i3 * n12 - i2 * n1;
        return i1 < in.s1 || i1 > in.e1 || i2 < in.s2 || i2 > in.e2 || i3 < in.s3 || i3 > in.e3;
    }
};

template <typename TS>
__global__ void __launch_bounds__(256) k_srcrec(TS *u, int64_t npoint, int64_t nsrc, const int64_t *src, const TS *w,
                                                int64_t nrec, const int64_t *rec, TS *tr, Carry<TS> c)
{
    if (blockIdx.x == 0) {
        for (int64_t i = threadIdx.x; i < nsrc; i += blockDim.x) {
            const int64_t j = src[i];
            if ((uint64_t)j >= (uint64_t)npoint) continue;
            u[j] = (TS)((double)(c.at(j) ? c.prev[j] : u[j]) + 1.0 * (double)w[i]);
        }
        __syncthreads();
        for (int64_t i = threadIdx.x; i < nrec; i += blockDim.x) {
            const int64_t j = rec[i];
            if (on_source(j, nsrc, src)) tr[i] = (uint64_t)j < (uint64_t)npoint ? u[j] : (TS)0;
        }
        return;
    }
    for (int64_t i = (int64_t)(blockIdx.x - 1) * blockDim.x + threadIdx.x; i < nrec;
         i += (int64_t)(gridDim.x - 1) * blockDim.x) {
        const int64_t j = rec[i];
        if (on_source(j, nsrc, src)) continue;
        const bool in = (uint64_t)j < (uint64_t)npoint;
        if (in && c.at(j)) u[j] = c.prev[j];
        tr[i] = in ? u[j] : (TS)0;
    }
}

// the receivers' points carried alone, before sources that take a launch of their own
template <typename TS>
__global__ void __launch_bounds__(256) k_carry(TS *u, int64_t npoint, int64_t nrec, const int64_t *rec, Carry<TS> c)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nrec; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = rec[i];
        if ((uint64_t)j < (uint64_t)npoint && c.at(j)) u[j] = c.prev[j];
    }
}

// the end of a reverse step alone (hsx_step_end.h)
template <typename TS>
__global__ void __launch_bounds__(256) k_reverse_end(ReverseEnd<TS> r)
{
    r.block(blockIdx.x);
}

// the imaging condition of two reverse steps in one pass over the gradient, for
// the grids that the tiled kernels do not take: mu1, mu2 the two outputs in
// order, q[0] .. q[3] the four wavefields, later ones first
template <typename TS>
struct Four {
    const TS *q[4];
};
template <typename TS>
__global__ void __launch_bounds__(256) k_imaging_pair(double *grad, const TS *mu1, const TS *mu2, Four<TS> w, Box b,
                                                      int64_t n1, int64_t n12, double scale)
{
    const int64_t N1 = b.n1(), N2 = b.n2(), rows = N2 * b.n3();
    for (int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.y; row < rows; row += (int64_t)gridDim.x * 4) {
        const int64_t base = (b.s2 + row % N2) * n1 + (b.s3 + row / N2) * n12 + b.s1;
        for (int64_t k = threadIdx.x; k < N1; k += 64) {
            const int64_t i = base + k;
            const double a = (double)w.q[0][i], c = (double)w.q[1][i], d = (double)w.q[2][i], e = (double)w.q[3][i];
            double x = grad[i];
            x += scale * (double)mu1[i] * ((a - 2.0 * c) + d);
            x += scale * (double)mu2[i] * ((c - 2.0 * d) + e);
            grad[i] = x;
        }
    }
}

// steps from which the check of the sources and receivers (two small launches and
// a wait, about 30 us) is worth the launch it saves on each step, 5 us
constexpr int64_t END_LEAST_STEPS = 24;

// sources up to which the imaging condition goes in pairs of steps
constexpr int64_t PAIR_SRC_MAX = 4096;

struct Dev {
    void *p = nullptr;
    ~Dev()
    {
        if (p) (void)hipFree(p);
    }
    int alloc(size_t bytes)
    {
        hipError_t e = dev_malloc(&p, bytes);
        return e == hipSuccess ? HSX_OK : hip_fail(e, "hipMalloc (adjoint buffers)");
    }
    char *c() const { return (char *)p; }
};

static int shot_checks(const hsx_grid *g, const void *coef, const hsx_shot *sh)
{
    int rc = check_grid(g);
    if (rc) return rc;
    if ((rc = check_ptr(coef, "coef")) || (rc = check_ptr(sh, "shot"))) return rc;
    if (sh->nt < 1) return fail(HSX_ERR_INVALID, "shot: nt = %lld", (long long)sh->nt);
    if (sh->nsrc < 0 || sh->nrec < 0) return fail(HSX_ERR_INVALID, "shot: negative source / receiver count");
    if (sh->nsrc > 0 && ((rc = check_ptr(sh->src_idx, "src_idx")) || (rc = check_ptr(sh->wavelet, "wavelet"))))
        return rc;
    if (sh->nrec > 0 && (rc = check_ptr(sh->rec_idx, "rec_idx"))) return rc;
    if (!(sh->dt > 0)) return fail(HSX_ERR_INVALID, "shot: dt must be > 0");
    return ensure_init();
}

static int zero(const hsx_grid *g, void *u, hipStream_t s)
{
    return hsx_array_op(g, HSX_ARRAY_FILL, u, nullptr, nullptr, 0.0, s);
}

static int imaging_pair(const hsx_grid *g, double *grad, const void *mu1, const void *mu2, const void *q0,
                        const void *q1, const void *q2, const void *q3, const Box &b, double scale, hipStream_t s)
{
    const int64_t rows = b.n2() * b.n3();
    const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>((rows + 3) / 4, 1 << 20));
    return dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        const Four<TS> w = {{(const TS *)q0, (const TS *)q1, (const TS *)q2, (const TS *)q3}};
        hipLaunchKernelGGL(k_imaging_pair<TS>, dim3(nb), dim3(64, 4), 0, s, grad, (const TS *)mu1, (const TS *)mu2, w, b,
                           g->n1, g->n1 * g->n2, scale);
        HSX_LAUNCHED("k_imaging_pair");
        return HSX_OK;
    });
}

// One forward step: out <- B(cur) step, source, record.  work (NULL: never, else
// step_end_check agreed): where end is set, the free surface of out, which the
// next step begins with, goes with the sources and receivers in one launch;
// *done says whether cur's was done like that, and on return whether out's was.
static int fwd_step(const hsx_grid *g, const void *coef, const hsx_shot *sh, void *out, const void *prev, void *cur,
                    int64_t n, void *traces, size_t es, const EndWork *work, bool end, bool *done, hipStream_t s)
{
    int rc = *done ? HSX_OK : hsx_free_surface(g, cur, 0x3F, s);
    if (!rc) rc = hsx_ac2_step_to(g, out, prev, cur, coef, s);
    *done = work && end;
    if (!rc && *done)
        return step_end_forward(g, out, sh->nsrc, sh->src_idx, (const char *)sh->wavelet + (size_t)n * sh->nsrc * es,
                                sh->nrec, sh->rec_idx,
                                traces && sh->nrec > 0 ? (char *)traces + (size_t)n * sh->nrec * es : nullptr, work, s);
    const bool record = sh->nrec > 0 && traces;
    const bool one = sh->nsrc > 0 && sh->nsrc <= SRCREC_MAX;
    if (!rc && record && (one || out != prev)) {
        const int64_t nrec = sh->nrec, npoint = g->n1 * g->n2 * g->n3;
        const unsigned nb = (unsigned)std::min<int64_t>((nrec + 255) / 256, 1024);
        rc = dispatch_types(g, [&](auto ts, auto) -> int {
            using TS = decltype(ts);
            const Carry<TS> c = {out != prev ? (const TS *)prev : (const TS *)nullptr, box_of(g->inner), g->n1,
                                 g->n1 * g->n2};
            if (one) {
                hipLaunchKernelGGL(k_srcrec<TS>, dim3(1 + nb), dim3(256), 0, s, (TS *)out, npoint, sh->nsrc, sh->src_idx,
                                   (const TS *)((const char *)sh->wavelet + (size_t)n * sh->nsrc * es), nrec,
                                   sh->rec_idx, (TS *)((char *)traces + (size_t)n * nrec * es), c);
                HSX_LAUNCHED("k_srcrec");
            } else {
                hipLaunchKernelGGL(k_carry<TS>, dim3(nb), dim3(256), 0, s, (TS *)out, npoint, nrec, sh->rec_idx, c);
                HSX_LAUNCHED("k_carry");
            }
            return HSX_OK;
        });
        if (one || rc) return rc;
    }
    if (!rc && sh->nsrc > 0)
        rc = hsx_inject(g, out, sh->nsrc, sh->src_idx, (const char *)sh->wavelet + (size_t)n * sh->nsrc * es, nullptr,
                        1.0, HSX_INJECT_ADD, s);
    if (!rc && record)
        rc = hsx_gather(g, out, sh->nrec, sh->rec_idx, (char *)traces + (size_t)n * sh->nrec * es, s);
    return rc;
}

} // namespace hsx

// Work buffers of hsx_gradient for one grid layout, nt, receiver count and
// checkpoint options, allocated once (hsx_adjoint_plan_create) and reused by
// every gradient of that geometry.
struct hsx_adjoint_plan {
    hsx_grid g;
    int64_t nt = 0, nrec = 0;
    hsx_adjoint_opts opt;
    size_t es = 4, bytes = 0, snap = 0;
    int64_t nseg = 0;
    hsx::Dev traces, res, crec, partial, msum, side, end, m1, m2, ck, fa, fb;
    std::vector<hsx::Dev> q;   // wavefields q^{m}, m from the segment start - 1
};

namespace hsx {

static int plan_checks(const hsx_grid *g, int64_t nt, int64_t nrec, const hsx_adjoint_opts *opt)
{
    int rc = check_grid(g);
    if (rc) return rc;
    if ((rc = check_ptr(opt, "opts"))) return rc;
    if (nt < 1) return fail(HSX_ERR_INVALID, "nt = %lld", (long long)nt);
    if (nrec < 0) return fail(HSX_ERR_INVALID, "negative receiver count");
    const int K = opt->ckpt_every;
    const int fmt = opt->ckpt_format;
    if (K < 0) return fail(HSX_ERR_INVALID, "ckpt_every %d < 0", K);
    if (fmt != HSX_CKPT_FP32 && fmt != HSX_CKPT_FP16 && fmt != HSX_CKPT_BF16)
        return fail(HSX_ERR_INVALID, "checkpoint format %d", fmt);
    if (fmt != HSX_CKPT_FP32 && g->storage != HSX_FP32)
        return fail(HSX_ERR_UNSUPPORTED, "16-bit checkpoints of FP64 wavefields");
    if (K == 0 && fmt != HSX_CKPT_FP32) return fail(HSX_ERR_INVALID, "full storage keeps every step in the storage type");
    if (opt->flags & ~(HSX_ADJ_RESIDUAL | HSX_ADJ_AUTOTUNE))
        return fail(HSX_ERR_INVALID, "adjoint flags 0x%x", opt->flags);
    for (int a = 0; a < g->dim; a++)
        if (g->inner[2 * a + 1] - g->inner[2 * a] < 2) return fail(HSX_ERR_INVALID, "grid too small for the imaging range");
    return ensure_init();
}

static bool same_layout(const hsx_grid &a, const hsx_grid &b)
{
    if (a.dim != b.dim || a.fd_order != b.fd_order || a.storage != b.storage || a.compute != b.compute ||
        a.n1 != b.n1 || a.n2 != b.n2 || a.n3 != b.n3)
        return false;
    for (int k = 0; k < 6; k++)
        if (a.inner[k] != b.inner[k]) return false;
    return true;
}

static int plan_run(hsx_adjoint_plan *P, const hsx_grid *g, const void *coef, const hsx_shot *sh, const void *d_obs,
                    double *grad, double *misfit, hipStream_t s)
{
    int rc;
    const int K = P->opt.ckpt_every;
    const int fmt = P->opt.ckpt_format;
    const bool given_residual = (P->opt.flags & HSX_ADJ_RESIDUAL) != 0;
    const size_t es = P->es, snap = P->snap;
    const int64_t npoint = g->n1 * g->n2 * g->n3;
    const int64_t nt = sh->nt, nrec = sh->nrec, ntr = nt * nrec, nseg = P->nseg;

    // imaging range: the inner points minus the boundary planes zeroed by B
    int64_t rim[6];
    for (int a = 0; a < 3; a++) {
        rim[2 * a] = g->inner[2 * a] + (a < g->dim ? 1 : 0);
        rim[2 * a + 1] = g->inner[2 * a + 1] - (a < g->dim ? 1 : 0);
    }
    const Box rimb = box_of(rim);
    const double img_scale = -1.0 / (sh->dt * sh->dt);
    auto &q = P->q;

    // Where the forward pass leaves q^m, m = -1 .. nt.  With full storage and
    // storage-type checkpoints the last segment (without checkpoints the only
    // one) goes straight to the buffers its reverse steps read, and the steps
    // themselves write the checkpoints: neither is computed twice or copied.
    // 16-bit checkpoints are restored in every segment, whose wavefields all
    // carry the same rounding.
    // (160 x 150 x 170 FP64 order 8, 60 steps: checkpoints every 10 steps 12.8 ->
    // 7.1 ms, full storage 9.4 -> 5.7, with the imaging below and the tile shapes)
    const bool in_place = K > 0 && fmt == HSX_CKPT_FP32;
    const int64_t n_last = K == 0 ? 0 : in_place ? (nseg - 1) * K : nt + 2;
    auto ck_at = [&](int64_t seg, int which) -> void * { return P->ck.c() + ((size_t)seg * 2 + which) * snap; };
    auto loc = [&](int64_t m) -> void * {
        if (m >= n_last - 1) return q[m - n_last + 1].p;
        if (in_place && m % K == 0) return ck_at(m / K, 0);
        if (in_place && (m + 1) % K == 0) return ck_at((m + 1) / K, 1);
        return m & 1 ? P->fa.p : P->fb.p;
    };
    auto save = [&](int64_t seg, const void *cur, const void *prev) -> int {
        return ckpt_encode_pair((const float *)cur, (const float *)prev, npoint, ck_at(seg, 0), ck_at(seg, 1), fmt, s);
    };
    auto restore = [&](int64_t seg, void *cur, void *prev) -> int {
        return ckpt_decode_pair(ck_at(seg, 0), ck_at(seg, 1), npoint, fmt, (float *)cur, (float *)prev, s);
    };

    // ---- forward pass (traces only when the residual is formed here)
    void *tr = given_residual ? nullptr : P->traces.p;
    bool merge = false, done = false;
    if (nt >= END_LEAST_STEPS && (rc = step_end_check(g, sh->nsrc, sh->src_idx, nrec, sh->rec_idx, (EndWork *)P->end.p,
                                                      &merge, s)))
        return rc;
    const EndWork *end = merge ? (const EndWork *)P->end.p : nullptr;
    if ((rc = zero(g, loc(-1), s)) || (rc = zero(g, loc(0), s))) return rc;
    for (int64_t n = 0; n < nt; n++) {
        if (K > 0 && !in_place && n % K == 0 && (rc = save(n / K, loc(n), loc(n - 1)))) return rc;
        // (a 16-bit checkpoint holds the wavefield before its free surface)
        const bool last = n + 1 == nt || (K > 0 && !in_place && (n + 1) % K == 0);
        if ((rc = fwd_step(g, coef, sh, loc(n + 1), loc(n - 1), loc(n), n, tr, es, end, !last, &done, s))) return rc;
    }

    // ---- residual and misfit
    const int nb = (int)std::max<int64_t>(1, std::min<int64_t>((ntr + 255) / 256, 4096));
    rc = dispatch_types(g, [&](auto ts, auto) -> int {
        using TS = decltype(ts);
        hipLaunchKernelGGL(k_residual<TS>, dim3(nb), dim3(256), 0, s, (const TS *)tr, (const TS *)d_obs,
                           (TS *)P->res.p, ntr, (double *)P->partial.p);
        HSX_LAUNCHED("k_residual");
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(64), 0, s, (const double *)P->partial.p, nb,
                           (double *)P->msum.p);
        HSX_LAUNCHED("k_sum_partials");
        return HSX_OK;
    });
    if (rc) return rc;
    if (nrec > 0 && (rc = hsx_gather(g, coef, nrec, sh->rec_idx, P->crec.p, s))) return rc;

    // ---- backward pass: mu^k for k = nt .. 1
    if ((rc = zero(g, P->m1.p, s)) || (rc = zero(g, P->m2.p, s))) return rc;
    void *mu1 = P->m1.p, *mu2 = P->m2.p;   // mu^{k+1}, mu^{k+2}
    // the imaging condition fused into the adjoint step's kernel where the
    // tiled kernels take the grid (exact arithmetic only), else its own pass
    const bool fuse_img = kernel_family() != HSX_KERNEL_REF && !contract_mode() && step_tiled(g);
    // the residual of step k - 1 goes into mu^{k+1}: for k = nt here, for the
    // others in the launch that ends reverse step k
    auto res_at = [&](int64_t k) { return P->res.c() + (size_t)(k - 1) * nrec * es; };
    if (nrec > 0 &&
        (rc = hsx_inject(g, mu2, nrec, sh->rec_idx, res_at(nt), P->crec.p, -1.0, HSX_INJECT_ADD, s)))
        return rc;
    // The imaging condition of two steps goes into the gradient together, in the
    // kernel of the second one (whose input is the first one's output): the
    // gradient, 16 bytes of traffic a point, moves half as often and two of six
    // wavefields less are read.  200^3 FP32 order 8, 100 steps, 16-bit checkpoints
    // every 20: 16.7 -> 14.1 ms, the imaging step 69 us every second time (a
    // plain step 28.7).  hold: the first of a pair, imaged with the next step;
    // q_up: its latest wavefield, in the second one.
    const bool pairs = sh->nsrc <= PAIR_SRC_MAX;
    bool bc_done = false;          // mu1's free surface went with the end of the step before
    auto back_step = [&](int64_t k, bool hold, const void *q_up, const void *qk, const void *qk1,
                         const void *qk2) -> int {
        // mu^k = 2 mu^{k+1} - (mu^{k+2} - c e^k) + c L mu^{k+1}: the residual
        // went into mu^{k+2} (mu2) before the step, so that the step's output is
        // mu^k complete and the imaging condition can be taken from it
        int r = bc_done ? HSX_OK : hsx_free_surface(g, mu1, 0x3F, s);
        bc_done = false;
        if (!r) {
            r = fuse_img && !hold ? tiled_ac2_step_img(g, mu2, mu1, coef, grad, qk, qk1, qk2, q_up, rim, img_scale, s)
                                  : HSX_ERR_UNSUPPORTED;
            if (r == HSX_ERR_UNSUPPORTED) {
                r = hsx_ac2_step(g, mu2, mu1, coef, s);                   // mu2 <- mu^k
                if (!r && !hold)
                    r = q_up ? imaging_pair(g, grad, mu1, mu2, q_up, qk, qk1, qk2, rimb, img_scale, s)
                             : hsx_imaging(g, grad, mu2, qk, qk1, qk2, rim, img_scale, -1, 0.0, s);
            }
        }
        // the source term of step k (reads mu^k in mu2) and the residual of
        // step k - 1 into mu^{k+1} (mu1): one launch
        const int64_t ns = sh->nsrc, nr = k >= 2 ? nrec : 0;
        if (!r && (ns > 0 || nr > 0)) {
            r = dispatch_types(g, [&](auto ts, auto) -> int {
                using TS = decltype(ts);
                const ReverseEnd<TS> e = {
                    grad, (const TS *)mu2, (const TS *)qk, (const TS *)qk1, (const TS *)qk2,
                    hold || q_up ? (double *)P->side.p : (double *)nullptr, (int)hold, ns, sh->src_idx,
                    ns > 0 ? (const TS *)((const char *)sh->wavelet + (size_t)(k - 1) * ns * es) : (const TS *)nullptr,
                    img_scale, rimb, g->n1, g->n1 * g->n2, (uint32_t)((ns + 255) / 256),
                    (uint32_t)std::min<int64_t>((nr + 255) / 256, 1024), (TS *)mu1, npoint, nr, sh->rec_idx,
                    nr > 0 ? (const TS *)res_at(k - 1) : (const TS *)nullptr, (const TS *)P->crec.p};
                // with the free surface of mu^k, which the next step reads
                if (k >= 2) {
                    const int r1 = step_end_reverse(g, mu2, e, s);
                    bc_done = r1 == HSX_OK;
                    if (r1 != HSX_ERR_UNSUPPORTED) return r1;
                }
                hipLaunchKernelGGL(k_reverse_end<TS>, dim3(e.nb_src + e.nb_rec), dim3(256), 0, s, e);
                HSX_LAUNCHED("k_reverse_end");
                return HSX_OK;
            });
        }
        std::swap(mu1, mu2);
        return r;
    };
    // reverse steps hi .. lo + 1 with q^m at at(m): pairs, after a single one if
    // their number is odd
    auto reverse = [&](int64_t hi, int64_t lo, auto at) -> int {
        for (int64_t k = hi; k > lo; k--) {
            const bool second = (k - lo) % 2 == 1;
            const int r = back_step(k, pairs && !second, pairs && second && k < hi ? at(k + 1) : nullptr, at(k),
                                    at(k - 1), at(k - 2));
            if (r) return r;
        }
        return HSX_OK;
    };
    if ((rc = reverse(nt, n_last, loc))) return rc;
    for (int64_t seg = in_place ? nseg - 2 : nseg - 1; seg >= 0; seg--) {
        const int64_t n0 = seg * K, n1 = std::min<int64_t>(n0 + K, nt);
        // q^m of this segment; of the storage-type checkpoints the segment's own
        // and the next one's serve as they lie, which leaves K - 2 steps to redo
        auto at = [&](int64_t m) -> void * {
            if (in_place && m <= n0) return ck_at(seg, m == n0 ? 0 : 1);
            if (in_place && m >= n1 - 1) return loc(m);
            return q[m - n0 + 1].p;
        };
        if (!in_place && (rc = restore(seg, at(n0), at(n0 - 1)))) return rc;
        const int64_t ne = in_place ? n1 - 2 : n1;
        done = false;
        for (int64_t n = n0; n < ne; n++)
            if ((rc = fwd_step(g, coef, sh, at(n + 1), at(n - 1), at(n), n, nullptr, es, end, n + 1 < ne, &done, s)))
                return rc;
        if ((rc = reverse(n1, n0, at))) return rc;
    }
    double m = 0.0;
    HSX_HIP(hipMemcpyAsync(&m, P->msum.p, sizeof(double), hipMemcpyDeviceToHost, s));
    HSX_HIP(hipStreamSynchronize(s));
    if (misfit) *misfit = 0.5 * m;
    return HSX_OK;
}

} // namespace hsx

using namespace hsx;

extern "C" {

int hsx_forward(const hsx_grid *g, const void *coef, const hsx_shot *sh, void *traces, void *stream)
{
    int rc = shot_checks(g, coef, sh);
    if (rc) return rc;
    if ((rc = check_ptr(traces, "traces"))) return rc;
    const size_t es = g->storage == HSX_FP64 ? 8 : 4;
    const size_t bytes = (size_t)(g->n1 * g->n2 * g->n3) * es;
    hipStream_t s = stream_of(stream);
    // both wavefields and the step ends' workspace
    const size_t each = (bytes + 255) / 256 * 256;
    struct Work {
        WorkBuf b;
        bool idle = false;
        ~Work() { work_give(b, idle); }
    } buf;
    if ((rc = work_take(2 * each + sizeof(EndWork), &buf.b))) return rc;
    void *prev = buf.b.p, *cur = (char *)prev + each;
    EndWork *work = (EndWork *)((char *)cur + each);
    bool merge = false, done = false;
    if (sh->nt >= END_LEAST_STEPS &&
        (rc = step_end_check(g, sh->nsrc, sh->src_idx, sh->nrec, sh->rec_idx, work, &merge, s)))
        return rc;
    const EndWork *end = merge ? work : nullptr;
    if ((rc = zero(g, prev, s)) || (rc = zero(g, cur, s))) return rc;
    for (int64_t n = 0; n < sh->nt; n++) {
        if ((rc = fwd_step(g, coef, sh, prev, prev, cur, n, traces, es, end, n + 1 < sh->nt, &done, s))) return rc;
        std::swap(prev, cur);
    }
    HSX_HIP(hipStreamSynchronize(s));   // the buffer may serve another call after the return
    buf.idle = true;
    return HSX_OK;
}

int hsx_adjoint_plan_create(const hsx_grid *g, int64_t nt, int64_t nrec, const hsx_adjoint_opts *opt,
                            hsx_adjoint_plan **out)
{
    if (!out) return fail(HSX_ERR_INVALID, "null plan pointer");
    *out = nullptr;
    int rc = plan_checks(g, nt, nrec, opt);
    if (rc) return rc;
    if ((opt->flags & HSX_ADJ_AUTOTUNE) && g->dim == 3 && (rc = hsx_autotune(g, 5, nullptr, nullptr))) return rc;
    hsx_adjoint_plan *P = new hsx_adjoint_plan();
    P->g = *g;
    P->nt = nt;
    P->nrec = nrec;
    P->opt = *opt;
    P->es = g->storage == HSX_FP64 ? 8 : 4;
    const int64_t npoint = g->n1 * g->n2 * g->n3;
    P->bytes = (size_t)npoint * P->es;
    // storage-type checkpoints of every step are full storage (the same values)
    if (opt->ckpt_every == 1 && opt->ckpt_format == HSX_CKPT_FP32) P->opt.ckpt_every = 0;
    const int64_t K = P->opt.ckpt_every;
    const int64_t ntr = nt * nrec;
    P->nseg = K == 0 ? 0 : (nt + K - 1) / K;
    P->snap = opt->ckpt_format == HSX_CKPT_FP32 ? (P->bytes + 255) / 256 * 256 : hsx_ckpt_bytes(npoint);
    auto bail = [&](int code) {
        delete P;
        return code;
    };
    if ((rc = P->traces.alloc(ntr * P->es)) || (rc = P->res.alloc(ntr * P->es)) || (rc = P->crec.alloc(nrec * P->es)) ||
        (rc = P->partial.alloc(4096 * sizeof(double))) || (rc = P->msum.alloc(sizeof(double))) ||
        (rc = P->side.alloc(PAIR_SRC_MAX * sizeof(double))) || (rc = P->end.alloc(sizeof(EndWork))) ||
        (rc = P->m1.alloc(P->bytes)) || (rc = P->m2.alloc(P->bytes)))
        return bail(rc);
    P->q.resize((K == 0 ? nt : std::min(K, nt)) + 2);
    for (auto &x : P->q)
        if ((rc = x.alloc(P->bytes))) return bail(rc);
    const int64_t ncks = opt->ckpt_format == HSX_CKPT_FP32 ? P->nseg - 1 : P->nseg;     // the last one: plan_run
    if (ncks > 0 && ((rc = P->ck.alloc((size_t)ncks * 2 * P->snap)) || (rc = P->fa.alloc(P->bytes)) ||
                     (rc = P->fb.alloc(P->bytes))))
        return bail(rc);
    *out = P;
    return HSX_OK;
}

int hsx_adjoint_plan_destroy(hsx_adjoint_plan *P)
{
    if (!P) return HSX_OK;
    (void)hipDeviceSynchronize();   // no kernel of a gradient may still use the buffers
    delete P;
    return HSX_OK;
}

int hsx_gradient_plan(hsx_adjoint_plan *P, const hsx_grid *g, const void *coef, const hsx_shot *sh, const void *d_obs,
                      double *grad, double *misfit, void *stream)
{
    if (!P) return fail(HSX_ERR_INVALID, "null plan");
    int rc = shot_checks(g, coef, sh);
    if (rc) return rc;
    if ((rc = check_ptr(d_obs, "d_obs")) || (rc = check_ptr(grad, "grad"))) return rc;
    if (!same_layout(*g, P->g)) return fail(HSX_ERR_INVALID, "gradient: grid layout differs from the plan's");
    if (sh->nt != P->nt || sh->nrec != P->nrec)
        return fail(HSX_ERR_INVALID, "gradient: nt / receiver count %lld / %lld, plan %lld / %lld", (long long)sh->nt,
                    (long long)sh->nrec, (long long)P->nt, (long long)P->nrec);
    return plan_run(P, g, coef, sh, d_obs, grad, misfit, stream_of(stream));
}

int hsx_gradient(const hsx_grid *g, const void *coef, const hsx_shot *sh, const void *d_obs,
                 const hsx_adjoint_opts *opt, double *grad, double *misfit, void *stream)
{
    int rc = shot_checks(g, coef, sh);
    if (rc) return rc;
    if ((rc = check_ptr(d_obs, "d_obs")) || (rc = check_ptr(grad, "grad")) || (rc = check_ptr(opt, "opts")))
        return rc;
    hsx_adjoint_plan *P = nullptr;
    if ((rc = hsx_adjoint_plan_create(g, sh->nt, sh->nrec, opt, &P))) return rc;
    rc = plan_run(P, g, coef, sh, d_obs, grad, misfit, stream_of(stream));
    hsx_adjoint_plan_destroy(P);   // plan_run has synchronised the stream (or failed)
    return rc;
}

} // extern "C"
