// Optimiser steps on the device: the L-BFGS two-loop recursion (lbfgs.c),
// its first-iteration gradient save (lbfgs_save.c) and the conjugate-gradient
// direction (conjugategrad.c).  Vector updates are FP32 elementwise in the
// reference's expression order; every dot product is reduced in FP64 (the
// reference sums in FP32 and all-reduces MPI_FLOAT) over a fixed grid of
// partial sums, so a call's result does not depend on scheduling.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>
#include "ifos_dev.h"

namespace ifos {

constexpr int kRedBlocks = 1024;  // partial sums per dot product
constexpr int kRedThreads = 256;  // 4 wavefronts

// block-wide FP64 sum of one value per thread (fixed tree order); t: the
// thread's index in the block
__device__ inline double block_sum(double v, double *sh, int t)
{
    sh[t] = v;
    __syncthreads();
    for (int s = kRedThreads / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    const double r = sh[0];
    __syncthreads();
    return r;
}

// Cells are walked a row (j, i) of the grid per wavefront, 64 k at a time: no
// index divisions, and a row of 276 cells fills 86 % of the lanes (256
// threads side by side along k: 54 %).
struct Rows {
    int64_t r, step, n;
};
__device__ inline Rows wave_rows(const DevGeom &g)
{
    const int y = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    return Rows{(int64_t)blockIdx.x * blockDim.y + y, (int64_t)gridDim.x * blockDim.y, (int64_t)g.nx * g.ny};
}
__device__ inline int64_t row_at(const DevGeom &g, int64_t r)
{
    const int j = (int)(r / g.nx) + 1, i = (int)(r % g.nx) + 1;
    return at(g, j, i, 1);
}

// ---- L-BFGS on compact vectors: [numpar][NY][NX][NZ], cell l = ((j-1)*NX +
// i-1)*NZ + k-1.  The two-loop recursion is a chain of passes over q, each
// pass applying the update of one pair and forming the dot product that the
// next needs, with the coefficients in device memory: 9 r + 1 vectors moved
// for r pairs instead of 10 r + 12, and no host round trip inside.
// The scalars of an update: state[0] y.s, [1] y.y, [2] the last dot product,
// [3] h0, [4 + w] alpha of slot w, [4 + bfgsnum + w] scale of slot w
// (bfgsscale, 1 / y.s)
struct Pack {
    float *g1, *g2;  // device-layout gradients (g2 used when numpar == 2)
    int numpar;
    int64_t n1;      // NX*NY*NZ
};

// lbfgs_save.c:31-53: y = grad
__global__ __launch_bounds__(kRedThreads) void k_lb_save(DevGeom g, Pack P, float *y)
{
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c = row_at(g, R.r), l = R.r * g.nz;
        for (int q = 0; q < P.numpar; ++q)
            for (int k = threadIdx.x; k < g.nz; k += 64) y[q * P.n1 + l + k] = +(q ? P.g2 : P.g1)[c + k];
    }
}

// lbfgs.c:45-71: y += -grad, q = grad, and the sums y.s, y.y (:74-88) and s.q
// (the first of the recursion, :94-116, whose newest pair this is)
__global__ __launch_bounds__(kRedThreads) void k_lb_first(DevGeom g, Pack P, float *q, float *y, const float *s,
                                                          double *part)
{
    __shared__ double sh[kRedThreads];
    double d[3] = {0.0, 0.0, 0.0};
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c = row_at(g, R.r), l = R.r * g.nz;
        for (int m = 0; m < P.numpar; ++m)
            for (int k = threadIdx.x; k < g.nz; k += 64) {
                const int64_t o = m * P.n1 + l + k;
                const float v = (m ? P.g2 : P.g1)[c + k], sv = s[o];
                const float yv = y[o] + -v;
                y[o] = yv;
                q[o] = v;
                d[0] += (double)yv * (double)sv;
                d[1] += (double)yv * (double)yv;
                d[2] += (double)sv * (double)v;
            }
    }
    const int t = (int)(threadIdx.y * 64 + threadIdx.x);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const double x = block_sum(d[m], sh, t);
        if (t == 0) part[3 * blockIdx.x + m] = x;
    }
}

// one pass of the recursion over the compact vectors, V floats at a time:
// q += a x (lbfgs.c:115: x = y_w, a = -alpha_w; :149: x = s_w, a = alpha_w -
// beta_w), q *= h0 where SCALE (:120-124), and the partial sums of z.q
template <int V, bool SCALE>
__global__ __launch_bounds__(kRedThreads) void k_lb_pass(float *q, const float *x, const float *z, int64_t n,
                                                         const double *state, int ia, int is, int up, double *part)
{
    typedef float vec __attribute__((ext_vector_type(V)));
    __shared__ double sh[kRedThreads];
    // the dot product this pass's coefficient comes from is state[2]: alpha =
    // scale * (s.q) on the way down, beta = scale * (y.q) on the way up
    const double co = state[is] * state[2];
    const float a = up ? (float)(state[ia] - co) : (float)(-co);
    const float h0 = SCALE ? (float)state[3] : 0.0f;
    double s = 0.0;
    const int64_t nv = n / V, step = (int64_t)gridDim.x * kRedThreads;
    for (int64_t l = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; l < nv; l += step) {
        vec qv = ((const vec *)q)[l];
        const vec xv = ((const vec *)x)[l], zv = ((const vec *)z)[l];
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float w = qv[e] + (a * xv[e]);
            if (SCALE) w = w * h0;
            qv[e] = w;
            s += (double)zv[e] * (double)w;
        }
        ((vec *)q)[l] = qv;
    }
    s = block_sum(s, sh, threadIdx.x);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// lbfgs.c:149 for the newest pair, then :157-178: bfgsgrad[w] = grad, grad = q
__global__ __launch_bounds__(kRedThreads) void k_lb_last(DevGeom g, Pack P, const float *q, const float *s, float *y,
                                                         const double *state, int ia, int is)
{
    const float a = (float)(state[ia] - state[is] * state[2]);
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c = row_at(g, R.r), l = R.r * g.nz;
        for (int m = 0; m < P.numpar; ++m)
            for (int k = threadIdx.x; k < g.nz; k += 64) {
                const int64_t o = m * P.n1 + l + k;
                float *G = m ? P.g2 : P.g1;
                y[o] = G[c + k];
                G[c + k] = q[o] + (s[o] * a);
            }
    }
}

// out[m] = sum over blocks of part[b*nd + m], m < nd (one workgroup)
__global__ __launch_bounds__(kRedThreads) void k_red_final(const double *part, int nblk, int nd, double *out)
{
    __shared__ double sh[kRedThreads];
    for (int m = 0; m < nd; ++m) {
        double s = 0.0;
        for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += part[b * nd + m];
        s = block_sum(s, sh, threadIdx.x);
        if (threadIdx.x == 0) out[m] = s;
    }
}

// after the first pass: the scalars of the new pair (lbfgs.c:74-88); ia >= 0
// (down the recursion): alpha of the slot whose dot product just arrived
__global__ void k_lb_scalars(double *state, int first, int ia, int is)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (first) {
        state[is] = 1.0 / state[0];
        state[3] = state[0] / state[1];
    }
    if (ia >= 0) state[ia] = state[is] * state[2];
}

// ---- conjugategrad.c on the device-layout fields
struct CgArgs {
    float *g[3], *p[6];
};

// conjugategrad.c:42-54 (cdf == 1): all six priors = grad
__global__ __launch_bounds__(kRedThreads) void k_cg_copy(DevGeom g, CgArgs A)
{
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c0 = row_at(g, R.r);
        for (int k = threadIdx.x; k < g.nz; k += 64) {
            const int64_t c = c0 + k;
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                const float v = A.g[n][c];
                A.p[n][c] = v;
                A.p[n + 3][c] = v;
            }
        }
    }
}

// conjugategrad.c:58-73: the six sums of the beta ratios, and prior1..3 = grad
__global__ __launch_bounds__(kRedThreads) void k_cg_dots(DevGeom g, CgArgs A, double *part)
{
    __shared__ double sh[kRedThreads];
    double s[6] = {0, 0, 0, 0, 0, 0};
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c0 = row_at(g, R.r);
        for (int k = threadIdx.x; k < g.nz; k += 64) {
            const int64_t c = c0 + k;
            float gv[3], pv[3];
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                gv[n] = A.g[n][c];
                pv[n] = A.p[n][c];
            }
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                s[2 * n] += (double)gv[n] * (double)(gv[n] - pv[n]);
                s[2 * n + 1] += (double)pv[n] * (double)pv[n];
                A.p[n][c] = gv[n];
            }
        }
    }
    const int t = (int)(threadIdx.y * 64 + threadIdx.x);
#pragma unroll
    for (int m = 0; m < 6; ++m) {
        const double x = block_sum(s[m], sh, t);
        if (t == 0) part[6 * blockIdx.x + m] = x;
    }
}

// conjugategrad.c:93-106: grad = prior4..6 * beta + grad; prior4..6 = grad
__global__ __launch_bounds__(kRedThreads) void k_cg_update(DevGeom g, CgArgs A, float b0, float b1, float b2)
{
    const float b[3] = {b0, b1, b2};
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c0 = row_at(g, R.r);
        for (int k = threadIdx.x; k < g.nz; k += 64) {
            const int64_t c = c0 + k;
            float v[3];
#pragma unroll
            for (int n = 0; n < 3; ++n) v[n] = (A.p[n + 3][c] * b[n]) + A.g[n][c];
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                A.g[n][c] = v[n];
                A.p[n + 3][c] = v[n];
            }
        }
    }
}

// workgroups of a row-walking kernel without partial sums
static unsigned row_grid(const ifos_geom *g)
{
    const int64_t b = ((int64_t)g->nx * g->ny + 3) / 4;
    return (unsigned)(b < 8192 ? b : 8192);
}

}  // namespace ifos

using namespace ifos;

struct ifos_lbfgs {
    ifos_geom g;
    DevGeom G;
    int numpar, bfgsnum;
    int64_t n1, n;            // cells, numpar * cells
    float *grad = nullptr;    // bfgsgrad [bfgsnum][n] (slot w at w-1)
    float *mod = nullptr;     // bfgsmod  [bfgsnum][n]
    float *q = nullptr;       // [n]
    double *part = nullptr;   // [kRedBlocks * 3]
    double *state = nullptr;  // [4 + 2 * bfgsnum] scalars of an update
    std::vector<double> scale;  // bfgsscale[1..bfgsnum] (index w-1), as state holds it
};

static int lb_slot(const ifos_lbfgs *b, int v)
{
    int w = v % b->bfgsnum;
    if (w == 0) w = b->bfgsnum;
    return w - 1;
}

extern "C" int ifos_lbfgs_create(const ifos_geom *g, int numpar, int bfgsnum, ifos_lbfgs **out)
{
    if (!g || !out || (numpar != 1 && numpar != 2) || bfgsnum < 1) {
        set_error("ifos_lbfgs_create: numpar must be 1 or 2 and bfgsnum >= 1");
        return IFOS_EINVAL;
    }
    *out = nullptr;
    ifos_lbfgs *b = new ifos_lbfgs;
    b->g = *g;
    b->G = make_dev_geom(g);
    b->numpar = numpar;
    b->bfgsnum = bfgsnum;
    b->n1 = (int64_t)g->nx * g->ny * g->nz;
    b->n = b->n1 * numpar;
    b->scale.assign(bfgsnum, 0.0);
    const size_t vb = (size_t)b->n * sizeof(float);
    int rc = hip_check(hipMalloc(&b->grad, vb * bfgsnum), "lbfgs grad");
    if (!rc) rc = hip_check(hipMalloc(&b->mod, vb * bfgsnum), "lbfgs mod");
    if (!rc) rc = hip_check(hipMalloc(&b->q, vb), "lbfgs q");
    const size_t sb = (4 + 2 * (size_t)bfgsnum) * sizeof(double);
    if (!rc) rc = hip_check(hipMalloc(&b->part, kRedBlocks * 3 * sizeof(double)), "lbfgs partials");
    if (!rc) rc = hip_check(hipMalloc(&b->state, sb), "lbfgs scalars");
    if (!rc) rc = zero_new(b->state, sb);
    // ifos3d.c:373-379: fmatrix / vector zero-fill
    if (!rc) rc = zero_new(b->grad, vb * bfgsnum);
    if (!rc) rc = zero_new(b->mod, vb * bfgsnum);
    if (!rc) rc = zero_wait();
    if (rc) {
        ifos_lbfgs_destroy(b);
        return rc;
    }
    *out = b;
    return IFOS_OK;
}

extern "C" void ifos_lbfgs_destroy(ifos_lbfgs *b)
{
    if (!b) return;
    (void)hipFree(b->grad);
    (void)hipFree(b->mod);
    (void)hipFree(b->q);
    (void)hipFree(b->part);
    (void)hipFree(b->state);
    delete b;
}

extern "C" float *ifos_lbfgs_mod(ifos_lbfgs *b, int w)
{
    if (!b || w < 1 || w > b->bfgsnum) return nullptr;
    return b->mod + (size_t)(w - 1) * b->n;
}

extern "C" float *ifos_lbfgs_grad(ifos_lbfgs *b, int w)
{
    if (!b || w < 1 || w > b->bfgsnum) return nullptr;
    return b->grad + (size_t)(w - 1) * b->n;
}

extern "C" int ifos_lbfgs_scale(const ifos_lbfgs *b, double *scale)
{
    if (!b || !scale) return IFOS_EINVAL;
    for (int w = 0; w < b->bfgsnum; ++w) scale[w] = b->scale[w];
    return IFOS_OK;
}

extern "C" int ifos_lbfgs_savegrad(ifos_lbfgs *b, const float *d_grad1, const float *d_grad2)
{
    if (!b || !d_grad1 || (b->numpar == 2 && !d_grad2)) return IFOS_EINVAL;
    const Pack P = {const_cast<float *>(d_grad1), const_cast<float *>(d_grad2), b->numpar, b->n1};
    hipLaunchKernelGGL(k_lb_save, dim3(row_grid(&b->g)), dim3(64, 4), 0, 0, b->G, P, b->grad);
    int rc = hip_check(hipGetLastError(), "k_lb_save");
    if (!rc) rc = hip_check(hipStreamSynchronize(0), "lbfgs_savegrad");
    return rc;
}

extern "C" int ifos_lbfgs_update(ifos_lbfgs *b, float *d_grad1, float *d_grad2, int iteration, double *h0_out)
{
    if (!b || !d_grad1 || (b->numpar == 2 && !d_grad2) || iteration < 2) {
        set_error("ifos_lbfgs_update: iteration must be >= 2 (iteration 1 saves the gradient)");
        return IFOS_EINVAL;
    }
    const int64_t n = b->n;
    const int M = b->bfgsnum;
    int m = iteration - M;
    if (m < 1) m = 1;
    double *st = b->state;
    auto grad = [&](int w) { return b->grad + (size_t)w * n; };
    auto mod = [&](int w) { return b->mod + (size_t)w * n; };
    auto red = [&](int nd, double *out) {
        hipLaunchKernelGGL(k_red_final, dim3(1), dim3(kRedThreads), 0, 0, b->part, kRedBlocks, nd, out);
    };
    auto scalars = [&](int first, int w) {
        hipLaunchKernelGGL(k_lb_scalars, dim3(1), dim3(64), 0, 0, st, first, w >= 0 ? 4 + w : -1, 4 + M + (w >= 0 ? w : 0));
    };
    // q += (up: alpha_w - beta_w, else -alpha_w) x, (* h0), then state[2] = z.q
    auto pass = [&](bool up, bool scale, int w, const float *x, const float *z) {
        // 16-byte vectors where every slot starts on such a boundary
        auto go = [&](auto v, auto sc) {
            hipLaunchKernelGGL((k_lb_pass<decltype(v)::value, decltype(sc)::value>), dim3(kRedBlocks),
                               dim3(kRedThreads), 0, 0, b->q, x, z, n, st, 4 + w, 4 + M + w, up ? 1 : 0, b->part);
        };
        if (n % 4 == 0 && scale) go(std::integral_constant<int, 4>{}, std::true_type{});
        else if (n % 4 == 0) go(std::integral_constant<int, 4>{}, std::false_type{});
        else if (scale) go(std::integral_constant<int, 1>{}, std::true_type{});
        else go(std::integral_constant<int, 1>{}, std::false_type{});
        red(1, st + 2);
    };
    // lbfgs.c:45-88: y_w = g_prev - g, q = g, rho_w = 1 / (y.s), h0 = (y.s) /
    // (y.y), and s_w.q
    const int wn = lb_slot(b, iteration - 1);
    const Pack P = {d_grad1, d_grad2, b->numpar, b->n1};
    hipLaunchKernelGGL(k_lb_first, dim3(kRedBlocks), dim3(64, 4), 0, 0, b->G, P, b->q, grad(wn), mod(wn), b->part);
    red(3, st);
    scalars(1, wn);
    // lbfgs.c:94-116: newest to oldest, alpha_w = rho_w s_w.q, q -= alpha_w y_w;
    // the oldest also multiplies by h0 (:120-124) and starts the way back
    for (int v = iteration - 1; v >= m; --v) {
        const int w = lb_slot(b, v);
        if (v > m) {
            pass(false, false, w, grad(w), mod(lb_slot(b, v - 1)));
            scalars(0, lb_slot(b, v - 1));
        } else {
            pass(false, true, w, grad(w), grad(w));
        }
    }
    // lbfgs.c:136-151: oldest to newest, beta = rho_w y_w.q, q += s_w (alpha_w - beta)
    for (int v = m; v < iteration - 1; ++v) {
        const int w = lb_slot(b, v);
        pass(true, false, w, mod(w), grad(lb_slot(b, v + 1)));
    }
    // the newest pair, and lbfgs.c:154-178: save this gradient in slot
    // iteration, grad = q
    hipLaunchKernelGGL(k_lb_last, dim3(row_grid(&b->g)), dim3(64, 4), 0, 0, b->G, P, b->q, mod(wn),
                       grad(lb_slot(b, iteration)), st, 4 + wn, 4 + M + wn);
    int rc = hip_check(hipGetLastError(), "ifos_lbfgs_update");
    std::vector<double> h(4 + 2 * (size_t)M);
    if (!rc) rc = hip_check(hipMemcpy(h.data(), st, h.size() * sizeof(double), hipMemcpyDeviceToHost), "lbfgs scalars");
    if (rc) return rc;
    b->scale[wn] = h[4 + M + wn];
    if (h0_out) *h0_out = h[3];
    return rc;
}

// conjugate's FP64 partial sums: allocated once per device on first use and
// kept for the life of the process (calls on one device share them; the
// optimiser's calls are serialised on the null stream)
static int cg_buffers(double **part, double **out)
{
    static double *s_part[64] = {}, *s_out[64] = {};
    int dev = 0;
    int rc = hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    if (dev < 0 || dev >= 64) {
        set_error("ifos_conjugate: device %d out of range", dev);
        return IFOS_EINVAL;
    }
    if (!s_part[dev]) {
        rc = hip_check(hipMalloc(&s_part[dev], kRedBlocks * 6 * sizeof(double)), "conjugate partials");
        if (!rc) rc = hip_check(hipMalloc(&s_out[dev], 6 * sizeof(double)), "conjugate sums");
        if (rc) {
            if (s_part[dev]) (void)hipFree(s_part[dev]);
            s_part[dev] = nullptr;
            s_out[dev] = nullptr;
            return rc;
        }
    }
    *part = s_part[dev];
    *out = s_out[dev];
    return IFOS_OK;
}

extern "C" int ifos_conjugate(const ifos_geom *g, float *const d_grad[3], float *const d_prior[6], float beta[3],
                              int cdf, double *sums)
{
    if (!g || !d_grad || !d_prior || !beta) return IFOS_EINVAL;
    const DevGeom G = make_dev_geom(g);
    CgArgs A;
    for (int n = 0; n < 3; ++n) A.g[n] = d_grad[n];
    for (int n = 0; n < 6; ++n) A.p[n] = d_prior[n];
    const unsigned gr = row_grid(g);
    beta[0] = beta[1] = beta[2] = 0.0f;  // conjugategrad.c:37
    if (cdf == 1) {
        hipLaunchKernelGGL(k_cg_copy, dim3(gr), dim3(64, 4), 0, 0, G, A);
        int rc = hip_check(hipGetLastError(), "k_cg_copy");
        if (!rc) rc = hip_check(hipStreamSynchronize(0), "ifos_conjugate");
        return rc;
    }
    double *part = nullptr, *out = nullptr;
    int rc = cg_buffers(&part, &out);
    double s[6] = {0, 0, 0, 0, 0, 0};
    if (!rc) {
        hipLaunchKernelGGL(k_cg_dots, dim3(kRedBlocks), dim3(64, 4), 0, 0, G, A, part);
        hipLaunchKernelGGL(k_red_final, dim3(1), dim3(kRedThreads), 0, 0, part, kRedBlocks, 6, out);
        rc = hip_check(hipGetLastError(), "k_cg_dots");
    }
    if (!rc) rc = hip_check(hipMemcpy(s, out, sizeof(s), hipMemcpyDeviceToHost), "conjugate sums copy");
    if (rc) return rc;
    if (sums)
        for (int m = 0; m < 6; ++m) sums[m] = s[m];
    // conjugategrad.c:78-90, clamps as written there: only beta[0] ends in
    // [0, 0.5] (the later tests read the already-clamped beta[0])
    if (cdf == 0) {
        if (std::fabs(s[1]) > 0.0) beta[0] = (float)(s[0] / s[1]);
        if (std::fabs(s[3]) > 0.0) beta[1] = (float)(s[2] / s[3]);
        if (std::fabs(s[5]) > 0.0) beta[2] = (float)(s[4] / s[5]);
    }
    if (beta[0] < 0) beta[0] = 0.0f;
    if (beta[0] < 0) beta[1] = 0.0f;
    if (beta[0] < 0) beta[2] = 0.0f;
    if (beta[0] > 0.5f) beta[0] = 0.5f;
    if (beta[0] > 0.5f) beta[1] = 0.5f;
    if (beta[0] > 0.5f) beta[2] = 0.5f;
    hipLaunchKernelGGL(k_cg_update, dim3(gr), dim3(64, 4), 0, 0, G, A, beta[0], beta[1], beta[2]);
    rc = hip_check(hipGetLastError(), "k_cg_update");
    if (!rc) rc = hip_check(hipStreamSynchronize(0), "ifos_conjugate");
    return rc;
}

// ---------------------------------------------------------------------------
// precongrad.c:28-336, modelupdate.c:26-160 and steplength.c:26-91.

namespace ifos {

// The source and receiver tapers are functions of the squared distance, an
// integer, and exactly 1 from kSrcD (r = 64: 1000 exp(-44.8) = 4e-17, so the
// double quotient is 1) and kRecD (r^2 = 64, the same exponent) on; rounded to
// float, as the tables hold them, they are 1 from 1199 and 35 on already.  The
// edge tapers are functions of one index each.  They are formed once per call in
// tables, and a cell multiplies only the factors of the points near its row.
constexpr int kSrcD = 4096, kRecD = 64;
struct PreconArgs {
    float *g[3];
    const int *src;  // [nsrc][3] grid x, y, z of the sources (iround(srcpos / D))
    const int *rec;  // [ntr][3] grid x, y, z of the receivers
    float *tsrc, *trec;  // [kSrcD], [kRecD] by squared distance
    float *ex, *ey, *ez; // [nx][2], [ny][2], [nz][2] by local index - 1
    int nsrc, ntr, damptype, free_surf, sh, rh;
    int nxg, nyg, nzg, posx, posy, posz;
};

// 1 / (1 + c * exp(e)) in double, stored to float as the reference does
__device__ inline float taper(double c, double e)
{
    return (float)(1.0 / (1.0 + c * exp(e)));
}

// global index of local index l: set only by the DAMPTYPE 1 and 2 loops
// (precongrad.c:45-47, :131-133); 0 elsewhere, as written there
__device__ inline int precon_index(const PreconArgs &A, int l, int pos, int n)
{
    return A.damptype == 1 || A.damptype == 2 ? l + pos * n : 0;
}

__global__ __launch_bounds__(256) void k_precon_tables(DevGeom g, PreconArgs A)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < kSrcD) {  // precongrad.c:135-150
        const float rr = (float)sqrt((double)t);
        A.tsrc[t] = taper(1000.0, -0.7 * (double)rr);
        return;
    }
    t -= kSrcD;
    if (t < kRecD) {  // precongrad.c:49-64, :152-166
        const float rr = (float)sqrt((double)t);
        A.trec[t] = taper(1000.0, -0.7 * (double)rr * (double)rr);
        return;
    }
    t -= kRecD;
    if (t < g.nx) {
        const int ii = precon_index(A, t + 1, A.posx, g.nx);
        A.ex[2 * t] = taper(2000.0, -0.6 * (double)(float)(ii * 1.0));
        A.ex[2 * t + 1] = taper(2000.0, -0.6 * (double)(float)((A.nxg - ii) * 1.0));
        return;
    }
    t -= g.nx;
    if (t < g.nz) {
        const int kk = precon_index(A, t + 1, A.posz, g.nz);
        A.ez[2 * t] = taper(2000.0, -0.6 * (double)(float)(kk * 1.0));
        A.ez[2 * t + 1] = taper(2000.0, -0.6 * (double)(float)((A.nzg - kk) * 1.0));
        return;
    }
    t -= g.nz;
    if (t >= g.ny) return;
    const int jj = precon_index(A, t + 1, A.posy, g.ny);
    float G0, G1;
    if (A.damptype != 3) {  // precongrad.c:65-113, :167-214, :283-330
        G0 = A.free_surf ? 0.0f : taper(2000.0, -0.6 * (double)(float)(jj * 1.0));
        G1 = taper(2000.0, -0.6 * (double)(float)((A.nyg - jj) * 1.0));
    } else {  // precongrad.c:222-236 (the x and z tests r < 0 never hold: ii, kk >= 0)
        float rr = (float)((jj - A.sh) * 1.0);
        G0 = rr < 0 ? 0.0f : taper(1000.0, -0.7 * (double)rr * (double)rr);
        rr = (float)((A.nyg - jj - A.rh) * 1.0);
        G1 = rr < 0 ? 0.0f : taper(1000.0, -0.7 * (double)rr);
    }
    A.ey[2 * t] = G0;
    A.ey[2 * t + 1] = G1;
}

// the factors of the points within squared distance D of the wavefront's 64
// cells of row (jj, ii), k0..k0+63, multiplied in the points' order: the lanes
// test 64 points at a time, then the near ones are taken one by one
template <int D>
__device__ inline void precon_points(const int *pts, int n, const float *table, int jj, int ii, int kk, float &a,
                                     float &b, float &d)
{
    const int lane = (int)threadIdx.x;
    const int k0 = __builtin_amdgcn_readfirstlane(kk);
    for (int base = 0; base < n; base += 64) {
        const int q = base + lane;
        int64_t row = D;
        int pz = 0;
        if (q < n) {
            const int64_t dx = ii - pts[3 * q], dy = jj - pts[3 * q + 1];
            pz = pts[3 * q + 2];
            row = dx * dx + dy * dy;
            const int64_t dz = pz < k0 ? (int64_t)k0 - pz : pz > k0 + 63 ? (int64_t)pz - (k0 + 63) : 0;
            if (row < D) row = row + dz * dz < D ? row : D;
        }
        unsigned long long near = __ballot(row < D);
        const int r32 = (int)(row < D ? row : D);
        while (near) {
            const int l = __ffsll(near) - 1;
            near &= near - 1;
            const int dz = kk - __builtin_amdgcn_readlane(pz, l);
            const int64_t r2 = __builtin_amdgcn_readlane(r32, l) + (int64_t)dz * dz;
            const float G = r2 < D ? table[r2] : 1.0f;
            a = a * G;
            b = b * G;
            d = d * G;
        }
    }
}

// one wavefront per 64 cells of a row.  Forming every taper of every point in
// every cell (an FP64 exp each) took 55 ms at 276^3 with 16 sources and 1024
// receivers; with this one an L-BFGS iteration's device work at that size
// (taper, direction, test model) went from 58 to 3.9 ms.
__global__ __launch_bounds__(256) void k_precon(DevGeom g, PreconArgs A)
{
    const int k = blockIdx.x * 64 + (int)threadIdx.x + 1;
    const int i = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (int)threadIdx.y + 1);
    const int j = blockIdx.z + 1;
    if (i > g.nx) return;  // whole wavefront
    const bool act = k <= g.nz;
    const int64_t c = at(g, j, i, act ? k : g.nz);
    float a = A.g[0][c], b = A.g[1][c], d = A.g[2][c];
    const int ii = precon_index(A, i, A.posx, g.nx), jj = precon_index(A, j, A.posy, g.ny),
              kk = precon_index(A, k, A.posz, g.nz);
    if (A.nsrc) precon_points<kSrcD>(A.src, A.nsrc, A.tsrc, jj, ii, kk, a, b, d);
    if (A.ntr) precon_points<kRecD>(A.rec, A.ntr, A.trec, jj, ii, kk, a, b, d);
    if (!act) return;
    const float *e[3] = {A.ey + 2 * (j - 1), A.ex + 2 * (i - 1), A.ez + 2 * (k - 1)};
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const float G0 = e[n][0], G1 = e[n][1];
        a = a * G0 * G1;
        b = b * G0 * G1;
        d = d * G0 * G1;
    }
    A.g[0][c] = a;
    A.g[1][c] = b;
    A.g[2][c] = d;
}

// block maxima of vp, vs, rho (modelupdate.c:59-74) and of |grad| (:86-95)
__global__ __launch_bounds__(kRedThreads) void k_mu_max(DevGeom g, const float *rho, const float *pi, const float *u,
                                                       const float *g1, const float *g2, const float *g3,
                                                       float *part)
{
    __shared__ float sh[6][kRedThreads];
    float m[6] = {0, 0, 0, 0, 0, 0};
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c0 = row_at(g, R.r);
        for (int k = threadIdx.x; k < g.nz; k += 64) {
            const int64_t c = c0 + k;
            const float r = rho[c];
            const float vp = (float)sqrt((double)(pi[c] / r));
            const float vs = (float)sqrt((double)(u[c] / r));
            if (vp > m[0]) m[0] = vp;
            if (vs > m[1]) m[1] = vs;
            if (r > m[2]) m[2] = r;
            if (fabsf(g1[c]) > m[3]) m[3] = fabsf(g1[c]);
            if (fabsf(g2[c]) > m[4]) m[4] = fabsf(g2[c]);
            if (fabsf(g3[c]) > m[5]) m[5] = fabsf(g3[c]);
        }
    }
    const int t = (int)(threadIdx.y * 64 + threadIdx.x);
    for (int q = 0; q < 6; ++q) sh[q][t] = m[q];
    __syncthreads();
    for (int s = kRedThreads / 2; s > 0; s >>= 1) {
        if (t < s)
            for (int q = 0; q < 6; ++q) sh[q][t] = fmaxf(sh[q][t], sh[q][t + s]);
        __syncthreads();
    }
    if (t < 6) part[6 * blockIdx.x + t] = sh[t][0];
}

// the six maxima over the blocks (none below 0): max[0..5]
__global__ __launch_bounds__(kRedThreads) void k_mu_final(const float *part, int nblk, float *max6)
{
    __shared__ float sh[kRedThreads];
    for (int q = 0; q < 6; ++q) {
        float m = 0.0f;
        for (int b = threadIdx.x; b < nblk; b += kRedThreads) m = fmaxf(m, part[6 * b + q]);
        sh[threadIdx.x] = m;
        __syncthreads();
        for (int s = kRedThreads / 2; s > 0; s >>= 1) {
            if ((int)threadIdx.x < s) sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + s]);
            __syncthreads();
        }
        if (threadIdx.x == 0) max6[q] = sh[0];
        __syncthreads();
    }
}

struct MuArgs {
    float *g[3], *rho, *pi, *u, *mod;  // mod: bfgsmod slot (compact) or null
    float step, s1, s2, s3, vp0, vs0, rho0;
    const float *max6;  // maxima of vp, vs, rho and of the gradients
    int lbfgs, numpar;
    int64_t ncell;
};

// modelupdate.c:97-157 (the gradient normalisation folded in as a division:
// modelupdate.c:84-115, without L-BFGS, by the gradients' maxima, when the vp
// and vs maxima are both nonzero)
__global__ __launch_bounds__(kRedThreads) void k_modelupdate(DevGeom g, MuArgs A)
{
    const float n1 = A.max6[3], n2 = A.max6[4], m5 = A.max6[5], n3 = m5 == 0.0f ? 1.0f : m5;
    const bool normalise = !A.lbfgs && n1 > 0.0f && n2 > 0.0f;
    for (Rows R = wave_rows(g); R.r < R.n; R.r += R.step) {
        const int64_t c0 = row_at(g, R.r), l0 = R.r * g.nz;
        for (int k = threadIdx.x; k < g.nz; k += 64) {
            const int64_t c = c0 + k;
            float gvp = A.g[0][c], gvs = A.g[1][c], grho = A.g[2][c];
            const float rho = A.rho[c], pi = A.pi[c], u = A.u[c];
            if (normalise) {
                gvp = gvp / n1;
                gvs = gvs / n2;
                grho = grho / n3;
                A.g[0][c] = gvp;
                A.g[1][c] = gvs;
                A.g[2][c] = grho;
            }
            const double vp = sqrt((double)(pi / rho)), vs = sqrt((double)(u / rho));
            const float vpnew = (float)(vp + (double)(((A.step * A.s1) * gvp) * A.vp0));
            const float vsnew = (float)(vs + (double)(((A.step * A.s2) * gvs) * A.vs0));
            const float rhonew = rho + (((A.s3 * A.step) * grho) * A.rho0);
            if (A.mod) {
                const int64_t l = l0 + k;
                A.mod[l] = (float)(((double)vpnew - vp) / (double)A.vp0);
                if (A.numpar > 1) A.mod[A.ncell + l] = (float)(((double)vsnew - vs) / (double)A.vs0);
            }
            A.u[c] = (rhonew * vsnew) * vsnew;
            A.pi[c] = (rhonew * vpnew) * vpnew;
            A.rho[c] = rhonew;
        }
    }
}

}  // namespace ifos

extern "C" int ifos_precon_grad(const ifos_geom *g, float *const d_grad[3], int damptype, const int *src_xyz, int nsrc,
                                const int *rec_xyz, int ntr, const int nglob[3], const int pos[3], void *stream)
{
    if (!g || !d_grad || damptype < 0 || damptype > 3 || nsrc < 0 || ntr < 0 || (nsrc && !src_xyz) ||
        (ntr && !rec_xyz)) {
        set_error("ifos_precon_grad: bad arguments (DAMPTYPE must be 0..3)");
        return IFOS_EINVAL;
    }
    const hipStream_t st = (hipStream_t)stream;
    const DevGeom G = make_dev_geom(g);
    PreconArgs A;
    for (int n = 0; n < 3; ++n) A.g[n] = d_grad[n];
    A.nsrc = damptype == 2 ? nsrc : 0;
    A.ntr = (damptype == 1 || damptype == 2) ? ntr : 0;
    A.damptype = damptype;
    A.free_surf = g->free_surf;
    A.sh = A.rh = g->fw + 40;  // precongrad.c:38-39
    A.nxg = nglob ? nglob[0] : g->nx;
    A.nyg = nglob ? nglob[1] : g->ny;
    A.nzg = nglob ? nglob[2] : g->nz;
    A.posx = pos ? pos[0] : 0;
    A.posy = pos ? pos[1] : 0;
    A.posz = pos ? pos[2] : 0;
    // positions and tables, stream-ordered
    const size_t np = (size_t)(A.nsrc + A.ntr) * 3, nt = (size_t)kSrcD + kRecD + 2 * ((size_t)g->nx + g->ny + g->nz);
    int *d = nullptr;
    int rc = hip_check(hipMallocAsync((void **)&d, (np + nt) * 4, st), "precon buffers");
    if (rc) return rc;
    if (A.nsrc)
        rc = hip_check(hipMemcpyAsync(d, src_xyz, (size_t)A.nsrc * 3 * sizeof(int), hipMemcpyHostToDevice, st), "src");
    if (!rc && A.ntr)
        rc = hip_check(hipMemcpyAsync(d + 3 * A.nsrc, rec_xyz, (size_t)A.ntr * 3 * sizeof(int),
                                      hipMemcpyHostToDevice, st), "rec");
    A.src = d;
    A.rec = d + 3 * A.nsrc;
    A.tsrc = (float *)(d + np);
    A.trec = A.tsrc + kSrcD;
    A.ex = A.trec + kRecD;
    A.ey = A.ex + 2 * g->nx;
    A.ez = A.ey + 2 * g->ny;
    if (!rc) {
        const int nt1 = kSrcD + kRecD + g->nx + g->ny + g->nz;
        hipLaunchKernelGGL(k_precon_tables, dim3((unsigned)((nt1 + 255) / 256)), dim3(256), 0, st, G, A);
        hipLaunchKernelGGL(k_precon, dim3((unsigned)((g->nz + 63) / 64), (unsigned)((g->nx + 3) / 4), (unsigned)g->ny),
                           dim3(64, 4), 0, st, G, A);
        rc = hip_check(hipGetLastError(), "k_precon");
    }
    if (!rc) rc = hip_check(hipStreamSynchronize(st), "ifos_precon_grad");
    (void)hipFreeAsync(d, st);
    return rc;
}

extern "C" int ifos_modelupdate(const ifos_geom *g, float *const d_grad[3], float *d_rho, float *d_pi, float *d_u,
                                float *d_bfgsmod, int numpar, int lbfgs, float step, const float weight[3], float vp0,
                                float vs0, float rho0, float maxima[3], void *stream)
{
    if (!g || !d_grad || !d_rho || !d_pi || !d_u || !weight || (lbfgs && !d_bfgsmod)) {
        set_error("ifos_modelupdate: bad arguments");
        return IFOS_EINVAL;
    }
    const hipStream_t st = (hipStream_t)stream;
    const DevGeom G = make_dev_geom(g);
    float *part = nullptr, m[6] = {0, 0, 0, 0, 0, 0};
    int rc = hip_check(hipMallocAsync((void **)&part, (kRedBlocks + 1) * 6 * sizeof(float), st), "modelupdate partials");
    if (rc) return rc;
    MuArgs A;
    for (int n = 0; n < 3; ++n) A.g[n] = d_grad[n];
    A.rho = d_rho;
    A.pi = d_pi;
    A.u = d_u;
    A.mod = lbfgs ? d_bfgsmod : nullptr;
    A.step = step;
    A.s1 = weight[0];
    A.s2 = weight[1];
    A.s3 = weight[2];
    A.vp0 = vp0;
    A.vs0 = vs0;
    A.rho0 = rho0;
    A.max6 = part + 6 * kRedBlocks;
    A.lbfgs = lbfgs;
    A.numpar = numpar;
    A.ncell = (int64_t)g->nx * g->ny * g->nz;
    hipLaunchKernelGGL(k_mu_max, dim3(kRedBlocks), dim3(64, 4), 0, st, G, d_rho, d_pi, d_u, d_grad[0], d_grad[1],
                       d_grad[2], part);
    hipLaunchKernelGGL(k_mu_final, dim3(1), dim3(kRedThreads), 0, st, part, kRedBlocks, part + 6 * kRedBlocks);
    hipLaunchKernelGGL(k_modelupdate, dim3(row_grid(g)), dim3(64, 4), 0, st, G, A);
    rc = hip_check(hipGetLastError(), "k_modelupdate");
    if (!rc) rc = hip_check(hipMemcpyAsync(m, part + 6 * kRedBlocks, sizeof m, hipMemcpyDeviceToHost, st), "max");
    if (!rc) rc = hip_check(hipStreamSynchronize(st), "ifos_modelupdate");
    (void)hipFreeAsync(part, st);
    if (rc) return rc;
    if (maxima)
        for (int q = 0; q < 3; ++q) maxima[q] = m[q];
    return rc;
}

// steplength.c:26-91: the parabola through (step[0..2], L2[0..2]) in T.
// The literals are double as in the reference, so T = float reproduces its
// float/double promotions (0.1 * step[1] formed in double, stored to float);
// T = double is the FP64 fit.
namespace ifos {
template <class T>
__host__ __device__ inline void steplength_t(T L2[4], T step[5], int lbfgs, int it_group, T teststep)
{
    T a = ((step[0] - step[1]) * (L2[0] - L2[2]) - (step[0] - step[2]) * (L2[0] - L2[1])) /
          (step[0] * step[2] * (step[0] - step[2]) + step[0] * step[1] * (step[1] - step[0]) +
           step[1] * step[2] * (step[2] - step[1]));
    T b = (L2[0] - L2[1]) / (step[0] - step[1]);
    b = b - a * (step[0] + step[1]);
    const T c = L2[0] - a * step[0] * step[0] - b * step[0];
    step[3] = 0;
    if (a > 0) step[3] = -b / (2 * a);
    if (a < 0) {
        if (L2[0] < L2[1] && L2[0] < L2[2]) step[3] = 0.1 * step[1];
        if (L2[1] < L2[0] && L2[1] < L2[2]) step[3] = step[1];
        if (L2[2] < L2[0] && L2[2] < L2[1]) step[3] = step[2];
    }
    if (step[3] > 2.5 * step[4]) step[3] = 2.5 * step[4];
    if (lbfgs && it_group > 1 && step[3] > 1.0) step[3] = 1.0;
    if (step[3] <= 0) step[3] = 0.1 * step[1];
    if (step[3] < 0.1 * step[1]) step[3] = 0.1 * step[1];
    L2[3] = a * step[3] * step[3] + b * step[3] + c;
    step[4] = step[3] / 2;
    if (step[4] < 0.2 * teststep) step[4] = 0.2 * teststep;
    if (step[4] > teststep) step[4] = teststep;
    if (lbfgs && it_group > 1) step[4] = 0.5;
}

// one thread: the FP64 fit where the FP64 misfits already are
__global__ void k_steplength64(double *L2, double *step, int lbfgs, int it_group, double teststep)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) steplength_t<double>(L2, step, lbfgs, it_group, teststep);
}
}  // namespace ifos

// steplength.c:26-91 on the host, in the reference's float arithmetic
extern "C" int ifos_steplength(float L2[4], float step[5], int lbfgs, int it_group, float teststep)
{
    if (!L2 || !step) return IFOS_EINVAL;
    ifos::steplength_t<float>(L2, step, lbfgs, it_group, teststep);
    return IFOS_OK;
}

extern "C" int ifos_steplength_f64(double *d_L2, double *d_step, int lbfgs, int it_group, double teststep,
                                   void *stream)
{
    if (!d_L2 || !d_step) {
        set_error("ifos_steplength_f64: null argument");
        return IFOS_EINVAL;
    }
    const hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(ifos::k_steplength64, dim3(1), dim3(64), 0, st, d_L2, d_step, lbfgs, it_group, teststep);
    return hip_check(hipGetLastError(), "k_steplength64");
}
