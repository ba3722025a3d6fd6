// dft.hip -- the chunked on-the-fly DFT (disc_fourier.c:28-62) of the one-shot
// and batched paths on gfx950: velocity snapshots of up to 32 samples folded
// into the accumulators in one pass, with the roundings of one discfourier
// call per sample.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "ifos_dev.h"

namespace ifos {

// chunked DFT: nsnap (<= CH) snapshots of one shot's v, every accumulator
// of the cell updated nsnap times in registers.  trig[(c*tstride + l)*2 +
// {0,1}] are the cos/sin factors of snapshot c (disc_fourier.c:42-44).  One thread
// per cell of [1..N]^3, shot and velocity component (blockIdx.z = shot * ny
// + j - 1, blockIdx.y = 3 * (i row block) + component), so a thread holds
// one component's snapshots and its two accumulators; the frequencies are
// walked in order with the next frequency's accumulators loaded while the
// current one is updated.  FIRST: the accumulators start at 0 and are not
// read, which saves their zeroing as well.  FULL: nsnap is CH, so that no
// term sits behind a test of its own; the tests also kept the trig factors'
// scalar loads one by one, each waited for before its term.
struct FBase {
    float *p[6];
};

template <int CH, bool KAHAN, bool FIRST, bool FULL>
__global__ __launch_bounds__(256) void k_dft_chunk(DevGeom g, const float *ring, int64_t rstride, int nsnap,
                                                  FBase F, FBase Cc, int64_t fshot, uint32_t tot, int nf,
                                                  const double *__restrict__ trig, int tstride)
{
    const int q = (int)(blockIdx.y % 3u);  // velocity component: accumulators q (Re) and 3 + q (Im)
    const int k = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int i = (int)(blockIdx.y / 3u) * blockDim.y + threadIdx.y + 1;
    const int j = (int)(blockIdx.z % (unsigned)g.ny) + 1;
    const int s = (int)(blockIdx.z / (unsigned)g.ny);
    if (k > g.nz || i > g.nx) return;
    const int64_t cell = at(g, j, i, k);
    const uint32_t vo = (uint32_t)cell * 4u;
    const int64_t fe = g.fbytes / 4;
    const float *rp = ring + (int64_t)s * rstride + (int64_t)q * fe + cell;
    float v[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (FULL || c < nsnap) v[c] = __builtin_nontemporal_load(rp + 3 * c * fe);
    rsrc_t r[2], rc[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        r[n] = make_rsrc(F.p[q + 3 * n] + (int64_t)s * fshot, tot);
        if (KAHAN) rc[n] = make_rsrc(Cc.p[q + 3 * n] + (int64_t)s * fshot, tot);
    }
    float a[2], cm[2], an[2], cn[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        a[n] = FIRST ? 0.0f : bload(r[n], vo, 0);
        cm[n] = KAHAN && !FIRST ? bload(rc[n], vo, 0) : 0.0f;
    }
#pragma unroll 1
    for (int l = 0; l < nf; ++l) {
        const uint32_t lo = (uint32_t)l * g.fbytes, ln = (uint32_t)min(l + 1, nf - 1) * g.fbytes;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            an[n] = FIRST ? 0.0f : bload(r[n], vo, ln);
            cn[n] = KAHAN && !FIRST ? bload(rc[n], vo, ln) : 0.0f;
        }
        const double *tr = trig + 2 * l;
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if (FULL || c < nsnap) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {  // n = 0: cos (Re), 1: sin (Im)
                    const double term = (double)v[c] * tr[c * 2 * tstride + n];
                    if (KAHAN) {
                        const float yv = (float)(term - (double)cm[n]);
                        const float t = a[n] + yv;
                        cm[n] = (t - a[n]) - yv;
                        a[n] = t;
                    } else {
                        a[n] = (float)(a[n] + term);
                    }
                }
            }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            bstore(a[n], r[n], vo, lo);
            if (KAHAN) bstore(cm[n], rc[n], vo, lo);
            a[n] = an[n];
            cm[n] = cn[n];
        }
    }
}

int dft_trig(const ifos_geom *g, const float *finv, int nf, int ntast, double *out)
{
    const int nsamp = g->nt / ntast;
    for (int back = 0; back < 2; ++back)
        for (int q = 0; q < nsamp; ++q) {
            const int nt = (q + 1) * ntast;
            float t = 0.0f;
            if (back == 0) t = nt * g->dt;
            if (back == 1) t = g->time - nt * g->dt;
            double *o = out + ((size_t)back * nsamp + q) * nf * 2;
            for (int l = 0; l < nf; ++l) {
                o[2 * l + 0] = cos(2.0 * t * finv[l] * M_PI) * g->dt * ntast;
                o[2 * l + 1] = sin(2.0 * t * finv[l] * M_PI) * g->dt * ntast;
            }
        }
    return nsamp;
}

static void dft_chunk_launch(int chunk, bool kahan, bool first, dim3 grid, dim3 block, hipStream_t st, const DevGeom &G,
                         const float *ring, int64_t rstride, int nsnap, const FBase &F, const FBase &C,
                         int64_t fshot, uint32_t tot, int nf, const double *trig, int tstride)
{
    auto launch = [&](auto ch, auto kh, auto fi, auto fu) {
        hipLaunchKernelGGL((k_dft_chunk<decltype(ch)::value, decltype(kh)::value, decltype(fi)::value,
                                        decltype(fu)::value>),
                           grid, block, 0, st, G, ring, rstride, nsnap, F, C, fshot, tot, nf, trig, tstride);
    };
    auto go = [&](auto ch) {
        auto full = [&](auto kh, auto fi) {
            if (nsnap == decltype(ch)::value) launch(ch, kh, fi, std::true_type{});
            else launch(ch, kh, fi, std::false_type{});
        };
        if (kahan && first) full(std::true_type{}, std::true_type{});
        else if (kahan) full(std::true_type{}, std::false_type{});
        else if (first) full(std::false_type{}, std::true_type{});
        else full(std::false_type{}, std::false_type{});
    };
    if (chunk <= 4) go(std::integral_constant<int, 4>{});
    else if (chunk <= 8) go(std::integral_constant<int, 8>{});
    else if (chunk <= 16) go(std::integral_constant<int, 16>{});
    else if (chunk <= 24) go(std::integral_constant<int, 24>{});
    else go(std::integral_constant<int, 32>{});
}

int launch_dft_chunk(const ifos_geom *g, int ns, const float *ring, int chunk, int nsnap, float *const Fp[6],
                     float *const Cp[6], int64_t fshot, const double *trig, int nf, bool first, hipStream_t st)
{
    DevGeom G = make_dev_geom(g);
    const size_t fe = ifos_field_elems(g);
    const int64_t rstride = (int64_t)chunk * 3 * (int64_t)fe;
    dim3 block(64, 4), grid((unsigned)((g->nz + 63) / 64), (unsigned)(3 * ((g->nx + 3) / 4)), (unsigned)(ns * g->ny));
    ProfScope ps_(IFOS_K_DFT, st);
    // the fields of a launch's frequencies stay below 4 GiB (the accumulators'
    // buffer offsets are 32-bit)
    const int most = (int)std::min<size_t>(IFOS_MAX_NF, 4294967295u / (fe * 4));
    for (int l0 = 0; l0 < nf; l0 += most) {
        const int n = std::min(most, nf - l0);
        FBase F, C = {};
        for (int q = 0; q < 6; ++q) {
            F.p[q] = Fp[q] + (size_t)l0 * fe;
            if (Cp) C.p[q] = Cp[q] + (size_t)l0 * fe;
        }
        const uint32_t tot = (uint32_t)(n * fe * 4);
        const double *tr = trig + 2 * l0;
        dft_chunk_launch(chunk, Cp != nullptr, first, grid, block, st, G, ring, rstride, nsnap, F, C, fshot, tot, n,
                         tr, nf);
        const int rc = hip_check(hipGetLastError(), "k_dft_chunk");
        if (rc) return rc;
    }
    return IFOS_OK;
}

}  // namespace ifos
