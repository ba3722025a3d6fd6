"""A gradient shot made of the library's per-routine entry points, in the
order of ifos3d.c:712-975: interior and CPML updates in launches of their own,
one discfourier call per sample, the point operations one by one.  These
kernels (slab kernels, interior marches, per-sample DFT) are not those of
ifos_ctx_run_shot and ifos_batch_run (whole-domain marches, chunked DFT, merged
point kernels), so the two sides of a comparison share gradient_F alone.  The
interface is ifosgpu.ShotContext's.
"""
import numpy as np


class RoutineShots:
    def __init__(self, ig, G, nf, ntr, prec):
        self.ig, self.G, self.prec = ig, G, prec
        self.f = [G.empty() for _ in range(9)]
        self.psi_s = [ig.DBuf((G.psi_elems(n),)) for n in range(9)]
        self.psi_v = [ig.DBuf((G.psi_elems(n),)) for n in range(9)]
        self.F = [G.empty(nf) for _ in range(12)]
        self.C = [G.empty(nf) for _ in range(12)] if prec == ig.DFT_KAHAN else None
        self.adj = ig.DBuf((3, ntr, G.nt + 2))
        self.visco, self.r = None, []

    def set_cpml(self, vppml, fpml):
        self.prof = self.ig.DBuf.from_numpy(self.ig.cpml_profiles(self.G, vppml, fpml))

    def set_freqs(self, finv, tast):
        self.finv = np.asarray(finv, np.float32)
        self.ntast = self.ig.ntast(self.finv[-1], tast, self.G.c.dt)

    def set_model(self, rho, pi, u):
        ig, G = self.ig, self.G
        m = [a.clone() for a in (rho, pi, u)]
        for a in m:
            ig.matcopy_wrap(G, a)
        avg = [G.empty() for _ in range(6)]
        ig.av_mat(G, m[0], m[2], avg)
        self.m = m + avg

    def set_visco(self, taus, taup, eta):
        ig, G = self.ig, self.G
        self.tau = [a.clone() for a in (taus, taup)]
        for a in self.tau:
            ig.matcopy_wrap(G, a)
        self.tav = [G.empty() for _ in range(3)]
        ig.av_tau(G, self.tau[0], self.tav)
        self.r = [G.empty(len(eta)) for _ in range(6)]
        self.visco = ig.visco_struct(self.r, *self.tau, *self.tav, eta)

    def _step(self, back, nt, d_syn):
        ig, G, f, m = self.ig, self.G, self.f, self.m
        ig.update_v(G, ig.REGION_INTERIOR, f, m, self.prof, self.psi_s)
        if back:
            ig.add_adjoint(G, f, self.rec, self.adj, self.ntr, nt, self.chain)
        else:
            ig.add_forces(G, f, m, self.src, self.sig, 1, nt)
        ig.update_v(G, ig.REGION_CPML, f, m, self.prof, self.psi_s)
        if back:
            ig.add_adjoint(G, f, self.rec, self.adj, self.ntr, nt, self.chain)
        for region in (ig.REGION_INTERIOR, ig.REGION_CPML):
            if self.visco is None:
                ig.update_s(G, region, f, m, self.prof, self.psi_v)
            else:
                ig.update_s_visco(G, region, f, m, self.visco, self.prof, self.psi_v)
        if not back:
            ig.psource(G, f, self.src, self.sig, 1, nt)
        if self.dft and nt % self.ntast == 0:
            q = slice(6 * back, 6 * back + 6)
            ig.discfourier(G, f, self.F[q], self.C[q] if self.C else None, self.finv, nt, self.ntast, back, self.prec)
        if G.c.free_surf:
            ig.surface(G, f, m)
        if not back:
            ig.seismo(G, f, self.rec, self.ntr, nt, G.nt, d_syn)

    def run_shot(self, src, rec_ijk, d_syn, grads, d_obs=None, want_adjoint=True):
        ig, G = self.ig, self.G
        rec = np.ascontiguousarray(rec_ijk, np.int32)
        self.ntr, self.dft = len(rec), want_adjoint
        self.rec, self.chain = ig.DBuf.from_numpy(rec), ig.DBuf.from_numpy(ig.rec_chain(rec))
        self.src = ig.DBuf.from_numpy(np.array([src[0], src[1], src[2], src[6]], np.int32))
        self.sig = ig.DBuf.from_numpy(ig.wavelet(G, 1, src[3], src[4], src[5]))
        for a in self.F + (self.C or []) + [d_syn, self.adj]:
            a.zero_()
        l2 = 0.0
        for back in range(2 if want_adjoint else 1):
            for a in self.f + self.psi_s + self.psi_v + self.r:
                a.zero_()
            if back:
                l2 = ig.residual(G, d_obs, d_syn, self.adj, self.ntr, G.nt)
            for nt in range(1, G.nt + 1):
                self._step(back, nt, d_syn)
        if want_adjoint:
            ig.gradient_F(G, self.F[:6], self.F[6:], self.m, self.finv, grads)
        return l2

    def dft_ptrs(self, back):
        return [a.data_ptr() for a in self.F[6 * back:6 * back + 6]]

    def close(self):
        self.__dict__.clear()
