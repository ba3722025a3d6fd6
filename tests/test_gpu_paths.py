"""Every form that the launch rules choose, at the sizes where it can go
wrong: march rows of 32 and 64 lanes with and without LDS staging at k depths
around multiples of both, on grids whose step fits the last-level cache and
past it; DFT chunks with a partial one and more frequencies than one launch
takes; gradient tiles' edges; vector forms of the optimiser passes; receivers
that share cells.  Against the oracle; where the other tests of a kernel ask
for equal bits, so do these.
"""
import os
import sys

import numpy as np
import pytest

import test_gpu_batch as tb
import test_gpu_kernels as tk
import test_gpu_optim as to
from helpers import max_ulp, small_grid
from pyoracle import Oracle

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
from optim_oracle import LbfgsOracle  # noqa: E402

pytestmark = pytest.mark.gpu


def _note(msg):
    print(msg, flush=True)


def _both_updates(ig, g, seed):
    """whole-domain velocity and stress update against the oracle, bit for bit"""
    o, rng, rho, pi, u, avg, prof, f, psi = tk._setup(g, seed)
    G = tk._geom(ig, g)
    dmodel, df, dpsi, dprof = tk._upload(ig, G, rho, pi, u, avg, f, psi, prof)
    box = o.box(g)
    for velocity in (True, False):
        fo, po = [a.copy() for a in f], [p.copy() for p in psi]
        if velocity:
            o.update_v(g, box, 1, fo, avg[3], avg[4], avg[5], [], None, None, None, 0)
            o.update_v_cpml(g, box, 1, fo, avg[3], avg[4], avg[5], [], None, None, None, 0, prof, po)
        else:
            o.update_s(g, box, fo, pi, u, avg[0], avg[1], avg[2])
            o.update_s_cpml(g, box, fo, pi, u, avg[0], avg[1], avg[2], prof, po)
        df = [G.to_dev(a) for a in f]
        dpsi = [ig.DBuf.from_numpy(p) for p in psi]
        (ig.update_v if velocity else ig.update_s)(G, ig.REGION_ALL, df, dmodel, dprof, dpsi)
        ig.sync()
        for n in range(9):
            assert max_ulp(g.interior(G.from_dev(df[n])), g.interior(fo[n])) == 0, tk.NAMES[n]
            assert np.array_equal(dpsi[n].numpy(), po[n]), f"velocity={velocity} psi[{n}]"


@pytest.mark.parametrize("tiles", [None, (4, 8, 0, 0, 0, 1, 1, 1), (8, 16, 0, 0, 0, 1, 1, 1), (2, 0, 0, 0, 0, 1, 1, 1),
                                   (4, 0, 0, 0, 1, 1, 1, 0), (4, 16, 0, 0, 0, 1, 1, 0)])
@pytest.mark.parametrize("nz", [63, 64, 65, 96, 97, 130])
def test_march_rows(nz, tiles):
    """rows of 64 (nz 64, 97) and of 32 lanes (65, 96, 130), whole rows below
    64; chunks of 8 and 16 planes with 5 left over of the 21 (a set chunk is
    kept), the automatic chunk (4 and 1 left), and the default's rule (None)"""
    import ifosgpu as ig
    _note(f"march rows nz={nz} tiles={tiles}")
    old = ig.get_plain_tiles()
    if tiles:
        ig.set_plain_tiles(tiles)
    try:
        _both_updates(ig, small_grid(nx=19, ny=21, nz=nz, fw=5), 3 + nz)
    finally:
        ig.set_plain_tiles(old)


# 17 words of 4 bytes a cell: past 256e6 bytes from 3.77e6 cells on
@pytest.mark.parametrize("nx,nz", [(157, 160), (122, 200), (126, 192), (90, 276)])
def test_march_rows_past_the_cache(nx, nz):
    """the default shape where a step is not cached: LDS staging with rows of
    32 (nz 160, 200: both updates, rows in 64s 1.2 and 1.14 x longer; 276:
    velocity only, 1.11 x) and of 64 (192)"""
    import ifosgpu as ig
    _note(f"large march {nx}x157x{nz}")
    _both_updates(ig, small_grid(nx=nx, ny=157, nz=nz, fw=9), 77)


@pytest.mark.parametrize("L", [1, 2, 4])
@pytest.mark.parametrize("nz", [65, 97])
def test_march_rows_visco(nz, L):
    import ifosgpu as ig
    old = ig.get_plain_tiles()
    ig.set_plain_tiles((4, 8, 0, 0, 0, 1, 1, 1))
    try:
        tk.test_visco_stress_update_regions((ig, ig), 1, 2, nz, L)
    finally:
        ig.set_plain_tiles(old)


@pytest.mark.parametrize("prec_name,nf,nt,free_surf", [("compat", 9, 70, 0), ("kahan", 11, 70, 0), ("kahan", 8, 50, 0),
                                                     ("compat", 2, 33, 1)])
def test_one_shot_chunks(prec_name, nf, nt, free_surf):
    """a one-shot context against the oracle and (up to 8 frequencies) the
    batched path: more
    frequencies than a launch takes, a last chunk that is not full, a force
    in the slab, receivers in the slab and several in one cell"""
    import ifosgpu as ig
    g = small_grid(nx=27, ny=25, nz=37, fw=6, nt=nt, free_surf=free_surf)
    srcs = [(3, 12, 20, 0.0, 50.0, 1e6, 4), (14, 11, 18, 0.0, 50.0, 1.0, 1)]
    rec = np.array([[9, 10, 19], [3, 4, 33], [9, 10, 19], [20, 12, 21], [9, 10, 19], [24, 3, 2]], np.int32)
    finv, tast = [35.0 + 5.0 * n for n in range(nf)], 100
    prec = ig.DFT_KAHAN if prec_name == "kahan" else ig.DFT_COMPAT
    _note(f"one-shot chunks {prec_name} nf={nf} nt={nt}")
    true, start = tb._models(g)
    G = tb._setup(ig, g, finv, tast, prec)
    ref = tb._plain(ig, G, g, true, start, srcs, rec, finv, tast, prec, one_shot=True)
    orc = tb._oracle(g, true, start, srcs, rec, finv, tast)
    for n in range(len(srcs)):
        for q in range(3):
            assert max_ulp(ref["syn"][n][q][:, 1:], orc["syn"][n][q][:, 1:]) == 0, f"synthetics, shot {n}"
    for n in range(3):
        a, want = g.interior(ref["grads"][n]), g.interior(orc["grads"][n])
        if prec_name == "compat":
            assert max_ulp(a, want) == 0, f"gradient {n}"
        else:
            assert tb.rel_l2(a, want) <= 1e-4, f"gradient {n}"
    if nf > 8:  # the batched path takes up to 8
        return
    out = tb._batched(ig, G, g, true, start, srcs, rec, finv, tast, prec, 7, True)
    for n in range(len(srcs)):
        assert max_ulp(out["syn"][n], ref["syn"][n]) == 0, f"batched synthetics, shot {n}"
    for n in range(3):
        assert max_ulp(out["grads"][n], ref["grads"][n]) == 0, f"batched gradient {n}"
    out["ctx"].close()


@pytest.mark.parametrize("nx,ny,nz", [(18, 16, 20), (17, 17, 21), (17, 18, 19), (19, 17, 21)])
@pytest.mark.parametrize("numpar", [1, 2])
def test_optimiser_vectors(nx, ny, nz, numpar):
    """L-BFGS passes by vectors of four words, where they divide the history's
    slots (5760 words, 11520, ...), and by single words (6069, 5814, 6783: 1 to
    3 over); the FP64 sums' order is the only difference, so to the few ulp of
    the other L-BFGS test"""
    import ifosgpu as ig
    g = small_grid(nx=nx, ny=ny, nz=nz, fw=4)
    _note(f"optimiser vectors {nx}x{ny}x{nz} numpar={numpar}")
    G = to._geom(ig, g)
    rng = np.random.default_rng(nx)
    n = numpar * g.nx * g.ny * g.nz
    o = LbfgsOracle(n, 2, dot="f64", vec=np.float32)
    lb = ig.Lbfgs(G, numpar, 2)
    try:
        grads = [to._field(g, rng) for _ in range(numpar)]
        flat = lambda gs: np.concatenate([g.interior(a).ravel() for a in gs])
        pair = lambda gs: ([G.to_dev(a) for a in gs] + [None])[:2]
        lb.savegrad(*pair(grads))
        o.savegrad(flat(grads))
        for it in range(1, 4):
            w = it % 2 or 2
            s = (0.01 * rng.standard_normal(n)).astype(np.float32)
            o.mod[w - 1] = s
            lb.mod(w).copy_from(ig.DBuf.from_numpy(s))
            grads = [(0.7 * a + 0.3 * to._field(g, rng)).astype(np.float32) for a in grads]
            d = pair(grads)
            h0 = lb.update(d[0], d[1], it + 1)
            q, h0_o = o.update(flat(grads), it + 1)
            assert h0 == pytest.approx(h0_o, rel=1e-12)
            got = np.concatenate([g.interior(G.from_dev(t)).ravel() for t in d[:numpar]])
            assert to._close(got, q), f"direction, iteration {it + 1}"
            for v in (1, 2):
                assert to._close(lb.grad(v).numpy(), o.grad[v - 1]), f"slot {v}"
    finally:
        lb.close()


@pytest.mark.parametrize("nx,ny,nz", [(13, 15, 63), (14, 16, 64), (15, 13, 65), (13, 17, 130)])
def test_gradient_and_hessian_tiles(nx, ny, nz):
    """rows of 64 cells (63, 64: 4 rows a tile) and of 32 (65, 130: 8 rows), rows
    and planes past a tile; tiles of 4 planes, as few as these"""
    import ifosgpu as ig
    _note(f"gradient and Hessian tiles {nx}x{ny}x{nz}")
    _gradient_and_hessian(ig, small_grid(nx=nx, ny=ny, nz=nz), [40.0, 60.0, 85.0], 2)


@pytest.mark.timeout(300)
@pytest.mark.parametrize("nx,ny,nz", [(233, 245, 276), (257, 260, 252)])
def test_gradient_and_hessian_long_tiles(nx, ny, nz):
    """8192 workgroups and more: tiles of 8 planes, 5 and 4 left over (ny), in
    rows of 32 (nz 276) and of 64 (252)"""
    import ifosgpu as ig
    tiles = -(-nz // 32) * -(-nx // 8) if nz == 276 else -(-nz // 64) * -(-nx // 4)
    assert tiles * -(-ny // 8) >= 8192
    _note(f"gradient and Hessian, long tiles {nx}x{ny}x{nz}")
    _gradient_and_hessian(ig, small_grid(nx=nx, ny=ny, nz=nz), [40.0], 1)


def _gradient_and_hessian(ig, g, finv, ntr):
    o = Oracle("f32")
    rng = np.random.default_rng(g.nz)
    rho, pi, u = tk.random_model(g, rng)
    nf = len(finv)
    Ff = [rng.standard_normal((nf,) + g.shape, np.float32) for _ in range(6)]
    Fb = [rng.standard_normal((nf * (ntr + 1),) + g.shape, np.float32) for _ in range(6)]
    for a in Ff + Fb:  # zero halos, as the DFT fields have
        a[:, :3] = 0; a[:, 3 + g.ny:] = 0; a[:, :, :3] = 0; a[:, :, 3 + g.nx:] = 0
        a[:, :, :, :3] = 0; a[:, :, :, 3 + g.nz:] = 0
    out = [rng.random(g.shape).astype(np.float32) for _ in range(3)]
    G = tk._geom(ig, g)
    dFf, dFb = [G.to_dev(a) for a in Ff], [G.to_dev(a) for a in Fb]
    dm = [G.to_dev(a) for a in (rho, pi, u)] + [G.empty() for _ in range(6)]
    ref, dev = [a.copy() for a in out], [G.to_dev(a) for a in out]
    o.hess_F(g, Ff, Fb, ref, rho, pi, u, finv, ntr)
    ig.hess_F(G, dFf, dFb, ntr, dm, finv, dev)
    ig.sync()
    for n in range(3):
        assert max_ulp(g.interior(G.from_dev(dev[n])), g.interior(ref[n])) == 0, f"hess{n + 1}"
    Fb = [np.ascontiguousarray(a[:nf]) for a in Fb]
    dFb = [G.to_dev(a) for a in Fb]
    ref, dev = [a.copy() for a in out], [G.to_dev(a) for a in out]
    o.gradient_F(g, Ff, Fb, ref, rho, pi, u, finv)
    ig.gradient_F(G, dFf, dFb, dm, finv, dev)
    ig.sync()
    for n in range(3):
        assert max_ulp(g.interior(G.from_dev(dev[n])), g.interior(ref[n])) == 0, f"grad{n + 1}"


@pytest.mark.parametrize("nx,ny,nz", [(17, 19, 47), (19, 17, 64), (15, 16, 65)])
def test_time_domain_gradient_tiles(nx, ny, nz):
    """the sample kernel's tiles: rows of 64 (nz 47, 64) and 32 lanes, rows and
    planes past a tile; bits, as the other test of this gradient"""
    import ifosgpu as ig
    import test_gpu_td as tt
    g = small_grid(nx=nx, ny=ny, nz=nz, fw=4, nt=40)
    _note(f"time-domain gradient tiles {nx}x{ny}x{nz}")
    src, rec = (8, 8, nz // 2, 0.0, 60.0, 1.0, 1), np.array([[3 + 2 * n, 6, nz // 2 + n] for n in range(6)], np.int32)
    o = Oracle("f32")
    start, true = tt._models(g, 3)
    obs = o.run_shot(g, *true, src, rec, [40.0], want_adjoint=False)["syn"]
    ref = o.run_shot(g, *start, src, rec, [40.0], obs=obs, want_history=True)
    want = [o.zeros(g) for _ in range(3)]
    o.td_gradient(g, ref["vfwd"], ref["vadj"], *start, want)
    G = tk._geom(ig, g)
    ctx = ig.ShotContext(G, 1, len(rec))
    ctx.set_cpml(4000.0, 50.0)
    ctx.set_model(*[G.to_dev(a) for a in start])
    grads = [G.empty() for _ in range(3)]
    ctx.run_shot_td(src, rec, ig.DBuf((3, len(rec), g.nt + 1)), grads, ig.DBuf.from_numpy(np.stack(obs)))
    ig.sync()
    for n in range(3):
        assert max_ulp(g.interior(G.from_dev(grads[n])), g.interior(want[n])) == 0, f"gradient {n + 1}"
    ctx.close()


@pytest.mark.parametrize("ntr", [1, 64, 200])
def test_precon_points(ntr):
    """tapers of many points, most of them far from a cell; the bound of the
    other taper test"""
    import ifosgpu as ig
    g = small_grid(nx=33, ny=19, nz=67, fw=4)
    _note(f"precon points ntr={ntr}")
    G = to._geom(ig, g)
    rng = np.random.default_rng(ntr)
    grads = [to._field(g, rng) for _ in range(3)]
    src = np.array([[1, 1, 1], [33, 19, 67]], np.int32)
    rec = np.stack([rng.integers(1, n + 1, ntr) for n in (33, 19, 67)], 1).astype(np.int32)
    d = [G.to_dev(a) for a in grads]
    ig.precon_grad(G, d, 2, src, rec)
    og = [g.interior(a).copy() for a in grads]
    to.pg_oracle(og, 2, src, rec, (g.nx, g.ny, g.nz), g.fw, 0)
    for n in range(3):
        assert to._max_ulp(g.interior(G.from_dev(d[n])), og[n]) <= 4, f"grad{n + 1}"


def test_exact_adjoint_shared_receivers():
    """receivers that share a cell, and ones in neighbouring cells whose
    injections share a word: as the other test of the exact adjoint"""
    import ifosgpu as ig
    import test_gpu_adjoint as ta
    g = ta._grid(nt=60)
    rec = np.array([[8, 17, 13], [9, 17, 13], [8, 17, 13], [8, 18, 13], [8, 17, 14], [24, 22, 26], [1, 1, 1],
                    [9, 17, 13]], np.int32)
    _note("exact adjoint, shared receivers")
    one = np.ones(g.shape)
    m = [a.astype(np.float32) for a in ta._model(4000.0 * one, 2300.0 * one, 2000.0 * one)]
    b = ta._bump(g, 11, 12, 13, 4)
    true = [a.astype(np.float32) for a in ta._model(4000.0 * (1 + 0.05 * b), 2300.0 * (1 + 0.05 * b), 2000.0 * one)]
    o = Oracle("f32")
    obs = o.run_shot(g, *true, ta.SRC, rec, [100.0], want_adjoint=False)["syn"]
    ref = o.run_shot_adj(g, *m, ta.SRC, rec, obs)
    G = tk._geom(ig, g)
    ctx = ig.ShotContext(G, 1, len(rec))
    ctx.set_cpml(4000.0, 50.0)
    ctx.set_model(*[G.to_dev(a) for a in m])
    d_syn = ig.DBuf((3, len(rec), g.nt + 1))
    grads = [G.empty() for _ in range(3)]
    J = ctx.run_shot_adj(ta.SRC, rec, d_syn, grads, ig.DBuf.from_numpy(np.stack(obs).astype(np.float32)))
    ig.sync()
    assert J == pytest.approx(ref["J"], rel=1e-6)
    for q in range(3):
        a, want = g.interior(G.from_dev(grads[q])), g.interior(ref["grads"][q])
        assert np.abs(want).max() > 0
        assert ta.rel_l2(a, want) <= 1e-4, f"gradient {q + 1}"
    ctx.close()
