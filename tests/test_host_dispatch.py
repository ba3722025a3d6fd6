"""The library's host code against a stand-in for the HIP runtime
(tests/standin/standin.c): which memory it holds, which launches it makes and
what it waits for, without a GPU.  The library's own objects are linked
against the stand-in; kernels do not run.
"""
import ctypes as C
import gc
import glob
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
OBJ = os.path.join(os.path.dirname(HERE), "ifos3d-dev_amd", "lib", "obj")


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    objs = [o for o in glob.glob(os.path.join(OBJ, "*.o")) if "dropin" not in o]
    if not objs:
        pytest.skip("the library's objects are not built here")
    d = tmp_path_factory.mktemp("standin")
    c, so = str(d / "standin.o"), str(d / "libifos3d_standin.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-Wall", "-c", os.path.join(HERE, "standin", "standin.c"), "-o", c],
                   check=True)
    subprocess.run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-o", so, *objs, c], check=True)
    return so


@pytest.fixture
def ig(standin):
    """ifosgpu on the stand-in library, with its log as ig.lib().standin_log()"""
    import ifosgpu
    old = ifosgpu._lib, ifosgpu.LIBPATH
    ifosgpu._lib, ifosgpu.LIBPATH = None, standin
    lib = ifosgpu.lib()
    lib.standin_log.restype = C.c_char_p
    lib.standin_held.restype = C.c_size_t
    lib.standin_clear()
    tiles = ifosgpu.get_plain_tiles()
    try:
        yield ifosgpu
    finally:
        gc.collect()
        ifosgpu.set_plain_tiles(tiles)
        ifosgpu._lib, ifosgpu.LIBPATH = old


def _log(ig):
    return [line.split() for line in ig.lib().standin_log().decode().splitlines()]


STREAM = C.c_void_p(0x5150)  # a stream other than the null stream
SRC = (10, 11, 12, 0.0, 60.0, 1.0, 1)
REC = np.array([[8, 9, 10], [12, 9, 14]], np.int32)


def _context(ig, nt=12, nf=2):
    G = ig.Geom(24, 22, 26, 5, 2.0, 2.0, 2.0, 2e-4, nt)
    ctx = ig.ShotContext(G, nf, len(REC))
    ctx.set_cpml(4000.0, 50.0)
    ctx.set_freqs([40.0 + 20.0 * n for n in range(nf)], 10)
    return G, ctx


def test_new_memory_is_zeroed_before_another_stream_sees_it(ig):
    """every fill of new memory on the null stream has been waited for before
    the call returns, and before the call's next work on another stream"""
    G, ctx = _context(ig)
    obs, syn = ig.DBuf((3, len(REC), G.nt + 1)), ig.DBuf((3, len(REC), G.nt + 1))
    grads, model = [G.empty() for _ in range(3)], [G.empty() for _ in range(3)]
    eta = np.array([0.1, 0.2], np.float32)
    calls = {
        "context": lambda: ig.ShotContext(G, 2, 4),
        "set_visco": lambda: ig.ShotContext(G, 1, 1).set_visco(model[0], model[1], eta, stream=STREAM),
        "time-domain": lambda: ctx.run_shot_td(SRC, REC, syn, grads, obs, stream=STREAM),
        "exact adjoint": lambda: ctx.run_shot_adj(SRC, REC, syn, grads, obs, stream=STREAM),
        "batch": lambda: ig.BatchContext(G, 2, 2, 2).set_model(*model),
        "l-bfgs": lambda: ig.Lbfgs(G, 2, 2),
    }
    for what, call in calls.items():
        ig.lib().standin_clear()
        keep = call()
        pending, fills = None, 0
        for line in _log(ig) + [["end"]]:
            if line[0] == "fill":
                pending, fills = line, fills + 1
            elif line[0] == "wait" and line[1] in ("all", "(nil)"):
                pending = None
            elif line[0] in ("launch", "copy") and line[-1] != "(nil)" or line[0] == "end":
                assert pending is None, f"{what}: {line} behind {pending}"
        assert fills > 0, what
        del keep


def _marches(ig):
    """(kernel, workgroups) of the march launches in the log"""
    return [(line[1], int(line[2])) for line in _log(ig) if line[0] == "launch" and
            any(k in line[1] for k in ("k_v_march", "k_s_march", "k_v_lds", "k_s_lds"))]


def _updates(ig, G, f, m, psi, prof):
    ig.lib().standin_clear()
    ig.update_v(G, ig.REGION_ALL, f, m, prof, psi)
    ig.update_s(G, ig.REGION_ALL, f, m, prof, psi)
    return _marches(ig)


def _region_call(ig, n=84):
    G = ig.Geom(n, n, n, 10, 2.0, 2.0, 2.0, 2e-4, 10)
    bufs = [G.empty() for _ in range(9)], [G.empty() for _ in range(9)], \
        [ig.DBuf((G.psi_elems(q),)) for q in range(9)], ig.DBuf((18 * 21,))
    return lambda: _updates(ig, G, *bufs)


@pytest.mark.parametrize("jc", [4, 8, 10, 30, 84])
@pytest.mark.parametrize("lds", [0, 1])
def test_a_set_chunk_is_kept(ig, jc, lds):
    """jc > 0 of a caller's shape is the number of planes of a tile, however
    few workgroups that makes: 84^3 in rows of 32 lanes is 3 x 11 tiles along k
    and i (8 rows a workgroup), grids are multiples of 8"""
    run = _region_call(ig)
    ig.set_plain_tiles((4, jc, 0, 0, 0, 1, 1, lds))
    tiles = 3 * 11 * -(-84 // jc)
    got = run()
    assert [n for _, n in got] == [-(-tiles // 8) * 8] * 2
    assert all(("_lds" in k) == bool(lds) for k, _ in got)
    ig.set_plain_tiles((4, 0, 0, 0, 0, 1, 1, lds))  # automatic: 4 planes here
    assert [n for _, n in run()] == [-(-3 * 11 * 21 // 8) * 8] * 2


def test_the_default_shape_comes_back(ig):
    """default -> another shape -> the shape read before: the launches of the
    default's rule again (register marches with 4 planes a tile at 84^3), for
    the region calls and for a batch"""
    run = _region_call(ig)
    first, old = run(), ig.get_plain_tiles()
    assert all("_march" in k for k, _ in first)
    ig.set_plain_tiles(old)
    assert run() == first
    ig.set_plain_tiles((4, 8, 0, 0, 0, 1, 1, 1))
    assert run() != first
    ig.set_plain_tiles(old)
    assert run() == first

    G = ig.Geom(84, 84, 84, 10, 2.0, 2.0, 2.0, 2e-4, 2)
    b = ig.BatchContext(G, 3, 1, 2)

    def shots():
        ig.lib().standin_clear()
        b.run([SRC] * 3, REC, want_adjoint=False)
        return _marches(ig)

    first = shots()
    assert all("_march" in k for k, _ in first)
    b.set_tiles(old, old)
    assert shots() == first
    b.set_tiles((8, 32, 0, 0, 0, 1, 1, 1), (8, 32, 0, 0, 0, 1, 1, 1))
    assert shots() != first
    b.set_tiles(old, old)
    assert shots() == first
    b.close()


def test_the_autotuner_times_and_keeps_the_default(ig):
    """where the default shape is the fastest candidate, the tuned batch makes
    the launches of one that was not tuned; set again from the tuner's answer too"""
    G = ig.Geom(84, 84, 84, 10, 2.0, 2.0, 2.0, 2e-4, 2)
    b = ig.BatchContext(G, 3, 1, 2)
    cands = b.tune_candidates()
    assert cands.count((4, 32, 0, 0, 0, 1, 1, 1)) == 1 and len(set(cands)) == len(cands)
    d = cands.index((4, 32, 0, 0, 0, 1, 1, 1))

    def shots():
        ig.lib().standin_clear()
        b.run([SRC] * 3, REC, want_adjoint=False)
        return _marches(ig)

    first = shots()
    ms = [2.0] * 2 * len(cands) + [100.0] * 16  # v and s of each candidate, then the fused step's
    ms[2 * d] = ms[2 * d + 1] = 1.0
    ig.lib().standin_times((C.c_float * len(ms))(*ms), len(ms))
    ig.lib().standin_clear()
    bv, bs, _ = b.autotune(reps=1)
    assert set(first) <= set(_marches(ig))
    assert bv == bs == cands[d]
    assert shots() == first
    b.set_tiles(bv, bs)
    assert shots() == first
    b.close()


@pytest.mark.parametrize("stream", [None, STREAM])
def test_a_shot_gives_its_snapshot_ring_back(ig, stream):
    """a sampling shot holds no more memory after it than before, whether it
    ends well or not; by hipFree, as a stream's pool may keep what it is given"""
    G, ctx = _context(ig)
    obs, syn = ig.DBuf((3, len(REC), G.nt + 1)), ig.DBuf((3, len(REC), G.nt + 1))
    grads = [G.empty() for _ in range(3)]
    before = ig.lib().standin_held()
    for rec, ok in ((REC, True), (REC, True), (np.array([[99, 1, 1]] * 2, np.int32), False)):
        ig.lib().standin_clear()
        if ok:
            ctx.run_shot(SRC, rec, syn, grads, d_obs=obs, stream=stream)
            log = _log(ig)
            assert 32 * 3 * 4 * G.field_elems() in [int(line[2]) for line in log if line[0] == "malloc"]
            assert any("k_dft_chunk" in line[1] for line in log if line[0] == "launch")
            assert [line[0] for line in log[-2:]] == ["wait", "free"] and log[-2][1] == "all"
        else:
            with pytest.raises(ig.IfosError):
                ctx.run_shot(SRC, rec, syn, grads, d_obs=obs, stream=stream)
        assert ig.lib().standin_held() == before
