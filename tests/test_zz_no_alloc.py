"""ddx_model_batch_noalloc (no reference counterpart; for callers that
cannot allocate device memory) against ddx_model_batch through the C ABI:
two calls in a row, the second with a smaller batch of smaller grids, each
member's seismograms bit for bit equal."""
import ctypes

import numpy as np
import pytest

import ddx
from ddx import synth

pytestmark = pytest.mark.gpu


def engine(c, ntime):
    d = ddx.make_desc(c["nx"], c["ny"], c["nz"], c["dx"], c["pml"], c["dt"], c["fm"], ntime, cfl_policy=1)
    e = ddx.Engine(d)
    e.set_model(c["vp"], c["vs"], c["rho"])
    e.set_wavelet(ddx.ricker(c["fm"], c["dt"], ntime))
    e.set_geometry(c["shots"], c["recv"])
    return e


def noalloc(engines):
    L = ddx.lib()
    f = L.ddx_model_batch_noalloc
    f.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_int), ctypes.c_int]
    n = len(engines)
    hs = (ctypes.c_void_p * n)(*[e.h.value for e in engines])
    sh = (ctypes.c_int * n)(*([0] * n))
    rc = f(hs, sh, n)
    if rc != 0:
        raise RuntimeError(f"ddx_model_batch_noalloc: {rc} {L.ddx_last_error(engines[0].h).decode()}")


def uneven(sizes, seed):
    out = []
    for q, (nx, ny, nz) in enumerate(sizes):
        vp, vs, rho = synth.homogeneous_noise(nx, ny, nz, seed=seed + q)
        shots = np.array([[nx // 2 * 10.0, ny // 2 * 10.0, 30.0]], np.float32)
        recv = np.array([[x * 10.0, ny // 3 * 10.0, 20.0] for x in range(2, nx - 2, 5)], np.float32)
        out.append(dict(nx=nx, ny=ny, nz=nz, dx=10.0, pml=8, dt=0.001, fm=20.0, vp=vp, vs=vs, rho=rho, shots=shots,
                        recv=recv))
    return out


@pytest.mark.parametrize("sizes", [[(40, 36, 30), (52, 30, 28), (34, 34, 34)], [(30, 26, 24), (28, 32, 22)]])
def test_noalloc_batch_equals_batch(sizes):
    nt = 60
    cs = uneven(sizes, seed=len(sizes))
    es = [engine(c, nt) for c in cs]
    try:
        for e in es:  # seismogram buffers and brick tables exist after one shot
            e.model_shot(0)
        ddx.model_batch(es)
        ref = [e.seismograms(0) for e in es]
        for e in es:
            e.reset_wave(0)
        noalloc(es)
        got = [e.seismograms(0) for e in es]
        for a, b in zip(got, ref):
            assert np.array_equal(a, b)
    finally:
        for e in es:
            e.close()


def test_noalloc_refuses_unprepared_context():
    c = uneven([(30, 26, 24)], seed=9)[0]
    e = engine(c, 20)
    try:
        with pytest.raises(RuntimeError, match="seismogram buffer"):
            noalloc([e])
    finally:
        e.close()


def test_noalloc_batch_above_the_one_launch_limit(monkeypatch):
    """Tuned members each small enough for half steps in one launch, the batch
    too large for it: the first context's shapes for separate launches may
    differ from those it runs shots with.  The batch needs no more than one
    shot of each member with the latter, whether the first context timed its
    shapes or took them from the cache, and of a member of another grid that
    was given them."""
    nt = 20
    for q, n in enumerate([(36, 33, 30), (70, 24, 22), (100, 20, 18), (130, 18, 20)]):
        sizes = [n, n, (n[0] - 9, n[1] + 5, n[2] + 3)]
        cs = uneven(sizes, seed=20 + q)
        cs[1] = cs[0]
        monkeypatch.setenv("DDX_WHOLE_CELLS", str(int(1.6 * np.prod([v + 16 for v in n]))))
        es = [engine(c, nt) for c in cs]
        try:
            for e in es[:2]:
                e.autotune(reps=1)
            for k in (0, 1):
                es[2].set_brick(k, ddx.PURE_FORWARD, *es[0].brick(k, ddx.PURE_FORWARD))
            ref = []
            for e in es:
                e.model_shot(0)
                ref.append(e.seismograms(0))
            for order in ([1, 0], [0, 1, 2], [1, 2]):
                noalloc([es[i] for i in order])
                for i in order:
                    assert np.array_equal(es[i].seismograms(0), ref[i]), (n, order, i)
        finally:
            for e in es:
                e.close()
