"""Half steps run as one launch (bricks, CPML cells, source and receivers)
against the separate kernels, and the CPML kernels' short division against
the general one: equal bit for bit."""
import numpy as np
import pytest

import ddx
import pyoracle as po
from cases import case, random_fields

pytestmark = pytest.mark.gpu

SHAPES = {
    "fp32": [(32, 8, 1, 4, 1), (64, 4, 1, 2, 1), (64, 4, 1, 2, 4), (64, 4, 1, 4, 4)],
    "bf16": [(32, 8, 1, 2, 2), (32, 8, 1, 4, 2), (64, 4, 1, 2, 2), (64, 4, 1, 4, 2)],
    "fp16": [(32, 8, 1, 4, 2), (64, 4, 1, 2, 2), (64, 4, 1, 4, 2)],
}


def engine(c, storage="fp32", shots=None, **kw):
    e = ddx.Engine(ddx.make_desc(c["nx"], c["ny"], c["nz"], c["dx"], c["pml"], c["dt"], c["fm"], c["ntime"],
                                 rec_width=c["rec_width"], cfl_policy=1, storage=storage, **kw))
    e.set_model(c["vp"], c["vs"], c["rho"])
    e.set_wavelet(po.ricker(c["fm"], c["dt"], c["ntime"]))
    e.set_geometry(c["shots"] if shots is None else shots, c["recv"])
    return e


# partial tiles on every axis; a row of exactly 64; several columns of bricks (256 cells x 16 rows)
GRIDS = [(75, 21, 19, 6), (64, 9, 8, 4), (300, 37, 9, 5)]


@pytest.mark.parametrize("grid,cached", [(GRIDS[0], 1), (GRIDS[0], 0), (GRIDS[1], 1), (GRIDS[2], 0)])
@pytest.mark.parametrize("storage", list(SHAPES))
def test_whole_half_steps_equal_separate_kernels(storage, grid, cached, monkeypatch):
    """cached: ordinary accesses to the updated cells, else streaming ones."""
    if not cached:
        monkeypatch.setenv("DDX_CACHED_CELLS", "0")
    nx, ny, nz, pml = grid
    c = case(nx=nx, ny=ny, nz=nz, pml=pml, ntime=20, rec_width=2)
    dx = c["dx"]
    # in the physical region, in a CPML corner, in the layers that no kernel updates
    shots = np.array([c["shots"][0], [-(pml - 3) * dx, -(pml - 2) * dx, 2 * dx],
                      [-pml * dx, 3 * dx, 3 * dx]], np.float32)
    ref = None
    for shape in [None] + SHAPES[storage]:
        monkeypatch.setenv("DDX_WHOLE_CELLS", "0" if shape is None else "1e9")
        e = engine(c, storage, shots)
        modes = [po.PURE_FORWARD, po.RTM_FORWARD, po.RTM_REVERSE]
        if shape is not None:
            for k in (0, 1):
                for m in modes:
                    e.set_brick(k, m, *shape)
        out = []
        fwi = [po.FWI] if storage == "fp32" else []
        for m in modes + fwi:
            if m == po.FWI and shape is not None and shape[4] == 1:
                for k in (0, 1):
                    e.set_brick(k, m, *shape)
            for s in (0, 1):
                for f, arr in enumerate(random_fields(e.ext_shape, seed=5 + m, scale=1e-3)):
                    e.set(s, f, arr)
            s = 1 if m == po.RTM_REVERSE else 0
            for _ in range(2):
                e.step_vel(s, m)
                e.step_stress(s, m)
            out += [e.get(s, f) for f in range(19 if m == po.FWI else 13)]
        for q in range(len(shots)):
            e.model_shot(q)
            out += [e.seismograms(q), e.get(0, ddx.SZZ)]
        e.rtm_shot(0)
        out += [e.image(q, 0) for q in range(5)]
        e.close()
        if ref is None:
            ref = out
            continue
        for i, (a, b) in enumerate(zip(ref, out)):
            assert np.array_equal(a, b, equal_nan=True), (shape, i)


def test_whole_batches_equal_separate_kernels(monkeypatch):
    """Fused batches of modelling and RTM shots of uneven grids, one member's
    shot in the CPML, in whole half steps and apart."""
    cs = [case(nx=41, ny=22, nz=20, ntime=24), case(nx=70, ny=18, nz=26, pml=5, ntime=24, seed=3)]
    outs = []
    for cells in ("0", "1e9"):
        monkeypatch.setenv("DDX_WHOLE_CELLS", cells)
        es = [engine(c, shots=s) for c, s in zip(cs, (None, np.array([[-20.0, 50.0, 40.0]], np.float32)))]
        ddx.model_batch(es)
        ddx.rtm_batch(es)
        outs.append([e.seismograms(0) for e in es] + [e.image(q, 0) for e in es for q in range(5)])
        for e in es:
            e.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("ring,scaling", [("fp32", 0), ("fp16", 0), ("fp16", 1), ("bf16", 1), ("bfp16", 0)])
def test_reverse_halves_equal_separate_kernels(ring, scaling, monkeypatch):
    """A reverse iteration in two launches against separate ones, for every
    boundary store, with subdomains, with the shot in and outside the region
    that the backward bricks update, alone and as a batch."""
    c = case(nx=70, ny=21, nz=19, pml=6, ntime=30, rec_width=2)
    shots = np.array([c["shots"][0], [-2 * c["dx"], 3 * c["dx"], 2 * c["dx"]]], np.float32)
    outs = []
    for cells in ("0", "1e9"):
        monkeypatch.setenv("DDX_WHOLE_CELLS", cells)
        out = []
        es = [engine(c, shots=shots, divide=d, ring_storage=ring) for d in ((1, 1, 1), (2, 1, 2))]
        for e in es:
            e.set_ring_scaling(scaling)
            for q in range(2):
                e.model_shot(q)
                e.rtm_shot(q)
                out += [e.image(i, 0) for i in range(5)] + [e.get(0, f) for f in range(10)]
        ddx.rtm_batch(es)
        out += [e.image(i, 0) for e in es for i in range(5)]
        for e in es:
            e.close()
        outs.append(out)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("grid", [(75, 21, 19, 6), (20, 9, 8, 4), (33, 10, 9, 5), (512, 9, 8, 5)])
def test_cpml_pairs_equal_one_cell_kernels(grid, monkeypatch):
    """Two x cells per thread against one: rows that begin or end inside a
    pair, slabs two cells thick, damping edges inside a pair, rows of more
    pairs than a block."""
    nx, ny, nz, pml = grid
    c = case(nx=nx, ny=ny, nz=nz, pml=pml, rec_width=2)
    monkeypatch.setenv("DDX_WHOLE_CELLS", "0")
    outs = []
    for cz in ("1", "0"):
        monkeypatch.setenv("DDX_PML_CZ", cz)
        e = engine(c)
        e.set_migration_model(c["vp"][::-1, ::-1, ::-1].copy(), c["vs"][::-1, ::-1, ::-1].copy(),
                              c["rho"][::-1, ::-1, ::-1].copy())
        for f, arr in enumerate(random_fields(e.ext_shape, seed=23, scale=1e-3)):
            e.set(0, f, arr)
        for m in (po.PURE_FORWARD, po.RTM_FORWARD, po.RTM_REVERSE):
            for _ in range(2):
                e.step_vel(0, m)
                e.step_stress(0, m)
        outs.append([e.get(0, f) for f in range(13)])
        e.close()
    for f, (a, b) in enumerate(zip(*outs)):
        assert np.array_equal(a, b), ddx.FIELD_NAMES[f]


@pytest.mark.parametrize("spacing", [(10.0, 10.0, 10.0), (7.3, 12.9, 0.3), (8.0, 1000.0, 3.0)])
def test_cpml_division_is_exact_at_every_magnitude(spacing, monkeypatch):
    """The one-cell CPML kernels divide by the spacing in three operations
    where that is exact, else in general; the LDS-tile kernels always in
    general.  Fields from subnormals to the largest floats, with zeros and
    infinities in some of them."""
    c = case(nx=20, ny=18, nz=16, pml=6)
    for scale in (1e-44, 1e-38, 3e-28, 1e-3, 1e30, 1e37, None):
        outs = []
        for cz in ("1", "18"):
            monkeypatch.setenv("DDX_PML_CZ", cz)
            e = ddx.Engine(ddx.make_desc(c["nx"], c["ny"], c["nz"], spacing[0], c["pml"], 1e-6, c["fm"], 10,
                                         dy=spacing[1], dz=spacing[2], cfl_policy=1))
            e.set_model(c["vp"], c["vs"], c["rho"])
            rng = np.random.default_rng(3)
            for f in range(13):
                a = rng.standard_normal(e.ext_shape)
                if scale is None:  # every magnitude side by side, zeros and a few infinities
                    a = np.sign(a) * 10.0 ** rng.uniform(-46, 37, e.ext_shape)
                    a[rng.random(e.ext_shape) < 0.3] = 0.0
                    a[rng.random(e.ext_shape) < 1e-3] = np.inf
                else:
                    a = a * scale
                e.set(0, f, a.astype(np.float32))
            for m in (po.PURE_FORWARD, po.RTM_REVERSE):
                e.step_vel(0, m)
                e.step_stress(0, m)
            outs.append([e.get(0, f) for f in range(10)])
            e.close()
        for f, (a, b) in enumerate(zip(*outs)):
            assert np.array_equal(a, b, equal_nan=True), (scale, ddx.FIELD_NAMES[f])


# Values a (three spacings) whose first-tap difference 9/8 a, divided by the
# spacing, lies just above 2^-90: the remainder of the short division is then
# no FP32 number, and for these a rounding it changes the quotient.
SMALL_SPACINGS = [
    ("0x1.44f05ep-20", ["0x1.dedd5ep-110", "0x1.26dfdp-110", "0x1.33fad4p-110", "0x1.c423fap-110", "0x1.8fb7ecp-110",
                        "0x1.4eb436p-110", "0x1.7581e6p-110", "0x1.9d564ap-110"]),
    ("0x1.953dfap-17", ["0x1.54e12cp-106", "0x1.8b19e4p-106", "0x1.31fe6p-106"]),
    ("0x1.204942p-15", ["0x1.4f1488p-104"]),
]


@pytest.mark.parametrize("whole,cz", [("1e9", "0"), ("0", "1"), ("0", "0")])
@pytest.mark.parametrize("spacing,values", SMALL_SPACINGS)
def test_cpml_division_by_small_spacings(spacing, values, whole, cz, monkeypatch):
    """The z difference of one plane of szz in the x layers over a small dz,
    in the whole half step, the one-cell and the paired CPML kernels, against
    the correctly rounded quotient: dt / rho is a power of two, so a velocity
    is the quotient's bits."""
    monkeypatch.setenv("DDX_WHOLE_CELLS", whole)
    monkeypatch.setenv("DDX_PML_CZ", cz)
    nx, ny, nz, pml = 20, 18, 16, 6
    dz = np.float32(float.fromhex(spacing))
    a = np.array([float.fromhex(v) for v in values], np.float32)
    e = ddx.Engine(ddx.make_desc(nx, ny, nz, 10.0, pml, 2.0 ** -10, 15.0, 10, dz=float(dz), cfl_policy=1))
    e.set_model(np.full((nz, ny, nx), 2500, np.float32), np.full((nz, ny, nx), 1400, np.float32),
                np.full((nz, ny, nx), 2048, np.float32))
    szz = np.zeros(e.ext_shape, np.float32)
    k = pml + nz // 2
    szz[k] = np.resize(a, szz[k].shape)
    e.set(0, ddx.SZZ, szz)
    e.step_vel(0, po.PURE_FORWARD)
    v = e.get(0, ddx.VZ)
    e.close()
    want = np.float32(2.0 ** -21) * ((np.float32(1.125) * szz[k]) / dz)
    rows = slice(pml, pml + ny)
    for cols in (slice(2, pml), slice(pml + nx, nx + 2 * pml - 2)):
        assert np.array_equal(v[k - 1, rows, cols], want[rows, cols])
        assert np.array_equal(v[k, rows, cols], -want[rows, cols])


@pytest.mark.parametrize("storage", ["fp32", "bf16"])
def test_continuous_batch_across_the_one_launch_limit(storage, monkeypatch):
    """Members join and leave so that a continuous batch lies below, above and
    again below the cells up to which half steps run as one launch: modelling
    and RTM members equal their single shots."""
    c = case(nx=70, ny=18, nz=20, pml=6, ntime=24, rec_width=2)
    d = case(nx=41, ny=22, nz=20, pml=6, ntime=36, rec_width=2, seed=3)
    monkeypatch.setenv("DDX_WHOLE_CELLS", str(int(1.5 * (70 + 12) * (18 + 12) * (20 + 12))))
    es = [engine(x, storage) for x in (c, d, c, d)]
    es[0].autotune(reps=1)
    want = []
    for e in es:
        e.model_shot(0)
        want.append(e.seismograms(0))
    for e in es[2:]:
        e.rtm_shot(0)
    images = [[e.image(i, 0) for i in range(5)] for e in es[2:]]
    for e in es[2:]:
        e.reset_images()
    b = ddx.Batch()
    done = []
    b.add(es[0])
    done += b.run(5)
    b.add(es[1])
    done += b.run(5)
    b.add(es[2], rtm=True)
    done += b.run(5)
    b.add(es[3], rtm=True)
    while len(b):
        done += b.run(50)
    assert len(done) == 4
    for e, w in zip(es[:2], want):
        assert np.array_equal(e.seismograms(0), w)
    for e, w in zip(es[2:], images):
        for i in range(5):
            assert np.array_equal(e.image(i, 0), w[i]), i
    b.close()
    for e in es:
        e.close()


@pytest.mark.parametrize("storage", ["fp32", "bf16"])
def test_backward_bricks_of_their_own(storage):
    """RTM with a shape set for the backward mode that is not the reverse
    mode's, alone and as a batch: the images of the default shapes."""
    c = case(nx=70, ny=21, nz=19, pml=6, ntime=30, rec_width=2)
    shapes = [None, ((64, 4, 1, 4, 1), (64, 2, 1, 8, 1)), ((64, 4, 1, 2, 2), (64, 2, 1, 4, 2))]
    ref = None
    for shape in shapes:
        es = [engine(c, storage) for _ in range(2)]
        for e in es:
            if shape is not None:
                for k in (0, 1):
                    e.set_brick(k, po.RTM_BACKWARD, *shape[k])
                    assert e.brick(k, po.RTM_BACKWARD) == shape[k]
            e.model_shot(0)
        es[0].rtm_shot(0)
        out = [es[0].image(i, 0) for i in range(5)]
        es[0].reset_images()
        ddx.rtm_batch(es)
        out += [e.image(i, 0) for e in es for i in range(5)]
        for e in es:
            e.close()
        if ref is None:
            ref = out
        for a, b in zip(ref, out):
            assert np.array_equal(a, b), shape


def test_autotune_times_every_shape(monkeypatch):
    """Every brick shape of the format is timed in launches of its own, on
    small grids too."""
    monkeypatch.setenv("DDX_WHOLE_CELLS", "0")
    shapes = 9 + 4 + 5 + 6  # one-cell, paired, lane exchange, LDS y arm

    def timed(c):
        e = engine(c)
        n = e.autotune(reps=1)
        e.close()
        return n

    a = case(nx=44, ny=50, nz=47, pml=5, ntime=10)
    assert timed(a) == 2 * 4 * shapes
    assert timed(a) == 0


@pytest.mark.parametrize("storage,tuned", [("fp32", False), ("fp32", True), ("bf16", False)])
def test_reverse_halves_limit_changes_no_image(storage, tuned, monkeypatch):
    """Whole half steps with the backward bricks in the reverse half steps'
    launches and in their own, alone and as a batch."""
    c = case(nx=70, ny=21, nz=19, pml=6, ntime=24, rec_width=2)
    outs = []
    for cells in ("0", "1e9"):
        monkeypatch.setenv("DDX_REV_CELLS", cells)
        es = [engine(c, storage) for _ in range(2)]
        for e in es:
            if tuned:
                e.autotune(reps=1)
            e.model_shot(0)
        es[0].rtm_shot(0)
        out = [es[0].image(i, 0) for i in range(5)]
        ddx.rtm_batch(es)
        outs.append(out + [e.image(i, 0) for e in es for i in range(5)])
        for e in es:
            e.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_autotune_cache_is_keyed_by_what_decides(monkeypatch):
    """Contexts share a tuner's choice where the same launches were timed for
    it only: not across the limits up to which half steps, and the halves of a
    reverse iteration, run as one launch."""

    def timed(**kw):
        e = engine(case(nx=60, ny=50, nz=47, ntime=10, **kw))
        n = e.autotune(reps=1)
        e.close()
        return n

    monkeypatch.setenv("DDX_WHOLE_CELLS", str(65 * 55 * 52))  # of the cells that half steps update
    monkeypatch.setenv("DDX_REV_CELLS", "0")
    timed(pml=5)
    assert timed(pml=5) == 0
    assert timed(pml=4) > 0  # small enough for whole half steps
    monkeypatch.setenv("DDX_WHOLE_CELLS", "1e9")
    assert timed(pml=5) == 0  # as that one
    monkeypatch.setenv("DDX_REV_CELLS", "1e9")
    assert timed(pml=5) > 0
    assert timed(pml=4) == 0


@pytest.mark.parametrize("first", [0, 1])
def test_batches_of_uneven_layers_in_separate_launches(first, monkeypatch):
    """Members with layers on both sides of the width up to which the CPML
    launches take one cell per thread, each side first: fused and continuous
    batches equal single shots."""
    monkeypatch.setenv("DDX_WHOLE_CELLS", "0")
    cs = [case(nx=33, ny=22, nz=20, pml=20, ntime=24, rec_width=2),
          case(nx=70, ny=18, nz=19, pml=6, ntime=24, rec_width=2, seed=3)]
    es = [engine(c) for c in (cs if first == 0 else cs[::-1])]
    want, images = [], []
    for e in es:
        e.model_shot(0)
        want.append(e.seismograms(0))
        e.rtm_shot(0)
        images.append([e.image(i, 0) for i in range(5)])
        e.reset_images()

    def check():
        for e, w in zip(es, want):
            assert np.array_equal(e.seismograms(0), w)

    ddx.model_batch(es)
    check()
    ddx.rtm_batch(es)
    for e, w in zip(es, images):
        assert all(np.array_equal(e.image(i, 0), w[i]) for i in range(5))
        e.reset_images()
    b = ddx.Batch()
    for rtm in (False, True):
        b.add(es[0], rtm=rtm)
        b.run(5)
        b.add(es[1], rtm=rtm)
        while len(b):
            b.run(50)
        check()
    for e, w in zip(es, images):
        assert all(np.array_equal(e.image(i, 0), w[i]) for i in range(5))
    b.close()
    for e in es:
        e.close()
