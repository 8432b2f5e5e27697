"""CMM exchange by message blocks (exchange mode 1).  Subdomains are windows of
one array per field, so a block is unpacked into the cells it was packed
from: with DDX_CMM_CHECK=1 those are overwritten with NaN in between, and
whatever a block does not bring shows."""
import numpy as np
import pytest

import ddx
import pyoracle as po
from cases import case, random_fields

pytestmark = pytest.mark.gpu

BATCHES = [(ddx.VX, ddx.VY, ddx.VZ), (ddx.SXX, ddx.SYY, ddx.SZZ, ddx.SXY, ddx.SXZ, ddx.SYZ),
           (ddx.SXX, ddx.SYY, ddx.SZZ, ddx.SXY, ddx.SXZ, ddx.SYZ, ddx.SAU)]
# layers a subdomain receives at its (z lo, z hi, y lo, y hi, x lo, x hi) side: the reach of the staggered 8th-order
# differences that read the field across it (PHY/fdtd3d_phy_mpi_1_host_meat.hpp:31-42)
WIDTHS = {ddx.VX: (3, 4, 3, 4, 4, 3), ddx.VY: (3, 4, 4, 3, 3, 4), ddx.VZ: (4, 3, 3, 4, 3, 4),
          ddx.SXX: (0, 0, 0, 0, 3, 4), ddx.SYY: (0, 0, 3, 4, 0, 0), ddx.SZZ: (3, 4, 0, 0, 0, 0),
          ddx.SXY: (0, 0, 4, 3, 4, 3), ddx.SXZ: (4, 3, 0, 0, 4, 3), ddx.SYZ: (4, 3, 4, 3, 0, 0),
          ddx.SAU: (3, 4, 3, 4, 3, 4)}


def engine(c, divide, storage, monkeypatch, check):
    monkeypatch.setenv("DDX_CMM_CHECK", str(check))
    e = ddx.Engine(ddx.make_desc(c["nx"], c["ny"], c["nz"], c["dx"], c["pml"], c["dt"], c["fm"], c["ntime"],
                                 divide=divide, rec_width=c["rec_width"], cfl_policy=1, storage=storage))
    e.set_model(c["vp"], c["vs"], c["rho"])
    e.set_wavelet(po.ricker(c["fm"], c["dt"], c["ntime"]))
    e.set_geometry(c["shots"], c["recv"])
    return e


@pytest.mark.parametrize("storage", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("divide", [(2, 2, 1), (3, 2, 2)])
def test_message_blocks_bring_every_boundary_layer(divide, storage, monkeypatch):
    """One exchange of each batch leaves every field as it was (no layer lost,
    none in another's place) and moves the batch's boundary layers, each read
    and written by the pack and by the unpack."""
    c = case(nx=40, ny=34, nz=30, ntime=10)
    e = engine(c, divide, storage, monkeypatch, 1)
    e.set_exchange(1)
    subs = [ddx.subdomain(e.desc, r) for r in range(int(np.prod(divide)))]
    for s in (0, 1):
        for f, arr in enumerate(random_fields(e.ext_shape, seed=31 + s)):
            e.set(s, f, arr)
        before = [e.get(s, f) for f in range(13)]
        for b, fields in enumerate(BATCHES):
            e.profile(4)
            e.halo_exchange(s, b)
            moved = e.class_time(4)[2]
            e.profile(-2)
            cells = 0
            for sub in subs:
                n = sub["ext_n"]
                for side, axis in enumerate((2, 2, 1, 1, 0, 0)):
                    if sub["neighbour"][side] >= 0:
                        face = n[(axis + 1) % 3] * n[(axis + 2) % 3]
                        cells += face * sum(WIDTHS[f][side] for f in fields)
            assert moved == 4 * (4 if storage == "fp32" else 2) * cells, (s, b)
            for f in range(13):
                assert np.array_equal(e.get(s, f), before[f]), (s, b, ddx.FIELD_NAMES[f])
    e.close()


@pytest.mark.parametrize("storage", ["fp32", "bf16"])
def test_shots_through_message_blocks(storage, monkeypatch):
    """Seismograms and RTM images through the blocks, ghosts overwritten
    before each unpack, equal those without an exchange; alone and batched."""
    c = case(nx=40, ny=34, nz=30, ntime=30, rec_width=2)
    outs = []
    for mode in (0, 1):
        es = [engine(c, d, storage, monkeypatch, mode) for d in ((2, 2, 1), (1, 2, 2))]
        out = []
        for e in es:
            e.set_exchange(mode)
            e.model_shot(0)
            out.append(e.seismograms(0))
        ddx.model_batch(es)
        out += [e.seismograms(0) for e in es]
        es[0].rtm_shot(0)
        out += [es[0].image(q, r) for q in range(5) for r in range(4)]
        ddx.rtm_batch(es)
        out += [e.image(q, r) for e in es for q in range(5) for r in range(4)]
        for e in es:
            e.close()
        outs.append(out)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
