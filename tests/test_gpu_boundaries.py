"""The boundary handlers of all faces in one launch, and face by face where an
axis has fewer than four planes, leave what the sweep over faces 0..5 leaves:
every mix of handlers, edges and corners included, from fields that hold
values everywhere; against the oracle, bit for bit."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W
from fdf_amd.boundary import BoundaryConfig

pytestmark = pytest.mark.gpu

FACES = ["-Xi", "+Xi", "-Eta", "+Eta", "-Zeta", "+Zeta"]
KINDS = [("WALL", "noslip"), ("NOGRAD", "allcopy"), ("INLET", "constant_velocity"), ("INLET", "parabolic")]


def _config(rng):
    cfg = BoundaryConfig()
    for f in FACES:
        t, h = KINDS[rng.integers(len(KINDS))]
        kw = {}
        if h == "constant_velocity":
            kw = dict(zip(("vx", "vy", "vz"), rng.normal(size=3)))
        elif h == "parabolic":  # writes nothing on an i- or j-face
            kw = dict(vmax=float(rng.uniform(0.5, 2)))
        cfg.set_face(f, t, h, **kw)
    return cfg


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(2, 2, 2), (2, 5, 6), (3, 3, 3), (5, 3, 2), (3, 4, 9), (17, 6, 5)])
@pytest.mark.parametrize("seed", range(6))
def test_sweep_over_the_faces(oracle, precision, dims, seed):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] boundaries", precision, dims, seed, flush=True)
    rng = np.random.default_rng([seed, *dims])
    coor = W.perturbed_cube(*dims, seed=seed, amp=0.1)
    cfg = _config(rng)
    csi, eta, zet, aj, ori = oracle.metrics(*dims, coor)
    ucat, ucont = rng.normal(size=(len(csi), 3)), rng.normal(size=(len(csi), 3))
    with PicGpu(precision=precision) as g:
        g.upload_grid(*dims, coor)
        g.compute_metrics()
        g.BoundarySystem_Create(cfg)
        g.upload_ucat(ucat)
        g.upload_ucont(ucont)
        g.SetEulerianFields(1)
        got = g.field(L.FIELD_UCAT), g.field(L.FIELD_UCONT)
    oracle.set_eulerian_fields(*dims, cfg, csi, eta, zet, 1, 0, (0.0, 0.0, 0.0), ori, ucat, ucont)
    assert np.array_equal(got[0].ravel(), ucat.ravel()), "ucat"
    assert np.array_equal(got[1].ravel(), ucont.ravel()), "ucont"
