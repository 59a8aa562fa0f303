"""Steps of a lane a particle (few particles, or few a cell) and of a workgroup
a tile give the staged path's particles, faces, counts and averages bit for
bit, on both sides of the lines between them, over calls that compact, lose
particles through the boundary and start from particles without a cell."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(precision, dims, coor, ucat, pos, dt, rk2, faces, staged):
    from fdf_amd.swarm import PicGpu

    with PicGpu(precision=precision) as g:
        g.upload_grid(*dims, coor)
        g.upload_ucat(ucat)
        g.set_particle_volume(1e-6)
        rng = np.random.default_rng(1)
        pid = rng.permutation(len(pos)).astype(np.int64)
        g.upload_particles(pos, pid=pid, P=rng.random(len(pos)))
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        for steps in (1, 18, 2):
            g.AdvanceSimulation(dt, steps, rk2=rk2, deposit_cells=True, deposit_faces=faces, staged=staged)
        d = g.download_particles()
        order = np.argsort(d["pid"], kind="stable")
        out = {k: v[order] for k, v in d.items()}
        out["count"], out["P"] = g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)
        if faces:
            for a in range(3):
                out["face%d" % a] = g.field(L.FIELD_IFACE + a)
        return out


SIZES = [((9, 10, 7), 1), ((9, 10, 7), 700), ((12, 11, 10), 65_536), ((12, 11, 10), 65_600), ((48, 47, 50), 84_000),
         ((48, 47, 50), 85_200)]
FORMS = [(True, True), (False, False), (False, True), (True, False)]
# in the large grids the line differs with faces only
CASES = [(d, n, *f) for d, n in SIZES for f in FORMS] + [((104, 104, 100), n, True, True) for n in (540_000, 541_500)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,rk2,faces", CASES)
def test_matches_staged(precision, dims, n, rk2, faces):
    print("[gpu-case] sparse steps", precision, dims, n, rk2, faces, flush=True)
    coor = W.perturbed_cube(*dims, seed=4, amp=0.2)
    ucat = W.ucat_random_fourier(coor, *dims, seed=4, nmodes=8)
    pos = np.random.default_rng(n).random((n, 3)) * 1.02 - 0.01
    dt = 0.9 / max(dims) / float(np.abs(ucat).max())
    a = _run(precision, dims, coor, ucat, pos, dt, rk2, faces, False)
    b = _run(precision, dims, coor, ucat, pos, dt, rk2, faces, True)
    for k in b:
        assert np.array_equal(a[k], b[k]), k
