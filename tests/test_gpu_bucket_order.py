"""Buckets of the particle index in PID order, whatever their size: cells of 1
to 700 particles, with PIDs that fit 32 bits and that do not, give the staged
path's averages of P and face sums bit for bit."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("sizes", [[1, 2, 7, 8, 9, 10, 15, 16, 17, 18, 63, 64, 65, 127, 128, 129, 700], list(range(18)),
                                   [12] * 64, [9, 0, 16, 0, 0, 30], [8, 9] * 100, [0, 17] * 40, [300]])
def test_averages_and_faces(precision, wide, sizes):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] bucket order", precision, wide, sizes, flush=True)
    dims = IM, JM, KM = (8, 4, 11)
    rng = np.random.default_rng(len(sizes))
    where = np.repeat(np.arange(len(sizes)), sizes)
    cell = np.stack([where % IM, where // IM % JM, where // (IM * JM)], axis=1).astype(np.int64)
    n = len(cell)
    order = rng.permutation(n)
    cell = cell[order]
    pos = (cell + 0.25 + 0.5 * rng.random((n, 3))) / dims
    pid = rng.permutation(n).astype(np.int64)
    if wide:
        pid += 1 << 40
    P = 101325.0 + rng.normal(size=n)
    ucat = rng.normal(size=((IM + 1) * (JM + 1) * (KM + 1) * 3))
    out = []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            g.upload_grid(IM, JM, KM, W.uniform_grid(IM, JM, KM))
            g.upload_ucat(ucat)
            g.upload_particles(pos, cell=cell, pid=pid, P=P)
            g.LocateAllParticlesInGrid()
            g.InterpolateAllFieldsToSwarm()
            g.AdvanceSimulation(1e-9, 3, rk2=True, deposit_cells=True, deposit_faces=True, staged=staged)
            out.append([g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)] +
                       [g.field(L.FIELD_IFACE + a) for a in range(3)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
