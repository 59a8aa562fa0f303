"""Crowded cells in PID order: sizes at which the stage-wise sort ranks a cell's
particles together and the step's index merges runs of 64 (65), a run's and a
merge's edges, runs without a partner, PIDs in order, nearly, in reverse and at
random, within 32 bits and beyond.  FP64 averages of P are numpy's sums in PID
order; both paths give the same averages and face sums bit for bit; the sorted
swarm lies by cell and PID."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = {"edges": [63, 64, 65, 66, 127, 128, 129, 130, 191, 192, 193, 255, 256, 257, 511, 512, 513, 514, 575, 576, 577, 1, 0, 5, 16, 17],
         "long": [1024, 1025, 2047, 4097, 6000, 640, 641, 0, 3], "many": [520] * 70 + [90] * 50}


def _pids(kind, n, where, rng):
    if kind == "random":
        return rng.permutation(n)
    if kind == "reverse":
        return np.arange(n)[::-1]
    p = np.arange(n)
    if kind == "nearly":  # in order but for neighbours up to 150 places apart, within and across runs
        p = np.argsort(np.arange(n) + rng.integers(0, 150, n) * (rng.random(n) < 0.2), kind="stable")
    return p


@pytest.mark.parametrize("precision,wide", [("fp64", False), ("fp64", True), ("fp32", False)])
@pytest.mark.parametrize("kind", ["random", "nearly", "order", "reverse"])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_long_buckets(precision, wide, kind, sizes):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] long buckets", precision, wide, kind, sizes, flush=True)
    dims = IM, JM, KM = (8, 4, 11)
    rng = np.random.default_rng(3)
    where = np.repeat(np.arange(len(SIZES[sizes])), SIZES[sizes])
    cell = np.stack([where % IM, where // IM % JM, where // (IM * JM)], axis=1).astype(np.int64)
    n = len(cell)
    pos = (cell + 0.25 + 0.5 * rng.random((n, 3))) / dims
    pid = np.ascontiguousarray(_pids(kind, n, where, rng)).astype(np.int64) + ((1 << 40) if wide else 0)
    P = 101325.0 + rng.normal(size=n)
    ucat = rng.normal(size=((IM + 1) * (JM + 1) * (KM + 1) * 3))
    out = []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            g.upload_grid(*dims, W.uniform_grid(*dims))
            g.upload_ucat(ucat)
            g.upload_particles(pos, cell=cell, pid=pid, P=P)
            g.LocateAllParticlesInGrid()
            g.InterpolateAllFieldsToSwarm()
            g.AdvanceSimulation(1e-9, 2, rk2=True, deposit_cells=True, deposit_faces=True, staged=staged)
            out.append([g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)] +
                       [g.field(L.FIELD_IFACE + a) for a in range(3)])
            if staged:
                d = g.download_particles()
                lin = d["cell"][:, 0] + IM * (d["cell"][:, 1] + JM * d["cell"][:, 2])
                assert np.array_equal(np.lexsort((d["pid"], lin)), np.arange(n))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    if precision == "fp64":
        avg = out[0][1].reshape(KM + 1, JM + 1, IM + 1)
        for k, m in enumerate(SIZES[sizes]):
            sel = np.flatnonzero(where == k)
            sel = sel[np.argsort(pid[sel])]
            want = np.cumsum(P[sel])[-1] / m if m else 0.0
            assert avg[k // (IM * JM), k // IM % JM, k % IM] == want, k
