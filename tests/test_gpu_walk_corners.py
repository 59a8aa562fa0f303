"""Corners of the locate's walks, against the oracle (cells, statuses and walk
iterations exact; FP64 weights bit for bit): positions that are not numbers or
infinite, which the FP32 records must leave to the full evaluation, and cells
with a degenerate face, which may be looked at ahead of a walk and are an error
only where a walk comes to them."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

ODD = (np.nan, np.inf, -np.inf, 3.5e38, -1e300)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [400, 20_000, 150_000, (1 << 18) + 1])  # 16 and 4 lanes a particle, one, lines
@pytest.mark.parametrize("start", ["origin", "near"])
def test_positions_that_are_no_points(oracle, precision, n, start):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] odd positions", precision, n, start, flush=True)
    IM, JM, KM = 6, 7, 49
    coor = W.perturbed_cube(IM, JM, KM, seed=13, amp=0.3)
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    cell = None
    if start == "near":
        cell = np.clip(np.floor(pos * [IM, JM, KM]).astype(np.int64) + rng.integers(-1, 2, (n, 3)), 0,
                       [IM - 1, JM - 1, KM - 1])
    k = 0
    for a, v in enumerate(ODD):
        for axes in ((0,), (1,), (2,), (0, 1), (0, 1, 2)):
            for ax in axes:
                pos[5 + 7 * k, ax] = ODD[(a + ax) % len(ODD)] if len(axes) > 1 else v
            k += 1
    rc, rw, rs, rsteps = oracle.locate(IM, JM, KM, coor, pos, cell=cell)
    with PicGpu(precision=precision, collect_walk_stats=True) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_particles(pos, cell=cell, status=np.full(n, 4, np.int64))
        g.LocateAllParticlesInGrid()
        steps, d = g.walk_steps(), g.download_particles()
    np.testing.assert_array_equal(d["status"], rs)
    np.testing.assert_array_equal(d["cell"], rc)
    np.testing.assert_array_equal(steps, rsteps)
    ok = rs == 1
    if precision == "fp64":
        assert np.array_equal(d["weight"][ok], rw[ok], equal_nan=True)
    else:
        np.testing.assert_allclose(d["weight"][ok], rw[ok], atol=1e-5, rtol=0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [16, 20_000])  # 16 and 4 lanes a particle
def test_degenerate_cell_beyond_the_walks(oracle, precision, n):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] degenerate cell", precision, n, flush=True)
    IM, JM, KM = 5, 5, 50
    coor = W.uniform_grid(IM, JM, KM)
    nodes = coor.reshape(KM + 1, JM + 1, IM + 1, 3)
    nodes[31, 2:4, 2, :] = nodes[31, 2, 2, :]  # an edge of cells at k 30 and 31 in the middle collapses
    nodes[31, 2:4, 3, :] = nodes[31, 2, 2, :]  # and with it the faces between them
    rng = np.random.default_rng(n)
    pos = (np.array([2.5, 2.5, 0.0]) + rng.random((n, 3)) * [0.01, 0.01, 29.4]) / [IM, JM, KM]
    rc, rw, rs, rsteps = oracle.locate(IM, JM, KM, coor, pos)
    assert (rs == 1).all()
    with PicGpu(precision=precision, collect_walk_stats=True) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_particles(pos, status=np.full(n, 4, np.int64))
        g.LocateAllParticlesInGrid()  # no walk comes to the degenerate cells
        steps, d = g.walk_steps(), g.download_particles()
        np.testing.assert_array_equal(d["cell"], rc)
        np.testing.assert_array_equal(steps, rsteps)
        pos[n // 2, 2] = 30.5 / KM  # one does
        g.upload_particles(pos, status=np.full(n, 4, np.int64))
        with pytest.raises(L.PicgpuError, match="DEGENERATE"):
            g.LocateAllParticlesInGrid()
