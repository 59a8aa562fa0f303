"""Walks from cell (0,0,0) that go through the LDS only while half of a
wavefront's lanes evaluate: few, half and most of the walks long, at the size
from which that form is used, against the oracle (cells, statuses and walk
iterations exact; FP64 weights bit for bit, FP32 within 1e-5)."""
import numpy as np
import pytest

from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

N = 1 << 18


def _grid(kind, rng):
    if kind == "tube":  # most walks leave the pipe after two or three iterations
        IM, JM, KM = 24, 24, 60
        th, rho, ph = rng.random(N), 0.99 * W.TUBE_A * np.sqrt(rng.random(N)), 2 * np.pi * rng.random(N)
        rr = W.TUBE_R + rho * np.cos(ph)
        a = -W.TUBE_SWEEP * th
        return IM, JM, KM, W.tube_grid(IM, JM, KM), np.stack([rr * np.cos(a), rr * np.sin(a), rho * np.sin(ph)], 1)
    IM, JM, KM = 9, 11, 37
    pos = rng.random((N, 3))
    near = rng.random(N) >= float(kind)
    pos[near] *= np.array([1 / IM, 1 / JM, 1 / KM])  # in or beside the first cell
    return IM, JM, KM, W.perturbed_cube(IM, JM, KM, seed=6, amp=0.3), pos


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["tube", "0.02", "0.5", "0.9"])
def test_few_and_many_long_walks(oracle, precision, kind):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] locate lines", precision, kind, flush=True)
    IM, JM, KM, coor, pos = _grid(kind, np.random.default_rng(12))
    rc, rw, rs, rsteps = oracle.locate(IM, JM, KM, coor, pos)
    with PicGpu(precision=precision, collect_walk_stats=True) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_particles(pos, status=np.full(N, 4, np.int64))
        g.LocateAllParticlesInGrid()
        steps, d = g.walk_steps(), g.download_particles()
    np.testing.assert_array_equal(d["status"], rs)
    np.testing.assert_array_equal(d["cell"], rc)
    np.testing.assert_array_equal(steps, rsteps)
    ok = rs == 1
    assert ok.any()
    if precision == "fp64":
        assert np.array_equal(d["weight"][ok].view(np.int64), rw[ok].view(np.int64))
    else:
        assert np.abs(d["weight"][ok] - rw[ok]).max() < 1e-5
