"""Walks from cell (0,0,0) through a long grid: several lanes a particle
(16, 4), the lines through LDS, walks ended by MAX_TRAVERSAL among the cells
looked ahead, and points on planes of the grid, which the FP32 filter
certifies nowhere along it; against the oracle (cells, statuses and walk
iterations exact; FP64 weights bit for bit, FP32 within 1e-5)."""
import numpy as np
import pytest

from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

IM, JM, KM = 5, 7, 53


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,cap", [(1, 1000), (3, 1000), (5, 1), (200, 2), (200, 17), (1021, 33), (16_384, 1000),
                                   (16_385, 1000), (16_390, 20), (131_072, 1000), (131_073, 1000),
                                   ((1 << 18) + 3, 1000)])
@pytest.mark.parametrize("grid", ["box", "cube"])
def test_walks_from_the_first_cell(oracle, precision, n, cap, grid):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] far walks", precision, n, cap, grid, flush=True)
    coor = W.uniform_grid(IM, JM, KM) if grid == "box" else W.perturbed_cube(IM, JM, KM, seed=8, amp=0.3)
    rng = np.random.default_rng(n + cap)
    pos = rng.random((n, 3)) * 1.02 - 0.01
    pos[3::41, 0] = 2 / IM  # on a plane of the box
    pos[4::41, 1] = 3 / JM + 1e-8
    pos[5::97] = [1e30, -1e30, 3e38]
    status = np.full(n, 4, np.int64)
    status[7::13] = 1  # skipped
    rc, rw, rs, rsteps = oracle.locate(IM, JM, KM, coor, pos, status=status, max_traversal=cap)
    with PicGpu(precision=precision, collect_walk_stats=True, max_traversal=cap) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_particles(pos, status=status)
        g.LocateAllParticlesInGrid()
        steps, d, st = g.walk_steps(), g.download_particles(), g.stats()
    walked = status != 1
    np.testing.assert_array_equal(d["status"], rs)
    np.testing.assert_array_equal(d["cell"][walked], rc[walked])
    np.testing.assert_array_equal(steps[walked], rsteps[walked])
    ok = walked & (rs == 1)
    if precision == "fp64":
        assert np.array_equal(d["weight"][ok].view(np.int64), rw[ok].view(np.int64))
    elif ok.any():
        assert np.abs(d["weight"][ok] - rw[ok]).max() < 1e-5
    assert st["located"] == ok.sum() and st["lost"] == (walked & (rs == 3)).sum()
    assert st["walk_iterations"] == rsteps[walked].sum() and st["walk_hist"].sum() == walked.sum()
