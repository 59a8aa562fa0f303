"""The locate kernel at the edges of its launch: particles per wavefront, the
lanes' refill, the FP32 filter of the FP64 walk and the FP64 evaluation's
lane groups, against the oracle (cells, statuses and walk iterations exact;
FP64 weights bit for bit, FP32 within 1e-5)."""
import numpy as np
import pytest

from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

IM, JM, KM = 11, 9, 21


def _points(n, coor, rng):
    """Points in and around the grid, some where the filter certifies nothing:
    on nodes, on edge and face centres, and far outside float range."""
    p = rng.random((n, 3)) * 1.1 - 0.05
    nodes = coor.reshape(KM + 1, JM + 1, IM + 1, 3)
    for t in range(0, n, 7):
        k, j, i = rng.integers(0, KM), rng.integers(0, JM), rng.integers(0, IM)
        b = nodes[k:k + 2, j:j + 2, i:i + 2].reshape(8, 3)
        p[t] = [b[0], 0.5 * (b[0] + b[1]), 0.25 * (b[0] + b[1] + b[2] + b[3])][t % 3]
    p[5::97] = [1e30, -1e30, 3e38]
    p[6::97] = [0.5, 1e200, 0.5]
    return p


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000, 4096 * 16 + 1, 300_001])
@pytest.mark.parametrize("start", ["origin", "near"])
def test_locate_sizes(oracle, precision, n, start):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] locate sizes", precision, n, start, flush=True)
    coor = W.perturbed_cube(IM, JM, KM, seed=21, amp=0.3)
    rng = np.random.default_rng(n)
    pos = _points(n, coor, rng)
    cell = None
    if start == "near":
        cell = np.clip(np.floor(np.clip(pos, 0, 1) * [IM, JM, KM]).astype(np.int64) + rng.integers(-2, 3, (n, 3)), -1,
                       [IM - 1, JM - 1, KM - 1])
    status = np.zeros(n, np.int64)
    status[3::11] = 1  # skipped
    rc, rw, rs, rsteps = oracle.locate(IM, JM, KM, coor, pos, cell=cell, status=status)
    with PicGpu(precision=precision, collect_walk_stats=True) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_particles(pos, cell=cell, status=status)
        g.LocateAllParticlesInGrid()
        steps, d, st = g.walk_steps(), g.download_particles(), g.stats()
    np.testing.assert_array_equal(d["status"], rs)
    walked = status != 1
    np.testing.assert_array_equal(d["cell"][walked], rc[walked])
    np.testing.assert_array_equal(steps[walked], rsteps[walked])
    ok = walked & (rs == 1)
    if precision == "fp64":
        assert np.array_equal(d["weight"][ok].view(np.int64), rw[ok].view(np.int64))
    elif ok.any():
        assert np.abs(d["weight"][ok] - rw[ok]).max() < 1e-5
    assert st["located"] == ok.sum() and st["lost"] == (walked & (rs == 3)).sum()
    assert st["walk_iterations"] == rsteps[walked].sum() and st["walk_hist"].sum() == walked.sum()
