"""The steps of a workgroup a tile, over calls that each start with enough
particles to take them, against the staged path bit for bit: start states
recomputed, in-step deposition, deferred particles beside the seams, the
compaction inside a call, crowded tiles, long walks.  Each call says which path
it took: only the tiles' steps launch k_step_deferred under its own name."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

FACES = (L.FIELD_IFACE, L.FIELD_JFACE, L.FIELD_KFACE)


def _advance(g, dt, steps, tiles, **kw):
    """One call; tiles: whether its steps go by tiles (None: not looked at)."""
    if tiles is None:
        return g.AdvanceSimulation(dt, steps, **kw)
    g.timing_reset()
    g.timing(True)
    g.timing_select("step_deferred")
    g.AdvanceSimulation(dt, steps, **kw)
    assert (g.timing_query("step_deferred")[1] > 0) == tiles, (g.n, tiles)
    g.timing(False)


def _start(g, dims, coor, ucat, pos, pid=None, P=None):
    g.upload_grid(*dims, coor)
    g.upload_ucat(ucat)
    g.set_particle_volume(1e-6)
    g.upload_particles(pos, pid=pid, P=P)
    g.LocateAllParticlesInGrid()
    g.InterpolateAllFieldsToSwarm()


def _result(g, faces):
    d = g.download_particles()
    o = np.argsort(d["pid"], kind="stable")
    out = {k: v[o] for k, v in d.items()}
    out["count"], out["P"] = g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)
    for a, f in enumerate(FACES if faces else ()):
        out["face%d" % a] = g.field(f)
    return out


def _same(a, b):
    assert a.keys() == b.keys()
    for k in b:
        assert np.array_equal(a[k], b[k]), k


def _workload(dims, n, seed, cells_a_step):
    coor = W.perturbed_cube(*dims, seed=seed, amp=0.2)
    ucat = W.ucat_random_fourier(coor, *dims, seed=seed, nmodes=8)
    rng = np.random.default_rng(n)
    return coor, ucat, rng.random((n, 3)) * 1.02 - 0.01, cells_a_step / max(dims) / float(np.abs(ucat).max()), rng


FORMS = [(True, True), (False, False), (False, True), (True, False)]
CASES = [(d, n, *f) for d, n in (((12, 11, 10), 150_000), ((48, 47, 50), 130_000)) for f in FORMS] + \
    [((104, 104, 100), 900_000, True, True), ((104, 104, 100), 900_000, True, False)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,rk2,faces", CASES)
def test_matches_staged(precision, dims, n, rk2, faces):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] tile steps", precision, dims, n, rk2, faces, flush=True)
    coor, ucat, pos, dt, rng = _workload(dims, n, 4, 0.2)
    pid, P = rng.permutation(n).astype(np.int64), rng.random(n)
    out = []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos, pid, P)
            for steps in (1, 18, 2):
                _advance(g, dt, steps, None if staged else True, rk2=rk2, deposit_cells=True, deposit_faces=faces,
                         staged=staged)
            out.append(_result(g, faces))
    _same(*out)


@pytest.mark.parametrize("precision,faces,line", [("fp64", False, 0.6), ("fp64", True, 0.5), ("fp32", False, 0.75),
                                                  ("fp32", True, 0.5)])
def test_line_in_large_grids(precision, faces, line):
    """Both sides of the line between lists and tiles in a grid of more than
    4096 tiles, on particles that stay: which path runs, and the staged path's results."""
    from fdf_amd.swarm import PicGpu

    dims = (104, 104, 100)
    ncell = 104 * 104 * 100
    print("[gpu-case] sparse line", precision, faces, line, flush=True)
    coor, ucat, _, dt, _ = _workload(dims, 1, 4, 0.1)
    for n, tiles in ((int(line * ncell) - 1, False), (int(line * ncell) + 1, True)):
        pos = 0.02 + 0.96 * np.random.default_rng(n).random((n, 3))
        out = []
        for staged in (False, True):
            with PicGpu(precision=precision) as g:
                _start(g, dims, coor, ucat, pos)
                _advance(g, dt, 2, None if staged else tiles, rk2=True, deposit_cells=True, deposit_faces=faces,
                         staged=staged)
                out.append(_result(g, faces))
        _same(*out)
