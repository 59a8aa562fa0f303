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


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,faces,tiles", [
    ((5, 4, 3), 420, True, False), ((5, 4, 3), 421, True, True), ((5, 4, 3), 20_000, False, False),
    ((24, 23, 17), 65_536, True, False), ((24, 23, 15), 65_536, True, True), ((1, 1, 1), 7, True, False),
    ((1, 1, 1), 8, True, True), ((1, 1, 1), 3_000, False, None), ((2, 1, 1), 3_000, False, False)])
def test_line_for_few_particles(precision, dims, n, faces, tiles):
    """Up to 65,536 particles: the list with faces up to seven a cell, without
    them always but in a single cell in FP32; the staged path's results."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] few particles", precision, dims, n, faces, flush=True)
    tiles = precision == "fp32" if tiles is None else tiles
    coor, ucat, _, dt, _ = _workload(dims, 1, 4, 0.01)
    pos = 0.1 + 0.8 * np.random.default_rng(n).random((n, 3))
    out = []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos)
            _advance(g, dt, 2, None if staged else tiles, rk2=True, deposit_cells=True, deposit_faces=faces,
                     staged=staged)
            out.append(_result(g, faces))
    _same(*out)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_crowded_tiles_with_fast_particles(oracle, precision):
    """Tiles of over ten thousand particles, most of which change cell in a step:
    queues and staged results overflow, walks are handed over and go on.  FP64:
    also the oracle's particles bit for bit."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] crowded tiles", precision, flush=True)
    dims, n, nsteps = (16, 16, 8), 110_000, 3
    coor = W.perturbed_cube(*dims, seed=31, amp=0.15)
    ucat = W.ucat_random_fourier(coor, *dims, seed=32)
    pos = 0.05 + 0.9 * np.random.default_rng(33).random((n, 3))
    dt = 1.5 / (np.abs(ucat).max() * max(dims))  # up to about 1.5 cells a step
    out = []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos)
            _advance(g, dt, nsteps, None if staged else True, rk2=True, deposit_cells=True, deposit_faces=True,
                     staged=staged)
            out.append(_result(g, True))
    _same(*out)
    if precision == "fp64":
        corner = oracle.center_to_corner(*dims, ucat)
        c, w, st, _ = oracle.locate(*dims, coor, pos, status=np.full(n, 4, np.int64))
        s = {"pos": pos.copy(), "vel": oracle.interp(*dims, corner, c, w), "cell": c, "weight": w, "status": st,
             "pid": np.arange(n, dtype=np.int64), "P": np.full(n, 101325.0)}
        for _ in range(nsteps):
            oracle.step(*dims, coor, corner, s, dt, rk2=True)
        for k in ("pid", "cell", "pos", "vel", "weight", "status"):
            assert np.array_equal(out[0][k], s[k]), k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_long_call_matches_staged(precision):
    """Twenty steps in one call, which compacts in its middle: the staged path's
    particles, deposits, processed particles and walk iterations."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] long tile call", precision, flush=True)
    dims, n = (24, 20, 40), 160_000
    coor, ucat, pos, dt, _ = _workload(dims, n, 7, 0.5)
    out, st = [], []
    for staged in (False, True):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos)
            _advance(g, dt, 20, None if staged else True, rk2=True, deposit_cells=True, deposit_faces=True,
                     staged=staged)
            out.append(_result(g, True))
            st.append(g.stats())
    _same(*out)
    assert st[0]["particle_steps"] == st[1]["particle_steps"]
    assert st[0]["walk_iterations"] == st[1]["walk_iterations"]
    assert 0 < len(out[0]["pid"]) < n


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_single_step_calls_match_one_call_twice(precision):
    """Twenty one-step calls, the compaction falling inside the sequence, give
    what one twenty-step call gives, and that gives it again, bit for bit."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] single tile steps", precision, flush=True)
    dims, n = (16, 16, 8), 200_000
    coor, ucat, pos, dt, _ = _workload(dims, n, 71, 0.3)
    out = []
    for calls in ([20], [1] * 20, [20]):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos)
            for k in calls:
                _advance(g, dt, k, True, rk2=True, deposit_cells=True, deposit_faces=True)
            live = g.n
            out.append(_result(g, True))
            assert live == len(out[-1]["pid"])
    _same(out[0], out[1])
    _same(out[0], out[2])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_faces_of_start_in_sparse_grids(precision):
    """With the faces of the last step's start the steps stay with the tiles at
    any number of particles: the end state of a call without that option, and
    the faces of one that ends a step before."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] faces of start", precision, flush=True)
    dims, n = (20, 18, 16), 3_000
    coor, ucat, pos, dt, _ = _workload(dims, n, 9, 0.5)
    out = []
    for steps, kw, tiles in ((5, dict(faces_of_start=True), True), (5, {}, False), (4, {}, False)):
        with PicGpu(precision=precision) as g:
            _start(g, dims, coor, ucat, pos)
            _advance(g, dt, steps, tiles, rk2=True, deposit_cells=True, deposit_faces=True, **kw)
            out.append(_result(g, True))
    for k in out[1]:
        assert np.array_equal(out[0][k], out[2][k] if k.startswith("face") else out[1][k]), k
