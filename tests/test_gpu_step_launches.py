"""The passes around the fused step's kernel at the edges of their launches,
against the oracle: the node velocities at every chunk length and remainder,
and the bucket order with its P averages over buckets of zero, one, up to
eight and more particles (FP64 bit for bit; FP32 within 1e-5)."""
import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("IM,JM,KM", [(1, 1, 1), (2, 3, 700), (15, 15, 3), (15, 16, 129), (96, 96, 61), (200, 170, 256)])
def test_node_velocities(oracle, precision, IM, JM, KM):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] node velocities", precision, IM, JM, KM, flush=True)
    coor = W.uniform_grid(IM, JM, KM)
    ucat = np.random.default_rng(IM + KM).standard_normal(3 * (IM + 1) * (JM + 1) * (KM + 1))
    with PicGpu(precision=precision) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_ucat(ucat)
        g.upload_particles(np.array([[0.5, 0.5, 0.5]]))
        g.InterpolateAllFieldsToSwarm()
        got = g.field(L.FIELD_CORNER_VELOCITY)
    ref = np.asarray(oracle.center_to_corner(IM, JM, KM, ucat)).reshape(-1)
    if precision == "fp64":
        assert np.array_equal(got.view(np.int64), ref.view(np.int64))
    else:
        # eight roundings of sums of at most 8 |u|
        assert np.abs(got - ref).max() <= 16 * 2.0 ** -24 * 8 * np.abs(ucat).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("per_cell", [0.3, 1, 7, 9, 40])
def test_bucket_order_and_averages(oracle, precision, wide, per_cell):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] bucket order", precision, wide, per_cell, flush=True)
    IM, JM, KM = 9, 5, 7
    n = int(per_cell * IM * JM * KM)
    rng = np.random.default_rng(n)
    coor = W.perturbed_cube(IM, JM, KM, seed=3, amp=0.2)
    ucat = W.ucat_random_fourier(coor, IM, JM, KM, seed=4)
    dt = 0.3 / (np.abs(ucat).max() * max(IM, JM, KM))
    pos = 0.05 + 0.9 * rng.random((n, 3))
    pid = rng.permutation(n).astype(np.int64) + ((1 << 33) if wide else 0)
    P = 101325.0 + 50.0 * rng.random(n)
    with PicGpu(precision=precision) as g:
        g.upload_grid(IM, JM, KM, coor)
        g.upload_ucat(ucat)
        g.upload_particles(pos, pid=pid, P=P)
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        g.AdvanceSimulation(dt, 3, deposit_cells=True, deposit_faces=True)
        d = g.download_particles()
        cnt, avg = g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)
        faces = [g.field(f) for f in (L.FIELD_IFACE, L.FIELD_JFACE, L.FIELD_KFACE)]
    value = np.empty(n)
    value[pid - pid.min()] = P
    ref_cnt = oracle.count_cells(IM, JM, KM, d["cell"])
    Pd = value[d["pid"] - pid.min()]
    if precision == "fp32":
        Pd = Pd.astype(np.float32).astype(np.float64)
    ref = oracle.scatter_P(IM, JM, KM, d["cell"], Pd, d["pid"], ref_cnt)
    refs = oracle.deposit_faces(IM, JM, KM, d["cell"], d["weight"], d["vel"], d["pid"])
    assert np.array_equal(cnt, ref_cnt)
    if precision == "fp64":
        assert np.array_equal(avg, ref)
        assert all(np.array_equal(a, b) for a, b in zip(faces, refs))
    else:
        assert np.abs(avg - ref).max() <= 1e-5 * 101375.0
        for a, b in zip(faces, refs):
            assert np.abs(a - b).max() <= 1e-5 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n,crowd", [(1, 0), (300, 0), (257, 257), (6000, 3000)])
def test_stage_sort(oracle, precision, wide, n, crowd):
    """The stage-wise sort: cells in order, PIDs in order within a cell (also
    with `crowd` particles in one cell), the particles without a cell after
    them; the averages and face sums of that swarm."""
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] stage sort", precision, wide, n, crowd, flush=True)
    IM, JM, KM = 9, 5, 7
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    pos[:crowd] = (np.array([4, 2, 3]) + rng.random((crowd, 3))) / [IM, JM, KM]
    pos[crowd + 3::11] += 2.0  # outside: no cell
    pid = rng.permutation(n).astype(np.int64) * 3 + ((1 << 33) if wide else 0)
    P = 101325.0 + 50.0 * rng.random(n)
    with PicGpu(precision=precision) as g:
        g.upload_grid(IM, JM, KM, W.uniform_grid(IM, JM, KM))
        g.upload_ucat(rng.standard_normal(3 * (IM + 1) * (JM + 1) * (KM + 1)))
        g.upload_particles(pos, pid=pid, P=P)
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        before = g.download_particles()
        g.ScatterAllParticleFieldsToEulerFields()
        g.DepositParticlesToFaces(1e-9)
        d = g.download_particles()
        avg = g.field(L.FIELD_P_AVERAGE)
        faces = [g.field(f) for f in (L.FIELD_IFACE, L.FIELD_JFACE, L.FIELD_KFACE)]
    flat = lambda c: np.where(c[:, 0] < 0, 1 << 40, c[:, 0] + IM * (c[:, 1] + JM * c[:, 2]))  # noqa: E731
    fb = flat(before["cell"])
    order = np.lexsort((np.where(fb < 1 << 40, before["pid"], np.arange(n)), fb))
    for k in d:
        np.testing.assert_array_equal(d[k], before[k][order])
    at = d["cell"][:, 0] >= 0
    c, w, v, ids = d["cell"][at], d["weight"][at], d["vel"][at], d["pid"][at]
    Pd = np.empty(3 * n)
    Pd[pid - pid.min()] = P
    Pd = Pd[ids - pid.min()]
    if precision == "fp32":
        Pd = Pd.astype(np.float32).astype(np.float64)
    ref = oracle.scatter_P(IM, JM, KM, c, Pd, ids, oracle.count_cells(IM, JM, KM, c))
    refs = oracle.deposit_faces(IM, JM, KM, c, w, v, ids)
    if precision == "fp64":
        assert np.array_equal(avg, ref)
        assert all(np.array_equal(a, b) for a, b in zip(faces, refs))
    else:
        assert np.abs(avg - ref).max() <= 1e-5 * 101375.0
        for a, b in zip(faces, refs):  # n terms of at most |v|, one rounding each
            assert np.abs(a - b).max() <= max(1e-5, n * 2.0 ** -24) * max(1.0, np.abs(b).max())
