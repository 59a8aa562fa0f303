"""Host arrays to and from the device: sizes around a chunk's end, odd tails,
the reuse of slots and the helper threads, every kind of array; whole numbers
and FP64 arrays bit for bit, FP32 ones rounded once."""
import threading

import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

IM, JM, KM = 7, 6, 5
CHUNK = 128 << 10  # the smallest chunk


def _swarm(n, seed):
    rng = np.random.default_rng(seed)
    return {"pos": rng.standard_normal((n, 3)), "vel": rng.standard_normal((n, 3)), "weight": rng.random((n, 3)),
            "cell": rng.integers(-1, [IM + 1, JM + 1, KM + 1], (n, 3)), "status": rng.integers(0, 5, n),
            "pid": rng.integers(-2 ** 62, 2 ** 62, n)}


def _check(d, s, precision):
    inside = ((s["cell"] >= 0) & (s["cell"] < [IM, JM, KM])).all(1)
    np.testing.assert_array_equal(d["cell"], np.where(inside[:, None], s["cell"], -1))
    for k in ("status", "pid", "pos"):
        np.testing.assert_array_equal(d[k], s[k])
    for k in ("vel", "weight"):
        want = s[k] if precision == "fp64" else s[k].astype(np.float32).astype(np.float64)
        np.testing.assert_array_equal(d[k], want)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 2, 3, CHUNK // 24 - 1, CHUNK // 24 + 1, CHUNK // 8, CHUNK // 8 + 1, 100_003, 700_001])
def test_round_trip(precision, n):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] transfer", precision, n, flush=True)
    s = _swarm(n, n)
    with PicGpu(precision=precision) as g:
        g.upload_grid(IM, JM, KM, W.uniform_grid(IM, JM, KM))
        g.upload_particles(s["pos"], vel=s["vel"], cell=s["cell"], weight=s["weight"], status=s["status"],
                           pid=s["pid"])
        _check(g.download_particles(), s, precision)
        s2 = _swarm(n, n + 1)  # again, over the first swarm, and without the optional arrays
        g.upload_particles(s2["pos"], cell=s2["cell"], status=s2["status"], pid=s2["pid"])
        s2["vel"], s2["weight"] = np.zeros((n, 3)), np.zeros((n, 3))
        _check(g.download_particles(), s2, precision)


def test_two_contexts_in_two_threads():
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] transfer from two threads", flush=True)
    out = {}

    def work(k):
        s = _swarm(300_000 + k, k)
        with PicGpu(precision="fp32" if k else "fp64") as g:
            g.upload_grid(IM, JM, KM, W.uniform_grid(IM, JM, KM))
            for _ in range(3):
                g.upload_particles(s["pos"], vel=s["vel"], cell=s["cell"], weight=s["weight"], status=s["status"],
                                   pid=s["pid"])
                out[k] = (g.download_particles(), s)

    ts = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for k in (0, 1):
        _check(*out[k], "fp32" if k else "fp64")


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 4, 5), (61, 53, 47), (128, 96, 100)])
def test_fields(oracle, precision, dims):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] fields", precision, dims, flush=True)
    I, J, K = dims
    n = 3 * I * J * K
    rng = np.random.default_rng(n)
    coor = W.uniform_grid(I, J, K)
    with PicGpu(precision=precision) as g:
        g.upload_grid(I, J, K, coor)
        g.upload_ucat(rng.standard_normal(3 * (I + 1) * (J + 1) * (K + 1)))
        g.upload_particles(rng.random((n, 3)))
        g.set_particle_volume(1e-9)
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        g.ScatterAllParticleFieldsToEulerFields()
        g.DepositParticlesToFaces(1e-9)
        d = g.download_particles()
        cnt, avg = g.field(L.FIELD_PARTICLE_COUNT), g.field(L.FIELD_P_AVERAGE)
        face = [g.field(L.FIELD_IFACE + a) for a in range(3)]
        frac = [g.field(L.FIELD_IFACE_VOLFRAC + a) for a in range(3)]
    ref = np.zeros((K + 1, J + 1, I + 1))
    np.add.at(ref, (d["cell"][:, 2], d["cell"][:, 1], d["cell"][:, 0]), 1.0)
    np.testing.assert_array_equal(cnt.reshape(-1), ref.reshape(-1))
    np.testing.assert_array_equal(avg.reshape(-1) > 0, ref.reshape(-1) > 0)
    for a in range(3):
        r = np.asarray(oracle.face_volfrac(I, J, K, coor, a, face[a], 1e-9)).reshape(-1)
        np.testing.assert_array_equal(frac[a].reshape(-1), r)
