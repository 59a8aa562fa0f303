"""Checks of tests/test_gpu_alloc.py, each run in a process of its own with
tests/alloc_shim.c between libpicgpu.so and the HIP runtime's allocations:
alloc_child.py SHIM CHECK [ARGUMENT...]."""
import ctypes as C
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library
shim.shim_limit.argtypes = [C.c_int64]
for _f in ("shim_used", "shim_peak", "shim_host_calls"):
    getattr(shim, _f).restype = C.c_int64
shim.shim_host_flags.restype = C.c_uint

import numpy as np  # noqa: E402

from fdf_amd import _lib as L  # noqa: E402
from fdf_amd import workloads as W  # noqa: E402
from fdf_amd.swarm import PicGpu  # noqa: E402


def coherent():
    """The slots that kernels and host threads share are coherent by their own flag."""
    with PicGpu(precision="fp64") as g:
        g.upload_grid(4, 4, 4, W.uniform_grid(4, 4, 4))
        g.upload_particles(np.full((100, 3), 0.5))
        assert (g.download_particles()["pos"] == 0.5).all()
    assert shim.shim_host_calls() >= 1
    assert shim.shim_host_flags() & 0x40000000, hex(shim.shim_host_flags())  # hipHostMallocCoherent


def no_pinned(precision, n):
    """Every kind of array, up and down, when pinned memory is refused: what a
    context with pinned slots gives, bit for bit."""
    n, (IM, JM, KM) = int(n), (23, 19, 31)
    rng = np.random.default_rng(n)
    coor = W.perturbed_cube(IM, JM, KM, seed=2)
    a = {"vel": rng.standard_normal((n, 3)), "weight": rng.random((n, 3)),
         "cell": rng.integers(-1, [IM + 1, JM + 1, KM + 1], (n, 3)), "status": rng.integers(0, 5, n),
         "pid": rng.permutation(n) - n // 2, "P": rng.random(n)}
    pos = rng.random((n, 3))
    ucat = rng.standard_normal(3 * (IM + 1) * (JM + 1) * (KM + 1))
    out = []
    for refuse in (0, 1):
        shim.shim_refuse_host(refuse)
        with PicGpu(precision=precision) as g:
            g.upload_grid(IM, JM, KM, coor)
            g.upload_ucat(ucat)
            g.upload_particles(pos, **a)
            d = [g.download_particles()]
            g.upload_particles(pos, pid=a["pid"])
            g.LocateAllParticlesInGrid()
            g.InterpolateAllFieldsToSwarm()
            g.ScatterAllParticleFieldsToEulerFields()
            g.DepositParticlesToFaces(1e-9)
            d.append(g.download_particles())
            d[1]["fields"] = np.concatenate([g.field(w).reshape(-1) for w in range(9)])
            out.append(d)
    assert shim.shim_host_calls() >= 2
    for x, y in zip(*out):
        for k in x:
            assert x[k].tobytes() == y[k].tobytes(), k


def _swarm(g, n, IM, JM, KM, fused):
    """A swarm through the sort's consumers (or the fused steps), some of it
    outside the grid; what the sort returns in its order, the steps' by PID."""
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3)) * 1.04 - 0.02
    g.upload_particles(pos, pid=rng.permutation(n).astype(np.int64), P=rng.random(n))
    g.LocateAllParticlesInGrid()
    g.InterpolateAllFieldsToSwarm()
    if fused:
        g.AdvanceSimulation(2e-4, 3, rk2=True, deposit_cells=True, deposit_faces=True)
    else:
        g.ScatterAllParticleFieldsToEulerFields()
        g.DepositParticlesToFaces(1e-9)
    d = g.download_particles()
    if fused:
        o = np.argsort(d["pid"], kind="stable")
        d = {k: v[o] for k, v in d.items()}
    d["fields"] = np.concatenate([g.field(w).reshape(-1) for w in range(9)])
    return d


def tight(precision, fused):
    """Calls that take the sort's records and the FP64 filter where there is
    memory do with what they need: a small swarm, which leaves room for them,
    then a large one, which needs it back; the results are the same bits."""
    fused, (IM, JM, KM) = fused == "fused", (24, 24, 40)
    small, large = 5_000, 90_000
    coor = W.perturbed_cube(IM, JM, KM, seed=3)
    ucat = W.ucat_random_fourier(coor, IM, JM, KM, seed=3, nmodes=4)
    spares = 32 * large + (128 * IM * JM * KM if precision == "fp64" else 0)

    def run():
        shim.shim_peak_reset()
        with PicGpu(precision=precision) as g:
            g.upload_grid(IM, JM, KM, coor)
            g.upload_ucat(ucat)
            return [_swarm(g, n, IM, JM, KM, fused) for n in (small, large)]

    used = shim.shim_used()
    want = run()
    need = shim.shim_peak() - used - spares
    shim.shim_limit(used + need)
    got = run()
    for x, y in zip(want, got):
        for k in x:
            assert x[k].tobytes() == y[k].tobytes(), k
    shim.shim_limit(used + need - 1)  # and without that, the error that it always was
    try:
        run()
    except L.PicgpuError as e:
        assert "NOMEM" in str(e), e
    else:
        raise AssertionError("ran in less than it needs")
    assert shim.shim_used() == used


if __name__ == "__main__":
    globals()[sys.argv[2]](*sys.argv[3:])
    print("ok")
