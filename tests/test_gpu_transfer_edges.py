"""Host arrays at the edges of a transfer's slots: one array of 8-byte elements
that just fills, just fits or just exceeds 512 KiB, three such slots, the sizes
from which a download (2 MiB) and an upload (4 MiB) take the large ring and
helper threads, the one from which slots are filled to 1 MiB (8 MiB), and each
slot's second and third use.  Whole numbers and FP64 arrays bit for bit."""
import ctypes as C

import numpy as np
import pytest

from fdf_amd import _lib as L
from fdf_amd import workloads as W

pytestmark = pytest.mark.gpu

SLOT = (512 << 10) // 8  # elements
SIZES = [SLOT - 1, SLOT, SLOT + 1, 3 * SLOT - 1, 3 * SLOT, 3 * SLOT + 1, 4 * SLOT - 1, 4 * SLOT, 8 * SLOT - 1, 8 * SLOT, 8 * SLOT + 1,
         16 * SLOT - 1, 16 * SLOT, 16 * SLOT + 1, 32 * SLOT + 1, 48 * SLOT + 3]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", SIZES)
def test_one_array_at_a_time(precision, n):
    from fdf_amd.swarm import PicGpu

    print("[gpu-case] transfer edges", precision, n, flush=True)
    IM, JM, KM = 7, 6, 5
    rng = np.random.default_rng(n)
    real = np.float64 if precision == "fp64" else np.float32
    s = {"pos": rng.standard_normal((n, 3)), "vel": rng.standard_normal((n, 3)),
         "cell": rng.integers(0, [IM, JM, KM], (n, 3)), "weight": rng.random((n, 3)),
         "status": rng.integers(0, 5, n), "pid": rng.integers(-2 ** 62, 2 ** 62, n)}
    with PicGpu(precision=precision) as g:
        g.upload_grid(IM, JM, KM, W.uniform_grid(IM, JM, KM))
        g.upload_particles(s["pos"], **{k: s[k] for k in s if k != "pos"})
        for k in s:
            out = np.full_like(s[k], 77)
            ptr = [out.ctypes.data_as(C.c_void_p) if q == k else None
                   for q in ("pos", "vel", "cell", "weight", "status", "pid")]
            L.check(g.lib.picgpu_download_particles(g.h, *ptr))
            want = s[k].astype(real).astype(np.float64) if k in ("vel", "weight") else s[k]
            assert np.array_equal(out, want), k
