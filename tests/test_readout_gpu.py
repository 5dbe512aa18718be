"""The moment readout against FP64 numpy at the edges of its line grouping:
one line, an odd number of lines, pair counts at and below the line where lines
are taken in twos, spins that leave threads without work, and phases past 2^30
(whose sine takes another reduction), among ordinary ones in one wave."""
import ctypes as C

import numpy as np
import pytest
import torch

from dsim_amd import lib as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


@pytest.mark.parametrize("n,lines", [(1, 1), (257, 3), (65535, 64), (65536, 64), (65537, 65)])
def test_readout_matches_fp64(n, lines):
    print(f"case readout spins {n} lines {lines}", flush=True)
    rng = np.random.default_rng(n + lines)
    # one axis a spin, so that the FP32 phase is one rounded product
    mom = np.zeros((3, n), np.float32)
    axis = rng.integers(0, 3, n)
    mom[axis, np.arange(n)] = rng.normal(size=n) * 10.0 ** rng.integers(-2, 3, n)
    mom[axis[::97], np.arange(n)[::97]] *= np.float32(2.0 ** 30)
    mag = rng.uniform(0.1, 1.0, n).astype(np.float32)
    comp = rng.integers(0, 4, n)
    g = rng.normal(size=(lines, 3)).astype(np.float32)
    f = D.lib().dsim_signal_moment_nalloc
    f.restype = C.c_int
    f.argtypes = [C.c_uint32] + [C.c_void_p] * 3 + [C.c_float, C.c_void_p, C.c_uint32, C.c_void_p,
                                                   C.c_float, C.c_void_p, C.c_void_p]
    t = [torch.from_numpy(a).cuda() for a in
         (mag, mom, (comp | (65535 << 8)).astype(np.int32), g)]
    out = torch.zeros((lines, 5), dtype=torch.float64, device="cuda")
    D.check(f(n, t[0].data_ptr(), t[1].data_ptr(), None, 0.0, t[2].data_ptr(), lines,
              t[3].data_ptr(), 0.5, out.data_ptr(), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    v = mom[axis, np.arange(n)]
    for j in range(lines):
        ph = (g[j][axis] * v) * np.float32(0.5)
        z = mag.astype(np.float64) * np.exp(1j * ph.astype(np.float64))
        ref = [abs(z.sum()) / n] + [abs(z[comp == c].sum()) / max((comp == c).sum(), 1)
                                    for c in range(4)]
        # n sums of terms at most 1, each to half an ulp of the sum so far
        np.testing.assert_allclose(got[j], ref, rtol=0, atol=1e-15 * n + 1e-14)
