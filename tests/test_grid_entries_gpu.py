"""A grid whose cells list more triangles than 32-bit places can number is
refused by the device build, before anything is written at those places."""
import numpy as np
import pytest

from dsim_amd import lib as D

pytestmark = pytest.mark.gpu


def test_too_many_grid_entries_are_refused():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    # 4200 triangles in each of 2^20 cells: 4.4e9 entries, 1.1e8 in 32 bits
    n = 4200
    rng = np.random.default_rng(1)
    V = np.concatenate([np.full((n, 1, 3), -1.0), np.full((n, 1, 3), 1.0),
                        rng.uniform(-1, 1, (n, 1, 3))], 1).reshape(-1, 3)
    T = np.arange(3 * n).reshape(n, 3)
    I = np.stack([np.arange(n) % 9, np.zeros(n, int), T[:, 0]], 1)
    print(f"case {n} triangles in each of 2^20 cells", flush=True)
    with pytest.raises(D.DsimError) as e:
        D.Substrate(V, T, I, device=True, grid="aabb", dims=(128, 128, 64), lo=(-1.0,) * 3,
                    cell=(2 / 128, 2 / 128, 2 / 64), eps=1e-5)
    assert e.value.code == -1 and "too fine" in str(e.value)
