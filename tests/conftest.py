import os
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) to run")


@pytest.fixture(scope="session")
def host_ctx():
    import vision_amd as va
    ctx = va.Context(-1)
    yield ctx
    ctx.close()


@pytest.fixture(scope="session")
def gpu_ctx():
    import vision_amd as va
    ctx = va.Context(0)
    yield ctx
    ctx.close()


def _wide_soup(extent, size, n=600, m=3000):
    """n triangles of about `size`, spread over +-extent in x and 20 sizes in y
    and z, one in three long in x, so that rays meet it although x is coarse;
    and m rays along z (a third of them slanted in y), 50 sizes away, at points
    of the triangles: positions, triangles, rays [m][8]."""
    rng = np.random.default_rng(5)
    c = np.stack([rng.uniform(-1, 1, n) * extent, *(rng.uniform(-1, 1, (2, n)) * size * 20)], 1)
    tri = c[:, None, :] + rng.normal(scale=size, size=(n, 3, 3)) * [1.0, 1.0, 0.1]
    tri[np.arange(n) % 3 == 0, :, 0] = np.array([-1.0, 1.0, 0.2]) * extent * 0.9
    at = np.einsum("mk,mkc->mc", rng.dirichlet([1, 1, 1], m), tri[rng.integers(0, n, m)])
    d = np.tile([0.0, 0.0, 1.0], (m, 1)) * np.where(rng.random(m) < 0.5, 1.0, -1.0)[:, None]
    d[: m // 3, 1] += rng.normal(scale=0.3, size=m // 3)
    d[m // 3: m // 2, 0] = -0.0
    rays = np.concatenate([at - d * size * 50, np.zeros((m, 1)), d, np.full((m, 1), 3e38)], 1).astype(np.float32)
    return tri.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3), rays


@pytest.fixture(scope="session")
def wide_soup():
    return _wide_soup
