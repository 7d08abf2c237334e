"""The radiance cache's kernels at the sizes their launches change: fewer rows
than a tile, a wave or a block, remainders, the size from which a lane encodes
sixteen rows, and lists longer than the workspace (which run in chunks).
Forward outputs of a list equal those of its parts bit for bit; gradients of a
batch are the size-weighted mean of its parts' gradients (the loss is a mean),
within the BF16 rounding of the layers' gradients."""
import json

import numpy as np
import pytest

import vision_amd as va
from vision_amd import scenegen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cache(gpu_ctx):
    sc = gpu_ctx.load_text(json.dumps(scenegen.cornell_box(16, 16))).build_accel()
    nrc = va.RadianceCache(sc)
    rng = np.random.default_rng(3)
    mlp = np.concatenate([rng.uniform(-a, a, n) for a, n in
                          [(np.sqrt(6 / 96), 2048), (np.sqrt(6 / 128), 4096), (np.sqrt(6 / 128), 4096),
                           (np.sqrt(6 / 67), 192)]]).astype(np.float32)
    nrc.set_params(mlp, rng.random(va.NRC_GRID_PARAMS, dtype=np.float32) - np.float32(0.5))
    yield nrc
    nrc.close()
    sc.close()


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 255, 1000, (1 << 19) - 1, (1 << 19) + 1, (4 << 20) + 77])
def test_forward_of_a_list_equals_its_parts(cache, n):
    rng = np.random.default_rng(n)
    pos = rng.uniform([-1.1, -0.1, -1.1], [1.1, 2.1, 1.1], (n, 3)).astype(np.float32)
    whole = cache.forward(pos)
    cut = n // 3 + 1
    parts = [cache.forward(p) for p in (pos[:cut], pos[cut:]) if len(p)]
    assert np.array_equal(whole.view(np.uint32), np.concatenate(parts).view(np.uint32))


def _apart(whole, ref):
    """The difference's norm in units of the tolerance: the gradients of three
    layers are rounded to bf16 (2^-9 of each value), scaled by 1 / n in the whole
    and by the parts' sizes in them, six roundings apart."""
    whole, ref = np.asarray(whole, np.float64), np.asarray(ref, np.float64)
    return np.linalg.norm(whole - ref) / (6 * 2.0 ** -9 * np.linalg.norm(ref))


# the last `tail` rows (those of a second chunk of the workspace, or the very
# last) have far larger targets, so that the sums are theirs.  They lie at one
# point, where they have the same output and gradients in proportion to their
# targets, and the last row has the largest: its share is 1 / 33 or more, 2.5
# tolerances, and so a row lost, taken twice or at another's position shows
@pytest.mark.parametrize("n,tail", [(2, 0), (17, 1), (127, 0), (129, 1), (4099, 0), (4099, 1), (70001, 0), (70001, 1),
                                    ((1 << 20) + 33, 0), ((1 << 20) + 33, 33)])
def test_gradients_are_the_mean_of_the_parts(cache, n, tail):
    rng = np.random.default_rng(n)
    s = np.concatenate([rng.uniform([-1, 0, -1], [1, 2, 1], (n, 3)), rng.exponential(0.5, (n, 3))], 1).astype(np.float32)
    if tail:
        s[-tail:, :3] = s[-1, :3]
        s[-tail:, 3:] = 1e4 * rng.uniform(1, 2, (tail, 3))
        s[-1, 3:] = 2e4
    cut = n // 2
    whole = cache.gradients(s)
    a, b = cache.gradients(s[:cut]), cache.gradients(s[cut:])
    for w, pa, pb in zip(whole, a, b):
        assert _apart(w, cut / n * np.asarray(pa, np.float64) + (n - cut) / n * np.asarray(pb, np.float64)) <= 1
    if tail:
        fewer = cache.gradients(s[:-1])
        for w, p in zip(whole, fewer):
            assert _apart(w, (n - 1) / n * np.asarray(p, np.float64)) > 2
