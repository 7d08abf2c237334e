"""The wavefront form's segmented queues on the MI355X: queues of one path, of
whole and ragged blocks of 256, and of fewer, as many and more blocks than
segments give the megakernel's film bit for bit and its ray counts."""
import numpy as np
import pytest

from vision_amd import scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,chunk", [((1, 1), 1), ((255, 1), 1), ((16, 16), 1), ((257, 1), 2), ((60, 64), 1),
                                        ((64, 64), 1), ((4097, 1), 1), ((67, 129), 3)])
@pytest.mark.parametrize("kind", ["diffuse", "materials"])
def test_queues_hold_every_path(gpu_ctx, tmp_path, kind, size, chunk):
    if kind == "diffuse":
        sc = gpu_ctx.load_text(scenegen.cornell_box(64, 64, max_depth=6))
    else:
        sc = gpu_ctx.load_text(scenegen.procedural_scene(tmp_path, n_instances=4, level=2, width=64, height=64,
                                                         max_depth=6, hdri=(64, 32), spectrum="hero"), str(tmp_path))
    sc.build_accel()
    sc.set_resolution(*size)
    sc.set_counting(True)
    got = []
    for mode in ("megakernel", "wavefront"):
        sc.set_kernel(mode, chunk_frames=chunk)
        sc.reset_film()
        sc.render(3)
        st = sc.stats()
        got.append((sc.film(0).view(np.uint32), st["rays"], st["node_fetches"], st["tri_fetches"]))
    assert np.array_equal(got[0][0], got[1][0])
    assert got[0][1:] == got[1][1:]
    sc.close()
