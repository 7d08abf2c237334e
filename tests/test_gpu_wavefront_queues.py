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


def _resident():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[1]) * 4096


def test_stage_times_hold_no_more_events_for_longer_jobs(gpu_ctx):
    """Stage times of a job of thousands of bounces add up within its time, one
    launch of each stage a bounce, and host memory does not grow with them (an
    event of its own for each stamp would be some 60 000 here)."""
    sc = gpu_ctx.load_text(scenegen.cornell_box(64, 64, max_depth=8, min_depth=8))
    sc.build_accel()
    sc.set_resolution(3, 3)
    sc.set_kernel("wavefront", chunk_frames=1)
    sc.render(16)
    before = _resident()
    sc.render(2000)
    grown = _resident() - before
    st = sc.stats()
    bounces = st["stage_launches"][0]
    assert 2000 < bounces <= 2000 * 8 and st["stage_launches"] == [bounces] * 3
    assert all(ms > 0 for ms in st["stage_ms"]) and sum(st["stage_ms"]) < st["kernel_ms"]
    assert grown < 4 << 20
    sc.close()
