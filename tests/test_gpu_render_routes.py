"""The megakernel form's fused jobs of several frames on the MI355X: whichever
way vs_render runs them (a lane a sample for the diffuse family, as wavefront
for every material, one lane a pixel where counters or adaptive sampling need
it), the film and the output buffer equal the frame-by-frame launches' bit for
bit, also continued from an earlier frame, at odd sizes, in several chunks and
without accumulation; and the workspace they run in is one of the context and
given back."""
import numpy as np
import pytest
import torch

import vision_amd as va
from vision_amd import scenegen

pytestmark = pytest.mark.gpu


def _scene(kind, folder):
    if kind == "diffuse":
        return scenegen.cornell_box(64, 64, max_depth=5)
    return scenegen.procedural_scene(folder, n_instances=4, level=2, width=64, height=64, max_depth=6, hdri=(64, 32),
                                     spectrum="srgb")


@pytest.mark.parametrize("kind", ["diffuse", "materials"])
@pytest.mark.parametrize("size,spp,first", [((1, 1), 3, 0), ((8, 8), 2, 0), ((9, 17), 3, 1), ((65, 63), 7, 2)])
@pytest.mark.parametrize("spectral", [0, 3, 4])
def test_fused_equals_frame_by_frame(gpu_ctx, tmp_path, kind, size, spp, first, spectral):
    sc = gpu_ctx.load_text(_scene(kind, tmp_path), str(tmp_path))
    sc.build_accel()
    sc.set_resolution(*size)
    if spectral:
        sc.set_spectrum(True, spectral)
    films = []
    for fused in (False, True):
        sc.reset_film()
        if first:
            sc.render(first, fused=False)
        sc.render(spp, fused=fused)
        assert sc.info()["frame_index"] == first + spp
        films.append((sc.film(0), sc.film(1)))
    for a, b in zip(*films):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    sc.set_counting(True)
    sc.reset_film()
    sc.render(first + spp)
    assert sc.stats()["rays"] > 0
    assert np.array_equal(sc.film(0).view(np.uint32), films[0][0].view(np.uint32))
    sc.close()


def test_last_frame_without_accumulation(gpu_ctx):
    s = scenegen.cornell_box(40, 24, max_depth=4)
    s["camera"]["param"]["radiance_collector"]["param"]["accumulation"] = 0
    sc = gpu_ctx.load_text(s)
    sc.build_accel()
    sc.render(3, fused=False)
    a = sc.film(0)
    sc.reset_film()
    sc.render(3)
    assert np.array_equal(a.view(np.uint32), sc.film(0).view(np.uint32))
    sc.close()


def test_depths_beyond_the_wavefronts_bounce_count(gpu_ctx, tmp_path):
    """A scene file's max_depth has no limit; the wavefront's path state keeps
    16 bits of the bounce, so deeper jobs stay with the megakernel."""
    s = _scene("materials", tmp_path)
    launches = []
    for depth in (65_535, 65_536):
        s["integrator"]["param"]["max_depth"] = depth
        sc = gpu_ctx.load_text(s, str(tmp_path))
        sc.build_accel()
        sc.render(4)
        launches.append(sc.stats()["launches"])
        sc.close()
    assert launches[0] > 1 and launches[1] == 1


@pytest.mark.parametrize("kind,spectral,depth,spp,size,routed", [
    ("diffuse", 0, 2, 2, (1, 1), True), ("diffuse", 0, 2, 1, (64, 64), False),
    ("diffuse", 0, 2, 2, (2048, 2048), True), ("diffuse", 0, 2, 2, (2048, 2049), False),
    ("diffuse", 4, 2, 2, (2048, 2048), True), ("diffuse", 3, 2, 3, (2049, 2048), False),
    ("materials", 0, 1, 3, (512, 512), True), ("materials", 0, 1, 3, (513, 512), False),
    ("materials", 0, 2, 3, (1024, 512), True), ("materials", 4, 2, 3, (1025, 512), False),
    ("materials", 0, 3, 3, (1024, 1024), True), ("materials", 0, 3, 8, (1025, 1024), False),
    ("materials", 0, 4, 3, (2048, 1024), True), ("materials", 0, 4, 4, (2049, 1024), False),
    ("materials", 0, 9, 3, (1024, 512), True), ("materials", 0, 9, 3, (1025, 512), False),
    ("materials", 0, 8, 4, (2048, 2048), True), ("materials", 0, 8, 4, (2049, 2048), False),
    ("materials", 0, 6, 2, (64, 64), False), ("materials", 0, 0, 3, (64, 64), False),
])
def test_routes(gpu_ctx, tmp_path, kind, spectral, depth, spp, size, routed):
    """One launch is the megakernel; both sides of each line of the rule."""
    sc = gpu_ctx.load_text(_scene(kind, tmp_path), str(tmp_path))
    sc.build_accel()
    sc.set_resolution(*size)
    sc.set_integrator(depth, 5, 1.0)
    if spectral:
        sc.set_spectrum(True, spectral)
    sc.render(spp)
    launches = sc.stats()["launches"]
    assert launches > 1 if routed else launches == 1
    assert not routed or kind == "materials" or launches == 2
    sc.close()


# a second chunk: of frames beyond a launch's grid, of samples beyond 32 M, and
# of the wavefront's paths beyond 32 M
@pytest.mark.parametrize("kind,size,spp,chunks", [("diffuse", (1, 1), 65_537, 2), ("diffuse", (1920, 1080), 17, 2),
                                                  ("materials", (1920, 1080), 17, 2)])
def test_jobs_of_several_chunks(gpu_ctx, tmp_path, kind, size, spp, chunks):
    sc = gpu_ctx.load_text(_scene(kind, tmp_path), str(tmp_path))
    sc.build_accel()
    sc.set_resolution(*size)
    sc.set_integrator(2 if kind == "diffuse" else 4, 5, 1.0)
    sc.render(spp)
    launches = sc.stats()["launches"]
    # per chunk: samples and accumulation; or begin, accumulation and four launches a bounce, after one of the job
    assert launches == 2 * chunks if kind == "diffuse" else launches >= 1 + chunks * (2 + 4 * 4)
    got = sc.film(0)
    sc.reset_film()
    sc.set_counting(True)  # one launch of the megakernel
    sc.render(spp)
    assert sc.stats()["launches"] == 1
    assert np.array_equal(sc.film(0).view(np.uint32), got.view(np.uint32))
    sc.close()


MB = 1 << 20


def _free():
    return torch.cuda.mem_get_info(0)[0]


def _load(ctx, folder, kind="materials"):
    sc = ctx.load_text(_scene(kind, folder), str(folder))
    sc.build_accel()
    sc.render(3)  # the kernels' code and scratch memory
    sc.set_kernel("megakernel")
    sc.set_resolution(256, 256)
    return sc


def test_scenes_share_a_workspace_that_is_given_back(tmp_path):
    # 256 x 256 at 64 samples: 4 M paths, 772 MB of state, and 67 MB of samples
    with va.Context(0) as ctx:
        scenes = [_load(ctx, tmp_path) for _ in range(3)] + [_load(ctx, tmp_path, "diffuse")]
        start = _free()
        scenes[0].render(64)
        one = start - _free()
        assert 700 * MB < one < 900 * MB
        for sc in scenes[1:]:
            sc.render(64)
            assert start - _free() < one + 100 * MB
        scenes[1].set_kernel("megakernel")
        assert start - _free() < 64 * MB
        scenes[1].render(64)
        assert start - _free() > 700 * MB
        scenes.pop().close()
        assert start - _free() < 64 * MB
        for sc in scenes:
            sc.close()


def test_workspace_makes_room_for_other_allocations(tmp_path):
    """A server's arena of more than is free beside the workspace (more than a
    gigabyte beyond what the device reports can still be had)."""
    with va.Context(0) as ctx:
        sc = _load(ctx, tmp_path)
        sc.render(256)  # 16 M paths, 3.1 GB
        film = sc.film(0)
        with va.Server(ctx, hbm_budget=_free() + 2500 * MB) as srv:
            job = srv.submit(srv.add_scene(sc), 64, 64, 2)
            srv.wait(job)
            assert srv.result(job, 0, (64, 64)).max() > 0
            # beside the arena, at most an eighth of what is free (and the pages of 14 buffers)
            start = _free()
            sc.reset_film()
            sc.render(256)
            held = -_free()
            sc.set_kernel("megakernel")
            assert held + _free() <= start // 8 + 32 * MB
            assert np.array_equal(sc.film(0).view(np.uint32), film.view(np.uint32))
        sc.close()


def test_workspace_makes_room_for_another_scenes_render(tmp_path):
    """A wavefront job that needs 7.6 GB of state where 2.5 GB are free beside
    the workspace's 6.1."""
    with va.Context(0) as ctx:
        a, b = _load(ctx, tmp_path), _load(ctx, tmp_path)
        for sc in (a, b):
            sc.set_resolution(1920, 1080)
            sc.set_integrator(2, 5, 1.0)
        b.set_kernel("wavefront", chunk_frames=1)
        b.render(1)
        b.set_kernel("wavefront", chunk_frames=20)
        a.set_integrator(4, 5, 1.0)
        a.render(16)
        rest = torch.empty(_free() - 2500 * MB, dtype=torch.uint8, device="cuda")
        b.reset_film()
        b.render(20)
        film = b.film(0)
        del rest
        torch.cuda.empty_cache()
        b.reset_film()
        b.render(20, fused=False)
        assert np.array_equal(b.film(0).view(np.uint32), film.view(np.uint32))
        b.close()
        a.close()
