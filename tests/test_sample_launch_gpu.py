"""The ray passes of a frame and of a batch: one launch per lobe (specular
validation and generation together) gives every image the same bits as a
launch per pass, which is what the per-pass timers switch to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("size", [(8, 8), (65, 33), (161, 90)])
def test_one_launch_per_lobe_equals_one_per_pass(vgi, size, storage):
    import torch

    from violet_amd import _lib, renderer, scene, serve

    w, h = size
    sc = scene.Scene(scene.make_scene(4000, seed=5, extent=8.0))
    spec = serve.ViewSpec(w, h, 20.0)
    names = ("spec_reservoir", "spec_hit_pos", "spec_hit_radiance", "diff_new_hit_pos_normal", "diff_new_hit_radiance",
             "diff_reservoir", "indirect_diffuse_raw", "indirect_specular_raw", "hash_grid_storage")

    def frames(timed):
        r = renderer.RestirRenderer(w, h, renderer.RestirConfig(storage=storage))
        out = []
        _lib.call("vgi_profiler_reset")
        _lib.call("vgi_profiler_enable", int(timed))
        try:
            for f in range(6):  # a diffuse validation frame (4) among them
                r.add_passes(sc, serve.view_frame_params(spec, f), f)
                torch.cuda.synchronize()
                out.append([r.read(n, np.uint8, (r.image(n)[1],)).copy() for n in names])
        finally:
            _lib.call("vgi_profiler_enable", 0)
        passes = set(_lib.profiler_read()) if timed else set()
        r.close()
        return out, passes

    one, _ = frames(False)
    each, passes = frames(True)
    assert {"ind_spec_sample_gen", "ind_spec_sample_validate", "ind_diff_sample_gen", "ind_diff_sample_validate"} <= passes
    for f, (a, b) in enumerate(zip(one, each)):
        for n, x, y in zip(names, a, b):
            assert np.array_equal(x, y), f"frame {f}: {n} differs"


@pytest.mark.parametrize("storage", [0, 1])
def test_batch_times_each_sample_pass(vgi, storage):
    """Views at different frames, so that one batch holds generation and validation of both lobes."""
    import torch

    from violet_amd import _lib, batch, renderer, scene, serve

    sc = scene.Scene(scene.make_scene(4000, seed=5, extent=8.0))
    specs = [serve.ViewSpec(65, 33, 20.0), serve.ViewSpec(40, 56, 140.0), serve.ViewSpec(8, 8, 260.0)]
    first = [0, 3, 2]
    names = ("spec_reservoir", "spec_hit_radiance", "diff_reservoir", "indirect_diffuse_raw", "indirect_specular_raw")
    parts = {f"batch_ind_{lobe}_sample_{what}" for lobe in ("diff", "spec") for what in ("gen", "validate")}

    def frames(only):
        b = batch.Batch()
        views = [renderer.RestirRenderer(s.width, s.height, renderer.RestirConfig(storage=storage)) for s in specs]
        for r, s, f0 in zip(views, specs, first):
            for f in range(f0):
                r.add_passes(sc, serve.view_frame_params(s, f), f)
        torch.cuda.synchronize()
        _lib.call("vgi_profiler_reset")
        _lib.call("vgi_profiler_only", (only or "").encode())
        _lib.call("vgi_profiler_enable", int(only is not None))
        try:
            for k in range(4):
                b.add_passes(sc, views, [serve.view_frame_params(s, f0 + k) for s, f0 in zip(specs, first)],
                             [f0 + k for f0 in first])
            torch.cuda.synchronize()
        finally:
            _lib.call("vgi_profiler_enable", 0)
            _lib.call("vgi_profiler_only", None)
        out = [r.read(n, np.uint8, (r.image(n)[1],)).copy() for r in views for n in names]
        seen = set(_lib.profiler_read())
        b.close()
        for r in views:
            r.close()
        return out, seen

    whole, _ = frames(None)
    every, seen = frames("")
    assert parts <= seen and not {"batch_ind_spec_sample", "batch_ind_diff_sample"} & seen
    one, seen_one = frames("batch_ind_spec_sample_validate")
    assert seen_one == {"batch_ind_spec_sample_validate"}
    shared, seen_shared = frames("batch_ind_spec_sample")
    assert seen_shared == {"batch_ind_spec_sample"}
    for a in (every, one, shared):
        assert all(np.array_equal(x, y) for x, y in zip(whole, a))
