"""The per-depth kernels and captured graphs under the tests of small renders, which the default extend
mode finishes in one directly launched kernel: those tests again with contexts that launch every depth
(extend_mode 3), and renders of several chunks above 2^18 paths, whose graphs hold both."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
import test_gpu_edges as edges
import test_gpu_forms as forms
import test_gpu_parity as parity
import test_zz_no_alloc as noalloc
from illume_amd._abi import render_params
from oracle.pyoracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.fixture
def per_depth(monkeypatch):
    class PerDepth(illume_amd.Context):
        def __init__(self, device=0, **opts):
            super().__init__(device, **dict(dict(extend_mode=3), **opts))
    monkeypatch.setattr(illume_amd, "Context", PerDepth)


@pytest.fixture
def ctx3(per_depth):
    with illume_amd.Context(0) as c:
        yield c


@pytest.fixture
def scenes(ctx3):
    out = {}
    for name, fn in [("cornell", S.cornell), ("tiny", S.tiny_mesh_scene), ("gold", lambda: S.gold_spheres(n=20))]:
        spec, st = fn()
        out[name] = (spec, st, ctx3.scene(spec))
    yield out
    for _, _, s in out.values():
        s.free()


@pytest.mark.parametrize("test", [forms.test_graph_replays_match_direct_launches, forms.test_two_pipelines_match_one])
def test_graphs_and_pipelines(scenes, test):
    test(scenes)


@pytest.mark.parametrize("order", [dict(sample_group=2, tile_rows=3, paths_in_flight=3000), dict(shade_sort=2),
                                   dict(shade_sort=1, paths_in_flight=5000), dict(camera_packets=2),
                                   dict(camera_packets=1, sample_group=1, tile_rows=1),
                                   dict(sched_fair=1, paths_in_flight=3000)])
def test_path_orders(ctx3, scenes, order):
    forms.test_path_order_leaves_results_unchanged(ctx3, scenes, order)


def test_layouts_and_triangle_tests(per_depth, ctx3, scenes):
    with illume_amd.Context(0, bvh_layout="quant8") as q, illume_amd.Context(0, tri_test="watertight") as w:
        forms.test_layout_switch_by_tune_matches_a_context_opened_with_it(q, scenes)
        forms.test_quantized_and_watertight_renders_agree(q, w, ctx3, scenes)


def test_spilling_stack_without_allocation(per_depth):
    """The extend kernels under FP32 nodes with their spill area in the scratch array."""
    noalloc.test_noalloc_equals_plain_render_with_spilling_stack()


@pytest.mark.parametrize("mode", [0, 3])
def test_spilling_stack_on_long_queues(mode):
    """The same scene with more than 2^18 paths: the default mode spills at its first depths too."""
    spec, st = S.subsurface(env_size=(256, 128))
    with illume_amd.Context(0, extend_mode=mode, paths_in_flight=1 << 21) as c:
        s = c.scene(spec)
        noalloc._same(c, s, render_params(**dict(st, width=400, height=300, spp=5, max_depth=12)))
        s.free()


@pytest.mark.parametrize("name,make", [("cornell", S.cornell), ("tiny_all_materials", S.tiny_mesh_scene),
                                       ("gold", S.gold_spheres)])
@pytest.mark.parametrize("layout", ["fp32", "quant8"])
def test_path_radiance_against_the_oracle(per_depth, name, make, layout):
    spec, st = make()
    with illume_amd.Context(0, bvh_layout=layout) as c:
        s, orc = c.scene(spec), OracleScene(spec)
        getattr(parity, "test_path_radiance_" + name)(c, (spec, st, s, orc))
        s.free()
        orc.free()


def test_ties_resolved_independently_of_the_walk(per_depth, ctx3):
    spec, st = S.subsurface()
    s = ctx3.scene(spec)
    parity.test_subsurface_ties_resolved_independently_of_the_walk(ctx3, (spec, st, s, None))
    s.free()


@pytest.mark.parametrize("maker", [edges._env_only, edges._spheres_only, edges._degenerate_mesh_scene])
def test_small_scenes(ctx3, maker):
    edges.test_small_scenes_render_like_oracle(ctx3, maker)


@pytest.mark.parametrize("mode", [0, 3])
@pytest.mark.parametrize("pipes", [1, 2])
def test_replayed_graphs_of_long_chunks(mode, pipes):
    """Three chunks of 2^19 paths, a fourth below 2^18 and chunks of two scenes, replayed between other
    renders: captured depths with the launch that finishes them, against direct launches in one pipeline."""
    spec, st = S.gold_spheres(n=20)
    other, ot = S.tiny_mesh_scene()
    p = render_params(**dict(st, width=512, height=256, spp=13, max_depth=9))
    q = render_params(**dict(ot, width=300, height=300, spp=4, max_depth=12))
    res = []
    for opts in (dict(extend_mode=3, use_graphs=0, pipes=1), dict(extend_mode=mode, use_graphs=1, pipes=pipes)):
        with illume_amd.Context(0, paths_in_flight=1 << 19, **opts) as c:
            s, t = c.scene(spec), c.scene(other)
            for _ in range(1 if not opts["use_graphs"] else 3):
                out = [c.render(s, p)]
                batch, info = c.render_batch([s, t, s], [p, q, q])
                hs = [c.submit(s, p), c.submit(t, q)]
                for h in hs:
                    h.wait(60000)
                out += [(a, px, None) for a, px in batch] + [h.result() + (None,) for h in hs]
                for h in hs:
                    h.free()
                res.append((out, info["segments"]))
            assert out[0][2]["chunks"] == 4
            s.free()
            t.free()
    ref, segs = res[0]
    for out, n in res[1:]:
        assert n == segs and out[0][2]["segments"] == ref[0][2]["segments"]
        for (a, px, _), (ra, rpx, _) in zip(out, ref):
            assert np.array_equal(a, ra, equal_nan=True) and np.array_equal(px, rpx)
