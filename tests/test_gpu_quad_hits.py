"""Closest hits by the walk with four lanes per ray, which finishes short queues: the extend kernels'
oracle tests with their queries sent to this walk, and queues of every length against those kernels."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
import test_gpu_edges as edges
import test_gpu_parity as parity
from conftest import random_rays
from deep_mesh import DEEP, shrinking_clusters
from oracle.pyoracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.fixture
def by_quads(monkeypatch):
    hits = illume_amd.Context.closest_hit
    monkeypatch.setattr(illume_amd.Context, "closest_hit", lambda self, scene, rays: hits(self, scene, rays, quad=True))


@pytest.mark.parametrize("name,make", [("cornell", S.cornell), ("tiny_all_materials", S.tiny_mesh_scene),
                                       ("gold_100k", S.gold_spheres)])
def test_scenes_against_the_oracle(by_quads, ctx, name, make):
    spec, st = make()
    s, orc = ctx.scene(spec), OracleScene(spec)
    getattr(parity, "test_closest_hit_" + name)(ctx, (spec, st, s, orc))
    s.free()
    orc.free()


def test_degenerate_and_axis_parallel(by_quads, ctx):
    edges.test_closest_hit_degenerate_and_axis_parallel(ctx)


@pytest.mark.parametrize("offset", [1e3, 1e4])
@pytest.mark.parametrize("layout", ["fp32", "quant8"])
def test_far_from_the_world_origin(by_quads, offset, layout):
    edges.test_closest_hit_far_from_the_world_origin(offset, layout)


# one ray; a quad more or less than a wave's 16 and 64; every wave with 16 and one more; past 2^18
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 5120 * 16 + 1, 1 << 18, (1 << 18) + 1])
@pytest.mark.parametrize("tri", ["mt", "watertight"])
def test_queues_of_every_length_match_the_extend_kernel(n, tri):
    rays = random_rays(-3, 3, n, seed=n)
    rays[::7, 3] = 0.0                               # axis-parallel planes
    rays[::11, 4:] = 0.0
    rays[:, 3:] /= np.maximum(np.linalg.norm(rays[:, 3:], axis=1, keepdims=True), np.float32(1e-9))
    spec, _ = S.tiny_mesh_scene(n=9)
    with illume_amd.Context(0, tri_test=tri, paths_in_flight=1 << 19) as c:
        s = c.scene(spec)
        for a, b in zip(c.closest_hit(s, rays, quad=True), c.closest_hit(s, rays)):
            assert np.array_equal(a, b)
        s.free()


@pytest.mark.parametrize("levels", sorted(DEEP))
def test_deep_trees(levels):
    """Rays from the innermost clusters outwards: a mesh that fills the walk's stacks, and one past them."""
    v, i = shrinking_clusters(*DEEP[levels])
    spec = dict(meshes=[dict(positions=v, indices=i, face_normals=True, leaf_size=4)],
                instances=[dict(mesh=0, material=0, transform=dict(translation=[0, 0, 0]))], spheres=[],
                materials=[dict(type="lambert", albedo=[0.5, 0.5, 0.5])], mediums=[], environment=None,
                camera=dict(fov=40.0, transform=dict(translation=[0, 0, -3])))
    rng = np.random.default_rng(3)
    o = rng.uniform(-1e-3, 1e-3, (20000, 3)) - [1e-3, 0, 0]
    d = rng.uniform([1, 0, 0], [1.5, 1, 1], (20000, 3)) - o
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1)
    with illume_amd.Context(0, paths_in_flight=1 << 16) as c:
        s = c.scene(spec)
        ref = c.closest_hit(s, rays)
        assert (ref[0] >= 0).sum() > 2000
        if 3 * levels + 1 <= 64:
            for a, b in zip(c.closest_hit(s, rays, quad=True), ref):
                assert np.array_equal(a, b)
        else:
            with pytest.raises(illume_amd.IlmError) as e:
                c.closest_hit(s, rays, quad=True)
            assert e.value.code == -9
        s.free()
