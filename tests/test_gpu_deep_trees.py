"""Scenes whose walk over FNodes needs exactly the 64 stack entries it has, and scenes that need more and
keep to the per-depth kernels and the packets over the other layouts: the same images as those give."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from illume_amd._abi import render_params
from deep_mesh import DEEP, shrinking_clusters

pytestmark = pytest.mark.gpu


def _spec(levels, instances):
    """Seen from the innermost clusters outwards, so that a walk has the outer ones still to visit."""
    v, i = shrinking_clusters(*DEEP[levels])
    place = [dict(translation=[0.0, 2.5 * k, 0.0], rotation=[15.0 * k, 0.0, 10.0 * k]) for k in range(instances)]
    return dict(meshes=[dict(positions=v, indices=i, face_normals=True, leaf_size=4)],
                instances=[dict(mesh=0, material=0, transform=t) for t in place], spheres=[],
                materials=[dict(type="lambert", albedo=[0.8, 0.7, 0.6])], mediums=[], environment=[0.9, 0.95, 1.0],
                camera=dict(fov=60.0, dof=1.0, aperture=0.0, transform=dict(translation=[-0.02, -0.01, -0.01], lookat=[1.2, 0.6, 0.6])))


# 3 * levels of the mesh + 1 + 3 * levels of the instances: 64, 70, 67
@pytest.mark.parametrize("levels,instances", [(21, 1), (23, 1), (21, 2)])
@pytest.mark.parametrize("layout,tri", [("fp32", "mt"), ("quant8", "mt"), ("fp32", "watertight")])
def test_walks_of_full_stacks_and_scenes_beyond_them(levels, instances, layout, tri):
    spec = _spec(levels, instances)
    other, st = S.tiny_mesh_scene()
    ps = [render_params(**dict(st, width=61, height=47, spp=3, max_depth=8)),        # one launch finishes it
          render_params(**dict(st, width=600, height=450, spp=2, max_depth=8))]      # above 2^18 paths at first
    out = []
    for opts in (dict(extend_mode=3, camera_packets=2), dict(), dict(extend_mode=3, camera_packets=1)):
        with illume_amd.Context(0, bvh_layout=layout, tri_test=tri, paths_in_flight=1 << 21, **opts) as c:
            s, t = c.scene(spec), c.scene(other)
            res = [c.render(s, p) for p in ps]
            batch, info = c.render_batch([s, t, s], [ps[0], ps[0], ps[1]])
            res += [(a, px, info) for a, px in batch] + [c.render_noalloc(s, ps[1])]
            out.append(res)
            s.free()
            t.free()
    assert out[0][0][2]["segments"] > 1.3 * 61 * 47 * 3      # the rays do hit something
    for res in out[1:]:
        for (a, px, info), (ra, rpx, rinfo) in zip(res, out[0]):
            assert np.array_equal(a, ra, equal_nan=True) and np.array_equal(px, rpx)
            assert info["segments"] == rinfo["segments"]
