"""Queues of at most 2^18 paths are finished in one launch with four lanes per ray (the default
extend mode): bit-identical to the per-depth kernels (extend_mode 3) whatever the path count."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from illume_amd._abi import render_params

pytestmark = pytest.mark.gpu

TAIL = 1 << 18
SCENES = {"cornell": S.cornell, "tiny": S.tiny_mesh_scene, "gold": lambda: S.gold_spheres(n=20),
          "medium": lambda: S.subsurface(n=12, env_size=(64, 32))}


@pytest.fixture(scope="module")
def pair():
    with illume_amd.Context(0, extend_mode=3) as a, illume_amd.Context(0) as b:
        yield a, b


# one path; a wave's four, 64 and 65; every wave of the launch with 4 and 5 paths; the limit itself, one row
# above it (the queue crosses the limit after some depths) and a queue that stays above it
@pytest.mark.parametrize("name,w,h,spp,depth", [
    ("tiny", 1, 1, 1, 12), ("tiny", 4, 1, 1, 12), ("cornell", 64, 1, 1, 8), ("tiny", 13, 5, 1, 1),
    ("medium", 160, 128, 1, 45), ("gold", 160, 128, 1, 16), ("medium", 5121, 5, 1, 45),
    ("tiny", 512, 512, 1, 12), ("tiny", 512, 513, 1, 12), ("cornell", 512, 513, 1, 8), ("medium", 333, 251, 7, 45),
    ("cornell", 700, 700, 3, 3)])
@pytest.mark.parametrize("layout,tri", [("fp32", "mt"), ("quant8", "mt"), ("fp32", "watertight")])
def test_short_queues_match_the_per_depth_kernels(name, w, h, spp, depth, layout, tri):
    spec, st = SCENES[name]()
    p = render_params(**dict(st, width=w, height=h, spp=spp, max_depth=depth))
    out = []
    for mode in (3, 0):
        with illume_amd.Context(0, extend_mode=mode, bvh_layout=layout, tri_test=tri, paths_in_flight=1 << 21) as c:
            s = c.scene(spec)
            out.append(c.render(s, p))
            if mode == 0:
                out.append(c.render(s, p))          # the captured graph again
                out.append(c.render_noalloc(s, p))
            s.free()
    ref = out[0]
    for a, px, info in out[1:]:
        assert np.array_equal(a, ref[0], equal_nan=True)
        assert np.array_equal(px, ref[1])
        assert info["segments"] == ref[2]["segments"]


def test_short_queues_of_several_scenes_match(pair):
    """A chunk of several scenes, below the limit and crossing it, served and batched."""
    reqs = [("cornell", 64, 48, 3), ("tiny", 50, 33, 5), ("gold", 40, 40, 2), ("medium", 31, 57, 3), ("tiny", 400, 300, 3)]
    res = []
    for c in pair:
        sc = {k: c.scene(SCENES[k]()[0]) for k in SCENES}
        ps = [render_params(**dict(SCENES[k]()[1], width=w, height=h, spp=n)) for k, w, h, n in reqs]
        small, i0 = c.render_batch([sc[r[0]] for r in reqs[:4]], ps[:4])
        big, i1 = c.render_batch([sc[r[0]] for r in reqs], ps)
        hs = [c.submit(sc[r[0]], p) for r, p in zip(reqs, ps)]
        served = []
        for h in hs:
            h.wait(60000)
            served.append(h.result())
            h.free()
        for s in sc.values():
            s.free()
        res.append((small + big + served, i0["segments"], i1["segments"]))
    for (a, ap), (b, bp) in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b, equal_nan=True) and np.array_equal(ap, bp)
    assert res[0][1:] == res[1][1:]


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 5120 * 16 + 1, TAIL, TAIL + 1])
def test_closest_hits_of_short_queues_match(pair, n):
    rng = np.random.default_rng(n)
    rays = np.concatenate([rng.uniform(-3, 3, (n, 3)), rng.normal(size=(n, 3))], 1)
    rays[::7, 3] = 0.0                               # axis-parallel planes
    rays[::11, 4:] = 0.0
    rays[:, 3:] /= np.maximum(np.linalg.norm(rays[:, 3:], axis=1, keepdims=True), 1e-9)
    spec, _ = S.tiny_mesh_scene(n=9)
    out = []
    for c in pair:
        s = c.scene(spec)
        out.append(c.closest_hit(s, rays))
        s.free()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("layout", ["fp32", "quant8"])
@pytest.mark.parametrize("w,h,spp", [(1024, 512, 1), (1024, 512, 2), (333, 331, 8), (96, 64, 64), (700, 701, 3),
                                     (1001, 703, 6)])
def test_camera_rays_per_lane_and_as_packets_match(w, h, spp, layout):
    """The default choice between packets and lanes for the first depth, and both by name, over
    queues of few and many rays per wave (whole and split, ragged, one to 64 samples a pixel)."""
    spec, st = SCENES["tiny"]()
    p = render_params(**dict(st, width=w, height=h, spp=spp, max_depth=3))
    out = []
    for packets in (0, 1, 2):
        with illume_amd.Context(0, extend_mode=3, camera_packets=packets, bvh_layout=layout) as c:
            s = c.scene(spec)
            out.append(c.render(s, p))
            s.free()
    for a, px, info in out[1:]:
        assert np.array_equal(a, out[0][0], equal_nan=True) and np.array_equal(px, out[0][1])
        assert info["segments"] == out[0][2]["segments"]


@pytest.mark.parametrize("graphs", [0, 1])
def test_descriptors_of_any_length_are_staged(graphs):
    """Chunks of 1, 33 and 64 requests after one another: only the parts in use of a chunk's
    descriptor reach the device, and what an earlier chunk left there is not read."""
    spec, st = S.tiny_mesh_scene()
    ps = [render_params(**dict(st, width=3 + 5 * (i % 9), height=2 + i, spp=1 + i % 4, max_depth=2 + i % 5)) for i in range(64)]
    with illume_amd.Context(0, use_graphs=graphs) as c:
        s = c.scene(spec)
        alone = [c.render(s, p) for p in ps]
        for n in (64, 1, 33, 64, 1):
            res, info = c.render_batch([s] * n, ps[:n])
            for (a, px), ref in zip(res, alone):
                assert np.array_equal(a, ref[0], equal_nan=True) and np.array_equal(px, ref[1])
            assert info["segments"] == sum(r[2]["segments"] for r in alone[:n])
        s.free()


@pytest.mark.parametrize("name", ["cornell", "tiny", "gold", "medium"])
@pytest.mark.parametrize("tri", ["mt", "watertight"])
@pytest.mark.parametrize("w,h,spp", [(65, 63, 1), (61, 67, 7), (40, 30, 64)])
def test_packets_over_fnodes_match_lanes(name, tri, w, h, spp):
    """Packets whose directions share an octant and packets that straddle an axis (the image's middle,
    rotated and unrotated instances), last packets that are not full, spheres; one scene and several."""
    spec, st = SCENES[name]()
    other, _ = S.tiny_mesh_scene(n=3)
    p = render_params(**dict(st, width=w, height=h, spp=spp, max_depth=2))
    out = []
    for packets in (1, 2):
        with illume_amd.Context(0, extend_mode=3, camera_packets=packets, tri_test=tri) as c:
            s, t = c.scene(spec), c.scene(other)
            both, info = c.render_batch([s, t, s], [p, p, p])
            out.append((c.render(s, p), both, info["segments"]))
            s.free()
            t.free()
    (a, b) = out
    assert np.array_equal(a[0][0], b[0][0], equal_nan=True) and np.array_equal(a[0][1], b[0][1])
    assert a[0][2]["segments"] == b[0][2]["segments"] and a[2] == b[2]
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(x[0], y[0], equal_nan=True) and np.array_equal(x[1], y[1])


@pytest.mark.parametrize("scenes,opts", [(2, {}), (6, {}), (2, dict(sched_fair=1)), (2, dict(pipes=1)), (2, dict(chunk_passes=3))])
def test_requests_of_several_scenes_in_chunks_of_their_own(scenes, opts):
    """Work of 2^19 paths and more per scene runs as one chunk per scene while few scenes have work, and
    joined otherwise: the images and the segment count are those of the requests alone either way."""
    names = ["tiny", "cornell", "gold", "tiny", "cornell", "tiny"][:scenes]
    with illume_amd.Context(0, **opts) as c:
        sc = [c.scene(SCENES[n]()[0]) for n in names]
        ps = [render_params(**dict(SCENES[n]()[1], width=400 + 8 * i, height=300, spp=6 - i % 3, max_depth=4 + i))
              for i, n in enumerate(names)]
        sc, ps = sc + sc[:1], ps + [render_params(**dict(SCENES["tiny"]()[1], width=31, height=17, spp=3, max_depth=5))]
        alone = [c.render(s, p) for s, p in zip(sc, ps)]
        res, info = c.render_batch(sc, ps)
        hs = [c.submit(s, p) for s, p in zip(sc, ps)]
        served = []
        for h in hs:
            h.wait(60000)
            served.append(h.result())
            h.free()
        for (a, px), (b, bx), ref in zip(res, served, alone):
            for x, y in ((a, ref[0]), (b, ref[0]), (px, ref[1]), (bx, ref[1])):
                assert np.array_equal(x, y, equal_nan=x.dtype == np.float32)
        assert info["segments"] == sum(r[2]["segments"] for r in alone)
        for s in sc[:-1]:
            s.free()


def test_renders_that_follow_their_counts_match_when_interleaved():
    """Renders whose depths are launched by the counts of the depths before them: one after another with
    other depths and sizes (a count left by an earlier render is not taken for a later one's), from two
    threads on two contexts, against contexts that launch every depth."""
    import threading
    reqs = [("medium", 400, 300, 3, 45), ("tiny", 520, 510, 1, 2), ("medium", 512, 513, 1, 3), ("tiny", 400, 300, 3, 4),
            ("cornell", 512, 513, 1, 5), ("medium", 333, 251, 7, 45), ("tiny", 640, 480, 2, 12)]
    with illume_amd.Context(0, extend_mode=3) as c:
        sc = {k: c.scene(SCENES[k]()[0]) for k in SCENES}
        ref = [c.render(sc[r[0]], render_params(**dict(SCENES[r[0]]()[1], width=r[1], height=r[2], spp=r[3], max_depth=r[4])))
               for r in reqs]
        for s in sc.values():
            s.free()
    bad = []

    def work(order):
        with illume_amd.Context(0) as c:
            sc = {k: c.scene(SCENES[k]()[0]) for k in SCENES}
            for i in order:
                k, w, h, spp, depth = reqs[i]
                p = render_params(**dict(SCENES[k]()[1], width=w, height=h, spp=spp, max_depth=depth))
                for call in (c.render, c.render_noalloc):
                    a, px, info = call(sc[k], p)
                    if not (np.array_equal(a, ref[i][0], equal_nan=True) and np.array_equal(px, ref[i][1]) and
                            info["segments"] == ref[i][2]["segments"]):
                        bad.append((call.__name__, reqs[i]))
            for s in sc.values():
                s.free()

    n = len(reqs)
    ts = [threading.Thread(target=work, args=(o,)) for o in (list(range(n)) * 2, list(range(n))[::-1] * 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
