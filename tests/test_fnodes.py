"""The FP32 BVH4 layout (FNodes) against the FP32 BVH2 nodes it is collapsed from (CPU)."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from deep_mesh import DEEP, shrinking_clusters

NO_CHILD = 0x7FFFFFFF
FLT_MAX = np.finfo(np.float32).max


def _grid(n):
    return dict(positions=np.random.default_rng(n).uniform(-1, 1, (3 * n, 3)).astype(np.float32),
                indices=np.arange(3 * n, dtype=np.int32).reshape(-1, 3))


def _mesh(name):
    if name in DEEP:
        v, i = shrinking_clusters(*DEEP[name])
        return dict(positions=v, indices=i)
    if name == "flat":      # coplanar, many equal centroids: boxes without volume, median splits
        m = _grid(900)
        m["positions"][:, 2] = 0.0
        m["positions"][:900] = m["positions"][0]
        return m
    return S.displaced_icosphere(name[1], 3) if name[0] == "sphere" else _grid(name[1])


@pytest.mark.parametrize("name", [("soup", 0), ("soup", 1), ("soup", 4), ("soup", 5), ("soup", 17), ("soup", 3000),
                                  ("sphere", 3), ("sphere", 40), "flat", 21, 23])
def test_fnodes_hold_the_bvh2_boxes_and_leaves(name):
    m = _mesh(name)
    pos, idx = m["positions"], m["indices"]
    b = illume_amd.bvh_build(pos, idx)
    raw, _, _, (root, _, depth, _), _ = illume_amd.bvh_device_layouts(pos, idx)
    box, child = b["f_boxes"], b["f_child"]
    assert (b["f_levels"] == 0) == (len(child) == 0)
    if root < 0 or root == NO_CHILD:      # a leaf or nothing: no FNodes
        assert len(child) == 0 and b["f_root"] == root
        return
    w = raw.view(np.float32).reshape(-1, 16)
    bchild = raw.view(np.int32).reshape(-1, 16)[:, 12:14]
    bbox = np.stack([w[:, [0, 2, 4, 1, 3, 5]], w[:, [6, 8, 10, 7, 9, 11]]], 1)

    def area(q):
        e = q[3:].astype(np.float64) - q[:3]
        return 0.0 if (e < 0).any() else e[0] * e[1] + e[1] * e[2] + e[2] * e[0]

    assert b["f_root"] == 0
    seen, leaves, levels, worst = set(), [], 0, 0
    todo = [(0, root, 1, 0)]              # FNode, BNode it was collapsed from, level, entries pending above
    while todo:
        f, n, level, pending = todo.pop()
        assert f not in seen
        seen.add(f)
        levels = max(levels, level)
        kids = [(bchild[n, 0], bbox[n, 0]), (bchild[n, 1], bbox[n, 1])]
        while len(kids) < 4:              # the inner child of largest area opens, the first of equal ones
            a = [area(q) if 0 <= c != NO_CHILD else -1.0 for c, q in kids]
            k = int(np.argmax(a))
            if a[k] < 0:
                break
            c = kids[k][0]
            kids[k:k + 1] = [(bchild[c, 0], bbox[c, 0]), (bchild[c, 1], bbox[c, 1])]
        worst = max(worst, pending + len(kids) - 1)
        for k in range(4):
            if k >= len(kids):
                assert child[f, k] == NO_CHILD
                assert np.all(box[f, k, :3] == FLT_MAX) and np.all(box[f, k, 3:] == -FLT_MAX)
                continue
            c, q = kids[k]
            assert np.array_equal(box[f, k], q)
            if c < 0:
                assert child[f, k] == c
                leaves.append(c)
            else:
                assert child[f, k] > f     # breadth first
                todo.append((int(child[f, k]), int(c), level + 1, pending + len(kids) - 1))
    assert seen == set(range(len(child)))
    assert sorted(leaves) == sorted(int(c) for c in bchild.ravel() if c < 0)      # every leaf once
    assert b["f_levels"] == levels <= max(depth, 1)
    # what the device's stacks are sized by: a node leaves at most three entries behind
    assert worst <= 3 * levels
    if name in DEEP:
        assert levels == name
