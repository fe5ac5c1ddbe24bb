"""Meshes whose trees are deep for their size: clusters of small triangles that shrink geometrically
towards the origin, each holding more triangles than the ones inside it together need, so the builder
splits off one cluster after another."""
import numpy as np


def shrinking_clusters(scales, ratio, growth, smallest, seed=5):
    rng = np.random.default_rng(seed)
    tris = []
    for k in range(scales):
        n = int(smallest * growth ** (scales - 1 - k))
        c = np.stack([rng.uniform(1, 1.5, n), rng.uniform(0, 1, n), rng.uniform(0, 1, n)], 1)
        tris.append(ratio ** -k * (c[:, None, :] + rng.uniform(-.04, .04, (n, 3, 3))))
    v = np.concatenate(tris).reshape(-1, 3).astype(np.float32)
    return v, np.arange(len(v), dtype=np.int32).reshape(-1, 3)


# FNodes on the longest path from the root: a lone instance's walk over FNodes then holds at most
# 3 * levels + 1 entries, 64 and 70 of the 64 its stacks have
DEEP = {21: (24, 1.8, 1.31, 8), 23: (22, 1.8, 1.31, 16)}
