"""Results come back as packed sums and pixel words through pinned memory, in pieces unpacked by
several threads: every pixel of every output equals the direct copies of render_noalloc."""
import threading

import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from illume_amd._abi import render_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cornell():
    with illume_amd.Context(0) as c:
        spec, st = S.cornell()
        s = c.scene(spec)
        yield c, s, st
        s.free()


def _p(st, w, h, **kw):
    return render_params(**dict(st, width=w, height=h, spp=1, max_depth=2, **kw))


# 1 to 5 pixels, a thread's 16384, one more piece than fits a whole number of 2^18 pixels
@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (128, 128), (127, 129), (512, 512), (513, 512), (1031, 767)])
def test_results_of_every_size_equal_direct_copies(cornell, w, h):
    c, s, st = cornell
    p = _p(st, w, h)
    a, px, _ = c.render(s, p)
    ref_a, ref_px, _ = c.render_noalloc(s, p)
    assert np.array_equal(a, ref_a) and np.array_equal(px, ref_px)
    assert px.max() > 0 or w * h < 100            # the picture is not all black
    a2, none, _ = c.render(s, p, want_pixels=False)
    none2, px2, _ = c.render(s, p, want_accum=False)
    assert none is None and none2 is None and np.array_equal(a2, a) and np.array_equal(px2, px)
    r = c.submit(s, p)
    r.wait(60000)
    a3, px3 = r.result()
    r.free()
    assert np.array_equal(a3, a) and np.array_equal(px3, px)


def test_batch_results_over_several_rounds(cornell):
    """More pieces than one round of staging holds (64), and more bytes (64 MB)."""
    c, s, st = cornell
    sizes = [(17 + k, 9) for k in range(70)] + [(1920, 1080)] * 3
    ps = [_p(st, w, h, first_sample=k) for k, (w, h) in enumerate(sizes)]
    out, _ = c.render_batch([s] * len(ps), ps)
    for p, (a, px) in list(zip(ps, out))[::9] + [(ps[-1], out[-1]), (ps[-2], out[-2])]:
        ref_a, ref_px, _ = c.render(s, p)
        assert np.array_equal(a, ref_a) and np.array_equal(px, ref_px)


def test_results_of_two_threads(cornell):
    """Two callers of one context: each gets its own image."""
    c, s, st = cornell
    ps = [_p(st, 640, 480), _p(st, 900, 700, first_sample=5)]
    ref = [c.render(s, p) for p in ps]
    bad = []

    def go(k):
        for _ in range(8):
            a, px, info = c.render(s, ps[k])
            if not (np.array_equal(a, ref[k][0]) and np.array_equal(px, ref[k][1])):
                bad.append(k)
    th = [threading.Thread(target=go, args=(k,)) for k in (0, 1)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not bad
