"""Results where the system gives no pinned memory, or less than a round of a batch asks for: plain and
batched renders return the same images through pageable copies, served requests are refused."""
import time

import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from illume_amd._abi import render_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def box():
    with illume_amd.Context(0, paths_in_flight=1 << 22) as c:
        spec, st = S.cornell()
        s = c.scene(spec)
        yield c, s, st
        s.free()


def _p(st, w, h, **kw):
    return render_params(**dict(st, width=w, height=h, spp=1, max_depth=2, **kw))


# bytes of the largest pinned buffer: none, one piece of 2^18 pixels, nearly a whole round
@pytest.mark.parametrize("limit", [0, 4 << 20, 60 << 20])
def test_results_without_pinned_memory(box, limit):
    c, s, st = box
    L = illume_amd.lib()
    # one pixel; a piece of 2^18 pixels and one more row; 12 MB in small images, then more than a round
    sizes = [(1, 1), (3, 1), (512, 513)] + [(400 + k, 300) for k in range(6)] + [(1920, 1080)] * 3
    ps = [_p(st, w, h, first_sample=k) for k, (w, h) in enumerate(sizes)]
    ref = [c.render(s, p) for p in ps]
    served = c.submit(s, ps[2])
    served.wait(60000)
    try:
        assert L.ilm_debug_pinned_limit(c.h, limit) == 0
        for p, (a, px, _) in zip(ps, ref):
            a1, px1, _ = c.render(s, p)
            a2, none, _ = c.render(s, p, want_pixels=False)
            none2, px2, _ = c.render(s, p, want_accum=False)
            assert none is None and none2 is None
            assert np.array_equal(a1, a) and np.array_equal(px1, px)
            assert np.array_equal(a2, a) and np.array_equal(px2, px)
        out, _ = c.render_batch([s] * len(ps), ps)
        for (a, px), r in zip(out, ref):
            assert np.array_equal(a, r[0]) and np.array_equal(px, r[1])
        t = time.perf_counter()
        c.render(s, ps[-1])
        print("1920x1080 with pinned buffers of at most %d MB: %.1f ms" % (limit >> 20, 1e3 * (time.perf_counter() - t)))
        # a result that was there before stays readable; a new request of that size is refused
        a, px = served.result()
        assert np.array_equal(a, ref[2][0]) and np.array_equal(px, ref[2][1])
        if limit < 16 * 1920 * 1080:
            with pytest.raises(illume_amd.IlmError) as e:
                c.submit(s, ps[-1])
            assert e.value.code == -2
    finally:
        assert L.ilm_debug_pinned_limit(c.h, (1 << 63) - 1) == 0
        served.free()
    a, px, _ = c.render(s, ps[-1])
    assert np.array_equal(a, ref[-1][0]) and np.array_equal(px, ref[-1][1])
    t = time.perf_counter()
    c.render(s, ps[-1])
    print("1920x1080 with pinned memory: %.1f ms" % (1e3 * (time.perf_counter() - t)))
