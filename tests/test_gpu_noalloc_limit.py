"""The largest image ilm_render_noalloc takes: 56 bytes a pixel beside 4096 paths, the chunk
descriptor and 2 KB of control block in the 128 MiB of the documented array."""
import numpy as np
import pytest

import illume_amd
import illume_amd.scenes as S
from illume_amd._abi import render_params

pytestmark = pytest.mark.gpu


def test_images_up_to_the_documented_limit_render():
    spec, st = S.cornell()
    with illume_amd.Context(0, paths_in_flight=1 << 20) as c:
        s = c.scene(spec)
        p = render_params(**dict(st, width=1567, height=1522, spp=1, max_depth=2))    # 10 pixels under
        ref, ref_px, ri = c.render(s, p)
        got, px, gi = c.render_noalloc(s, p)
        assert np.array_equal(got, ref) and np.array_equal(px, ref_px) and gi["segments"] == ri["segments"]
        assert gi["chunks"] > 100
        with pytest.raises(illume_amd.IlmError) as e:                                 # 1 pixel over
            c.render_noalloc(s, render_params(**dict(st, width=1115, height=2139, spp=1, max_depth=2)))
        assert e.value.code == -9
        s.free()
