"""rtq_trace_host at the sizes where its buffers change (pinned host memory, the
context's scratch, the call's own): the records of the same rays traced in
device memory, also after a call of another size and a refused one."""
import numpy as np
import pytest

from realtimeraytracing_amd import HIT_DTYPE, RTQ_TRACE_ANY, RtqError, devmem, scenes
from conftest import first_diff, hits_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(rtq_ctx):
    sc = rtq_ctx.upload(*scenes.soup_scene(2000, seed=21))
    sc.build()
    yield sc
    sc.release()


@pytest.mark.parametrize("n", [1, 63, 32_767, 32_768, 32_769, 262_144, 262_145])
def test_host_sizes(rtq_ctx, scene, n):
    rays = scenes.random_rays(n, n, (0, 0, 0), (1, 1, 1))
    rays["tmax"][::3] = 0.3
    d, h = devmem.to_device(rays), devmem.empty(n, HIT_DTYPE)
    for flags in (0, RTQ_TRACE_ANY):
        scene.trace(d.data_ptr(), n, h.data_ptr(), flags)
        rtq_ctx.synchronize()
        want = devmem.to_host(h, HIT_DTYPE)
        got = scene.trace_host(rays, flags)
        assert hits_equal(got, want), first_diff(got, want)
    with pytest.raises(RtqError):
        scene.trace_host(rays, 1 << 30)
    assert np.array_equal(scene.trace_host(rays[:1], RTQ_TRACE_ANY), want[:1])
