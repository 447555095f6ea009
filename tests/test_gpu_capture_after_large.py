"""A launch sizes the traversal scratch for every launch of fewer rays on the same
nodes, which may then be captured, under the default chunks and under chunks so
long that the large launch itself has few of them."""
import numpy as np
import pytest

from realtimeraytracing_amd import HIT_DTYPE, Context, devmem, scenes
from conftest import hits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [128, 4096])
def test_fewer_rays_captured(torch_mod, chunk):
    torch = torch_mod
    many, fewer, base = 8_400_000, [2_000_000, 300_000, 5000], 40_000
    with Context(0) as ctx:
        ctx.set_launch_params(refill=32, chunk=chunk)
        sc = ctx.upload(*scenes.soup_scene(60_000, seed=6))
        assert sc.build().depth > 14      # more than the stack entries in LDS
        rays = devmem.to_device(scenes.random_rays(base, 7, (0, 0, 0), (1, 1, 1))).repeat(many // base)
        hits = devmem.empty(many, HIT_DTYPE)
        torch.cuda.synchronize()
        sc.trace(rays.data_ptr(), many, hits.data_ptr())
        ctx.synchronize()
        want = devmem.to_host(hits[:max(fewer) * HIT_DTYPE.itemsize], HIT_DTYPE)
        for n in fewer:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                sc.trace(rays.data_ptr(), n, hits.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
            for _ in range(3):
                hits.zero_()
                graph.replay()
                torch.cuda.synchronize()
                got = devmem.to_host(hits[:n * HIT_DTYPE.itemsize], HIT_DTYPE)
                assert hits_equal(got, want[:n])
        assert np.count_nonzero(want["id"] >= 0) > 0
