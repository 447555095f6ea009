"""How a launch's rays are split into chunks, XCD queues and waves: every ray is
traced and nothing else is written, at the edges of the split (a few rays, fewer
than the XCDs, one wave per SIMD, the step to waves of 200 rays, chunks of one
ray and of more rays than an XCD's part) and with items of uneven sizes."""
import numpy as np
import pytest

import oracle
from realtimeraytracing_amd import HIT_DTYPE, RAY_DTYPE, RTQ_TRACE_ANY, Context, devmem, scenes
from conftest import first_diff, hits_equal

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 63, 64, 65, 1021, 2047, 2049, 65535, 65536, 65537, 300001, 819201, 1400003]
MOST = SIZES[-1]
POISON = 0xA5


class Work:
    def __init__(self):
        tris, models = scenes.soup_scene(700, seed=3)
        base = scenes.random_rays(20000, 5, (0, 0, 0), (1, 1, 1))
        self.ctx = Context(0)
        self.scene = self.ctx.upload(tris, models)
        self.scene.build(node_width=8)
        want, _, _ = oracle.trace_bvh(self.scene.export_ref(), oracle.world_vertices(tris, models), base)
        at = np.arange(MOST) % len(base)      # neighbours differ, and so do equal offsets of two parts
        self.want = want[at]
        self.rays = devmem.to_device(base[at])
        self.hits = devmem.empty(MOST + 16, HIT_DTYPE)

    def poison(self):
        self.hits.fill_(POISON)
        devmem.synchronize()

    def check(self, n, any_hit=False, at=0):
        self.ctx.synchronize()
        got = devmem.to_host(self.hits, HIT_DTYPE)
        if any_hit:
            assert np.array_equal(got["id"][at:at + n] >= 0, self.want["id"][at:at + n] >= 0)
        else:
            assert hits_equal(got[at:at + n], self.want[at:at + n]), first_diff(got[at:at + n], self.want[at:at + n])
        return got


@pytest.fixture(scope="module")
def work(rtq_ctx):   # a context of its own: the launch settings are changed
    w = Work()
    yield w
    w.ctx.close()


@pytest.mark.parametrize("n", SIZES)
def test_every_ray_once(work, n):
    for flags in (0, RTQ_TRACE_ANY):
        for call in (work.scene.trace, work.scene.trace_noalloc):
            for _ in range(2):    # the counters are as the first launch found them
                work.poison()
                call(work.rays.data_ptr(), n, work.hits.data_ptr(), flags)
                got = work.check(n, flags != 0)
                assert (got[n:].view(np.uint8) == POISON).all()


@pytest.mark.parametrize("chunk", [1, 3, 64, 65, 4096])
def test_chunk_setting(work, chunk):
    try:
        work.ctx.set_launch_params(32, chunk)
        for n in (9, 2049, 70001):
            work.poison()
            work.scene.trace(work.rays.data_ptr(), n, work.hits.data_ptr())
            work.check(n)
    finally:
        work.ctx.set_launch_params(32, 128)


@pytest.mark.parametrize("sizes", [[1], [0, 5, 0, 1], [1] * 64, [100000, 3, 0, 70001, 8], [1000] * 63 + [400000]])
def test_items_of_uneven_sizes(work, sizes):
    ray, hit = RAY_DTYPE.itemsize, HIT_DTYPE.itemsize
    specs, at = [], 0
    for n in sizes:
        specs.append((work.scene, work.rays.data_ptr() + at * ray, n, work.hits.data_ptr() + at * hit, 0))
        at += n
    items = work.ctx.items(specs)
    batch = work.ctx.batch(items)
    try:
        for launch in (lambda: work.ctx.trace_batch(items), batch.launch, batch.launch):
            work.poison()
            launch()
            got = work.check(at)
            assert (got[at:].view(np.uint8) == POISON).all()
    finally:
        batch.destroy()
