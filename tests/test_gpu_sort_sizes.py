"""Radix sort at the sizes where its path changes: one workgroup with 2 or 8
pairs per thread, tiles of 2,048 pairs, tiles of 8,192, and the remainders of
each; every number of digit passes; keys of one digit and of few values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _keys(rng, n, bits, kind):
    top = (1 << bits) - 1
    if kind == "random":
        return rng.integers(0, top, n, dtype=np.uint32, endpoint=True)
    if kind == "equal":
        return np.full(n, top, np.uint32)
    if kind == "few":
        return (rng.integers(0, 3, n, dtype=np.uint32) * np.uint32(top // 2)).astype(np.uint32)
    return np.sort(rng.integers(0, top, n, dtype=np.uint32, endpoint=True))[::-1].copy()


@pytest.mark.parametrize("kind", ["random", "equal", "few", "descending"])
@pytest.mark.parametrize("n,bits", [
    (1, 32), (63, 8), (64, 30), (65, 16), (1024, 24), (2047, 30), (2048, 32), (2049, 30), (8191, 16), (8192, 24),
    (8193, 30), (10240, 8), (10241, 24), (524287, 30), (524288, 16), (524289, 30), (532480, 24), (532481, 8)])
def test_sort_sizes(rtq_ctx, torch_mod, n, bits, kind):
    torch = torch_mod
    keys = _keys(np.random.default_rng(n + bits), n, bits, kind)
    vals = np.arange(n, dtype=np.uint32)
    dk = torch.from_numpy(keys.view(np.int32).copy()).cuda()
    dv = torch.from_numpy(vals.view(np.int32).copy()).cuda()
    rtq_ctx.sort_pairs(dk.data_ptr(), dv.data_ptr(), n, bits)
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(dk.cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(dv.cpu().numpy().view(np.uint32), vals[order])


@pytest.mark.parametrize("kind", ["random", "few"])
def test_sort_with_one_set_of_status_words(rtq_ctx, torch_mod, kind):
    """Past 2,048 tiles the passes share one set of look-back words, cleared before
    each."""
    test_sort_sizes(rtq_ctx, torch_mod, 2049 * 8192 - 5, 32, kind)
