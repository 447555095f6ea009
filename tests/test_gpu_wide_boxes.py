"""Quantised boxes of the 8-wide nodes, byte by byte against a float64
restatement, where levels end before, at and past a workgroup's 64 nodes; and a
refit of unmoved triangles, which writes the same nodes again."""
import numpy as np
import pytest

from realtimeraytracing_amd import scenes

pytestmark = pytest.mark.gpu


def _exponent(extent):
    e = -126
    while e < 127 and np.ldexp(255.0, e) < extent:
        e += 1
    return e


def _restated(raw, cl, n, pad):
    """Words 0-15 of every node, from the exported cluster boxes."""
    none, f32 = 0xFFFFFFFF, np.float32
    left, right, boxes = cl["left"], cl["right"], cl["boxes"]
    nc = 2 * n - 1
    count, first = np.ones(nc, np.int64), np.zeros(nc, np.int64)
    for c in range(nc):
        if left[c] != none:
            count[c] = count[left[c]] + count[right[c]]
    for c in range(nc - 1, -1, -1):
        if left[c] != none:
            first[left[c]] = first[c]
            first[right[c]] = first[c] + count[left[c]]
    cluster = {(int(first[c]), int(count[c])): c for c in range(nc)}
    ranges = [None] * len(raw)
    out = np.zeros((len(raw), 16), np.uint32)
    for k in range(len(raw) - 1, -1, -1):
        kids = []
        for j in range(bin(int(raw[k, 3]) >> 24).count("1")):
            ref = int(raw[k, 16 + j])
            kids.append(((ref >> 3) & 0x0FFFFFFF, (ref & 7) + 1) if ref & 0x80000000 else ranges[ref])
        ranges[k] = (kids[0][0], sum(c for _, c in kids))
        b = boxes[[cluster[r] for r in kids]]
        lo, hi = b["min"] - f32(pad), b["max"] + f32(pad)
        org, top = lo.min(axis=0), hi.max(axis=0)
        planes = np.zeros((3, 2, 8), np.uint8)
        planes[:, 0] = 255
        meta = ((1 << len(kids)) - 1) << 24
        for q in range(3):
            e = _exponent(float(top[q]) - float(org[q]))
            meta |= (e + 127) << (8 * q)
            for side, v, up in ((0, lo, np.floor), (1, hi, np.ceil)):
                g = up((v[:, q].astype(np.float64) - float(org[q])) / np.ldexp(1.0, e))
                planes[q, side, :len(kids)] = np.clip(g, 0, 255).astype(np.uint8)
        out[k, :3] = org.view(np.uint32)
        out[k, 3] = meta
        out[k, 4:] = planes.reshape(-1).view(np.uint32)
    return out


@pytest.mark.parametrize("n,leaf", [(1, 1), (2, 1), (9, 1), (64, 1), (450, 1), (513, 1), (700, 2), (6000, 4)])
def test_wide_boxes(rtq_ctx, n, leaf):
    sc = rtq_ctx.upload(scenes.soup(n, seed=3 * n), scenes.identity_models())
    try:
        info = sc.build(16, leaf, 0, node_width=8)
        raw = sc.export_wide()
        want = _restated(raw, sc.export_clusters(), n, info.box_pad)
        assert np.array_equal(raw[:, :16], want)
        sc.refit()
        assert np.array_equal(sc.export_wide(), raw)
    finally:
        sc.release()
