"""Batches of basic-variation flames with one to four colours: one kernel
kind holds them all (kinds run one after another), and each renders what it
renders alone: counts and statistics exactly, colour sums to the rounding of
their order of addition (a sum of n terms of one sign is off by at most
n * 2^-53 of itself, so two orders by n * 2^-52, n the cell's count)."""

import json
import re

import numpy as np
import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu


def flame(k, colours, size):
    d = json.loads(re.sub(r"^\s*//.*$", "", read_flame("batch/flame_%d.json" % k), flags=re.M))
    d["color_dimensions"], d["size"] = colours, [size, size]
    for x in d["xforms"]:
        x["color"] = (x["color"] + [0.25, 0.75])[:colours]
    return json.dumps(d)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("colours, kinds", [([3, 3, 3], 1), ([1, 3, 2, 4, 3], 1),
                                            ([0, 3, 4], 2), ([3, 5], 2)])
def test_colour_counts_share_a_kind(ffr_mod, precision, colours, kinds):
    print(f"batch kinds {precision} {colours}", flush=True)
    texts = [flame(1040 + i, c, 300 + 7 * i) for i, c in enumerate(colours)]
    samples = [9_000_001 + 1000 * i for i in range(len(texts))]
    rs, alone = ([ffr_mod.BufferRenderer(t, precision=precision, seed=i, batch_size=1024)
                  for i, t in enumerate(texts)] for _ in range(2))
    with ffr_mod.Batch(rs) as batch:
        assert len(batch.shapes()) == kinds
        for _ in range(2):
            assert all(batch.render(samples))
    for a, b, n in zip(rs, alone, samples):
        assert b.render(n) and b.render(n)
        wa, wb = a.read_buffer(), b.read_buffer()
        assert np.array_equal(a.counts(wa), b.counts(wb))
        assert a.samples_plotted == b.samples_plotted
        assert np.array_equal(a.xform_distribution(), b.xform_distribution())
        if a.color_dims:
            ca, cb = a.colors(wa), b.colors(wb)
            n = a.counts(wa).astype(np.float64).reshape(-1, 1)
            assert np.all(np.abs(ca - cb) <= n * 2.0 ** -52 * np.abs(cb))
        a.close()
        b.close()


def test_launches_are_counted(ffr_mod, monkeypatch):
    """one per kind, and those of the rounds of miss records"""
    print("batch launches", flush=True)
    monkeypatch.setenv("FFR_MISS", "0")
    rs = [ffr_mod.BufferRenderer(flame(1069, c, 1000), precision="fp32", seed=1, batch_size=256)
          for c in (0, 3)]
    n = 30000 * 256
    with ffr_mod.Batch(rs) as batch:
        assert all(batch.render([n, n])) and batch.last_stats.launches == 2
    monkeypatch.setenv("FFR_MISS", "1")
    with_records = [ffr_mod.BufferRenderer(flame(1069, c, 1000), precision="fp32", seed=1,
                                           batch_size=256) for c in (0, 3)]
    with ffr_mod.Batch(with_records) as batch:
        assert all(batch.render([n, n])) and batch.last_stats.launches == 2  # a round each
        monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 22))
        assert all(batch.render([n, n]))
        assert any(r.record_use[1] for r in with_records) and batch.last_stats.launches > 4
    for r in rs + with_records:
        r.close()
