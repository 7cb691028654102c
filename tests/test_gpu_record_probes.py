"""The timed probes of a renderer in steady use (cell cache, compiled kernel)
run the launch they choose for: with miss records where the render takes them,
their binning included and every walker at its end.  They leave no trace:
renders around them equal those without records or probes, in a record memory
that holds every miss and in one so small that the probes' walkers pause."""

import json
import re

import numpy as np
import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu

SAMPLES, BATCH = 32768 * 300, 300


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("probe", ["FFR_CACHE_PROBE_SAMPLES", "FFR_COMPILED_PROBE_SAMPLES"])
def test_probes_with_records(ffr_mod, monkeypatch, probe, precision, small):
    print(f"record probes {probe} {precision} small={small}", flush=True)
    text = read_flame("batch/flame_1069.json")
    kw = dict(precision=precision, seed=9, batch_size=BATCH, binned=0)
    monkeypatch.setenv("FFR_MISS", "0")
    b = ffr_mod.BufferRenderer(text, compiled=0, **kw)
    monkeypatch.setenv("FFR_MISS", "1")
    a = ffr_mod.BufferRenderer(text, **kw)
    monkeypatch.setenv(probe, "1")
    if small:
        monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 22))
    for k in range(4):  # (the second render probes)
        assert a.render(SAMPLES)
        monkeypatch.delenv(probe)
        assert b.render(SAMPLES)
        monkeypatch.setenv(probe, "1")
        if a.last_stats.cache_slots:
            records, pauses = a.record_use
            assert records > 0 and (pauses > 0) == small
        wa, wb = a.read_buffer(), b.read_buffer()
        assert np.array_equal(a.counts(wa), b.counts(wb))
        n = a.counts(wa).astype(np.float64).reshape(-1, 1)
        ca, cb = a.colors(wa), b.colors(wb)
        assert np.all(np.abs(ca - cb) <= n * 2.0 ** -52 * np.abs(cb))
        assert a.samples_iterated == b.samples_iterated
        assert a.samples_plotted == b.samples_plotted
        assert np.array_equal(a.xform_distribution(), b.xform_distribution())
    a.close()
    b.close()


def test_probe_is_not_cut_short(ffr_mod, monkeypatch):
    """In a record memory that its walkers use up at once, a cached launch takes
    many rounds and the launch without the cache is far faster; a probe that
    timed the first round alone would keep the cache."""
    print("record probe with pauses", flush=True)
    d = json.loads(re.sub(r"^\s*//.*$", "", read_flame("batch/flame_1069.json"), flags=re.M))
    for key in ("color_dimensions", "color_speed"):
        d.pop(key, None)
    for x in d["xforms"]:
        x.pop("color")
    monkeypatch.setenv("FFR_MISS", "1")
    monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 22))
    monkeypatch.setenv("FFR_CACHE_PROBE_SAMPLES", "1")
    r = ffr_mod.BufferRenderer(json.dumps(d), precision="fp32", seed=9, batch_size=1024,
                               binned=0, compiled=0)
    assert r.render(24576 * 1024) and r.record_use[1] > 0
    assert r.render(24576 * 1024) and r.last_stats.cache_slots == 0
    r.close()
