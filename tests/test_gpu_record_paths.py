"""Miss records in the kernels that renders run on them: each case forces the
records (FFR_MISS=1) and checks that they were made, and in a small record
memory that workgroups paused for their binning; buffers and statistics then
equal those of the same render with every miss an atomic (FFR_MISS=0,
table-driven kernels; the compiled kernel of the catalogue flame is compared
with itself, as its FP32 trigonometry rounds otherwise than the table-driven
kernel's).  Counts and statistics exactly, colour sums to the
rounding of their order of addition: a sum of n terms of one sign is off by at
most n * 2^-53 of itself, so two orders by n * 2^-52, n the cell's count.

Kernels: three colours of the basic variations (three colour registers), one
and four; counts; the whole catalogue's kernel; more transforms than the byte
counters hold; the flame's compiled kernel; tasks of several walkers a lane; a
bad-value limit that is reached while records wait."""

import json
import re

import numpy as np
import pytest

import flames as TF
from conftest import read_flame

pytestmark = pytest.mark.gpu

SEED = 0x5EED0031
SAMPLES, BATCH = 5_000_011, 211  # 23697 walkers, the last of 55 samples


def basic(colours, size, repeat=1):
    d = json.loads(re.sub(r"^\s*//.*$", "", read_flame("batch/flame_1069.json"), flags=re.M))
    d["size"] = [size, size - 7]
    d["xforms"] = [json.loads(json.dumps(x)) for x in d["xforms"] for _ in range(repeat)]
    for k, x in enumerate(d["xforms"]):
        x["weight"] *= 1.0 + 0.1 * k
        x["color"] = (x["color"] + [0.25])[:colours]
    if colours:
        d["color_dimensions"] = colours
    else:
        for key in ("color_dimensions", "color_speed"):
            d.pop(key, None)
        for x in d["xforms"]:
            x.pop("color")
    return json.dumps(d)


def catalogue(colours):
    d = json.loads(basic(colours, 900))
    for x, n in zip(d["xforms"], ("bent", "handkerchief", "julian", "pdj", "blob", "rings") * 2):
        x["variations"] = [TF.variation(n, 0.5, 2), TF.variation("sinusoidal", 0.5, 2)]
    return json.dumps(d)


FLAMES = {
    "basic_c3": lambda: basic(3, 1200),
    "basic_c1": lambda: basic(1, 1200),
    "basic_c4": lambda: basic(4, 1200),
    "basic_counts": lambda: basic(0, 1200),
    "basic_many_xforms": lambda: basic(3, 1200, repeat=4),
    "catalogue_c3": lambda: catalogue(3),
    "catalogue_counts": lambda: catalogue(0),
    "linear_c3": lambda: TF.color_flame(3, size=1200),
}
MODES = {"fp32": dict(precision="fp32"), "fp64": dict(precision="fp64"),
         "u32": dict(precision="fp32", word=32)}


def same_buffers(a, b):
    wa, wb = a.read_buffer(), b.read_buffer()
    assert np.array_equal(a.counts(wa), b.counts(wb))
    if a.color_dims:
        ca, cb = a.colors(wa), b.colors(wb)
        n = a.counts(wa).astype(np.float64).reshape(-1, 1)
        assert np.all(np.abs(ca - cb) <= n * 2.0 ** -52 * np.abs(cb))
    assert a.samples_iterated == b.samples_iterated
    assert a.samples_plotted == b.samples_plotted
    assert np.array_equal(a.xform_distribution(), b.xform_distribution())
    assert a.point_extremes == b.point_extremes
    assert a.last_stats.n_bad == b.last_stats.n_bad


def make(ffr, monkeypatch, text, records, **kw):
    monkeypatch.setenv("FFR_MISS", "1" if records else "0")
    r = ffr.BufferRenderer(text, seed=SEED, batch_size=BATCH, binned=0, **kw)
    monkeypatch.delenv("FFR_MISS")
    return r


def missed(r):
    s = r.last_stats
    return (s.atomics - s.flush_atomics) // r.cell_words


def check(ffr, monkeypatch, text, small, compiled, reference=0, **kw):
    a = make(ffr, monkeypatch, text, True, compiled=compiled, **kw)
    b = make(ffr, monkeypatch, text, False, compiled=reference, **kw)
    if small:
        monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 21))
    for _ in range(2):
        assert a.render(SAMPLES) and b.render(SAMPLES)
        assert a.last_stats.compiled == compiled
        records, pauses = a.record_use
        assert b.record_use == (0, 0)
        if small:
            assert 0 < records <= missed(a) and pauses > 0
        else:
            assert records == missed(a) > 0 and pauses == 0
        same_buffers(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("name", sorted(FLAMES))
def test_table_kernels(ffr_mod, monkeypatch, name, mode, small):
    if mode == "u32" and "counts" not in name:
        pytest.skip("float colour sums keep their per-sample adds")
    print(f"records {name} {mode} small={small}", flush=True)
    check(ffr_mod, monkeypatch, FLAMES[name](), small, 0, **MODES[mode])


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("name, mode", [("basic_c3", "fp32"), ("basic_c3", "fp64"),
                                        ("basic_counts", "fp32"), ("basic_counts", "fp64"),
                                        ("basic_many_xforms", "fp32"),
                                        ("catalogue_c3", "fp32")])
def test_compiled_kernels(ffr_mod, monkeypatch, name, mode, small):
    print(f"records compiled {name} {mode} small={small}", flush=True)
    check(ffr_mod, monkeypatch, FLAMES[name](), small, 1, int("catalogue" in name),
          **MODES[mode])


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("mode", ["fp32", "fp64"])
def test_tasks_of_several_walkers_a_lane(ffr_mod, monkeypatch, mode, small):
    print(f"records, tasks of three walkers a lane {mode} small={small}", flush=True)
    monkeypatch.setenv("FFR_TASK_ROUNDS", "3")
    check(ffr_mod, monkeypatch, FLAMES["basic_c3"](), small, 0, **MODES[mode])


@pytest.mark.parametrize("rounds", [1, 3])
@pytest.mark.parametrize("small", [False, True])
def test_batch(ffr_mod, monkeypatch, small, rounds):
    print(f"records in a batch small={small} rounds={rounds}", flush=True)
    monkeypatch.setenv("FFR_TASK_ROUNDS", str(rounds))
    flames = [("basic_c3", "fp32"), ("basic_many_xforms", "fp32"), ("basic_c3", "fp64"),
              ("basic_counts", "u32"), ("catalogue_c3", "fp32"), ("linear_c3", "fp32")]
    rs = [make(ffr_mod, monkeypatch, FLAMES[n](), True, **MODES[m]) for n, m in flames]
    alone = [make(ffr_mod, monkeypatch, FLAMES[n](), False, **MODES[m]) for n, m in flames]
    samples = [SAMPLES - 100_003 * i for i in range(len(rs))]
    if small:
        monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 21))
    with ffr_mod.Batch(rs) as batch:
        for _ in range(3):
            assert all(batch.render(samples))
            for a, b, n in zip(rs, alone, samples):
                assert b.render(n)
                # (in the small memory one flame's misses may all come when
                # it is used up)
                assert int(not small) <= a.record_use[0] <= missed(a)
                same_buffers(a, b)
            assert sum(a.record_use[0] for a in rs) > 0
            assert (sum(a.record_use[1] for a in rs) > 0) == small
    for r in rs + alone:
        r.close()


@pytest.mark.parametrize("small", [False, True])
def test_bad_value_limit_with_records_waiting(ffr_mod, monkeypatch, small):
    print(f"records, bad-value limit small={small}", flush=True)
    d = json.loads(basic(3, 1200))
    total = sum(x["weight"] for x in d["xforms"])
    d["xforms"].append({"weight": 0.0005 * total, "color": [0.5, 0.5, 0.5],
                        "variations": [{"name": "linear", "weight": 1.0}],
                        "pre_affine": {"A": [[1e14, 0], [0, 1e14]], "b": [0, 0]}})
    r = make(ffr_mod, monkeypatch, json.dumps(d), True, precision="fp32", bad_value_limit=300)
    if small:
        monkeypatch.setenv("FFR_MISS_BYTES", str(1 << 21))
    assert not r.render(SAMPLES)
    assert r.last_stats.n_bad > 300 and r.record_use[0] > 0
    assert r.histogram_stats()[0] == r.samples_plotted
    r.close()


@pytest.mark.parametrize("compiled", [0, 1])
@pytest.mark.parametrize("mode", ["fp32", "fp64"])
@pytest.mark.parametrize("name", ["basic_c3", "basic_c1", "basic_c4", "basic_many_xforms"])
def test_binned_records(ffr_mod, monkeypatch, name, mode, compiled):
    """binned accumulation of the basic variations, in passes of 2^20 records"""
    print(f"binned records {name} {mode} compiled={compiled}", flush=True)
    text = FLAMES[name]()
    b = make(ffr_mod, monkeypatch, text, False, compiled=0, **MODES[mode])
    monkeypatch.setenv("FFR_BIN_PASS_RECORDS", str(1 << 20))
    a = ffr_mod.BufferRenderer(text, seed=SEED, batch_size=BATCH, binned=1, compiled=compiled,
                               **MODES[mode])
    for _ in range(2):
        assert a.render(SAMPLES) and b.render(SAMPLES)
        assert a.last_stats.binned == 1 and a.last_stats.compiled == compiled
        same_buffers(a, b)
    a.close()
    b.close()
