"""Split walkers on the GPU: renders of few walkers run each walker's
iterations as segments on many lanes.  A segment starts from a guess some
iterations before its first and must enter it with the state its left
neighbour ends with, bit for bit, so the buffer's counts and the statistics
must equal those of the unsplit walkers (cell_cache 0) bit for bit; colour
sums (8-byte words) to the rounding of their order of addition: a cell of n
samples is summed in two orders, each off by at most n * 2^-53 of the sum of
its (positive) terms, n < 2^17 here, so 2^-35 covers both.

A split render makes no global atomic add per sample (`atomics` 0); one
whose segments do not join, or that meets a bad value, runs unsplit behind
it and makes them.
"""

import json
import re

import numpy as np
import pytest

import flames as TF
from conftest import read_flame

pytestmark = pytest.mark.gpu

SEED = 0x5EED0011


def headline(w=97, h=61, speed=None):
    d = json.loads(re.sub(r"^\s*//.*$", "", read_flame("random_color_3840x2160.json"),
                          flags=re.M))
    d["size"] = [w, h]
    if speed is not None:
        d["color_speed"] = speed
    return d


def catalogue():
    """variations of the whole catalogue that draw no words, a final xform"""
    d = headline(64, 80)
    names = ["bent", "handkerchief", "disc", "bubble", "fisheye", "cylinder"]
    for x, n in zip(d["xforms"], names):
        x["variations"] = [TF.variation(n, 0.6, 2), TF.variation("sinusoidal", 0.4, 2)]
    d["final_xform"] = {"variations": [TF.variation("sinusoidal", 1.0, 2)],
                        "color": [0.1, 0.5, 0.9], "color_speed": 0.3}
    return json.dumps(d)


def sine_3d():
    d = json.loads(TF.tetrahedron(24))
    for x in d["xforms"]:
        x["variations"].append({"name": "sinusoidal", "weight": 0.2})
    return json.dumps(d)


FLAMES = {
    "headline": lambda: json.dumps(headline()),
    # a colour that keeps 7/8 of itself per iteration: a longer run-up
    "slow_colour": lambda: json.dumps(headline(speed=0.125)),
    "catalogue": catalogue,
    "one_d": lambda: TF.one_d(nonlinear=True),
    "sine_3d": sine_3d,
    "rotations": TF.rotations,
    "tied_weights": TF.tied_weights,     # more xforms than byte-packed counters
    "tetrahedron": TF.tetrahedron,
}
# samples, batch: one walker; walkers not a multiple of a workgroup's, the
# last of one sample; short walkers whose segments lie within reach of the
# start; an odd batch, most segments of the last walker unused
SHAPES = [(70_000, 70_000), (401 * 333 + 1, 333), (5_000, 40), (9 * 4_099 + 17, 4_099)]


def renderers(ffr, text, mode, batch, **kw):
    prec, word = {"fp64": ("fp64", 64), "fp32": ("fp32", 64), "fp32u32": ("fp32", 32)}[mode]
    return [ffr.BufferRenderer(text, precision=prec, word=word, seed=SEED, batch_size=batch,
                               cell_cache=c, **kw) for c in (-1, 0)]


def assert_same(a, b):
    wa, wb = a.read_buffer(), b.read_buffer()
    assert np.array_equal(a.counts(wa), b.counts(wb))
    assert a.samples_iterated == b.samples_iterated
    assert a.samples_plotted == b.samples_plotted
    assert np.array_equal(a.xform_distribution(), b.xform_distribution())
    assert a.point_extremes == b.point_extremes
    assert a.last_stats.n_bad == b.last_stats.n_bad
    if a.color_dims:
        ca, cb = a.colors(wa), b.colors(wb)
        assert np.all(np.abs(ca - cb) <= 2.0 ** -35 * np.abs(cb))


@pytest.mark.parametrize("mode", ["fp64", "fp32", "fp32u32"])
@pytest.mark.parametrize("name", sorted(FLAMES))
def test_split_equals_unsplit(ffr_mod, name, mode):
    text = FLAMES[name]()
    if mode == "fp32u32" and "color_dimensions" in text:
        pytest.skip("colour flames with 4-byte words run unsplit")
    for samples, batch in SHAPES:
        print(f"split {name} {mode} {samples} {batch}", flush=True)
        a, b = renderers(ffr_mod, text, mode, batch)
        for _ in range(2):  # the second continues the streams
            assert a.render(samples) and b.render(samples)
            assert a.last_stats.atomics == 0 < b.last_stats.atomics
            assert_same(a, b)
        a.close()
        b.close()


@pytest.mark.parametrize("mode", ["fp64", "fp32"])
def test_split_failure_runs_unsplit(ffr_mod, mode):
    """bad values; maps that keep distances (rotations of the plane, whose
    segments never join); a colour that is never blended"""
    turn = json.loads(TF.rotations())
    for k, x in enumerate(turn["xforms"]):
        c, s = np.cos(0.7 + k), np.sin(0.7 + k)
        x["pre_affine"] = {"A": [[c, -s], [s, c]], "b": [0.0, 0.0]}
        x["variations"] = [{"name": "linear", "weight": 0.5}, {"name": "sinusoidal",
                                                               "weight": 0.6}]
        x.pop("post_affine", None)
    keep = headline(speed=0.0)
    for name, text in (("bad", TF.occasional_bad()), ("turn", json.dumps(turn)),
                       ("keep", json.dumps(keep))):
        print(f"split failure {name} {mode}", flush=True)
        a, b = renderers(ffr_mod, text, mode, 3_000, bad_value_limit=10 ** 9)
        for _ in range(2):
            assert a.render(300_001) and b.render(300_001)
            assert_same(a, b)
        a.close()
        b.close()


def test_split_stops_at_the_bad_value_limit(ffr_mod):
    a, b = renderers(ffr_mod, TF.expanding(), "fp64", 1_000, bad_value_limit=3)
    assert not a.render(100_000) and not b.render(100_000)
    assert a.last_stats.n_bad >= 4
    s, _, _ = a.histogram_stats()
    assert s == a.samples_plotted
    a.close()
    b.close()
