"""Seeded caches miss 0.75 to 0.9 of what unseeded ones do, by flame and by
run, so what they miss says nothing about the line from which renders take
miss records: a renderer judges by what it missed unseeded, at that size."""

import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu


def renderer(ffr, flame, precision):
    return ffr.BufferRenderer(read_flame("batch/flame_%d.json" % flame), precision=precision,
                              seed=3, binned=0, compiled=0)


def uses(r, sizes):
    out = []
    for n in sizes:
        assert r.render(n)
        out.append(r.record_use[0] > 0)
    return out


def test_under_the_line_with_caches_that_gain_little(ffr_mod):
    """0.125 words, seeded 0.113: 0.9 of it; FP32 renders take records from
    0.13 on"""
    print("miss seeded 1009", flush=True)
    r = renderer(ffr_mod, 1009, "fp32")
    assert uses(r, [1 << 28] * 6) == [True] + [False] * 5
    r.close()


@pytest.mark.parametrize("precision, flame", [
    ("fp64", 1105),  # 0.301 words, seeded 0.230; the line at 0.3
    ("fp64", 1251),  # 0.301, 0.234
    ("fp32", 1098),  # 0.130, 0.103; the line at 0.13
])
def test_on_the_line(ffr_mod, precision, flame):
    """Either choice may come of it; once a render takes records again, the
    next ones do."""
    print(f"miss seeded {precision} {flame}", flush=True)
    r = renderer(ffr_mod, flame, precision)
    got = uses(r, [1 << 28] * 10)[1:]
    assert sorted(got) == got or all(got), got
    r.close()


def test_sizes_in_turn(ffr_mod):
    """0.16 words at 2^28 samples, which fill the device, and too few for
    2^26, which do not: what one size missed does not move the other"""
    print("miss seeded sizes", flush=True)
    r = renderer(ffr_mod, 1166, "fp32")
    uses(r, [1 << 28, 1 << 26])
    assert uses(r, [1 << 28, 1 << 26] * 3) == [True, False] * 3
    r.close()
