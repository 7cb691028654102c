"""Flames of the basic variations whose walkers settle beyond the number range
(an expanding map under the 1e15 up to which the kernel of the basic
variations takes a flame): every iteration is a bad value, and the points
recorded are the reference's, infinities where it has infinities and NaN where
it has NaN.  (The scales are such that walkers pass the range about when they have
settled: an infinite coordinate makes the point NaN an iteration later.)  That
kernel pads short variation lists with terms of weight 0; a
zero times an infinite point must not make a NaN of it.  Against the CPU
oracle, bit for bit (the maps that are drawn are linear)."""

import json

import numpy as np
import pytest

from test_gpu_parity import assert_same_stats, gpu_render, oracle_render

pytestmark = pytest.mark.gpu


def flame(scale, colours):
    lin = {"name": "linear", "weight": 1.0}
    xfs = [{"weight": 1.0, "variations": [lin],
            "pre_affine": {"A": [[scale, 0.0], [0.0, 0.9]], "b": [0.1, 0.2]}},
           {"weight": 0.4, "variations": [{"name": "linear", "weight": 0.9}],
            "pre_affine": {"A": [[0.5, 0.1], [0.0, 0.5]], "b": [0.3, 0.0]},
            "post_affine": {"A": [[1.0, 0.0], [0.0, 1.0]], "b": [0.0, 0.5]}},
           # never drawn: makes it a flame of the basic variations
           {"weight": 1e-30, "variations": [{"name": n, "weight": 0.3}
                                            for n in ("polar", "spherical", "swirl")]}]
    d = {"dimensions": 2, "size": [40, 30], "bounds": [[-2, 2], [-2, 2]], "xforms": xfs}
    if colours:
        d.update(color_dimensions=colours, color_speed=0.5)
        for k, x in enumerate(xfs):
            x["color"] = [0.2 + 0.3 * k] * colours
    return json.dumps(d)


def points(ids, pts):
    """as a sorted list of texts (NaN equals NaN there)"""
    return sorted(repr((int(i), [float(v) for v in p])) for i, p in zip(ids, pts))


KERNELS = {"default": {}, "lanes": dict(cell_cache=0), "cached": dict(cell_cache=1),
           "binned": dict(binned=1), "compiled": dict(cell_cache=1, compiled=1),
           "compiled binned": dict(binned=1, compiled=1)}


@pytest.mark.parametrize("kernel", sorted(KERNELS))
@pytest.mark.parametrize("colours", [0, 3, 2])
@pytest.mark.parametrize("mode, scale", [("fp32u64", 140.0), ("fp32u64", 300.0),
                                         ("fp64", 1.3e8)])
def test_recorded_points(ffr_mod, oracle_mod, mode, scale, colours, kernel):
    print(f"settle overflow {mode} {scale} {colours} {kernel}", flush=True)
    text = flame(scale, colours)
    a, ok = gpu_render(ffr_mod, text, 3_001, 97, mode, settle=-1, bad_value_limit=10 ** 9,
                       **KERNELS[kernel])
    ref = oracle_render(oracle_mod, text, 3_001, 97, mode, settle=-1, bv_limit=10 ** 9,
                        threads=1, bv_cap=4096)
    assert ok and ref.success and ref.n_bad > 1_000
    assert a.last_stats.n_bad == ref.n_bad
    got, want = points(*a.bad_values()), points(ref.bad_xforms, ref.bad_points)
    assert any("inf" in w for w in want)
    assert got == want
    assert np.array_equal(a.counts(a.read_buffer()).ravel(), ref.counts.ravel())
    assert_same_stats(a, ref, 2)
    a.close()
