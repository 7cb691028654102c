"""The walker kernel's choices by flame against the CPU oracle, bit-exact on
linear flames: one to five colour components (three and four registers, and
memory), one to five variation terms a transform (their lists are padded to
three), with and without post-affine maps, and affine entries on both sides
of the 1e15 up to which the kernel of the basic variations takes a flame.
Counts and statistics exact, colour sums within 1e-12 relative (device
atomics add in another order)."""

import json

import numpy as np
import pytest

from test_gpu_parity import assert_same_stats, gpu_render, oracle_render

pytestmark = pytest.mark.gpu


def flame(r, terms, scale=None, post=False):
    rng = np.random.default_rng(17 + 8 * r + terms)
    xfs = []
    for k in range(3):
        w = rng.uniform(0.2, 1.0, terms)
        x = {"weight": 1.0 + k,
             "variations": [{"name": "linear", "weight": float(v)} for v in 0.9 * w / w.sum()],
             "pre_affine": {"A": (rng.uniform(-1, 1, (2, 2)) * 0.5).tolist(),
                            "b": rng.uniform(-1, 1, 2).tolist()}}
        if post and k != 1:
            x["post_affine"] = {"A": [[0.9, 0.1], [-0.1, 0.9]], "b": [0.05, -0.02]}
        if r:
            x["color"] = rng.uniform(0, 1, r).tolist()
            x["color_speed"] = 0.25 * (k + 1)
        xfs.append(x)
    if scale:
        xfs.append({"weight": 0.004, "variations": [{"name": "linear", "weight": 1.0}],
                    "pre_affine": {"A": [[scale, 0], [0, scale]], "b": [0, 0]}})
    doc = {"dimensions": 2, "size": [83, 61], "bounds": [[-2, 2], [-2, 2]], "xforms": xfs}
    if r:
        doc.update(color_dimensions=r, color_speed=0.5)
    return json.dumps(doc)


def check(ffr, oracle, text, mode, dims=2, cache=-1):
    print(f"walker kind {mode}", flush=True)
    kw = {"settle": 20}
    a, ok = gpu_render(ffr, text, 200_001, 97, mode, bad_value_limit=10 ** 9, cell_cache=cache, **kw)
    ref = oracle_render(oracle, text, 200_001, 97, mode, bv_limit=10 ** 9, **kw)
    assert ok
    words = a.read_buffer()
    assert np.array_equal(a.counts(words).ravel(), ref.counts.ravel())
    if a.color_dims:
        c, cr = a.colors(words).ravel(), ref.colors.ravel()
        assert np.allclose(c, cr, rtol=1e-12, atol=1e-12 * np.abs(cr).max())
    assert_same_stats(a, ref, dims)
    a.close()


@pytest.mark.parametrize("mode", ["fp64", "fp32u64"])
@pytest.mark.parametrize("cache", [0, 1])
@pytest.mark.parametrize("r", [0, 1, 2, 3, 4, 5])
def test_colours_and_terms(ffr_mod, oracle_mod, r, cache, mode):
    for terms in (1, 2, 3, 4, 5):
        check(ffr_mod, oracle_mod, flame(r, terms, post=terms % 2 == 0), mode, cache=cache)


@pytest.mark.parametrize("mode", ["fp64", "fp32u64"])
@pytest.mark.parametrize("scale", [1e8, 0.99e15, 1.01e15, 1e25])
def test_affine_range(ffr_mod, oracle_mod, scale, mode):
    check(ffr_mod, oracle_mod, flame(3, 2, scale=scale), mode)
