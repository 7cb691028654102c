"""Which renders take miss records: by the words a sample that miss the cell
cache, which seeded caches of renders with records lower (a flame near the
line must not change its mind with each render), and by the walkers: a launch
that does not fill the device hides its atomics."""

import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu


def uses(ffr, flame, samples, renders, **kw):
    r = ffr.BufferRenderer(read_flame("batch/flame_%d.json" % flame), seed=3, binned=0,
                           compiled=0, **kw)
    out = []
    for n in (samples if isinstance(samples, list) else [samples] * renders):
        assert r.render(n)
        out.append(r.record_use[0] > 0)
    r.close()
    return out


@pytest.mark.parametrize("flame, kept", [
    (1034, False),  # 0.04 words
    (1135, False),  # 0.104 with atomics, 0.086 with records
    (1167, False),  # 0.124, 0.097
    (1166, True),   # 0.164, 0.128
    (1040, True),   # 0.48
])
def test_the_choice_is_kept(ffr_mod, flame, kept):
    print(f"miss line {flame}", flush=True)
    got = uses(ffr_mod, flame, 1 << 28, 6, precision="fp32")
    assert got == [True] + [kept] * 5


@pytest.mark.parametrize("precision, flame, samples, records", [
    ("fp32", 1069, 1 << 26, [True, True, True]),     # 2.4 words, a quarter of the lanes
    ("fp32", 1082, 1 << 26, [True, False, False]),   # 0.43
    ("fp32", 1069, 1 << 25, [False, True, True]),    # 2.4, an eighth
    ("fp32", 1017, 1 << 25, [False, False, False]),  # 0.86, an eighth
    ("fp32", 1082, 1 << 27, [True, True, True]),     # 0.44, half
    ("fp32", 1000, 1 << 27, [True, False, False]),   # 0.22, half
    ("fp64", 1017, 1 << 25, [False, False, False]),  # 0.84, a quarter
    ("fp64", 1069, 1 << 26, [True, True, True]),     # 2.4, half
    ("fp64", 1069, 1 << 25, [False, True, True]),    # 2.4, a quarter
    ("fp64", 1241, 1 << 27, [True, True, True]),     # 0.34, all
    ("fp64", 1166, 1 << 27, [True, False, False]),   # 0.16, all
])
def test_launches_that_do_not_fill_the_device(ffr_mod, precision, flame, samples, records):
    print(f"miss line {precision} {flame} {samples}", flush=True)
    assert uses(ffr_mod, flame, samples, len(records), precision=precision) == records


def test_a_tuned_batch_knows_its_misses(ffr_mod):
    """two flames of 0.44 and 0.48 words in FP64, where a batch takes records
    from 0.75 on: a first pass that knows nothing takes them"""
    print("miss line of a tuned batch", flush=True)
    for tuned in (False, True):
        rs = [ffr_mod.BufferRenderer(read_flame("batch/flame_%d.json" % k), precision="fp64",
                                     seed=k) for k in (1048, 1040)]
        samples = [1 << 27] * 2
        with ffr_mod.Batch(rs) as batch:
            if tuned:
                batch.tune(samples, 1.0 / 8)
            assert all(batch.render(samples))
            assert all((r.record_use[0] == 0) == tuned for r in rs)
            assert all(batch.render(samples))
            assert all(r.record_use[0] == 0 for r in rs)
        for r in rs:
            r.close()
