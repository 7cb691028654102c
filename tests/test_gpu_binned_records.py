"""Binned colour records of every size on the GPU: one to four colour
components of FP32 or FP64 walkers (records of 16, 32 and 48 bytes), few
tiles and more than 3072 (the scatter's smaller chunks), several chunks a
block with a ragged last one.  Counts and statistics equal the atomic
path's; colour sums to the rounding of their order of addition, 1e-12
relative.  (8-byte words only: the atomic path of 4-byte words rounds to
float on every add, and a cell of 6e4 samples strays by up to 6e4 * 2^-24 of
its sum, so it is no reference for these sums; test_gpu_binned_colour.py
has the float build's words.)"""

import numpy as np
import pytest

import flames as TF

pytestmark = pytest.mark.gpu

SEED = 0x5EED0012


@pytest.mark.parametrize("size,samples,batch", [(64, 300_001, 700), (4000, 2_500_003, 1_111)])
@pytest.mark.parametrize("r", [1, 2, 3, 4])
@pytest.mark.parametrize("mode", ["fp64", "fp32u64"])
def test_record_sizes(ffr_mod, mode, r, size, samples, batch):
    text = TF.color_flame(r, size=size)
    print(f"records {mode} r={r} size={size}", flush=True)
    kw = {"precision": "fp64" if mode == "fp64" else "fp32", "seed": SEED, "batch_size": batch}
    a = ffr_mod.BufferRenderer(text, binned=1, **kw)
    b = ffr_mod.BufferRenderer(text, binned=0, **kw)
    for _ in range(2):
        assert a.render(samples) and b.render(samples)
    assert a.last_stats.binned == 1 and b.last_stats.binned == 0
    wa, wb = a.read_buffer(), b.read_buffer()
    assert np.array_equal(a.counts(wa), b.counts(wb))
    ca, cb = a.colors(wa), b.colors(wb)
    assert np.allclose(ca, cb, rtol=1e-12, atol=1e-12 * np.abs(cb).max())
    assert a.samples_plotted == b.samples_plotted
    assert a.point_extremes == b.point_extremes
    a.close()
    b.close()
