"""The image stage's tone table on the GPU: counts below the table's size
(65536, or a quarter of the cells) take their level from it, larger ones
compute it.  Buffers hold counts on both sides of the edge, sizes down to one
cell (an empty table) and up to a full one, and one row past a whole number
of workgroups; every pixel against the CPU oracle, with the bar of the image
tests: both libraries' log and pow are within an ulp, which moves a pixel by
one where its exact value lies within an ulp of a boundary, so at most one
pixel in 10000 (and one) may be off by one."""

import numpy as np
import pytest

import flames as TF

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("word", [64, 32])
@pytest.mark.parametrize("w,h", [(1, 1), (3, 1), (5, 3), (257, 1), (97, 61), (600, 441)])
def test_tone_table_edges(ffr_mod, oracle_mod, word, w, h):
    text = TF.color_flame(3, size=64).replace("[64, 64]", f"[{w}, {h}]")
    r = ffr_mod.BufferRenderer(text, precision="fp64" if word == 64 else "fp32", word=word)
    cells = w * h
    edge = min(65536, cells // 4)
    rng = np.random.default_rng(w * 1000 + h)
    counts = rng.choice([0, 1, 2, 3, max(edge - 1, 1), edge + 0, edge + 1, 70_000, 5_000_000],
                        size=cells).astype(np.int64)
    counts[0] = 5_000_000
    real = np.float64 if word == 64 else np.float32
    buf = np.zeros((cells, 4), dtype=np.uint64 if word == 64 else np.uint32)
    buf[:, 0] = counts
    buf[:, 1:] = (counts[:, None] * rng.random((cells, 3))).astype(real).view(buf.dtype)
    r.write_buffer(buf.reshape(-1))
    for mode in (ffr_mod.IMG_MONO, ffr_mod.IMG_GRAY, ffr_mod.IMG_COLOR):
        for bits in (8, 16):
            for gamma in (1.0, 2.2):
                img, info = r.render_image(mode, gamma, bits)
                st, ref, _, _ = oracle_mod.tonemap(buf.reshape(-1), w, h, 4, mode, gamma, bits)
                assert st == 0 and info.hist_max == 5_000_000
                assert info.hist_min == int(counts.min())
                d = np.abs(img.astype(np.int64) - ref.astype(np.int64))
                assert int(d.max()) <= 1 and np.count_nonzero(d) <= max(1, d.size // 10000)
    assert r.histogram_stats() == (int(counts.sum()), int(counts.min()), int(counts.max()))
    r.close()


def test_empty_histogram_writes_no_pixel(ffr_mod):
    r = ffr_mod.BufferRenderer(TF.color_flame(3, size=64))
    n = r.image_bytes(ffr_mod.IMG_COLOR, 8)
    dev = ffr_mod.DeviceMemory(n, fill=0x5A)
    with pytest.raises(ffr_mod.FfrError, match="empty"):
        r.render_image_device(dev.ptr, n, ffr_mod.IMG_COLOR, 2.2, 8)
    assert np.all(dev.to_host() == 0x5A)
    dev.close()
    r.close()
