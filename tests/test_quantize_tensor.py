"""quantize_tensor encodes full blocks with vector code of its own: byte for byte what quantize_block_all (pinned to the
reference) gives for each block, on data that sits on the edges of the rounding rules."""
import numpy as np
import pytest

import innova_amd as ia
from innova_amd import block_codec

LEVELS = np.array([0.126, 0.3976, 0.4528, 0.6508, 0.9275, 1.2392, 1.5104, 1.5995, 2.0522, 2.7178], np.float32)


def _data(kind, n, rng):
    if kind == "normal":
        return rng.standard_normal(n).astype(np.float32) * np.float32(0.02)
    if kind == "halfway":                                  # points between levels, and the floats next to them
        mid = np.concatenate([(LEVELS[1:] + LEVELS[:-1]) / 2, [0.0, 1.0]]).astype(np.float32)
        v = rng.choice(np.concatenate([mid, -mid]), n).astype(np.float32)
        return np.nextafter(v, rng.choice([-9.0, 9.0], n).astype(np.float32))
    if kind == "zeros":
        return np.where(rng.random(n) < 0.5, np.float32(0.0), np.float32(-0.0))
    if kind == "tiny":
        return (rng.integers(-3, 4, n) * np.float32(2.0 ** -148)).astype(np.float32)
    w = rng.standard_normal(n).astype(np.float32)          # "special": values that leave the vector path
    w[::97] = rng.choice(np.array([np.inf, -np.inf, np.nan, 3e38, 1e30, 0.0], np.float32), w[::97].size)
    return w


@pytest.mark.parametrize("n", [256, 256 * 8, 256 * 9 + 1, 256 * 17 + 255])
@pytest.mark.parametrize("kind", ["normal", "halfway", "zeros", "tiny", "special"])
def test_blocks_equal_the_block_encoder(kind, n):
    rng = np.random.default_rng(n + len(kind))
    w = _data(kind, n, rng)
    for fmts in list(ia.Format) + [None]:
        nb = (n + 255) // 256
        fm = np.full(nb, int(fmts), np.uint8) if fmts is not None else rng.integers(0, 13, nb).astype(np.uint8)
        payload, blocks = block_codec.quantize_tensor(w, fm, threads=3)
        for b in range(nb):
            idx, cb = block_codec.quantize_block_all(int(fm[b]), w[256 * b:256 * b + 256])
            at, ct = int(blocks[b]["idx_off"]), int(blocks[b]["cb_off"])
            assert np.array_equal(payload[at:at + blocks[b]["idx_bytes"]], idx), (fmts, b)
            assert np.array_equal(payload[ct:ct + blocks[b]["cb_bytes"]], cb), (fmts, b)


def _thresholds(levels):
    """Floats around the points at which the nearest level changes."""
    lv = np.sort(np.concatenate([levels, -levels])).astype(np.float32)
    t = ((lv[1:] + lv[:-1]) / 2).astype(np.float32)
    around = [t]
    for way in (np.float32(9.0), np.float32(-9.0)):
        v = t
        for _ in range(3):
            v = np.nextafter(v, way)
            around.append(v)
    return np.concatenate(around)


def _block_of_rms_one(values, rng):
    """256 weights that hold `values` and whose RMS rounds to 1."""
    w = np.empty(256, np.float64)
    w[:values.size] = values
    rest = 256 - values.size - 1
    left = 256.0 - float((values.astype(np.float64) ** 2).sum()) - 0.5
    fill = rng.standard_normal(rest)
    w[values.size:255] = fill * np.sqrt(left / float((fill ** 2).sum()))
    w = w.astype(np.float32).astype(np.float64)
    w[255] = np.sqrt(256.0 - float((w[:255] ** 2).sum()))
    return rng.permutation(w.astype(np.float32))


# Shares of sixteen blocks and more, whose sums run side by side, in every mix of formats; quotients on both sides of every threshold (found in the
# weights instead of dividing each) at scales of any size, those among them at which t * scale passes a power of two; run means and scales around 2^-24,
# the smallest magnitude that becomes a half
@pytest.mark.parametrize("scale", [1.0, 0.02, 0.0137, 0.99999994, 1.0000001, 0.5 / 0.5252, 3e-11, 1.7e-12, 7e-13, 6e-8, 2.0 ** -24, 1.9e-7, 4e20])
@pytest.mark.parametrize("threads", [1, 2])
def test_wide_shares_equal_the_block_encoder(scale, threads):
    rng = np.random.default_rng(int(abs(np.log(scale)) * 1000) + threads)
    l4 = np.array([0.126, 0.3976, 0.6508, 0.9275, 1.2392, 1.5995, 2.0522, 2.7178], np.float32)
    l2 = np.array([0.4528, 1.5104], np.float32)
    edges = [_thresholds(l4), _thresholds(l2)]
    blocks_of = [_block_of_rms_one(np.asarray(edges[i % 2]), rng) for i in range(37)] + [rng.standard_normal(256).astype(np.float32) for _ in range(10)]
    w = (np.concatenate(blocks_of + [rng.standard_normal(77).astype(np.float32)]) * np.float32(scale)).astype(np.float32)
    w[256 * 40:256 * 41] = np.where(rng.random(256) < 0.5, np.float32(0.0), np.float32(-0.0))
    w[256 * 41 + 5] = np.float32(2e29)                     # leaves the vector path
    nb = (w.size + 255) // 256
    for fm in [np.full(nb, f, np.uint8) for f in range(13)] + [rng.integers(0, 13, nb).astype(np.uint8), rng.integers(0, 2, nb).astype(np.uint8),
                                                               rng.choice(np.array([7, 9, 10, 11], np.uint8), nb)]:
        payload, blocks = block_codec.quantize_tensor(w, fm, threads=threads)
        for b in range(nb):
            idx, cb = block_codec.quantize_block_all(int(fm[b]), w[256 * b:256 * b + 256])
            at, ct = int(blocks[b]["idx_off"]), int(blocks[b]["cb_off"])
            assert np.array_equal(payload[at:at + blocks[b]["idx_bytes"]], idx), (int(fm[b]), b)
            assert np.array_equal(payload[ct:ct + blocks[b]["cb_bytes"]], cb), (int(fm[b]), b)


def test_unknown_formats_are_refused_wherever_they_stand():
    w = np.ones(256 * 50, np.float32)
    for at in (0, 13, 49):
        fm = np.zeros(50, np.uint8)
        fm[at] = 15
        with pytest.raises(ia._lib.OilHipError):
            block_codec.quantize_tensor(w, fm, threads=2)
