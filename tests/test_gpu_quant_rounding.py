"""The quantizer's codes at and next to the rounding boundaries (its fast
rounding must hand exactly those to the double division), for block scales
over the whole float range, against the oracle bit for bit."""

import numpy as np
import pytest

import llmi_hip as H
import oracle as O

pytestmark = pytest.mark.gpu


def blocks_at_halves(rng, count, top):
    """Blocks of 32 whose other weights are (n + 1/2) scales, n < top, moved by
    -2 .. 2 ulps, or ordinary; one weight fixes the scale at 2^e * m / top."""
    e = rng.integers(-149, 121, count)
    e[: count // 2] = rng.integers(-12, 3, count // 2)
    scale = np.ldexp(np.where(rng.random(count) < 0.5, 1.0, 1.0 + rng.random(count)), e)
    n = rng.integers(0, int(top), (count, 32)) + 0.5
    v = (n * scale[:, None] * rng.choice([-1.0, 1.0], (count, 32))).astype(np.float32)
    for _ in range(2):
        up = rng.integers(-1, 2, v.shape)
        v = np.where(up == 0, v, np.nextafter(v, np.where(up > 0, np.inf, -np.inf).astype(np.float32)))
    v[:, rng.integers(0, 32)] = (top * scale * rng.choice([-1.0, 1.0], count)).astype(np.float32)
    return np.nan_to_num(v.astype(np.float32), posinf=3e38, neginf=-3e38)


@pytest.mark.parametrize("qt,top", [(O.Q8_0, 127.0), (O.Q4_0, 8.0)])
@pytest.mark.parametrize("out,n_in", [(130, 256), (64, 33), (67, 95), (1, 32), (200, 1)])
def test_codes_at_rounding_boundaries(qt, top, out, n_in):
    rng = np.random.default_rng(out * 7 + n_in)
    nblk = -(-n_in // 32)
    w = blocks_at_halves(rng, out * nblk, top).reshape(out, nblk * 32)[:, :n_in].copy()
    w[0, : min(n_in, 40)] = 0.0
    if out > 2:  # ties of the largest |v|: its first occurrence gives Q4_0's scale its sign
        w[1] = np.where(rng.random(n_in) < 0.5, 3.0, -3.0)
    want_d, want_s = O.oracle().quantize(w.reshape(-1), out, n_in, qt)
    data, scales = H.quantize(w.reshape(-1), out, n_in, qt)
    tiled, tiled_s = H.Weight.quantize(w.reshape(-1), out, n_in, qt).download()
    for got_d, got_s in ((data, scales), (tiled, tiled_s)):
        assert np.array_equal(got_d, want_d)
        assert np.array_equal(got_s.view(np.uint32), want_s.view(np.uint32))
