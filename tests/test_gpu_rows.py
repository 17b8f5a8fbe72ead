"""The exact products of more than one input row on the matrix cores
(csrc/qrows.hip above 8 rows, csrc/qfew.hpp up to 8) against the oracle, bit
for bit, on the shapes where their tiles and their dispatch can go wrong."""

import numpy as np
import pytest

import llmi_hip as H
import oracle as O
import synth

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# (rows, out, in): one side and the other of a 16- and 32-row tile, of a
# 16-output group and a 64-row tile, of a partial block and a whole one, of
# one block per wavefront (4, 8, 16 wavefronts) and several; 16 x 16 tiles up
# to 256 (16 wavefronts a tile), up to 1408 / 2560 (8), up to 8191 (16 rows a
# wavefront) and from 8192 (32 rows, but 16 for few groups of 16, an odd
# number of them); in the last two also one block, partial, and one to 31 of
# its elements.
SHAPES = [(9, 1, 1), (16, 15, 31), (17, 16, 32), (31, 17, 33), (32, 63, 63), (33, 65, 512), (15, 64, 513),
          (40, 130, 1055), (100, 700, 260), (48, 1500, 1024), (257, 1416, 64), (260, 1500, 1037), (529, 3900, 96),
          (545, 3890, 35), (11, 131073, 33), (41, 43700, 64), (33, 43690, 35),
          (545, 3890, 31), (544, 3900, 127), (545, 3890, 1), (545, 3890, 97), (48, 12000, 29), (48, 12000, 130)]


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,out,n_in", SHAPES)
def test_tile_edges_match_oracle(qt, rows, out, n_in):
    """Also with x only 4-byte aligned, and next to values that must not be
    read as its padding."""
    orc = O.oracle()
    w = synth.normal(out * 5 + n_in, out * n_in, 0.0, 0.02)
    x = synth.normal(rows * 11 + n_in, rows * n_in, 0.0, 1.0)
    bias = synth.normal(3, out, 0.0, 0.5)
    data, scales = orc.quantize(w, out, n_in, qt)
    dev = H.Weight.upload(data, scales, out, n_in, qt)
    want = orc.matmul(x, rows, n_in, data, scales, qt, out, bias)
    around = np.full(rows * n_in + 9, np.nan, dtype=np.float32)
    around[1 : 1 + rows * n_in] = x
    xd, bd = H.DeviceBuffer.from_array(around), H.DeviceBuffer.from_array(bias)
    yd = H.DeviceBuffer.from_array(np.full(rows * out + 64, 7.0, dtype=np.float32))
    dev.matmul_dev(xd.ptr + 4, rows, bd.ptr, yd.ptr)
    H.synchronize()
    got = yd.download(np.float32)
    assert np.array_equal(bits(got[: rows * out]), bits(want))
    assert np.all(got[rows * out :] == 7.0)


def test_rows_past_32_bit_offsets():
    """Rows of 2^25 elements and more: 16 of them are out of a 32-bit byte
    offset's reach."""
    orc = O.oracle()
    rows, out, n_in = 11, 2, 2**25 + 37
    rng = np.random.default_rng(25)
    w = np.resize(rng.standard_normal(1000003, dtype=np.float32), out * n_in)
    x = np.resize(rng.standard_normal(999983, dtype=np.float32), rows * n_in)
    data, scales = orc.quantize(w, out, n_in, O.Q4_0)
    got = H.Weight.upload(data, scales, out, n_in, O.Q4_0).matmul(x, rows, None)
    want = orc.matmul(x, rows, n_in, data, scales, O.Q4_0, out, None)
    assert np.array_equal(bits(got), bits(want))


# 2..8 rows: one side and the other of 4 rows a matrix instruction, of a
# 64-row tile, of a partial block; 16-row tiles (at most 64 tiles and 64
# blocks), long rows on few tiles, and 16, 8 and 4 wavefronts per 64-row tile
# with fewer, as many and more blocks than wavefronts; rows of 32 and of more
# blocks, and those on as many row chunks of 1, 2 and 4 as there are CUs, and
# on one more.
FEW = [(2, 64, 33), (3, 63, 32), (4, 4161, 31), (5, 4200, 32), (8, 4097, 513), (7, 8256, 70), (4, 8192, 288),
       (3, 32832, 100), (8, 32770, 97), (5, 32768, 160), (2, 32768, 64), (6, 200, 2100), (4, 130, 2048), (3, 8300, 2100),
       (8, 2000, 1024), (8, 2048, 1025), (8, 2049, 1056), (3, 8192, 1600), (4, 8193, 2048), (7, 8192, 1500), (5, 8193, 1030),
       (8, 2000, 1279), (8, 2000, 1281), (5, 4100, 1290)]


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,out,n_in", FEW)
def test_few_rows_match_oracle(qt, rows, out, n_in):
    """Single and grouped; x between values that must not be read as its
    padding."""
    orc = O.oracle()
    w = synth.normal(out + 5 * n_in, out * n_in, 0.0, 0.02)
    x = synth.normal(rows * 17 + n_in, rows * n_in, 0.0, 1.0)
    bias = synth.normal(4, out, 0.0, 0.5)
    data, scales = orc.quantize(w, out, n_in, qt)
    dev = H.Weight.upload(data, scales, out, n_in, qt)
    want = orc.matmul(x, rows, n_in, data, scales, qt, out, bias)
    around = np.full(rows * n_in + 9, np.nan, dtype=np.float32)
    around[1 : 1 + rows * n_in] = x
    xd, bd = H.DeviceBuffer.from_array(around), H.DeviceBuffer.from_array(bias)
    yd = [H.DeviceBuffer.from_array(np.full(rows * out + 64, 7.0, dtype=np.float32)) for _ in range(2)]
    dev.matmul_dev(xd.ptr + 4, rows, bd.ptr, yd[0].ptr)
    H.Group([(dev, xd.ptr + 4, yd[1].ptr, rows, bd.ptr)]).launch()
    H.synchronize()
    for y in yd:
        got = y.download(np.float32)
        assert np.array_equal(bits(got[: rows * out]), bits(want))
        assert np.all(got[rows * out :] == 7.0)


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("shapes", [[(8, 200, 1600), (8, 130, 2048)], [(8, 200, 1600), (8, 130, 576)],
                                    [(8, 200, 1600), (3, 130, 1100)], [(1, 200, 1600), (8, 130, 2048)],
                                    [(2, 2000, 2048), (2, 130, 1000), (3, 70, 700)], [(2, 100, 96), (2, 3000, 700), (7, 60, 64)],
                                    [(5, 700, 576), (5, 130, 2100), (8, 100, 3000), (1, 64, 4100)]])
def test_groups_of_few_rows_match_oracle(qt, shapes):
    """Products of long rows on few tiles together, with others that want
    another kind of tile or chunk, and beside one row; the same of the other
    type in the same group."""
    orc = O.oracle()
    keep, items, wants = [], [], []
    for qt, (rows, out, n_in) in [(t, sh) for sh in shapes for t in (qt, O.Q8_0 + O.Q4_0 - qt)]:
        w = synth.normal(out + 5 * n_in, out * n_in, 0.0, 0.02)
        x = synth.normal(rows * 17 + n_in, rows * n_in, 0.0, 1.0)
        data, scales = orc.quantize(w, out, n_in, qt)
        wants.append(orc.matmul(x, rows, n_in, data, scales, qt, out, None))
        xd, yd = H.DeviceBuffer.from_array(x), H.DeviceBuffer.from_array(np.full(rows * out, 7.0, dtype=np.float32))
        keep.append((xd, yd))
        items.append((H.Weight.upload(data, scales, out, n_in, qt), xd.ptr, yd.ptr, rows, None))
    H.Group(items).launch()
    H.synchronize()
    for (_, yd), want in zip(keep, wants):
        assert np.array_equal(bits(yd.download(np.float32)), bits(want))


@pytest.mark.parametrize("rows,out,n_in", [(5, 4500, 96), (24, 4500, 96), (5, 200, 1101), (8, 5000, 1119), (24, 4500, 65)])
@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
def test_extreme_rows_stay_in_their_rows(qt, rows, out, n_in):
    """Subnormal, zero, huge and infinite activations, also in a partial last
    block: each row's results are the oracle's, whatever its neighbours in the
    tile hold."""
    orc = O.oracle()
    w = synth.normal(1, out * n_in, 0.0, 0.02)
    x = synth.normal(2, rows * n_in, 0.0, 1.0).reshape(rows, n_in)
    x[0] *= np.float32(1e-42)
    x[1] = -0.0
    x[2] *= np.float32(1e36)
    x[3, 7] = np.inf
    x[4, n_in - 1] = -np.inf
    data, scales = orc.quantize(w, out, n_in, qt)
    scales[::7] *= np.float32(1e-12)
    dev = H.Weight.upload(data, scales, out, n_in, qt)
    got = dev.matmul(x.reshape(-1), rows, None)
    want = orc.matmul(x.reshape(-1), rows, n_in, data, scales, qt, out, None)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(bits(got)[~nan], bits(want)[~nan])


# fp32 weights (csrc/f32.hip): 16- and 32-row tiles of the matrix-core form,
# outputs around its 64- and 32-output tiles, elements around a 64-element
# step, a 16-element chunk and the scalar rest.
@pytest.mark.parametrize("rows,out,n_in", [(2, 40000, 500), (16, 8001, 64), (16, 5000, 79), (17, 3000, 128),
                                           (32, 2911, 255), (33, 1600, 1003), (70, 1100, 16), (5, 90000, 31)])
def test_f32_rows_match_single_rows_and_oracle(rows, out, n_in):
    """Every output against the one-row product (tests/test_gpu_f32.py holds
    that one to the oracle), some of them against the oracle's dot."""
    orc = O.oracle()
    w = synth.normal(out + 3 * n_in, out * n_in, 0.0, 0.02)
    x = synth.normal(rows + n_in, rows * n_in, 0.0, 1.0)
    x[: n_in // 2] *= np.float32(1e-30)  # products that underflow to either zero
    w[: n_in // 2] *= np.float32(-1e-16)
    bias = synth.normal(6, out, 0.0, 0.5)
    bias[::5] = -0.0
    dev = H.Weight.quantize(w, out, n_in, H.F32)
    around = np.full(rows * n_in + 9, np.nan, dtype=np.float32)
    around[1 : 1 + rows * n_in] = x
    xd, bd = H.DeviceBuffer.from_array(around), H.DeviceBuffer.from_array(bias)
    yd = H.DeviceBuffer.from_array(np.full(rows * out + 64, 7.0, dtype=np.float32))
    dev.matmul_dev(xd.ptr + 4, rows, bd.ptr, yd.ptr)
    H.synchronize()
    got = yd.download(np.float32)
    want = np.concatenate([dev.matmul(x[r * n_in : (r + 1) * n_in], 1, bias) for r in range(rows)])
    assert np.array_equal(bits(got[: rows * out]), bits(want))
    for i in np.random.default_rng(n_in).integers(0, rows * out, 60):
        r, o = divmod(int(i), out)
        d = np.float32(orc.dot(x[r * n_in : (r + 1) * n_in], w[o * n_in : (o + 1) * n_in])) + bias[o]
        assert bits(got[i : i + 1])[0] == bits(np.float32([d]))[0]
    assert np.all(got[rows * out :] == 7.0)
