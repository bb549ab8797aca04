"""The order of the row reductions' sums, bit for bit: a lane's own columns in
order, then the butterfly over the wave's 64 lanes (partners 32, 16, 8, 4, 2 and
1 apart). Each is read off an output that shows the sum itself: LayerNorm with
an eps that drowns the variance gives x - mean times a power of two; a softmax
whose exponentials are powers of two gives their sum's reciprocal."""
import numpy as np
import pytest

import mxenc
from mxenc import from_bf16_bits, to_bf16_bits

pytestmark = pytest.mark.gpu

F = np.float32


@pytest.fixture(scope="module")
def ctx():
    c = mxenc.Context(0)
    yield c
    c.close()


def butterfly(lanes):
    """[rows, 64] -> [rows], in fp32."""
    v = lanes.astype(F)
    for o in (32, 16, 8, 4, 2, 1):
        v = v + v[:, np.arange(64) ^ o]
    return v[:, 0]


def lane_sums(v, per):
    """Row sums before the butterfly: lane l holds columns l * per .. of each
    group of 64 * per, fours added in pairs."""
    rows, cols = v.shape
    groups = -(-cols // (64 * per))
    w = np.zeros((rows, groups * 64 * per), F)
    w[:, :cols] = v
    w = w.reshape(rows, groups, 64, per)
    s = np.zeros((rows, 64), F)
    for i in range(groups):
        if per == 4:
            s = s + ((w[:, i, :, 0] + w[:, i, :, 1]) + (w[:, i, :, 2] + w[:, i, :, 3]))
        else:
            for e in range(per):
                s = s + w[:, i, :, e]
    return s


@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("cols", [128, 384, 640, 768, 1024, 1280, 2048])
@pytest.mark.parametrize("with_y", [False, True])
def test_layernorm_sums(ctx, i8, cols, with_y):
    print("case", i8, cols, with_y, flush=True)
    rows = 37
    rng = np.random.default_rng(cols)
    x = (rng.standard_normal((rows, cols)) * 2.0 ** rng.integers(-12, 10, (rows, cols))).astype(F)
    y = to_bf16_bits(rng.standard_normal((rows, cols)).astype(F)) if with_y else None
    x[:, 0] = 0.0
    if with_y:
        y[:, 0] = 0
    v = x + from_bf16_bits(y) if with_y else x
    per = 4 if i8 or cols % 256 == 0 else 2
    mean = butterfly(lane_sums(v, per)) / F(cols)
    dx, dy = ctx.put(x), ctx.put(y) if with_y else None
    one, zero = ctx.put(np.ones(cols, F)), ctx.put(np.zeros(cols, F))
    out = ctx.empty((rows, cols), F)
    eps = float(2.0 ** 60)  # 1 / sqrt(var + eps) is 2^-30: the rest is exact
    if i8:
        mxenc.layernorm_i8(ctx, dx, dy, one, zero, eps, rows, cols, out, one,
                           ctx.empty((rows, cols), np.int8), ctx.empty((rows,), F))
    else:
        mxenc.layernorm(ctx, dx, dy, one, zero, eps, rows, cols, out_f32=out)
    got = -out.host()[:, 0] * F(2.0 ** 30)
    assert np.array_equal(got, mean)


@pytest.mark.parametrize("cols", [8, 64, 120, 128, 136, 512, 1024])
def test_softmax_sums(ctx, cols):
    print("case", cols, flush=True)
    rows = 37
    # arguments whose product with log2(e) is a whole number in fp32: 2^-k is exact
    table = {}
    for k in range(25):
        d = F(-k / 1.4426950408889634)
        for c in (d, np.nextafter(d, F(-99)), np.nextafter(d, F(99))):
            if F(c * F(1.4426950408889634)) == F(-k):
                table[k] = c
    ks = np.array(sorted(table))
    assert ks.size > 15 and ks[0] == 0
    rng = np.random.default_rng(cols)
    k = rng.choice(ks, (rows, cols))
    k[np.arange(rows), rng.integers(0, cols, rows)] = 0  # the row's maximum
    x = np.array([table.get(i, F(0)) for i in range(25)], F)[k]
    e = (2.0 ** -k.astype(np.float64)).astype(F)
    inv = F(1) / butterfly(lane_sums(e, 8))
    dx = ctx.put(x)
    mxenc.softmax_rows(ctx, dx, rows, cols, cols, variant=mxenc.MX_SOFTMAX_POLY)
    assert np.array_equal(dx.host(), e * inv[:, None])
