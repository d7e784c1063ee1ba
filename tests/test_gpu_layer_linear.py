"""``rfsn_layer_linear`` against float64: one row, the streamed rows (up to 64) and the tiles (past 64), at the
edges of their row, output and k ranges.

A plain result is one fp16 rounding (2^-11 |y|) of fp32 sums of k products with weights kept to 2^-23 (and to
2^-37, or 2^-39 of their row's largest): bounded by 2^-20 sum |x w| for the k here.  Behind it each fp16 cast point may add 2^-11 of its value once more."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 16, 17, 33, 64, 65, 129, 200, 520]
SHAPES = [(64, 64), (192, 320), (640, 128), (2048, 68), (8192, 64), (128, 4100)]  # k, n (the last: larger tiles)


def _t(a, device):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def _data(rows, k, n, seed):
    g = np.random.default_rng(seed)
    x = g.standard_normal((rows, k), dtype=np.float32).astype(np.float16)
    w = [((g.random((m, k), dtype=np.float32) * 2 - 1) / np.float32(k ** 0.5)) for m in (n, n, 64)]
    return g, x, w


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("k,n", SHAPES)
def test_plain_and_residual(device, rows, k, n):
    from apple_amd import kernels as K

    g, x, w = _data(rows, k, n, rows * k + n)
    xd = _t(x, device)
    x64 = x.astype(np.float64)
    outs = K.layer_linear(xd, [_t(m, device) for m in w])
    for o, m in zip(outs, w):
        y, mag = x64 @ m.T.astype(np.float64), np.abs(x64) @ np.abs(m.T.astype(np.float64))
        assert np.all(np.abs(o.cpu().numpy() - y) <= np.abs(y) * 2.0 ** -11 + mag * 2.0 ** -20 + 2.0 ** -25)
    res = g.standard_normal((rows, n), dtype=np.float32).astype(np.float16)
    o, = K.layer_linear(xd, [_t(w[0], device)], K.LINEAR_RESIDUAL, residual=_t(res, device))
    y, mag = x64 @ w[0].T.astype(np.float64), np.abs(x64) @ np.abs(w[0].T.astype(np.float64))
    want = res.astype(np.float64) + y
    assert np.all(np.abs(o.cpu().numpy() - want) <= (np.abs(want) + np.abs(y)) * 2.0 ** -11 + mag * 2.0 ** -20 + 2.0 ** -24)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("k,n", SHAPES)
def test_norm_swiglu(device, rows, k, n):
    from apple_amd import kernels as K

    g, x, w = _data(rows, k, n, rows + k * n)
    nw = (1 + 0.1 * g.standard_normal(k, dtype=np.float32)).astype(np.float32)
    o, = K.layer_linear(_t(x, device), [_t(m, device) for m in w[:2]], K.LINEAR_SWIGLU, norm=(_t(nw, device), 1e-5))
    x64 = x.astype(np.float64)
    a = (x64 / np.sqrt((x64 ** 2).mean(-1, keepdims=True) + 1e-5) * nw).astype(np.float16).astype(np.float64)
    gate, up = (a @ m.T.astype(np.float64) for m in w[:2])
    want = gate / (1 + np.exp(-gate)) * up
    # cast points: the normed row (flips of one rounding move a product by up to 2^-10 of sum |x w| / sqrt(k)),
    # gate (its relative step grows by at most 1 + |gate| through the sigmoid), act, up, the product
    tol = (np.abs(want) * (4 + np.abs(gate)) * 2.0 ** -11
           + (np.abs(up) + np.abs(gate) + 1) * 2.0 ** -10)
    assert np.all(np.abs(o.cpu().numpy() - want) <= tol)


@pytest.mark.parametrize("rows", [1, 3, 40, 70])
@pytest.mark.parametrize("D", [64, 128])
def test_rope_from_frequencies_and_from_tables(device, rows, D):
    import torch
    from apple_amd import kernels as K

    g = np.random.default_rng(rows + D)
    k, hq, hkv = 256, 6, 2
    x = g.standard_normal((rows, k), dtype=np.float32).astype(np.float16)
    w = [(g.standard_normal((h * D, k), dtype=np.float32) / 16) for h in (hq, hkv, hkv)]
    inv = 500000.0 ** (-np.arange(0, D, 2) / D)
    ang = (np.arange(rows)[:, None] + 777) * inv[None]
    cos, sin = (np.concatenate([f(ang)] * 2, -1).astype(np.float32) for f in (np.cos, np.sin))
    xd, wd = _t(x, device), [_t(m, device) for m in w]
    a = K.layer_linear(xd, wd, head_dim=D, inv_freq=_t(inv, device), pos0=777)
    b = K.layer_linear(xd, wd, head_dim=D, tables=(_t(cos, device), _t(sin, device)))
    plain = K.layer_linear(xd, wd)
    for i in range(3):
        y = plain[i].cpu().numpy().astype(np.float64).reshape(rows, -1, D)
        want = y if i == 2 else y * cos[:, None] + np.concatenate([-y[..., D // 2:], y[..., :D // 2]], -1) * sin[:, None]
        for o in (a[i], b[i]):
            err = np.abs(o.cpu().numpy().astype(np.float64).reshape(rows, -1, D) - want)
            assert np.all(err <= np.abs(want) * 2.0 ** -11 + np.abs(y).max() * 2.0 ** -22)
    assert torch.equal(a[2], plain[2])


@pytest.mark.parametrize("rows", [1, 5, 20, 50, 90])
def test_weights_outside_the_first_scale(device, rows):
    """Weights past fp16's range at the kernel's scale (and one that is infinite) repeat the block at one that fits."""
    from apple_amd import kernels as K

    g, x, w = _data(rows, 256, 128, rows)
    x = (x.astype(np.float32) * 1e-3).astype(np.float16)
    m = w[0].copy()
    m[3, 5], m[70, 7], m[127, 255] = 40.0, -3e5, 1e7
    o, = K.layer_linear(_t(x, device), [_t(m, device)])
    y, mag = x.astype(np.float64) @ m.T.astype(np.float64), np.abs(x.astype(np.float64)) @ np.abs(m.T.astype(np.float64))
    # at a smaller scale a weight keeps 2^-38 of its row's largest
    small = np.abs(x.astype(np.float64)).sum(-1, keepdims=True) * np.abs(m).max(-1)[None] * 2.0 ** -38
    assert np.all(np.abs(o.cpu().numpy() - y) <= np.abs(y) * 2.0 ** -11 + mag * 2.0 ** -20 + small + 2.0 ** -25)
    m[9, 9] = np.inf
    o, = K.layer_linear(_t(x, device), [_t(m, device)])
    o = o.cpu().numpy()
    assert np.all(np.isinf(o[:, 9]) | (x[:, 9] == 0))
    ok = np.abs(o - y) <= np.abs(y) * 2.0 ** -11 + mag * 2.0 ** -20 + small + 2.0 ** -25
    assert np.all(np.delete(ok, 9, 1))


@pytest.mark.parametrize("rows", [1, 5, 20, 50, 90, 300])
@pytest.mark.parametrize("k", [192, 256])
def test_small_weights(device, rows, k):
    """Rows of small weights (all of a matrix, or single rows among ordinary ones) keep their precision."""
    from apple_amd import kernels as K

    g, x, w = _data(rows, k, 128, rows + k)
    x = (x.astype(np.float32) * 4096).astype(np.float16)
    small, mixed = w[0] * np.float32(2.0 ** -26), w[1].copy()
    mixed[::5] *= np.float32(2.0 ** -26)
    mixed[7], mixed[8] = 0, small[8] * np.float32(2.0 ** -90)
    mixed[9, 0] = 5e-5  # the largest of a row of 2^-26
    x64 = x.astype(np.float64)
    for m in (small, mixed):
        o, = K.layer_linear(_t(x, device), [_t(m, device)])
        y, mag = x64 @ m.T.astype(np.float64), np.abs(x64) @ np.abs(m.T.astype(np.float64))
        row = np.abs(x64).sum(-1, keepdims=True) * np.abs(m).max(-1)[None] * 2.0 ** -38  # 2^-39, rounded twice
        f = np.abs(y) < 65000  # the ordinary rows' sums may leave fp16's range
        assert np.all(np.abs(o.double().cpu().numpy() - y)[f] <= (np.abs(y) * 2.0 ** -11 + mag * 2.0 ** -20 + row + 2.0 ** -25)[f])


def _ieee(x, w):
    """x w^T in float64 with the infinities and NaN of a float32 sum: what meets each product, in any order."""
    fin = np.where(np.isfinite(x), x, 0).astype(np.float64)
    y = fin @ w.T.astype(np.float64)
    inf = np.where(np.isinf(x), np.sign(np.where(np.isinf(x), x, 0)), 0).astype(np.float64)
    up = np.maximum(inf, 0) @ np.maximum(w, 0).T + np.maximum(-inf, 0) @ np.maximum(-w, 0).T
    down = np.maximum(inf, 0) @ np.maximum(-w, 0).T + np.maximum(-inf, 0) @ np.maximum(w, 0).T
    nan = np.isnan(x).any(-1, keepdims=True) | (np.isinf(x).astype(np.float64) @ (w == 0).T.astype(np.float64) > 0)
    y[up > 0], y[down > 0] = np.inf, -np.inf
    y[nan | ((up > 0) & (down > 0))] = np.nan
    return y


@pytest.mark.parametrize("rows", [1, 2, 20, 50, 70, 300])
@pytest.mark.parametrize("k,n", [(192, 128), (256, 128), (256, 4100)])
def test_infinite_inputs(device, rows, k, n):
    """An infinite x is infinite in every output its weights lead to, whether a weight has a low half or not, down to
    the smallest; two of opposite sign, or one that meets a weight of 0, give NaN; other rows are untouched."""
    from apple_amd import kernels as K

    g, x, w = _data(rows, k, n, rows * k + n)
    m = w[0].copy()
    m[::3] = m[::3].astype(np.float16)          # no low half
    m[5, 100], m[6, 100], m[7, 100] = 0.0, 2.0 ** -60, -(2.0 ** -60)
    m[1::7, 30] = np.abs(m[1::7, 30])
    plain = x.astype(np.float64) @ m.T.astype(np.float64)
    x[0, 100] = np.inf
    if rows > 1:
        x[rows - 1, 30], x[rows - 1, 31] = -np.inf, np.inf
    if rows > 20:
        x[17, 3], x[18, 64] = np.nan, -np.inf
    want = _ieee(x, m)
    res = np.ones((rows, n), np.float16)
    for o, add in ((K.layer_linear(_t(x, device), [_t(m, device)])[0], 0.0),
                   (K.layer_linear(_t(x, device), [_t(m, device)], K.LINEAR_RESIDUAL, residual=_t(res, device))[0], 1.0)):
        o = o.double().cpu().numpy()
        assert np.array_equal(np.isnan(o), np.isnan(want)) and np.array_equal(o[np.isinf(want)], want[np.isinf(want)])
        f = np.isfinite(want)
        assert np.all(np.abs(o[f] - want[f] - add) <= (np.abs(want[f]) + add) * 2.0 ** -10 + 2.0 ** -12)
    # SwiGLU of the same: gate and up past the norm's infinities (none here) as their products make them
    act, = K.layer_linear(_t(x, device), [_t(m, device), _t(w[1], device)], K.LINEAR_SWIGLU)
    act = act.double().cpu().numpy()
    with np.errstate(all="ignore"):
        gate, up = want, _ieee(x, w[1])
        ref = (gate * (1 / (1 + np.exp(-gate)))) * up
    assert np.array_equal(np.isnan(act), np.isnan(ref))
    assert np.array_equal(act[np.isinf(ref)], ref[np.isinf(ref)])


@pytest.mark.parametrize("k", [64, 192, 320, 2048, 2112, 8192, 8256, 32768])
def test_one_row_infinite_weights(device, k):
    """Infinite weights anywhere in a row, of one row of x: at the ends of k, of its 2,048-wide rounds and of the
    quarters that waves share from 8,192 on (the loads past a wave's share are not its own), and the widest k."""
    from apple_amd import kernels as K

    g, x, w = _data(1, k, 128, k)
    x = np.where(x == 0, np.float16(1), x)
    quarter = k // 4 if k >= 8192 else k
    spots = sorted({0, k - 1, k - 4, k // 2, min(2047, k - 1), min(2048, k - 1), quarter - 1, quarter % k, 2 * quarter % k})
    m = w[0].copy()
    for i, c in enumerate(spots):
        m[3 * i, c] = np.inf if i % 2 else -np.inf
    res = np.zeros((1, 128), np.float16)
    x64 = x.astype(np.float64)
    want = x64 @ w[0].T.astype(np.float64)
    mag = np.abs(x64) @ np.abs(w[0].T.astype(np.float64))
    for i, c in enumerate(spots):
        want[0, 3 * i] = np.inf * m[3 * i, c] * float(x[0, c])
    for o in (K.layer_linear(_t(x, device), [_t(m, device)])[0],
              K.layer_linear(_t(x, device), [_t(m, device)], K.LINEAR_RESIDUAL, residual=_t(res, device))[0]):
        o = o.double().cpu().numpy()
        assert np.array_equal(np.isinf(o), np.isinf(want)) and not np.isnan(o).any()
        f = np.isfinite(want)
        assert np.array_equal(o[~f], np.sign(want[~f]) * np.inf)
        assert np.all(np.abs(o[f] - want[f]) <= np.abs(want[f]) * 2.0 ** -11 + mag[f] * 2.0 ** -20 + 2.0 ** -24)


def test_refusals(device):
    import torch
    from apple_amd import kernels as K

    x = torch.zeros(2, 64, dtype=torch.float16, device=device)
    w = torch.zeros(8, 64, device=device)
    with pytest.raises(ValueError):
        K.layer_linear(x[:, :32].contiguous(), [w[:, :32].contiguous()])  # k below one MFMA run
    with pytest.raises(ValueError):
        K.layer_linear(x, [w[:6].contiguous()])                           # n not a multiple of 4
    with pytest.raises(ValueError):
        K.layer_linear(x, [w], head_dim=64, inv_freq=torch.ones(32, dtype=torch.float64, device=device))
