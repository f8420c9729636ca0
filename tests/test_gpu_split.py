"""The tower's convolution on split f16 operands (azh_tower.hpp): fp32
operands as two f16 parts under a power of two per board and per output
channel, three matrix products per pair, fp32 sums.

- every workgroup shape gives the same bits, within the fp32 summation bound
  K * u * sum|w||x| of float64, at channel counts that leave the last 32-channel
  chunk, co tile or quad part-filled, on every board size;
- scaling a board or a channel's weights by a power of two scales the outputs
  by it, bit for bit, across the whole range of the scales: they only move
  exponents;
- a value far above the rest of its board, or a weight far above the rest of
  its channel's, costs the sums that do not see it no precision;
- boards holding infinities or NaN, and channels with such weights, come out as
  the same products in fp32 give them, the same bits in every shape and in
  every form of a pass, and other boards and channel blocks as without them.
"""
import numpy as np
import pytest

import build
import oracle as O
from _util import U, bitwise_equal, conv_exact_and_bound, to_hip_cfg

pytestmark = pytest.mark.gpu

TILINGS = range(build.conv_tiling_count())


def _data(seed, n, cin, cout, B):
    rng = np.random.default_rng(seed)
    x = np.maximum(rng.standard_normal((B, cin, n * n)), 0).astype(np.float32)
    w = (rng.standard_normal((cout, cin * 9)) * np.sqrt(2.0 / (cin * 9))).astype(np.float32)
    return x, w


def _raw(hip, x, w, tiling=-1):
    cout = w.shape[0]
    return hip.probe_conv3x3(x, w, np.ones(cout, np.float32), np.zeros(cout, np.float32), relu=False, tiling=tiling)


@pytest.mark.parametrize("n,cin,cout,B", [(5, 16, 16, 3), (5, 48, 33, 2), (9, 32, 64, 3), (9, 80, 130, 2),
                                          (13, 16, 20, 2), (13, 96, 96, 2), (19, 112, 113, 2), (19, 144, 16, 2)])
def test_every_tiling_and_the_fp32_bound(hip, n, cin, cout, B):
    x, w = _data(n + cin + cout, n, cin, cout, B)
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs[1:]:
        assert bitwise_equal(o, outs[0])
    exact, mag = conv_exact_and_bound(x, w)
    assert (np.abs(outs[0] - exact) <= cin * 9 * U * mag + 1e-30).all()


# The smallest shapes stage four chunks of 32 input channels at a time: exactly
# one such round, a round and part of a chunk, two whole rounds, and two with
# one chunk left; blocks and column groups past the edge.
@pytest.mark.parametrize("n,cin,cout,B", [(19, 128, 17, 1), (13, 144, 16, 2), (9, 256, 33, 1), (5, 272, 16, 2)])
def test_staging_rounds(hip, n, cin, cout, B):
    x, w = _data(n * cin + cout, n, cin, cout, B)
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs[1:]:
        assert bitwise_equal(o, outs[0])
    exact, mag = conv_exact_and_bound(x, w)
    assert (np.abs(outs[0] - exact) <= cin * 9 * U * mag + 1e-30).all()


@pytest.mark.parametrize("kx,kw", [(0, 0), (90, -60), (-90, 60), (-20, -70), (60, 50)])
def test_powers_of_two_only_move_exponents(hip, kx, kw):
    x, w = _data(7, 9, 32, 32, 3)
    base = _raw(hip, x, w)
    scaled = x.copy()
    scaled[1] *= np.float32(2.0 ** kx)   # one board of the batch
    ws = w.copy()
    ws[5] *= np.float32(2.0 ** kw)       # one output channel
    got = _raw(hip, scaled, ws)
    want = base.copy()
    want[1] *= np.float32(2.0 ** kx)
    want[:, 5] *= np.float32(2.0 ** kw)
    assert np.isfinite(want).all() and bitwise_equal(got, want)


def _fp32_grade(got, exact, mag, K):
    """Within the bound of any fp32 order, and as close as the fp32 matrix
    units' sums of random terms: K / 4 additions that each round a partial sum,
    the partial sums no larger than the whole, in quadrature."""
    err = np.abs(got.astype(np.float64) - exact)
    assert (err <= K * U * mag).all()
    rms = np.sqrt((err ** 2).mean() / (exact ** 2).mean())
    assert rms <= U * np.sqrt(K / 4), f"{rms:.2e} of the sums"


@pytest.mark.parametrize("spread", [8, 14, 17, 20, 24, 30, 40, 90])
@pytest.mark.parametrize("n,F", [(5, 16), (9, 64), (13, 32), (19, 144)])
def test_a_value_far_above_its_board(hip, n, F, spread):
    """One activation 2^spread times the others' scale: the sums whose window
    does not hold it, and the other boards', are as good as without it."""
    x, w = _data(41 + n, n, F, F, 2)
    clean = _raw(hip, x, w)
    at = (n // 2) * n + n // 2
    x[1, F // 2, at] = np.float32(2.0 ** spread)
    exact, mag = conv_exact_and_bound(x, w)
    rows, cols = np.divmod(np.arange(n * n), n)
    away = (np.abs(rows - n // 2) > 1) | (np.abs(cols - n // 2) > 1)
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs[1:]:
        assert bitwise_equal(o, outs[0])
    assert bitwise_equal(outs[0][0], clean[0])
    _fp32_grade(outs[0][1][:, away], exact[1][:, away], mag[1][:, away], F * 9)
    assert (np.abs(outs[0][1] - exact[1]) <= F * 9 * U * mag[1]).all()


@pytest.mark.parametrize("spread", [8, 14, 17, 20, 24, 30, 40, 90])
@pytest.mark.parametrize("n,F", [(9, 64), (19, 128)])
@pytest.mark.parametrize("few", [False, True])
def test_a_weight_far_above_its_channel(hip, n, F, spread, few):
    """One weight 2^spread times the others of its channel, on an input that is
    zero; few: all but five of the others are zero."""
    x, w = _data(43 + n, n, F, F, 2)
    x[:, 5] = 0
    if few:
        w[3] = 0
        w[3, 11::2 * F] = 0.01 + np.arange(5, dtype=np.float32) / 97
    w[3, 5 * 9 + 4] = np.float32(2.0 ** spread)
    exact, mag = conv_exact_and_bound(x, w)
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs[1:]:
        assert bitwise_equal(o, outs[0])
    _fp32_grade(outs[0][:, 3], exact[:, 3], mag[:, 3], F * 9)
    rest = np.delete(np.arange(F), 3)
    _fp32_grade(outs[0][:, rest], exact[:, rest], mag[:, rest], F * 9)


def test_boards_of_zeros_and_of_denormals(hip):
    x, w = _data(47, 9, 32, 32, 3)
    x[0] = 0
    x[1] *= np.float32(2.0 ** -122)
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    exact, mag = conv_exact_and_bound(x, w)
    for o in outs:
        assert bitwise_equal(o, outs[0]) and not o[0].any()
        assert (np.abs(o - exact) <= 32 * 9 * (U * mag + 2.0 ** -149)).all()


@pytest.mark.parametrize("n,F", [(5, 16), (9, 64), (19, 128)])
def test_infinities_and_nan(hip, n, F):
    B = 3
    x, w = _data(11 + n, n, F, F, B)
    clean = _raw(hip, x, w)
    x[1, 3, 4] = np.inf
    x[1, 7, n * n - 1] = np.nan
    for weights in (False, True):
        if weights:
            w[2, 9 + 4] = -np.inf
        with np.errstate(invalid="ignore"):
            exact, mag = conv_exact_and_bound(x, w)
        inf, fin = np.isinf(exact), np.isfinite(exact)
        outs = [_raw(hip, x, w, t) for t in TILINGS]
        for o in outs:
            assert np.array_equal(o, outs[0], equal_nan=True)
            assert np.array_equal(np.isnan(o), np.isnan(exact))
            assert np.array_equal(np.isinf(o), inf) and np.array_equal(o[inf], exact[inf])
            assert (np.abs(o[fin] - exact[fin]) <= F * 9 * U * mag[fin] + 1e-30).all()
            if not weights:
                assert bitwise_equal(o[0], clean[0]) and bitwise_equal(o[2], clean[2])


@pytest.mark.parametrize("cfg", [O.make_cfg(5, 2, 20), O.make_cfg(9, 2, 48), O.make_cfg(13, 1, 32),
                                 O.make_cfg(19, 2, 128)])
@pytest.mark.parametrize("value", [np.inf, 2.0 ** 22, 2.0 ** 60])
def test_infinite_inputs_same_bits_in_every_form(hip, cfg, value):
    """Positions of which one holds an infinity, or a value far above the rest: the one-launch forms (a board
    in LDS, a board resident) and the per-layer launches agree bit for bit,
    and the other positions are untouched."""
    net = O.random_network(cfg, 77)
    B = 70 if cfg.board != 19 else 3
    inp = np.random.default_rng(5).integers(0, 2, (B, cfg.planes, cfg.area)).astype(np.float32)
    bad = inp.copy()
    bad[1, 0, 3] = value
    with hip.Runner(to_hip_cfg(hip, cfg), net.tensors(), B, 1) as r:
        r.set_resident_tower(2)
        clean, one = r.infer(inp), r.infer(bad)
        r.set_resident_tower(0)
        r.set_small_tower(False)
        per_layer = r.infer(bad)
    rest = np.delete(np.arange(B), 1)
    for a, b, c in zip(one, per_layer, clean):
        assert bitwise_equal(a[rest], c[rest]) and bitwise_equal(b[rest], c[rest])
        assert np.array_equal(a[1], b[1], equal_nan=True)


@pytest.mark.parametrize("n,F", [(5, 20), (9, 64), (13, 40), (19, 128)])
def test_infinite_weight_stays_in_its_channel_block(hip, n, F):
    """One infinite weight: the 16 channels of its block are summed from the
    weights as given (channel 1's span 2^30, the large one on an input that is
    zero, so that no rounding of it may show in the small ones' sums), the
    others have the bits they have without it."""
    F = -(-F // 16) * 16
    x, w = _data(23 + n, n, F, F + 4, 2)
    x[:, 0] = 0
    w[1] *= np.float32(2.0 ** -30)
    w[1, 4] = 1.0
    clean = _raw(hip, x, w)
    w[3, 5 * 9 + 4] = np.inf
    with np.errstate(invalid="ignore"):
        exact, mag = conv_exact_and_bound(x, w)
    fin = np.isfinite(exact)
    assert not fin[:, 3].any() and fin[:, :3].all()
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs:
        assert np.array_equal(o, outs[0], equal_nan=True)
        assert bitwise_equal(o[:, 16:], clean[:, 16:])
        assert np.array_equal(np.isnan(o), np.isnan(exact)) and (o[np.isinf(exact)] == exact[np.isinf(exact)]).all()
        assert (np.abs(o[fin] - exact[fin]) <= F * 9 * U * mag[fin]).all()


@pytest.mark.parametrize("n,F", [(5, 16), (9, 64), (19, 144)])
def test_few_weights_below_the_parts(hip, n, F):
    """A channel whose sums are made by three weights 2^-30 of its largest, on
    a board with an infinity in a corner: away from it the sums see every bit
    of them, and the infinity meets them as it would the weights as given."""
    x, w = _data(31 + n, n, F, F, 2)
    x[:, 0] = 0
    x[1, 2, 0] = np.inf
    w[1] = 0
    w[1, :9] = 1.0
    for c, tap in ((1, 4), (5, 0), (F - 1, 8)):
        w[1, c * 9 + tap] = np.float32(2.0 ** -30 * (1.1 + 0.3 * c))
    w[2, 2 * 9 + 4] = np.float32(-2.0 ** -40)   # below both parts; meets the infinity
    with np.errstate(invalid="ignore"):
        exact, mag = conv_exact_and_bound(x, w)
    fin = np.isfinite(exact)
    assert exact[1, 2, 0] == -np.inf
    outs = [_raw(hip, x, w, t) for t in TILINGS]
    for o in outs:
        assert np.array_equal(o, outs[0], equal_nan=True)
        assert np.array_equal(np.isnan(o), np.isnan(exact)) and (o[np.isinf(exact)] == exact[np.isinf(exact)]).all()
        assert (np.abs(o[1][fin[1]] - exact[1][fin[1]]) <= F * 9 * U * mag[1][fin[1]]).all()


@pytest.mark.parametrize("cfg", [O.make_cfg(5, 2, 20), O.make_cfg(9, 2, 48), O.make_cfg(13, 2, 32),
                                 O.make_cfg(19, 2, 128)])
def test_infinite_weights_same_bits_in_every_form(hip, cfg):
    net = O.random_network(cfg, 78)
    t = net.tensors()
    t["block0.conv2.w"][5 * 9 * cfg.filters + 4] = np.inf
    t["block1.conv1.w"][2 * 9 * cfg.filters + 13] = -np.inf
    B = 70 if cfg.board != 19 else 3
    inp = np.random.default_rng(6).integers(0, 2, (B, cfg.planes, cfg.area)).astype(np.float32)
    with hip.Runner(to_hip_cfg(hip, cfg), t, B, 1) as r:
        r.set_resident_tower(2)
        one = r.infer(inp)
        r.set_resident_tower(0)
        r.set_small_tower(False)
        per_layer = r.infer(inp)
    for a, b in zip(one, per_layer):
        assert np.array_equal(a, b, equal_nan=True)
