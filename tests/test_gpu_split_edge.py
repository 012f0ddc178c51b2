"""The stride-2 and the transposed convolutions on three bf16 parts, at the
edges of their tiles (128 pixels, 64 channels), channel chunks (16, by groups
of 8) and value ranges, against the oracle.

Tolerance: a product in parts is within 2^-23 of the f32 one and the sum of
up to 9 * 100 of them is rounded in f32 as before, so the 1e-5 relative bound of
the other operator tests holds with the same margin, at any scale."""
import numpy as np
import pytest

import oracle_api as O
from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5
# one group of 8 and less; an odd number of groups; ragged channels; one pixel
# past a 32 x 4 tile and past a 16 x 8 one; M past 32, 64, 96
SHAPES = [(5, 33, 6, 8), (24, 96, 9, 67), (100, 70, 19, 12), (16, 130, 66, 34), (3, 1, 2, 2)]


def _case(kind, cin, cout, h, w):
    rng = np.random.default_rng(cin * 5 + cout + h)
    x = rng.standard_normal((cin, h, w), np.float32)
    shape = (cout, cin, 3, 3) if kind == "down" else (cin, cout, 3, 3)
    wt = (rng.standard_normal(shape) * np.sqrt(2.0 / (cin * 9))).astype(np.float32)
    return x, wt


def _ref(kind, x, wt):
    if kind == "down":
        return O.conv2d(x, wt, None, pad=1, stride=2, reflect=True)
    return O.conv_transpose(x, wt, np.zeros(wt.shape[1], np.float32))


def _run(eng, kind, x, wt):
    if kind == "down":
        return eng.op_conv2d(x, wt, None, 2)
    m = wt.shape[1]
    return eng.op_conv_transpose(x, wt, np.zeros(m, np.float32), np.ones(m, np.float32), np.zeros(m, np.float32),
                                 relu=False)


@pytest.mark.parametrize("kind", ["down", "up"])
@pytest.mark.parametrize("cin,cout,h,w", SHAPES)
def test_any_magnitude(engine, kind, cin, cout, h, w):
    x, wt = _case(kind, cin, cout, h, w)
    ref = _ref(kind, x, wt)
    for sx, sw in ((1.0, 1.0), (2.0**-90, 2.0**20), (2.0**60, 2.0**-30)):
        got = _run(engine, kind, x * np.float32(sx), wt * np.float32(sw))
        assert rel_err(got.astype(np.float64) / (sx * sw), ref) < TOL
    for s in (np.logspace(-6, 6, cin), np.logspace(6, -6, cin)):  # rising and falling
        xs = x * s.astype(np.float32)[:, None, None]
        assert rel_err(_run(engine, kind, xs, wt), _ref(kind, xs, wt)) < TOL


@pytest.mark.parametrize("kind", ["down", "up"])
def test_nonfinite(engine, kind):
    """What reads an infinity or a NaN is not finite, the rest is unchanged."""
    cin, cout, h, w = 24, 40, 12, 40
    x, wt = _case(kind, cin, cout, h, w)
    ref = _ref(kind, x, wt)
    for v in (np.inf, -np.inf, np.nan):
        x[9, 6, 20] = v
        got = _run(engine, kind, x, wt)
        hit = np.zeros(ref.shape[1:], bool)
        if kind == "down":
            hit[3, 10] = True  # an even row and column: one output's centre
        else:
            hit[11:14, 39:42] = True
        assert not np.isfinite(got[:, hit]).any()
        assert rel_err(got[:, ~hit], ref[:, ~hit]) < TOL
