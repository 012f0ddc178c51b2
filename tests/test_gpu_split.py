"""The kernels that multiply f32 values as three bf16 parts, where the split can
go wrong: tiny and huge values, values that grow or fall along the channels,
ragged channel counts against the 8- and 16-channel groups, infinities and NaNs.

Tolerance: a product in parts is within 2^-23 of the f32 one and the sum of up
to 1152 of them is rounded in f32 as before, so the 1e-5 relative bound of the
other operator tests holds with the same margin, at any scale."""
import numpy as np
import pytest

import oracle_api as O
from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _case(cin, cout, h, w, k, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((cin, h, w), np.float32)
    wt = (rng.standard_normal((cout, cin, k, k)) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32)
    return x, wt


def _ref(x, wt):
    k = wt.shape[2]
    return O.conv2d(x, wt, None, pad=k // 2, stride=1, reflect=True)


# 1x1: below one 16-channel step, one fill, several fills; a plane past the
# small tiles' range (64 x 64 tiles: more than 512).  3x3: one group of 8, an
# odd number of groups, ragged channels.
SHAPES = [(5, 33, 6, 7, 1), (24, 96, 5, 9, 1), (400, 40, 8, 8, 1), (100, 200, 190, 100, 1), (96, 65, 190, 188, 1),
          (8, 64, 9, 20, 3), (24, 70, 6, 36, 3), (13, 8, 11, 75, 3)]


@pytest.mark.parametrize("cin,cout,h,w,k", SHAPES)
def test_any_magnitude(engine, cin, cout, h, w, k):
    x, wt = _case(cin, cout, h, w, k, cin + cout)
    ref = _ref(x, wt)
    for sx, sw in ((1.0, 1.0), (2.0**-90, 2.0**20), (2.0**60, 2.0**-30), (2.0**-20, 2.0**-60)):
        print(f"case {cin}->{cout} {h}x{w} k{k} x*{sx:g} w*{sw:g}", flush=True)
        got = engine.op_conv2d(x * np.float32(sx), wt * np.float32(sw))
        assert rel_err(got.astype(np.float64) / (sx * sw), ref) < TOL


@pytest.mark.parametrize("cin,cout,h,w,k", SHAPES)
@pytest.mark.parametrize("rising", [True, False])
def test_magnitudes_along_the_channels(engine, cin, cout, h, w, k, rising):
    """Channels from 1e-6 to 1e6, either way round."""
    x, wt = _case(cin, cout, h, w, k, 3 * cin + cout)
    s = np.logspace(-6, 6, cin).astype(np.float32)
    x *= (s if rising else s[::-1])[:, None, None]
    assert rel_err(engine.op_conv2d(x, wt), _ref(x, wt)) < TOL


@pytest.mark.parametrize("cin,cout,h,w,k", [s for s in SHAPES if s[4] == 1])
def test_nonfinite_pointwise(engine, cin, cout, h, w, k):
    """An infinity gives what the f32 products give, a NaN a NaN, and the other
    pixels of the tile keep their values."""
    x, wt = _case(cin, cout, h, w, k, 5 * cin + cout)
    ref = _ref(x, wt)
    x[1, 0, 1], x[3, 2, 3] = np.inf, -np.inf
    x[2, 4, 4] = np.nan
    got = engine.op_conv2d(x, wt)
    bad = np.zeros((h, w), bool)
    bad[0, 1] = bad[2, 3] = bad[4, 4] = True
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[:, 0, 1], wt[:, 1, 0, 0] * np.float32(np.inf))
        assert np.array_equal(got[:, 2, 3], wt[:, 3, 0, 0] * np.float32(-np.inf))
    assert np.isnan(got[:, 4, 4]).all()
    assert rel_err(got[:, ~bad], ref[:, ~bad]) < TOL


@pytest.mark.parametrize("cin,cout,h,w,k", [s for s in SHAPES if s[4] == 3])
def test_nonfinite_3x3(engine, cin, cout, h, w, k):
    """A Winograd tile that reads an infinity or a NaN gives no finite value
    where the direct sum gives none, and tiles that do not read it keep theirs."""
    x, wt = _case(cin, cout, h, w, k, 7 * cin + cout)
    ref = _ref(x, wt)
    for v in (np.inf, np.nan):
        x[2, 3, 9] = v
        got = engine.op_conv2d(x, wt)
        assert not np.isfinite(got[:, 2:5, 8:11]).any()
        far = np.ones((h, w), bool)
        far[1:6, 4:16] = False  # the tiles of up to two rows by four columns that read row 3, column 9
        assert rel_err(got[:, far], ref[:, far]) < TOL
