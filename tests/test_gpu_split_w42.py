"""The two-dimensional Winograd F(2x4, 3x3) kernel on three bf16 parts, where it
can go wrong: the edges of its 4-row x 64-pixel blocks (planes one row or
pixel past them, widths that are and are not multiples of 4, whose columns the
lanes take from their neighbours), ragged channels against its 8- and
16-channel groups, and the range of the values.

Tolerance: a product in parts is within 2^-23 of the f32 one and the sum of up
to 100 * 9 of them is rounded in f32 as before, so the 1e-5 relative bound of
the other operator tests holds with the same margin, at any scale."""
import numpy as np
import pytest

import oracle_api as O
from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5
SHAPES = [(8, 64, 9, 20), (24, 70, 6, 36), (13, 8, 11, 75), (16, 33, 4, 64), (100, 65, 5, 68), (40, 64, 8, 129),
          (3, 5, 2, 4)]


@pytest.fixture(scope="module")
def w42(pkg):
    with pytest.MonkeyPatch.context() as mp:
        mp.setenv("LAMA_FFC_WINO", "42")
        eng = pkg.hip_engine.Engine()
    yield eng
    eng.close()


def _case(cin, cout, h, w):
    rng = np.random.default_rng(cin * 3 + cout + w)
    x = rng.standard_normal((cin, h, w), np.float32)
    return x, (rng.standard_normal((cout, cin, 3, 3)) * np.sqrt(2.0 / (cin * 9))).astype(np.float32)


def _ref(x, wt):
    return O.conv2d(x, wt, None, pad=1, stride=1, reflect=True)


@pytest.mark.parametrize("cin,cout,h,w", SHAPES)
def test_any_magnitude(w42, cin, cout, h, w):
    x, wt = _case(cin, cout, h, w)
    ref = _ref(x, wt)
    for sx, sw in ((1.0, 1.0), (2.0**-90, 2.0**20), (2.0**60, 2.0**-30)):
        got = w42.op_conv2d(x * np.float32(sx), wt * np.float32(sw))
        assert rel_err(got.astype(np.float64) / (sx * sw), ref) < TOL
    for s in (np.logspace(-6, 6, cin), np.logspace(6, -6, cin)):  # rising and falling
        xs = x * s.astype(np.float32)[:, None, None]
        assert rel_err(w42.op_conv2d(xs, wt), _ref(xs, wt)) < TOL


@pytest.mark.parametrize("w", [40, 75])
def test_nonfinite(w42, w):
    """No finite value where the direct sum gives none; tiles that do not read
    the value keep theirs."""
    x, wt = _case(24, 40, 12, w)
    ref = _ref(x, wt)
    for ch, v in ((2, np.inf), (18, np.nan)):
        x[ch, 5, 9] = v
        got = w42.op_conv2d(x, wt)
        assert not np.isfinite(got[:, 4:7, 8:11]).any()
        far = np.ones((12, w), bool)
        far[2:8, 4:16] = False  # the tiles of 2 rows x 4 pixels that read row 5, column 9
        assert rel_err(got[:, far], ref[:, far]) < TOL
