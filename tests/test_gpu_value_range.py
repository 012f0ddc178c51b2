"""Every convolution kernel keeps its values apart: an output depends on the inputs
its sum (or its Winograd tile) reads and on nothing else of the workgroup's tile,
at any magnitude f32 holds, whatever the other channels and pixels are.

Tolerance: a product of two values in three bf16 parts is within 2^-23 of the
f32 one and the sum of up to 64 * 49 of them is rounded in f32 as before, so the
1e-5 relative bound of the other operator tests holds with the same margin.  At
the bottom of the range, values of about 2^-114 are off by up to half of the
smallest bf16, 2^-134: 1e-6 of them."""
import numpy as np
import pytest

import oracle_api as O
from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5

# kind: (cin, cout, h, w) of one tile or a few.  pw: the 32-pixel and the
# 64-pixel tiles, with 48 and 80 channels ending in the middle of the 32 that two
# waves share; w43, w42: F(4,3) and F(2x4, 3x3)
CASES = [("pw", 24, 96, 5, 9), ("pw", 13, 33, 6, 7), ("pw", 24, 48, 5, 9), ("pw", 96, 65, 190, 188),
         ("pw", 40, 80, 190, 188), ("w43", 24, 70, 6, 36), ("w43", 13, 8, 11, 75), ("w42", 24, 70, 8, 36),
         ("w42", 13, 8, 11, 75), ("down", 24, 70, 19, 24), ("up", 24, 70, 9, 24), ("head", 4, 64, 19, 33),
         ("head", 3, 33, 9, 40), ("tail", 40, 3, 17, 60)]


@pytest.fixture(scope="module")
def run(pkg, engine):
    with pytest.MonkeyPatch.context() as mp:
        mp.setenv("LAMA_FFC_WINO", "42")
        w42 = pkg.hip_engine.Engine()

    def f(kind, x, wt):
        print(f"case {kind} {x.shape} -> {wt.shape}", flush=True)
        if kind == "up":
            m = wt.shape[1]
            zero, one = np.zeros(m, np.float32), np.ones(m, np.float32)
            return engine.op_conv_transpose(x, wt, zero, one, zero, relu=False)
        if kind == "tail":
            return engine.op_tail(x, wt, np.zeros(3, np.float32))
        return (w42 if kind == "w42" else engine).op_conv2d(x, wt, None, 2 if kind == "down" else 1)

    yield f
    w42.close()


def _case(kind, cin, cout, h, w, seed):
    rng = np.random.default_rng(seed)
    k = {"pw": 1, "head": 7, "tail": 7}.get(kind, 3)
    x = rng.uniform(-1, 1, (cin, h, w)).astype(np.float32)
    shape = (cin, cout, k, k) if kind == "up" else (cout, cin, k, k)
    return x, (rng.standard_normal(shape) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32)


def _ref(kind, x, wt):
    if kind == "up":
        return O.conv_transpose(x, wt, np.zeros(wt.shape[1], np.float32))
    if kind == "pw":
        return O.conv2d(x, wt, None, pad=0, stride=1, reflect=True)
    if kind in ("head", "tail"):
        z = O.conv2d(O.reflect_pad(x, 3), wt, None, pad=0, stride=1, reflect=False)
        return 1.0 / (1.0 + np.exp(-z.astype(np.float64))) if kind == "tail" else z
    return O.conv2d(x, wt, None, pad=1, stride=2 if kind == "down" else 1, reflect=True)


def _reads(kind, shape, y, x):
    """The outputs that may depend on input pixel (y, x): those whose sum reads it,
    and for the Winograd kernels those of a tile that does."""
    if kind == "up":
        ys, xs = (2 * y - 1, 2 * y + 2), (2 * x - 1, 2 * x + 2)
    elif kind == "down":
        ys, xs = (y // 2, (y + 1) // 2 + 1), (x // 2, (x + 1) // 2 + 1)
    else:
        r = {"pw": 0, "head": 3, "tail": 3}.get(kind, 1)
        ys, xs = (y - r, y + r + 1), (x - r, x + r + 1)
        if kind in ("w43", "w42"):  # tiles of four columns; w42: and two rows
            xs = (xs[0] // 4 * 4, (xs[1] + 3) // 4 * 4)
        if kind == "w42":
            ys = (ys[0] // 2 * 2, (ys[1] + 1) // 2 * 2)
    hit = np.zeros(shape[1:], bool)
    hit[max(0, ys[0]):ys[1], max(0, xs[0]):xs[1]] = True
    return hit


@pytest.mark.parametrize("kind,cin,cout,h,w", CASES)
def test_ends_of_the_range(run, kind, cin, cout, h, w):
    x, wt = _case(kind, cin, cout, h, w, cin + w)
    ref = _ref(kind, x, wt)
    for sx, sw in ((2.0**-114, 2.0**100), (2.0**100, 2.0**-100), (2.0**119, 2.0**-100), (2.0**-100, 2.0**118)):
        got = run(kind, x * np.float32(sx), wt * np.float32(sw))
        if kind == "tail":  # the sigmoid of a sum that is scaled by a power of two
            z = -np.log(1.0 / ref - 1.0) * (sx * sw)
            ok = np.abs(z) < 80
            assert rel_err(got[ok], (1.0 / (1.0 + np.exp(-z)))[ok]) < TOL
        else:
            assert rel_err(got.astype(np.float64) / (sx * sw), ref) < TOL, (sx, sw)


@pytest.mark.parametrize("kind,cin,cout,h,w", CASES)
@pytest.mark.parametrize("v", [1e12, 1e30, np.inf, np.nan])
def test_other_pixels_of_the_tile(run, kind, cin, cout, h, w, v):
    """A huge, infinite or NaN pixel leaves alone what does not read it."""
    x, wt = _case(kind, cin, cout, h, w, 3 * cin + w)
    ref = _ref(kind, x, wt)
    py, px = (2, 5) if kind == "pw" else (h // 2, w // 2 + 2)
    x[:, py, px] = v
    got = run(kind, x, wt)
    hit = _reads(kind, ref.shape, py, px)
    assert hit.any() and (~hit).any()
    assert rel_err(got[:, ~hit], ref[:, ~hit]) < TOL
    if not np.isfinite(v) and kind != "tail":
        direct = _reads(kind if kind in ("up", "down", "pw", "head") else "3x3", ref.shape, py, px)
        assert not np.isfinite(got[:, direct]).any()


@pytest.mark.parametrize("kind,cin,cout,h,w", CASES)
def test_weights_that_undo_the_range_of_the_channels(run, kind, cin, cout, h, w):
    """Channels 2^40 apart whose weights bring them together again."""
    x, wt = _case(kind, cin, cout, h, w, 5 * cin + w)
    s = (2.0 ** np.round(np.linspace(-20, 20, cin))).astype(np.float32)
    np.random.default_rng(cin).shuffle(s)
    ws = s[:, None, None, None] if kind == "up" else s[None, :, None, None]
    assert rel_err(run(kind, x * s[:, None, None], wt / ws), _ref(kind, x, wt)) < TOL


@pytest.mark.parametrize("c,h,w", [(24, 5, 9), (13, 6, 7), (96, 190, 188)])
def test_values_keep_their_24_bits(run, c, h, w):
    """A 1x1 convolution with unit weights returns its input, bit for bit."""
    rng = np.random.default_rng(c)
    x = rng.standard_normal((c, h, w), np.float32) * (10.0 ** rng.uniform(-12, 12, (c, h, w))).astype(np.float32)
    assert np.array_equal(run("pw", x, np.eye(c, dtype=np.float32)[:, :, None, None]), x)
