"""The backend's standing workloads, each built exactly as specified, on the GPU
against the CPU oracle:

* the bench workload: 512x512, the brush-stroke mask that
  bench.py draws (synth_mask_strokes(0.25, seed 2)), blurred-noise image
  seed 1, the seed-0 weights -- both as bench.py loads them (plain BN
  statistics) and with calibrated BN statistics;
* 256x256 with one seeded 64-wide x 96-tall rectangle, plain and
  calibrated weights;
* the SpectralTransform alone, 18 blocks with distinct weights on
  384 x 64 x 64 N(0,1) inputs, every stage of each block.

Whole passes are checked at every plan step (relative L2 error <= 1e-3, the
per-layer bound) through lama_hip_forward_steps; the sigmoid
output value by value (within 1/255 wherever its pre-activation is
well-conditioned, see _check_output); and the production path
(lama_hip_forward: three streams, no step synchronisation) must equal the
step-synchronised pass bit for bit.  The 8-bit result is checked through
lama_hip_inpaint (device build_input and composite): within 1 level max and
0.1 mean of the oracle's composite, unmasked pixels bit-exact."""
import numpy as np
import pytest

import oracle_api as O
from conftest import rel_err

pytestmark = pytest.mark.gpu

STEP_TOL = 1e-3


@pytest.fixture(scope="module")
def plain_engine(pkg, weights_dir):
    eng = pkg.hip_engine.Engine()
    eng.load_weights(pkg.host_api.Store(weights_dir["plain"]))
    yield eng
    eng.close()


@pytest.fixture(scope="module")
def weights(weights_dir):
    return {k: O.read_safetensors(weights_dir[k]) for k in ("plain", "cal")}


@pytest.fixture(scope="module")
def oracles(weights):
    return {k: O.OracleNet(v) for k, v in weights.items()}


def _ill_conditioned(W, step27, co, y, x):
    """The output convolution at pixel (co, y, x) recomputed in f64 from the
    oracle's step-27 input: True when |v| <= 1e-3 * sum |terms|, i.e. when an
    input perturbation within the per-layer bound (1e-3 relative) can move v
    across zero and flip the saturated sigmoid."""
    wt = np.asarray(W["model.34.weight"], np.float64)[co]
    patch = step27[:, y:y + 7, x:x + 7].astype(np.float64)
    terms = wt * patch
    v = terms.sum() + float(W["model.34.bias"][co])
    return abs(v) <= 1e-3 * (np.abs(terms).sum() + abs(float(W["model.34.bias"][co])))


def _check_output(label, got, ref, step27, W, h, w):
    """The sigmoid output: within 1/255 of the oracle at every value whose
    pre-activation is well-conditioned.  With the plain fixture weights the
    activations grow ~4x per resblock and the tail's pre-activations reach
    ~1e10, so the sigmoid is saturated and a value whose pre-activation cancels
    to near zero can flip between 0 and 1 under f32 rounding; those values are
    shown to be ill-conditioned one by one, and must be rare."""
    bad = np.argwhere(np.abs(got - ref) > 1.0 / 255)
    assert len(bad) <= 1e-5 * got.size, (label, len(bad))
    s27 = step27.reshape(64, h + 6, w + 6)
    for co, y, x in bad:
        assert _ill_conditioned(W, s27, co, y, x), (label, co, y, x, got[co, y, x], ref[co, y, x])
    return {(int(y), int(x)) for _, y, x in bad}


def _check_pass(pkg, eng, net, W, img, mask, label):
    H = pkg.host_api
    h, w = mask.shape
    x = H.build_input(img, mask)
    print(f"case {label}: {h}x{w}", flush=True)
    ref, ref_steps = net.forward(x, steps=True)
    got, got_steps = eng.forward_steps(x, list(range(29)))
    for s in range(28):
        e = rel_err(got_steps[s], ref_steps[s])
        assert e < STEP_TOL, f"{label} step {s}: rel err {e:.3e}"
    flips = _check_output(label, got, ref, ref_steps[27], W, h, w)
    # the production schedule (overlapped streams, no per-step drains)
    prod = eng.forward(x)
    assert np.array_equal(prod, got), "stream schedule differs from the step-synchronised one"
    # the device-side inpaint flow: the same pass, composited on the device
    u8, net_out = eng.inpaint(img, mask, net_out=True)
    assert np.array_equal(net_out, prod)
    u8r = O.composite(img, mask, ref, 0, 0)
    d = np.abs(u8.astype(int) - u8r.astype(int))
    for y, x in flips:
        d[y, x] = 0  # shown ill-conditioned above
    assert d.max() <= 1 and d.mean() <= 0.1, (label, d.max(), d.mean())
    assert np.array_equal(u8[mask == 0], img[mask == 0])
    assert np.array_equal(u8, O.composite(img, mask, net_out, 0, 0))
    return len(flips)


@pytest.mark.parametrize("kind", ["plain", "cal"])
def test_config3_bench_workload_512(pkg, engine, plain_engine, oracles, weights, kind):
    H = pkg.host_api
    img = H.synth_image(512, 512, 1)
    mask, cov = H.synth_mask_strokes(512, 512, 0.25, 2)
    assert 0.2 < cov < 0.3
    eng = plain_engine if kind == "plain" else engine
    flips = _check_pass(pkg, eng, oracles[kind], weights[kind], img, mask, f"512x512 {kind}")
    if kind == "cal":
        assert flips == 0


@pytest.mark.parametrize("kind", ["plain", "cal"])
def test_config0_256_rect_64x96(pkg, engine, plain_engine, oracles, weights, kind):
    H = pkg.host_api
    img = H.synth_image(256, 256, 1)
    mask, (x0, y0) = H.synth_mask_rect(256, 256, 64, 96, 2)
    assert mask.sum() // 255 == 64 * 96
    assert mask[y0:y0 + 96, x0:x0 + 64].all()
    eng = plain_engine if kind == "plain" else engine
    flips = _check_pass(pkg, eng, oracles[kind], weights[kind], img, mask, f"256x256 {kind}")
    if kind == "cal":
        assert flips == 0


def test_config2_spectral_transform_18_blocks(plain_engine, oracles):
    """FFCs 0..17 (model.5.conv1 .. model.13.conv2), each on its
    own seeded N(0,1) 384 x 64 x 64 input: f, spectrum, FU conv, f + ifft
    and the output each within 1e-3 of the oracle."""
    net = oracles["plain"]
    names = ["f", "spectrum", "fu", "f+ifft"]
    for k in range(18):
        x = np.random.default_rng(1000 + k).standard_normal((384, 64, 64)).astype(np.float32)
        print(f"case spectral block {k}", flush=True)
        ref, ref_st = net.spectral(k, x, stages=True)
        got, got_st = plain_engine.spectral(k, x, stages=True)
        for i in range(4):
            e = rel_err(got_st[i], ref_st[i])
            assert e < STEP_TOL, f"block {k} {names[i]}: rel err {e:.3e}"
        e = rel_err(got, ref)
        assert e < STEP_TOL, f"block {k} out: rel err {e:.3e}"


@pytest.mark.parametrize("hw", [(75, 75), (32, 17)])
def test_spectral_transform_other_planes(plain_engine, oracles, hw):
    """The isolated SpectralTransform at the 600x600 bottleneck (75 = 3 * 5 * 5,
    the reference's opposite-sign Bluestein rule) and a ragged plane."""
    h, w = hw
    x = np.random.default_rng(7).standard_normal((384, h, w)).astype(np.float32)
    print(f"case spectral {h}x{w}", flush=True)
    ref, ref_st = oracles["plain"].spectral(3, x, stages=True)
    got, got_st = plain_engine.spectral(3, x, stages=True)
    for i in range(4):
        assert rel_err(got_st[i], ref_st[i]) < STEP_TOL, i
    assert rel_err(got, ref) < STEP_TOL


def test_spectral_rejects_bad_index(pkg, plain_engine):
    with pytest.raises(pkg.hip_engine.HipError, match="outside 0..35"):
        plain_engine.spectral(36, np.zeros((384, 8, 8), np.float32))
