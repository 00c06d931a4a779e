"""The VAE convolutions that run as products of BF16 parts (vae.hip,
conv_split_kernel): single convolutions against float64 at the sizes where
the tiles, rings and slots can go wrong, and a whole decoder whose last
blocks are long enough for the large tile, under the contract of
test_gpu_vae.py (max |device - f64| <= 4 max |oracle - f64| + 1e-6).

A single convolution is held to two measures.  Its root-mean-square distance
from float64 is no larger than that of the same sum taken as one FP32 fma
chain, K roundings of the growing sum (the kernel rounds 6 K / 16 times;
measured 0.70 to 0.90 of the chain's): leaving out one of the six products adds
9 to 53 times it, the three that are left out 0.02 to 0.08.  And where every
output is one product of integers, whose parts' products and sums FP32 holds
exactly, it is exact: 24-bit values against powers of two need x2 w0 or x0 w2,
12-bit values x1 w1."""
import numpy as np
import pytest

from oracle import oracle as O
import yue2_rs_amd as y2

from test_gpu_vae import _selftest
from vae_files import conv_case, conv_f64, decode_f64, oracle_ops, synthetic_vae, write_vae_dir

pytestmark = pytest.mark.gpu

# (transpose, cin, cout, kernel, stride, padding, dilation, frames)
SHAPES = [
    (False, 16, 17, 7, 1, 3, 1, 1),      # one row, one 16-channel group, a part of one column block
    (False, 16, 40, 7, 1, 27, 9, 300),   # the widest reach of the 7-tap slots, several row tiles
    (False, 48, 130, 5, 1, 2, 1, 65),    # a tile and a row; two blocks of padded columns
    (False, 32, 33, 1, 1, 0, 1, 64),     # one tap, a whole tile
    (False, 16, 64, 8, 1, 64, 18, 200),  # eight taps, reach 126
    (False, 128, 20, 2, 1, 32, 65, 129),
    (True, 32, 64, 20, 10, 5, 1, 40),    # ten phases of two taps
    (True, 16, 33, 12, 4, 2, 1, 7),      # three taps a phase
    (False, 16, 32, 7, 1, 3, 1, 49410),  # the large tile, a ragged last one
    (True, 16, 64, 8, 4, 2, 1, 12300),
]


def _sequential(transpose, x, w, bias, kernel, stride, padding, dilation, length):
    """The convolution as one float32 fma chain (a product and its sum are
    exact to 53 bits before they are rounded)."""
    x = x.astype(np.float64)
    y = np.zeros((length, w.shape[1] if transpose else w.shape[0]), np.float32)
    for j in range(kernel):
        if transpose:
            out = np.arange(x.shape[0]) * stride + j * dilation - padding
            ok = (out >= 0) & (out < length)
            out, src = out[ok], np.flatnonzero(ok)
        else:
            src = np.arange(length) * stride + j * dilation - padding
            ok = (src >= 0) & (src < x.shape[0])
            out, src = np.flatnonzero(ok), src[ok]
        for i in range(x.shape[1]):
            y[out] = x[src, i, None] * (w[i, :, j] if transpose else w[:, i, j]) + y[out]
    return y + bias


def _rms(a):
    return np.sqrt(np.mean(np.square(a, dtype=np.float64)))


@pytest.mark.parametrize("shape", SHAPES)
def test_convolution_shapes(gpu, shape):
    transpose, cin, cout, kernel, stride, padding, dilation, frames = shape
    x, w, b, want = conv_case(*shape)
    print(shape, flush=True)
    got = _selftest(transpose, cin, cout, kernel, stride, padding, dilation, x, w, b, want.shape[0])
    plain = _sequential(transpose, x, w, b, kernel, stride, padding, dilation, want.shape[0])
    print(f"rms from float64: {_rms(got - want):.3g}, one chain {_rms(plain - want):.3g}", flush=True)
    assert _rms(got - want) <= _rms(plain - want)
    # and no single output: four times the largest of the chain's
    assert np.abs(got - want).max() <= 4 * np.abs(plain - want).max()


@pytest.mark.parametrize("bits_x,bits_w", [(24, 0), (0, 24), (12, 12)])
@pytest.mark.parametrize("shape", SHAPES)
def test_all_parts_enter(gpu, shape, bits_x, bits_w):
    transpose, cin, cout, kernel, stride, padding, dilation, frames = shape
    rng = np.random.default_rng(frames + bits_x)

    def values(bits, size):  # of the given bits, the last one set; or 1, 2, 4
        v = rng.integers(1 << (bits - 1), 1 << bits, size) | 1 if bits else 1 << rng.integers(0, 3, size)
        return (v * rng.choice([-1, 1], size)).astype(np.float32)

    # rows with one input channel each, no two of them under one output
    x = np.zeros((frames, cin), np.float32)
    rows = np.arange(0, frames, -(-kernel // stride) if transpose else dilation * (kernel - 1) + 1)
    x[rows, rng.integers(0, cin, rows.size)] = values(bits_x, rows.size)
    w = values(bits_w, (cin, cout, kernel) if transpose else (cout, cin, kernel))
    bias = np.zeros(cout, np.float32)
    want = conv_f64(transpose, x, w, bias, kernel, stride, padding, dilation)
    assert np.count_nonzero(want)
    got = _selftest(transpose, cin, cout, kernel, stride, padding, dilation, x, w, bias, want.shape[0])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("frames", [1, 37, 1601])
def test_decode_with_both_tiles(gpu, tmp_path, frames):
    cfg, t = synthetic_vae(seed=11, channels=32, c_mults=(1, 2), strides=(4, 8))
    t = {n: a * np.float32(0.5) if n.endswith("weight_g") else a for n, a in t.items()}
    vae = y2.Vae(write_vae_dir(tmp_path, cfg, t))
    z = np.random.default_rng(frames).standard_normal((frames, 16)).astype(np.float32)
    print(f"{frames} frames", flush=True)
    got, exact = vae.decode(z), decode_f64(cfg, t, z)
    oracle = oracle_ops(cfg, t).run(z)
    assert np.abs(got - exact).max() <= 4 * np.abs(oracle - exact).max() + 1e-6
    vae.close()


def _long_vae(seed, **kw):
    cfg, t = synthetic_vae(seed=seed, channels=32, c_mults=(1, 2), strides=(4, 8), **kw)
    return cfg, {n: a * np.float32(0.5) if n.endswith("weight_g") else a for n, a in t.items()}


@pytest.mark.parametrize("arguments", ["ordinary", "large"])
def test_tiles_equal_the_whole_decode(gpu, tmp_path, arguments):
    """Tiles on the 64 x 64 kernel tile equal the whole decode, whose last
    blocks take the 256 x 128 one, bit for bit; also where some of SnakeBeta's
    arguments are past the range of its series (one channel, beside others in
    the same wave)."""
    cfg, t = _long_vae(12)
    if arguments == "large":
        for n in t:
            if n.endswith(".alpha"):
                t[n][3] = np.log(2e5)
    vae = y2.Vae(write_vae_dir(tmp_path, cfg, t))
    z = np.random.default_rng(8).standard_normal((1601, 16)).astype(np.float32)
    full, tiled = vae.decode(z), vae.decode_tiled(z, 64, vae.required_halo(64))
    vae.close()
    assert np.array_equal(full.view(np.uint32), tiled.view(np.uint32))


def _sine_squared(which, x):
    out = np.empty_like(x)
    rc = y2.lib().yue2_hip_selftest_math(which, x.ctypes.data, out.ctypes.data, x.size)
    assert rc == 0, y2.lib().yue2_hip_last_error().decode()
    return out.astype(np.float64)


@pytest.mark.parametrize("limit", [1.0, 10.0, 100.0, 1e4, 1e5])
def test_sine_squared(gpu, limit):
    """SnakeBeta's sin(x)^2 is no further from float64 than the square of the
    library's sinf: in the largest and the root-mean-square difference, and in
    the largest relative one, which multiples of pi and their neighbours
    decide."""
    rng = np.random.default_rng(int(limit))
    n = 1 << 21
    near = np.arange(1, int(limit / np.pi) + 1) * np.pi
    near = np.resize(near, n // 2).astype(np.float32) if near.size else rng.uniform(0, limit, n // 2).astype(np.float32)
    near = (near.view(np.int32) + rng.integers(-2, 3, near.size).astype(np.int32)).view(np.float32)
    x = np.concatenate([rng.uniform(-limit, limit, n), limit * np.exp(rng.uniform(-20, 0, n // 2)), near])
    x = x.astype(np.float32)
    want = np.sin(x.astype(np.float64)) ** 2
    measures = []
    for which in (19, 20):
        d = _sine_squared(which, x) - want
        measures.append([np.abs(d).max(), np.sqrt(np.mean(d * d)), (np.abs(d) / np.maximum(want, 1e-300)).max()])
    print(f"to {limit}: series {measures[0]}, sinf {measures[1]}", flush=True)
    assert all(a <= b for a, b in zip(*measures))


def test_sine_squared_of_what_is_not_finite(gpu):
    x = np.resize(np.array([np.inf, -np.inf, np.nan, 0.0], np.float32), 256)
    got = _sine_squared(19, x)
    assert np.isnan(got[x != 0]).all() and (got[x == 0] == 0).all()


HUGE = 3.4e38  # rounds to an infinite BF16 value
# (place, value): the activation at (70, 5) or the weight of output 2, input 5, tap 1
EXTREMES = [("x", np.inf), ("x", -np.inf), ("x", np.nan), ("x", HUGE), ("x", -HUGE), ("w", HUGE), ("w", -np.inf),
            ("w", np.nan)]


@pytest.mark.parametrize("place,value", EXTREMES)
@pytest.mark.parametrize("shape", [(False, 32, 40, 7, 1, 3, 1, 200), (False, 32, 33, 1, 1, 0, 1, 100),
                                   (True, 16, 64, 8, 4, 2, 1, 90), (False, 16, 32, 7, 1, 3, 1, 33000)])
def test_extreme_operands(gpu, shape, place, value):
    """Operands without finite BF16 parts give what FP32 arithmetic gives, and
    the outputs that they do not enter stay as they are."""
    transpose, cin, cout, kernel, stride, padding, dilation, frames = shape
    x, w, b, plain = conv_case(*shape)
    if place == "x":
        x[70, 5] = value
    else:
        tap = min(1, kernel - 1)
        w[(5, 2, tap) if transpose else (2, 5, tap)] = value
    with np.errstate(all="ignore"):
        want = conv_f64(transpose, x, w, b, kernel, stride, padding, dilation).astype(np.float32)
    got = _selftest(transpose, cin, cout, kernel, stride, padding, dilation, x, w, b, want.shape[0])
    same = np.abs(want - plain) < 1e30
    assert not same.all() and np.abs(got - plain)[same].max() <= 1e-5
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~same & ~np.isnan(want)
    assert np.array_equal(np.isinf(got[ok]), np.isinf(want[ok])) and np.array_equal(np.sign(got[ok]), np.sign(want[ok]))
    ok &= np.isfinite(want)
    # one product of full size: its rounding and those of the sum, which may
    # round again after each of the few products that follow
    assert (np.abs(got[ok] - want[ok]) <= 1e-6 * np.abs(want[ok])).all()


def test_infinite_activations_through_the_last_tanh(gpu, tmp_path):
    """An ELU decoder whose last unit overflows: its 1-tap convolution turns
    one infinite input into infinities of both signs, ELU those into infinity
    and -1, and the last convolution (weights of one sign) and tanh into
    finite audio."""
    cfg, t = _long_vae(13, snake=False)
    last = max(int(n.split(".")[2]) for n in t if n.startswith("decoder.layers."))
    t[f"decoder.layers.{last - 2}.layers.4.layers.1.bias"][0] = np.inf
    name = f"decoder.layers.{last}.weight_v"
    t[name] = np.abs(t[name])
    vae = y2.Vae(write_vae_dir(tmp_path, cfg, t))
    z = np.random.default_rng(8).standard_normal((40, 16)).astype(np.float32)
    got = vae.decode(z)
    vae.close()
    assert (got == 1.0).all()
