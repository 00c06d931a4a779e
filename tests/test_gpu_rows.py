"""The multi-row decode-order forward (rows.hip) against token steps.

Model::forward_phase over n ids (src/model.rs:469-477) is what n calls of one
id compute, bit for bit: the logits of the last row and every cached key and
value.  One-id calls run the token step, which the other tests pin to the
oracle; the first case here is pinned to the oracle directly.  Sizes sit at
the edges of the kernels: 16 queries per wave, 32-row tiles, 64-key blocks,
128 rows per attention workgroup, contraction lengths of fewer than eight
64-element lines and of a count that eight does not divide, the 256-block
limit past which blocks are added in pairs.  The instructions that this rests
on are compared with the oracle's fma chains in themselves: the FP32 MFMAs over
ordinary, wide-ranging and denormal operands, and the attention's own copy of
the exponential."""
import numpy as np
import pytest

from oracle import oracle as O
from yue2_rs_amd import synthetic
from yue2_rs_amd.api import Config
import yue2_rs_amd as y2

from helpers import bits, rb

pytestmark = pytest.mark.gpu


def _config(hidden, heads, kv_heads, head_dim, inter, layers=2, vocab=4096):
    return Config(hidden_size=hidden, num_hidden_layers=layers, num_attention_heads=heads,
                  num_key_value_heads=kv_heads, head_dim=head_dim, intermediate_size=inter, vocab_size=vocab,
                  max_position_embeddings=24576, rms_norm_eps=1e-6, rope_theta=10000.0)


SHAPES = {
    "d64": _config(1024, 16, 4, 64, 2816),          # 16, 16, 44 lines
    "d128": _config(1280, 10, 5, 128, 3456),        # 20, 20, 54 lines
    "small": _config(320, 4, 2, 64, 448),           # 5, 4, 7 lines
    "wide": _config(4096, 32, 8, 128, 14336, layers=1),
}


@pytest.fixture(scope="module", params=list(SHAPES), ids=list(SHAPES))
def shape(request, gpu, oracle_threads):
    ck = synthetic.checkpoint(SHAPES[request.param], seed=5)
    gm = y2.Model.open(ck)
    yield request.param, ck, gm
    gm.close()


def _filled(gm, context, capacity, seed):
    c, cfg = y2.Cache(gm, capacity), gm.config
    if context:
        rng = np.random.default_rng(seed)
        shape = (cfg.num_hidden_layers, context, cfg.num_key_value_heads * cfg.head_dim)
        c.load(rb(rng.standard_normal(shape)), rb(rng.standard_normal(shape)), context)
    return c


def _check(gm, context, n, seed, phase=0):
    cap = context + n + 3
    ids = synthetic.prompt(n + 1, gm.config.vocab_size, seed)
    a, b = _filled(gm, context, cap, seed), _filled(gm, context, cap, seed)
    print(f"context {context}, {n} ids", flush=True)
    got = gm.forward_phase(ids[:n], a, phase)
    for t in ids[:n]:
        want = gm.forward_phase([t], b, phase)
    assert a.length == b.length == context + n
    assert np.array_equal(bits(got), bits(want)), "last row's logits differ"
    for x, y in zip(a.export(context, n), b.export(context, n)):
        assert np.array_equal(bits(x), bits(y)), "cached rows differ"
    # and a step on top of the multi-row cache
    assert np.array_equal(bits(gm.forward(ids[n:], a)), bits(gm.forward(ids[n:], b)))
    a.close()
    b.close()


@pytest.mark.parametrize("n", [4, 15, 16, 17, 32, 33, 64, 65, 129, 300])
def test_prompt_equals_token_steps(shape, n):
    _check(shape[2], 0, n, seed=n)


@pytest.mark.parametrize("context,n", [(1, 5), (63, 5), (100, 37), (500, 130)])
def test_append_equals_token_steps(shape, context, n):
    _check(shape[2], context, n, seed=context + n)


@pytest.mark.parametrize("context,n", [(16290, 32), (16255, 130), (16256, 129), (16400, 35)])
def test_long_append_equals_token_steps(shape, context, n):
    if shape[0] in ("d64", "d128"):
        _check(shape[2], context, n, seed=context + n)


# from 256 workgroups of 128 rows on: as many as it takes, the last workgroup
# with n rows.  Past 16320 keys they run the attention kernels of long
# contexts: rows on both sides of the 256th block in one call (15000 cached
# keys), or all of them past it, ending in an odd and in an even number of
# blocks
@pytest.mark.parametrize("context,n", [(0, 1), (15000, 7), (16300, 128), (16400, 60)])
def test_many_rows_equal_token_steps(shape, context, n):
    name, _, gm = shape
    if name in ("d64", "d128"):
        heads = gm.config.num_attention_heads
        rows = 128 * (255 // heads) + n
        assert heads * -(-rows // 128) >= 256, "fewer workgroups than the long-context kernels are for"
        assert context == 0 or context + rows > 255 * 64
        _check(gm, context, rows, seed=n)


def test_more_rows_than_a_pass_takes(shape):
    """4096 rows go through the layers at a time: the second pass attends the
    first one's rows."""
    if shape[0] == "small":
        _check(shape[2], 0, 4096 + 37, seed=3)


def test_longest_prompt(shape):
    """24000 ids in one call: six passes, the last of them in the kernels of
    long contexts."""
    if shape[0] == "d64":
        _check(shape[2], 0, 24000, seed=6)


@pytest.mark.parametrize("step_kernel", [True, False])
def test_norm_fallbacks_counted(shape, step_kernel):
    """yue2_hip_norm_fallbacks counts a prompt's rows as it counts token
    steps."""
    gm, n = shape[2], 301
    ids = np.asarray(synthetic.prompt(n, gm.config.vocab_size, 9), np.int32)
    logits = np.empty(gm.config.vocab_size, np.float32)
    gm.set_step_kernel(step_kernel)
    counts = []
    for cuts in ([n], [1] * n):
        c, before, at = y2.Cache(gm, n), gm.norm_fallbacks(), 0
        for k in cuts:
            last = logits.ctypes.data if at + k == n else None
            assert y2.lib().yue2_hip_forward(gm._h, c._h, ids[at:].ctypes.data, k, 0, last) == 0
            at += k
        counts.append(gm.norm_fallbacks() - before)
        c.close()
    gm.set_step_kernel(True)
    assert counts[0] == counts[1] > 0


# (head_dim, context, rows, position of the id whose value overflows): in the
# middle of a wave's queries and of a block; in the last row of a block; a few
# rows past the 256th block; in the kernels of long contexts, with rows on both
# sides of it
@pytest.mark.parametrize("head_dim,context,n,at", [(64, 0, 83, 70), (128, 0, 83, 70), (64, 5, 200, 122), (128, 5, 40, 30),
                                                   (64, 16400, 40, 30), (128, 16400, 40, 30),
                                                   (64, 15000, 2048, 1400), (128, 15000, 2048, 1400)])
def test_rows_before_an_infinite_value(gpu, head_dim, context, n, at):
    """A row attends the keys up to its own: what is computed for it does not
    depend on the ids after it, also where a later id's value row overflows
    to infinity (0 * inf would be NaN)."""
    cfg = _config(1024, 16, 4, head_dim, 512, vocab=64)
    ck = synthetic.checkpoint(cfg, seed=3)
    # component 0 of the embedding: only id 63 has one, its only one, and it
    # overflows dimension 0 of its value in the first layer
    embed = ck.embed_tokens.reshape(cfg.vocab_size, -1)
    embed[:, 0] = 0
    embed[63] = 0
    embed[63, 0] = 0x3f80
    v = ck.layers[0].v_proj.reshape(-1, cfg.hidden_size)
    v[:] = 0
    v[0, 0] = 0x7f00  # 1.7e38; the norm makes the component 32
    rng = np.random.default_rng(n)
    v[1:, 1:] = (rb(0.02 * rng.standard_normal(v[1:, 1:].shape)).view(np.uint32) >> 16).astype(np.uint16)
    gm = y2.Model.open(ck)
    ids = np.asarray(synthetic.prompt(n, 63, 4), np.int32)
    print(f"head_dim {head_dim}, context {context}, {n} ids", flush=True)
    rows = []
    for special in (63, 7):
        ids[at] = special
        c = _filled(gm, context, context + n, 2)
        gm.forward_phase(ids, c, 0)
        rows.append([a[:, context:] for a in c.export(context, n)])
        c.close()
    gm.close()
    assert np.isinf(rows[0][1][0, at, 0]) and not np.isfinite(rows[0][0][1, at]).any(), "the id does not overflow"
    for x, y in zip(*rows):
        assert np.isfinite(y[:, :at]).all()
        assert np.array_equal(bits(x[:, :at]), bits(y[:, :at])), "rows before the infinity differ"


def test_prompt_equals_oracle(gpu, oracle_threads):
    ck = synthetic.checkpoint(SHAPES["d64"], seed=6)
    gm, om = y2.Model.open(ck), O.Model(ck)
    ids = synthetic.prompt(83, gm.config.vocab_size, 4)
    oc = O.Cache(om, 90)
    cache, got = gm.prefill_phase(ids, 90)
    assert np.array_equal(bits(got), bits(om.forward(ids, oc)))
    for x, y in zip(cache.export(), oc.arrays()):
        assert np.array_equal(bits(x), bits(y[:, :83]))
    gm.close()


def _selftest(which, x):
    out = np.empty_like(x)
    rc = y2.lib().yue2_hip_selftest_math(which, x.ctypes.data, out.ctypes.data, x.size)
    assert rc == 0, y2.lib().yue2_hip_last_error().decode()
    return out


# operands: the exponents they are spread over
@pytest.mark.parametrize("low,high", [(-1, 1), (-60, 60), (-80, -60), (-149, -120), (-149, 20)])
@pytest.mark.parametrize("which,side,rows", [(22, 16, 16), (23, 32, 16)])
def test_fp32_mfma_is_the_fma_chain(gpu, which, side, rows, low, high):
    rng = np.random.default_rng(which + high + 200)
    groups, n = 128, 2 * side * 8
    x = (rng.uniform(1, 2, groups * n) * 2.0 ** rng.integers(low, high, groups * n)).astype(np.float32)
    x *= rng.choice(np.array([-1, 1], np.float32), x.size)
    x[rng.random(x.size) < 0.02] = 0.0
    got = _selftest(which, x).reshape(groups, rows, side)
    L = O.lib()
    x = x.reshape(groups, 2, side, 8)
    want = np.empty_like(got)
    for g in range(groups):
        for r in range(rows):
            a = x[g, 0, r if side == rows else 2 * r + (g & 1)].ctypes.data
            for c in range(side):
                want[g, r, c] = L.y2o_dot_f32(a, x[g, 1, c].ctypes.data, 8)
    assert np.array_equal(bits(got), bits(want))


def test_attention_exponential(gpu):
    """Every f32 from -2^-27 down to -128, and the ends, against the library's
    other exponential, which test_gpu_math.py holds to the oracle's."""
    lo, hi = (int(np.float32(-v).view(np.uint32)) for v in (2.0 ** -27, 128.0))
    ends = np.array([0.0, -0.0, -1e-30, -1e-45, -150.0, -3e38, -np.inf, np.nan], np.float32)
    for at in range(lo, hi, 1 << 26):
        x = np.arange(at, at + (1 << 26), dtype=np.uint64).clip(lo, hi).astype(np.uint32).view(np.float32).copy()
        x[:8] = ends
        got, want = _selftest(21, x), _selftest(0, x)
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got)[~nan], bits(want)[~nan])
