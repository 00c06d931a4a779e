"""The scratch that a model keeps between its multi-row calls (runtime.h,
Scratch): kept up to 2 GiB, given back when a call needed more, and given back
when any other allocation of the library runs out of memory.  Requests beyond
the device's memory stand for the latter: they fail before anything is read."""
import ctypes as C
import time

import numpy as np
import pytest

from yue2_rs_amd import synthetic
from yue2_rs_amd.api import Config
import yue2_rs_amd as y2

from helpers import bits

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _free():
    free, total = C.c_size_t(), C.c_size_t()
    hip = C.CDLL("libamdhip64.so")
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _settled(at_least):
    """The free memory, once it is at_least (the driver clears what it gets
    back in its own time), or after five seconds."""
    until = time.monotonic() + 5
    while _free() < at_least and time.monotonic() < until:
        time.sleep(0.02)
    return _free()


def _too_large_cache(gm):
    with pytest.raises(y2.Yue2Error):
        y2.Cache(gm, 2**31 - 1)


def _too_large_gemm(gm):
    word = np.zeros(1, np.float32).ctypes.data
    assert y2.lib().yue2_hip_selftest_gemm(word, word, word, 1 << 30, 1, 1 << 16) < 0


@pytest.mark.parametrize("request_", [_too_large_cache, _too_large_gemm], ids=["cache", "selftest"])
def test_scratch_given_back_to_a_failing_allocation(gpu, request_):
    gm = y2.Model.open(synthetic.checkpoint(synthetic.REDUCED, seed=0))
    ids = synthetic.prompt(16000, gm.config.vocab_size, 1)
    cache = y2.Cache(gm, 16000)
    want = gm.forward_phase(ids, cache, 0)
    del cache
    kept = _free()
    request_(gm)
    assert _settled(kept + 64 * MIB) >= kept + 64 * MIB, "the scratch was kept"  # 4096 rows: 100 MiB
    cache = y2.Cache(gm, 16000)
    assert np.array_equal(bits(gm.forward_phase(ids, cache, 0)), bits(want))
    gm.close()


def test_large_scratch_given_back(gpu):
    """A prompt whose rows take 2.9 GB; then one that takes 0.9 GB."""
    cfg = Config(hidden_size=4096, num_hidden_layers=1, num_attention_heads=32, num_key_value_heads=8, head_dim=128,
                 intermediate_size=16384, vocab_size=4096, max_position_embeddings=24576, rms_norm_eps=1e-6,
                 rope_theta=10000.0)
    gm = y2.Model.open(synthetic.checkpoint(cfg, seed=0))
    free = {}
    for n in (64, 24576, 8192):
        cache, _ = gm.prefill_mfma(synthetic.prompt(n, cfg.vocab_size, 1), 24576)
        cache.close()
        free[n] = _settled(free.get(64, 0) - 64 * MIB if n == 24576 else 0)
    gm.close()
    assert free[24576] >= free[64] - 64 * MIB, "more than 2 GiB were kept"
    assert free[8192] <= free[64] - 512 * MIB, "the scratch was not kept"
