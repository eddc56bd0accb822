"""The tiled prefill's exact attention on int8 digit planes.

Cached fp16 values below 127 are four base-256 digits, and the digit sums are
put together in fp64 and rounded once, as the f64 forms' (Q3T_PF_ATT_INT=0)
are: the same bits at every length, but for an fp64 rounding that meets a tie
of the fp32 one (about one in 2^28, none in these rows); a cache with larger values or
infinities runs the f64 bodies of the same kernels.  Row counts are the edges
of the 64-row tiles, odd tile counts (the dealt-out middle tile) and the row
lengths where the softmax changes its register count.
"""
import sys

import numpy as np
import pytest

from qwen3_tts_amd import config as qcfg
from qwen3_tts_amd.device import Device
from qwen3_tts_amd.synth import Weights

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def model():
    cfg = qcfg.tiny()
    dev = Device(cfg)
    dev.upload_weights(Weights(cfg, "q8_0", seed=29))
    yield cfg, dev
    dev.close()


def both(dev, rows, past, monkeypatch):
    out = []
    for env in ("0", "1"):
        monkeypatch.setenv("Q3T_PF_ATT_INT", env)
        out.append(dev.prefill(rows, past))
    return out


def same(out, what):
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True), what


@pytest.mark.parametrize("past,n", [(0, 65), (0, 128), (0, 129), (63, 65), (1, 191), (300, 321), (1000, 88), (1980, 70),
                                    (2490, 130), (3996, 100), (4000, 100)])
def test_digit_attention_equals_f64(model, monkeypatch, past, n):
    """(4000, 100) is past the longest row of the digit form."""
    cfg, dev = model
    dev.kv_reserve(past + n)
    rng = np.random.default_rng(past + n)
    if past:
        shape = (past, cfg.n_kv_head, cfg.head_dim)
        for layer in range(cfg.n_layers):
            kv = rng.standard_normal((2,) + shape) * np.exp2(rng.integers(-14, 4, (2,) + shape))
            kv.reshape(-1)[rng.integers(0, kv.size, 64)] = np.resize([0.0, 126.9375, -126.9375, 2.0**-24, -(2.0**-24)], 64)
            kv = np.clip(kv, -126.9375, 126.9375).astype(np.float16)
            dev.kv_write(layer, kv[0], kv[1])
    rows = (rng.standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    say(f"[gpu] digit attention, {n} rows at {past}")
    same(both(dev, rows, past, monkeypatch), (past, n))


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("value", [127.0, -300.0, np.inf])
def test_values_without_digits_take_f64(model, monkeypatch, which, value):
    """One value of 127 or more in one layer's cache; the next call, with that value gone, is back on digits."""
    cfg, dev = model
    past, n = 70, 130
    dev.kv_reserve(past + n)
    rng = np.random.default_rng(7)
    kv = rng.standard_normal((2, past, cfg.n_kv_head, cfg.head_dim)).astype(np.float16)
    rows = (rng.standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    for layer in range(cfg.n_layers):
        dev.kv_write(layer, kv[0], kv[1])
    plain = both(dev, rows, past, monkeypatch)
    same(plain, "plain")
    bad = kv.copy()
    bad[0 if which == "k" else 1, 33, 0, 5] = value
    dev.kv_write(0, bad[0], bad[1])
    say(f"[gpu] {which} = {value} in the cache")
    wide = both(dev, rows, past, monkeypatch)
    same(wide, (which, value))
    assert not np.array_equal(wide[0][0], plain[0][0], equal_nan=True)
    dev.kv_write(0, kv[0], kv[1])
    again = both(dev, rows, past, monkeypatch)
    same(again, "again")
    same([plain[0], again[1]], "plain and again")


@pytest.mark.parametrize("value", [-300.0, np.inf])
def test_values_without_digits_in_a_contexts_first_prefill(model, monkeypatch, value):
    """The flag of such values is allocated, cleared and set by the first prefill that wants digits."""
    cfg, _ = model
    past, n = 70, 130
    kv = np.random.default_rng(8).standard_normal((2, past, cfg.n_kv_head, cfg.head_dim)).astype(np.float16)
    kv[0, 33, 0, 5] = value
    rows = (np.random.default_rng(9).standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    out = []
    for env in ("0", "1"):
        monkeypatch.setenv("Q3T_PF_ATT_INT", env)
        dev = Device(cfg)
        try:
            dev.upload_weights(Weights(cfg, "q8_0", seed=29))
            dev.kv_reserve(past + n)
            for layer in range(cfg.n_layers):
                dev.kv_write(layer, kv[0], kv[1])
            say(f"[gpu] first prefill, k = {value} in the cache, digits {env}")
            out.append(dev.prefill(rows, past))
        finally:
            dev.close()
    same(out, value)
