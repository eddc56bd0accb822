"""Short Q8_0 prefills and text projections on the few-row GEMMs.

A Q8_0 model's prefill of 3 to 16 rows (2 to 63 behind enough history) and its
text projection of 2 to 64 ids run on the multi-stream decode's few-row
kernels (16-row activation tiles, K split over workgroups).  Sums are exact fp64 sums rounded once, so every row equals the
tiled prefill's and the GEMV's bit for bit; the row counts are the edges of
the 16-row tiles and of the range.
"""
import sys

import numpy as np
import pytest

from qwen3_tts_amd import config as qcfg
from qwen3_tts_amd.device import Device
from qwen3_tts_amd.synth import Weights

pytestmark = pytest.mark.gpu

ROWS = [2, 3, 9, 16, 17, 33, 48, 64, 65]


def say(*a):
    print(*a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module", params=["tiny", "tiny_mtp", "wide"])
def model(request):
    cfg = {"tiny": qcfg.tiny, "tiny_mtp": qcfg.tiny_mtp,
           # K splits above the 0.6B shapes' (2048 and 6144 wide, the 1.7B layout's)
           "wide": lambda: qcfg.tiny(n_layers=1, cp_layers=1, hidden=2048, ffn=6144, n_head=16, n_kv_head=8,
                                     text_embd=2048)}[request.param]()
    dev = Device(cfg)
    dev.upload_weights(Weights(cfg, "q8_0", seed=23))
    yield cfg, dev
    dev.close()


@pytest.mark.parametrize("kv", [1, 30])
@pytest.mark.parametrize("past", [0, 170])
def test_short_prefill_equals_other_paths(model, monkeypatch, kv, past):
    cfg, dev = model
    dev.kv_set_type(kv)
    dev.kv_reserve(256)
    rng = np.random.default_rng(past + kv)
    hist = (rng.standard_normal((170, cfg.hidden_size)) * 0.05).astype(np.float32)
    rows = (rng.standard_normal((65, cfg.hidden_size)) * 0.05).astype(np.float32)
    step = (rng.standard_normal(cfg.hidden_size) * 0.05).astype(np.float32)
    for n in ROWS:
        got = []
        for env in (None, "1", "0"):
            if env is None:
                monkeypatch.delenv("Q3T_PREFILL_MFMA", raising=False)
            else:
                monkeypatch.setenv("Q3T_PREFILL_MFMA", env)
            say(f"[gpu] prefill of {n} rows at {past}, cache type {kv}, path {env}")
            if past:
                dev.prefill(hist, 0)
            hid, logits = dev.prefill(rows[:n], past)
            # a step over the rows' cache entries
            got.append((hid, logits) + dev.talker_step(step, past + n))
        for other in got[1:]:
            for a, b in zip(got[0], other):
                assert np.array_equal(a, b), (n, float(np.abs(a - b).max()))


@pytest.mark.parametrize("side", [-1, 0])
@pytest.mark.parametrize("n,line", [(17, 60), (32, 60), (33, 320), (48, 320), (49, 600), (63, 600), (64, 600)])
def test_short_prefill_on_both_sides_of_its_lines(model, monkeypatch, n, line, side):
    """More than 16 rows take the few-row GEMMs from `line` cached positions on, times the layer's weights over the
    15,728,640 of the 0.6B layers; 64 rows never."""
    cfg, dev = model
    weights = cfg.hidden_size * ((2 * cfg.n_head + 2 * cfg.n_kv_head) * cfg.head_dim + 3 * cfg.ffn_size)
    past = -(-line * weights // 15728640) + side
    dev.kv_set_type(1)
    dev.kv_reserve(past + n + 1)
    rng = np.random.default_rng(past + n)
    kv = rng.standard_normal((2, past, cfg.n_kv_head, cfg.head_dim)).astype(np.float16)
    for layer in range(cfg.n_layers):
        dev.kv_write(layer, kv[0], kv[1])
    rows = (rng.standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    step = (rng.standard_normal(cfg.hidden_size) * 0.05).astype(np.float32)
    got = []
    for env in (None, "1", "0"):
        if env is None:
            monkeypatch.delenv("Q3T_PREFILL_MFMA", raising=False)
        else:
            monkeypatch.setenv("Q3T_PREFILL_MFMA", env)
        say(f"[gpu] prefill of {n} rows at {past}, path {env}")
        got.append(dev.prefill(rows, past) + dev.talker_step(step, past + n))
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b), float(np.abs(a - b).max())


def test_short_text_projection_equals_other_paths(model, monkeypatch):
    cfg, dev = model
    ids = np.random.default_rng(3).integers(0, cfg.text_vocab, 65).astype(np.int32)
    for n in [1] + ROWS:
        got = []
        for env in (None, "1", "0"):
            if env is None:
                monkeypatch.delenv("Q3T_PREFILL_MFMA", raising=False)
            else:
                monkeypatch.setenv("Q3T_PREFILL_MFMA", env)
            say(f"[gpu] text projection of {n} ids, path {env}")
            got.append(dev.text_proj(ids[:n]))
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2]), n
