"""The int8 prefill GEMM's tiles, through the text projection.

Its row counts pick the tile (64 x 64, 64 x 32 with the blocks over two wave
pairs, 32 x 32 with stages of eight or four blocks); every sum is an exact
fp64 sum rounded once, so the rows equal the GEMV path's bit for bit on each
side of the rule's lines and at remainders of 1 and 31 rows.
"""
import sys

import numpy as np
import pytest

from qwen3_tts_amd import config as qcfg
from qwen3_tts_amd.device import Device
from qwen3_tts_amd.synth import Weights

pytestmark = pytest.mark.gpu



def test_text_projection_tiles_equal_gemv(monkeypatch):
    """2,048 wide: 64 x 32 from 12 tiles of 32 rows on (353), 64 x 64 from 28 tiles of 64 rows on (1,729)."""
    counts = (65, 128, 351, 352, 353, 415, 1728, 1729, 1823)
    cfg = qcfg.tiny(hidden=2048, n_layers=1, cp_layers=1, text_embd=2048)
    dev = Device(cfg)
    try:
        dev.upload_weights(Weights(cfg, "q8_0", seed=31))
        ids = np.random.default_rng(2048).integers(0, cfg.text_vocab, max(counts)).astype(np.int32)
        monkeypatch.setenv("Q3T_PREFILL_MFMA", "0")
        want = dev.text_proj(ids)
        monkeypatch.setenv("Q3T_PREFILL_MFMA", "1")
        for n in counts:
            print(f"[gpu] text projection of {n} ids", file=sys.stderr, flush=True)
            assert np.array_equal(dev.text_proj(ids[:n]), want[:n]), n
    finally:
        dev.close()


@pytest.mark.parametrize("n", [33, 65, 97])
def test_prefill_with_a_128_wide_projection_equals_gemv(monkeypatch, n):
    """One query head: the output projection's K is 128, one stage of four blocks."""
    cfg = qcfg.tiny(n_head=1, n_kv_head=1)
    dev = Device(cfg)
    try:
        dev.upload_weights(Weights(cfg, "q8_0", seed=37))
        dev.kv_reserve(n)
        rows = (np.random.default_rng(n).standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
        got = []
        for env in ("0", "1"):
            monkeypatch.setenv("Q3T_PREFILL_MFMA", env)
            print(f"[gpu] prefill of {n} rows, path {env}", file=sys.stderr, flush=True)
            got.append(dev.prefill(rows, 0))
        for a, b in zip(*got):
            assert np.array_equal(a, b)
    finally:
        dev.close()
