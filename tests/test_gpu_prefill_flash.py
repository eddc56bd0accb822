"""The fast attention of the tiled F16 prefill (scores, softmax and P.V in one kernel) and its GEMM tiles.

Its rows against the exact form's (Q3T_PF_EXACT=1) over the edges of the 64-row and 64-position tiles, behind
cached positions whose keys grow or shrink with the position, so that a row's weight lies late or early in its
sweep, and with a bfloat16 cache.  Tolerance: the probabilities are rounded to 11 bits (bfloat16: 8), each
GEMM input to 11, so a row moves by a few 2^-12 (2^-9) of its largest value per layer; two layers, with room for
the sums' own spread, stay within 2^-8 (2^-6).  The second layer's q comes from sums that the two forms round
differently, and a q element that falls the other way moves by 2^-10 (2^-7) of itself: against the grown keys (up
to 30, q up to 3, scale 2^-3.5) a score then moves by 30 * 3 * 2^-3.5 * 2^-10 = 2^-7 (2^-4), and the weight it carries
by as much; those rows get twice the tolerance.
"""
import sys

import numpy as np
import pytest
import torch

from qwen3_tts_amd import config as qcfg
from qwen3_tts_amd.device import Device
from qwen3_tts_amd.synth import Weights

pytestmark = pytest.mark.gpu
BF16 = 30


def say(*a):
    print(*a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module", params=["f16", "bf16"])
def model(request):
    cfg = qcfg.tiny()
    dev = Device(cfg)
    dev.upload_weights(Weights(cfg, "f16", seed=31))
    if request.param == "bf16":
        dev.kv_set_type(BF16)
    yield cfg, dev, request.param == "bf16"
    dev.close()


SIZES = [(0, 64), (0, 65), (0, 127), (0, 193), (1, 64), (63, 65), (10, 119), (300, 321), (3000, 70)]


@pytest.mark.parametrize("past,n,growth", [(p, n, g) for p, n in SIZES for g in (0.0, 2.0, -2.0) if p or not g])
def test_flash_attention_against_exact(model, monkeypatch, past, n, growth):
    cfg, dev, bf = model
    dev.kv_reserve(past + n)
    rng = np.random.default_rng(past + n)
    for layer in range(cfg.n_layers if past else 0):
        kv = rng.standard_normal((2, past, cfg.n_kv_head, cfg.head_dim)).astype(np.float32)
        kv[0] *= np.exp(growth * np.linspace(-1, 1, past))[:, None, None]
        if bf:
            k, v = (torch.from_numpy(a).bfloat16().view(torch.int16).numpy().view(np.uint16) for a in kv)
        else:
            k, v = kv.astype(np.float16)
        dev.kv_write(layer, k, v)
    rows = (rng.standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    out = {}
    for exact in ("1", "0"):
        monkeypatch.setenv("Q3T_PF_EXACT", exact)
        out[exact] = dev.prefill(rows, past)[0].astype(np.float64)
    rel = np.abs(out["0"] - out["1"]).max(axis=1) / np.abs(out["1"]).max(axis=1)
    say(f"[gpu] fast attention, {n} rows at {past}, growth {growth}, bf16 {bf}: rel max {rel.max():.2e}")
    assert rel.max() > 0          # the fast form ran
    assert rel.max() <= (2.0**-6 if bf else 2.0**-8) * (2 if growth else 1)


@pytest.mark.parametrize("kv", ["f16", "bf16"])
@pytest.mark.parametrize("past,n", [(1, 64), (37, 65), (100, 200), (700, 129), (2900, 100)])
def test_flash_probabilities_are_normalised_then_rounded(monkeypatch, past, n, kv):
    """Every score zero (no Q weights), V one in the cache and zero in the new rows: a row of c positions is
    past * p with p the 16-bit rounding of fp32(1 / c), the sum of c ones taken in full.  The products are
    whole multiples of p below 2^12, exact in any order, and the output projection copies one attention value
    to each of the hidden dims 128 .. 255, beside ones in the dims before, so the values come out whole."""
    monkeypatch.setenv("Q3T_PF_EXACT", "0")
    cfg = qcfg.tiny(n_layers=1)
    w = Weights(cfg, "f16", seed=41)
    blk = "talker.blk.0."
    for name in ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_down"):
        w[blk + name + ".weight"][2][:] = 0
    w["talker.output_norm.weight"][2][:] = 1
    m = np.arange(128)
    wo = w[blk + "attn_output.weight"][2].reshape(cfg.hidden_size, cfg.n_head * cfg.head_dim)
    wo[128 + m, 4 * m + m % 4] = 1
    dev = Device(cfg)
    try:
        dev.upload_weights(w)
        if kv == "bf16":
            dev.kv_set_type(BF16)
        dev.kv_reserve(past + n)
        shape = (past, cfg.n_kv_head, cfg.head_dim)
        one = np.uint16(0x3F80) if kv == "bf16" else np.float16(1)
        dev.kv_write(0, np.zeros(shape, type(one)), np.full(shape, one))
        rows = np.zeros((n, cfg.hidden_size), np.float32)
        rows[:, :128] = 1
        say(f"[gpu] uniform attention, {n} rows at {past}, cache {kv}")
        hid = dev.prefill(rows, past)[0]
    finally:
        dev.close()
    p = torch.from_numpy((1.0 / np.arange(past + 1, past + n + 1)).astype(np.float32))
    p = (p.bfloat16() if kv == "bf16" else p.half()).double().numpy()
    want = (past * p).astype(np.float16)
    got = (hid[:, 128:] / hid[:, :1]).astype(np.float16)
    wrong = int((got != want[:, None]).sum())
    assert wrong == 0, f"{wrong} of {got.size} values"


@pytest.mark.parametrize("which,value", [("k", np.inf), ("k", -np.inf), ("k", np.nan), ("v", np.inf), ("v", np.nan)])
def test_flash_attention_of_values_that_are_not_finite(monkeypatch, which, value):
    """One such value in the cached history of one layer: the rows that are not finite are the exact form's (an
    infinite key turns into a score of either sign, and a row of the one sign has no weight there), the others
    within the bound of the fp16 rows above."""
    cfg = qcfg.tiny(n_layers=1)
    past, n = 70, 130
    rng = np.random.default_rng(11)
    kv = rng.standard_normal((2, past, cfg.n_kv_head, cfg.head_dim)).astype(np.float16)
    kv["kv".index(which), 33, 0, 5] = value
    rows = (rng.standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
    dev = Device(cfg)
    try:
        dev.upload_weights(Weights(cfg, "f16", seed=47))
        dev.kv_reserve(past + n)
        dev.kv_write(0, kv[0], kv[1])
        out = {}
        for exact in ("1", "0"):
            monkeypatch.setenv("Q3T_PF_EXACT", exact)
            say(f"[gpu] {which} = {value} in the cache, exact {exact}")
            out[exact] = dev.prefill(rows, past)[0].astype(np.float64)
    finally:
        dev.close()
    finite = np.isfinite(out["1"]).all(axis=1)
    assert np.array_equal(np.isfinite(out["0"]).all(axis=1), finite)
    assert np.isnan(out["0"][~finite]).all() and (~finite).any()
    if which == "k" and not np.isnan(value):
        assert finite.any()
        rel = np.abs(out["0"] - out["1"])[finite].max(axis=1) / np.abs(out["1"][finite]).max(axis=1)
        assert 0 < rel.max() <= 2.0**-8, rel.max()


@pytest.mark.parametrize("n", [65, 1100])
def test_fast_form_of_one_head(monkeypatch, n):
    """One head: the output projection's K of 128 is half of the four stages that the small tiles hold
    otherwise (32 x 32 tiles at 65 rows, 64 x 64 at 1,100); the bound of the fp16 rows above, and the fast
    form ran."""
    cfg = qcfg.tiny(hidden=512, n_head=1, n_kv_head=1)
    dev = Device(cfg)
    try:
        dev.upload_weights(Weights(cfg, "f16", seed=43))
        dev.kv_reserve(n)
        rows = (np.random.default_rng(n).standard_normal((n, cfg.hidden_size)) * 0.05).astype(np.float32)
        out = {}
        for exact in ("1", "0"):
            monkeypatch.setenv("Q3T_PF_EXACT", exact)
            say(f"[gpu] one head, {n} rows, exact {exact}")
            out[exact] = dev.prefill(rows, 0)[0].astype(np.float64)
    finally:
        dev.close()
    rel = np.abs(out["0"] - out["1"]).max(axis=1) / np.abs(out["1"]).max(axis=1)
    assert 0 < rel.max() <= 2.0**-8, rel.max()


@pytest.mark.parametrize("n", [40, 65, 200, 600, 2049])
@pytest.mark.parametrize("hidden,ffn", [(256, 512), (1024, 3072)])
def test_fast_gemm_tiles_against_exact(monkeypatch, hidden, ffn, n):
    """The fast GEMM's tiles and stage counts: the shortest K (four stages, all in flight at once), rows
    below and past a tile, few and many workgroups.  Every input is rounded to 11 bits and summed in fp32, in the same order
    whatever the tile: the bound of the fp16 rows above."""
    cfg = qcfg.tiny(hidden=hidden, ffn=ffn, n_layers=1)
    monkeypatch.setenv("Q3T_PREFILL_MFMA", "1")
    dev = Device(cfg)
    try:
        dev.upload_weights(Weights(cfg, "f16", seed=37))
        dev.kv_reserve(n)
        rows = (np.random.default_rng(n).standard_normal((n, hidden)) * 0.05).astype(np.float32)
        out = {}
        for exact in ("1", "0"):
            monkeypatch.setenv("Q3T_PF_EXACT", exact)
            out[exact] = dev.prefill(rows, 0)[0].astype(np.float64)
    finally:
        dev.close()
    rel = np.abs(out["0"] - out["1"]).max(axis=1) / np.abs(out["1"]).max(axis=1)
    say(f"[gpu] fast GEMM tiles, {n} rows of {hidden}, {ffn}: rel max {rel.max():.2e}")
    assert 0 < rel.max() <= 2.0**-8
