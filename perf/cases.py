"""Performance cases of the framework: what a user of it runs, through its public entry points.

Every case is one call, or the few calls that belong together, on a device context that holds its weights
already: the text projection of a prompt, one talker step, the code predictor, a prompt prefill, a whole
generate(), several utterances decoded together, and the vocoder's streaming window and whole decode.  Shapes
are the package's own layouts (config.full_06b, config.full_17b, vocoder.full); weights are synthetic in the
package's tensor list (N(0, 0.02), norm gains around 1) and the same for every seed, as a program keeps one
model; the inputs (token ids, rows, speaker, codes, sampling seeds) come from the seed.
"""
import functools
import os
import sys
import zlib

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3-tts.cpp_amd"))

from qwen3_tts_amd import config, driver, synth, vocoder  # noqa: E402
from qwen3_tts_amd.device import Device  # noqa: E402

NO_EOS = -1e4          # EOS biased off, as bench.py does: every frame does its full work
BF16 = 30              # ggml's type id, as Device.kv_set_type takes it


def listed():
    return [
        # a sentence handed over in pieces: a few ids through the two-matrix text MLP, a latency-bound call
        {"name": "proj_9_q8", "kind": "proj", "model": "0.6b", "wtype": "q8_0", "n": 9},
        # a long text in one call (an audiobook chapter's prompt), an odd count
        {"name": "proj_1501_f16", "kind": "proj", "model": "0.6b", "wtype": "f16", "n": 1501},
        # one decode step for a program that drives the frame loop itself, mid-utterance
        {"name": "step_q8_kv512", "kind": "step", "model": "0.6b", "wtype": "q8_0", "kv": "f16", "past": 512},
        # the same far into a long utterance with unquantised weights and a bfloat16 cache
        {"name": "step_f16_kv3001_bf16", "kind": "step", "model": "0.6b", "wtype": "f16", "kv": "bf16", "past": 3001},
        # the prompt of a voice clone: 200 reference frames and the layout rows around them
        {"name": "prefill_q8_209", "kind": "prefill", "model": "0.6b", "wtype": "q8_0", "n": 209, "past": 0},
        # a long cloned history resumed in one call, quantised weights
        {"name": "prefill_q8_1600", "kind": "prefill", "model": "0.6b", "wtype": "q8_0", "n": 1600, "past": 0},
        # the long-context prompt of the package's configuration tests, F16 weights, one row past full tiles
        {"name": "prefill_f16_2049", "kind": "prefill", "model": "0.6b", "wtype": "f16", "n": 2049, "past": 0},
        # the whole thing for one utterance: prompt rows, prefill and the frame loop (two seconds of speech)
        {"name": "generate_q8", "kind": "generate", "model": "0.6b", "wtype": "q8_0", "ids": 64, "frames": 24,
         "temperature": 0.9},
        # the same with the larger layout, greedy
        {"name": "generate_q8_17b", "kind": "generate", "model": "1.7b", "wtype": "q8_0", "ids": 33, "frames": 16,
         "temperature": 0.0},
        # a server: 16 utterances with caches of 128 to 2,048 positions, a short prompt each, decoded together
        {"name": "streams_16_q8", "kind": "streams", "model": "0.6b", "wtype": "q8_0", "streams": 16, "rows": 10,
         "frames": 12, "past_lo": 128, "past_hi": 2048},
        # the streaming vocoder's steady state: 25 new frames behind 48 of context, codes on the device
        {"name": "voc_window_25_48", "kind": "window", "new": 25, "context": 48, "start": 100},
        # an utterance of 20 seconds decoded whole, codes from the host
        {"name": "voc_decode_241", "kind": "decode", "n": 241},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["proj", "step", "predict", "prefill", "prefill", "generate", "streams", "window", "decode"])
    wtype = rng.choice(["q8_0", "f16"])
    if kind == "proj":
        return {"kind": kind, "model": "0.6b", "wtype": wtype, "n": _log(rng, 3, 1500)}
    if kind == "step":
        return {"kind": kind, "model": "0.6b", "wtype": wtype, "kv": rng.choice(["f16", "bf16"]),
                "past": _log(rng, 16, 3500)}
    if kind == "predict":
        return {"kind": kind, "model": rng.choice(["0.6b", "1.7b"]), "wtype": wtype}
    if kind == "prefill":
        return {"kind": kind, "model": "0.6b", "wtype": wtype, "n": _log(rng, 9, 2048),
                "past": rng.choice([0, 0, rng.randrange(1, 400)])}
    if kind == "generate":
        return {"kind": kind, "model": rng.choice(["0.6b", "0.6b", "1.7b"]), "wtype": wtype,
                "ids": _log(rng, 9, 400), "frames": rng.randrange(6, 25), "temperature": rng.choice([0.0, 0.9])}
    if kind == "streams":
        lo = _log(rng, 16, 600)
        return {"kind": kind, "model": "0.6b", "wtype": wtype, "streams": rng.randrange(2, 17),
                "rows": _log(rng, 9, 39), "frames": rng.randrange(4, 11), "past_lo": lo,
                "past_hi": lo + rng.randrange(100, 1400)}
    if kind == "window":
        return {"kind": kind, "new": _log(rng, 1, 60), "context": rng.choice([48, 48, rng.randrange(0, 48)]),
                "start": rng.randrange(0, 200)}
    return {"kind": kind, "n": _log(rng, 4, 241)}


# ---------------------------------------------------------------- weights and contexts
def _cfg(case):
    return config.full_17b() if case["model"] == "1.7b" else config.full_06b()


def _tensor(name, ttype, ne):
    """One synthetic tensor on the GPU: fp32 values [ne1][ne0] for F32 / F16 tensors (already rounded), or
    (int8 quants [ne1][ne0/32][32], fp16 scales [ne1][ne0/32]) for Q8_0."""
    g = torch.Generator(device="cuda").manual_seed(zlib.crc32(name.encode()))
    x = torch.randn(ne[1], ne[0], generator=g, device="cuda") * 0.02
    if ttype == synth.F32:
        return x + 1.0 if name.endswith("norm.weight") else x
    if ttype == synth.F16:
        return x.half()
    b = x.view(ne[1], ne[0] // 32, 32)
    d = b.abs().amax(-1) / 127.0
    return torch.round(b / d[..., None]).clamp(-127, 127).to(torch.int8), d.half()


def _raw(t):
    """The tensor in ggml's memory layout (Q8_0: 34-byte blocks)."""
    if isinstance(t, tuple):
        q, d = t
        blocks = torch.cat([d.contiguous().view(torch.uint8).view(*d.shape, 2), q.view(torch.uint8)], -1)
        return blocks.reshape(-1).cpu().numpy()
    return t.reshape(-1).cpu().numpy()


def _history(layer, n, dtype):
    """n cached K and V rows of one talker layer (N(0, 1), as normed keys and values are of that size)."""
    g = torch.Generator(device="cuda").manual_seed(1000 + layer)
    kv = torch.randn(2, 4096, 8, 128, generator=g, device="cuda")[:, :n]
    return kv.to(dtype)


def _bits(t):
    t = t.contiguous()
    return t.cpu().numpy() if t.dtype == torch.float16 else t.view(torch.int16).cpu().numpy().view(np.uint16)


def _past(case):
    """Each stream's cached positions, spread evenly over the case's range in a mixed order."""
    b = case["streams"]
    at = np.linspace(case["past_lo"], case["past_hi"], b).astype(int)
    return [int(at[(i * 7) % b]) if b % 7 else int(at[i]) for i in range(b)]


@functools.lru_cache(maxsize=1)
def _handle(key):
    """The context that a program keeps: weights uploaded, caches reserved and, where the case has one, the
    cached history written.  One at a time, so that cases do not share a card's memory."""
    case = dict(key)
    if case["kind"] in ("window", "decode"):
        cfg = vocoder.full()
        v = vocoder.VocDevice(cfg, vocoder.VocWeights(cfg, seed=7).tensors)
        v.reserve(case["new"] + case["context"] if case["kind"] == "window" else case["n"])
        return v
    cfg = _cfg(case)
    dev = Device(cfg, 0)
    for name, ttype, ne in synth.tensor_specs(cfg, case["wtype"]):
        dev.upload(name, ttype, ne, _raw(_tensor(name, ttype, ne)))
    if case["kind"] == "streams":
        past = _past(case)
        dev.streams_reserve(case["streams"], max(past) + case["rows"] + case["frames"] + 8)
        for layer in range(cfg.n_layers):
            k, v = _history(layer, max(past), torch.float16).cpu().numpy()
            for b, n in enumerate(past):
                dev.stream_kv_write(b, layer, k[:n], v[:n])
        return dev
    if case.get("kv") == "bf16":
        dev.kv_set_type(BF16)
    dev.kv_reserve(case.get("past", 0) + case.get("n", 1) + case.get("ids", 0) + case.get("frames", 0) + 32)
    if case.get("past"):
        for layer in range(cfg.n_layers):
            k, v = _history(layer, case["past"], torch.bfloat16 if case.get("kv") == "bf16" else torch.float16)
            dev.kv_write(layer, _bits(k), _bits(v))
    return dev


def prepare(case, seed):
    h = _handle(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind in ("window", "decode"):
        n = case["start"] + case["new"] if kind == "window" else case["n"]
        codes = rng.integers(0, 2048, (n, 16)).astype(np.int32)
        if kind == "window":        # the frame loop's code rows, already on the device
            codes = torch.from_numpy(codes).cuda()
            torch.cuda.synchronize()
        return {"case": case, "h": h, "codes": codes}
    cfg = _cfg(case)
    d = cfg.hidden_size
    s = {"case": case, "h": h, "cfg": cfg}
    if kind == "proj":
        s["ids"] = rng.integers(0, cfg.text_vocab, case["n"]).astype(np.int32)
    elif kind == "step":
        s["x"] = (rng.standard_normal(d) * 0.05).astype(np.float32)
    elif kind == "predict":
        s["hidden"] = rng.standard_normal(d).astype(np.float32)
        s["prev"] = rng.integers(0, cfg.cp_vocab, 15).astype(np.int32)
        s["cb0"] = int(rng.integers(0, 2048))
    elif kind == "prefill":
        s["rows"] = (rng.standard_normal((case["n"], d)) * 0.05).astype(np.float32)
    elif kind == "generate":
        s["ids"] = rng.integers(0, 151643, case["ids"]).astype(np.int32)
        s["speaker"] = rng.standard_normal(d).astype(np.float32)
        s["seed"] = int(seed) & 0xFFFFFFFF
    else:
        s["rows"], s["args"] = [], []
        for b, n in enumerate(_past(case)):
            s["rows"].append((rng.standard_normal((case["rows"], d)) * 0.05).astype(np.float32))
            s["args"].append(dict(trailing=(rng.standard_normal((4, d)) * 0.05).astype(np.float32),
                                  tts_pad=(rng.standard_normal(d) * 0.05).astype(np.float32),
                                  n_past=n + case["rows"], max_len=case["frames"], eos_bias=NO_EOS,
                                  temperature=0.9 if b % 2 else 0.0, top_k=50 if b % 2 else 0, seed=int(seed) + b))
        s["past"] = _past(case)
    return s


def run(s):
    case, h = s["case"], s["h"]
    kind = case["kind"]
    if kind == "proj":
        return h.text_proj(s["ids"])
    if kind == "step":
        logits, hidden = h.talker_step(s["x"], case["past"])
        return {"logits": logits, "hidden": hidden}
    if kind == "predict":           # one frame's 15 codes, and the single-pass form beside it
        codes, logits = h.code_pred(s["hidden"], s["cb0"])
        return {"single": h.predict_codes(s["hidden"], s["prev"]), "codes": codes, "logits": logits}
    if kind == "prefill":
        hidden, logits = h.prefill(s["rows"], case["past"])
        return {"hidden": hidden, "logits": logits}
    if kind == "generate":
        rows, trailing, pad = driver.build_prefill(h, s["cfg"], s["ids"], s["speaker"])
        _, logits = h.prefill(rows, 0, want_hidden=False)
        t = case["temperature"]
        h.frames_begin(trailing, pad, rows.shape[0], case["frames"], temperature=t, top_k=50 if t > 0 else 0,
                       eos_bias=NO_EOS, seed=s["seed"])
        codes = [h.frames_run(min(8, case["frames"] - i))[0] for i in range(0, case["frames"], 8)]
        return {"prompt": rows, "trailing": trailing, "logits": logits, "codes": np.concatenate(codes)}
    if kind == "streams":
        for b, rows in enumerate(s["rows"]):
            h.stream_prefill(b, rows, s["past"][b])
        h.streams_begin(s["args"])
        codes, _ = h.streams_run(case["frames"])
        return {"codes": np.stack(codes), "logits": np.stack([h.stream_logits(b) for b in range(case["streams"])])}
    if kind == "window":
        n = case["start"] + case["new"]
        return h.decode_window(None, case["start"], n, case["context"], n_frames=n, device_ptr=s["codes"].data_ptr())
    return h.decode(s["codes"])


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(cfg, wtype, prefix):
    per = {synth.F32: 4.0, synth.F16: 2.0, synth.Q8_0: 34 / 32}
    return sum(per[t] * ne[0] * ne[1] for name, t, ne in synth.tensor_specs(cfg, wtype) if name.startswith(prefix))


def _layer_params(cfg, d, ffn):
    qd, kd = cfg.n_head * cfg.head_dim, cfg.n_kv_head * cfg.head_dim
    return d * (qd + 2 * kd) + qd * d + 3 * d * ffn


def _rows_work(cfg, wtype, n, past):
    """n talker rows after `past` cached positions, one row's head."""
    kv_row = 2 * cfg.n_kv_head * cfg.head_dim * 2 * cfg.n_layers
    pairs = n * past + n * (n + 1) / 2
    b = _weight_bytes(cfg, wtype, "talker.blk.") + 2 * cfg.codec_vocab * cfg.hidden_size + kv_row * (past + n)
    b += 2 * 4 * n * cfg.hidden_size
    f = 2.0 * n * cfg.n_layers * _layer_params(cfg, cfg.hidden_size, cfg.ffn_size)
    f += 4.0 * cfg.n_layers * cfg.n_head * cfg.head_dim * pairs + 2.0 * cfg.codec_vocab * cfg.hidden_size
    return b, f


def _frame_work(cfg, wtype, lengths):
    """One frame of len(lengths) utterances: a talker step each and 15 passes of the code predictor."""
    n = len(lengths)
    cp = _weight_bytes(cfg, wtype, "code_pred.blk.") + _weight_bytes(cfg, wtype, "code_pred.mtp_proj")
    b = 15 * cp + _weight_bytes(cfg, wtype, "code_pred.lm_head.")
    f = 2.0 * n * (16 * cfg.cp_layers * _layer_params(cfg, cfg.cp_hidden, cfg.cp_ffn)
                   + 15 * cfg.cp_vocab * cfg.cp_hidden)
    b += _weight_bytes(cfg, wtype, "talker.blk.") + 2 * cfg.codec_vocab * cfg.hidden_size
    for n_kv in lengths:
        tb, tf = _rows_work(cfg, wtype, 1, n_kv)
        b += 2 * cfg.n_kv_head * cfg.head_dim * 2 * cfg.n_layers * (n_kv + 1)
        f += tf
    return b, f


def _proj_work(cfg, wtype, n):
    te, d = cfg.text_embd_dim, cfg.hidden_size
    return _weight_bytes(cfg, wtype, "talker.text_proj") + 2 * n * te + 4 * n * d, 2.0 * n * te * (te + d)


def _voc_work(n, new):
    c = vocoder.full()
    params = sum(np.prod(ne) * (2 if t == synth.F16 else 4) for name, t, ne, *_ in vocoder.tensor_specs(c)
                 if "codebook" not in name and "usage" not in name)
    f = 2.0 * n * 16 * c.codebook_dim * c.hidden
    f += 2.0 * n * (3 * c.hidden * c.latent + 2 * c.latent * c.hidden)
    f += 2.0 * n * c.n_layers * (4 * c.hidden * c.latent + 3 * c.hidden * c.ffn)
    rows = n
    for _ in range(2):
        f += 2.0 * rows * 2 * c.latent * c.latent
        rows *= 2
        f += 2.0 * rows * (7 * c.latent + 2 * c.latent * c.cnx_ffn)
    f += 2.0 * rows * 7 * c.latent * c.decoder_dim
    ch = c.decoder_dim
    for s, k in zip(c.rates, c.dec_kernel):
        co = ch // 2
        f += 2.0 * rows * k * ch * co
        rows = (rows - 1) * s
        f += 2.0 * rows * 3 * 8 * co * co
        ch = co
    f += 2.0 * rows * 7 * ch
    return params + n * 16 * 4 + 4 * c.samples_for_frames(new), f


def work(case):
    kind = case["kind"]
    if kind == "window":
        b, f = _voc_work(min(case["context"], case["start"]) + case["new"], case["new"])
    elif kind == "decode":
        b, f = _voc_work(case["n"], case["n"])
    else:
        cfg, wtype = _cfg(case), case["wtype"]
        if kind == "proj":
            b, f = _proj_work(cfg, wtype, case["n"])
        elif kind == "step":
            b, f = _rows_work(cfg, wtype, 1, case["past"])
        elif kind == "prefill":
            b, f = _rows_work(cfg, wtype, case["n"], case["past"])
        elif kind == "predict":
            cp = _weight_bytes(cfg, wtype, "code_pred.blk.") + _weight_bytes(cfg, wtype, "code_pred.mtp_proj")
            b = 16 * cp + 2 * _weight_bytes(cfg, wtype, "code_pred.lm_head.")
            f = 2.0 * (17 * cfg.cp_layers * _layer_params(cfg, cfg.cp_hidden, cfg.cp_ffn)
                       + 30 * cfg.cp_vocab * cfg.cp_hidden)
        elif kind == "generate":
            b, f = _proj_work(cfg, wtype, case["ids"])
            n = 10
            for add in [_rows_work(cfg, wtype, n, 0)] + [_frame_work(cfg, wtype, [n + i])
                                                         for i in range(case["frames"])]:
                b, f = b + add[0], f + add[1]
        else:
            b = f = 0.0
            for n in _past(case):
                add = _rows_work(cfg, wtype, case["rows"], n)
                b, f = b + add[0], f + add[1]
            for i in range(case["frames"]):
                add = _frame_work(cfg, wtype, [n + case["rows"] + i for n in _past(case)])
                b, f = b + add[0], f + add[1]
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("generate", "streams", "predict"):
        # codes are whole numbers, the decode's sums are exact in 64 bits and rounded once, and a stream's codes
        # equal the utterance's own: the same codes and logits, whatever the order of a sum
        return "exact"
    if kind in ("window", "decode"):
        return {"rel": 2e-2}
    if kind == "proj":
        return {"rel": 1e-2 if case["wtype"] == "q8_0" else 1e-3}
    return {"rel": 5e-2 if case["wtype"] == "q8_0" else 5e-3}


# ---------------------------------------------------------------- the same in 64 bits, plain torch
class _W64:
    def __init__(self, cfg, wtype):
        self.specs = {name: (t, ne) for name, t, ne in synth.tensor_specs(cfg, wtype)}

    def __getitem__(self, name):
        ttype, ne = self.specs[name]
        t = _tensor(name, ttype, ne)
        if isinstance(t, tuple):
            return (t[0].double() * t[1].double()[..., None]).reshape(ne[1], ne[0])
        return t.double().reshape(-1) if ne[1] == 1 else t.double()


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, theta):
    half = x.shape[-1] // 2
    i = torch.arange(half, dtype=torch.float64, device="cuda")
    a = pos[:, None].double() * theta ** (-i / half)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def _causal(q, k, v, past):
    """q [n][heads][hd] over k, v [past + n][kv heads][hd]"""
    n, heads, hd = q.shape
    out = torch.empty_like(q)
    mask = torch.arange(k.shape[0], device="cuda")[None] > torch.arange(n, device="cuda")[:, None] + past
    for h in range(heads):
        g = h // (heads // k.shape[1])
        s = (q[:, h] @ k[:, g].T.contiguous() / hd ** 0.5).masked_fill(mask, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ v[:, g]
    return out


def _talker64(case, x):
    cfg, past = _cfg(case), case["past"]
    w = _W64(cfg, case["wtype"])
    n = x.shape[0]
    pos = torch.arange(past, past + n, device="cuda")
    for layer in range(cfg.n_layers):
        p = f"talker.blk.{layer}."
        h = _rms(x, w[p + "attn_norm.weight"], cfg.rms_eps)
        q, k, v = ((h @ w[p + f"attn_{c}.weight"].T).view(n, -1, cfg.head_dim) for c in "qkv")
        q = _rope(_rms(q, w[p + "attn_q_norm.weight"], cfg.rms_eps), pos, cfg.rope_theta)
        k = _rope(_rms(k, w[p + "attn_k_norm.weight"], cfg.rms_eps), pos, cfg.rope_theta)
        if past:
            hk, hv = _history(layer, past, torch.bfloat16 if case.get("kv") == "bf16" else torch.float16).double()
            k, v = torch.cat([hk, k]), torch.cat([hv, v])
        x = x + _causal(q, k, v, past).reshape(n, -1) @ w[p + "attn_output.weight"].T
        h = _rms(x, w[p + "ffn_norm.weight"], cfg.rms_eps)
        f = torch.nn.functional.silu(h @ w[p + "ffn_gate.weight"].T) * (h @ w[p + "ffn_up.weight"].T)
        x = x + f @ w[p + "ffn_down.weight"].T
    h = _rms(x, w["talker.output_norm.weight"], cfg.rms_eps)
    return h, (h[-1:] @ w["talker.codec_head.weight"].T)[0]


class _Voc64:
    def __init__(self):
        self.c = vocoder.full()
        self.w = vocoder.VocWeights(self.c, seed=7)

    def t(self, name):
        _, ne, a = self.w["tok_dec." + name]
        return torch.from_numpy(a).cuda().double().reshape(tuple(reversed(ne)))

    def linear(self, x, name, bias=None):
        w = self.t(name)
        y = x @ w.reshape(w.shape[0], -1).T
        return y if bias is None else y + self.t(bias)

    def conv(self, x, name, dil=1):
        w = self.t(name + ".weight")            # [out][in][taps], causal
        k = w.shape[-1]
        x = torch.cat([x.new_zeros((k - 1) * dil, x.shape[1]), x])
        n = x.shape[0] - (k - 1) * dil
        return sum(x[i * dil:i * dil + n] @ w[:, :, i].T for i in range(k)) + self.t(name + ".bias")

    def conv_t(self, x, name, stride, crop):
        w = self.t(name + ".weight")            # [in][out][taps]
        k, n = w.shape[-1], x.shape[0]
        y = x.new_zeros((n - 1) * stride + k, w.shape[1])
        for i in range(k):
            y[i:i + (n - 1) * stride + 1:stride] += x @ w[:, :, i]
        return y[crop:y.shape[0] - crop] + self.t(name + ".bias")

    def snake(self, x, a):
        return x + torch.sin(x * torch.exp(self.t(a + ".alpha"))) ** 2 * torch.exp(-self.t(a + ".beta"))

    def __call__(self, codes, pos0):
        c, F = self.c, torch.nn.functional
        x = 0
        for q in range(c.n_codebooks):
            p = "vq_first.0." if q == 0 else f"vq_rest.{q - 1}."
            rows = self.t(p + "codebook") / self.t(p + "usage").clamp(min=1e-5)[:, None]
            x = x + self.linear(rows[codes[:, q].long()], f"vq_{'first' if q == 0 else 'rest'}.output_proj.weight")
        x = self.conv(x, "pre_conv")
        x = self.linear(x, "pre_tfm.input_proj.weight", "pre_tfm.input_proj.bias")
        n, hd = x.shape[0], c.latent // c.n_heads
        pos = torch.arange(pos0, pos0 + n, device="cuda")
        for layer in range(c.n_layers):
            p = f"pre_tfm.blk.{layer}."
            h = _rms(x, self.t(p + "attn_norm.weight"), c.rms_eps)
            q, k, v = (self.linear(h, p + f"attn_{s}.weight").view(n, c.n_heads, hd) for s in "qkv")
            a = _causal(_rope(q, pos, c.rope_theta), _rope(k, pos, c.rope_theta), v, 0).reshape(n, -1)
            x = x + self.linear(a, p + "attn_output.weight") * self.t(p + "attn_scale")
            h = _rms(x, self.t(p + "ffn_norm.weight"), c.rms_eps)
            f = F.silu(self.linear(h, p + "ffn_gate.weight")) * self.linear(h, p + "ffn_up.weight")
            x = x + self.linear(f, p + "ffn_down.weight") * self.t(p + "ffn_scale")
        x = _rms(x, self.t("pre_tfm.norm.weight"), c.rms_eps)
        x = self.linear(x, "pre_tfm.output_proj.weight", "pre_tfm.output_proj.bias")
        for i in range(2):
            p = f"upsample.{i}."
            x = self.conv_t(x, p + "conv", 2, 0)
            w = self.t(p + "dwconv.weight")
            h = torch.cat([x.new_zeros(6, x.shape[1]), x])
            h = sum(h[j:j + x.shape[0]] * w[:, 0, j] for j in range(7)) + self.t(p + "dwconv.bias")
            h = F.layer_norm(h, (h.shape[-1],), self.t(p + "norm.weight"), self.t(p + "norm.bias"), eps=1e-6)
            h = F.gelu(self.linear(h, p + "pwconv1.weight", p + "pwconv1.bias"), approximate="tanh")
            x = x + self.linear(h, p + "pwconv2.weight", p + "pwconv2.bias") * self.t(p + "gamma")
        x = self.conv(x, "dec.0.conv")
        for b, (s, k) in enumerate(zip(c.rates, c.dec_kernel)):
            p = f"dec.{b + 1}."
            x = self.conv_t(self.snake(x, p + "snake"), p + "conv_t", s, k - s)
            for r, dil in ((2, 1), (3, 3), (4, 9)):
                q = p + f"res.{r}."
                h = self.conv(self.snake(x, q + "act1"), q + "conv1", dil)
                x = x + self.conv(self.snake(h, q + "act2"), q + "conv2")
        return torch.tanh(self.conv(self.snake(x, "dec.5.snake"), "dec.6.conv")[:, 0])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("generate", "streams", "predict"):
        return None        # chains of sampled tokens: each pass's input is the token before it
    s = prepare(case, seed)
    if kind == "window":
        first = max(0, case["start"] - case["context"])
        return _Voc64()(s["codes"][first:], first)[vocoder.full().samples_for_frames(case["start"] - first):]
    if kind == "decode":
        return _Voc64()(torch.from_numpy(s["codes"]).cuda(), 0)
    if kind == "proj":
        cfg = s["cfg"]
        w = _W64(cfg, case["wtype"])
        x = w["talker.text_embd.weight"][torch.from_numpy(s["ids"]).long().cuda()]
        x = x @ w["talker.text_proj.fc1.weight"].T + w["talker.text_proj.fc1.bias"]
        return torch.nn.functional.silu(x) @ w["talker.text_proj.fc2.weight"].T + w["talker.text_proj.fc2.bias"]
    x = torch.from_numpy(s["rows"] if kind == "prefill" else s["x"][None]).cuda().double()
    hidden, logits = _talker64(case, x)
    return {"logits": logits, "hidden": hidden if kind == "prefill" else hidden[0]}
