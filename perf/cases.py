"""Performance cases of the SwiftKV decode-attention stage, through its Python entry points.

Three kinds of work, as a decoder around the stage issues it:

  decode   one decode step of `layers` layers: per layer one call of swiftkv_attention (FP32 or
           Q15.17 inputs) or swiftkv_attention_partials (the split-K partial sums of the Q/K/V
           projection), every sequence at one position or at positions of its own;
  prefill  a prompt of `position` tokens appended layer by layer (swiftkv_append_tokens), and the
           first decode step over it, whose outputs depend on every appended row;
  exact    the integer-compatibility step (swiftkv_attention_exact), whose results equal the
           reference's bit for bit; split-K partials go through convert_partials_q17 first, as
           that entry takes Q15.17 words.

A step may be repeated on the same state: it writes the same row at the same position again.  The
appended row stays in the cache, where the same call attends to it, so the attention outputs (and
the A14 words and E8M0 codes the O projection reads) show it.
"""
import importlib
import random

import numpy as np
import torch

MODEL, HEADS, DIM, GROUP = 4096, 32, 128, 32
TOKEN_BYTES = HEADS * 288          # INT8 codes and FP32 group scales of one token, all heads
REFERENCE_POSITIONS = 4096
MAX_POSITIONS = 32768

_kept = {}


def _package():
    return importlib.import_module("4pe_u250_amd")


def _context():
    """The one context (stream, workspace) that a program keeps for its GPU."""
    if "ctx" not in _kept:
        _kept["ctx"] = _package().Context(0)
    return _kept["ctx"]


def _rope_lut(positions):
    """The RoPE table: the reference's 4096 positions, or the extended one."""
    n = REFERENCE_POSITIONS if positions <= REFERENCE_POSITIONS else MAX_POSITIONS
    if n not in _kept:
        _kept[n] = _package().RopeLut.generate(_context(), n)
    return _kept[n]


def _case(kind, batch, position, layers, name=None, ragged=False, inputs="f32", dist="normal", outliers=False,
          a14=False):
    c = {"kind": kind, "batch": batch, "position": position, "layers": layers, "ragged": ragged, "inputs": inputs,
         "dist": dist, "outliers": outliers, "a14": a14}
    return dict(c, name=name) if name else c


def listed():
    return [
        # The first tokens of a conversation: the smallest calls, where the launch and the host count.
        _case("decode", 1, 127, 32, "decode_b1_p127"),
        # One user at the reference's last position, heavy-tailed K channels: latency of the whole stack.
        _case("decode", 1, 4095, 32, "decode_b1_p4095", outliers=True, a14=True),
        # A few users mid-conversation, Q15.17 words from an integer pipeline.
        _case("decode", 3, 1777, 32, "decode_b3_p1777_q17", inputs="q17", a14=True),
        # A small serving batch at full context.
        _case("decode", 8, 4095, 8, "decode_b8_p4095"),
        # The throughput workload: batch 64 at full context (4 of its 32 layers).
        _case("decode", 64, 4095, 4, "decode_b64_p4095", a14=True),
        # Continuous batching: sequences of 256 to 4096 tokens, fed by the projection's split-K partials.
        _case("decode", 64, 4095, 4, "decode_b64_ragged_parts4", ragged=True, inputs="parts4"),
        # Long contexts, past the reference's bound, heavy-tailed values.
        _case("decode", 16, 32511, 1, "decode_b16_p32511_t3", dist="t3"),
        # A full-length prompt and its first token.
        _case("prefill", 1, 4095, 16, "prefill_n4095"),
        # A short prompt of odd length, Q15.17 words.
        _case("prefill", 1, 333, 32, "prefill_n333_q17", inputs="q17", a14=True),
        # Bit-exact decoding of one sequence (comparing a deployment with the reference).
        _case("exact", 1, 4095, 8, "exact_b1_p4095", outliers=True, a14=True),
        # Bit-exact decoding of a few sequences from the projection's partials.
        _case("exact", 5, 1501, 8, "exact_b5_p1501_parts4", inputs="parts4", a14=True),
        # A bit-exact serving batch.
        _case("exact", 64, 4095, 1, "exact_b64_p4095", a14=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(lo * (hi / lo) ** rng.random() + rng.random()))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "exact", "exact"])
    if kind == "prefill":
        batch, position = 1, _log_int(rng, 64, 4095)
        budget = 16 * 4095
    else:
        batch = _log_int(rng, 1, 64)
        # token-layers: those of the largest listed case of the kind, less for decoding, whose small batches
        # read at a lower rate
        budget = (3 if kind == "decode" else 1) * 64 * 4096
        top = 4095 if kind == "exact" or batch > 16 else 32511
        position = _log_int(rng, 127, min(top, budget // batch - 1))
    most = 8 if kind == "exact" else 32
    layers = max(1, min(most, budget // (batch * (position + 1)))) if rng.random() < 0.8 else 1
    ragged = kind != "prefill" and batch > 1 and rng.random() < 0.4
    if kind == "prefill":
        inputs = rng.choice(["f32", "f32", "q17"])
    else:
        inputs = rng.choice(["f32", "f32", "q17", "parts2", "parts4"])
    return _case(kind, batch, position, layers, ragged=ragged, inputs=inputs, dist=rng.choice(["normal", "normal", "t3"]),
                 outliers=rng.random() < 0.3, a14=rng.random() < 0.5)


def _positions(case):
    """Cached tokens of each sequence before the step: one position, or lengths from a sixteenth of it up."""
    if not case["ragged"]:
        return [case["position"]] * case["batch"]
    r = random.Random(case["batch"] * 65537 + case["position"])
    lo = (case["position"] + 1) // 16
    return [case["position"]] + [r.randint(max(1, lo), case["position"]) for _ in range(case["batch"] - 1)]


def _values(gen, shape, dist):
    x = torch.randn(shape, generator=gen, device="cuda")
    if dist == "t3":     # Student-t(3) of unit variance
        chi = sum(torch.randn(shape, generator=gen, device="cuda").square_() for _ in range(3))
        x = x / (chi / 3.0).sqrt_() / 3.0 ** 0.5
    return x


def _generator(seed, *what):
    key = seed
    for w in what:
        key = (key * 1000003 + w + 1) % (1 << 62)
    return torch.Generator("cuda").manual_seed(key)


def _outlier_channels(seed):
    return torch.from_numpy(np.random.RandomState(seed % (1 << 31)).choice(MODEL, MODEL // 100, replace=False)).cuda()


def _history(case, seed, layer, seq, n):
    """FP32 k and v rows [n][4096] that fill tokens [0, n) of a sequence's layer."""
    gen = _generator(seed, 1, layer, seq)
    k, v = _values(gen, (n, MODEL), case["dist"]), _values(gen, (n, MODEL), case["dist"])
    if case["outliers"]:
        k[:, _outlier_channels(seed)] *= 20.0
    return k, v


def _to_q17(x):
    """Q15.17 words of FP32 values: half-even, saturated."""
    return (x.double() * 131072.0).round_().clamp_(-2.0 ** 31, 2.0 ** 31 - 1).to(torch.int32)


def _step_inputs(case, seed):
    """q, k, v of the step: [layers][batch][4096], or split-K partials [layers][parts][batch][4096]."""
    shape = (case["layers"], case["batch"], MODEL)
    got = []
    for i in range(3):
        gen = _generator(seed, 2, i)
        if case["inputs"].startswith("parts"):
            parts = int(case["inputs"][5:])
            x = torch.randn((shape[0], parts) + shape[1:], generator=gen, device="cuda") / parts ** 0.5
        else:
            x = _values(gen, shape, case["dist"])
        if i == 1 and case["outliers"]:
            x[..., _outlier_channels(seed)] *= 20.0
        got.append(_to_q17(x) if case["inputs"] == "q17" else x)
    return got


def prepare(case, seed):
    skv, ctx = _package(), _context()
    positions = _positions(case)
    batch, layers, top = case["batch"], case["layers"], max(positions)
    lut = _rope_lut(top + 1)
    kv = skv.KVCache(ctx, layers=layers, max_batch=batch, max_seq_len=top + 1)
    st = {"case": case, "kv": kv, "lut": lut, "positions": positions if batch > 1 else positions[0]}
    prompts = []
    for layer in range(layers):
        for seq in range(batch):
            n = positions[seq]
            k, v = _history(case, seed, layer, seq, n)
            if case["kind"] == "prefill":
                prompts.append((_to_q17(k), _to_q17(v)) if case["inputs"] == "q17" else (k, v))
                continue
            torch.cuda.synchronize()
            skv.swiftkv_append_tokens(ctx, k.data_ptr(), v.data_ptr(), kv, lut, layer, seq, 0, n)
            ctx.synchronize()
    st["prompts"] = prompts
    st["inputs"] = _step_inputs(case, seed)
    kind = torch.int32 if case["kind"] == "exact" else torch.float32
    st["out"] = torch.zeros((layers, batch, MODEL), dtype=kind, device="cuda")
    if case["inputs"].startswith("parts") and case["kind"] == "exact":
        st["words"] = [torch.zeros((batch, MODEL), dtype=torch.int32, device="cuda") for _ in range(3)]
    if case["a14"]:
        st["a14"] = torch.zeros((layers, batch, MODEL // GROUP, 56), dtype=torch.uint8, device="cuda")
        st["e8m0"] = torch.zeros((layers, batch, MODEL // GROUP), dtype=torch.uint8, device="cuda")
    q, k, v = st["inputs"]
    a14, e8m0 = st.get("a14"), st.get("e8m0")
    # The device addresses of each layer's tensors, as a program that owns its buffers holds them.
    st["args"] = [(q[i].data_ptr(), k[i].data_ptr(), v[i].data_ptr(), a14[i].data_ptr() if case["a14"] else None,
                   e8m0[i].data_ptr() if case["a14"] else None, st["out"][i].data_ptr()) for i in range(layers)]
    st["prompt_args"] = [(pk.data_ptr(), pv.data_ptr()) for pk, pv in prompts]
    st["word_args"] = [w.data_ptr() for w in st.get("words", ())]
    torch.cuda.synchronize()
    return st


class _Raw:
    """A device address with the interface of the package's buffers."""

    def __init__(self, ptr):
        self.ptr = ptr


def run(st):
    skv, ctx, case = _package(), _context(), st["case"]
    kv, lut, pos, kind, batch = st["kv"], st["lut"], st["positions"], case["kind"], case["batch"]
    q17 = case["inputs"] == "q17"
    parts = int(case["inputs"][5:]) if case["inputs"].startswith("parts") else 1
    for layer, (q, k, v, a14, e8m0, out) in enumerate(st["args"]):
        if kind == "prefill":
            pk, pv = st["prompt_args"][layer]
            skv.swiftkv_append_tokens(ctx, pk, pv, kv, lut, layer, 0, 0, case["position"], q17=q17)
        if kind == "exact":
            if parts > 1:
                for src, dst in zip((q, k, v), st["word_args"]):
                    ctx.convert_partials_q17(_Raw(src), _Raw(dst), batch * MODEL, parts)
                q, k, v = st["word_args"]
            skv.swiftkv_attention_exact(ctx, q, k, v, kv, lut, a14, e8m0, layer, pos, out, q17=parts > 1 or q17)
        elif parts > 1:
            skv.swiftkv_attention_partials(ctx, q, k, v, parts, kv, lut, a14, e8m0, layer, pos, out)
        else:
            skv.swiftkv_attention(ctx, q, k, v, kv, lut, a14, e8m0, layer, pos, out, q17=q17)
    return {"out": st["out"], "a14": st["a14"], "e8m0": st["e8m0"]} if case["a14"] else {"out": st["out"]}


def work(case):
    positions, layers, batch = _positions(case), case["layers"], case["batch"]
    parts = int(case["inputs"][5:]) if case["inputs"].startswith("parts") else 1
    tokens = sum(positions)
    step = tokens * TOKEN_BYTES + batch * (TOKEN_BYTES + 3 * parts * MODEL * 4 + MODEL * 4 + 512)
    if case["a14"]:
        step += batch * (MODEL // GROUP) * 57
    flops = (tokens + batch) * HEADS * 4 * DIM
    if case["kind"] == "prefill":
        step += tokens * (2 * MODEL * 4 + TOKEN_BYTES + 512)
    return {"bytes": layers * step, "flops": layers * flops}


def tolerance(case):
    # The integer step is defined bit for bit.  The FP32 step sums up to 32768 FP32 products per output in an
    # order of its own; a 14-bit word turns where that moves a value over a rounding boundary.
    if case["kind"] == "exact":
        return "exact"
    # Over the listed cases the split sizes and launch shapes differ among themselves by up to rel 1.2e-6, max
    # 6.5e-6 and 3.5e-4 of the packed bytes; four times that.
    return {"rel": 5e-6, "max": 2.6e-5, "differ": 0.0014}


# ---------------------------------------------------------------- the same in 64 bits, in plain torch


def _rope_values(pos0, n):
    """Q1.17 (cos, sin) of positions [pos0, pos0 + n): RNE(2^17 cos|sin(p theta^(-j/64))), theta = 10000."""
    freq = 1.0 / np.power(10000.0, np.arange(DIM // 2) / (DIM // 2))
    ang = np.arange(pos0, pos0 + n, dtype=np.float64)[:, None] * freq
    cs = np.stack([np.cos(ang), np.sin(ang)])
    return torch.from_numpy(np.clip(np.rint(cs * 131072.0), -262144, 262143).astype(np.int64)).cuda()


def _rotate(x, cs):
    """Rotation of adjacent channel pairs, x [n][4096] int64: floor shift, saturated."""
    a, b = x.view(-1, HEADS, DIM // 2, 2).unbind(-1)
    c, s = cs[0][:, None], cs[1][:, None]
    both = torch.stack([(a * c - b * s) >> 17, (a * s + b * c) >> 17], -1)
    return both.clamp_(-2 ** 31, 2 ** 31 - 1).view(-1, HEADS, DIM)


def _dequantized(x):
    """INT8 codes times their power-of-two scale per 32 channels, x [n][32][128] int64, as float64."""
    g = x.view(x.shape[0], HEADS, DIM // GROUP, GROUP)
    mag = g.abs()
    msb = torch.frexp(mag.amax(-1, keepdim=True).double()).exponent.to(torch.int64) - 1
    s = (msb - 6).clamp_(min=0)
    rnd = torch.where(s > 0, torch.ones_like(s) << (s - 1).clamp(min=0), torch.zeros_like(s))
    code = ((mag + rnd) >> s).clamp_(max=127) * g.sign()
    return torch.ldexp(code.double(), s - 17).view(x.shape)


def _reduced(x, case):
    """Q15.17 words (int64) of a step's inputs of one layer, [batch][4096]."""
    if case["inputs"] == "q17":
        return x.to(torch.int64)
    if case["inputs"] == "parts2":
        x = x[0] + x[1]
    elif case["inputs"] == "parts4":
        x = (x[0] + x[1]) + (x[2] + x[3])
    return _to_q17(x).to(torch.int64)


def exact(case, seed):
    if case["kind"] == "exact":
        return None     # whole numbers, the same in every implementation
    positions, inputs = _positions(case), _step_inputs(case, seed)
    out = torch.zeros((case["layers"], case["batch"], MODEL), dtype=torch.float64, device="cuda")
    cs = _rope_values(0, max(positions) + 1)
    for layer in range(case["layers"]):
        q, k, v = (_reduced(x[layer], case) for x in inputs)
        for seq, n in enumerate(positions):
            at = cs[:, n:n + 1]
            kh, vh = _history(case, seed, layer, seq, n)
            scores, values, chunk = [], [], 4096
            query = _rotate(q[seq:seq + 1], at)[0].double() / 131072.0
            for t in range(0, n, chunk):
                m = min(n, t + chunk)
                kd = _dequantized(_rotate(_to_q17(kh[t:m]).to(torch.int64), cs[:, t:m]))
                scores.append(torch.matmul(kd.transpose(0, 1).contiguous(), query[:, :, None])[:, :, 0])
                values.append(_dequantized(_to_q17(vh[t:m]).to(torch.int64).view(-1, HEADS, DIM)).float())
            kd = _dequantized(_rotate(k[seq:seq + 1], at))
            scores.append(torch.matmul(kd.transpose(0, 1).contiguous(), query[:, :, None])[:, :, 0])
            values.append(_dequantized(v[seq:seq + 1].view(1, HEADS, DIM)).float())     # 8 bits and a power of two
            weights = torch.softmax(torch.cat(scores, 1) / DIM ** 0.5, 1)
            t = 0
            for x in values:
                w = weights[:, t:t + x.shape[0]].contiguous()
                out[layer, seq] += torch.matmul(w[:, None], x.double().transpose(0, 1).contiguous())[:, 0].reshape(-1)
                t += x.shape[0]
    return {"out": out, "a14": None, "e8m0": None} if case["a14"] else {"out": out}
