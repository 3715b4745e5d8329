"""The work that is measured: matrix products against GGUF block weights as an inference program issues them.

Four kinds of pass, all through the public entry points of `HipGpu`:

  mm       one projection, `HipGpu.mm`, issued eagerly: decode (m = 1), speculative verify (m = 2 .. 16), small batches
           and prefill chunks (m up to 2048), in the formats a GGUF file of a dense model holds
  decode   the projections of one decode step as one recorded chain: q/k/v, o, gate/up, down, head, one `mm_multi` call a
           stage (the repository's benchmark step)
  layer    one decode layer of a mixed-format file with its norms and the gated activation, as one recorded chain
  moe      router and expert feed-forward of one mixture layer, `HipGpu.moe_ffn_routed`, issued eagerly

Weights are random blocks of each format (uniform codes and sub-scales, normally distributed scales), activations and
router logits N(0, 1).  Everything is made on the GPU from the seed.
"""
import math

import torch

from __graft_entry__ import load_package

pkg = load_package()

FORMATS = {"q4_k": pkg.Q4_K, "q5_k": pkg.Q5_K, "q6_k": pkg.Q6_K, "q8_0": pkg.Q8_0, "iq4_xs": pkg.IQ4_XS}
ACT = {"auto": pkg.ACT_AUTO, "q8k": pkg.ACT_Q8K}
# no pass is larger than these: the longest prefill product listed, and the bytes of the largest output head
MOST_MACS = 4096 * 14336 * 2048
MOST_BYTES = 512_000_000

_gpu = None


def gpu():
    """The one device handle of the process, as an inference program holds it."""
    global _gpu
    if _gpu is None:
        _gpu = pkg.HipGpu(0)
    return _gpu


# ---- the cases -------------------------------------------------------------------------------------------------------

def _mm(name, fmt, n, k, m, x="f32", act="auto"):
    return {"name": name, "kind": "mm", "fmt": fmt, "n": n, "k": k, "m": m, "x": x, "act": act}


def listed():
    return [
        # one small projection of one token (k or v of grouped-query attention): launches and latency are what counts
        _mm("token_kv_q4k", "q4_k", 1024, 4096, 1),
        # one square projection of one token on a Q8_0 file, f32 activations
        _mm("token_square_q8_0", "q8_0", 4096, 4096, 1),
        # a whole decode step over a Q4_K file of an 8B-shaped model, the head included
        {"name": "decode_step_q4k", "kind": "decode", "hidden": 4096, "kv": 1024, "ff": 14336, "vocab": 128256},
        # a decode layer of a mixed file (v and down kept finer), odd feed-forward width, norms and activation included
        {"name": "decode_layer_mixed", "kind": "layer", "hidden": 4096, "kv": 1024, "ff": 11008, "v": "q6_k", "down": "q6_k"},
        # speculative verify of a handful of draft positions against the largest output head
        _mm("verify_head_q6k", "q6_k", 151936, 4096, 5, x="bf16"),
        # a small batch of concurrent requests against a 4-bit non-linear file
        _mm("batch_iq4xs", "iq4_xs", 14336, 4096, 24),
        # an ordinary prefill chunk, and the longest one on the other feed-forward shape
        _mm("prefill_gate_q4k", "q4_k", 14336, 4096, 512, x="bf16"),
        _mm("prefill_down_q4k", "q4_k", 4096, 14336, 2048, x="bf16"),
        # the last, ragged chunk of a prompt on a finer file: no size a multiple of a tile
        _mm("prefill_ragged_q6k", "q6_k", 6914, 2816, 333),
        # a short prefill chunk in the CPU path's arithmetic (int8 activations), the option for parity with it
        _mm("chunk_int8_q4k", "q4_k", 14336, 4096, 128, x="bf16", act="q8k"),
        # a mixture layer, 128 experts and top 8, for one token and for a prefill chunk
        {"name": "moe_token", "kind": "moe", "tokens": 1, "experts": 128, "ksel": 8, "d": 2048, "ff": 768, "down": "q4_k"},
        {"name": "moe_batch", "kind": "moe", "tokens": 256, "experts": 128, "ksel": 8, "d": 2048, "ff": 768, "down": "q4_k"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    return max(lo, min(hi, _log(rng, lo, hi) // step * step))


def draw(rng):
    kind = rng.choice(["mm", "mm", "mm", "mm", "decode", "layer", "moe", "moe"])
    if kind == "mm":
        fmt = rng.choice(["q4_k", "q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "q8_0", "iq4_xs"])
        k = _mult(rng, 1024, 14336, 256)
        n = rng.choice([_log(rng, 512, 32768), _mult(rng, 512, 32768, 64)])
        m = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 2048)])
        if m <= 16 and k <= 8192 and rng.random() < 0.15:      # an output head
            n = _log(rng, 32000, 152064)
        while n * k > 480_000_000:
            n //= 2
        m = max(1, min(m, MOST_MACS // (n * k)))
        act = "q8k" if fmt in ("q4_k", "q5_k", "q6_k") and rng.random() < 0.25 else "auto"
        return {"kind": "mm", "fmt": fmt, "n": n, "k": k, "m": m, "x": rng.choice(["f32", "bf16"]), "act": act}
    if kind in ("decode", "layer"):
        hidden = _mult(rng, 1024, 5120, 256)
        kv = max(256, hidden // rng.choice([1, 4, 8]) // 64 * 64)
        ff = int(hidden * rng.uniform(2.5, 3.75)) // 256 * 256
        if kind == "decode":
            return {"kind": "decode", "hidden": hidden, "kv": kv, "ff": ff, "vocab": _log(rng, 32000, 128256)}
        return {"kind": "layer", "hidden": hidden, "kv": kv, "ff": ff, "v": rng.choice(["q4_k", "q5_k", "q6_k"]),
                "down": rng.choice(["q4_k", "q5_k", "q6_k"])}
    return {"kind": "moe", "tokens": rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 512)]),
            "experts": rng.choice([32, 64, 96, 128]), "ksel": rng.choice([4, 6, 8]), "d": _mult(rng, 1024, 3072, 256),
            "ff": _mult(rng, 512, 1024, 256), "down": rng.choice(["q4_k", "q4_k", "q6_k"])}


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weights(g, fmt, n, k):
    """Random blocks of a format for an [n][k] matrix, as bytes on the GPU, with 16 spare bytes behind them."""
    block, per = pkg.runtime.BLOCK_SHAPE[FORMATS[fmt]]
    nb = n * (k // per)
    whole = torch.zeros(nb * block + 16, dtype=torch.uint8, device="cuda")
    raw = whole[:nb * block].view(nb, block)
    words = torch.randint(-2**63, 2**63 - 1, ((nb * block + 7) // 8,), generator=g, device="cuda", dtype=torch.int64)
    raw.copy_(words.view(torch.uint8)[:nb * block].view(nb, block))

    def put(at, values):
        raw[:, at:at + 2] = values.abs().to(torch.float16).view(torch.uint8).view(nb, 2)

    if fmt == "q8_0":
        put(0, _normal(g, nb, 1) * (0.02 / 127))
        codes = raw[:, 2:]
        codes[codes == 128] = 0                                # codes lie in [-127, 127]
    elif fmt in ("q4_k", "q5_k"):
        put(0, _normal(g, nb, 1) * 0.01)
        put(2, _normal(g, nb, 1) * 0.01)
    elif fmt == "q6_k":
        scales = raw[:, 192:208]
        scales.copy_(((scales & 63).to(torch.int8) - 32).view(torch.uint8))
        put(208, _normal(g, nb, 1) * 0.01)
    else:
        put(0, _normal(g, nb, 1) * (0.01 / 127))
    return whole


class _Held:
    """What a program keeps for a pass: device tensors, their handles in the library, the outputs."""

    def __init__(self):
        self.tensors, self.out = [], {}

    def buf(self, tensor):
        self.tensors.append(tensor)
        return gpu().wrap(tensor.data_ptr(), tensor.numel() * tensor.element_size())

    def lin(self, g, fmt, n, k):
        return gpu().lin_wrap(FORMATS[fmt], n, k, self.buf(_weights(g, fmt, n, k)))

    def new(self, *shape, dtype=torch.float32):
        return torch.zeros(*shape, dtype=dtype, device="cuda")

    def result(self, name, *shape, dtype=torch.float32):
        self.out[name] = self.new(*shape, dtype=dtype)
        return self.buf(self.out[name])


def _prepare_mm(case, g, s):
    n, k, m = case["n"], case["k"], case["m"]
    s.w = s.lin(g, case["fmt"], n, k)
    x = _normal(g, m, k)
    s.x = s.buf(x if case["x"] == "f32" else x.to(torch.bfloat16))
    s.y = s.result("y", m, n)


def _record(s, issue):
    """Run the launches once eagerly, then record them: what a program does for the step it replays per token."""
    torch.cuda.synchronize()
    issue()
    gpu().submit()
    gpu().capture_begin()
    issue()
    s.graph = gpu().capture_end()


def _prepare_decode(case, g, s):
    h, kv, ff, vocab = case["hidden"], case["kv"], case["ff"], case["vocab"]
    stages = [("attn", h, [("q", h), ("k", kv), ("v", kv)]), ("o", h, [("o", h)]), ("ffn", h, [("gate", ff), ("up", ff)]),
              ("down", ff, [("down", h)]), ("head", h, [("logits", vocab)])]
    calls = []
    for _, k, rows in stages:
        calls.append((s.buf(_normal(g, k)), [s.lin(g, "q4_k", n, k) for _, n in rows], [s.result(name, n) for name, n in rows]))

    def issue():
        for x, ws, ys in calls:
            gpu().mm_multi(x, ws, ys)
    _record(s, issue)
    s.calls = calls


def _prepare_layer(case, g, s):
    h, kv, ff = case["hidden"], case["kv"], case["ff"]
    x, attn, mid = s.buf(_normal(g, h)), s.buf(_normal(g, h)), s.buf(_normal(g, h))
    g1, g2 = s.buf(1 + 0.1 * _normal(g, h)), s.buf(1 + 0.1 * _normal(g, h))
    qkv = [s.lin(g, "q4_k", h, h), s.lin(g, "q4_k", kv, h), s.lin(g, case["v"], kv, h)]
    wo, wg, wu = s.lin(g, "q4_k", h, h), s.lin(g, "q4_k", ff, h), s.lin(g, "q4_k", ff, h)
    wd = s.lin(g, case["down"], h, ff)
    outs = [s.result(name, n) for name, n in (("q", h), ("k", kv), ("v", kv))]
    o, act, down = s.result("o", h), s.result("act", ff), s.result("down", h)
    xq, xs = s.buf(s.new(h, dtype=torch.int8)), s.buf(s.new(h // 256))

    def issue():
        d = gpu()
        d.rmsnorm_quant_q8k(x, g1, 1e-5, 1, h, xq, xs)
        d.mm_q8k_multi(xq, xs, qkv, outs)
        d.mm_multi(attn, [wo], [o])
        d.rmsnorm_quant_q8k(mid, g2, 1e-5, 1, h, xq, xs)
        d.ffn_gu_q8k(xq, xs, wg, wu, act)
        d.mm_multi(act, [wd], [down])
    _record(s, issue)
    s.calls = (x, attn, mid, g1, g2, qkv, wo, wg, wu, wd, outs, o, act, down, xq, xs)


def _prepare_moe(case, g, s):
    t, e, d, ff, ksel = case["tokens"], case["experts"], case["d"], case["ff"], case["ksel"]
    s.gate, s.up, s.down = s.lin(g, "q4_k", e * ff, d), s.lin(g, "q4_k", e * ff, d), s.lin(g, case["down"], e * d, ff)
    s.x, s.logits = s.buf(_normal(g, t, d)), s.buf(_normal(g, t, e))
    s.idx, s.wgt, s.y = s.result("idx", t, ksel, dtype=torch.int32), s.result("wgt", t, ksel), s.result("y", t, d)


def prepare(case, seed):
    s = _Held()
    s.case = dict(case)
    {"mm": _prepare_mm, "decode": _prepare_decode, "layer": _prepare_layer, "moe": _prepare_moe}[case["kind"]](case, _rng(seed), s)
    torch.cuda.synchronize()                                   # the library works on a stream of its own
    return s


def run(state):
    c, s = state.case, state
    if c["kind"] == "mm":
        gpu().mm(s.x, s.w, s.y, c["m"], x_dtype=pkg.X_BF16 if c["x"] == "bf16" else pkg.X_F32, act_mode=ACT[c["act"]])
    elif c["kind"] == "moe":
        gpu().moe_ffn_routed(s.x, c["tokens"], c["d"], c["ff"], c["experts"], c["ksel"], s.logits, s.idx, s.wgt, s.gate,
                             s.up, s.down, s.y)
    else:
        s.graph.launch()
    return s.out


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _matrix(fmt, n, k):
    return n * pkg.row_bytes(FORMATS[fmt], k)


def work(case):
    if case["kind"] == "mm":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": _matrix(case["fmt"], n, k) + m * (k * (2 if case["x"] == "bf16" else 4) + 4 * n), "flops": 2 * m * n * k}
    if case["kind"] == "moe":
        t, e, d, ff, ksel = case["tokens"], case["experts"], case["d"], case["ff"], case["ksel"]
        touched = e * (1 - (1 - ksel / e) ** t)                # experts that any token chose, on average
        per = 2 * _matrix("q4_k", ff, d) + _matrix(case["down"], d, ff)
        return {"bytes": int(touched * per) + t * (8 * d + 4 * e + 8 * ksel), "flops": 2 * t * ksel * 3 * d * ff}
    h, kv, ff = case["hidden"], case["kv"], case["ff"]
    decode = case["kind"] == "decode"
    mats = [("q4_k", h, h), ("q4_k", kv, h), ("q4_k" if decode else case["v"], kv, h), ("q4_k", h, h), ("q4_k", ff, h),
            ("q4_k", ff, h), ("q4_k" if decode else case["down"], h, ff)]
    if decode:
        mats.append(("q4_k", case["vocab"], h))
    ios = 4 * (3 * h + ff + sum(n for _, n, _ in mats)) if decode else 4 * (5 * h + 3 * h + 2 * kv + 2 * ff)
    return {"bytes": sum(_matrix(*a) for a in mats) + ios, "flops": sum(2 * n * k for _, n, k in mats)}


def tolerance(case):
    """About four times what the path shows against the same product in 64 bits.  Integer dots scaled in f32 and f32
    weights against f32 activations: 0.5 - 2e-7.  f16 operands under f32 sums: 2e-4 (activations rounded) to 3e-4 (weights
    too).  Where an activation is quantized again between two products, one of its int8 codes may round the other way
    after a last-bit difference: up to 3e-4 of one token's output."""
    if case["kind"] == "mm":
        float_rows = case["fmt"] in ("q8_0", "iq4_xs")
        f16 = case["act"] == "auto" and case["m"] >= 4 and (float_rows or case["m"] >= 32)
        return {"rel": 1.2e-3} if f16 else {"rel": 1e-6}
    return {"rel": 1e-6} if case["kind"] == "decode" else {"rel": 1e-3}
