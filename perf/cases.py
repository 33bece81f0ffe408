"""The work that programs have this framework do, as measurable cases.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call (inputs,
packed weights, a decoder with its graph), ``run`` is one pass through the public entry points,
``work`` the bytes and operations that pass cannot do without, ``exact`` its result in 64 bits from
plain torch and ``tolerance`` how far two correct implementations of the same precision may be
apart.  The kinds:

* ``weight``: activations times a packed weight, ``linalg.matvec`` for one row and
  ``linalg.matmul_nt`` for more -- every projection of a quantised model, decode and prefill;
* ``mx``: two packed operands on ``linalg.matmul_nt`` (4- or 6-bit activations and weights);
* ``dense``: ``linalg.matmul`` of two ordinary matrices, the right one row-major;
* ``quantize``: ``quantize_mx`` of activations, the step before an ``mx`` product;
* ``unpack``: ``PackedTensor.unpack``, a packed weight decoded for ordinary use;
* ``prefill`` / ``decode``: the decoder's prompt pass, and one replayed decode step.
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tinygrad-dx12_amd"))

from tinygrad_mi355x.codegen import linalg  # noqa: E402
from tinygrad_mi355x.codegen.decomp.mi355x import PackedTensor, quantize_mx  # noqa: E402
from tinygrad_mi355x.decoder import Decoder, DecoderConfig, random_weights  # noqa: E402

DEVICE = "cuda"
BITS = {"int4": 4, "uint4": 4, "fp4_e2m1": 4, "fp6_e2m3": 6, "fp6_e3m2": 6}
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
MAX_NEW = 128  # tokens a decoder state has room for past its prompt


def listed():
    return [
        # one token through a 4096 x 4096 INT4 projection: the smallest call, a 9 MB stream
        dict(name="matvec_int4_4096", kind="weight", fmt="int4", group=32, m=1, n=4096, k=4096, out="float16"),
        # one token through an FP4 up projection: batch-1 decode's largest product
        dict(name="matvec_fp4_14336", kind="weight", fmt="fp4_e2m1", group=32, m=1, n=14336, k=4096, out="bfloat16"),
        # 64 sequences decoding together, or a short prompt, through the same projection
        dict(name="linear_fp4_m64", kind="weight", fmt="fp4_e2m1", group=32, m=64, n=14336, k=4096, out="bfloat16"),
        # a 512-token prompt through stacked q|k|v rows in INT4
        dict(name="linear_int4_m512", kind="weight", fmt="int4", group=128, m=512, n=6144, k=4096, out="float16"),
        # a 2048-token prompt through an FP6 feed-forward projection
        dict(name="linear_fp6_m2048", kind="weight", fmt="fp6_e3m2", group=32, m=2048, n=11008, k=4096, out="bfloat16"),
        # 4-bit activations and weights, a large prefill batch
        dict(name="mx_fp4_4096", kind="mx", fa="fp4_e2m1", fb="fp4_e2m1", m=4096, n=14336, k=4096, out="bfloat16"),
        # 6-bit activations on 4-bit weights, a prompt of an odd length
        dict(name="mx_fp6_fp4_m1001", kind="mx", fa="fp6_e2m3", fb="fp4_e2m1", m=1001, n=4096, k=4096, out="bfloat16"),
        # an unquantised layer: relu(A @ B)'s product without the epilogue
        dict(name="dense_bf16_4096", kind="dense", dtype="bfloat16", m=4096, n=4096, k=4096, out="bfloat16"),
        # the activations of a prompt on their way into a 4-bit product
        dict(name="quantize_fp4_4096", kind="quantize", fmt="fp4_e2m1", dtype="bfloat16", rows=4096, k=4096),
        # a packed weight decoded for a program that wants it in bf16
        dict(name="unpack_fp4_14336", kind="unpack", fmt="fp4_e2m1", group=32, n=14336, k=4096, out="bfloat16"),
        # the decoder's two halves: eight 512-token prompts (two layers: more of them repeat the same work, and
        # through random weights a rounding that flips a sharp attention row grows with every layer), and one
        # token for each of eight sequences
        dict(name="prefill_b8", kind="prefill", batch=8, prompt=512, layers=2),
        dict(name="decode_b8", kind="decode", batch=8, prompt=512, layers=8),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _k(rng, high=14336):
    """A contraction length: rows of packed weights in real models are whole multiples of 128."""
    return 128 * _log_int(rng, 4, high // 128)


def draw(rng):
    kind = rng.choice(["weight", "weight", "weight", "weight", "mx", "mx", "dense", "quantize", "unpack", "prefill",
                       "decode"])
    if kind == "weight":
        fmt = rng.choice(["int4", "uint4", "fp4_e2m1", "fp6_e2m3", "fp6_e3m2"])
        group = rng.choice([32, 64, 128]) if fmt in ("int4", "uint4") else 32
        out = rng.choice(["float16" if fmt in ("int4", "uint4") else "bfloat16", "float32"])
        return dict(kind=kind, fmt=fmt, group=group, m=_log_int(rng, 1, 4096), n=_log_int(rng, 512, 16384), k=_k(rng),
                    out=out)
    if kind == "mx":
        fa = rng.choice(["fp4_e2m1", "fp6_e2m3", "fp6_e3m2"])
        fb = rng.choice(["fp4_e2m1", "fp6_e2m3"])
        return dict(kind=kind, fa=fa, fb=fb, m=_log_int(rng, 17, 4096), n=_log_int(rng, 512, 16384), k=_k(rng),
                    out=rng.choice(["bfloat16", "float32"]))
    if kind == "dense":
        return dict(kind=kind, dtype=rng.choice(["bfloat16", "float16"]), m=_log_int(rng, 17, 4096),
                    n=8 * _log_int(rng, 64, 1024), k=64 * _log_int(rng, 8, 128), out=rng.choice(["bfloat16", "float32"]))
    if kind == "quantize":
        return dict(kind=kind, fmt=rng.choice(["fp4_e2m1", "fp6_e2m3", "fp6_e3m2"]),
                    dtype=rng.choice(["bfloat16", "float16", "float32"]), rows=_log_int(rng, 1, 8192),
                    k=32 * _log_int(rng, 16, 448))
    if kind == "unpack":
        fmt = rng.choice(["int4", "uint4", "fp4_e2m1", "fp6_e2m3", "fp6_e3m2"])
        group = rng.choice([32, 64, 128]) if fmt in ("int4", "uint4") else 32
        return dict(kind=kind, fmt=fmt, group=group, n=_log_int(rng, 64, 14336), k=4 * _log_int(rng, 128, 2048),
                    out=rng.choice(["bfloat16", "float16", "float32"]))
    batch = rng.randint(1, 8)
    prompt = _log_int(rng, 2, 512) if kind == "prefill" else _log_int(rng, 16, 1024)
    return dict(kind=kind, batch=batch, prompt=prompt, layers=2)


# ------------------------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _packed(fmt, n, k, group, g):
    """A packed weight as a quantised model stores it: INT4 codes over their whole range with fp16
    scales per group, N(0, 0.02) weights MX-quantised with E8M0 scales per 32 otherwise."""
    if fmt in ("int4", "uint4"):
        data = torch.randint(0, 256, ((n * k + 1) // 2,), dtype=torch.uint8, device=DEVICE, generator=g)
        scales = (torch.rand((n, -(-k // group)), device=DEVICE, generator=g) * 0.003 + 0.002).to(torch.float16)
        return PackedTensor(data, fmt, (n, k), scales, group)
    if k % 32 == 0:
        return quantize_mx(torch.randn((n, k), device=DEVICE, generator=g) * 0.02, fmt)
    data = torch.randint(0, 256, ((n * k * BITS[fmt] + 7) // 8,), dtype=torch.uint8, device=DEVICE, generator=g)
    scales = torch.randint(118, 124, (n, -(-k // 32)), dtype=torch.uint8, device=DEVICE, generator=g)
    return PackedTensor(data, fmt, (n, k), scales.view(torch.float8_e8m0fnu), 32)


def _activations(m, k, dtype, g):
    return torch.randn((m, k), device=DEVICE, generator=g).to(dtype)


def _new_positions(case):
    """The cache positions that a pass fills."""
    return (0, case["prompt"]) if case["kind"] == "prefill" else (case["prompt"], case["prompt"] + 1)


def _config(case):
    return DecoderConfig(layers=case["layers"])


def _decoder_inputs(case, seed):
    cfg, g = _config(case), _generator(seed)
    weights = random_weights(cfg, DEVICE, seed)
    prompts = torch.randint(0, cfg.vocab, (case["batch"], case["prompt"]), device=DEVICE, generator=g)
    tokens = torch.randint(0, cfg.vocab, (case["batch"],), dtype=torch.int32, device=DEVICE, generator=g)
    caches = None
    if case["kind"] == "decode":  # keys and values of earlier tokens
        shape = (cfg.layers, case["batch"], cfg.kv_heads, case["prompt"], cfg.head_dim)
        caches = [torch.randn(shape, device=DEVICE, generator=g).to(torch.bfloat16) for _ in range(2)]
    return cfg, weights, prompts, tokens, caches


def _operands(case, seed):
    """The inputs of every kind but the decoder's."""
    g, kind = _generator(seed), case["kind"]
    if kind == "weight":
        xdt = torch.float16 if case["fmt"] in ("int4", "uint4") else torch.bfloat16
        return _packed(case["fmt"], case["n"], case["k"], case["group"], g), _activations(case["m"], case["k"], xdt, g)
    if kind == "mx":
        a = quantize_mx(_activations(case["m"], case["k"], torch.bfloat16, g), case["fa"])
        return a, _packed(case["fb"], case["n"], case["k"], 32, g)
    if kind == "dense":
        dt = DTYPES[case["dtype"]]
        return (_activations(case["m"], case["k"], dt, g),
                (torch.randn((case["k"], case["n"]), device=DEVICE, generator=g) * 0.02).to(dt))
    if kind == "quantize":
        return (_activations(case["rows"], case["k"], DTYPES[case["dtype"]], g),)
    return (_packed(case["fmt"], case["n"], case["k"], case["group"], g),)


def prepare(case, seed):
    if case["kind"] not in ("prefill", "decode"):
        ops = _operands(case, seed)
        if case["kind"] == "weight" and case["m"] == 1:
            ops = (ops[0], ops[1][0])
        return dict(case=case, ops=ops)
    cfg, weights, prompts, tokens, caches = _decoder_inputs(case, seed)
    t = case["prompt"]
    dec = Decoder(weights, cfg, case["batch"], t + MAX_NEW, t)
    state = dict(case=case, dec=dec, prompts=prompts)
    if case["kind"] == "decode":
        # the prompts are in the cache and one step has run eagerly, as generate() does before it captures
        dec.k_cache[:, :, :, :t], dec.v_cache[:, :, :, :t] = caches
        state["tokens"], state["pos"] = tokens, torch.full_like(dec.pos, t)
        dec.tokens[:case["batch"]].copy_(tokens)
        dec.pos.fill_(t)
        dec.step()
        state["graph"] = dec.capture()
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "weight":
        w, x = state["ops"]
        out = DTYPES[case["out"]]
        return linalg.matvec(w, x, out) if case["m"] == 1 else linalg.matmul_nt(x, w, dtype=out)
    if kind == "mx":
        a, b = state["ops"]
        return linalg.matmul_nt(a, b, dtype=DTYPES[case["out"]])
    if kind == "dense":
        a, b = state["ops"]
        return linalg.matmul(a, b, dtype=DTYPES[case["out"]])
    if kind == "quantize":
        q = quantize_mx(state["ops"][0], case["fmt"])
        return dict(data=q.data, scales=q.scales.view(torch.uint8))
    if kind == "unpack":
        return state["ops"][0].unpack(DTYPES[case["out"]])
    dec = state["dec"]
    if kind == "prefill":
        dec.prefill(state["prompts"])
    else:
        dec.tokens[:dec.batch].copy_(state["tokens"])  # the sequences' newest tokens, at the position after the prompt
        dec.pos.copy_(state["pos"])
        current = torch.cuda.current_stream()
        dec.graph_stream.wait_stream(current)
        state["graph"].launch()
        current.wait_stream(dec.graph_stream)
    first, end = _new_positions(case)
    return dict(logits=dec.logits, k=dec.k_cache[:, :, :, first:end], v=dec.v_cache[:, :, :, first:end])


# --------------------------------------------------------------------------------- what it takes
def _packed_bytes(fmt, n, k, group):
    scale = 2 if fmt in ("int4", "uint4") else 1
    return n * k * BITS[fmt] / 8 + n * -(-k // group) * scale


def work(case):
    kind = case["kind"]
    if kind in ("weight", "mx", "dense"):
        m, n, k = case["m"], case["n"], case["k"]
        size = DTYPES[case["out"]].itemsize
        if kind == "weight":
            read = _packed_bytes(case["fmt"], n, k, case["group"]) + 2 * m * k
        elif kind == "mx":
            read = _packed_bytes(case["fa"], m, k, 32) + _packed_bytes(case["fb"], n, k, 32)
        else:
            read = 2 * (m * k + k * n)
        return dict(bytes=read + m * n * size, flops=2 * m * n * k)
    if kind == "quantize":
        rows, k = case["rows"], case["k"]
        return dict(bytes=rows * k * DTYPES[case["dtype"]].itemsize + _packed_bytes(case["fmt"], rows, k, 32),
                    flops=3 * rows * k)
    if kind == "unpack":
        n, k = case["n"], case["k"]
        return dict(bytes=_packed_bytes(case["fmt"], n, k, case["group"]) + n * k * DTYPES[case["out"]].itemsize,
                    flops=n * k)
    cfg = _config(case)
    b, t = case["batch"], case["prompt"]
    rows = b * t if kind == "prefill" else b
    pairs = b * t * (t + 1) / 2 if kind == "prefill" else b * (t + 1)  # (query, key) positions
    d, width = cfg.hidden, cfg.heads * cfg.head_dim
    weights = cfg.qkv_rows * d + d * width + 3 * d * cfg.ffn
    cache = 2 * 2 * cfg.layers * b * (t + (kind == "decode")) * cfg.kv_heads * cfg.head_dim
    return dict(bytes=cfg.weight_bytes_per_token() + cache + 2 * rows * d + 4 * b * cfg.vocab,
                flops=cfg.layers * (2 * rows * weights + 4 * pairs * width) + 2 * b * cfg.vocab * d)


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "unpack"):
        return "exact"
    if kind in ("prefill", "decode"):
        return dict(rel=1e-2, max=0.2)  # 16-bit activations between the layers' products
    # about four times the distance from the 64-bit product rounded once to the same type: sums of up to
    # 14336 products in fp32, and the last place of a 16-bit result where two sums straddle a tie
    return {"float32": dict(rel=2e-6, max=2e-5), "float16": dict(rel=2.5e-4, max=4e-3),
            "bfloat16": dict(rel=2.5e-4, max=2e-2)}[case["out"]]


# ------------------------------------------------------------------------------ 64-bit results
def _table(fmt):
    """The value of every code of a format."""
    if fmt == "int4":
        return [float(c - 16 if c > 7 else c) for c in range(16)]
    if fmt == "uint4":
        return [float(c) for c in range(16)]
    e_bits, m_bits, bias = {"fp4_e2m1": (2, 1, 1), "fp6_e2m3": (2, 3, 1), "fp6_e3m2": (3, 2, 3)}[fmt]
    values = []
    for c in range(1 << BITS[fmt]):
        e, f = (c >> m_bits) & ((1 << e_bits) - 1), c & ((1 << m_bits) - 1)
        mag = math.ldexp(f + (1 << m_bits), e - bias - m_bits) if e else math.ldexp(f, 1 - bias - m_bits)
        values.append(-mag if c >> (e_bits + m_bits) else mag)
    return values


def _dequantised(w):
    """A packed matrix in 64 bits: codes from the little-endian bit stream, times their scales."""
    n, k = w.shape
    d = w.data.to(torch.int64)
    if BITS[w.format] == 4:
        codes = torch.stack((d & 15, d >> 4), -1).reshape(-1)[:n * k]
    else:
        d = torch.nn.functional.pad(d, (0, -d.numel() % 3)).reshape(-1, 3)
        word = d[:, 0] | (d[:, 1] << 8) | (d[:, 2] << 16)
        codes = torch.stack([(word >> s) & 63 for s in (0, 6, 12, 18)], -1).reshape(-1)[:n * k]
    values = torch.tensor(_table(w.format), dtype=torch.float64, device=d.device)[codes].reshape(n, k)
    if w.scales.dtype is torch.float8_e8m0fnu:
        s = torch.exp2(w.scales.view(torch.uint8).double() - 127)
    else:
        s = w.scales.double()
    return values * s.repeat_interleave(w.block_size, 1)[:, :k]


def _rounded(x, dtype):
    return x.to(torch.float32).to(dtype).double()


def _norm(h, weight, eps):
    return h / torch.sqrt(h.square().mean(-1, keepdim=True) + eps) * weight.double()


def _rope(x, pos, base):
    half = x.shape[-1] // 2
    angle = pos.double()[:, None] * base ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    c, s = angle.cos(), angle.sin()
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat((lo * c - hi * s, hi * c + lo * s), -1)


def _decoder_pass(cfg, weights, tokens, start, caches):
    """One pass over tokens [B, T] at positions start ..: the logits of the last token, with the k and
    v of the new positions written to ``caches``.  Activations and caches are rounded to 16 bits where
    the decoder's storage is; everything between is 64-bit."""
    b, t = tokens.shape
    heads, kv, hd = cfg.heads, cfg.kv_heads, cfg.head_dim
    pos = torch.arange(start, start + t, device=DEVICE)
    blocked = torch.arange(start + t, device=DEVICE)[None, :] > pos[:, None]
    h = weights.embed[tokens].double()
    for layer, (kc, vc) in zip(weights.layers, caches):
        x = _rounded(_norm(h, layer.attn_norm, cfg.eps), torch.float16)
        qkv = (x @ _dequantised(layer.wqkv).T).reshape(b, t, heads + 2 * kv, hd).transpose(1, 2)
        q = _rope(qkv[:, :heads], pos, cfg.rope_base)
        kc[:, :, start:start + t] = _rounded(_rope(qkv[:, heads:heads + kv], pos, cfg.rope_base), torch.bfloat16)
        vc[:, :, start:start + t] = _rounded(qkv[:, heads + kv:], torch.bfloat16)
        out = torch.empty((b, heads, t, hd), dtype=torch.float64, device=DEVICE)
        for i in range(heads):  # one head at a time bounds the score matrices
            k, v = kc[:, i * kv // heads, :start + t], vc[:, i * kv // heads, :start + t]
            scores = torch.matmul(q[:, i], k.transpose(1, 2).contiguous()) / math.sqrt(hd)
            out[:, i] = torch.matmul(scores.masked_fill(blocked, -math.inf).softmax(-1), v)
        attn = _rounded(out.transpose(1, 2).reshape(b, t, heads * hd), torch.float16)
        h = h + attn @ _dequantised(layer.wo).T
        x = _rounded(_norm(h, layer.ffn_norm, cfg.eps), torch.bfloat16)
        gu = x @ _dequantised(layer.w_gate_up).T
        gate, up = gu[..., 0::2], gu[..., 1::2]
        act = _rounded(gate / (1 + torch.exp(-gate)) * up, torch.bfloat16)
        h = h + act @ _dequantised(layer.w_down).T
    x = _rounded(_norm(h[:, -1], weights.final_norm, cfg.eps), torch.bfloat16)
    return x @ weights.lm_head.double().T


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # codes and exponents: whole numbers
    if kind == "unpack":
        return _dequantised(_operands(case, seed)[0])
    if kind == "weight":
        w, x = _operands(case, seed)
        y = x.double() @ _dequantised(w).T
        return y[0] if case["m"] == 1 else y
    if kind == "mx":
        a, b = _operands(case, seed)
        return _dequantised(a) @ _dequantised(b).T
    if kind == "dense":
        a, b = _operands(case, seed)
        return a.double() @ b.double()
    cfg, weights, prompts, tokens, caches = _decoder_inputs(case, seed)
    first, end = _new_positions(case)
    shape = (cfg.layers, case["batch"], cfg.kv_heads, end, cfg.head_dim)
    k, v = (torch.zeros(shape, dtype=torch.float64, device=DEVICE) for _ in range(2))
    if kind == "decode":
        k[:, :, :, :first], v[:, :, :, :first] = caches
        prompts = tokens[:, None].long()
    logits = _decoder_pass(cfg, weights, prompts, first, list(zip(k, v)))
    return dict(logits=logits, k=k[:, :, :, first:], v=v[:, :, :, first:])
