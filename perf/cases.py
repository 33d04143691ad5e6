"""The work that a program using this library has it do, as cases to time and
to check: the attention calls of a CrossDiT block, the VAE's attention block
and the linear layers, each through the entry point that such a program
calls, with its descriptors, weights, tables and workspaces made beforehand.

Kinds of case:
  self    visual self-attention: 3-D RoPE on Q and K, optionally the
          query/key RMSNorm ahead of it, over a (T, Hp, Wp) token grid
  text    self-attention of a text block: RMSNorm and 1-D RoPE
  cross   text cross-attention, optionally with an F16 padding mask or the
          query/key RMSNorm
  vae     the VAE's attention block: one head of 512
  linear  a linear layer with bias; the weight either BF16 and kept, or
          stored in blocks (Q8_0, Q4_0) and expanded by the call
  load    a block weight expanded to BF16 rows, as a model load does it once
          per weight

Operand forms of the attention cases ("ops"): "bf16" and "f16" are Q, K and V
in that type; "ref" is Q F32 with K and V F16 (the graph's own cast done
before); "f32" is all three F32, K and V cast to F16 by the call.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kandinsky.cpp_amd"))

import kd_fa  # noqa: E402
import kd_mm  # noqa: E402

DEV = "cuda:0"
HEADS, D, D_VAE = 32, 128, 512
AXES, SCALE_FACTOR, THETA = (32, 48, 48), (1.0, 2.0, 2.0), 10000.0
EPS = 1e-6
SIXTEEN = {"bf16": torch.bfloat16, "f16": torch.float16, "ref": torch.float16, "f32": torch.float16}
QTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "ref": torch.float32, "f32": torch.float32}
KTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "ref": torch.float16, "f32": torch.float32}
OUT = {"f32": torch.float32, "bf16": torch.bfloat16}
BLOCK = {"q8_0": kd_mm.TYPE_Q8_0, "q4_0": kd_mm.TYPE_Q4_0}


def listed():
    return [
        # the smallest video: 5 latent frames of 16 x 16 patches, as the CPU-runnable configuration has it
        dict(name="self_1280_f16", kind="self", t=5, hp=16, wp=16, batch=1, ops="f16", norm=False, ws=True, out="f32"),
        # a short clip of an odd size in the graph's own operand types, from the projections on, guided pair
        dict(name="self_6510_f32_norm", kind="self", t=7, hp=30, wp=31, batch=2, ops="f32", norm=True, ws=True, out="f32"),
        # 512 x 512, 121 frames, guided pair: the layer that most of a generation's time goes to
        dict(name="self_31744_bf16", kind="self", t=31, hp=32, wp=32, batch=2, ops="bf16", norm=False, ws=True, out="f32"),
        # a text block's self-attention over a prompt of 300 tokens: latency and launches count
        dict(name="text_300_f32_norm", kind="text", l=300, batch=2, ops="f32", norm=True, ws=True, out="f32"),
        # cross-attention of the same clip to prompts padded to 256 tokens
        dict(name="cross_256_mask_bf16", kind="cross", lq=31744, lk=256, batch=2, ops="bf16", mask=True, norm=False, ws=True, out="f32"),
        # cross-attention to an unpadded prompt as the graph hands it over: Q F32, K and V F16, no mask
        dict(name="cross_300_ref", kind="cross", lq=31744, lk=300, batch=2, ops="ref", mask=False, norm=False, ws=False, out="f32"),
        # the image decoder's attention over a 64 x 64 latent
        dict(name="vae_4096", kind="vae", l=4096, ops="ref"),
        # the time embedding's and the modulations' layers: one row per guided branch
        dict(name="linear_2_bf16w", kind="linear", m=2, n=16384, k=4096, w="bf16", x="f32", bias=True),
        # a text block's projection over the prompt, its Q8_0 weight expanded by the call
        dict(name="linear_300_q8", kind="linear", m=300, n=4096, k=4096, w="q8_0", x="f32", bias=True),
        # a visual block's projection at the smallest video
        dict(name="linear_1280_bf16w", kind="linear", m=1280, n=4096, k=4096, w="bf16", x="f32", bias=True),
        # the same projection at 121 frames, guided pair
        dict(name="linear_63488_bf16w", kind="linear", m=63488, n=4096, k=4096, w="bf16", x="f32", bias=True),
        # one feed-forward weight of a Q4_0 model file expanded at load
        dict(name="load_q4_16384x4096", kind="load", n=16384, k=4096, w="q4_0"),
    ]


def log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["self", "self", "text", "cross", "cross", "vae", "linear", "linear", "linear", "linear", "load"])
    if kind == "self":
        hp, wp = rng.randint(8, 36), rng.randint(8, 36)
        ops = rng.choice(["bf16", "f16", "ref", "f32"])
        t = max(1, min(log_int(rng, 64, 31744), 31744 - hp * wp) // (hp * wp))
        return dict(kind=kind, t=t, hp=hp, wp=wp, batch=rng.choice([1, 2]), ops=ops, norm=rng.random() < 0.5,
                    ws=ops == "f32" or rng.random() < 0.75, out=rng.choice(["f32", "f32", "bf16"]))
    if kind == "text":
        return dict(kind=kind, l=log_int(rng, 16, 512), batch=rng.choice([1, 2]), ops=rng.choice(["bf16", "ref", "f32"]),
                    norm=True, ws=True, out=rng.choice(["f32", "f32", "bf16"]))
    if kind == "cross":
        return dict(kind=kind, lq=log_int(rng, 64, 31744), lk=log_int(rng, 16, 512), batch=rng.choice([1, 2]),
                    ops=rng.choice(["bf16", "f16", "ref"]), mask=rng.random() < 0.35, norm=rng.random() < 0.35,
                    ws=True, out=rng.choice(["f32", "f32", "bf16"]))
    if kind == "vae":
        return dict(kind=kind, l=log_int(rng, 64, 16384), ops=rng.choice(["bf16", "ref"]))
    n, k = rng.choice([(4096, 4096), (16384, 4096), (4096, 16384), (4096, 1024), (1024, 4096), (1536, 3584), (64, 4096)])
    if kind == "load":
        return dict(kind=kind, n=n, k=k, w=rng.choice(["q8_0", "q4_0"]))
    return dict(kind=kind, m=log_int(rng, 1, 63488), n=n, k=k, w=rng.choice(["bf16", "bf16", "q8_0", "q4_0"]),
                x=rng.choice(["f32", "f32", "bf16"]), bias=rng.random() < 0.75)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def normal(gen, shape, dtype, scale=1.0):
    x = torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)
    return (x * scale if scale != 1.0 else x).to(dtype)


def frequencies(n):
    return torch.exp(torch.arange(n, dtype=torch.float64) * (-math.log(THETA) / n))


def rope_rows(positions, dim, scale):
    a = positions.to(torch.float64)[:, None] * frequencies(dim // 2) / scale
    return torch.stack((a.cos(), a.sin()), dim=-1).flatten(-2)


def table_of(case):
    """(L, 128) F32 rows of interleaved (cos, sin)."""
    if case["kind"] == "text":
        return rope_rows(torch.arange(case["l"]), D, 1.0).float().to(DEV)
    t, hp, wp = case["t"], case["hp"], case["wp"]
    i = torch.arange(t * hp * wp)
    at = (i // (hp * wp), i // wp % hp, i % wp)
    return torch.cat([rope_rows(at[j], AXES[j], SCALE_FACTOR[j]) for j in range(3)], dim=1).float().to(DEV)


def lengths(case):
    if case["kind"] == "self":
        n = case["t"] * case["hp"] * case["wp"]
        return n, n
    if case["kind"] == "cross":
        return case["lq"], case["lk"]
    return case["l"], case["l"]


def padding_mask(gen, batch, lq, lk):
    """F16 (batch, 1, lq, lk): 0 on each prompt's own tokens, -inf on its padding."""
    valid = torch.randint(max(1, lk // 8), lk + 1, (batch,), generator=gen, device=DEV)
    row = torch.zeros((batch, 1, 1, lk), dtype=torch.float16, device=DEV)
    row.masked_fill_(torch.arange(lk, device=DEV) >= valid[:, None, None, None], float("-inf"))
    # rows padded to whole 16-byte chunks, as the library asks of a mask's stride
    mask = torch.zeros((batch, 1, lq, (lk + 7) // 8 * 8), dtype=torch.float16, device=DEV)[..., :lk]
    return mask.copy_(row.expand(batch, 1, lq, lk))


def attention_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    lq, lk = lengths(case)
    ops = case["ops"]
    if case["kind"] == "vae":
        heads, dim, batch = 1, D_VAE, 1
    else:
        heads, dim, batch = HEADS, D, case["batch"]
    q = normal(gen, (batch, heads, lq, dim), QTYPE[ops])
    k = normal(gen, (batch, heads, lk, dim), KTYPE[ops])
    v = normal(gen, (batch, heads, lk, dim), KTYPE[ops])
    got = dict(q=q, k=k, v=v, mask=None, table=None, wq=None, wk=None)
    if case["kind"] in ("self", "text"):
        got["table"] = table_of(case)
    if case.get("norm"):
        got["wq"] = 1.0 + normal(gen, (D,), torch.float32, 0.1)
        got["wk"] = 1.0 + normal(gen, (D,), torch.float32, 0.1)
    if case.get("mask"):
        got["mask"] = padding_mask(gen, batch, lq, lk)
    return got


def blocks_of(w, kind):
    """Weight rows (N, K) as Q8_0 or Q4_0 blocks: uint8 (N, K / 32 * block bytes)."""
    n, k = w.shape
    b = w.reshape(n, k // 32, 32)
    if kind == "q8_0":
        d = (b.abs().amax(-1, keepdim=True) / 127.0).half()
        q = torch.where(d > 0, b / d.float(), torch.zeros_like(b)).round().clamp(-127, 127).to(torch.int8)
        data = q.view(torch.uint8)
    else:
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        d = (top / -8.0).half()
        q = torch.where(d != 0, b / d.float(), torch.zeros_like(b)).add(8.5).trunc().clamp(0, 15).to(torch.uint8)
        data = q[..., :16] | (q[..., 16:] << 4)
    return torch.cat((d.view(torch.uint8), data), dim=-1).reshape(n, -1).contiguous()


def values_of(blocks, kind, k):
    """The F32 values of such blocks, rounded to BF16: (N, K)."""
    n = blocks.shape[0]
    b = blocks.reshape(n, k // 32, -1)
    d = b[..., :2].contiguous().view(torch.float16).float()
    if kind == "q8_0":
        q = b[..., 2:].contiguous().view(torch.int8).float()
    else:
        q = torch.cat((b[..., 2:] & 15, b[..., 2:] >> 4), dim=-1).float() - 8.0
    return (q * d).reshape(n, k).bfloat16()


def weight_of(gen, case):
    w = normal(gen, (case["n"], case["k"]), torch.float32, case["k"] ** -0.5)
    return w.bfloat16() if case["w"] == "bf16" else blocks_of(w, case["w"])


def linear_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    w = weight_of(gen, case)
    if case["kind"] == "load":
        return dict(w=w)
    x = normal(gen, (case["m"], case["k"]), torch.float32 if case["x"] == "f32" else torch.bfloat16)
    bias = normal(gen, (case["n"],), torch.float32, 0.1) if case["bias"] else None
    return dict(w=w, x=x, bias=bias)


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------

def prepare(case, seed):
    if case["kind"] in ("linear", "load"):
        s = linear_inputs(case, seed)
        if case["w"] != "bf16":
            s["w"] = kd_mm.QuantWeight(s["w"], BLOCK[case["w"]], case["k"])
        s["kind"] = case["kind"]
        if case["kind"] == "linear":
            s["dst"] = torch.empty((case["m"], case["n"]), dtype=torch.float32, device=DEV)
            s["desc"] = kd_mm.make_desc(s["w"], s["x"], s["bias"], s["dst"])
            need = kd_mm.workspace_size(s["desc"])
            s["ws"] = torch.empty(need, dtype=torch.uint8, device=DEV) if need else None
        return s
    s = attention_inputs(case, seed)
    q, v = s["q"], s["v"]
    s["kind"] = "attention"
    s["dst"] = torch.empty(kd_fa.out_shape(q, v), dtype=OUT[case.get("out", "f32")], device=DEV)
    s["desc"] = kd_fa.make_desc(q, s["k"], v, s["mask"], s["dst"], 1.0 / q.shape[-1] ** 0.5)
    s["rope"] = kd_fa.rope_table(s["table"]) if s["table"] is not None else None
    s["norm"] = kd_fa.qk_norm(s["wq"], s["wk"], EPS) if s["wq"] is not None else None
    need = kd_fa.workspace_size_full(s["desc"], s["rope"], s["norm"]) if case.get("ws", True) else 0
    s["ws"] = torch.empty(need, dtype=torch.uint8, device=DEV) if need else None
    return s


def run(state):
    if state["kind"] == "load":
        return kd_mm.dequant(state["w"])
    if state["kind"] == "linear":
        status = kd_mm.run_desc(state["desc"], state["ws"])
    else:
        status = kd_fa.run_desc(state["desc"], state["rope"], None, state["ws"], state["norm"])
    if status != kd_fa.OK:
        raise kd_fa.KdFaError(status, state["kind"])
    return state["dst"]


# ---------------------------------------------------------------------------
# what a pass needs, and how exact its results are
# ---------------------------------------------------------------------------

WEIGHT_BYTES = {"bf16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32}


def work(case):
    if case["kind"] in ("linear", "load"):
        n, k = case["n"], case["k"]
        bytes_w = n * k * WEIGHT_BYTES[case["w"]]
        if case["kind"] == "load":
            return {"bytes": bytes_w + 2 * n * k, "flops": 0}
        m = case["m"]
        return {"bytes": bytes_w + m * k * (4 if case["x"] == "f32" else 2) + m * n * 4, "flops": 2 * m * n * k}
    lq, lk = lengths(case)
    pairs, dim = (1, D_VAE) if case["kind"] == "vae" else (case["batch"] * HEADS, D)
    qb = 4 if QTYPE[case["ops"]] == torch.float32 else 2
    kb = 4 if KTYPE[case["ops"]] == torch.float32 else 2
    ob = 4 if case.get("out", "f32") == "f32" else 2
    total = pairs * dim * (lq * (qb + ob) + 2 * lk * kb)
    if case["kind"] in ("self", "text"):
        total += lq * D * 4
    if case.get("mask"):
        total += case["batch"] * lq * lk * 2
    return {"bytes": total, "flops": 4 * pairs * lq * lk * dim}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "linear":
        # products of the same BF16 values summed in F32: 4e-7 off the 64-bit sums at 4,096 terms, up to 16,384 of them here
        return {"rel": 4e-6, "max": 4e-5}
    # the weights of the keys are rounded to K's type (F16: 2.1e-4 off the 64-bit result, BF16: 1.7e-3), as is a 16-bit
    # output (BF16, both: 2.3e-3)
    return {"rel": 1e-2, "max": 0.1} if "bf16" in (case["ops"], case.get("out")) else {"rel": 8e-4, "max": 1e-2}


def rotated(x, table):
    """Interleaved pairs of x (..., L, 128) turned by the table's rows, in F32."""
    c, s = table[:, 0::2], table[:, 1::2]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * s, x0 * s + x1 * c), dim=-1).flatten(-2)


def operand(x, weight, table, dtype):
    """One head's rows normalised and rotated, then rounded to the products' type, as 64-bit values."""
    x = x.float()
    if weight is not None:
        mean = x.double().square().mean(-1, keepdim=True).float()
        x = x * (1.0 / (mean + EPS).sqrt()) * weight
    if table is not None:
        x = rotated(x, table)
    return x.to(dtype).double()


def exact(case, seed):
    """The call's result from its operands as the products see them, in 64 bits."""
    if case["kind"] == "load":
        return values_of(linear_inputs(case, seed)["w"], case["w"], case["k"])
    if case["kind"] == "linear":
        s = linear_inputs(case, seed)
        w = (s["w"] if case["w"] == "bf16" else values_of(s["w"], case["w"], case["k"])).double()
        y = torch.empty((case["m"], case["n"]), dtype=torch.float64, device=DEV)
        for i in range(0, case["m"], 8192):
            y[i:i + 8192] = s["x"][i:i + 8192].bfloat16().double() @ w.T
        return y if s["bias"] is None else y + s["bias"].double()
    s = attention_inputs(case, seed)
    q, k, v = s["q"], s["k"], s["v"]
    batch, heads, lq, dim = q.shape
    dtype = SIXTEEN[case["ops"]]
    out = torch.empty((batch, lq, heads, dim), dtype=torch.float64, device=DEV)
    step = max(64, (1 << 27) // max(1, k.shape[2]))
    for b in range(batch):
        mask = s["mask"][b, 0].double() if s["mask"] is not None else None
        for h in range(heads):
            kk = operand(k[b, h], s["wk"], s["table"], dtype).T.contiguous()
            vv = v[b, h].to(dtype).double()
            qq = operand(q[b, h], s["wq"], s["table"], dtype)
            for i in range(0, lq, step):
                p = (qq[i:i + step] @ kk).mul_(1.0 / dim ** 0.5)
                if mask is not None:
                    p += mask[i:i + step]
                out[b, i:i + step, h] = torch.softmax(p, dim=-1) @ vv
    return out
