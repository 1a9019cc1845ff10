"""Performance cases of the library: the calls its users make, through the Python entry points they call.

A case is one kind of call (`op`) with its sizes, types and options:

  attn       fmha_forward: prompt processing (causal) and the attention of image models (none, odd key counts)
  attn_bwd   fmha_backward: the training step's attention gradients
  gemm       run_gemm on 16-bit operands: from one decode row to a whole batch of tokens, both storage orders of the
             weights, fused bias / activation, sizes that no tile divides; scratch as gemm_workspace_bytes asks for it
  gemm_f32   run_gemm on fp32, the default type of the programs behind the custom call
  int4       int4_gemm / int4_gemm_ws: weight-only quantised linears, decode rows and prompts; `layers` products in a
             row, each with its own weights, as a model's blocks issue them
  fp8        fp8_gemm: e4m3 linears with per-tensor scales
  decode     GptjDecoder.step: a whole decode step on int4 weights and an fp16 cache

Inputs have the distributions of the benchmark's configurations.  Everything a program keeps between calls (weights,
outputs, scratch, the decoder's descriptors) is made by prepare(); run() is the call itself.
"""
import importlib
import math

import torch

xmk = importlib.import_module("intel-extension-for-openxla_amd")

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPILOGUES = {"none": xmk.EPI_DEFAULT, "bias": xmk.EPI_BIAS, "gelu": xmk.EPI_GELU, "bias_relu": xmk.EPI_BIAS_RELU,
             "bias_gelu": xmk.EPI_BIAS_GELU}
# the decode step's model: the GPT-J-6B shape of the benchmark's decode configuration
D_MODEL, HEADS, HEAD_DIM, ROTARY, D_FF, VOCAB, GROUP = 4096, 16, 256, 64, 16384, 50400, 128
MAX_FLOPS = 1.0e12  # a drawn case stays below the 8192^3 product


def listed():
    return [
        # prompt processing of a long batch: the benchmark's headline attention
        dict(name="attn_causal", op="attn", dtype="bf16", b=8, n=32, f=2048, t=2048, h=128, causal=True, bias=False, lse=False),
        # the smallest attention of an image model's network: cross attention to 77 text tokens, latency only
        dict(name="attn_cross_small", op="attn", dtype="f16", b=2, n=8, f=64, t=77, h=160, causal=False, bias=False, lse=False),
        # training: gradients of the headline attention
        dict(name="attn_backward", op="attn_bwd", dtype="bf16", b=8, n=32, s=2048, h=128, causal=True),
        # the largest dense product
        dict(name="gemm_8192", op="gemm", dtype="bf16", m=8192, n=8192, k=8192, rhs_t=False, epi="none"),
        # a linear layer over a prompt of 512 tokens
        dict(name="gemm_bias_512", op="gemm", dtype="bf16", m=512, n=4096, k=4096, rhs_t=False, epi="bias"),
        # four decode rows through a dense MLP projection
        dict(name="gemm_rows", op="gemm", dtype="f16", m=4, n=4096, k=16384, rhs_t=False, epi="bias"),
        # no dimension is even: rows of neither operand nor output start on a vector boundary
        dict(name="gemm_odd", op="gemm", dtype="bf16", m=1023, n=5003, k=2047, rhs_t=False, epi="bias_gelu"),
        # a linear layer of a program in its default precision
        dict(name="gemm_f32", op="gemm_f32", m=2048, n=2048, k=1024, rhs_t=False, epi="bias"),
        # one token through the MLP up-projections of eight blocks
        dict(name="int4_decode", op="int4", m=1, k=4096, n=16384, group=128, layers=8, bias=True),
        # a prompt of 512 tokens through one quantised projection
        dict(name="int4_prompt", op="int4", m=512, k=4096, n=16384, group=128, layers=1, bias=True),
        # a short prompt (or a large decode batch) through an fp8 projection
        dict(name="fp8_linear", op="fp8", m=256, n=16384, k=4096, rhs_t=True, bias=False, d_scale=False),
        # a whole decode step, four sequences with full caches
        dict(name="decode_step", op="decode", layers=28, batch=4, position=2047, capacity=2048),
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """A size spread over the logarithm of lo..hi; a multiple of `step`."""
    return max(step, _log(rng, lo, hi) // step * step)


def _fit(m, n, k, limit, step=1):
    """The three sizes of a product, the largest halved until 2 m n k fits the limit."""
    d = [m, n, k]
    while 2.0 * d[0] * d[1] * d[2] > limit:
        i = d.index(max(d))
        d[i] = max(step, d[i] // 2 // step * step)
    return d


def _draw_attn(rng):
    h = rng.choice([40, 64, 80, 128, 160, 256])
    f = _log(rng, 32, 8192)
    kind = rng.choice(["self", "causal", "cross"])
    t = rng.choice([77, _log(rng, 16, 512)]) if kind == "cross" else f
    b, n = rng.choice([1, 2, 4, 8]), rng.randint(4, 32)
    while 4.0 * b * n * f * t * h > 5.0e11:
        b, n = max(1, b // 2), max(1, n // 2)
    bias = rng.random() < 0.2 and b * n * f * t <= 1 << 28
    return dict(op="attn", dtype=rng.choice(["bf16", "f16"]), b=b, n=n, f=f, t=t, h=h, causal=kind == "causal", bias=bias,
                lse=kind != "cross" and rng.random() < 0.5)


def _draw_attn_bwd(rng):
    h = rng.choice([64, 64, 80, 128, 128, 256])
    s = _log(rng, 64, 4096)
    b, n = rng.choice([1, 2, 4, 8]), rng.randint(4, 32)
    while 10.0 * b * n * s * s * h > 6.0e11:
        b, n = max(1, b // 2), max(1, n // 2)
    return dict(op="attn_bwd", dtype=rng.choice(["bf16", "f16"]), b=b, n=n, s=s, h=h, causal=rng.random() < 0.7)


def _draw_gemm(rng):
    step = rng.choice([1, 8, 8, 64])
    m, n, k = _fit(_log(rng, 1, 8192), _size(rng, 64, 16384, step), _size(rng, 64, 16384, step), MAX_FLOPS, step)
    if step == 1:
        n, k = n | 1, k | 1
    return dict(op="gemm", dtype=rng.choice(["bf16", "f16"]), m=m, n=n, k=k, rhs_t=rng.random() < 0.4,
                epi=rng.choice(["none", "bias", "gelu", "bias_relu", "bias_gelu"]))


def _draw_gemm_f32(rng):
    step = rng.choice([1, 4, 64])
    m, n, k = _fit(_log(rng, 4, 4096), _size(rng, 64, 4096, step), _size(rng, 64, 4096, step), 1.0e11, step)
    if step == 1:
        n, k = n | 1, k | 1
    return dict(op="gemm_f32", m=m, n=n, k=k, rhs_t=rng.random() < 0.4, epi=rng.choice(["none", "bias", "bias_relu", "gelu"]))


def _draw_int4(rng):
    group = rng.choice([32, 64, 128, 128, 256])
    k, n = _size(rng, 1024, 16384, group), _size(rng, 1024, 16384, 8)
    m = _log(rng, 1, 2048)
    return dict(op="int4", m=m, k=k, n=n, group=group, layers=rng.randint(1, 8) if m <= 32 else 1, bias=rng.random() < 0.5)


def _draw_fp8(rng):
    step = rng.choice([1, 16, 16, 64])
    m, n, k = _fit(_log(rng, 1, 8192), _size(rng, 64, 16384, step), _size(rng, 64, 16384, step), MAX_FLOPS, step)
    if step == 1:
        n, k = n | 1, k | 1
    return dict(op="fp8", m=m, n=n, k=k, rhs_t=rng.random() < 0.6, bias=rng.random() < 0.4, d_scale=rng.random() < 0.2)


def _draw_decode(rng):
    capacity = _size(rng, 64, 2048, 8)
    return dict(op="decode", layers=rng.randint(2, 28), batch=rng.randint(1, 8), position=rng.randint(capacity // 2, capacity - 1),
                capacity=capacity)


def draw(rng):
    """A case of the ranges above; an op is as likely as the listed cases of that op are many."""
    return rng.choice([_draw_attn, _draw_attn, _draw_attn_bwd, _draw_gemm, _draw_gemm, _draw_gemm, _draw_gemm, _draw_gemm_f32,
                       _draw_int4, _draw_int4, _draw_fp8, _draw_decode])(rng)


# ------------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, scale=1.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _uniform(g, shape, lo, hi):
    return torch.empty(shape, device="cuda", dtype=torch.float16).uniform_(lo, hi, generator=g)


def _int4_linear(g, k, n, group, bias):
    """Uniform random nibbles, scales U(0.001, 0.02), zero points U(0, 15)."""
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    return qw, _uniform(g, (k // group, n), 0.001, 0.02), _uniform(g, (k // group, n), 0.0, 15.0), \
        _normal(g, (n,), torch.float16, 0.02) if bias else None


def _fp8(g, shape):
    x = torch.randn(shape, generator=g, device="cuda")
    scale = (x.abs().max() / 448.0).reshape(1)
    return (x / scale).to(torch.float8_e4m3fn), scale


def prepare(case, seed):
    g, op = _generator(seed), case["op"]
    c = case
    if op == "attn":
        dt = DTYPES[c["dtype"]]
        q = _normal(g, (c["b"], c["n"], c["f"], c["h"]), dt)
        k, v = (_normal(g, (c["b"], c["n"], c["t"], c["h"]), dt) for _ in range(2))
        return dict(op=op, q=q, k=k, v=v, out=torch.empty_like(q), causal=c["causal"],
                    bias=_normal(g, (c["b"], c["n"], c["f"], c["t"]), dt) if c["bias"] else None,
                    lse=torch.empty((c["b"] * c["n"], c["f"]), device="cuda") if c["lse"] else None)
    if op == "attn_bwd":
        dt, shape = DTYPES[c["dtype"]], (c["b"], c["n"], c["s"], c["h"])
        q, k, v, d_out = (_normal(g, shape, dt) for _ in range(4))
        out, lse = torch.empty_like(q), torch.empty((c["b"] * c["n"], c["s"]), device="cuda")
        xmk.fmha_forward(q, k, v, out, lse=lse, causal=c["causal"])
        return dict(op=op, q=q, k=k, v=v, out=out, d_out=d_out, lse=lse, causal=c["causal"])
    if op in ("gemm", "gemm_f32"):
        dt = DTYPES[c.get("dtype", "f32")]
        m, n, k = c["m"], c["n"], c["k"]
        a = _normal(g, (m, k), dt, k ** -0.5)
        b = _normal(g, (n, k) if c["rhs_t"] else (k, n), dt)
        out = torch.empty((m, n), device="cuda", dtype=dt)
        need = xmk.gemm_workspace_bytes(a, b, out, rhs_transpose=c["rhs_t"])
        return dict(op=op, a=a, b=b, out=out, rhs_t=c["rhs_t"], epi=EPILOGUES[c["epi"]],
                    bias=_normal(g, (n,), dt) if c["epi"].startswith("bias") else None,
                    ws=torch.empty((need,), device="cuda", dtype=torch.uint8) if need else None)
    if op == "int4":
        m, k, n = c["m"], c["k"], c["n"]
        linears = [_int4_linear(g, k, n, c["group"], c["bias"]) for _ in range(c["layers"])]
        need = xmk.int4_gemm_workspace_bytes(m, k, n)
        return dict(op=op, act=_normal(g, (m, k), torch.float16), linears=linears, group=c["group"],
                    outs=[torch.empty((m, n), device="cuda", dtype=torch.float16) for _ in linears],
                    ws=torch.empty((need,), device="cuda", dtype=torch.uint8) if need else None)
    if op == "fp8":
        m, n, k = c["m"], c["n"], c["k"]
        (a, sa), (b, sb) = _fp8(g, (m, k)), _fp8(g, (n, k) if c["rhs_t"] else (k, n))
        return dict(op=op, a=a, b=b, sa=sa, sb=sb, out=torch.empty((m, n), device="cuda", dtype=torch.bfloat16), rhs_t=c["rhs_t"],
                    bias=_normal(g, (n,), torch.bfloat16, 8.0) if c["bias"] else None,
                    d_scale=torch.full((1,), 0.5, device="cuda") if c["d_scale"] else None)
    if op == "decode":
        n_layer, batch, cap = c["layers"], c["batch"], c["capacity"]
        kv = [_normal(g, (n_layer, batch, HEADS, cap, HEAD_DIM), torch.float16) for _ in range(2)]
        ones, zeros = torch.ones((D_MODEL,), device="cuda").half(), torch.zeros((D_MODEL,), device="cuda").half()
        layers = [dict(ln_gamma=ones, ln_beta=zeros, qkv=_int4_linear(g, D_MODEL, 3 * D_MODEL, GROUP, False),
                       out_proj=_int4_linear(g, D_MODEL, D_MODEL, GROUP, False), fc_in=_int4_linear(g, D_MODEL, D_FF, GROUP, True),
                       fc_out=_int4_linear(g, D_FF, D_MODEL, GROUP, True), k_cache=kv[0][i], v_cache=kv[1][i])
                  for i in range(n_layer)]
        cfg = xmk.GptjConfig(n_layer, HEADS, HEAD_DIM, ROTARY, D_MODEL, D_FF, VOCAB, GROUP, batch, cap, 1e-5)
        dec = xmk.GptjDecoder(cfg, layers, ones, zeros, _int4_linear(g, D_MODEL, VOCAB, GROUP, True))
        return dict(op=op, dec=dec, hidden=_normal(g, (batch, D_MODEL), torch.float16), position=c["position"], kv=kv,
                    logits=torch.empty((batch, VOCAB), device="cuda", dtype=torch.float16))
    raise ValueError(op)


# ------------------------------------------------------------------------------------------------ the calls
def run(s):
    op = s["op"]
    if op == "attn":
        xmk.fmha_forward(s["q"], s["k"], s["v"], s["out"], bias=s["bias"], lse=s["lse"], causal=s["causal"])
        return [s["out"]] if s["lse"] is None else [s["out"], s["lse"]]
    if op == "attn_bwd":
        return xmk.fmha_backward(s["q"], s["k"], s["v"], s["out"], s["d_out"], s["lse"], causal=s["causal"])
    if op in ("gemm", "gemm_f32"):
        return xmk.run_gemm(s["a"], s["b"], s["out"], rhs_transpose=s["rhs_t"], bias=s["bias"], epilogue=s["epi"], workspace=s["ws"])
    if op == "int4":
        for (qw, scales, zeros, bias), out in zip(s["linears"], s["outs"]):
            if s["ws"] is None:
                xmk.int4_gemm(s["act"], qw, scales, zeros, out, group=s["group"], bias=bias)
            else:
                xmk.int4_gemm_ws(s["act"], qw, scales, zeros, out, s["ws"], group=s["group"], bias=bias)
        return s["outs"]
    if op == "fp8":
        return xmk.fp8_gemm(s["a"], s["b"], s["sa"], s["sb"], s["out"], rhs_transpose=s["rhs_t"], d_scale=s["d_scale"], bias=s["bias"])
    s["dec"].step(s["hidden"], s["position"], s["logits"])
    return [s["logits"]] + s["kv"]  # the step appends a row to the caches


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    """Each input read once, each output written once; the operations of the mathematics (causal: half the scores;
    the backward's five products, not the kernels' recomputation)."""
    c, op = case, case["op"]
    if op == "attn":
        units, scores = c["b"] * c["n"], c["f"] * c["t"] * (0.5 if c["causal"] else 1.0)
        return {"bytes": units * (2.0 * (2 * c["f"] + 2 * c["t"]) * c["h"] + (2.0 * scores if c["bias"] else 0.0) + (4.0 * c["f"] if c["lse"] else 0.0)),
                "flops": 4.0 * units * scores * c["h"]}
    if op == "attn_bwd":
        units = c["b"] * c["n"]
        return {"bytes": units * (16.0 * c["s"] * c["h"] + 4.0 * c["s"]),
                "flops": 10.0 * units * c["s"] * c["s"] * c["h"] * (0.5 if c["causal"] else 1.0)}
    if op in ("gemm", "gemm_f32"):
        m, n, k, size = c["m"], c["n"], c["k"], 4.0 if op == "gemm_f32" else 2.0
        return {"bytes": size * (m * k + k * n + m * n + (n if c["epi"].startswith("bias") else 0)), "flops": 2.0 * m * n * k}
    if op == "int4":
        m, k, n = c["m"], c["k"], c["n"]
        each = k * n / 2.0 + 4.0 * (k // c["group"]) * n + 2.0 * m * n + (2.0 * n if c["bias"] else 0.0)
        return {"bytes": c["layers"] * each + 2.0 * m * k, "flops": c["layers"] * 2.0 * m * n * k}
    if op == "fp8":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 1.0 * (m * k + k * n) + 2.0 * m * n + (2.0 * n if c["bias"] else 0.0), "flops": 2.0 * m * n * k}
    params = c["layers"] * (4.0 * D_MODEL * D_MODEL + 2.0 * D_MODEL * D_FF) + D_MODEL * VOCAB
    keys = c["position"] + 1
    kv = c["layers"] * 4.0 * c["batch"] * keys * D_MODEL
    return {"bytes": params * (0.5 + 4.0 / GROUP) + kv + 2.0 * c["batch"] * VOCAB,
            "flops": 2.0 * c["batch"] * params + c["layers"] * 4.0 * c["batch"] * keys * D_MODEL}


def tolerance(case):
    """What the storage types give: results rounded once to 16 bits from fp32 sums; attention rounds the softmax weights
    to 16 bits too; a decode step chains a hundred such roundings."""
    op = case["op"]
    if op == "gemm_f32":
        return {"rel": 1e-5}
    if op in ("attn", "attn_bwd"):
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}
    if op == "gemm":
        return {"rel": 4e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
    if op == "int4":
        return {"rel": 2e-3}
    if op == "fp8":
        return {"rel": 4e-3}
    return {"rel": 5e-3}
