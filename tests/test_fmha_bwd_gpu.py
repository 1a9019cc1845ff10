"""GPU parity: fused attention backward through the C ABI (xmk_fmha_bwd) against the oracle's
float64 closed form (pinned by finite differences in tests/test_oracle_math.py).

Tolerance: error relative to the tensor's scale (oracle.rel_err's first figure) <= 1e-2 as for the
forward outputs.  The elementwise figure (eps = rms(ref)) is held to 1e-2 for fp16 on every shape
(measured maximum 3.9e-3) and, for bf16, to 1.5 times the measured maximum of each group of cases:
8e-2 on the small shapes (measured 5.3e-2) and 1.5e-1 on the shapes with thousands of rows
(measured 9.9e-2: the maximum over 1.5 M elements of a rounding-dominated error sits further out
in the tail).  P, dS and the forward output O (which enters through D = rowsum(dO o O)) are rounded
to the 16-bit operand type before the products that consume them, here as in the reference
(xetla/sdp/fmha_backward.h:195-196); with three mantissa bits fewer than fp16 that rounding is the
bf16 error, largest under a causal mask, where late keys receive few terms, and the same for the
fused kernels and for the GEMM composition (XMK_FMHA_BWD_COMPOSED=1, which test_backward_composition
runs in a child process).  The reference's own attention test allows atol 3e-2 for bf16 and 1e-2 for
fp16 on O(1) outputs (test/jax_ut.patch:997)."""
import numpy as np
import pytest
import torch

from util import to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-2
TOL_ELEM = {"bf16": 8e-2, "fp16": 1e-2}        # small shapes
TOL_ELEM_LARGE = {"bf16": 1.5e-1, "fp16": 1e-2}  # thousands of rows


def _run(xmk, oracle, name, B, N, F, T, H, causal, use_bias, seed=0, tol_elem=None):
    dt = oracle.BF16 if name == "bf16" else oracle.F16
    tdt = torch.bfloat16 if name == "bf16" else torch.float16
    q = oracle.from_f32(oracle.normal((B, N, F, H), seed + 1), dt)
    k = oracle.from_f32(oracle.normal((B, N, T, H), seed + 2), dt)
    v = oracle.from_f32(oracle.normal((B, N, T, H), seed + 3), dt)
    g = oracle.from_f32(oracle.normal((B, N, F, H), seed + 4), dt)
    bias = oracle.from_f32(oracle.normal((B, N, F, T), seed + 5), dt) if use_bias else None
    scale = H ** -0.5
    dq, dk, dv = oracle.fmha_bwd(q, k, v, g, dt, scale, bias=bias, causal=causal)
    kind = "bf16" if name == "bf16" else "f16"
    tq, tk, tv, tg = (to_dev(x, kind) for x in (q, k, v, g))
    tb = None if bias is None else to_dev(bias, kind)
    out = torch.empty_like(tq)
    lse = torch.empty((B * N, F), dtype=torch.float32, device="cuda")
    xmk.fmha_forward(tq, tk, tv, out, bias=tb, lse=lse, causal=causal)
    gq, gk, gv = xmk.fmha_backward(tq, tk, tv, out, tg, lse, bias=tb, causal=causal)
    torch.cuda.synchronize()
    errs = {}
    for nm, got, ref in (("dq", gq, dq), ("dk", gk, dk), ("dv", gv, dv)):
        ge, ee = oracle.rel_err(got.float().cpu().numpy(), ref.astype(np.float32),
                                label=f"fmha_bwd {nm} {name} [{B},{N},{F}x{T},{H}] causal={causal} bias={use_bias}")
        errs[nm] = (ge, ee)
        assert ge <= TOL and ee <= (tol_elem or TOL_ELEM[name]), (nm, ge, ee)
    return errs


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("causal,use_bias", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("F,T,H", [(128, 128, 64), (200, 136, 128), (64, 77, 40), (257, 64, 256)])
def test_backward_shapes(xmk, oracle, name, causal, use_bias, F, T, H):
    _run(xmk, oracle, name, 2, 3, F, T, H, causal, use_bias)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,N,F,T,H", [
    # (not a single key: its softmax is constant, dQ and dK are exactly zero and an error relative to them has no bound)
    (1, 1, 2, 3, 128), (1, 3, 129, 513, 64), (1, 2, 640, 127, 80), (1, 3, 385, 129, 256),  # one grid: passes of different widths
    (96, 4, 64, 65, 64), (96, 4, 33, 128, 128),                                         # the most work-groups it takes
    (97, 4, 65, 64, 64), (97, 4, 128, 40, 128), (43, 3, 32, 64, 256),                   # one more: a launch per pass
])
def test_backward_one_grid_or_three_launches(xmk, oracle, causal, B, N, F, T, H):
    """fp16: few work-groups run all passes as one grid, on statistics formed before; more, a launch per pass."""
    _run(xmk, oracle, "fp16", B, N, F, T, H, causal, False, seed=F + T)


def test_backward_large(xmk, oracle):
    """Many blocks with a bias and a causal mask; the elementwise bound of the large shapes."""
    errs = _run(xmk, oracle, "bf16", 1, 12, 2048, 2048, 64, True, True, seed=9, tol_elem=TOL_ELEM_LARGE["bf16"])
    print(errs)


_COMPOSED_CHILD = """
import sys
sys.path.insert(0, {tests!r}); sys.path.insert(0, {root!r})
import importlib
import oracle
import test_fmha_bwd_gpu as t
xmk = importlib.import_module("intel-extension-for-openxla_amd")
t._run(xmk, oracle, "fp16", 2, 3, 200, 136, 128, True, True)
t._run(xmk, oracle, "bf16", 2, 3, 257, 64, 256, False, False)
# more units than fit one workspace chunk (score buffers are capped at 1 GiB)
t._run(xmk, oracle, "bf16", 1, 12, 2048, 2048, 64, True, False, seed=9, tol_elem=t.TOL_ELEM_LARGE["bf16"])
print("composed ok")
"""


def test_backward_composition():
    """The GEMM composition (the path behind XMK_FMHA_BWD_COMPOSED=1) in a child process, since the
    switch is read once per process: bias, head size 256, and chunking over units."""
    import os
    import subprocess
    import sys
    tests = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, XMK_FMHA_BWD_COMPOSED="1")
    r = subprocess.run([sys.executable, "-c", _COMPOSED_CHILD.format(tests=tests, root=os.path.dirname(tests))],
                       env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "composed ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.parametrize("name,causal", [("bf16", True), ("fp16", False)])
def test_backward_fused_long(xmk, oracle, name, causal):
    """The fused kernels over many blocks in both directions (16 key blocks, 8 owner blocks), ragged
    ends in F and T; the elementwise bound of the large shapes."""
    errs = _run(xmk, oracle, name, 1, 3, 1000, 1016, 128, causal, False, seed=21, tol_elem=TOL_ELEM_LARGE[name])
    print(errs)


def test_backward_errors(xmk):
    q = torch.zeros((1, 1, 8, 64), dtype=torch.float16, device="cuda")
    lse = torch.zeros((1, 8), dtype=torch.float32, device="cuda")
    with pytest.raises(xmk.XmkError) as e:
        xmk.fmha_backward(q.float(), q.float(), q.float(), q.float(), q.float(), lse)
    assert e.value.code == xmk.INTERNAL and "Invalid MHA datatype" in e.value.message
    q2 = torch.zeros((1, 1, 8, 60), dtype=torch.float16, device="cuda")
    with pytest.raises(xmk.XmkError) as e:
        xmk.fmha_backward(q2, q2, q2, q2, q2, lse)
    assert e.value.code == xmk.UNIMPLEMENTED


def test_backward_on_a_side_stream(xmk):
    """The call's scratch belongs to the stream it runs on: tensors made on the current stream while the side stream is
    still busy do not get its memory, and the gradients are those of a call on the current stream."""
    B, N, S, H = 1, 4, 512, 128
    q, k, v, g = (torch.randn((B, N, S, H), device="cuda").bfloat16() for _ in range(4))
    out, lse = torch.empty_like(q), torch.empty((B * N, S), device="cuda")
    xmk.fmha_forward(q, k, v, out, lse=lse, causal=True)
    ref = xmk.fmha_backward(q, k, v, out, g, lse, causal=True)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    a = torch.randn((4096, 4096), device="cuda").bfloat16()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(20):  # keeps the side stream busy for a few milliseconds
            b = torch.empty_like(a)
            xmk.run_gemm(a, a, b)
    got = xmk.fmha_backward(q, k, v, out, g, lse, causal=True, stream=side)
    junk = [torch.full((n,), 0xff, dtype=torch.uint8, device="cuda") for n in (1 << 12, 1 << 16, 1 << 18, 1 << 20, 1 << 22, 1 << 24) for _ in range(4)]
    torch.cuda.synchronize()
    assert len(junk) == 24 and all(torch.equal(x, y) for x, y in zip(got, ref))


def _rows_agree(nm, a, b, ulp):
    """Two ways to the same sums of products of factors that are rounded alike.  Each result is rounded once (one spacing of it,
    `ulp` of its size at most), and a few of the rounded factors may fall on the other side of a rounding boundary (less than as
    much again); what remains of a row whose exact gradients cancel is the noise of 32-bit sums."""
    a, b = a.float(), b.float()
    diff, size = (a - b).norm(dim=-1), a.norm(dim=-1)
    assert torch.isfinite(b).all(), nm
    over = diff - 2 * ulp * size - 1e-5 * a.shape[-1] ** 0.5
    at = int(over.argmax())
    assert over.max().item() <= 0, (nm, at, diff.flatten()[at].item(), size.flatten()[at].item())


@pytest.mark.parametrize("name,causal", [("bf16", True), ("fp16", True), ("fp16", False)])
@pytest.mark.parametrize("B,N,F,T,H,parts", [
    (10, 16, 130, 257, 128, 1), (13, 16, 257, 130, 80, 1), (29, 9, 33, 65, 256, 1), (12, 11, 129, 1, 200, 1), (130, 4, 1, 64, 72, 1),
    (57, 47, 100, 96, 128, 2),
    # whole query blocks: the loads past a unit's last one, and past the last unit's, start where the workspace ends
    (11, 16, 256, 256, 128, 1), (23, 16, 128, 128, 96, 1), (29, 9, 128, 65, 256, 1), (57, 47, 128, 96, 128, 2),
])
def test_backward_with_kept_score_gradients(xmk, name, causal, B, N, F, T, H, parts):
    """dS kept in the workspace (all units at once, or as many as a smaller workspace holds) against a call with the least
    workspace, which forms it twice, row by row; and the units at the ends of the parts against float64."""
    import ctypes as C
    L, tdt = xmk.lib(), torch.bfloat16 if name == "bf16" else torch.float16
    L.xmk_fmha_bwd_best_workspace_bytes.restype = C.c_size_t
    u = [C.c_uint32(x) for x in (B, N, H, F, T)]
    g = torch.Generator(device="cuda")
    g.manual_seed(F * T + H)
    q, d_o = (torch.randn((B, N, F, H), generator=g, device="cuda", dtype=tdt) for _ in range(2))
    k, v = (torch.randn((B, N, T, H), generator=g, device="cuda", dtype=tdt) for _ in range(2))
    out, lse = torch.empty_like(q), torch.empty((B * N, F), device="cuda")
    xmk.fmha_forward(q, k, v, out, lse=lse, causal=causal)
    least = L.xmk_fmha_bwd_workspace_bytes(*u)
    best = L.xmk_fmha_bwd_best_workspace_bytes(*u, C.c_int32(causal))
    assert best > least and (best - least) % (B * N) == 0
    results = []
    for size in (least, least + (best - least) // (B * N) * -(-B * N // parts)):
        ws = torch.full((size,), 0xff, dtype=torch.uint8, device="cuda")
        grads = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        p = [C.c_void_p(x.data_ptr()) for x in (q, k, v, out, d_o, lse, *grads, ws)]
        rc = L.xmk_fmha_bwd(*p[:3], None, *p[3:9], C.c_int32(xmk.BF16 if name == "bf16" else xmk.F16), *u, C.c_float(H ** -0.5),
                            C.c_int32(causal), p[9], C.c_size_t(size), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert rc == 0
        results.append(grads)
    ulp = 2.0 ** (-7 if name == "bf16" else -10)  # relative spacing of the results, and of the dS that enter them, at most
    for nm, a, b in zip(("dq", "dk", "dv"), *results):
        _rows_agree(nm, a, b, ulp)
    each = -(-B * N // parts)
    for unit in {0, each - 1, each % (B * N), B * N - 1}:
        Q, K, V, O, G = (x.flatten(0, 1)[unit].double() for x in (q, k, v, out, d_o))
        S = Q @ K.T * H ** -0.5
        if causal:
            S.masked_fill_(torch.ones_like(S).triu(1).bool(), float("-inf"))
        P = torch.exp(S - lse[unit].double()[:, None])
        dS = P * (G @ V.T - (G * O).sum(1, keepdim=True)) * H ** -0.5
        for nm, got, ref in zip(("dq", "dk", "dv"), results[1], (dS @ K, dS.T @ Q, P.T @ G)):
            err = (got.flatten(0, 1)[unit].double() - ref).abs().max().item()
            assert err <= TOL * max(ref.abs().max().item(), 1e-2), (nm, unit, err)


def test_backward_where_memory_is_short(xmk):
    """The scratch that keeps dS (88 MiB here) is one the call can do without: where there is room for it or for the gradients
    (33 MiB) but not for both, the call runs with the least scratch."""
    B, N, S, H = 1, 44, 1024, 128
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    q, k, v, d_o = (torch.randn((B, N, S, H), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(4))
    out, lse = torch.empty_like(q), torch.empty((B * N, S), device="cuda")
    xmk.fmha_forward(q, k, v, out, lse=lse)
    want = xmk.fmha_backward(q, k, v, out, d_o, lse)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = (S * S * 2 * N) + (8 << 20)
    before = torch.cuda.memory_reserved()
    torch.cuda.set_per_process_memory_fraction((before + room) / torch.cuda.mem_get_info()[1])
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            torch.empty((room + (16 << 20),), dtype=torch.uint8, device="cuda")
        got = xmk.fmha_backward(q, k, v, out, d_o, lse)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    torch.cuda.synchronize()
    assert torch.cuda.memory_reserved() <= before + room
    for nm, a, b in zip(("dq", "dk", "dv"), want, got):
        _rows_agree(nm, a, b, 2.0 ** -7)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,N,F,T,H", [(40, 9, 33, 65, 128), (29, 9, 100, 257, 80), (29, 9, 33, 65, 256)])
def test_backward_infinite_key_without_weight(xmk, causal, B, N, F, T, H):
    """A key with an infinity that no query gives any weight (behind the last query of a causal call, or a score of minus
    infinity for every query) has gradients of zero, also where dS is kept and the last tile of queries is not full."""
    import ctypes as C
    L = xmk.lib()
    u = [C.c_uint32(x) for x in (B, N, H, F, T)]
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    q, d_o = (torch.randn((B, N, F, H), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    k, v = (torch.randn((B, N, T, H), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    key = T - 3
    q[..., 5] = q[..., 5].abs() + 0.5
    k[:, :, key, 5] = float("inf") if causal else float("-inf")
    out, lse = torch.empty_like(q), torch.empty((B * N, F), device="cuda")
    xmk.fmha_forward(q, k, v, out, lse=lse, causal=causal)
    assert L.xmk_fmha_bwd_best_workspace_bytes(*u, C.c_int32(causal)) > L.xmk_fmha_bwd_workspace_bytes(*u)
    _, dk, dv = xmk.fmha_backward(q, k, v, out, d_o, lse, causal=causal)
    assert torch.isfinite(out).all() and torch.isfinite(dk).all() and torch.isfinite(dv).all()
    assert not dk[:, :, key].any() and not dv[:, :, key].any()


@pytest.mark.parametrize("causal,use_bias", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("name,B,N,F,T,H", [
    ("bf16", 1, 3, 130, 203, 72), ("fp16", 1, 3, 203, 130, 96), ("fp16", 1, 3, 97, 257, 136), ("bf16", 1, 3, 257, 97, 160), ("fp16", 1, 2, 130, 131, 168),
    ("bf16", 29, 9, 33, 65, 96), ("bf16", 40, 9, 33, 65, 96), ("fp16", 29, 9, 65, 33, 160),  # dS kept: the last two
])
def test_backward_head_size_classes(xmk, oracle, name, causal, use_bias, B, N, F, T, H):
    """Classes of head sizes at their last size and just past the one below, ragged in F and T, in one grid, with dS kept and
    (with a bias) in launches of their own."""
    _run(xmk, oracle, name, B, N, F, T, H, causal, use_bias, seed=9)


@pytest.mark.parametrize("B,N,F,T,H", [(29, 9, 33, 65, 160), (9, 17, 257, 130, 136), (130, 4, 64, 33, 96)])
def test_backward_with_kept_score_gradients_head_size_classes(xmk, B, N, F, T, H):
    test_backward_with_kept_score_gradients(xmk, "bf16", True, B, N, F, T, H, 1)
