"""GPU parity: int4 dequantisation (bit-exact) and the int4 weight-only GEMM, through the C ABI."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from util import to_bits, to_dev

pytestmark = pytest.mark.gpu


def _case(oracle, m, k, n, group, seed):
    qw = oracle.words((k // 8, n), seed)
    s = oracle.from_f32(oracle.uniform((k // group, n), seed + 1, 0.001, 0.02), oracle.F16)
    z = oracle.from_f32(oracle.uniform((k // group, n), seed + 2, 0.0, 15.0), oracle.F16)
    act = oracle.from_f32(oracle.normal((m, k), seed + 3), oracle.F16)
    return act, qw, s, z


@pytest.mark.parametrize("k,n,group", [(4096, 16384, 128), (256, 64, 32), (512, 1024, 64), (1024, 200, 256)])
def test_int4_dequant_bit_exact(xmk, oracle, k, n, group):
    _, qw, s, z = _case(oracle, 1, k, n, group, 100 + n)
    ref = oracle.int4_dequant(qw, s, z, group)
    w = torch.empty((k, n), dtype=torch.float16, device="cuda")
    xmk.int4_dequant(to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16"), w, group=group)
    torch.cuda.synchronize()
    assert np.array_equal(to_bits(w), ref)


@pytest.mark.parametrize("m", [1, 8, 32])
def test_int4_gemm_gptj_mlp_shape(xmk, oracle, m):
    """benchmark configuration 3: K=4096, N=16384, group 128, M in {1, 8, 32}; <= 1e-2 vs fp32 recompute."""
    k, n, group = 4096, 16384, 128
    act, qw, s, z = _case(oracle, m, k, n, group, 7)
    _, ref = oracle.int4_gemm(act, qw, s, z, group)
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    xmk.int4_gemm(to_dev(act, "f16"), to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16"), out,
                  group=group)
    torch.cuda.synchronize()
    g, e = oracle.rel_err(out.float().cpu().numpy(), ref)
    print(f"int4 m={m}: max|d|/max|ref|={g:.2e} elementwise={e:.2e}")
    assert g <= 1e-2 and e <= 1e-2
    # against act @ fp16-rounded weights the difference is the weights' fp16 rounding only
    _, ref16 = oracle.int4_gemm(act, qw, s, z, group, round_weights=True)
    assert oracle.rel_err(out.float().cpu().numpy(), ref16)[0] <= 1e-2


@pytest.mark.parametrize("m,k,n,group,with_bias", [
    (1, 4096, 4096, 128, False),    # attention projections of the decode step (narrow-N path)
    (4, 4096, 4096, 128, False),
    (4, 16384, 4096, 128, True),    # fc_out
    (3, 256, 8, 32, True),          # smallest legal N
    (17, 512, 200, 64, True),       # ragged N (not a multiple of the block's columns), two row tiles
    (33, 256, 72, 256, False),      # M > 32: second launch
    (16, 1024, 1024, 128, True),
    (2, 512, 136, 128, True),       # 2-4 rows and 5-8 rows take the variants that feed the rows spread out
    (6, 1024, 200, 64, False),
    (7, 4096, 4096, 128, True),
    (36, 256, 72, 32, True),        # 32 rows + 4 in a second launch
    (40, 512, 264, 128, False),     # 32 rows + 8
    # 9 to 32 rows (one or two 16-row tiles per wave), group sizes 32 to 128
    (12, 1024, 1024, 32, True),     # one row tile, group 32
    (9, 512, 200, 64, False),       # ragged N
    (25, 16384, 264, 128, True),    # 16 groups per wave
    (32, 8192, 1024, 64, False),
    (20, 256, 72, 128, False),      # fewer groups than waves
    (31, 640, 136, 128, True),      # 5 groups: waves with one group and waves with none
    (48, 4096, 1024, 128, True),    # 32 rows + 16 in a second launch
    # more than eight groups per wave: the straight-line part is followed by the loop, which ends on an
    # odd count (9 and 11 groups per wave) and after one group of the loop (9)
    (10, 9216, 264, 128, True), (5, 5632, 136, 64, False), (30, 9216, 72, 128, False),
    # more than 256 column blocks with 2 to 16 rows: four-wave work-groups (ragged last block; 9 groups over 4 waves)
    (4, 512, 16640, 128, True), (12, 256, 16448, 64, False), (6, 1152, 16400, 128, True), (3, 128, 16392, 32, False),
    # 16 groups per wave with the activations staged through LDS (eight-wave and four-wave forms): the reads of
    # both staging buffers inside the loop have to wait for their loads
    (32, 16384, 1024, 128, False), (6, 8192, 16400, 128, True),
    # groups of 256 channels run as two batches of 128 with the same scale and zero point
    (1, 2048, 512, 256, True), (8, 1024, 264, 256, False), (32, 4096, 256, 256, True), (4, 4096, 4096, 256, False),
])
def test_int4_gemm_shapes(xmk, oracle, m, k, n, group, with_bias):
    act, qw, s, z = _case(oracle, m, k, n, group, 1000 + m + n)
    bias = oracle.from_f32(oracle.normal((n,), 55), oracle.F16) if with_bias else None
    _, ref = oracle.int4_gemm(act, qw, s, z, group, bias=bias)
    out = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
    xmk.int4_gemm(to_dev(act, "f16"), to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16"), out,
                  group=group, bias=None if bias is None else to_dev(bias, "f16"))
    torch.cuda.synchronize()
    g, e = oracle.rel_err(out.float().cpu().numpy(), ref)
    assert g <= 1e-2 and e <= 1e-2, (g, e)


def test_int4_gemm_linearity_full_size(xmk, oracle):
    """Size-independent property at the full shape: f(a1 + a2) == f(a1) + f(a2) within rounding."""
    k, n, group = 4096, 16384, 128
    _, qw, s, z = _case(oracle, 1, k, n, group, 7)
    dq, ds, dz = to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16")
    a1 = torch.randn((8, k), device="cuda").half()
    a2 = torch.randn((8, k), device="cuda").half()
    a3 = (a1.float() + a2.float()).half()
    outs = []
    for a in (a1, a2, a3):
        o = torch.empty((8, n), dtype=torch.float16, device="cuda")
        xmk.int4_gemm(a, dq, ds, dz, o, group=group)
        outs.append(o.float())
    torch.cuda.synchronize()
    err = (outs[2] - outs[0] - outs[1]).abs().max().item() / outs[2].abs().max().item()
    assert err < 1e-2


@pytest.mark.parametrize("m,k,n,group,with_bias,dense", [(256, 512, 1024, 128, True, False), (200, 1024, 328, 64, False, False),
                                                          (2000, 1024, 1032, 32, True, True)])
def test_int4_gemm_many_rows_with_scratch(xmk, oracle, m, k, n, group, with_bias, dense):
    """Prompt-sized row counts: with the scratch xmk_int4_gemm_workspace_bytes asks for, the row tiles run or,
    with enough rows, the weights are dequantised into it once and the dense fp16 GEMM runs; without it the row
    tiles run.  All within 1e-2 of the fp32 recompute, and of the recompute from fp16-rounded weights."""
    act, qw, s, z = _case(oracle, m, k, n, group, 2000 + m)
    bias = oracle.from_f32(oracle.normal((n,), 56), oracle.F16) if with_bias else None
    _, ref = oracle.int4_gemm(act, qw, s, z, group, bias=bias)
    _, ref16 = oracle.int4_gemm(act, qw, s, z, group, bias=bias, round_weights=True)
    need = xmk.int4_gemm_workspace_bytes(m, k, n)
    assert need == k * n * 2
    assert xmk.int4_gemm_workspace_bytes(32, k, n) == 0   # decode-sized calls never ask for scratch
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device="cuda")
    dev = [to_dev(act, "f16"), to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16")]
    dbias = None if bias is None else to_dev(bias, "f16")
    outs = []
    for scratch in (ws, None):
        out = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
        xmk.int4_gemm_ws(*dev, out, scratch, group=group, bias=dbias)
        torch.cuda.synchronize()
        for r in (ref, ref16):
            g, e = oracle.rel_err(out.float().cpu().numpy(), r)
            assert g <= 1e-2 and e <= 1e-2, (scratch is not None, g, e)
        outs.append(out.float())
    assert bool((ws != 0xff).any()) == dense
    assert (outs[0] - outs[1]).abs().max().item() <= 1e-2 * outs[1].abs().max().item()


@pytest.mark.parametrize("m,k,n,group", [
    # 32-row tiles, eight waves on one reduction: one row past a tile, one column block, odd step count, every group size
    (41, 1056, 72, 32), (64, 3136, 136, 64), (65, 4096, 1000, 128), (96, 2304, 64, 256),
    # the same with four waves: a single step (and less than one), more than one round of work-groups
    (41, 32, 8, 32), (49, 512, 200, 64), (70, 1024, 8200, 128), (67, 768, 6152, 256),
    # 64 rows x 128 columns on eight and on four waves
    (128, 640, 16328, 128), (97, 768, 16264, 256), (128, 1056, 16328, 32), (100, 1088, 16384, 64),
    (255, 512, 16392, 256), (200, 384, 4000, 128), (250, 480, 8000, 32), (130, 320, 9000, 64),
    # 64 rows x 256 columns
    (310, 128, 16400, 128), (300, 256, 16400, 256), (257, 224, 16400, 32), (383, 192, 16328, 64),
])
def test_int4_gemm_row_tiles(xmk, oracle, m, k, n, group):
    """Products of more than 32 rows, without scratch: every tile shape at the edges of its rows, columns and steps.
    The error is the output's rounding, 2^-11 of a value, plus that of the fp32 sums: a group's sum of a (16 + q)
    stays below 31 * 4 sqrt(group), is rounded eight times per 128 k and scaled by up to 0.02, and the K / group
    groups' errors add like noise."""
    act, qw, s, z = _case(oracle, m, k, n, group, 3000 + m + n)
    bias = oracle.from_f32(oracle.normal((n,), 57), oracle.F16) if m % 2 else None
    _, ref = oracle.int4_gemm(act, qw, s, z, group, bias=bias)
    guard = 64  # rows before and behind the result stay as they were
    out = torch.full((m + 2 * guard, n), 7.0, dtype=torch.float16, device="cuda")
    xmk.int4_gemm(to_dev(act, "f16"), to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16"), out[guard:guard + m],
                  group=group, bias=None if bias is None else to_dev(bias, "f16"))
    torch.cuda.synchronize()
    got = out[guard:guard + m].float().cpu().numpy()
    ref = np.asarray(ref, np.float32).reshape(m, n)
    assert np.all(np.abs(got - ref) <= np.abs(ref) * 2.0 ** -11 + 2.0 ** -24 * 31 * 4 * k ** 0.5 * 8 * 0.02)
    assert bool((out[:guard] == 7).all()) and bool((out[guard + m:] == 7).all())


@pytest.mark.parametrize("m,k,n,group", [(64, 4096, 512, 32), (128, 4096, 8200, 64), (64, 8192, 1024, 128),
                                         (300, 4096, 16328, 128), (96, 4096, 1024, 256)])
def test_int4_gemm_row_tiles_keep_the_direct_kernel_s_precision(xmk, m, k, n, group):
    """Activations of one sign and zero points near the weights' mean: the sums of a and of a q are large and all but cancel,
    so an offset that stays on the weights until the end of a chain costs bits of the result.  Against 64 bits the row
    tiles may be no further off than the kernel for 32 rows and fewer; the 1 % is ten times the noise of a norm over the
    m n > 30000 rounding errors of each."""
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    act = torch.randn((m, k), generator=g, device="cuda").abs().half()
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    s = torch.empty((k // group, n), device="cuda", dtype=torch.float16).uniform_(0.001, 0.02, generator=g)
    z = torch.empty_like(s).uniform_(7.0, 8.0, generator=g)
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((qw[:, None, :] >> shifts[None, :, None]) & 15).reshape(k, n).double()
    rows = torch.arange(k, device="cuda") // group
    ref = act.double() @ ((q - z[rows].double()) * s[rows].double())
    tiles, direct = (torch.empty((m, n), dtype=torch.float16, device="cuda") for _ in range(2))
    xmk.int4_gemm(act, qw, s, z, tiles, group=group)
    for m0 in range(0, m, 32):
        xmk.int4_gemm(act[m0:m0 + 32], qw, s, z, direct[m0:m0 + 32], group=group)
    err, bound = (((x.double() - ref).norm() / ref.norm()).item() for x in (tiles, direct))
    print(f"int4 row tiles {m}x{k}x{n} group {group}: error {err:.3e}, direct kernel {bound:.3e}")
    assert err <= 1.01 * bound


@pytest.mark.parametrize("m,k,n,group", [(64, 256, 200, 32), (70, 1024, 8200, 128), (128, 640, 16328, 64), (100, 256, 16384, 256),
                                         (310, 128, 16400, 128)])
def test_int4_gemm_row_tiles_single_products(xmk, m, k, n, group):
    """Rows with one activation that is not zero, from the smallest subnormal to the largest finite value: with scale 1 and
    zero point 0 a result is one rounded product, so the weights' form in the matrix cores is exact up to the row sum that is taken
    off it: 16 a and 16 a + q a are both exact in fp32, and so is their difference."""
    g = torch.Generator(device="cuda").manual_seed(m)
    bits = torch.linspace(0, 0x7bff, m, device="cuda").to(torch.int16)
    bits[:7] = torch.tensor([1, 2, 3, 0x3fe, 0x3ff, 0x400, 0x401], dtype=torch.int16)
    values = bits.view(torch.float16) * torch.where(torch.arange(m, device="cuda") % 3 == 0, -1.0, 1.0).half()
    at = torch.randint(0, k, (m,), generator=g, device="cuda")
    act = torch.zeros((m, k), device="cuda", dtype=torch.float16)
    act[torch.arange(m, device="cuda"), at] = values
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    s = torch.ones((k // group, n), device="cuda", dtype=torch.float16)
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    xmk.int4_gemm(act, qw, s, torch.zeros_like(s), out, group=group)
    q = (qw[at // 8] >> (4 * (at % 8)).int()[:, None]) & 15
    assert torch.equal(out, (values.double()[:, None] * q.double()).half())


def test_int4_gemm_row_tiles_keep_rows_apart(xmk, oracle):
    """An infinity in one row of the activations reaches no other row, also where a step reaches past the end of K."""
    m, k, n, group = 70, 160, 200, 32
    act, qw, s, z = _case(oracle, m, k, n, group, 77)
    a = to_dev(act, "f16")
    outs = []
    for bad in (False, True):
        b = a.clone()
        if bad:
            b[41, 0] = float("inf")
        out = torch.empty((m, n), dtype=torch.float16, device="cuda")
        xmk.int4_gemm(b, to_dev(qw, "u32"), to_dev(s, "f16"), to_dev(z, "f16"), out, group=group)
        torch.cuda.synchronize()
        outs.append(out)
    keep = [i for i in range(m) if i != 41]
    assert torch.equal(outs[0][keep], outs[1][keep])


@pytest.mark.parametrize("m,k,n,group,with_ws", [
    (65, 1056, 72, 32, False), (70, 1024, 8200, 128, False), (128, 640, 16328, 128, True), (255, 512, 16392, 256, True),
    (310, 128, 16400, 64, True), (96, 2304, 64, 256, True),
    (2000, 1024, 1032, 32, True)])  # (the dense product)
def test_int4_gemm_row_tiles_infinite_activations(xmk, m, k, n, group, with_ws):
    """Rows with infinite activations: infinities of the products' signs, NaN where a weight is zero or two products cancel,
    as weight by weight (which the dense product on the dequantised weights gives too).  Integer zero points, so that a
    sixteenth of the weights is zero.  The other rows are as they are without them."""
    g = torch.Generator(device="cuda").manual_seed(m)
    act = torch.randn((m, k), generator=g, device="cuda").half()
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    s = torch.empty((k // group, n), device="cuda", dtype=torch.float16).uniform_(0.001, 0.02, generator=g)
    z = torch.randint(0, 16, s.shape, generator=g, device="cuda").half()
    bias = torch.randn((n,), generator=g, device="cuda").half()
    bad = act.clone()
    at = {3: [(0, 1.0)], 33: [(k - 1, -1.0)], m - 1: [(7, 1.0), (k // 2, 1.0)], 40: [(k // 2 + 5, float("nan"))],
          41: [(i, 1.0) for i in range(k)]}
    for row, entries in at.items():
        for i, v in entries:
            bad[row, i] = v * float("inf")
    ws = torch.empty((max(1, xmk.int4_gemm_workspace_bytes(m, k, n)),), dtype=torch.uint8, device="cuda") if with_ws else None
    outs = []
    for a in (act, bad):
        outs.append(torch.empty((m, n), dtype=torch.float16, device="cuda"))
        xmk.int4_gemm_ws(a, qw, s, z, outs[-1], ws, group=group, bias=bias)
    keep = torch.tensor([i for i in range(m) if i not in at], device="cuda")
    assert torch.equal(outs[0][keep], outs[1][keep])
    for row, entries in at.items():
        i = torch.tensor([e[0] for e in entries], device="cuda")
        q = ((qw[i // 8] >> (4 * (i % 8)).int()[:, None]) & 15).float()
        ref = (bad[row, i].float()[:, None] * ((q - z[i // group].float()) * s[i // group].float())).sum(0)
        got = outs[1][row]
        assert torch.equal(got.isnan(), ref.isnan()), row
        assert torch.equal(got[~ref.isnan()], ref[~ref.isnan()].half()), row


def test_int4_forced_tile_takes_every_row_count():
    """XMK_INT4_TILE (read once per process) keeps int4_gemm_kernel and its forced tile where the row tiles would run."""
    program = """
import importlib, torch
xmk = importlib.import_module("intel-extension-for-openxla_amd")
a = torch.ones((64, 256), device="cuda", dtype=torch.float16)
qw = torch.full((32, 128), 0x33333333, device="cuda", dtype=torch.int32)
s = torch.ones((2, 128), device="cuda", dtype=torch.float16)
out = torch.zeros((64, 128), device="cuda", dtype=torch.float16)
xmk.int4_gemm(a, qw, s, s, out, group=128)
assert bool((out == 512).all())
"""
    for forced in (None, "2,8"):
        env = dict(os.environ, XMK_TRACE="1")
        env.pop("XMK_INT4_TILE", None)
        if forced:
            env["XMK_INT4_TILE"] = forced
        r = subprocess.run([sys.executable, "-c", program], env=env, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr
        assert ("row tiles" in r.stderr) == (forced is None) and ("words_per_lane=2 waves=8" in r.stderr) == (forced is not None), r.stderr


def test_int4_errors(xmk):
    a = torch.zeros((1, 256), dtype=torch.float16, device="cuda")
    qw = torch.zeros((32, 64), dtype=torch.int32, device="cuda")
    sz = torch.zeros((2, 64), dtype=torch.float16, device="cuda")
    out = torch.zeros((1, 64), dtype=torch.float16, device="cuda")
    with pytest.raises(xmk.XmkError) as e:
        xmk.int4_gemm(a, qw, sz, sz, out, group=100)
    assert e.value.code == xmk.INVALID_ARGUMENT
    with pytest.raises(xmk.XmkError) as e:
        xmk.int4_gemm(a, qw, sz, sz, out, group=8)
    assert e.value.code == xmk.UNIMPLEMENTED
    # the same contract on the dense path
    a2 = torch.zeros((256, 256), dtype=torch.float16, device="cuda")
    out2 = torch.zeros((256, 64), dtype=torch.float16, device="cuda")
    ws = torch.empty((xmk.int4_gemm_workspace_bytes(256, 256, 64),), dtype=torch.uint8, device="cuda")
    with pytest.raises(xmk.XmkError) as e:
        xmk.int4_gemm_ws(a2, qw, sz, sz, out2, ws, group=8)
    assert e.value.code == xmk.UNIMPLEMENTED


@pytest.mark.parametrize("m", [1, 3, 7, 16, 20])
@pytest.mark.parametrize("n", [8, 232, 240, 256, 272, 504, 1032, 4096, 4104, 4608, 8192, 8200])
def test_int4_gemm_every_block_once(xmk, m, n):
    """Numbers of column blocks on both sides of the lines between block widths, and of sixteen: whole numbers with scale 1 and
    zero point 0, whose sums (below 64 * 15) fp16 holds exactly."""
    k, group = 64, 32
    g = torch.Generator(device="cuda").manual_seed(n + m)
    act = torch.randint(-1, 2, (m, k), generator=g, device="cuda").half()
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    s, z = torch.ones((k // group, n), device="cuda").half(), torch.zeros((k // group, n), device="cuda").half()
    out = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float16)
    xmk.int4_gemm(act, qw, s, z, out, group=group)
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((qw[:, None, :] >> shifts[None, :, None]) & 15).reshape(k, n)
    assert torch.equal(out.double().cpu(), act.double().cpu() @ q.double().cpu())


@pytest.mark.parametrize("m,k,n,group", [(65, 1056, 72, 32), (128, 640, 16328, 128), (64, 768, 200, 64), (310, 512, 16400, 64), (49, 512, 200, 128)])
def test_int4_gemm_row_tiles_infinite_scales(xmk, m, k, n, group):
    """Infinite and NaN scales and zero points: their columns come out as from the kernel for 32 rows and fewer, which forms a
    group's difference of sums before it is scaled (groups of 256 in two parts, whose infinities may cancel: left out); the other
    columns are as they are without them."""
    g = torch.Generator(device="cuda").manual_seed(m + k)
    act = torch.randn((m, k), generator=g, device="cuda").half()
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    s = torch.empty((k // group, n), device="cuda", dtype=torch.float16).uniform_(0.001, 0.02, generator=g)
    z = torch.empty_like(s).uniform_(0.0, 15.0, generator=g)
    plain = torch.empty((m, n), dtype=torch.float16, device="cuda")
    xmk.int4_gemm(act, qw, s, z, plain, group=group)
    inf = float("inf")
    s[0, 3], s[k // group - 1, 8], s[1, 20], z[1, 33], z[0, 40] = inf, -inf, float("nan"), inf, -inf
    bad = [3, 8, 20, 33, 40]
    tiles, direct = torch.empty_like(plain), torch.empty_like(plain)
    xmk.int4_gemm(act, qw, s, z, tiles, group=group)
    for m0 in range(0, m, 32):
        xmk.int4_gemm(act[m0:m0 + 32], qw, s, z, direct[m0:m0 + 32], group=group)
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[bad] = False
    assert torch.equal(tiles[:, keep], plain[:, keep])
    assert not bool(direct[:, bad].isfinite().any())
    assert torch.equal(tiles[:, bad].nan_to_num(nan=7.0), direct[:, bad].nan_to_num(nan=7.0))


@pytest.mark.parametrize("m,k,n,group", [(65, 1056, 72, 32), (64, 768, 200, 64), (49, 512, 200, 128), (310, 512, 16400, 64), (70, 1024, 136, 256)])
def test_int4_gemm_row_tiles_infinite_scales_without_a_sum(xmk, m, k, n, group):
    """Infinite scales on differences of zero (rows of zero activations, groups whose weights are their zero points) and on groups
    whose infinities have opposite signs: NaN.  Whole numbers, so that every sum is exact, against the formula group by group (in
    parts of 128, as the products are formed), which the kernel for 32 rows and fewer gives too."""
    g = torch.Generator(device="cuda").manual_seed(m + k)
    act = torch.randint(-3, 4, (m, k), generator=g, device="cuda").half()
    act[[0, 33, m - 1]] = 0
    act[5, :group] = 0
    qw = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device="cuda", dtype=torch.int32)
    qw[group // 8:2 * group // 8, 12] = 0x44444444
    s = torch.full((k // group, n), 0.5, device="cuda", dtype=torch.float16)
    z = torch.randint(0, 16, s.shape, generator=g, device="cuda").half()
    z[1, 12] = 4
    inf = float("inf")
    s[0, 3] = s[1, 12] = s[0, 20] = s[1, 20] = s[0, 41] = s[0, 50] = s[0, 51] = inf
    s[1, 41] = s[k // group - 1, 60] = -inf
    z[1, 50], z[0, 51], z[1, 61] = -inf, inf, inf
    bias = torch.randint(-3, 4, (n,), generator=g, device="cuda").half()
    out, few = (torch.empty((m, n), dtype=torch.float16, device="cuda") for _ in range(2))
    xmk.int4_gemm(act, qw, s, z, out, group=group, bias=bias)
    for m0 in range(0, m, 32):
        xmk.int4_gemm(act[m0:m0 + 32], qw, s, z, few[m0:m0 + 32], group=group, bias=bias)
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((qw[:, None, :] >> shifts[None, :, None]) & 15).reshape(k, n).double().cpu()
    a, s, z, ref = act.double().cpu(), s.double().cpu(), z.double().cpu(), bias.double().cpu().expand(m, n)
    part = min(group, 128)
    for k0 in range(0, k, part):
        rows, gr = slice(k0, k0 + part), k0 // group
        diff = a[:, rows] @ q[rows] - a[:, rows].sum(1, keepdim=True) * z[gr]
        ref = ref + diff * s[gr]
    ref = ref.half()
    assert bool(ref[:, [3, 12, 20, 41]].isnan().any(0).all()) and bool(ref[:, [3, 20, 41]].isinf().any(0).all())
    for got in (out.cpu(), few.cpu()):
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.nan_to_num(nan=7.0), ref.nan_to_num(nan=7.0))
