"""Output forms of the bf16 ping-pong GEMM (gemm_pp.hip): every op with every operand type, one and two
accumulators, on 128-, 192- and 256-row tiles, against float64 of the same bf16 operands."""

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

# K % 64 != 0: the direct-to-LDS loops need whole 64-deep steps, so these run on the ping-pong kernel.
# Rows: 128-row tiles with a remainder inside a subtile; 192 and 256 rows where whole rounds of them are cheaper.
SIZES = [(301, 136), (8171, 136), (16371, 136)]


def _rel(a, b):
    return float((a.double() - b).abs().max() / b.abs().max())


def _gemm(M, N, K, n_acc, outs, gpu, seed, scaled, **kw):
    from torch_helion.hip import ops

    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
    ws = [(torch.randn(K, N, generator=g, device=gpu) * 0.1).bfloat16() for _ in range(n_acc)]
    if scaled:
        kw.update(sumsq=True, rscale_mask=(1 << n_acc) - 1, inv_k=1.0 / K, eps=1e-5)
    ops.gemm(ops.GemmCall(M, N, K, n_acc, x, ops.pack_rhs(ws, torch.bfloat16), outs, **kw))
    torch.cuda.synchronize()
    xd = x.double()
    r = torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) if scaled else 1.0
    return [(xd @ w.double()) * r for w in ws]


def _rope_ref(acc, part, cos, sin, period):
    M, N = acc.shape
    hd = cos.shape[1]
    rows = torch.arange(M, device=acc.device) % period
    c, s = cos.double()[rows].repeat(1, N // hd), sin.double()[rows].repeat(1, N // hd)
    if part is None:
        h = acc.view(M, N // hd, hd)
        part = torch.cat((-h[..., hd // 2:], h[..., :hd // 2]), -1).reshape(M, N)
    return acc * c + part * s


def _same_bits(o16, o32):
    bad = o16 != o32.bfloat16()
    assert not bad.any(), f"{int(bad.sum())} differ, first at {bad.nonzero()[0].tolist()}, by up to " \
        f"{float((o16.float() - o32).abs()[bad].max())}"


# fp32 outputs: K = 136 products of bf16 values are exact in fp32, their sum rounds at most K times by 2^-24 of
# the magnitudes' sum (about 12 times the root-mean-square here): 136 * 12 * 2^-24 = 1e-4 of the largest at the
# very worst, 1e-6 in practice. Softplus uses the hardware exp and log (1 ulp of terms of order 1).
TOL = 1e-5


@pytest.mark.parametrize("M,K", SIZES)
@pytest.mark.parametrize("op", ["ADD", "SOFTPLUS_ADD", "MUL"])
@pytest.mark.parametrize("n_acc,a,xdt", [(1, 0, torch.bfloat16), (1, 0, torch.float32), (2, 1, torch.bfloat16),
                                         (2, 0, torch.float32)])
def test_extra_operand(gpu, M, K, op, n_acc, a, xdt):
    from torch_helion.hip import abi, ops

    N = 2048 if n_acc == 1 else 1024
    announce(f"gemm pp {op} M={M} N={N} K={K} n_acc={n_acc} a={a} {xdt}")
    code = getattr(abi, f"EPI_{op}")
    g = torch.Generator(device=gpu).manual_seed(M + a)
    x = torch.randn(M, N, generator=g, device=gpu).to(xdt)
    xw = torch.randn(M, 264, generator=g, device=gpu).to(xdt)
    o16, o32 = torch.empty(M, N, dtype=torch.bfloat16, device=gpu), torch.empty(M, N, device=gpu)
    lone = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    win = torch.full((M, 264), 7.0, device=gpu)  # a window that starts and ends inside tiles, its own operand
    w0 = N - 264 - 8
    outs = [ops.EpiSpec(code, o16, a=a, e=0), ops.EpiSpec(code, o32, a=a, e=0),
            ops.EpiSpec(code, win, a=a, e=1, cols=(w0, w0 + 264)), ops.EpiSpec(code, lone, a=a, e=0)]
    acc = _gemm(M, N, K, n_acc, outs, gpu, M, True, extras=[x, xw])[a]

    def ref(v, e):
        e = e.double()
        return v * e if op == "MUL" else torch.nn.functional.softplus(v + e) if op == "SOFTPLUS_ADD" else v + e

    assert _rel(o32, ref(acc, x)) < TOL
    _same_bits(o16, o32)
    assert torch.equal(lone, o16)
    assert _rel(win, ref(acc[:, w0:w0 + 264], xw)) < TOL


@pytest.mark.parametrize("M,K", SIZES)
@pytest.mark.parametrize("hd,period", [(64, 100), (128, 7), (256, 4096)])
def test_rope(gpu, M, K, hd, period):
    """Heads of 64, 128 and 256 (a whole tile), tables shorter than 16 rows, than M, and longer."""
    from torch_helion.hip import abi, ops

    N = 2048
    announce(f"gemm pp rope M={M} N={N} K={K} hd={hd} period={period}")
    g = torch.Generator(device=gpu).manual_seed(hd)
    cos, sin = torch.randn(period, hd, generator=g, device=gpu), torch.randn(period, hd, generator=g, device=gpu)
    q16, q32 = torch.empty(M, 1536, dtype=torch.bfloat16, device=gpu), torch.empty(M, 1536, device=gpu)
    v16 = torch.empty(M, 512, dtype=torch.bfloat16, device=gpu)
    outs = [ops.EpiSpec(abi.EPI_ROPE, q16, cols=(0, 1536)), ops.EpiSpec(abi.EPI_ROPE, q32, cols=(0, 1536)),
            ops.EpiSpec(abi.EPI_ACC, v16, cols=(1536, 2048))]
    acc, = _gemm(M, N, K, 1, outs, gpu, M, True, rope_cos=cos, rope_sin=sin, rope_head_dim=hd, rope_period=period)
    assert _rel(q32, _rope_ref(acc, None, cos, sin, period)[:, :1536]) < TOL
    _same_bits(q16, q32)
    assert _rel(v16, acc[:, 1536:]) < 2.0**-8


@pytest.mark.parametrize("M,K", SIZES)
@pytest.mark.parametrize("hd", [64, 128])
def test_two_accumulators_rope(gpu, M, K, hd):
    """k and v as two accumulators (a wave holds whole heads of one), v through SILU; and ROPE_PAIR, whose partner
    values are the second accumulator, beside an ACC output of that one."""
    from torch_helion.hip import abi, ops

    N, period = 1024, 50
    announce(f"gemm pp two-accumulator rope M={M} N={N} K={K} hd={hd}")
    g = torch.Generator(device=gpu).manual_seed(hd)
    cos, sin = torch.randn(period, hd, generator=g, device=gpu), torch.randn(period, hd, generator=g, device=gpu)
    kw = dict(rope_cos=cos, rope_sin=sin, rope_head_dim=hd, rope_period=period)

    def empty(dt):
        return torch.empty(M, N, dtype=dt, device=gpu)

    k32, k16, v32 = empty(torch.float32), empty(torch.bfloat16), empty(torch.float32)
    acc = _gemm(M, N, K, 2, [ops.EpiSpec(abi.EPI_ROPE, k16, a=0), ops.EpiSpec(abi.EPI_ROPE, k32, a=0),
                             ops.EpiSpec(abi.EPI_SILU, v32, a=1)], gpu, M, True, **kw)
    assert _rel(k32, _rope_ref(acc[0], None, cos, sin, period)) < TOL
    _same_bits(k16, k32)
    assert _rel(v32, torch.nn.functional.silu(acc[1])) < TOL
    p32, p16, a32 = empty(torch.float32), empty(torch.bfloat16), empty(torch.float32)
    acc = _gemm(M, N, K, 2, [ops.EpiSpec(abi.EPI_ROPE_PAIR, p32, a=0, b=1), ops.EpiSpec(abi.EPI_ACC, a32, a=1),
                             ops.EpiSpec(abi.EPI_ROPE_PAIR, p16, a=0, b=1)], gpu, M, False, **kw)
    assert _rel(p32, _rope_ref(acc[0], acc[1], cos, sin, period)) < TOL
    _same_bits(p16, p32)
    assert _rel(a32, acc[1]) < TOL


@pytest.mark.parametrize("n_acc", [1, 2])
def test_in_place_residual(gpu, n_acc):
    """The residual operand's own buffer as the output: rows are read before they are written, 256-row tiles and a
    ragged end included."""
    from torch_helion.hip import abi, ops

    M, N, K = 4099, 2048 // n_acc, 136
    announce(f"gemm pp in-place residual n_acc={n_acc}")
    g = torch.Generator(device=gpu).manual_seed(5)
    x = torch.randn(M, N, generator=g, device=gpu)
    x0, o16 = x.double(), torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    acc = _gemm(M, N, K, n_acc, [ops.EpiSpec(abi.EPI_ADD, o16, e=0), ops.EpiSpec(abi.EPI_ADD, x, e=0)], gpu, 3, False,
                extras=[x])[0]
    assert _rel(x, acc + x0) < TOL
    _same_bits(o16, x)
