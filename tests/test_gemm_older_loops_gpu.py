"""The bf16 main loops that the ping-pong kernel leaves: persistent (128 and 256 rows) and direct (64 rows, one and
two workgroups per CU), each call's loop asserted (th_gemm_route), against float64 of the same bf16 operands.

fp32 outputs are compared at 1e-5 of the largest value: at most 576 products that are exact in fp32, each sum
rounded by 2^-24 of magnitudes a dozen times the typical result, 1e-6 in practice."""

import pytest
import torch

from conftest import announce
from test_gemm_pp_epilogue_gpu import _rel, _rope_ref, _same_bits

pytestmark = pytest.mark.gpu

TOL = 1e-5


class _Case:
    def __init__(self, gpu, M, N, K, n_acc, **kw):
        g = torch.Generator(device=gpu).manual_seed(M + N + K)
        self.gpu, self.shape, self.gen, self.kw = gpu, (M, N, K, n_acc), g, kw
        self.x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
        self.ws = [(torch.randn(K, N, generator=g, device=gpu) * 0.1).bfloat16() for _ in range(n_acc)]

    def out(self, dtype, cols=None):
        return torch.full((self.shape[0], cols or self.shape[1]), 7.0, dtype=dtype, device=self.gpu)

    def run(self, outs, loop, rows=None, scaled=True):
        """Launches the call, checks that it runs on ``loop`` and returns the float64 accumulators."""
        from torch_helion.hip import abi, ops

        M, N, K, n_acc = self.shape
        announce(f"gemm {loop} M={M} N={N} K={K} n_acc={n_acc}")
        if scaled:
            self.kw.update(sumsq=True, rscale_mask=(1 << n_acc) - 1, inv_k=1.0 / K, eps=1e-5)
        call = ops.GemmCall(M, N, K, n_acc, self.x, ops.pack_rhs(self.ws, torch.bfloat16), outs, **self.kw)
        route = ops.gemm_route(call)
        assert route[0] == getattr(abi, f"LOOP_BF16_{loop}") and rows in (None, route[1]), route
        ops.gemm(call)
        torch.cuda.synchronize()
        xd = self.x.double()
        parts = self.kw.get("rs_parts")
        ss = parts.double().sum(-1, keepdim=True) if parts is not None else xd.square().sum(-1, keepdim=True)
        r = torch.rsqrt(ss / K + 1e-5) if scaled else 1.0
        return [(xd @ w.double()) * r for w in self.ws]


@pytest.mark.parametrize("M,rows", [(16371, 256), (4099, 128)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_persistent_residual_and_row_parts(gpu, M, rows, xdt):
    """A residual with bf16 and fp32 outputs, the row scale from the producer's partial sums (K = 64: one step, which
    the ping-pong loop does not take)."""
    from torch_helion.hip import abi, ops

    c = _Case(gpu, M, 2048, 64, 1)
    x = torch.randn(M, 2048, generator=c.gen, device=gpu).to(xdt)
    ss = torch.empty(M, device=gpu)
    c.kw.update(extras=[x], sumsq_out=ss, rs_parts=torch.rand(M, 12, generator=c.gen, device=gpu))
    o16, o32 = c.out(torch.bfloat16), c.out(torch.float32)
    acc, = c.run([ops.EpiSpec(abi.EPI_ADD, o16, e=0), ops.EpiSpec(abi.EPI_ADD, o32, e=0)], "PERSISTENT", rows)
    assert _rel(o32, acc + x.double()) < TOL
    _same_bits(o16, o32)
    assert _rel(ss, c.kw["rs_parts"].double().sum(-1)) < TOL


@pytest.mark.parametrize("M,N,K", [(16371, 2052, 192), (8190, 2052, 512)])
def test_persistent_unaligned_rows(gpu, M, N, K):
    """N % 8 == 4: output and operand rows that no loop can access in 16-byte pieces; the row scale from the
    producer's partial sums."""
    from torch_helion.hip import abi, ops

    c = _Case(gpu, M, N, K, 1)
    x = torch.randn(M, N, generator=c.gen, device=gpu).bfloat16()
    c.kw.update(extras=[x], rs_parts=torch.rand(M, 12, generator=c.gen, device=gpu))
    o16, o32, s16 = c.out(torch.bfloat16), c.out(torch.float32), c.out(torch.bfloat16)
    acc, = c.run([ops.EpiSpec(abi.EPI_MUL, o16, e=0), ops.EpiSpec(abi.EPI_MUL, o32, e=0),
                  ops.EpiSpec(abi.EPI_SILU, s16)], "PERSISTENT")
    assert _rel(o32, acc * x.double()) < TOL
    _same_bits(o16, o32)
    assert _rel(s16, torch.nn.functional.silu(acc)) < 2.0**-8


@pytest.mark.parametrize("M,K,rows,hd", [(16371, 256, 256, 128), (16371, 128, 256, 64), (8190, 64, 128, 64),
                                         (8190, 512, 128, 32)])
def test_persistent_rope(gpu, M, K, rows, hd):
    from torch_helion.hip import abi, ops

    N, period = 2048, 100
    c = _Case(gpu, M, N, K, 1)
    cos, sin = (torch.randn(period, hd, generator=c.gen, device=gpu) for _ in range(2))
    c.kw.update(rope_cos=cos, rope_sin=sin, rope_head_dim=hd, rope_period=period)
    q16, q32 = c.out(torch.bfloat16), c.out(torch.float32)
    acc, = c.run([ops.EpiSpec(abi.EPI_ROPE, q16), ops.EpiSpec(abi.EPI_ROPE, q32)], "PERSISTENT", rows)
    assert _rel(q32, _rope_ref(acc, None, cos, sin, period)) < TOL
    _same_bits(q16, q32)


@pytest.mark.parametrize("M,K,rows", [(16371, 512, 256), (4090, 64, 128)])
@pytest.mark.parametrize("hd", [64, 128])
def test_persistent_two_accumulators(gpu, M, K, rows, hd):
    """k (rotated) and v in one launch: heads of 64 fit a wave's columns, heads of 128 need a whole accumulator
    per wave."""
    from torch_helion.hip import abi, ops

    N, period = 1024, 100
    c = _Case(gpu, M, N, K, 2)
    cos, sin = (torch.randn(period, hd, generator=c.gen, device=gpu) for _ in range(2))
    c.kw.update(rope_cos=cos, rope_sin=sin, rope_head_dim=hd, rope_period=period)
    k16, k32, v32 = c.out(torch.bfloat16), c.out(torch.float32), c.out(torch.float32)
    acc = c.run([ops.EpiSpec(abi.EPI_ROPE, k16, a=0), ops.EpiSpec(abi.EPI_ACC, v32, a=1),
                 ops.EpiSpec(abi.EPI_ROPE, k32, a=0)], "PERSISTENT", rows)
    assert _rel(k32, _rope_ref(acc[0], None, cos, sin, period)) < TOL
    _same_bits(k16, k32)
    assert _rel(v32, acc[1]) < TOL


@pytest.mark.parametrize("M,N,K,n_acc,rows", [(16371, 2560, 64, 1, 256), (8190, 1000, 512, 3, 256), (4090, 1024, 512, 4, 128)])
def test_persistent_windows_and_more_accumulators(gpu, M, N, K, n_acc, rows):
    from torch_helion.hip import abi, ops

    c = _Case(gpu, M, N, K, n_acc)
    cuts = [0, 64, 136, N - 512, N]
    if n_acc == 1:
        outs = [(0, b, e) for b, e in zip(cuts, cuts[1:])]
    else:
        outs = [(i, 0, N) for i in range(n_acc)]
    dst = [c.out(torch.float32, e - b) for _, b, e in outs]
    acc = c.run([ops.EpiSpec(abi.EPI_ACC, d, a=a, cols=(b, e)) for d, (a, b, e) in zip(dst, outs)], "PERSISTENT", rows)
    for d, (a, b, e) in zip(dst, outs):
        assert _rel(d, acc[a][:, b:e]) < TOL


@pytest.mark.parametrize("M,N,K", [(2000, 2196, 512), (2048, 2196, 512), (1000, 5004, 256), (130, 2196, 512)])
@pytest.mark.parametrize("scaled", [True, False])
def test_direct_one_accumulator_256_columns(gpu, M, N, K, scaled):
    """64 x 256 tiles: 288, 288 and 320 of them, two workgroups per CU, and 27, one per CU."""
    from torch_helion.hip import abi, ops

    c = _Case(gpu, M, N, K, 1)
    o16, o32 = c.out(torch.bfloat16), c.out(torch.float32)
    acc, = c.run([ops.EpiSpec(abi.EPI_ACC, o16), ops.EpiSpec(abi.EPI_ACC, o32)], "DIRECT", 64, scaled)
    assert _rel(o32, acc) < TOL
    _same_bits(o16, o32)
