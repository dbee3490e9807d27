"""Which main loop th_gemm takes (th_gemm_route; no GPU): pinned to shapes on which every loop was timed."""

import pytest
import torch

from torch_helion.hip import abi, ops


class _Fake:
    """A device matrix that only has a shape, a type and an aligned address."""

    def __init__(self, rows, cols, dtype):
        self.shape, self.dtype = (rows, cols), dtype

    def data_ptr(self):
        return 1 << 20

    def dim(self):
        return 2

    def stride(self, i):
        return self.shape[1] if i == 0 else 1

    def is_contiguous(self):
        return True


def _call(M, N, K, form, copy32=False):
    bf, f32, E = torch.bfloat16, torch.float32, ops.EpiSpec
    n_acc, kw, w = 1, {}, []
    if form == "acc2":
        n_acc, outs = 2, [E(abi.EPI_ACC, _Fake(M, N, bf)), E(abi.EPI_ACC, _Fake(M, N, bf), a=1)]
    elif form == "acc":
        outs = [E(abi.EPI_ACC, _Fake(M, N, bf))]
    elif form in ("add", "add_fp32", "add_parts"):
        outs = [E(abi.EPI_ADD, _Fake(M, N, bf), e=0)]
        kw["extras"] = [_Fake(M, N, bf if form == "add" else f32)]
        if form == "add_parts":
            kw.update(sumsq=True, rscale_mask=1, rs_parts=_Fake(M, 64, f32))
    elif form == "windows":
        w = [0, N // 2 // 8 * 8, N - 304, N - 176, N - 48, N]
        outs = [E(abi.EPI_ACC, _Fake(M, e - b, bf), cols=(b, e)) for b, e in zip(w, w[1:])]
        kw.update(sumsq=True, rscale_mask=1)
    elif form == "swiglu":
        n_acc, outs = 2, [E(abi.EPI_SWIGLU, _Fake(M, N, bf), a=0, b=1)]
        kw.update(sumsq=True, rscale_mask=3)
    else:  # ropeHD, qkvHD
        hd = int(form.lstrip("ropeqkv"))
        kw.update(sumsq=True, rscale_mask=1, rope_cos=_Fake(2048, hd, f32), rope_sin=_Fake(2048, hd, f32),
                  rope_head_dim=hd, rope_period=2048)
        if form.startswith("rope"):
            outs = [E(abi.EPI_ROPE, _Fake(M, N, bf))]
        else:
            q = N * 2 // 3 // hd * hd
            k = (N - q) // 2 // hd * hd
            outs = [E(abi.EPI_ROPE, _Fake(M, q, bf), cols=(0, q)), E(abi.EPI_ROPE, _Fake(M, k, bf), cols=(q, q + k)),
                    E(abi.EPI_ACC, _Fake(M, N - q - k, bf), cols=(q + k, N))]
    if copy32:
        outs.insert(1, E(outs[0].op, _Fake(M, N, f32), a=outs[0].a, b=outs[0].b, e=outs[0].e))
    return ops.GemmCall(M, N, K, n_acc, _Fake(M, K, bf), _Fake(N, K, bf), outs, **kw)


@pytest.fixture(scope="module", autouse=True)
def _lib():
    if not abi.library_path().exists():
        pytest.skip("libth_hip.so not built (run __graft_entry__.build())")


D, P, PP = abi.LOOP_BF16_DIRECT, abi.LOOP_BF16_PERSISTENT, abi.LOOP_BF16_PINGPONG


# (us, one MI355X: direct 64-row / persistent 128 or 256 rows / ping-pong at its best rows)
@pytest.mark.parametrize("M,N,K,form,loops", [
    (200, 2048, 2048, "rope64", (D,)),          # 30.8 / - / 33.5
    (1000, 2048, 2048, "rope64", (D,)),         # 32.8 / - / 34.5
    (500, 3072, 2048, "qkv64", (D,)),           # 33.7 / - / 34.8
    (4096, 1024, 1024, "rope64", (D, P)),       # 18.4 / 19.3 / 24.9
    (4096, 1024, 1024, "acc", (D, P)),          # 14.0 / 14.3 / 15.9
    (2000, 2048, 576, "acc", (D,)),             # 12.3 / - / 13.7
    (16384, 2048, 192, "acc", (P,)),            # - / 29.5 / 33.5
    (16384, 2048, 320, "acc", (P,)),            # - / 36.1 / 41.5
    (16384, 2048, 576, "acc", (P,)),            # - / 48.5 / 51.9
    (16384, 128, 1024, "acc2", (D,)),           # 25.0 / - / 27.1 (after the kernel that writes the lhs)
    (2067, 20352, 256, "add", (PP,)),           # - / 74.1 / 53.7
    (16384, 2192, 512, "windows", (PP,)),       # - / 86.2 / 68.0
    (500, 2192, 512, "windows", (PP,)),         # 16.8 / - / 15.4
    (4096, 2048, 2048, "rope64", (PP,)),        # - / 46.0 / 42.4
    (16384, 6144, 4096, "qkv128", (PP,)),       # - / 731.7 / 680.8
    (16384, 1024, 2048, "add_parts", (PP,)),    # - / 84.2 / 79.1
    (8192, 1024, 2048, "add", (PP,)),           # - / 60.0 / 35.7
    (16384, 14336, 4096, "swiglu", (PP,)),      # - / 3106 / 2847
    (3001, 4096, 14336, "add", (PP,)),          # - / 411 / 283
    (3001, 4096, 136, "acc", (PP,)),            # (K % 64: no direct loop)
])
def test_takes_the_measured_faster_loop(M, N, K, form, loops):
    assert ops.gemm_route(_call(M, N, K, form))[0] in loops


@pytest.mark.parametrize("M,N,K,form,rows", [
    (16384, 14336, 4096, "swiglu", 256),        # 2847, 192 rows 3300
    (3001, 4096, 14336, "add", 192),            # 283, 128 rows 320, 256 rows 300
    (1500, 2048, 4096, "acc", 128),
])
def test_tile_rows(M, N, K, form, rows):
    loop, tile_rows, cols, us = ops.gemm_route(_call(M, N, K, form))
    assert (loop, tile_rows, cols) == (PP, rows, 256) and us > 0


def test_estimate_counts_the_steps_that_run():
    """The ping-pong loop runs an even number of 64-deep steps: K = 4160 costs what K = 4224 does."""
    a, b = ops.gemm_route(_call(4096, 4096, 4160, "acc")), ops.gemm_route(_call(4096, 4096, 4224, "acc"))
    assert a[0] == b[0] == PP and a[3] == b[3]


@pytest.mark.parametrize("M", [64, 700, 2000, 4096, 16384])
@pytest.mark.parametrize("N,K,form", [(8192, 256, "swiglu"), (2048, 192, "acc"), (1024, 2048, "add_fp32"), (4096, 4096, "add")])
def test_a_copy_beside_an_output_changes_nothing(M, N, K, form):
    assert ops.gemm_route(_call(M, N, K, form)) == ops.gemm_route(_call(M, N, K, form, copy32=True))


@pytest.mark.parametrize("M,N,K,slices", [(32, 64, 256, 8), (32, 64, 260, 9), (128, 512, 512, 16), (32, 64, 16384, 64)])
def test_fp32_workspace_holds_the_slices_that_run(M, N, K, slices):
    """fp32 split-K: slices are whole 32-wide steps, so no more of them are asked for than K has steps."""
    bn = 64 if N <= 64 else 128
    Mp, Npk = -(-M // 32) * 32, -(-N // bn) * bn
    assert ops.gemm_workspace_bytes(M, N, K, 1, torch.float32) == slices * Mp * (Npk + 1) * 4
