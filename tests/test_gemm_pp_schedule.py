"""The ping-pong GEMM's K loop as compiled: what its schedule counts on (loads that stay in
flight for one and a half K steps) holds only if the compiler adds no wait of its own."""

import re
import shutil
import subprocess

import pytest

from torch_helion.hip import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(TM, sumsq, n_acc): assembly text} of every instance of gemm_bf16_pp_kernel."""
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc not on PATH")
    out = tmp_path_factory.mktemp("asm") / "gemm_pp.s"
    cmd = [build.hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", str(build.CSRC / "gemm_pp.hip"), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    text = out.read_text()
    found = {}
    for name, body in re.findall(r"^(\S*gemm_bf16_pp_kernel\S*):.*?\n(.*?)^\.Lfunc_end", text, re.S | re.M):
        found[tuple(int(x) for x in re.search(r"ILi(\d)ELb(\d)ELi(\d)E", name).groups())] = body
    assert len(found) == 12
    return found


def _steady_loop(body: str) -> list[str]:
    """The shortest backward-branch span that holds both MFMAs and direct-to-LDS loads."""
    lines = body.split("\n")
    at = {m.group(1): i for i, l in enumerate(lines) if (m := re.match(r"(\.LBB\S+):", l))}
    spans = []
    for i, l in enumerate(lines):
        m = re.match(r"\s+s_c?branch\S*\s+(\.LBB\S+)", l)
        if m and at.get(m.group(1), i) < i:
            span = lines[at[m.group(1)]:i]
            if any("v_mfma" in x for x in span) and any("global_load_lds" in x for x in span):
                spans.append(span)
    return min(spans, key=len)


def test_k_loop_keeps_loads_in_flight(kernels):
    for (tm, sumsq, n_acc), body in kernels.items():
        loop = _steady_loop(body)
        what = f"TM={tm} sumsq={sumsq} n_acc={n_acc}"
        # two K steps: 64-deep, four 16-deep MFMAs on 2 TM subtiles, 4 + TM loads each
        assert sum("v_mfma" in l for l in loop) == 2 * 4 * 2 * tm, what
        assert sum("global_load_lds" in l for l in loop) == 2 * (4 + tm), what
        # The kernel's own waits leave a step's loads (4 + TM) and at least a phase's of the step before in flight.
        waits = [int(m.group(1)) for l in loop if (m := re.search(r"vmcnt\((\d+)\)", l))]
        assert len(waits) == 8 and min(waits) >= 4 + tm + 2 + tm // 2, f"{what}: {waits}"


def test_no_spills(kernels):
    for key, body in kernels.items():
        assert "scratch_" not in body, f"{key}: registers spill to scratch memory"


def test_wide_buffer_stores_take_no_scalar_offset(kernels):
    """The compiler keeps a wait between a 16-byte store and the next write of its data registers only for stores
    without a register as scalar offset; with one, the last lanes' data was overwritten."""
    for key, body in kernels.items():
        stores = re.findall(r"buffer_store_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], (\S+) ", body)
        assert stores and set(stores) == {"0"}, key
