"""Cost model on the CPU: the GEMM tile choice mirrors th_gemm's, the calibration fit
recovers the parameters that generated its samples, and merged sibling launches are
priced with the fitted merged-launch factor (the planner's merge-or-split decision);
and the counters tool's per-symbol table."""

from __future__ import annotations

import dataclasses

import pytest
import torch


def test_gemm_tiles_mirror_th_gemm():
    """The tile that th_gemm says it would run (th_gemm_route; no GPU), over rows, columns and depths on both
    sides of every rule: 64-, 128- and 256-row loops, ping-pong rows, partial K steps, ragged columns."""
    from test_gemm_route import _Fake
    from torch_helion.cost_models.roofline import gemm_tiles
    from torch_helion.hip import abi, ops

    if not abi.library_path().exists():
        pytest.skip("libth_hip.so not built (run __graft_entry__.build())")
    bf = torch.bfloat16
    seen = set()
    for n_acc in (1, 2, 3):
        for N in (48, 128, 512, 768, 1000, 1024, 1280, 2048, 4096, 8200, 50280):
            for K in (64, 192, 576, 1000, 2048, 14336):
                for M in (1, 64, 300, 1500, 4096, 8192, 16384):
                    outs = [ops.EpiSpec(abi.EPI_ACC, _Fake(M, N, bf), a=i) for i in (0,)]
                    loop, bm, cols, _ = ops.gemm_route(ops.GemmCall(M, N, K, n_acc, _Fake(M, K, bf), _Fake(N, K, bf), outs))
                    assert gemm_tiles(N, n_acc, M, "bfloat16", 256, K) == (bm, cols // n_acc), (M, N, K, n_acc)
                    seen.add((loop, bm))
    assert {l for l, _ in seen} == {abi.LOOP_BF16_STAGED, abi.LOOP_BF16_DIRECT, abi.LOOP_BF16_PERSISTENT,
                                    abi.LOOP_BF16_PINGPONG}
    assert {bm for l, bm in seen if l == abi.LOOP_BF16_PINGPONG} == {128, 192, 256}


def _rec(kernel, cat, ideal, waves, measured):
    return {"run": "r", "kernel": kernel, "category": cat, "ideal_us": ideal, "waves": waves,
            "measured_us": measured, "bound": "mfma"}


def test_calibration_fit_recovers_parameters():
    """Samples generated from known parameters: the weighted NNLS fit returns them, the
    merged-launch factor is the one the merged samples carry, and predict() reproduces
    every sample."""
    from torch_helion.cost_models.calibrate import fit, predict

    eff, tile, fixed, factor = 0.5, 10.0, 8.0, 1.25
    recs = [_rec(f"k{i}", "gemm_bf16", ideal, waves, ideal / eff + waves * tile + fixed)
            for i, (ideal, waves) in enumerate([(5, 1), (40, 2), (100, 4), (300, 4), (800, 8), (20, 0.25),
                                                (2, 0.0625)])]
    recs += [_rec(f"m{i}", "gemm_bf16_merged", ideal, waves, factor * (ideal / eff + waves * tile + fixed))
             for i, (ideal, waves) in enumerate([(60, 3), (3, 1), (150, 5)])]
    c = fit(recs)
    assert c["efficiency"]["gemm_bf16"] == pytest.approx(eff, rel=1e-3)
    assert c["tile_us"]["gemm_bf16"] == pytest.approx(tile, rel=1e-3)
    assert c["fixed_us"]["gemm_bf16"] == pytest.approx(fixed, abs=0.01)
    assert c["merged_launch_factor"] == pytest.approx(factor, abs=1e-3)
    assert c["kernels_fitted"] == {"gemm_bf16": 7, "gemm_bf16_merged": 3}
    for r in recs:
        assert predict(r, c) == pytest.approx(r["measured_us"], rel=2e-3)


def test_calibration_counts_a_repeated_shape_once():
    """24 equal layers whose shape does not follow the other kernels' line move the fit no further than one."""
    from torch_helion.cost_models.calibrate import distinct, fit

    recs = [_rec(f"k{i}", "gemm_bf16", ideal, waves, 2 * ideal + 10 * waves + 8)
            for i, (ideal, waves) in enumerate([(5, 1), (40, 2), (100, 4), (300, 4), (800, 8), (20, 0.25)])]
    odd = [_rec(f"layer{i}", "gemm_bf16", 27.0, 1.0, 90.0 + i) for i in range(25)]
    d = distinct(recs + odd)
    assert len(d) == 7 and d[-1]["measured_us"] == 102.0
    assert fit(d) == fit(recs + [{**odd[0], "measured_us": 102.0}])


def test_calibration_without_merged_samples_has_no_factor():
    from torch_helion.cost_models.calibrate import fit

    recs = [_rec(f"k{i}", "gemm_bf16", ideal, waves, 2 * ideal + 10 * waves + 8)
            for i, (ideal, waves) in enumerate([(5, 1), (40, 2), (100, 4), (300, 8)])]
    assert "merged_launch_factor" not in fit(recs)


@pytest.fixture(scope="module")
def mamba_program(tmp_path_factory):
    from targets.mamba import MambaConfig, build_mamba_block
    from torch_helion import CompileConfig, compile_model

    cfg = MambaConfig(batch=2, seq=64, d_model=256, expand=2, headdim=32, d_state=32, chunk=32, n_layers=1)
    m = build_mamba_block(cfg)
    x = m.example_inputs(seed=0)
    res = compile_model(m, x, CompileConfig(run_name="cm", results_dir=tmp_path_factory.mktemp("cm"), backend="none",
                                            planner_mode="greedy", reference_check=False))
    return res.program


def _sibling_group(program):
    """GEMM kernels reading the same lhs over the same K (the in-projection's parts), with
    the accumulators each uses."""
    from torch_helion.hip.epilogue import match_epilogue

    by_lhs: dict = {}
    for k in program.kernels:
        if k.kind == "gemm" and k.gemms:
            by_lhs.setdefault((k.arg("lhs").tensor, k.k_extent), []).append(k)
    group = max(by_lhs.values(), key=len)
    assert len(group) >= 2, "the Mamba in-projection lowers to several GEMM kernels on one lhs"
    return [(k.name, len({o.a for o in match_epilogue(k).outs})) for k in group]


def test_merge_decision_follows_merged_launch_factor(mamba_program):
    """The merged price is the GEMM model of the concatenated weights times the fitted
    factor; the split price does not depend on it; a large enough factor turns the
    decision to split, and the plan report shows both prices."""
    from torch_helion.cost_models.hw_spec import HardwareSpec
    from torch_helion.optimizer.planner import launch_merge_report, price_launch_merges

    hw = HardwareSpec.load()
    assert hw.calibration.get("efficiency", {}).get("gemm_bf16"), "the shipped spec carries a bf16 GEMM fit"

    def with_factor(f):
        return dataclasses.replace(hw, raw={**hw.raw, "calibration": {**hw.calibration, "merged_launch_factor": f}})

    group = _sibling_group(mamba_program)
    one = price_launch_merges(mamba_program, [group], with_factor(1.0))[0]
    big = price_launch_merges(mamba_program, [group], with_factor(50.0))[0]
    assert big.split_us == pytest.approx(one.split_us)
    assert big.merged_us == pytest.approx(50.0 * one.merged_us)
    assert not big.merged and big.to_dict()["merged"] is False
    rep = launch_merge_report([one, big])
    assert f"{big.merged_us:,.1f}" in rep and f"{big.split_us:,.1f}" in rep
    assert rep.rstrip().endswith("| split |")


def test_counter_table_groups_by_symbol():
    """The counters tool's table: one row per kernel symbol (parameters dropped), averaged over
    its positions, longest total first; a dispatch above --split-us gets a row of its own."""
    from torch_helion.hip.counters import by_symbol

    def pos(sym, us, util, fetch):
        return {"symbol": sym, "duration_us": us, "mfma_util": util, "clock_ghz": 2.0, "FETCH_SIZE": fetch,
                "WRITE_SIZE": 1024.0}

    g = "void th::gemm<256, 1>(th::GemmK)"
    rows = by_symbol([pos(g, 90.0, 0.3, 2048.0), pos("th::carry(th::SsdK)", 20.0, 0.0, 1024.0), pos(g, 110.0, 0.5, 4096.0),
                      pos(g, 1800.0, 0.47, 8192.0)], split_us=1000.0).splitlines()
    assert rows[2] == "| `th::gemm<256, 1> (long)` | 1 | 1800.0 | 47.0% | 2.00 | 8.0 | 1.0 |"
    assert rows[3] == "| `th::gemm<256, 1>` | 2 | 100.0 | 40.0% | 2.00 | 3.0 | 1.0 |"
    assert rows[4] == "| `th::carry` | 1 | 20.0 | 0.0% | 2.00 | 1.0 | 1.0 |"
    assert len(by_symbol([pos(g, 90.0, 0.3, 2048.0), pos(g, 1800.0, 0.4, 2048.0)]).splitlines()) == 3
