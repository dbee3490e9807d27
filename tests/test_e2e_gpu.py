"""End to end on the GPU: compile_model(backend="hip") vs the CPU oracle.

fp32 programs: max relative error (max|a-b| / max|b|) <= 1e-4 against the
oracle in float64. bf16 programs: max-abs error <= 2e-2 against the oracle in
float32 on the same (bf16) weights and inputs.
"""

from __future__ import annotations

import functools

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _oracle(model, cfg, x, dtype, storage=None, round_residual=False):
    from oracle.llama import block_forward

    w = {k: v.detach().to(dtype) for k, v in model.state_dict().items() if not k.startswith(("rope", "attn_bias"))}
    return block_forward(x.to(dtype), w, heads=cfg.heads, kv_heads=cfg.n_kv, eps=cfg.eps, theta=cfg.rope_theta,
                         causal=cfg.causal, rope=(model.rope_cos.to(dtype), model.rope_sin.to(dtype)), dtype=dtype,
                         storage=storage, round_residual=round_residual)


def _compile(model, x, tmp_path, name, **cfg):
    from torch_helion import CompileConfig, compile_model

    return compile_model(model, x, CompileConfig(run_name=name, results_dir=tmp_path, backend="hip",
                                                 planner_mode="greedy", **cfg))


CASES = {
    "mha_bf16": dict(batch=2, seq=128, hidden=256, heads=4, intermediate=512, dtype=torch.bfloat16),
    "gqa_causal_bf16": dict(batch=2, seq=256, hidden=512, heads=8, kv_heads=2, intermediate=1024, causal=True,
                            dtype=torch.bfloat16, rope_theta=500000.0),
    "gqa_causal_bf16_hd128": dict(batch=1, seq=384, hidden=1024, heads=8, kv_heads=4, intermediate=2048, causal=True,
                                  dtype=torch.bfloat16),
}


@pytest.mark.parametrize("case", list(CASES))
def test_llama_block_bf16(gpu, tmp_path, case):
    from targets.llama_block import LlamaBlockConfig, build_llama_block

    announce(f"e2e llama {case}")
    cfg = LlamaBlockConfig(**CASES[case])
    model = build_llama_block(cfg, seed=0)
    x = model.example_inputs(seed=0)
    res = _compile(model, x, tmp_path, case)
    assert res.validation["ok"], res.validation
    # the pre-rotated RoPE siblings are re-fused: q alone and (k, v) as 2 accumulators
    fused = [p for p in res.device_program.plans.values() if p.get("rope_fused")]
    assert fused and all(p["n_acc"] <= 3 for p in fused), res.device_program.plans
    out = res.run(*x)[0].float().cpu()
    ref = _oracle(model, cfg, x[0], torch.float32)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max().item() < 2e-2
    # the fp32 copy of the output against the oracle with the program's bf16 storage points
    out32 = res.device_program.outputs(fp32=True)[0].float().cpu()
    ref_store = _oracle(model, cfg, x[0], torch.float32, storage=torch.bfloat16)
    assert (out32 - ref_store).abs().max().item() < 1e-2


def test_llama_block_bf16_residual_in_bf16(gpu, tmp_path):
    """residual_fp32=False and fp32_outputs=False (the eager model's precision): no fp32 copies are
    allocated and the residual stream is the bf16 buffer. Gate: the reference's normalised error
    max|a-b| / max|b| <= 2e-2 against the fp32 oracle (outputs reach ~3.6 here, where one bf16 ulp
    is 0.0156, so the 2e-2 max-abs bar sits at about one ulp of storage rounding), and agreement with
    the oracle that rounds to bf16 at the same storage points to within 1e-2 normalised."""
    from targets.llama_block import LlamaBlockConfig, build_llama_block

    announce("e2e llama bf16 residual")
    cfg = LlamaBlockConfig(**CASES["gqa_causal_bf16_hd128"])
    model = build_llama_block(cfg, seed=0)
    x = model.example_inputs(seed=0)
    res = _compile(model, x, tmp_path, "bf16res", residual_fp32=False, fp32_outputs=False)
    assert res.validation["ok"], res.validation
    assert not res.device_program.shadow, list(res.device_program.shadow)
    out = res.run(*x)[0].float().cpu()
    ref = _oracle(model, cfg, x[0], torch.float32)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max().item() / ref.abs().max().item() < 2e-2
    ref_store = _oracle(model, cfg, x[0], torch.float32, storage=torch.bfloat16)
    assert (out - ref_store).abs().max().item() / ref_store.abs().max().item() < 1e-2


def test_llama_block_c1_fp32(gpu, tmp_path):
    """BASELINE config 0 (C1): fp32, B=1, S=128, d=512, 8x64 MHA, FFN 1376, causal."""
    from targets.llama_block import build_llama_block, config_c1

    announce("e2e llama C1 fp32")
    cfg = config_c1()
    model = build_llama_block(cfg, seed=0)
    x = model.example_inputs(seed=0)
    res = _compile(model, x, tmp_path, "c1")
    out = res.run(*x)[0].double().cpu()
    ref = _oracle(model, cfg, x[0], torch.float64)
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    assert rel < 1e-4, rel
    kinds = [k.kind for k in res.program.kernels]
    assert kinds == ["gemm", "attention", "gemm", "gemm", "gemm"], kinds


def test_device_program_reruns_are_identical(gpu, tmp_path):
    """Two runs on the same inputs give bit-identical outputs (no atomics in reductions)."""
    from targets.llama_block import LlamaBlockConfig, build_llama_block

    announce("e2e determinism")
    cfg = LlamaBlockConfig(**CASES["gqa_causal_bf16"])
    model = build_llama_block(cfg, seed=1)
    x = model.example_inputs(seed=1)
    res = _compile(model, x, tmp_path, "det")
    a = res.run(*x)[0].clone()
    b = res.run(*x)[0].clone()
    assert torch.equal(a, b)


def _mamba_oracle(model, cfg, x):
    from oracle.mamba import backbone_forward

    return backbone_forward(x.double(), {k: v.double() for k, v in model.state_dict().items()}, cfg)


def test_mamba_block_fp32_conv_groups(gpu, tmp_path):
    import math

    from targets.mamba import MambaConfig, build_mamba_block

    announce("e2e mamba fp32 conv ngroups=1")
    cfg = MambaConfig(batch=2, seq=256, d_model=256, expand=2, headdim=64, d_state=64, chunk=64, n_layers=1,
                      ngroups=1, use_conv=True, dtype=torch.float32, a_log_range=(0.0, math.log(16.0)))
    m = build_mamba_block(cfg, seed=0)
    x = m.example_inputs(seed=0)
    res = _compile(m, x, tmp_path, "mamba_fp32")
    kinds = [k.kind for k in res.program.kernels]
    assert "ssd_chunked" in kinds and "conv1d" in kinds, kinds
    out = res.run(*x)[0].double().cpu()
    ref = _mamba_oracle(m, cfg, x[0])
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    assert rel < 1e-4, rel


@pytest.mark.parametrize("fp32_copies", [True, False])
def test_mamba_layer_c2_bf16(gpu, tmp_path, fp32_copies):
    """BASELINE config 1 (C2): Mamba-2 block bf16, B=2, L=1024, d=512, 16 heads x 64, N=64, G=1, conv 4, chunk 64;
    with the fp32 residual and output copies, and at the eager model's precision (bf16 throughout)."""
    from targets.mamba import build_mamba_block, config_c2

    announce(f"e2e mamba C2 bf16 fp32_copies={fp32_copies}")
    cfg = config_c2()
    m = build_mamba_block(cfg, seed=0)
    x = m.example_inputs(seed=0)
    res = _compile(m, x, tmp_path, "mamba_c2", residual_fp32=fp32_copies, fp32_outputs=fp32_copies)
    assert res.validation["ok"], res.validation
    out = res.device_program.outputs(fp32=True)[0].double().cpu()
    ref = _mamba_oracle(m, cfg, x[0])
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    assert rel < 2e-2, rel
    assert (out - ref).abs().max().item() < 5e-2


def test_mamba_layer_c2_merged_in_projection(gpu, tmp_path):
    """merge_siblings=True: the three in-projection GEMMs of the Mamba layer (B|C, dt, z|x) launch as one
    th_gemm over concatenated weights with column-windowed outputs; same results as the separate launches."""
    from targets.mamba import build_mamba_block, config_c2

    announce("e2e mamba C2 merged in-projection")
    cfg = config_c2()
    m = build_mamba_block(cfg, seed=0)
    x = m.example_inputs(seed=0)
    sep = _compile(m, x, tmp_path, "c2_sep", residual_fp32=False, fp32_outputs=False, merge_siblings=False)
    mer = _compile(m, x, tmp_path, "c2_mer", residual_fp32=False, fp32_outputs=False, merge_siblings=True)
    auto = _compile(m, x, tmp_path, "c2_auto", residual_fp32=False, fp32_outputs=False)  # 2048 rows: merged
    assert len(auto.device_program.launches) == len(mer.device_program.launches)
    assert mer.validation["ok"], mer.validation
    merged = [l for l in mer.device_program.launches if "+" in l.kernel]
    assert merged and len(merged[0].info["merged"]) == 3, [l.kernel for l in mer.device_program.launches]
    assert len(mer.device_program.launches) == len(sep.device_program.launches) - 2
    a = sep.run(*x)[0].float().cpu()
    b = mer.run(*x)[0].float().cpu()
    # same products, one accumulator instead of three: fp32 sums in a different tile order
    assert (a - b).abs().max().item() / a.abs().max().item() < 1e-2


def test_mamba_layer_c2_merged_convs(gpu, tmp_path):
    """merge_convs (the default): the x, B and C convolutions of the layer run as one th_conv1d_causal
    launch over the xBC channels side by side (inputs and outputs are column windows of two shared
    buffers); bit-identical to one launch per convolution, two launches fewer."""
    from targets.mamba import build_mamba_block, config_c2

    announce("e2e mamba C2 merged convolutions")
    cfg = config_c2()
    m = build_mamba_block(cfg, seed=0)
    x = m.example_inputs(seed=0)
    sep = _compile(m, x, tmp_path, "c2_convsep", merge_convs=False, merge_siblings=False)
    mer = _compile(m, x, tmp_path, "c2_convmer", merge_siblings=False)
    assert mer.validation["ok"], mer.validation
    convs = [l for l in mer.device_program.launches if l.kind == "conv1d"]
    assert len(convs) == 1 and len(convs[0].info["merged"]) == 3, [l.kernel for l in mer.device_program.launches]
    assert convs[0].info["width"] == cfg.d_inner + 2 * cfg.d_bc
    assert len(mer.device_program.launches) == len(sep.device_program.launches) - 2
    for a, b in zip(sep.run(*x), mer.run(*x)):
        assert torch.equal(a.cpu(), b.cpu())
    a32, b32 = sep.device_program.outputs(fp32=True)[0], mer.device_program.outputs(fp32=True)[0]
    assert torch.equal(a32.cpu(), b32.cpu())


@pytest.mark.parametrize("which", ["llama_gqa_bf16", "mamba_c2_bf16"])
def test_graph_replays_match_eager(gpu, tmp_path, which):
    """The captured HIP graph of a whole program reproduces the eager launch sequence bit for bit,
    on every replay, with eager runs and synchronisations between replays and after new inputs."""
    announce(f"e2e graph replay {which}")
    if which == "mamba_c2_bf16":
        from targets.mamba import build_mamba_block, config_c2

        model = build_mamba_block(config_c2(), seed=0)
    else:
        from targets.llama_block import LlamaBlockConfig, build_llama_block

        model = build_llama_block(LlamaBlockConfig(**CASES["gqa_causal_bf16"]), seed=2)
    x1, x2 = model.example_inputs(seed=0), model.example_inputs(seed=5)
    res = _compile(model, x1, tmp_path, f"graph_{which}")
    dp = res.device_program

    def eager(x):
        dp.set_inputs(list(x))
        dp.launch_all()
        torch.cuda.synchronize()
        return [o.clone() for o in dp.outputs()] + [o.clone() for o in dp.outputs(fp32=True)]

    ref1, ref2 = eager(x1), eager(x2)
    dp.set_inputs(list(x1))
    dp.capture()
    for i, (x, ref) in enumerate([(x1, ref1), (x1, ref1), (x2, ref2), (x1, ref1)]):
        dp.set_inputs(list(x))
        for o in dp.outputs() + dp.outputs(fp32=True):  # a replay that writes nothing must fail
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        dp.replay()
        torch.cuda.synchronize()
        got = [o.clone() for o in dp.outputs()] + [o.clone() for o in dp.outputs(fp32=True)]
        for g, r in zip(got, ref):
            assert torch.equal(g, r), (which, i)
        eager(x2 if i % 2 else x1)  # ordinary eager work between replays


def _decode_case(cfg, pos, seed):
    from targets.llama_block import build_llama_block

    torch.manual_seed(seed)
    m = build_llama_block(cfg, seed=seed)
    sd = {k: v for k, v in m.state_dict().items() if not k.startswith(("rope", "attn_bias"))}
    g = torch.Generator().manual_seed(seed + 1)
    x = torch.randn(cfg.batch, cfg.hidden, generator=g).bfloat16()
    kc = torch.randn(cfg.batch, cfg.seq, cfg.n_kv, cfg.head_dim, generator=g).bfloat16()
    vc = torch.randn(cfg.batch, cfg.seq, cfg.n_kv, cfg.head_dim, generator=g).bfloat16()
    return sd, x, kc, vc


def _spec_quantised(sd: dict[str, torch.Tensor]) -> dict[str, torch.Tensor]:
    """The decode configuration's weights as the BASELINE specifies them, computed here
    independently of the product: every projection W [out, in] quantised per output
    channel, s_n = max|W[n, :]| / 448, q = e4m3(W / s_n), dequantised to q * s_n in fp32;
    the norm gains unchanged."""
    out = {}
    for k, v in sd.items():
        w = v.detach().float()
        if k.endswith("_proj.weight"):
            s = w.abs().amax(1, keepdim=True) / 448.0
            w = (w / s).to(torch.float8_e4m3fn).float() * s
        out[k] = w
    return out


@pytest.mark.parametrize("which", ["small", "medium", "medium_unfolded", "c5"])
def test_decode_step_fp8_vs_oracle(gpu, which):
    """Decode step with e4m3 weights: the block output and the cache entries it writes at ``pos``
    against the oracle's decode step in fp32 on the BASELINE's quantisation (plain W quantised
    per output channel, gains on the activations), built by the test itself. Hidden sizes that
    are multiples of 1024 (medium, C5) apply the post-attention gain in the o-projection's
    finishing pass; medium_unfolded runs the same block with its own pass for it."""
    from oracle.llama import decode_step
    from targets.llama_block import LlamaBlockConfig, config_c5
    from torch_helion.hip.decode import DecodeBlock

    if which == "c5":
        cfg, pos = config_c5(), 4096
    elif which.startswith("medium"):
        cfg, pos = LlamaBlockConfig(batch=4, seq=80, hidden=1024, heads=8, kv_heads=2, intermediate=2048, causal=True,
                                    dtype=torch.bfloat16, rope_theta=500000.0), 71
    else:
        cfg, pos = LlamaBlockConfig(batch=4, seq=80, hidden=256, heads=4, kv_heads=2, intermediate=512, causal=True,
                                    dtype=torch.bfloat16, rope_theta=500000.0), 77
    announce(f"e2e decode fp8 {which} pos={pos}")
    sd, x, kc, vc = _decode_case(cfg, pos, seed=3)
    w_spec = _spec_quantised(sd)
    assert w_spec["input_norm.weight"].std() > 0.01      # the gains are not all one: the test sees where they go
    blk = DecodeBlock(sd, hidden=cfg.hidden, heads=cfg.heads, kv_heads=cfg.n_kv, intermediate=cfg.intermediate,
                      eps=cfg.eps, rope_theta=cfg.rope_theta, batch=cfg.batch, max_len=cfg.seq, device=gpu,
                      fold_gain=which != "medium_unfolded")
    assert blk.fold_gain == (which in ("medium", "c5"))
    eff = blk.effective_weights()
    for k, v in w_spec.items():
        assert torch.equal(eff[k], v), k                  # the product quantises exactly as specified
    blk.k_cache.copy_(kc.to(gpu))
    blk.v_cache.copy_(vc.to(gpu))
    blk.step(x.to(gpu), pos)
    torch.cuda.synchronize()
    out = blk.out32.cpu().double()
    kw = dict(heads=cfg.heads, kv_heads=cfg.n_kv, eps=cfg.eps, theta=cfg.rope_theta)
    ref, kn, vn = decode_step(x, w_spec, kc, vc, pos, **kw)
    ref_b, kn_b, vn_b = decode_step(x, w_spec, kc, vc, pos, storage=torch.bfloat16, **kw)
    floor = (ref_b - ref).abs().max().item()
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    assert rel < 2e-2, rel
    # max-abs bar: twice the bf16 rounding floor, i.e. twice the distance of a step that rounds the
    # same intermediates to bf16 from the unrounded step (a correct kernel's error is a draw from the
    # same distribution; the factor covers the draw and roundings placed differently inside kernels)
    assert (out - ref).abs().max().item() <= 2 * floor, ((out - ref).abs().max().item(), floor)
    # the cache entries are stored in bf16: the same twice-the-floor bar, per tensor
    for got, want, want_b in ((blk.k_cache[:, pos], kn, kn_b), (blk.v_cache[:, pos], vn, vn_b)):
        err = (got.double().cpu() - want).abs().max().item()
        assert err <= 2 * (want_b - want).abs().max().item(), err
    # positions before pos are untouched
    assert torch.equal(blk.k_cache[:, :pos].cpu(), kc[:, :pos])


@pytest.mark.parametrize("which", ["small", "c5"])
def test_compile_model_decode_fp8_vs_oracle(gpu, tmp_path, which):
    """The decode step through compile_model: a LlamaDecodeBlock (e4m3 weights quantised as the
    BASELINE specifies, gains on the activations) compiles to a Program with e4m3 weight
    tensors and an attention_decode kernel; on the device its output (fp32 copy) and the new
    key/value rows, written straight into the cache inputs at pos, meet the same bars as the
    hand-assembled step against the oracle's decode step on the spec weights."""
    from oracle.llama import decode_step
    from targets.llama_block import LlamaBlockConfig, build_llama_block, config_c5
    from targets.llama_decode import PROJECTIONS, LlamaDecodeBlock

    if which == "c5":
        cfg, pos = config_c5(), 4096
    else:
        cfg, pos = LlamaBlockConfig(batch=4, seq=80, hidden=256, heads=4, kv_heads=2, intermediate=512, causal=True,
                                    dtype=torch.bfloat16, rope_theta=500000.0), 77
    announce(f"e2e compile_model decode fp8 {which} pos={pos}")
    sd, x, kc, vc = _decode_case(cfg, pos, seed=3)
    m = LlamaDecodeBlock(build_llama_block(cfg, seed=3), pos).eval()
    w_spec = _spec_quantised(sd)
    for short, name in PROJECTIONS.items():
        deq = getattr(m, f"{short}_q").float() * getattr(m, f"{short}_s")[:, None]
        assert torch.equal(deq, w_spec[name]), name
    res = _compile(m, (x, kc, vc), tmp_path, f"decode_{which}", device_check=False, reference_check=False,
                   verify_passes=False)
    prog = res.program
    assert [k.kind for k in prog.kernels].count("attention_decode") == 1
    assert all(prog.tensors[k.arg(g.rhs).tensor].dtype == "float8_e4m3fn" for k in prog.kernels
               if k.kind == "gemm" for g in k.gemms)
    dp = res.device_program
    # q and k|v read the same input: one e4m3 launch over both, on column windows
    assert any(l.info.get("weights") == "float8_e4m3fn" and len(l.info.get("merged", [])) == 2
               for l in dp.launches), [l.kernel for l in dp.launches]
    # hidden a multiple of 1024 (C5): the o-projection stores gate/up's gained operand and its row
    # sums, so gate/up has no gain pre-pass; at hidden 256 gate/up scales its rows itself
    folded = [l.info.get("gain_out_for") for l in dp.launches if l.info.get("gain_out_for")]
    from_producer = [l.kernel for l in dp.launches if l.info.get("row_sums_from_producer")]
    assert len(folded) == (1 if which == "c5" else 0) and from_producer == folded, (folded, from_producer)
    dp.run([x, kc, vc])
    torch.cuda.synchronize()
    out, k_dev, v_dev = (t.double().cpu() for t in dp.outputs(fp32=True))
    rope = (m.rope_cos.expand(pos + 1, -1), m.rope_sin.expand(pos + 1, -1))
    kw = dict(heads=cfg.heads, kv_heads=cfg.n_kv, eps=cfg.eps, theta=cfg.rope_theta, rope=rope)
    ref, kn, vn = decode_step(x, w_spec, kc, vc, pos, **kw)
    ref_b, kn_b, vn_b = decode_step(x, w_spec, kc, vc, pos, storage=torch.bfloat16, **kw)
    floor = (ref_b - ref).abs().max().item()
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    mx = (out - ref).abs().max().item()
    print(f"decode {which}: normalised {rel:.3e}, max-abs {mx:.4f}, bf16 floor {floor:.4f}", flush=True)
    assert rel < 2e-2, rel
    assert mx <= 2 * floor, (mx, floor)
    for got, want, want_b in ((k_dev, kn, kn_b), (v_dev, vn, vn_b)):
        err = (got - want).abs().max().item()
        assert err <= 2 * (want_b - want).abs().max().item(), err
    # the new rows live in the cache inputs at pos; the rows before pos are untouched
    L, hk, hd = cfg.seq, cfg.n_kv, cfg.head_dim
    k_cache = dp.tensor("k_cache").view(cfg.batch, L, hk, hd)
    assert torch.equal(k_cache[:, pos].double().cpu(), k_dev)
    assert torch.equal(k_cache[:, :pos].cpu(), kc[:, :pos])


def _lm_check(res, model, cfg, ids, prefix: int, layers=None):
    """Logits of the HIP program (fp32 copy) for sequence 0's first ``prefix`` tokens
    against the oracle's model_forward in float64 on those tokens alone (the model is
    causal, so a prefix of the output depends only on the same prefix of the input)."""
    from oracle.mamba import model_forward

    dp = res.device_program
    dp.run([ids])
    torch.cuda.synchronize()
    out = dp.outputs(fp32=True)[0].reshape(cfg.batch, cfg.seq, cfg.vocab)[0, :prefix].double().cpu()
    w = {k: v.detach() for k, v in model.state_dict().items()}
    ref = model_forward(ids[:1, :prefix], w, cfg)[0]
    return float((out - ref).abs().max() / ref.abs().max()), float((out - ref).abs().max())


def test_mamba_lm_fp32_small(gpu, tmp_path):
    """Token ids -> th_embedding -> 2 Mamba-2 layers -> tied head (vocab 1000, not a
    multiple of 32) in fp32: 1e-4 relative to the oracle."""
    import math

    from targets.mamba import MambaConfig, build_mamba_model

    announce("e2e mamba lm fp32 small")
    cfg = MambaConfig(batch=2, seq=128, d_model=128, expand=2, headdim=32, d_state=32, chunk=64, n_layers=2, ngroups=1,
                      use_conv=True, dtype=torch.float32, a_log_range=(0.0, math.log(16.0)), vocab=1000)
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)[0]
    res = _compile(m, (ids,), tmp_path, "lm_fp32")
    assert [l.entry for l in res.device_program.launches][0] == "th_embedding"
    rel, _ = _lm_check(res, m, cfg, ids, cfg.seq)
    assert rel < 1e-4, rel
    with pytest.raises(IndexError):
        res.device_program.set_inputs([ids.clone().fill_(cfg.vocab)])


def test_mamba_lm_c4_shapes_two_layers(gpu, tmp_path):
    """BASELINE config 3 (C4) at full width and length with 2 of its 24 layers and 2 of
    its 8 sequences: d=1024, 32 heads x 64, N=128, chunk 256, vocab 50280 tied, bf16."""
    from targets.mamba import build_mamba_model, config_c4
    from torch_helion import CompileConfig, compile_model

    announce("e2e mamba lm C4 shapes, 2 layers")
    cfg = config_c4()
    cfg.n_layers, cfg.batch = 2, 2
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)[0]
    res = compile_model(m, (ids,), CompileConfig(run_name="lm_c4", results_dir=tmp_path, backend="hip",
                                                 planner_mode="greedy", device_check=False))
    kinds = [k.kind for k in res.program.kernels]
    assert kinds[0] == "embedding" and kinds.count("ssd_chunked") == 2
    rel, mx = _lm_check(res, m, cfg, ids, 384)
    assert rel < 2e-2, (rel, mx)


def test_mamba_lm_merged_in_projection_activation_gain(gpu, tmp_path):
    """norm_gain='activation' with merge_siblings=True: the in-projection GEMMs unfold the same
    norm gain, so they merge into one launch over the unfolded weights behind one shared
    normalised-lhs launch; the logits match the separate launches (each output column is the
    same dot product in the same K order)."""
    from targets.mamba import build_mamba_model, config_c4

    announce("e2e mamba lm merged in-projection, activation-side gain")
    cfg = config_c4()
    cfg.n_layers, cfg.batch, cfg.seq, cfg.vocab = 2, 1, 512, 4096
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)
    kw = dict(device_check=False, fp32_outputs=False, norm_gain="activation")
    sep = _compile(m, ids, tmp_path, "lm_sep", merge_siblings=False, **kw)
    mer = _compile(m, ids, tmp_path, "lm_mer", merge_siblings=True, **kw)
    merged = [l for l in mer.device_program.launches if "+" in l.kernel and l.entry == "th_gemm"]
    assert len(merged) == 2 and all(l.info["gain_on_activation"] for l in merged), \
        [l.kernel for l in mer.device_program.launches]
    # the gated norm before each out-projection folds into the scan (its gain) and the
    # GEMM (its row scale): one scan per layer names its GEMM, which has no norm launch
    for res in (sep, mer):
        folds = {l.info["norm_gain_for"] for l in res.device_program.launches if l.info.get("norm_gain_for")}
        assert len(folds) == cfg.n_layers
        for l in res.device_program.launches:
            if l.kernel in folds:
                assert l.entry == "th_gemm" and l.info.get("row_sums_from_producer"), (l.kernel, l.entry, l.info)
    a = sep.run(*ids)[0].float().cpu()
    b = mer.run(*ids)[0].float().cpu()
    assert (a - b).abs().max().item() / a.abs().max().item() < 1e-3


@pytest.mark.parametrize("fp32_copies", [True, False])
def test_llama_block_c3_full(gpu, tmp_path, fp32_copies):
    """BASELINE config 2 (C3) at its full size: Llama-3-8B-shaped block, bf16, B=8, S=2048,
    32/8 heads x 128, FFN 14336, causal, through compile_model. Sequence 0 of the output
    against the oracle in float64: normalised error <= 2e-2, and max-abs at most twice the bf16
    floor (the same block storing q, k, v, the attention output, the MLP's residual operand and
    the SwiGLU product in bf16, against the unrounded block).
    Both storage variants: fp32 copies of the residual stream and the output (the compiled
    default; the output's fp32 copy is compared), and none (residual_fp32=False,
    fp32_outputs=False: the program bench.py times), whose bf16 output is compared against a
    floor that also rounds the residual stream and the output to bf16."""
    from targets.llama_block import build_llama_block, config_c3

    announce(f"e2e llama C3 full size (B=8, S=2048), fp32 copies {fp32_copies}")
    cfg = config_c3()
    model = build_llama_block(cfg, seed=0)
    x = model.example_inputs(seed=0)
    res = _compile(model, x, tmp_path, "c3_full", device_check=False, reference_check=False, verify_passes=False,
                   residual_fp32=fp32_copies, fp32_outputs=fp32_copies)
    res.device_program.run(list(x))
    torch.cuda.synchronize()
    out = res.device_program.outputs(fp32=fp32_copies)[0].reshape(cfg.batch, cfg.seq, cfg.hidden)[0].double().cpu()
    x0 = x[0][:1]
    ref = _oracle(model, cfg, x0, torch.float64)[0]
    emu = _oracle(model, cfg, x0, torch.float64, storage=torch.bfloat16, round_residual=not fp32_copies)[0]
    floor = (emu - ref).abs().max().item()
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    mx = (out - ref).abs().max().item()
    print(f"C3 full (fp32 copies {fp32_copies}): normalised {rel:.3e}, max-abs {mx:.4f}, bf16 floor {floor:.4f}",
          flush=True)
    assert torch.isfinite(out).all()
    assert rel < 2e-2, rel
    assert mx <= 2 * floor, (mx, floor)


@functools.lru_cache(maxsize=1)
def _c4_reference(prefix: int):
    """Sequence 0's first ``prefix`` tokens of the C4 model in float64: the oracle's logits and
    the bf16 floor (the compiled program evaluated in float64 with exact weights and every
    kernel output rounded to its declared dtype), computed once for both storage variants."""
    import tempfile

    from oracle import interpret as oi
    from oracle.mamba import model_forward
    from targets.mamba import build_mamba_model, config_c4
    from torch_helion import CompileConfig, compile_model

    cfg = config_c4()
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)[0]
    w = {k: v.detach() for k, v in m.state_dict().items()}
    ids0 = ids[:1, :prefix]
    ref = model_forward(ids0, w, cfg)[0]
    small = type(cfg)(**{**cfg.__dict__, "batch": 1, "seq": prefix})
    ms = build_mamba_model(small, seed=0)
    rs = compile_model(ms, (ids0,), CompileConfig(run_name="c4_floor", results_dir=tempfile.mkdtemp(), backend="none",
                                                  planner_mode="greedy", reference_check=False, verify_passes=False))
    fs = rs.graph.fold_sources
    params = {n: fs[n][0].double().reshape(-1, 1) * fs[n][1].double() if n in fs else v
              for n, v in rs.graph.params.items()}
    emu = oi.program_outputs(rs.program, params, [ids0], storage="declared")[0].reshape(ref.shape)
    return ref, (emu - ref).abs().max().item()


@pytest.mark.parametrize("fp32_outputs", [True, False])
def test_mamba_lm_c4_full(gpu, tmp_path, fp32_outputs):
    """BASELINE config 3 (C4) at its full size: token ids -> embedding -> 24 Mamba-2 layers
    (d=1024, 32 heads x 64, N=128, chunk 256) -> final norm -> tied head (vocab 50280), bf16,
    B=8, L=2048, with the norm gains on the activation side (norm_gain="activation").
    The logits of sequence 0's first 256 tokens (their fp32 copy, or with fp32_outputs=False,
    the program bench.py times, the bf16 logits themselves) against the oracle's model_forward
    in float64 on those tokens. The bf16 floor is the compiled program evaluated in float64
    with exact weights and every kernel output rounded to its declared dtype (bf16 logits
    included): max-abs must stay within twice the floor's, and the normalised error within
    2e-2 or, where the floor itself is above that, within 1.25 times the floor's normalised
    error. This bar was set after the plain 2e-2 gate failed at 2.5%: 24 layers of bf16
    activations put the floor at 2.4% here and the eager bf16 model at 3.8%; the rounding of
    the MFMA operands alone, with every other intermediate exact, already costs 1.3%."""
    from targets.mamba import build_mamba_model, config_c4
    from torch_helion import CompileConfig, compile_model

    announce(f"e2e mamba lm C4 full size (24 layers, B=8, L=2048), fp32 outputs {fp32_outputs}")
    cfg = config_c4()
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)[0]
    res = compile_model(m, (ids,), CompileConfig(run_name="c4_full", results_dir=tmp_path, backend="hip",
                                                 planner_mode="greedy", device_check=False, reference_check=False,
                                                 verify_passes=False, norm_gain="activation",
                                                 fp32_outputs=fp32_outputs))
    assert [k.kind for k in res.program.kernels].count("ssd_chunked") == 24
    assert any(p.get("gain_on_activation") for p in res.device_program.plans.values())
    prefix = 256
    dp = res.device_program
    dp.run([ids])
    torch.cuda.synchronize()
    out = dp.outputs(fp32=fp32_outputs)[0].reshape(cfg.batch, cfg.seq, cfg.vocab)[0, :prefix].double().cpu()
    del res, dp
    ref, floor = _c4_reference(prefix)
    floor_rel = floor / ref.abs().max().item()
    rel = ((out - ref).abs().max() / ref.abs().max()).item()
    mx = (out - ref).abs().max().item()
    print(f"C4 full (fp32 outputs {fp32_outputs}): normalised {rel:.3e} (floor {floor_rel:.3e}), "
          f"max-abs {mx:.4f} (floor {floor:.4f})", flush=True)
    assert torch.isfinite(out).all()
    assert rel <= max(2e-2, 1.25 * floor_rel), (rel, floor_rel)
    assert mx <= 2 * floor, (mx, floor)


@pytest.mark.parametrize("norm_gain", ["fold", "activation"])
def test_buffer_reuse_is_bit_exact(gpu, tmp_path, norm_gain):
    """Liveness-based buffer reuse changes where intermediates live, not what is computed:
    a 6-layer bf16 Mamba-2 LM gives bit-identical logits with and without reuse (eager and
    graph replay), while its intermediates hold well under half the bytes."""
    import math

    from targets.mamba import MambaConfig, build_mamba_model

    announce(f"e2e buffer reuse, norm_gain={norm_gain}")
    cfg = MambaConfig(batch=2, seq=512, d_model=256, expand=2, headdim=64, d_state=64, chunk=128, n_layers=6,
                      ngroups=1, use_conv=True, dtype=torch.bfloat16, a_log_range=(0.0, math.log(16.0)), vocab=4000)
    m = build_mamba_model(cfg, seed=0)
    ids = m.example_inputs(seed=0)[0]
    outs = {}
    for reuse in (False, True):
        res = _compile(m, (ids,), tmp_path, f"reuse_{reuse}", device_check=False, reference_check=False,
                       verify_passes=False, reuse_buffers=reuse, norm_gain=norm_gain)
        dp = res.device_program
        dp.run([ids])
        torch.cuda.synchronize()
        outs[reuse] = dp.outputs(fp32=True)[0].clone()
        if reuse:
            rep = dp.memory_report()
            assert rep["pool_bytes"] < 0.5 * rep["without_reuse_bytes"], rep
            dp.capture()
            for _ in range(3):
                dp.replay()
                torch.cuda.synchronize()
                assert torch.equal(dp.outputs(fp32=True)[0], outs[True])
    assert torch.equal(outs[True], outs[False])


@pytest.mark.parametrize("heads,kv_heads,seq", [(8, 4, 200), (16, 8, 129)])
def test_llama_rotary_projections_merged(gpu, heads, kv_heads, seq, tmp_path):
    """q, k and v of a grouped-query bf16 block as one launch (heads of 128 and 64) against two launches."""
    from targets.llama_block import LlamaBlockConfig, build_llama_block
    from torch_helion import CompileConfig, compile_model

    cfg = LlamaBlockConfig(batch=2, seq=seq, hidden=1024, heads=heads, kv_heads=kv_heads, intermediate=512, causal=True,
                           dtype=torch.bfloat16)
    model = build_llama_block(cfg, seed=3)
    x = model.example_inputs(seed=3)
    outs = []
    for merge in (None, False):
        res = compile_model(model, x, CompileConfig(run_name=f"rotary_{merge}", results_dir=tmp_path, device_check=False,
                                                    reference_check=False, verify_passes=False, merge_siblings=merge))
        outs.append(res.run(*x)[0].clone())
        merged = [l for l in res.device_program.launches if "+" in l.kernel]
        assert len(merged) == (1 if merge is None else 0)
        assert [(p.members, p.merged) for p in res.device_program.launch_merges] == [(l.info["merged"], True) for l in merged]
    torch.cuda.synchronize()
    # The products are the same sums in the same order. Two launches may run on another kernel than one, whose
    # fp32 row sums of squares add up in another order: the row scales then differ by a few 2^-24, which moves a
    # bf16 rounding here and there (q, k, v, the attention output, the MLP's operands), each by 2^-8 of the value
    # at most: under 2^-8 of the result's 2-norm even if every value moved.
    a, b = outs[0].double(), outs[1].double()
    assert float((a - b).norm() / b.norm()) < 2.0**-8
    # And row by row, so that no few rows are wrong: the output's own rounding (2^-8 of the row), and four bf16
    # roundings in a row in what is added to the residual (projections, attention output, MLP input and operand).
    d, r = a - b, b - x[0].to(b.device).double().reshape(b.shape)
    assert bool((d.norm(dim=-1) < 2.0**-8 * b.norm(dim=-1) + 4 * 2.0**-8 * r.norm(dim=-1)).all())


def test_llama_rotary_projections_priced(gpu, tmp_path):
    """Where two launches of the rotary projections are estimated the faster (both fill whole rounds of tiles, one
    does not), merge_siblings=None keeps them apart and says so in the plan; True merges all the same."""
    from targets.llama_block import LlamaBlockConfig, build_llama_block
    from torch_helion import CompileConfig, compile_model

    cfg = LlamaBlockConfig(batch=4, seq=2048, hidden=2048, heads=32, kv_heads=8, intermediate=256, causal=True,
                           dtype=torch.bfloat16)
    model = build_llama_block(cfg, seed=3)
    x = model.example_inputs(seed=3)
    for merge in (None, True):
        res = compile_model(model, x, CompileConfig(run_name=f"priced_{merge}", results_dir=tmp_path, device_check=False,
                                                    reference_check=False, verify_passes=False, merge_siblings=merge))
        merged = [l for l in res.device_program.launches if "+" in l.kernel]
        assert len(merged) == (1 if merge else 0)
        if merge:
            assert not res.device_program.launch_merges  # (nothing was priced)
            continue
        price, = res.device_program.launch_merges
        assert not price.merged
        plan = next(tmp_path.rglob(f"*priced_{merge}*/05_plan/plan.md"), None) or next(tmp_path.rglob("plan.md"))
        assert " + ".join(price.members) in plan.read_text()
