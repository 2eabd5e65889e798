"""Parity of the device-resident decision-model forward with the reference, through the C ABI.

* The four forward goldens (crates/raya-cli/tests/forward_golden.rs): every traced stage
  on the valid rows at 1e-5, probabilities and features at 1e-6.  fixture-h64 has
  head_dim 32 (separate RoPE kernel), fixture-h128 head_dim 64 (RoPE fused into the
  QKV GEMM epilogue).
* Padding invariance (forward_golden.rs:238-262).
* A batch of sequences with different lengths and markers against the oracle's
  Network::forward run one sequence at a time, on random models of both head dims.
"""
import json
import os

import numpy as np
import pytest

import oracle
from oracle import forward as F
from raya_amd import Mask
from raya_amd import model as M
from tests.conftest import GOLDEN

pytestmark = pytest.mark.gpu

FWD = os.path.join(GOLDEN, "forward")
LAYER_TOL, PROB_TOL = 1e-5, 1e-6
CASES = ["short", "medium", "padded", "fastpath_off"]


def load_case(name):
    from safetensors.numpy import load_file

    meta = json.load(open(os.path.join(FWD, name, "meta.json")))
    cdir = os.path.normpath(os.path.join(FWD, name, meta["config_dir"]))
    wpath = os.path.normpath(os.path.join(FWD, name, meta["weights_file"]))
    g = load_file(os.path.join(FWD, name, "tensors.safetensors"))
    return F.load_config(cdir), M.Model.load(cdir, wpath), g, meta["input"]["unpadded_length"]


def golden_input(g, valid, cut=None):
    ids = g["input_ids"][0] if cut is None else g["input_ids"][0][:cut]
    return M.ForwardInput(ids, valid, g["marker_pos"][0], g["marker_mask"][0], int(g["qtype"][0]))


def stages(cfg):
    v = [("embedding_output", LAYER_TOL)]
    v += [(f"encoder_layer_{i:02d}", LAYER_TOL) for i in range(cfg.layers)]
    v += [(n, LAYER_TOL) for n in ("encoder_final_norm", "encoder_output", "type_emb_add", "head_input")]
    v += [(f"head_layer_{i:02d}", LAYER_TOL) for i in range(cfg.head_layers)]
    v += [("marker_states", LAYER_TOL), ("logits", LAYER_TOL), ("probabilities", PROB_TOL),
          ("act_features", PROB_TOL), ("pooled", LAYER_TOL), ("act_logits", LAYER_TOL)]
    return v


@pytest.mark.parametrize("case", CASES)
def test_forward_matches_golden(case):
    cfg, model, g, valid = load_case(case)
    print(f"case {case}: valid {valid} of {g['input_ids'].shape[1]}", flush=True)
    tr = M.Trace()
    out = model.forward(golden_input(g, valid), trace=tr)
    assert tr.names() == [n for n, _ in stages(cfg)]
    seq = g["input_ids"].shape[1]
    worst = {}
    for name, tol in stages(cfg):
        want = g[name].astype(np.float32)
        shape, got = tr.get(name)
        assert shape == want.shape, name
        if want.ndim == 3 and want.shape[1] == seq:
            want, got = want[:, :valid], got[:, :valid]
        worst[name] = float(np.abs(got - want).max())
        assert worst[name] <= tol, (name, worst[name])
    print(case, {k: f"{v:.1e}" for k, v in worst.items()})
    for name, arr in (("logits", out.logits), ("probabilities", out.probabilities),
                      ("act_logits", out.act_logits), ("pooled", out.pooled)):
        assert np.array_equal(arr, tr.get(name)[1].reshape(arr.shape)), name
    assert np.array_equal(out.features, tr.get("act_features")[1].reshape(4))


def test_padding_does_not_change_valid_rows():
    cfg, model, g, valid = load_case("padded")
    a, b = M.Trace(), M.Trace()
    model.forward(golden_input(g, valid), trace=a)
    model.forward(golden_input(g, valid, cut=valid), trace=b)
    for name in ("embedding_output", "encoder_layer_00", "encoder_layer_02", "head_layer_00"):
        x, y = a.get(name)[1][:, :valid], b.get(name)[1][:, :valid]
        assert np.abs(x - y).max() <= 1e-5, name
    for name in ("logits", "probabilities", "act_logits", "pooled"):
        assert np.abs(a.get(name)[1] - b.get(name)[1]).max() <= 1e-5, name


# --- random models against the oracle -------------------------------------------------------

def make_model(tmp_path, hidden, heads, layers=3, inter=None, head_layers=2, vocab=300, acts=2,
               local_attention=16, seed=0, dtype=np.float32):
    from safetensors.numpy import save_file

    inter = inter or 2 * hidden
    enc = {"hidden_size": hidden, "intermediate_size": inter, "num_hidden_layers": layers,
           "num_attention_heads": heads, "global_attn_every_n_layers": 2,
           "local_attention": local_attention, "max_position_embeddings": 4096,
           "vocab_size": vocab, "norm_eps": 1e-5, "norm_bias": False, "attention_bias": False,
           "mlp_bias": False, "hidden_activation": "gelu",
           "rope_parameters": {"full_attention": {"rope_theta": 160000.0},
                               "sliding_attention": {"rope_theta": 10000.0}}}
    agent = {"head_layers": head_layers, "act_costs": {f"a{i}": 0.1 for i in range(acts - 1)}}
    d = tmp_path / f"m{hidden}_{heads}_{seed}"
    os.makedirs(d / "encoder", exist_ok=True)
    json.dump(enc, open(d / "encoder" / "config.json", "w"))
    json.dump(agent, open(d / "rl_agent_config.json", "w"))
    cfg = F.load_config(str(d))
    rng = np.random.default_rng(seed)
    w = {}
    for name, shape in F.expected_names(cfg):
        if name.endswith("norm.weight") or name.endswith(("norm1.weight", "norm2.weight")) \
                or name == "scorer.0.weight":
            x = 1.0 + 0.1 * rng.standard_normal(shape)
        else:
            x = 0.05 * rng.standard_normal(shape)
        w[name] = x.astype(dtype)
    save_file(w, str(d / "model.safetensors"))
    return cfg, str(d), {k: v.astype(np.float32) for k, v in w.items()}


def random_batch(rng, cfg, b, seq, k):
    ids = rng.integers(1, cfg.vocab, size=(b, seq)).astype(np.uint32)
    valid = rng.integers(max(4, seq // 4), seq + 1, size=b)
    valid[0] = seq
    pos = np.zeros((b, k), np.int64)
    mask = np.zeros((b, k), bool)
    for i in range(b):
        nk = rng.integers(1, k + 1)
        pos[i, :nk] = np.sort(rng.choice(valid[i], size=nk, replace=False))
        mask[i, :nk] = True
        mask[i, 0] = True
    qtype = rng.integers(0, 3, size=b)
    return ids, valid, pos, mask, qtype


@pytest.mark.parametrize("hidden,heads,inter", [(128, 2, None), (64, 2, None), (256, 4, None), (96, 2, None),
                                                (128, 2, 200)])
def test_batch_matches_oracle_per_sequence(tmp_path, hidden, heads, inter):
    """hidden 256: the row-in-registers LayerNorm (rows of a multiple of 256 floats); hidden 96:
    not a multiple of 64, so the LayerNorms stay kernels of their own (the others fold them
    into the GEMMs); intermediate size 200: not a multiple of 16, so the MLP's output GEMM
    pads its depth and the norms stay unfolded."""
    cfg, cdir, w = make_model(tmp_path, hidden, heads, inter=inter)
    model = M.Model.load(cdir)
    rng = np.random.default_rng(hidden)
    ids, valid, pos, mask, qtype = random_batch(rng, cfg, b=5, seq=200, k=4)
    print(f"hidden {hidden} heads {heads}: valid {valid.tolist()}", flush=True)
    out = model.forward_batch(ids, valid, pos, mask, qtype)
    for i in range(len(valid)):
        want = F.forward(cfg, w, ids[i], int(valid[i]), pos[i], mask[i], int(qtype[i]))
        for name, tol in (("logits", LAYER_TOL), ("probabilities", PROB_TOL),
                          ("act_logits", LAYER_TOL), ("features", PROB_TOL), ("pooled", LAYER_TOL)):
            got, exp = getattr(out, name)[i], getattr(want, name)
            assert np.abs(got - exp).max() <= tol, (i, name, float(np.abs(got - exp).max()))
        # the same sequence alone on the device gives the same outputs
        one = model.forward(M.ForwardInput(ids[i], int(valid[i]), pos[i], mask[i], int(qtype[i])))
        assert np.abs(one.act_logits - out.act_logits[i]).max() <= 1e-6


def test_local_mask_override_matches_oracle(tmp_path):
    """The throughput option: BlockDiag(64) on local layers, global layers stay Full."""
    cfg, cdir, w = make_model(tmp_path, 128, 2, layers=2, head_layers=0)
    model = M.Model.load(cdir)
    rng = np.random.default_rng(3)
    ids, valid, pos, mask, qtype = random_batch(rng, cfg, b=3, seq=300, k=3)
    tr = M.Trace()
    out = model.forward_batch(ids, valid, pos, mask, qtype, trace=tr, local_mask=Mask.block_diag(64))
    for i in range(3):
        want = F.forward(cfg, w, ids[i], int(valid[i]), pos[i], mask[i], int(qtype[i]),
                         local_mask=(oracle.MASK_BLOCKDIAG, 64))
        v = int(valid[i])
        got = tr.get("encoder_layer_01")[1][i, :v]
        assert np.abs(got - want.trace["encoder_layer_01"][:v]).max() <= LAYER_TOL
        assert np.abs(out.act_logits[i] - want.act_logits).max() <= LAYER_TOL


def test_half_precision_weights_are_widened_exactly(tmp_path):
    """F16 weights give the same outputs as the F32 file holding their widened values."""
    from safetensors.numpy import save_file

    cfg, cdir16, w = make_model(tmp_path, 128, 2, layers=2, seed=7, dtype=np.float16)
    cfg, cdir32, _ = make_model(tmp_path / "f32", 128, 2, layers=2, seed=7, dtype=np.float16)
    save_file(w, os.path.join(cdir32, "model.safetensors"))  # widened on the host by numpy
    rng = np.random.default_rng(4)
    batch = random_batch(rng, cfg, b=2, seq=64, k=2)
    a = M.Model.load(cdir16).forward_batch(*batch)
    b = M.Model.load(cdir32).forward_batch(*batch)
    assert np.array_equal(a.act_logits, b.act_logits) and np.array_equal(a.pooled, b.pooled)


def test_stage_timing_spans_and_outputs_unchanged():
    """Profiling records one span per stage (level 1) and per layer kernel (level 2)
    without changing any output."""
    cfg, model, g, valid = load_case("medium")
    inp = golden_input(g, valid)
    print(f"stage timing: {cfg.layers} layers, {cfg.head_layers} head layers", flush=True)
    base = model.forward(inp)
    assert model.stage_times() == []
    model.set_profiling(1)
    out1 = model.forward(inp)
    names1 = [n for n, _ in model.stage_times()]
    want1 = (["embedding"] + [f"encoder_layer_{i:02d}" for i in range(cfg.layers)] + ["final_norm"]
             + [f"head_layer_{i:02d}" for i in range(cfg.head_layers)] + ["scorer_and_act_head"])
    assert names1 == want1
    assert all(ms > 0.0 for _, ms in model.stage_times())
    model.set_profiling(2)
    out2 = model.forward(inp)
    names2 = [n for n, _ in model.stage_times()]
    # the fixture's width (a multiple of 64) folds both LayerNorms into the GEMMs that read them
    ops = ["qkv", "attention", "attn_out", "mlp_in_geglu", "mlp_out"]
    for i in range(cfg.layers):
        layer = f"encoder_layer_{i:02d}"
        subs = [n.split("/")[1] for n in names2 if n.startswith(layer + "/")]
        assert subs == ops, (layer, subs)
    times = dict(model.stage_times())
    for i in range(cfg.layers):
        layer = f"encoder_layer_{i:02d}"
        parts = sum(ms for n, ms in times.items() if n.startswith(layer + "/"))
        assert parts <= times[layer] * 1.001 + 1e-3
    model.set_profiling(0)
    out0 = model.forward(inp)
    assert model.stage_times() == []
    for o in (out1, out2, out0):
        for f in ("logits", "probabilities", "act_logits", "features", "pooled"):
            assert np.array_equal(getattr(o, f), getattr(base, f)), f
    with pytest.raises(M.InputError):
        model.set_profiling(3)


def test_base_width_layers_match_oracle(tmp_path):
    """The bench model's layer width at reduced depth: hidden 768, 12 heads of 64 (RoPE fused
    into the QKV GEMM), GeGLU 3072, Sliding(64) local layers (local_attention 128), LayerNorm
    rows of 768 held in registers, one head layer; three sequences up to 300 tokens against the
    oracle's Network::forward one sequence at a time.

    The goldens' 1e-5 per stage and 1e-6 on probabilities are set for the reference's small
    fixtures (d <= 128).  At d = 768 the contractions run over 768 and 3,072 terms in another
    order than the reference's sequential sums, so the 768-wide outputs (pooled, act_logits)
    are held to the fp32 bar of max-abs 1e-4 and rel-L2 1e-5 (measured: pooled 5.6e-5
    max-abs, 5.4e-6 rel-L2; act_logits 2.3e-5), the logits (magnitude ~1.4) to the goldens'
    1e-5 (measured 6.8e-6, about 60 units in the last place after four layers) and the
    probabilities to 5e-6 (measured 1.3e-6: |dp_i| <= p_i (1 - p_i) |dz_i - dz_j|)."""
    cfg, cdir, w = make_model(tmp_path, 768, 12, layers=3, inter=3072, head_layers=1, vocab=500,
                              local_attention=128, seed=11)
    model = M.Model.load(cdir)
    rng = np.random.default_rng(12)
    ids, valid, pos, mask, qtype = random_batch(rng, cfg, b=3, seq=300, k=3)
    print(f"hidden 768 heads 12: valid {valid.tolist()}", flush=True)
    out = model.forward_batch(ids, valid, pos, mask, qtype)
    for i in range(len(valid)):
        want = F.forward(cfg, w, ids[i], int(valid[i]), pos[i], mask[i], int(qtype[i]))
        for name in ("logits", "probabilities", "act_logits", "features", "pooled"):
            got = getattr(out, name)[i].astype(np.float64)
            exp = np.asarray(getattr(want, name), np.float64)
            err = np.abs(got - exp)
            rel = float(np.sqrt((err ** 2).sum() / max((exp ** 2).sum(), 1e-30)))
            print(f"  seq {i} {name}: max-abs {err.max():.2e} rel-L2 {rel:.2e}")
            assert err.max() <= 1e-4 and rel <= 1e-5, (i, name, float(err.max()), rel)
        assert np.abs(out.logits[i] - want.logits).max() <= LAYER_TOL
        assert np.abs(out.probabilities[i] - want.probabilities).max() <= 5e-6


def test_split_k_in_every_epilogue(tmp_path):
    """16 tokens at hidden 1,024 and intermediate size 256: the QKV GEMM (folded norm, RoPE), the GeGLU
    GEMM (folded norm) and the Wo GEMM (residual, row statistics) divide their depth among workgroups and
    sum the partials in a second launch, the MLP's output GEMM at 3,072.  Bars as at the base width."""
    from tests.test_gemm_plan import plan

    d, room = 1024, 1 << 40
    for inter, heads in ((256, 16), (3072, 16)):
        n_splits = {"qkv": plan(16, 3 * d, d, 0, True, True, room)[3], "wo": plan(16, d, d, 0, True, True, room)[3],
                    "geglu": plan(16, inter, d, 3, True, True, room)[3], "mlp_wo": plan(16, d, inter, 0, True, True, room)[3]}
        assert all(n_splits[x] > 1 for x in (("qkv", "wo", "geglu") if inter == 256 else ("qkv", "wo", "mlp_wo"))), n_splits
        cfg, cdir, w = make_model(tmp_path, d, heads, layers=2, inter=inter, head_layers=0, vocab=100, seed=31)
        model = M.Model.load(cdir)
        rng = np.random.default_rng(32)
        ids, valid, pos, mask, qtype = random_batch(rng, cfg, b=1, seq=16, k=2)
        out = model.forward_batch(ids, valid, pos, mask, qtype)
        want = F.forward(cfg, w, ids[0], 16, pos[0], mask[0], int(qtype[0]))
        for name in ("logits", "probabilities", "act_logits", "features", "pooled"):
            got, exp = getattr(out, name)[0].astype(np.float64), np.asarray(getattr(want, name), np.float64)
            err = np.abs(got - exp)
            rel = float(np.sqrt((err ** 2).sum() / max((exp ** 2).sum(), 1e-30)))
            print(f"  inter {inter} {name}: max-abs {err.max():.2e} rel-L2 {rel:.2e}")
            assert err.max() <= 1e-4 and rel <= 1e-5, (inter, name, float(err.max()), rel)


@pytest.mark.parametrize("case", ["medium", "padded"])
def test_folded_norms_match_the_layernorm_kernels(case, monkeypatch):
    """The pre-LN LayerNorms folded into the GEMMs (statistics from the residual GEMM,
    normalisation in the next GEMM's epilogue) against the LayerNorm kernels
    (RAYA_LN_FUSION=0) on the same model: every stage within the goldens' 1e-5, both paths
    within 1e-5 of the golden."""
    cfg, model, g, valid = load_case(case)
    inp = golden_input(g, valid)
    fused = M.Trace()
    model.forward(inp, trace=fused)
    monkeypatch.setenv("RAYA_LN_FUSION", "0")
    plain = M.Trace()
    model.forward(inp, trace=plain)
    seq = g["input_ids"].shape[1]
    worst = 0.0
    for name, tol in stages(cfg):
        a, b = fused.get(name)[1], plain.get(name)[1]
        if a.ndim == 3 and a.shape[1] == seq:
            a, b = a[:, :valid], b[:, :valid]
        err = float(np.abs(a - b).max())
        worst = max(worst, err)
        assert err <= tol, (name, err)
    print(f"{case}: folded vs kernel LayerNorm, worst stage difference {worst:.2e}", flush=True)


@pytest.mark.parametrize("kappa", [5.0, 50.0])
def test_folded_norms_on_rows_far_from_zero(tmp_path, monkeypatch, kappa):
    """Residual rows 10 and 100 sigma from zero through the folded pre-LN LayerNorms.

    Every Wo gets kappa added to all its entries, so each attention output row adds the
    same kappa * sum(ctx row) to all hidden columns: the residual stream's rows drift to
    |mean| / sigma of about 2 kappa by the second layer (checked on the oracle's trace),
    where a fold that removed the mean after the contraction cancels catastrophically.
    The rank-1 term also multiplies every rounding of the context by about kappa * sqrt(d),
    on the oracle as on the device, so the stages are held to the LayerNorm kernels' own
    distance from the oracle (RAYA_LN_FUSION=0 on the same model): the folded path within
    twice that distance plus one f32 unit of the stage's magnitude, at every stage, and the
    outputs within twice that distance or the goldens' 1e-5, whichever is larger."""
    from safetensors.numpy import save_file

    cfg, cdir, w = make_model(tmp_path, 128, 2, layers=3, inter=256, head_layers=1, seed=21)
    for i in range(cfg.layers):
        name = f"encoder.layers.{i}.attn.Wo.weight"
        w[name] = (w[name] + np.float32(kappa)).astype(np.float32)
    save_file(w, os.path.join(cdir, "model.safetensors"))
    model = M.Model.load(cdir)
    rng = np.random.default_rng(22)
    ids, valid, pos, mask, qtype = random_batch(rng, cfg, b=3, seq=96, k=3)
    print(f"kappa {kappa}: valid {valid.tolist()}", flush=True)
    fused, plain = M.Trace(), M.Trace()
    out_f = model.forward_batch(ids, valid, pos, mask, qtype, trace=fused)
    monkeypatch.setenv("RAYA_LN_FUSION", "0")
    out_p = model.forward_batch(ids, valid, pos, mask, qtype, trace=plain)
    names = [f"encoder_layer_{i:02d}" for i in range(cfg.layers)] + ["encoder_final_norm", "head_layer_00"]
    for i in range(len(valid)):
        v = int(valid[i])
        want = F.forward(cfg, w, ids[i], v, pos[i], mask[i], int(qtype[i]))
        h = want.trace["encoder_layer_01"][:v].astype(np.float64)
        drift = float(np.median(np.abs(h.mean(1)) / h.std(1)))
        assert drift >= kappa, drift
        for name in names:
            ref = want.trace[name][:v]
            ef = float(np.abs(fused.get(name)[1][i, :v] - ref).max())
            ep = float(np.abs(plain.get(name)[1][i, :v] - ref).max())
            unit = float(np.spacing(np.float32(np.abs(ref).max())))
            print(f"  seq {i} {name}: folded {ef:.2e}, LayerNorm kernels {ep:.2e} (drift {drift:.0f} sigma)")
            assert ef <= 2 * ep + unit, (i, name, ef, ep)
        for name in ("logits", "probabilities", "act_logits", "pooled"):
            ef = float(np.abs(getattr(out_f, name)[i] - getattr(want, name)).max())
            ep = float(np.abs(getattr(out_p, name)[i] - getattr(want, name)).max())
            print(f"  seq {i} {name}: folded {ef:.2e}, LayerNorm kernels {ep:.2e}")
            assert ef <= max(2 * ep, LAYER_TOL), (i, name, ef, ep)
