"""The work this framework is timed on: attention launches, encoder GEMMs, the post-LN layer and
the decision model, called as a program calls them.

`listed()` holds the fixed cases, `draw(rng)` one more of the same ranges.  `prepare` makes what a
program has in hand before the call (inputs, weights, handles), `run` is one pass through the
public entry points and returns its whole outputs, `exact` the same outputs from plain torch in
64 bits.  Inputs are N(0, 1), weights N(0, 0.02), as in the throughput benchmark; lengths of a
padded batch are spread evenly over their range and dealt to the sequences by the seed.
"""
import json
import math
import os
import tempfile

import numpy as np
import torch

import raya_amd as R
from raya_amd import _capi as C
from raya_amd.checkpoint import MODERNBERT_BASE, expected_params, write_config
from raya_amd.layers import PostLNLayer
from raya_amd.model import Model

ACTS = {"none": C.RAYA_EPI_NONE, "gelu": C.RAYA_EPI_GELU, "relu": C.RAYA_EPI_RELU, "geglu": C.RAYA_EPI_GEGLU}
HIDDEN, HEADS, FFN = 768, 12, 3072  # the model's layers
REF_BLOCK, REF_WINDOW = 128, 64     # Block3's block, Window64's half-width
AGENT = {"head_layers": 0, "act_costs": {"abstain": 0.1}}
HEAD_EPS = 1e-5


def _attention(name, batch, heads, seq, head_dim, mask, arg, lo, packed=False):
    return {"name": name, "kind": "attention", "batch": batch, "heads": heads, "seq": seq, "head_dim": head_dim,
            "mask": mask, "arg": arg, "valid_lo": lo, "packed": packed}


def _gemm(name, m, n, k, act, bias, residual):
    return {"name": name, "kind": "gemm", "m": m, "n": n, "k": k, "act": act, "bias": bias, "residual": residual}


def listed():
    return [
        # The benchmark's headline: a padded batch, every query in its own 64-token block.
        _attention("attn_blockdiag64_b32_l2048", 32, 12, 2048, 64, "block_diag", 64, 512),
        # One short sequence under the reference's own mask: launch and latency.
        _attention("attn_block3_b1_l512", 1, 12, 512, 64, "block3", 0, 512),
        # The reference bench's largest shape: 16 heads of 8192 rows under Block3.
        _attention("attn_block3_h16_l8192", 1, 16, 8192, 64, "block3", 0, 8192),
        # A local layer of the model: Sliding(64) on a padded batch, read out of the packed QKV projection.
        _attention("attn_sliding64_b16_l1000_packed", 16, 12, 1000, 64, "sliding", 64, 200, packed=True),
        # A global layer of the model on longer sequences: every key.
        _attention("attn_full_b4_l2048_packed", 4, 12, 2048, 64, "full", 0, 1024, packed=True),
        # A wider head at a ragged length.
        _attention("attn_block3_d128_b2_l3000", 2, 8, 3000, 128, "block3", 0, 3000),
        # The trait's own call: host slices in and out, copies included.
        {"name": "attend_host_block3_l512", "kind": "attend_host", "heads": 12, "seq": 512, "head_dim": 64,
         "mask": "block3", "arg": 0},
        # The largest projection input of the encoder benchmark: 21,405 packed tokens through Wqkv.
        _gemm("gemm_qkv_m21405", 21405, 3 * HIDDEN, HIDDEN, "none", True, False),
        # The act head's first Linear on a batch: few rows, a depth (hidden + 4) of no round size.
        _gemm("gemm_act_head_m64", 64, 256, HIDDEN + 4, "gelu", True, False),
        # One post-LN layer as BERT writes it, 16 sequences of 1024 tokens.
        {"name": "postln_b16_l1024", "kind": "postln", "batch": 16, "seq": 1024, "valid_lo": 1024,
         "mask": "block_diag", "arg": 64},
        # One 512-token predict through the 12-layer decision model: the serving call.
        {"name": "predict_l512", "kind": "model", "batch": 1, "seq": 512, "valid_lo": 512, "markers": 2},
        # The encoder benchmark: 64 padded sequences of up to 512 tokens in one pass.
        {"name": "encoder_b64_l512", "kind": "model", "batch": 64, "seq": 512, "valid_lo": 128, "markers": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["attention", "gemm", "postln", "model", "attend_host"], [9, 8, 3, 2, 2])[0]
    if kind in ("attention", "attend_host"):
        mask, arg = rng.choice([("block_diag", 64), ("block_diag", 128), ("block_diag", 32), ("block3", 0),
                                ("window64", 0), ("sliding", 64), ("sliding", rng.randint(4, 256)), ("full", 0)])
        heads, dim = rng.randint(2, 16), rng.choice([64, 64, 64, 32, 40, 96, 128])
        if kind == "attend_host":
            return {"kind": kind, "heads": heads, "seq": _log_int(rng, 17, 2048), "head_dim": dim, "mask": mask,
                    "arg": arg}
        seq = _log_int(rng, 33, 8192)
        batch = _log_int(rng, 1, max(1, min(32, 65536 // seq)))
        case = _attention(None, batch, heads, seq, dim, mask, arg, rng.randint(max(1, seq // 4), seq),
                          packed=rng.random() < 0.4)
        while case["batch"] > 1 and work(case)["flops"] > 4e11:
            case["batch"] //= 2
    elif kind == "gemm":
        k = 16 * _log_int(rng, 4, 192) if rng.random() < 0.6 else _log_int(rng, 64, 3072)
        case = _gemm(None, _log_int(rng, 1, 21405), _log_int(rng, 64, 6144), k, rng.choice(list(ACTS)),
                     rng.random() < 0.7, rng.random() < 0.4)
        if case["act"] == "geglu":
            case["n"] = max(32, case["n"] // 2)
    elif kind == "postln":
        seq = _log_int(rng, 48, 2048)
        case = {"kind": kind, "batch": _log_int(rng, 1, max(1, 16384 // seq)), "seq": seq,
                "valid_lo": rng.randint(max(1, seq // 4), seq)}
        case["mask"], case["arg"] = rng.choice([("block_diag", 64), ("block3", 0), ("sliding", 64), ("full", 0)])
    else:
        seq = _log_int(rng, 16, 4096)
        case = {"kind": kind, "batch": _log_int(rng, 1, max(1, 8192 // seq)), "seq": seq,
                "valid_lo": rng.randint(max(8, seq // 4), seq), "markers": rng.randint(2, 6)}
    case.pop("name", None)
    return case


# --- masks, lengths and the work of a pass ----------------------------------------------------

def _mask(case):
    name, arg = case["mask"], case["arg"]
    return {"block3": R.Mask.BLOCK3, "window64": R.Mask.WINDOW64, "full": R.Mask.FULL}.get(name) or (
        R.Mask.sliding(arg) if name == "sliding" else R.Mask.block_diag(arg))


def _ranges(mask, arg, v):
    """(lo, hi) of the keys each row i < v sees."""
    i = np.arange(v, dtype=np.int64)
    if mask == "block3":
        lo, hi = (i // REF_BLOCK - 1) * REF_BLOCK, (i // REF_BLOCK + 2) * REF_BLOCK
    elif mask == "block_diag":
        lo, hi = i // arg * arg, (i // arg + 1) * arg
    elif mask == "full":
        lo, hi = 0 * i, 0 * i + v
    else:
        w = REF_WINDOW if mask == "window64" else arg
        lo, hi = i - w, i + w + 1
    return np.maximum(lo, 0), np.minimum(hi, v)


def _pairs(mask, arg, lengths):
    total = 0
    for v in lengths:
        lo, hi = _ranges(mask, arg, int(v))
        total += int((hi - lo).sum())
    return total


def _lengths(case):
    """Evenly spread over [valid_lo, seq]: the same total for every seed."""
    return np.linspace(case["valid_lo"], case["seq"], case["batch"]).round().astype(np.int64) \
        if case["batch"] > 1 else np.array([case["seq"]], np.int64)


def _dealt(case, seed):
    return np.random.default_rng([seed, 7]).permutation(_lengths(case))


def _model_masks():
    """(mask, arg, rope base) of every layer: each third sees every key, the rest a sliding window."""
    c = MODERNBERT_BASE
    rope = c["rope_parameters"]
    return [("full", 0, rope["full_attention"]["rope_theta"]) if i % c["global_attn_every_n_layers"] == 0 else
            ("sliding", c["local_attention"] // 2, rope["sliding_attention"]["rope_theta"])
            for i in range(c["num_hidden_layers"])]


def work(case):
    kind = case["kind"]
    if kind in ("attention", "attend_host"):
        h, s, d = case["heads"], case["seq"], case["head_dim"]
        lengths = _lengths(case) if kind == "attention" else [s]
        return {"bytes": 4 * (3 * h * d * int(sum(lengths)) + len(lengths) * h * s * d),
                "flops": 4 * d * h * _pairs(case["mask"], case["arg"], lengths)}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        rows = 2 * n if case["act"] == "geglu" else n
        return {"bytes": 4 * (m * k + rows * k + m * n + rows * case["bias"] + m * n * case["residual"]),
                "flops": 2 * m * rows * k}
    lengths = _lengths(case)
    if kind == "postln":
        tokens = case["batch"] * case["seq"]
        weights = 4 * HIDDEN * HIDDEN + 2 * HIDDEN * FFN + 9 * HIDDEN + FFN
        return {"bytes": 4 * (2 * tokens * HIDDEN + weights),
                "flops": 2 * tokens * HIDDEN * (4 * HIDDEN + 2 * FFN)
                + 4 * HIDDEN * _pairs(case["mask"], case["arg"], lengths)}
    layers, tokens = _model_masks(), int(lengths.sum())
    per_token = 2 * HIDDEN * (4 * HIDDEN + 3 * FFN)
    weights = len(layers) * HIDDEN * (4 * HIDDEN + 3 * FFN)
    return {"bytes": 4 * (weights + tokens * (HIDDEN + 1) + case["batch"] * HIDDEN),
            "flops": len(layers) * tokens * per_token
            + 4 * HIDDEN * sum(_pairs(mask, arg, lengths) for mask, arg, _ in layers)}


# --- inputs -----------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1 + seed)


def _randn(gen, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=gen).mul_(std)


def _attention_inputs(case, seed):
    b, h, s, d = case.get("batch", 1), case["heads"], case["seq"], case["head_dim"]
    gen = _gen(seed)
    return [_randn(gen, b, h, s, d) for _ in range(3)]


def _gemm_inputs(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    rows = 2 * n if case["act"] == "geglu" else n
    gen = _gen(seed)
    a, w = _randn(gen, m, k), _randn(gen, rows, k, std=0.02)
    bias = _randn(gen, rows, std=0.02) if case["bias"] else None
    return a, w, bias, _randn(gen, m, n) if case["residual"] else None


def _postln_inputs(case, seed):
    gen = _gen(seed)
    d, f = HIDDEN, FFN
    x = _randn(gen, case["batch"], case["seq"], d)
    w = {"wqkv": _randn(gen, 3 * d, d, std=0.02), "wo": _randn(gen, d, d, std=0.02),
         "w1": _randn(gen, f, d, std=0.02), "w2": _randn(gen, d, f, std=0.02)}
    for name, n in (("bqkv", 3 * d), ("bo", d), ("b1", f), ("b2", d), ("ln1_b", d), ("ln2_b", d)):
        w[name] = _randn(gen, n, std=0.02)
    for name in ("ln1_w", "ln2_w"):
        w[name] = 1.0 + _randn(gen, d, std=0.02)
    return x, w


def _model_weights(folder, seed):
    """Every parameter of the 12-layer model, in the checkpoint's order, on the GPU."""
    gen = _gen(seed)
    out = {}
    for name, shape in expected_params(folder):
        x = _randn(gen, *shape, std=0.02)
        if name.endswith(("norm.weight", "norm1.weight", "norm2.weight")) or name in ("scorer.0.weight",
                                                                                     "temperature"):
            x += 1.0
        out[name] = x
    return out


def _save(path, tensors):
    """A safetensors file: the header's length, the header, the tensors' bytes."""
    header, at = {}, 0
    for name, t in tensors.items():
        n = t.numel() * 4
        header[name] = {"dtype": "F32", "shape": list(t.shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(path, "wb") as f:
        f.write(len(text).to_bytes(8, "little"))
        f.write(text)
        for t in tensors.values():
            f.write(memoryview(t.cpu().numpy().reshape(-1)).cast("B"))


def _model_inputs(case, seed):
    """Token ids with a leading CLS id, lengths, markers at the first positions, question types."""
    b, s, k = case["batch"], case["seq"], case["markers"]
    rng = np.random.default_rng([seed, 3])
    ids = rng.integers(1000, MODERNBERT_BASE["vocab_size"], (b, s)).astype(np.uint32)
    ids[:, 0] = MODERNBERT_BASE["cls_token_id"]
    pos = np.tile(np.arange(1, k + 1, dtype=np.uint64), (b, 1))
    return ids, _dealt(case, seed).astype(np.uint64), pos, np.ones((b, k), np.uint8), \
        rng.integers(0, 3, b).astype(np.uint64)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attention":
        b, h, s, d = case["batch"], case["heads"], case["seq"], case["head_dim"]
        qkv = _attention_inputs(case, seed)
        layouts = None
        if case["packed"]:  # [batch][seq][q | k | v][heads][head_dim], the projection's own layout
            rows = torch.stack([x.transpose(1, 2) for x in qkv], dim=2).reshape(b, s, 3 * h * d).contiguous()
            qkv = [rows[:, :, i * h * d:] for i in range(3)]
            lay, out = (s * 3 * h * d, d, 3 * h * d), torch.empty(b, s, h * d, device="cuda")
            layouts = {"shape": (b, h, s, d), "q": lay, "k": lay, "v": lay, "out": (s * h * d, d, h * d)}
        else:
            out = torch.empty(b, h, s, d, device="cuda")
        return {"kind": kind, "kernel": R.HipAttention(), "qkv": qkv, "out": out, "mask": _mask(case),
                "layouts": layouts, "valid": torch.from_numpy(_dealt(case, seed).astype(np.int32)).cuda()}
    if kind == "attend_host":
        h, s, d = case["heads"], case["seq"], case["head_dim"]
        qkv = [x.cpu().numpy().reshape(-1) for x in _attention_inputs(case, seed)]
        return {"kind": kind, "kernel": R.HipAttention(), "qkv": qkv, "out": np.empty(h * s * d, np.float32),
                "shape": R.AttnShape(h, s, d), "params": R.AttnParams.new(_mask(case), s, d)}
    if kind == "gemm":
        a, w, bias, residual = _gemm_inputs(case, seed)
        return {"kind": kind, "gemm": R.HipGemm(), "a": a, "w": w, "bias": bias, "residual": residual,
                "act": ACTS[case["act"]], "out": torch.empty(case["m"], case["n"], device="cuda")}
    if kind == "postln":
        x, w = _postln_inputs(case, seed)
        return {"kind": kind, "layer": PostLNLayer(w, HEADS, mask=_mask(case)), "x": x, "out": torch.empty_like(x),
                "valid": torch.from_numpy(_dealt(case, seed).astype(np.int32)).cuda()}
    with tempfile.TemporaryDirectory() as folder:
        write_config(folder, MODERNBERT_BASE, AGENT)
        _save(os.path.join(folder, "model.safetensors"), _model_weights(folder, seed))
        model = Model.load(folder)
    return {"kind": kind, "model": model, "inputs": _model_inputs(case, seed)}


def run(state):
    kind = state["kind"]
    if kind == "attention":
        state["kernel"].attend_batched(*state["qkv"], state["out"], state["valid"], state["mask"],
                                       layouts=state["layouts"])
        return state["out"]
    if kind == "attend_host":
        state["kernel"].attend(state["shape"], state["params"], *state["qkv"], state["out"])
        return state["out"]
    if kind == "gemm":
        state["gemm"].matmul_nt_device(state["out"], state["a"], state["w"], bias=state["bias"],
                                       activation=state["act"], residual=state["residual"])
        return state["out"]
    if kind == "postln":
        return state["layer"].forward(state["x"], state["valid"], out=state["out"])
    o = state["model"].forward_batch(*state["inputs"])
    return [o.logits, o.probabilities, o.act_logits, o.features, o.pooled]


def tolerance(case):
    # About four times what the start shows against 64 bits, over the listed cases and draws.
    kind = case["kind"]
    if kind in ("attention", "attend_host"):
        return {"rel": 4e-6}
    if kind == "gemm":
        return {"rel": 4e-6}
    if kind == "postln":
        return {"rel": 2e-6}
    return {"rel": 1.2e-5}


# --- the same in 64 bits ----------------------------------------------------------------------

def _attend64(q, k, v, mask, arg, valid):
    """q, k, v [heads, rows, dim] in float64: the rows below valid attend, the rest are zero."""
    out = torch.zeros_like(q)
    lo, hi = _ranges(mask, arg, valid)
    scale = 1.0 / math.sqrt(q.shape[2])
    step = 512
    keys = torch.arange(valid, device=q.device)
    lo_t, hi_t = torch.from_numpy(lo).to(q.device), torch.from_numpy(hi).to(q.device)
    for r0 in range(0, valid, step):
        r1 = min(r0 + step, valid)
        k0, k1 = int(lo[r0:r1].min()), int(hi[r0:r1].max())
        s = torch.matmul(q[:, r0:r1] * scale, k[:, k0:k1].transpose(1, 2).contiguous())
        j = keys[k0:k1]
        s.masked_fill_((j < lo_t[r0:r1, None]) | (j >= hi_t[r0:r1, None]), -math.inf)
        out[:, r0:r1] = torch.matmul(torch.softmax(s, -1), v[:, k0:k1].contiguous())
    return out


def _norm64(x, w, b, eps):
    y = torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps) * w
    return y if b is None else y + b


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _exact_model(case, seed):
    with tempfile.TemporaryDirectory() as folder:
        write_config(folder, MODERNBERT_BASE, AGENT)
        w = _model_weights(folder, seed)
    ids, valid, pos, _, qtype = _model_inputs(case, seed)
    d, hd, eps = HIDDEN, HIDDEN // HEADS, MODERNBERT_BASE["norm_eps"]
    valid = [int(x) for x in valid]
    starts = np.concatenate([[0], np.cumsum(valid)]).astype(np.int64)
    token = torch.from_numpy(np.concatenate([ids[b, :v] for b, v in enumerate(valid)]).astype(np.int64)).cuda()
    place = torch.from_numpy(np.concatenate([np.arange(v) for v in valid]).astype(np.float32)).cuda()
    lin = lambda x, name: x @ w[name].double().T
    h = _norm64(w["encoder.embeddings.tok_embeddings.weight"][token].double(),
                w["encoder.embeddings.norm.weight"].double(), None, eps)
    for i, (mask, arg, theta) in enumerate(_model_masks()):
        p = f"encoder.layers.{i}"
        x = h if i == 0 else _norm64(h, w[f"{p}.attn_norm.weight"].double(), None, eps)
        qkv = lin(x, f"{p}.attn.Wqkv.weight").reshape(-1, 3, HEADS, hd)
        # The rotary angles are the model's own 32-bit numbers: position times 1 / theta^(2i / dim).
        inv = 1.0 / torch.pow(torch.tensor(theta, dtype=torch.float32),
                              torch.arange(0, hd, 2, dtype=torch.float32) / hd)
        angle = (place[:, None] * inv.cuda()).double()
        cos, sin = angle.cos()[:, None, None], angle.sin()[:, None, None]
        a, b = qkv[:, :2, :, :hd // 2], qkv[:, :2, :, hd // 2:]
        qk = torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        ctx = torch.empty_like(h)
        for r0, v in zip(starts, valid):
            q3 = [t[r0:r0 + v].transpose(0, 1).contiguous() for t in (qk[:, 0], qk[:, 1], qkv[:, 2])]
            ctx[r0:r0 + v] = _attend64(*q3, mask, arg, v).transpose(0, 1).reshape(v, d)
        h = h + lin(ctx, f"{p}.attn.Wo.weight")
        wi = lin(_norm64(h, w[f"{p}.mlp_norm.weight"].double(), None, eps), f"{p}.mlp.Wi.weight")
        h = h + lin(_gelu64(wi[:, :FFN]) * wi[:, FFN:], f"{p}.mlp.Wo.weight")
    h = _norm64(h, w["encoder.final_norm.weight"].double(), None, eps)
    first = torch.from_numpy(starts[:-1]).cuda()
    add = w["type_emb.weight"].double()[torch.from_numpy(qtype.astype(np.int64)).cuda()]
    states = h[first[:, None] + torch.from_numpy(pos.astype(np.int64)).cuda()] + add[:, None]
    x = _norm64(states, w["scorer.0.weight"].double(), w["scorer.0.bias"].double(), HEAD_EPS)
    x = _gelu64(lin(x, "scorer.1.weight") + w["scorer.1.bias"].double())
    logits = (lin(x, "scorer.3.weight") + w["scorer.3.bias"].double())[..., 0]
    probs = torch.softmax(logits, -1)
    n = max(case["markers"], 2)
    top = probs.topk(2, -1).values
    entropy = -(probs * probs.clamp_min(1e-9).log()).sum(-1)
    feats = torch.stack([top[:, 0], top[:, 0] - top[:, 1], entropy / math.log(n),
                         torch.full_like(entropy, n / 255.0)], -1)
    pooled = h[first] + add
    x = _gelu64(lin(torch.cat([pooled, feats], -1), "act_head.0.weight") + w["act_head.0.bias"].double())
    act = lin(x, "act_head.2.weight") + w["act_head.2.bias"].double()
    return [t.cpu().numpy() for t in (logits, probs, act, feats, pooled)]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("attention", "attend_host"):
        q, k, v = _attention_inputs(case, seed)
        valid = [case["seq"]] if kind == "attend_host" else _dealt(case, seed)
        out = torch.stack([_attend64(q[b].double(), k[b].double(), v[b].double(), case["mask"], case["arg"], int(n))
                           for b, n in enumerate(valid)])
        if kind == "attend_host":
            return out.reshape(-1).cpu().numpy()
        return out.transpose(1, 2).reshape(q.shape[0], q.shape[2], -1) if case["packed"] else out
    if kind == "gemm":
        a, w, bias, residual = _gemm_inputs(case, seed)
        y = a.double() @ w.double().T
        y = y if bias is None else y + bias.double()
        n = case["n"]
        y = {"none": lambda: y, "gelu": lambda: _gelu64(y), "relu": lambda: y.clamp_min(0.0),
             "geglu": lambda: _gelu64(y[:, :n]) * y[:, n:]}[case["act"]]()
        return y if residual is None else y + residual.double()
    if kind == "postln":
        x, w = _postln_inputs(case, seed)
        x, w = x.double(), {name: t.double() for name, t in w.items()}
        b, s, d = x.shape
        qkv = (x @ w["wqkv"].T + w["bqkv"]).reshape(b, s, 3, HEADS, d // HEADS)
        ctx = torch.stack([_attend64(*(qkv[i, :, j].transpose(0, 1).contiguous() for j in range(3)), case["mask"],
                                     case["arg"], int(n)).transpose(0, 1).reshape(s, d)
                           for i, n in enumerate(_dealt(case, seed))])
        y = _norm64(x + ctx @ w["wo"].T + w["bo"], w["ln1_w"], w["ln1_b"], 1e-12)
        f = _gelu64(y @ w["w1"].T + w["b1"])
        return _norm64(y + f @ w["w2"].T + w["b2"], w["ln2_w"], w["ln2_b"], 1e-12)
    return _exact_model(case, seed)
