"""The 128-row attention kernel (head_dim 64 and 128) on three-part bfloat16 products, forced with RAYA_ATTN_ITEMS=128:
edges of its tiles and waves under every mask it takes, strided and padded batches, non-finite
operands, and its instrumented copy.

Bars as in test_attention_gpu.py: max-abs 1e-5 and rel-L2 1e-5 against the oracle's Naive (an fp32
reordering bar; the parts carry all 24 bits of every operand), exact zeros on padded rows.
"""
import numpy as np
import pytest
import torch

import oracle
import raya_amd as R
from raya_amd import synth

pytestmark = pytest.mark.gpu

MASKS = {"block3": (R.Mask.BLOCK3, oracle.MASK_BLOCK3, 128, 0), "full": (R.Mask.FULL, oracle.MASK_FULL, 0, 0),
         "sliding64": (R.Mask.sliding(64), oracle.MASK_SLIDING, 0, 64),
         "sliding7": (R.Mask.sliding(7), oracle.MASK_SLIDING, 0, 7),
         "sliding200": (R.Mask.sliding(200), oracle.MASK_SLIDING, 0, 200)}


@pytest.fixture(autouse=True)
def items128(monkeypatch):
    monkeypatch.setenv("RAYA_ATTN_ITEMS", "128")


def inputs(seed, h, s, d=64):
    return [synth.normal(1000 * seed + i, h * s * d).reshape(h, s, d) for i in range(3)]


def naive(q, k, v, name, valid, scale=0.125):
    _, kind, block, window = MASKS[name]
    return oracle.naive_attend(q, k, v, kind, valid, scale, block=block, window=window)


def close(got, want):
    assert np.isfinite(got).all()
    diff = np.abs(got - want)
    assert diff.max() <= 1e-5, diff.max()
    assert np.sqrt((diff.astype(np.float64) ** 2).sum()) <= 1e-5 * np.sqrt((want.astype(np.float64) ** 2).sum())


@pytest.mark.parametrize("name", list(MASKS))
@pytest.mark.parametrize("seq", [1, 31, 33, 64, 127, 129, 300, 513])
@pytest.mark.parametrize("d", [64, 128])
def test_edges(hip_attention, name, seq, d):
    """One launch of sequences whose valid lengths end at, before and after every kind of edge."""
    h = 2
    lens = sorted({max(0, min(seq, n)) for n in (0, 1, 16, 32, 65, 128, 130, 257, seq - 1, seq)})
    qkv = [inputs(100 + n, h, seq, d) for n in range(len(lens))]
    dev = [torch.from_numpy(np.stack([x[i] for x in qkv])).cuda() for i in range(3)]
    out = torch.full_like(dev[0], 7.0)
    print(f"{name} seq {seq} lens {lens}", flush=True)
    hip_attention.attend_batched(*dev, out, torch.tensor(lens, dtype=torch.int32, device="cuda"), MASKS[name][0],
                                 0.125)
    got = out.cpu().numpy()
    for b, n in enumerate(lens):
        assert (got[b, :, n:] == 0).all()
        if n:
            close(got[b, :, :n], naive(*qkv[b], name, n)[:, :n])


@pytest.mark.parametrize("name", ["block3", "full", "sliding64"])
@pytest.mark.parametrize("scale", [-0.2, 0.0, 0.125])
def test_packed_projection_and_scales(hip_attention, name, scale):
    """Heads read out of a [batch][seq][3 heads dim] projection with padded rows between."""
    b, h, s, d, pad = 2, 3, 260, 64, 8
    width = 3 * h * d + pad
    rows = torch.from_numpy(synth.normal(77, b * s * width).reshape(b, s, width)).cuda()
    out = torch.full((b, s, h * d + 4), 9.0, device="cuda")
    lay = (s * width, d, width)
    hip_attention.attend_batched(rows, rows[:, :, h * d:], rows[:, :, 2 * h * d:], out,
                                 torch.tensor([s, 200], dtype=torch.int32, device="cuda"), MASKS[name][0], scale,
                                 layouts={"shape": (b, h, s, d), "q": lay, "k": lay, "v": lay,
                                          "out": (s * (h * d + 4), d, h * d + 4)})
    got, x = out.cpu().numpy(), rows.cpu().numpy()
    assert (got[:, :, h * d:] == 9.0).all()
    for i, n in enumerate((s, 200)):
        q, k, v = (np.ascontiguousarray(x[i, :, j * h * d:(j + 1) * h * d].reshape(s, h, d).transpose(1, 0, 2))
                   for j in range(3))
        have = got[i, :, :h * d].reshape(s, h, d).transpose(1, 0, 2)
        assert (have[:, n:] == 0).all()
        close(have[:, :n], naive(q, k, v, name, n, scale)[:, :n])


@pytest.mark.parametrize("name", list(MASKS))
@pytest.mark.parametrize("operand", [0, 1, 2])
@pytest.mark.parametrize("d", [64, 128])
def test_non_finite_operands_match_the_reference(hip_attention, name, operand, d):
    """Inf, -Inf, NaN and 3.4e38 in one row of q, k or v at a time: NaN and Inf where Naive has
    them, its values elsewhere."""
    h, s, valid = 1, 300, 290
    for at, value in ((0, np.inf), (63, -np.inf), (130, np.nan), (valid - 1, -np.inf), (200, 3.4e38)):
        x = inputs(9, h, s, d)
        x[operand][0, at, 5] = value
        with np.errstate(all="ignore"):
            want = naive(*x, name, valid)
        out = np.full(h * s * d, 7.0, np.float32)
        hip_attention.attend(R.AttnShape(h, s, d), R.AttnParams(MASKS[name][0], 128, valid, 0.125),
                             *(t.reshape(-1) for t in x), out)
        got = out.reshape(want.shape)
        assert np.array_equal(np.isnan(got), np.isnan(want)), (at, value)
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), (at, value)
        ok = np.isfinite(want)
        assert (np.abs(got[ok] - want[ok]) <= 1e-5 * np.maximum(1.0, np.abs(want[ok]))).all(), (at, value)


@pytest.mark.parametrize("name", ["block3", "full", "sliding64"])
@pytest.mark.parametrize("d", [64, 128])
def test_error_is_no_larger_than_the_fp32_kernels(hip_attention, monkeypatch, name, d):
    """RMS distance from float64 attention, against the 64-row kernel's on the fp32 instruction."""
    h, s = 4, 1024
    x = inputs(5, h, s, d)
    dev = [torch.from_numpy(t[None]).cuda() for t in x]
    valid = torch.tensor([s], dtype=torch.int32, device="cuda")
    outs = {}
    for items in ("128", "64"):
        monkeypatch.setenv("RAYA_ATTN_ITEMS", items)
        outs[items] = torch.empty_like(dev[0])
        hip_attention.attend_batched(*dev, outs[items], valid, MASKS[name][0], 0.125)
    q, k, v = (t[0].double() for t in dev)
    i = torch.arange(s, device="cuda")
    seen = {"block3": (i[:, None] // 128 - i[None] // 128).abs() <= 1, "full": (i[:, None] >= 0) & (i[None] >= 0),
            "sliding64": (i[:, None] - i[None]).abs() <= 64}[name]
    w = torch.softmax((torch.matmul(q, k.transpose(1, 2).contiguous()) * 0.125).masked_fill(~seen, -np.inf), -1)
    want = torch.matmul(w, v)
    rms = {n: float(((o[0].double() - want) ** 2).mean().sqrt()) for n, o in outs.items()}
    print(name, rms)
    assert rms["128"] <= 1.05 * rms["64"]


@pytest.mark.parametrize("name", ["block3", "sliding64"])
@pytest.mark.parametrize("d", [64, 128])
def test_stages(hip_attention, name, d):
    """The instrumented copy: the same outputs, the tiles of 16 rows x 64 keys it computes (two to
    a wave of 32 rows that meets the tile, one if its second 16 are padding)."""
    seq, heads, lens = 512, 2, [512, 300]
    dev = [torch.from_numpy(np.stack([inputs(n, heads, seq, d)[i] for n in (1, 2)])).cuda() for i in range(3)]
    valid = torch.tensor(lens, dtype=torch.int32, device="cuda")
    mask = MASKS[name][0]
    plain = torch.empty_like(dev[0])
    hip_attention.attend_batched(*dev, plain, valid, mask)
    timed = torch.empty_like(plain)
    st = hip_attention.attend_batched_stages(*dev, timed, valid, mask)
    assert torch.equal(timed, plain)
    assert st.qk > 0 and st.softmax > 0 and st.pv > 0 and st.load_wait > 0
    n = 0
    for v in lens:
        for q0 in range(0, v, 128):
            lo = mask.key_range(q0, v).start
            hi = mask.key_range(min(q0 + 128, v) - 1, v).stop
            for kt in range(lo, hi, 64):
                for w in range(q0, min(q0 + 128, v), 32):
                    a, z = mask.key_range(w, v), mask.key_range(min(w + 31, v - 1), v)
                    meets = any(t < z.stop and t + 32 > a.start for t in (kt, kt + 32))
                    n += (2 if w + 16 < v else 1) if meets else 0
    assert st.tiles == n * heads


@pytest.mark.parametrize("name", ["block3", "full", "sliding200"])
@pytest.mark.parametrize("d", [64, 128])
def test_out_may_be_q(hip_attention, name, d):
    """q overwritten by its own outputs, some of them not finite: the same bits as in a separate out."""
    h, s = 3, 300
    q, k, v = (torch.from_numpy(x[None]).cuda() for x in inputs(11, h, s, d))
    q[0, 0, 70, 1] = float("nan")
    q[0, 1, 129, 0] = float("inf")
    v[0, 2, 40, 3] = float("nan")
    valid = torch.tensor([290], dtype=torch.int32, device="cuda")
    out = torch.full_like(q, 7.0)
    hip_attention.attend_batched(q, k, v, out, valid, MASKS[name][0], 0.125)
    assert not torch.isfinite(out).all()
    hip_attention.attend_batched(q, k, v, q, valid, MASKS[name][0], 0.125)
    assert torch.equal(q.view(torch.int32), out.view(torch.int32))


@pytest.mark.parametrize("name", list(MASKS))
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("eq,ek,ev", [(0, 0, -120), (124, -124, 0), (-124, 124, 0), (-79, 79, 0), (-82, 82, 0), (100, -100, 100),
                                      (0, 0, 81), (0, 0, 120), (60, -60, -90)])
def test_operands_of_any_size(hip_attention, name, d, eq, ek, ev):
    """Operands of 2^eq, 2^ek and 2^ev, scores of order one: rel-L2 1e-5 around float64 as at every
    other size (the smallest lose no bits, the largest are left to the fp32 body)."""
    h, s, valid = 2, 300, 290
    x = [torch.from_numpy(t[None]).cuda() * 2.0 ** e for t, e in zip(inputs(21, h, s, d), (eq, ek, ev))]
    out = torch.full_like(x[0], 7.0)
    hip_attention.attend_batched(*x, out, torch.tensor([valid], dtype=torch.int32, device="cuda"), MASKS[name][0], 0.125)
    assert (out[:, :, valid:] == 0).all()
    q, k, v = (t[0, :, :valid].double() for t in x)
    kind, block, window = MASKS[name][1:]
    i = torch.arange(valid, device="cuda")
    seen = {oracle.MASK_BLOCK3: (i[:, None] // 128 - i[None] // 128).abs() <= 1, oracle.MASK_FULL: i[:, None] >= i[None] * 0,
            oracle.MASK_SLIDING: (i[:, None] - i[None]).abs() <= window}[kind]
    w = torch.softmax((torch.matmul(q, k.transpose(1, 2).contiguous()) * 0.125).masked_fill(~seen, -np.inf), -1)
    want = torch.matmul(w, v) * 2.0 ** -ev
    got = out[0, :, :valid].double() * 2.0 ** -ev
    assert float((got - want).norm() / want.norm()) <= 1e-5
    assert float((got - want).abs().max()) <= 1e-5


@pytest.mark.parametrize("d", [64, 128])
def test_tiny_weights_of_huge_values(hip_attention, d):
    """Keys that weigh about 2^-112 with V of 2^104: their part of the sum counts as much as the rest."""
    h, s = 1, 256
    q, k, v = (torch.from_numpy(t[None]).cuda() for t in inputs(22, h, s, d))
    q[:], k[:] = 0.0, 0.0
    q[..., 0] = 1.0
    k[..., ::2, 0] = -112 * float(np.log(2)) * 8 + 0.1 * k[..., ::2, 1]
    v[..., ::2, :] *= 2.0 ** 104
    v[..., 1::2, :] *= 2.0 ** -8
    out = torch.full_like(q, 7.0)
    hip_attention.attend_batched(q, k, v, out, torch.tensor([s], dtype=torch.int32, device="cuda"), R.Mask.FULL, 0.125)
    w = torch.softmax(torch.matmul(q[0].double(), k[0].double().transpose(1, 2).contiguous()) * 0.125, -1)
    want = torch.matmul(w, v[0].double())
    # The exponents' own rounding: -112 with 24 bits is off by 2^-18, its weight by 2.6e-6.
    assert float((out[0].double() - want).norm() / want.norm()) <= 2e-5


def attend(hip_attention, x, lens, mask):
    out = torch.full_like(x[0], 7.0)
    hip_attention.attend_batched(*x, out, torch.tensor(lens, dtype=torch.int32, device="cuda"), mask)
    return out


@pytest.mark.parametrize("seq", [4096, 2000, 500, 260, 100])
@pytest.mark.parametrize("name", ["block3", "full", "sliding200"])
@pytest.mark.parametrize("d", [64, 128])
def test_item_orders(hip_attention, monkeypatch, name, seq, d):
    """Every order of the items computes each of them once: whole pairs per XCD, their tiles rotated
    from pair to pair (32, 16, 4, 3 and 1 tiles a pair), units of 1, 2 and 4 tiles, and 7 pairs (the scattered
    order).  The same bits as the sequences' own launches."""
    for b, h in ((4, 2), (24, 1), (7, 1)):
        if b * seq > 20000:
            continue
        lens = [seq, max(1, seq // 3), 0, min(seq, 129), min(seq, 128), 1, seq - 1][:b] + [seq // 2] * (b - 7)
        x = [torch.from_numpy(synth.normal(31 + i, b * h * seq * d).reshape(b, h, seq, d)).cuda() for i in range(3)]
        monkeypatch.delenv("RAYA_ATTN_ORDER", raising=False)
        want = torch.cat([attend(hip_attention, [t[i:i + 1].contiguous() for t in x], lens[i:i + 1], MASKS[name][0])
                          for i in range(b)])
        for order in (None, "pairs", "rot1", "rot2", "rot4"):
            if order:
                monkeypatch.setenv("RAYA_ATTN_ORDER", order)
            assert torch.equal(attend(hip_attention, x, lens, MASKS[name][0]), want), (b, h, order)


@pytest.mark.parametrize("b", [2, 3, 16, 17])
@pytest.mark.parametrize("d", [64, 128])
def test_longest_first_at_its_limit_and_packed(hip_attention, b, d):
    """Full batches of up to 16 sequences run longest first, ties and empty ones included; 17 do not.
    Also read out of rows of [heads dim + 8] floats."""
    h, s = 3, 300
    lens = [(37 * i + 150) % 301 if i % 5 else 200 for i in range(b)]
    lens[-1] = 0
    x = [torch.from_numpy(synth.normal(91 + i, b * h * s * d).reshape(b, h, s, d)).cuda() for i in range(3)]
    want = torch.cat([attend(hip_attention, [t[i:i + 1].contiguous() for t in x], lens[i:i + 1], R.Mask.FULL)
                      for i in range(b)])
    assert torch.equal(attend(hip_attention, x, lens, R.Mask.FULL), want)
    width = h * d + 8
    rows = [torch.zeros(b, s, width, device="cuda") for _ in x]
    for r, t in zip(rows, x):
        r[:, :, :h * d] = t.permute(0, 2, 1, 3).reshape(b, s, h * d)
    out = torch.full((b, s, width), 9.0, device="cuda")
    lay = (s * width, d, width)
    hip_attention.attend_batched(*rows, out, torch.tensor(lens, dtype=torch.int32, device="cuda"), R.Mask.FULL,
                                 layouts={"shape": (b, h, s, d), "q": lay, "k": lay, "v": lay, "out": lay})
    assert torch.equal(out[:, :, :h * d].reshape(b, s, h, d).permute(0, 2, 1, 3), want)
    assert (out[:, :, h * d:] == 9.0).all()


# Batch, heads, seq, head_dim, mask and the item height that a launch takes, on either side of each line.
CHOICES = [(2, 9, 1024, 64, R.Mask.BLOCK3, "128"), (1, 143, 100, 64, R.Mask.BLOCK3, "64"), (2, 72, 100, 64, R.Mask.FULL, "128"),
           (1, 12, 896, 64, R.Mask.FULL, "128"), (1, 12, 768, 64, R.Mask.FULL, "16"), (1, 16, 768, 64, R.Mask.BLOCK3, "128"),
           (1, 16, 760, 64, R.Mask.BLOCK3, "64"), (2, 6, 768, 64, R.Mask.FULL, "16"),
           (1, 12, 768, 128, R.Mask.BLOCK3, "16"), (1, 18, 1024, 128, R.Mask.BLOCK3, "128"),
           (23, 3, 442, 128, R.Mask.FULL, "64"), (23, 4, 442, 128, R.Mask.FULL, "128"),
           (64, 3, 130, 64, R.Mask.BLOCK3, "64"), (64, 3, 200, 64, R.Mask.BLOCK3, "128"),
           (4, 8, 1024, 64, R.Mask.sliding(128), "128"), (4, 8, 1024, 64, R.Mask.sliding(127), "64"),
           (5, 8, 1024, 64, R.Mask.sliding(128), "64"), (6, 8, 1024, 64, R.Mask.sliding(128), "128"),
           (4, 8, 1024, 128, R.Mask.sliding(256), "128"), (4, 8, 1024, 128, R.Mask.sliding(255), "64"),
           (6, 8, 1024, 128, R.Mask.sliding(256), "64"), (8, 8, 1024, 128, R.Mask.sliding(256), "128"),
           (16, 17, 300, 64, R.Mask.FULL, "128"), (17, 17, 300, 64, R.Mask.FULL, "128"),
           (8, 12, 1024, 64, R.Mask.block_diag(128), "64"), (8, 12, 1024, 64, R.Mask.WINDOW64, "64"),
           (8, 12, 1024, 96, R.Mask.FULL, "64")]


@pytest.mark.parametrize("b,h,s,d,mask,rows", CHOICES)
def test_default_dispatch(hip_attention, monkeypatch, b, h, s, d, mask, rows):
    """What a launch takes by itself: the bits of that height forced, which on other kernels differ,
    within the bar of the oracle on two sequences."""
    lens = [(97 * i) % (s // 2) + s // 2 + 1 if i else s for i in range(b)]
    x = [torch.from_numpy(synth.normal(51 + i, b * h * s * d).reshape(b, h, s, d)).cuda() for i in range(3)]
    monkeypatch.delenv("RAYA_ATTN_ITEMS")
    got = attend(hip_attention, x, lens, mask)
    for forced in ("16", "64", "128"):
        monkeypatch.setenv("RAYA_ATTN_ITEMS", forced)
        same = torch.equal(attend(hip_attention, x, lens, mask), got)
        no_kernel = forced == "128" and (d not in (64, 128) or mask.kind in (R.Mask.WINDOW64.kind, R.Mask.block_diag(1).kind))
        assert same == (forced == rows) or no_kernel, (forced, same)
    kind, block, window = {R.Mask.BLOCK3.kind: (oracle.MASK_BLOCK3, 128, 0), R.Mask.FULL.kind: (oracle.MASK_FULL, 0, 0),
                           R.Mask.sliding(1).kind: (oracle.MASK_SLIDING, 0, mask.arg),
                           R.Mask.WINDOW64.kind: (oracle.MASK_WINDOW64, 128, 0),
                           R.Mask.block_diag(1).kind: (oracle.MASK_BLOCKDIAG, mask.arg, 0)}[mask.kind]
    for i in (0, b - 1):
        q, k, v = (t[i].cpu().numpy() for t in x)
        want = oracle.naive_attend(q, k, v, kind, lens[i], R.kernels.default_scale(d), block=block, window=window)
        close(got[i, :, :lens[i]].cpu().numpy(), want[:, :lens[i]])
        assert (got[i, :, lens[i]:] == 0).all()


@pytest.mark.parametrize("name", ["block3", "full", "sliding200"])
@pytest.mark.parametrize("d", [64, 128])
def test_masks_are_exact(hip_attention, name, d):
    """V one-hot on key j: exactly the rows that see it get its weight, and the other dims stay zero."""
    seq, mask = 400, MASKS[name][0]
    q, k, _ = (torch.from_numpy(t[None]).cuda() for t in inputs(41, 1, seq, d))
    for j in (0, 63, 64, 127, 128, 255, 256, 399):
        v = torch.zeros_like(q)
        v[0, 0, j, j % d] = 1.0
        out = attend(hip_attention, [q, k, v], [seq], mask)[0, 0].cpu()
        want = torch.tensor([mask.allows(i, j) for i in range(seq)])
        assert torch.equal(out[:, j % d] > 0, want)
        out[:, j % d] = 0
        assert (out == 0).all()


def test_random_sweep_against_the_oracle(hip_attention):
    """36 random batched launches: batch 1-4, heads 1-3, seq 1-700, both head dims, every mask with a
    kernel and windows from 1 to past seq, valid lengths anywhere (clamped into [0, seq] by the entry
    point), negative and doubled scales."""
    rng = np.random.default_rng(2025)
    for case in range(36):
        b, h, s, d = int(rng.integers(1, 5)), int(rng.integers(1, 4)), int(rng.integers(1, 701)), (64, 128)[case % 2]
        arg = int(rng.integers(1, s + 80))
        mask, kind, block, window = [MASKS["block3"], MASKS["full"], (R.Mask.sliding(arg), oracle.MASK_SLIDING, 0, arg)][case % 3]
        valid = rng.integers(-3, s + 4, size=b).astype(np.int32)
        clamped = np.clip(valid, 0, s).astype(np.int32)
        scale = R.kernels.default_scale(d) * float(rng.choice([1.0, -1.0, 2.0]))
        q, k, v = (rng.standard_normal((b, h, s, d)).astype(np.float32) for _ in range(3))
        print(f"case {case}: b{b} h{h} s{s} d{d} {mask} valid {valid.tolist()} scale {scale:.4f}", flush=True)
        want = oracle.naive_attend_batched(q, k, v, kind, clamped, scale, block=block, window=window)
        out = torch.full((b, h, s, d), float("nan"), device="cuda")
        hip_attention.attend_batched(*(torch.from_numpy(x).cuda() for x in (q, k, v)), out, torch.from_numpy(valid).cuda(),
                                     mask, scale=scale)
        got = out.cpu().numpy()
        if (clamped > 0).any():
            close(np.concatenate([got[i, :, :n].reshape(-1) for i, n in enumerate(clamped)]),
                  np.concatenate([want[i, :, :n].reshape(-1) for i, n in enumerate(clamped)]))
        for i, n in enumerate(clamped):
            assert (got[i, :, n:] == 0).all()


def test_full_size_block3_by_default_against_float64(hip_attention, monkeypatch):
    """The 32 x 12 x 2048 Block3 batch (valid lengths 512 to 2048) as a launch takes it by itself, every
    output against float64 on the device."""
    monkeypatch.delenv("RAYA_ATTN_ITEMS")
    b, h, s, d = 32, 12, 2048, 64
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = [torch.randn(b, h, s, d, device="cuda", generator=gen) for _ in range(3)]
    lens = [int(n) for n in synth.integers(77, b, 512, 2048)]
    out = attend(hip_attention, x, lens, R.Mask.BLOCK3)
    blk = torch.arange(s, device="cuda") // 128
    near = (blk[:, None] - blk[None]).abs() <= 1
    worst = total = norm = 0.0
    for i, n in enumerate(lens):
        q, k, v = (t[i, :, :n].double() for t in x)
        w = torch.softmax((torch.matmul(q, k.transpose(1, 2).contiguous()) * 0.125).masked_fill(~near[:n, :n], -np.inf), -1)
        want = torch.matmul(w, v)
        diff = out[i, :, :n].double() - want
        worst, total, norm = max(worst, float(diff.abs().max())), total + float((diff ** 2).sum()), norm + float((want ** 2).sum())
        assert (out[i, :, n:] == 0).all()
    print(f"max-abs {worst:.2e}, rel-L2 {(total / norm) ** 0.5:.2e}")
    assert worst <= 1e-5 and (total / norm) ** 0.5 <= 1e-6
