"""The GEMM's three-part bfloat16 products where they can go wrong: the edges of every tile,
depths that a slab does not divide, unaligned rows, operands of very different sizes, and operands
whose parts do not sum to them (Inf, NaN, values above the largest bfloat16).

Bar: the reordering bound 2 k 2^-24 sum |a b| around the float64 product
(specs/009-gemm-backend-comparison/spec.md:24), which the sequential fp32 result meets.  The six
part products leave out at most 2^-24 of a product and are summed smallest first, with 6
roundings per 16 k, so they meet it from k = 2 on; at k = 1 the one product is rounded once.  Non-finite results are compared with
Reference::matmul_nt's.
"""
import numpy as np
import pytest
import torch

import oracle
from raya_amd import _capi as C
from tests.test_gemm_plan import plan

pytestmark = pytest.mark.gpu

GEGLU = C.RAYA_EPI_GEGLU


def check(out, a, b):
    k = a.shape[1]
    a64, b64 = a.double(), b.double()
    want = a64 @ b64.T
    bound = 2 * k * 2.0 ** -24 * (a64.abs() @ b64.abs().T)
    worst = float(((out.double() - want).abs() - bound).max())
    assert worst <= 0, worst


# Sizes one row and column short of a whole tile or past it, with whole and padded depths (the tile and
# depth of each are pinned further down).
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (33, 65, 128), (31, 63, 200), (257, 65, 15), (257, 2303, 768),
                                   (321, 2177, 744), (513, 2305, 768), (511, 2303, 780), (1023, 2305, 768),
                                   (1025, 2049, 100), (2047, 2305, 768), (2100, 2300, 720), (4097, 3073, 768),
                                   (8193, 2300, 64)])
def test_tile_edges(hip_gemm, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", generator=gen)
    b = torch.randn(n, k, device="cuda", generator=gen)
    out = torch.full((m, n + 3), 9.0, device="cuda")
    hip_gemm.matmul_nt_device(out[:, :n], a, b)
    check(out[:, :n], a, b)
    assert (out[:, n:] == 9.0).all()


NONE = C.RAYA_EPI_NONE
# By tile (rows x weight rows), whole depths, padded ones in 16-byte chunks, and others: sizes that take it,
# one row and one column short of a whole tile or past it.
TILE_EDGES = [
    (32, 64, NONE, [(31, 63, 256), (33, 65, 256), (1, 1, 256), (31, 65, 780), (33, 63, 780), (31, 63, 333), (33, 65, 333)]),
    (64, 64, NONE, [(63, 65, 128), (65, 63, 128), (63, 65, 100), (65, 63, 132), (63, 63, 67), (65, 65, 131)]),
    (64, 128, NONE, [(8193, 127, 128), (255, 4097, 128), (8193, 127, 100), (255, 4097, 100), (4097, 255, 67), (255, 4097, 67)]),
    (128, 128, NONE, [(8193, 257, 256), (511, 4097, 768), (8193, 255, 780), (511, 4097, 780), (4097, 513, 333), (8193, 257, 333)]),
    (256, 128, NONE, [(8193, 511, 256), (1023, 4097, 256), (8193, 513, 132), (1023, 4097, 780), (8193, 513, 131), (8193, 511, 333)]),
    (256, 256, NONE, [(16383, 1023, 64), (4095, 3073, 256), (16385, 513, 768)]),
    (32, 64, GEGLU, [(31, 33, 256), (33, 31, 256), (31, 33, 780), (33, 31, 333)]),
    (64, 64, GEGLU, [(63, 33, 128), (65, 31, 128), (63, 33, 100), (65, 33, 67)]),
    (64, 128, GEGLU, [(8193, 63, 128), (127, 4097, 128), (8193, 63, 100), (65, 4097, 131)]),
    (128, 128, GEGLU, [(8193, 129, 256), (2047, 1023, 256), (8193, 127, 780), (8193, 129, 333)]),
    (256, 128, GEGLU, [(8193, 255, 256), (511, 4097, 256), (8193, 257, 132), (8193, 257, 131)]),
    (256, 256, GEGLU, [(16383, 511, 64), (2047, 3073, 256)]),
]


@pytest.mark.parametrize("rows,cols,act,m,n,k", [(r, c, a, *x) for r, c, a, sizes in TILE_EDGES for x in sizes])
def test_every_tile_at_its_edges(hip_gemm, rows, cols, act, m, n, k):
    """Each tile with every kind of depth it takes, plain and with a bias and a residual: the bound, carried
    through GeGLU as in test_gemm_gpu.py (GELU's slope is at most 1.13)."""
    assert plan(m, n, k, act, vec=k % 4 == 0)[:2] == (rows, cols)
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    rows_b = 2 * n if act == GEGLU else n
    a = torch.randn(m, k, device="cuda", generator=gen)
    b = 0.1 * torch.randn(rows_b, k, device="cuda", generator=gen)
    bias, res = torch.randn(rows_b, device="cuda", generator=gen), torch.randn(m, n, device="cuda", generator=gen)
    y = a.double() @ b.double().T
    err = 2 * k * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T)
    for extra in (False, True):
        out = res.clone() if extra else torch.full((m, n), 9.0, device="cuda")
        hip_gemm.matmul_nt_device(out, a, b, bias=bias if extra else None, activation=act, residual=out if extra else None)
        want, tol = (y + bias.double(), err + 2.0 ** -24 * (y.abs() + bias.abs())) if extra else (y, err)
        if act == GEGLU:
            x, g = want[:, :n], want[:, n:]
            gx = torch.nn.functional.gelu(x)
            tol = 1.13 * tol[:, :n] * g.abs() + (gx.abs() + 1.13 * tol[:, :n]) * tol[:, n:] + 1e-6 * (gx * g).abs()
            want = gx * g
        if extra:
            want = want + res.double()
            tol = tol + 2.0 ** -23 * (want.abs() + res.abs())
        worst = float(((out.double() - want).abs() - tol).max())
        assert worst <= 0, (extra, worst)


@pytest.mark.parametrize("m,n,k", [(40, 70, 131), (600, 500, 67), (5000, 777, 333)])
def test_unaligned_rows(hip_gemm, m, n, k):
    """Operand rows that start one float past a 16-byte boundary, at every alignment of the depth."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    for extra in range(4):
        a = torch.randn(m, k + 1 + extra, device="cuda", generator=gen)[:, 1:k + 1]
        b = torch.randn(n, k + 1 + extra, device="cuda", generator=gen)[:, 1:k + 1]
        out = torch.empty(m, n, device="cuda")
        hip_gemm.matmul_nt_device(out, a, b)
        check(out, a, b)


@pytest.mark.parametrize("m,n,k", [(50, 70, 96), (2100, 2300, 128)])
def test_operands_over_the_whole_exponent_range(hip_gemm, m, n, k):
    """Elements from 2^-60 to 2^60 in one row: each part keeps the operand's own exponent, so the
    bound holds element by element, also where only a row's smallest elements meet b."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    scale = 2.0 ** torch.randint(-60, 61, (m, k), device="cuda", generator=gen)
    a = torch.randn(m, k, device="cuda", generator=gen) * scale
    b = torch.randn(n, k, device="cuda", generator=gen)
    b[::2] *= (scale[:1] < 1).float()  # every other row of b meets the small half of a's first row only
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, a, b)
    check(out, a, b)


@pytest.mark.parametrize("m,n,k", [(40, 70, 2), (40, 70, 3), (33, 65, 20), (300, 200, 96), (2100, 2300, 64)])
@pytest.mark.parametrize("exponent", [-149, -133, -126, -118, -110, -100])
def test_tiny_operands(hip_gemm, m, n, k, exponent):
    """Operands from 2^exponent down, subnormals among them, times operands of about 2^80 (no
    output is subnormal): all their bits count, on either side."""
    gen = torch.Generator(device="cuda").manual_seed(k - exponent)
    for swap in (False, True):
        tiny = torch.randn(n if swap else m, k, device="cuda", dtype=torch.float64, generator=gen)
        tiny = (tiny * 2.0 ** exponent).float()
        big = torch.randn(m if swap else n, k, device="cuda", generator=gen) * 2.0 ** 80
        a, b = (big, tiny) if swap else (tiny, big)
        out = torch.empty(m, n, device="cuda")
        hip_gemm.matmul_nt_device(out, a, b)
        check(out, a, b)


def test_tiny_weights_behind_a_folded_norm(hip_gemm):
    """Weights of about 2^-122 and rows normalised on the way in: within the bound around the
    64-bit product of the normalised rows, whose own rounding adds one unit per product."""
    m, n, k = 70, 132, 16
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = 2.0 + torch.randn(m, k, device="cuda", generator=gen)
    b = (torch.randn(n, k, device="cuda", generator=gen).double() * 2.0 ** -122).float()
    mean, rstd = x.double().mean(1), 1.0 / x.double().std(1, unbiased=False)
    rows = torch.zeros(m, 4, device="cuda")
    rows[:, 0] = mean.float()
    rows[:, 1] = (mean - mean.float().double()).float()
    rows[:, 2] = rstd.float()
    sums = torch.empty(n, device="cuda")
    hip_gemm.weight_row_sums(b, sums)
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, x, b, in_row_stats=rows, in_weight_sums=sums)
    norm = (x.double() - mean[:, None]) * rstd[:, None]
    want = norm @ b.double().T
    bound = (2 * k + 8) * 2.0 ** -24 * (norm.abs() @ b.double().abs().T)
    worst = float(((out.double() - want).abs() / bound).max())
    assert worst <= 1, worst


@pytest.mark.parametrize("m,n,k", [(268435456 + 77, 1, 2), (128 * (0x7FFFFFFF // 256), 1, 1), (3, 300000001, 1)])
def test_very_tall_and_wide_outputs(hip_gemm, m, n, k):
    """Grids past 2^22 workgroups; rows and columns checked at both ends and in between."""
    a = torch.arange(m * k, device="cuda", dtype=torch.int32).remainder_(4093).float().reshape(m, k)
    b = torch.arange(n * k, device="cuda", dtype=torch.int32).remainder_(61).float().reshape(n, k)
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, a, b)
    for r0 in range(0, m, max(1, m // 7)):
        for c0 in range(0, n, max(1, n // 7)):
            x, y = a[r0:r0 + 2000], b[c0:c0 + 2000]
            assert torch.equal(out[r0:r0 + 2000, c0:c0 + 2000], x @ y.T)
    assert torch.equal(out[-300:, -300:], a[-300:] @ b[-300:].T)


@pytest.mark.parametrize("m,n", [(1, 1), (40, 70), (300, 200), (2100, 2300)])
@pytest.mark.parametrize("exponent", [0, -100, 100])
def test_depth_one_is_the_rounded_product(hip_gemm, m, n, exponent):
    """One product has one rounding."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    a = torch.randn(m, 1, device="cuda", generator=gen) * 2.0 ** exponent
    b = torch.randn(n, 1, device="cuda", generator=gen)
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, a, b)
    assert torch.equal(out, a * b.reshape(1, n))


@pytest.mark.parametrize("m,n,k", [(40, 70, 3), (300, 200, 96), (2100, 2300, 64)])
@pytest.mark.parametrize("ea,eb", [(100, -100), (104, -60), (106, -106), (120, -120), (41, 40), (70, 45)])
def test_large_operands_and_sums(hip_gemm, m, n, k, ea, eb):
    """Finite operands from about 2^105, whose scaled parts overflow, and finite sums from about
    2^82, on either side of both lines."""
    gen = torch.Generator(device="cuda").manual_seed(ea)
    a = torch.randn(m, k, device="cuda", generator=gen) * 2.0 ** ea
    b = torch.randn(n, k, device="cuda", generator=gen) * 2.0 ** eb
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, a, b)
    assert torch.isfinite(out).all()
    check(out, a, b)


@pytest.mark.parametrize("m,n,k", [(40, 70, 96), (300, 200, 100), (2100, 2300, 64)])
def test_non_finite_operands(hip_gemm, m, n, k):
    """Inf, NaN and 3.4e38 in single elements of a and b: NaN and Inf where the reference has
    them, its values (the bound) elsewhere, and the outputs that meet none of them unchanged.
    The two huge values share a column, so that an output's exact sum overflows whenever one of
    its products does: where two huge products cancel, a sum overflows or not by its order."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k)).astype(np.float32)
    b[3, 5] = 0.0  # 0 * Inf
    plain = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(plain, torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda())
    x, y = a.copy(), b.copy()
    for row, col, v in ((0, 5, np.inf), (7, k - 1, -np.inf), (m - 1, 0, np.nan), (33, 2, 3.4e38)):
        x[row, col] = v
    for row, col, v in ((1, 4, np.inf), (n - 1, k - 2, np.nan), (35, 2, -3.4e38)):
        y[row, col] = v
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    got = out.cpu().numpy()
    rows, cols = [0, 7, 33, m - 1], [1, 35, n - 1]
    with np.errstate(all="ignore"):
        for i, j in [(r, slice(None)) for r in rows] + [(slice(None), c) for c in cols]:
            xa, yb = (x[i:i + 1], y) if isinstance(i, int) else (x, y[j:j + 1])
            want = oracle.matmul_nt(np.ascontiguousarray(xa), np.ascontiguousarray(yb)).reshape(-1)
            have = got[i, j].reshape(-1)
            assert np.array_equal(np.isnan(have), np.isnan(want))
            assert np.array_equal(have[np.isinf(want)], want[np.isinf(want)])
            ok = np.isfinite(want)
            bound = 2 * k * 2.0 ** -24 * (np.abs(xa).astype(np.float64) @ np.abs(yb).astype(np.float64).T).reshape(-1)
            assert (np.abs(have[ok].astype(np.float64) - want[ok]) <= bound[ok]).all()
    keep = np.ones((m, n), bool)
    keep[rows] = False
    keep[:, cols] = False
    assert np.array_equal(got[keep], plain.cpu().numpy()[keep])


@pytest.mark.parametrize("k", [1, 2, 5, 31, 32, 33, 64, 100, 131])
@pytest.mark.parametrize("offset", [0, 1])
def test_exact_outputs_at_every_depth(hip_gemm, k, offset):
    """Rows whose parts overflow (values from 2^120) are computed from the unsplit operands: every
    remainder of the 32 k that a step takes, of aligned rows and of rows one float past a boundary."""
    m, n = 70, 66
    gen = torch.Generator(device="cuda").manual_seed(k)
    a = torch.zeros(m, k + 4 - k % 4 + 4, device="cuda")[:, offset:k + offset]
    b = torch.zeros(n, k + 4 - k % 4 + 4, device="cuda")[:, offset:k + offset]
    a.copy_(torch.randn(m, k, device="cuda", generator=gen))
    b.copy_(torch.randn(n, k, device="cuda", generator=gen) * 2.0 ** -60)
    a[::3] *= 2.0 ** 120
    out = torch.empty(m, n, device="cuda")
    hip_gemm.matmul_nt_device(out, a, b)
    assert torch.isfinite(out).all()
    check(out, a, b)
