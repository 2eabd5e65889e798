"""The GEMM's choice of tile and split, on the CPU: what sizes it takes and what it launches for them."""
import ctypes

import pytest

from raya_amd import _capi as C

MAX_BLOCKS = 0x7FFFFFFF // 256


def plan(m, n, k, act=C.RAYA_EPI_NONE, vec=True, whole=False, room=0):
    """(tile rows, tile weight rows, threads, splits, workgroups), or None where the size is refused."""
    f = C.lib().raya_gemm_plan
    f.argtypes = [ctypes.c_int] * 6 + [ctypes.c_uint64, ctypes.POINTER(ctypes.c_int64)]
    out = (ctypes.c_int64 * 5)()
    return tuple(out) if f(m, n, k, act, vec, whole, room, out) == 0 else None


def blocks(m, n, act):
    out_bn = 64 if act == C.RAYA_EPI_GEGLU else 128
    return -(-m // 128) * -(-n // out_bn)


@pytest.mark.parametrize("act", [C.RAYA_EPI_NONE, C.RAYA_EPI_GEGLU])
@pytest.mark.parametrize("vec", [False, True])
def test_sizes_taken_and_refused(act, vec):
    """Outputs of up to 2^31 / 256 blocks of 128 x 128 are taken, whatever their shape, on a grid of
    fewer than 2^32 threads that covers them; larger ones are refused, past 2^31 rows included."""
    top = 128 * MAX_BLOCKS
    cols = top // (2 if act == C.RAYA_EPI_GEGLU else 1)
    sizes = [(268435392, 64), (268435393, 64), (268435457, 1), (top, 1), (top - 127, 1), (top + 1, 1), (2 ** 30 + 128, 1),
             (2 ** 31 - 1, 1), (1, cols), (1, cols + 1), (128, cols), (129, cols), (100, cols - 1), (2 ** 19, 2 ** 19),
             (370000, 370000), (3000, 2 ** 25), (1, 1)]
    for m, n in sizes:
        for k in (1, 4, 64, 768):
            p = plan(m, n, k, act, vec)
            assert (p is not None) == (blocks(m, n, act) <= MAX_BLOCKS), (m, n, k)
            if p is not None:
                bm, bn, threads, splits, groups = p
                out_bn = bn // 2 if act == C.RAYA_EPI_GEGLU else bn
                assert groups == -(-m // bm) * -(-n // out_bn) * splits and groups * threads < 2 ** 32
