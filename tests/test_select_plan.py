"""The score pass's plan (asa::select_plan: waves per block, LDS rings, candidate
keys per row) over k, head dimension, dtype and key count, on the host."""
import ctypes
import itertools

import pytest

F32, BF16 = 0, 1


class Dims(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("BH", "H", "NQ", "NK", "D", "hd", "k", "nQB", "nKB")] + \
               [("alpha", ctypes.c_float), ("scale", ctypes.c_float)]


class Plan(ctypes.Structure):
    _fields_ = [("waves", ctypes.c_int), ("ring", ctypes.c_bool), ("cap", ctypes.c_int),
                ("needs", ctypes.c_size_t)]


@pytest.fixture(scope="module")
def plan():
    from splash_attention import _lib

    f = getattr(_lib.load(), "_ZN3asa11select_planERKNS_4DimsEibmi")
    f.restype = Plan
    f.argtypes = [ctypes.POINTER(Dims), ctypes.c_int, ctypes.c_bool, ctypes.c_size_t, ctypes.c_int]

    def call(k, hd, dtype, nk, blocks=1024, lds=160 * 1024, scores=False, scale=0.125):
        d = Dims(blocks, 1, 64, nk, 64 if hd <= 64 else 128, hd, k, 1, -(-nk // 64), 1.5, scale)
        return f(ctypes.byref(d), dtype, scores, lds, 256)

    return call


@pytest.mark.parametrize("nk", [64, 4096, 131072, 400000, 500000, 700000, 850000, 950336, 1425472, 1671232,
                                1687616])
@pytest.mark.parametrize("dtype,hd,blocks", itertools.product([F32, BF16], [64, 80, 128], [64, 1024]))
def test_lists_keep_room_for_the_candidates(plan, nk, dtype, hd, blocks):
    """A row lists at least k + 4 keys (an overflow round drops cap - k), and
    the eight-wave and ring variants, which take LDS from the lists, do not
    hold fewer than random rows need (about 1.15 k) where the variant with
    neither (the one of a negative scale) holds more."""
    for k in range(1, 129):
        p, plain = plan(k, hd, dtype, nk, blocks), plan(k, hd, dtype, nk, blocks, scale=-0.125)
        assert (plain.waves, plain.ring) == (4, False)
        if p.cap < 0:
            assert p.needs > 160 * 1024 and plain.cap < 0
            continue
        assert k + 4 <= p.cap <= 256, (k, p.cap)
        assert p.cap >= min(k + k // 8 + 16, plain.cap), (k, p.waves, p.ring, p.cap, plain.cap)


def test_smaller_lds_refuses_only_below_the_least_list(plan):
    """As LDS shrinks, a plan is refused only where k + 4 keys per row do not
    fit, and the bytes it then names are enough."""
    for k, hd, dtype in itertools.product((1, 8, 50, 64, 128), (64, 128), (F32, BF16)):
        for scores in (False, True):
            refused = 0
            for lds in range(160 * 1024, 0, -1024):
                p = plan(k, hd, dtype, 8192, lds=lds, scores=scores)
                if p.cap < 0:
                    assert p.needs > lds
                    refused = refused or lds
                else:
                    assert not refused
                    assert p.needs == 0
            assert refused and plan(k, hd, dtype, 8192, lds=p.needs, scores=scores).cap >= k + 4
