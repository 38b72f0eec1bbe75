"""The field operations of volta-zk_amd/csrc/gl64.hpp and gl64_shift.hpp that
take or give words above p - 1 (built for the host from the same headers,
libgl64_check.so), against Python big integers.  CPU only."""
import ctypes
import pathlib
import random

import pytest

from test_shift_arithmetic import EDGE, P

LIB = pathlib.Path(__file__).resolve().parent.parent / "volta-zk_amd" / "libgl64_check.so"


@pytest.fixture(scope="module")
def glc():
    if not LIB.exists():
        pytest.fail("libgl64_check.so missing: run volta-zk_amd/build.py (or __graft_entry__.build())")
    L = ctypes.CDLL(str(LIB))
    u64, ptr = ctypes.c_uint64, ctypes.POINTER(ctypes.c_uint64)
    for name, res, args in [("glc_mul_pow2", u64, [u64, ctypes.c_int]), ("glc_mul32x4", u64, [u64, u64]),
                            ("glc_sub", u64, [u64, u64]), ("glc_add_lazy", u64, [u64, u64]),
                            ("glc_fold96_lazy", u64, [u64, ctypes.c_uint32]),
                            ("glc_bfly_lazy", None, [ptr, ptr, ctypes.c_int]),
                            ("glc_dft_lazy", None, [ptr, ctypes.c_int])]:
        f = getattr(L, name)
        f.restype, f.argtypes = res, args
    return L


# Words from p on (and the largest u64): values that only the lazy forms meet.
LAZY = [P, P + 1, (1 << 64) - 1, (1 << 64) - 2, (1 << 64) - (1 << 31), P + 12345]


def test_lazy_forms_of_any_word(glc):
    """add_lazy, sub and the butterflies on any u64 u, the shifts on any u64: right
    mod p, and the difference canonical whenever its first operand is."""
    rnd = random.Random(11)
    words = LAZY + EDGE + [rnd.randrange(1 << 64) for _ in range(30)]
    for e in range(192):
        w = pow(2, e, P)
        for x in LAZY + EDGE + words[-8:]:
            if e % 96:
                assert glc.glc_mul_pow2(x, e) == x * w % P, (e, x)
            y = rnd.choice(EDGE if e % 96 == 0 else words)
            u, v = ctypes.c_uint64(x), ctypes.c_uint64(y)
            glc.glc_bfly_lazy(ctypes.byref(u), ctypes.byref(v), e)
            assert (u.value % P, v.value % P) == ((x + w * y) % P, (x - w * y) % P), (e, x, y)
    for a in words:
        for b in EDGE:
            assert glc.glc_add_lazy(a, b) % P == (a + b) % P
            assert glc.glc_sub(a, b) % P == (a - b) % P
        for hi in (0, 1, 0xFFFF, 0x80000000, 0xFFFFFFFF):
            assert glc.glc_fold96_lazy(a, hi) % P == (a + (hi << 64)) % P
        assert glc.glc_mul32x4(a, words[-1]) == a * words[-1] % P


@pytest.mark.parametrize("log", [4, 5])
def test_dft_with_lazy_outputs(glc, log):
    """Every output right mod p and output 0 canonical, on edge values in every
    position and on constant rows (whose sums wrap at every stage)."""
    n, rnd = 1 << log, random.Random(13 + log)
    w = pow(2, 78 << (5 - log), P)
    rows = [[e] * n for e in EDGE] + [[rnd.choice(EDGE) for _ in range(n)] for _ in range(40)]
    rows += [[P - 1 if (i >> b) & 1 else 0 for i in range(n)] for b in range(log)]
    for x in rows:
        v = (ctypes.c_uint64 * n)(*[x[int(f"{i:0{log}b}"[::-1], 2)] for i in range(n)])
        glc.glc_dft_lazy(v, log)
        want = [sum(x[j] * pow(w, j * k, P) for j in range(n)) % P for k in range(n)]
        assert [t % P for t in v] == want
        assert v[0] == want[0]
