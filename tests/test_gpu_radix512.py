"""Passes of radix 2^9 (two LDS rounds per tile, ntt_reg.hip) for two-plane (Fp2)
transforms and without a column table: batches on both sides of where two planes
take the radix (2^21 elements), both plans (2^17: gather of 2^9 and columns of 2^8;
2^18: both 2^9), the column pass that builds its own twiddles, and every input
count of the two-plane gather (2^25 points, ragged lengths)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 0xFFFF_FFFF_0000_0001


def rand_rows(seed, rows, n, planes):
    x = np.random.default_rng(seed).integers(0, P, size=(rows, n, planes), dtype=np.uint64)
    x[0, :3] = [[P - 1] * planes, [0] * planes, [0xFFFFFFFF] * planes]
    x[-1, -1] = P - 1
    return x


def check(oracle, got, host):
    for comp in range(host.shape[2]):
        want = oracle.ntt_forward_batch(np.ascontiguousarray(host[:, :, comp]))
        assert (got[:, :, comp] == want).all(), comp


@pytest.mark.parametrize("bits,rows", [(17, 15), (17, 16), (17, 17), (18, 7), (18, 8), (18, 9)])
def test_fp2_batches(backend, oracle, bits, rows):
    from volta_mi355x import FP2
    n = 1 << bits
    host = rand_rows(bits + rows, rows, n, 2)
    inp = backend.upload_device(host.reshape(-1, 2), FP2)
    out = backend.ntt_fp2_batch_device(inp, rows, n)
    got = backend.download_device(out).view(np.uint64).reshape(rows, n, 2)
    for b in (inp, out):
        backend.free_device(b)
    check(oracle, got, host)


@pytest.mark.parametrize("planes,rows", [(2, 8), (1, 1), (1, 3)])
def test_without_the_column_table(oracle, planes, rows):
    """2^18 points inside a coarse timing scope, where tables may not grow, on a
    context that has only the twiddles: one Fp2 row before the scope takes radix
    2^6 and builds the tables of that."""
    from volta_mi355x import FP2, Backend
    n = 1 << 18
    host = rand_rows(planes, rows, n, planes)
    with Backend(timing_policy=1) as b:
        one = b.upload_device(rand_rows(9, 1, n, 2).reshape(-1, 2), FP2)
        b.free_device(b.ntt_fp2_batch_device(one, 1, n))
        inp = b.upload_device(host.reshape(-1, 2), FP2) if planes == 2 else b.upload_device(host.reshape(-1))
        out = b.alloc_device(rows * n * planes, np.uint64)
        live = b.get_stats()["live_device_bytes"]
        f = b.lib.volta_cuda_ntt_fp2_batch_device if planes == 2 else b.lib.volta_cuda_ntt_fp_batch_device
        assert b.lib.volta_cuda_begin_coarse_timing(b.raw, 3) == 0
        assert f(b.raw, inp.id, 0, rows, n, out.id, 0) == 0, b.last_error()
        assert b.lib.volta_cuda_end_coarse_timing(b.raw) == 0
        assert b.get_stats()["live_device_bytes"] == live
        got = b.download_device(out).reshape(rows, n, planes)
    check(oracle, got, host)


@pytest.fixture(scope="module")
def powers(backend):
    """2^25 resident powers c, c^2, .. of one Fp2 element, and c."""
    c = (0x123456789ABCDEF1, P - 98765)
    buf = backend.fp2_powers_device(c, 1 << 25)
    yield buf, c
    backend.free_device(buf)


# step 1 of the gather reads ceil(32 len / n) of its 32 inputs, rounded up to a
# compiled count (1, 2, 4, 9, 16, 32): lengths at and one past each
@pytest.mark.parametrize("k,more", [(1, 0), (1, 1), (2, 0), (2, 1), (4, 0), (4, 1), (9, 0), (9, 1), (16, 0), (16, 1),
                                    (32, -1), (32, 0)])
def test_x4_2_25_ragged_lengths(backend, oracle, powers, k, more):
    """The transform of c^1 .. c^len (more powers behind it, which it must not
    read) is c ((c w^j)^len - 1) / (c w^j - 1) at w^j: sampled outputs."""
    buf, c = powers
    n = 1 << 25
    length = k * (n // 32) + more
    out = backend.x4_ntt_fp2_device(buf, length, n)
    w = oracle.x4_root_of_unity(25)
    rng = np.random.default_rng(k)
    picks = {0, 1, n // 2, n - 1} | {int(j) for j in rng.integers(0, n, size=60)}
    try:
        for j in sorted(picks):
            cw = oracle.fp2_mul(c, oracle.fp2_pow(w, j))
            top, bottom = oracle.fp2_pow(cw, length), (oracle.fp_sub(cw[0], 1), cw[1])
            top = (oracle.fp_sub(top[0], 1), top[1])
            want = oracle.fp2_mul(c, oracle.fp2_mul(top, oracle.fp2_inv(bottom)))
            got = tuple(int(v) for v in backend.download_device(out, j, 1).view(np.uint64))
            assert got == tuple(int(v) for v in want), j
    finally:
        backend.free_device(out)
