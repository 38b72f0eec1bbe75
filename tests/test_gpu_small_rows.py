"""Rows of 2^8 .. 2^12 points through the one-pass small-row transform
(ntt_small.hip), bit-exact against the oracle: each size, row counts on both sides
of where it takes over and that leave the last workgroup part-filled, lengths on
both sides of every input count, message rows, both directions, offsets and edge
values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 0xFFFF_FFFF_0000_0001


def field(seed, shape):
    x = np.random.default_rng(seed).integers(0, P, size=shape, dtype=np.uint64)
    x.reshape(-1)[: min(4, x.size)] = [P - 1, 0, 1, 0xFFFFFFFF][: min(4, x.size)]
    return x


@pytest.mark.parametrize("bits", [8, 9, 10, 11, 12])
@pytest.mark.parametrize("total", [0, 1 << 20, 5 << 18])
@pytest.mark.parametrize("more", [-1, 0, 1, 7])
def test_both_directions(backend, oracle, bits, total, more):
    n = 1 << bits
    rows = max(1, total // n + more)
    x = field(bits + rows, (rows, n))
    inp = backend.upload_device(x.reshape(-1))
    out = backend.ntt_fp_batch_device(inp, rows, n)
    back = backend.ntt_fp_inverse_batch_device(out, rows, n)
    got, trip = backend.download_device(out).reshape(rows, n), backend.download_device(back).reshape(rows, n)
    for b in (inp, out, back):
        backend.free_device(b)
    assert (got == oracle.ntt_forward_batch(x)).all()
    assert (trip == x).all()


@pytest.mark.parametrize("bits", [8, 9, 10, 11, 12])
def test_lengths(backend, oracle, bits):
    n, m = 1 << bits, (1 << bits) // 16
    rows = (1 << 20) // n + 3
    for length in (1, 4 * m, 4 * m + 1, 6 * m, 6 * m + 1, 8 * m, 8 * m + 1, n - 1, n):
        x = field(length, (rows, length))
        msgs = backend.upload_device(x.reshape(-1))
        out = backend.ntt_fp_encode_device(msgs, rows, length, n)
        got = backend.download_device(out).reshape(rows, n)
        for b in (msgs, out):
            backend.free_device(b)
        assert (got == oracle.ntt_encode_batch(x, n)).all()


@pytest.mark.parametrize("bits", [8, 9, 10, 11, 12])
@pytest.mark.parametrize("total", [0, 1 << 20])
def test_message_rows(backend, oracle, bits, total):
    n = 1 << bits
    rows = total // n + 1
    for cols, pad in ((n // 4, 0), (n // 4, 16), (n // 8, n // 8), (n // 2 - 3, 7), (1, 1), (n - 9, 9), (n, 0)):
        rng = np.random.default_rng(cols)
        w = rng.integers(-32768, 32768, size=(rows, cols), dtype=np.int16)
        pads = field(pad, (rows, max(pad, 1)))
        dw, dp = backend.upload_device(w.reshape(-1)), backend.upload_device(pads.reshape(-1))
        out = backend.pcs_encode_device(dw, 0, dp, 0, rows, cols, pad, n)
        got = backend.download_device(out).reshape(rows, n)
        for b in (dw, dp, out):
            backend.free_device(b)
        want = oracle.pcs_encode_i16(w.reshape(-1), pads.reshape(-1) if pad else None, rows, cols, pad, n)
        assert (got == want.reshape(rows, n)).all()


def test_offsets_leave_the_rest_alone(backend, oracle):
    n, rows = 512, 2059
    x = field(5, (rows, n))
    inp = backend.upload_device(np.concatenate([np.full(3, 7, np.uint64), x.reshape(-1)]))
    out = backend.upload_device(np.full(rows * n + 10, 9, np.uint64))
    backend._check(backend.lib.volta_cuda_ntt_fp_batch_device(backend.raw, inp.id, 3, rows, n, out.id, 5))
    got = backend.download_device(out)
    for b in (inp, out):
        backend.free_device(b)
    assert (got[5:-5].reshape(rows, n) == oracle.ntt_forward_batch(x)).all()
    assert (got[:5] == 9).all() and (got[-5:] == 9).all()
