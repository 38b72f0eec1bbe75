"""GPU transforms of rows whose elements sit at the field's edges (0, 1, p - 1,
2^32 - 1, 2^32, ...), bit-exact against the oracle: constant rows, rows that
alternate 0 and p - 1 with every power-of-two period, and random mixes, so that
carries, borrows and sums equal to p occur in every butterfly stage."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 0xFFFF_FFFF_0000_0001
EDGE = np.array([0, 1, 2, 0xFFFFFFFF, 0x100000000, 0x100000001, P - 1, P - 2, P - 0xFFFFFFFF, 1 << 63,
                 0xFFFFFFFE00000002, 0x8000000080000000], dtype=np.uint64)


def edge_rows(n):
    j = np.arange(n, dtype=np.uint64)
    rows = [np.full(n, e, np.uint64) for e in (1, P - 1, 0xFFFFFFFF, 0x100000000)]
    rows += [np.where((j >> np.uint64(b)) & np.uint64(1), np.uint64(P - 1), np.uint64(0))
             for b in range(0, n.bit_length() - 1, 3)]
    g = np.random.Generator(np.random.PCG64(n))
    rows += [EDGE[g.integers(0, len(EDGE), n)] for _ in range(4)]
    return np.stack(rows)


@pytest.mark.parametrize("bits", [6, 12, 13, 14, 15, 16, 17])
def test_edge_rows_forward_and_inverse(backend, oracle, bits):
    n = 1 << bits
    host = edge_rows(n)
    inp = backend.upload_device(host.reshape(-1))
    out = backend.ntt_fp_batch_device(inp, len(host), n)
    back = backend.ntt_fp_inverse_batch_device(out, len(host), n)
    got, round_trip = backend.download_device(out), backend.download_device(back)
    for b in (inp, out, back):
        backend.free_device(b)
    assert (got.reshape(host.shape) == oracle.ntt_forward_batch(host)).all()
    assert (round_trip.reshape(host.shape) == host).all()


@pytest.mark.parametrize("bits,rate", [(13, 4), (14, 4), (15, 8), (17, 4)])
def test_edge_rows_with_zero_tails(backend, oracle, bits, rate):
    n, m = 1 << bits, (1 << bits) // rate
    host = edge_rows(m)
    msgs = backend.upload_device(host.reshape(-1))
    out = backend.ntt_fp_encode_device(msgs, len(host), m, n)
    got = backend.download_device(out).reshape(len(host), n)
    for b in (msgs, out):
        backend.free_device(b)
    assert (got == oracle.ntt_encode_batch(host, n)).all()
