"""The opening's small kernels at the edges of their dispatch, bit-exact against
the oracle: mask rows spread over the GPU and their rejected draws, equality
rows with each number of outputs per thread, dots of whole, of cut and of many
short rows; mask rows and dots also inside a coarse timing scope, where
workspaces may not grow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 0xFFFF_FFFF_0000_0001
# the 6th raw draw of row 0 in domain 0x19664BCA is rejected for this seed
# (rust/volta-accel/src/lib.rs:7517-7528)
from test_gpu_pcs import KAT_SEED  # noqa: E402


def fp2(seed, n):
    return np.random.default_rng(seed).integers(0, P, size=(n, 2), dtype=np.uint64)


@pytest.mark.parametrize("rows,count", [(1, 8192), (2, 8193), (7, 66561), (1024, 8199), (1025, 8192), (3, 511), (5, 1024),
                                        (2, 1537), (7, 4097)])
def test_long_rows_with_and_without_a_rejection(backend, oracle, rows, count):
    for domain in (0x19664BCA, 0x19664BCB, 0x19664BCA):  # a rejected row, none, and again
        d = backend.chacha8_prover_secret_fp_rows_device(KAT_SEED, domain, rows, count)
        got = backend.download_device(d).reshape(rows, count)
        backend.free_device(d)
        assert (got == oracle.fp_rows(KAT_SEED, domain, rows, count)).all()


@pytest.mark.parametrize("rows,dims", [(1, 0), (1, 1), (1, 16), (6, 15), (1, 17), (3, 17), (64, 13), (97, 13), (129, 13)])
def test_equality_rows(backend, oracle, rows, dims):
    pts = fp2(rows + dims, rows * dims)
    buf = backend.upload_device(pts, pts_dtype()) if dims else None
    out = backend.logup_eq_rows_device(buf, rows, dims)
    got = backend.download_device(out).view(np.uint64).reshape(-1, 2)
    for b in (buf, out):
        if b is not None:
            backend.free_device(b)
    want = oracle.eq_rows(pts, rows, dims)
    assert (got == np.asarray(want).reshape(-1, 2)).all()


def pts_dtype():
    from volta_mi355x import FP2
    return FP2


@pytest.mark.parametrize("rows,length", [(1, 1), (1, 4096), (1, 4097), (1, 100000), (6, 32768), (97, 8200), (255, 8193),
                                         (256, 8193), (300, 5000), (1, 8191), (1, 8192), (128, 8192), (256, 512),
                                         (257, 1), (257, 512), (257, 513), (3000, 300)])
def test_row_dots(backend, oracle, rows, length):
    stride = length + 3
    a, b = fp2(length, rows * stride), fp2(length + 1, rows * length)
    a[:4] = P - 1
    da, db = backend.upload_device(a, pts_dtype()), backend.upload_device(b, pts_dtype())
    out = backend.fp2_row_dots_device(da, 0, stride, db, 0, length, rows, length)
    got = backend.download_device(out).view(np.uint64).reshape(rows, 2)
    for x in (da, db, out):
        backend.free_device(x)
    assert (got == np.asarray(oracle.fp2_row_dots(a, stride, b, length, rows, length)).reshape(rows, 2)).all()


def test_without_workspaces_in_a_coarse_scope(oracle):
    from volta_mi355x import Backend
    with Backend(timing_policy=1) as b:
        rows, count, length = 2, 8200, 20000
        out = b.alloc_device(rows * count, np.uint64)
        x, y = fp2(1, length), fp2(2, length)
        dx, dy = b.upload_device(x, pts_dtype()), b.upload_device(y, pts_dtype())
        dot = b.alloc_device(1, pts_dtype())
        seed = (np.frombuffer(bytes(KAT_SEED), np.uint8)).copy()
        import ctypes
        cs = (ctypes.c_uint8 * 32).from_buffer(seed)
        live = b.get_stats()["live_device_bytes"]
        assert b.lib.volta_cuda_begin_coarse_timing(b.raw, 2) == 0
        assert b.lib.volta_cuda_chacha8_prover_secret_fp_rows_device(b.raw, out.id, 0, cs, 0x19664BCA, rows, count) == 0
        assert b.lib.volta_cuda_end_coarse_timing(b.raw) == 0
        got = b.download_device(out).reshape(rows, count)
        assert b.lib.volta_cuda_begin_coarse_timing(b.raw, 2) == 0
        assert b.lib.volta_cuda_fp2_row_dots_device(b.raw, dx.id, 0, length, dy.id, 0, length, dot.id, 0, 1, length) == 0
        assert b.lib.volta_cuda_end_coarse_timing(b.raw) == 0
        assert b.get_stats()["live_device_bytes"] == live
        assert (got == oracle.fp_rows(KAT_SEED, 0x19664BCA, rows, count)).all()
        want = np.asarray(oracle.fp2_row_dots(x, length, y, length, 1, length)).reshape(1, 2)
        assert (b.download_device(dot).view(np.uint64).reshape(1, 2) == want).all()
