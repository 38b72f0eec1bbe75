"""Message rows lift(w) || pads || 0 of 2^13 and 2^14 points through the one-pass
transform (ntt_rr.hip): each choice of blocks on both sides of its bounds, odd
column and pad counts, on the host emulation of the kernel's phases and on the
GPU, bit-exact against the oracle."""
import ctypes
import pathlib

import numpy as np
import pytest

import oracle

P = 0xFFFF_FFFF_0000_0001
LIB = pathlib.Path(__file__).resolve().parent.parent / "volta-zk_amd" / "libgl64_check.so"
# (bits, cols, pad) in blocks of M = 2^bits / 32: 8 M and 4 M with pads of at most
# 2 M, everything else up to 16 M and up to n
SHAPES = [(13, 2048, 512), (13, 2048, 1), (13, 2048, 513), (13, 1024, 512), (13, 1024, 513), (13, 1, 1),
          (13, 1000, 77), (13, 2047, 2049), (13, 4095, 0), (13, 4096, 1), (13, 5001, 3191), (13, 8192, 0),
          (14, 4096, 0), (14, 4096, 512), (14, 4096, 1024), (14, 4096, 1025), (14, 2048, 512), (14, 3001, 129),
          (14, 8191, 2), (14, 16383, 1)]


def inputs(rows, cols, pad):
    rng = np.random.default_rng(7 * cols + pad)
    w = rng.integers(-32768, 32768, size=(rows, cols), dtype=np.int16)
    w[0, : min(4, cols)] = [-32768, 32767, -1, 0][: min(4, cols)]
    pads = rng.integers(0, P, size=(rows, max(pad, 1)), dtype=np.uint64)
    pads[0, 0] = P - 1
    return w, pads


@pytest.mark.parametrize("bits,cols,pad", SHAPES)
def test_emulated_rows(bits, cols, pad):
    glc = ctypes.CDLL(str(LIB))
    vp, sz = ctypes.c_void_p, ctypes.c_size_t
    glc.glc_ntt_rr_msg.argtypes = [vp, vp, vp, sz, sz, sz, sz, sz, vp]
    n, rows = 1 << bits, 3
    w, pads = inputs(rows, cols, pad)
    fwd = np.ascontiguousarray(oracle.ntt_twiddles(n))
    got = np.zeros((rows, n), dtype=np.uint64)
    assert glc.glc_ntt_rr_msg(fwd.ctypes.data, w.ctypes.data, pads.ctypes.data, cols, pad, bits, rows, 2,
                              got.ctypes.data) == 0
    want = oracle.pcs_encode_i16(w.reshape(-1), pads.reshape(-1) if pad else None, rows, cols, pad, n)
    assert (got == want.reshape(rows, n)).all()


# row counts on both sides of where the one pass takes over from the pass engine's two
# (5/8 of 256 CUs at 2^13, half of them at 2^14), and more rows than workgroups
@pytest.mark.gpu
@pytest.mark.parametrize("bits,cols,pad", SHAPES)
@pytest.mark.parametrize("rows", [1, -1, 0, 1030])
def test_device_rows(backend, bits, cols, pad, rows):
    n = 1 << bits
    rows = rows if rows > 0 else (160 if bits == 13 else 128) + rows
    w, pads = inputs(rows, cols, pad)
    dw, dp = backend.upload_device(w.reshape(-1)), backend.upload_device(pads.reshape(-1))
    msgs = backend.pcs_messages_device(dw, 0, dp, 0, rows, cols, pad, n)
    chain = backend.ntt_fp_batch_device(msgs, rows, n)
    fused = backend.pcs_encode_device(dw, 0, dp, 0, rows, cols, pad, n)
    got, got2 = backend.download_device(chain), backend.download_device(fused)
    for b in (dw, dp, msgs, chain, fused):
        backend.free_device(b)
    want = oracle.pcs_encode_i16(w.reshape(-1), pads.reshape(-1) if pad else None, rows, cols, pad, n).reshape(-1)
    assert (got == want).all() and (got2 == want).all()
