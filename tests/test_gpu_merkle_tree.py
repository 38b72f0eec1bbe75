"""The Merkle levels (subtrees of up to ten levels per workgroup, joins by one
lane or by a quad of lanes) and the chunk runs of the column hash, bit-exact
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 0xFFFF_FFFF_0000_0001


def tree_of(backend, m):
    rows, cols = m.shape
    buf = backend.upload_device(m.reshape(-1))
    tree = backend.hash_fp_tree_device(buf, rows, cols)
    got = backend.download_device(tree.storage).reshape(2 * cols - 1, 32)
    backend.free_device_merkle_tree(tree)
    backend.free_device(buf)
    return got


# one workgroup's sizes on both sides of the quad switch (256), of its limit
# (1,024), then one and two rounds of subtrees
@pytest.mark.parametrize("bits", [0, 1, 2, 5, 7, 8, 9, 10, 11, 12, 16, 18, 19])
def test_tree_levels(backend, oracle, bits):
    m = np.random.Generator(np.random.PCG64(bits)).integers(0, P, size=(3, 1 << bits), dtype=np.uint64)
    leaves = oracle.hash_fp_columns(m, *m.shape)
    assert (tree_of(backend, m) == oracle.merkle_tree(leaves).reshape(-1, 32)).all()


# runs of one and two chunks per thread, with a short last run and a short last
# chunk (the columns decide which: 64 columns to a wave)
@pytest.mark.parametrize("rows,bits", [(129, 6), (700, 8), (1300, 10), (300, 18), (140, 19)])
def test_chunk_runs(backend, oracle, rows, bits):
    m = np.random.Generator(np.random.PCG64(rows)).integers(0, P, size=(rows, 1 << bits), dtype=np.uint64)
    got = tree_of(backend, m)
    leaves = oracle.hash_fp_columns(m, rows, 1 << bits)
    assert (got[:1 << bits] == leaves.reshape(-1, 32)).all()


# runs of four chunks: nine chunks in 2^17 columns (runs of 4, 4 and 1), three in
# 2^19 (one run of 3); the rows repeat with a period of 251, so that the columns of
# a large matrix cost little to make, and a sample of the leaves is hashed again
@pytest.mark.parametrize("rows,bits,fp2", [(1030, 17, False), (300, 19, False), (515, 17, True)])
def test_long_chunk_runs(backend, oracle, rows, bits, fp2):
    from volta_mi355x import FP2
    cols, w = 1 << bits, 2 if fp2 else 1
    block = np.random.Generator(np.random.PCG64(rows)).integers(0, P, size=(251, cols * w), dtype=np.uint64)
    buf = backend.alloc_device(rows * cols, FP2 if fp2 else np.uint64)
    for r in range(0, rows, 251):
        part = block[: min(251, rows - r)].reshape(-1)
        backend.upload_into(buf, r * cols, part.view(FP2) if fp2 else part)
    tree = (backend.hash_fp2_tree_device if fp2 else backend.hash_fp_tree_device)(buf, rows, cols)
    got = backend.download_device(tree.storage).reshape(2 * cols - 1, 32)
    backend.free_device_merkle_tree(tree)
    backend.free_device(buf)
    picks = np.unique(np.concatenate([[0, 1, 63, 64, cols - 65, cols - 1],
                                      np.random.default_rng(bits).integers(0, cols, size=2000)]))
    picked = block.reshape(251, cols, w)[:, picks][np.arange(rows) % 251]
    if fp2:
        want = oracle.hash_fp2_columns(np.ascontiguousarray(picked), rows, len(picks))
    else:
        want = oracle.hash_fp_columns(np.ascontiguousarray(picked[:, :, 0]), rows, len(picks))
    assert (got[picks] == want.reshape(-1, 32)).all()
    assert (got == oracle.merkle_tree(got[:cols].copy()).reshape(-1, 32)).all()


def hash_in_scope(b, rows, cols, seed):
    """(tree, matrix) of a hash inside a coarse timing scope, where nothing may be allocated."""
    m = np.random.Generator(np.random.PCG64(seed)).integers(0, P, size=(rows, cols), dtype=np.uint64)
    buf, tree = b.upload_device(m.reshape(-1)), b.alloc_device((2 * cols - 1) * 32, np.uint8)
    live = b.get_stats()["live_device_bytes"]
    assert b.lib.volta_cuda_begin_coarse_timing(b.raw, 4) == 0
    rc = b.lib.volta_cuda_hash_fp_tree_device(b.raw, buf.id, 0, rows, cols, tree.id, 0)
    assert rc == 0, b.last_error()
    assert b.lib.volta_cuda_end_coarse_timing(b.raw) == 0
    assert b.get_stats()["live_device_bytes"] == live
    got = b.download_device(tree).reshape(-1, 32)
    for x in (buf, tree):
        b.free_device(x)
    return got, m


# columns of up to four chunks need no workspace as one run, so a new context
# hashes them inside a scope; after columns of five chunks (two runs of at most
# four) there is space for columns of eight
@pytest.mark.parametrize("warm,rows", [(0, 129), (0, 300), (0, 512), (520, 1024)])
def test_hash_where_workspaces_may_not_grow(oracle, warm, rows):
    from volta_mi355x import Backend
    cols = 1 << 10
    with Backend(timing_policy=1) as b:
        if warm:
            tree_of(b, np.ones((warm, cols), np.uint64))
        got, m = hash_in_scope(b, rows, cols, rows)
    assert (got == oracle.merkle_tree(oracle.hash_fp_columns(m, rows, cols)).reshape(-1, 32)).all()
