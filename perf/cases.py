"""Timed workloads of the Ligero commitment library, through its public entry points.

Every case is work that a prover built on this library asks for: committing a
weight matrix (placements, masking pads, encode, BLAKE3 tree, root), encoding
with the proximity combinations, encoding u64 rows, opening a commitment, and
the transforms of the evaluation-domain and extension-field steps.  Outputs are
field elements, hashes and bytes: they are compared bit for bit.

``listed()`` holds the configurations of this repository's benchmark and
production layouts plus a small and two mid-size commitments; ``draw()`` gives
further sizes over the same ranges, odd ones among them.
"""
from __future__ import annotations

import pathlib
import sys

import numpy as np
import torch

_ROOT = pathlib.Path(__file__).resolve().parents[1]
if str(_ROOT / "volta-zk_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "volta-zk_amd"))

from volta_mi355x import accel, ligero, workloads  # noqa: E402

P = accel.P
FP2 = accel.FP2
CACHE_LIMIT = 64 << 30  # resident cache kept between workloads, bytes

_backend = None


def backend() -> accel.Backend:
    """The one context a prover process keeps (timing as the reference's report
    runs it: counters only, no events around each call)."""
    global _backend
    if _backend is None:
        _backend = accel.Backend(timing_policy=1)
    return _backend


# ---- the cases ------------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # The smallest commitments: a bias or a test-size matrix, where the
        # number of launches and the latency of each decide.
        dict(name="commit_small", kind="commit", rows=24, col_bits=6, pad=16, code_bits=8, layout=""),
        # A narrow projection matrix with an odd number of rows, codewords of 2^12.
        dict(name="commit_4096", kind="commit", rows=1531, col_bits=10, pad=128, code_bits=12, layout=""),
        # A layer matrix on the 2^13 layout with masking pads.
        dict(name="commit_8192_pads", kind="commit", rows=8192, col_bits=11, pad=512, code_bits=13, layout=""),
        # The reference's production weights commitment: 48 tensors, 24,576 x 2^13 -> 2^15.
        dict(name="commit_weights", kind="commit", rows=24576, col_bits=13, pad=512, code_bits=15, layout="weights"),
        # The reference's production embedding commitment: 2,080 x 2^15 -> 2^17.
        dict(name="commit_embed", kind="commit", rows=2080, col_bits=15, pad=512, code_bits=17, layout="embed"),
        # One c_attn matrix (C2): encode and two challenge-power combinations.
        dict(name="encode_c_attn", kind="encode", rows=1024, col_bits=11, code_bits=13, combinations=2),
        # The full GPT-2-small weight matrix (C3), the headline step.
        dict(name="encode_gpt2", kind="encode", rows=1 << 16, col_bits=11, code_bits=13, combinations=2),
        # u64 rows at rate 1/4 with one combination of all rows (C1).
        dict(name="rows_16384", kind="rows", rows=256, msg_len=1 << 12, code_bits=14, combinations=1),
        # u64 rows at rate 1/8 (C4), packed four i16 lanes to an element.
        dict(name="rows_32768", kind="rows", rows=1 << 15, msg_len=1 << 12, code_bits=15, combinations=0),
        # Long transforms in both directions, a combination and an opening's
        # columns (C5).
        dict(name="transform_2_24", kind="transform", rows=64, bits=24, queries=256),
        # The opening of an embedding commitment: 6 block claims, 120 queries.
        dict(name="open_embed", kind="open", rows=2080, col_bits=15, pad=512, code_bits=17, claims=6, queries=120),
        # An extension-field codeword: evaluations to coefficients, transform at
        # rate 1/8, and the folds of the proximity test.
        dict(name="x4_2_24", kind="x4", bits=21, code_bits=24, folds=12),
    ]


def _log(rng, lo: float, hi: float) -> int:
    """An integer spread over the logarithm of [lo, hi]."""
    return max(int(lo), min(int(hi), int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["commit", "commit", "encode", "rows", "transform", "open", "x4"])
    most = 1 << 27  # codeword elements of a drawn case
    if kind in ("commit", "open"):
        code_bits = rng.randint(8 if kind == "commit" else 10, 17)
        col_bits = code_bits - rng.choice([2, 2, 3])
        pad = _log(rng, 8, min(512, 1 << (code_bits - 2)))
        rows = _log(rng, 8, min(20000, most >> code_bits))
        if kind == "commit":
            return dict(kind=kind, rows=rows, col_bits=col_bits, pad=pad, code_bits=code_bits, layout="")
        rows = max(rows, 32)
        return dict(kind=kind, rows=rows, col_bits=col_bits, pad=pad, code_bits=code_bits, claims=rng.randint(1, 16),
                    queries=rng.randint(20, 150))
    if kind == "encode":
        code_bits = rng.randint(11, 15)
        return dict(kind=kind, rows=_log(rng, 16, min(60000, most >> code_bits)),
                    col_bits=code_bits - rng.choice([2, 2, 3]), code_bits=code_bits, combinations=rng.randint(1, 3))
    if kind == "rows":
        code_bits = rng.randint(9, 16)
        return dict(kind=kind, rows=_log(rng, 8, min(40000, most >> code_bits)),
                    msg_len=_log(rng, 1 << (code_bits - 4), (1 << code_bits) - 1), code_bits=code_bits,
                    combinations=rng.randint(0, 2))
    if kind == "transform":
        bits = rng.randint(12, 22)
        return dict(kind=kind, rows=_log(rng, 1, min(64, most >> bits)), bits=bits, queries=rng.randint(20, 300))
    code_bits = rng.randint(12, 23)
    return dict(kind=kind, bits=code_bits - rng.choice([1, 2, 3]), code_bits=code_bits,
                folds=rng.randint(4, code_bits - 3))


# ---- inputs ---------------------------------------------------------------------------------

class _Region:
    """Device memory of a resident buffer as torch sees it."""

    def __init__(self, ptr: int, shape, typestr: str, keep):
        self.keep = keep
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False),
                                         "version": 3, "strides": None}


class _Owned:
    """Resident buffers of one result, returned to the pool with it."""

    def __init__(self, b, bufs):
        self.b, self.bufs = b, list(bufs)

    def __del__(self):
        for buf in self.bufs:
            self.b.free_device(buf)


_TYPES = {np.dtype(np.uint64): "<i8", np.dtype(np.int16): "<i2", np.dtype(np.uint8): "|u1"}


def _tensor(b, buf, keep, shape=None):
    """A resident buffer as a tensor: u64 words as int64 (torch's widest), Fp2 as pairs of them."""
    n = buf.len * 2 if buf.dtype == FP2 else buf.len
    typestr = "<i8" if buf.dtype == FP2 else _TYPES[buf.dtype]
    return torch.as_tensor(_Region(b.device_ptr(buf), shape or (n,), typestr, keep), device="cuda")


def _resident(b, t: torch.Tensor, dtype):
    """A resident buffer holding the tensor's values (through a second one, so
    that the library alone knows the address of what the program keeps)."""
    n = t.numel() // 2 if dtype == FP2 else t.numel()
    stage = b.alloc_device(n, dtype)
    b.synchronize()  # torch writes on a stream of its own
    _tensor(b, stage, None).copy_(t.reshape(-1))
    torch.cuda.synchronize()
    buf = b.alloc_device(n, dtype)
    b.copy_device_rows(stage, 0, n, buf, 0, n, 1, n)
    b.synchronize()
    b.free_device(stage)
    return buf


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(g, n: int) -> torch.Tensor:
    """Quantised weights: i16 ~ N(0, 2000^2), rounded and clipped."""
    return torch.randn(n, generator=g, device="cuda").mul_(2000.0).round_().clamp_(-32768, 32767).to(torch.int16)


def _field(g, n: int) -> torch.Tensor:
    """Uniform field elements in [0, p) as int64 words."""
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (n,), generator=g, device="cuda", dtype=torch.int64)
    high = (x < 0) & (x > -(1 << 32))  # words from p on
    x[high] += (1 << 32) - 1
    return x


def _fp2(rng: np.random.Generator, count: int) -> np.ndarray:
    return rng.integers(0, P, size=(count, 2), dtype=np.uint64)


class _State:
    """A case's inputs on the device; its buffers go back to the pool with it."""

    def __init__(self, b, case):
        self.b, self.case, self.bufs = b, case, []

    def keep(self, buf):
        self.bufs.append(buf)
        return buf

    def __del__(self):
        for buf in self.bufs:
            self.b.free_device(buf)


def prepare(case: dict, seed: int) -> _State:
    b = backend()
    if b.memory_breakdown()[2] > CACHE_LIMIT:
        b.lib.volta_cuda_trim_resident_cache(b.raw)
    s = _State(b, case)
    g, rng, kind = _gen(seed), np.random.Generator(np.random.PCG64(seed)), case["kind"]
    if kind in ("commit", "open", "encode"):
        s.params = ligero.LigeroParams(case["rows"], case["col_bits"], case.get("pad", 0), case["code_bits"],
                                       case.get("queries", 0))
        s.seed = rng.bytes(32)
    if kind == "commit":
        total = case["rows"] << case["col_bits"]
        slots = {"weights": workloads.c3_weights_slots, "embed": workloads.c3_embed_slots}
        if case["layout"]:
            shapes, packed = slots[case["layout"]]()
            assert packed == total
        else:
            shapes = [workloads.TensorSlot("w", case["rows"], 1 << case["col_bits"], 0, 1 << case["col_bits"])]
        s.tensors = [(t, s.keep(_resident(b, _weights(g, t.k * t.n), np.int16))) for t in shapes]
        if case["layout"]:
            s.placements = [ligero.ResidentWeightPlacement(buf, 0, t.k, t.n, t.offset, t.stride, total)
                            for t, buf in s.tensors]
        else:
            # one block of whole rows: consecutive placements of power-of-two row counts
            s.placements, row = [], 0
            while row < case["rows"]:
                k = 1 << ((case["rows"] - row).bit_length() - 1)
                cols = 1 << case["col_bits"]
                s.placements.append(ligero.ResidentWeightPlacement(s.tensors[0][1], row * cols, k, cols, row * cols,
                                                                   cols, total))
                row += k
    elif kind == "encode":
        s.weights = s.keep(_resident(b, _weights(g, case["rows"] << case["col_bits"]), np.int16))
        s.challenges = [tuple(int(v) for v in c) for c in _fp2(rng, case["combinations"])]
    elif kind == "rows":
        s.msgs = s.keep(_resident(b, _field(g, case["rows"] * case["msg_len"]), np.uint64))
        k = case["combinations"]
        s.coeffs = s.keep(_resident(b, _field(g, 2 * k * case["rows"]), FP2)) if k else None
    elif kind == "transform":
        n = 1 << case["bits"]
        s.rows = s.keep(_resident(b, _field(g, case["rows"] * n), np.uint64))
        s.coeffs = s.keep(_resident(b, _field(g, 2 * case["rows"]), FP2))
        s.columns = rng.integers(0, n, size=case["queries"], dtype=np.uint32)
    elif kind == "open":
        p = s.params
        w = _resident(b, _weights(g, p.rows * p.cols), np.int16)
        _, s.matrix = ligero.finish_resident_commit(b, w, p, s.seed)
        s.bufs += [s.matrix.weights, s.matrix.pads, s.matrix.encoded, s.matrix.tree.storage]
        # claims on blocks of rows: the largest power of two that fits, then smaller ones
        s.claims = []
        for k in range(case["claims"]):
            bits = max(0, (p.rows.bit_length() - 1) - k)
            at = int(rng.integers(0, p.rows >> bits)) << bits
            s.claims.append((at << p.col_bits, _fp2(rng, p.col_bits + bits)))
        s.challenge = tuple(int(v) for v in _fp2(rng, 1)[0])
        s.queries = rng.integers(0, p.code_len, size=case["queries"], dtype=np.uint32)
    elif kind == "x4":
        s.evals = s.keep(_resident(b, _field(g, 2 << case["bits"]), FP2))
        s.challenges = [tuple(int(v) for v in c) for c in _fp2(rng, case["folds"])]
    else:
        raise ValueError(f"unknown case kind {kind!r}")
    b.synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------

def run(s: _State):
    b, case, kind = s.b, s.case, s.case["kind"]
    if kind == "commit":
        root, m = ligero.commit_resident_from_device(b, s.placements, s.params, s.seed)
        own = _Owned(b, (m.weights, m.pads, m.encoded, m.tree.storage))
        return {"root": np.frombuffer(root, np.uint8), "encoded": _tensor(b, m.encoded, own),
                "pads": _tensor(b, m.pads, own), "tree": _tensor(b, m.tree.storage, own)}
    if kind == "encode":
        enc, _ = ligero.commit_encode_resident(b, s.weights, s.params, fused=False)
        u = ligero.proximity_combinations(b, s.weights, None, s.params, s.challenges)
        own = _Owned(b, (enc, u))
        return {"encoded": _tensor(b, enc, own), "combinations": _tensor(b, u, own)}
    if kind == "rows":
        bufs = [b.ntt_fp_encode_device(s.msgs, case["rows"], case["msg_len"], 1 << case["code_bits"])]
        if s.coeffs is not None:
            bufs.append(b.combine_rows_fp_device(s.msgs, case["rows"], case["msg_len"], s.coeffs,
                                                 case["combinations"]))
        own = _Owned(b, bufs)
        return [_tensor(b, x, own) for x in bufs]
    if kind == "transform":
        rows, n = case["rows"], 1 << case["bits"]
        fwd = b.ntt_fp_batch_device(s.rows, rows, n)
        inv = b.ntt_fp_inverse_batch_device(fwd, rows, n)
        u = b.combine_rows_fp_device(fwd, rows, n, s.coeffs, 1)
        cols = b.pcs_gather_columns_device(fwd, rows, n, s.columns)
        own = _Owned(b, (fwd, inv, u, cols))
        return {"forward": _tensor(b, fwd, own), "inverse": _tensor(b, inv, own), "combination": _tensor(b, u, own),
                "columns": _tensor(b, cols, own)}
    if kind == "open":
        out = ligero.open_rows_resident(b, s.matrix, s.claims, s.challenge, s.queries, s.seed)
        out["mask_root"] = np.frombuffer(out["mask_root"], np.uint8)
        return {k: v.view(np.int64) if v.dtype == np.uint64 else v for k, v in out.items()}
    # x4: coefficients of the multilinear evaluations, codeword, folds
    size, n = 1 << case["bits"], 1 << case["code_bits"]
    coeffs = b.alloc_device(size, FP2)
    b.copy_device_rows(s.evals, 0, size, coeffs, 0, size, 1, size)
    b.fp2_mobius_inverse_inplace_device(coeffs)
    arena = b.alloc_device(2 * n, FP2)
    b.x4_ntt_fp2_device(coeffs, size, n, out=arena)
    at, length = 0, n
    for c in s.challenges:
        b.x4c_direct_fold_arena_into_arena(arena, at * 16, length, (at + length) * 16, c)
        at, length = at + length, length // 2
    own = _Owned(b, (coeffs, arena))
    return {"coefficients": _tensor(b, coeffs, own), "codewords": _tensor(b, arena, own)[:2 * (at + length)]}


def work(case: dict) -> dict:
    """Bytes: each input read once and each output written once.  The work is
    integer arithmetic mod p, so no floating-point operations are counted."""
    kind, rows = case["kind"], case.get("rows", 1)
    if kind in ("commit", "open"):
        cols, n = 1 << case["col_bits"], 1 << case["code_bits"]
        if kind == "commit":
            size = 2 * rows * cols
            if case["layout"] == "weights":
                size = 2 * 12 * (768 * 4096 + 768 * 768 + 768 * 3072 + 3072 * 768)
            elif case["layout"] == "embed":
                size = 2 * (50257 + 1024) * 768
            return {"bytes": size + 8 * rows * (n + case["pad"]) + 32 * (2 * n - 1), "flops": 0}
        msg, k, q = cols + case["pad"], case["claims"], case["queries"]
        read = 2 * rows * cols + 8 * rows * case["pad"] + q * (8 * rows + 32 * case["code_bits"])
        wrote = 16 * (k + 1) * msg + q * (8 * rows + 16 * (k + 1) + 64 * case["code_bits"])
        return {"bytes": read + wrote, "flops": 0}
    if kind == "encode":
        cols, n = 1 << case["col_bits"], 1 << case["code_bits"]
        return {"bytes": rows * (2 * cols + 8 * n) + 16 * case["combinations"] * cols, "flops": 0}
    if kind == "rows":
        k, m = case["combinations"], case["msg_len"]
        return {"bytes": 8 * rows * (m + (1 << case["code_bits"])) + 16 * k * (rows + m), "flops": 0}
    if kind == "transform":
        n = 1 << case["bits"]
        return {"bytes": 24 * rows * n + 16 * (rows + n) + 12 * case["queries"] * rows, "flops": 0}
    size, n = 1 << case["bits"], 1 << case["code_bits"]
    return {"bytes": 16 * (2 * size + 2 * n - (n >> case["folds"])), "flops": 0}


def tolerance(case: dict):
    """Residues, hashes and bytes: every correct implementation gives the same."""
    return "exact"


def exact(case: dict, seed: int):
    """The outputs are whole numbers, compared bit for bit; none is a rounded value."""
    return None
