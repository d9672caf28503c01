"""admp_pairwise_compute_noalloc (the entry point that allocates nothing) against
admp_pairwise_compute on the same pairs, through the C ABI: every short-range
kind, both precisions, two calls in a row with the second on a smaller system
(fewer sites and pairs), so results cannot lean on the first call's scratch.
Tolerance: 1e-12 relative (both evaluate the same per-pair arithmetic and differ
only in the order of the FP64 sums)."""
import ctypes

import numpy as np
import pytest
import torch

from dmff_amd import _lib as L
from tests.systems import pairwise_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _subsystem(kind, n):
    """The kind's test system restricted to its first n sites."""
    pos, box, pairs, m, prm = pairwise_case(kind)
    keep = (pairs[:, 0] < n) & (pairs[:, 1] < n)
    return pos[:n], box, pairs[keep], m, prm[:n]


def _with_context(kind, prec, pos, box, pairs, m, prm):
    from dmff_amd.admp.engine import Engine
    eng = Engine(len(pos), 0, False, False, 0.0, (0, 0, 0), 9.0, precision=prec, device=DEV)
    eng.set_topology(None, None, {})
    eng.set_pairs(torch.as_tensor(pairs))
    E, g = eng.pairwise_compute(kind, pos, box, prm, m)
    return float(E[0]), g["pos"][0].cpu().numpy(), g["box"][0].cpu().numpy(), g["prm"][0].cpu().numpy()


def _noalloc(kind, prec, pos, box, pairs, m, prm, int64=True):
    lib = L.load()
    n, npr = len(pos), prm.shape[1]
    dev = torch.device(DEV)
    P = torch.as_tensor(pos, dtype=F64, device=dev).contiguous()
    B = torch.as_tensor(box, dtype=F64, device=dev).contiguous()
    pr = torch.as_tensor(pairs.astype(np.int64 if int64 else np.int32), device=dev).contiguous()
    Q = torch.as_tensor(prm, dtype=F64, device=dev).contiguous()
    ms = np.ascontiguousarray(m, dtype=np.float64)
    E = torch.full((1,), 7.0, dtype=F64, device=dev)
    gp = torch.full((n, 3), 7.0, dtype=F64, device=dev)   # stale values: the call must clear them
    gb = torch.full((3, 3), 7.0, dtype=F64, device=dev)
    gq = torch.full((n, npr), 7.0, dtype=F64, device=dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    st = lib.admp_pairwise_compute_noalloc(kind, L.ADMP_MIXED if prec == "mixed" else L.ADMP_FP64, n, _p(P), _p(B),
                                           _p(pr), len(pairs), 1 if int64 else 0, _p(Q), npr,
                                           ms.ctypes.data_as(ctypes.c_void_p), len(ms), 1, _p(E), _p(gp), _p(gb),
                                           _p(gq), ctypes.c_void_p(stream))
    assert st == L.ADMP_OK, lib.admp_last_error(None)
    torch.cuda.synchronize()
    return float(E[0]), gp.cpu().numpy(), gb.cpu().numpy(), gq.cpu().numpy()


def _rel(a, b):
    a, b = np.asarray(a, dtype=np.float64).ravel(), np.asarray(b, dtype=np.float64).ravel()
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("n_pairs", [1, 2047, 2048, 2049, None])
def test_noalloc_chunks_and_full_site_table(order, n_pairs):
    """1,728 sites, more than one chunk's table of sites holds, on a jittered lattice: a chunk
    less one pair, one chunk, one more, and every pair inside 5 A; the shuffled list fills the
    table.  Tolerance as above."""
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), -1).reshape(-1, 3) * 2.5
    pos, box = g + rng.uniform(-0.4, 0.4, g.shape), np.eye(3) * 30.0
    d = pos[:, None] - pos[None]
    d -= np.round(d / 30.0) * 30.0
    i, j = np.nonzero(np.triu((d ** 2).sum(-1) < 25.0, 1))
    pairs = np.stack([i, j, np.zeros_like(i)], 1)
    if order == "shuffled":
        pairs = pairs[rng.permutation(len(pairs))]
    pairs = pairs[:n_pairs]
    prm = rng.uniform(2.0, 4.0, (len(pos), 4))
    m = np.array([0.0, 0.0, 0.0, 1.0, 1.0, 1.0])
    ref = _with_context(2, "fp64", pos, box, pairs, m, prm)
    got = _noalloc(2, "fp64", pos, box, pairs, m, prm)
    errs = [abs(got[0] - ref[0]) / abs(ref[0])] + [_rel(got[k], ref[k]) for k in (1, 2, 3)]
    print(f"{order} {len(pairs)} pairs: {errs}", flush=True)
    assert max(errs) < 1e-12


@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("n_pairs", [255, 256, 257, 65536, 65537, 131073, 262144, 262145, None])
def test_noalloc_chunk_lengths(order, n_pairs):
    """The lattice with pairs inside 12 A: list lengths at which a chunk's length doubles (256 to
    2048 pairs); the longest shuffled list fills the table.  Tolerance as above."""
    rng = np.random.default_rng(7)
    g = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), -1).reshape(-1, 3) * 2.5
    pos, box = g + rng.uniform(-0.4, 0.4, g.shape), np.eye(3) * 30.0
    d = pos[:, None] - pos[None]
    d -= np.round(d / 30.0) * 30.0
    i, j = np.nonzero(np.triu((d ** 2).sum(-1) < 144.0, 1))
    pairs = np.stack([i, j, np.zeros_like(i)], 1)
    assert len(pairs) > 262145
    if order == "shuffled":
        pairs = pairs[rng.permutation(len(pairs))]
    pairs = pairs[:n_pairs]
    prm = rng.uniform(2.0, 4.0, (len(pos), 4))
    m = np.array([0.0, 0.0, 0.0, 1.0, 1.0, 1.0])
    ref = _with_context(2, "fp64", pos, box, pairs, m, prm)
    got = _noalloc(2, "fp64", pos, box, pairs, m, prm)
    errs = [abs(got[0] - ref[0]) / abs(ref[0])] + [_rel(got[k], ref[k]) for k in (1, 2, 3)]
    print(f"{order} {len(pairs)} pairs: {errs}", flush=True)
    assert max(errs) < 1e-12


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", [1, 2, 3, 4])
def test_noalloc_equals_context_entry_point_twice(kind, prec):
    for n, int64 in ((60, True), (37, False)):
        case = _subsystem(kind, n)
        ref = _with_context(kind, prec, *case)
        got = _noalloc(kind, prec, *case, int64=int64)
        errs = [abs(got[0] - ref[0]) / abs(ref[0])] + [_rel(got[k], ref[k]) for k in (1, 2, 3)]
        print(f"kind {kind} {prec} n={n} pairs={len(case[2])}: E {got[0]:.15e} ref {ref[0]:.15e} "
              f"errors E/pos/box/prm {errs}", flush=True)
        assert max(errs) < 1e-12, (kind, prec, n, errs)


def test_noalloc_argument_errors():
    lib = L.load()
    ms = np.ones(6)
    z = ctypes.c_void_p(0)
    st = lib.admp_pairwise_compute_noalloc(9, 0, 10, z, z, z, 0, 1, z, 2, ms.ctypes.data_as(ctypes.c_void_p), 6, 0,
                                           z, z, z, z, z)
    assert st == 1 and b"kind" in lib.admp_last_error(None)
    st = lib.admp_pairwise_compute_noalloc(1, 0, 10, z, z, z, 0, 1, z, 3, ms.ctypes.data_as(ctypes.c_void_p), 6, 0,
                                           z, z, z, z, z)
    assert st == 1 and b"n_prm" in lib.admp_last_error(None)
    st = lib.admp_pairwise_compute_noalloc(1, 0, 1 << 28, z, z, z, 0, 1, z, 2, ms.ctypes.data_as(ctypes.c_void_p),
                                           6, 0, z, z, z, z, z)
    assert st == 1 and b"n_atoms" in lib.admp_last_error(None)
