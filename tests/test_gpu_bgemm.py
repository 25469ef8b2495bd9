"""The large-batch GEMM (k_bgemm) through batched_dequant_matmul, at the edges
of its tiles: 32 tokens per tile and 1..4 tiles per workgroup, 128 / 256 rows
per workgroup, 256-value steps (Q8_0 rows may end inside one), K splits.

The oracle is float64 over the dequantized weight and the oracle's own Q8_0
codes of each row.  Tolerance: every output is a sum of at most K/32 block
terms (plus one offset per 256 values), each rounded a few times; every
intermediate is at most twice A = sum over blocks of max|w| * sum|x|, so with
r = K/32 + 16 roundings of relative size 2^-24 the error stays below
2 r A 2^-24 (weights here are zero-mean normals, so a Q4_K block's offset and
centred codes are both within twice its largest weight)."""
import ctypes as C

import numpy as np
import pytest

from flarellm_amd import FL_Q4K, FL_Q8_0
from flarellm_amd import synth as S
from flarellm_amd._lib import check

pytestmark = pytest.mark.gpu


def _check(backend, oracle, fmt, rows, cols, batch, edit=None):
    import torch

    print(f"[bgemm] fmt={fmt} {rows}x{cols} batch={batch}", flush=True)
    w = S.quantize(S.normal(rows + 7 * cols, 0, rows * cols, 0, 0.02).reshape(rows, cols), fmt)
    W = backend.upload(S.QWeight(w, fmt, rows, cols))
    x = S.normal(batch + cols, 0, batch * cols, 0.0, 1.0).reshape(batch, cols)
    if edit is not None:
        edit(x)
    got = backend.batched_dequant_matmul(W, torch.from_numpy(x).cuda()).cpu().numpy()
    W.free()
    ok = np.isfinite(x).all(axis=1)
    wd = oracle.dequant(w, fmt, rows, cols).astype(np.float64)
    xd = np.zeros((batch, cols))
    for t in np.flatnonzero(ok):
        q, s = oracle.quantize_q8(x[t])
        xd[t] = (q.reshape(-1, 32).astype(np.float64) * s.astype(np.float64)[:, None]).reshape(-1)
    want = xd @ wd.T
    A = np.abs(xd).reshape(batch, -1, 32).sum(2) @ np.abs(wd).reshape(rows, -1, 32).max(2).T
    bound = 2 * (cols // 32 + 16) * A * 2.0 ** -24
    err = np.abs(got - want)
    assert (err[ok] <= bound[ok]).all(), float((err[ok] / np.maximum(bound[ok], 1e-30)).max())
    assert not np.isfinite(got[~ok]).any()


@pytest.mark.parametrize("fmt,rows,cols", [(FL_Q4K, 130, 256), (FL_Q4K, 257, 1536), (FL_Q8_0, 33, 32),
                                           (FL_Q8_0, 131, 544), (FL_Q8_0, 256, 2080)])
@pytest.mark.parametrize("batch", [17, 32, 33, 97, 128, 129, 300])
def test_tile_edges(backend, oracle, fmt, rows, cols, batch):
    _check(backend, oracle, fmt, rows, cols, batch)


@pytest.mark.parametrize("fmt,rows,cols,batch", [(FL_Q4K, 4096, 4096, 70), (FL_Q8_0, 2048, 8192, 77),
                                                 (FL_Q4K, 1024, 14336, 40), (FL_Q8_0, 64, 64, 2100),
                                                 (FL_Q4K, 6145, 512, 520)])
def test_splits_and_pieces(backend, oracle, fmt, rows, cols, batch):
    """Deep K splits, batches larger than one piece, many token groups."""
    _check(backend, oracle, fmt, rows, cols, batch)


# (format, token tiles, waves, K split): every kernel the planner picks from,
# whole and split rows, at ragged sizes
VARIANTS = [(FL_Q8_0, 1, 4, False, 102, 256, 17), (FL_Q8_0, 1, 4, True, 102, 544, 17),
            (FL_Q8_0, 2, 4, False, 12260, 256, 65), (FL_Q8_0, 2, 4, True, 129, 800, 1134),
            (FL_Q8_0, 2, 8, False, 13436, 256, 136), (FL_Q8_0, 2, 8, True, 133, 1344, 1347),
            (FL_Q8_0, 3, 8, False, 9476, 256, 388), (FL_Q8_0, 3, 8, True, 131, 2368, 1712),
            (FL_Q8_0, 4, 8, False, 11080, 256, 488), (FL_Q8_0, 4, 8, True, 133, 6176, 1253),
            (FL_Q4K, 1, 4, False, 100, 256, 17), (FL_Q4K, 1, 4, True, 103, 1024, 17),
            (FL_Q4K, 2, 4, False, 10844, 256, 336), (FL_Q4K, 2, 4, True, 9277, 1792, 34),
            (FL_Q4K, 2, 8, False, 13084, 256, 132), (FL_Q4K, 2, 8, True, 129, 2304, 897),
            (FL_Q4K, 3, 8, False, 13059, 256, 262), (FL_Q4K, 3, 8, True, 129, 3584, 1168),
            (FL_Q4K, 4, 8, False, 13229, 256, 392), (FL_Q4K, 4, 8, True, 135, 6400, 1231)]


@pytest.mark.parametrize("fmt,tt,nw,split,rows,cols,batch", VARIANTS)
def test_every_variant(backend, oracle, fmt, tt, nw, split, rows, cols, batch):
    plan = (C.c_int32 * 6)()
    check(backend.lib.fl_plan_batched_matmul(fmt, rows, cols, batch, 0, plan), backend.ctx)
    assert (plan[0], plan[1], plan[4] > 1) == (tt, nw, split), tuple(plan)
    _check(backend, oracle, fmt, rows, cols, batch)


@pytest.mark.parametrize("fmt", [FL_Q4K, FL_Q8_0])
def test_odd_values(backend, oracle, fmt):
    """Zero rows, tiny and large magnitudes, and rows that are not finite
    (which reach no other token)."""

    def edit(x):
        x[0] = 0.0
        x[1] *= 1e-30
        x[2] *= 1e6
        x[3, 5] = np.inf
        x[34, :32] = np.inf
        x[35] = 0.0
        x[35, 7] = 3.0

    _check(backend, oracle, fmt, 160, 512, 40, edit)


@pytest.mark.parametrize("fmt,rows,cols,batch", [(FL_Q4K, 257, 1536, 300), (FL_Q8_0, 131, 2080, 333)])
@pytest.mark.parametrize("mib", [1, 0])
def test_little_workspace(backend, oracle, fmt, rows, cols, batch, mib):
    """More rows than the workspace's limit holds: fewer at a time, 32 at least."""
    from flarellm_amd import _lib as L

    backend.set_option(L.FL_OPT_WORKSPACE_MIB, mib)
    try:
        _check(backend, oracle, fmt, rows, cols, batch)
    finally:
        backend.set_option(L.FL_OPT_WORKSPACE_MIB, -1)
