"""The bounded top-k selection (2049 to 8192 blocks, topk <= 64): row counts
around the score tiles and the kernels' class counts, batch elements that
leave few or no whole tiles, ties beyond the listed columns, NaN scores, and
scores out of fp32's range, bit for bit against the oracle."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from oracle.select import select_blocks_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(pq, pk, cu_sb, topk, forced, force_self=True):
    nb, d = pk.shape
    cu = torch.arange(nb + 1, dtype=torch.int32)  # one-token blocks: pooled = given
    sb = torch.tensor(cu_sb, dtype=torch.int32)
    q = pq.view(nb, 1, d)
    topk_idx, compact = H.select_blocks(q.to(DEV), q.to(DEV), sb.to(DEV), cu.to(DEV), topk,
                                        forced, force_self, pooled_k=pk.to(DEV))
    ref = select_blocks_ref(q.numpy(), pk.view(nb, 1, d).numpy(), sb.numpy(), topk, forced,
                            force_self)
    np.testing.assert_array_equal(compact.cpu().numpy(), ref)
    np.testing.assert_array_equal(topk_idx.cpu().numpy(), ref)


@pytest.mark.parametrize("nb,topk", [(2049, 1), (2176, 64), (4096, 32), (4097, 33), (6144, 16),
                                     (6145, 64), (8191, 8), (8192, 64)])
def test_sizes(nb, topk):
    g = torch.Generator().manual_seed(nb + topk)
    _check(torch.randn(nb, 32, generator=g), torch.randn(nb, 32, generator=g), [0, nb], topk,
           [3, 3, nb - 1, nb, -1][:topk])


@pytest.mark.parametrize("cu_sb", [[0, 100, 1124, 2148, 2600], [7, 1032, 2090, 2090, 2599]])
@pytest.mark.parametrize("topk", [5, 64])
def test_batch_elements(cu_sb, topk):
    g = torch.Generator().manual_seed(topk)
    _check(torch.randn(2600, 32, generator=g), torch.randn(2600, 32, generator=g), cu_sb, topk,
           [2, 50, 1030], force_self=topk == 5)


@pytest.mark.parametrize("kind", ["equal", "nan", "few_finite", "huge", "tiny", "clustered"])
def test_scores(kind):
    nb, topk, d = 2300, 32, 32
    g = torch.Generator().manual_seed(9)
    pq, pk = torch.zeros(nb, d), torch.zeros(nb, d)
    pq[:, 0] = 1.0
    pk[:, 0] = torch.randn(nb, generator=g)
    if kind == "equal":         # every column ties with the bound
        pk[:, 0] = 0.25
    elif kind == "nan":         # ranked last, by id
        pk[::2, 0] = float("nan")
    elif kind == "few_finite":  # fewer scores than picks
        pk[:, 0] = float("nan")
        pk[5::500, 0] = -1.0
    elif kind == "huge":        # fp64 scores beyond fp32, both signs, infinities
        pq[:, 0] = 1e30
        pk[:, 0] *= 1e30
        pk[100:110, 0] = float("inf")
        pk[200:210, 0] = -float("inf")
    elif kind == "tiny":        # below fp32's smallest numbers
        pq[:, 0] = 1e-30
        pk[:, 0] *= 1e-25
    else:                       # the best scores are neighbours
        pk[:, 0] = -(torch.arange(nb) - 1200).abs() / 64.0
    _check(pq, pk, [0, nb], topk, [1])


@pytest.mark.parametrize("nb,topk", [(2880, 64), (2881, 33), (4881, 32), (8192, 64)])
@pytest.mark.parametrize("kind", ["equal", "nan", "late", "steps"])
def test_ties_in_pieces(nb, topk, kind):
    # more columns at the bound than are listed: pieces of 960 columns
    pq, pk = torch.zeros(nb, 32), torch.zeros(nb, 32)
    pq[:, 0] = 1.0
    i = torch.arange(nb)
    if kind == "equal":
        pk[:, 0] = 0.25
    elif kind == "nan":
        pk[:, 0] = float("nan")
    elif kind == "late":    # a few columns above the ties in every piece
        pk[(i % 960 == 959) | (i == nb - 1), 0] = 1.0 + nb
    else:                   # the better columns come later, piece by piece
        pk[:, 0] = (i // 700).float()
    _check(pq, pk, [0, nb], topk, [1, 960, nb - 2, 961])


def test_ties_cost_no_scan_per_pick():
    # one layer's scores all equal (zero projections) or NaN (a diverged step)
    # against ordinary ones: the same pass over the scores, some more ranking
    nb, topk = 4881, 32
    cu = torch.arange(nb + 1, dtype=torch.int32, device=DEV)
    sb = torch.tensor([0, nb], dtype=torch.int32, device=DEV)
    q, k = torch.randn(2, nb, 4, 64, device=DEV)

    def best(keys):
        times = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            H.select_blocks(q, keys, sb, cu, topk)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    usual = best(k)
    for value in (0.25, float("nan")):
        assert best(torch.full_like(k, value)) <= 2 * usual
