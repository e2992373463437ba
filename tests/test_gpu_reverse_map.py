"""The reverse query map's stable counting sort (lsrm_reverse_query_map)
against its oracle, bit for bit, at the edges of its parts: groups of 64
queries, chunks, windows of 4096 blocks, rows of whole 16-byte pieces and
others, rows that list a block twice, padding and ids out of range."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from oracle.revmap import reverse_query_map_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,nb", [
    (1, 1, 1), (63, 4, 7), (64, 3, 40), (65, 16, 40), (130, 33, 300), (4097, 8, 4095),
    (1000, 12, 4096), (1000, 16, 4097), (700, 32, 8193), (20011, 4, 462), (3001, 64, 70)])
@pytest.mark.parametrize("rows", ["distinct", "repeated", "one_block"])
@pytest.mark.parametrize("batch", [1, 3])
def test_counting_sort(n, k, nb, rows, batch):
    if batch > min(n, nb):
        pytest.skip("an element for every sequence")
    gen = torch.Generator().manual_seed(n * 131 + k)
    hkv = 2
    cu_q = [n * i // batch for i in range(batch + 1)]
    cu_sb = [nb * i // batch for i in range(batch + 1)]
    nbb = cu_sb[1]
    if rows == "one_block":  # every listing in one block's segment
        topk = torch.full((hkv, n, k), nbb - 1, dtype=torch.int32)
        topk[:, :, 1:] = -1
    elif rows == "repeated":
        topk = torch.randint(-2, nbb + 2, (hkv, n, k), generator=gen, dtype=torch.int32)
        topk[:, ::3] = topk[:, ::3, :1]  # one id in every slot
    else:
        start = torch.randint(0, max(1, nbb), (hkv, n, 1), generator=gen)
        topk = ((start + torch.arange(k)) % max(nbb, k)).to(torch.int32)
    dev = torch.device("cuda:0")
    t = [torch.tensor(x, dtype=torch.int32) for x in (cu_q, cu_sb)]
    cu_rev, rev = H.reverse_query_map(topk.to(dev), t[0].to(dev), t[1].to(dev), nb)
    ref_cu, ref_lists = reverse_query_map_ref(topk.numpy(), t[0].numpy(), t[1].numpy(), nb)
    assert np.array_equal(cu_rev.cpu().numpy(), ref_cu)
    got = rev.cpu().numpy()
    for h in range(hkv):
        assert np.array_equal(got[h, :ref_cu[h, -1]], np.asarray(ref_lists[h], dtype=np.int32))
