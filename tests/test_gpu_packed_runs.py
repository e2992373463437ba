"""dK/dV over short run tiles taken query by query (key-centric backward plans
with 8 or more query heads per kv head): runs of every length around half a
tile, mixed with grouped single queries and whole tiles, duplicates and empty
rows, against the fp32 oracle; run to run bitwise."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from helpers import assert_attn_close
from oracle.attention import sel_attn_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("g,d", [(8, 64), (16, 32), (16, 128), (64, 32)])
@pytest.mark.parametrize("batch", [1, 2])
def test_backward_mixed_runs(g, d, batch):
    gen = torch.Generator().manual_seed(g + d)
    tq = 128 // g
    lens = [1, 1, tq // 2, 1, tq // 2 + 1, 2, tq, 1, tq + 1, 3, 1, 1, 1, 2 * tq - 1]
    lens = (lens * (700 // sum(lens) + 1))
    n, hkv, nb, topk = sum(lens), 2, 12, 5
    sizes = np.full(nb, n // nb)
    sizes[-1] += n - sizes.sum()
    cu = torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32)
    half = nb // batch
    cu_sb = torch.tensor([0, half, nb] if batch == 2 else [0, nb], dtype=torch.int32)
    cu_q = torch.tensor([0, int(cu[half]), n] if batch == 2 else [0, n], dtype=torch.int32)
    rows = torch.stack([torch.randperm(half, generator=gen)[:topk]
                        for _ in range(hkv * len(lens))]).view(hkv, len(lens), topk)
    rows[:, 3::7, 1] = rows[:, 3::7, 0]  # a block listed twice
    rows[:, 5::11] = -1                  # runs that attend nothing
    rows = rows.repeat_interleave(torch.tensor(lens), dim=1).to(torch.int32).contiguous()
    q, do = (torch.randn(n, hkv * g, d, generator=gen).to(torch.bfloat16) * 0.5
             for _ in range(2))
    k, v = (torch.randn(n, hkv, d, generator=gen).to(torch.bfloat16) * 0.5 for _ in range(2))
    scale = d ** -0.5
    dev = [t.to(DEV) for t in (q, k, v, rows, cu_sb, cu, cu_q)]
    plan = H.SelAttnPlan(q.shape, k.shape, *dev[3:], backward=True, key_centric=True)
    got = []
    for _ in range(2):
        o, lse = plan.fwd(*dev[:3], scale)
        got.append((o, lse) + plan.bwd(do.to(DEV), *dev[:3], o, lse, scale))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    o, lse, dq, dk, dv, _ = got[0]
    qf, kf, vf = (t.float().requires_grad_() for t in (q, k, v))
    ref, _ = sel_attn_ref(qf, kf, vf, rows, cu_sb, cu, cu_q, scale)
    ref.backward(do.float())
    for name, a, b in (("out", o, ref), ("dq", dq, qf.grad), ("dk", dk, kf.grad),
                       ("dv", dv, vf.grad)):
        assert_attn_close(a, b.detach(), name)
