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


def test_packed_plan_run_without_flags():
    # A key-centric backward plan also serves the entry point without plan
    # flags: with runs of three equal rows only (no grouped tile), every query
    # is in the packed map and must still be found there.
    gen = torch.Generator().manual_seed(3)
    n, hkv, g, d, nb, topk = 384, 2, 16, 32, 8, 3
    rows = torch.stack([torch.randperm(nb, generator=gen)[:topk] for _ in range(hkv * n // 3)])
    rows = rows.view(hkv, n // 3, topk).repeat_interleave(3, dim=1).to(torch.int32).contiguous()
    cu = torch.arange(nb + 1, dtype=torch.int32) * (n // nb)
    cu_sb, cu_q = (torch.tensor([0, x], dtype=torch.int32) for x in (nb, n))
    q, do = (torch.randn(n, hkv * g, d, generator=gen).to(torch.bfloat16) * 0.5
             for _ in range(2))
    k, v = (torch.randn(n, hkv, d, generator=gen).to(torch.bfloat16) * 0.5 for _ in range(2))
    q, k, v, do, rows, cu_sb, cu, cu_q = (t.to(DEV) for t in (q, k, v, do, rows, cu_sb, cu, cu_q))
    plan = H.SelAttnPlan(q.shape, k.shape, rows, cu_sb, cu, cu_q, backward=True, key_centric=True)
    o, lse = plan.fwd(q, k, v, d ** -0.5)
    want = plan.bwd(do, q, k, v, o, lse, d ** -0.5)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    delta = torch.empty(hkv * g, n, dtype=torch.float32, device=DEV)
    p = H._ptr
    assert H.lib().lsrm_sel_attn_bwd_run(
        p(do), p(q), p(k), p(v), p(o), p(lse), H.BF16, n, n, hkv * g, hkv, d, p(rows), topk,
        p(cu_sb), p(cu), nb, p(cu_q), 1, d ** -0.5, p(dq), p(dk), p(dv), p(delta), p(plan.ws),
        plan.ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
    assert float(dk.float().abs().max()) > 0
    for a, b in zip((dq, dk, dv, delta), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("run,listed", [(5, False), (4, True), (1, True)])
@pytest.mark.parametrize("key_centric", [True, False])
def test_query_map_counts_as_used_only_if_it_lists(run, listed, key_centric):
    # Runs longer than half a tile are neither packed nor grouped: dK/dV runs
    # without the map's steps (they cost 3 to 10% of its time), whether or not
    # the plan is key-centric.  The word lies two behind the backward marker.
    gen = torch.Generator().manual_seed(run)
    n, hkv, g, d, nb, topk = 640, 2, 16, 32, 40, 3
    rows = torch.stack([torch.randperm(nb, generator=gen)[:topk] for _ in range(hkv * n // run)])
    rows = rows.view(hkv, n // run, topk).repeat_interleave(run, dim=1).to(torch.int32)
    cu = torch.arange(nb + 1, dtype=torch.int32) * (n // nb)
    cu_sb, cu_q = (torch.tensor([0, x], dtype=torch.int32) for x in (nb, n))
    rows, cu_sb, cu, cu_q = (t.contiguous().to(DEV) for t in (rows, cu_sb, cu, cu_q))
    plan = H.SelAttnPlan((n, hkv * g, d), (n, hkv, d), rows, cu_sb, cu, cu_q, backward=True,
                         key_centric=key_centric)
    plan.ws.zero_()  # and built again: the memory may hold an older plan's words
    p = H._ptr
    assert H.lib().lsrm_sel_attn_plan2(
        p(rows), n, n, hkv * g, hkv, d, topk, p(cu_sb), p(cu), nb, p(cu_q), 1, plan.flags,
        p(plan.ws), plan.ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
    words = plan.ws[:plan.ws.numel() // 4 * 4].view(torch.int32).cpu()
    at = (words == 0x4c42574b).nonzero().flatten().tolist()
    assert len(at) == 1
    grouped = run == 1  # without the key-centric part only grouped tiles are listed
    assert (int(words[at[0] + 2]) > 0) == (listed if key_centric else grouped)
