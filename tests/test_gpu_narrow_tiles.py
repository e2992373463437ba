"""Run tiles of at most 32 rows at head dim 32, split over the keys between the
waves (forward and dQ): tile widths around 32 and 64 rows, key streams around
the 32-key blocks, one wave's turn and the token map's limit, empty streams,
repeated blocks, and scores that keep raising the running maximum, against the
fp32 oracle; run to run bitwise.  Results do not depend on a tile's width
beyond the order of the fp32 sums."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from helpers import assert_attn_close
from oracle.attention import sel_attn_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _grad_close(a, b, dtype, what):
    # A stream of a few keys gathers the gradients of all its rows, so sizes
    # vary: the suite's tolerance for values of size 1, and beyond it two
    # roundings (P or dS, then the result) of half a unit in the last place
    # each, relative to the value.
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    a, b = a.float().cpu(), b.detach()
    assert torch.isfinite(a).all(), what
    assert ((a - b).abs() <= 2e-2 + ulp * b.abs()).all(), \
        f"{what}: {float(((a - b).abs() - ulp * b.abs()).max()):.3e}"
    assert float((a - b).abs().mean()) <= 2e-3 + ulp * float(b.abs().mean())


@pytest.mark.parametrize("keys", [1, 31, 33, 128, 129, 257, 2047, 2100])
@pytest.mark.parametrize("g,dtype", [(1, torch.bfloat16), (4, torch.float16),
                                     (16, torch.bfloat16)])
@pytest.mark.parametrize("scores", ["plain", "rising"])
@pytest.mark.parametrize("key_centric", [False, True])
def test_narrow_tiles(keys, g, dtype, scores, key_centric):
    # (a key-centric plan lists the narrow tiles apart at every size; nothing
    # here is grouped, so nothing runs gathered)
    gen = torch.Generator().manual_seed(keys * 7 + g)
    d, hkv, topk = 32, 2, 3
    # widths in queries; neighbours of 8 or more queries share no block, so
    # they are not grouped
    lens = [w for w in (33, 64, 32, 9, 65, 31, 40, 8) if w * g <= 256] or [4, 2, 8, 3, 9, 1]
    lens = lens * 2
    # every third block holds the rest of the keys of a stream, the others few
    sizes = [max(1, keys - 2), 1, 1] * len(lens)
    n = sum(lens)
    nk = sum(sizes)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32)
    nb = len(sizes)
    rows = torch.stack([torch.arange(3) + 3 * i for i in range(len(lens))])
    if keys < 3:
        rows[:, 1:] = -1
    rows[1, 1:] = -1
    rows[1, 0] = -1                    # a tile that attends nothing
    rows[2, 1] = rows[2, 0]            # a block listed twice
    rows = rows.repeat_interleave(torch.tensor(lens), 0).expand(hkv, -1, -1).to(torch.int32)
    cu_sb = torch.tensor([0, nb], dtype=torch.int32)
    cu_q = torch.tensor([0, n], dtype=torch.int32)
    q = (0.5 * torch.randn(n, hkv * g, d, generator=gen)).to(dtype)
    do = (0.5 * torch.randn(n, hkv * g, d, generator=gen)).to(dtype)
    k, v = ((0.5 * torch.randn(nk, hkv, d, generator=gen)).to(dtype) for _ in range(2))
    if scores == "rising":  # the maximum moves by more than the rescaling step
        q = (q.abs() + 0.5).to(dtype)
        ramp = torch.linspace(-6, 6, nk)[:, None, None]
        k = (ramp + 0.1 * k.float()).to(dtype)
    scale = d ** -0.5
    rows = rows.contiguous()
    dev = [t.to(DEV) for t in (q, k, v, rows, cu_sb, cu, cu_q)]
    plan = H.SelAttnPlan(q.shape, k.shape, *dev[3:], backward=True, key_centric=key_centric)
    got = []
    for _ in range(2):
        o, lse = plan.fwd(*dev[:3], scale)
        got.append((o, lse) + plan.bwd(do.to(DEV), *dev[:3], o, lse, scale))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    o, lse, dq, dk, dv, delta = got[0]
    qf, kf, vf = (t.float().requires_grad_() for t in (q, k, v))
    ref, lse_ref = sel_attn_ref(qf, kf, vf, rows, cu_sb, cu, cu_q, scale)
    ref.backward(do.float())
    assert_attn_close(o, ref.detach(), "out")
    fin = torch.isfinite(lse_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), fin)
    # 16-bit inputs, fp32 products: a score of size s is off by under s * 2^-18
    err = (lse.cpu()[fin] - lse_ref.detach()[fin]).abs()
    assert float(err.max()) <= 2e-2
    delta_ref = (o.float().cpu() * do.float()).sum(-1).transpose(0, 1)
    torch.testing.assert_close(delta.cpu(), delta_ref, rtol=1e-4, atol=1e-4)
    _grad_close(dq, qf.grad, dtype, "dq")
    _grad_close(dk, kf.grad, dtype, "dk")
    _grad_close(dv, vf.grad, dtype, "dv")


def _passes(nq, g, dtype, sizes, listed, gen, key_centric=True):
    """Forward and dQ of nq queries that all list the same blocks, and of
    those queries among as many as fill a 128-row tile -> the two results for
    the nq queries.  Key-centric plans list narrow tiles apart whatever the
    stream's length."""
    d, hkv, full = 32, 2, 128 // g
    nk = sum(sizes)
    q, do = (torch.randn(full, hkv * g, d, generator=gen).to(dtype) for _ in range(2))
    k, v = (torch.randn(nk, hkv, d, generator=gen).to(dtype).to(DEV) for _ in range(2))
    cu = torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32, device=DEV)
    cu_sb = torch.tensor([0, len(sizes)], dtype=torch.int32, device=DEV)
    res = []
    for n in (nq, full):
        rows = torch.tensor(listed, dtype=torch.int32).expand(hkv, n, -1).contiguous().to(DEV)
        cu_q = torch.tensor([0, n], dtype=torch.int32, device=DEV)
        x = [t[:n].contiguous().to(DEV) for t in (q, do)]
        plan = H.SelAttnPlan(x[0].shape, k.shape, rows, cu_sb, cu, cu_q, backward=True,
                             key_centric=key_centric)
        o, lse = plan.fwd(x[0], k, v, d ** -0.5)
        dq = plan.bwd(x[1], x[0], k, v, o, lse, d ** -0.5)[0]
        res.append([o[:nq].cpu(), lse[:, :nq].cpu(), dq[:nq].cpu()])
    return res


@pytest.mark.parametrize("nq,g", [(3, 16), (4, 16), (33, 1), (64, 1), (10, 4)])
@pytest.mark.parametrize("blocks", [3, 40])
def test_wider_tiles_are_run_tiles(nq, g, blocks):
    # 33 to 64 rows: the kernel of a full tile, so the same bits
    gen = torch.Generator().manual_seed(nq)
    a, b = _passes(nq, g, torch.bfloat16, [61] * blocks, list(range(blocks)), gen)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("nq,g,blocks,size", [(2, 16, 40, 61), (32, 1, 40, 61), (8, 4, 33, 63)])
def test_narrow_tiles_over_long_streams_are_run_tiles(nq, g, blocks, size):
    # Streams beyond the token map, not key-centric: splitting the tiles costs
    # a little there, so they run as run tiles and give their bits.
    gen = torch.Generator().manual_seed(nq * blocks)
    a, b = _passes(nq, g, torch.bfloat16, [size] * blocks, list(range(blocks)), gen,
                   key_centric=False)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_wide_blocks_launch_no_narrow_kernel():
    # 4096 queries in blocks of 128 rows: no separate kernel for short tiles.
    n, hkv, d, blk = 4096, 2, 32, 128
    nb = n // blk
    rows = (torch.arange(nb)[:, None] + torch.arange(4)) % nb
    rows = rows.repeat_interleave(blk, 0).expand(hkv, -1, -1).to(torch.int32).contiguous().to(DEV)
    cu = (torch.arange(nb + 1, dtype=torch.int32) * blk).to(DEV)
    cu_sb, cu_q = (torch.tensor([0, x], dtype=torch.int32, device=DEV) for x in (nb, n))
    q, k, v = torch.randn(3, n, hkv, d, device=DEV).to(torch.bfloat16)
    plan = H.SelAttnPlan(q.shape, k.shape, rows, cu_sb, cu, cu_q, backward=True)
    o, lse = plan.fwd(q, k, v, d ** -0.5)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA],
                                acc_events=True) as prof:
        plan.fwd(q, k, v, d ** -0.5, o, lse)
        plan.bwd(q, q, k, v, o, lse, d ** -0.5)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("sel_attn_fwd_kernel" in x for x in names), names
    assert not any("narrow" in x for x in names), names


@pytest.mark.parametrize("nq,g", [(2, 16), (1, 16), (32, 1), (19, 1), (8, 4)])
@pytest.mark.parametrize("blocks,size", [(1, 3), (1, 50), (3, 61), (40, 61)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_narrow_tiles_round_as_run_tiles(nq, g, blocks, size, dtype):
    # One reference for P whatever the tile's width: the same 16-bit P, so the
    # results differ by the order of the fp32 sums alone.  That is less than
    # 2440 * 2^-24 < 2^-12 of the sums' terms at most and near 50 * 2^-24 as a
    # random walk, against a rounding step of 2^-8 (bf16) or 2^-11 (fp16) of
    # the result: far fewer than one result in fifty rounds the other way.
    gen = torch.Generator().manual_seed(nq + blocks)
    a, b = _passes(nq, g, dtype, [size] * blocks, list(range(blocks)), gen)
    torch.testing.assert_close(a[1], b[1], rtol=0, atol=1e-5)
    for x, y in ((a[0], b[0]), (a[2], b[2])):
        assert float((x != y).float().mean()) <= 0.02


def test_list_by_width_only_where_it_is_read():
    # One run tile per query: a plan for head dim 64 leaves the list by width
    # unwritten, one for head dim 32 writes it; run at head dim 32, both give
    # the same rows up to the order of the fp32 sums.
    gen = torch.Generator().manual_seed(5)
    n, hkv, g, d, nb, topk, flags = 2048, 2, 32, 32, 1500, 8, H.PLAN_BACKWARD
    rows = (torch.arange(n)[:, None] + torch.arange(topk) * 7) % nb
    rows = rows.expand(hkv, -1, -1).to(torch.int32).contiguous().to(DEV)
    cu = (torch.arange(nb + 1, dtype=torch.int32) * 33).to(DEV)
    cu_sb, cu_q = (torch.tensor([0, x], dtype=torch.int32, device=DEV) for x in (nb, n))
    q, do = (torch.randn(n, hkv * g, d, generator=gen).to(torch.bfloat16).to(DEV)
             for _ in range(2))
    k, v = (torch.randn(nb * 33, hkv, d, generator=gen).to(torch.bfloat16).to(DEV)
            for _ in range(2))
    untouched, results = {}, {}
    for plan_d in (32, 64):
        plan = H.SelAttnPlan(q.shape, k.shape, rows, cu_sb, cu, cu_q, backward=True)
        plan.ws.fill_(0x5a)
        p = H._ptr
        assert H.lib().lsrm_sel_attn_plan2(
            p(rows), n, k.shape[0], hkv * g, hkv, plan_d, topk, p(cu_sb), p(cu), nb, p(cu_q), 1,
            flags, p(plan.ws), plan.ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
        untouched[plan_d] = int((plan.ws == 0x5a).sum())
        o, lse = plan.fwd(q, k, v, d ** -0.5)
        results[plan_d] = (o, lse) + plan.bwd(do, q, k, v, o, lse, d ** -0.5)
    assert untouched[64] - untouched[32] >= 7 * hkv * n  # (some bytes are the filler)
    # 16-bit rounding steps of the few values that round otherwise; an output
    # that does moves its row's delta by up to 2^-8 |o| |do|, two of a row by
    # twice that
    step = 2.0 ** -7 * float(results[32][0].abs().max()) * float(do.abs().max())
    for i, (a, b) in enumerate(zip(*results.values())):
        torch.testing.assert_close(a, b, rtol=2.0 ** -7, atol=step if i == 5 else 2e-3)
