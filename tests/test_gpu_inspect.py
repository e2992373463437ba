"""The one-pass row checks of a selection (lsrm_sel_attn_inspect): metadata
bits and the count of rows that differ from the row before them, for both
kernel forms (rows of a power-of-two number of 16-byte pieces, and any other
row), against an evaluation on the CPU."""

import pytest
import torch

import lsrm_hip as H

pytestmark = pytest.mark.gpu

PREFIX, EMPTY = 16, 32


def _expected(rows, cu_q, cu_sb):
    bits = 0
    for e in range(len(cu_q) - 1):
        part = rows[:, cu_q[e]:cu_q[e + 1]]
        valid = (part >= 0) & (part < cu_sb[e + 1] - cu_sb[e])
        if part.shape[1] and not valid.any(-1).all():
            bits |= EMPTY
        if (valid[..., 1:] & ~valid[..., :-1]).any():
            bits |= PREFIX
    return bits, int((rows[:, 1:] != rows[:, :-1]).any(-1).sum())


# (25037 rows of 256 ids: more than one pass of the bounded grid)
@pytest.mark.parametrize("k,n", [(k, n) for k in (1, 3, 4, 8, 12, 16, 32, 64, 128, 256)
                                 for n in (1, 2, 65, 513, 1030)] + [(256, 25037)])
@pytest.mark.parametrize("bad", ["none", "prefix", "empty", "unaligned"])
def test_inspect_matches_row_by_row(k, n, bad):
    gen = torch.Generator().manual_seed(k * 10007 + n)
    hkv, nb = 2, 300
    split = n // 3  # two batch elements, the boundary inside a wave's rows
    cu_q, cu_sb = [0, split, n], [0, 270, nb]
    rows = torch.randint(0, 30, (hkv, n, k), generator=gen, dtype=torch.int32)
    rows[:, 1::2] = rows[:, 0:n - n % 2:2]  # runs of two equal rows
    if n > 2:  # runs across the batch boundary and one late difference
        rows[0, n - 1] = rows[0, n - 2]
        rows[1, n - 1] = rows[1, n - 2]
        rows[1, n - 1, k - 1] += 1
    if bad == "prefix" and k > 1:
        rows[1, n - 1, k - 2] = -1      # a valid entry after an invalid one
    if bad == "empty":
        rows[0, n // 2] = -1
        rows[1, n - 1, k // 2:] = 500   # out of range, as padding
    dev = torch.device("cuda:0")
    cu_blk = torch.arange(nb + 1, dtype=torch.int32, device=dev) * 4
    t = [torch.tensor(x, dtype=torch.int32, device=dev) for x in (cu_sb, cu_q)]
    cu_k = torch.tensor([0, 270 * 4, nb * 4], dtype=torch.int32, device=dev)
    if bad == "unaligned":  # rows that start 4 bytes past a 16-byte boundary
        pad = torch.empty(rows.numel() + 1, dtype=torch.int32, device=dev)
        dev_rows = pad[1:].view(rows.shape)
        dev_rows.copy_(rows)
    else:
        dev_rows = rows.to(dev)
    want = _expected(rows, cu_q, cu_sb)
    assert H.inspect_selection(dev_rows, t[0], cu_blk, t[1], cu_k, nb * 4) == want
    assert H.validate(dev_rows, t[0], cu_blk, t[1], cu_k, nb * 4) == want[0]
