"""Block means of launches of few waves (pool_pieces_small): row widths of
whole and broken 256-byte pieces in every type, sizes on both sides of the
rule's line, blocks of a few rows, empty blocks in great number, rows outside
every block and chunk edges, bit for bit against the oracle; two tensors in one
call as two calls."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from oracle.pool import block_mean_pool_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _offsets(n, kind, gen):
    if kind == "even":
        return list(range(0, n, 37)) + [n]
    if kind == "few":  # blocks of 0 to 9 rows
        cuts = torch.randint(0, 10, (n,), generator=gen).cumsum(0).tolist()
        return [0] + [c for c in cuts if c < n] + [n]
    if kind == "empties":  # up to 200 empty blocks in a row, some at a chunk's edge
        cuts = torch.randint(0, n + 1, (40,), generator=gen).tolist() + [0, n, 64, 128][:4]
        cuts = [min(c, n) for c in cuts for _ in range(1 + 50 * (c % 5 == 0))]
        return sorted(cuts)
    return sorted(min(n, c) for c in (n // 5, n // 5 + 3, n // 2, n // 2, max(0, n - 70)))


@pytest.mark.parametrize("dtype,c", [(torch.bfloat16, 256), (torch.float16, 1536),
                                     (torch.float32, 64), (torch.float32, 192),
                                     (torch.bfloat16, 192)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1029, 4099])
@pytest.mark.parametrize("kind", ["even", "few", "empties", "uncovered"])
def test_small_pool(dtype, c, n, kind):
    gen = torch.Generator().manual_seed(n + c)
    x, y = (torch.randn(n, c, generator=gen).to(dtype) for _ in range(2))
    cu = torch.tensor(_offsets(n, kind, gen), dtype=torch.int32)
    ref = [block_mean_pool_ref(t.float().numpy(), cu.numpy()) for t in (x, y)]
    got = H.block_mean_pool(x.to(DEV), cu.to(DEV), torch.float32).cpu().numpy()
    np.testing.assert_array_equal(got, ref[0])
    a, b = H.block_mean_pool2(x.to(DEV), y.to(DEV), cu.to(DEV), torch.float32, torch.float32)
    np.testing.assert_array_equal(a.cpu().numpy(), ref[0])
    np.testing.assert_array_equal(b.cpu().numpy(), ref[1])


@pytest.mark.parametrize("n", [65536, 65537])  # 2048 waves, and one chunk more
def test_both_sides_of_the_line(n):
    gen = torch.Generator().manual_seed(n)
    x = torch.randn(n, 256, generator=gen).to(torch.bfloat16)
    cu = torch.tensor(list(range(0, n, 91)) + [n], dtype=torch.int32)
    got = H.block_mean_pool(x.to(DEV), cu.to(DEV), torch.float32).cpu().numpy()
    np.testing.assert_array_equal(got, block_mean_pool_ref(x.float().numpy(), cu.numpy()))


def test_short_blocks_cost_little():
    # Blocks of one row, once 84 us against 31 now (8.7 in blocks of 64 rows).
    # The calls take about 17 us of the host, so the ratio lies between 1.8 and
    # 3.6 (once 5.8 to 10).
    x = torch.randn(4096, 256, device=DEV).to(torch.bfloat16)
    times = []
    for rows in (1, 64):
        cu = torch.arange(0, 4097, rows, dtype=torch.int32, device=DEV)
        best = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(30):
                H.block_mean_pool(x, cu)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        times.append(min(best))
    assert times[0] <= 4.5 * times[1]
