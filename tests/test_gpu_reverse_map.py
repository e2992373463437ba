"""The reverse query map's stable counting passes (lsrm_reverse_query_map, and
the masked and slot-encoded maps of a plan) against its oracle, bit for bit, at
the edges of their parts: steps of 64 listings, chunks of one unit and of
several, one pass and two, windows of 4096 buckets, rows of whole 16-byte pieces
and others, rows that list a block twice, padding and ids out of range."""

import numpy as np
import pytest
import torch

import lsrm_hip as H
from oracle.revmap import reverse_query_map_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _chunk_lens(hkv, n, k, nb):
    # csrc/plan.hip (rev_one_pass, rev_chunks, build_query_reverse_map): queries
    # per chunk of the only pass, or of the first of two and pairs per chunk of
    # the second.
    one = nb <= 2048 or (nb <= 8192 and hkv * n * k >= 1 << 25)
    waves, counts = (1024, 4 << 20) if one else (4096, 2 << 20)

    def length(items, unit, buckets):
        c = max(1, min(-(-waves // hkv), counts // (hkv * buckets), -(-items // unit)))
        return max(unit, -(-(-(-items // c)) // unit) * unit)
    if one:
        return [length(n, 64, nb)]
    half = -(-(nb - 1).bit_length() // 2)
    return [length(n, 64, 1 << half), length(n * k, 1024, -(-nb // (1 << half)))]


def _check_map(topk, cu_q, cu_sb, nb):
    t = [torch.tensor(x, dtype=torch.int32) for x in (cu_q, cu_sb)]
    cu_rev, rev = H.reverse_query_map(topk.to(DEV), t[0].to(DEV), t[1].to(DEV), nb)
    ref_cu, ref_lists = reverse_query_map_ref(topk.numpy(), t[0].numpy(), t[1].numpy(), nb)
    assert np.array_equal(cu_rev.cpu().numpy(), ref_cu)
    got = rev.cpu().numpy()
    for h in range(topk.shape[0]):
        assert np.array_equal(got[h, :ref_cu[h, -1]], np.asarray(ref_lists[h], dtype=np.int32))


SIZES = [(n, k, nb, batch) for n, k, nb in (
    (1, 1, 1), (63, 4, 7), (64, 3, 40), (65, 16, 40), (130, 33, 300), (4097, 8, 1023),
    (1000, 12, 1024), (1000, 16, 1025), (700, 32, 8193), (20011, 4, 462), (3001, 64, 70),
    (2000, 65, 2049), (300, 256, 4096), (1, 2, 5000))
    for batch in (1, 3) if batch <= min(n, nb)]  # queries and blocks for every sequence


@pytest.mark.parametrize("n,k,nb,batch", SIZES)
@pytest.mark.parametrize("rows", ["distinct", "repeated", "one_block"])
def test_counting_sort(n, k, nb, batch, rows):
    gen = torch.Generator().manual_seed(n * 131 + k)
    hkv = 2
    assert _chunk_lens(hkv, n, k, nb)[0] == 64  # longer chunks: below
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
    _check_map(topk, cu_q, cu_sb, nb)


# Chunks of several units: many heads, or so many blocks that few chunks' counts fit.
@pytest.mark.parametrize("hkv,n,k,nb,lens", [
    (32, 20011, 4, 300, [640]), (48, 10007, 6, 1000, [512]), (32, 33001, 32, 8192, [2112]),
    (32, 20011, 16, 4097, [192, 3072]), (2, 20011, 16, 60000, [64, 1024])])
@pytest.mark.parametrize("twice", ["some_groups", "few_rows", "none"])
def test_longer_chunks(hkv, n, k, nb, lens, twice):
    gen = torch.Generator().manual_seed(n + k + nb)
    assert _chunk_lens(hkv, n, k, nb) == lens
    length = lens[0]
    cut = n // 3  # an element's edge inside a group
    cu_q, cu_sb = [0, cut, n], [0, nb // 3, nb]
    few = max(2 * k, nb // 2000)  # the blocks of a head's segments: many queries in each
    start = torch.randint(0, few, (hkv, n, 1), generator=gen)
    topk = ((start + torch.arange(k)) % few).to(torch.int32) * ((nb // 3 - 1) // few)
    group = torch.arange(n) // 64
    if twice == "some_groups":     # groups with repeated rows between others
        topk[:, group % 3 == 1, 1] = topk[:, group % 3 == 1, 0]
    elif twice == "few_rows":      # one row of a group, in every fourth chunk or so
        topk[:, 77::64 * 13, k - 1] = topk[:, 77::64 * 13, 0]
    topk[:, group % 7 == 3] = -1   # groups that list nothing
    topk[:, 5 * length:7 * length] = -1  # whole chunks that list nothing
    topk[:, ::11, k // 2:] = nb    # out of range, as padding
    _check_map(topk, cu_q, cu_sb, nb)


def test_two_windows_of_buckets():
    # more than 8192 buckets in a pass: the first of two, at 2^26 blocks and more
    nb, n, k = (1 << 26) + 5, 517, 3
    ids = torch.arange(n * k).view(1, n, k) * 43261 % nb
    ids[:, ::5, 2] = ids[:, ::5, 1]
    ids[:, 7::9, 0] = nb - 1
    ids[:, 3::9, 0] = 0
    _check_map(ids.to(torch.int32), [0, n], [0, nb], nb)


def _map_ms(nb, twice, hkv=2, n=131072, k=16):
    gen = torch.Generator(device=DEV).manual_seed(nb)
    start = torch.randint(0, nb, (hkv, n, 1), generator=gen, device=DEV)
    topk = ((start + torch.arange(k, device=DEV) * (nb // k - 1)) % nb).to(torch.int32)
    if twice:
        topk[..., 1] = topk[..., 0]
    cu_q, cu_sb = (torch.tensor([0, x], dtype=torch.int32, device=DEV) for x in (n, nb))
    times = []
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        H.reverse_query_map(topk, cu_q, cu_sb, nb)
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


def test_repeated_blocks_and_many_blocks_cost_little():
    # Rows that list a block twice take the same steps as others (once 1.3 ms
    # against 0.32 at 4881 blocks), and many blocks one more pass (once 0.71 ms
    # at 30000 blocks against 0.12 at 462).  The calls include the host's read
    # of the result's size and its copy.
    assert _map_ms(4881, True) <= 1.5 * _map_ms(4881, False)
    assert _map_ms(30000, False) <= 3 * _map_ms(462, False)


def _find_map(ws, cu_ref, lists):
    """Whether the plan's workspace holds the offsets `cu_ref` [hkv, nb + 1]
    (256-byte aligned) followed by the listings of every head, cap apart."""
    raw, pat = ws.tobytes(), cu_ref.tobytes()
    at = raw.find(pat)
    while at >= 0:
        if at % 256 == 0:
            rev = (at + len(pat) + 255) // 256 * 256
            cap = lists[1]
            if all(raw[rev + 4 * h * cap:rev + 4 * (h * cap + len(x))] == x.tobytes()
                   for h, x in enumerate(lists[0])):
                return True
        at = raw.find(pat, at + 4)
    return False


@pytest.mark.parametrize("hkv,nb,k,lens", [(32, 500, 4, [640]), (24, 3000, 8, [128, 1024]),
                                           (2, 60000, 6, [64, 1024]), (4, 700, 4, [128])])
@pytest.mark.parametrize("key_centric", [False, True])
def test_masked_and_encoded_maps_of_a_plan(hkv, nb, k, lens, key_centric):
    # One query head per kv head: windows of 96 queries are either one run of
    # equal rows (a run tile) or rows that all differ (a grouped tile, whose
    # queries alone the plan's query map lists; a key-centric plan's own map
    # lists them as q * k + slot, too).
    n = 96 * 210
    assert _chunk_lens(hkv, n, k, nb) == lens
    gen = torch.Generator().manual_seed(nb + k)
    window = torch.arange(n) // 96
    token = (window % 4 == 0) | (window % 11 == 5)
    token[96 * 40:96 * 55] = False
    start = torch.randint(0, nb // 2 - 1, (hkv, n), generator=gen)
    start = start // 2 * 2 + torch.arange(n) % 2       # neighbours differ
    start[:, ~token] = nb // 2 + (window[~token] * 7) % (nb // 4)
    topk = (start[:, :, None] + torch.arange(k) * 3) % nb
    twice = token & (torch.arange(n) % 192 == 9)
    topk[:, twice, 1] = topk[:, twice, 0]
    topk = topk.to(torch.int32).contiguous()
    cu_blk = torch.arange(nb + 1, dtype=torch.int32)
    cu_sb, cu_q = (torch.tensor([0, x], dtype=torch.int32) for x in (nb, n))
    plan = H.SelAttnPlan((n, hkv, 64), (nb, hkv, 64), topk.to(DEV), cu_sb.to(DEV), cu_blk.to(DEV),
                         cu_q.to(DEV), backward=True, key_centric=key_centric)
    marked = torch.where(token[None, :, None], topk, torch.tensor(-1, dtype=torch.int32))
    cu_ref, lists = reverse_query_map_ref(marked.numpy(), cu_q.numpy(), cu_sb.numpy(), nb)
    base = -plan.ws.data_ptr() % 256
    ws = plan.ws[base:].cpu().numpy()
    assert _find_map(ws, cu_ref, (lists, n * k))
    if key_centric:
        slots = []
        for h in range(hkv):
            x = marked[h].numpy().reshape(-1)
            at = np.nonzero(x >= 0)[0]
            slots.append(at[np.argsort(x[at], kind="stable")].astype(np.int32))
        assert _find_map(ws, cu_ref, (slots, n * k))
