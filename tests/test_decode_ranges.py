"""How a decode step's blocks of 32 keys are shared by its workgroups (csrc/grouped_attn.hip, find_range): the
arithmetic, and the kernel at its edges against fp32."""
import math

import numpy as np
import pytest
import torch

from agentcontrolplane_amd import ops


def cut(blocks, P, paired, ranges):
    """(aligned, ranges of a workgroup, blocks of one) as the kernel finds them."""
    total, seqs = sum(blocks), len(blocks)
    share, spare = -(-total // P), P - seqs
    if not ranges or (share <= 32 and spare >= 0):
        even, most = (share + 3) // 4 * 4, share + share // 4 + 4
        if seqs <= 64 and sum(-(-n // even) for n in blocks) <= P:
            return True, 1, even
        if spare >= 0 and max(blocks) <= most:
            return True, 1, most
        if not ranges:
            return True, 1, max(4, (share + 7) // 8 * 4)
        each = -(-total // spare) if spare else most + 1
        return (True, 1, max(4, each)) if each <= most else (False, 1, max(4, share))
    return (False, 2, (share + 1) // 2) if share > 32 and paired else (False, 1, max(4, share))


def parts(blocks, P, paired, ranges):
    """{workgroup of a key head: [(other head's, range, sequence, from, to, goes on)]}"""
    aligned, count, each = cut(blocks, P, paired, ranges)
    before = np.concatenate([[0], np.cumsum([-(-n // each) if aligned else n for n in blocks])])
    out = {}
    for item in range(P if ranges else 2 * P + len(blocks)):
        first = item if aligned else item * count * each
        if first >= before[-1]:
            continue
        seq = int(np.searchsorted(before, first, "right")) - 1
        at, mine = (first - int(before[seq])) * (each if aligned else 1), []
        if aligned:
            mine.append((0, item, seq, at, min(blocks[seq], at + each), False))
        for j in range(0 if aligned else count):
            left, goes_on = each, False
            while left > 0 and seq < len(blocks):
                to = min(blocks[seq], at + left)
                mine.append((j, item * count + j, seq, at, to, goes_on))
                left -= to - at
                seq, at = (seq, to) if to < blocks[seq] else (seq + 1, 0)
                goes_on = True
        out[item] = mine
    return out, (aligned, each, before)


@pytest.mark.parametrize("ranges", [False, True])
@pytest.mark.parametrize("P,paired", [(64, True), (16, True), (7, False), (1, True), (256, True)])
def test_every_block_has_one_workgroup(P, paired, ranges):
    """Of either head, whose partial results have places of their own in the workspace, which are those that
    the merge reads."""
    gen = np.random.default_rng(P)
    for _ in range(150):
        top = int(np.exp(gen.uniform(0, np.log(3000))))
        blocks = gen.integers(1, top + 1, int(np.exp(gen.uniform(0, np.log(400))))).tolist()
        shares, (aligned, each, before) = parts(blocks, P, paired, ranges)
        for head in (0, 1):
            seen, slots = {s: [] for s in range(len(blocks))}, {}
            for mine in shares.values():
                for j, r, s, at, to, goes_on in mine:
                    # the two workgroups of a pair of heads change heads for their second range
                    if cut(blocks, P, paired, ranges)[1] == 2 or head == 0:
                        assert 0 <= at < to <= blocks[s]
                        seen[s].append((at, to))
                        if (at, to) != (0, blocks[s]):
                            slot = 2 * r + (to < blocks[s] and goes_on)
                            assert slot not in slots and slot < 2 * (2 * P + len(blocks))
                            slots[slot] = s
            if head and not slots and not any(seen.values()):
                continue
            for s, n in enumerate(blocks):
                assert [a for a, _ in seen[s]] == [0] + [b for _, b in seen[s][:-1]]
                assert seen[s][-1][1] == n
                if aligned:
                    first, k, ahead = int(before[s]), -(-n // each), 0
                else:
                    first = int(before[s]) // each
                    k = (int(before[s]) + n - 1) // each - first + 1
                    ahead = first * each < before[s]
                if k > 1:
                    assert {2 * (first + i) + (i == 0 and ahead) for i in range(k)} == {
                        t for t, q in slots.items() if q == s}


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d", [(8, 8, 128), (32, 8, 128), (6, 3, 128), (4, 2, 256)])
@pytest.mark.parametrize("lens", [
    [1, 0, 33, 32, 31] + [4100] + [64] * 60,            # one long sequence among short ones
    [2048] * 65,                                        # ranges that end where sequences do
    [37 + 211 * i % 1900 for i in range(70)],           # in the middle of them
    [5] * 200 + [9000],
], ids=["long", "even", "ragged", "many"])
@pytest.mark.parametrize("form", ["plain", "window"])
def test_decode_by_ranges(H, G, d, lens, form):
    gen = torch.Generator("cuda").manual_seed(len(lens) + H)
    block, window = 16, (500, 40) if form == "window" else (None, 0)
    n_blocks = [-(-max(n, 1) // block) for n in lens]
    table = torch.zeros(len(lens), max(n_blocks), dtype=torch.int32, device="cuda")
    order = torch.randperm(sum(n_blocks), generator=gen, device="cuda").int()
    for row, pages in zip(table, order.split(n_blocks)):
        row[: len(pages)] = pages
    k, v = (torch.randn(len(order), block, G, d, generator=gen, device="cuda").bfloat16()
            for _ in range(2))
    q = torch.randn(len(lens), H, d, generator=gen, device="cuda").bfloat16()
    out = torch.full_like(q, 7.0)
    hip, rest = ops._hip(), (1 << 30, False)
    seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    keep = hip._WHOLE_GROUPS
    try:
        hip._WHOLE_GROUPS = 1 << 30  # cut, however many sequences
        hip._grouped_decode(out, q, k, v, table, seq_lens, None, None, None, d ** -0.5, 0.0,
                            window[0] or 1 << 30, rest[0], window[1], rest[1])
    finally:
        hip._WHOLE_GROUPS = keep
    for b, n in enumerate(lens):
        if n == 0:
            assert (out[b] == 0).all()
            continue
        pages = table[b, : n_blocks[b]].long()
        keys, values = (c[pages].view(-1, G, d)[:n].float().repeat_interleave(H // G, 1) for c in (k, v))
        s = torch.einsum("nhd,hd->nh", keys, q[b].float()) * d ** -0.5
        if window[0]:
            p = torch.arange(n, device="cuda")[:, None]
            s = s.masked_fill((p <= n - 1 - window[0]) & (p >= window[1]), -math.inf)
        w = torch.softmax(s, 0)
        want = (w.unsqueeze(-1) * values).sum(0)
        # fp32 but for the result, and sums of up to 9000 terms in it
        slack = 2.0 ** -8 * want.abs() + 2.0 ** -20 * (w.unsqueeze(-1) * values.abs()).sum(0) + 1e-4
        assert ((out[b].float() - want).abs() <= slack).all(), (b, n)
