"""How a decode step's blocks of 32 keys are shared by its workgroups (csrc/grouped_attn.hip, find_range): the
arithmetic, and the kernel at its edges against fp32."""
import math

import numpy as np
import pytest
import torch

from agentcontrolplane_amd import ops


def two_rounds(blocks, pieces, shared_from=12):
    """[(pieces, blocks of one)] of the sequences where all are for about two rounds of workgroups: at most
    ``pieces`` and one for every sequence."""
    half = max(1, (sum(blocks) + 2 * pieces - 1) // (2 * pieces))
    size = 4 * (max(min(half, 3), (half + 1) // 2) if max(blocks) > 4 * half else half)
    out = []
    for n in blocks:
        k, each = max(1, (n + size - (0 if size < shared_from else size // 4) - 1) // size), size
        if k * size < n:
            each = 4 * -(-n // (4 * k))
            k = -(-n // each)
        out.append((k, each))
    return out


@pytest.mark.parametrize("shared_from", [12, 16])
@pytest.mark.parametrize("pieces", [1, 7, 25, 128, 1024])
def test_pieces_fit_their_workspace(pieces, shared_from):
    gen = np.random.default_rng(pieces)
    for _ in range(400):
        top = int(np.exp(gen.uniform(0, np.log(40000))))
        blocks = gen.integers(0, top + 1, int(np.exp(gen.uniform(0, np.log(1000))))).tolist()
        parts = two_rounds(blocks, pieces, shared_from)
        assert sum(k for k, _ in parts) <= pieces + len(blocks)
        for n, (k, each) in zip(blocks, parts):
            assert k * each >= n and (k == 1 or (k - 1) * each < n)


def cut(blocks, P, paired, ranges, shared_from):
    """(aligned, ranges of a workgroup, blocks of one or of each sequence's pieces) as the kernel finds them."""
    total, seqs = sum(blocks), len(blocks)
    share, spare = -(-total // P), P - seqs
    if not ranges or (share <= 32 and spare >= 0):
        even, most = (share + 3) // 4 * 4, share + share // 4 + 4
        if seqs <= 64 and sum(-(-n // even) for n in blocks) <= P:
            return True, 1, [even] * seqs
        if spare >= 0 and max(blocks) <= most:
            return True, 1, [most] * seqs
        if not ranges:
            return True, 1, [each for _, each in two_rounds(blocks, 2 * P, shared_from)]
        each = -(-total // spare) if spare else most + 1
        return (True, 1, [max(4, each)] * seqs) if each <= most else (False, 1, max(4, share))
    return (False, 2, (share + 1) // 2) if share > 32 and paired else (False, 1, max(4, share))


def parts(lens, P, paired, ranges, shared_from):
    """{(workgroup, one of two heads): [(head, range, sequence, from, to, goes on)]} of sequences of so many
    blocks, as the workgroups go on; a sequence without a block has a turn of one"""
    turns = [max(1, n) for n in lens]
    aligned, count, each = cut(turns, P, paired, ranges, shared_from)
    before = np.concatenate([[0], np.cumsum([-(-n // e) for n, e in zip(turns, each)] if aligned else turns)])
    out = {}
    items = P if ranges else 2 * P + len(lens)
    assert not aligned or before[-1] <= items
    for item in range(items):
        first = item if aligned else item * count * each
        if first >= before[-1]:
            continue
        for at in (0, 1):
            seq = int(np.searchsorted(before, first, "right")) - 1
            left = size = each[seq] if aligned else each
            head, r, on, start = at, item * count, False, (first - int(before[seq])) * (size if aligned else 1)
            mine = out[item, at] = []
            while True:
                to = min(lens[seq], start + left)
                mine.append((head, r, seq, start, to, on))
                left -= max(1, to - start)
                if aligned:
                    break
                on = left > 0
                if not on:  # the next range, of the other head
                    r, head, left = r + 1, head ^ 1, size
                    if count == 1 or r % 2 == 0:
                        break
                stays = not on and to < lens[seq]
                seq, start = (seq, to) if stays else (seq + 1, 0)
                if seq == len(lens):
                    break
    return out, (aligned, each, before)


@pytest.mark.parametrize("ranges,shared_from", [(False, 16), (False, 12), (True, None)])
@pytest.mark.parametrize("P,paired", [(64, True), (16, True), (7, False), (1, True), (256, True)])
def test_every_block_has_one_workgroup(P, paired, ranges, shared_from):
    """Of either head, whose partial results have places of their own in the workspace, which are those that
    the merge reads.  Sequences of no block are written once for either head."""
    gen = np.random.default_rng(P)
    for _ in range(120):
        top = int(np.exp(gen.uniform(0, np.log(3000))))
        lens = gen.integers(0, top + 1, int(np.exp(gen.uniform(0, np.log(400))))).tolist()
        shares, (aligned, each, before) = parts(lens, P, paired, ranges, shared_from)
        seen, slots = {}, {}
        for mine in shares.values():
            # a second range is of the other head
            assert len({head for head, *_ in mine}) == len({r for _, r, *_ in mine})
            for head, r, s, start, to, on in mine:
                assert 0 <= start <= to <= lens[s] and (start < to or lens[s] == 0)
                seen.setdefault((head, s), []).append((start, to))
                if (start, to) != (0, lens[s]):
                    slot = 2 * r + (to < lens[s] and on)
                    assert (head, slot) not in slots and slot < 2 * (2 * P + len(lens))
                    slots[head, slot] = s
        for head in (0, 1):
            places = {}
            for (h, slot), s in slots.items():
                if h == head:
                    places.setdefault(s, set()).add(slot)
            for s, n in enumerate(lens):
                own = sorted(seen[head, s])
                assert [a for a, _ in own] == [0] + [b for _, b in own[:-1]] and own[-1][1] == n
                turn = max(1, n)
                if aligned:
                    first, k, ahead = int(before[s]), -(-turn // each[s]), 0
                else:
                    first = int(before[s]) // each
                    k = (int(before[s]) + turn - 1) // each - first + 1
                    ahead = first * each < before[s]
                # one part is written by its workgroup, several are what the merge reads
                assert (k > 1) == (s in places)
                if k > 1:
                    assert places[s] == {2 * (first + i) + (i == 0 and ahead) for i in range(k)}


LENS = {
    "long": [1, 0, 33, 32, 31] + [4100] + [64] * 60,     # one long sequence among short ones
    "even": [2048] * 65,                                 # ranges that end where sequences do
    "ragged": [37 + 211 * i % 1900 for i in range(70)],  # in the middle of them
    "many": [5] * 200 + [9000],
}


def check_decode(H, G, d, lens, block=16, window=None, keep=0, cap=0.0, form=""):
    """A step whose keys are cut, however many sequences, against fp32.  form: what else a layer has."""
    gen = torch.Generator("cuda").manual_seed(len(lens) + H)
    n_blocks = [-(-max(n, 1) // block) for n in lens]
    table = torch.zeros(len(lens), max(n_blocks), dtype=torch.int32, device="cuda")
    order = torch.randperm(sum(n_blocks), generator=gen, device="cuda").int()
    for row, pages in zip(table, order.split(n_blocks)):
        row[: len(pages)] = pages
    k, v = (torch.randn(len(order), block, G, d, generator=gen, device="cuda").bfloat16()
            for _ in range(2))
    q = torch.randn(len(lens), H, d, generator=gen, device="cuda").bfloat16()
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    sink = rand(H) if "sink" in form else None
    bias = rand(H, 100) if "bias" in form else None
    gate = rand(len(lens), H).bfloat16() if "gate" in form else None
    sigmoid = "sigmoid" in form
    out = torch.full_like(q, 7.0)
    hip = ops._hip()
    seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    whole = hip._WHOLE_GROUPS
    try:
        hip._WHOLE_GROUPS = 1 << 30
        hip._grouped_decode(out, q, k, v, table, seq_lens, sink, bias, gate, d ** -0.5, cap, window or 1 << 30,
                            1 << 30, keep, sigmoid)
    finally:
        hip._WHOLE_GROUPS = whole
    for b, n in enumerate(lens):
        if n == 0:
            assert (out[b] == 0).all()
            continue
        pages = table[b, : n_blocks[b]].long()
        keys, values = (c[pages].view(-1, G, d)[:n].float().repeat_interleave(H // G, 1) for c in (k, v))
        s = torch.einsum("nhd,hd->nh", keys, q[b].float()) * d ** -0.5
        if cap:
            s = cap * torch.tanh(s / cap)
        p = torch.arange(n, device="cuda")[:, None]
        if bias is not None:
            s = s + bias[:, (n - 1 - p[:, 0]).clamp(max=99)].T
        if window:
            s = s.masked_fill((p <= n - 1 - window) & (p >= keep), -math.inf)
        if sigmoid:
            w = torch.sigmoid(s)
        elif sink is not None:
            w = torch.softmax(torch.cat([s, sink[None]]), 0)[:-1]
        else:
            w = torch.softmax(s, 0)
        g = 1.0 if gate is None else torch.sigmoid(gate[b].float())[:, None]
        want = g * (w.unsqueeze(-1) * values).sum(0)
        # fp32 but for the result, and sums of up to 9000 terms in it
        slack = 2.0 ** -8 * want.abs() + 2.0 ** -20 * g * (w.unsqueeze(-1) * values.abs()).sum(0) + 1e-4
        assert ((out[b].float() - want).abs() <= slack).all(), (b, n)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G", [(8, 8), (16, 8), (32, 8)])
@pytest.mark.parametrize("lens", ["long", "ragged"])
@pytest.mark.parametrize("form,block,cap,window", [
    ("sink", 32, 5.0, None), ("sink gate", 6, 0.0, 500), ("sigmoid bias", 16, 0.0, None), ("bias", 8, 5.0, None),
    ("sigmoid", 64, 5.0, 300),
])
def test_decode_by_ranges_of_other_forms(H, G, lens, form, block, cap, window):
    """What only a sequence's first part or a whole sequence has, pages of other sizes."""
    check_decode(H, G, 128, LENS[lens], block, window, 0, cap, form)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d,lens", [
    (64, 8, 128, "long"), (64, 8, 128, "even"), (64, 8, 128, "ragged"), (64, 8, 128, "many"),
    (40, 4, 128, "ragged"), (16, 1, 128, "long"), (32, 8, 128, [130 + 199 * i for i in range(19)]),
    (8, 8, 128, [8000, 1, 0, 300]), (4, 2, 128, [900] * 70), (2, 1, 128, [40] * 90 + [5000]),
    (64, 8, 256, [510 + 82 * i for i in range(24)]), (16, 2, 256, "long"), (64, 8, 256, "many"),
], ids=str)
@pytest.mark.parametrize("form", ["", "sink", "sigmoid"])
def test_decode_by_pieces(H, G, d, lens, form):
    """Without ranges: many query heads a key head, and few sequences."""
    check_decode(H, G, d, LENS[lens] if isinstance(lens, str) else lens, form=form)
