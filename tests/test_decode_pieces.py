"""The arithmetic by which a decode step's keys are cut into pieces (csrc/grouped_attn.hip,
find_range, for pieces of about two rounds of workgroups): at most pieces + sequences."""
import numpy as np
import pytest


def quotient(n, d):
    """As the kernel divides, with a reciprocal that may be off by one unit in either direction."""
    n, d = np.asarray(n, np.int64), np.asarray(d, np.int64)
    for step in (-1, 0, 1):
        by = (np.float32(1) / d.astype(np.float32)).view(np.int32) + np.int32(step)
        by = by.view(np.float32)
        q = (n.astype(np.float32) * by).astype(np.int64)
        more = ((n - q * d).astype(np.float32) * by).astype(np.int64)
        q = q + more
        rest = n - q * d
        assert (np.abs(q * d) < 1 << 31).all()  # no overflow on the way
        yield q + (rest >= d) - (rest < 0)


def test_quotient_is_exact():
    gen = np.random.default_rng(1)
    d = np.concatenate([np.arange(1, 3000), gen.integers(1, 1 << 29, 20000),
                        gen.integers(1, 1 << 12, 20000)])
    top = (1 << 30) - 1
    for shift in (0, 3, 8, 15, 22):
        n = gen.integers(0, top + 1, d.shape) >> shift
        near = n // d * d  # multiples and one less
        for x in (n, near, np.maximum(near - 1, 0), np.full_like(d, top)):
            for q in quotient(x, d):
                assert (q == x // d).all()


def cut(blocks, pieces):
    """[(pieces, blocks of one)] of the sequences."""
    half = max(1, (sum(blocks) + 2 * pieces - 1) // (2 * pieces))
    size = 4 * (max(min(half, 3), (half + 1) // 2) if max(blocks) > 4 * half else half)
    out = []
    for n in blocks:
        k, each = max(1, (n + size - (0 if size < 12 else size // 4) - 1) // size), size
        if k * size < n:
            each = 4 * -(-n // (4 * k))
            k = -(-n // each)
        out.append((k, each))
    return out


@pytest.mark.parametrize("pieces", [1, 7, 25, 128, 1024])
def test_pieces_fit_their_workspace(pieces):
    gen = np.random.default_rng(pieces)
    for _ in range(400):
        top = int(np.exp(gen.uniform(0, np.log(40000))))
        blocks = gen.integers(0, top + 1, int(np.exp(gen.uniform(0, np.log(1000))))).tolist()
        parts = cut(blocks, pieces)
        assert sum(k for k, _ in parts) <= pieces + len(blocks)
        for n, (k, each) in zip(blocks, parts):
            assert k * each >= n and (k == 1 or (k - 1) * each < n)
