"""CPU: where fla_scan_split cuts sequences.  Host arithmetic, whose tables the kernels index memory with."""
import ctypes
import random

import pytest

CHUNK, CUS = 64, 256


def _plan(bounds, N, T, H, slabs, reverse, kind):
    """The plan and, for a packed batch, its tables (from buffers with guard words behind them)."""
    from fla_amd import _backend as be
    fn, sp = be.lib().fla_scan_split, be.Split()
    offs = None if bounds is None else (ctypes.c_int64 * len(bounds))(*bounds)
    if not fn(offs, N, T, H, slabs, reverse, kind, ctypes.byref(sp), None, None, None):
        return None
    if bounds is None:
        return sp, None, None, None
    sizes = [2 * sp.nseg, 2 * sp.nsub, N + 1]
    tables = [(ctypes.c_int32 * (n + 8))(*([-7] * (n + 8))) for n in sizes]
    again = be.Split()
    assert fn(offs, N, T, H, slabs, reverse, kind, ctypes.byref(again), *tables)
    for name in ("sub_chunks", "ratio", "nseg", "nsub", "slots"):
        assert getattr(sp, name) == getattr(again, name)
    assert all(list(t[n:]) == [-7] * 8 for t, n in zip(tables, sizes))
    seg, sub, base = (list(t[:n]) for t, n in zip(tables, sizes))
    return sp, list(zip(seg[::2], seg[1::2])), list(zip(sub[::2], sub[1::2])), base


def _check(sp, seg, sub, base, chunks, H, slabs, reverse, kind):
    """``chunks``: chunks of every sequence; ``seg`` and the others None for sequences of equal length."""
    kind &= 7   # (8: the delta rule with 64 key channels)
    assert sp.sub_chunks > 0 and sp.ratio > 0 and (kind in (0, 3) or sp.ratio == 1)
    subs = [max(1, -(-c // sp.sub_chunks)) for c in chunks]
    segs = [-(-s // sp.ratio) for s in subs]
    assert max(segs) > 1                                 # something is cut,
    assert sum(segs) * H * slabs <= CUS                  # every workgroup of the scan has a CU of its own,
    assert sp.slots == sum(subs)                         # and every sub-block a slot
    # the sub-blocks the first pass forms: all whose end another segment begins at (and those whose transition a backward wants)
    def formed(n):
        return range(sp.ratio, subs[n]) if reverse else range(subs[n] if kind == 2 else (segs[n] - 1) * sp.ratio)
    if seg is None:
        assert len(set(chunks)) == 1 and sp.nseg == segs[0] and sp.nsub == subs[0]
        return
    assert sorted(seg) == [(n, s) for n in range(len(chunks)) for s in range(segs[n])] and sp.nseg == len(seg)
    assert sorted(sub) == [(n, j) for n in range(len(chunks)) for j in formed(n)] and sp.nsub == len(sub)
    assert base == [sum(subs[:n]) for n in range(len(chunks) + 1)]
    last = [i for i, (n, s) in enumerate(seg) if s == segs[n] - 1]
    assert last == list(range(len(seg) - len(last), len(seg)))     # the shorter last pieces start last


@pytest.mark.parametrize("kind", [0, 1, 2, 3, 9, 10])
def test_packed_batches(kind):
    rng, cut = random.Random(kind), 0
    for _ in range(3000):
        N = rng.randint(1, 40)
        longest = int(2 ** rng.uniform(4, 18))
        bounds = [0]
        for _ in range(N):
            bounds.append(bounds[-1] + (0 if rng.random() < 0.1 else rng.randint(1, longest)))
        H, slabs, reverse = rng.choice((1, 2, 3, 4, 8, 16, 32)), rng.choice((1, 2, 4)), rng.randint(0, 1)
        got = _plan(bounds, N, bounds[-1], H, slabs, reverse, kind)
        if got:
            cut += 1
            _check(*got, [-(-(b - a) // CHUNK) for a, b in zip(bounds, bounds[1:])], H, slabs, reverse, kind)
    assert cut > 300


@pytest.mark.parametrize("kind", [0, 1, 2, 3, 9, 10])
def test_sequences_of_equal_length(kind):
    cut = 0
    for N in (1, 2, 3, 5, 8, 16, 33, 128):
        for T in (1, 64, 704, 833, 1600, 4096, 5003, 8192, 100001, 262144):
            for H in (1, 2, 3, 4, 16, 64, 128):
                for slabs in (1, 2, 4):
                    for reverse in (0, 1):
                        got = _plan(None, N, T, H, slabs, reverse, kind)
                        if got:
                            cut += 1
                            _check(*got, [-(-T // CHUNK)] * N, H, slabs, reverse, kind)
    assert cut > 100


def test_forward_and_backward_of_the_delta_rule_are_cut_alike():
    """The backward folds with the transitions the forward left, slot by slot."""
    rng = random.Random(5)
    for trial in range(600):
        kind = (2, 10)[trial % 2]
        bounds = [0]
        for _ in range(rng.randint(1, 12)):
            bounds.append(bounds[-1] + rng.randint(0, 20000))
        N, H, slabs = len(bounds) - 1, rng.choice((1, 2, 4, 8)), rng.choice((1, 2))
        f, r = (_plan(bounds, N, bounds[-1], H, slabs, reverse, kind) for reverse in (0, 1))
        assert (f is None) == (r is None)
        if f:
            assert (f[0].sub_chunks, f[0].slots, f[3]) == (r[0].sub_chunks, r[0].slots, r[3]) and f[1] == r[1]


def test_nothing_to_cut():
    assert _plan([0, 0, 0], 2, 0, 1, 1, 0, 0) is None
    assert _plan(None, 1, 0, 1, 1, 0, 0) is None
    assert _plan(None, 0, 64, 1, 1, 0, 0) is None
    assert _plan(None, 1, 64 * 200, 512, 2, 0, 0) is None
    for kind in (-1, 5, 8, 11, 12, 13, 16):   # no such kinds: the key channels go with the delta rule's
        assert _plan(None, 1, 64 * 200, 2, 2, 0, kind) is None


@pytest.mark.parametrize("kind,heads,chunks,cut", [
    # kind 0, GLA, 1, the delta rule's forward, 2, one that keeps its intermediates, 3, the plain scan of chunk_simple_gla; K = V =
    # 128, so two slabs a head
    (0, 16, 12, True), (0, 32, 12, True), (0, 64, 16, False), (0, 64, 20, False), (0, 64, 24, True),
    (1, 4, 24, False), (1, 4, 32, True), (1, 8, 24, False), (1, 8, 28, False), (1, 8, 33, True), (1, 12, 36, False), (1, 12, 40, True),
    (1, 16, 24, False), (1, 16, 32, False), (1, 16, 37, False), (1, 16, 42, True), (1, 24, 44, False), (1, 24, 52, True),
    (1, 32, 40, False), (1, 32, 56, False), (1, 32, 68, True), (1, 48, 128, False), (2, 4, 23, False), (2, 4, 32, True),
    (2, 8, 20, False), (2, 8, 28, True), (2, 12, 36, False), (2, 16, 32, False), (2, 16, 40, False), (2, 16, 44, False),
    (2, 16, 56, True), (2, 24, 72, False), (2, 24, 80, True), (2, 32, 96, False), (2, 32, 128, True),
    (3, 4, 12, False), (3, 4, 16, True), (3, 12, 16, False), (3, 12, 20, True), (3, 16, 16, False), (3, 16, 20, False),
    (3, 16, 24, True), (3, 32, 24, False), (3, 32, 36, False), (3, 32, 40, True), (3, 48, 64, False), (3, 64, 64, False)])
def test_cut_where_it_pays(kind, heads, chunks, cut):
    """The cuts that were measured to lose (delta-rule forward of 16 heads, 32 chunks: 48 us uncut, 52 cut; plain scan of 32
    heads, 24 chunks: 31 uncut, 35 cut) are not made, also not in a packed batch whose other sequences are short."""
    for reverse in (0, 1):
        for bounds in (None, [0, chunks * CHUNK], [0, chunks * CHUNK, chunks * CHUNK + 3]):
            N = 1 if bounds is None else len(bounds) - 1
            if N > 1 and cut:   # (what the short sequence takes lengthens the segments)
                continue
            assert (_plan(bounds, N, chunks * CHUNK, heads, 2, reverse, kind) is not None) == cut


@pytest.mark.parametrize("kind,heads,slabs,chunks,cut", [
    # kinds 1 and 2 with 128 key channels and 64 value channels, and (+ 8) with 64 key channels
    (1, 4, 1, 20, False), (1, 4, 1, 28, True), (1, 16, 1, 24, False), (1, 16, 1, 28, False), (1, 16, 1, 36, True), (1, 16, 1, 48, False),
    (1, 32, 1, 32, False), (1, 32, 1, 48, False), (1, 32, 1, 64, False), (2, 16, 1, 24, False), (2, 16, 1, 32, True),
    (2, 32, 1, 40, False), (2, 32, 1, 64, False), (9, 4, 2, 20, False), (9, 4, 2, 24, True), (9, 16, 2, 28, False),
    (9, 16, 2, 36, True), (9, 32, 2, 48, False), (9, 8, 1, 20, False), (9, 8, 1, 24, True), (9, 32, 1, 28, False), (9, 32, 1, 40, True),
    (9, 64, 1, 64, False), (10, 8, 1, 20, True), (10, 16, 2, 24, False), (10, 16, 2, 32, True), (10, 32, 2, 64, False),
    (10, 32, 1, 48, True)])
def test_cut_where_it_pays_with_other_head_dims(kind, heads, slabs, chunks, cut):
    """The delta rule with head dims other than 128 and 128, on both sides of the measured lines (32 heads of 128 keys and 64 values,
    32 chunks: 50 us uncut, 68 cut)."""
    for reverse in (0, 1):
        got = _plan(None, 1, chunks * CHUNK, heads, slabs, reverse, kind)
        assert (got is not None) == cut
        if cut:
            _check(*got, [chunks], heads, slabs, reverse, kind)


@pytest.mark.parametrize("heads,slabs,chunks,cut", [
    (4, 4, 16, False), (4, 4, 32, True), (8, 4, 24, False), (8, 4, 48, True), (16, 4, 32, False), (16, 4, 48, True),
    (24, 4, 64, False), (24, 4, 96, True), (32, 4, 64, False), (8, 1, 16, False), (8, 1, 24, True), (32, 1, 24, False),
    (32, 1, 32, True), (64, 1, 32, False), (96, 1, 48, False), (128, 1, 48, False)])
def test_state_gradients_are_cut_where_it_pays(heads, slabs, chunks, cut):
    """The reverse scan of GLA's backward (kind 4), on both sides of the measured lines."""
    for bounds in (None, [0, chunks * CHUNK]):
        got = _plan(bounds, 1, chunks * CHUNK, heads, slabs, 1, 4)
        assert (got is not None) == cut
        if cut:
            _check(*got, [chunks], heads, slabs, 1, 0)


@pytest.mark.parametrize("kind,heads,chunks,cut", [
    (1, 16, [54, 94, 77], False), (1, 16, [46, 42, 40, 40], False), (1, 16, [60, 20, 20, 20], False), (1, 16, [80, 171], True),
    (1, 16, [48, 40], False), (1, 8, [54, 94, 77], True), (3, 16, [46, 42, 40, 40], False), (3, 16, [54, 94, 77], True),
    (0, 16, [46, 42, 40, 40], True), (2, 8, [30, 10, 10], False), (2, 8, [20, 63, 49, 26], False),
    (2, 8, [80, 40], True)])
def test_packed_batches_are_cut_where_it_pays(kind, heads, chunks, cut):
    """The measured packed batches: segments are as long as room for all of them makes them (delta rule, 16 heads, 54, 94 and
    77 chunks in segments of 32: 132 us uncut, 146 cut)."""
    bounds = [0]
    for c in chunks:
        bounds.append(bounds[-1] + c * CHUNK - 5)
    for reverse in (0, 1):
        assert (_plan(bounds, len(chunks), bounds[-1], heads, 2, reverse, kind) is not None) == cut
