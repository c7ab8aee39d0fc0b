"""Launches of few pairs: prism_bsa_fwd_tile over prism_tile_lists rows (one
workgroup per query tile, the pair forward's bits), prism_part_union and the
split dQ / dK/dV launches over it.

Lists of 0 to 6 entries around the copy pipeline's depth, tile counts that are
not multiples of the groups of 8 or of the 32-bit bitmap words, a list range of
more than one bitmap window (8,192 tiles), rows without a list, key masks,
split launches with and without whole pairs."""
import math

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import bits_equal, host, say
from tests.test_gpu_torch_ops import UTILS

pytestmark = pytest.mark.gpu


def make(seed, BH, Ntq, Ntk, D, longest, masked):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    t = lambda n: torch.randn((1, BH, n * 64, D), device="cuda", generator=g).to(torch.bfloat16)
    q, do, k, v = t(Ntq), t(Ntq), t(Ntk), t(Ntk)
    lens = rng.integers(0, min(longest, Ntk) + 1, BH * Ntq).astype(np.int32)
    lens[: min(7, lens.size)] = np.minimum(np.arange(min(7, lens.size)), Ntk)
    cols = np.concatenate([np.sort(rng.choice(Ntk, n, replace=False)) for n in lens] + [np.zeros(1)]).astype(np.int32)
    start = (np.cumsum(lens) - lens).astype(np.int64)
    dev = lambda a: torch.from_numpy(a).to("cuda")
    valid = torch.rand((Ntk * 64,), device="cuda", generator=g) < 0.8 if masked else None
    return q, k, v, do, (dev(start), dev(lens), dev(cols)), valid


@pytest.mark.parametrize("shape", [(1, 2, 2, 64, 2, False), (3, 6, 10, 64, 6, True), (2, 10, 40, 128, 40, True),
                                   (1, 4, 8202, 64, 60, False)], ids=str)
def test_tile_forward_equals_pair_forward(shape):
    from prism_amd import ops
    BH, Ntq, Ntk, D, longest, masked = shape
    say("tile forward", shape)
    q, k, v, _, lists, valid = make(1, BH, Ntq, Ntk, D, longest, masked)
    tm, sm = ops.tile_masks(valid), 1.0 / math.sqrt(D)
    rows = ops.tile_lists(*lists, Ntq, tm, Ntk)
    st, ln, cl = (host(t) for t in rows)
    s0, l0, c0 = (host(t) for t in lists)
    full = None if tm is None else host(tm) == -1
    for r in range(BH * Ntq):
        t = c0[s0[r]: s0[r] + l0[r]]
        part = np.zeros_like(t) if full is None else (~full[t]).astype(np.int32)
        assert np.array_equal(cl[st[r]: st[r] + ln[r]], t << 3 | part << 2 | 1 << (r % 2)), r
    o1, l1 = ops.bsa_fwd(q, k, v, tm, ops.pair_union(*lists, Ntq, tm, col_tiles=Ntk), sm)
    o2, l2 = ops.bsa_fwd_tile(q, k, v, tm, rows, sm)
    assert bits_equal(host(o1), host(o2)) and bits_equal(host(l1), host(l2))


def called(monkeypatch):
    """The names of the operators that run from here on."""
    from prism_amd import ops
    names, run = [], ops._op
    monkeypatch.setattr(ops, "_op", lambda name, *args: (names.append(name), run(name, *args))[1])
    return names


# (BH, Nt, width, D, operators after tile_masks): both sides of every line of
# the rule that picks the forward of given lists
ROUTES = [(2, 128, 9, 64, ["tile_lists", "bsa_fwd_tile"]),
          (2, 130, 9, 128, ["pair_union", "bsa_fwd"]),
          (4, 256, 70, 64, ["pair_union", "bsa_fwd"]),
          (2, 640, 16, 64, ["pair_tiles", "quad_union", "pair_order", "bsa_fwd_quad"]),
          (2, 642, 16, 64, ["pair_union", "bsa_fwd"]),
          (2, 640, 16, 128, ["pair_union", "bsa_fwd"]),
          (2, 636, 16, 64, ["pair_union", "bsa_fwd"]),
          (2, 640, 17, 64, ["pair_union", "bsa_fwd"]),
          (2, 514, 64, 64, ["pair_union", "bsa_fwd"]),
          (2, 514, 65, 64, ["pair_tiles", "pair_union", "launch_order", "bsa_fwd"]),
          (2, 1026, 129, 128, ["pair_union", "pair_order", "bsa_fwd"]),
          (2, 1026, 128, 128, ["pair_union", "bsa_fwd"]),
          (2, 1282, 130, 64, ["pair_union", "pair_order", "bsa_fwd"]),
          (16, 512, 5, 64, ["pair_tiles", "quad_union", "pair_order", "bsa_fwd_quad"]),
          (64, 130, 5, 64, ["pair_union", "bsa_fwd"])]


@pytest.mark.parametrize("shape", ROUTES, ids=str)
def test_given_lists_forward_routes(shape, monkeypatch):
    """attn_fwd_bsa_varlen: the kernels and launch orders of the rule, and the
    bits of the pair forward over neighbouring pairs whichever it takes (empty
    lists, unsorted rows, key masks)."""
    from prism_amd import bsa_interface, ops
    BH, Nt, W, D, want = shape
    say("forward route", shape)
    g = torch.Generator(device="cuda").manual_seed(W)
    q, k, v = (torch.randn((1, BH, Nt * 64, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    idx = torch.sort(torch.rand((1, BH, Nt, Nt), device="cuda", generator=g), -1).indices[..., :W].contiguous()
    lens = torch.randint(0, W + 1, (1, BH, Nt), device="cuda", generator=g, dtype=torch.int32)
    valid = torch.rand((Nt * 64,), device="cuda", generator=g) < 0.8
    tm, sm = ops.tile_masks(valid), 1.0 / math.sqrt(D)
    union = ops.pair_union(*bsa_interface._lists_from_dense(idx, lens), Nt, tm, col_tiles=Nt)
    ref = ops.bsa_fwd(q, k, v, tm, union, sm)
    names = called(monkeypatch)
    got = bsa_interface.attn_fwd_bsa_varlen(q, k, v, sm, idx, lens, kv_valid_mask=valid)
    assert [n for n in names if n != "tile_masks"] == want
    assert all(bits_equal(host(a), host(b)) for a, b in zip(ref, got))


# (whole, splits): every pair split, some, none
@pytest.mark.parametrize("shape", [(1, 2, 2, 64, 2, False, 0, 2), (3, 6, 10, 64, 6, True, 3, 3),
                                   (2, 10, 40, 128, 40, True, 4, 5), (2, 16, 24, 128, 24, False, 16, 1),
                                   (1, 4, 8202, 64, 60, False, 0, 16)], ids=str)
def test_split_backward(shape):
    from prism_amd import ops
    BH, Ntq, Ntk, D, longest, masked, whole, splits = shape
    say("split backward", shape)
    q, k, v, do, lists, valid = make(2, BH, Ntq, Ntk, D, longest, masked)
    tm, sm = ops.tile_masks(valid), 1.0 / math.sqrt(D)
    kv = None if valid is None else valid.to(torch.uint8)
    klists = ops.transpose_lists(*lists, BH, Ntq, Ntk)
    qpair, kpair = ops.pair_tiles(*lists, Ntq, Ntk), ops.pair_tiles(*klists, Ntk, Ntq)
    qun = ops.pair_union(*lists, Ntq, tm, col_tiles=Ntk, pairmap=qpair)
    kun = ops.pair_union(*klists, Ntk, None, col_tiles=Ntq, pairmap=kpair)
    kwhole = min(whole, BH * Ntk // 2)
    qit = ops.part_union(*lists, Ntq, whole, splits, tm, col_tiles=Ntk, pairmap=qpair)
    kit = ops.part_union(*klists, Ntk, kwhole, splits, None, col_tiles=Ntq, pairmap=kpair)
    for un, it, w in ((qun, qit, whole), (kun, kit, kwhole)):
        us, ul, uc = (host(t) for t in un)
        s, n, c = (host(t) for t in it)
        assert n.size == w + (ul.size - w) * splits
        # the items of a pair take little more than the pair's own row
        assert c.size <= uc.size + 8 * (n.size - w)
        for i in range(n.size):
            p, part = (i, -1) if i < w else (w + (i - w) // splits, (i - w) % splits)
            e = uc[us[p]: us[p] + ul[p]]
            assert np.array_equal(c[s[i]: s[i] + n[i]], e if part < 0 else e[(e >> 6) % splits == part]), i
    o, lse = ops.bsa_fwd(q, k, v, tm, qun, sm, qpair)
    m2, delta = ops.lse_to_m2(lse), ops.bwd_preprocess(o, do)
    ref = ops.bsa_bwd(q, k, v, do, m2, delta, kv, tm, qun, kun, sm, qpair, kpair)
    order = lambda u: torch.randperm(u[1].numel(), device="cuda").int()
    one = (order(qit), order(kit))
    got = [ops.bsa_bwd(q, k, v, do, m2, delta, kv, tm, qit, kit, sm, qpair, kpair, *od, q_split=(whole, splits),
                       k_split=(kwhole, splits)) for od in (one, (None, None))]
    for name, a, b, c in zip(("dq", "dk", "dv"), ref, *got):
        assert bits_equal(host(b), host(c)), name  # the launch order changes nothing
        # the same float32 products in another order of summation, rounded to
        # bf16 once: at most one bf16 step (2^-7 of the value) apart, plus the
        # float32 rounding of at most 60 x 64 terms, well below 2^-10 of the
        # tensor's root mean square
        x, y = a.float(), b.float()
        assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 2.0 ** -10 * x.pow(2).mean().sqrt()).all()), name
        if splits == 1:
            assert bits_equal(host(a), host(b)), name


def _close(x, y, name):
    """The same float32 products in another order of summation: as in
    test_split_backward."""
    x, y = x.float(), y.float()
    assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 2.0 ** -10 * x.pow(2).mean().sqrt()).all()), name


def _call(kind):
    """(function of q, k, v; their tokens; sides that are split): a clip of 576
    tiles, attended by itself, by 300 audio tokens, and attending to them."""
    from prism_amd import flash_attn_bsa_3d_dynamic, flash_attn_bsa_cross
    grid = (16, 32, 72)
    S = grid[0] * grid[1] * grid[2]
    if kind == "self":
        return (lambda q, k, v: flash_attn_bsa_3d_dynamic(q, k, v, grid, method="ivpq", sparsity=0.9)), S, S, "qk"
    if kind == "audio_queries":
        return (lambda q, k, v: flash_attn_bsa_cross(q, k, v, "1d", "3d", k_grid_size=grid, sparsity=0.75)), 300, S, "q"
    return (lambda q, k, v: flash_attn_bsa_cross(q, k, v, "3d", "1d", q_grid_size=grid, sparsity=0.5)), S, 300, "k"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kind", ["self", "audio_queries", "audio_keys"])
def test_split_through_the_layers(kind, D, monkeypatch):
    """A training step whose dQ and / or dK/dV is split, key lists beside the
    forward or before it: the gradients of whole lists to the order of
    summation, the same bits from both overlap settings, the forward's bits
    untouched."""
    from prism_amd import ops
    fn, Sq, Sk, sides = _call(kind)
    say("split layer", kind, D)
    g = torch.Generator(device="cuda").manual_seed(11)
    make_t = lambda S: torch.randn((1, 2, S, D), device="cuda", generator=g).to(torch.bfloat16)
    q, k, v, do = make_t(Sq), make_t(Sk), make_t(Sk), make_t(Sq)

    def step(overlap, split):
        monkeypatch.undo()
        monkeypatch.setattr(ops, "OVERLAP_SIDE_WORK", overlap)
        if not split:
            monkeypatch.setattr(ops, "split_plan", lambda kernel, heads, per_head, entries, D: (heads * per_head, 1))
        names = called(monkeypatch)
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = fn(*x)
        plan = o.grad_fn.plan
        assert (plan._q.split is not None) == (split and "q" in sides)
        assert (plan._k.split is not None) == (split and "k" in sides)
        assert plan._q.source is None and plan._k.source is None
        o.backward(do)
        assert ("bsa_bwd_dq_split" in names) == (split and "q" in sides)
        assert ("bsa_bwd_dkdv_split" in names) == (split and "k" in sides)
        return [o.detach()] + [t.grad for t in x]

    whole, apart, beside = step(True, False), step(False, True), step(True, True)
    assert bits_equal(host(whole[0]), host(beside[0]))
    for name, w, a, b in zip(("O", "dQ", "dK", "dV"), whole, apart, beside):
        assert bits_equal(host(a), host(b)), name
        _close(w, b, name)


@pytest.mark.parametrize("D", [64, 128])
def test_split_given_lists(D, monkeypatch):
    """attn_bwd_bsa_varlen over lists long enough to be split, with key masks."""
    from prism_amd import bsa_interface, ops
    BH, Nt, W = 2, 514, 70
    say("split given lists", D)
    g = torch.Generator(device="cuda").manual_seed(12)
    q, k, v, do = (torch.randn((1, BH, Nt * 64, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(4))
    idx = torch.sort(torch.rand((1, BH, Nt, Nt), device="cuda", generator=g), -1).indices[..., :W]
    idx, lens = torch.sort(idx, -1).values, torch.randint(0, W + 1, (1, BH, Nt), device="cuda", generator=g, dtype=torch.int32)
    valid = torch.rand((Nt * 64,), device="cuda", generator=g) < 0.8
    o, lse = bsa_interface.attn_fwd_bsa_varlen(q, k, v, 0.1, idx, lens, kv_valid_mask=valid)

    def back():
        out = [torch.empty_like(t) for t in (q, k, v)]
        return bsa_interface.attn_bwd_bsa_varlen(do, q, k, v, o, *out, 0.1, lse, idx, lens, kv_valid_mask=valid)

    names = called(monkeypatch)
    split = back()
    assert "bsa_bwd_dq_split" in names and "bsa_bwd_dkdv_split" in names
    monkeypatch.setattr(ops, "split_plan", lambda kernel, heads, per_head, entries, D: (heads * per_head, 1))
    names.clear()
    for name, w, x in zip(("dQ", "dK", "dV"), back(), split):
        _close(w, x, name)
    assert "bsa_bwd_dq" in names and "bsa_bwd_dkdv" in names


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("grid,audio", [((7, 16, 16), 0), ((9, 30, 52), 0), ((7, 20, 24), 460)], ids=str)
def test_small_and_large_launches_agree(grid, audio, D, monkeypatch):
    """Single tiles and dense lists of small launches against pairs or quads
    and compact or dense lists of large ones: the same output and gradients,
    bit for bit (lists too short to be split)."""
    from prism_amd import flash_attn_bsa_cross, ops
    from prism_amd.adapter import run_bsa_uniform
    S = grid[0] * grid[1] * grid[2]
    say("small and large", grid, audio, D)
    g = torch.Generator(device="cuda").manual_seed(13)
    make_t = lambda n: torch.randn((1, 2, n, D), device="cuda", generator=g).to(torch.bfloat16)
    q, k, v, do = make_t(audio or S), make_t(S), make_t(S), make_t(audio or S)
    outs = []
    for keep, compact in ((ops.KEEP_DENSE_BYTES, True), (-1, True), (-1, False)):
        monkeypatch.setattr(ops, "KEEP_DENSE_BYTES", keep)
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        if audio:
            o = flash_attn_bsa_cross(*x, "1d", "3d", k_grid_size=grid, sparsity=0.75)
        else:
            o = run_bsa_uniform(*x, grid, {"sparsity": 0.75, "cdf_threshold": 0.9, "compact_lists": compact})
        assert o.grad_fn.plan._q.small == (keep > 0)
        o.backward(do)
        outs.append([host(t) for t in (o, *(t.grad for t in x))])
    for other in outs[1:]:
        for name, a, b in zip(("O", "dQ", "dK", "dV"), outs[0], other):
            assert bits_equal(a, b), name


def test_split_plan_covers_the_gpu():
    """split_plan cuts only launches of a few rounds over long lists, at a
    group boundary, and never makes more items than it has workgroups for
    eight rounds."""
    from prism_amd import ops
    for kernel in (1, 2):
        for heads, per_head in ((1, 1), (5, 16), (3, 720), (1, 37), (24, 2000)):
            for entries in (32, 511, 512, 6900):
                whole, splits = ops.split_plan(kernel, heads, per_head, entries, 128)
                pairs = heads * per_head
                assert 0 <= whole <= pairs and 1 <= splits <= 16
                assert (whole == pairs) == (splits == 1)
                assert splits == 1 or (entries >= 512 and (whole % per_head) % 4 == 0)
                assert whole + (pairs - whole) * splits <= max(pairs, 8 * 512)


def test_operators_opcheck():
    from prism_amd import ops
    q, k, v, do, lists, _ = make(3, 1, 4, 6, 64, 6, False)
    P = torch.ops.prism

    def chk(op, args):
        torch.library.opcheck(op.default, args, test_utils=UTILS)

    rows = ops.tile_lists(*lists, 4, None, 6)
    chk(P.tile_lists, (*lists, 4, 6, None))
    chk(P.bsa_fwd_tile, (q, k, v, None, *rows, 0.125))
    items = ops.part_union(*lists, 4, 1, 2, None, col_tiles=6)
    chk(P.part_union, (*lists, 4, 6, None, None, 1, 2))
    o, lse = ops.bsa_fwd_tile(q, k, v, None, rows, 0.125)
    m2, delta = ops.lse_to_m2(lse), ops.bwd_preprocess(o, do)
    chk(P.bsa_bwd_dq_split, (q, k, v, do, m2, delta, None, *items, None, None, 0.125, 1, 2))
    kit = ops.part_union(*ops.transpose_lists(*lists, 1, 4, 6), 6, 1, 2, None, col_tiles=4)
    chk(P.bsa_bwd_dkdv_split, (q, k, v, do, m2, delta, None, *kit, None, None, 0.125, 1, 2))


@pytest.mark.parametrize("heads,per_head", [(1, 1), (3, 7), (2, 1024), (5, 1025), (2, 2600), (1, 5000), (1, 16384),
                                            (2, 16500)], ids=str)
def test_launch_order(heads, per_head):
    """Each run longest first, then the lower list; total the sum; chunked
    orders the same ranks dealt to the XCDs; lengths past the sort key's
    range still give a permutation."""
    from prism_amd import ops
    n = heads * per_head
    rng = np.random.default_rng(n)
    u = rng.integers(0, 40, n).astype(np.int32)
    ulen = torch.from_numpy(u).to("cuda")
    say("launch order", (heads, per_head))
    seg = -(-per_head // -(-per_head // 16384))
    runs = [np.arange(b, min(b + seg, n)) for b in range(0, n, seg)]
    want = np.concatenate([r[np.argsort(-u[r], kind="stable")] for r in runs])
    order, total = ops.launch_order(ulen, heads, 1 << 40)
    assert np.array_equal(host(order), want) and int(total) == int(u.sum())
    chunked = host(ops.launch_order(ulen, heads, 1 << 40, 4)[0])
    for r in runs:
        ranks, got = want[r], chunked[r]
        for c in range(len(r) // 32):
            for x in range(8):
                seg_x = 7 - x if c & 1 else x
                assert np.array_equal(got[32 * c + x: 32 * c + 32: 8], ranks[32 * c + 4 * seg_x: 32 * c + 4 * seg_x + 4])
        tail = len(r) // 32 * 32
        assert np.array_equal(got[tail:], ranks[tail:])
    if n <= 16384:
        assert np.array_equal(host(ops.launch_order(ulen, heads, 0)[0]), np.argsort(-u, kind="stable"))
    big = ops.launch_order(ulen * 100000, heads, 1 << 40)[0]
    assert np.array_equal(np.sort(host(big)), np.arange(n))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shared", [True, False])
def test_fwd_either_walks_one(D, shared):
    """The device's choice (quads when the tiles of a quad share their lists,
    pairs when they do not) changes no bit; the kernel not chosen writes
    nothing."""
    from prism_amd import ops
    BH, Nt, W = 2, 16, 5
    say("fwd either", D, shared)
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((1, BH, Nt * 64, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    rng = np.random.default_rng(5)
    rows = [np.sort(rng.choice(Nt, W, replace=False)) for _ in range(BH * Nt)]
    if shared:
        rows = [rows[r // 8] for r in range(BH * Nt)]
    dev = lambda a, t: torch.from_numpy(np.ascontiguousarray(a)).to("cuda", t)
    lists = (dev(np.arange(BH * Nt) * W, torch.int64), dev(np.full(BH * Nt, W), torch.int32),
             dev(np.concatenate(rows), torch.int32))
    pm = ops.pair_tiles(*lists, Nt)
    pairs, quads = ops.pair_union(*lists, Nt, pairmap=pm), ops.quad_union(*lists, Nt, pairmap=pm)
    po, pt = ops.launch_order(pairs[1], BH, 0)
    qo, qt = ops.launch_order(quads[1], BH, 0)
    assert (2 * int(pt) >= 3 * int(qt)) == shared
    want = ops.bsa_fwd(q, k, v, None, pairs, 0.1, pm)
    got = ops.bsa_fwd_either(q, k, v, None, pairs, po, pt, quads, qo, qt, 0.1, pm)
    assert all(bits_equal(host(a), host(b)) for a, b in zip(want, got))
    # the choice is the totals': the other way round on the same lists
    zero = torch.zeros_like(pt)
    for a, b in ((zero, qt), (pt, zero)):
        got = ops.bsa_fwd_either(q, k, v, None, pairs, None, a, quads, None, b, 0.1, pm)
        assert all(bits_equal(host(x), host(y)) for x, y in zip(want, got))
    torch.library.opcheck(torch.ops.prism.launch_order.default, (pairs[1], 8, 1), test_utils=UTILS)
    torch.library.opcheck(torch.ops.prism.bsa_fwd_either.default,
                          (q, k, v, None, *pairs, po, pt, *quads, qo, qt, pm, 0.1), test_utils=UTILS)
