"""Work lists of one attention call, shared by the dynamic-shape and the
uniform / cross plans: the tile unions that the forward, dQ and dK/dV kernels
walk, their launch orders, which kernels the call takes, and what is kept from
the forward to the backward.

The reference's kernels take one list per 64-token tile (bsa_interface.py
:328-523) and need none of this; the lists here come from the same selection.
"""
from __future__ import annotations

import torch

from . import ops


class _Side:
    """The lists that one side's kernels walk (queries: forward and dQ, keys:
    dK/dV), built when first asked for."""

    def __init__(self, source, rows, cols, BH, D, keys, tmasks):
        self.source = source      # the per-tile lists (start, len, cols)
        self.rows, self.cols, self.BH, self.D, self.keys, self.tmasks = rows, cols, BH, D, keys, tmasks
        self.group = 32 if keys else 64
        pairs = BH * (rows // 2)
        # a side of a few rounds of workgroups: its dense lists are kept as
        # they are (at most ops.KEEP_DENSE_BYTES)
        self.small = (pairs < 8 * 8 * self.group
                      and 4 * max(2 * pairs * cols, source[2].numel()) <= ops.KEEP_DENSE_BYTES)
        self._pairmap = self._pairs = self._items = None
        self.split = None         # (whole, splits) of items
        self._orders = {}

    @property
    def pairmap(self):
        """Tiles paired inside each group of 8 by list overlap (fewest idle
        wave slots)."""
        if self._pairmap is None:
            self._pairmap = ops.pair_tiles(*self.source, self.rows, self.cols)
        return self._pairmap

    def union(self):
        return ops.pair_union(*self.source, self.rows, self.tmasks, col_tiles=self.cols, pairmap=self.pairmap)

    @property
    def pairs(self):
        """Pair unions."""
        if self._pairs is None:
            self._pairs = self.union()
        return self._pairs

    @pairs.setter
    def pairs(self, value):
        self._pairs = value

    @property
    def items(self):
        """The backward's lists: the work items of a split launch where a
        launch over the pairs would leave the GPU partly idle, else the pairs."""
        if self._items is None and self.small:
            whole, splits = ops.split_plan(2 if self.keys else 1, self.BH, self.rows // 2, self.cols, self.D)
            if splits > 1:
                self.split = (whole, splits)
                self._items = ops.part_union(*self.source, self.rows, whole, splits, self.tmasks, col_tiles=self.cols,
                                             pairmap=self.pairmap)
        return self.pairs if self._items is None else self._items

    def order(self, lists):
        """Launch order over pairs or items."""
        key = "items" if lists is self._items else "pairs"
        if key not in self._orders:
            self._orders[key] = ops.items_order(lists[1], self.group, self.BH, self.cache_bytes)
        return self._orders[key]

    @property
    def cache_bytes(self):
        """bf16 operand rows that the lists index (K and V, or Q and dO)."""
        return self.BH * self.cols * 64 * self.D * 4


class WorkLists:
    """Base of the plans.  A plan sets qstart, qlen, qcols (its per-query-tile
    key lists) and calls _build_query_lists.

    A query side of fewer than eight rounds of workgroups walks pairs (its
    forward single tiles when there are few), whatever the quad switches say; a
    larger one walks pairs or quads, as the switches and the lists say."""

    def _build_query_lists(self, BH, Ntq, Ntk, D, tmasks, compact, dq_quads):
        self._BH, self._Ntq, self._Ntk, self._D = BH, Ntq, Ntk, D
        self.tmasks = tmasks
        # compact lists: what the backward keeps of a large side is stored as
        # CSR, O(nnz) memory instead of pairs x Nt
        self.compact = compact
        self._settled = False
        self._csr = None
        self._q = _Side((self.qstart, self.qlen, self.qcols), Ntq, Ntk, BH, D, False, tmasks)
        self._k = None
        self._few = self._q.small and BH * Ntq // 2 <= ops.TILE_PAIRS
        # quad unions (two pairs of a group per workgroup: four query tiles per
        # staged K / V tile); quads: the call may walk them, dq_quads: dQ too
        self.quads = ops.QUADS and Ntq % 4 == 0
        self.dq_quads = self.quads and dq_quads
        self._qquad = self._qquad_order = self._qquad_total = None
        self._shown = {}
        if self.quads and not self._q.small:
            self._qquad = self._query_quads()
            self._qquad_order, self._qquad_total = ops.launch_order(self._qquad[1], BH, self._q.cache_bytes)
        self.klists = None
        self.keys_ready = None  # event of a key-list build on the side stream

    def _query_quads(self):
        return ops.quad_union(*self._q.source, self._Ntq, self.tmasks, col_tiles=self._Ntk, pairmap=self.qpair)

    # ------------------------------------------------ the lists, for inspection
    def _union_of(self, name, side):
        """A side's pair unions.  A small side's kernels may walk other lists,
        and keep them dense: its unions are built when asked for, as CSR once a
        compact plan has settled."""
        if side is None or not side.small:
            return None if side is None else side.pairs
        if name not in self._shown:
            u = side.union()
            if self._settled and self.compact:
                u = (*ops.csr_lists(ops.csr_offsets(u[1])[0]), ops.lists_to_csr(*u)[1])
            self._shown[name] = u
        return self._shown[name]

    @property
    def qunion(self):
        """Query-side pair unions (CSR once a compact plan has settled)."""
        return self._union_of("q", self._q)

    @property
    def kunion(self):
        """Key-side pair unions, once build_key_lists has run."""
        return self._union_of("k", self._k)

    @property
    def qpair(self):
        return self._q.pairmap

    @property
    def kpair(self):
        return None if self._k is None else self._k.pairmap

    @property
    def qorder(self):
        """A launch order of the pair kernels over qunion."""
        if "qorder" not in self._shown:
            self._shown["qorder"] = ops.pair_order(self.qunion[1], 64)
        return self._shown["qorder"]

    @property
    def korder(self):
        if "korder" not in self._shown and self._k is not None:
            self._shown["korder"] = ops.pair_order(self.kunion[1], 32)
        return self._shown.get("korder")

    @property
    def qquadmap(self):
        return self.qpair if self.quads else None

    @property
    def qquad(self):
        """Quad unions (None where the call cannot walk them or has released
        them); a small query side builds them when asked."""
        if self._qquad is None and self._q.small and (self.dq_quads if self._settled else self.quads):
            self._qquad = self._query_quads()
        return self._qquad

    @property
    def qquad_order(self):
        if self._qquad_order is None and self.qquad is not None:
            self._qquad_order = ops.pair_order(self._qquad[1], 32)
        return self._qquad_order

    # ------------------------------------------------ key-side lists
    def build_key_lists_side(self):
        """build_key_lists on the side stream, after the work queued so far on
        the current stream."""
        if self._k is not None:
            return
        _, self.keys_ready = ops.side_launch(
            self.qcols.device, self.build_key_lists, reads=(self.qstart, self.qlen, self.qcols),
            produces=lambda _: (*self.klists, self._k.pairmap, *self._k.items, self._k.order(self._k.items),
                                self._csr.offsets[1] if self._csr is not None else None))

    def join_side(self):
        """Make the current stream wait for a side-stream key-list build (the
        stream fork is joined where it was opened, so a captured or
        backward-less forward leaves no dangling dependency)."""
        if self.keys_ready is not None:
            torch.cuda.current_stream().wait_event(self.keys_ready)
            self.keys_ready = None

    def build_key_lists(self):
        """Per-key-tile query lists, their pairing, unions and launch order
        (the dK/dV side), built on first use."""
        self.join_side()
        if self._k is not None:
            return
        Ntq, Ntk = self._Ntq, self._Ntk
        self.klists = ops.transpose_lists(self.qstart, self.qlen, self.qcols, self._BH, Ntq, Ntk)
        self._k = k = _Side(self.klists, Ntk, Ntq, self._BH, self._D, True, None)
        k.order(k.items)
        if self._csr is not None and not k.small:
            self._csr.add(1, k.pairs)

    def key_lists(self):
        self.build_key_lists()
        return self.kunion

    # ------------------------------------------------ from forward to backward
    def _start_compaction(self):
        """Sizes of the large sides' unions, copied to the host without
        waiting."""
        if self.compact and self._csr is None:
            self._csr = ops.DeferredCompaction(3)
            if not self._q.small:
                self._csr.add(0, self._q.pairs)
                if self.dq_quads:
                    self._csr.add(2, self._qquad)
            if self._k is not None and not self._k.small:
                self._csr.add(1, self._k.pairs)

    def settle(self):
        """Keep only what the backward reads: each side's lists (a large
        side's pair unions, and the quad unions when dQ walks them, as CSR when
        the plan is compact, with one batched host read of their sizes),
        pairings and launch orders.  A large side's per-tile lists (1.0 GB
        query-side and 0.66 GB key-side at a 21 x 90 x 160 grid with 5 heads)
        and the forward-only quad unions are released."""
        if self._settled:
            return
        self.build_key_lists()
        self._start_compaction()
        if self.dq_quads and not self._q.small and ops.DQ_QUADS is None:
            sizes = None if self._csr is None else self._csr.sizes()
            self.dq_quads = sizes is not None and sizes[0] >= ops.DQ_QUAD_RATIO * sizes[2]
        if not self.dq_quads and not self._q.small:
            self._qquad = None
        if self._csr is not None:
            self._q._pairs, self._k._pairs = self._csr.finish([self._q._pairs, self._k._pairs])
            if self._qquad is not None:
                self._qquad = self._csr.fill(2, self._qquad)
            self._csr = None
        if not self.dq_quads or self._q.small:  # not walked by the backward
            self._qquad = self._qquad_order = None
        for side in (self._q, self._k):
            if not side.small:
                side.source = None
        self._shown.pop("q", None)
        self._shown.pop("k", None)
        self.qcols = None
        self.klists = None
        self.sel = {key: val for key, val in self.sel.items() if key != "tiles"}
        self._settled = True

    def list_bytes(self) -> int:
        """Bytes of the work lists that the plan holds (small sides: of the
        pair unions that stand for theirs)."""
        ts = [*self.qunion, self.qstart, self.qlen]
        for lists in (self._qquad, self.kunion, self.klists):
            if lists is not None:
                ts += list(lists)
        if self.qcols is not None:
            ts.append(self.qcols)
        return sum(t.numel() * t.element_size() for t in ts)

    def sum_lens(self) -> int:
        """Executed (query tile, key tile) pairs (host sync)."""
        return int(self.qlen.sum().item())

    # ------------------------------------------------ the attention launches
    def attend(self, sm_scale: float, grads: bool):
        """o and lse in tile order; with grads the backward's lists are built
        beside the forward kernel (or before it), and the per-tile lists
        released."""
        if grads:
            if not self._q.small:
                self._start_compaction()
            if ops.OVERLAP_SIDE_WORK:
                self.build_key_lists_side()
            else:
                self.build_key_lists()
        qkv, q = (self.q_re, self.k_re, self.v_re, self.tmasks), self._q
        if self._few:
            out = ops.bsa_fwd_tile(*qkv, ops.tile_lists(*q.source, self._Ntq, self.tmasks, self._Ntk), sm_scale)
        elif self.quads and not q.small:
            order, total = ops.launch_order(q.pairs[1], self._BH, q.cache_bytes, ops.FWD_CHUNK)
            out = ops.bsa_fwd_either(*qkv, q.pairs, order, total, self._qquad, self._qquad_order, self._qquad_total,
                                     sm_scale, q.pairmap)
        else:
            out = ops.bsa_fwd(*qkv, q.pairs, sm_scale, q.pairmap, q.order(q.pairs))
        self.join_side()  # queued after the forward kernel: the key lists still run beside it
        if grads:
            self.settle()  # release the per-tile lists; compact the unions while the forward runs
        return out

    def attend_backward(self, do_re, lse, delta, sm_scale: float, after_dkdv):
        """dq, dk, dv in tile order."""
        self.build_key_lists()
        q, k = self._q, self._k
        quads = self.dq_quads and not q.small
        qlists, klists = self._qquad if quads else q.items, k.items
        return ops.bsa_bwd(self.q_re, self.k_re, self.v_re, do_re, ops.lse_to_m2(lse), delta, self.kv_valid,
                           self.tmasks, qlists, klists, sm_scale, q.pairmap, k.pairmap,
                           self._qquad_order if quads else q.order(qlists), k.order(klists), after_dkdv=after_dkdv,
                           q_quads=quads, q_split=q.split, k_split=k.split)


__all__ = ["WorkLists"]
