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
        self.source = source      # the per-tile lists (start, len, cols), until release()
        self.rows, self.cols, self.BH, self.D, self.keys, self.tmasks = rows, cols, BH, D, keys, tmasks
        self.group = 32 if keys else 64
        pairs = BH * (rows // 2)
        # a side of a few rounds of workgroups whose lists take little room:
        # what its backward walks is kept dense (ops.KEEP_DENSE_BYTES)
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

    @property
    def pairs(self):
        """Pair unions (None once a split side is released)."""
        if self._pairs is None and self.source is not None:
            self._pairs = ops.pair_union(*self.source, self.rows, self.tmasks, col_tiles=self.cols,
                                         pairmap=self.pairmap)
        return self._pairs

    @property
    def items(self):
        """The backward's lists: the work items of a split launch where a
        launch over the pairs would leave the GPU partly idle, else the pairs."""
        if self._items is None and self.small and self.source is not None:
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

    def release(self, walked=True):
        """Keep the backward's lists, their order (if it walks them) and the
        pairing alone."""
        items = self.items
        if walked:
            self.order(items)
        if self._items is not None:
            self._pairs = None
            self._orders.pop("pairs", None)
        self.source = None

    def compact(self, pairs):
        """The pair unions as CSR: the same rows and entries."""
        self._pairs = pairs

    def tensors(self):
        """Every list, pairing and order that the side holds."""
        for lists in (self.source, self._pairs, self._items):
            yield from lists or ()
        yield self._pairmap
        yield from self._orders.values()

    @property
    def cache_bytes(self):
        """bf16 operand rows that the lists index (K and V, or Q and dO)."""
        return self.BH * self.cols * 64 * self.D * 4


class WorkLists:
    """Base of the plans.  A plan sets qstart, qlen, qcols (its per-query-tile
    key lists) and calls _build_query_lists.

    A side of fewer than eight rounds of workgroups whose lists fit
    ops.KEEP_DENSE_BYTES is small: its backward walks pairs, split where that
    fills the GPU, its forward pairs or, when there are few, single tiles,
    whatever the quad switches say.  A larger one walks pairs or quads, as the
    switches and the lists say."""

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
        # staged K / V tile) of a large side; quads: the switches and tile
        # counts allow them, dq_quads: for dQ too
        self.quads = ops.QUADS and Ntq % 4 == 0
        self.dq_quads = self.quads and dq_quads
        self.qquad = self.qquad_order = self._qquad_total = None
        if self.quads and not self._q.small:
            self.qquad = ops.quad_union(*self._q.source, Ntq, tmasks, col_tiles=Ntk, pairmap=self.qpair)
            self.qquad_order, self._qquad_total = ops.launch_order(self.qquad[1], BH, self._q.cache_bytes)
        self.klists = None
        self.keys_ready = None  # event of a key-list build on the side stream

    # ------------------------------------------------ the lists, for callers that launch the kernels themselves
    @property
    def qunion(self):
        """Query-side pair unions (CSR once a compact plan of a large side has
        settled; None once a split side has)."""
        return self._q.pairs

    @property
    def kunion(self):
        """Key-side pair unions, once build_key_lists has run."""
        return None if self._k is None else self._k.pairs

    @property
    def qpair(self):
        return self._q.pairmap

    @property
    def kpair(self):
        return None if self._k is None else self._k.pairmap

    @property
    def qorder(self):
        """A launch order over qunion (launches that all run at once go without one)."""
        return ops.launch_order(self.qunion[1], self._BH, self._q.cache_bytes)[0]

    @property
    def korder(self):
        return None if self._k is None else ops.launch_order(self.kunion[1], self._BH, self._k.cache_bytes)[0]

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
                    self._csr.add(2, self.qquad)
            if self._k is not None and not self._k.small:
                self._csr.add(1, self._k.pairs)

    def settle(self):
        """Keep only what the backward reads: each side's lists, their launch
        order and the pairing.  A large side's are its pair unions (or, where dQ
        walks them, the quad unions beside them), as CSR when the plan is
        compact, with one batched host read of their sizes; a small side's its
        pair unions or split items.  The per-tile lists (1.0 GB query-side and
        0.66 GB key-side at a 21 x 90 x 160 grid with 5 heads) and the
        forward-only quad unions are released."""
        if self._settled:
            return
        self.build_key_lists()
        self._start_compaction()
        if self.qquad is not None and self.dq_quads and ops.DQ_QUADS is None:
            sizes = None if self._csr is None else self._csr.sizes()
            self.dq_quads = sizes is not None and sizes[0] >= ops.DQ_QUAD_RATIO * sizes[2]
        if not self.dq_quads:  # not walked by the backward
            self.qquad = self.qquad_order = None
        if self._csr is not None:
            for i, side in enumerate((self._q, self._k)):
                if not side.small:
                    side.compact(self._csr.fill(i, side.pairs))
            if self.qquad is not None:
                self.qquad = self._csr.fill(2, self.qquad)
            self._csr = None
        self._q.release(walked=self.qquad is None)
        self._k.release()
        self.qcols = None
        self.klists = None
        self.sel = {key: val for key, val in self.sel.items() if key != "tiles"}
        self._settled = True

    def list_bytes(self) -> int:
        """Bytes of the work lists, pairings and launch orders that the plan holds."""
        held = [self.qstart, self.qlen, self.qcols, self.qquad_order, *(self.qquad or ()), *(self.klists or ())]
        for side in (self._q, self._k):
            if side is not None:
                held += side.tensors()
        return sum({id(t): t.numel() * t.element_size() for t in held if t is not None}.values())

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
            out = ops.bsa_fwd_either(*qkv, q.pairs, order, total, self.qquad, self.qquad_order, self._qquad_total,
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
        quads = self.qquad is not None
        qlists, klists = self.qquad if quads else q.items, k.items
        return ops.bsa_bwd(self.q_re, self.k_re, self.v_re, do_re, ops.lse_to_m2(lse), delta, self.kv_valid,
                           self.tmasks, qlists, klists, sm_scale, q.pairmap, k.pairmap,
                           self.qquad_order if quads else q.order(qlists), k.order(klists), after_dkdv=after_dkdv,
                           q_quads=quads, q_split=q.split, k_split=k.split)


__all__ = ["WorkLists"]
