"""Dynamic-block-shape block-sparse attention, MI355X implementation.

Drop-in for hymm/models/modules/block_sparse_attention/dynamic_block_attention.py
of the reference: ``flash_attn_bsa_3d_dynamic`` keeps its signature, return
contract, errors and autograd behaviour (gradients flow to q, k, v only).

Pipeline (all HIP kernels of libprism_bsa.so, one host sync for N_b):
  (1) zone statistics + shape ids      prism_zone_stats / _gradient / _shapes
  (2) zone layout (block/tile maps)    prism_zone_layout
  (3) rearranged rows + block means    prism_gather_pool (q, k, v)
  (4) fp32 block scores + selection    prism_block_scores, prism_select_tiles
  (5) tile lists per query tile        prism_tile_rows
  (6) block-sparse attention           prism_bsa_fwd / prism_bsa_bwd_*
  (7) back to THW order                prism_scatter_rows
Deliberate differences from the reference: block
means and scores are fp32 (the reference pools and scores in q's dtype) and
every reduction uses one fixed order, so zone statistics, shape ids and
selected sets are reproducible bit for bit.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import ops
from .dynamic_block_shape import ALL_CANDIDATE_SHAPES, ZONE_SIZE, _gradient_and_shapes
from .worklists import WorkLists

_TILE = 64  # kernel tile (dynamic_block_attention.py:15)


# ------------------------------------------------------------------ geometry helpers (API parity)
def _build_rearrange_index(shape_ids, ZT, ZH, ZW, H, W, device):
    """src_idx[S], inv_idx[S] int64 (dynamic_block_attention.py:107-135)."""
    return ops.rearrange_index(shape_ids.to(device), (ZT * ZONE_SIZE, H, W))


def _build_block_tile_maps(shape_ids, ZT, ZH, ZW, device):
    """(block_id_of_tile [N_tiles], kblock_tiles [N_b+1, 2], N_b, N_tiles)
    (dynamic_block_attention.py:138-170)."""
    lay = ops.ZoneLayout(shape_ids.to(device), (ZT * ZONE_SIZE, ZH * ZONE_SIZE, ZW * ZONE_SIZE))
    first = lay.block_first_tile[: lay.N_b + 1].to(torch.int64)
    two = (first[1:] - first[:-1]) == 2
    kbt = torch.full((lay.N_b + 1, 2), lay.Nt, device=device, dtype=torch.int64)
    kbt[: lay.N_b, 0] = first[:-1]
    kbt[: lay.N_b, 1] = torch.where(two, first[:-1] + 1, torch.full_like(first[:-1], lay.Nt))
    return lay.block_id_of_tile.to(torch.int64), kbt, lay.N_b, lay.Nt


# ------------------------------------------------------------------ selection (steps 3-5)
class _Plan(WorkLists):
    """Everything the attention kernels need for one call, built under no_grad."""

    def __init__(self, q, k, v, grid, shape_ids, valid_mask, sparsity, cdf_threshold, sm_scale,
                 compute_padded_queries=False, box=None, keep_scores=False, compact_lists=False):
        B, H, _, D = q.shape
        self.lay = ops.ZoneLayout(shape_ids, grid, box)
        lay = self.lay
        self.B, self.H, self.S, self.D = B, H, lay.S, D
        self.grid = grid
        gq = ops.gather_pool(q, lay, valid_mask, rows=True, pool=True, counts=True)
        gk = ops.gather_pool(k, lay, valid_mask, rows=True, pool=True)
        gv = ops.gather_pool(v, lay, valid_mask, rows=True)
        self.q_re, self.k_re, self.v_re = gq["rows"], gk["rows"], gv["rows"]
        # zone-grid positions outside the input grid are invalid tokens
        masked = valid_mask is not None or lay.padded
        self.kv_valid = gq["valid_re"] if masked else None
        self.block_count = gq["block_count"]
        self.tile_count = gq["tile_count"]
        scores = ops.block_scores(gq["block_mean"].view(B * H, lay.N_b, D), gk["block_mean"].view(B * H, lay.N_b, D),
                                  self.block_count if masked else None)
        sel = ops.select_tiles(scores, sparsity, cdf_threshold, sm_scale, lay.block_first_tile,
                               self.tile_count if masked else None)
        # the [B*H, N_b, N_b] scores (564 MB at 2K) are freed once the lists
        # exist, as the reference frees them per head; kept only on request
        self.scores = scores if keep_scores else None
        del scores
        self.sel = sel
        skip = masked and not compute_padded_queries
        self.qstart, self.qlen = ops.tile_rows(sel["ntiles"], lay.block_id_of_tile, B * H, lay.Nt, lay.N_b,
                                               sel["tcap"], self.tile_count if skip else None)
        self.qcols = sel["tiles"].view(-1)
        # key validity words of padded key tiles, and the work lists
        tmasks = ops.tile_masks(self.kv_valid) if masked else None
        self._build_query_lists(B * H, lay.Nt, lay.Nt, D, tmasks, compact_lists, ops.DQ_QUADS is not False)


class _DynBSA(torch.autograd.Function):
    """Attention over a _Plan with gradients to the THW q, k, v
    (_dyn_bsa_kernel, dynamic_block_attention.py:71-101, plus the autograd of
    the gathers :250-252 and the scatter :329)."""

    @staticmethod
    def forward(ctx, q, k, v, plan: _Plan, sm_scale: float):
        o_re, lse = plan.attend(sm_scale, any(ctx.needs_input_grad[:3]))
        ctx.plan = plan
        ctx.sm_scale = sm_scale
        ctx.in_dtypes = (q.dtype, k.dtype, v.dtype)
        ctx.save_for_backward(o_re, lse)
        return ops.scatter_rows(o_re, plan.lay, q.dtype)

    @staticmethod
    def backward(ctx, do):
        plan: _Plan = ctx.plan
        o_re, lse = ctx.saved_tensors
        lay = plan.lay
        gd = ops.gather_pool(do.contiguous(), lay, None, rows=True, dot_with=o_re)
        do_re, delta = gd["rows"], gd["rowdot"]
        tq, tk, tv = ctx.in_dtypes
        side = {}

        def scatter_dkdv(dk_re, dv_re):
            # dK and dV back to THW order on the side stream, during the dQ kernel
            if ops.OVERLAP_SIDE_WORK and ops.OVERLAP_DKDV_SCATTER:
                side["dkdv"] = ops.side_launch(
                    dk_re.device, lambda: (ops.scatter_rows(dk_re, lay, tk), ops.scatter_rows(dv_re, lay, tv)),
                    reads=(dk_re, dv_re), produces=lambda out: out)

        dq_re, dk_re, dv_re = plan.attend_backward(do_re, lse, delta, ctx.sm_scale, scatter_dkdv)
        dq = ops.scatter_rows(dq_re, lay, tq)
        if "dkdv" in side:
            (dk, dv), done = side["dkdv"]
            torch.cuda.current_stream().wait_event(done)
        else:
            dk = ops.scatter_rows(dk_re, lay, tk)
            dv = ops.scatter_rows(dv_re, lay, tv)
        return dq, dk, dv, None, None


def plan_dynamic(q, k, v, grid_padded, *, method, sparsity=0.9375, cdf_threshold=None, audio_token_norms=None,
                 valid_mask=None, lambda_a=0.5, tau_128=0.15, lambda_128=1.0, shape_ids=None,
                 compute_padded_queries=False, input_grid=None, keep_scores=False, compact_lists=False) -> _Plan:
    """Steps (1)-(5) of flash_attn_bsa_3d_dynamic: shape ids, layout, pooled
    scores, selection and tile lists (no attention).

    With input_grid (Ti, Hi, Wi) inside grid_padded, q, k, v, the audio norms
    and valid_mask cover the input grid only (S = Ti Hi Wi): the zero padding
    and padding mask of wan_video_dit.py:342-400 are applied inside the
    kernels, with results identical to padding first.  compute_padded_queries
    defaults to False here, the adapters' setting (flash_attn_bsa_3d_dynamic
    passes True unless told otherwise).  keep_scores keeps the fp32 block
    scores on the plan (plan.scores) for inspection.  compact_lists makes
    plan.settle() keep the two pair unions in compact CSR form (O(nnz)
    memory, one host read for both); the plan keeps every list until then."""
    B, Hn, S, D = q.shape
    T, H, W = grid_padded
    box = tuple(input_grid) if input_grid is not None else (T, H, W)
    assert box[0] * box[1] * box[2] == S
    assert all(0 < b <= g for b, g in zip(box, (T, H, W)))
    assert T % ZONE_SIZE == 0 and H % ZONE_SIZE == 0 and W % ZONE_SIZE == 0
    if sparsity is None and cdf_threshold is None:
        raise ValueError("Either sparsity or cdf_threshold must be provided")
    if method not in ("ivpq", "penalty") and shape_ids is None:
        raise ValueError(f"unknown dynamic-block method: {method!r}")
    sm_scale = 1.0 / (D ** 0.5)
    with torch.no_grad():
        if shape_ids is not None:
            shape_ids = torch.as_tensor(shape_ids, device=q.device)
        else:
            shape_ids = _gradient_and_shapes(v.detach(), audio_token_norms, (T, H, W), method, lambda_a, tau_128,
                                             lambda_128, valid_mask, box)[2]
        return _Plan(q.detach(), k.detach(), v.detach(), (T, H, W), shape_ids, valid_mask, sparsity, cdf_threshold,
                     sm_scale, compute_padded_queries, box, keep_scores, compact_lists)


def flash_attn_bsa_3d_dynamic(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    grid_padded: Tuple[int, int, int],
    *,
    method: str,
    sparsity: Optional[float] = 0.9375,
    cdf_threshold: Optional[float] = None,
    audio_token_norms: Optional[torch.Tensor] = None,
    valid_mask: Optional[torch.Tensor] = None,
    lambda_a: float = 0.5,
    tau_128: float = 0.15,
    lambda_128: float = 1.0,
    shape_ids: Optional[torch.Tensor] = None,
    return_shape_ids: bool = False,
    compute_padded_queries: bool = True,
    input_grid: Optional[Tuple[int, int, int]] = None,
    compact_lists: bool = True,
):
    """Dynamic-block-shape BSA for video self-attention; returns [B,H,S,D] in
    THW order (dynamic_block_attention.py:194-332).  q, k, v: [B,H,S,D] THW
    order on the GPU, grid padded to multiples of 8; float32 or bfloat16
    (attention itself runs in bf16 MFMA with fp32 accumulation).

    With a valid_mask, query tiles that hold no valid token are padding the
    caller slices away (wan_video_dit.py:429-431).  Like the reference, this
    function attends for them by default (their pooled query is 0, so the
    threshold keeps ~p of all blocks).  compute_padded_queries=False (not in
    the reference's signature; the adapters use it) gives them empty lists
    instead: their output rows are 0, and outputs at valid positions and all
    gradients of valid tokens are the same either way when the incoming
    gradient is 0 at padded positions (as the caller's unpadding makes it).

    input_grid (not in the reference's signature) takes the caller's unpadded
    grid: q, k, v [B,H,Ti*Hi*Wi,D], audio norms and valid_mask then cover it,
    grid_padded is its round-up to multiples of 8, and the output (and the
    gradients) come back unpadded.  This is the padding, valid mask and
    unpadding of wan_video_dit.py:342-431 done inside the gather and scatter
    kernels; the result equals padding first and slicing after, bit for bit.

    When gradients are needed, the forward releases the per-tile lists once
    the backward's lists exist.  compact_lists (not in the reference's
    signature; default True) keeps those of a long launch in compact CSR form
    until the backward (O(nnz) memory, one host read of their sizes made while
    the forward kernel runs); False keeps them as dense pairs x Nt buffers.  A
    short launch's (fewer than eight rounds of workgroups) are kept dense either
    way, about 32 MB a side at most.  Results are identical either way."""
    plan = plan_dynamic(q, k, v, grid_padded, method=method, sparsity=sparsity, cdf_threshold=cdf_threshold,
                        audio_token_norms=audio_token_norms, valid_mask=valid_mask, lambda_a=lambda_a,
                        tau_128=tau_128, lambda_128=lambda_128, shape_ids=shape_ids,
                        compute_padded_queries=compute_padded_queries, input_grid=input_grid,
                        compact_lists=compact_lists)
    sm_scale = 1.0 / (q.shape[-1] ** 0.5)
    out = _DynBSA.apply(q, k, v, plan, sm_scale)
    if return_shape_ids:
        return out, plan.lay.shape_ids
    return out


__all__ = ["flash_attn_bsa_3d_dynamic", "plan_dynamic", "ALL_CANDIDATE_SHAPES"]
