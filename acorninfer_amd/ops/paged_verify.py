"""Speculative-verify attention over the paged cache.

Drop-in for acorninfer/ops/paged_verify.py (`paged_verify_attention`,
:96-123): the m = spec_num + 1 window positions of each sequence are scored
together, each with causal visibility inside the window. Row (b, j) sees
seq_lens[b] - (m - 1 - j) tokens (its history plus the window's first j + 1
tokens); seq_lens counts the whole window, and the window's k/v are already in
the pages (`PagedKVCache.scatter_verify`).

A window is a short prefill whose prefix is in the cache: it runs on the
query-tiled prefill kernel (`acorn_paged_prefill_attention_ws`), which reads a
sequence's K/V once for the whole window and divides a long context over
several workgroups. Rows stay independent as in K3: what a later token's V
holds, infinities and NaN included, reaches no earlier row. Eight windows of
five over 1024..8192 tokens take 41 us; as one K3 row per window token, the form
below, 109, each row reading the context for itself. Shapes the prefill kernel is not built for (fp32, head
sizes other than 64 / 128, pages under 16 tokens) and one-token windows, which
are decode, keep it: the window is flattened to B*m query rows and the
split/combine kernels of decode run over them.
"""
from __future__ import annotations

import torch

from acorninfer_amd._lib import check, dtype_code, lib, ptr, require_gpu, stream_ptr
from acorninfer_amd.ops.paged_attention import (paged_decode_attention, prefill_supported,
                                                prefill_workspace)

__all__ = ["paged_verify_attention"]


def paged_verify_attention(q: torch.Tensor, k_pages: torch.Tensor, v_pages: torch.Tensor,
                           tables: torch.Tensor, seq_lens: torch.Tensor,
                           num_splits: int) -> torch.Tensor:
    """q [B, m, H, D] (normed + roped, positions len .. len+m-1); k/v_pages
    [NB, P, KV, D] (read only); tables [B, MP] int32; seq_lens [B] int32 =
    len + m. Returns [B, m, H, D] in q.dtype: row j is the window-causal
    attention output at position len + j (a row that sees no token is NaN).
    num_splits applies to the K3 form; the prefill kernel plans its own. Shape
    contracts raise AssertionError as the reference's do (paged_verify.py:
    110-118)."""
    require_gpu(q, k_pages, v_pages, tables, seq_lens)
    B, M, H, D = q.shape
    NB, P, KV, _ = k_pages.shape
    assert M >= 1, "verify window must be non-empty"
    assert D & (D - 1) == 0 and P & (P - 1) == 0, "D and P must be power-of-2"
    assert H % KV == 0, "GQA requires H divisible by KV"
    assert num_splits >= 1
    assert v_pages.shape == k_pages.shape
    assert tables.shape[0] == B and seq_lens.shape[0] == B
    assert k_pages.is_contiguous() and v_pages.is_contiguous()
    assert tables.is_contiguous() and seq_lens.is_contiguous()
    assert tables.dtype == torch.int32 and seq_lens.dtype == torch.int32
    if M > 1 and B > 0 and prefill_supported(q.dtype, D, P, H, KV):
        assert k_pages.dtype == q.dtype == v_pages.dtype
        assert k_pages.shape[3] == D
        assert tables.shape[1] >= 1, "tables must hold at least one page per sequence"
        q2 = q.contiguous()
        out = torch.empty_like(q2)
        W = tables.shape[1]
        ws = prefill_workspace(B, B * M, M, H, KV, D, P, W, q.device)
        rc = lib().acorn_paged_prefill_attention_ws(
            ptr(q2), ptr(k_pages), ptr(v_pages), ptr(tables), None, ptr(seq_lens), None, ptr(out),
            B, B * M, M, H, KV, D, P, NB, W, float(D ** -0.5), dtype_code(q2), ptr(ws),
            0 if ws is None else ws.numel(), stream_ptr(q.device))
        check(rc, "paged_verify_attention")
        return out
    # row (b, j): sequence b's table, length seq_lens[b] - (m - 1 - j)
    row_tables = tables.repeat_interleave(M, dim=0)
    back = torch.arange(M - 1, -1, -1, device=seq_lens.device, dtype=torch.int32)
    row_lens = (seq_lens[:, None] - back[None, :]).reshape(-1).contiguous()
    out = paged_decode_attention(q.reshape(B * M, H, D), k_pages, v_pages, row_tables,
                                 row_lens, num_splits)
    return out.view(B, M, H, D)
