"""Batched fused entry points of the verify-and-sample path.

These are the chain-of-k versions of the reference's per-position rules:
the reference verifies one position per pipeline lane and prunes every
descendant of a rejected lane (sglang_recurrent/loopspec/pipeline.py:365-412),
which, over k draft positions, is exactly an accept-prefix scan.
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib


def _check_rows(t: torch.Tensor, what: str) -> None:
    _lib.require_cuda(t, what)
    if t.stride(-1) != 1:
        raise ValueError(f"{what}: the vocabulary axis must be contiguous")


def argmax_rows(logits: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """Row-wise argmax of CUDA logits [M, V] with torch.argmax tie/NaN rules.

    Returns int64 [M]. Replaces torch.argmax in GreedyDecisionPolicy.queue
    (sglang_recurrent/loopspec/decisions.py:116).
    """
    _check_rows(logits, "argmax")
    if logits.dim() != 2:
        raise ValueError("argmax_rows expects [rows, vocab] logits")
    rows, vocab = logits.shape
    if out is None:
        out = torch.empty(rows, dtype=torch.int64, device=logits.device)
    elif out.shape != (rows,) or out.dtype != torch.int64 or not out.is_contiguous():
        raise ValueError("argmax_rows: out must be contiguous int64 [rows]")
    nbytes = _lib.query("ls_argmax_rows_workspace", rows, vocab)
    ws = _lib.WORKSPACE.get(logits.device, nbytes, "argmax", keep=_status_header_bytes())
    _lib.call(
        "ls_argmax_rows", logits.data_ptr(), _lib.dtype_code(logits), rows, vocab, logits.stride(0),
        out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream(logits.device),
    )
    return out


def lm_head_argmax(hidden: torch.Tensor, weight: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """Greedy token of each row straight from the hidden states: argmax_n of
    hidden [M, H] @ weight[V, H]^T (bf16, fp32 accumulation), one fused pass
    that never writes the [M, V] logits.

    Returns int64 [M]. Replaces the vocabulary head's logits
    (sglang_recurrent/modeling/components.py:175-194) followed by torch.argmax
    in GreedyDecisionPolicy.queue (sglang_recurrent/loopspec/decisions.py:116).
    A row whose two largest logits lie within fp32 accumulation rounding may
    return either index.
    """
    _lib.require_cuda(hidden, "lm_head_argmax")
    _lib.require_cuda(weight, "lm_head_argmax")
    if hidden.dim() != 2 or weight.dim() != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError("lm_head_argmax expects hidden [M, H] and weight [V, H]")
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("lm_head_argmax: bf16 hidden states and weight only")
    if hidden.stride(1) != 1 or weight.stride(1) != 1:
        raise ValueError("lm_head_argmax: the hidden axis must be contiguous")
    rows, h = hidden.shape
    vocab = weight.shape[0]
    if out is None:
        out = torch.empty(rows, dtype=torch.int64, device=hidden.device)
    elif out.shape != (rows,) or out.dtype != torch.int64 or not out.is_contiguous():
        raise ValueError("lm_head_argmax: out must be contiguous int64 [rows]")
    nbytes = _lib.query("ls_lm_head_argmax_workspace", rows, vocab)
    ws = _lib.WORKSPACE.get(hidden.device, nbytes, "lm_head")
    _lib.call(
        "ls_lm_head_argmax", hidden.data_ptr(), hidden.stride(0), weight.data_ptr(), weight.stride(0),
        _lib.dtype_code(hidden), rows, h, vocab, out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream(hidden.device),
    )
    return out


def lm_head_logits(hidden: torch.Tensor, weight: torch.Tensor, out: torch.Tensor | None = None,
                   dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """The vocabulary head's logits [M, V] (float32 or bf16) from hidden [M, H]
    and weight [V, H] (bf16, fp32 MFMA accumulation): the logits producer of
    sglang_recurrent/modeling/components.py:175-194 for the rows that sample.
    `out` may be a row-strided view (e.g. [B, k+1, V] target positions)."""
    _lib.require_cuda(hidden, "lm_head_logits")
    _lib.require_cuda(weight, "lm_head_logits")
    if hidden.dim() != 2 or weight.dim() != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError("lm_head_logits expects hidden [M, H] and weight [V, H]")
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("lm_head_logits: bf16 hidden states and weight only")
    if hidden.stride(1) != 1 or weight.stride(1) != 1:
        raise ValueError("lm_head_logits: the hidden axis must be contiguous")
    rows, h = hidden.shape
    vocab = weight.shape[0]
    if out is None:
        out = torch.empty((rows, vocab), dtype=dtype, device=hidden.device)
    if out.dim() != 2 or out.shape != (rows, vocab) or out.stride(1) != 1:
        raise ValueError("lm_head_logits: out must be [rows, vocab] with a contiguous vocabulary axis")
    if out.dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("lm_head_logits: float32 or bf16 logits only")
    _lib.call(
        "ls_lm_head_logits", hidden.data_ptr(), hidden.stride(0), weight.data_ptr(), weight.stride(0),
        _lib.dtype_code(hidden), rows, h, vocab, out.data_ptr(), out.stride(0), _lib.dtype_code(out),
        _lib.stream(hidden.device),
    )
    return out


def lm_head_greedy_verify(hidden: torch.Tensor, weight: torch.Tensor, k: int,
                          draft_tokens: torch.Tensor | None = None, *, accept_len: torch.Tensor | None = None,
                          tokens: torch.Tensor | None = None,
                          row_argmax: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """greedy_verify from the hidden states: the head's argmax of every endpoint
    row (as lm_head_argmax) and the accept-prefix scan, without logits.

    hidden [B * rpg, H] bf16, rows ordered (b, j): the k + 1 target positions,
    then, when draft_tokens [B, k] is not given, the k draft positions. Returns
    (accept_len int32 [B], tokens int64 [B, k+1]) as greedy_verify does.
    Replaces the vocabulary head's logits (components.py:175-194) and the
    greedy final-endpoint rule (decisions.py:116, 157-170) along the accept
    prefix (pipeline.py:365-412).
    """
    _lib.require_cuda(hidden, "lm_head_greedy_verify")
    _lib.require_cuda(weight, "lm_head_greedy_verify")
    if hidden.dim() != 2 or weight.dim() != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError("lm_head_greedy_verify expects hidden [B * rows, H] and weight [V, H]")
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("lm_head_greedy_verify: bf16 hidden states and weight only")
    if hidden.stride(1) != 1 or weight.stride(1) != 1:
        raise ValueError("lm_head_greedy_verify: the hidden axis must be contiguous")
    if not 1 <= k <= 64:
        raise ValueError("lm_head_greedy_verify: need 1 <= k <= 64")
    rpg = k + 1 if draft_tokens is not None else 2 * k + 1
    rows, h = hidden.shape
    if rows % rpg != 0:
        raise ValueError(f"lm_head_greedy_verify: {rows} rows are not whole groups of {rpg}")
    batch = rows // rpg
    vocab = weight.shape[0]
    dev = hidden.device
    if draft_tokens is not None:
        _lib.require_cuda(draft_tokens, "lm_head_greedy_verify")
        if draft_tokens.shape != (batch, k):
            raise ValueError("lm_head_greedy_verify: draft_tokens must be [B, k]")
        draft_tokens = draft_tokens.to(torch.int64).contiguous()
    if accept_len is None:
        accept_len = torch.empty(batch, dtype=torch.int32, device=dev)
    if tokens is None:
        tokens = torch.empty((batch, k + 1), dtype=torch.int64, device=dev)
    if accept_len.shape != (batch,) or accept_len.dtype != torch.int32 or not accept_len.is_contiguous():
        raise ValueError("lm_head_greedy_verify: accept_len must be contiguous int32 [B]")
    if tokens.shape != (batch, k + 1) or tokens.dtype != torch.int64 or not tokens.is_contiguous():
        raise ValueError("lm_head_greedy_verify: tokens must be contiguous int64 [B, k+1]")
    if row_argmax is not None and (row_argmax.shape != (batch, rpg) or row_argmax.dtype != torch.int64
                                   or not row_argmax.is_contiguous()):
        raise ValueError("lm_head_greedy_verify: row_argmax must be contiguous int64 [B, rows per element]")
    ws = _lib.WORKSPACE.get(dev, _lib.query("ls_lm_head_argmax_workspace", rows, vocab), "lm_head")
    _lib.call(
        "ls_lm_head_greedy_verify", hidden.data_ptr(), hidden.stride(0), weight.data_ptr(), weight.stride(0),
        _lib.dtype_code(hidden), batch, k, h, vocab, _lib.ptr(draft_tokens), accept_len.data_ptr(),
        tokens.data_ptr(), _lib.ptr(row_argmax), ws.data_ptr(), ws.numel(), _lib.stream(dev),
    )
    return accept_len, tokens


def greedy_verify(
    target_logits: torch.Tensor,
    draft_logits: torch.Tensor | None = None,
    draft_tokens: torch.Tensor | None = None,
    *,
    accept_len: torch.Tensor | None = None,
    tokens: torch.Tensor | None = None,
    row_argmax: torch.Tensor | None = None,
    workspace: torch.Tensor | None = None,
    check: bool = False,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Greedy chain verification in one launch.

    target_logits: [B, k+1, V]; draft_logits: [B, k, V] (same dtype) or
    draft_tokens: int64 [B, k]. Returns (accept_len int32 [B], tokens int64
    [B, k+1]); tokens[b, :accept_len+1] are the target argmaxes (accepted
    drafts then the correction/bonus token), the rest are -1. If row_argmax
    (int64 [B, 2k+1]) is given it receives every row's argmax. With
    check=True the call waits for the launch and raises RuntimeError when the
    workspace's status word reports a key poll that timed out (the outputs are
    then not valid); the default leaves the launch asynchronous and the check
    to check_greedy_status.
    """
    _check_rows(target_logits, "greedy_verify")
    if target_logits.dim() != 3:
        raise ValueError("target_logits must be [B, k+1, V]")
    batch, kp1, vocab = target_logits.shape
    k = kp1 - 1
    if k < 1:
        raise ValueError("greedy_verify needs at least one draft position")
    dev = target_logits.device
    if draft_logits is not None:
        _check_rows(draft_logits, "greedy_verify")
        if draft_logits.shape != (batch, k, vocab) or draft_logits.dtype != target_logits.dtype:
            raise ValueError("draft_logits must be [B, k, V] with the target's dtype")
        d_ptr, d_bs, d_ps = draft_logits.data_ptr(), draft_logits.stride(0), draft_logits.stride(1)
        tok_ptr = None
    else:
        if draft_tokens is None:
            raise ValueError("greedy_verify needs draft_logits or draft_tokens")
        if draft_tokens.shape != (batch, k) or draft_tokens.dtype != torch.int64:
            raise ValueError("draft_tokens must be int64 [B, k]")
        draft_tokens = draft_tokens.contiguous()
        d_ptr, d_bs, d_ps, tok_ptr = None, 0, 0, draft_tokens.data_ptr()
    # a step is a few microseconds of kernel: only what the caller passed is checked
    if accept_len is None:
        accept_len = torch.empty(batch, dtype=torch.int32, device=dev)
    elif accept_len.shape != (batch,) or accept_len.dtype != torch.int32 or not accept_len.is_contiguous():
        raise ValueError("accept_len must be contiguous int32 [B]")
    if tokens is None:
        tokens = torch.empty((batch, kp1), dtype=torch.int64, device=dev)
    elif tokens.shape != (batch, kp1) or tokens.dtype != torch.int64 or not tokens.is_contiguous():
        raise ValueError("tokens must be contiguous int64 [B, k+1]")
    if row_argmax is not None and (
        row_argmax.shape != (batch, 2 * k + 1) or row_argmax.dtype != torch.int64 or not row_argmax.is_contiguous()
    ):
        raise ValueError("row_argmax must be contiguous int64 [B, 2k+1]")
    ws = workspace if workspace is not None else _lib.WORKSPACE.get(
        dev, _lib.query("ls_greedy_verify_workspace", batch, k, vocab), "greedy", keep=_status_header_bytes())
    _lib.call(
        "ls_greedy_verify",
        target_logits.data_ptr(), target_logits.stride(0), target_logits.stride(1),
        d_ptr, d_bs, d_ps, tok_ptr,
        _lib.dtype_code(target_logits), batch, k, vocab,
        accept_len.data_ptr(), tokens.data_ptr(), _lib.ptr(row_argmax),
        ws.data_ptr(), ws.numel(), _lib.stream(dev),
    )
    if check:
        check_greedy_status(dev, ws)
    return accept_len, tokens


def _status_header_bytes() -> int:
    """Bytes of a greedy workspace up to and including its status word (the
    part a grown workspace keeps)."""
    return _lib.query("ls_greedy_status_offset") + 4


def greedy_status_word(workspace: torch.Tensor) -> torch.Tensor | None:
    """int32 view of the sticky status word of an argmax / greedy-verify
    workspace, or None for a workspace too small to hold one (no launch with
    split rows used it). Bit 0 (LS_GREEDY_KEY_TIMEOUT): a split's key did not
    become visible within the kernel's poll limit, so rows of the launches since
    the word was last cleared may be wrong."""
    off = _lib.query("ls_greedy_status_offset")
    if workspace.numel() < off + 4:
        return None
    return workspace[off:off + 4].view(torch.int32)


def check_greedy_status(device: torch.device | str, workspace: torch.Tensor | None = None) -> None:
    """Wait for the device's stream and raise RuntimeError if the status word
    of `workspace` (default: the argmax and greedy-verify workspaces cached for
    the device) is set; the word and the workspace's key slots are cleared, so
    later launches read normally."""
    device = torch.device(device)
    spaces = [workspace] if workspace is not None else [
        _lib.WORKSPACE.get(device, 0, tag) for tag in ("argmax", "greedy")]
    for ws in spaces:
        if greedy_status_word(ws) is None:
            continue
        status = ctypes.c_uint32(0)
        _lib.call("ls_greedy_workspace_status", ws.data_ptr(), ws.numel(), ctypes.addressof(status),
                  _lib.stream(device))
        if status.value:
            raise RuntimeError(f"greedy argmax: a split key was not visible within the poll limit "
                               f"(status {status.value:#x}); the results of these launches are not valid")


def greedy_verify_workspace_bytes(batch: int, k: int, vocab: int) -> int:
    return _lib.query("ls_greedy_verify_workspace", batch, k, vocab)


def _history_args(history: torch.Tensor | None, history_len: torch.Tensor | None, groups: int, dev):
    if history is None:
        return None, 0, None
    _lib.require_cuda(history, "repetition penalty history")
    if history.dtype != torch.int32 or history.dim() != 2 or history.stride(-1) != 1 or history.shape[0] < groups:
        raise ValueError("history must be int32 [rows, L] with contiguous ids")
    if history_len is None:
        history_len = torch.full((history.shape[0],), history.shape[1], dtype=torch.int32, device=dev)
    if history_len.dtype != torch.int32 or not history_len.is_contiguous() or history_len.shape[0] < groups:
        raise ValueError("history_len must be contiguous int32 [rows]")
    return history.data_ptr(), history.stride(0), history_len.data_ptr()


def speculative_verify(
    target_logits: torch.Tensor,
    draft_logits: torch.Tensor,
    draft_tokens: torch.Tensor,
    uniforms: torch.Tensor,
    temperature: float = 1.0,
    top_p: float = 1.0,
    *,
    penalty: float = 1.0,
    history: torch.Tensor | None = None,
    history_len: torch.Tensor | None = None,
    top_k: int = 0,
    accept_len: torch.Tensor | None = None,
    tokens: torch.Tensor | None = None,
    workspace: torch.Tensor | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Lossless speculative verification of a chain of k draft positions.

    target_logits [B, k+1, V] and draft_logits [B, k, V] (same dtype), draft
    tokens int64 [B, k] (sampled from the filtered draft distributions),
    uniforms float32 [B, 2k+1]: u[:, i] accept position i, u[:, k+i] the residual
    draw after a rejection at i, u[:, 2k] the bonus draw. Returns
    (accept_len int32 [B], tokens int64 [B, k+1]); see ls_spec_verify.
    """
    _check_rows(target_logits, "speculative_verify")
    _check_rows(draft_logits, "speculative_verify")
    if target_logits.dim() != 3:
        raise ValueError("target_logits must be [B, k+1, V]")
    batch, kp1, vocab = target_logits.shape
    k = kp1 - 1
    dev = target_logits.device
    if draft_logits.shape != (batch, k, vocab) or draft_logits.dtype != target_logits.dtype:
        raise ValueError("draft_logits must be [B, k, V] with the target's dtype")
    if draft_tokens.shape != (batch, k) or draft_tokens.dtype != torch.int64:
        raise ValueError("draft_tokens must be int64 [B, k]")
    if uniforms.shape != (batch, 2 * k + 1) or uniforms.dtype != torch.float32:
        raise ValueError("uniforms must be float32 [B, 2k+1]")
    draft_tokens = draft_tokens.contiguous()
    uniforms = uniforms.contiguous()
    if accept_len is None:
        accept_len = torch.empty(batch, dtype=torch.int32, device=dev)
    if tokens is None:
        tokens = torch.empty((batch, kp1), dtype=torch.int64, device=dev)
    h_ptr, h_stride, hl_ptr = _history_args(history, history_len, batch, dev) if penalty != 1.0 else (None, 0, None)
    nbytes = _lib.query("ls_spec_verify_workspace", batch, k, vocab)
    ws = workspace if workspace is not None else _lib.WORKSPACE.get(dev, nbytes, "spec")
    _lib.call(
        "ls_spec_verify",
        target_logits.data_ptr(), target_logits.stride(0), target_logits.stride(1),
        draft_logits.data_ptr(), draft_logits.stride(0), draft_logits.stride(1),
        draft_tokens.data_ptr(), uniforms.data_ptr(), _lib.dtype_code(target_logits),
        batch, k, vocab, float(temperature), float(top_p), int(top_k), float(penalty),
        h_ptr, h_stride, hl_ptr, accept_len.data_ptr(), tokens.data_ptr(),
        ws.data_ptr(), ws.numel(), _lib.stream(dev),
    )
    return accept_len, tokens


def stream_read_probe(target_logits: torch.Tensor, draft_logits: torch.Tensor, out: torch.Tensor | None = None
                      ) -> torch.Tensor:
    """Read-ceiling calibration (ls_stream_read_probe): reads greedy_verify's
    rows with its kernel's grid and loads and keeps only an exclusive-or of
    the words (int32, one per wave). Its duration bounds greedy_verify's from
    below."""
    _check_rows(target_logits, "stream_read_probe")
    _check_rows(draft_logits, "stream_read_probe")
    batch, kp1, vocab = target_logits.shape
    k = kp1 - 1
    words = _lib.query("ls_stream_read_probe_words", batch, k)
    if out is None:
        out = torch.zeros(words, dtype=torch.int32, device=target_logits.device)  # words past the grid stay 0
    _lib.call(
        "ls_stream_read_probe",
        target_logits.data_ptr(), target_logits.stride(0), target_logits.stride(1),
        draft_logits.data_ptr(), draft_logits.stride(0), draft_logits.stride(1),
        _lib.dtype_code(target_logits), batch, k, vocab, out.data_ptr(), out.numel(),
        _lib.stream(target_logits.device),
    )
    return out


def spec_verify_workspace_bytes(batch: int, k: int, vocab: int) -> int:
    return _lib.query("ls_spec_verify_workspace", batch, k, vocab)


def sample_logits(
    logits: torch.Tensor,
    uniforms: torch.Tensor,
    temperature: float = 1.0,
    top_p: float = 1.0,
    *,
    penalty: float = 1.0,
    history: torch.Tensor | None = None,
    history_len: torch.Tensor | None = None,
    top_k: int = 0,
    out: torch.Tensor | None = None,
) -> torch.Tensor:
    """Filter each row of logits [R, V] and draw one token per row (int64 [R])."""
    _check_rows(logits, "sample_logits")
    if logits.dim() != 2:
        raise ValueError("logits must be [rows, vocab]")
    rows, vocab = logits.shape
    dev = logits.device
    if uniforms.shape != (rows,) or uniforms.dtype != torch.float32:
        raise ValueError("uniforms must be float32 [rows]")
    uniforms = uniforms.contiguous()
    if out is None:
        out = torch.empty(rows, dtype=torch.int64, device=dev)
    h_ptr, h_stride, hl_ptr = _history_args(history, history_len, rows, dev) if penalty != 1.0 else (None, 0, None)
    ws = _lib.WORKSPACE.get(dev, _lib.query("ls_sample_logits_workspace", rows, vocab), "sample")
    _lib.call(
        "ls_sample_logits", logits.data_ptr(), logits.stride(0), _lib.dtype_code(logits), rows, vocab,
        float(temperature), float(top_p), int(top_k), float(penalty), h_ptr, h_stride, hl_ptr,
        uniforms.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream(dev),
    )
    return out


def filter_logits(
    logits: torch.Tensor,
    temperature: float = 1.0,
    top_p: float = 1.0,
    *,
    top_p_rows: torch.Tensor | None = None,
    top_k: int = 0,
    want_probs: bool = False,
    want_filtered: bool = True,
) -> dict[str, torch.Tensor]:
    """Dense filtering of logits [R, V]; returns a dict with 'filtered' (new
    float32 [R, V]), optionally 'probs' (unfiltered softmax), 'cutoff' and
    'mass' (float32 [R])."""
    _check_rows(logits, "filter_logits")
    if logits.dim() != 2:
        raise ValueError("logits must be [rows, vocab]")
    rows, vocab = logits.shape
    dev = logits.device
    res: dict[str, torch.Tensor] = {
        "cutoff": torch.empty(rows, dtype=torch.float32, device=dev),
        "mass": torch.empty(rows, dtype=torch.float32, device=dev),
    }
    if want_probs:
        res["probs"] = torch.empty((rows, vocab), dtype=torch.float32, device=dev)
    if want_filtered:
        res["filtered"] = torch.empty((rows, vocab), dtype=torch.float32, device=dev)
    if top_p_rows is not None:
        if top_p_rows.dtype != torch.float32 or top_p_rows.numel() < rows:
            raise ValueError("top_p_rows must be float32 with at least one entry per row")
        top_p_rows = top_p_rows.reshape(-1).contiguous()
    probs, filt = res.get("probs"), res.get("filtered")
    ws = _lib.WORKSPACE.get(dev, _lib.query("ls_filter_logits_workspace", rows, vocab), "filter")
    _lib.call(
        "ls_filter_logits", logits.data_ptr(), logits.stride(0), _lib.dtype_code(logits), rows, vocab,
        float(temperature), float(top_p), _lib.ptr(top_p_rows), int(top_k),
        _lib.ptr(probs), probs.stride(0) if probs is not None else 0,
        _lib.ptr(filt), filt.stride(0) if filt is not None else 0,
        res["cutoff"].data_ptr(), res["mass"].data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream(dev),
    )
    return res
