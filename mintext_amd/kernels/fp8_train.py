"""The blockwise-fp8 expert layer's training step as one autograd node.

The composition of ``moe_experts_forward_fp8_train`` (route, gate_up GEMM, SwiGLU, down GEMM, combine;
bzantium/mintext mintext/modules/moe.py:161-221) with the same codes, scales and products as its
separate steps, in which every operand is quantised by the kernel that makes it:

* tokens: quantised per token, gathered by the gate_up GEMM; their transposed codes for the weight
  gradient gathered from the tokens in the backward (no sorted copy);
* SwiGLU output and the gradients of both products' outputs: both codes from one pass, the bf16 SwiGLU
  output never written;
* weights: the forward's and the backward's codes from one read.

Between its passes the node holds the gate_up and down products, a copy of the tokens and, as far as
that is no more than what the separate steps hold, codes that the backward reads (``kept_codes``); the
rest is quantised again in the backward.  ``gate_up`` and ``down`` are saved for that, and for autograd's
check that they were not changed in place.
"""
from __future__ import annotations

import torch

from .. import _lib as L
from .fp8 import SCALE_MODES, _entry, quantize_fp8_rows, quantize_fp8_weights, quantize_fp8_weights_t, tgmm_fp8
from .moe_dispatch import _as_i32, _combine, route_indices

_ROWS, _GATHER, _SWIGLU = 0, 1, 2


def experts_fp8_train_supported(x, topk_indices, topk_weights, gate_up, down, scales) -> bool:
    """Whether ``experts_fp8_train`` takes these arguments: bf16 tokens, widths in tiles of 256,
    tokens aligned for 16-byte loads (a sorted copy of others is) and 32-bit operand offsets (the other
    forms, and what has to raise, take the separate steps)."""
    if scales not in SCALE_MODES or x.dtype != torch.bfloat16 or x.dim() != 2 or topk_indices.dim() != 2:
        return False
    if gate_up.dim() != 3 or down.dim() != 3 or gate_up.dtype != down.dtype:
        return False
    if gate_up.dtype not in (torch.bfloat16, torch.float32) or topk_weights.dtype not in (torch.bfloat16, torch.float32):
        return False
    if x.is_contiguous() and x.data_ptr() % 16:
        return False
    N, D = x.shape
    E, D2, two_i = gate_up.shape
    I = two_i // 2
    K = topk_indices.shape[1]
    if N < 1 or K < 1 or topk_indices.shape[0] != N or topk_weights.shape != topk_indices.shape or E > 1023:
        return False
    if D2 != D or two_i % 2 or tuple(down.shape) != (E, I, D) or D < 256 or I < 256 or D % 256 or I % 256:
        return False
    C = (N * K + 127) // 128 + E
    return max(D, two_i) * max(128 * C, N * K) < 2 ** 32 and D * two_i < 2 ** 32


def _weights(w, p2, both):
    """(forward codes, scales, dlhs codes, scales); the latter None unless ``both``."""
    dev = w.device
    if not both:
        return *quantize_fp8_weights(w, scales=SCALE_MODES[p2]), None, None
    w = w.contiguous()
    E, kin, kout = w.shape
    f8, f32 = torch.float8_e4m3fn, torch.float32
    wq = torch.empty((E, kout, kin), dtype=f8, device=dev)
    ws = torch.empty((E, kout // 128, kin // 128), dtype=f32, device=dev)
    wqt = torch.empty((E, kin, kout), dtype=f8, device=dev)
    wst = torch.empty((E, kin // 128, kout // 128), dtype=f32, device=dev)
    L.call("mtx_quant_fp8_weights_both", L.ptr(w), L.dtype_code(w.dtype), E, kin, kout, p2, L.ptr(wq), L.ptr(ws),
           L.ptr(wqt), L.ptr(wst), L.stream(dev))
    return wq, ws, wqt, wst


def kept_codes(N, K, D, I, E):
    """Which operands of the backward keep their codes from the forward: (SwiGLU output, gate_up, down).
    The others are made in the backward, from the copy of the tokens, the gate_up product and the weights,
    with the same bits.

    The separate steps hold the sorted tokens and the SwiGLU output in bf16, 2 M (D + I) bytes that this
    node does not; of those the copy of the tokens takes 2 N D.  Codes are kept while they fit the rest, in
    the order of what making them again costs, so that a layer never holds more between its passes than
    the separate steps.  Nor does it at its backward's peak, in the gate_up gradients: there the
    separate steps have given back the SwiGLU output but hold one more copy of the gate_up codes."""
    M = N * K
    left = 2 * D * (M - N) + 2 * I * min(M, E * D)
    kept = []
    chunk_rows = 128 * ((M + 127) // 128 + E)
    for size in (I * (chunk_rows + chunk_rows // 32), 2 * E * D * I, E * D * I):
        kept.append(size + size // 1024 <= left)
        left -= size + size // 1024 if kept[-1] else 0
    return kept


def _operands(source, a, row_index, div, M, F, E, blocks, p2, chunks, rows, grouped):
    """(row codes, row scales, transposed codes, transposed scales) of ``mtx_quant_fp8_operands``."""
    dev = a.device
    f8, f32 = torch.float8_e4m3fn, torch.float32
    rq = torch.empty((M, F), dtype=f8, device=dev) if rows else None
    rs = torch.empty((M, F // 128), dtype=f32, device=dev) if rows else None
    C = L.query("mtx_fp8_grouped_chunks", M, E)
    xt = torch.empty((F * 128 * C,), dtype=f8, device=dev) if grouped else None
    xts = torch.empty(((F // 128) * C if blocks else F * C,), dtype=f32, device=dev) if grouped else None
    L.call("mtx_quant_fp8_operands", source, L.ptr(a), L.ptr(row_index), div, a.shape[0], M, F, E, int(blocks), p2,
           L.ptr(rq), L.ptr(rs), L.ptr(xt), L.ptr(xts), L.ptr(chunks), L.stream(dev))
    return rq, rs, xt, xts


def _tile_list(M, E, dev):
    """Workspace of an fp8 product: the tile list, at its smallest tiles of 64 rows (the partial tiles that
    ``mtx_gmm_workspace_size`` has room for besides, 64 MB, are of the bf16 products)."""
    return L.workspace(256 + 16 * ((M + 63) // 64 + E + 1), dev)


def _gmm(entry, xq, xs, wq, ws, gs, M, kin, kout, E, cols):
    """One product of ``entry`` ([E, kin, kout] weights), ``cols`` output columns."""
    dev = xq.device
    out = torch.empty((M, cols), dtype=torch.bfloat16, device=dev)
    wsp = _tile_list(M, E, dev)
    L.call(entry, L.ptr(xq), L.ptr(xs), L.ptr(wq), L.ptr(ws), L.ptr(gs), M, kin, kout, E, L.ptr(out), L.ptr(wsp),
           wsp.numel(), L.stream(dev))
    return out


def _chunks(gs, M):
    ws = L.workspace(L.query("mtx_fp8_grouped_workspace_size", gs.numel()), gs.device)
    L.call("mtx_fp8_chunks", L.ptr(gs), M, gs.numel(), L.ptr(ws), ws.numel(), L.stream(gs.device))
    return ws


class _ExpertsFP8Train(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, topk_indices, topk_weights, gate_up, down, scales, grad):
        p2 = int(scales == "pow2")
        dev = L.require_device(x, topk_indices, topk_weights, gate_up, down)
        given, x = x, x.contiguous()
        N, D = x.shape
        K = topk_indices.shape[1]
        E, _, two_i = gate_up.shape
        I, M = two_i // 2, N * K
        need_x, _, _, need_dgu, need_ddn = (grad and n for n in ctx.needs_input_grad[:5])
        through = need_x or need_dgu  # the gradient goes on to the gate_up product
        keep_y, keep_gu, keep_dn = kept_codes(N, K, D, I, E)
        si, gs, inv = route_indices(_as_i32(topk_indices), E)
        xq, xs = quantize_fp8_rows(x, scales=scales)
        guq, gus, guqt, gust = _weights(gate_up, p2, need_x and keep_gu)
        h = torch.empty((M, two_i), dtype=torch.bfloat16, device=dev)
        wsp = _tile_list(M, E, dev)
        L.call("mtx_gmm_fp8_gathered", L.ptr(xq), L.ptr(xs), N, L.ptr(si), K, L.ptr(guq), L.ptr(gus), L.ptr(gs), M, D,
               two_i, E, p2, L.ptr(h), L.ptr(wsp), wsp.numel(), L.stream(dev))
        del xq, xs, guq, gus, wsp
        # without a gradient of h, its SwiGLU's codes are less than h
        keep_y = need_ddn and (keep_y or not through)
        yq, ys, yt, yts = _operands(_SWIGLU, h, None, 1, M, I, E, False, p2, _chunks(gs, M), True, keep_y)
        dnq, dns, dnqt, dnst = _weights(down, p2, through and keep_dn)
        out = _gmm(_entry("mtx_gmm_fp8", scales), yq, ys, dnq, dns, gs, M, I, D, E, D)
        del yq, ys, dnq, dns
        w = topk_weights.contiguous()
        res = _combine(out, inv, w, N, K, torch.result_type(out, w))
        # the tokens may be changed in place before the backward (the separate steps read their sorted copy)
        tokens = (x.clone() if x.data_ptr() == given.data_ptr() else x) if need_dgu else None
        ctx.save_for_backward(gate_up, down, w, h if through else None, out, inv, gs, guqt, gust, dnqt, dnst, tokens,
                              si if need_dgu else None, yt, yts)
        ctx.cfg = (N, K, D, I, E, scales, x.dtype)
        return res

    @staticmethod
    def backward(ctx, dout):
        gate_up, down, w, h, out, inv, gs, guqt, gust, dnqt, dnst, tokens, si, yt, yts = ctx.saved_tensors
        N, K, D, I, E, scales, x_dtype = ctx.cfg
        p2, M = int(scales == "pow2"), N * K
        need_x, _, need_w, need_dgu, need_ddn = ctx.needs_input_grad[:5]
        need_dgu, need_ddn = need_dgu and tokens is not None, need_ddn and (yt is not None or h is not None)
        dev = L.require_device(dout)
        dout = dout.contiguous()
        if dout.dtype not in (torch.float32, torch.bfloat16):
            dout = dout.float()
        dY = torch.empty_like(out)
        dw = torch.empty_like(w) if need_w else None
        L.call("mtx_unroute_bwd", L.ptr(dout), L.dtype_code(dout.dtype), L.ptr(out), L.dtype_code(out.dtype), L.ptr(inv),
               L.ptr(w), L.dtype_code(w.dtype), N, K, D, L.ptr(dY), L.ptr(dw), L.stream(dev))
        dx = dgu = ddn = None
        through = need_x or need_dgu  # the gradient goes on to the gate_up product
        if through or need_ddn:
            chunks = _chunks(gs, M)
            dyq, dys, dyt, dyts = _operands(_ROWS, dY, None, 1, M, D, E, True, p2, chunks, through, need_ddn)
            del dY
        # the peak of a backward: each operand is given back after its last reader, and the product that goes
        # on comes before the weight gradient
        if through:
            if dnqt is None:
                dnqt, dnst = quantize_fp8_weights_t(down, scales=scales)
            dinter = _gmm(_entry("mtx_gmm_fp8_dlhs", scales), dyq, dys, dnqt, dnst, gs, M, I, D, E, I)
            del dyq, dys, dnqt, dnst
        if need_ddn:
            if yt is None:
                _, _, yt, yts = _operands(_SWIGLU, h, None, 1, M, I, E, False, p2, chunks, False, True)
            ddn = tgmm_fp8(yt, yts, dyt, dyts, gs, M, I, D, scales=scales).to(down.dtype)
            del yt, yts, dyt, dyts
        if through:
            dh = torch.empty_like(h)
            L.call("mtx_swiglu_bwd", L.ptr(h), L.ptr(dinter), L.MTX_BF16, M, I, L.ptr(dh), L.stream(dev))
            del dinter
            dhq, dhs, dht, dhts = _operands(_ROWS, dh, None, 1, M, 2 * I, E, True, p2, chunks, need_x, need_dgu)
            del dh
            if need_x:
                if guqt is None:
                    guqt, gust = quantize_fp8_weights_t(gate_up, scales=scales)
                dsorted = _gmm(_entry("mtx_gmm_fp8_dlhs", scales), dhq, dhs, guqt, gust, gs, M, D, 2 * I, E, D)
                del dhq, dhs, guqt, gust
                dx = _combine(dsorted, inv, None, N, K, x_dtype)
                del dsorted
            if need_dgu:
                _, _, xt, xts = _operands(_GATHER, tokens, si, K, M, D, E, False, p2, chunks, False, True)
                dgu = tgmm_fp8(xt, xts, dht, dhts, gs, M, D, 2 * I, scales=scales).to(gate_up.dtype)
        return dx, None, dw, dgu, ddn, None, None


def experts_fp8_train(x, topk_indices, topk_weights, gate_up, down, scales: str):
    """[N, D] tokens -> [N, D] in result_type(bf16, topk_weights); see the module's docstring.
    Gradients reach x, topk_weights, gate_up and down."""
    return _ExpertsFP8Train.apply(x, topk_indices, topk_weights, gate_up, down, scales, torch.is_grad_enabled())
