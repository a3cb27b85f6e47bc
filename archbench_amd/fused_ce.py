"""Chunked linear + cross-entropy that never materialises the full (N, V) logits, on MI355X.

Same interface and arithmetic as archbench/fused_ce.py:20-57 (``fused_linear_cross_entropy(x, target, weight,
num_chunks=8, ignore_index=-100)`` -> mean token cross-entropy; the forward computes every gradient and the
backward only scales them).  Per pass of rows: logits = x W^T and the two gradient products dx = dlogits W,
dW += dlogits^T x (fp32 accumulation) are plain library GEMMs (hipBLASLt through torch); between them one HIP kernel
(``ops.cross_entropy_fwd_bwd_``) computes each row's loss and overwrites the logits with
dloss * (softmax - onehot), reading and writing the chunk once.  ``num_chunks`` bounds the memory: a pass takes the
rows of one chunk and as many more as fit in the room that the accumulation in place saves (_rows_per_pass).  With
288 GB of HBM even one chunk for 32768 tokens (3.3 GB of logits) is cheap to hold; with one pass the weight gradient
comes straight out of one GEMM in the weight's dtype, the fastest configuration on MI355X.
"""

from __future__ import annotations

import torch

from . import _lib, ops


def fused_ce_available() -> bool:
    """True when the HIP library is built (the kernel path has no fallback)."""
    try:
        _lib.load()
    except _lib.GDNLibraryError:
        return False
    return True


_KERNEL_DTYPES = (torch.bfloat16, torch.float32)
_TILE = 256  # rows and columns of the GEMMs' output tiles


def _rows_per_pass(N: int, num_chunks: int, d: int, es: int) -> int:
    """Rows per pass: a chunk's ceil(N / num_chunks), plus what fits in the memory a second fp32 copy of dW [V, d] would
    take (an accumulation out of place held one): two thirds of it as logits [rows, V] of es bytes, the last third left
    for dx's partial products (_dx_split).  Every pass reads and writes dW once and runs products of its rows' size:
    N = 8192, d = 1024, V = 50304 in eight passes of 1024 rows took 6.2 ms (dx on 80 of 256 CUs, 72 us a pass copying
    dW), in four of 2048 3.3 ms."""
    C = -(-N // num_chunks)
    if C >= N:
        return max(N, 1)
    most = C + 8 * d // (3 * es)
    rows = -(-N // -(-N // most))
    return min(most, -(-rows // _TILE) * _TILE, N)


def _dx_split(rows: int, d: int, V: int) -> int:
    """Parts of the contraction over V in dx = dlogits W: as one product it has rows/256 x d/256 output tiles for 256
    CUs (rows 2048, d 1024: 32, 308 us); in S parts, batched and summed in fp32, S times as many (S = 8: 197 us).  The
    parts hold whole 16-byte pieces of a row and take at most a third of dW's fp32 size."""
    if rows == 0:
        return 1
    tiles = -(-rows // _TILE) * -(-d // _TILE)
    S = min(256 // tiles, V // (3 * rows), 16)
    while S > 1 and V % (8 * S):
        S -= 1
    return max(S, 1)


# Below this a call that takes dx in parts and scales by the HIP pass waits for its launches, not for its kernels (measured
# 314 to 330 us, at N 128 to 1024 and V 32000 and 50304; without the two 215 to 263, at V 8192).
_HOST_US = 320


def _outlasts_host(N: int, d: int, V: int) -> bool:
    """Whether a call's kernels take longer than its launches, so that extra calls which shorten them pay.  In us: dx's
    product in one part (its chain over V alone takes about 3.5 ns a class while the tiles leave CUs idle: V 8192, 32000
    and 50304 at 128 to 1024 rows 15 to 45, 97 to 175 and 146 to 242; in the parts of _dx_split 13 to 35, 28 to 91 and
    35 to 118), 6 N d V operations at 0.6 PFLOP/s, and the passes over W's size with torch's scaling of its gradient.
    By this count and measured, without / with the two: N 128 to 1024 at V 8192 43 to 146, 252 / 345 us; N 210, d 768, V
    32000 262, 278 / 318; N 1024, d 512, V 32000 345, 350 / 258 to 334; N 128, d 1024, V 50304 448, 420 / 289 to 324."""
    return 3.5e-3 * V + V * d * (1e-8 * N + 4e-6) > _HOST_US


def _dx(dlogits: torch.Tensor, weight: torch.Tensor, out: torch.Tensor | None, parts: bool) -> torch.Tensor:
    """dlogits [rows, V] W [V, d], written to ``out`` if given; with ``parts`` in parts where that can be done."""
    rows, V = dlogits.shape
    d = weight.shape[1]
    # 16-byte rows throughout; not under an autocast that would change a dtype, nor into the gradient of an x laid out
    # feature by feature (dx has x's strides)
    parts = (parts and dlogits.dtype == weight.dtype == torch.bfloat16 and d % 8 == 0 and weight.is_contiguous()
             and (out is None or (out.dtype == torch.bfloat16 and out.is_contiguous())))
    S = _dx_split(rows, d, V) if parts else 1
    if S == 1:
        return dlogits @ weight if out is None else out.copy_(dlogits @ weight)
    if out is None:
        out = dlogits.new_empty(rows, d)
    products = torch.bmm(dlogits.view(rows, S, V // S).transpose(0, 1), weight.view(S, V // S, d),
                         out_dtype=torch.float32)
    ops.sum_parts_(products, out)
    return out


def _scaled(t: torch.Tensor, s: torch.Tensor, hip: bool) -> torch.Tensor:
    """s t for a 0-d s, the product in fp32 and rounded once.  The HIP pass (``hip``) runs at the copy rate, 41 us for 64M
    bf16 elements and 2.9 for 4M where torch's product with a 0-d tensor takes 163 and 13.6 (with a 1-d one 19 for 25M,
    HIP 15), but as an op it costs the host 20 us more in a backward."""
    if t.dtype not in (torch.bfloat16, torch.float32):  # an fp16 weight under autocast
        return t * s
    if hip and t.numel() >= 1 << 22 or torch.is_grad_enabled():
        return ops.scaled(t, s)
    # a 1-d s, which takes part in the type promotion: torch rounds a 0-d one to t's dtype first
    try:
        return torch.mul(t, s.reshape(1), out=torch.empty_like(t))
    except RuntimeError:  # a batch of factors (is_grads_batched), which out= does not take; a second pass otherwise
        return (t * s.reshape(1)).to(t.dtype)


class _FusedLinearCE(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, target, weight, num_chunks: int, ignore_index: int):
        N, d = x.shape
        C = _rows_per_pass(N, num_chunks, d, x.element_size())
        outlasts = ctx.outlasts_host = _outlasts_host(N, d, weight.shape[0])
        total = target.ne(ignore_index).sum().clamp_min(1)
        dloss = total.float().reciprocal().reshape(1)  # device scalar: no host sync
        if C >= N:
            logits = x @ weight.t()
            loss_rows = ops.cross_entropy_fwd_bwd_(logits, target, dloss, ignore_index)[0]
            dx = _dx(logits, weight, None, outlasts).to(x.dtype)
            if num_chunks == 1 or logits.dtype == weight.dtype:
                # dW needs no accumulation across passes, so the GEMM writes it in the weight's dtype directly (fp32
                # accumulation inside, one rounding -- where several passes round at the end)
                dw = logits.t() @ x
            else:  # under autocast an fp32 weight's gradient over several chunks keeps its fp32 sums, also in one pass
                dw = torch.mm(logits.t(), x.to(logits.dtype), out_dtype=torch.float32)
        else:
            loss_rows = torch.empty(N, device=x.device, dtype=torch.float32)
            dx, dw = torch.empty_like(x), None
            for s in range(0, N, C):
                e = min(s + C, N)
                c_x = x[s:e]
                logits = c_x @ weight.t()
                loss_rows[s:e] = ops.cross_entropy_fwd_bwd_(logits, target[s:e], dloss, ignore_index)[0]
                _dx(logits, weight, dx[s:e], outlasts)
                if dw is None:
                    dw = torch.mm(logits.t(), c_x, out_dtype=torch.float32)
                else:  # in place
                    torch.addmm(dw, logits.t(), c_x, out_dtype=torch.float32, out=dw)
                del logits
        ctx.save_for_backward(dx, dw.to(weight.dtype))
        return loss_rows.sum() / total

    @staticmethod
    def backward(ctx, dout):
        dx, dw = ctx.saved_tensors
        return _scaled(dx, dout, ctx.outlasts_host), None, _scaled(dw, dout, ctx.outlasts_host), None, None


def fused_linear_cross_entropy(x, target, weight, num_chunks: int = 8, ignore_index: int = -100):
    """x (B, T, H), target (B, T), weight (V, H) -> mean token cross-entropy (fused_ce.py:55-57)."""
    return _FusedLinearCE.apply(x.reshape(-1, x.shape[-1]), target.reshape(-1), weight, num_chunks, ignore_index)
