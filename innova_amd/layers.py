"""Host mirror of the decode-step pieces of Qwen35Engine around the quantized matmuls
(src/adapters/tools/qwen35_engine.cpp: rmsnorm :39-44, mlp_step :611-621, embedding lookup :756-760)."""
from __future__ import annotations

from . import _lib
from .weights import DeviceWeights


def rmsnorm(x, w, out=None):
    """out = x * r * (1 + w), r = 1 / sqrt(mean(x^2) + 1e-6), per row of a float32 cuda tensor [..., n]."""
    import torch
    assert x.is_cuda and w.is_cuda and x.dtype == torch.float32 and w.dtype == torch.float32 and x.is_contiguous()
    n = w.numel()
    rows = x.numel() // n
    if out is None:
        out = torch.empty_like(x)
    _lib.check(_lib.lib().oilhip_rmsnorm_f32(x.data_ptr(), w.data_ptr(), n, rows, out.data_ptr(), _lib.current_stream()))
    return out


def gemv_rmsnorm(w: DeviceWeights, x, norm_w, out=None):
    """y = W . rmsnorm(x; norm_w): the norm in front of a projection, formed inside the GEMV for one OIL4 row."""
    y = (_lib._native or _lib.native()).gemv_rmsnorm(w._h, x, norm_w, out, w.rows, w.cols)
    if y is not None:
        return y
    import torch
    assert x.is_cuda and x.dtype == torch.float32 and x.is_contiguous() and norm_w.is_cuda and norm_w.dtype == torch.float32
    M = w._rows(x, torch.float32)
    if out is None:
        out = x.new_empty((M, w.rows))
    # xn and the scratch of mlp_step go back to torch's allocator when these return, while the launches may still be queued:
    # the allocator hands a block out again in the order of the stream it came from, which is the stream they run on
    xn = torch.empty_like(x)
    args = w.handle, x.data_ptr(), norm_w.data_ptr(), out.data_ptr(), M, xn.data_ptr()
    ws = _lib.graph_workspace(M, w)
    if ws is not None:
        _lib.check(_lib.lib().oilhip_gemv_rmsnorm_f32_ws(*args, ws[0].data_ptr(), ws[1], _lib.current_stream()))
    else:
        _lib.check(_lib.lib().oilhip_gemv_rmsnorm_f32(*args, _lib.current_stream()))
    return out


def mlp_step(gate_up: DeviceWeights, down: DeviceWeights, x, out=None, norm_w=None):
    """y = down(siluf(gate x') * up x'), x' = rmsnorm(x; norm_w) or x; gate_up = the gate and up projections stacked
    (DeviceWeights.stack_rows)."""
    y = (_lib._native or _lib.native()).mlp_step(gate_up._h, down._h, x, norm_w, out, down.rows, gate_up.cols, down.cols)
    if y is not None:
        return y
    import torch
    assert x.is_cuda and x.dtype == torch.float32 and x.is_contiguous()
    M, F = gate_up._rows(x, torch.float32), down.cols
    if out is None:
        out = x.new_empty((M, down.rows))
    scratch = x.new_empty((3 * F + gate_up.cols) * M)
    args = (gate_up.handle, down.handle, x.data_ptr(), norm_w.data_ptr() if norm_w is not None else None, out.data_ptr(), M,
            scratch.data_ptr())
    ws = _lib.graph_workspace(M, gate_up, down)
    if ws is not None:
        _lib.check(_lib.lib().oilhip_mlp_step_f32_ws(*args, ws[0].data_ptr(), ws[1], _lib.current_stream()))
    else:
        _lib.check(_lib.lib().oilhip_mlp_step_f32(*args, _lib.current_stream()))
    return out


def embed_rows(w: DeviceWeights, ids, out=None):
    """Rows ids[i] of a quantized [vocab][cols] tensor decoded to float32 [n][cols]; ids: int32 cuda tensor."""
    if out is None:
        y = (_lib._native or _lib.native()).embed_rows(w._h, ids, w.cols)
        if y is not None:
            return y
    import torch
    assert ids.is_cuda and ids.dtype == torch.int32 and ids.is_contiguous()
    n = ids.numel()
    if out is None:
        out = torch.empty((n, w.cols), dtype=torch.float32, device=ids.device)
    _lib.check(_lib.lib().oilhip_embed_rows_f32(w.handle, ids.data_ptr(), n, out.data_ptr(), _lib.current_stream()))
    return out
