"""C = A @ B for the model's linear layers (the reference's kernel 3).

The reference writes its own tiled Triton GEMM (kernels/tiled_matmul.py) and
measures it against cuBLAS. On MI355X the plain library GEMM is hipBLASLt,
reached through torch.matmul; this module keeps the reference's entry point,
argument checks and AssertionErrors (kernels/tiled_matmul.py:135-140) so the
model code and the reference's tests call it unchanged. fp32 operands use
IEEE fp32 (torch's default, allow_tf32 off), as the reference's
input_precision="ieee" does.

Decode-time calls carry one row per sequence in the batch. There a GEMM is a
single pass over B's bytes, so bf16/fp16 products with M <= 2 go to the
library's skinny kernel (lsfa_gemv: one launch, a K-split pass over B at HBM
rate whose last workgroup per column block sums the fp32 partials and rounds
once), which hipBLASLt's general tiles reach at a fraction of the bandwidth.
From 3 to 32 rows, products whose widths are multiples of 128 run on a second
kernel that computes them on MFMA while W streams through registers, with the
SwiGLU activation formed as x is loaded. Measured on MI355X over the
LLaMA-3-8B decode projections at 8 and 32 rows (us, graph replays, weights
that no cache holds), this kernel against hipBLASLt: q/k/v 13.5 and 16.4
against 51.9 and 54.1, o 10.9 and 13.7 against 21.9 and 20.9, gate/up 42.3 and
46.2 against 56.1 and 56.8, down 23.1 and 27.2 against 71.0 and 61.4, LM head
165 and 177 against 190 and 198; so such products go to it, small single ones
above 8 rows apart (MFMA_MIN_*). Calls that
autograd, a tracer or autocast has to see stay on torch's operators at every
row count (_library_only). The norm
is folded into the launch at up to 2 rows only. Above 32 rows the same kernel
runs over blocks of 64 rows (lsfa_gemm_group) as long as the launch has at most
one tile of 64 x 128 per CU (GEMM_*); there it beats hipBLASLt's larger tiles
(figures in csrc/fa_gemv_mfma.hip), beyond that it loses to them.

Projections that share their input (a decoder's q/k/v, gate/up) go through
matmul_shared_input, which runs them as one lsfa_gemv_group launch over their
concatenated columns when they qualify for the skinny kernel.
add_rmsnorm_matmul_shared_input also folds the residual add + RMSNorm that
precedes such projections into that launch (the norm computed exactly as
fused_add_rmsnorm computes it).

lsfa_gemv's workspace carries arrival counters (its first
LSFA_GEMV_COUNTER_BYTES) that must start at zero and that every call leaves
at zero, so this module keeps one workspace per (device, stream), zeroes its
counter bytes once when it is created, and reuses it for every call on that
stream (stream order keeps the calls apart). Workspaces start at 16 MB, so
they rarely grow. A graph capture gets a workspace of its own, from the
graph's memory pool, whose fill it records: the graph clears its 256 KB of
counters before its first product on every replay, whatever ran before it, and
shares neither counters nor partials with eager calls or with another graph
that may run at the same time. (Captures share a stream: torch captures on one
default capture stream per device.) The cache is bounded: it holds one eager
workspace and the last capture's per stream, and at most MAX_CACHED_STREAMS
streams without a capture, the least recently used going first.
"""
import collections
import threading

import torch
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from .. import _lib

_interpreter = torch._C._functorch.peek_interpreter_stack
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_tracing = torch._C._get_tracing_state

SKINNY_MAX_ROWS = 32  # what lsfa_gemv takes (more than 8 rows: MFMA kernel only)
AUTO_MAX_ROWS = 2    # rows that every product (and the fused norm / SwiGLU inputs) routes to it
# From 3 to this many rows, products of up to this many columns in all, every
# matrix a multiple of 128 wide, run on the library's MFMA kernel.
MFMA_AUTO_ROWS = 32
MFMA_AUTO_MAX_COLS = 128 * (_lib.GEMV_COUNTER_BYTES // 64)
MFMA_MAX_STRIDE = 1 << 25  # of W's rows: 32 of them in a 31-bit byte offset
# A matrix by itself has to be large enough for the pass over it to outweigh the
# launch and the split's reduction (a group saves launches too, and runs from 256 x
# 256 on). Measured against hipBLASLt in us: up to 16 rows K of 1536 or 2.4 million
# elements (at 9 rows 768 x 768 6.5 against 5.3, 512 x 1024 6.2 against 4.2, 2048 x 512
# 7.2 against 7.8; up to 256 columns all the same); above 16 rows, where hipBLASLt is
# faster on them, 9.4 million (at 17 rows 5120 x 1024 14.6 against 11.2, 4096 x 2048 13.8
# against 11.2, 3072 x 3072 12.1 against 17.8). Up to 8 rows all go to the kernel.
MFMA_MIN_K, MFMA_MIN_ELEMS, MFMA_MIN_ELEMS_17 = 1536, 9 << 18, 9 << 20
# Above MFMA_AUTO_ROWS rows, lsfa_gemm_group runs launches of this many tiles of
# 64 x 128 whose K is at least GEMM_MIN_K or which group several matrices (a
# short K alone: 2048 -> 2048 at 128 rows 15.7 us against hipBLASLt's 12.6; few
# tiles: 4096 -> 1024 at 48 rows 19.0 against 14.6). Fewer than GEMM_FEW_TILES
# need more: a matrix by itself a K of 8192 or 2048 columns (4096 -> 1024 at 128 rows
# 19.2 against 16.3, 4096 -> 256 at 512 21.5 against 15.0; 8192 -> 1024 0.72 times
# hipBLASLt's time), two matrices a K of 1024 (512 -> 512 + 512 at 192 rows 11.2
# against 10.5). Over 64 rows and 8192 columns a matrix by itself is hipBLASLt's
# (4096 -> 14336 at 128 rows 44.4 against 41.7).
GEMM_MIN_TILES, GEMM_FEW_TILES, GEMM_MAX_TILES, GEMM_MIN_K = 16, 32, 256, 4096

MAX_CACHED_STREAMS = 8


class _Entry:
    __slots__ = ("buf", "captured", "graph_buf")

    def __init__(self):
        self.buf = None        # the workspace of eager calls
        self.captured = 0      # the last graph capture on the stream (lsfa_capture_id)
        self.graph_buf = None  # its workspace


# (device index, stream handle) -> _Entry, least recently used first
_workspaces = collections.OrderedDict()
_workspaces_lock = threading.Lock()


def _workspace(device, stream, nbytes):
    with _workspaces_lock:
        return _workspace_locked(device, stream, nbytes)


def _workspace_locked(device, stream, nbytes):
    key = (device.index, stream)
    entry = _workspaces.pop(key, None) or _Entry()
    capture = _lib.capture_id(stream) if torch.cuda.is_current_stream_capturing() else 0
    if capture and entry.captured != capture:
        entry.captured, entry.graph_buf = capture, None
    buf = entry.graph_buf if capture else entry.buf
    if buf is None or buf.numel() < nbytes:
        buf = torch.empty(max(nbytes, 16 << 20), dtype=torch.uint8, device=device)
        buf[:_lib.GEMV_COUNTER_BYTES].zero_()
        if capture:
            entry.graph_buf = buf
        else:
            entry.buf = buf
    _workspaces[key] = entry
    while len(_workspaces) > MAX_CACHED_STREAMS:
        victim = next((k for k, e in _workspaces.items() if not e.captured), None)
        if victim is None:
            break
        del _workspaces[victim]
    return buf


def release_workspaces():
    """Frees every cached skinny-GEMM workspace. (Those that captured graphs
    recorded live in the graphs' own memory pools.)"""
    with _workspaces_lock:
        _workspaces.clear()


def _skinny_ok(a: torch.Tensor, b: torch.Tensor, max_rows: int = SKINNY_MAX_ROWS) -> bool:
    ok = (a.shape[0] <= max_rows and a.dtype in (torch.bfloat16, torch.float16)
          and a.stride(1) == 1 and b.stride(1) == 1 and b.shape[1] % 8 == 0
          and b.stride(0) % 8 == 0 and b.stride(0) >= b.shape[1] and b.data_ptr() % 16 == 0)
    if ok and a.shape[0] > 8:  # the MFMA kernel's conditions
        ok = (b.shape[1] % 128 == 0 and a.shape[1] % 8 == 0 and a.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0)
    return ok


def skinny_matmul(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """C = A @ B for a [M <= 32, K], b [K, N] (bf16/fp16, N % 8 == 0, rows of
    b 16-byte aligned) through lsfa_gemv; fp32 accumulation, one rounding."""
    assert _skinny_ok(a, b), ("skinny_matmul needs M <= 8 (or up to 32 with N % 128 == 0 and 16-byte aligned a "
                              "rows), bf16/fp16, unit column strides, N % 8 == 0")
    assert a.shape[1] == b.shape[0] and a.dtype == b.dtype and a.is_cuda and b.is_cuda, (
        "a [M, K] and b [K, N] must share K, dtype and device")
    M, K = a.shape
    N = b.shape[1]
    if out is None:
        out = torch.empty(M, N, dtype=a.dtype, device=a.device)
    assert out.shape == (M, N) and out.dtype == a.dtype and out.is_cuda and out.stride(1) == 1, (
        "out must be [M, N] in a's dtype with unit column stride")
    if M == 0 or N == 0:
        return out
    if K == 0:
        return out.zero_()
    args = _lib.GemvArgs(x=a.data_ptr(), w=b.data_ptr(), y=out.data_ptr(), workspace=None, workspace_bytes=0,
                         x_stride=a.stride(0), w_stride=b.stride(0), y_stride=out.stride(0),
                         dtype=_lib.TORCH_TO_LSFA[a.dtype], m=M, k=K, n=N)
    nbytes = _lib.gemv_workspace_size(args)
    with _lib.device_guard(a.device):
        stream = _lib.current_stream(a.device)
        if nbytes:
            ws = _workspace(a.device, stream, nbytes)
            args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
        _lib.gemv(args, stream)
    return out


_ZEROS = (0, 0, 0, 0)


def _group_args(a, bs, outs, gate=None, norm=(0, 0, 0, 0, 0, 0.0)):
    """lsfa_gemv_group_args of [a @ b for b in bs] into outs, no workspace yet;
    norm: (weight, residual, residual_out, their strides, eps)."""
    pad = _ZEROS[len(bs):]
    return _lib.pack(
        _lib.GemvGroupArgs, a.data_ptr(), 0, 0, a.stride(0), *((0, 0) if gate is None else (gate.data_ptr(), gate.stride(0))),
        *[b.data_ptr() for b in bs], *pad, *[o.data_ptr() for o in outs], *pad, *[b.stride(0) for b in bs], *pad,
        *[o.stride(0) for o in outs], *pad, *[b.shape[1] for b in bs], *pad, _lib.TORCH_TO_LSFA[a.dtype], a.shape[0],
        a.shape[1], len(bs), *norm, 0)


def _run_group(args, device, size=_lib.gemv_group_workspace_size, launch=_lib.gemv_group):
    nbytes = size(args)
    with _lib.device_guard(device):
        stream = _lib.current_stream(device)
        if nbytes:
            ws = _workspace(device, stream, nbytes)
            args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
        launch(args, stream)


def _empty_outs(a, bs):
    return [torch.empty(a.shape[0], b.shape[1], dtype=a.dtype, device=a.device) for b in bs]


def skinny_matmul_group(a: torch.Tensor, bs, outs=None, gate: torch.Tensor = None):
    """[a @ b for b in bs] for up to four b sharing a (each as for
    skinny_matmul) in one lsfa_gemv_group launch. With gate (a's shape and
    dtype), the products read F.silu(gate) * a instead of a, rounded as torch
    rounds it."""
    assert 1 <= len(bs) <= _lib.GEMV_MAX_GROUP, f"1..{_lib.GEMV_MAX_GROUP} matrices per group"
    assert gate is None or (gate.shape == a.shape and gate.dtype == a.dtype and gate.stride(1) == 1), (
        "gate must match a's shape and dtype, with unit column stride")
    assert all(_skinny_ok(a, b) and b.shape[0] == a.shape[1] and b.dtype == a.dtype for b in bs), (
        "every matrix must qualify for skinny_matmul with the shared input")
    M, K = a.shape
    assert a.is_cuda and all(b.is_cuda for b in bs), "GPU tensors expected"
    if outs is None:
        outs = [torch.empty(M, b.shape[1], dtype=a.dtype, device=a.device) for b in bs]
    assert len(outs) == len(bs) and all(
        o.shape == (M, b.shape[1]) and o.dtype == a.dtype and o.is_cuda and o.stride(1) == 1 for o, b in zip(outs, bs)), (
        "outs must be [M, N_i] in a's dtype with unit column stride")
    if M == 0 or sum(b.shape[1] for b in bs) == 0:
        return outs
    if K == 0:
        return [o.zero_() for o in outs]
    _run_group(_group_args(a, bs, outs, gate), a.device)
    return outs


def _sizes_fit(rows: int, k: int, cols) -> bool:
    """Whether products of these sizes (rows and columns of a, columns of each
    b) are routed to a kernel of the library, if nothing else is against it.
    Arithmetic only, and asked first: a call that stays on torch anyway is short
    enough (5 us at 64 rows of 1024 x 1024) for the other tests to show. (Sizes
    that a tracer passes are symbols: no test of them becomes a guard.)"""
    if torch.compiler.is_compiling():
        return False
    if rows <= AUTO_MAX_ROWS:
        return True
    total = 0
    for n in cols:
        if n % 128:
            return False
        total += n
    if k % 8:
        return False
    alone = len(cols) == 1
    if rows <= MFMA_AUTO_ROWS:
        if alone and rows > 16:
            return MFMA_MIN_ELEMS_17 <= k * total <= k * MFMA_AUTO_MAX_COLS
        return total <= MFMA_AUTO_MAX_COLS and (not alone or rows <= 8 or total <= 256 or k >= MFMA_MIN_K
                                                or k * total >= MFMA_MIN_ELEMS)
    tiles = total // 128 * ((rows + 63) // 64)
    if tiles < GEMM_MIN_TILES or tiles > GEMM_MAX_TILES:
        return False
    if alone:
        return (k >= GEMM_MIN_K and (tiles >= GEMM_FEW_TILES or k >= 2 * GEMM_MIN_K or total >= 2048)
                and (rows <= 64 or total <= 8192))
    return tiles >= GEMM_FEW_TILES or k >= 1024 or len(cols) > 2


def _library_only(*tensors) -> bool:
    """Whether a call on these tensors has to go through torch's own operators:
    a gradient is recorded (reverse or forward mode), a subclass, mode or
    transform looks at the operators, autocast to another type is on, or one
    is sparse. (A default device is a mode too, but one that only places new
    tensors.) To be asked before anything reads an address or a stride: what a
    transform or tracer passes has no address, a sparse tensor neither."""
    if torch.compiler.is_compiling():
        return True
    grad = torch.is_grad_enabled()
    for t in tensors:
        kind = type(t)
        if ((kind is not torch.Tensor and kind is not torch.nn.Parameter) or (grad and t.requires_grad)
                or t.layout is not torch.strided):
            return True
    return (forward_ad._current_level >= 0 or _interpreter() is not None or _dispatch_modes() > 0
            or (_function_modes() > 0 and any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()))
            or _tracing() is not None
            or (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != tensors[0].dtype))


def _mfma_ok(a: torch.Tensor, bs) -> bool:
    """Whether the MFMA kernel takes these products (beyond _skinny_ok)."""
    return (AUTO_MAX_ROWS < a.shape[0] <= MFMA_AUTO_ROWS and sum(b.shape[1] for b in bs) <= MFMA_AUTO_MAX_COLS
            and all(_skinny_ok(a, b) and b.shape[1] % 128 == 0 and b.stride(0) <= MFMA_MAX_STRIDE for b in bs)
            and a.shape[1] % 8 == 0 and _rows_addressable(a) and a.stride(0) >= a.shape[1])


def _auto_skinny(a: torch.Tensor, bs) -> bool:
    """Whether matmul / matmul_shared_input route these products, which are not
    _library_only, to the skinny kernels (see AUTO_MAX_ROWS and MFMA_AUTO_*)."""
    if not (len(bs) <= _lib.GEMV_MAX_GROUP and a.ndim == 2 and a.is_cuda and all(
            b.ndim == 2 and b.device == a.device and b.dtype == a.dtype and b.shape[0] == a.shape[1] for b in bs)):
        return False
    if a.shape[0] <= AUTO_MAX_ROWS:
        return all(_skinny_ok(a, b, AUTO_MAX_ROWS) for b in bs)
    return _mfma_ok(a, bs)


def _skinny_run(a: torch.Tensor, bs):
    """skinny_matmul_group where _auto_skinny holds (its conditions are checked)."""
    if 0 in a.shape or sum(b.shape[1] for b in bs) == 0:
        return skinny_matmul_group(a, bs)
    outs = _empty_outs(a, bs)
    _run_group(_group_args(a, bs, outs), a.device)
    return outs


def _gemm_ok(a: torch.Tensor, bs) -> bool:
    """Whether lsfa_gemm_group takes these products, which are not
    _library_only, and is the faster route."""
    return (len(bs) <= _lib.GEMV_MAX_GROUP and a.ndim == 2 and a.is_cuda and a.shape[0] > MFMA_AUTO_ROWS
            and a.dtype in (torch.bfloat16, torch.float16) and a.shape[1] > 0 and a.shape[1] % 8 == 0
            and _rows_addressable(a) and a.shape[1] <= a.stride(0) <= 1 << 23 and all(
                b.ndim == 2 and b.device == a.device and b.dtype == a.dtype and b.shape[0] == a.shape[1]
                and b.shape[1] % 128 == 0 and b.shape[1] > 0 and _rows_addressable(b)
                and b.shape[1] <= b.stride(0) <= MFMA_MAX_STRIDE for b in bs)
            and _sizes_fit(*a.shape, [b.shape[1] for b in bs]))


def _gemm_group(a: torch.Tensor, bs):
    """[a @ b for b in bs] through lsfa_gemm_group (_gemm_ok holds)."""
    outs = _empty_outs(a, bs)
    _run_group(_group_args(a, bs, outs), a.device, _lib.gemm_group_workspace_size, _lib.gemm_group)
    return outs


def matmul_shared_input(a: torch.Tensor, bs):
    """[matmul(a, b) for b in bs]: one grouped launch when the products
    qualify for the library's kernels together, else one matmul each."""
    if (a.ndim == 2 and all(b.ndim == 2 for b in bs) and _sizes_fit(*a.shape, [b.shape[1] for b in bs])
            and not _library_only(a, *bs)):
        if _auto_skinny(a, bs):
            return _skinny_run(a, bs)
        if _gemm_ok(a, bs):
            return _gemm_group(a, bs)
    return [matmul(a, b) for b in bs]


def swiglu_matmul(gate: torch.Tensor, up: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """matmul(F.silu(gate) * up, b), the activation folded into the skinny
    kernels' load of their input when the product qualifies for them."""
    if (gate.ndim == 2 and gate.shape[0] <= MFMA_AUTO_ROWS and gate.shape == up.shape
            and gate.dtype == up.dtype == b.dtype and gate.is_cuda and up.device == gate.device and b.device == gate.device and b.ndim == 2 and b.shape[0] == up.shape[1]
            and not _library_only(gate, up, b)
            and gate.stride(1) == 1 and (_skinny_ok(up, b, AUTO_MAX_ROWS) or (
                _mfma_ok(up, [b]) and _rows_addressable(gate) and gate.stride(0) >= gate.shape[1]))):
        return skinny_matmul_group(up, [b], gate=gate)[0]
    return matmul(torch.nn.functional.silu(gate) * up, b)


def _rows_addressable(t: torch.Tensor) -> bool:
    return t.stride(-1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0


def add_rmsnorm_matmul_shared_input(x, residual, weight, eps, bs, write_residual=True):
    """(outs, h) for h = x + residual (x alone when residual is None) and
    outs = [matmul(rmsnorm(h) * weight, b) for b in bs], the norm as
    fused_add_rmsnorm computes it. Products of at most AUTO_MAX_ROWS rows run
    as one skinny launch that also forms the norm (and writes h, when
    write_residual and residual is given); others run fused_add_rmsnorm (or
    rmsnorm) then matmul_shared_input. h is residual's replacement, as from
    fused_add_rmsnorm, or x itself when residual is None."""
    from .fused_rmsnorm_residual import fused_add_rmsnorm, rmsnorm
    assert x.ndim == 2 and weight.ndim == 1 and weight.shape[0] == x.shape[1], "x [M, K] and weight [K] expected"
    M, K = x.shape
    fused = (len(bs) <= _lib.GEMV_MAX_GROUP and x.is_cuda and x.dtype in (torch.bfloat16, torch.float16)
             and M <= AUTO_MAX_ROWS and not _library_only(x, weight, *bs, *(() if residual is None else (residual,)))
             and weight.device == x.device and (residual is None or residual.device == x.device)
             and K % 8 == 0 and _rows_addressable(x) and weight.is_contiguous() and weight.data_ptr() % 16 == 0
             and weight.dtype == x.dtype and (residual is None or (residual.shape == x.shape and residual.dtype == x.dtype
                                                                   and _rows_addressable(residual)))
             and all(b.ndim == 2 and b.device == x.device and b.dtype == x.dtype and b.shape[0] == K
                     and _skinny_ok(x, b, AUTO_MAX_ROWS) for b in bs))
    if not fused:
        normed, h = (fused_add_rmsnorm(x, residual, weight, eps) if residual is not None
                     else (rmsnorm(x, weight, eps), x))
        return matmul_shared_input(normed, bs), h
    h = torch.empty_like(x) if (residual is not None and write_residual) else None
    outs = [torch.empty(M, b.shape[1], dtype=x.dtype, device=x.device) for b in bs]
    if M == 0:
        return outs, (h if residual is not None else x)
    _run_group(_group_args(x, bs, outs, norm=(
        weight.data_ptr(), residual.data_ptr() if residual is not None else 0, h.data_ptr() if h is not None else 0,
        residual.stride(0) if residual is not None else 0, h.stride(0) if h is not None else 0, float(eps))), x.device)
    return outs, (h if residual is not None else x)


def matmul(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """C = A @ B. a: [M, K], b: [K, N], same dtype, both on the GPU."""
    assert a.ndim == 2 and b.ndim == 2, f"expected 2D matrices, got {a.ndim}D and {b.ndim}D"
    assert a.shape[1] == b.shape[0], f"inner dims must match: a is {tuple(a.shape)}, b is {tuple(b.shape)}"
    assert a.is_cuda and b.is_cuda, "the gfx950 path needs GPU tensors"
    assert a.dtype == b.dtype, f"dtype mismatch: a={a.dtype} b={b.dtype}"
    if _sizes_fit(*a.shape, b.shape[1:]) and not _library_only(a, b):
        if _auto_skinny(a, [b]):
            return _skinny_run(a, [b])[0]
        if _gemm_ok(a, [b]):
            return _gemm_group(a, [b])[0]
    return torch.matmul(a, b)
