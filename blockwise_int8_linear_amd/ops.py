"""Operator launchers with the reference's names, signatures and output layouts
(triton_functions.py:221-233, :492-500, :142-168), running hand-written gfx950 kernels through the
C ABI of libbi8.so.  Like the reference's launchers they allocate their outputs with torch.empty on the
input's device, enqueue on the current stream and return without synchronizing.

The calls themselves (allocation, operand checks, launch) are native code, ``_bi8_torch`` (csrc/bi8_torch.cpp).
There is one code path: device tensors, HIP kernels.  A CPU tensor trips the same assertion as in the
reference (``assert x.is_cuda``); a missing libbi8.so raises.
"""
from __future__ import annotations

import torch

from . import _lib
from . import block_linear_config

_DT = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


def ceil_div(n: int, d: int) -> int:
    return -(n // -d)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    """hipStream_t of torch's current stream on t's device (the raw getter is ~2 us cheaper than the Stream object)"""
    if _raw_stream is not None:
        return _raw_stream(t.device.index)
    return torch.cuda.current_stream(t.device).cuda_stream


class _NoGuard:
    def __enter__(self):
        return None

    def __exit__(self, *a):
        return False


_NO_GUARD = _NoGuard()
_multi_device = None


def _on_device(t: torch.Tensor):
    """Context that makes t's device current for the launch; free on a one-GPU machine."""
    global _multi_device
    if _multi_device is None:
        _multi_device = torch.cuda.device_count() > 1
    return torch.cuda.device(t.device) if _multi_device else _NO_GUARD


def _float_operand(x: torch.Tensor) -> torch.Tensor:
    if x.dtype not in _DT:
        raise TypeError(f"unsupported dtype {x.dtype}: expected float32, bfloat16 or float16")
    return x if x.stride(-1) == 1 or x.numel() == 0 else x.contiguous()


def _rows(x: torch.Tensor) -> torch.Tensor:
    """2-D tensor whose rows are contiguous (leading dimension = stride(0))."""
    if x.is_contiguous():
        return x
    if x.numel() and (x.stride(1) != 1 or (x.shape[0] > 1 and x.stride(0) < x.shape[1])):
        return x.contiguous()
    return x


def _ld(x: torch.Tensor) -> int:
    return x.stride(0) if x.shape[0] > 1 else max(x.shape[1], 1)


def _scales_out(s: torch.Tensor) -> torch.Tensor:
    t = block_linear_config.SHARED_EXP_TORCH_TYPE
    return s if t == torch.float32 else s.to(t)       # the reference's store casts to the scale dtype (:216, :227)


def quantize_block_rowwise(x: torch.Tensor, fblock_size=None):
    """x [M,K] -> (int8 codes [M,K], absmax scales [ceil(K/B), M]); triton_functions.py:221-233."""
    m, k = x.shape
    assert x.is_cuda
    return _lib.native().quantize_rowwise(x, fblock_size or block_linear_config.GROUP_SIZE, block_linear_config.SHARED_EXP_TORCH_TYPE)


def quantize_block_transposed(x: torch.Tensor, fblock_size=None):
    """Same result as ``quantize_block_rowwise(x.t().contiguous())`` (block_linear.py:93-94, :100-103) in one
    pass over x:  x [R,C] -> (int8 [C,R], scales [ceil(R/B), C])."""
    r, c = x.shape
    assert x.is_cuda
    return _lib.native().quantize_transposed(x, fblock_size or block_linear_config.GROUP_SIZE, block_linear_config.SHARED_EXP_TORCH_TYPE)


_FAST_BLOCKS = (32, 64, 128)


def _code_buffer(rows: int, cols: int, device, pad: bool):
    """int8 [rows, cols]; with `pad`, a view of a buffer whose rows are padded with zero codes to a multiple of 128
    (what the tiled GEMM kernels want of a contraction dimension), so that no padded copy is needed later"""
    if pad and cols % 128 != 0 and rows > 0 and cols > 0:
        ld = ceil_div(cols, 128) * 128
        store = torch.empty((rows, ld), device=device, dtype=torch.int8)
        store[:, cols:].zero_()
        return store[:, :cols], store
    t = torch.empty((rows, cols), device=device, dtype=torch.int8)
    return t, t


def _quantize_block_dual(x: torch.Tensor, fblock_size, pad: bool, colsum: bool = False):
    r, c = x.shape
    assert x.is_cuda
    x = _rows(_float_operand(x))
    pad = pad and fblock_size in _FAST_BLOCKS
    q, q_store = _code_buffer(r, c, x.device, pad)
    qt, qt_store = _code_buffer(c, r, x.device, pad)
    s = torch.empty((ceil_div(c, fblock_size), r), device=x.device, dtype=torch.float32)
    st = torch.empty((ceil_div(r, fblock_size), c), device=x.device, dtype=torch.float32)
    lib = _lib.load()
    if colsum:
        # the column sums of x from the same read (the bias gradient when x is the output gradient)
        sums = torch.empty((c,), device=x.device, dtype=x.dtype)
        ws = torch.empty((ceil_div(r, 128) * c,), device=x.device, dtype=torch.float32)
        with _on_device(x):
            rc = lib.bi8_quantize_dual_colsum(x.data_ptr(), _DT[x.dtype], q.data_ptr(), s.data_ptr(), qt.data_ptr(), st.data_ptr(),
                                              sums.data_ptr(), ws.data_ptr(), ws.numel() * 4, r, c, _ld(x), max(q_store.shape[1], 1),
                                              max(qt_store.shape[1], 1), fblock_size, _stream(x))
        _lib.check(rc, "bi8_quantize_dual_colsum")
        return q, _scales_out(s), qt, _scales_out(st), q_store, qt_store, sums
    with _on_device(x):
        rc = lib.bi8_quantize_dual(x.data_ptr(), _DT[x.dtype], q.data_ptr(), s.data_ptr(), qt.data_ptr(), st.data_ptr(),
                                   r, c, _ld(x), max(q_store.shape[1], 1), max(qt_store.shape[1], 1), fblock_size, _stream(x))
    _lib.check(rc, "bi8_quantize_dual")
    return q, _scales_out(s), qt, _scales_out(st), q_store, qt_store


def quantize_block_dual_colsum(x: torch.Tensor, fblock_size=None):
    """``quantize_block_dual(x)`` plus ``x.sum(dim=0)`` (fp32 accumulation, result in x's dtype) from the same pass
    over x: the output gradient's two quantizations and the bias gradient of block_linear.py:92, :101-103, :110.
    Returns (q, scales, qT, scalesT, column sums)."""
    out = _quantize_block_dual(x, fblock_size or block_linear_config.GROUP_SIZE, pad=False, colsum=True)
    return out[0], out[1], out[2], out[3], out[6]


def quantize_block_dual(x: torch.Tensor, fblock_size=None):
    """``quantize_block_rowwise(x)`` and ``quantize_block_transposed(x)`` from one pass over x:
    x [R,C] -> (int8 [R,C], scales [ceil(C/B), R], int8 [C,R], scales [ceil(R/B), C]), the same bits as the two calls.
    A training step needs both directions of X, W and G (block_linear.py:77-78, :92-94, :100-103)."""
    return _quantize_block_dual(x, fblock_size or block_linear_config.GROUP_SIZE, pad=False)[:4]


def dequantize_block_rowwise(x: torch.Tensor, state_x: torch.Tensor, fblock_size=None):
    """int8 [M,K] + scales [ceil(K/B), M] -> [M,K] of INPUT_OUTPUT_TORCH_TYPE; triton_functions.py:492-500."""
    assert x.is_cuda
    M, K = x.shape
    return _lib.native().dequantize(x, state_x, fblock_size or block_linear_config.GROUP_SIZE, block_linear_config.INPUT_OUTPUT_TORCH_TYPE)


def int8_matmul_block64_rowwise_dequantize(a, b, state_x, state_w, bias=None):
    """a int8 [M,K], b int8 [K,N] (any strides), state_x [K/B, M], state_w [K/B, N], bias [N] or None
    -> [M,N] of INPUT_OUTPUT_TORCH_TYPE; triton_functions.py:142-168.  B = GROUP_SIZE at call time.
    (b.t() with contiguous rows is what the kernels read and what the reference's callers pass, W_int8.t(),
    block_linear.py:80; anything else is copied into that layout once.)"""
    assert a.is_cuda and b.is_cuda
    assert a.dtype == torch.int8 and b.dtype == torch.int8, "operands must be int8 codes"
    assert a.shape[1] == b.shape[0], "incompatible dimensions"
    block = block_linear_config.GROUP_SIZE
    M, K = a.shape
    scratch = None
    if M > 16 or block == 32:
        # what the call runs: K padded to a multiple of 128, blocks of 256, 512, ... at 128
        lib, run_block = _lib.load(), 128 if block > 128 and block & (block - 1) == 0 else block
        scratch = _workspace(lib, M, b.shape[1], ceil_div(K, 128) * 128, run_block, a.device, _stream(a))[0]
    return _lib.native().gemm(a, b, state_x, state_w, bias, block, block_linear_config.INPUT_OUTPUT_TORCH_TYPE, scratch)


_ws_need = {}                       # (M, N, K, block) -> bytes of scratch memory the library's split of K wants (0: none)


def _workspace(lib, M, N, K, block, device, stream):
    """Scratch memory for a GEMM of fewer output tiles than compute units (the library then splits K over the
    workgroups and sums the pieces): (tensor or None, bytes).  What a shape wants is asked once; the memory (at most 48 MiB) is
    the call's own, from torch's allocator on the current stream: the split and its sum are two launches, and those of two
    threads that use one stream may be queued in between one another.
    (Up to 16 rows at blocks 64 / 128 run the one-pass decode kernels whatever they are given: not asked.)"""
    if M <= 16 and block != 32:
        return None, 0
    key = (M, N, K, block)
    need = _ws_need.get(key)
    if need is None:
        need = _ws_need[key] = lib.bi8_gemm_workspace_bytes(M, N, K, block)
    return (torch.empty(need, device=device, dtype=torch.uint8), need) if need else (None, 0)


_FEW_ROWS = 2
_FEW_ROWS_LDS = 64 * 1024


def _few_rows_lds(M: int, K: int, block: int, elem_bytes: int) -> int:
    """LDS bytes of the one-launch few-row kernel: scales of the K-blocks (whole 1 KiB runs of K plus one, in multiples
    of 16) for 4 + 16 rows, the activations' codes, 1 KiB of slack, the un-quantized activations"""
    return ceil_div((ceil_div(K, 1024) + 1) * (1024 // block), 16) * 16 * 80 + (1 if M <= 1 else 2) * K + 1024 + M * K * elem_bytes


def linear_few_rows(x, W_int8, state_W, bias=None):
    """``quantize_block_rowwise(x)`` followed by ``int8_matmul_block64_rowwise_dequantize(x_int8, W_int8.t(),
    state_x, state_W, bias)`` (BlockInt8Linear.infer, block_linear.py:141-144) as ONE kernel, for the few-row case of
    token-by-token decode: x [M,K] float with 1 <= M <= 2, W_int8 [N,K] and state_W [K/B, N] the cached weights.
    Returns the same bits as the two launchers, or None when the operands are outside what the fused kernel covers
    (the caller then runs the two launchers)."""
    plan = few_rows_plan(x, _rows(W_int8), state_W if state_W.is_contiguous() else state_W.contiguous(), bias)
    return None if plan is None else plan(_rows(x))


def few_rows_plan(x, W_int8, state_W, bias):
    """``linear_few_rows`` for activations of x's shape and dtype against these weights under the present
    ``block_linear_config``: ``call(x) -> output or None``, or None when the one-launch kernel does not cover the case.  The
    closure holds the tensors it was made from; make a new one when the weights' buffers, the bias or the configuration change."""
    block = block_linear_config.GROUP_SIZE
    dtype = block_linear_config.INPUT_OUTPUT_TORCH_TYPE
    K = x.shape[-1]
    M = x.numel() // K if K else 0
    N = W_int8.shape[0]
    if not (1 <= M <= _FEW_ROWS and block in (64, 128) and K > 0 and K % 128 == 0 and N > 0 and x.dtype == dtype
            and x.dtype in _DT and W_int8.dtype == torch.int8 and state_W.dtype == torch.float32
            and W_int8.stride(1) == 1 and state_W.is_contiguous() and _few_rows_lds(M, K, block, x.element_size()) <= _FEW_ROWS_LDS):
        return None
    assert x.is_cuda and W_int8.is_cuda
    assert W_int8.shape[1] == K and tuple(state_W.shape) == (K // block, N), "incompatible dimensions"
    few_rows = _lib.native().few_rows

    def call(x):
        return few_rows(x, W_int8, state_W, bias, block, dtype)

    return call


def int8_matmul_block_partials(a, b, fblock_size=None):
    """The GEMM kernel's int32 block partials, before any scaling: int32 [ceil(K/B), M, N]
    (what ``tl.dot`` yields at triton_functions.py:115).  Parity/debug operator."""
    block = fblock_size or block_linear_config.GROUP_SIZE
    assert a.is_cuda and b.is_cuda
    assert a.dtype == torch.int8 and b.dtype == torch.int8, "operands must be int8 codes"
    assert a.shape[1] == b.shape[0], "incompatible dimensions"
    a, w = _rows(a), _rows(b.t())
    M, K = a.shape
    N = w.shape[0]
    p = torch.empty((ceil_div(K, block), M, N), device=a.device, dtype=torch.int32)
    with _on_device(a):
        rc = _lib.load().bi8_gemm_nt_partials(a.data_ptr(), w.data_ptr(), p.data_ptr(), M, N, K, _ld(a), _ld(w),
                                              block, _stream(a))
    _lib.check(rc, "bi8_gemm_nt_partials")
    return p
