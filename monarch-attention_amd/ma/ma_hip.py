"""Host side of the HIP implementation: marshals torch tensors into the C ABI.

``monarch_attention_hip`` has the signature of the reference's implementation
functions (``MonarchAttentionFn``, ma/monarch_attention.py:11-13; the torch
one is ``monarch_attention_torch``, ma/ma_torch.py:65-73):

    fn(q, k, v, attn_mask, T, B, pre_pad) -> Tensor

q, k ``(E, H, N, D)``; v ``(E, H, N, Dv)`` (its dtype is the output dtype and
may differ from q/k, as in ``get_matrix``); ``attn_mask`` ``(E, N)`` bool /
int / float, truthy = keep, or ``None``.  Inputs may be arbitrary strided views
with a contiguous last dimension (models pass permuted ``(E, N, H, D)``
buffers); nothing is padded or copied on the host - the kernels apply the
reference's zero padding (ma/ma_torch.py:81-86) by index arithmetic and write
only the N real rows.  PyTorch provides the device buffers (output, workspace)
and the stream; all arithmetic happens in libma_hip.so, and the way from tensors
to its parameter blocks is native as well (csrc/ma_host.cpp).
"""
from __future__ import annotations

import os

import torch

from . import _hip_lib as L

Tensor = torch.Tensor

_DTYPES = {torch.float32: L.MA_F32, torch.float16: L.MA_F16, torch.bfloat16: L.MA_BF16}
_MASK_DTYPES = {torch.bool: L.MA_MASK_U8, torch.uint8: L.MA_MASK_U8, torch.int8: L.MA_MASK_U8, torch.int16: L.MA_MASK_I16,
                torch.int32: L.MA_MASK_I32, torch.int64: L.MA_MASK_I64, torch.float16: L.MA_MASK_F16,
                torch.bfloat16: L.MA_MASK_BF16, torch.float32: L.MA_MASK_F32, torch.float64: L.MA_MASK_F64}

# default variant of monarch_attention_hip; tests and the benchmark switch it
# per call through the `variant` keyword
DEFAULT_VARIANT = "auto"

# Does this process own the GPU while its forward calls run - no other stream,
# thread or process competing for compute units?  Only then may 'auto' resolve
# to the 'fused' kernel, whose workgroups wait for each other and so must all be
# on the device together (MA_FLAG_DEVICE_EXCLUSIVE).  Off unless the environment
# says MA_HIP_DEVICE_EXCLUSIVE=1 or the application sets this attribute; 'auto'
# then stays with kernels that make progress beside any other work.
DEVICE_EXCLUSIVE = os.environ.get("MA_HIP_DEVICE_EXCLUSIVE", "") not in ("", "0")

# extra ma_fwd_params.flags for the failure-path tests (MA_FLAG_TEST_NO_SPIN)
_TEST_FLAGS = 0


def _load_host():
    """lib/_ma_host.so (csrc/ma_host.cpp), bound to the library the ctypes layer has loaded and checked."""
    import importlib.machinery
    import importlib.util

    L.load()
    path = L.host_path()
    if not os.path.exists(path):
        raise ImportError(f"_ma_host.so not found at {path}: build it with `python monarch-attention_amd/build.py`")
    loader = importlib.machinery.ExtensionFileLoader("_ma_host", path)
    host = importlib.util.module_from_spec(importlib.util.spec_from_loader("_ma_host", loader))
    loader.exec_module(host)
    host.bind(L.library_path())
    return host


class _LazyHost:
    """Loads the extension at the first call: importing the package needs no built library."""

    def __getattr__(self, name):
        global _HOST
        _HOST = _load_host()
        return getattr(_HOST, name)


_HOST = _LazyHost()


def sync_status() -> int:
    """The sticky error word of the one-launch kernels, over all cached
    workspaces (synchronises the device): 0 = every wait between workgroups was
    satisfied; 1 = a bounded wait ran out (results of that call are invalid);
    2 = a producer ran on another XCD than its consumer (the device does not
    deal workgroup ids to XCDs the way the one-launch kernels are built on)."""
    worst = 0
    for buf in _HOST.workspaces():
        torch.cuda.synchronize(buf.device)
        worst = max(worst, int(buf[4:8].view(torch.int32).item()))
    return worst


def clear_workspace_cache() -> None:
    """Drop the cached per-stream workspaces (frees their device memory once the
    work queued on them is complete)."""
    _HOST.clear()


def _check_inputs(q: Tensor, k: Tensor, v: Tensor, attn_mask, T: int, B: int) -> None:
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor, got {type(t).__name__}")
        if t.dim() != 4:
            raise ValueError(f"{name} must have shape (E, H, N, D), got {tuple(t.shape)}")
    if q.shape != k.shape:
        raise ValueError(f"q and k must have the same shape, got {tuple(q.shape)} and {tuple(k.shape)}")
    if v.shape[:3] != q.shape[:3]:
        raise ValueError(f"v must share (E, H, N) with q, got {tuple(v.shape)} vs {tuple(q.shape)}")
    if q.dtype != k.dtype:
        raise TypeError(f"q and k must have the same dtype, got {q.dtype} and {k.dtype}")
    if q.dtype not in _DTYPES or v.dtype not in _DTYPES:
        raise TypeError(f"supported dtypes are float32, float16, bfloat16; got q {q.dtype}, v {v.dtype}")
    if not (q.device == k.device == v.device):
        raise ValueError("q, k and v must be on the same device")
    if min(q.shape) < 1 or v.shape[-1] < 1:
        raise ValueError(f"empty tensors are not supported, got q {tuple(q.shape)}, v {tuple(v.shape)}")
    if not isinstance(B, int) or B < 1:
        raise ValueError(f"block size B must be a positive int, got {B!r}")
    if not isinstance(T, int) or T < 1:
        raise ValueError(f"number of steps T must be a positive int, got {T!r}")
    if attn_mask is not None:
        if attn_mask.shape != (q.shape[0], q.shape[2]):
            raise ValueError(f"attn_mask must have shape (E, N) = {(q.shape[0], q.shape[2])}, "
                             f"got {tuple(attn_mask.shape)}")
        if attn_mask.device != q.device:
            raise ValueError("attn_mask must be on the same device as q")
    if q.device.type != "cuda":
        raise ValueError(f"the 'hip' implementation needs tensors on a GPU, got {q.device}")


def make_params(q: Tensor, k: Tensor, v: Tensor, mask_u8, out: Tensor, T: int, B: int, pre_pad: bool,
                variant: str = "auto", eps: float = 1e-12) -> L.FwdParams:
    """Fill a ``ma_fwd_params`` (workspace fields left empty)."""
    if variant not in L.VARIANTS:
        raise ValueError(f"unknown variant {variant!r}; available: {', '.join(L.VARIANTS)}")
    E, H, N, D = q.shape
    p = L.FwdParams()
    p.q, p.k, p.v, p.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    p.mask = mask_u8.data_ptr() if mask_u8 is not None else None
    p.mask_dtype = _MASK_DTYPES[mask_u8.dtype] if mask_u8 is not None else L.MA_MASK_U8
    p.E, p.H, p.N, p.D, p.Dv = E, H, N, D, v.shape[-1]
    p.B, p.T, p.pre_pad = B, T, int(bool(pre_pad))
    p.dtype_qk, p.dtype_v = _DTYPES[q.dtype], _DTYPES[v.dtype]
    p.variant = L.VARIANTS[variant]
    for name, t in (("q_stride", q), ("k_stride", k), ("v_stride", v), ("out_stride", out)):
        s = t.stride()
        setattr(p, name, (L.C.c_int64 * 3)(s[0], s[1], s[2]))
    if mask_u8 is not None:
        p.mask_stride = (L.C.c_int64 * 2)(*mask_u8.stride())
    p.eps = eps
    return p


def _variant_code(variant: str | None) -> int:
    code = L.VARIANTS.get(variant or DEFAULT_VARIANT)
    if code is None:
        raise ValueError(f"unknown variant {variant or DEFAULT_VARIANT!r}; available: {', '.join(L.VARIANTS)}")
    return code


def _flags() -> int:
    return _TEST_FLAGS | L.MA_FLAG_DEVICE_EXCLUSIVE if DEVICE_EXCLUSIVE else _TEST_FLAGS


def _refused(q, k, v, attn_mask, T, B):
    """The host extension did not take these arguments: raise what is wrong with them."""
    _check_inputs(q, k, v, attn_mask, T, B)
    if attn_mask is not None and attn_mask.dtype not in _MASK_DTYPES:
        raise TypeError(f"attn_mask dtype {attn_mask.dtype} is not supported")
    raise ValueError(f"T = {T} and B = {B} must fit 32 bits")


def monarch_attention_hip(q: Tensor, k: Tensor, v: Tensor, attn_mask: Tensor | None, T: int, B: int,
                          pre_pad: bool, *, variant: str | None = None, keep_state: bool = True) -> Tensor:
    """MonarchAttention forward on the current HIP stream; returns a new
    ``(E, H, N, Dv)`` tensor of ``v.dtype`` in v's memory layout (contiguous for
    contiguous v; backed by ``(E, N, H, Dv)`` when v is such a permuted view).
    Differentiable with respect to q, k and v: when one of them requires grad
    (and grad mode is on) the call is recorded as one autograd node that keeps
    the states of the steps and whose backward is ``ma_bwd_kept``.  The states
    are saved tensors like q, k and v (2T - 1 of q's size and one of v's).
    ``keep_state=False`` keeps none of them: the forward then runs as an
    unrecorded call does, the LDS-resident kernels included, and the backward
    runs the steps again - for callers who need the memory, or who leave grad
    mode on where no backward follows.  (A module takes it as an implementation:
    ``register_impl("hip_lean", functools.partial(monarch_attention_hip,
    keep_state=False))``.)  There is no forward-mode derivative: dual tensors raise ``NotImplementedError``.

    The one-launch kernels wait for each other's workgroups with bounded waits:
    a call whose wait ran out is reported by a RuntimeError from the first later
    call on the same stream that finds its error word set."""
    out = _HOST.forward(q, k, v, attn_mask, T, B, pre_pad, _variant_code(variant), _flags(), keep_state)
    if out is None:
        _refused(q, k, v, attn_mask, T, B)
    return out


def monarch_matrix_hip(q: Tensor, k: Tensor, attn_mask: Tensor | None, T: int, B: int, pre_pad: bool, *,
                       variant: str | None = None) -> Tensor:
    """Dense ``(E, H, N, N)`` fp32 attention matrix of q and k: what the forward
    pass returns for an fp32 identity as v (``MonarchAttention.get_matrix``,
    ma/monarch_attention.py:61-66), written entry by entry by ``ma_matrix``
    without the identity and without the ``(E, H, Np, N)`` intermediate.
    ``variant`` ('auto', 'generic' or 'staged') selects the kernels of the T
    steps.  Raises ``NotImplementedError`` when the padded sequence is beyond
    what the kernel holds on chip."""
    A = _HOST.matrix(q, k, attn_mask, T, B, pre_pad, _variant_code(variant), 0)
    if A is None:
        _refused(q, k, q, attn_mask, T, B)
    return A


def monarch_attention_hip_backward(q: Tensor, k: Tensor, v: Tensor, attn_mask: Tensor | None, dout: Tensor, T: int,
                                   B: int, pre_pad: bool, *, variant: str | None = None):
    """Gradients ``(dq, dk, dv)`` of ``monarch_attention_hip(q, k, v, attn_mask, T, B, pre_pad)``
    for the output gradient ``dout`` - what autograd through the reference's
    ``monarch_attention_torch`` (ma/ma_torch.py:65-108) yields.  ``ma_bwd`` runs
    the T steps again (``variant`` 'auto', 'generic' or 'staged' picks their
    kernels) and then the backward kernels, all on the current stream."""
    grads = _HOST.backward(q, k, v, attn_mask, dout, T, B, pre_pad, _variant_code(variant), 0)
    if grads is None:
        if dout.shape != v.shape or dout.device != v.device:
            raise ValueError(f"dout must have the shape of the output {tuple(v.shape)}, got {tuple(dout.shape)}")
        _refused(q, k, v, attn_mask, T, B)
    return grads
