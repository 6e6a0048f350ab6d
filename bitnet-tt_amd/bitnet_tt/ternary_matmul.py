"""The ternary matmul op: drop-in for ``ttnn.experimental.ternary_matmul``.

bitnet-tt calls ``ttnn.experimental.ternary_matmul(x, W, use_packed_ternary=True,
norm_weight=..., norm_epsilon=...)`` from ``Linear.__call__``
(src/bitnet_tt/layers/bitlinear.py:336-341) and from the decode loop's fused
RMSNorm->QKV (src/bitnet_tt/inference/generator_batch32.py:721-727).  Here the
same call runs one launch sequence of libbtl.so (``btl_bitlinear_fused``):

    [RMSNorm(norm_weight, norm_epsilon) ->] per-token int8 absmax quant ->
    int8 x ternary GEMM (int32, exact) -> epilogue -> bf16

The epilogue applies the activation dequantisation ``a/127`` and the weight
scale(s) in one multiply (Linear's separate ``multiply(out, weight_scale)``,
bitlinear.py:351-352, folds into it), optionally ``relu(g)^2 * u`` for the
gate||up weight (ffn.py:164-170) and a residual add.  There is no other
backend: inputs must live on a ROCm device and libbtl.so must be built.
"""

from __future__ import annotations

import functools
import os
from dataclasses import dataclass, field

from . import _native as N

EPILOGUES = {"none": N.EPI_SCALE, "scale": N.EPI_SCALE, "relu2_mul": N.EPI_RELU2_MUL}

# Check-after-call mode: every call synchronises its device and raises
# RuntimeError at the call when a bounded wait of a fused decode launch ran
# out, as the reference's op raises at its call (bitlinear.py:329-330).  Off by
# default (a synchronisation per call; not allowed inside a graph capture);
# on with set_check_after_call(True) or BTL_CHECK_AFTER_CALL=1, or per call.
_check_after_call = os.environ.get("BTL_CHECK_AFTER_CALL", "0") not in ("", "0")


def set_check_after_call(enabled: bool) -> None:
    """Turn the check-after-call mode on or off for every later call."""
    global _check_after_call
    _check_after_call = bool(enabled)


def check_after_call_enabled() -> bool:
    return _check_after_call


@dataclass
class PackedTernaryWeight:
    """A ternary weight in the GEMM's device layout.

    ``data``: int32 tensor (N/32, ceil(K/128), 256) on the device, made by
    :func:`bitnet_tt.kernels.pack.repack_for_gemm` from the reference tile
    format.  ``segment_scales``/``segment_ends`` are the per-projection weight
    scales of a fused weight (Q|K|V, gate|up) with their exclusive column ends.
    """

    data: "object"
    in_features: int
    out_features: int
    segment_scales: tuple = (1.0,)
    segment_ends: tuple = field(default_factory=tuple)

    def __post_init__(self):
        if not self.segment_ends:
            self.segment_ends = (self.out_features,)

    @property
    def device(self):
        return self.data.device

    @property
    def nbytes(self) -> int:
        return self.data.numel() * 4


def ternary_matmul(
    input_tensor_a,
    input_tensor_b,
    *,
    use_packed_ternary: bool = True,
    norm_weight=None,
    norm_epsilon: float | None = None,
    compute_kernel_config=None,
    weight_scale=None,
    epilogue: str = "none",
    residual=None,
    splitk: int = 0,
    acc_out=None,
    xq_out=None,
    check_errors: bool | None = None,
):
    """``y = epilogue(quant(norm(a)) @ W)`` in bf16.

    input_tensor_a: bf16 [..., M, K] on a ROCm device.
    input_tensor_b: :class:`PackedTernaryWeight` (or its ``data`` tensor).
    norm_weight / norm_epsilon: RMSNorm gain [K] (any shape with K elements)
        and epsilon, fused in front of the quantiser when given.
    weight_scale: None -> the weight's own segment scales; a float or a
        sequence of per-segment floats overrides them.
    epilogue: "none" (scale), or "relu2_mul" for a gate||up weight (output has
        N/2 columns).
    residual: optional bf16 [..., M, N] added to the output (may be the output
        buffer's owner tensor; the result is returned as a new tensor unless
        ``residual`` is also the destination, see :func:`ternary_matmul_into`).
    acc_out / xq_out: optional int32 [M, N] / int8 [M, K] tensors receiving the
        exact accumulators and the quantised activations (parity checks).
    compute_kernel_config: accepted for signature compatibility; the gfx950
        path has a single (exact) accumulation mode.
    check_errors: True synchronises after the launch and raises RuntimeError
        if a bounded wait of a fused decode launch ran out (None: the mode set
        by :func:`set_check_after_call`).
    """
    import torch

    if not use_packed_ternary:
        raise ValueError("only the packed ternary path exists on this backend")
    w = input_tensor_b
    if not isinstance(w, PackedTernaryWeight):
        if w.dim() != 3 or w.shape[-1] != 256:
            raise ValueError("input_tensor_b must be a PackedTernaryWeight or an int32 (N/32, KS, 256) tensor")
        w = PackedTernaryWeight(w, input_tensor_a.shape[-1], w.shape[0] * 32)
    x = input_tensor_a
    N.require_cuda(x, "input_tensor_a")
    if x.dtype != torch.bfloat16:
        raise ValueError("input_tensor_a must be bfloat16")
    K = x.shape[-1]
    if K != w.in_features:
        raise ValueError(f"input has K={K}, weight expects {w.in_features}")
    Nf = w.out_features
    epi = EPILOGUES.get(epilogue)
    if epi is None:
        raise ValueError(f"unknown epilogue {epilogue!r}")
    M = x.numel() // K
    n_out = Nf // 2 if epi == N.EPI_RELU2_MUL else Nf
    out = torch.empty(x.shape[:-1] + (n_out,), dtype=torch.bfloat16, device=x.device)
    ternary_matmul_into(
        x, w, out, norm_weight=norm_weight, norm_epsilon=norm_epsilon, weight_scale=weight_scale,
        epilogue=epilogue, residual=residual, splitk=splitk, acc_out=acc_out, xq_out=xq_out,
        check_errors=check_errors,
    )
    return out


# The library reads these arrays during the call and never writes them.
_cached_segments = functools.lru_cache(maxsize=4096)(N.segments_arrays)


def _segments(scales, ends):
    """segments_arrays of a weight's segments, kept by their values: a scale
    may be any object that converts to a float (a tensor or array may change
    in place between calls).  Zeros are not kept: 0.0 and -0.0 are equal keys."""
    if type(sum(scales) + sum(ends)) is not float or 0.0 in scales:  # not plain numbers
        return N.segments_arrays(scales, ends)
    return _cached_segments(tuple(scales), tuple(ends))


@functools.lru_cache(maxsize=4096)
def _fused_bytes(index: int, m: int, k: int, n: int, epi: int, splitk: int) -> tuple[int, int]:
    """(workspace bytes, error word offset) of a fused call on device ``index``."""
    L = N.lib()
    return int(L.btl_fused_workspace_bytes(m, k, n, epi, splitk)), int(L.btl_fused_error_offset())


def check(device=None) -> None:
    """Raise RuntimeError if a bounded wait of a fused decode launch on
    ``device`` ran out since the last check (the launch then returned invalid
    bf16 values).  Synchronises the device; call it at synchronisation points.
    The reference surfaces op failures as RuntimeError
    (src/bitnet_tt/layers/bitlinear.py:329-330)."""
    N.check_errors(device)


def ternary_matmul_into(
    x,
    w: PackedTernaryWeight,
    out,
    *,
    norm_weight=None,
    norm_epsilon: float | None = None,
    weight_scale=None,
    epilogue: str = "none",
    residual=None,
    splitk: int = 0,
    acc_out=None,
    xq_out=None,
    check_errors: bool | None = None,
):
    """Same as :func:`ternary_matmul` writing into ``out`` (no allocation once
    the per-stream workspace exists, so the call can be captured in a graph).
    ``residual`` may be ``out`` itself for an in-place residual add."""
    import torch

    K = w.in_features
    Nf = w.out_features
    M = x.numel() // K
    epi = EPILOGUES[epilogue]
    N.require_cuda(x, "x")
    N.require_cuda(out, "out")
    if out.dtype != torch.bfloat16:
        raise ValueError("out must be bfloat16")
    n_out = Nf // 2 if epi == N.EPI_RELU2_MUL else Nf
    if out.numel() != M * n_out:
        raise ValueError(f"out has {out.numel()} elements, expected {M}x{n_out}")
    gamma = res = acc = xq = None  # addresses
    eps = 0.0
    if residual is not None:
        N.require_cuda(residual, "residual")
        if residual.numel() != M * n_out or residual.dtype != torch.bfloat16:
            raise ValueError("residual must be bf16 with the output's shape")
        res = residual.data_ptr()
    if acc_out is not None:
        N.require_cuda(acc_out, "acc_out")
        if acc_out.dtype != torch.int32 or acc_out.numel() != M * Nf:
            raise ValueError("acc_out must be int32 [M, N]")
        acc = acc_out.data_ptr()
    if xq_out is not None:
        N.require_cuda(xq_out, "xq_out")
        if xq_out.dtype != torch.int8 or xq_out.numel() != M * K:
            raise ValueError("xq_out must be int8 [M, K]")
        xq = xq_out.data_ptr()
    if norm_weight is not None:
        if norm_epsilon is None:
            raise ValueError("norm_weight needs norm_epsilon")
        N.require_cuda(norm_weight, "norm_weight")
        if norm_weight.dtype != torch.bfloat16 or norm_weight.numel() != K:
            raise ValueError("norm_weight must be bf16 with K elements")
        gamma = norm_weight.data_ptr()
        eps = float(norm_epsilon)
    if weight_scale is None:
        sc, en, nseg = _segments(w.segment_scales, w.segment_ends)
    elif isinstance(weight_scale, (int, float)):
        sc, en, nseg = N.segments_arrays((float(weight_scale),), (Nf,))
    else:
        scales = tuple(float(s) for s in weight_scale)
        if len(scales) != len(w.segment_ends):
            raise ValueError("weight_scale needs one value per weight segment")
        sc, en, nseg = N.segments_arrays(scales, tuple(w.segment_ends))
    index = x.device.index
    stream = N.raw_stream(index)
    if type(splitk) is not int:
        splitk = int(splitk)
    nbytes, off = _fused_bytes(index, M, K, Nf, epi, splitk)
    ws, ws_bytes, _ = N.workspace_ptr(index, nbytes, "bitlinear", off, stream)
    rc = N.lib().btl_bitlinear_fused(x.data_ptr(), M, K, K, gamma, eps, w.data.data_ptr(), Nf, sc, en, nseg, epi, res,
                                     out.data_ptr(), acc, xq, ws, ws_bytes, splitk, stream)
    if rc != N.BTL_OK:
        N.check(rc, "btl_bitlinear_fused")
    if _check_after_call if check_errors is None else check_errors:
        N.check_errors(x.device)
    return out
