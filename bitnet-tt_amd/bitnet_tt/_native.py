"""ctypes binding of libbtl.so, the gfx950 BitLinear library (include/btl.h).

The library is the only compute path of this package: every device operation
goes through it, and a missing or stale library raises instead of falling back
to anything else.  Tensors are passed as raw device pointers together with the
current HIP stream of the calling thread (``torch.cuda.current_stream()``), so
calls are stream-ordered and can be recorded into a HIP graph.
"""

from __future__ import annotations

import collections
import ctypes
import itertools
import os
import threading
import weakref

_HERE = os.path.dirname(os.path.abspath(__file__))
# BTL_LIBRARY names another build of the same library (the host-sanitizer
# build of tests/host_asan.sh); the default is the in-tree product build.
LIB_PATH = os.environ.get("BTL_LIBRARY") or os.path.join(_HERE, "_lib", "libbtl.so")

# Status codes and epilogue modes (include/btl.h).
BTL_OK = 0
STATUS_NAMES = {
    1: "BTL_ERR_NULL",
    2: "BTL_ERR_SHAPE",
    3: "BTL_ERR_ALIGN",
    4: "BTL_ERR_WORKSPACE",
    5: "BTL_ERR_ARG",
    6: "BTL_ERR_LAUNCH",
}
EPI_SCALE = 0
EPI_RELU2_MUL = 1
MAX_SEGMENTS = 4
MAX_K = 16384

_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_I = ctypes.c_int
_F = ctypes.c_float
_SZ = ctypes.c_size_t



class LayerWeight(ctypes.Structure):
    """btl_layer_weight_t: one BitLinear of a btl_decode_step launch."""

    _fields_ = [
        ("wdev", ctypes.c_void_p),
        ("seg_scale", ctypes.c_float * MAX_SEGMENTS),
        ("seg_end", ctypes.c_int64 * MAX_SEGMENTS),
        ("nseg", ctypes.c_int),
        ("gamma", ctypes.c_void_p),
    ]


def layer_weight(w, gamma) -> LayerWeight:
    """LayerWeight of a PackedTernaryWeight and the RMSNorm gain of its input."""
    n = len(w.segment_scales)
    if not 1 <= n <= MAX_SEGMENTS:
        raise ValueError(f"1..{MAX_SEGMENTS} weight-scale segments are supported, got {n}")
    lw = LayerWeight()
    lw.wdev = w.data.data_ptr()
    for i in range(MAX_SEGMENTS):
        lw.seg_scale[i] = float(w.segment_scales[i]) if i < n else 0.0
        lw.seg_end[i] = int(w.segment_ends[i]) if i < n else 0
    lw.nseg = n
    lw.gamma = gamma.data_ptr()
    return lw


_LWP = ctypes.POINTER(LayerWeight)

# name -> (argtypes, restype); the exported C ABI, one entry per declaration.
EXPORTS = {
    "btl_last_error": ([], ctypes.c_char_p),
    "btl_version": ([], _I),
    "btl_check_coresident": ([_I64, _I64, _I64], _I),
    "btl_packed_tile_count": ([_I64, _I64], _I64),
    "btl_packed_dram_bytes": ([_I64, _I64], _I64),
    "btl_devlayout_words": ([_I64, _I64], _I64),
    "btl_act_bytes": ([_I64, _I64], _I64),
    "btl_choose_splitk": ([_I64, _I64, _I64, _I], _I),
    "btl_gemm_tiling": ([_I64, _I64, _I64, _I, _I, _P], _I),
    "btl_gemm_workspace_bytes": ([_I64, _I64, _I64, _I, _I], _I64),
    "btl_fused_workspace_bytes": ([_I64, _I64, _I64, _I, _I], _I64),
    "btl_fused_prefill_form": ([_I64, _I64, _I64, _I], _I),
    "btl_fused_error_offset": ([], _I64),
    "btl_weight_quant_scratch_bytes": ([_I64], _I64),
    "btl_weight_quant_ternary": ([_P, _I64, _F, _P, _P, _P, _SZ, _P], _I),
    "btl_weight_quant_pack": ([_P, _I64, _I64, _F, _P, _P, _P, _SZ, _P], _I),
    "btl_pack_tiles": ([_P, _I64, _I64, _P, _P], _I),
    "btl_unpack_tiles": ([_P, _I64, _I64, _P, _P], _I),
    "btl_repack": ([_P, _I64, _I64, _P, _P], _I),
    "btl_quant_absmax": ([_P, _I64, _I64, _I64, _P, _F, _P, _P, _P, _P, _P, _P, _P], _I),
    "btl_rmsnorm": ([_P, _I64, _I64, _I64, _P, _F, _P, _P], _I),
    "btl_gemm_i8t2": (
        [_P, _P, _P, _I64, _I64, _I64, _P, _P, _P, _I, _I, _P, _P, _P, _P, _SZ, _I, _P],
        _I,
    ),
    "btl_bitlinear_fused": (
        [_P, _I64, _I64, _I64, _P, _F, _P, _I64, _P, _P, _I, _I, _P, _P, _P, _P, _P, _SZ, _I, _P],
        _I,
    ),
    "btl_bitlinear_fused_noalloc": (
        [_P, _I64, _I64, _I64, _P, _F, _P, _I64, _P, _P, _I, _I, _P, _P, _P, _P, _P, _I, _P],
        _I,
    ),
    "btl_decode_step_workspace_bytes": ([_I64, _I64, _I64, _I64, _I64], _I64),
    "btl_decode_step_error_offset": ([], _I64),
    "btl_decode_step_prepare": ([_I64, _I64, _I64, _I64, _I64, _LWP, _P, _SZ], _I),
    "btl_decode_step": ([_I64, _I64, _I64, _I64, _I64, _F, _P, _P, _P, _P, _P, _SZ, _P], _I),
    "btl_decode_step_floor": ([_I64, _I64, _I64, _I64, _I64, _P, _SZ, _P], _I),
    "btl_decode_step_clear_share": ([_I, _I64, _P, _I64], _I),
    "btl_decode_step_attention_prepare": ([_I64, _I64, _I64, _I64, _I64, _P, _P, _P, _SZ], _I),
    "btl_decode_step_full": (
        [_I64, _I64, _I64, _I64, _I64, _F, _I64, _I64, _P, _P, _P, _I, _F, _P, _P, _P, _P, _P, _SZ, _P],
        _I,
    ),
    "btl_gemm_i8t2_dot4": ([_P, _P, _I64, _I64, _I64, _P, _P, _P], _I),
    "btl_lm_head_weight_bytes": ([_I64, _I64], _I64),
    "btl_lm_head_workspace_bytes": ([], _I64),
    "btl_lm_head_repack": ([_P, _I64, _I64, _P, _P], _I),
    "btl_lm_head": ([_P, _I64, _I64, _I64, _P, _P, _P, _P, _SZ, _P], _I),
    "btl_decode_attention_workspace_bytes": ([_I64, _I64, _I64, _I64], _I64),
    "btl_decode_attention_error_offset": ([_I64, _I64], _I64),
    "btl_decode_attention_split_bytes": ([_I64, _I64, _I64], _I64),
    "btl_decode_attention_split": ([_P, _I64, _I64, _I64, _I64, _I64, _P, _P, _P, _I, _F, _P, _P, _P, _P, _SZ, _P,
                                    _SZ, _P], _I),
    "btl_decode_attention": ([_P, _I64, _I64, _I64, _I64, _I64, _P, _P, _P, _I, _F, _P, _P, _P, _P, _SZ, _P], _I),
}


class NativeLibraryError(RuntimeError):
    """libbtl.so is missing or unusable; there is no other compute path."""


_lib = None
_lock = threading.Lock()


def lib() -> ctypes.CDLL:
    """Load libbtl.so once and declare every exported signature."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise NativeLibraryError(
                f"{LIB_PATH} is not built; build it with __graft_entry__.build() "
                "(hipcc --offload-arch=gfx950). The BitLinear path has no other backend."
            )
        L = ctypes.CDLL(LIB_PATH)
        for name, (args, res) in EXPORTS.items():
            fn = getattr(L, name)
            fn.argtypes = args
            fn.restype = res
        _lib = L
    return _lib


def last_error() -> str:
    msg = lib().btl_last_error()
    return msg.decode() if msg else ""


def check(rc: int, what: str) -> None:
    if rc != BTL_OK:
        raise RuntimeError(f"{what} failed with {STATUS_NAMES.get(rc, rc)}: {last_error()}")


def ptr(t) -> ctypes.c_void_p | None:
    """Device pointer of a tensor (None passes NULL)."""
    if t is None:
        return None
    return ctypes.c_void_p(t.data_ptr())


def require_cuda(t, name: str) -> None:
    if t is None:
        return
    if not t.is_cuda:
        raise ValueError(
            f"{name} must be a tensor on a ROCm GPU device; the BitLinear path runs only "
            "through the gfx950 kernels"
        )
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


def _resolve_raw_stream():
    """current_stream(index).cuda_stream without the Stream object around it
    (1.7 us a call) where this torch has it."""
    import torch

    global _raw_stream
    _raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (
        lambda index: torch.cuda.current_stream(index).cuda_stream)
    return _raw_stream


_raw_stream = None


def raw_stream(index: int) -> int:
    """Handle of the calling thread's current stream on device ``index``."""
    return (_raw_stream or _resolve_raw_stream())(index)


def stream_of(device) -> ctypes.c_void_p:
    import torch

    if isinstance(device, torch.device) and device.type == "cuda" and device.index is not None:
        return ctypes.c_void_p(raw_stream(device.index))
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def segments_arrays(scales, ends):
    """Host arrays for the per-segment epilogue scales."""
    n = len(scales)
    if not 1 <= n <= MAX_SEGMENTS:
        raise ValueError(f"1..{MAX_SEGMENTS} weight-scale segments are supported, got {n}")
    sc = (ctypes.c_float * n)(*[float(s) for s in scales])
    en = (ctypes.c_int64 * n)(*[int(e) for e in ends])
    return sc, en, n


# Per (device, stream) workspace.  Calls on one stream are ordered, so they
# can share it; the activation kernel of every fused call clears the split-K
# counters it uses.  A workspace that holds one object's prepared state (the
# decode step's weight table) is that object's own on each stream: its key
# ends with the object's owner_id(), and it goes when the object does.
_workspaces: dict = {}
# workspace_ptr's lookups: (kind, device index, stream, error offset, owner) ->
# (address, bytes, buffer).  Emptied whenever a workspace is made or released.
_fast: dict = {}
# Held while the tables change or are read as a whole.  Not reentrant: a
# finalizer may run inside (at any allocation) and must not change them then.
_ws_lock = threading.Lock()
_owner_ids = itertools.count(1)
_owners: "weakref.WeakKeyDictionary" = weakref.WeakKeyDictionary()
# Owners that went while the lock was held; released by the next workspace().
_dead_owners: "collections.deque" = collections.deque()
# Workspaces that went with unread error words: (key, buffer, offsets), read
# and dropped by check_errors, or the oldest where a new one is made and there
# are more than _RETIRED_MAX.  _late_errors: what the latter found.
_retired: list = []
_late_errors: list = []
_RETIRED_MAX = 16


def owner_id(obj) -> int:
    """The number of ``obj`` whose workspaces are released with it (a copy of
    ``obj`` gets its own)."""
    n = _owners.get(obj)
    if n is None:
        n = _owners.setdefault(obj, next(_owner_ids))
        weakref.finalize(obj, _release_owner, n).atexit = False
    return n


def _release_owner(n: int) -> None:
    _dead_owners.append(n)
    if _ws_lock.acquire(blocking=False):
        try:
            _bury()
        finally:
            _ws_lock.release()


def _bury() -> None:
    """Release the workspaces of the owners that are gone (lock held)."""
    while _dead_owners:
        n = _dead_owners.popleft()
        _fast.clear()
        for key in [k for k in _workspaces if len(k) == 4 and k[3] == n]:
            _retire(key, _workspaces.pop(key))
            _error_words.pop(key, None)


def _retire(key, buf) -> None:
    """A workspace that is replaced or released (lock held)."""
    _prepared_for.pop(buf.data_ptr(), None)
    _reset_hooks.pop(buf.data_ptr(), None)
    offsets = sorted(_error_words.get(key, ()))
    if offsets:
        _retired.append((key, buf, offsets))


def _set_words(key, buf, offsets) -> list:
    """The error words of a workspace that are set: [(key, offset, value)]."""
    import torch

    words = [(key, off, int(buf[off:off + 4].view(torch.int32).item())) for off in offsets]
    return [w for w in words if w[2]]


def workspace_ptr(index: int, nbytes: int, kind: str, error_offset: int, stream: int, owner: int = 0):
    """(address, bytes) of :func:`workspace` on device ``index`` and the current
    stream, whose handle is ``stream``."""
    key = (kind, index, stream, error_offset, owner)
    hit = _fast.get(key)
    if hit is None or hit[1] < nbytes:
        import torch

        with _ws_lock:
            buf = _workspace(torch.device("cuda", index), nbytes, kind, error_offset, owner)
            hit = _fast[key] = (buf.data_ptr(), buf.numel(), buf)
    return hit


def _key(kind: str, device, stream: int, owner: int) -> tuple:
    return (kind, _device_key(device), stream) + ((owner,) if owner else ())


def has_workspace(device, nbytes: int, kind: str = "bitlinear", owner: int = 0) -> bool:
    """True when the current stream already owns a workspace of nbytes."""
    import torch

    buf = _workspaces.get(_key(kind, device, torch.cuda.current_stream(device).cuda_stream, owner))
    return buf is not None and buf.numel() >= nbytes


# Byte offsets of the sticky error words each workspace holds (a bounded wait
# of a kernel that ran out sets one; see check_errors).
_error_words: dict = {}
# What a workspace was prepared for (data_ptr -> owner object), for launches
# whose workspace holds host-prepared state (the decode step's weight table).
_prepared_for: dict = {}


# Host-side set-up to redo after a workspace has been zero-filled by
# check_errors (data_ptr -> callable), for workspaces whose start state is not
# all zeros (the decode step's weight table and operand tiles).
_reset_hooks: dict = {}


def workspace_prepared_for(buf):
    return _prepared_for.get(buf.data_ptr())


def set_workspace_reset(buf, fn) -> None:
    _reset_hooks[buf.data_ptr()] = fn


def set_workspace_prepared_for(buf, owner) -> None:
    _prepared_for[buf.data_ptr()] = owner


def _device_key(device) -> str:
    import torch

    d = torch.device(device)
    if d.index is None:
        d = torch.device(d.type, torch.cuda.current_device())
    return str(d)


def workspace(device, nbytes: int, kind: str = "bitlinear", error_offset: int | None = None, owner: int = 0):
    """Zero-filled device workspace of at least nbytes for the current stream.

    kind separates workspaces whose layouts differ ("bitlinear" for
    btl_bitlinear_fused / btl_gemm_i8t2, "step" for btl_decode_step).  A
    workspace that grows is replaced by a fresh zero-filled one; the old one
    is released in stream order, after the calls that used it (one with an error
    word once check_errors has read it).
    ``owner`` (owner_id) makes it one object's own.  ``error_offset`` registers
    the byte offset of a sticky error word inside the workspace, which
    :func:`check_errors` reads."""
    with _ws_lock:
        return _workspace(device, nbytes, kind, error_offset, owner)


def _workspace(device, nbytes: int, kind: str, error_offset: int | None, owner: int):
    """workspace() with the lock held."""
    import torch

    _bury()
    key = _key(kind, device, torch.cuda.current_stream(device).cuda_stream, owner)
    buf = _workspaces.get(key)
    if buf is None or buf.numel() < nbytes:
        _fast.clear()
        if buf is not None:
            _retire(key, buf)
        while len(_retired) > _RETIRED_MAX and not torch.cuda.is_current_stream_capturing():
            old = _retired.pop(0)
            torch.cuda.synchronize(old[0][1])
            _late_errors.extend(_set_words(*old))
        size = max(int(nbytes), 1 << 20)
        buf = torch.zeros(size, dtype=torch.uint8, device=device)
        _prepared_for.pop(buf.data_ptr(), None)
        _reset_hooks.pop(buf.data_ptr(), None)
        _workspaces[key] = buf
    if error_offset is not None:
        _error_words.setdefault(key, set()).add(int(error_offset))
    return buf


def check_errors(device=None) -> None:
    """Raise RuntimeError if any kernel on ``device`` set its sticky error word.

    The kernels that hand data between workgroups of one launch (the fused
    decode BitLinear, the decode step, decode attention) never hang: a wait
    that exceeds its spin limit sets a sticky error word in the call's
    workspace and the kernel finishes with invalid outputs.  This reads every
    registered error word of the device's workspaces (all streams) after a
    device synchronisation.  When one is set, the affected workspaces are
    zero-filled in place (the start state of their launch counters) and the
    host-side set-up registered for them (set_workspace_reset: the decode
    step's weight table and operand tiles) is redone, so later calls and
    graphs captured on them work again; RuntimeError names them: the outputs
    of the calls since the last check are not valid."""
    import torch

    dev = _device_key(device if device is not None else "cuda")
    with _ws_lock:
        live = [(k, b, sorted(_error_words.get(k, ()))) for k, b in _workspaces.items() if k[1] == dev]
        gone = [r for r in _retired if r[0][1] == dev]
        _retired[:] = [r for r in _retired if r[0][1] != dev]
        bad = [e for e in _late_errors if e[0][1] == dev]
        _late_errors[:] = [e for e in _late_errors if e[0][1] != dev]
    if gone or any(offsets for _, _, offsets in live):
        torch.cuda.synchronize(dev)
    for r in gone:
        bad += _set_words(*r)
    reset = []
    for r in live:
        found = _set_words(*r)
        bad += found
        if found:
            reset.append(r[1])
    if not bad:
        return
    for buf in reset:
        buf.zero_()
        torch.cuda.synchronize(dev)
        hook = _reset_hooks.get(buf.data_ptr())
        if hook is not None:
            hook()
        else:
            _prepared_for.pop(buf.data_ptr(), None)
    torch.cuda.synchronize(dev)
    what = ", ".join(f"{k[0]} workspace (stream {k[2]:#x}) word at byte {off} = {w}" for k, off, w in bad)
    raise RuntimeError(
        f"a kernel on {dev} set its error word ({what}): a bounded wait ran out, or a decode-attention position "
        "was out of range; the outputs of the calls since the last check are invalid, and the workspaces have "
        "been reset"
    )


def gemm_tiling(M: int, K: int, N: int, epilogue: int = EPI_SCALE, rowsum_given: bool = True) -> dict:
    """The tiling btl_gemm_i8t2 runs for a shape (a planning query)."""
    info = (ctypes.c_int32 * 6)()
    check(lib().btl_gemm_tiling(M, K, N, epilogue, int(bool(rowsum_given)), info), "btl_gemm_tiling")
    kind = ("decode", "tiles", "wide")[info[0]]
    return {"kind": kind, "rows": info[1], "col_tiles": info[2], "splitk": info[3], "k_groups": info[4],
            "tiles_per_wave": info[5]}
