"""Host side of the MI355X transformer-block hot path.

Mirrors the operator surface the reference's model builders use
(`Dense`, `RMSNorm`, `Functional.cmul`, `ScaledDotProductAttention`,
the rotary-table builders) on top of the C-ABI HIP library `libdthip.so`
declared in `include/dt_hip.h`.  torch is used for device memory and streams
only; every operator below runs hand-written gfx950 kernels, the common calls
through `_dthost.so` (csrc/dt_host.cpp), all others through ctypes, and raises
if the library is missing or a call fails.  There is no CPU path.
"""
from __future__ import annotations

import ctypes
import os
import struct
import subprocess
import warnings
from dataclasses import dataclass
from typing import Optional, Sequence

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libdthip.so")
CSRC = os.path.join(_HERE, "csrc")

DT_OK, DT_INVALID, DT_NO_KERNEL, DT_OOM, DT_DEVICE_ERROR = 0, -1, -2, -3, -4
_STATUS = {0: "DT_OK", -1: "DT_INVALID", -2: "DT_NO_KERNEL", -3: "DT_OOM", -4: "DT_DEVICE_ERROR"}

# every symbol include/dt_hip.h declares
ABI_SYMBOLS = (
    "dt_version",
    "dt_init",
    "dt_qx_bytes",
    "dt_depalettize_f16",
    "dt_dense_qx_f16",
    "dt_dense_qx_heads_f16",
    "dt_dense_qx_grouped_f16",
    "dt_dense_workspace_bytes",
    "dt_dense_qx_grouped_ws_f16",
    "dt_dense_scratch_bytes",
    "dt_dense_qx_grouped_scratch_f16",
    "dt_dense_qx_post_f16",
    "dt_qk_norm_rope_f16",
    "dt_layernorm_modulate_f16",
    "dt_layernorm_f16",
    "dt_sdpa_f16",
    "dt_sdpa_workspace_bytes",
    "dt_sdpa_f16_static",
    "dt_lora_branch_f32_f16",
    "dt_lora_dense_scratch_bytes",
    "dt_lora_dense_f16",
)

STATIC_SCRATCH_BYTES = 64 << 20  # DT_SDPA_STATIC_SCRATCH_BYTES


class DtError(RuntimeError):
    def __init__(self, fn: str, status: int):
        super().__init__(f"{fn} failed: {_STATUS.get(status, status)}")
        self.status = status


class _QxWeight(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("qbits", ctypes.c_int32), ("nib", ctypes.c_int32), ("count", ctypes.c_int64)]


class _View4(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("stride_b", ctypes.c_int64), ("stride_s", ctypes.c_int64),
                ("stride_h", ctypes.c_int64)]


class _HeadEpilogue(ctypes.Structure):
    _fields_ = [("gamma", ctypes.c_void_p), ("rot", ctypes.c_void_p), ("rot_pos0", ctypes.c_int64),
                ("eps", ctypes.c_float), ("head_dim", ctypes.c_int32)]


class _DensePost(ctypes.Structure):
    _fields_ = [("activation", ctypes.c_int32), ("gate", ctypes.c_void_p), ("residual", ctypes.c_void_p),
                ("ld_residual", ctypes.c_int64), ("scale", ctypes.c_float), ("addend", ctypes.c_void_p),
                ("ld_addend", ctypes.c_int64), ("gate_f32", ctypes.c_void_p), ("multiplicand", ctypes.c_void_p),
                ("ld_multiplicand", ctypes.c_int64)]


class _DenseGroup(ctypes.Structure):
    _fields_ = [("M", ctypes.c_int64), ("K", ctypes.c_int64), ("X", ctypes.c_void_p), ("ldx", ctypes.c_int64),
                ("W", ctypes.c_void_p), ("n_weights", ctypes.c_int32), ("bias", ctypes.c_void_p),
                ("Y", ctypes.c_void_p), ("ldy", ctypes.c_void_p), ("epi", ctypes.c_void_p),
                ("post", ctypes.c_void_p)]


class _LoraPair(ctypes.Structure):
    _fields_ = [("down", ctypes.c_void_p), ("up", ctypes.c_void_p), ("ld_up", ctypes.c_int64), ("rank", ctypes.c_int32),
                ("f32", ctypes.c_int32), ("scale", ctypes.c_float)]


# The first four as struct formats: a launch's arrays are packed in one go (a ctypes structure costs a microsecond each,
# which for a conditioning row's six projections is more than the kernel takes).
_FMT_WEIGHT, _FMT_EPI, _FMT_POST, _FMT_GROUP = "Qiiq", "QQqfi", "i4xQQqf4xQqQQq", "qqQqQi4xQQQQQ"
for _fmt, _cls in ((_FMT_WEIGHT, _QxWeight), (_FMT_EPI, _HeadEpilogue), (_FMT_POST, _DensePost), (_FMT_GROUP, _DenseGroup)):
    assert struct.calcsize("=" + _fmt) == ctypes.sizeof(_cls)


class _Segment(ctypes.Structure):
    _fields_ = [("view", _View4), ("len", ctypes.c_int64), ("gamma", ctypes.c_void_p)]


def build(verbose: bool = False) -> str:
    """Compile libdthip.so for gfx950, and these operators' way to it, with the Makefile under csrc/ (always recompiles)."""
    cmd = ["make", "-C", CSRC, "-B", "-j8", "python"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if verbose or res.returncode != 0:
        print(res.stdout)
    if res.returncode != 0:
        raise RuntimeError("building libdthip.so failed")
    return LIB_PATH


_lib = None


def lib():
    """The loaded C-ABI library.  Raises if it has not been built: there is no fallback."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with __graft_entry__.build() or `make -C {CSRC} python`; "
                "this package has no CPU or PyTorch fallback"
            )
        L = ctypes.CDLL(LIB_PATH)
        vp, i32, i64, f32 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64, ctypes.c_float
        L.dt_version.restype = ctypes.c_char_p
        L.dt_version.argtypes = []
        L.dt_init.restype = i32
        L.dt_init.argtypes = [ctypes.c_int]
        L.dt_qx_bytes.restype = i64
        L.dt_qx_bytes.argtypes = [i32, i32, i64]
        L.dt_depalettize_f16.restype = i32
        L.dt_depalettize_f16.argtypes = [vp, ctypes.POINTER(_QxWeight), vp]
        L.dt_dense_qx_f16.restype = i32
        L.dt_dense_qx_f16.argtypes = [vp, i64, i64, vp, i64, ctypes.POINTER(_QxWeight), i32,
                                      ctypes.POINTER(vp), ctypes.POINTER(vp), ctypes.POINTER(i64), ctypes.c_uint32]
        L.dt_dense_qx_heads_f16.restype = i32
        L.dt_dense_qx_heads_f16.argtypes = [vp, i64, i64, vp, i64, ctypes.POINTER(_QxWeight), i32,
                                            ctypes.POINTER(vp), ctypes.POINTER(vp), ctypes.POINTER(i64),
                                            ctypes.POINTER(_HeadEpilogue), ctypes.c_uint32]
        L.dt_qk_norm_rope_f16.restype = i32
        L.dt_dense_qx_post_f16.restype = i32
        L.dt_dense_qx_post_f16.argtypes = [vp, i64, i64, vp, i64, ctypes.POINTER(_QxWeight), i32,
                                           ctypes.POINTER(vp), ctypes.POINTER(vp), ctypes.POINTER(i64),
                                           ctypes.POINTER(_DensePost), ctypes.c_uint32]
        L.dt_dense_qx_grouped_f16.restype = i32
        L.dt_dense_qx_grouped_f16.argtypes = [vp, i32, ctypes.POINTER(_DenseGroup), ctypes.c_uint32]
        L.dt_dense_workspace_bytes.restype = ctypes.c_size_t
        L.dt_dense_workspace_bytes.argtypes = [i32, vp]
        L.dt_dense_qx_grouped_ws_f16.restype = i32
        L.dt_dense_qx_grouped_ws_f16.argtypes = [vp, i32, vp, ctypes.c_uint32, vp, ctypes.c_size_t]
        L.dt_dense_scratch_bytes.restype = ctypes.c_size_t
        L.dt_dense_scratch_bytes.argtypes = [i32, vp]
        L.dt_dense_qx_grouped_scratch_f16.restype = i32
        L.dt_dense_qx_grouped_scratch_f16.argtypes = L.dt_dense_qx_grouped_ws_f16.argtypes
        L.dt_qk_norm_rope_f16.argtypes = [vp, _View4, i32, i64, i32, i32, vp, f32, i32, vp, i64, f32]
        L.dt_layernorm_modulate_f16.restype = i32
        L.dt_layernorm_modulate_f16.argtypes = [vp, i64, i64, vp, i64, vp, vp, i32, f32, vp, i64]
        L.dt_layernorm_f16.restype = i32
        L.dt_layernorm_f16.argtypes = [vp, i64, i64, vp, i64, vp, vp, f32, vp, i64]
        L.dt_sdpa_f16.restype = i32
        L.dt_sdpa_f16.argtypes = [vp, i32, i32, i32, i32, i32, ctypes.POINTER(_Segment), i32,
                                  ctypes.POINTER(_Segment), ctypes.POINTER(_Segment), vp, vp, f32, _View4, f32,
                                  vp, vp, vp, ctypes.c_size_t]
        L.dt_sdpa_f16_static.restype = i32
        L.dt_sdpa_f16_static.argtypes = L.dt_sdpa_f16.argtypes[:-2]
        L.dt_lora_branch_f32_f16.restype = i32
        L.dt_lora_branch_f32_f16.argtypes = [vp, i64, i64, vp, i64, vp, i32, vp, i64, f32, vp, vp, i64]
        pair = [ctypes.POINTER(_DensePost), ctypes.POINTER(_LoraPair)]
        L.dt_lora_dense_scratch_bytes.restype = ctypes.c_size_t
        L.dt_lora_dense_scratch_bytes.argtypes = [i64, i64, vp, i64, ctypes.POINTER(_QxWeight), vp, i64, *pair]
        L.dt_lora_dense_f16.restype = i32
        L.dt_lora_dense_f16.argtypes = [vp, i64, i64, vp, i64, ctypes.POINTER(_QxWeight), vp, vp, i64, *pair, ctypes.c_uint32, vp,
                                        ctypes.c_size_t]
        L.dt_sdpa_workspace_bytes.restype = ctypes.c_size_t
        L.dt_sdpa_workspace_bytes.argtypes = [i32, i32, i32, i32, i64, i64, i32, i32]
        _lib = L
    return _lib


_native = None


def _host():
    """The operators' native way to the library (csrc/dt_host.cpp), or None where there is none that loads beside this torch: every
    operator's results are the same without it, in more of the host's time and, for LoRA layers, more launches."""
    global _native
    if _native is None:
        lib(), _torch()  # (whose libraries it is linked against)
        path, host = os.path.join(_HERE, "_dthost.so"), False
        if os.path.exists(path):
            import importlib.util

            try:
                spec = importlib.util.spec_from_file_location("_dthost", path)
                host = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(host)
                host.classes(QxTensor, HeadEpilogue, DensePost)
            except ImportError as e:
                host = False
                warnings.warn(f"{path} does not load ({e}); calls go through ctypes.  Build it against this torch: "
                              f"`make -C {CSRC} python`", RuntimeWarning)
        _native = host  # (whole: another thread may be looking)
    return _native or None


def _check(fn: str, status: int):
    if status != DT_OK:
        raise DtError(fn, status)


def _torch():
    import torch

    return torch


def _stream_ptr(stream=None):
    torch = _torch()
    # (given the device's number, torch looks the stream up without asking for the device first: 1 us instead of 3)
    s = stream if stream is not None else torch.cuda.current_stream(torch.cuda.current_device())
    return ctypes.c_void_p(s.cuda_stream)


class _on:
    """Makes `stream` torch's current stream for the body of an operator, so that the tensors the operator
    allocates, the copies it makes (`clone`, `contiguous`) and the kernels it launches are all ordered on that one
    stream, and torch's allocator ties every temporary's reuse to it.  None = leave the current stream alone."""

    def __init__(self, stream):
        self.ctx = None if stream is None else _torch().cuda.stream(stream)

    def __enter__(self):
        if self.ctx is not None:
            self.ctx.__enter__()

    def __exit__(self, *exc):
        if self.ctx is not None:
            self.ctx.__exit__(*exc)


def _stream_scoped(fn):
    """Runs an operator with its `stream=` argument as torch's current stream (see _on)."""
    import functools
    import inspect

    names = list(inspect.signature(fn).parameters)
    at = names.index("stream")

    @functools.wraps(fn)
    def wrapped(*args, **kwargs):
        stream = kwargs.get("stream", args[at] if len(args) > at else None)
        if stream is None:
            return fn(*args, **kwargs)
        with _on(stream):
            return fn(*args, **kwargs)

    return wrapped


def _f16_cuda(t, name):
    torch = _torch()
    if not (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == torch.float16):
        raise TypeError(f"{name} must be a CUDA float16 tensor")
    return t


# --------------------------------------------------------------------------
# palettized weights
# --------------------------------------------------------------------------

# Elements per palette block for each codec.  Derived from the shipped model
# sizes (about 0.25 bit/weight of palette overhead for q6p/q8p, 0.5 for
# q4p/q5p); the library itself takes (qbits, nib) at run time.
CODEC = {"q4p": (4, 512), "q5p": (5, 1024), "q6p": (6, 4096), "q7p": (7, 8192), "q8p": (8, 16384)}


def qx_bytes(qbits: int, nib: int, count: int) -> int:
    return int(lib().dt_qx_bytes(qbits, nib, count))


def pack_indices(qbits: int, idx: np.ndarray) -> np.ndarray:
    """MSB-first bit stream of `qbits`-wide indices (host-side producer of the format).
    Eight indices always fill exactly `qbits` bytes: build each group as one 64-bit
    big-endian number and cut it into bytes."""
    idx = np.asarray(idx, dtype=np.uint8).reshape(-1)
    n = idx.size
    nbytes = (n * qbits + 7) // 8
    if qbits == 8:
        return idx.copy()
    groups = (n + 7) // 8
    padded = np.zeros(groups * 8, dtype=np.uint64)
    padded[:n] = idx & ((1 << qbits) - 1)
    padded = padded.reshape(groups, 8)
    val = np.zeros(groups, dtype=np.uint64)
    for j in range(8):
        val |= padded[:, j] << np.uint64(qbits * (7 - j))
    out = np.empty((groups, qbits), dtype=np.uint8)
    for i in range(qbits):
        out[:, i] = (val >> np.uint64(8 * (qbits - 1 - i))).astype(np.uint8)
    return out.reshape(-1)[:nbytes].copy()


def pack_qx(qbits: int, nib: int, palettes: np.ndarray, idx: np.ndarray) -> np.ndarray:
    """Packed buffer from per-block fp16 palettes [nblocks, 2^q] and indices [count]."""
    idx = np.asarray(idx, dtype=np.uint8).reshape(-1)
    palettes = np.ascontiguousarray(palettes, dtype=np.float16)
    count = idx.size
    nblocks = (count + nib - 1) // nib
    if palettes.shape != (nblocks, 1 << qbits):
        raise ValueError(f"palettes must be [{nblocks}, {1 << qbits}]")
    full = count // nib
    pal_bytes = 2 << qbits
    blk_bytes = nib * qbits // 8 if (nib * qbits) % 8 == 0 else None
    chunks = []
    if blk_bytes is not None and full > 0:
        # all full blocks at once
        packed = pack_indices(qbits, idx[: full * nib]).reshape(full, blk_bytes)
        body = np.empty((full, pal_bytes + blk_bytes), dtype=np.uint8)
        body[:, :pal_bytes] = palettes[:full].view(np.uint8).reshape(full, pal_bytes)
        body[:, pal_bytes:] = packed
        chunks.append(body.reshape(-1))
        start = full
    else:
        start = 0
    for b in range(start, nblocks):
        chunks.append(palettes[b].view(np.uint8).reshape(-1))
        chunks.append(pack_indices(qbits, idx[b * nib:(b + 1) * nib]))
    return np.concatenate(chunks) if chunks else np.zeros(0, np.uint8)


@dataclass
class QxTensor:
    """A weight as `store.read(codec: [.jit, .q?p])` leaves it: packed, on the device.

    qbits == 16 means a plain fp16 [out, in] tensor (data is then a float16 tensor)."""

    data: "object"  # torch uint8 (packed) or float16 tensor on the GPU
    qbits: int
    nib: int
    shape: tuple  # (out, in)

    @property
    def count(self) -> int:
        return int(self.shape[0]) * int(self.shape[1])

    def _c(self) -> _QxWeight:
        return _QxWeight(self.data.data_ptr(), self.qbits, self.nib, self.count)

    @staticmethod
    def from_packed(packed: np.ndarray, qbits: int, nib: int, shape, device="cuda") -> "QxTensor":
        torch = _torch()
        want = qx_bytes(qbits, nib, int(shape[0]) * int(shape[1]))
        packed = np.ascontiguousarray(packed, dtype=np.uint8)
        if packed.size != want:
            raise ValueError(f"packed buffer has {packed.size} bytes, layout needs {want}")
        # pad so the device buffer is a whole number of dwords
        buf = np.zeros((packed.size + 15) // 16 * 16, dtype=np.uint8)
        buf[: packed.size] = packed
        return QxTensor(torch.from_numpy(buf).to(device), qbits, nib, (int(shape[0]), int(shape[1])))

    @staticmethod
    def from_f16(w, device="cuda") -> "QxTensor":
        torch = _torch()
        if isinstance(w, np.ndarray):
            w = torch.from_numpy(np.ascontiguousarray(w, dtype=np.float16))
        w = w.to(device).contiguous()
        return QxTensor(w, 16, 0, tuple(w.shape))

    def dequantize(self, stream=None, out=None):
        """fp16 [out, in] tensor (K0): what a CPU read of the same key followed by Tensor<Float16>(from:) holds.
        `out`: a contiguous fp16 tensor of that shape to fill instead of a new one."""
        torch = _torch()
        if out is not None and (out.dtype != torch.float16 or tuple(out.shape) != tuple(self.shape)
                                or not out.is_contiguous() or out.device != self.data.device):
            raise ValueError("out must be a contiguous fp16 tensor of the weight's shape on its device")
        with _on(stream):
            if self.qbits == 16:
                return self.data.clone() if out is None else out.copy_(self.data)
            if out is None:
                out = torch.empty(self.shape, dtype=torch.float16, device=self.data.device)
            w = self._c()
            _check("dt_depalettize_f16", lib().dt_depalettize_f16(_stream_ptr(stream), ctypes.byref(w), out.data_ptr()))
            return out


# --------------------------------------------------------------------------
# operators (names and argument meaning follow the reference's Model DSL)
# --------------------------------------------------------------------------

class GEMMFlag:
    """Functional.GEMMFlag: permissions to compute at a given precision, not requests (Models/Flux1.swift:134, 162,
    229-231).  `Int8` is what FlashAttentionLevel.quantized adds to an attention's flags (`[.Int8, .Float16]`,
    Models/UNetProtocol.swift:14-19): this library computes such calls with its fp16 kernel (fp16 operands, fp32
    accumulation and statistics), which every combination of these flags permits."""
    Float16 = 1
    Float32 = 2
    Int8 = 4


@dataclass
class HeadEpilogue:
    """Per-head RMSNorm and RoPE fused behind a Dense: gamma [head_dim] or None, rot [>= rot_pos0 + M, head_dim] or None."""

    gamma: "object" = None
    rot: "object" = None
    rot_pos0: int = 0
    eps: float = 1e-6
    head_dim: int = 128


def _per_weight(entries, n, what):
    """One entry per weight: a shorter list leaves the rest None."""
    entries = list(entries)
    if len(entries) > n:
        raise IndexError(f"{len(entries)} {what} for {n} weights")
    return entries + [None] * (n - len(entries))


def _pack_epilogues(epilogues, M):
    vals = []
    for e in epilogues:
        if e is None:
            vals += (0, 0, 0, 0.0, 128)
            continue
        if e.rot is not None:
            _f16_cuda(e.rot, "rot")
            if e.rot.dim() != 2 or e.rot.shape[1] != e.head_dim or not e.rot.is_contiguous() \
                    or e.rot.shape[0] < e.rot_pos0 + M:
                raise ValueError("rot must be a contiguous [>= rot_pos0 + M, head_dim] table")
        if e.gamma is not None and (_f16_cuda(e.gamma, "gamma").numel() != e.head_dim or not e.gamma.is_contiguous()):
            raise ValueError("gamma must hold head_dim elements")
        vals += (0 if e.gamma is None else e.gamma.data_ptr(), 0 if e.rot is None else e.rot.data_ptr(), e.rot_pos0, e.eps,
                 e.head_dim)
    return struct.pack("=" + _FMT_EPI * len(epilogues), *vals)


def _marshal_dense(x, weights, biases, outs, epilogues, posts):
    """One Dense problem: (what it keeps alive, its packed dt_dense_group, its outputs, M)."""
    _f16_cuda(x, "x")
    K = x.shape[-1]
    x2 = x if x.dim() == 2 else x.reshape(-1, K)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    M = x2.shape[0]
    n = len(weights)
    vals = []
    for w in weights:
        if w.shape[1] != K:
            raise ValueError(f"weight {w.shape} does not match input width {K}")
        vals += (w.data.data_ptr(), w.qbits, w.nib, w.count)
    outs = [x.new_empty((M, w.shape[0])) for w in weights] if outs is None else list(outs)
    ptrs = [0 if b is None else _f16_cuda(b, "bias").data_ptr() for b in _per_weight(biases, n, "biases")]
    if len(outs) != n:
        raise ValueError("weights and outs must be of one length")
    ys = [o.data_ptr() for o in outs]
    strides = [o.stride(0) for o in outs]
    # (a problem with both is for the library to refuse)
    epi = b"" if epilogues is None else _pack_epilogues(_per_weight(epilogues, n, "epilogues"), M)
    post = b"" if posts is None else _pack_posts(_per_weight(posts, n, "posts"), weights, M, ys, outs)
    arrays = ctypes.create_string_buffer(struct.pack(f"={_FMT_WEIGHT * n}{2 * n}Q{n}q", *vals, *ptrs, *ys, *strides) + epi + post)
    base = ctypes.addressof(arrays)
    tails = base + 48 * n
    # (the stride of a single row says nothing: that of a [K, 1] tensor's transpose is 1)
    group = struct.pack("=" + _FMT_GROUP, M, K, x2.data_ptr(), x2.stride(0) if M > 1 else K, base, n, base + 24 * n, base + 32 * n, base + 40 * n,
                        0 if epilogues is None else tails, 0 if posts is None else tails + len(epi))
    return (x2, arrays), group, outs, M


# Rows up to which the library streams the weights (kRowsMax in csrc/dt_dense_rows.h) and uses no workspace, so that it is
# not asked how much (0.5 us of a conditioning row's 22).  The few such calls that it gives to the tiled kernel after all
# -- plain fp16 weights with over 16 rows and 8192 features, palettes that do not fit the LDS -- run uncut from here.
_ROWS_MAX = 64
# The smallest blocks and the most bytes of fp16 that the library copies palettized weights in (kDepalMinNib in
# csrc/dt_depalettize.h, kDenseMaxExpand in csrc/dt_dense.hip).
_COPIED_NIB, _COPIED_BYTES = 512, 512 << 20
_BESIDE_INPUTS = 2048  # from which on a LoRA layer's down projection may get a stream of its own


def _scratch(like, need, least):
    """(what holds it, address, bytes) of scratch memory on the device of `like`, 256-byte aligned: `need` bytes, or where
    the device is that full the `least` that the call cannot do without.  torch's allocator hands the block out again in
    stream order, so it may be dropped as soon as the call is enqueued."""
    if not need:
        return None, None, 0
    torch = _torch()
    try:
        ws = like.new_empty(need + 255, dtype=torch.uint8)
        return ws, (ws.data_ptr() + 255) & ~255, need
    except torch.OutOfMemoryError:
        if need == least:
            raise
    return _scratch(like, least, least)


def _enqueue_dense(problems, flags, stream):
    """Enqueues Dense problems -- (x, weights, biases, outs, epilogues, posts) each -- together, with the scratch memory
    that lets the library look palettized weights up ahead of the launch where X has many rows, and cut tiles along K where
    there are too few of them for the chip.  Returns their outputs."""
    host = _native or _host()
    if host is not None:
        got = host.dense(problems, flags, _scratch)
        if type(got) is list:
            return got
        if got is not None:
            _check(*(("dt_dense_qx_grouped_scratch_f16", got + 1000) if got < -500 else ("dt_dense_qx_grouped_ws_f16", got)))
    packed = [_marshal_dense(*p) for p in problems]
    groups = b"".join(g for _, g, _, _ in packed)  # (what they point to lives in `packed` until the call returns)
    n, L = len(packed), lib()
    need = L.dt_dense_scratch_bytes(n, groups) if any(M > _ROWS_MAX for _, _, _, M in packed) else 0
    like = problems[0][0]
    ws, at, got = _scratch(like, need, 0)
    if need and not got:  # the device is too full for copies of the weights; cutting takes less
        ws, at, got = _scratch(like, L.dt_dense_workspace_bytes(n, groups), 0)
    need = got
    if need:
        _check("dt_dense_qx_grouped_scratch_f16",
               L.dt_dense_qx_grouped_scratch_f16(_stream_ptr(stream), n, groups, flags, at, need))
    else:
        _check("dt_dense_qx_grouped_ws_f16", L.dt_dense_qx_grouped_ws_f16(_stream_ptr(stream), n, groups, flags, None, 0))
    return [_shape_outs(p[0], M, outs, p[3] is None) for p, (_, _, outs, M) in zip(problems, packed)]


def _shape_outs(x, M, outs, made):
    if made and x.dim() == 2:
        return outs
    lead = tuple(x.shape[:-1])
    return [o if o is None or o.shape[0] != M or not o.is_contiguous() else o.reshape(lead + (o.shape[-1],)) for o in outs]


def dense_multi(x, weights: Sequence[QxTensor], biases: Sequence[Optional[object]], outs=None, flags: int = 0,
                stream=None, epilogues: Optional[Sequence[Optional[HeadEpilogue]]] = None):
    """Several Dense ops that share the input, one launch (x_q / x_k / x_v).  `epilogues[i]` (optional) fuses the
    per-head RMSNorm / RoPE that follows projection i."""
    if stream is None:
        return _enqueue_dense([(x, weights, biases, outs, epilogues, None)], flags, None)[0]
    with _on(stream):
        return _enqueue_dense([(x, weights, biases, outs, epilogues, None)], flags, stream)[0]


ACT_NONE, ACT_GELU_TANH, ACT_SWISH, ACT_GELU_ERF = 0, 1, 2, 3


class DensePost:
    """Elementwise tail of one projection, in this order: scalar `scale`, fp16 `addend` [M, N] (the low-rank branch of a
    LoRADense, Models/LoRA.swift:117-140; a residual of an fp16 stream), fp16 `multiplicand` [M, N] (the gated
    feed-forward `fc10(x) .* GELU()(fc11(x))`, Models/UNet.swift:510-513), activation (ACT_*), per-feature fp16 gate [N], fp32 residual [M, N] that the
    result is accumulated into (`x + (y .* gate).to(of: x)`, Models/Flux1.swift:250).  A float32 gate multiplies in
    fp32 on the way into the residual instead (`x + out.to(of: x) .* chunks[2]`, Models/Wan.swift:159).  With
    `residual` given and `keep_output=False` the fp16 result itself is not written."""

    def __init__(self, activation: int = ACT_NONE, gate=None, residual=None, keep_output: bool = True,
                 scale: float = 1.0, addend=None, multiplicand=None):
        self.activation, self.gate, self.residual, self.keep_output = activation, gate, residual, keep_output
        self.scale, self.addend, self.multiplicand = scale, addend, multiplicand


def _pack_posts(posts, weights, M, Y, outs):
    """dt_dense_post array for the DensePost tails of one problem; clears Y / outs entries that only accumulate."""
    torch = _torch()
    vals = []
    for i, p in enumerate(posts):
        if p is None:
            vals += (ACT_NONE, 0, 0, 0, 1.0, 0, 0, 0, 0, 0)
            continue
        N = weights[i].shape[0]
        if float(p.scale) == 0.0:
            # dt_dense_post.scale == 0 means "no scale" in the C ABI (a zero-initialised struct is a plain Dense)
            raise ValueError("DensePost.scale must not be 0 (the library reads 0 as 'no scale'); a zero result "
                             "needs no Dense")
        g16 = g32 = None
        if p.gate is not None:
            if isinstance(p.gate, torch.Tensor) and p.gate.dtype == torch.float32:  # product formed in fp32 (Wan)
                if not p.gate.is_cuda:
                    raise TypeError("gate must be a CUDA tensor")
                g32 = p.gate
            else:
                g16 = _f16_cuda(p.gate, "gate")
            if p.gate.numel() != N or not p.gate.is_contiguous():
                raise ValueError("gate must hold one value per output feature")
        rp, ldr = 0, 0
        if p.residual is not None:
            r = p.residual
            if not (isinstance(r, torch.Tensor) and r.is_cuda and r.dtype == torch.float32):
                raise TypeError("residual must be a float32 CUDA tensor")
            r2 = r.reshape(-1, N) if r.dim() != 2 else r
            if r2.shape != (M, N) or r2.stride(1) != 1 or r2.data_ptr() != r.data_ptr():
                raise ValueError("residual must be an [M, N] view with contiguous rows")
            rp, ldr = r2.data_ptr(), r2.stride(0)
            if not p.keep_output:
                Y[i] = 0
                outs[i] = None
        ap, lda = 0, 0
        if p.addend is not None:
            a2 = _f16_cuda(p.addend, "addend")
            a2 = a2.reshape(-1, N) if a2.dim() != 2 else a2
            if a2.shape != (M, N) or a2.stride(1) != 1 or a2.data_ptr() != p.addend.data_ptr():
                raise ValueError("addend must be an [M, N] view with contiguous rows")
            ap, lda = a2.data_ptr(), a2.stride(0)
        mp, ldm = 0, 0
        if p.multiplicand is not None:
            m2 = _f16_cuda(p.multiplicand, "multiplicand")
            m2 = m2.reshape(-1, N) if m2.dim() != 2 else m2
            if m2.shape != (M, N) or m2.stride(1) != 1 or m2.data_ptr() != p.multiplicand.data_ptr():
                raise ValueError("multiplicand must be an [M, N] view with contiguous rows")
            mp, ldm = m2.data_ptr(), m2.stride(0)
        vals += (p.activation, 0 if g16 is None else g16.data_ptr(), rp, ldr, float(p.scale), ap, lda,
                 0 if g32 is None else g32.data_ptr(), mp, ldm)
    return struct.pack("=" + _FMT_POST * len(weights), *vals)


def dense_post(x, weights: Sequence[QxTensor], biases: Sequence[Optional[object]], posts: Sequence[Optional[DensePost]],
               outs=None, flags: int = 0, stream=None):
    """Dense ops sharing `x`, each followed by its DensePost tail inside the GEMM epilogue (the feed-forward's
    linear1 -> GELU and the gated residual additions of a transformer block).  Returns the fp16 outputs (None where
    a projection only accumulates into its residual)."""
    if stream is None:
        return _enqueue_dense([(x, weights, biases, outs, None, posts)], flags, None)[0]
    with _on(stream):
        return _enqueue_dense([(x, weights, biases, outs, None, posts)], flags, stream)[0]


def dense_grouped(problems: Sequence[dict], flags: int = 0, stream=None):
    """Independent Dense problems enqueued together (the context and image projections of a joint block).  Each
    problem is a dict with the arguments of dense_multi or dense_post: x, weights, biases, and optionally outs and
    either epilogues or posts.  Returns one list of outputs per problem (None where a projection only accumulates
    into its residual)."""
    if not problems:
        return []
    with _on(stream):
        return _enqueue_dense([(p["x"], p["weights"], p["biases"], p.get("outs"), p.get("epilogues"), p.get("posts"))
                               for p in problems], flags, stream)


class Dense:
    """Dense(count:noBias:flags:name:) -- y = x W^T + b with W [count, in] (Models/Flux1.swift:161-176)."""

    def __init__(self, count: int, noBias: bool = False, flags: int = 0, name: str = ""):
        self.count, self.noBias, self.flags, self.name = count, noBias, flags, name
        self.weight: Optional[QxTensor] = None
        self.bias = None

    def __call__(self, x, stream=None):
        if self.weight is None:
            raise RuntimeError(f"Dense {self.name!r}: weight not loaded")
        if self.weight.shape[0] != self.count:
            raise ValueError(f"Dense {self.name!r}: weight has {self.weight.shape[0]} rows, count is {self.count}")
        b = None if self.noBias else self.bias
        return dense_multi(x, [self.weight], [b], flags=self.flags, stream=stream)[0]


class LoRANetworkConfiguration:
    """rank / scale / highPrecision of the low-rank branch (Models/LoRA.swift:4-22)."""

    def __init__(self, rank: int, scale: float = 1.0, highPrecision: bool = False):
        self.rank, self.scale, self.highPrecision = rank, scale, highPrecision


class LoRADense:
    """LoRADense(count:configuration:noBias:flags:name:) -- dense(x) + up(scale * down(x)) with the palettized base
    left packed and the fp16 low-rank pair applied beside it (Models/LoRA.swift:85-142; running the LoRA separately
    is the preferred mode for quantized models, Models/UNetProtocol.swift:696-697).  dt_lora_dense_f16: the down
    projection, then the Dense kernel on the base, whose epilogue multiplies with `up` and adds the branch.  What that does not take (few
    rows, widths off the tiled kernels' grid, ranks for which it is slower, palettized pairs) goes out as Dense calls: base and down projection (with the
    scale in its epilogue), in one call or side by side, then the up projection, whose epilogue adds the base projection's
    result.  Every intermediate is rounded to fp16 as the reference's separate ops round, either way.  With
    `highPrecision` the pair is fp32 (`down.data` / `up.data` float32 tensors): the branch is computed as
    fp16(up(scale * down(float(x)))) in fp32 throughout (Models/LoRA.swift:117-139)."""

    def __init__(self, count: int, configuration: LoRANetworkConfiguration, noBias: bool = False, flags: int = 0,
                 name: str = ""):
        self.count, self.configuration, self.noBias, self.flags, self.name = count, configuration, noBias, flags, name
        self.weight: Optional[QxTensor] = None
        self.bias = None
        self.down: Optional[QxTensor] = None  # [rank, in] fp16
        self.up: Optional[QxTensor] = None    # [count, rank] fp16

    def _padded(self):
        """The pair with the rank padded by zero rows / columns to the tiled kernel's K granule (64): the zeros add
        nothing, so the results are the same bit for bit, and the up projection avoids the any-shape kernel."""
        # keyed on the identity of the pair's tensors (held here, so that their addresses cannot be handed to other
        # tensors while the cache lives), their in-place modification counters, the rank and the count
        src = (self.down.data, self.up.data)
        key = (self.down.data._version, self.up.data._version, self.configuration.rank, self.count,
               tuple(self.down.shape), tuple(self.up.shape))
        held = getattr(self, "_pad_src", None)
        if held is None or held[0] is not src[0] or held[1] is not src[1] or getattr(self, "_pad_key", None) != key:
            self._pad_src = src
            r = self.configuration.rank
            rp = (r + 63) // 64 * 64
            dn, up = self.down, self.up
            if rp != r and self.down.qbits == 16 and self.up.qbits == 16:
                torch = _torch()
                d = torch.zeros((rp, dn.shape[1]), dtype=torch.float16, device=dn.data.device)
                d[:r] = dn.data
                u = torch.zeros((self.count, rp), dtype=torch.float16, device=up.data.device)
                u[:, :r] = up.data
                dn, up = QxTensor(d, 16, 0, tuple(d.shape)), QxTensor(u, 16, 0, tuple(u.shape))
            self._pad_key, self._pad = key, (dn, up)
        return self._pad

    @staticmethod
    def _down_beside_base(M, K, weight, rank, capturing) -> bool:
        """Whether the down projection of M rows runs on a second stream beside the base projection.  On few workgroups it takes as
        long as K is, 60 us at 64 x 13824, unless it shares the base projection's launch.  Two streams cost a captured graph 12
        us, and a caller that waits for the host 65 (us, one call / two streams, rank 16: in a graph 64 x 13824 -> 5120 q6p 137 /
        93, 64 x 5120 -> 5120 63 / 54, 48 x 5120 -> 5120 56 / 51, 1024 x 12288 -> 3072 in blocks of 128 200 / 178, 64 x 3072 -> 3072 39
        / 39, with over 64 rows and blocks too small to be copied, means over the other sizes: K = 2048 .. 2303 0.96 of the time, 2304 ..
        3071 0.93, 1536 .. 2047 0.99; and the other way round 32 x 13824 -> 5120 88 / 91, 48 x 3072 -> 3072 34 / 37, 1024 x 1280 -> 1280 in blocks of 256 48 / 53;
        otherwise 64 x 13824 -> 5120 137 / 118, 1024 x 12288 -> 3072 in blocks of 128 190 / 170, and the other way round 64 x 12288 ->
        3072 113 / 131, 1024 x 3072 -> 3072 in blocks of 256 86 / 123)."""
        if weight.qbits == 16 or K < _BESIDE_INPUTS or M <= 32 or M * K < 64 * 3072:
            return False
        if not (K >= 3072 and M * K >= (60 * 13824 if M <= _ROWS_MAX else 8 << 20) or capturing()):
            return False
        if M <= _ROWS_MAX or weight.nib < _COPIED_NIB or 2 * weight.count > _COPIED_BYTES:
            return True
        # What can be copied mostly is, with that many rows, and asking takes the host 6 us of a layer that waits for it
        # (2800 x 3072 -> 512: 38 us, 45 with the question).  A graph asks once.
        if not capturing():
            return False
        # the call as the library sees it, as far as it looks at addresses
        ws = (_QxWeight * 2)(_QxWeight(4096, weight.qbits, weight.nib, weight.count), _QxWeight(4096, 16, 0, rank * K))
        ys, strides = (ctypes.c_void_p * 2)(4096, 4096), (ctypes.c_int64 * 2)(weight.shape[0], rank)
        at = ctypes.addressof
        group = (_DenseGroup * 1)(_DenseGroup(M, K, 4096, K, at(ws), 2, None, at(ys), at(strides), None, None))
        # nothing is copied where the call has no use for more than the workspace that cutting takes
        return lib().dt_dense_scratch_bytes(1, group) == lib().dt_dense_workspace_bytes(1, group)

    def _fused(self, x, b, post, stream):
        """The layer through dt_lora_dense_f16 as a list of its output, or None where it runs as Dense calls (us, those / this: 4608 x 3072
        -> 3072 q6p, rank 16, 104 / 95; 300 x 1280 -> 1280 q8p 28 / 22)."""
        high, rank = self.configuration.highPrecision, self.configuration.rank
        host = _native or _host()
        # (what the library would answer no to by its widths alone is not asked: 4 us of a small layer's 22)
        if host is None or not (high or rank <= 32) or not isinstance(x, _torch().Tensor) or x.dim() < 1 \
                or x.numel() <= _ROWS_MAX * x.shape[-1] or x.shape[-1] % 64:
            return None
        dn, up = (self.down, self.up) if high else self._padded()
        if dn.shape[1] != x.shape[-1] or dn.qbits not in (16, 32) or up.qbits not in (16, 32) \
                or dn.data.dtype != (_torch().float32 if high else _torch().float16):
            return None
        if not high:
            rank = (rank + 15) // 16 * 16  # (of the padded pair's 64)
        problem = (x, [self.weight], [b], None, None, None if post is None else [post])
        if stream is None and x.is_cuda and x.device.index != _torch().cuda.current_device():
            stream = _torch().cuda.current_stream(x.device)  # (a layer runs where x is)
        if stream is None:
            got = host.lora(problem, dn.data, up.data, rank, up.shape[1], self.configuration.scale, self.flags, _scratch)
        else:
            with _on(stream):
                got = host.lora(problem, dn.data, up.data, rank, up.shape[1], self.configuration.scale, self.flags, _scratch)
        if got is not None and type(got) is not list:
            _check("dt_lora_dense_f16", got)
        return got

    def __call__(self, x, post: Optional[DensePost] = None, stream=None):
        if self.weight is None:
            raise RuntimeError(f"LoRADense {self.name!r}: weight not loaded")
        b = None if self.noBias else self.bias
        # no matching LoRA keys: plain Dense.  A scale of zero makes the branch up(0 * down(x)) = 0 exactly, and
        # adding zero changes nothing: the same plain Dense
        if self.configuration.rank <= 0 or self.down is None or self.up is None or self.configuration.scale == 0:
            if post is None:
                return dense_multi(x, [self.weight], [b], flags=self.flags, stream=stream)[0]
            return dense_post(x, [self.weight], [b], [post], flags=self.flags, stream=stream)[0]
        if self.down.shape[0] != self.configuration.rank or self.up.shape != (self.count, self.configuration.rank):
            raise ValueError(f"LoRADense {self.name!r}: down / up shapes do not match rank and count")
        if self.weight.shape[0] != self.count:
            raise ValueError(f"LoRADense {self.name!r}: weight has {self.weight.shape[0]} rows, count is {self.count}")
        p = post or DensePost()
        if p.scale != 1.0 or p.addend is not None or p.multiplicand is not None:
            raise ValueError(f"LoRADense {self.name!r}: the tail may carry an activation, a gate and a residual only")
        got = self._fused(x, b, post, stream)
        if got is not None:
            return got[0]
        if self.configuration.highPrecision:
            return self._high_precision(x, b, p, stream)
        dn, up = self._padded()
        # Base and down projection share x.  One call puts them into one launch where the base weight is copied to fp16 for it (the
        # down projection's few tiles then run on compute units that the base projection leaves idle), and where they are
        # short the host has no time for more.  The up projection's epilogue adds the base projection's result and then runs
        # the tail.  (fp16(base) + fp16(branch) rounds the same whichever of the two is the addend.)
        down_post = DensePost(scale=self.configuration.scale)
        torch, K = _torch(), self.weight.shape[1]
        if K >= _BESIDE_INPUTS and self._down_beside_base(
                _f16_cuda(x, "x").numel() // K, K, self.weight, dn.shape[0],
                torch.cuda.is_current_stream_capturing if stream is None else lambda: _capturing(stream)):
            main = stream if stream is not None else torch.cuda.current_stream(x.device)
            side = _side_stream(x.device)
            side.wait_stream(main)
            down = dense_post(x, [dn], [None], [down_post], stream=side)[0]
            # (making a stream current that is so already costs 8 us)
            at = stream if x.device.index == torch.cuda.current_device() else main
            base = dense_multi(x, [self.weight], [b], flags=self.flags, stream=at)[0]
            main.wait_stream(side)  # every use of x and `down` on the side stream is ordered before what follows on `main`
            # `down` came from the side stream's pool and is read on `main`: its memory must not go back to that pool's
            # next user before `main` has passed this point
            down.record_stream(main)
        else:
            base, down = dense_post(x, [self.weight, dn], [b, None], [None, down_post], flags=self.flags, stream=stream)
        rows = x.dim() == 2  # (what has the shape already is not reshaped: 1 us each of 38)
        tail = DensePost(p.activation, p.gate, p.residual, p.keep_output, addend=base if rows else base.reshape(-1, self.count))
        out = dense_post(down, [up], [None], [tail], stream=stream)[0]
        return out if out is None or rows else out.reshape(*x.shape[:-1], self.count)


def _lora_high_precision(self, x, b, p, stream):
    """out = dense(x) + fp16(up32(scale * down32(float(x)))), then the tail: the fp32 branch, then the base projection with
    the sum in its epilogue."""
    torch = _torch()
    dn, up = self.down.data, self.up.data
    if dn.dtype != torch.float32 or up.dtype != torch.float32 or not dn.is_contiguous() or not up.is_contiguous():
        raise TypeError(f"LoRADense {self.name!r}: highPrecision takes contiguous float32 down / up weights")
    _f16_cuda(x, "x")
    K, r = x.shape[-1], self.configuration.rank
    if dn.shape[1] != K or self.weight.shape[1] != K:  # (the branch goes out ahead of the Dense, which would say so)
        raise ValueError(f"LoRADense {self.name!r}: weight or down do not match input width {K}")
    main = stream if stream is not None else torch.cuda.current_stream(x.device)
    with _on(main):  # a copy, if the view needs one, belongs on the caller's stream
        x2 = x if x.dim() == 2 else x.reshape(-1, K)
        if x2.stride(-1) != 1:
            x2 = x2.contiguous()
        M = x2.shape[0]
        # (on the caller's stream: the base projection waits for the branch, so there is nothing to run it beside)
        T = torch.empty((M, r), dtype=torch.float32, device=x.device)
        branch = torch.empty((M, self.count), dtype=torch.float16, device=x.device)
        st = lib().dt_lora_branch_f32_f16(_stream_ptr(main), M, K, x2.data_ptr(), x2.stride(0), dn.data_ptr(), r,
                                          up.data_ptr(), self.count, float(self.configuration.scale), T.data_ptr(),
                                          branch.data_ptr(), branch.stride(0))
        _check("dt_lora_branch_f32_f16", st)
    tail = DensePost(p.activation, p.gate, p.residual, p.keep_output, addend=branch)
    out = dense_post(x2, [self.weight], [b], [tail], flags=self.flags, stream=main)[0]
    return out if out is None or x.dim() == 2 else out.reshape(*x.shape[:-1], self.count)


LoRADense._high_precision = _lora_high_precision

_SIDE_STREAMS = {}


def _side_stream(device):
    """One extra stream per device (default priority) for work that may run beside the caller's stream."""
    torch = _torch()
    key = torch.device(device).index if torch.device(device).index is not None else torch.cuda.current_device()
    if key not in _SIDE_STREAMS:
        _SIDE_STREAMS[key] = torch.cuda.Stream(device=key)
    return _SIDE_STREAMS[key]


def _capturing(stream) -> bool:
    """Whether what is enqueued on `stream` becomes part of a graph."""
    with _on(stream):
        return _torch().cuda.is_current_stream_capturing()


def _view4(t) -> _View4:
    if t.dim() != 4 or t.stride(3) != 1:
        raise ValueError("expected a [B, S, H, D] tensor with contiguous D")
    return _View4(t.data_ptr(), t.stride(0), t.stride(1), t.stride(2))


def qk_norm_rope_(x, gamma=None, eps: float = 1e-6, norm_per_head: bool = True, rot=None, rot_pos0: int = 0,
                  post_scale: float = 1.0, stream=None):
    """In place on [B, S, H, D]: RMSNorm (per head, or over the whole row), then cmul with `rot`, then a scale."""
    _f16_cuda(x, "x")
    B, S, H, D = x.shape
    if rot is not None:
        _f16_cuda(rot, "rot")
        if rot.dim() != 2 or rot.shape[1] != D or not rot.is_contiguous() or rot.shape[0] < rot_pos0 + S:
            raise ValueError("rot must be a contiguous [>= rot_pos0 + S, D] table")
    if gamma is not None:
        _f16_cuda(gamma, "gamma")
        want = D if norm_per_head else H * D
        if gamma.numel() != want or not gamma.is_contiguous():
            raise ValueError(f"gamma must hold {want} elements")
    st = lib().dt_qk_norm_rope_f16(
        _stream_ptr(stream), _view4(x), B, S, H, D, None if gamma is None else gamma.data_ptr(), eps,
        1 if norm_per_head else 0, None if rot is None else rot.data_ptr(), rot_pos0, post_scale)
    _check("dt_qk_norm_rope_f16", st)
    return x


class RMSNorm:
    """RMSNorm(epsilon:axis:name:) on [B, S, H, D] (axis [3], per head) or [B, S, C] (axis [2], whole row)."""

    def __init__(self, epsilon: float, axis: Sequence[int], name: str = ""):
        self.epsilon, self.axis, self.name = epsilon, list(axis), name
        self.weight = None

    def __call__(self, x, stream=None):
        with _on(stream):
            y = x.clone()
            if x.dim() == 4 and self.axis == [3]:
                return qk_norm_rope_(y, self.weight, self.epsilon, True, stream=stream)
            if x.dim() == 3 and self.axis == [2]:
                qk_norm_rope_(_as_heads(y), self.weight, self.epsilon, False, stream=stream)
                return y
            raise DtError("RMSNorm", DT_NO_KERNEL)


MOD_F16, MOD_F32, MOD_AFFINE_F32 = 0, 1, 2


@_stream_scoped
def layernorm_modulate(x, scale=None, shift=None, epsilon: float = 1e-6, out=None, stream=None, affine: bool = False):
    """LayerNorm(epsilon:, axis: [last], elementwiseAffine: false) of the fp32 stream `x` [..., C], then the adaLN
    modulation, fp16 out.  fp16 `scale` / `shift` [C]: `norm(x).to(.Float16) .* scale + shift` (Models/Flux1.swift:
    172-173); fp32 ones: `(norm(x) .* (scale + 1) + shift).to(.Float16)` (Models/Wan.swift:217-221), or with
    `affine=True` the LayerNorm's own fp32 weight and bias, `norm(x) * scale + shift` (Models/Wan.swift:160-161)."""
    torch = _torch()
    if not (isinstance(x, torch.Tensor) and x.is_cuda and x.dtype == torch.float32):
        raise TypeError("x must be a float32 CUDA tensor")
    C = x.shape[-1]
    x2 = x.reshape(-1, C)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    M = x2.shape[0]
    mods = [t for t in (scale, shift) if t is not None]
    dtypes = {t.dtype for t in mods}
    if len(dtypes) > 1 or not dtypes <= {torch.float16, torch.float32}:
        raise TypeError("scale and shift must both be float16 or both be float32")
    for t in mods:
        if not t.is_cuda or t.numel() != C or not t.is_contiguous():
            raise ValueError("scale / shift must be contiguous CUDA vectors of C elements")
    mod = MOD_F32 if dtypes == {torch.float32} else MOD_F16
    if affine:
        if mod != MOD_F32:
            raise TypeError("affine LayerNorm takes float32 weight and bias")
        mod = MOD_AFFINE_F32
    if out is None:
        out = torch.empty((M, C), dtype=torch.float16, device=x.device)
    elif out.dtype != torch.float16 or out.shape != (M, C) or out.stride(1) != 1:
        raise ValueError("out must be an [M, C] float16 view with contiguous rows")
    st = lib().dt_layernorm_modulate_f16(_stream_ptr(stream), M, C, x2.data_ptr(), x2.stride(0),
                                         None if scale is None else scale.data_ptr(),
                                         None if shift is None else shift.data_ptr(), mod, float(epsilon),
                                         out.data_ptr(), out.stride(0))
    _check("dt_layernorm_modulate_f16", st)
    return out.reshape(tuple(x.shape[:-1]) + (C,)) if out.is_contiguous() else out


@_stream_scoped
def layernorm16(x, weight=None, bias=None, epsilon: float = 1e-5, out=None, stream=None):
    """LayerNorm(epsilon:, axis: [last]) with fp16 affine `weight` / `bias` [C] on an fp16 tensor [..., C], fp16 out
    (the norms of a UNet transformer block, Models/UNet.swift:530, 544, 554)."""
    host = _native or _host()
    if host is not None and out is None:
        got = host.layernorm16(x, weight, bias, epsilon)
        if type(got) is int:
            _check("dt_layernorm_f16", got)
        if got is not None:
            return got
    torch = _torch()
    _f16_cuda(x, "x")
    C = x.shape[-1]
    x2 = x.reshape(-1, C)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    M = x2.shape[0]
    for t in (weight, bias):
        if t is not None and (_f16_cuda(t, "weight / bias").numel() != C or not t.is_contiguous()):
            raise ValueError("weight / bias must be contiguous vectors of C elements")
    if out is None:
        out = torch.empty((M, C), dtype=torch.float16, device=x.device)
    elif out.dtype != torch.float16 or out.shape != (M, C) or out.stride(1) != 1:
        raise ValueError("out must be an [M, C] float16 view with contiguous rows")
    st = lib().dt_layernorm_f16(_stream_ptr(stream), M, C, x2.data_ptr(), x2.stride(0),
                                None if weight is None else weight.data_ptr(), None if bias is None else bias.data_ptr(),
                                float(epsilon), out.data_ptr(), out.stride(0))
    _check("dt_layernorm_f16", st)
    return out.reshape(tuple(x.shape[:-1]) + (C,)) if out.is_contiguous() else out


class LayerNorm:
    """LayerNorm(epsilon:axis:elementwiseAffine:) on the last axis.  Of an fp32 tensor, result cast to fp16
    (`xNorm1(x).to(.Float16)`, Models/Flux1.swift:172-173; with fp32 `weight` / `bias` `xNorm3(out).to(.Float16)`,
    Models/Wan.swift:160-161); of an fp16 tensor with fp16 `weight` / `bias` (Models/UNet.swift:530)."""

    def __init__(self, epsilon: float, axis: Sequence[int], elementwiseAffine: bool = True, name: str = ""):
        self.epsilon, self.axis, self.elementwiseAffine, self.name = epsilon, list(axis), elementwiseAffine, name
        self.weight = None
        self.bias = None

    def __call__(self, x, stream=None):
        if self.axis != [x.dim() - 1]:
            raise ValueError("LayerNorm: only the last axis is supported")
        if x.dtype == _torch().float16:
            if self.elementwiseAffine and (self.weight is None or self.bias is None):
                raise RuntimeError(f"LayerNorm {self.name!r}: weight / bias not loaded")
            return layernorm16(x, self.weight if self.elementwiseAffine else None,
                               self.bias if self.elementwiseAffine else None, self.epsilon, stream=stream)
        if not self.elementwiseAffine:
            return layernorm_modulate(x, None, None, self.epsilon, stream=stream)
        if self.weight is None or self.bias is None:
            raise RuntimeError(f"LayerNorm {self.name!r}: weight / bias not loaded")
        return layernorm_modulate(x, self.weight, self.bias, self.epsilon, stream=stream, affine=True)


def _as_heads(y):
    B, S, C = y.shape
    for d in (128, 64, 32, 16, 8, 2):
        if C % d == 0:
            return y.view(B, S, C // d, d)
    raise DtError("RMSNorm", DT_NO_KERNEL)


class Functional:
    @staticmethod
    def cmul(left, right, stream=None):
        """Complex multiply on adjacent pairs; `right` is the [1, S, 1, D] (or [S, D]) rotary table."""
        with _on(stream):
            y = left.clone()
            rot = right.reshape(-1, right.shape[-1]).contiguous()
            return qk_norm_rope_(y, None, 0.0, True, rot=rot, stream=stream)


class ScaledDotProductAttention:
    """ScaledDotProductAttention(scale:isCausal:hasAttentionMask:flags:multiHeadOutputProjectionFused:name:)
    (Models/Flux1.swift:228-232, Models/UNet.swift:122-155).  Inputs [B, S, H, D]; returns [B, Sq, Hq, D], or
    [B, Sq, Hq*D] when the unify-heads projection is fused (then `.weight` [HD, HD] fp16 and `.bias`)."""

    def __init__(self, scale: float, isCausal: bool = False, hasAttentionMask: bool = False, flags: int = 0,
                 multiHeadOutputProjectionFused: bool = False, name: str = ""):
        if isCausal or hasAttentionMask:
            raise DtError("ScaledDotProductAttention(isCausal/hasAttentionMask)", DT_NO_KERNEL)
        self.scale, self.flags, self.fused, self.name = float(scale), flags, multiHeadOutputProjectionFused, name
        self.weight = None
        self.bias = None

    def __call__(self, queries, keys, values, stream=None):
        return sdpa_segments([queries], [keys], [values], self.scale,
                             Wo=self.weight if self.fused else None, bo=self.bias if self.fused else None,
                             stream=stream)


@_stream_scoped
def sdpa_segments(q_segs, k_segs, v_segs, scale, gamma_q=None, gamma_k=None, rot_q=None, rot_k=None,
                  eps: float = 1e-6, Wo=None, bo=None, out=None, stream=None, static_scratch: bool = False):
    """Attention over a joint sequence given as segments (text || image without a concat).
    gamma_q / gamma_k: per-segment per-head RMSNorm weights (or None); rot_*: [S, D] tables.
    static_scratch: stage through the library's fixed per-GPU array (dt_sdpa_f16_static) instead of a workspace
    allocated here; with `out` given the call then allocates nothing.  Requests beyond STATIC_SCRATCH_BYTES raise
    DtError(DT_OOM); calls that may overlap on one GPU must not both use it."""
    host = _native or _host()
    if host is not None and not static_scratch and Wo is None and bo is None:
        got = host.sdpa(q_segs, k_segs, v_segs, scale, gamma_q or None, gamma_k or None, rot_q, rot_k, eps, out, _scratch)
        if type(got) is int:
            _check("dt_sdpa_f16", got)
        if got is not None:
            return got
    torch = _torch()
    L = lib()
    for t in list(q_segs) + list(k_segs) + list(v_segs):
        _f16_cuda(t, "q/k/v")
    B, _, Hq, D = q_segs[0].shape
    Hk = k_segs[0].shape[2]
    Sq = sum(t.shape[1] for t in q_segs)
    Skv = sum(t.shape[1] for t in k_segs)
    nq, nk = len(q_segs), len(k_segs)
    gq = gamma_q or [None] * nq
    gk = gamma_k or [None] * nk

    def segs(ts, gs):
        arr = (_Segment * len(ts))()
        for i, (t, g) in enumerate(zip(ts, gs)):
            arr[i] = _Segment(_view4(t), t.shape[1], None if g is None else _f16_cuda(g, "gamma").data_ptr())
        return arr

    qa, ka, va = segs(q_segs, gq), segs(k_segs, gk), segs(v_segs, [None] * nk)
    # only K is staged for a fused norm / rotation (the queries are handled inside the attention kernel)
    prep = any(g is not None for g in gk) or rot_k is not None
    fused = Wo is not None
    if out is None:
        shape = (B, Sq, Hq * D) if fused else (B, Sq, Hq, D)
        out = torch.empty(shape, dtype=torch.float16, device=q_segs[0].device)
    if fused:
        ov = _View4(out.data_ptr(), out.stride(0), out.stride(1), 0)
    else:
        ov = _view4(out)
    rq = None if rot_q is None else _f16_cuda(rot_q, "rot_q").data_ptr()
    rk = None if rot_k is None else _f16_cuda(rot_k, "rot_k").data_ptr()
    wo = None if Wo is None else _f16_cuda(Wo, "Wo").data_ptr()
    bo_p = None if bo is None else _f16_cuda(bo, "bo").data_ptr()
    if static_scratch:
        st = L.dt_sdpa_f16_static(_stream_ptr(stream), B, Hq, Hk, D, nq, qa, nk, ka, va, rq, rk, eps, ov, scale, wo, bo_p)
        _check("dt_sdpa_f16_static", st)
        return out
    need = L.dt_sdpa_workspace_bytes(B, Hq, Hk, D, Sq, Skv, int(prep), int(fused))
    ws, at = None, None
    if need:
        staged = sum((b + 255) // 256 * 256 for b in (prep * B * Skv * Hk * D * 2, fused * B * Sq * Hq * D * 2))
        ws, at, need = _scratch(out, need, staged)
    st = L.dt_sdpa_f16(_stream_ptr(stream), B, Hq, Hk, D, nq, qa, nk, ka, va, rq, rk, eps, ov, scale, wo, bo_p, at, need)
    _check("dt_sdpa_f16", st)
    return out


# --------------------------------------------------------------------------
# rotary tables (host side, as in the reference: computed on the CPU in double,
# stored as float, cast to fp16 on upload)
# --------------------------------------------------------------------------

def _axis_table(pos: np.ndarray, dim: int) -> np.ndarray:
    k = np.arange(dim // 2, dtype=np.float64)
    theta = pos.astype(np.float64)[:, None] * 1.0 / np.power(10000.0, k * 2 / dim)
    out = np.empty((pos.size, dim), dtype=np.float32)
    out[:, 0::2] = np.cos(theta)
    out[:, 1::2] = np.sin(theta)
    return out


def Flux1RotaryPositionEmbedding(height: int, width: int, tokenLength: int, referenceSizes=(), channels: int = 128):
    """[tokenLength + height*width + sum(ref), channels] float32 table (Models/Flux1.swift:5-119), heads = 1."""
    assert channels % 16 == 0
    dim0, dim1 = channels // 8, channels * 7 // 16
    pos0 = [np.zeros(tokenLength + height * width)]
    ys, xs = np.divmod(np.arange(height * width), width)
    pos1 = [np.zeros(tokenLength), ys]
    pos2 = [np.zeros(tokenLength), xs]
    h = w = 0
    for (rh, rw) in referenceSizes:
        hoff = woff = 0
        if rh + h > rw + w:
            woff = w
        else:
            hoff = h
        ys, xs = np.divmod(np.arange(rh * rw), rw)
        pos0.append(np.ones(rh * rw))
        pos1.append(ys + hoff)
        pos2.append(xs + woff)
        h, w = max(h, rh + hoff), max(w, rw + woff)
    p0, p1, p2 = (np.concatenate(p) for p in (pos0, pos1, pos2))
    return np.concatenate([_axis_table(p0, dim0), _axis_table(p1, dim1), _axis_table(p2, dim1)], axis=1)


def WanRotaryPositionEmbedding(height: int, width: int, time: int, channels: int = 128):
    """[time*height*width, channels] float32 table (Models/Wan.swift:5-46), heads = 1."""
    assert channels % 16 == 0
    dim1 = (channels // 6) * 2
    dim0 = channels - 2 * dim1
    i = np.arange(time * height * width)
    t, rem = np.divmod(i, height * width)
    y, x = np.divmod(rem, width)
    return np.concatenate([_axis_table(t, dim0), _axis_table(y, dim1), _axis_table(x, dim1)], axis=1)


# --------------------------------------------------------------------------
# work units (Models/InstructionCount/InstructionCount.swift:4-17)
# --------------------------------------------------------------------------

def DenseInstructionCount(rows: int, input: int, output: int) -> int:
    assert rows >= 0 and input >= 0 and output >= 0
    return rows * output * input


def ScaledDotProductAttentionInstructionCount(batchSize, heads, headDimension, sequenceDimensionA,
                                              sequenceDimensionB) -> int:
    return batchSize * heads * (2 * headDimension + 5) * sequenceDimensionA * sequenceDimensionB
