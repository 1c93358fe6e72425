"""The gfx950 kernels as torch ops, over the C ABI of libflash_lab_hip.so.

This module replaces the reference's compiled op registry (csrc/bindings.cpp:7-42). Importing it
loads the kernel library and the native ops over it (csrc/torch_ops.cpp, libflash_lab_torch.so) and
registers, under torch.ops.flash_lab, ops with the reference's names and schemas:

    attention_mma_pipelined / attention_mma
        (Tensor q, Tensor k, Tensor v, bool causal, float softmax_scale) -> (Tensor, Tensor)
    decode_splitkv / decode_inplace
        (Tensor q, Tensor k_cache, Tensor v_cache, Tensor seq_lens, float softmax_scale,
         int num_splits) -> (Tensor, Tensor)
    decode_splitkv_paged / decode_inplace_paged: the same with block_tables after seq_lens
    smoke_axpy(Tensor x, Tensor y, float alpha) -> Tensor
    mma_tile_test(Tensor a, Tensor b, bool trans_b) -> Tensor

Each op allocates its outputs (and its workspace) with torch on the input's device, passes the
current stream, and raises RuntimeError with the library's message when a call fails. Nothing here
synchronizes, reads seq_lens on the host or allocates outside torch's caching allocator, so the ops
can be captured in a HIP graph. If a library cannot be loaded, importing this module raises
ImportError; there is no other code path. Also here: the library's own entry points through ctypes,
for what the ops do not offer (plans, knobs, the allocation-free decode).
"""

from __future__ import annotations

import contextlib
import ctypes
import functools
import math
import os
from pathlib import Path

import torch

LIB_NAME = "libflash_lab_hip.so"
LIB_PATH = Path(os.environ.get("FLASH_LAB_HIP_LIB", Path(__file__).with_name(LIB_NAME)))

ERR_WORKSPACE = 4  # enum fl_status
DTYPE_CODES = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


class AttnParams(ctypes.Structure):
    """fl_attn_params of include/flash_lab_hip.h."""

    _fields_ = [
        ("q", ctypes.c_void_p),
        ("k", ctypes.c_void_p),
        ("v", ctypes.c_void_p),
        ("o", ctypes.c_void_p),
        ("lse", ctypes.c_void_p),
        *[
            (f"{t}_{s}_stride", ctypes.c_int64)
            for t in ("q", "k", "v", "o")
            for s in ("batch", "seq", "head")
        ],
        ("batch", ctypes.c_int32),
        ("seqlen_q", ctypes.c_int32),
        ("seqlen_k", ctypes.c_int32),
        ("heads", ctypes.c_int32),
        ("heads_kv", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("causal", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("softmax_scale", ctypes.c_double),
    ]


class DecodeParams(ctypes.Structure):
    """fl_decode_params of include/flash_lab_hip.h."""

    _fields_ = [
        ("q", ctypes.c_void_p),
        ("k_cache", ctypes.c_void_p),
        ("v_cache", ctypes.c_void_p),
        ("o", ctypes.c_void_p),
        ("lse", ctypes.c_void_p),
        ("seq_lens", ctypes.c_void_p),
        ("q_batch_stride", ctypes.c_int64),
        ("q_head_stride", ctypes.c_int64),
        ("k_batch_stride", ctypes.c_int64),
        ("k_seq_stride", ctypes.c_int64),
        ("k_head_stride", ctypes.c_int64),
        ("v_batch_stride", ctypes.c_int64),
        ("v_seq_stride", ctypes.c_int64),
        ("v_head_stride", ctypes.c_int64),
        ("o_batch_stride", ctypes.c_int64),
        ("o_head_stride", ctypes.c_int64),
        ("batch", ctypes.c_int32),
        ("heads", ctypes.c_int32),
        ("heads_kv", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("max_seqlen", ctypes.c_int32),
        ("num_splits", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("softmax_scale", ctypes.c_double),
        ("workspace", ctypes.c_void_p),
        ("workspace_bytes", ctypes.c_size_t),
        ("block_tables", ctypes.c_void_p),
        ("block_tables_stride", ctypes.c_int64),
        ("page_size", ctypes.c_int32),
        ("num_blocks", ctypes.c_int32),
    ]


# Every symbol include/flash_lab_hip.h declares, with its ctypes signature.
SIGNATURES = {
    "fl_attention_fwd": (ctypes.c_int, [ctypes.POINTER(AttnParams), ctypes.c_void_p]),
    "fl_attention_plan": (
        ctypes.c_int,
        [
            ctypes.POINTER(AttnParams),
            ctypes.c_int32,
            ctypes.c_int32,
            ctypes.POINTER(ctypes.c_int32),
            ctypes.POINTER(ctypes.c_size_t),
        ],
    ),
    "fl_attention_fwd_split": (
        ctypes.c_int,
        [
            ctypes.POINTER(AttnParams),
            ctypes.c_int32,
            ctypes.c_int32,
            ctypes.c_void_p,
            ctypes.c_size_t,
            ctypes.c_void_p,
        ],
    ),
    "fl_decode_plan": (
        ctypes.c_int,
        [
            ctypes.POINTER(DecodeParams),
            ctypes.c_int32,
            ctypes.c_int32,
            ctypes.c_int32,
            ctypes.POINTER(ctypes.c_int32),
            ctypes.POINTER(ctypes.c_size_t),
        ],
    ),
    "fl_decode_schedule": (
        ctypes.c_int,
        [
            ctypes.POINTER(DecodeParams),
            ctypes.c_int32,
            ctypes.POINTER(ctypes.c_int32),
            ctypes.POINTER(ctypes.c_int32),
            ctypes.POINTER(ctypes.c_size_t),
        ],
    ),
    "fl_decode_balanced": (
        ctypes.c_int,
        [ctypes.POINTER(DecodeParams), ctypes.c_int32, ctypes.c_void_p],
    ),
    "fl_decode": (ctypes.c_int, [ctypes.POINTER(DecodeParams), ctypes.c_void_p]),
    "fl_decode_noalloc": (ctypes.c_int, [ctypes.POINTER(DecodeParams), ctypes.c_void_p]),
    "fl_smoke_axpy": (
        ctypes.c_int,
        [
            ctypes.c_void_p,
            ctypes.c_void_p,
            ctypes.c_float,
            ctypes.c_void_p,
            ctypes.c_int64,
            ctypes.c_void_p,
        ],
    ),
    "fl_mfma_tile_test": (
        ctypes.c_int,
        [
            ctypes.c_void_p,
            ctypes.c_void_p,
            ctypes.c_void_p,
            ctypes.c_int32,
            ctypes.c_int32,
            ctypes.c_void_p,
        ],
    ),
    "fl_set_knob": (ctypes.c_int, [ctypes.c_int32, ctypes.c_int64]),
    "fl_get_knob": (ctypes.c_int64, [ctypes.c_int32]),
    "fl_last_error": (ctypes.c_char_p, []),
    "fl_version": (ctypes.c_char_p, []),
}


def load_library(path: Path = LIB_PATH) -> ctypes.CDLL:
    """Loads the library and attaches the C signatures. torch is imported first, so the HIP
    runtime the library links against is the one torch already loaded."""
    if not path.exists():
        raise ImportError(
            f"{path} is missing; build it with `python flash-attention-lab_amd/csrc/build.py`"
        )
    try:
        lib = ctypes.CDLL(str(path))
    except OSError as exc:
        raise ImportError(f"could not load {path}: {exc}") from exc
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    return lib


LIB = load_library()

TORCH_LIB_PATH = Path(__file__).with_name("libflash_lab_torch.so")
# The library functions that fl_torch_bind takes, in its order.
TORCH_BOUND = ("fl_attention_plan", "fl_attention_fwd_split", "fl_decode_plan", "fl_decode_schedule", "fl_decode",
               "fl_decode_balanced", "fl_last_error")


def load_torch_ops(path: Path = TORCH_LIB_PATH) -> ctypes.CDLL:
    """Loads the native ops (which registers them with torch) and binds them to LIB's functions."""
    if not path.exists():
        raise ImportError(
            f"{path} is missing; build it with `python flash-attention-lab_amd/csrc/build.py`"
        )
    try:
        ops = ctypes.CDLL(str(path))
    except OSError as exc:
        raise ImportError(f"could not load {path}: {exc}") from exc
    ops.fl_torch_bind.restype = None
    ops.fl_torch_bind.argtypes = [ctypes.c_void_p] * len(TORCH_BOUND)
    ops.fl_torch_bind(*(ctypes.cast(getattr(LIB, name), ctypes.c_void_p) for name in TORCH_BOUND))
    return ops



def _check(rc: int) -> None:
    if rc != 0:
        raise RuntimeError(LIB.fl_last_error().decode())


# Routing overrides of the library (enum fl_knob): test and experiment hooks that pin a call to
# one of the kernels. None restores the built-in rule.
KNOBS = {"prefill_pp_min_wg": 0, "decode_mfma_min_group": 1, "decode_wg_per_cu": 2,
         "decode_mfma_span": 3, "prefill_causal_stream": 4}


def set_knob(name: str, value: int | None) -> None:
    _check(LIB.fl_set_knob(KNOBS[name], -1 if value is None else int(value)))


def get_knob(name: str) -> int | None:
    value = LIB.fl_get_knob(KNOBS[name])
    return None if value == -1 else value


@contextlib.contextmanager
def knob(name: str, value: int | None):
    """Sets a routing knob for the duration of the block, then restores its previous value."""
    previous = get_knob(name)
    set_knob(name, value)
    try:
        yield
    finally:
        set_knob(name, previous)


def _stream(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


class _on_device:
    """Makes `device` current for the call when it is not already (the role of the reference's
    OptionalCUDAGuard)."""

    def __init__(self, device: torch.device):
        self.device = device
        self.ctx = None

    def __enter__(self):
        if self.device.index is not None and self.device.index != torch.cuda.current_device():
            self.ctx = torch.cuda.device(self.device)
            self.ctx.__enter__()

    def __exit__(self, *exc):
        if self.ctx is not None:
            self.ctx.__exit__(*exc)


@functools.lru_cache(maxsize=None)
def cu_count(index: int) -> int:
    return torch.cuda.get_device_properties(index).multi_processor_count


def _require(cond: bool, message: str, *args) -> None:
    """Raises RuntimeError(message % args) unless cond; the message is only formatted on failure
    (these checks run on every op call)."""
    if not cond:
        raise RuntimeError(message % args if args else message)


def _check_cuda(**tensors: torch.Tensor) -> None:
    for name, x in tensors.items():
        _require(x.is_cuda, "%s must be a CUDA tensor", name)


# ----------------------------------------------------------------------------------------------
# Decode


def _decode_params(q, k_cache, v_cache, seq_lens, o, lse, softmax_scale,
                   block_tables=None) -> DecodeParams:
    batch, heads, head_dim = q.shape
    if block_tables is not None:
        # [num_blocks, page_size, H_kv, D] caches: the batch strides are block strides.
        p = _decode_params(q, k_cache, v_cache, seq_lens, o, lse, softmax_scale)
        p.max_seqlen = block_tables.shape[1] * k_cache.shape[1]
        p.block_tables = block_tables.data_ptr()
        p.block_tables_stride = block_tables.stride(0)
        p.page_size = k_cache.shape[1]
        p.num_blocks = k_cache.shape[0]
        return p
    return DecodeParams(
        q.data_ptr(),
        k_cache.data_ptr(),
        v_cache.data_ptr(),
        o.data_ptr(),
        lse.data_ptr(),
        seq_lens.data_ptr(),
        q.stride(0),
        q.stride(1),
        *k_cache.stride()[:3],
        *v_cache.stride()[:3],
        o.stride(0),
        o.stride(1),
        batch,
        heads,
        k_cache.shape[2],
        head_dim,
        k_cache.shape[1],
        1,
        DTYPE_CODES[q.dtype],
        float(softmax_scale),
        None,
        0,
    )


def decode_noalloc(q, k_cache, v_cache, seq_lens, o, lse, softmax_scale: float, num_splits: int,
                   block_tables=None) -> int:
    """fl_decode_noalloc on caller-provided outputs o [B, H, D] and lse [B, H]: the split workspace
    is the library's own scratch array, so nothing is allocated. num_splits 0 takes the planned
    count. Returns the split count used. The arguments are taken as valid (the public ops check
    them); this is the allocation-free path for callers that manage their own buffers."""
    p = _decode_params(q, k_cache, v_cache, seq_lens, o, lse, softmax_scale, block_tables)
    index = q.device.index if q.device.index is not None else torch.cuda.current_device()
    splits, ws_bytes = ctypes.c_int32(), ctypes.c_size_t()
    _check(LIB.fl_decode_plan(ctypes.byref(p), int(num_splits), 1, cu_count(index),
                              ctypes.byref(splits), ctypes.byref(ws_bytes)))
    p.num_splits = splits.value
    with _on_device(q.device):
        _check(LIB.fl_decode_noalloc(ctypes.byref(p), _stream(q.device)))
    return splits.value


def decode_schedule(batch, heads, heads_kv, head_dim, max_seqlen, dtype, page_size=0,
                    cu_count_=256) -> tuple[int, int, int]:
    """(num_splits, workgroups, workspace bytes) of a decode call that asks for no split count:
    workgroups > 0 (and num_splits 0) for a balanced one. Host-only."""
    p = DecodeParams()
    p.batch, p.heads, p.heads_kv, p.head_dim, p.max_seqlen = batch, heads, heads_kv, head_dim, max_seqlen
    p.dtype = DTYPE_CODES[dtype]
    if page_size:  # only whether the cache is paged, and its page size, count here
        p.block_tables, p.page_size, p.num_blocks = 16, page_size, 1
    splits, wgs, ws = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_size_t()
    _check(LIB.fl_decode_schedule(ctypes.byref(p), cu_count_, ctypes.byref(splits), ctypes.byref(wgs),
                                  ctypes.byref(ws)))
    return splits.value, wgs.value, ws.value


def decode_plan(batch, heads, heads_kv, head_dim, max_seqlen, dtype, num_splits=0,
                allow_splits=True, cu_count_=256) -> tuple[int, int]:
    """(num_splits, workspace bytes) the library picks for a decode shape; host-only."""
    p = DecodeParams()
    p.batch, p.heads, p.heads_kv, p.head_dim, p.max_seqlen = batch, heads, heads_kv, head_dim, max_seqlen
    p.dtype = DTYPE_CODES[dtype]
    splits = ctypes.c_int32()
    ws = ctypes.c_size_t()
    _check(LIB.fl_decode_plan(ctypes.byref(p), num_splits, int(allow_splits), cu_count_,
                              ctypes.byref(splits), ctypes.byref(ws)))
    return splits.value, ws.value


# ----------------------------------------------------------------------------------------------
# Op registration


def _register() -> None:
    lib = "flash_lab"

    @torch.library.custom_op(
        f"{lib}::smoke_axpy", mutates_args=(), device_types="cuda",
        schema="(Tensor x, Tensor y, float alpha) -> Tensor",
    )
    def smoke_axpy(x: torch.Tensor, y: torch.Tensor, alpha: float) -> torch.Tensor:
        _check_cuda(x=x, y=y)
        _require(x.dtype == torch.float32 and y.dtype == torch.float32, "x and y must be fp32")
        _require(x.shape == y.shape, "x and y must have the same shape")
        xc, yc = x.contiguous(), y.contiguous()
        out = torch.empty_like(xc)
        with _on_device(x.device):
            _check(
                LIB.fl_smoke_axpy(
                    xc.data_ptr(), yc.data_ptr(), float(alpha), out.data_ptr(), xc.numel(),
                    _stream(x.device),
                )
            )
        return out

    @smoke_axpy.register_fake
    def _(x, y, alpha):
        return torch.empty_like(x, memory_format=torch.contiguous_format)

    @torch.library.custom_op(
        f"{lib}::mma_tile_test", mutates_args=(), device_types="cuda",
        schema="(Tensor a, Tensor b, bool trans_b) -> Tensor",
    )
    def mma_tile_test(a: torch.Tensor, b: torch.Tensor, trans_b: bool) -> torch.Tensor:
        _check_cuda(a=a, b=b)
        _require(a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16, "a and b must be bf16")
        _require(a.dim() == 2 and a.shape[0] == 16 and a.shape[1] in (16, 32, 64),
                 "a must be [16, K]")
        k = a.shape[1]
        want = (k, 16) if trans_b else (16, k)
        _require(tuple(b.shape) == want, "b must be [K, 16] with trans_b, else [16, K]")
        ac, bc = a.contiguous(), b.contiguous()
        c = torch.empty((16, 16), dtype=torch.float32, device=a.device)
        with _on_device(a.device):
            _check(
                LIB.fl_mfma_tile_test(
                    ac.data_ptr(), bc.data_ptr(), c.data_ptr(), k, int(bool(trans_b)),
                    _stream(a.device),
                )
            )
        return c

    @mma_tile_test.register_fake
    def _(a, b, trans_b):
        return a.new_empty((16, 16), dtype=torch.float32)


# The attention and decode ops, native (csrc/torch_ops.cpp): loading the library registers them, and
# they call the functions of the kernel library loaded above.
TORCH_LIB = load_torch_ops()
_register()

OPS = (
    "attention_mma_pipelined",
    "attention_mma",
    "decode_splitkv",
    "decode_inplace",
    "decode_splitkv_paged",
    "decode_inplace_paged",
    "smoke_axpy",
    "mma_tile_test",
)


def default_scale(head_dim: int) -> float:
    return 1.0 / math.sqrt(head_dim)
