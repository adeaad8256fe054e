"""ctypes binding of libmoegemm.so (the C ABI declared in include/moegemm.h).

The library is built in-tree next to this file (``csrc/Makefile`` or ``__graft_entry__.build()``).
Nothing here falls back to another implementation: when the library or a GPU is missing, every
launch raises ``RuntimeError``, mirroring the reference's "Triton with an active CUDA driver is
required" error (reference kernels/grouped_gemm.py:626-627, kernels/matmul.py:342-343).
"""

from __future__ import annotations

import ctypes
import os
import threading
from functools import lru_cache
from pathlib import Path

LIBRARY_PATH = Path(__file__).resolve().with_name("libmoegemm.so")

ABI_VERSION = 9
OK = 0
ERR_INVALID = -1
ERR_NO_KERNEL = -2
ERR_LAUNCH = -3

DTYPE_F16 = 0
DTYPE_BF16 = 1
DTYPE_F32 = 2
PRECISION_IEEE = 0
PRECISION_TF32 = 1

DTYPE_NAMES = {DTYPE_F16: "fp16", DTYPE_BF16: "bf16", DTYPE_F32: "fp32"}

_i32 = ctypes.c_int32
_i64 = ctypes.c_int64
_vp = ctypes.c_void_p

# Exported symbol -> (restype, argtypes).  tests/test_native_abi.py checks this against the header.
SIGNATURES = {
    "moegemm_abi_version": (ctypes.c_int, []),
    "moegemm_last_error": (ctypes.c_char_p, []),
    "moegemm_kernel_count": (ctypes.c_int, [ctypes.c_int]),
    "moegemm_kernel_info": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, ctypes.POINTER(_i32)]),
    "moegemm_grouped_gemm": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "moegemm_grouped_gemm_stealing": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _i32, _vp],
    ),
    "moegemm_grouped_gemm_swiglu": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "moegemm_kernel_swiglu": (ctypes.c_int, [ctypes.c_int, ctypes.c_int]),
    "moegemm_splitk_workspace_bytes": (ctypes.c_int, [_i32, _i32, _i32, _i32, ctypes.POINTER(_i64)]),
    "moegemm_matmul_splitk": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_matmul_splitk_any": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_grouped_gemm_splitk_any": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_kernel_layouts": (ctypes.c_int, [ctypes.c_int, ctypes.c_int]),
    "moegemm_matmul_splitk_noalloc": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "moegemm_grouped_gemm_splitk": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_streamk_workspace_bytes": (ctypes.c_int, [_i32, _i32, _i32, _i32, ctypes.POINTER(_i64)]),
    "moegemm_matmul_streamk": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_grouped_gemm_streamk": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
         _i32, _i32, _i32, _vp, _i64, _i32, _vp],
    ),
    "moegemm_grouped_mm_offs": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "moegemm_grouped_mm_offs_swiglu": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "moegemm_grouped_mm_offs_stealing": (
        ctypes.c_int,
        [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _i32, _vp],
    ),
    "moegemm_matmul": (
        ctypes.c_int,
        [_vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64, _i32, _i32,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
}


class NativeUnavailable(RuntimeError):
    """libmoegemm.so is missing or does not match this binding."""


@lru_cache(maxsize=1)
def library() -> ctypes.CDLL:
    path = Path(os.environ.get("MOEGEMM_LIBRARY", LIBRARY_PATH))
    if not path.exists():
        raise NativeUnavailable(
            f"native library {path} is not built; run `make -C moe-gemm-parallel-bench_amd/csrc` "
            "or __graft_entry__.build()"
        )
    try:
        lib = ctypes.CDLL(str(path))
    except OSError as exc:  # missing ROCm runtime, wrong architecture, ...
        raise NativeUnavailable(f"cannot load {path}: {exc}") from exc
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    version = lib.moegemm_abi_version()
    if version != ABI_VERSION:
        raise NativeUnavailable(f"{path} has ABI version {version}, this binding expects {ABI_VERSION}")
    return lib


def available() -> bool:
    try:
        library()
        return True
    except NativeUnavailable:
        return False


def last_error() -> str:
    return library().moegemm_last_error().decode("utf-8", "replace")


def check(status: int) -> None:
    """Map a native status to the reference's exception types."""
    if status == OK:
        return
    message = last_error()
    if status == ERR_INVALID:
        raise ValueError(message)
    raise RuntimeError(message)


@lru_cache(maxsize=None)
def compiled_kernels(dtype_code: int) -> tuple[tuple[int, int, int, int, int, int, int], ...]:
    """(block_m, block_n, block_k, num_warps, num_stages, lds_bytes, waves_m) per compiled kernel."""
    lib = library()
    out = (_i32 * 7)()
    rows = []
    for index in range(lib.moegemm_kernel_count(dtype_code)):
        check(lib.moegemm_kernel_info(dtype_code, index, out))
        rows.append(tuple(int(v) for v in out))
    return tuple(rows)


@lru_cache(maxsize=None)
def swiglu_tiles(dtype_code: int) -> frozenset:
    """Tile keys (block_m, block_n, block_k, num_warps, num_stages) that can run the SwiGLU epilogue."""
    lib = library()
    keys = set()
    for index, row in enumerate(compiled_kernels(dtype_code)):
        status = lib.moegemm_kernel_swiglu(dtype_code, index)
        if status < 0:
            check(status)
        if status == 1:
            keys.add(tuple(row[:5]))
    return frozenset(keys)


# Operand layouts of the LDS-DMA kernels: 0 row-major, else these bits; GENERAL runs the general kernel, and
# STRIDED (an operand without a unit stride) the element-wise one.
GENERAL = -1
STRIDED = -2
A_TRANSPOSED = 1
B_TRANSPOSED = 2
# vector_layout argument of the grouped launches per layout (MOEGEMM_LAYOUT_* for transposed operands).
LAYOUT_FLAGS = {STRIDED: 0x40000, GENERAL: 0, 0: 1, 1: 0x10001, 2: 0x20001, 3: 0x30001}


GENERAL_SPLIT = 4  # moegemm_kernel_layouts' bit for a general tile with a split-K kernel


@lru_cache(maxsize=None)
def layout_tiles(dtype_code: int, layout: int) -> frozenset:
    """Tile keys whose LDS-DMA kernel is compiled for an operand layout (``GENERAL_SPLIT``: whose
    general tile has a split-K kernel)."""
    lib = library()
    keys = set()
    for index, row in enumerate(compiled_kernels(dtype_code)):
        mask = lib.moegemm_kernel_layouts(dtype_code, index)
        if mask < 0:
            check(mask)
        if mask >> layout & 1:
            keys.add(tuple(row[:5]))
    return frozenset(keys)


def split_tiles(dtype_code: int, layout: int) -> frozenset:
    """Tile keys that can split K over operands of this layout."""
    if layout == STRIDED:
        return frozenset()
    return layout_tiles(dtype_code, GENERAL_SPLIT if layout == GENERAL else layout)


_COPIED_PAST_K = 1024  # K rows past the matrix that a tile's zero slices may address


def _operand_layout(tensor, x_dim: int) -> int:
    """0 when one operand's rows run along K, 1 when they run along its M or N dimension ``x_dim``
    (either way in aligned 16-byte chunks within the kernels' 32-bit offsets), else -1."""
    extent, k = tensor.shape[x_dim], tensor.shape[1 - x_dim]
    sx, sk = tensor.stride(x_dim), tensor.stride(1 - x_dim)
    if tensor.data_ptr() % 16:
        return -1
    if sk == 1 and sx % 8 == 0 and sx >= k and k % 8 == 0 and PANEL_ROWS * sx * 2 < _TWO_GIB:
        return 0
    if sx == 1 and sk % 8 == 0 and sk >= extent and extent % 8 == 0 and (k + _COPIED_PAST_K) * sk * 2 < _TWO_GIB:
        return 1
    return -1


def strided_or(layout: int, a, b) -> int:
    """``layout``, or STRIDED for general operands of which one has no unit stride: no tile stages such an
    operand in chunks, or splits its K."""
    return STRIDED if layout == GENERAL and (1 not in a.stride() or 1 not in b.stride()) else layout


def transposed_layout(a, b, c) -> int:
    """Layout of 16-bit operands of which at least one is transposed (1, 2 or 3), else GENERAL: the
    library's rule (api.hip fast_layout) after its row-major one."""
    n = b.shape[1]
    scm, scn = c.stride()
    if scn != 1 or n % 8 or scm % 4 or scm < n or c.data_ptr() % 8 or PANEL_ROWS * scm * 2 >= _TWO_GIB:
        return GENERAL
    la, lb = _operand_layout(a, 0), _operand_layout(b, 1)
    if la < 0 or lb < 0:
        return GENERAL
    return (A_TRANSPOSED if la == 1 else 0) | (B_TRANSPOSED if lb == 0 else 0) or GENERAL


@lru_cache(maxsize=4096)
def splitk_workspace_bytes(tiles: int, splits: int, block_m: int, block_n: int) -> int:
    out = _i64(0)
    check(library().moegemm_splitk_workspace_bytes(tiles, splits, block_m, block_n, ctypes.byref(out)))
    return int(out.value)


def streamk_workspace_bytes(tail_tiles: int, grid: int, block_m: int, block_n: int) -> int:
    out = _i64(0)
    check(library().moegemm_streamk_workspace_bytes(tail_tiles, grid, block_m, block_n, ctypes.byref(out)))
    return int(out.value)


PANEL_ROWS = 256  # the largest block_m of the menu
_TWO_GIB = 1 << 31


def panels_fit(k: int, sam: int, sbk: int, scm: int) -> bool:
    """Byte-range limits of the LDS-DMA kernels' 32-bit buffer offsets, as the library checks them:
    A and C are addressed through one resource per tile of at most PANEL_ROWS rows (any number of
    rows in all), B through one resource running to the end of the [k, n] matrix."""
    return PANEL_ROWS * sam * 2 < _TWO_GIB and PANEL_ROWS * scm * 2 < _TWO_GIB and k * sbk * 2 < _TWO_GIB


def streamk_tail(tiles: int, grid: int, k: int, block_k: int) -> int:
    """Tail tiles of a stream-K launch (0 when stream-K does not apply): the remainder r of
    ``tiles`` over a ``grid`` of workgroups, so the whole tiles fill exact rounds and the r tail
    tiles are spread over every workgroup.  0 when there is no remainder, or when the tail is too
    thin for the library's limit of 64 pieces per tile."""
    if tiles <= 0 or grid <= 0:
        return 0
    tail = tiles % grid
    if tail == 0:
        return 0
    kt = -(-k // block_k)
    per_run = tail * kt // grid
    if per_run < 1 or -(-kt // per_run) + 1 > 64:
        return 0
    return tail


# Split-K workspaces, one per (device, stream).  A workspace is never released once handed out, so
# a captured graph that recorded its address stays valid; a larger need allocates a new one.
_SPLITK_WORKSPACES: dict[tuple[int, int], list] = {}
_SPLITK_MIN_BYTES = 32 << 20


def _refuse_allocation_under_capture(what: str) -> None:
    """A buffer made inside graph capture would be zeroed only when the graph replays, so an eager
    launch on that stream before the first replay would read stale counters: refuse instead."""
    import torch

    if torch.cuda.is_available() and torch.cuda.is_current_stream_capturing():
        raise RuntimeError(f"the {what} for this stream does not exist yet and cannot be created during graph "
                           "capture; make the first call on this stream outside capture")


_SPLITK_MAX_SPLITS, _SPLITK_MAX_TILES = 64, 65536  # the split-K launches' limits (moegemm.h)

# Split-K scratch of operands outside the row-major 16-bit layout (fp32, unaligned, transposed).  They must
# run wherever a launch without scratch would, so theirs is kept apart from the workspaces above: only eager
# launches use it, in the order of the one stream it belongs to, and no captured graph holds its address
# (two graphs captured on one stream, or a graph beside eager calls on its capture stream, may replay at
# once).  Each buffer is made on its own stream and used on no other, so dropping one is safe at any
# time: its memory is reused in that stream's order.  At most 33 streams hold one (torch's stream pool and
# the default stream), as large as the last growth asked for.
_EAGER_SCRATCH: dict[tuple[int, int], object] = {}
_EAGER_SCRATCH_STREAMS = 33
_EAGER_SCRATCH_LOCK = threading.Lock()


def capturing() -> bool:
    """Whether the current stream records a graph."""
    import torch

    return torch.cuda.is_current_stream_capturing()


def eager_scratch(device, stream_handle: int, tiles: int, splits: int, block_m: int, block_n: int):
    """Zero-initialised split-K scratch for one launch on the current stream of ``device``; None when the
    launch has to run whole: past the library's limits, under graph capture, or out of memory."""
    import torch

    if splits > _SPLITK_MAX_SPLITS or tiles > _SPLITK_MAX_TILES or capturing():
        return None
    nbytes = splitk_workspace_bytes(tiles, splits, block_m, block_n)
    key = (torch.device(device).index or 0, int(stream_handle))
    held = _EAGER_SCRATCH.get(key)
    if held is not None and held.numel() >= nbytes:
        return held
    try:
        buffer = torch.zeros(nbytes, dtype=torch.uint8, device=device)
    except torch.cuda.OutOfMemoryError:
        return None
    with _EAGER_SCRATCH_LOCK:
        _EAGER_SCRATCH.pop(key, None)
        while len(_EAGER_SCRATCH) >= _EAGER_SCRATCH_STREAMS:
            _EAGER_SCRATCH.pop(next(iter(_EAGER_SCRATCH)))
        _EAGER_SCRATCH[key] = buffer
    return buffer


class TuningScratch:
    """What a tuner's timings use in place of ``eager_scratch``: one buffer for all candidates, which run one
    after the other, given back when the ``with`` block ends.  The tuner's own captured graphs may use it:
    each is replayed and dropped before the next candidate runs."""

    def __init__(self):
        import torch

        self._home = torch.cuda.current_stream()
        self._buffer = None

    def __enter__(self):
        return self

    def __exit__(self, *error):
        import torch

        if self._buffer is not None:
            torch.cuda.synchronize(self._buffer.device)  # whatever a failed candidate left on another stream
            self._buffer = None

    def __call__(self, device, stream_handle: int, tiles: int, splits: int, block_m: int, block_n: int):
        import torch

        if splits > _SPLITK_MAX_SPLITS or tiles > _SPLITK_MAX_TILES:
            return None
        nbytes = splitk_workspace_bytes(tiles, splits, block_m, block_n)
        if self._buffer is None or self._buffer.numel() < nbytes:
            if capturing():
                return None
            torch.cuda.synchronize(device)  # as in __exit__
            self._buffer = None
            with torch.cuda.stream(self._home):  # one stream's memory, whichever stream times
                self._buffer = torch.zeros(nbytes, dtype=torch.uint8, device=device)
            torch.cuda.current_stream(device).wait_stream(self._home)
        return self._buffer


def splitk_workspace(device, stream_handle: int, nbytes: int):
    """A zero-initialised uint8 device tensor of at least ``nbytes`` for this device and stream."""
    import torch

    key = (torch.device(device).index or 0, int(stream_handle))
    held = _SPLITK_WORKSPACES.setdefault(key, [])
    if not held or held[-1].numel() < nbytes:
        _refuse_allocation_under_capture("split-K workspace")
        held.append(torch.zeros(max(nbytes, _SPLITK_MIN_BYTES), dtype=torch.uint8, device=device))
    return held[-1]


# Work-stealing tile queues, one per (device, stream), zeroed once and never released (launches
# leave them zero; a captured graph keeps a valid address).
QUEUE_BYTES = 4352
NOALLOC_SCRATCH_BYTES = 64 * 1024 * 1024 + 256 * 1024  # MOEGEMM_NOALLOC_SCRATCH_BYTES
TILE_SCHEDULES = ("static", "stealing")
# Schedules of homogeneous grouped launches: also "streamk" (whole tiles in exact rounds, then a
# stream-K tail; fp16/bf16 vector layouts).
GROUPED_SCHEDULES = TILE_SCHEDULES + ("streamk",)
_TILE_QUEUES: dict[tuple[int, int], object] = {}


def tile_queue(device, stream_handle: int):
    """The zero-initialised MOEGEMM_QUEUE_BYTES device buffer for this device and stream."""
    import torch

    key = (torch.device(device).index or 0, int(stream_handle))
    queue = _TILE_QUEUES.get(key)
    if queue is None:
        _refuse_allocation_under_capture("work-stealing tile queue")
        queue = torch.zeros(QUEUE_BYTES // 4, dtype=torch.int32, device=device)
        _TILE_QUEUES[key] = queue
    return queue


def dtype_code(dtype) -> int:
    import torch

    codes = {torch.float16: DTYPE_F16, torch.bfloat16: DTYPE_BF16, torch.float32: DTYPE_F32}
    if dtype not in codes:
        raise ValueError(f"unsupported dtype {dtype}; expected float16, bfloat16 or float32")
    return codes[dtype]


def precision_code(input_precision: str, dtype_code_value: int) -> int:
    if input_precision not in ("ieee", "tf32"):
        raise ValueError(f"input_precision must be 'ieee' or 'tf32', got {input_precision!r}")
    # Like tl.dot, TF32 only changes fp32 operands; 16-bit operands are exact in any mode.
    if input_precision == "tf32" and dtype_code_value == DTYPE_F32:
        return PRECISION_TF32
    return PRECISION_IEEE


def current_stream_handle(device) -> int:
    import torch

    # The raw handle: building a torch.cuda.Stream object for it took about 2 us of a 11 us call.
    index = device.index
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)
