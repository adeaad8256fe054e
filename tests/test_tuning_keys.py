"""Tuned options are kept by operand layout: operands of one shape and one set of strides run other kernels
when their alignment differs."""

from __future__ import annotations

import contextlib

import pytest
import torch

from kernels import _native, grouped_gemm, matmul


def _offset(rows, cols, dtype, skip):
    return torch.zeros(rows * cols + 8, dtype=dtype)[skip:skip + rows * cols].view(rows, cols)


@pytest.fixture
def tuned(monkeypatch):
    """Launches of CPU operands through a tuner that takes its first candidate; yields the keys it filled."""
    library = _native.library()

    class Nothing:
        def __getattr__(self, name):
            return (lambda *args: 0) if name.startswith(("moegemm_matmul", "moegemm_grouped")) else getattr(library, name)

    monkeypatch.setattr(_native, "library", Nothing)
    monkeypatch.setattr(_native, "current_stream_handle", lambda device: 7)
    monkeypatch.setattr(_native, "TuningScratch", contextlib.nullcontext)
    monkeypatch.setattr(_native, "eager_scratch", lambda *args: None)
    monkeypatch.setattr(_native, "capturing", lambda: False)
    monkeypatch.setattr(matmul, "_device_signature", lambda device: 950256)
    monkeypatch.setattr(matmul, "_validate_matrices", lambda a, b, c: (a.shape[0], b.shape[1], a.shape[1]))
    for module in (matmul, grouped_gemm):
        monkeypatch.setattr(module, "_require_runtime", lambda tensor=None: None)
        monkeypatch.setattr(module, "_tune", lambda options, launch, twin=None, fallback=None: (options[0], options[0]))
    monkeypatch.setattr(grouped_gemm, "_check_workspace", lambda ws: _native.dtype_code(ws.a[0].dtype))
    monkeypatch.setattr(matmul, "_AUTOTUNE_CACHE", {})
    monkeypatch.setattr(grouped_gemm, "_GROUPED_AUTOTUNE_CACHE", {})


def test_aligned_and_unaligned_matrices_are_tuned_apart(tuned):
    m, k, n = 64, 256, 64
    b, c = _offset(k, n, torch.bfloat16, 0), _offset(m, n, torch.bfloat16, 0)
    for count, skip in enumerate((1, 0, 2, 8), 1):  # 2 and 4 bytes past alignment: GENERAL; 0 and 16: row-major
        a = _offset(m, k, torch.bfloat16, skip)
        matmul.launch_matmul(a, b, c)
        assert len(matmul._AUTOTUNE_CACHE) == min(count, 2)
    # Transposed storage: its candidates are the tiles compiled for it, whatever an unaligned view chose.
    wt = [_offset(n, k, torch.bfloat16, skip).t() for skip in (1, 0)]
    for w in wt:
        matmul.launch_matmul(_offset(m, k, torch.bfloat16, 0), w, c)
    assert len(matmul._AUTOTUNE_CACHE) == 4
    assert list(matmul._AUTOTUNE_CACHE.values())[-1][0].tile_key in _native.layout_tiles(_native.DTYPE_BF16, 2)


def test_aligned_and_unaligned_groups_are_tuned_apart(tuned):
    for count, skip in enumerate((1, 0, 2, 8), 1):
        a = [_offset(64, 256, torch.float16, skip) for _ in range(2)]
        b, c = ([_offset(*shape, torch.float16, 0) for _ in range(2)] for shape in ((256, 64), (64, 64)))
        grouped_gemm.launch_grouped(grouped_gemm.workspace_from_tensors(a, b, c))
        assert len(grouped_gemm._GROUPED_AUTOTUNE_CACHE) == min(count, 2)


def test_repeated_untuned_calls_search_no_menu(tuned, monkeypatch):
    """An untuned call's tile is looked up, not searched for again: the search took as long as a small launch."""
    operands = []
    for dtype, flip in ((torch.bfloat16, True), (torch.bfloat16, False), (torch.float32, False)):
        b = _offset(104, 264, dtype, 0).t() if flip else _offset(264, 104, dtype, 0)
        operands.append((_offset(24, 264, dtype, 0), b, _offset(24, 104, dtype, 0)))
    for a, b, c in operands:
        matmul.launch_matmul(a, b, c, autotune=False)

    def searched(dtype=None):
        raise AssertionError("the menu was searched")

    monkeypatch.setattr(matmul, "_menu", searched)
    for a, b, c in operands:
        matmul.launch_matmul(a, b, c, autotune=False)
