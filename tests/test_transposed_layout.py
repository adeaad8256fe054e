"""Operand layouts of the LDS-DMA kernels: the Python rule against the library's, and the kernels on
transposed operands (linear weights [N, K], backward products) against exact integer products."""

from __future__ import annotations

import random

import pytest
import torch

from kernels import _native

CODES = {torch.float16: _native.DTYPE_F16, torch.bfloat16: _native.DTYPE_BF16}


def test_layout_rule_matches_the_library():
    """The split-K entry checks layouts before its workspace, so operands it accepts fail on the
    missing workspace instead, and nothing is launched."""
    from kernels.matmul import _operand_layout

    rng = random.Random(5)
    storage = torch.empty(1 << 20, dtype=torch.bfloat16)
    seen = set()
    for _ in range(4000):
        m, n, k = (rng.choice((8, 40, 64, 77, 136)) for _ in range(3))
        k += 128  # two K ranges of the tile below, so the workspace is needed
        views = []
        for rows, cols in ((m, k), (k, n), (m, n)):
            swap = rng.random() < (0.5 if cols != n or rows != m else 0.05)
            extent = rows if swap else cols
            pitch = extent + rng.choice((0, 0, 8, -extent % 8, 1, 4))
            inner = 2 if rng.random() < 0.05 else 1
            strides = (inner, pitch) if swap else (pitch, inner)
            views.append(storage.as_strided((rows, cols), strides, rng.choice((0, 0, 8, 4, 1))))
        a, b, c = views
        layout = _operand_layout(a, b, c)
        status = _native.library().moegemm_matmul_splitk_any(
            a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, *a.stride(), *b.stride(), *c.stride(),
            _native.DTYPE_BF16, 0, 128, 256, 64, 8, 8, 3, 2, 0, None, 0, 0, None)
        assert status == _native.ERR_INVALID
        accepted = "workspace" in _native.last_error()
        assert accepted != ("vector layout" in _native.last_error())
        assert accepted == (layout >= 0), (layout, a.stride(), b.stride(), c.stride(), m, n, k)
        # What the row-major entry refused before stays refused there.
        status = _native.library().moegemm_matmul_splitk(
            a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, *a.stride(), *b.stride(), *c.stride(),
            _native.DTYPE_BF16, 64, 64, 64, 8, 4, 4, 2, 0, None, 0, 0, None)
        assert ("workspace" in _native.last_error()) == (layout == 0)
        seen.add(layout)
    assert seen == {-1, 0, 1, 2, 3}


def test_compiled_layouts_are_reported():
    assert _native.layout_tiles(_native.DTYPE_F32, 0) == frozenset()
    for code in CODES.values():
        every = {tuple(row[:5]) for row in _native.compiled_kernels(code)}
        assert _native.layout_tiles(code, 0) == every
        for layout in (1, 2, 3):
            assert _native.layout_tiles(code, layout) and _native.layout_tiles(code, layout) <= every
    assert _native.library().moegemm_kernel_layouts(_native.DTYPE_BF16, 10_000) < 0


def _operand(rows, cols, transposed, pad, dtype, gen):
    """Integers in {-1, 0, 1} as a row-major or transposed view whose padding and neighbourhood hold
    NaN: a copy that took anything past the operand's extents would show."""
    shape = (cols, rows) if transposed else (rows, cols)
    storage = torch.full((shape[0] + 16, shape[1] + pad), float("nan"), device="cuda", dtype=dtype)
    values = torch.randint(-1, 2, shape, generator=gen, device="cuda", dtype=torch.int32).to(dtype)
    view = storage[:shape[0], :shape[1]]
    view.copy_(values)
    return view.t() if transposed else view


def _cases():
    # (m, k, n): one chunk; partial tiles in every direction; several tiles, K past the stages and
    # no multiple of the slice; M = 1 and odd M (rows along K), odd K (both operands along M and N).
    for layout in (1, 2, 3):
        for shape in ((8, 8, 8), (40, 72, 136), (264, 328, 520), (512, 1032, 256)):
            yield layout, shape
    yield from ((2, (1, 136, 24)), (2, (77, 264, 72)), (1, (72, 77, 136)), (1, (264, 1, 264)), (1, (8, 641, 8)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(CODES), ids=str)
@pytest.mark.parametrize("layout,shape", list(_cases()))
def test_transposed_operands_every_tile(layout, shape, dtype):
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels.matmul import KernelConfig, _operand_layout, last_matmul_split, launch_matmul

    m, k, n = shape
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    a = _operand(m, k, bool(layout & 1), 8, dtype, gen)
    b = _operand(k, n, bool(layout & 2), 16, dtype, gen)
    expected = (a.double() @ b.double()).to(dtype)  # exact in fp32, so rounded once either way
    for tile in sorted(_native.layout_tiles(CODES[dtype], layout)):
        for splits in (1, 3):
            print(f"transposed layout={layout} shape={shape} tile={tile} splits={splits}", flush=True)
            guard = torch.full((m + 2, n + 8), float("nan"), device="cuda", dtype=dtype)
            c = guard[1:m + 1, :n]
            assert _operand_layout(a, b, c) == layout
            launch_matmul(a, b, c, KernelConfig(*tile[:3], 2, *tile[3:]), autotune=False, split_k=splits,
                          b_stream=splits & 1)
            torch.cuda.synchronize()
            assert last_matmul_split() == splits
            assert torch.equal(c, expected), (tile, splits)
            assert torch.isnan(guard[:, n:]).all() and torch.isnan(guard[0]).all() and torch.isnan(guard[-1]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [1, 2, 3])
@pytest.mark.parametrize("schedule", ["static", "stealing"])
def test_transposed_groups(layout, schedule):
    """Unequal problems of one layout take its kernels; a group that mixes layouts stays general."""
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels.grouped_gemm import _group_layout, launch_grouped, workspace_from_tensors

    gen = torch.Generator(device="cuda").manual_seed(layout)
    shapes = [(72, 136, 264), (8, 264, 520), (264, 72, 136), (136, 520, 8)]
    for mixed in (False, True):
        a, b, c = [], [], []
        for i, (m, k, n) in enumerate(shapes):
            lay = 0 if mixed and i == 1 else layout
            a.append(_operand(m, k, bool(lay & 1), 8, torch.bfloat16, gen))
            b.append(_operand(k, n, bool(lay & 2), 8, torch.bfloat16, gen))
            c.append(torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16))
        ws = workspace_from_tensors(a, b, c)
        assert _group_layout(ws, _native.DTYPE_BF16) == (-1 if mixed else layout)
        print(f"transposed group layout={layout} schedule={schedule} mixed={mixed}", flush=True)
        launch_grouped(ws, autotune=False, tile_schedule=schedule)
        torch.cuda.synchronize()
        for x, y, z in zip(a, b, c):
            assert torch.equal(z, (x.double() @ y.double()).to(z.dtype))


def _column_view_group(count, m, n, device):
    """K = 1 and A the transposed view of a [1, M] tensor: contiguous to torch, M-contiguous by its strides."""
    a = [torch.arange(m, device=device).sub(3 + i).to(torch.bfloat16).view(1, m).t() for i in range(count)]
    b = [torch.arange(n, device=device).remainder(5 + i).to(torch.bfloat16).view(1, n) for i in range(count)]
    return a, b, [torch.full((m, n), float("nan"), device=device, dtype=torch.bfloat16) for _ in range(count)]


def test_homogeneous_groups_are_never_transposed():
    from kernels.grouped_gemm import _group_layout, workspace_from_tensors

    a, b, c = _column_view_group(2, 64, 128, "cpu")
    assert a[0].stride() == (1, 64) and _native.transposed_layout(a[0], b[0], c[0]) == 1
    ws = workspace_from_tensors(a, b, c)
    assert ws.homogeneous and _group_layout(ws, _native.DTYPE_BF16) == _native.GENERAL
    unequal = workspace_from_tensors([a[0], a[1][:56]], b, [c[0], c[1][:56]])
    assert not unequal.homogeneous and _group_layout(unequal, _native.DTYPE_BF16) == 1


@pytest.mark.parametrize("flag", [0x10001, 0x20001, 0x30001])
def test_homogeneous_launches_refuse_a_transposed_promise(flag):
    """Checked before the workspace, so nothing is launched."""
    lib, tables, tile = _native.library(), (64, 64, 64), (128, 128, 64, 8, 4, 4)
    for status in (
            lib.moegemm_grouped_gemm(*tables, None, None, 2, 64, 128, 256, 1, 0, _native.DTYPE_BF16, 0, *tile, 0, flag,
                                     0, None),
            lib.moegemm_grouped_gemm_splitk(*tables, 2, 64, 128, 256, _native.DTYPE_BF16, *tile, 2, 0, flag, None, 0,
                                            0, None),
            lib.moegemm_grouped_gemm_splitk_any(*tables, 2, 64, 128, 256, _native.DTYPE_BF16, 0, *tile, 2, 0, flag,
                                                None, 0, 0, None),
            lib.moegemm_grouped_gemm_streamk(*tables, 2, 64, 128, 256, _native.DTYPE_BF16, *tile, 1, 1, flag, None, 0,
                                             0, None)):
        assert status == _native.ERR_INVALID and "homogeneous groups are row-major" in _native.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("autotune", [False, True])
def test_column_view_groups_launch(autotune):
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels.grouped_gemm import launch_grouped, workspace_from_tensors

    a, b, c = _column_view_group(2, 64, 128, "cuda")
    ws = workspace_from_tensors(a, b, c)
    print(f"column view group autotune={autotune}", flush=True)
    launch_grouped(ws, autotune=autotune)
    torch.cuda.synchronize()
    for x, y, z in zip(a, b, c):
        assert torch.equal(z, (x.double() @ y.double()).to(z.dtype))


def test_untuned_ragged_configs_are_compiled():
    from kernels.matmul import _menu, select_ragged_config

    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        for mean in (1, 4, 5, 64, 256, 257, 4096):
            for n in (1, 64, 128, 129, 1023, 1024, 7168):
                for groups in (2, 32):
                    assert select_ragged_config(mean, n, 512, dtype, groups=groups).tile_key in _menu(dtype)


def test_unequal_groups_default_to_the_ragged_rule():
    from kernels.grouped_gemm import build_grouped_workspace
    from kernels.matmul import select_config, select_ragged_config

    ragged = build_grouped_workspace([(8, 64, 256), (40, 64, 256), (72, 64, 256)], torch.bfloat16, device="cpu")
    assert ragged.config == select_ragged_config(40, 256, 64, torch.bfloat16, groups=3, rows=(8, 40, 72))
    # Tiles that fit one round of 256 CUs: (1 + 3 + 5) M tiles of 16 rows by 4 (28, 29) N tiles of 64.
    for n, tile in ((256, (16, 64)), (1792, (16, 64)), (1856, (64, 64))):
        few = build_grouped_workspace([(8, 64, n), (40, 64, n), (72, 64, n)], torch.bfloat16, device="cpu")
        assert (few.config.block_m, few.config.block_n) == tile
    # 512 columns, 2 N tiles: 129 problems of up to 128 rows are two rounds of 256 CUs in either tile; of
    # 129 to 256 rows three rounds of 128-row tiles against two, and 128 such problems two against one.
    for tall, count, block_m in ((128, 129, 128), (256, 129, 128), (256, 128, 256)):
        ws = build_grouped_workspace([(tall - i % 2, 8, 512) for i in range(count)], torch.bfloat16, device="cpu")
        assert ws.config.block_m == block_m, (tall, count)
    equal = build_grouped_workspace([(40, 64, 256)] * 3, torch.bfloat16, device="cpu")
    assert equal.config == select_config(40, 256, 64, torch.bfloat16)


@pytest.mark.parametrize("mean,mib,expected", [(64, 257, 1), (65, 4096, 0), (4, 256, 0), (1, 384, 0), (1, 512, 1)])
def test_untuned_b_stream_rule(mean, mib, expected):
    from kernels.matmul import ragged_b_stream

    assert ragged_b_stream(mean, mib << 20) == expected


@pytest.mark.gpu
def test_untuned_routed_groups_stream_large_weights():
    """Above the cache's size all three untuned routes run non-temporal copies; a named policy, a named
    config and small weights keep theirs; the results are the same bytes."""
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels import grouped_mm
    from kernels.grouped_gemm import launch_grouped, workspace_from_tensors
    from kernels.grouped_mm import last_grouped_mm_b_stream, last_grouped_mm_config

    gen = torch.Generator(device="cuda").manual_seed(9)
    rows = [5, 0, 40, 3, 16, 1, 0, 31]
    g, k, n = len(rows), 4096, 4608  # 288 MiB
    a = torch.randint(-1, 2, (sum(rows), k), generator=gen, device="cuda").to(torch.bfloat16)
    b = torch.randint(-1, 2, (g, k, n), generator=gen, device="cuda", dtype=torch.int8).to(torch.bfloat16)
    offs = torch.tensor(rows, device="cuda").cumsum(0).to(torch.int32)
    print("untuned b_stream, expert-sorted", flush=True)
    streamed = grouped_mm(a, b, offs, autotune=False)
    assert last_grouped_mm_b_stream() == 1
    plain = grouped_mm(a, b, offs, autotune=False, b_stream=0)
    assert last_grouped_mm_b_stream() == 0
    grouped_mm(a, b, offs, config=last_grouped_mm_config())
    assert last_grouped_mm_b_stream() == 0
    grouped_mm(a, b[:, :, :4096].contiguous(), offs, autotune=False)  # 256 MiB
    assert last_grouped_mm_b_stream() == 0
    first, spans = 0, []
    for e, count in enumerate(rows):
        if count:
            spans.append((e, first, first + count))
        first += count
    expected = torch.cat([(a[x:y].double() @ b[e].double()).to(a.dtype) for e, x, y in spans])
    assert torch.equal(streamed, expected) and torch.equal(plain, expected)
    print("untuned b_stream, pointer group", flush=True)
    c = torch.empty_like(expected)
    spans = spans + [(1, 0, 5), (6, 5, 45)]  # every expert's weights
    outs = [c[x:y] for _, x, y in spans[:-2]] + [torch.empty_like(c[x:y]) for _, x, y in spans[-2:]]
    ws = workspace_from_tensors([a[x:y] for _, x, y in spans], [b[e] for e, _, _ in spans], outs)
    launch_grouped(ws, autotune=False)
    assert ws.b_stream == 1
    torch.cuda.synchronize()
    assert torch.equal(c, expected)
