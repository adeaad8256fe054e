"""Which operands the general tile stages in chunks with unsigned 32-bit offsets: the rule alone on the
CPU, and operands with negative pitches (reversed views, which only C callers can pass) on the GPU."""

from __future__ import annotations

import random
import subprocess
from pathlib import Path

import pytest
import torch

CSRC = Path(__file__).resolve().parents[1] / "moe-gemm-parallel-bench_amd" / "csrc"
PROGRAM = """
#include <cstdio>
#include "general_route.h"
int main() {
  int f32, es, bm, bn; long long m, n, k, s[4];
  while (std::scanf("%d %d %d %d %lld %lld %lld %lld %lld %lld %lld", &f32, &es, &bm, &bn, &m, &n, &k, s, s + 1, s + 2,
                    s + 3) == 11) {
    const moegemm::ChunkRoute r = moegemm::chunk_route(f32, es, bm, bn, m, n, k, s[0], s[1], s[2], s[3]);
    std::printf("%d %d %d %d %d\\n", r.a_rows, r.a_cols, r.b_rows, r.b_cols, r.chunked());
  }
}
"""
TILES = ((256, 256, 64), (256, 128, 32), (128, 256, 64), (64, 64, 64), (16, 64, 128), (16, 512, 64))


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    folder = tmp_path_factory.mktemp("route")
    (folder / "route.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), "-o", str(folder / "route"), str(folder / "route.cpp")],
                   check=True)

    def run(rows):
        text = "\n".join(" ".join(map(str, row)) for row in rows)
        done = subprocess.run([str(folder / "route")], input=text, capture_output=True, text=True, check=True)
        return [tuple(int(v) for v in line.split()) for line in done.stdout.splitlines()]

    return run


def test_chunked_offsets_stay_inside_32_bits(route):
    """Every offset of an accepted operand, in exact integers, is what unsigned 32-bit arithmetic gives."""
    rng = random.Random(2)
    pitches = (-(1 << 33), -4096, -1, 0, 1, 7, 4096, (1 << 21) - 1, 1 << 21, 1 << 22, 1 << 23, 1 << 24, 1 << 31, 1 << 33)
    rows = []
    for _ in range(20000):
        bm, bn, _ = rng.choice(TILES)
        f32 = rng.random() < 0.5
        m, n, k = (rng.choice((1, 7, 8, 300, 70000)) for _ in range(3))
        strides = [rng.choice(pitches + (1,) * 14) for _ in range(4)]
        rows.append((int(f32), 4 if f32 else 2, bm, bn, m, n, k, *strides))
    slices = {(bm, bn): bk for bm, bn, bk in TILES}
    accepted = 0
    for row, (a_rows, a_cols, b_rows, b_cols, chunked) in zip(rows, route(rows)):
        _, es, bm, bn, m, n, k, sam, sak, sbk, sbn = row
        assert chunked == ((a_rows or a_cols) and (b_rows or b_cols))
        for rows_k, rows_x, x, pitch_k, pitch_x in ((a_rows, a_cols, bm, sam, sak), (b_rows, b_cols, bn, sbn, sbk)):
            if rows_k:
                assert 0 <= (x - 1) * pitch_k * es + (k - 1) * es < 1 << 32 and pitch_k >= 0
            if rows_x:
                assert 0 <= (slices[bm, bn] - 1) * pitch_x * es + x * es < 1 << 32 and pitch_x >= 0
        accepted += chunked
    assert accepted > 500


def test_ordinary_strides_are_chunked_and_negative_ones_are_not(route):
    rows, expected = [], []
    for bm, bn, _ in TILES:
        for f32, es in ((1, 4), (0, 2)):
            for sam in (100, 101, 0, -100):  # a broadcast row has pitch 0
                for sbn in (100, 0, -100):
                    rows.append((f32, es, bm, bn, 50, 60, 100, sam, 1, 1, sbn))
                    expected.append((int(sam >= 0), 0, int(sbn >= 0), 0, int(sam >= 0 and sbn >= 0)))
            for sak in (50, -50):
                for sbk in (60, -60):
                    rows.append((f32, es, bm, bn, 50, 60, 100, 1, sak, sbk, 1))
                    a, b = int(sak >= 0 and bm >= 32), int(sbk >= 0)
                    expected.append((0, a, 0, b, a & b))
    assert route(rows) == expected


def _reversed_rows(storage):
    """Base address and strides of ``storage`` seen with its rows in falling order."""
    base = storage.data_ptr() + (storage.shape[0] - 1) * storage.stride(0) * storage.element_size()
    return base, -storage.stride(0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("splits", [1, 3])
def test_negative_pitches(dtype, splits):
    """Reversed A rows and B rows (row-major), and reversed columns of transposed storage, in every tile."""
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels import _native
    from kernels.matmul import _menu

    m, k, n = 70, 203, 67
    code = _native.dtype_code(dtype)
    gen = torch.Generator(device="cuda").manual_seed(8)
    a = torch.randint(-2, 3, (m, k), generator=gen, device="cuda").to(dtype)
    b = torch.randint(-2, 3, (k, n), generator=gen, device="cuda").to(dtype)
    at, bt = a.t().contiguous(), b.t().contiguous()
    lib, stream = _native.library(), _native.current_stream_handle(a.device)
    a_rev, a_pitch = _reversed_rows(a)    # A with its rows reversed
    b_rev, b_pitch = _reversed_rows(b)    # B with its rows (K) reversed
    at_rev, at_pitch = _reversed_rows(at)  # A with its columns (K) reversed
    bt_rev, bt_pitch = _reversed_rows(bt)  # B with its columns reversed
    forms = (
        (a_rev, (a_pitch, 1), b.data_ptr(), (n, 1), a.flip(0).double() @ b.double()),
        (a.data_ptr(), (k, 1), b_rev, (b_pitch, 1), a.double() @ b.flip(0).double()),
        (at_rev, (1, at_pitch), b_rev, (b_pitch, 1), a.flip(1).double() @ b.flip(0).double()),
        (a.data_ptr(), (k, 1), bt_rev, (1, bt_pitch), a.double() @ b.flip(1).double()),
    )
    for bm, bn, bk, warps, stages in _menu(dtype):
        if splits > 1 and (bm, bn, bk, warps, stages) not in _native.split_tiles(code, _native.GENERAL):
            continue
        tiles = -(-m // bm) * -(-n // bn)
        scratch = torch.zeros(_native.splitk_workspace_bytes(tiles, splits, bm, bn), dtype=torch.uint8, device="cuda")
        for form, (pa, sa, pb, sb, expected) in enumerate(forms):
            print(f"negative pitch form={form} {dtype} tile={(bm, bn, bk)} splits={splits}", flush=True)
            c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
            tile = (bm, bn, bk, 8, warps, stages)
            if splits > 1:
                status = lib.moegemm_matmul_splitk_any(pa, pb, c.data_ptr(), m, n, k, *sa, *sb, n, 1, code, 0, *tile,
                                                       splits, 0, scratch.data_ptr(), scratch.numel(), 0, stream)
            else:
                status = lib.moegemm_matmul(pa, pb, c.data_ptr(), m, n, k, *sa, *sb, n, 1, code, 0, *tile, 0, 0, stream)
            _native.check(status)
            torch.cuda.synchronize()
            assert torch.equal(c, expected.to(dtype)), (form, tile)


def _strided(rows, cols, dtype, device, gen):
    """Integers as every second column of every second row: no unit stride."""
    wide = torch.full((2 * rows, 2 * cols), float("nan"), device=device, dtype=dtype)
    view = wide[::2, ::2]
    return view.copy_(torch.randint(-2, 3, (rows, cols), generator=gen, device=device).to(dtype))


def test_strided_operands_take_their_own_layout():
    from kernels import _native
    from kernels.grouped_gemm import _group_layout, workspace_from_tensors
    from kernels.matmul import _operand_layout

    gen = torch.Generator().manual_seed(1)
    for dtype, code in ((torch.float32, _native.DTYPE_F32), (torch.float16, _native.DTYPE_F16)):
        a, b, c = torch.zeros((24, 40), dtype=dtype), torch.zeros((40, 32), dtype=dtype), torch.zeros((24, 32), dtype=dtype)
        odd = _strided(24, 40, dtype, "cpu", gen)
        assert _native.strided_or(_operand_layout(odd, b, c), odd, b) == _native.STRIDED
        assert _native.strided_or(_operand_layout(a, b, c), a, b) == (_native.GENERAL if code == _native.DTYPE_F32 else 0)
        assert _native.strided_or(_operand_layout(a.t(), b, c), a.t().contiguous().t(), b) != _native.STRIDED
        both = workspace_from_tensors([odd, odd[:8]], [b, b], [c, c[:8].clone()])
        mixed = workspace_from_tensors([odd, a[:8]], [b, b], [c, c[:8].clone()])
        assert _group_layout(both, code) == _native.STRIDED and _group_layout(mixed, code) == _native.GENERAL
        assert _native.split_tiles(code, _native.STRIDED) == frozenset()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("shape", [(1, 1, 1), (70, 5, 67), (129, 203, 131)])
def test_strided_operands_every_tile(dtype, shape):
    """Alone and in groups whose problems all are strided, or only one is; K below and above one chunk."""
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    from kernels.grouped_gemm import launch_grouped, workspace_from_tensors
    from kernels.matmul import KernelConfig, _menu, launch_matmul

    m, k, n = shape
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    a, b = _strided(m, k, dtype, "cuda", gen), _strided(k, n, dtype, "cuda", gen)
    flat = b.contiguous()
    expected = (a.double() @ b.double()).to(dtype)
    for bm, bn, bk, warps, stages in _menu(dtype):
        cfg = KernelConfig(bm, bn, bk, 8, warps, stages)
        for precision in ("ieee", "tf32"):
            print(f"strided {dtype} shape={shape} tile={cfg.tile_key} {precision}", flush=True)
            c = torch.full((m, n + 3), float("nan"), device="cuda", dtype=dtype)[:, 1:n + 1]
            launch_matmul(a, b, c, cfg, precision, autotune=False)
            torch.cuda.synchronize()
            assert torch.equal(c, expected), cfg
        for second in (b, flat):
            outs = [torch.full((m, n), float("nan"), device="cuda", dtype=dtype) for _ in range(2)]
            ws = workspace_from_tensors([a, a.contiguous() if second is flat else a], [b, second], outs)
            for schedule in ("static", "stealing"):
                for z in outs:
                    z.fill_(float("nan"))
                launch_grouped(ws, config=cfg, autotune=False, tile_schedule=schedule)
                torch.cuda.synchronize()
                assert all(torch.equal(z, expected) for z in outs), (cfg, schedule)
