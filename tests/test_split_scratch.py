"""Split-K scratch of operands that are not row-major 16-bit ones (fp32, unaligned, transposed): which
launches get it, who may share it, and what is left of it when the tuner is done."""

from __future__ import annotations

import pytest
import torch

from kernels import _native, grouped_gemm, matmul
from kernels.matmul import KernelConfig

TILES = {torch.float32: KernelConfig(64, 64, 32, 2, 4, 2), torch.bfloat16: KernelConfig(64, 64, 64, 2, 4, 4)}
FORMS = ("fp32", "tf32", "unaligned", "transposed")


def _operands(form, device, m=64, k=1024, n=64):
    dtype = torch.float32 if "32" in form else torch.bfloat16
    gen = torch.Generator(device=device).manual_seed(3)

    def ints(rows, cols):
        return torch.randint(-2, 3, (rows, cols), generator=gen, device=device).to(dtype)

    a, b = ints(m, k), ints(k, n)
    if form == "unaligned":
        a = torch.empty((m * k + 1,), device=device, dtype=dtype)[1:].view(m, k).copy_(a)
    if form == "transposed":
        b = b.t().contiguous().t()
    return a, b, torch.full((m, n), float("nan"), device=device, dtype=dtype)


class _Recorder:
    """Stands in for the library: notes the entry points called (and their arguments) and launches nothing."""

    def __init__(self, real):
        self._real, self.calls = real, []

    def __getattr__(self, name):
        if name.startswith(("moegemm_matmul", "moegemm_grouped_gemm")):
            return lambda *args: self.calls.append((name, args)) or 0
        return getattr(self._real, name)


@pytest.fixture
def recorder(monkeypatch):
    library = _Recorder(_native.library())
    state = {"capturing": False}
    monkeypatch.setattr(_native, "library", lambda: library)
    monkeypatch.setattr(_native, "current_stream_handle", lambda device: state.get("stream", 77))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(matmul, "_device_signature", lambda device: 950256)
    monkeypatch.setattr(matmul, "_validate_matrices", lambda a, b, c: (*a.shape[:1], b.shape[1], a.shape[1]))
    monkeypatch.setattr(matmul, "_require_runtime", lambda tensor=None: None)
    monkeypatch.setattr(grouped_gemm, "_require_runtime", lambda tensor=None: None)
    monkeypatch.setattr(grouped_gemm, "_check_workspace", lambda ws: _native.dtype_code(ws.a[0].dtype))
    monkeypatch.setattr(_native, "_EAGER_SCRATCH", {})
    monkeypatch.setattr(_native, "_SPLITK_WORKSPACES", {})
    library.state = state
    return library


def _launch(form, group):
    a, b, c = _operands(form, "cpu")
    precision = "tf32" if form == "tf32" else "ieee"
    if group:
        ws = grouped_gemm.workspace_from_tensors([a, a], [b, b], [c, c.clone()])
        grouped_gemm.launch_grouped(ws, precision, TILES[a.dtype], autotune=False, split_k=4)
        return ws.split_k
    matmul.launch_matmul(a, b, c, TILES[a.dtype], precision, autotune=False, split_k=4)
    return matmul.last_matmul_split()


@pytest.mark.parametrize("form,group", [(f, g) for f in FORMS for g in (False, True) if not (g and f == "transposed")])
def test_captured_launches_hold_no_scratch(recorder, form, group):
    """Warmed on the capturing stream or not: a graph that held the stream's scratch could replay beside
    another launch that uses it.  Eager calls split, and with their own buffer."""
    assert _launch(form, group) == 4
    name, args = recorder.calls.pop()
    assert name.endswith("splitk_any") and _native._EAGER_SCRATCH[0, 77].data_ptr() in args
    assert not _native._SPLITK_WORKSPACES
    recorder.state["capturing"] = True
    assert _launch(form, group) == 1
    name, args = recorder.calls.pop()
    assert name in ("moegemm_matmul", "moegemm_grouped_gemm")
    assert _native._EAGER_SCRATCH[0, 77].data_ptr() not in args


def test_launches_run_whole_without_memory(recorder, monkeypatch):
    def no_memory(*args, **kwargs):
        raise torch.cuda.OutOfMemoryError("no memory")

    monkeypatch.setattr(torch, "zeros", no_memory)
    assert _launch("fp32", False) == 1 and recorder.calls.pop()[0] == "moegemm_matmul"
    assert _launch("fp32", True) == 1 and recorder.calls.pop()[0] == "moegemm_grouped_gemm"


def test_scratch_grows_in_place_and_few_streams_hold_one(recorder):
    small = _native.eager_scratch("cpu", 1, 4, 2, 64, 64)
    assert _native.eager_scratch("cpu", 1, 2, 4, 64, 64) is small
    large = _native.eager_scratch("cpu", 1, 8, 2, 64, 64)
    assert large.numel() > small.numel() and list(_native._EAGER_SCRATCH) == [(0, 1)]
    assert not large.any() and not small.any()
    for stream in range(40):
        _native.eager_scratch("cpu", stream, 4, 2, 64, 64)
    assert len(_native._EAGER_SCRATCH) == _native._EAGER_SCRATCH_STREAMS
    assert _native.eager_scratch("cpu", 1, 4, 65, 64, 64) is None
    assert _native.eager_scratch("cpu", 1, 65537, 2, 64, 64) is None


def test_tuner_names_the_best_candidate_that_does_not_split(monkeypatch):
    times = {("a", 4): 1.0, ("a", 1): 3.0, ("b", 1): 2.0, ("b", 2): 1.5}
    last = []
    monkeypatch.setattr(matmul, "_warm_clocks", lambda launch: None)
    monkeypatch.setattr(matmul, "hot_autotune_bench", lambda launch, q: (launch(), [times[last.pop()]])[1])
    assert matmul._tune(times, last.append, fallback=lambda o: o[1] == 1) == (("a", 4), ("b", 1))
    times[("a", 1)] = 0.5
    assert matmul._tune(times, last.append, fallback=lambda o: o[1] == 1) == (("a", 1), ("a", 1))
    assert matmul._tune(times, last.append, fallback=lambda o: o[1] == 3) == (("a", 1), None)


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_graphs_beside_eager_calls_of_their_capture_stream(form):
    """Two graphs captured on one stream after eager split calls there, replayed on two streams beside eager
    calls on the capture stream: every result is the eager one."""
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    a, b, _ = _operands(form, "cuda")
    expected = (a.double() @ b.double()).to(a.dtype)
    cfg, precision = TILES[a.dtype], "tf32" if form == "tf32" else "ieee"
    outs = [torch.empty_like(expected) for _ in range(3)]

    def launch(c):
        matmul.launch_matmul(a, b, c, cfg, precision, autotune=False, split_k=4)

    home, others, graphs = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)], []
    print(f"graphs beside eager calls form={form}", flush=True)
    torch.cuda.synchronize()
    with torch.cuda.stream(home):
        launch(outs[2])
        assert matmul.last_matmul_split() == 4
    home.synchronize()
    assert torch.equal(outs[2], expected)
    for c in outs[:2]:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=home):
            launch(c)
        assert matmul.last_matmul_split() == 1
        graphs.append(graph)
    for _ in range(10):
        for c in outs:
            c.fill_(float("nan"))
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, others):
            with torch.cuda.stream(stream):
                graph.replay()
        with torch.cuda.stream(home):
            launch(outs[2])
        torch.cuda.synchronize()
        for c in outs:
            assert torch.equal(c, expected)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["fp32", "transposed"])
def test_tuning_keeps_only_the_scratch_of_its_choice(form):
    if not torch.cuda.is_available():
        pytest.skip("ROCm GPU unavailable")
    a, b, c = _operands(form, "cuda", 328, 2056, 264)
    rows = {key: sum(t.numel() for t in held) for key, held in _native._SPLITK_WORKSPACES.items()}
    _native._EAGER_SCRATCH.clear()
    print(f"tuning scratch form={form}", flush=True)
    matmul.launch_matmul(a, b, c)
    torch.cuda.synchronize()
    assert torch.equal(c, (a.double() @ b.double()).to(a.dtype))
    assert {key: sum(t.numel() for t in held) for key, held in _native._SPLITK_WORKSPACES.items()} == rows
    held = dict(_native._EAGER_SCRATCH)
    assert set(held) <= {(a.device.index, _native.current_stream_handle(a.device))}
    if matmul.last_matmul_split() > 1:
        cfg = matmul.last_matmul_config(None)
        tiles = -(-328 // cfg.block_m) * -(-264 // cfg.block_n)
        nbytes = _native.splitk_workspace_bytes(tiles, matmul.last_matmul_split(), cfg.block_m, cfg.block_n)
        assert [t.numel() for t in held.values()] == [nbytes]
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    c.fill_(float("nan"))
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        matmul.launch_matmul(a, b, c)
    assert matmul.last_matmul_split() == 1
    for _ in range(3):
        c.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, (a.double() @ b.double()).to(a.dtype))
