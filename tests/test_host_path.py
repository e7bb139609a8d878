"""What hawk.run and a prepared launcher hand the GPU, call by call, recorded on
the CPU: the launches are stubs, the planes CPU tensors, everything between
them the runtime's own."""

from __future__ import annotations

import pytest

import hawk_amd as hawk
from hawk_amd import Mutable, Scalar


@hawk.kernel
def three(x: Scalar, a: Mutable[Scalar], o: Mutable[Scalar], b: Mutable[Scalar]):
    a = hawk.sum(x * 2.0)
    o = hawk.sum(x, policy="ordered")
    b = hawk.max(x)


@pytest.fixture
def recorded(monkeypatch):
    """``calls``: every (entry, arguments) that would have crossed into the GPU."""
    from hawk_amd import _core, runtime
    calls = []

    class Entry:
        def __init__(self, name):
            self.name = name

        def run(self, block, base, count, n, **kw):
            calls.append((self.name, (block, base, count, n)))

        def prepared(self, block, base, count, n, **kw):
            return lambda: self.run(block, base, count, n)

    class Library:
        def __init__(self, code):
            pass

        def entry(self, name):
            return Entry(name)

    def record(name):
        return lambda *args: calls.append((name, args))
    monkeypatch.setattr(_core, "DeviceLibrary", Library)
    for name in ("rows_finish_many", "ordered_sum", "ordered_scatter", "keyed_ordered_sum", "keyed_sample_sum",
                 "keyed_log_fold", "band_ordered_sum"):
        monkeypatch.setattr(_core, name, record(name))
    monkeypatch.setattr(runtime, "_on", lambda stream: runtime._nullcontext())
    monkeypatch.setattr(runtime, "_current_stream", lambda: 0)
    monkeypatch.setattr(runtime.DeviceKernel, "check_planes",
                        lambda self, arrays, n_samples=None, rows=(): arrays["x"].shape[-1])
    return calls


def _load(tmp_path, *kernels):
    hawk.build(list(kernels), tmp_path)
    return [hawk.load(tmp_path, k.name) for k in kernels]


def _both_ways(k, n, stream, **planes):
    """One run's recorded calls come from hawk.run's launch path, then from a launcher."""
    k._run(dict(planes), 0, n, n, stream, False)
    yield
    k.prepare(stream=stream, **planes)()
    yield


def _cells(n):
    import torch
    return torch.ones(n, dtype=torch.float64), *(torch.zeros(1, dtype=torch.float64) for _ in range(3))


def test_reductions_of_their_own_cells_finish_in_one_call(tmp_path, recorded):
    (k,) = _load(tmp_path, three)
    x, a, o, b = _cells(100)
    for _ in _both_ways(k, 100, 0, x=x, a=a, o=o, b=b):
        assert [name for name, _ in recorded] == ["three", "rows_finish_many", "ordered_sum"]
        assert [job.out for job in recorded[1][1][0]] == [a.data_ptr(), b.data_ptr()]
        recorded.clear()


def test_reductions_that_share_a_cell_keep_the_kernels_order(tmp_path, recorded):
    """Two reductions bound to one cell: each in a call of its own, where the
    kernel has it, so the last one's value stays."""
    (k,) = _load(tmp_path, three)
    x, a, o, _ = _cells(100)
    for b in (a, o):
        for _ in _both_ways(k, 100, 0, x=x, a=a, o=o, b=b):
            assert [name for name, _ in recorded] == ["three", "rows_finish_many", "ordered_sum", "rows_finish_many"]
            assert [[job.out for job in recorded[i][1][0]] for i in (1, 3)] == [[a.data_ptr()], [b.data_ptr()]]
            recorded.clear()
