"""What hawk.run and a prepared launcher hand the GPU, call by call, recorded on
the CPU: the launches are stubs, the planes CPU tensors, everything between
them the runtime's own."""

from __future__ import annotations

from pathlib import Path

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
                        lambda self, arrays, n_samples=None, rows=(): next(
                            x.shape[-1] for name, x in arrays.items() if self.planes[name]["role"] in
                            runtime._PER_SAMPLE))
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


def _work_pointers(calls, planes) -> set:
    """The addresses a run's calls work in: every pointer but the caller's planes'."""
    mine = {x.data_ptr() for x in planes.values()}
    found = set()
    for _name, args in calls:
        for a in args:
            for v in ([p for job in a for p in (job.hi, job.lo, job.out)] if hasattr(a, "_length_") else [a]):
                if isinstance(v, int) and v > 1 << 20 and v not in mine:
                    found.add(v)
    return found


def _kernels_with_scratch(n):
    import torch
    from hawk_amd import Grid, Index, Kernel, Table
    from hawk_amd import examples as E

    @hawk.kernel
    def keyed(lane: Grid["key", "sample":200], x: Scalar, o: Mutable["key"], c: Mutable["key"]):
        o = hawk.sum(x * 2.0, over="sample", policy="ordered")
        c = hawk.sum(x, over="sample")

    @hawk.kernel
    def table(lane: Grid["key", "sample":100], t: Table["key", "w":2], x: Scalar) -> Scalar:
        return hawk.sum(t.at(key=lane.key, w=0) * x + t.at(key=lane.key, w=1), over="sample", policy="ordered")
    back = Kernel("table_vjp", hawk.diff.vjp(table, wrt=("t",)))

    def d(*shape):
        return torch.ones(*shape, dtype=torch.float64)
    return [(three, dict(x=d(n), a=d(1), o=d(1), b=d(1))),
            (E.chain, dict(x=d(n), key=torch.zeros(n, dtype=torch.int32), y=d(n), total=d(1), bins=d(64))),
            (keyed, dict(x=d(n), o=d(n // 200), c=d(n // 200))),
            (back, dict(t=d(n // 50), x=d(n), bar_out=d(n // 100), bar_t=d(n // 50)))]


def test_each_stream_has_its_own_workspace(tmp_path, recorded):
    """Calls on two streams may run at once, so nothing one works in is the
    other's: not the scratch of a team stage, not a plane the stage writes for
    it, not a launcher's.  Runs on one stream share, and so do its launchers."""
    cases = _kernels_with_scratch(2000)
    for k, (_, planes) in zip(_load(tmp_path, *(c[0] for c in cases)), cases):
        used = {}
        for stream in (0, 7, 0, 7):
            for way, _ in enumerate(_both_ways(k, 2000, stream, **planes)):
                here = _work_pointers(recorded, planes)
                assert here and used.setdefault((stream, way), here) == here, (k.name, stream)
                recorded.clear()
        assert not (used[0, 0] | used[0, 1]) & (used[7, 0] | used[7, 1]), k.name


def test_runs_of_many_sizes_hold_a_multiple_of_the_largest(tmp_path, recorded):
    """hawk.run over ever new sample counts holds, for every scratch tensor, at
    most half more than the largest needs and twice that outgrown; a size seen
    before works where it did, and a launcher's addresses are its own."""
    sizes = [2000 + 200 * i for i in range(40)]
    kernels = [case[0] for case in _kernels_with_scratch(2000)]
    calls = {n: [case[1] for case in _kernels_with_scratch(n)] for n in sizes}
    for i, k in enumerate(_load(tmp_path, *kernels)):
        launch = k.prepare(stream=0, **calls[sizes[0]][i])
        recorded.clear()
        launch()
        mine = _work_pointers(recorded, calls[sizes[0]][i])
        seen = {}
        for n in sizes * 2:
            recorded.clear()
            k._run(dict(calls[n][i]), 0, n, n, 0, False)
            here = _work_pointers(recorded, calls[n][i])
            assert here and not here & mine and seen.setdefault(n, here) == here
        work = k._workspace(0, calls[sizes[0]][i]["x"].device)
        for key, buffer in work._buffers.items():
            need = max(x.numel() * x.element_size() for held, x in work.items() if held[:2] == key)
            assert buffer.numel() <= max(8, 1.5 * need)
        assert sum(x.numel() for x in work._outgrown) <= 2 * sum(x.numel() for x in work._buffers.values())
        recorded.clear()
        launch()
        assert _work_pointers(recorded, calls[sizes[0]][i]) == mine


def test_each_stream_has_its_own_trip_count_and_finish_counter(tmp_path, recorded):
    """The words the runtime itself binds: another stream's are rewritten
    while this one's launch reads them."""
    import torch
    from hawk_amd import examples as E
    (k,) = _load(tmp_path, E.osc_finish_xauto)
    planes = {name: torch.zeros(50, dtype=torch.bool if name == "terminated" else torch.float64)
              for name in ("t_final", "terminated", "x", "v", "t")}
    mine = {x.data_ptr() for x in planes.values()}
    used = {}
    for stream in (0, 7, 0):
        for steps in (3, 4):
            k._run(dict(planes, dt=0.5), 0, 50, 50, stream, False, steps=steps)
            here = {held[1] for held in k._held_slots if held[0] == "p"} - mine
            assert len(here) == 2 and used.setdefault(stream, here) == here
            word = k._workspace(stream, planes["x"].device)[("word", "")]
            assert int(word) == steps and word.data_ptr() in here
    assert not used[0] & used[7]


def test_a_cut_chain_crosses_in_planes_of_its_stream_one_call_at_a_time(tmp_path, recorded):
    """A cut chain's crossing planes are a stream's own, and a call's segments
    run with no other call's between them."""
    import threading

    import torch
    from hawk_amd import examples as E
    chained = hawk.chain(*E.CHAIN_MEMBERS, name="cut")
    hawk.build([chained], tmp_path, register_line=32)
    k = hawk.load(tmp_path, "cut")
    planes = {name: torch.zeros(tuple(info["shape"]) + (40,), dtype=torch.float64)
              for name, info in k.planes.items()}
    mine = {x.data_ptr() for x in planes.values()}
    used = {}
    for stream in (0, 7, 0):
        here = {x.data_ptr() for _, p in k._bindings(planes, stream=stream) for x in p.values()} - mine
        assert here and used.setdefault(stream, here) == here
    assert not used[0] & used[7]
    with k._lock:
        other = threading.Thread(target=lambda: hawk.run(k, stream=7, **planes))
        other.start()
        other.join(0.2)
        assert other.is_alive() and not recorded
    other.join(10)
    assert len(recorded) == len(k.segments) > 1


def test_loading_a_kernel_imports_no_torch(tmp_path):
    """hawk.load of a kernel with no code object of its own, and the load of
    any other past its code object, leave torch alone."""
    import subprocess
    import sys
    from hawk_amd import examples as E
    hawk.build([E.mm16, E.energy], tmp_path)
    text = """
import sys
import hawk_amd as hawk
from hawk_amd import _core
class Library:
    def __init__(self, code): pass
    def entry(self, name): return name
class Block:
    def __init__(self, descriptor): pass
_core.DeviceLibrary, _core.ArgBlock = Library, Block
for name in ("mm16", "energy"):
    hawk.load(sys.argv[1], name)
    assert "torch" not in sys.modules, name
"""
    done = subprocess.run([sys.executable, "-c", text, str(tmp_path)], capture_output=True, text=True,
                          cwd=Path(__file__).resolve().parent.parent)
    assert done.returncode == 0, done.stderr
