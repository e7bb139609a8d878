"""The routes a team stage picks by size and alignment, each at the sizes
where it can go wrong (edges of tiles, remainders, planes that start inside a
line), against the oracle or against an independent computation."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _unit(tmp_path, kernels, mode="float64"):
    import hawk_amd as hawk
    hawk.build(kernels, tmp_path, mode=mode)
    return [hawk.load(tmp_path, k.name) for k in kernels]


def _plane(a, gpu, shift=0):
    """``a`` on the device, its first element ``shift`` elements past an allocation's start."""
    import torch
    flat = torch.from_numpy(np.ascontiguousarray(a)).reshape(-1)
    held = torch.empty(flat.numel() + shift, dtype=flat.dtype, device=gpu)
    held[shift:] = flat.to(gpu)
    return held[shift:].view(a.shape)


@pytest.mark.parametrize("mode", ["float32", "float64"])
@pytest.mark.parametrize("n, shift", [(32, 0), (64, 0), (64, 1), (4128, 0), (4128, 3), (4127, 0), (100, 0)])
def test_mm16_streamed_and_cached(tmp_path, gpu, mode, n, shift):
    """Whole-line planes stream, others (a row that is no multiple of 128
    bytes, a plane starting inside a line) go through the cache.  On small
    integers every partial sum is exact, so both give the exact product."""
    from hawk_amd import examples as E
    import hawk_amd as hawk
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(n + shift)
    A, B, C = (g.integers(-8, 9, size=(16, 16, n)).astype(dt) for _ in range(3))
    fwd, vjp = _unit(tmp_path, [E.mm16, E.mm16_vjp], mode)
    zero = np.zeros((16, 16, n), dt)
    got, bar_A, bar_B = (_plane(zero, gpu, shift) for _ in range(3))
    a, b, c = (_plane(x, gpu, shift) for x in (A, B, C))
    hawk.run(fwd, A=a, B=b, C=got, layout="samples_last")
    hawk.run(vjp, A=a, B=b, bar_C=c, bar_A=bar_A, bar_B=bar_B, layout="samples_last")
    for x, (X, Y) in ((got, (A, B)), (bar_A, (C, B.transpose(1, 0, 2))), (bar_B, (A.transpose(1, 0, 2), C))):
        assert np.array_equal(x.cpu().numpy(), np.einsum("ikn,kjn->ijn", X, Y))


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("cells, n, keys", [
    (8192, 60_000, "zipf"), (8193, 60_000, "zipf"), (9000, 9000 * 31, "one"), (9000, 9000 * 32, "one"),
    (12_289, 100, "uniform"), (20_000, 20_000 * 191, "zipf"), (20_000, 20_000 * 192, "sorted"),
    (65_537, 65_537, "uniform"), (65_537, 400_003, "sorted"), (65_600, 700_001, "zipf"), (65_600, 300_000, "one"),
    (289_792, 600_001, "zipf"), (289_793, 600_001, "zipf"), (1 << 20, 5_000, "uniform"), (70_000, 0, "uniform"), (5_000_001, 700, "uniform")])
def test_ordered_scatter_walks(tmp_path, gpu, mode, cells, n, keys):
    """Few chunks, many cells and their neighbours on the other walk: the
    serial walk's bits, skip keys and infinities among the lanes, and the bad
    keys reported with every other lane added."""
    import hawk_amd as hawk
    import oracle_lib as O
    import torch
    from hawk_amd import HawkError
    from hawk_amd import examples as E
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(cells + n)
    key = {"uniform": lambda: g.integers(0, cells, n), "sorted": lambda: np.sort(g.integers(0, cells, n)),
           "zipf": lambda: (g.zipf(1.1, n) - 1) % cells, "one": lambda: np.full(n, cells - 3)}[keys]().astype(np.int32)
    key[::11] = -1
    x = (g.normal(size=n) * np.exp(g.normal(size=n))).astype(dt)
    x[5::1001] = np.inf
    acc0 = np.linspace(1.0, 2.0, cells).astype(dt)
    (k,) = _unit(tmp_path, [E.ordered_add], mode)
    planes = {"x": torch.from_numpy(x).to(gpu)}
    for bad in (False, True):
        if bad and n:
            key[n // 2], key[n - 1] = cells, -2
        acc = torch.from_numpy(acc0).to(gpu)
        print(f"scatter cells={cells} n={n} {keys} {mode} bad={bad}", flush=True)
        call = dict(key=torch.from_numpy(key).to(gpu), acc=acc, **planes)
        if bad and n:
            with pytest.raises(HawkError, match="outside"):
                hawk.run(k, **call)
        else:
            hawk.run(k, **call)
        want, status = O.ordered_scatter(key, x, acc0)
        assert bool(status[1:].any()) == (bad and n > 0)
        assert acc.cpu().numpy().tobytes() == want.tobytes()


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("cells, n", [(33, 4097), (64, 64 * 300 + 5), (1000, 1000 * 256 + 63), (20_000, 20_000 * 192)])
@pytest.mark.parametrize("each", [1, 2, 3, 5, 8, 9, 64, "heads"])
def test_ordered_scatter_peers(gpu, mode, cells, n, each):
    """Windows whose keys have no peers, one, a block's worth, one more and a
    whole window's, and head keys of unequal runs: the serial walk's bits,
    negative zeros among the values."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(cells + n)
    if each == "heads":
        key = np.minimum(g.geometric(0.5, n) - 1, 32)
    else:
        # a stride of 15 and of 8 keeps neighbours in one class of either split
        key = (np.arange(n) // each * 120) % cells
        key[n // 2:] = np.roll(key[n // 2:], 7)
    key = key.astype(np.int32)
    x = (g.normal(size=n) * np.exp(g.normal(size=n))).astype(dt)
    x[::3] = -0.0
    acc0 = np.full(cells, -0.0, dt)
    want, _ = O.ordered_scatter(key, x, acc0)
    fn = _core.ordered_scatter_f32 if mode == "float32" else _core.ordered_scatter
    kd, xd, acc = (torch.from_numpy(a).to(gpu) for a in (key, x, acc0))
    scratch = torch.empty(_core.ordered_scatter_scratch_bytes(n, cells), dtype=torch.uint8, device=gpu)
    status = torch.zeros(257, dtype=torch.int32, device=gpu)
    print(f"scatter peers cells={cells} n={n} each={each} {mode}", flush=True)
    fn(kd.data_ptr(), xd.data_ptr(), n, acc.data_ptr(), cells, scratch.data_ptr(), status.data_ptr(),
       torch.cuda.current_stream().cuda_stream)
    assert acc.cpu().numpy().tobytes() == want.tobytes()
    assert not status[1:].any()


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("cells, chunks", [(12_289, 95), (12_289, 96), (16_384, 95), (16_384, 96), (16_385, 96),
                                           (20_000, 192), (65_600, 130)])
def test_ordered_scatter_long_runs(gpu, mode, cells, chunks):
    """Runs of one key of every length about a window, in the class of one wave
    of the tail and sorted over all cells, on both sides of the walks' lines:
    the serial walk's bits, negative zeros and an infinity among the values."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    dt = np.float32 if mode == "float32" else np.float64
    n = cells * chunks + 77
    assert _core.scatter_chunks(n, cells) == chunks
    g = np.random.default_rng(cells + chunks)
    x = (g.normal(size=n) * np.exp(g.normal(size=n))).astype(dt)
    x[::3] = -0.0
    x[n // 2] = np.inf
    acc0 = np.full(cells, -0.0, dt)
    fn = _core.ordered_scatter_f32 if mode == "float32" else _core.ordered_scatter
    xd = torch.from_numpy(x).to(gpu)
    scratch = torch.empty(_core.ordered_scatter_scratch_bytes(n, cells), dtype=torch.uint8, device=gpu)
    status = torch.zeros(257, dtype=torch.int32, device=gpu)
    lengths = np.array([1, 2, 63, 64, 65, 127, 128, 129, 192, 200, 1000])
    run = np.repeat(np.arange(n // 100), np.resize(lengths, n // 100))[:n]
    run = np.concatenate([run, np.zeros(n - run.size, run.dtype)])
    high = 12_288 if cells > 12_296 else 0
    for key in (high + run * 8 % max(8, cells - high), np.arange(n) * cells // n, np.full(n, cells - 1)):
        key = np.minimum(key, cells - 1).astype(np.int32)
        want, _ = O.ordered_scatter(key, x, acc0)
        kd, acc = torch.from_numpy(key).to(gpu), torch.from_numpy(acc0).to(gpu)
        print(f"scatter runs cells={cells} chunks={chunks} {mode}", flush=True)
        fn(kd.data_ptr(), xd.data_ptr(), n, acc.data_ptr(), cells, scratch.data_ptr(), status.data_ptr(),
           torch.cuda.current_stream().cuda_stream)
        assert acc.cpu().numpy().tobytes() == want.tobytes()
        assert not status[1:].any()


@pytest.mark.parametrize("mode", ["float64", "float32"])
def test_ordered_scatter_partials(gpu, mode):
    """Every number of chunks around the fold's blocks of 32 and groups of 8:
    the serial walk's bits."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    dt = np.float32 if mode == "float32" else np.float64
    fn = _core.ordered_scatter_f32 if mode == "float32" else _core.ordered_scatter
    for chunks in (1, 2, 7, 8, 9, 31, 32, 33, 40, 41, 63, 64, 65, 95, 96, 97, 128, 255, 256):
        for cells in (7, 300):
            n = cells * chunks + cells // 2
            assert _core.scatter_chunks(n, cells) == chunks
            g = np.random.default_rng(n)
            key, x = g.integers(-1, cells, n).astype(np.int32), g.normal(size=n).astype(dt)
            acc0 = g.normal(size=cells).astype(dt)
            want, _ = O.ordered_scatter(key, x, acc0)
            kd, xd, acc = (torch.from_numpy(a).to(gpu) for a in (key, x, acc0))
            scratch = torch.full((_core.ordered_scatter_scratch_bytes(n, cells),), 255, dtype=torch.uint8, device=gpu)
            status = torch.zeros(257, dtype=torch.int32, device=gpu)
            fn(kd.data_ptr(), xd.data_ptr(), n, acc.data_ptr(), cells, scratch.data_ptr(), status.data_ptr(),
               torch.cuda.current_stream().cuda_stream)
            assert acc.cpu().numpy().tobytes() == want.tobytes(), (chunks, cells)


def _per_key(group, policy):
    import hawk_amd as hawk
    from hawk_amd import Grid, Kernel, Scalar

    @hawk.kernel
    def key_total(lane: Grid["key", "sample":group], x: Scalar) -> Scalar:
        return hawk.sum(x, over="sample", policy=policy)
    return Kernel("key_total", key_total.program)


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("keys, group", [
    (9, 1), (7, 31), (8, 32), (5, 33), (3, 64), (5, 65), (6, 128), (5, 129), (3, 256), (5, 257), (5, 512), (4, 513),
    (5, 1024), (5, 1025), (3, 2048), (511, 2049), (512, 2049), (2, 256 * 32 + 1), (2, 131_072), (2, 131_073),
    (600, 8193)])
def test_keyed_default_sum_routes(tmp_path, gpu, mode, keys, group):
    """Rows of eight lanes, every number of rows a step and a key can hold: the
    oracle's bits, with infinities, NaN and signed zeros among the values."""
    import hawk_amd as hawk
    import oracle_lib as O
    import torch
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(keys * 7 + group)
    x = (g.normal(size=keys * group) * 2.0 ** g.integers(-20, 20, keys * group)).astype(dt)
    x[g.random(x.size) < 0.1] = -0.0
    if keys > 2:
        x[group // 2], x[2 * group - 1] = np.inf, np.nan
    (k,) = _unit(tmp_path, [_per_key(group, "auto")], mode)
    out = torch.full((keys,), 7.0, dtype=torch.float32 if mode == "float32" else torch.float64, device=gpu)
    hawk.run(k, x=torch.from_numpy(x).to(gpu), out=out)
    want = O.keyed_sample_sum(x, group)
    got = out.cpu().numpy()
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all() and got[~nan].tobytes() == want[~nan].tobytes()


def test_default_sums_of_more_keys_than_sixteen_waves_each_launch(gpu):
    """2^22 keys of 8193 float32 samples: sixteen waves a key would pass the
    2^32 - 1 threads of a launch, four do not.  A 137 GB plane, its first and
    last keys checked."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    keys, group = 1 << 22, 8193
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < keys * group * 4 + (4 << 30):
        pytest.skip("the plane does not fit the memory that is free")
    u = torch.empty(keys * group, dtype=torch.float32, device=gpu)
    ends = np.random.default_rng(22).normal(size=2 * group).astype(np.float32)
    u[:group], u[-group:] = (torch.from_numpy(e).to(gpu) for e in (ends[:group], ends[group:]))
    out = torch.zeros(keys, dtype=torch.float32, device=gpu)
    _core.keyed_sample_sum_f32(u.data_ptr(), keys * group, group, out.data_ptr(),
                               torch.cuda.current_stream().cuda_stream)
    got = torch.stack((out[0], out[-1])).cpu().numpy()
    del u
    torch.cuda.empty_cache()
    assert got.tobytes() == O.keyed_sample_sum(ends, group).tobytes()


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("keys, group", [
    (9, 1), (70, 3), (257, 16), (5, 17), (7, 33), (1025, 64), (5, 65), (9, 128), (5, 129), (6, 256), (5, 257),
    (7, 512), (5, 513), (3, 1023), (5, 1024), (5, 1025), (511, 2047), (512, 2047), (2, 65_536), (2, 65_537),
    (3, 131_073), (1, 1), (1, 1000), (1, 65_536), (1, 65_537), (1, 65_536 * 9 + 5), (1, 65_536 * 40 - 1)])
def test_ordered_sum_routes(tmp_path, gpu, mode, keys, group):
    """Keyed and plain ordered sums at the edges of their kernels: the fixed
    tree's bits per key, with infinities and signed zeros among the values."""
    import hawk_amd as hawk
    import oracle_lib as O
    import torch
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(keys * 11 + group)
    x = (g.normal(size=keys * group) * 2.0 ** g.integers(-20, 20, keys * group)).astype(dt)
    x[g.random(x.size) < 0.1] = -0.0
    if keys > 2:
        x[group // 2] = np.inf
    (k,) = _unit(tmp_path, [_per_key(group, "ordered")], mode)
    out = torch.full((keys,), 7.0, dtype=torch.float32 if mode == "float32" else torch.float64, device=gpu)
    hawk.run(k, x=torch.from_numpy(x).to(gpu), out=out)
    assert out.cpu().numpy().tobytes() == O.keyed_ordered_sum(x, group).tobytes()


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("rows", [1, 7, 8, 9, 16, 31, 32, 33, 40, 63, 64, 65, 72, 95, 96, 127, 128, 129, 193])
def test_ordered_sum_batches(gpu, mode, rows):
    """Every kind of last batch a virtual lane can have, whole, one row short of
    a group and one past: the fixed tree's bits."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    dt = np.float32 if mode == "float32" else np.float64
    g = np.random.default_rng(rows)
    x = (g.normal(size=65_536 * rows) * 2.0 ** g.integers(-10, 10, 65_536 * rows)).astype(dt)
    x[g.random(x.size) < 0.05] = -0.0
    u, out = torch.from_numpy(x).to(gpu), torch.full((1,), 7.0, dtype=torch.float32 if mode == "float32" else
                                                     torch.float64, device=gpu)
    scratch = torch.zeros(_core.ordered_sum_scratch_bytes(), dtype=torch.uint8, device=gpu)
    fn = _core.ordered_sum_f32 if mode == "float32" else _core.ordered_sum
    for n in (65_536 * rows, 65_536 * rows - 1, 65_536 * (rows - 1) + 1, 65_536 * rows - 40_000):
        fn(u.data_ptr(), n, out.data_ptr(), scratch.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert out.cpu().numpy().tobytes() == O.keyed_ordered_sum(x[:n], n).tobytes(), n


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("rows", [1, 255, 256, 257, 4095, 4096, 4097, 2 * 4096, 128 * 4096 + 1, 129 * 4096,
                                  1024 * 4096, 1025 * 4096 + 17])
def test_rows_finish_together(gpu, mode, rows):
    """Every kind of reduction's rows finished in one call, at the edges of the
    leaves and of the levels' forms: each the oracle's bits, NaN and infinities
    included (seventeen jobs: more than one launch takes)."""
    import oracle_lib as O
    import torch
    from hawk_amd import _core
    f32 = mode == "float32"
    dt = np.float32 if f32 else np.float64
    g = np.random.default_rng(rows)
    hi = (g.normal(size=rows) * 2.0 ** g.integers(-10, 10, rows)).astype(dt)
    lo = (hi * g.uniform(-1, 1, rows) * (2.0 ** -25 if f32 else 2.0 ** -54)).astype(dt)
    odd = hi.copy()
    odd[g.integers(0, rows, 3)] = (np.nan, np.inf, -np.inf)
    inf = hi.copy()
    inf[rows // 2] = np.inf
    planes = {k: torch.from_numpy(v).to(gpu) for k, v in (("hi", hi), ("lo", lo), ("odd", odd), ("inf", inf))}
    finish = O.rows_finish_f32 if f32 else O.rows_finish
    jobs = [("hi", _core.ROWS_SUM, finish(hi, lo)), ("odd", _core.ROWS_MAX, O.rows_extreme(odd, "max")),
            ("odd", _core.ROWS_MIN, O.rows_extreme(odd, "min")), ("inf", _core.ROWS_SUM, finish(inf, lo))]
    if not f32:
        jobs.append(("hi", _core.ROWS_BAND, O.band_rows_finish(hi, lo)))
    jobs += [jobs[i % 3] for i in range(17 - len(jobs))]
    out = torch.full((len(jobs),), 7.0, dtype=planes["hi"].dtype, device=gpu)
    call = (_core.RowsJob * len(jobs))()
    for i, (plane, op, _want) in enumerate(jobs):
        call[i].hi, call[i].lo, call[i].op = planes[plane].data_ptr(), planes["lo"].data_ptr(), op
        call[i].out = out.data_ptr() + i * out.element_size()
    scratch = torch.empty(_core.rows_finish_many_scratch_bytes(rows, len(jobs)), dtype=torch.uint8, device=gpu)
    _core.rows_finish_many(call, rows, f32, scratch.data_ptr(), torch.cuda.current_stream().cuda_stream)
    got = out.cpu().numpy()
    want = np.array([w for *_, w in jobs], dt)
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all() and got[~nan].tobytes() == want[~nan].tobytes()


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("n", [1, 6, 127, 1001, 70_003])
def test_sample_major_stage(tmp_path, gpu, mode, n):
    """Every vector and matrix plane sample-major: the stage over (N, w) planes
    gives the component-major run's bits; so does the copying path (a plane
    marked the other way, a strided plane, planes that share memory), which the
    rule must pick there, and a partial range touches only its samples."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Mutable, Scalar, Vector
    from hawk_amd import examples as E
    from hawk_amd.runtime import _PER_SAMPLE, _WRITTEN

    @hawk.kernel
    def total_vec(v: Vector[3], w: Mutable[Vector[2]], s: Mutable[Vector[3]]):
        w = hawk.math.vec(v[0] + v[1], v[2])
        s = hawk.sum(v * 2.0)

    dt = torch.float32 if mode == "float32" else torch.float64
    g = torch.Generator(device=gpu).manual_seed(n)
    for k in _unit(tmp_path, [E.energy, E.energy_vjp, E.spd_solve, E.spd_solve_vjp, E.twobody, total_vec], mode):
        ins, major = {}, set()
        for name in k.caller_planes():
            info = k.planes[name]
            if info["role"] == "uniform":
                ins[name] = 1.0
                continue
            shape = tuple(info["shape"]) + ((n,) if info["role"] in _PER_SAMPLE else ())
            ins[name] = torch.randn(shape, dtype=dt, device=gpu, generator=g)
            if name == "A":
                ins[name] += 20.0 * torch.eye(6, dtype=dt, device=gpu)[:, :, None]
            if info["shape"] and info["role"] in _PER_SAMPLE:
                major.add(name)
        assert set(k.sidecar["sample_major"]["planes"]) == major

        def run(change=lambda planes: planes, direct=True, **kw):
            planes = {name: x.movedim(-1, 0).contiguous() if name in major else x.clone() if torch.is_tensor(x) else x
                      for name, x in ins.items()}
            call = change(dict(planes))
            first = [name for name in major if not isinstance(call[name], hawk.layout.Marked)
                     or call[name].axis == "samples_first"]
            plain = {name: getattr(x, "array", x) for name, x in call.items()}
            assert k.takes_rows(plain, first, "plain") == direct
            hawk.run(k, layout="samples_first", **call, **kw)
            return {name: x.movedim(0, -1).contiguous() if name in first else x
                    for name, x in plain.items() if torch.is_tensor(x)}

        want = {name: x.clone() for name, x in ins.items() if torch.is_tensor(x)}
        hawk.run(k, layout="samples_last", **{**ins, **want})

        def same(got):
            for name, x in want.items():
                assert got[name].cpu().numpy().tobytes() == x.cpu().numpy().tobytes(), (k.name, name)
        same(run())
        one = sorted(major)[0]
        if len(major) > 1 and n != 6:
            same(run(lambda p: {**p, one: hawk.samples_last(ins[one].clone())}, direct=False))
        read = [m for m in sorted(major) if k.planes[m]["role"] not in _WRITTEN]
        if n > 1:
            wide = torch.empty((2 * n,) + tuple(k.planes[read[0]]["shape"]), dtype=dt, device=gpu)
            wide[::2] = ins[read[0]].movedim(-1, 0)
            same(run(lambda p: {**p, read[0]: wide[::2]}, direct=False))
        if k.name == "twobody":                          # stepping a state in place
            got = run(lambda p: {**p, "r": p["r0"], "v": p["v0"]}, direct=False)
            assert got["r"].cpu().numpy().tobytes() == want["r"].cpu().numpy().tobytes()
            assert got["v"].cpu().numpy().tobytes() == want["v"].cpu().numpy().tobytes()
        if n > 100 and not k.team:
            part = run(base=5, count=n - 60)
            for name, x in want.items():
                assert torch.equal(part[name][..., 5:n - 55], x[..., 5:n - 55])
                assert torch.equal(part[name][..., :5], ins[name][..., :5])
                assert torch.equal(part[name][..., n - 55:], ins[name][..., n - 55:])


def test_sample_major_banded_and_tables(tmp_path, gpu):
    """The stage over (N, w) planes in the banded mode, with its band rows, and
    beside tables: the component-major run's bits."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Grid, Mutable, Scalar, Table, Vector

    @hawk.kernel
    def banded_vec(v: Vector[3], w: Mutable[Vector[2]], s: Mutable[Scalar]):
        w = hawk.math.vec(v[0] * v[1], v[2])
        s = hawk.sum(v[0] * v[2])

    @hawk.kernel
    def by_key(lane: Grid["key", "sample":5], t: Table["key", "w":3], v: Vector[3], w: Mutable[Vector[2]]):
        w = hawk.math.vec(v[0] * t.at(key=lane.key, w=0), v[1] + v[2] * t.at(key=lane.key, w=2))
    n = 10_005
    g = torch.Generator(device=gpu).manual_seed(5)
    v = torch.randn(3, n, dtype=torch.float64, device=gpu, generator=g)
    table = torch.randn(n // 5 * 3, dtype=torch.float64, device=gpu, generator=g)
    for kernel, mode, more in ((banded_vec, "banded", dict(s=torch.zeros(1, dtype=torch.float64, device=gpu))),
                               (by_key, "float64", dict(t=table)), (by_key, "banded", dict(t=table))):
        (k,) = _unit(tmp_path, [kernel], mode)
        last, first = (dict(more, v=p, w=torch.full(shape, 7.0, dtype=torch.float64, device=gpu))
                       for p, shape in ((v, (2, n)), (v.t().contiguous(), (n, 2))))
        hawk.run(k, layout="samples_last", **last)
        cell = more["s"].clone() if "s" in more else None
        assert k.takes_rows(first, ["v", "w"], "plain")
        hawk.run(k, layout="samples_first", **first)
        assert torch.equal(first["w"].t(), last["w"]) and not (last["w"] == 7.0).any()
        assert cell is None or (torch.equal(more["s"], cell) and float(cell) != 0.0)


def test_plain_calls_direct_and_general(tmp_path, gpu):
    """hawk.run's direct path for plain calls and its general path: the same
    planes or the same refusal, call by call, and each call on the path that
    its planes say (True: the direct one)."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import examples as E
    n = 1001
    direct, general = (_unit(tmp_path, [E.scale, E.energy_vjp, E.spd_solve]) for _ in range(2))
    taken = []

    def watched(run_direct):
        def run(*args):
            taken.append(run_direct(*args))
            return taken[-1]
        return run
    for k in general:
        k._direct = None
    for k in direct:
        assert k._direct is not None
        k.run_direct = watched(k.run_direct)

    def t(*shape, dtype=torch.float64, device=gpu):
        return torch.randn(*shape, dtype=torch.float64, generator=torch.Generator().manual_seed(3)).to(dtype).to(device)
    x, v, bar = t(n), t(3, n), t(n)
    scale = dict(x=x, a=2.0, b=1.0)
    vjp = dict(v=v, bar_out=bar, bar_v=t(3, n))
    rows = dict(v=v.t().contiguous(), bar_out=bar, bar_v=t(n, 3))
    a = t(6, 6, 6) + 20.0 * torch.eye(6, dtype=torch.float64, device=gpu)[:, :, None]
    small = dict(v=t(3, 3), bar_out=t(3), bar_v=t(3, 3))
    calls = [(0, True, dict(scale, out=t(n))), (0, True, dict(scale, out=t(n), base=7, count=500)),
             (0, True, dict(scale, out=t(n), base=7)), (0, True, dict(scale, out=t(n), count=0)),
             (0, True, dict(scale, a=3, out=t(n))), (0, True, dict(scale, out=t(n), n_samples=n)),
             (0, False, dict(scale, out=t(n), n_samples=n - 1)), (0, False, dict(scale, out=t(n), base=-1)),
             (0, False, dict(scale, out=t(n), count=n + 1)), (0, False, dict(scale, out=t(n), base=True)),
             (0, False, dict(scale, a=True, out=t(n))), (0, False, dict(scale, a=np.float64(2.0), out=t(n))),
             (0, False, dict(scale, a=x, out=t(n))), (0, False, dict(scale)),
             (0, False, dict(scale, out=t(n), other=x)), (0, False, dict(scale, out=t(n - 1))),
             (0, False, dict(scale, out=t(n, 1))), (0, False, dict(scale, out=t(n, dtype=torch.float32))),
             (0, False, dict(scale, out=t(n, device="cpu"))), (0, False, dict(scale, out=t(2 * n)[::2])),
             (0, False, dict(scale, out=torch.nn.Parameter(t(n)))), (0, True, dict(x=t(0), a=1.0, b=1.0, out=t(0))),
             (0, False, dict(scale, out=t(n), layout="rows")), (0, False, dict(scale, out=t(n), steps=1)),
             (0, False, dict(scale, out=t(n), entry="range")),
             (0, True, dict(scale, out=t(n), stream=torch.cuda.Stream())),
             (1, True, vjp), (1, True, rows), (1, True, dict(vjp, layout="samples_last")),
             (1, True, dict(rows, layout="samples_first")), (1, False, dict(rows, layout="samples_last")),
             (1, False, dict(vjp, layout="samples_first")), (1, False, dict(vjp, v=rows["v"])),
             (1, False, dict(rows, v=hawk.samples_first(rows["v"]))), (1, False, small),
             (1, True, dict(small, layout="samples_first")), (1, True, dict(small, layout="samples_last")),
             (2, False, dict(A=a, b=t(6, 6), x=t(6, 6))),
             (2, True, dict(A=a, b=t(6, 6), x=t(6, 6), layout="samples_last")),
             (2, True, dict(A=a.movedim(-1, 0).contiguous(), b=t(6, 6), x=t(6, 6), layout="samples_first"))]
    for which, plain, call in calls * 2:             # twice: fresh and held bindings
        done = []
        taken.clear()
        for k in (direct[which], general[which]):
            # fresh output planes a side, the same values in both
            planes = {name: p.clone() if type(p) is torch.Tensor and p.is_contiguous()
                      and name in ("out", "bar_v", "x") and which + (name == "out") else p for name, p in call.items()}
            torch.cuda.synchronize()
            try:
                hawk.run(k, **planes)
                torch.cuda.synchronize()
                done.append({name: p.detach().cpu().numpy().tobytes() for name, p in planes.items()
                             if isinstance(p, torch.Tensor)})
            except Exception as e:
                done.append((type(e), str(e)))
        said = (which, {name: getattr(p, "shape", p) for name, p in call.items()}, done)
        assert done[0] == done[1], said
        assert any(taken) == plain, said


def test_refused_param_leaves_bindings(tmp_path, gpu):
    """A call refused at a Param, after a plane before it has moved, leaves the
    binding of the last run: the next call over the moved plane reads it."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import examples as E
    scale, = _unit(tmp_path, [E.scale])
    first, second = (torch.full((1001,), value, dtype=torch.float64, device=gpu) for value in (1.0, 5.0))
    out = torch.empty_like(first)
    hawk.run(scale, x=first, a=2.0, b=1.0, out=out)
    want = out.clone()
    hawk.run(scale, x=second, a=2.0, b=1.0, out=out)
    moved = out.clone()
    assert not torch.equal(want, moved)
    hawk.run(scale, x=first, a=2.0, b=1.0, out=out)
    with pytest.raises(OverflowError):
        hawk.run(scale, x=second, a=10 ** 400, b=1.0, out=out)
    hawk.run(scale, x=second, a=2.0, b=1.0, out=out)
    assert torch.equal(out, moved)


@pytest.mark.parametrize("mode", ["float64", "float32"])
def test_a_param_of_the_other_zero_is_bound(tmp_path, gpu, mode):
    """A call with -0.0 after one with 0.0 (and the reverse) runs on its own
    zero, on the direct path and the general one: 1 * a keeps the sign."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Param, Scalar

    @hawk.kernel
    def times(x: Scalar, a: Param) -> Scalar:
        return x * a
    x = torch.ones(100, dtype=torch.float32 if mode == "float32" else torch.float64, device=gpu)
    for direct in (True, False):
        (k,) = _unit(tmp_path, [times], mode)
        if not direct:
            k._direct = None
        for a in (0.0, -0.0, -0.0, 0.0, 1.0, -0.0, 0):
            out = torch.full_like(x, 7.0)
            hawk.run(k, x=x, a=a, out=out)
            want = np.full(100, a, out.cpu().numpy().dtype)
            assert out.cpu().numpy().tobytes() == want.tobytes(), (direct, a)


@pytest.mark.parametrize("n", [1, 5000, 300_000])
def test_reductions_into_one_cell_leave_the_last(tmp_path, gpu, n):
    """Reductions that share a cell are written in the kernel's order."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Mutable, Scalar

    @hawk.kernel
    def three(x: Scalar, a: Mutable[Scalar], o: Mutable[Scalar], b: Mutable[Scalar]):
        a = hawk.sum(x * 2.0)
        o = hawk.sum(x, policy="ordered")
        b = hawk.max(x)
    (k,) = _unit(tmp_path, [three])
    x = torch.arange(n, dtype=torch.float64, device=gpu) % 1024 + 1.0
    one, two = (torch.zeros(1, dtype=torch.float64, device=gpu) for _ in range(2))
    for cells, want in (((one, two, one), x.max()), ((one, one, one), x.max()), ((two, one, one), x.max()),
                        ((one, one, two), x.sum())):
        for call in (lambda **p: hawk.run(k, **p), lambda **p: k.prepare(**p)()):
            call(x=x, a=cells[0], o=cells[1], b=cells[2])
            assert float(one) == float(want), (n, call)


def test_two_streams_of_one_kernel(tmp_path, gpu):
    """One kernel's runs and launchers on two streams at once: each ends with
    the cells of its own inputs."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Index, Mutable, Scalar

    @hawk.kernel
    def all_of(x: Scalar, key: Index, a: Mutable[Scalar], b: Mutable[Scalar], o: Mutable[Scalar],
               bins: Mutable[Scalar]):
        a = hawk.sum(x * x)
        b = hawk.max(x)
        o = hawk.sum(x * 2.0, policy="ordered")
        hawk.scatter(bins, policy="ordered")[key] += x * 3.0
    (k,) = _unit(tmp_path, [all_of])
    n, cells = 300_007, 30_000
    streams, sides = [torch.cuda.Stream() for _ in range(2)], []
    for i in range(2):
        g = torch.Generator(device=gpu).manual_seed(i)
        sides.append(dict(x=torch.randn(n, dtype=torch.float64, device=gpu, generator=g) + 10.0 * i,
                          key=torch.randint(0, cells, (n,), dtype=torch.int32, device=gpu, generator=g),
                          bins=torch.zeros(cells, dtype=torch.float64, device=gpu),
                          **{c: torch.zeros(1, dtype=torch.float64, device=gpu) for c in "abo"}))
    want = []
    for p in sides:                                   # one stream alone
        hawk.run(k, **p)
        want.append({name: x.clone() for name, x in p.items()})
    torch.cuda.synchronize()
    launchers = [k.prepare(stream=s, **p) for s, p in zip(streams, sides)]
    for way in ("run", "launcher"):
        for turn in range(20):
            for s, p, launch in zip(streams, sides, launchers):
                with torch.cuda.stream(s):
                    for name in ("bins", "a", "b", "o"):
                        p[name].zero_()
                    hawk.run(k, check=False, **p) if way == "run" else launch()
        torch.cuda.synchronize()
        for p, w in zip(sides, want):
            for name in p:
                assert torch.equal(p[name], w[name]), (way, name)


def test_captured_calls_keep_their_scratch(tmp_path, gpu):
    """A graph of a launcher and one of hawk.run on the same stream, replayed
    with other inputs between eager runs of larger and smaller sizes there: the
    eager results, every time."""
    import hawk_amd as hawk
    import torch
    from hawk_amd import Index, Mutable, Scalar

    @hawk.kernel
    def all_of(x: Scalar, key: Index, a: Mutable[Scalar], b: Mutable[Scalar], o: Mutable[Scalar],
               bins: Mutable[Scalar]):
        a = hawk.sum(x * x)
        b = hawk.max(x)
        o = hawk.sum(x * 2.0, policy="ordered")
        hawk.scatter(bins, policy="ordered")[key] += x * 3.0
    (k,) = _unit(tmp_path, [all_of])

    def planes(n, seed):
        g = torch.Generator(device=gpu).manual_seed(seed)
        return dict(x=torch.randn(n, dtype=torch.float64, device=gpu, generator=g),
                    key=torch.randint(0, 20_000, (n,), dtype=torch.int32, device=gpu, generator=g),
                    bins=torch.zeros(20_000, dtype=torch.float64, device=gpu),
                    **{c: torch.zeros(1, dtype=torch.float64, device=gpu) for c in "abo"})
    n = 50_001
    inputs = [planes(n, seed) for seed in range(3)]
    want = []
    for p in inputs:
        hawk.run(k, **p)
        want.append({name: x.clone() for name, x in p.items()})
    p = planes(n, 9)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    launch = k.prepare(stream=side, **p)
    graphs = []
    for call in (launch, lambda: hawk.run(k, check=False, **p)):
        with torch.cuda.stream(side):
            call()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            call()
        graphs.append(graph)
    for turn, other in enumerate((1_000, 400_003, 100, 900_001)):
        for graph in graphs:
            source, result = inputs[turn % 3], want[turn % 3]
            with torch.cuda.stream(side):
                hawk.run(k, check=False, **planes(other, turn))
                for name in ("x", "key"):
                    p[name].copy_(source[name])
                p["bins"].zero_()
                graph.replay()
            side.synchronize()
            for name in p:
                assert torch.equal(p[name], result[name]), (turn, name)


def test_work_beside_a_launch_is_on_its_stream(gpu):
    """Resets, fills and allocations go to the launch's stream, the default
    stream inside another one's context included."""
    import torch
    from hawk_amd import runtime
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    for current in (torch.cuda.default_stream(), side):
        for stream in (0, side.cuda_stream, other.cuda_stream):
            with torch.cuda.stream(current):
                with runtime._on(stream):
                    assert torch.cuda.current_stream().cuda_stream == stream
                assert torch.cuda.current_stream() == current
