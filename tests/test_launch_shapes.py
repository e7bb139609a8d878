"""The launch shape a build gives a stage, by its planes, operations and tables."""

from __future__ import annotations

import pytest

import hawk_amd as hawk
from hawk_amd import Grid, Index, Mutable, Scalar, Table, Vector


@hawk.kernel
def rows4(a: Vector[2], b: Mutable[Vector[2]]):
    b = a * 2.0


@hawk.kernel
def rows5(a: Vector[3], b: Mutable[Vector[2]]):
    b = hawk.math.vec(a[0] + a[1], a[2])


@hawk.kernel
def rows8(a: Vector[4], b: Mutable[Vector[4]]):
    b = a * 2.0


@hawk.kernel
def rows9(a: Vector[3], b: Vector[3], c: Mutable[Vector[3]]):
    c = a + b


@hawk.kernel
def rows16(a: Vector[8], b: Mutable[Vector[8]]):
    b = a * 2.0


@hawk.kernel
def rows17(a: Vector[8], s: Scalar, b: Mutable[Vector[8]]):
    b = a * s


def _shape(tmp_path, kernel, mode):
    launch = hawk.build([kernel], tmp_path, mode=mode).sidecar(kernel.name)["launch"]
    return launch["block"], launch["per_thread"]


@pytest.mark.parametrize("mode, kernel, shape", [
    ("float32", rows5, (256, 1)), ("float32", rows8, (256, 1)), ("float32", rows9, (256, 1)),
    ("float32", rows16, (256, 1)), ("float32", rows17, (128, 1)), ("float64", rows4, (128, 1)),
    ("float64", rows5, (256, 1)), ("float64", rows8, (256, 1)), ("float64", rows9, (128, 1))])
def test_streams_by_their_bytes(tmp_path, mode, kernel, shape):
    """Workgroups of 256 between 32 (float32: 16) and 64 plane bytes a sample."""
    assert _shape(tmp_path, kernel, mode) == shape


@hawk.kernel
def light(lane: Grid["key", "sample":64], t: Table["key", "w":3], x: Scalar, y: Mutable[Scalar]):
    s = 0.0 * x
    for i in range(3):
        s = s * x + t.at(key=lane.key, w=i)
    y = s


@hawk.kernel
def heavy(lane: Grid["key", "sample":4], t: Table["key", "w":24], x: Scalar, y: Mutable[Scalar]):
    s = 0.0 * x
    for i in range(24):
        s = s * x + t.at(key=lane.key, w=i)
    y = s


@hawk.kernel
def strided(lane: Grid["key", "sample":4], t: Table["s":4096], x: Scalar, y: Mutable[Scalar]):
    y = x * t.at(s=lane.sample * 3 + lane.key)


@hawk.kernel
def spread(lane: Grid["key", "sample":4], t: Table["s":4096], x: Scalar, y: Mutable[Scalar]):
    y = x * t.at(s=(lane.flat * 7919) % 4096)


@hawk.kernel
def by_plane(lane: Grid["key", "sample":4], t: Table["s":4096], i: Index, x: Scalar, y: Mutable[Scalar]):
    y = x * t.at(s=i)


@pytest.mark.parametrize("mode", ["float64", "float32"])
@pytest.mark.parametrize("kernel, shape", [(light, (256, 2)), (heavy, (256, 1)), (strided, (256, 2)),
                                           (spread, (1024, 2)), (by_plane, (1024, 2))])
def test_tables_by_how_they_are_read(tmp_path, mode, kernel, shape):
    """Along the lanes two samples a thread, or one in a heavy stage; scattered
    by arithmetic or by a plane the gather's shape."""
    assert _shape(tmp_path, kernel, mode) == shape
