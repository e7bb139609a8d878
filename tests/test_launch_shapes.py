"""The launch shape a build gives a stage, by its planes, operations and tables."""

from __future__ import annotations

import pytest

import hawk_amd as hawk
from hawk_amd import Mutable, Scalar, Vector


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
