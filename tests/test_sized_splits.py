"""Into how many runs the keys of rows over one cached vector go: never more than 64, never runs of less than two tiles, twice the
workgroups only where every run keeps its share."""
import types

import pytest

from tiny_llm_infer_amd.kernels.ops import HipOps


def splits(rows, reach, units=16, key_heads=1, window=None, keep=0):
    stub = types.SimpleNamespace(sized_splits=None, SIZED_WORKGROUPS=HipOps.SIZED_WORKGROUPS, SIZED_SPLIT_KEYS=HipOps.SIZED_SPLIT_KEYS,
                                 SIZED_WIDE_KEYS=HipOps.SIZED_WIDE_KEYS)
    return HipOps._sized_splits(stub, rows, reach, units, key_heads, window, keep)


@pytest.mark.parametrize("rows, reach, want", [(1, 128, 4), (1, 8192, 64), (8, 4096, 32), (8, 8192, 64), (16, 2048, 16), (16, 4096, 32),
                                               (32, 1024, 8), (32, 2048, 16), (64, 512, 4), (64, 1024, 8), (128, 256, 2), (128, 512, 4),
                                               (300, 256, 1), (512, 8192, 1), (2000, 8192, 1)])
def test_runs_of_rows(rows, reach, want):
    assert splits(rows, reach) == want


def test_what_was_not_measured_stays():
    assert splits(32, 8192, units=32) == 8 and splits(32, 8192, keep=4) == 8          # other kernel; kept first keys
    assert splits(32, 8192, window=500) == 8 and splits(16, 8192, units=32, key_heads=2) == 16


@pytest.mark.parametrize("rows, reach, want", [(8, 8192, 32), (1, 8192, 64), (16, 8192, 32), (64, 1024, 8)])
def test_narrow_vectors_go_into_fewer_runs(rows, reach, want):
    """Short vectors are read faster than many runs' sums of them are merged: 64 runs only where there are no more rows."""
    stub = types.SimpleNamespace(sized_splits=None, SIZED_WORKGROUPS=HipOps.SIZED_WORKGROUPS, SIZED_SPLIT_KEYS=HipOps.SIZED_SPLIT_KEYS,
                                 SIZED_WIDE_KEYS=HipOps.SIZED_WIDE_KEYS)
    assert HipOps._sized_splits(stub, rows, reach, 16, 1, None, 0, 128) == want
