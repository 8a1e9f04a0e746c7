"""The list-based launcher's checks, made before anything touches the GPU:
which block ids and table lengths it takes, and whose error comes first."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from memforge_amd import _native as nat
from memforge_amd.kernels._varlen import padded_tables_host, run_varlen


def _run(tables, seq_ids, positions, blocks=8, **kw):
    pool = nat.PoolView.from_bshd(torch.zeros((blocks, 16, 1, 32)), torch.zeros((blocks, 16, 1, 32)))
    q = torch.zeros((len(seq_ids), 2, 32))
    run_varlen(q, torch.empty_like(q), pool, tables, seq_ids, positions, None, 1, **kw)


@pytest.mark.parametrize("tables,positions,match", [
    ([[0, 8], [1]], [16, 3], "table of sequence 0 names a block outside the pool of 8"),
    ([[0], [-1]], [3, 3], "table of sequence 1 names a block outside"),
    ([[0], [1]], [3, 16], "sequence 1 needs 2 blocks but its block table has 1"),
    ([[9], [1]], [3, 16], "table of sequence 0 names a block outside"),  # the first sequence's fault comes first
])
def test_bad_tables_are_refused(tables, positions, match):
    with pytest.raises(IndexError, match=match):
        _run(tables, [0, 1], positions)


@pytest.mark.parametrize("tables,positions,kw", [
    ([[0, 99], [1, -5]], [15, 0], {}),                       # entries past what is read may hold anything
    ([[7], [1]], [40, 2], {"pool_lens": [16, 2]}),           # in-flight keys need no block
])
def test_good_tables_reach_the_device_check(tables, positions, kw):
    with pytest.raises(ValueError, match="runs on the GPU"):  # the next check: these tensors are on the CPU
        _run(tables, [0, 1], positions, **kw)


def test_padded_tables_are_int32_rows():
    got = padded_tables_host([[3, 1], [], [5]])
    assert got.dtype == np.int32 and got.tolist() == [[3, 1], [0, 0], [5, 0]]
