"""Tied groups of an augmenting path, taken row by row with the columns in
registers (K > 64), against the pinned C oracle: bit-exact mappings.

The padding columns of N > M are one such group of N - M members; square
inputs with repeated values make small groups, rows with many joins (handed
back to the position-by-position scan) and groups of two.  Shapes lie at the
edges of the chunk counts (65, 127..129, 512/513) and above the 1024 columns
up to which rows are cached.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import torchmatch_amd  # noqa: F401
from oracle import jv

pytestmark = pytest.mark.gpu

SHAPES = [(4, 65, 64), (4, 65, 20), (3, 127, 126), (3, 128, 90), (3, 129, 129), (2, 190, 257),
          (2, 300, 193), (2, 512, 470), (2, 513, 511), (1, 769, 700), (1, 1100, 1060)]


def _cost(kind: str, shape, g) -> np.ndarray:
    b, n, m = shape
    if kind == "uniform":
        return g.random(shape, dtype=np.float32)
    if kind == "tied":  # a few values: rows with many joins
        return g.integers(0, 7, shape).astype(np.float32)
    if kind == "pairs":  # every column twice: groups of two
        half = g.random((b, n, (m + 1) // 2), dtype=np.float32)
        return np.ascontiguousarray(np.repeat(half, 2, axis=2)[:, :, :m])
    c = g.standard_normal(shape).astype(np.float32)  # masked, either sign
    c[g.random(shape) < 0.3] = np.inf
    return c


@pytest.mark.parametrize("kind", ["uniform", "tied", "pairs", "masked"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_tied_groups_match_oracle(shape, kind, device):
    c = _cost(kind, shape, np.random.default_rng(sum(shape) + len(kind)))
    print(f"{kind} {shape}", flush=True)
    x = torch.from_numpy(c).to(device)
    got = torch.ops.assignment.jonker_dense_batch(x).cpu().numpy()
    np.testing.assert_array_equal(got, jv.jv_dense_batch(c))
    got = torch.ops.assignment.jonker_compact_batch(x).cpu().numpy()
    np.testing.assert_array_equal(got, jv.jv_compact_batch(c))
