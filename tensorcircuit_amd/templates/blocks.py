"""Ansatz blocks (the reference's templates/blocks.py) and the HEA layer used
by the statevector benchmarks."""
from __future__ import annotations

from typing import Any

import numpy as np

import torch

from .. import gates as G


def _rows(param: Any, nrows: int) -> Any:
    """The first ``nrows`` rows of angles.  Those of a tensor are split by two
    levels of unbind, whose backward is a stack each: an angle taken by
    ``param[r, i]`` costs two select nodes, and in backward a fill, a copy and
    an addition of the whole of ``param`` each."""
    if isinstance(param, torch.Tensor) and param.dim() >= 2:
        rows = param.unbind(0)
        return [rows[r].unbind(0) for r in range(nrows)]
    return [_Row(param, r) for r in range(nrows)]


class _Row:
    def __init__(self, param: Any, r: int):
        self.param, self.r = param, r

    def __getitem__(self, i: int) -> Any:
        return self.param[self.r, i]


def example_block(c: Any, param: Any, nlayers: int = 2, is_split: bool = False) -> Any:
    """H on every qubit, then ``nlayers`` of exp1(ZZ) ladders and rx
    (templates/blocks.py:113-152); ``param`` reshaped to [2*nlayers, n]."""
    n = c._nqubits
    param = param.reshape(2 * nlayers, n) if hasattr(param, "reshape") else np.reshape(param, (2 * nlayers, n))
    rows = _rows(param, 2 * nlayers)
    for i in range(n):
        c.H(i)
    for j in range(nlayers):
        for i in range(n - 1):
            c.exp1(i, i + 1, unitary=G._zz_matrix, theta=rows[2 * j][i])
        for i in range(n):
            c.rx(i, theta=rows[2 * j + 1][i])
    return c


def hea_layers(c: Any, param: Any, nlayers: int, barrier: bool = True) -> Any:
    """Per layer: ry on every qubit, rz on every qubit, CNOT chain i -> i+1;
    ``param`` laid out [2*nlayers, n] (row 2j = ry of layer j, row 2j+1 = rz),
    the indexing idiom of tests/test_backends.py:426-442."""
    n = c._nqubits
    rows = _rows(param, 2 * nlayers)
    for j in range(nlayers):
        for i in range(n):
            c.ry(i, theta=rows[2 * j][i])
        for i in range(n):
            c.rz(i, theta=rows[2 * j + 1][i])
        for i in range(n - 1):
            c.cnot(i, i + 1)
        if barrier:
            c.barrier_instruction()
    return c
