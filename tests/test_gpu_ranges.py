"""Calls at the ends of their ranges."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def np_of(t):
    return t.detach().cpu().numpy()


def test_tables_of_many_parameter_sets(gpu):
    """Two programs whose parameter sets fit one launch of 2^32 threads each
    but not together."""
    from tensorcircuit_amd import _lib, engine

    B = 9_000_000
    th = torch.rand(B, 1, device=gpu) * 6.0 - 3.0
    items = []
    for kind in (_lib.G_RX, _lib.G_RY):
        prog = engine.Program(1, [engine.GateSpec(kind, (0,), 0, 0.0, 1.0, None)], 1, fuse=1)
        items.append((prog, th, torch.full((B, 2), 7.0, dtype=torch.complex64, device=gpu)))
    engine.forward_multi(items, "complex64")
    c, s = torch.cos(0.5 * th.double()), torch.sin(0.5 * th.double())
    # entries within one unit of the last place of a float, one product each
    for (_, _, st), one in zip(items, (torch.complex(0 * s, -s), torch.complex(s, 0 * s))):
        ref = torch.cat([torch.complex(c, 0 * c), one], dim=1)
        assert float((st - ref).abs().max()) <= 4 * 2.0**-24
