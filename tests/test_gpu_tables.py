"""GPU parity of the table-driven kernels at the sizes where their tiles,
staged tables and remainders can go wrong, against the complex128 CPU oracle.

Tolerances: a sum of T products in a type of unit roundoff u is off by at
most (T + c) u times the sum of magnitudes; each test names its T and takes
c for the few operations around the sum.
"""
import numpy as np
import pytest
import torch

from oracle import statevector as sv

pytestmark = pytest.mark.gpu

UNIT = {torch.complex64: 2.0**-24, torch.complex128: 2.0**-53}
DTYPES = (torch.complex64, torch.complex128)


def np_of(t):
    return t.detach().cpu().numpy()


def random_states(rng, batch, n):
    s = rng.standard_normal((batch, 2**n)) + 1j * rng.standard_normal((batch, 2**n))
    return s / np.linalg.norm(s, axis=1, keepdims=True)


# (qubits, terms, letters): states smaller than a wave, one tile exactly, a
# tile and a bit, several tiles; 600 terms of one flip group (Z only) and 700
# mixed ones fill more than one chunk of staged terms
@pytest.mark.parametrize("n,T,letters", [(1, 3, 4), (3, 6, 4), (4, 9, 4), (5, 40, 4), (7, 30, 4), (10, 33, 4),
                                         (11, 700, 4), (12, 600, "z"), (13, 300, "xz"), (14, 25, 4), (15, 700, "z")])
def test_pauli_tile(gpu, n, T, letters):
    from tensorcircuit_amd import engine

    rng = np.random.default_rng(1000 * n + T)
    alphabet = {4: [0, 1, 2, 3], "z": [0, 3], "xz": [0, 0, 0, 0, 0, 0, 1, 3]}[letters]
    codes = rng.choice(alphabet, size=(T, n)).astype(np.int8)
    w = rng.standard_normal(T)
    terms = [(float(w[k]), list(codes[k])) for k in range(T)]
    wsum = np.abs(w).sum()
    s = random_states(rng, 3, n)
    ham = engine.PauliSum(n, codes, w, jit=0)
    alpha = np.array([0.5, -1.0, 2.0])
    for dt in DTYPES:
        st = torch.as_tensor(s).to(dt).cuda()
        sd = np_of(st).astype(np.complex128)
        # T weights summed, then one product and sum per flip group (<= T)
        tol = (2 * T + 8) * UNIT[dt] * wsum
        e = np_of(ham.expect(st))
        hs = np_of(ham.apply(st, torch.as_tensor(alpha).cuda()))
        for b in range(3):
            assert abs(e[b] - sv.pauli_sum_expectation(sd[b], n, terms)) <= tol
            ref = alpha[b] * sv.pauli_sum_apply(sd[b], n, terms)
            assert np.abs(hs[b] - ref).max() <= 2.0 * tol
