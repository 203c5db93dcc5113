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


def test_launches_of_many_small_states(gpu):
    """2^26 states of four qubits: a wave each is 2^32 threads."""
    from tensorcircuit_amd import _lib, engine

    n, B = 4, (1 << 26) + 5
    x = np.array([[0, 1], [1, 0]])
    prog = engine.Program(n, [engine.GateSpec(_lib.G_MAT, (q,), -1, 0.0, 1.0, x) for q in (0, 3)], 0, fuse=1)
    st = torch.zeros(B, 16, dtype=torch.complex64, device=gpu)
    prog.forward(None, B, "complex64", out=st)
    ref = torch.zeros(16, dtype=torch.complex64, device=gpu)
    ref[0b1001] = 1.0
    for part in st.split(1 << 22):
        assert bool((part == ref).all())
    codes = [[1, 0, 0, 0], [0, 0, 0, 3]]
    hs = engine.PauliSum(n, codes, [2.0, 1.0], jit=0).apply(st)
    ref = torch.zeros(16, dtype=torch.complex64, device=gpu)
    ref[0b0001], ref[0b1001] = 2.0, -1.0
    for part in hs.split(1 << 22):
        assert bool((part == ref).all())


def test_multi_program_launch_of_many_states(gpu):
    """Programs whose tiles come to 2^32 threads when they share a launch."""
    from tensorcircuit_amd import _lib, engine

    x = np.array([[0, 1], [1, 0]])
    items = []
    for n, B in ((4, 9_000_000), (12, 3), (5, 9_000_000)):
        prog = engine.Program(n, [engine.GateSpec(_lib.G_MAT, (0,), -1, 0.0, 1.0, x)], 0, fuse=1)
        items.append((prog, None, torch.zeros(B, 1 << n, dtype=torch.complex64, device=gpu)))
    engine.forward_multi(items, "complex64")
    for prog, _, st in items:
        ref = torch.zeros(st.shape[1], dtype=torch.complex64, device=gpu)
        ref[st.shape[1] // 2] = 1.0
        for part in st.split(1 << 22):
            assert bool((part == ref).all())


def test_terms_of_many_states(gpu):
    """65535 states x 1100 strings: 2^26 sums, a wave each."""
    from tensorcircuit_amd import engine

    T, B = 1100, 65535
    ham = engine.PauliSum(1, [[3]] * T, np.ones(T))
    st = torch.zeros(B, 2, dtype=torch.complex64, device=gpu)
    st[:, 1] = 1.0
    e = ham.expect_terms(st)
    assert bool((e.real == -1.0).all()) and bool((e.imag == 0.0).all())


def draws(p, u):
    from tensorcircuit_amd import engine

    n = p.shape[1].bit_length() - 1
    return engine.sample_prob_indices(p.cuda(), n, torch.as_tensor(u)).cpu().numpy()


# one stretch of 64 indices, one chunk of 1024, several chunks, more than 256
# and more than 4096 of them: the running sums over indices without weight
# (behind, before and between those with weight) stay what they are, so that
# no such index is drawn, least of all for u = 0
@pytest.mark.parametrize("n", [2, 6, 9, 10, 12, 18, 19, 20, 23])
def test_draws_have_weight(gpu, n):
    N = 1 << n
    reps = 2 if n > 20 else 10 if n > 12 else 40
    for dt in (torch.float32, torch.float64):
        for seed in range(reps):
            rng = np.random.default_rng(1000 * n + seed)
            w = rng.random((3, N))
            cut = int(rng.integers(1, N))
            w[0, cut:] = 0.0
            w[1, N // 2:] = 0.0
            w[2] *= np.repeat(rng.random(max(N // 32, 1)) < 0.3, min(N, 32))  # 32 at a time
            w[2, rng.integers(0, N)] = 1.0
            p = torch.as_tensor(w).to(dt)
            u = np.concatenate([np.zeros((3, 1)), rng.random((3, 200))], axis=1)
            # r on the running sums themselves
            cdf = np.cumsum(p.double().numpy(), axis=1)
            at = rng.integers(0, N, (3, 50))
            u = np.concatenate([u, np.maximum(0.0, 1.0 - np.take_along_axis(cdf, at, 1) / cdf[:, -1:])], axis=1)
            u = np.where(u < 1.0, u, 0.5)
            got = draws(p, u)
            drawn = np.take_along_axis(p.numpy(), got, 1)
            assert (drawn > 0).all(), (dt, seed, np.argwhere(~(drawn > 0))[:5])


@pytest.mark.parametrize("shots", [1, 70])
def test_draws_from_one_qubit(gpu, shots):
    rng = np.random.default_rng(shots)
    p = torch.as_tensor([[0.25, 0.75], [1.0, 0.0], [0.0, 2.0], [3.0, 1.0]])
    u = rng.random((4, shots))
    r = p.numpy().sum(axis=1, keepdims=True) * (1.0 - u)
    for dt in (torch.float32, torch.float64):
        assert (draws(p.to(dt), u) == (r > p.numpy()[:, :1])).all()


@pytest.mark.parametrize("kind", ["rx", "ry"])
@pytest.mark.parametrize("jit", [0, 1])
def test_angles_of_many_turns(gpu, kind, jit):
    """Rotations by angles of up to 10^9, reduced to one turn without loss."""
    from tensorcircuit_amd import _lib, engine

    n = 10
    th = np.array([0.3, -2.0, 3.0, 4.0, 9.5, 1e3, -1e5, 1e7, 12345678.9, -1e9])
    code = {"rx": _lib.G_RX, "ry": _lib.G_RY}[kind]
    prog = engine.Program(n, [engine.GateSpec(code, (q,), q, 0.0, 1.0, None) for q in range(n)], n, fuse=1, jit=jit)
    got = np_of(prog.forward(torch.as_tensor(th)[None].to(gpu), 1, "complex128")[0])[0]
    ref = np.ones(1)
    for t in th:
        c, s = np.cos(0.5 * t), np.sin(0.5 * t)
        ref = np.kron(ref, [c, -1j * s if kind == "rx" else s])
    # ten rotations, each of up to three shears with two rounded constants
    assert np.abs(got - ref).max() <= 10 * 3 * 4 * 2.0**-53


@pytest.mark.parametrize("hermitian", [True, False])
def test_sparse_cotangent_that_is_not_finite(gpu, hermitian):
    """A cotangent with a NaN part shows in the gradient, also where only its
    real part counts (A = A^dagger)."""
    from tensorcircuit_amd import engine

    N = 64
    rng = np.random.default_rng(5)
    m = rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))
    if hermitian:
        m = m + m.conj().T
    x = torch.as_tensor(rng.standard_normal((2, N)) + 0j).to(gpu)
    a = engine.CsrMatrix(torch.as_tensor(m).to(gpu).to_sparse_csr(), 6, torch.complex128)
    assert a.hermitian == hermitian
    for bad in (complex(1.0, float("nan")), complex(float("nan"), 1.0), complex(0.0, float("inf"))):
        y = a.vjp(x, torch.tensor([bad, 1.0 + 0j], device=gpu))
        assert not torch.isfinite(torch.view_as_real(y[0])).any()
        assert torch.isfinite(torch.view_as_real(y[1])).all()


# tables of 1, 2, 5, 24, 60 and 300 entries: up to 256 parameter sets to a
# block, one set and part of one; batches that leave the last block part empty
@pytest.mark.parametrize("n,gates", [(1, 1), (2, 2), (3, 5), (4, 3), (6, 24), (8, 60), (10, 300)])
@pytest.mark.parametrize("batch", [2, 5, 129, 257])
def test_tables_sharing_blocks(gpu, n, gates, batch):
    from tensorcircuit_amd import _lib, engine

    kinds = (_lib.G_RX, _lib.G_RZ, _lib.G_RY, _lib.G_PHASE)
    specs = [engine.GateSpec(kinds[g % 4], (g % n,), g, 0.0, 1.0, None) for g in range(gates)]
    prog = engine.Program(n, specs, gates, fuse=1)
    for dt, rdt in (("complex64", torch.float32), ("complex128", torch.float64)):
        p = torch.randn(batch, gates, dtype=rdt, device=gpu)
        st, _ = prog.forward(p, batch, dt)
        for b in sorted({0, 1, batch // 2, batch - 2, batch - 1}):
            assert torch.equal(st[b], prog.forward(p[b:b + 1], 1, dt)[0][0])


# many states run by tiles, one state straight from memory: one tile, several,
# flips that leave it; 33 strings (a second chunk), Z only, and one to seven
# strings (the lines between the two ways)
@pytest.mark.parametrize("n,T,batch", [(9, 33, 1100), (10, 40, 700), (11, 33, 300), (12, 90, 150), (13, 64, 60),
                                       (12, 1, 150), (12, 2, 150), (12, 3, 1500), (11, 7, 1300)])
@pytest.mark.parametrize("letters", [(0, 1, 2, 3), (0, 3), (0, 0, 0, 1, 3)])
def test_pauli_strings_by_tiles_and_without(gpu, n, T, batch, letters):
    from tensorcircuit_amd import engine

    rng = np.random.default_rng(100 * n + T)
    codes = rng.choice(letters, size=(T, n)).astype(np.int8)
    w = rng.standard_normal(T)
    ham = engine.PauliSum(n, codes, w)
    a = torch.as_tensor(rng.standard_normal((batch, T))).to(gpu)
    for dt, unit in ((torch.complex64, 2.0**-24), (torch.complex128, 2.0**-53)):
        st = torch.randn(batch, 1 << n, dtype=dt, device=gpu)
        st /= torch.linalg.vector_norm(st, dim=1, keepdim=True)
        e, y = ham.expect_terms(st), ham.apply_terms(st, a)
        for b in (0, 1, batch // 2, batch - 1):
            # sums of 2^n products of total size one in 64 bits
            assert float((e[b] - ham.expect_terms(st[b])[0]).abs().max()) <= np.abs(w).max() * n * 2.0**-50
            # sums of T in 64 bits, rounded once
            size = float((a[b].abs() * torch.as_tensor(np.abs(w)).to(gpu)).sum() * st[b].abs().max())
            assert float((y[b] - ham.apply_terms(st[b], a[b:b + 1])[0]).abs().max()) <= 4 * (unit + T * 2.0**-53) * size
        # a state that starts between 16-byte boundaries
        buf = torch.empty((1 << n) + 1, dtype=dt, device=gpu)
        buf[1:] = st[0]
        assert float((e[0] - ham.expect_terms(buf[1:])[0]).abs().max()) <= np.abs(w).max() * n * 2.0**-50
        y0 = ham.apply_terms(buf[1:], a[:1])[0]
        assert float((y[0] - y0).abs().max()) <= 4 * (unit + T * 2.0**-53) * float(
            (a[0].abs() * torch.as_tensor(np.abs(w)).to(gpu)).sum() * st[0].abs().max())


@pytest.mark.parametrize("n", [13, 14, 16])
@pytest.mark.parametrize("dtype,bits", [("complex64", 14), ("complex128", 13)])
def test_widest_adjoint_tiles(gpu, n, dtype, bits):
    """128 KiB tiles, the widest that a CU's LDS holds, against 32 KiB ones."""
    from tensorcircuit_amd import _lib, engine

    kinds = (_lib.G_RX, _lib.G_RZ, _lib.G_RY, _lib.G_RZZ)
    specs = [engine.GateSpec(kinds[g % 4], (g % n, (g + 3) % n)[: 2 if g % 4 == 3 else 1], g, 0.0, 1.0, None)
             for g in range(6 * n)]
    ham = engine.PauliSum(n, [[3, 3] + [0] * (n - 2), [0] * (n - 1) + [1]], [0.7, 1.1])
    p = torch.randn(2, len(specs), dtype=torch.float32 if dtype == "complex64" else torch.float64, device=gpu)
    (e, g), (e2, g2) = (engine.Program(n, specs, len(specs), fuse=1, adj_tile_bits=b).energy_grad(p, ham, 2, dtype)
                        for b in (bits, 11))
    # 6 n gates on states of norm one, each rounded a few times per amplitude
    unit = 2.0**-24 if dtype == "complex64" else 2.0**-53
    assert float((e - e2).abs().max()) <= 16 * len(specs) * unit and float((g - g2).abs().max()) <= 16 * len(specs) * unit


def test_sums_of_many_states(gpu):
    """2^26 inner products and energies of one-qubit states: a wave each."""
    from tensorcircuit_amd import engine

    B = (1 << 26) + 3
    st = torch.zeros(B, 2, dtype=torch.complex64, device=gpu)
    st[:, 1] = 1.0
    st[-1, 1] = 3.0
    got = engine.inner(st, st, 1).real
    assert bool((got[:-1] == 1.0).all()) and float(got[-1]) == 9.0
    del got
    e = engine.PauliSum(1, [[3], [1]], [2.0, 1.0], jit=0).expect(st).real
    assert bool((e[:-1] == -2.0).all()) and float(e[-1]) == -18.0
