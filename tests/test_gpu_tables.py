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


def _long_runs(n):
    """Runs that overflow one staged chunk or one staged op: 45 merged
    diagonals (27 trainable) on four qubits, 40 rotations of one qubit,
    every CX order, and permutation gates before, between and after them."""
    ops = []
    for i in range(27):
        ops.append(("rz" if i % 3 else "rzz", (i % 4,) if i % 3 else (i % 4, (i + 1) % 4), 0.1 + 0.05 * i))
    ops += [("cz", (0, 1), 0.0), ("s", (2,), 0.0), ("t", (3,), 0.0)] * 6
    ops += [(("ry", "rx")[i % 2], (i % 2,), 0.3 - 0.02 * i) for i in range(40)]
    ops += [("cnot", (a, b), 0.0) for a in range(4) for b in range(4) if a != b]
    ops += [("ry", (q,), 0.2 * (q + 1)) for q in range(n)]
    ops += [("swap", (0, n - 1), 0.0), ("x", (1,), 0.0), ("cnot", (n - 1, 0), 0.0), ("swap", (3, 1), 0.0)]
    return ops


# states smaller than a wave of threads, one tile, a tile and more; few gates
# and enough to fill several chunks of staged tables
@pytest.mark.parametrize("n,gates", [(4, 12), (4, 0), (5, 30), (7, 60), (9, 25), (10, 0), (11, 90), (12, 400), (13, 0),
                                     (14, 120), (18, 26)])
def test_tile_pass(gpu, n, gates):
    import tensorcircuit_amd as tc
    from tensorcircuit_amd import engine
    from test_gpu_jit import _circuit, _random_ops, _terms

    rng = np.random.default_rng(31 * n + gates)
    ops = _random_ops(rng, n, gates) if gates else _long_runs(n)
    c, oops = _circuit(tc, n, ops)
    specs, thetas = c._lower()
    terms = _terms(rng, n, 5)
    wsum = sum(abs(t[0]) for t in terms)
    ham = engine.PauliSum(n, [t[1] for t in terms], [t[0] for t in terms], jit=0)
    prog = engine.Program(n, specs, len(thetas), fuse=1, jit=0)
    B = 3
    params = np.array([float(np.real(t)) for t in thetas])[None, :] + rng.normal(0, 0.3, size=(B, len(thetas)))
    inputs = random_states(rng, B, n)
    for dt in DTYPES:
        name = str(dt).split(".")[1]
        p = torch.as_tensor(params).to(torch.float32 if dt == torch.complex64 else torch.float64).cuda()
        pd = np_of(p).astype(np.float64)
        # each gate turns a unit state with a few roundings
        tol = 8 * (len(ops) + 4) * UNIT[dt]
        st, _ = prog.forward(p, B, name)
        e, g = prog.energy_grad(p, ham, B, name)
        si = torch.as_tensor(inputs).to(dt).cuda()
        gs = torch.as_tensor(inputs[::-1].copy()).to(dt).cuda()
        out, _ = prog.forward(p, B, name, inputs=si)
        gp, gi = prog.vjp(p, None, out, gs, B, name, True)
        for b in range(B):
            assert np.abs(np_of(st)[b] - sv.run_ops(n, oops, pd[b])).max() <= tol
            e_ref, g_ref = sv.adjoint_value_and_grad(n, oops, pd[b], terms)
            assert abs(float(e[b]) - e_ref) <= 2 * tol * wsum
            assert np.abs(np_of(g)[b] - g_ref).max() <= 4 * tol * wsum
            # U^dagger of the output's cotangent, and of the output itself
            ref = sv.run_ops(n, oops, pd[b], inputs[b])
            assert np.abs(np_of(out)[b] - ref).max() <= 2 * tol
            lhs = np.vdot(np_of(gs)[b].astype(np.complex128), ref)
            rhs = np.vdot(np_of(gi)[b].astype(np.complex128), inputs[b])
            assert abs(lhs - rhs) <= 4 * tol
        assert torch.isfinite(gp).all()


def test_tile_pass_multi(gpu):
    """Programs of 3 (per-gate), 4, 7, 9, 12 and 13 qubits in shared launches
    against single runs, from |0..0> and from given states."""
    import tensorcircuit_amd as tc
    from tensorcircuit_amd import engine
    from test_gpu_jit import _circuit, _random_ops

    rng = np.random.default_rng(77)
    for dt in DTYPES:
        name = str(dt).split(".")[1]
        rdt = torch.float32 if dt == torch.complex64 else torch.float64
        items, ref = [], []
        start = []
        for n, B in ((3, 2), (4, 5), (7, 1), (9, 70), (12, 3), (13, 2)):
            ops = _random_ops(rng, n, 10 * n)
            c, oops = _circuit(tc, n, ops)
            specs, thetas = c._lower()
            prog = engine.Program(n, specs, len(thetas), fuse=1, jit=0)
            p = torch.as_tensor(rng.uniform(0, 6, size=(B, len(thetas)))).to(rdt).cuda()
            start.append(torch.as_tensor(random_states(rng, B, n)).to(dt).cuda())
            items.append((prog, p, torch.empty(B, 1 << n, dtype=dt, device="cuda")))
        for zero in (True, False):
            if not zero:
                for it, s in zip(items, start):
                    it[2].copy_(s)
            engine.forward_multi(items, name, init_zero=zero)
            for (prog, p, st), s in zip(items, start):
                one, _ = prog.forward(p, p.shape[0], name, inputs=None if zero else s)
                assert torch.equal(st, one)


# rows of no entry, one, a few and many (a group of lanes per row from 1 to
# 64); Hermitian or not
@pytest.mark.parametrize("n,mean,hermitian", [(1, 1, True), (3, 2, False), (6, 0.3, False), (7, 30, True),
                                              (9, 5, False), (9, 200, False), (11, 12, True)])
def test_csr(gpu, n, mean, hermitian):
    from tensorcircuit_amd import engine

    rng = np.random.default_rng(int(100 * n + mean))
    N = 1 << n
    m = (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))) * (rng.random((N, N)) < mean / N)
    m[N // 2] = 0
    if N > 2:
        m[1] = rng.standard_normal(N)  # a full row
    if hermitian:
        m = m + m.conj().T
    x = random_states(rng, 3, n)
    g = rng.standard_normal(3) + 1j * rng.standard_normal(3)
    for dt in DTYPES:
        c = engine.CsrMatrix(torch.as_tensor(m).to(dt).cuda().to_sparse_csr(), n, dt)
        assert c.hermitian == hermitian
        xd, gd = torch.as_tensor(x).to(dt).cuda(), torch.as_tensor(g).to(dt).cuda()
        mr, xr, gr = (np_of(torch.as_tensor(v).to(dt)).astype(np.complex128) for v in (m, x, g))
        # sums in fp64; the result is rounded once
        tol = 4 * UNIT[dt] * np.abs(mr).sum(axis=1).max()
        ax, dx = xr @ mr.T, xr @ mr.conj()
        assert np.abs(np_of(c.matvec(xd)) - ax).max() <= tol
        assert np.abs(np_of(c.matvec(xd, dagger=True)) - dx).max() <= tol
        ref = gr.conj()[:, None] * ax + gr[:, None] * dx
        assert np.abs(np_of(c.vjp(xd, gd)) - ref).max() <= 8 * tol
        # a lazily conjugated cotangent
        assert np.abs(np_of(c.vjp(xd, torch.conj(gd))) - (gr[:, None] * ax + gr.conj()[:, None] * dx)).max() <= 8 * tol
        for b in range(3):
            assert abs(complex(c.expect(xd[b])) - np.vdot(xr[b], ax[b])) <= max(tol, 1e-12) * np.sqrt(N)


# one stretch, several, one chunk, 16 chunks (one search level), more than
# 4096 chunks (two tiles of the scan); sparse weights, and draws at both ends
@pytest.mark.parametrize("n,shots", [(1, 5), (3, 40), (6, 17), (8, 100), (10, 1), (11, 333), (14, 2000), (15, 64),
                                     (23, 500)])
def test_sample_levels(gpu, n, shots):
    from tensorcircuit_amd import engine

    rng = np.random.default_rng(500 + n)
    N = 1 << n
    for dt in (torch.float32, torch.float64):
        p = torch.as_tensor(rng.random((2, N)) * (rng.random((2, N)) < (0.3 if n > 3 else 1.0))).to(dt)
        p[:, 0] = 0.0
        p[:, -1] = 0.0
        u = rng.random((2, shots))
        u[0, 0] = 0.0  # r = total
        got = engine.sample_prob_indices(p.cuda(), n, torch.as_tensor(u)).cpu().numpy()
        pd = p.to(torch.float64).numpy()
        for b in range(2):
            cdf = np.cumsum(pd[b])
            r = cdf[-1] * (1.0 - u[b])
            if cdf[-1] == 0:  # no weight (n = 1 here): the first index
                assert (got[b] == 0).all()
                continue
            assert (pd[b][got[b]] > 0).all()
            # the running sums agree to about N units in the last place
            slack = N * 2.0**-52 * cdf[-1]
            assert (cdf[got[b]] >= r - slack).all()
            assert (cdf[got[b]] - pd[b][got[b]] <= r + slack).all()


# (qubits, strings, letters): less than a wave, the last size with one
# amplitude per thread and the first with eight, one tile (2^11 or 2^12
# amplitudes) and several, the second chunk of 32 staged strings, flips that
# stay in the tile and flips that leave it
@pytest.mark.parametrize("n,T,letters", [(1, 4, 4), (2, 9, 4), (5, 32, 4), (6, 33, 4), (8, 40, 4), (9, 128, 4),
                                         (11, 33, 4), (12, 257, 4), (13, 90, "z"), (14, 131, "xz")])
def test_pauli_strings(gpu, n, T, letters):
    from tensorcircuit_amd import engine

    rng = np.random.default_rng(77 * n + T)
    alphabet = {4: [0, 1, 2, 3], "z": [0, 3], "xz": [0, 0, 0, 0, 0, 0, 1, 3]}[letters]
    codes = rng.choice(alphabet, size=(T, n)).astype(np.int8)
    w = rng.standard_normal(T)
    a = rng.standard_normal((3, T))
    a[:, rng.integers(0, T, T // 3)] = 0.0
    ham = engine.PauliSum(n, codes, w)
    s = random_states(rng, 3, n)
    for dt in DTYPES:
        st = torch.as_tensor(s).to(dt).cuda()
        sd = np_of(st).astype(np.complex128)
        e = np_of(ham.expect_terms(st))
        out = np_of(ham.apply_terms(st, torch.as_tensor(a).cuda()))
        for b in range(3):
            ref = np.zeros(2**n, dtype=np.complex128)
            for t in range(T):
                p = sv.pauli_sum_apply(sd[b], n, [(1.0, list(codes[t]))])
                # 2^n products summed in 64 bits; their magnitudes sum to 1
                assert abs(e[b, t] - w[t] * np.vdot(sd[b], p)) <= 1.01 * (2**n + 8) * 2.0**-53 * abs(w[t])
                ref += a[b, t] * w[t] * p
            # T products summed in 64 bits, then one rounding to the state's type
            tol = (2 * T + 8) * 2.0**-53 * np.abs(a[b] * w).sum() + 2 * UNIT[dt] * np.abs(ref).max()
            assert np.abs(out[b] - ref).max() <= tol


# (qubits, gates, batch, type of pass): partial sums of all passes side by
# side, one or many per gate, and (the last two: more than 64 MiB of them) of
# one pass at a time; also the per-gate kernels
@pytest.mark.parametrize("n,gates,batch,fuse", [(3, 20, 5, 1), (6, 90, 3, 1), (13, 60, 2, 1), (14, 70, 3, 0),
                                                (4, 310, 30000, 1), (3, 150, 60000, 0)])
def test_gradient_sums(gpu, n, gates, batch, fuse):
    from tensorcircuit_amd import _lib, engine

    rng = np.random.default_rng(gates + batch)
    specs, ops = [], []
    kinds = [("x", _lib.G_RX), ("y", _lib.G_RY), ("z", _lib.G_RZ)]
    for i in range(gates):
        name, kind = kinds[i % 3]
        q = int(rng.integers(n))
        # every third gate shares its parameter with the one before
        p = i - 1 if i % 3 == 2 else i
        specs.append(engine.GateSpec(kind, (q,), p, 0.0, 1.0, None))
        ops.append((name, q, p))
        if i % 7 == 0:
            cx = np.eye(4)[[0, 1, 3, 2]].astype(np.complex128)
            a, b = (int(x) for x in rng.choice(n, 2, replace=False))
            specs.append(engine.GateSpec(_lib.G_MAT, (a, b), -1, 0.0, 1.0, cx))
            ops.append(("cx", a, b))
    prog = engine.Program(n, specs, gates, fuse=fuse)
    codes, w = rng.integers(0, 4, size=(4, n)).astype(np.int8), rng.standard_normal(4)
    ham = engine.PauliSum(n, codes, w, jit=0)
    terms = [(float(w[k]), list(codes[k])) for k in range(4)]
    params = torch.as_tensor(rng.uniform(-2, 2, (batch, gates)))
    e, g = prog.energy_grad(params.cuda(), ham, batch, "complex128")
    e, g = np_of(e), np_of(g)
    pauli = {"x": np.array([[0, 1], [1, 0]]), "y": np.array([[0, -1j], [1j, 0]]), "z": np.diag([1, -1])}

    def turn(s, m, q):
        return np.einsum("ij,ajb->aib", m, s.reshape(2**q, 2, -1)).reshape(-1)

    for b in (0, batch // 2, batch - 1):
        th = params[b].numpy()
        s = np.zeros(2**n, dtype=np.complex128)
        s[0] = 1.0
        for name, q, p in ops:
            if name == "cx":
                idx = np.arange(2**n)
                s = s[np.where(idx >> (n - 1 - q) & 1, idx ^ (1 << (n - 1 - p)), idx)]
            else:
                s = turn(s, np.cos(th[p] / 2) * np.eye(2) - 1j * np.sin(th[p] / 2) * pauli[name], q)
        lam = sv.pauli_sum_apply(s, n, terms)
        ref_e, ref = np.vdot(s, lam).real, np.zeros(gates)
        for name, q, p in reversed(ops):
            if name == "cx":
                idx = np.arange(2**n)
                src = np.where(idx >> (n - 1 - q) & 1, idx ^ (1 << (n - 1 - p)), idx)
                s, lam = s[src], lam[src]
            else:
                ref[p] += np.imag(np.vdot(lam, turn(s, pauli[name], q)))
                m = np.cos(th[p] / 2) * np.eye(2) + 1j * np.sin(th[p] / 2) * pauli[name]
                s, lam = turn(s, m, q), turn(lam, m, q)
        # each gate is off by a few units of rounding of the state it acts on,
        # there and back, for state and adjoint (of norm <= sum |w|); two
        # gates at most share a parameter
        tol = 2 * (16 * gates + 2**n) * 2.0**-53 * np.abs(w).sum()
        assert abs(e[b] - ref_e) <= tol
        assert np.abs(g[b] - ref).max() <= tol


# compiled passes: merged diagonals of one, two and more qubits (rz, rzz,
# phase, T, CZ, alone and in runs) between rotations and CNOTs; widths of one
# tile, one tile exactly and several, where a pass's diagonals are over
# their first entries but for one
@pytest.mark.parametrize("n,gates", [(10, 3), (10, 40), (11, 80), (13, 120), (14, 200), (20, 90)])
def test_compiled_diagonals(gpu, n, gates):
    from tensorcircuit_amd import _lib, engine

    rng = np.random.default_rng(31 * n + gates)
    t = np.diag([1.0, np.exp(0.25j * np.pi)])
    cz, cx = np.diag([1.0, 1, 1, -1]).astype(np.complex128), np.eye(4)[[0, 1, 3, 2]].astype(np.complex128)
    pick = ["ry", "rz", "rz", "rzz", "phase", "t", "cz", "cx", "rx"]
    one = {"ry": _lib.G_RY, "rz": _lib.G_RZ, "phase": _lib.G_PHASE, "rx": _lib.G_RX}
    specs, p = [engine.GateSpec(_lib.G_RZ, (n - 1,), 0, 0.0, 1.0, None)], 1
    for _ in range(gates):
        name = pick[rng.integers(len(pick))]
        a, b = (int(x) for x in rng.choice(n, 2, replace=False))
        if name in one:
            specs.append(engine.GateSpec(one[name], (a,), p, 0.0, 1.0, None))
            p += 1
        elif name == "rzz":
            specs.append(engine.GateSpec(_lib.G_RZZ, (a, b), p, 0.0, 1.0, None))
            p += 1
        else:
            q = (a,) if name == "t" else (a, b)
            specs.append(engine.GateSpec(_lib.G_MAT, q, -1, 0.0, 1.0, {"t": t, "cz": cz, "cx": cx}[name]))
    codes, w = rng.integers(0, 4, size=(5, n)).astype(np.int8), rng.standard_normal(5)
    ham = engine.PauliSum(n, codes, w, jit=0)
    params = torch.as_tensor(rng.uniform(-4, 4, (2, p)))
    # one kernel per gate
    plain = engine.Program(n, specs, p, fuse=0)
    ref, _ = plain.forward(params.cuda(), 2, "complex128")
    re, rg = plain.energy_grad(params.cuda(), ham, 2, "complex128")
    prog = engine.Program(n, specs, p, fuse=1, jit=1)
    for dt, name in ((torch.complex64, "complex64"), (torch.complex128, "complex128")):
        th = params.cuda().to(torch.float32 if dt == torch.complex64 else torch.float64)
        if dt == torch.complex64:  # the angles as they were rounded
            ref, _ = plain.forward(th.double(), 2, "complex128")
            re, rg = plain.energy_grad(th.double(), ham, 2, "complex128")
        else:
            ref, _ = plain.forward(params.cuda(), 2, "complex128")
            re, rg = plain.energy_grad(params.cuda(), ham, 2, "complex128")
        psi, _ = prog.forward(th, 2, name)
        e, g = prog.energy_grad(th, ham, 2, name)
        # a gate moves a normalised state by a few units of rounding; there
        # and back for state and adjoint, whose norm is at most sum |w|
        tol = 4 * (4 + len(specs)) * UNIT[dt]
        assert np.abs(np_of(psi) - np_of(ref)).max() <= tol
        assert np.abs(np_of(e) - np_of(re)).max() <= 2 * tol * np.abs(w).sum()
        assert np.abs(np_of(g) - np_of(rg)).max() <= 4 * tol * np.abs(w).sum()


# rx and ry of compiled passes as shears: small angles, angles near pi and
# beyond, and middling ones, with and without diagonals
@pytest.mark.parametrize("n,gates,diag", [(10, 30, True), (10, 30, False), (13, 120, True), (15, 200, True)])
def test_compiled_rotations(gpu, n, gates, diag):
    from tensorcircuit_amd import _lib, engine

    rng = np.random.default_rng(5 * n + gates)
    cx = np.eye(4)[[0, 1, 3, 2]].astype(np.complex128)
    specs, p = [], 0
    for _ in range(gates):
        k = rng.integers(4 if diag else 3)
        a, b = (int(x) for x in rng.choice(n, 2, replace=False))
        if k == 2:
            specs.append(engine.GateSpec(_lib.G_MAT, (a, b), -1, 0.0, 1.0, cx))
            continue
        specs.append(engine.GateSpec([_lib.G_RX, _lib.G_RY, None, _lib.G_RZ][k], (a,), p, 0.0, 1.0, None))
        p += 1
    th = rng.normal(0, 0.2, (3, p))
    th[1, : p // 2] += 2 * np.pi  # cosines near -1
    th[1, p // 3] = 3.1
    th[2] = rng.uniform(1.2, 1.6, p)
    th = torch.as_tensor(th).cuda()
    ref, _ = engine.Program(n, specs, p, fuse=0).forward(th.float().double(), 3, "complex128")
    exact, _ = engine.Program(n, specs, p, fuse=0).forward(th, 3, "complex128")
    prog = engine.Program(n, specs, p, fuse=1, jit=1)
    # each gate moves a normalised state by a few units of rounding
    for name, x, want in (("complex64", th.float(), ref), ("complex128", th, exact)):
        psi, _ = prog.forward(x, 3, name)
        tol = 4 * (4 + len(specs)) * UNIT[psi.dtype]
        assert np.abs(np_of(psi) - np_of(want)).max() <= tol


# angles of a circuit as Python numbers and as tensors of other shapes, types
# and devices, and angles taken from rows of a larger tensor
def test_mixed_angles(gpu):
    import tensorcircuit_amd as tc
    from tensorcircuit_amd.templates import blocks

    x = [0.3, -0.7, 1.1, 0.4, -0.2, 0.9]

    def energy(a):
        c = tc.Circuit(3)
        for i in range(3):
            c.ry(i, theta=a[i])
            c.rx(i, theta=a[i + 3])
        c.cnot(0, 1)
        c.cnot(1, 2)
        return tc.backend.real(c.expectation_ps(z=[0, 2]))

    want = float(energy(x))
    mixed = [0.3, torch.tensor(-0.7, dtype=torch.float64), torch.tensor([1.1]).cuda(), torch.tensor(0.4 + 0.0j),
             torch.tensor([[-0.2]], dtype=torch.float64), torch.tensor(0.9).cuda()]
    same = [torch.tensor(v, dtype=torch.complex64) for v in x]
    for a in (mixed, same, [torch.tensor([v]) for v in x]):
        assert abs(float(energy(a)) - want) <= 32 * UNIT[torch.complex64]
    # rows: more of them, and longer, than the circuit has
    p = torch.as_tensor(np.random.default_rng(3).normal(size=(6, 5)), dtype=torch.float32).cuda().requires_grad_(True)

    def layers(f, q):
        c = tc.Circuit(4)
        f(c, q, 2)
        return tc.backend.real(c.expectation_ps(z=[1], x=[2]))

    e = layers(blocks.hea_layers, p)
    g = torch.autograd.grad(e, p)[0]
    cut = p.detach().cpu().numpy()[:4, :4]
    assert abs(float(e) - float(layers(blocks.hea_layers, cut))) <= 128 * UNIT[torch.complex64]
    q = torch.as_tensor(cut).cuda().requires_grad_(True)
    h = torch.autograd.grad(layers(blocks.example_block, q.reshape(-1)), q)[0]
    assert h.shape == q.shape and torch.isfinite(h).all()
    assert g[:4, :4].abs().sum() > 0 and g[4:].abs().sum() == 0 and g[:, 4].abs().sum() == 0


# the first pass reads given inputs itself: table-driven, compiled and
# matrix-core passes, and the copy before per-gate kernels, circuits without
# gates and inputs off a 16-byte boundary; against the same passes in place
@pytest.mark.parametrize("n,opts", [(3, {}), (6, {}), (13, {}), (13, {"jit": 1}), (14, {"jit": 1, "ckpt_every": 1}),
                                    (5, {"fuse": 0}), (12, {"mfma": 2}), (15, {"mfma": 2}), (4, {"empty": 1})])
def test_forward_inputs(gpu, n, opts):
    from tensorcircuit_amd import _lib, engine, fusion, workloads

    rng = np.random.default_rng(n)
    opts = {"fuse": 1, **opts}
    if opts.get("mfma"):
        prog, p = engine.Program(n, fusion.fuse(workloads.brickwork(n, 4, seed=2), n), 0, **opts), 0
    else:
        specs, p = [], 0
        for i in range(0 if opts.pop("empty", 0) else 4 * n):
            specs.append(engine.GateSpec((_lib.G_RX, _lib.G_RY, _lib.G_RZ)[i % 3], (i % n,), p, 0.0, 1.0, None))
            p += 1
            if i % n == n - 1:
                specs.append(engine.barrier())
        prog = engine.Program(n, specs, p, **opts)
    for dt in DTYPES[:1] if opts.get("mfma") else DTYPES:
        name = {torch.complex64: "complex64", torch.complex128: "complex128"}[dt]
        th = torch.as_tensor(rng.normal(size=(3, p))).cuda() if p else None
        flat = torch.as_tensor(rng.standard_normal(3 * 2**n + 1) + 1j * rng.standard_normal(3 * 2**n + 1)).to(dt).cuda()
        for x in (flat[:-1], flat[1:], torch.conj(flat[:-1])):
            x = x.reshape(3, 2**n)
            before = x.clone()
            want, wck = prog.forward(th, 3, name, inputs=x, want_ckpts=True, out=torch.empty_like(before))
            got, ck = prog.forward(th, 3, name, inputs=x, want_ckpts=True)
            assert torch.equal(got, want) and torch.equal(ck, wck) and torch.equal(x, before)
            assert got.data_ptr() != x.data_ptr()


# Pauli sums whose 14-bit tiles would take fewer passes (XX on every pair of
# qubits), at the qubit counts that keep 12-bit tiles, and with a string that
# only a 14-bit tile holds; the entry point with a fixed scratch accepts the
# batches that 14-bit tiles allow, in parts
@pytest.mark.parametrize("n,wide", [(14, False), (15, False), (17, True), (15, True)])
def test_pauli_tile_widths(gpu, n, wide):
    import ctypes

    from tensorcircuit_amd import _lib, engine

    rng = np.random.default_rng(n + wide)
    pairs = [(i, j) for i in range(n) for j in range(i)]
    T = len(pairs) + 2
    codes = np.zeros((T, n), dtype=np.int8)
    for t, (i, j) in enumerate(pairs):
        codes[t, i] = codes[t, j] = 1 + t % 2
    codes[T - 2, 1:3] = 3
    codes[T - 1, : 9 if wide else 1] = 1  # 9 flips above the 4 low bits, or 1
    w = rng.standard_normal(T)
    terms = [(float(w[t]), list(codes[t])) for t in range(T)]
    ham = engine.PauliSum(n, codes, w, jit=0)
    s = random_states(rng, 2, n)
    for dt in DTYPES:
        st = torch.as_tensor(s).to(dt).cuda()
        sd = np_of(st).astype(np.complex128)
        # T weights summed, then one product and sum per flip group (<= T)
        tol = (2 * T + 8) * UNIT[dt] * np.abs(w).sum()
        e, h = np_of(ham.expect(st)), np_of(ham.apply(st))
        for b in range(2):
            assert abs(e[b] - sv.pauli_sum_expectation(sd[b], n, terms)) <= tol
            assert np.abs(h[b] - sv.pauli_sum_apply(sd[b], n, terms)).max() <= 2 * tol
    if n == 15 and not wide:
        nb = ctypes.c_int64()
        _lib.lib.tcm_pauli_workspace_bytes(ham.handle, _lib.TCM_C64, 1000, ctypes.byref(nb))
        batch = 3 * (8 << 20) // (2 * (nb.value // 1000))  # half as much again as the scratch holds
        st = torch.as_tensor(s[:1]).to(torch.complex64).cuda().expand(batch, -1).contiguous()
        out = torch.empty(batch, 2, dtype=torch.float64, device="cuda")
        want = np_of(ham.expect(st[:1]))[0]
        _lib.check(_lib.lib.tcm_expect_pauli_sum_noalloc(ham.handle, _lib.TCM_C64, st.data_ptr(), batch, out.data_ptr(),
                                                         engine._stream()), "tcm_expect_pauli_sum_noalloc")
        assert (np_of(out)[:, 0] == want.real).all()


# lambda less E psi in the first reverse pass: one partial sum of the energy,
# many, and more than the pass sums itself; gates that are not unitary and
# given inputs keep lambda as it is.  A constant added to the Hamiltonian
# (identity string) makes E large beside the gradients.
@pytest.mark.parametrize("n,dtype,keep", [(6, "complex64", ""), (12, "complex64", ""), (15, "complex128", ""),
                                          (18, "complex64", "inputs"), (8, "complex128", "gate"),
                                          (19, "complex128", "")])
def test_energy_shift(gpu, n, dtype, keep):
    from tensorcircuit_amd import _lib, engine

    rng = np.random.default_rng(n)
    specs, p = [], 0
    for i in range(2 * n):
        specs.append(engine.GateSpec((_lib.G_RY, _lib.G_RZ, _lib.G_RX)[i % 3], (i % n,), p, 0.0, 1.0, None))
        p += 1
        if i % n == n - 1:
            for q in range(n - 1):
                specs.append(engine.GateSpec(_lib.G_MAT, (q, q + 1), -1, 0.0, 1.0,
                                             np.eye(4)[[0, 1, 3, 2]].astype(np.complex128)))
    if keep == "gate":
        specs.insert(3, engine.GateSpec(_lib.G_MAT, (1,), -1, 0.0, 1.0, np.diag([1.0, 0.9]).astype(np.complex128)))
    codes = np.zeros((n + 1, n), dtype=np.int8)
    codes[np.arange(n), np.arange(n)] = 1 + np.arange(n) % 3
    w = np.append(rng.standard_normal(n), 50.0)
    th = torch.as_tensor(rng.normal(0, 0.3, (2, p))).cuda()
    prog = engine.Program(n, specs, p, fuse=1, jit=0)
    args = {}
    if keep == "inputs":
        args["inputs"] = torch.as_tensor(random_states(rng, 2, n)).cuda()
    x = th if dtype == "complex128" else th.float()
    with_one = engine.PauliSum(n, codes, w, jit=0)
    without = engine.PauliSum(n, codes[:n], w[:n], jit=0)
    kw = {k: v.to(torch.complex64 if dtype == "complex64" else torch.complex128) for k, v in args.items()}
    e1, g1 = prog.energy_grad(x, with_one, 2, dtype, **kw)
    # the gradient of the constant is zero: <psi|psi> does not depend on the
    # angles of unitary gates; per-gate kernels in 64 bits as the reference
    ref = engine.Program(n, specs, p, fuse=0)
    h = without if keep != "gate" else with_one
    e0, g0 = ref.energy_grad(x.double(), h, 2, "complex128",
                             **{k: v.to(torch.complex128) for k, v in kw.items()})
    u = 2.0**-24 if dtype == "complex64" else 2.0**-53
    # roundings of each gate on psi and lambda (of norm <= sum |w|), there and back
    tol = 4 * (len(specs) + 4) * u * np.abs(w).sum()
    assert np.abs(np_of(g1) - np_of(g0)).max() <= tol
    shift = 50.0 if keep != "gate" else 0.0
    assert np.abs(np_of(e1) - np_of(e0) - shift).max() <= tol
