"""Performance cases: the work that programs built on this package do, through
its public entry points, from single small circuits to states that fill
gigabytes.

A case is a dict of plain values with a ``kind``:

* ``energy_grad`` -- one step of a variational optimiser: energies and
  parameter gradients of a batch of parameter sets (``Program.energy_grad``).
* ``forward``     -- simulation of one large circuit: final state and energy.
* ``uneven``      -- circuits of different qubit counts run together
  (``forward_multi``), states and energies.
* ``blocks``      -- a deep circuit of fixed gates, fused into dense 5-qubit
  blocks, applied to an input state.
* ``circuit``     -- the drop-in API: a ``Circuit`` rebuilt on each call under
  ``backend.value_and_grad``, as a TensorCircuit training loop does.
* ``hamiltonian`` -- a many-term Pauli sum on given states: energies and
  H|psi> (Lanczos, variance, imaginary time).
* ``terms``       -- every Pauli string of a list by itself, and the weighted
  application that is its backward (shadow tomography, QAOA statistics).
* ``sparse``      -- expectation of a sparse matrix and its gradient in the
  state.
* ``sample``      -- measurement shots of a given state.

Angles are those of a variational run after its start: normal around zero.
States are random product states with some noise, normalised.
"""
import functools
import math

import numpy as np
import torch

import tensorcircuit_amd as tc
from tensorcircuit_amd import _lib, engine, fusion, quantum, workloads
from tensorcircuit_amd.templates import blocks, measurements

DEV = "cuda"
CDT = {"complex64": torch.complex64, "complex128": torch.complex128}
RDT = {"complex64": torch.float32, "complex128": torch.float64}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # one call of a small variational eigensolver: launches and latency
        {"name": "energy_grad 12q", "kind": "energy_grad", "ansatz": "hea", "n": 12, "layers": 4, "batch": 1,
         "dtype": "complex64", "ckpt": 0},
        # a population of parameter sets of a mid-size circuit, an odd width
        {"name": "energy_grad 17q x33", "kind": "energy_grad", "ansatz": "hea", "n": 17, "layers": 8, "batch": 33,
         "dtype": "complex64", "ckpt": 0},
        # double precision, and the ring of ZZ couplings of a QAOA circuit
        {"name": "energy_grad 18q x3 c128", "kind": "energy_grad", "ansatz": "qaoa", "n": 18, "layers": 6, "batch": 3,
         "dtype": "complex128", "ckpt": 0},
        # the benchmark's circuit (24 qubits, 20 layers, checkpoints)
        {"name": "energy_grad 24q x4", "kind": "energy_grad", "ansatz": "hea", "n": 24, "layers": 20, "batch": 4,
         "dtype": "complex64", "ckpt": 5},
        # the benchmark's single large state
        {"name": "forward 26q", "kind": "forward", "ansatz": "hea", "n": 26, "layers": 10, "dtype": "complex64"},
        # circuits of 10 to 18 qubits side by side
        {"name": "uneven 10..18q", "kind": "uneven", "ansatz": "hea", "lo": 10, "hi": 18, "layers": 6, "batch": 21,
         "dtype": "complex64"},
        # a random circuit in dense blocks on the matrix cores
        {"name": "blocks 26q", "kind": "blocks", "n": 26, "depth": 20},
        # a training loop written against the Circuit API
        {"name": "circuit 10q", "kind": "circuit", "n": 10, "layers": 3},
        # a fermionic Hamiltonian (hopping strings) on a few states
        {"name": "hamiltonian 18q 200t", "kind": "hamiltonian", "n": 18, "terms": 200, "batch": 4,
         "dtype": "complex64"},
        # 59 separate strings of a 20-qubit state
        {"name": "terms 20q 59t", "kind": "terms", "n": 20, "terms": 59, "batch": 1, "dtype": "complex64"},
        # a transverse-field Ising matrix in sparse form
        {"name": "sparse 18q", "kind": "sparse", "n": 18, "dtype": "complex64"},
        # shots of a 24-qubit state
        {"name": "sample 24q", "kind": "sample", "n": 24, "shots": 100003, "dtype": "complex64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["energy_grad", "energy_grad", "forward", "uneven", "blocks", "circuit", "hamiltonian",
                       "terms", "sparse", "sample"])
    dtype = "complex128" if rng.random() < 0.3 else "complex64"
    c = {"kind": kind}
    if kind == "energy_grad":
        n = rng.randint(4, 22 if dtype == "complex64" else 20)
        layers = rng.randint(1, 10)
        # the batch of the largest listed case holds 2^26 amplitudes
        most = max(1, min(1024, (1 << (25 if dtype == "complex64" else 23)) >> n))
        c.update(ansatz=rng.choice(["hea", "qaoa"]), n=n, layers=layers, batch=_log_int(rng, 1, most), dtype=dtype,
                 ckpt=rng.choice([0, 0, 3]))
    elif kind == "forward":
        c.update(ansatz=rng.choice(["hea", "qaoa"]), n=rng.randint(6, 25), layers=rng.randint(1, 8), dtype=dtype)
    elif kind == "uneven":
        lo = rng.randint(8, 13)
        c.update(ansatz=rng.choice(["hea", "qaoa"]), lo=lo, hi=lo + rng.randint(1, 5), layers=rng.randint(2, 8),
                 batch=rng.randint(2, 40), dtype=dtype)
    elif kind == "blocks":
        c.update(n=rng.randint(14, 26), depth=rng.randint(4, 19))
    elif kind == "circuit":
        c.update(n=rng.randint(4, 18), layers=rng.randint(1, 4))
    elif kind == "hamiltonian":
        c.update(n=rng.randint(6, 19), terms=_log_int(rng, 10, 400), batch=rng.randint(1, 6), dtype=dtype)
    elif kind == "terms":
        c.update(n=rng.randint(6, 21), terms=_log_int(rng, 4, 120), batch=rng.randint(1, 4), dtype=dtype)
    elif kind == "sparse":
        c.update(n=rng.randint(6, 20), dtype=dtype)
    else:
        c.update(n=rng.randint(6, 25), shots=_log_int(rng, 50, 1 << 19), dtype=dtype)
    return c


# ---------------------------------------------------------------------------
# circuits, as (rotation factors and parameter slots) gate lists
# ---------------------------------------------------------------------------


@functools.lru_cache(maxsize=64)
def _ansatz(kind, n, layers):
    """(gates, number of parameters); gates: ("rot", pauli, qubits, slot) =
    exp(-i theta/2 P), ("cnot", a, b), ("h", q), ("barrier",)."""
    gates, p = [], 0
    if kind == "qaoa":
        gates += [("h", q) for q in range(n)]
    for _ in range(layers):
        if kind == "hea":
            for pauli in ("y", "z"):
                for q in range(n):
                    gates.append(("rot", pauli, (q,), p))
                    p += 1
            gates += [("cnot", q, q + 1) for q in range(n - 1)]
        else:
            for q in range(n if n > 2 else 1):
                gates.append(("rot", "zz", (q, (q + 1) % n), p))
                p += 1
            for q in range(n):
                gates.append(("rot", "x", (q,), p))
                p += 1
        gates.append(("barrier",))
    return gates, p


_KIND = {"x": _lib.G_RX, "y": _lib.G_RY, "z": _lib.G_RZ, "zz": _lib.G_RZZ}
_H = np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2.0)
_CNOT = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]], dtype=np.complex128)


@functools.lru_cache(maxsize=64)
def _program(kind, n, layers, ckpt):
    gates, p = _ansatz(kind, n, layers)
    specs = []
    for g in gates:
        if g[0] == "rot":
            specs.append(engine.GateSpec(_KIND[g[1]], g[2], g[3], 0.0, 1.0, None))
        elif g[0] == "cnot":
            specs.append(engine.GateSpec(_lib.G_MAT, (g[1], g[2]), -1, 0.0, 1.0, _CNOT))
        elif g[0] == "h":
            specs.append(engine.GateSpec(_lib.G_MAT, (g[1],), -1, 0.0, 1.0, _H))
        else:
            specs.append(engine.barrier())
    return engine.get_program(n, specs, p, fuse=1, ckpt_every=ckpt)


@functools.lru_cache(maxsize=64)
def _tfim(n):
    codes, w = workloads.tfim_terms(n)
    return engine.get_pauli(n, codes, w)


@functools.lru_cache(maxsize=64)
def _strings(n, terms):
    """Pauli codes and weights of a lattice-fermion kind of Hamiltonian:
    densities (Z, ZZ) and Jordan-Wigner hoppings (X Z..Z X and Y Z..Z Y)."""
    rng = np.random.default_rng(1000 * n + terms)
    codes = np.zeros((terms, n), dtype=np.int8)
    for t in range(terms):
        a, b = sorted(rng.choice(n, size=2, replace=False))
        if t % 4 == 0:
            codes[t, a] = 3
        elif t % 4 == 1:
            codes[t, a] = codes[t, b] = 3
        else:
            codes[t, a:b + 1] = 3
            codes[t, a] = codes[t, b] = 1 if t % 4 == 2 else 2
    return codes, rng.normal(size=terms)


@functools.lru_cache(maxsize=64)
def _many(n, terms):
    return engine.get_pauli(n, *_strings(n, terms))


@functools.lru_cache(maxsize=16)
def _csr(n, dtype):
    codes, w = workloads.tfim_terms(n)
    with tc.runtime_dtype(dtype):
        return engine.CsrMatrix(quantum.PauliStringSum2COO(codes, w), n, CDT[dtype])


@functools.lru_cache(maxsize=16)
def _blocks(n, depth):
    specs = workloads.brickwork(n, depth, seed=7)
    return engine.Program(n, fusion.fuse(specs, n), 0, fuse=1, mfma=2)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _angles(g, shape, dtype):
    return 0.2 * torch.randn(shape, generator=g, device=DEV, dtype=torch.float64).to(RDT[dtype])


def _states(g, batch, n, dtype):
    """Random product states with a tenth of their weight in noise."""
    ang = math.pi * torch.rand((batch, n, 2), generator=g, device=DEV, dtype=torch.float64)
    psi = torch.ones((batch, 1), dtype=CDT[dtype], device=DEV)
    for q in range(n):
        one = torch.polar(torch.sin(0.5 * ang[:, q, 0]), 2.0 * ang[:, q, 1])
        pair = torch.stack([torch.cos(0.5 * ang[:, q, 0]).to(one.dtype), one], dim=1).to(CDT[dtype])
        psi = (psi.view(batch, -1, 1) * pair.view(batch, 1, 2)).view(batch, -1)
    noise = torch.randn((batch, 1 << n, 2), generator=g, device=DEV, dtype=RDT[dtype])
    psi = psi + math.sqrt(0.1 / (2 << n)) * torch.view_as_complex(noise)
    return psi / torch.linalg.vector_norm(psi, dim=1, keepdim=True)


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = {"kind": kind, "case": case}
    if kind in ("energy_grad", "forward"):
        p = _ansatz(case["ansatz"], case["n"], case["layers"])[1]
        s["params"] = _angles(g, (case.get("batch", 1), p), case["dtype"])
        s["prog"] = _program(case["ansatz"], case["n"], case["layers"], case.get("ckpt", 0))
        s["ham"] = _tfim(case["n"])
    elif kind == "uneven":
        s["items"], s["hams"] = [], []
        for n in range(case["lo"], case["hi"] + 1):
            prog = _program(case["ansatz"], n, case["layers"], 0)
            params = _angles(g, (case["batch"], prog.nparams), case["dtype"])
            s["items"].append((prog, params, torch.empty(case["batch"], 1 << n, dtype=CDT[case["dtype"]], device=DEV)))
            s["hams"].append(_tfim(n))
    elif kind == "blocks":
        s["prog"] = _blocks(case["n"], case["depth"])
        s["psi"] = _states(g, 1, case["n"], "complex64")
    elif kind == "circuit":
        n, layers = case["n"], case["layers"]
        codes, w = workloads.tfim_terms(n)

        def energy(param):
            c = tc.Circuit(n)
            blocks.example_block(c, param, layers)
            return tc.backend.real(measurements.pauli_sum_expectation(c, codes, w))

        s["vag"] = tc.backend.value_and_grad(energy)
        s["params"] = _angles(g, (2 * layers, n), "complex64")
    elif kind in ("hamiltonian", "terms"):
        s["psi"] = _states(g, case["batch"], case["n"], case["dtype"])
        s["ham"] = _many(case["n"], case["terms"])
        if kind == "terms":
            s["weights"] = torch.randn((case["batch"], case["terms"]), generator=g, device=DEV, dtype=torch.float64)
    elif kind == "sparse":
        s["psi"] = _states(g, 1, case["n"], case["dtype"]).reshape(-1).requires_grad_(True)
        s["h"] = _csr(case["n"], case["dtype"])
    else:
        s["psi"] = _states(g, 1, case["n"], case["dtype"]).reshape(-1)
        s["uniforms"] = torch.rand(case["shots"], generator=g, device=DEV, dtype=torch.float64)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "energy_grad":
        e, grad = s["prog"].energy_grad(s["params"], s["ham"], case["batch"], case["dtype"])
        # the optimiser's tensors have the type of the angles
        return e.to(s["params"].dtype), grad.to(s["params"].dtype)
    if kind == "forward":
        psi, _ = s["prog"].forward(s["params"], 1, case["dtype"])
        return psi, s["ham"].expect(psi).to(psi.dtype)
    if kind == "uneven":
        engine.forward_multi(s["items"], case["dtype"])
        return [(psi, h.expect(psi).to(psi.dtype)) for (_, _, psi), h in zip(s["items"], s["hams"])]
    if kind == "blocks":
        return s["prog"].forward(None, 1, "complex64", inputs=s["psi"])[0]
    if kind == "circuit":
        return s["vag"](s["params"])
    if kind == "hamiltonian":
        return s["ham"].expect(s["psi"]).to(s["psi"].dtype), s["ham"].apply(s["psi"])
    if kind == "terms":
        return s["ham"].expect_terms(s["psi"]).to(s["psi"].dtype), s["ham"].apply_terms(s["psi"], s["weights"])
    if kind == "sparse":
        e = torch.real(engine.csr_expectation(s["h"], s["psi"], case["n"]))
        return e.detach(), torch.autograd.grad(e, s["psi"])[0]
    return quantum.measurement_counts(s["psi"], case["shots"], format="sample_int", status=s["uniforms"])


def work(case):
    """Bytes: inputs and outputs once (a state that only exists inside a pass
    counts nothing).  Flops: 6 per amplitude and rotation (a real rotation of
    a pair as three multiply-adds on each component), for the state, and in a
    reverse sweep for state and adjoint, with 4 for the gradient."""
    kind = case["kind"]
    amp = 8 if case.get("dtype", "complex64") == "complex64" else 16
    if kind in ("energy_grad", "forward"):
        p, b = _ansatz(case["ansatz"], case["n"], case["layers"])[1], case.get("batch", 1)
        state = float(b << case["n"])
        if kind == "energy_grad":
            return {"bytes": amp * p * b, "flops": state * p * (6 * 3 + 4)}
        return {"bytes": amp * state, "flops": state * p * 6}
    if kind == "uneven":
        nb = fl = 0.0
        for n in range(case["lo"], case["hi"] + 1):
            nb += amp * float(case["batch"] << n)
            fl += 6.0 * (case["batch"] << n) * _ansatz(case["ansatz"], n, case["layers"])[1]
        return {"bytes": nb, "flops": fl}
    if kind == "blocks":
        # a one-qubit matrix costs 14 flops an amplitude
        return {"bytes": 16.0 * (1 << case["n"]), "flops": 14.0 * case["n"] * case["depth"] * (1 << case["n"])}
    if kind == "circuit":
        n, p = case["n"], 2 * case["layers"] * case["n"]
        return {"bytes": 8.0 * p, "flops": float(1 << n) * p * (6 * 3 + 4)}
    if kind in ("hamiltonian", "terms"):
        state = float(case["batch"] << case["n"])
        return {"bytes": 2 * amp * state, "flops": 8.0 * case["terms"] * state}
    if kind == "sparse":
        nnz = float((case["n"] + 1) << case["n"])
        return {"bytes": (8 + amp) * nnz + (8 + 2 * amp) * (1 << case["n"]), "flops": 8.0 * nnz}
    return {"bytes": amp * float(1 << case["n"]) + 16.0 * case["shots"], "flops": 4.0 * (1 << case["n"])}


# ---------------------------------------------------------------------------
# the same values in 64 bits by plain torch
# ---------------------------------------------------------------------------


def _split(psi, n, q):
    return psi.view(psi.shape[0], 1 << q, 2, 1 << (n - 1 - q))


def _pauli1(psi, n, pauli, q):
    v = _split(psi, n, q)
    if pauli == "z":
        ph = torch.tensor([1.0, -1.0], dtype=torch.complex128, device=psi.device).view(1, 1, 2, 1)
        return (v * ph).reshape(psi.shape)
    v = v.flip(2)
    if pauli == "y":
        v = v * torch.tensor([-1j, 1j], dtype=torch.complex128, device=psi.device).view(1, 1, 2, 1)
    return v.reshape(psi.shape)


def _pauli(psi, n, paulis, qubits):
    for a, q in zip(paulis, qubits):
        psi = _pauli1(psi, n, a, q)
    return psi


def _rotate(psi, n, pauli, qubits, half):
    """exp(-i half P) psi, half [batch, 1]."""
    c, s = torch.cos(half).view(-1, 1, 1, 1), torch.sin(half).view(-1, 1, 1, 1)
    if pauli in ("z", "zz"):
        sign = torch.tensor([1.0, -1.0], dtype=torch.float64, device=psi.device)
        if pauli == "z":
            return (_split(psi, n, qubits[0]) * (c - 1j * s * sign.view(1, 1, 2, 1))).view(psi.shape)
        a, b = sorted(qubits)
        v = psi.view(psi.shape[0], 1 << a, 2, 1 << (b - a - 1), 2, 1 << (n - 1 - b))
        zz = sign.view(1, 1, 2, 1, 1, 1) * sign.view(1, 1, 1, 1, 2, 1)
        return (v * (c - 1j * s * zz.view(1, 2, 1, 2)).view(-1, 1, 2, 1, 2, 1)).view(psi.shape)
    coef = torch.tensor([-1j, -1j] if pauli == "x" else [-1.0, 1.0], dtype=torch.complex128, device=psi.device)
    v = _split(psi, n, qubits[0])
    return torch.addcmul(v * c, v.flip(2), s * coef.view(1, 1, 2, 1)).view(psi.shape)


def _undo_or_do(psi, n, g, params, sign):
    if g[0] == "rot":
        return _rotate(psi, n, g[1], g[2], (0.5 * sign) * params[:, g[3]].view(-1, 1))
    if g[0] == "cnot":
        v = _split(psi, n, g[1]).clone()
        v = v.view(psi.shape[0], 1 << g[1], 2, 1 << (g[2] - g[1] - 1), 2, 1 << (n - 1 - g[2]))
        v[:, :, 1] = v[:, :, 1].flip(3)
        return v.view(psi.shape)
    if g[0] == "h":
        v = _split(psi, n, g[1])
        s = math.sqrt(0.5)
        return torch.stack([s * (v[:, :, 0] + v[:, :, 1]), s * (v[:, :, 0] - v[:, :, 1])], dim=2).reshape(psi.shape)
    return psi


def _string(psi, n, codes):
    paulis = [("", "x", "y", "z")[int(c)] for c in codes]
    return _pauli(psi, n, [a for a in paulis if a], [q for q, a in enumerate(paulis) if a])


def _apply_sum(psi, n, codes, w):
    out = torch.zeros_like(psi)
    for c, x in zip(codes, w):
        out += float(x) * _string(psi, n, c)
    return out


def _inner(a, b):
    return torch.sum(torch.conj(a) * b, dim=1)


def _zero(b, n):
    psi = torch.zeros(b, 1 << n, dtype=torch.complex128, device=DEV)
    psi[:, 0] = 1
    return psi


def _forward(gates, n, params):
    psi = _zero(params.shape[0], n)
    for g in gates:
        psi = _undo_or_do(psi, n, g, params, 1.0)
    return psi


def _energy_grad(gates, n, params):
    psi = _forward(gates, n, params)
    lam = _apply_sum(psi, n, *workloads.tfim_terms(n))
    e = torch.real(_inner(psi, lam))
    grad = torch.zeros_like(params)
    for g in reversed(gates):
        if g[0] == "rot":
            grad[:, g[3]] += torch.imag(_inner(lam, _pauli(psi, n, g[1], g[2])))
        psi = _undo_or_do(psi, n, g, params, -1.0)
        lam = _undo_or_do(lam, n, g, params, -1.0)
    return e, grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    s = prepare(case, seed)
    with torch.no_grad():
        if kind in ("energy_grad", "forward"):
            gates = _ansatz(case["ansatz"], case["n"], case["layers"])[0]
            params = s["params"].double()
            if kind == "energy_grad":
                return _energy_grad(gates, case["n"], params)
            psi = _forward(gates, case["n"], params)
            return psi, _inner(psi, _apply_sum(psi, case["n"], *workloads.tfim_terms(case["n"])))
        if kind == "uneven":
            out = []
            for n, (_, params, _) in zip(range(case["lo"], case["hi"] + 1), s["items"]):
                psi = _forward(_ansatz(case["ansatz"], n, case["layers"])[0], n, params.double())
                out.append((psi, _inner(psi, _apply_sum(psi, n, *workloads.tfim_terms(n)))))
            return out
        if kind == "blocks":
            n, psi = case["n"], s["psi"].to(torch.complex128)
            for sp in workloads.brickwork(n, case["depth"], seed=7):
                if len(sp.qubits) == 2:  # CZ
                    a, b = sp.qubits
                    v = psi.view(1 << a, 2, 1 << (b - a - 1), 2, 1 << (n - 1 - b))
                    v[:, 1, :, 1] *= -1
                else:
                    v, m = _split(psi, n, sp.qubits[0]), sp.mat
                    x, y = v[:, :, 0], v[:, :, 1]
                    psi = torch.stack([complex(m[0, 0]) * x + complex(m[0, 1]) * y,
                                       complex(m[1, 0]) * x + complex(m[1, 1]) * y], dim=2).reshape(psi.shape)
            return psi
        if kind == "circuit":
            n, layers = case["n"], case["layers"]
            gates = [("h", q) for q in range(n)]
            for j in range(layers):
                gates += [("rot", "zz", (q, q + 1), 2 * j * n + q) for q in range(n - 1)]
                gates += [("rot", "x", (q,), (2 * j + 1) * n + q) for q in range(n)]
            # exp1 turns by twice its angle
            scale = torch.ones(2 * layers, n, dtype=torch.float64, device=DEV)
            scale[0::2] = 2.0
            e, grad = _energy_grad(gates, n, (s["params"].double() * scale).reshape(1, -1))
            return e.reshape(()), grad.reshape(2 * layers, n) * scale
        psi = s["psi"].detach().to(torch.complex128).reshape(-1, 1 << case["n"])
        if kind == "sparse":
            hp = _apply_sum(psi, case["n"], *workloads.tfim_terms(case["n"]))
            return torch.real(_inner(psi, hp)).reshape(()), (2.0 * hp).reshape(-1)
        codes, w = _strings(case["n"], case["terms"])
        if kind == "hamiltonian":
            hp = _apply_sum(psi, case["n"], codes, w)
            return _inner(psi, hp), hp
        each, out = [], torch.zeros_like(psi)
        for t in range(case["terms"]):
            p = float(w[t]) * _string(psi, case["n"], codes[t])
            each.append(_inner(psi, p))
            out += s["weights"][:, t].view(-1, 1) * p
        return torch.stack(each, dim=1), out
