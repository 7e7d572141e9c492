"""The work this framework is timed on: whole calls a user's program makes.

Six kinds of work, one per public way in:

* ``quil``    -- an interpreted Quil program on ``make_qvm``: gate by gate, a
  MEASURE on every other qubit, amplitudes read back.  The smallest calls.
* ``plain``   -- a gate list applied one ``apply_matrix`` call per gate (the
  bit-exact path), then measure-all shots.
* ``program`` -- a gate list compiled once (tile passes or dense blocks on the
  matrix cores) and replayed from |0...0>, then expectations, marginals, shots
  or amplitudes.
* ``batch``   -- many QAOA MaxCut instances of uneven sizes in one batch.
* ``density`` -- a noisy program on the density-matrix machine.
* ``noisy``   -- one noisy trajectory on the pure-state machine.

Everything a case uses (angles, graphs, Haar unitaries, uniforms) is drawn
from the seed here, so ``exact`` can follow the same circuit in 64 bits with
torch alone.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from qvm_amd import planner as P
from qvm_amd.batch import Batch
from qvm_amd.density import DensityQVM
from qvm_amd.noise import NoisyQVM
from qvm_amd.qvm import make_qvm
from qvm_amd.state import HipPureState

# ---------------------------------------------------------------------------
# Cases


def listed():
    return [
        # the QVM server's everyday request: a few qubits, interpreted, measured
        dict(name="quil_n11", kind="quil", n=11, layers=2),
        # inner loop of a variational algorithm: a small compiled ansatz, replayed
        dict(name="vqe_n14", kind="program", circuit="layered", n=14, depth=4, dtype="f64", fma=False,
             mode="tiled", k=0, shots=0),
        # the CPU-runnable benchmark configuration (20 qubits, 20 layers, 10^4 shots)
        dict(name="plain_n20", kind="plain", circuit="layered", n=20, depth=20, dtype="f64", shots=10000),
        # layers of the headline configuration at its full 16 GiB state, 10^6 shots
        dict(name="plain_n30", kind="plain", circuit="layered", n=30, depth=1, dtype="f64", shots=1000000),
        # QFT of a product state compiled with the default options, odd size
        dict(name="qft_n27", kind="program", circuit="qft", n=27, depth=1, dtype="f64", fma=False,
             mode="tiled", k=0, shots=10000),
        # random 1q/2q mix, FP64 with contracted tiles
        dict(name="mix_n28", kind="program", circuit="mix", n=28, depth=20, dtype="f64", fma=True,
             mode="tiled", k=0, shots=10000),
        # the precision configuration's circuit in complex FP32 at 30 qubits
        dict(name="haar_n30_f32", kind="program", circuit="haar_cz", n=30, depth=20, dtype="f32", fma=True,
             mode="tiled", k=0, shots=0),
        # dense 6-qubit unitaries, as a fusing compiler emits them
        dict(name="dense_n24", kind="program", circuit="dense", n=24, depth=4, dtype="f64", fma=False,
             mode="fused", k=6, shots=1000),
        # QAOA parameter sweep with shots, FP64
        dict(name="qaoa64_f64", kind="batch", count=64, nmin=10, nmax=24, dtype="f64", shots=1024),
        # the same sweep for its expectations only, FP32
        dict(name="qaoa96_f32", kind="batch", count=96, nmin=10, nmax=24, dtype="f32", shots=0),
        # noisy circuit on the density-matrix machine
        dict(name="density_n12", kind="density", n=12, layers=2),
        # one noisy trajectory
        dict(name="noisy_n24", kind="noisy", n=24, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds; every kind over its own range."""
    kind = rng.choice(["quil", "plain", "plain", "program", "program", "program", "program", "batch", "density",
                       "noisy"])
    if kind == "quil":
        return dict(kind="quil", n=rng.randint(3, 20), layers=rng.randint(1, 4))
    if kind == "plain":
        n = rng.randint(8, 29)
        return dict(kind="plain", circuit=rng.choice(["layered", "qft", "haar_cz", "mix"]), n=n,
                    depth=rng.randint(1, 1 if n > 27 else 3 if n > 24 else 20),
                    dtype=rng.choice(["f64", "f64", "f32"]), shots=_log(rng, 1, 100000))
    if kind == "program":
        circuit = rng.choice(["layered", "qft", "haar_cz", "mix", "qaoa", "dense"])
        n = rng.randint(9, 28)
        dtype = rng.choice(["f64", "f64", "f32"])
        if circuit == "dense":
            k = rng.randint(3, 6)
            return dict(kind="program", circuit=circuit, n=min(n, 26), depth=rng.randint(1, 4), dtype=dtype,
                        fma=False, mode="fused", k=k, shots=_log(rng, 1, 1000) if dtype == "f64" else 0)
        mode = rng.choice(["tiled", "tiled", "tiled", "fused"])
        return dict(kind="program", circuit=circuit, n=n, depth=rng.randint(1, 4 if n > 24 else 16), dtype=dtype,
                    fma=mode == "tiled" and rng.random() < 0.6, mode=mode, k=rng.randint(3, 5) if mode == "fused" else 0,
                    shots=_log(rng, 1, 10000) if dtype == "f64" and n > 14 else 0)
    if kind == "batch":
        nmax = rng.choice([12, 16, 18, 20, 22, 24])
        dtype = rng.choice(["f64", "f32"])
        return dict(kind="batch", count=_log(rng, 4, 64), nmin=8 if nmax < 18 else 10, nmax=nmax, dtype=dtype,
                    shots=_log(rng, 16, 1024) if dtype == "f64" else 0)
    if kind == "density":
        return dict(kind="density", n=rng.randint(3, 12), layers=rng.randint(1, 3))
    return dict(kind="noisy", n=rng.randint(5, 25), layers=rng.randint(1, 2))


# ---------------------------------------------------------------------------
# Gate matrices and circuits (Quil convention: the first qubit of a gate is the
# most significant bit of its matrix index)

_H = np.array([[1, 1], [1, -1]], dtype=np.complex128) * math.sqrt(0.5)
_X = np.array([[0, 1], [1, 0]], dtype=np.complex128)
_Y = np.array([[0, -1j], [1j, 0]], dtype=np.complex128)
_Z = np.diag([1, -1]).astype(np.complex128)
_CNOT = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]], dtype=np.complex128)
_CZ = np.diag([1, 1, 1, -1]).astype(np.complex128)
_SWAP = np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], dtype=np.complex128)


def _cis(x):
    return complex(math.cos(x), math.sin(x))


def _rx(t):
    c, s = math.cos(t / 2), math.sin(t / 2)
    return np.array([[c, -1j * s], [-1j * s, c]], dtype=np.complex128)


def _rz(t):
    return np.array([[_cis(-t / 2), 0], [0, _cis(t / 2)]], dtype=np.complex128)


def _rzz(t):
    return np.diag([_cis(-t / 2), _cis(t / 2), _cis(t / 2), _cis(-t / 2)]).astype(np.complex128)


def _cphase(t):
    return np.diag([1, 1, 1, _cis(t)]).astype(np.complex128)


def _haar(rng, k):
    d = 1 << k
    z = np.array([[complex(rng.gauss(0, 1), rng.gauss(0, 1)) for _ in range(d)] for _ in range(d)])
    q, r = np.linalg.qr(z)
    r = np.diag(r)
    return np.ascontiguousarray(q * (r / np.abs(r)))


def _pair(rng, n):
    a = rng.randrange(n)
    b = rng.randrange(n - 1)
    return a, b + 1 if b >= a else b


def _circuit(case, rng):
    """The case's gate list: (matrix, qubits) pairs."""
    n, depth, out = case["n"], case["depth"], []
    if case["circuit"] == "layered":
        for layer in range(depth):
            for q in range(n):
                out.append((_rx(rng.uniform(0, 2 * math.pi)), [q]))
                out.append((_rz(rng.uniform(0, 2 * math.pi)), [q]))
            out += [(_CNOT, [i, i + 1]) for i in range(layer % 2, n - 1, 2)]
    elif case["circuit"] == "qft":
        # of a random product state
        out += [(_rx(rng.uniform(0, 2 * math.pi)), [q]) for q in range(n)]
        for q in range(n - 1, -1, -1):
            out.append((_H, [q]))
            out += [(_cphase(math.pi / 2 ** (q - j)), [q, j]) for j in range(q - 1, -1, -1)]
        out += [(_SWAP, [i, n - 1 - i]) for i in range(n // 2)]
    elif case["circuit"] == "haar_cz":
        for _ in range(depth):
            out += [(_haar(rng, 1), [q]) for q in range(n)]
            order = rng.sample(range(n), n)
            out += [(_CZ, [order[i], order[i + 1]]) for i in range(0, n - 1, 2)]
    elif case["circuit"] == "mix":
        for _ in range(depth * n):
            if rng.random() < 0.6:
                out.append((_haar(rng, 1), [rng.randrange(n)]))
            else:
                out.append((_CNOT if rng.random() < 0.5 else _CZ, list(_pair(rng, n))))
    elif case["circuit"] == "qaoa":
        out += [(_H, [q]) for q in range(n)]
        for _ in range(depth):
            g, b = rng.uniform(0, math.pi), rng.uniform(0, math.pi / 2)
            out += [(_rzz(g), list(_pair(rng, n))) for _ in range(3 * n // 2)]
            out += [(_rx(b), [q]) for q in range(n)]
    else:
        for _ in range(depth):
            out += [(_haar(rng, 1), [q]) for q in range(n)]
            order = rng.sample(range(n), n)
            k = case["k"]
            out += [(_haar(rng, k), order[b * k:(b + 1) * k]) for b in range(n // k)]
    return out


def _regular3(n, rng):
    """A random simple 3-regular graph on n (even) vertices."""
    while True:
        points = [v for v in range(n) for _ in range(3)]
        rng.shuffle(points)
        edges = {tuple(sorted(points[i:i + 2])) for i in range(0, 3 * n, 2)}
        if len(edges) == 3 * n // 2 and all(a != b for a, b in edges):
            return sorted(edges)


def _instances(case, rng):
    """(n, edges, gammas, betas) per QAOA instance; the sizes of the range
    come up in turn, so every seed has the same mix of them."""
    sizes = range(case["nmin"] + case["nmin"] % 2, case["nmax"] + 1, 2)
    out = []
    for i in range(case["count"]):
        n, p = sizes[i % len(sizes)], 1 + (i // len(sizes)) % 4
        out.append((n, _regular3(n, rng), [rng.uniform(0, math.pi) for _ in range(p)],
                    [rng.uniform(0, math.pi / 2) for _ in range(p)]))
    return out


def _qaoa(n, edges, gammas, betas):
    out = [(_H, [q]) for q in range(n)]
    for g, b in zip(gammas, betas):
        out += [(_rzz(g), list(e)) for e in edges]
        out += [(_rx(b), [q]) for q in range(n)]
    return out


def _ring(n):
    return [(i, (i + 1) % n) for i in range(n)]


def _steps(case, rng):
    """The instructions of a Quil case: (gate name, angle or None, qubits)."""
    n, out = case["n"], []
    noisy = case["kind"] != "quil"
    for layer in range(case["layers"]):
        out += [("RX", rng.uniform(0, 2 * math.pi), [q]) for q in range(n)]
        out += [("H", None, [q]) if noisy else ("RZ", rng.uniform(0, 2 * math.pi), [q]) for q in range(n)]
        out += [("CNOT", None, [i, i + 1]) for i in range(layer % 2, n - 1, 2)]
        if noisy:
            out += [("I", None, [q]) for q in range(n)]
    return out


def _quil(case, steps):
    lines = ["DECLARE ro BIT[%d]" % case["n"]]
    for name, angle, qubits in steps:
        lines.append("%s%s %s" % (name, "" if angle is None else "(%r)" % angle, " ".join(map(str, qubits))))
    if case["kind"] == "quil":
        lines += ["MEASURE %d ro[%d]" % (q, q) for q in range(0, case["n"], 2)]
    return "\n".join(lines) + "\n"


def _noise(case, rng):
    """Kraus lists of the noisy gates: H followed by a Pauli channel, I as
    amplitude damping, CNOT followed by correlated dephasing."""
    n, out = case["n"], {}
    for q in range(n):
        px, py, pz = (rng.uniform(0.002, 0.02) for _ in range(3))
        out["H", (q,)] = [math.sqrt(1 - px - py - pz) * _H, math.sqrt(px) * _X @ _H, math.sqrt(py) * _Y @ _H,
                          math.sqrt(pz) * _Z @ _H]
        g = rng.uniform(0.01, 0.1)
        out["I", (q,)] = [np.array([[1, 0], [0, math.sqrt(1 - g)]], dtype=np.complex128),
                          np.array([[0, math.sqrt(g)], [0, 0]], dtype=np.complex128)]
        if q + 1 < n:
            p = rng.uniform(0.005, 0.03)
            out["CNOT", (q, q + 1)] = [math.sqrt(1 - p) * _CNOT, math.sqrt(p) * np.kron(_Z, _Z) @ _CNOT]
    return out


# ---------------------------------------------------------------------------
# One pass


def prepare(case, seed):
    rng = random.Random(int(seed))
    kind = case["kind"]
    st = {"case": case}
    if kind in ("quil", "density", "noisy"):
        steps = _steps(case, rng)
        kraus = _noise(case, rng) if kind != "quil" else {}
        draws = [rng.random() for _ in range(len(steps) + 2 * case["n"] + 8)]
        if kind == "quil":
            qvm = make_qvm(case["n"])
        elif kind == "density":
            qvm = DensityQVM(case["n"], noisy_gate_definitions=kraus)
        else:
            qvm = NoisyQVM(case["n"], noisy_gate_definitions=kraus)
        qvm.load_program(_quil(case, steps))
        st.update(qvm=qvm, draws=draws)
    elif kind in ("plain", "program"):
        gates = _circuit(case, rng)
        state = HipPureState(case["n"], case["dtype"], fma_tiles=case.get("fma", False))
        st["state"] = state
        if kind == "plain":
            st["plan"] = P.plan_plain(gates, case["n"])
        else:
            st["program"] = P.compile_gates(state, gates, mode=case["mode"], merge_1q=case["fma"],
                                            kmax=case["k"] or 4)
        st["u"] = np.random.RandomState(int(seed) % (1 << 32)).random_sample(case["shots"])
    else:
        inst = _instances(case, rng)
        count, shots = case["count"], case["shots"]
        u = np.random.RandomState(int(seed) % (1 << 32)).random_sample(count * shots) if shots else None
        st["batch"] = Batch([_qaoa(*i) for i in inst], [i[0] for i in inst], case["dtype"],
                            edges=[i[1] for i in inst], shots=shots, uniforms=u, fma_tiles=True)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("quil", "density", "noisy"):
        qvm = st["qvm"]
        qvm.rng = iter(st["draws"]).__next__
        qvm.reset_quantum_state()
        qvm.run()
        if kind == "quil":
            return {"bits": np.array(qvm.memory["ro"]), "amplitudes": qvm.amplitudes()}
        if kind == "density":
            return {"probabilities": qvm.measurement_probabilities()}
        marginals = np.array([qvm.state.prob_excited(q) for q in range(case["n"])])
        return {"marginals": marginals, "bits": np.array(qvm.measure_all()[1])}
    if kind == "batch":
        b = st["batch"]
        b.run()
        expectations, shots = b.results()
        # a batch of FP32 states gives its costs in FP32
        out = {"cost": expectations if case["dtype"] == "f64" else expectations.astype(np.float32)}
        if case["shots"]:
            out["shots"] = shots
        return out
    state = st["state"]
    state.reset_zero()
    if kind == "plain":
        P.execute_plan(state, st["plan"])
        return {"shots": state.sample_measure_all(st["u"])}
    st["program"].run()
    n, real = case["n"], np.float64 if case["dtype"] == "f64" else np.float32
    out = {"zz": real(state.expectation_zz(_ring(n)))}
    if case["dtype"] == "f32":
        out["marginals"] = np.array([state.prob_excited(q) for q in range(n)], dtype=real)
    if n <= 14:
        out["amplitudes"] = state.amplitudes().astype(np.complex128 if case["dtype"] == "f64" else np.complex64)
    if case["shots"]:
        out["shots"] = state.sample(st["u"])
    return out


# ---------------------------------------------------------------------------
# What one pass cannot do without


def _flops(U, n):
    """Floating-point operations of one gate: 6 per complex product (2 for the
    sum) of a row's nonzero entries other than 1, over the rows it changes."""
    d = U.shape[0]
    total = 0
    for r in range(d):
        nz = np.nonzero(U[r])[0]
        if len(nz) == 1 and U[r, nz[0]] == 1:
            continue
        total += 8 * len(nz) - 2
    return float(total) * 2.0 ** n / d


def _moved(U):
    """Share of the amplitudes a gate can change."""
    return float(np.mean(np.any(U != np.eye(U.shape[0]), axis=1)))


def work(case):
    rng = random.Random(1)
    kind = case["kind"]
    if kind in ("quil", "noisy"):
        n, steps = case["n"], _steps(case, rng)
        # every gate is a call of its own: the amplitudes in and out
        byte = 32.0 * 2.0 ** n * len(steps)
        if kind == "quil":
            return {"bytes": byte + 48.0 * 2.0 ** n * ((n + 1) // 2), "flops": 14.0 * 2.0 ** n * len(steps)}
        return {"bytes": byte + 16.0 * 2.0 ** n * (len(steps) + n), "flops": 14.0 * 2.0 ** n * len(steps)}
    if kind == "density":
        n, steps = case["n"], _steps(case, rng)
        return {"bytes": 32.0 * 4.0 ** n * len(steps), "flops": 30.0 * 4.0 ** n * len(steps)}
    if kind == "batch":
        byte = flops = 0.0
        for n, edges, gam, bet in _instances(case, rng):
            amp = 16.0 if case["dtype"] == "f64" else 8.0
            byte += 2 * amp * 2.0 ** n  # the state written, then read for its cost and shots
            flops += 2.0 ** n * (14 * n + len(gam) * (6 * len(edges) + 14 * n))
        return {"bytes": byte, "flops": flops}
    n, amp = case["n"], 16.0 if case["dtype"] == "f64" else 8.0
    gates = _circuit(case, rng)
    flops = sum(_flops(U, n) for U, _ in gates)
    if kind == "plain":  # every gate is a call of its own
        return {"bytes": amp * 2.0 ** n * (2 * sum(_moved(U) for U, _ in gates) + 2), "flops": flops}
    sweeps = 2 + (n if case["dtype"] == "f32" else 0) + (1 if case["shots"] else 0)
    return {"bytes": amp * 2.0 ** n * sweeps, "flops": flops}


# ---------------------------------------------------------------------------
# The same in 64 bits with torch alone


def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda" if torch.cuda.is_available() else "cpu")
    psi[0] = 1
    return psi


def _parts(psi, bits):
    """psi's slices by the values of the given index bits: slices[j], bit i
    of j being the value of index bit bits[i]."""
    n = psi.numel().bit_length() - 1
    order = sorted(range(len(bits)), key=lambda i: -bits[i])
    shape, top = [], n
    for i in order:
        shape += [1 << (top - bits[i] - 1), 2]
        top = bits[i]
    v = psi.view(shape + [1 << top])
    out = []
    for j in range(1 << len(bits)):
        at = []
        for i in order:
            at += [slice(None), (j >> i) & 1]
        out.append(v[tuple(at)])
    return out


def _apply(psi, U, qubits):
    nat = list(reversed(qubits))
    src = _parts(psi, nat)
    new = torch.empty_like(psi)
    dst = _parts(new, nat)
    for r in range(U.shape[0]):
        acc = None
        for c in np.nonzero(U[r])[0]:
            term = src[c] * complex(U[r, c]) if U[r, c] != 1 else src[c]
            acc = term if acc is None else acc + term
        dst[r].copy_(acc) if acc is not None else dst[r].zero_()
    return new


def _prob(psi):
    return psi.real.square() + psi.imag.square()


def _zz(p, edges):
    total = 0.0
    for a, b in edges:
        s = _parts(p, [a, b])
        total += float(s[0].sum() + s[3].sum() - s[1].sum() - s[2].sum())
    return total


def _marginals(p, n):
    return np.array([float(_parts(p, [q])[1].sum()) for q in range(n)])


def _matrix(name, angle):
    return {"RX": lambda: _rx(angle), "RZ": lambda: _rz(angle), "H": lambda: _H, "CNOT": lambda: _CNOT,
            "I": lambda: np.eye(2, dtype=np.complex128)}[name]()


def exact(case, seed):
    rng = random.Random(int(seed))
    kind, n = case["kind"], case.get("n", 0)
    if kind == "plain" or (kind == "program" and n > 28):
        return None  # shots only, or beyond 20 seconds
    if kind == "program":
        psi = _zero(n)
        for U, q in _circuit(case, rng):
            psi = _apply(psi, U, q)
        p = _prob(psi)
        out = {"zz": np.float64(_zz(p, _ring(n)))}
        if case["dtype"] == "f32":
            out["marginals"] = _marginals(p, n)
        if n <= 14:
            out["amplitudes"] = psi.cpu().numpy()
        if case["shots"]:
            out["shots"] = None
        return out
    if kind == "batch":
        cost = []
        for m, edges, gammas, betas in _instances(case, rng):
            psi = torch.full_like(_zero(m), 2.0 ** (-m / 2))
            zz = torch.zeros(1 << m, dtype=torch.float64, device=psi.device)
            for a, b in edges:
                s = _parts(zz, [a, b])
                for j, sign in enumerate((1, -1, -1, 1)):
                    s[j].add_(sign)
            for g, b in zip(gammas, betas):
                psi = psi * torch.polar(torch.ones_like(zz), zz * (-g / 2))
                for q in range(m):
                    psi = _apply(psi, _rx(b), [q])
            cost.append(float((_prob(psi) * zz).sum()))
        out = {"cost": np.array(cost)}
        if case["shots"]:
            out["shots"] = None
        return out
    steps = _steps(case, rng)
    kraus = _noise(case, rng) if kind != "quil" else {}
    draws = iter([rng.random() for _ in range(len(steps) + 2 * n + 8)])
    if kind == "density":
        rho = _zero(2 * n)
        for name, angle, qubits in steps:
            ops = kraus.get((name, tuple(qubits)), [_matrix(name, angle)])
            # vec(K rho K^H): K on the row bits (q + n), conj(K) on the column bits
            S = sum(np.kron(K, K.conj()) for K in ops)
            rho = _apply(rho, S, [q + n for q in qubits] + list(qubits))
        d = 1 << n
        return {"probabilities": rho.view(d, d).diagonal().real.cpu().numpy().copy()}
    psi = _zero(n)
    for name, angle, qubits in steps:
        ops = kraus.get((name, tuple(qubits)))
        if ops is None:
            psi = _apply(psi, _matrix(name, angle), qubits)
            continue
        r, total = next(draws), 0.0
        for K in ops:
            trial = _apply(psi, K, qubits)
            weight = float(_prob(trial).sum())
            total += weight
            if total >= r:
                break
        psi = trial / math.sqrt(weight)
    if kind == "noisy":
        return {"marginals": _marginals(_prob(psi), n), "bits": None}
    for q in range(0, n, 2):
        p1 = float(_prob(_parts(psi, [q])[1]).sum())
        bit = 0 if p1 == 0.0 else 1 if next(draws) <= p1 else 0
        psi = psi.clone()
        parts = _parts(psi, [q])
        parts[1 - bit].zero_()
        parts[bit].mul_(1 / math.sqrt(p1 if bit else 1 - p1))
    return {"bits": None, "amplitudes": psi.cpu().numpy()}
