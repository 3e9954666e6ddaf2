"""The workloads whose speed is tracked, each through the package's public entry points.

A case is a dict of plain values. ``prepare(case, seed)`` makes what a program
holds before the timed call (circuit, plan, handle, inputs; all numbers come
from the seed, the circuit's wiring from the case), ``run(state)`` is one pass,
``work(case)`` what a pass cannot do without, and ``exact(case, seed)`` the
outputs in 64 bits by plain torch/numpy statevector arithmetic.

Kinds of case and what they stand for:

gates    a circuit gate by gate (``State.apply_gates``), the reference driver's
         unpartitioned run
part     a partitioned circuit on the FP64 part path (``State.apply_part``),
         the drop-in for the reference's gather_and_execute_on
fused    the same on the matrix cores, FP64 or FP32-split products
chain    the BF16-split paths with the moving layout (the benchmark's path)
sample   read-out of a state in hand: P(1) of every qubit, then shots of the
         whole register
energy   <H> of a Heisenberg chain on a state in hand, term by term, as a
         variational program evaluates it
batch    one step of a variational loop over many small circuits: new
         parameters, one run, <Z> of each
qaoa     one evaluation of many QAOA MaxCut instances at new angles
mlp      one step on the cost model: predictions and all gradients

A circuit pass starts from |0...0> (reset) and ends with what the program
reads: the state itself up to 20 qubits, above that P(1) and Pauli
expectations of a few qubits and, on the FP64 paths, shots of a register, as
the QASM driver does. Results of the split-precision paths and of complex64
states are returned in single precision, which is what those paths carry.
"""
import math
import random

import numpy as np
import torch

from hisvsim_amd import batch as circuit_batch
from hisvsim_amd import capi, costmodel, qaoa
from hisvsim_amd.circuit import Gate, gate_amplitudes, gaussian_state, qft, random_layered
from hisvsim_amd.partition import chain_parts, closure_parts

LOW = 5          # slots the device adds to wide parts
READ_QUBITS = 20  # widest state a pass reads back whole
SHOTS = 10       # the driver's shots per run


def listed():
    return [
        # the smallest call: a few dozen gates on a tiny register, where each
        # launch and each conversion counts (interactive use, unit tests)
        {"name": "gates_n10", "kind": "gates", "circuit": "layered", "n": 10, "depth": 4, "dtype": "complex128"},
        # an ordinary partitioned run whose state is read back
        {"name": "part_n19", "kind": "part", "circuit": "layered", "n": 19, "depth": 8, "k": 12,
         "dtype": "complex128"},
        # the largest: a 34 GB state on the FP64 part path, with the driver's read-outs
        {"name": "part_n31", "kind": "part", "circuit": "layered", "n": 31, "depth": 4, "k": 12,
         "dtype": "complex128"},
        # fused unitaries with FP64 products, QFT in 7-qubit parts
        {"name": "fused64_n28", "kind": "fused", "circuit": "qft", "n": 28, "depth": 0, "k": 7, "mode": "f64",
         "dtype": "complex128"},
        # fused unitaries with FP32-split products at an odd size
        {"name": "fused32_n25", "kind": "fused", "circuit": "layered", "n": 25, "depth": 5, "k": 6,
         "mode": "f32split", "dtype": "complex128"},
        # the benchmark's path: two-piece BF16 products, 13-qubit chain parts
        {"name": "chain_n30", "kind": "chain", "circuit": "layered", "n": 30, "depth": 12, "k": 13,
         "mode": "bf16split", "dtype": "complex128"},
        # its FP32-class form on a complex64 state, a QFT
        {"name": "chain_x3_c64_n27", "kind": "chain", "circuit": "qft", "n": 27, "depth": 0, "k": 13,
         "mode": "bf16x3", "dtype": "complex64"},
        # sampling a register: 1000 shots of every qubit, marginals first
        {"name": "sample_n24", "kind": "sample", "n": 24, "shots": 1000, "dtype": "complex128"},
        # term-by-term energy of a complex64 state
        {"name": "energy_c64_n28", "kind": "energy", "n": 28, "depth": 2, "dtype": "complex64"},
        # a variational step over uneven small circuits
        {"name": "batch_192", "kind": "batch", "instances": 192, "nmin": 8, "nmax": 18, "wiring": 0,
         "dtype": "complex128"},
        # one QAOA evaluation of a batch of uneven instances
        {"name": "qaoa_256", "kind": "qaoa", "instances": 256, "nmin": 12, "nmax": 22, "wiring": 0},
        # the cost model's forward and backward pass
        {"name": "mlp_6000", "kind": "mlp", "samples": 6000, "hidden": 64},
    ]


def draw(rng):
    """One more case of the listed ranges; the width of a state is drawn
    evenly, so the amplitudes are spread over their logarithm."""
    kind = rng.choice(["gates", "part", "fused", "chain", "sample", "energy", "batch", "qaoa", "mlp"])
    dtype = rng.choice(["complex128", "complex64"])
    circuit = rng.choice(["layered", "qft"])
    if kind == "gates":
        return {"kind": kind, "circuit": circuit, "n": rng.randint(6, 24), "depth": rng.randint(1, 6), "dtype": dtype}
    if kind == "part":
        return {"kind": kind, "circuit": circuit, "n": rng.randint(12, 29), "depth": rng.randint(2, 8),
                "k": rng.randint(9, 12), "dtype": dtype}
    if kind == "fused":
        return {"kind": kind, "circuit": circuit, "n": rng.randint(14, 27), "depth": rng.randint(2, 6),
                "k": rng.randint(5, 7), "mode": rng.choice(["f64", "f32split"]), "dtype": dtype}
    if kind == "chain":
        return {"kind": kind, "circuit": circuit, "n": rng.randint(16, 30), "depth": rng.randint(4, 12),
                "k": rng.choice([12, 13]), "mode": rng.choice(["bf16split", "bf16x3"]), "dtype": dtype}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(10, 24),
                "shots": int(round(math.exp(rng.uniform(math.log(10), math.log(1000))))), "dtype": dtype}
    if kind == "energy":
        return {"kind": kind, "n": rng.randint(10, 28), "depth": rng.randint(1, 3), "dtype": dtype}
    if kind == "batch":
        return {"kind": kind, "instances": int(round(math.exp(rng.uniform(math.log(8), math.log(192))))),
                "nmin": rng.randint(4, 10), "nmax": rng.randint(11, 18), "wiring": rng.randint(1, 9999),
                "dtype": dtype}
    if kind == "qaoa":
        return {"kind": kind, "instances": int(round(math.exp(rng.uniform(math.log(8), math.log(256))))),
                "nmin": rng.randint(8, 13), "nmax": rng.randint(14, 22), "wiring": rng.randint(1, 9999)}
    return {"kind": kind, "samples": int(round(math.exp(rng.uniform(math.log(300), math.log(20000))))),
            "hidden": rng.choice([32, 64, 96])}


# ---- circuits ---------------------------------------------------------------

def _circuit(case, seed):
    """The case's gates: wiring from its sizes alone, angles from the seed."""
    n = case["n"]
    rng = np.random.default_rng([seed, 11])

    def u3(q):
        return Gate("U3", (q,), (), tuple(float(x) for x in rng.uniform(0.0, 2 * math.pi, 3)))

    if case.get("circuit", "layered") == "qft":
        return [u3(q) for q in range(n)] + qft(n)   # on a product state
    return [u3(g.targets[0]) if g.name == "U3" else g for g in random_layered(n, case["depth"], seed=n)]


def _readout(case, seed):
    """The qubits measured, the Pauli strings read and the shots' uniforms."""
    n = case["n"]
    r = random.Random(n)
    qubits = sorted(r.sample(range(n), min(4, n)))
    paulis = []
    for letters in ("XX", "YZ", "ZY", "ZZ"):
        a, b = r.sample(range(n), 2)
        paulis.append("%s%d %s%d" % (letters[0], a, letters[1], b))
    return qubits, paulis, np.random.default_rng([seed, 13]).random(SHOTS)


def _single(case):
    return case["dtype"] == "complex64" or case.get("mode") in ("f32split", "bf16split", "bf16x3")


def _random_state(case, seed):
    """Amplitudes as a deep random circuit leaves them: i.i.d. complex Gaussian."""
    return gaussian_state(case["n"], seed)


def _layered_state(case, seed):
    """A state in hand, made on the FP64 part path."""
    s = capi.State(case["n"], case["dtype"])
    gates = _circuit(case, seed)
    if case["n"] < 12:
        s.apply_gates(gates)
    else:
        for p in closure_parts(gates, 12, always=range(LOW)):
            s.apply_part(p, 0)
    s.synchronize()
    return s


def _bonds(n):
    return ["%s%d %s%d" % (p, q, p, q + 1) for q in range(n - 1) for p in "XYZ"]


def _batch_instances(case, seed):
    """(n, gates) per instance; the circuits' shapes from the case, the angles from the seed."""
    shape = np.random.default_rng([case["wiring"], 17])
    rng = np.random.default_rng([seed, 19])
    out = []
    for _ in range(case["instances"]):
        n = int(shape.integers(case["nmin"], case["nmax"] + 1))
        layers = int(shape.integers(2, 7))
        out.append((n, circuit_batch.ansatz(n, layers, rng.uniform(0, 2 * math.pi, 2 * n * layers))))
    return out


def _batch_masks(case):
    r = random.Random(case["wiring"])
    return [r.getrandbits(case["nmin"]) | 1 for _ in range(case["instances"])]


def _qaoa_instances(case, seed):
    insts = qaoa.make_batch(case["instances"], case["wiring"], (case["nmin"], case["nmax"]))
    rng = np.random.default_rng([seed, 23])
    return [qaoa.Instance(i.n, i.edges, [float(x) for x in rng.uniform(0, math.pi, i.p)],
                          [float(x) for x in rng.uniform(0, math.pi, i.p)]) for i in insts]


def _mlp_data(case, seed):
    """Features in the cost model's range, targets a smooth function of them, and the network's weights."""
    rng = np.random.default_rng([seed, 29])
    n, f, h = case["samples"], costmodel.N_FEATURES, case["hidden"]
    x = rng.uniform(0.0, 1.3, (n, f)).astype(np.float32)
    y = (x.sum(axis=1) / f + 0.3 * np.sin(3 * x[:, 0]) + 0.05 * rng.standard_normal(n)).astype(np.float32)
    w = np.concatenate([rng.uniform(-1, 1, f * h) * math.sqrt(6.0 / f), 0.1 * rng.uniform(-1, 1, h),
                        rng.uniform(-1, 1, h * h) * math.sqrt(6.0 / h), 0.1 * rng.uniform(-1, 1, h),
                        rng.uniform(-1, 1, h) * math.sqrt(6.0 / h), 0.1 * rng.uniform(-1, 1, 1)]).astype(np.float32)
    return x, y, w


# ---- prepare and run --------------------------------------------------------

def _plan(case, gates):
    """(parts, lows) as the driver and the benchmark plan each path."""
    kind = case["kind"]
    if kind == "part":
        return closure_parts(gates, min(case["k"], case["n"]), always=range(LOW)), None
    if kind == "fused":
        return closure_parts(gates, case["k"]), None
    if kind == "chain":
        return chain_parts(gates, case["k"], LOW, beam=(16, 8))
    return None, None


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("gates", "part", "fused", "chain"):
        st["gates"] = _circuit(case, seed)
        st["parts"], st["lows"] = _plan(case, st["gates"])
        st["qubits"], st["paulis"], st["uniforms"] = _readout(case, seed)
        st["state"] = capi.State(case["n"], case["dtype"])
    elif kind == "sample":
        st["state"] = capi.State(case["n"], case["dtype"])
        st["state"].write(_random_state(case, seed))
        st["uniforms"] = np.random.default_rng([seed, 13]).random(case["shots"])
    elif kind == "energy":
        st["state"] = _layered_state(case, seed)
    elif kind == "batch":
        insts = _batch_instances(case, seed)
        st["batch"] = circuit_batch.CircuitBatch(insts, case["dtype"])
        circuit_batch.apply_tuning(st["batch"])
        st["batch"].run()   # plans and captures
        st["lists"] = [g for _, g in insts]
        st["masks"] = _batch_masks(case)
    elif kind == "qaoa":
        insts = _qaoa_instances(case, seed)
        st["batch"] = qaoa.QAOABatch(insts)
        qaoa.apply_tuning(st["batch"])
        st["batch"].run()   # plans and captures
        st["gammas"], st["betas"] = [i.gammas for i in insts], [i.betas for i in insts]
    else:
        st["x"], st["y"], w = _mlp_data(case, seed)
        st["model"] = costmodel.MLP(costmodel.N_FEATURES, case["hidden"])
        st["model"].set_params(w)
    return st


def _run_circuit(st):
    case, s, kind = st["case"], st["state"], st["case"]["kind"]
    s.reset()
    if kind == "gates":
        s.apply_gates(st["gates"])
    elif kind == "part":
        for p in st["parts"]:
            s.apply_part(p, 0)
    elif kind == "fused":
        for p in st["parts"]:
            s.apply_fused(p, case["mode"])
    else:
        s.apply_fused_chain(st["parts"], st["lows"], case["mode"], renormalize=True)
    if case["n"] <= READ_QUBITS:
        amps = s.read()
        return {"state": amps.astype(np.complex64) if _single(case) else amps}
    values = [s.probability(q, 1) for q in st["qubits"]] + [s.expectation(p) for p in st["paulis"]]
    if _single(case):
        return {"values": np.array(values, np.float32)}
    return {"values": np.array(values), "samples": s.measure(st["qubits"], st["uniforms"])}


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind in ("gates", "part", "fused", "chain"):
        return _run_circuit(st)
    if kind == "sample":
        s, n = st["state"], case["n"]
        return {"p1": np.array([s.probability(q, 1) for q in range(n)]),
                "samples": s.measure(list(range(n)), st["uniforms"])}
    if kind == "energy":
        terms = np.array([st["state"].expectation(t) for t in _bonds(case["n"])])
        terms = terms.astype(np.float32) if _single(case) else terms
        return {"terms": terms, "energy": terms.sum(keepdims=True)}
    if kind == "batch":
        b = st["batch"]
        b.set_gates(st["lists"])
        b.run()
        z = b.expect_z(st["masks"])
        return {"z": z.astype(np.float32) if _single(case) else z}
    if kind == "qaoa":
        st["batch"].set_angles(st["gammas"], st["betas"])
        return {"cost": st["batch"].run().astype(np.float32)}   # complex64 states
    loss, grads = st["model"].gradient(st["x"], st["y"])
    return {"prediction": st["model"].predict(st["x"]), "loss": np.float32(loss), "gradient": grads}


# ---- what a pass cannot do without --------------------------------------------

def _elem(case):
    return 16 if case["dtype"] == "complex128" else 8


def _gate_flops(gates, n):
    """14 flops per amplitude of a dense pair, 6 per phase."""
    return float(sum((14 if g.name in ("U3", "H", "RY", "RX") else 6) * gate_amplitudes(g, n) for g in gates))


def work(case):
    """bytes: per gate (gates) or per part of the plan (part, fused, chain) the
    state read and written once, per read-out the amplitudes it depends on read
    once; per batch instance the state written once. flops: the gates'."""
    kind = case["kind"]
    if kind in ("gates", "part", "fused", "chain"):
        n, size = case["n"], _elem(case)
        full = float(size) * 2 ** n
        gates = _circuit(case, 0)
        parts, _ = _plan(case, gates)
        if kind == "gates":
            moved = 2.0 * size * sum(gate_amplitudes(g, n) for g in gates)
        else:
            moved = 2.0 * full * len(parts)
        moved += full                                    # reset
        if n <= READ_QUBITS:
            moved += full + 16.0 * 2 ** n                # read on the device, written on the host
        else:
            moved += 4 * full / 2 + 4 * full + (0 if _single(case) else full)
        flops = 8.0 * 2 ** n * sum(2 ** case["k"] for _ in parts) if kind == "fused" else _gate_flops(gates, n)
        return {"bytes": moved, "flops": flops}
    if kind == "sample":
        full = float(_elem(case)) * 2 ** case["n"]
        return {"bytes": case["n"] * full / 2 + full, "flops": 3.0 * 2 ** case["n"] * (case["n"] / 2 + 1)}
    if kind == "energy":
        full = float(_elem(case)) * 2 ** case["n"]
        terms = 3 * (case["n"] - 1)
        return {"bytes": terms * full, "flops": 4.0 * terms * 2 ** case["n"]}
    if kind == "batch":
        insts = _batch_instances(case, 0)
        return {"bytes": 2.0 * _elem(case) * sum(2 ** n for n, _ in insts) + 256.0 * sum(len(g) for _, g in insts),
                "flops": sum(_gate_flops(g, n) for n, g in insts)}
    if kind == "qaoa":
        insts = _qaoa_instances(case, 0)
        return {"bytes": 8.0 * sum((1 + 2 * i.p) * 2 ** i.n for i in insts),
                "flops": float(sum(i.p * (6 + 10 * i.n) * 2 ** i.n for i in insts))}
    n, f, h = case["samples"], costmodel.N_FEATURES, case["hidden"]
    p = f * h + h + h * h + h + h + 1
    return {"bytes": 4.0 * (2 * n * (f + 1) + n + 4 * p), "flops": 2.0 * n * (f * h + h * h + h) * 4}


# ---- the same in 64 bits, by plain tensor arithmetic -----------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _matrix(g):
    """2x2 of a one-target gate, as the reference's functors define it."""
    p, name = g.params, g.name
    if name == "U3":     # with the reference's global phase
        t, a, b = p
        c, s = math.cos(t / 2), math.sin(t / 2)
        e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
        return [[c * e(-(a + b) / 2), -s * e((b - a) / 2)], [s * e((a - b) / 2), c * e((a + b) / 2)]]
    if name == "H":
        r = 1 / math.sqrt(2.0)
        return [[r, r], [r, -r]]
    if name == "RY":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return [[c, -s], [s, c]]
    if name == "RX":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return [[c, -1j * s], [-1j * s, c]]
    if name == "RZ":
        return [[complex(math.cos(p[0] / 2), -math.sin(p[0] / 2)), 0],
                [0, complex(math.cos(p[0] / 2), math.sin(p[0] / 2))]]
    if name == "Z":
        return [[1, 0], [0, -1]]
    if name == "R1":
        return [[1, 0], [0, complex(math.cos(p[0]), math.sin(p[0]))]]
    raise ValueError(name)


def _at(v, n, fixed):
    """The view of the 2^n amplitudes with the given qubits fixed."""
    v = v.view(-1)
    shape, index, at = [], [], n
    for q in sorted(fixed, reverse=True):
        shape += [2 ** (at - q - 1), 2]
        index += [slice(None), fixed[q]]
        at = q
    return v.view(*shape, 2 ** at)[tuple(index)]


def _apply(v, n, g):
    if g.name == "SWAP":
        a, b = g.targets
        x, y = _at(v, n, {a: 0, b: 1}), _at(v, n, {a: 1, b: 0})
        t = x.clone()
        x.copy_(y)
        y.copy_(t)
        return
    t, on = g.targets[0], {c: 1 for c in g.controls}
    m = _matrix(g)
    x, y = _at(v, n, {**on, t: 0}), _at(v, n, {**on, t: 1})
    if m[0][1] == 0 and m[1][0] == 0:
        if m[0][0] != 1:
            x.mul_(m[0][0])
        y.mul_(m[1][1])
        return
    new = x * m[0][0]
    new.add_(y, alpha=m[0][1])
    y.mul_(m[1][1])
    y.add_(x, alpha=m[1][0])
    x.copy_(new)


def _simulate(n, gates):
    v = torch.zeros(2 ** n, dtype=torch.complex128, device=_device())
    v[0] = 1
    for g in gates:
        _apply(v, n, g)
    return v


def _mass(v):
    return float(torch.linalg.vector_norm(torch.view_as_real(v).reshape(-1)).item()) ** 2


def _p1(v, n, q):
    return _mass(_at(v, n, {q: 1}))


def _pauli2(v, n, text):
    """<P> of a string on two qubits."""
    (pa, a), (pb, b) = ((t[0], int(t[1:])) for t in text.split())
    one = {"X": lambda i: (1 - i, 1), "Y": lambda i: (1 - i, 1j if i == 0 else -1j), "Z": lambda i: (i, (-1) ** i)}
    total = 0
    for i in (0, 1):
        for j in (0, 1):
            (ti, ci), (tj, cj) = one[pa](i), one[pb](j)
            x, y = _at(v, n, {a: i, b: j}), _at(v, n, {a: ti, b: tj})
            total += ci * cj * complex((y.conj() * x).sum().item())
    return total.real


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gates", "part", "fused", "chain"):
        n = case["n"]
        if _device() == "cpu" and n > READ_QUBITS:
            return None
        v = _simulate(n, _circuit(case, seed))
        if n <= READ_QUBITS:
            return {"state": v.cpu().numpy()}
        qubits, paulis, _ = _readout(case, seed)
        values = np.array([_p1(v, n, q) for q in qubits] + [_pauli2(v, n, p) for p in paulis])
        return {"values": values} if _single(case) else {"values": values, "samples": None}
    if kind == "sample":
        v = torch.from_numpy(_random_state(case, seed)).to(_device())
        if case["dtype"] == "complex64":
            v = v.to(torch.complex64).to(torch.complex128)   # what the state holds
        return {"p1": np.array([_p1(v, case["n"], q) for q in range(case["n"])]), "samples": None}
    if kind == "energy":
        v = _simulate(case["n"], _circuit(case, seed))
        terms = np.array([_pauli2(v, case["n"], t) for t in _bonds(case["n"])])
        return {"terms": terms, "energy": np.array([terms.sum()])}
    if kind == "batch":
        out = []
        for (n, gates), mask in zip(_batch_instances(case, seed), _batch_masks(case)):
            p = _simulate(n, gates).abs().square()
            for q in range(n):
                if mask >> q & 1:
                    _at(p, n, {q: 1}).neg_()
            out.append(float(p.sum()))
        return {"z": np.array(out)}
    if kind == "qaoa":
        out = []
        for i in _qaoa_instances(case, seed):
            x = torch.arange(2 ** i.n, device=_device())
            cut = torch.zeros(2 ** i.n, dtype=torch.float64, device=_device())
            for a, b in i.edges:
                cut += ((x >> a) ^ (x >> b)) & 1
            v = torch.full((2 ** i.n,), 2.0 ** (-i.n / 2), dtype=torch.complex128, device=_device())
            for g, b in zip(i.gammas, i.betas):
                v *= torch.exp(-0.5j * g * (len(i.edges) - 2 * cut))
                for q in range(i.n):
                    _apply(v, i.n, Gate("RX", (q,), (), (2 * b,)))
            out.append(float((v.abs().square() * cut).sum()))
        return {"cost": np.array(out)}
    x, y, w = (torch.from_numpy(a).double() for a in _mlp_data(case, seed))
    f, h = costmodel.N_FEATURES, case["hidden"]
    w.requires_grad_(True)
    w1, b1, w2, b2, w3, b3 = torch.split(w, [f * h, h, h * h, h, h, 1])
    a = torch.relu(x @ w1.view(f, h) + b1)
    a = torch.relu(a @ w2.view(h, h) + b2)
    out = a @ w3 + b3
    loss = ((out - y) ** 2).mean()
    loss.backward()
    return {"prediction": out.detach().numpy(), "loss": loss.item(), "gradient": w.grad.numpy()}
