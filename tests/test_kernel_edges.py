"""Kernels and dispatch rules at the sizes where they can go wrong: tile edges,
remainders, the smallest and the largest of a rule's range. Each against the
restatements under oracle/ or plain numpy in 64 bits."""
import os

import numpy as np
import pytest

from oracle import mlp_ref


@pytest.mark.gpu
@pytest.mark.parametrize("in_features,hidden,n", [(1, 1, 1), (3, 17, 5), (14, 64, 32), (14, 64, 33), (16, 16, 31),
                                                  (15, 15, 64), (31, 48, 2051), (14, 200, 700), (5, 700, 40)])
def test_mlp_contractions_at_tile_edges(in_features, hidden, n):
    """Result tiles of 16, four samples per MFMA, slices of the samples (one,
    several, a short last one; one when the tiles alone fill the chip) against
    float64, at the bar of the network's other tests."""
    from hisvsim_amd.costmodel import MLP
    rng = np.random.default_rng(n)
    m = MLP(in_features, hidden, seed=3)
    p = m.params().astype(np.float64)
    X = rng.normal(size=(n, in_features)).astype(np.float32)
    y = rng.normal(size=n).astype(np.float32)
    want, _ = mlp_ref.forward(p, X, in_features, hidden)
    assert np.abs(m.predict(X) - want).max() <= 1e-4 * max(1.0, np.abs(want).max())
    loss, g = m.gradient(X, y)
    rl, rg = mlp_ref.loss_and_grad(p, X, y, in_features, hidden)
    assert abs(loss - rl) <= 1e-4 * rl
    assert np.abs(g - rg).max() <= 1e-4 * max(1.0, np.abs(rg).max())
    m.close()


def _stored(n, dtype, seed):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=2 ** n) + 1j * rng.normal(size=2 ** n)
    a /= np.linalg.norm(a)
    return a if dtype == "complex128" else a.astype(np.complex64).astype(complex)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 3, 9, 10, 11, 13, 20])
def test_read_outs_at_unit_and_grid_edges(n, dtype):
    """Norm, P(0) of every qubit and Pauli strings (no X, X on the lowest
    qubit alone, on the highest alone, random) where a state is less than a
    16-byte unit's block, one block, several. At most 64 roundings of partial
    sums below 1 in a row: 1e-14, and the sums in numpy as much again."""
    from hisvsim_amd import capi
    from oracle.oracle import pauli_expectation
    a = _stored(n, dtype, n)
    p = np.abs(a) ** 2
    i = np.arange(2 ** n)
    rng = np.random.default_rng(n + 50)
    full = 2 ** n - 1
    strings = [(0, 1), (0, full), (1, 0), (1, 1), (1, full), (1 << (n - 1), 0), (full, full)]
    strings += [(int(rng.integers(0, 2 ** n)), int(rng.integers(0, 2 ** n))) for _ in range(12)]
    with capi.State(n, dtype) as s:
        s.write(a)
        assert abs(s.norm2() - p.sum()) <= 1e-13
        for q in range(n):
            p0 = p[(i >> q) & 1 == 0].sum()
            assert abs(s.probability(q, 0) - p0) <= 1e-13
            assert abs(s.probability(q, 1) - (1 - p0)) <= 1e-13
        for x, z in strings:
            want = pauli_expectation(a, x, z)
            assert abs(s.expectation((x, z)) - want.real) <= 1e-13, (x, z)


def _walk_states():
    """(name, n, dtype, amplitudes) where the measurement walk's integer sums
    can go wrong: one wavefront's chunk and several, changes of binade at and
    inside chunks, exact ties, empty chunks, all mass in one amplitude."""
    out = []
    for n, dtype in ((14, "complex128"), (15, "complex128"), (15, "complex64"), (16, "complex128"),
                     (18, "complex64"), (20, "complex128")):
        out.append(("gaussian", n, dtype, _stored(n, dtype, n)))
    out.append(("uniform", 16, "complex128", np.full(2 ** 16, 2.0 ** -8, complex)))
    a = np.zeros(2 ** 15, complex)
    a[0], a[1:] = np.sqrt(0.5), 2.0 ** -27     # each |a|^2 half an ulp of the sum so far
    out.append(("ties", 15, "complex128", a))
    a = _stored(17, "complex128", 3)
    a[: 2 ** 15] = 0
    a[2 ** 16: 2 ** 16 + 2 ** 14] = 0
    out.append(("gaps", 17, "complex128", a))
    a = _stored(16, "complex128", 4) * 2.0 ** -12
    a[40000] = 1.0
    out.append(("peak", 16, "complex128", a))
    out.append(("large", 16, "complex128", _stored(16, "complex128", 5) * 3.0))   # norm^2 = 9
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name,n,dtype,a", _walk_states(), ids=lambda v: v if isinstance(v, str) else "")
def test_measurement_walk_is_the_serial_sum(name, n, dtype, a):
    """Uniforms on and just below the serial FP64 sum, in every chunk (so that
    every chunk with mass is walked and the sum is serial from 0): the outcome
    is the first amplitude whose sum exceeds the uniform, to the last bit."""
    from hisvsim_amd import capi
    p = a.real * a.real + a.imag * a.imag
    cum = np.cumsum(p)
    rng = np.random.default_rng(n)
    chunk = max(1, 2 ** n // 1024)
    at = (np.arange(0, 2 ** n, chunk)[:, None] + rng.integers(0, chunk, (2 ** n // chunk, 3))).ravel()
    edge = np.concatenate([np.arange(chunk - 1, 2 ** n, chunk), at])
    u = np.sort(np.concatenate([cum[edge], np.nextafter(cum[edge], 0.0), [0.0, -0.5, cum[-1] * 1.01]]))
    # a chunk without a uniform below its end would be passed by its mass
    want = np.searchsorted(cum, u, side="right")
    with capi.State(n, dtype) as s:
        s.write(a)
        got = s.measure(list(range(n)), u) @ (1 << np.arange(n))
    inside = want < 2 ** n
    assert np.array_equal(got[inside], want[inside])
    assert np.all(got[~inside] == 2 ** n - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(13, 512), (12, 256), (8, 128), (11, 512)])
def test_qaoa_passes_at_chunk_edges(orc, shape):
    """Instances of one chunk (whole in LDS, 13 qubits in registers), just
    wider (a high chunk over all but a few qubits), with every split of a
    13-qubit chunk into low and high qubits up to the widest the shape takes;
    no layer to four; angles on both sides of |cos b| = |sin b| (odd and even
    numbers of layers past it) and at 0, pi/2 and pi. <C> and the state
    against the CPU oracle: complex64 states, the bars of the batch's tests."""
    from hisvsim_amd.qaoa import Instance, QAOABatch, circuit, cut_values, random_3regular
    bits, threads = shape
    rng = np.random.default_rng(bits)
    insts = []
    for n in sorted({2, 3, 4, bits - 1, bits, bits + 1, bits + 2, bits + 4, min(bits + 6, 17), 13, 14}):
        edges = random_3regular(n, rng) if n >= 4 else [(0, n - 1)]
        for p in range(5):
            betas = [float(x) for x in rng.uniform(0, np.pi, p)]
            insts.append(Instance(n, edges, [float(x) for x in rng.uniform(0, np.pi, p)], betas))
        insts.append(Instance(n, edges, [0.3, 0.9, 1.7], [0.0, np.pi / 2, np.pi]))
    with QAOABatch(insts) as b:
        b.tune("chunk_bits", bits)
        b.tune("threads", threads)
        for _ in range(2):
            got = b.run()
        for i, inst in enumerate(insts):
            amps = np.zeros(2 ** inst.n, complex)
            amps[0] = 1
            orc.apply_gates(amps, circuit(inst))
            want = float(np.sum(np.abs(amps) ** 2 * cut_values(inst.n, inst.edges)))
            assert abs(got[i] - want) <= 1e-5 * max(1.0, abs(want)), (inst.n, inst.p)
            assert np.abs(b.state(i) - amps).max() <= 2e-6, (inst.n, inst.p)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n,qubits", [(12, (0,)), (12, (5, 7, 8, 9, 10, 11)), (12, (0, 1, 2, 3, 4, 5, 6)),
                                      (13, (0, 4, 8, 12)), (13, (1, 5, 9, 2, 12)), (14, (3, 7, 11, 12, 13)),
                                      (15, (8, 9, 10, 11, 12, 13, 14)), (16, (0, 2, 6, 10, 13, 14, 15))])
def test_fused_f64_steps_match_the_gates(n, qubits, dtype):
    """The FP64 fused path as 4-qubit steps on a tile (part qubits below, in
    and above the tile's low slots, all bank classes as rows, the smallest
    state), and where it stays one dense product (a gate on five qubits, more
    steps than the product is worth), against the gates one by one: 1e-12,
    complex64 states at their rounding of one pass, 2^-24 times the largest
    amplitude a few times over."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    rng = np.random.default_rng(n * 100 + len(qubits))
    a = _stored(n, dtype, 7)
    lists = []
    for count in (1, 4, 12, 40):
        gs = []
        for _ in range(count):
            q = [int(x) for x in rng.permutation(qubits)]
            th = [float(x) for x in rng.uniform(0, 6, 3)]
            gs.append(Gate("U3", (q[0],), (), tuple(th)))
            if len(q) > 1:
                gs += [Gate("Z", (q[1],), (q[0],)), Gate("R1", (q[0],), (q[1],), (th[0],)),
                       Gate("RZZ", (q[0], q[1]), (), (th[1],)), Gate("SWAP", (q[1], q[0]))]
            if len(q) > 3:
                gs.append(Gate("RY", (q[3],), (q[0], q[1], q[2]), (th[2],)))
        lists.append(gs)
    if len(qubits) > 4:
        lists.append(lists[1] + [Gate("X", (qubits[0],), tuple(qubits[1:5]))])
    tol = 1e-12 if dtype == "complex128" else 2.0 ** -20 * np.abs(a).max()
    with capi.State(n, dtype) as s, capi.State(n, "complex128") as r:
        for gs in lists:
            s.write(a)
            s.apply_fused(gs, "f64")
            r.write(a)
            r.apply_gates(gs)
            assert np.abs(s.read() - r.read()).max() <= tol


@pytest.mark.gpu
def test_fused_f64_unitarity_is_the_parts():
    """Accepted and refused as before: a gate that is not unitary followed by
    its inverse is a unitary part; alone it is none."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    n, m = 13, np.array([[2.0, 0.5], [0.25, 1.0]])
    g = Gate("C1", (3,), (), tuple(m.ravel()))
    inv = Gate("C1", (3,), (), tuple(np.linalg.inv(m).ravel()))
    far = [Gate("H", (q,)) for q in (3, 4, 5, 6, 7)]
    a = _stored(n, "complex128", 1)
    with capi.State(n) as s:
        s.write(a)
        s.apply_fused([g] + [inv], "f64")
        assert np.abs(s.read() - a).max() <= 1e-12
        with pytest.raises(capi.HsvError) as e:
            s.apply_fused([g] + far, "f64")
        assert e.value.code == -6
        with pytest.raises(capi.HsvError) as e:
            s.apply_fused([Gate("H", (q,)) for q in range(8)], "f64")
        assert e.value.code == -5


def _some_gates(rng, qubits, count):
    from hisvsim_amd.circuit import Gate
    gs = []
    for _ in range(count):
        q = [int(x) for x in rng.permutation(qubits)]
        th = [float(x) for x in rng.uniform(0, 6, 3)]
        gs.append(Gate("U3", (q[0],), (), tuple(th)))
        if len(q) > 1:
            gs += [Gate("X", (q[1],), (q[0],)), Gate("RZZ", (q[0], q[1]), (), (th[1],)), Gate("SWAP", (q[1], q[0]))]
    return gs


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(12))
def test_passes_skip_only_what_is_zero(seed):
    """From |0...0>, whatever acts in between on whatever qubits (gates, parts
    on each kernel, fused parts, chains, permutations, projections,
    renormalisations, reads, writes of a range, resets): the state equals the
    one of the same calls on a state that was written, where nothing is known
    to be zero. 1e-12 (the FP64 paths; the chain runs the same passes on
    both, so its rounding is the same or that of zeros)."""
    from hisvsim_amd import capi
    n, rng = 15, np.random.default_rng(seed)
    zero = np.zeros(2 ** n, complex)
    zero[0] = 1
    with capi.State(n) as a, capi.State(n) as b:
        for _ in range(14):
            b.write(b.read())        # forgets what b knows
            pick = [int(x) for x in rng.permutation(n)[:int(rng.integers(1, 6))]]
            op = rng.choice(["gates", "part", "reg", "lds", "f64", "f32split", "chain", "permute", "project",
                             "renormalize", "write", "reset", "measure"],
                            p=[.2, .15, .08, .07, .1, .06, .08, .1, .03, .03, .03, .04, .03])
            gs = _some_gates(rng, pick, int(rng.integers(1, 4)))
            perm = [int(x) for x in rng.permutation(n)]
            at = int(rng.integers(0, 2 ** n - 4))
            u = rng.random(5)
            for s in (a, b):
                s.tune("part_kernel", {"reg": 1, "lds": 0}.get(op, 2))
                if op == "gates":
                    s.apply_gates(gs)
                elif op in ("part", "reg", "lds"):
                    s.apply_part(gs, 0)
                elif op in ("f64", "f32split"):
                    s.apply_fused(gs, "f64")
                elif op == "chain":
                    s.apply_fused_chain([gs], [list(range(5))], "bf16x3")
                elif op == "permute":
                    s.permute_qubits(perm)
                elif op == "project":
                    q = pick[0]
                    s.project([q], [0 if s.probability(q, 0) > 0.4 else 1])
                elif op == "renormalize":
                    s.renormalize()
                elif op == "write":
                    s.write(np.full(3, 0.01 + 0.02j), at)
                elif op == "reset":
                    s.reset()
                else:
                    s.measure(list(range(n)), u)
            tol = 1e-12 if op != "chain" else 1e-6
            x, y = a.read(), b.read()
            assert np.abs(x - y).max() <= tol, op
            if op == "chain":        # past a chain both go on from the same amplitudes
                a.reset()
                b.reset()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("threads", [64, 256, 512])
def test_new_parameters_equal_a_new_batch(threads, dtype):
    """set_gates with plain new angles, with a phase that becomes and stops
    being a sign flip and with matrices that change their kind, on instances
    with tile plans and with LDS sweeps: bit for bit the states of a batch
    made with those gates."""
    from hisvsim_amd.batch import CircuitBatch, ansatz
    from hisvsim_amd.circuit import Gate
    sizes = [3, 6, 8, 10, 11, 12, 14]

    def gates(seed, phase, swap):
        rng = np.random.default_rng(seed)
        out = []
        for n in sizes:
            m = np.array([[0, 1], [1, 0]]) if swap else np.diag([1, np.exp(0.3j)])
            mid = [Gate("MATRIX", (1,), (), (1, 0, 0, complex(np.cos(phase), np.sin(phase)) if phase else -1.0)),
                   Gate("MATRIX", (n - 1,), (0,), tuple(complex(x) for x in m.ravel())),
                   Gate("RZZ", (0, n - 1), (), (float(rng.uniform(0, 6)),)), Gate("C1", (2,), (), (1, 0, 0, 1j))]
            out.append(ansatz(n, 2, rng.uniform(0, 6, 4 * n)) + mid + ansatz(n, 2, rng.uniform(0, 6, 4 * n)))
        return out

    first = gates(1, 0.7, False)
    with CircuitBatch(list(zip(sizes, first)), dtype) as b:
        b.tune("threads", threads)
        b.run()
        for seed, phase, swap in ((2, 0.9, False), (3, 0, False), (4, 0, True), (5, 1.1, True), (6, 0.2, False)):
            new = gates(seed, phase, swap)
            b.set_gates(new)
            b.run()
            with CircuitBatch(list(zip(sizes, new)), dtype) as c:
                c.tune("threads", threads)
                c.run()
                for i in range(len(sizes)):
                    assert np.array_equal(b.state(i), c.state(i)), (seed, sizes[i])


@pytest.mark.parametrize("gates", [
    [("X", (1,), (), ())], [("U3", (3,), (), (1.5, 2, np.float64(0.3)))], [("C1", (0,), (1, 2), (1j, 2, 3.5, 1 + 2j))],
    [("RXFRAC", (2,), (), (3, 4))], [("MATRIX", (0, 1), (), tuple(range(16)))], [("H", [4], [True], [])],
    [("x", (1,), (2,), ())], [("RZ", (np.int64(1),), (), (0.5,))], [("RX", (1,), (), (np.complex64(1),))], []])
def test_native_gate_records_equal_the_python_ones(gates):
    """capi.gate_array (native where the list is plain, Python where not),
    also into a used array, against to_hsv_gate."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    gs = [Gate(*g) for g in gates]
    used = capi.gate_array([Gate("C1", (9,), (7, 8), (1j, 2j, 3j, 4j))] * 3)
    for arr in (capi.gate_array(gs), capi.gate_array(tuple(gs), used)):
        for g, d in zip(gs, arr):
            assert bytes(d) == bytes(capi.to_hsv_gate(g))


@pytest.mark.parametrize("gate", [("NOTAGATE", (0,), (), ()), ("X", tuple(range(6)), (), ()), ("X", ("a",), (), ()),
                                  ("RXFRAC", (0,), (), (1j, 2)), ("U3", (0,), (), tuple(range(17)))])
def test_native_gate_records_refuse_what_python_refuses(gate):
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    with pytest.raises(Exception) as want:
        capi.to_hsv_gate(Gate(*gate))
    with pytest.raises(type(want.value)):
        capi.gate_array([Gate("X", (0,)), Gate(*gate)])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 5, 9, 12, 13, 14])
def test_gate_lists_equal_the_gates_one_by_one(n, dtype):
    """Lists below and above the length that takes one launch, longer than
    the kernel's chunk of records, on states below, at and beyond a
    workgroup's LDS, from |0...0> (qubits untouched so far above the touched
    ones) and from a written state: the same bits as gate by gate."""
    from hisvsim_amd import capi
    rng = np.random.default_rng(n)
    a = _stored(n, dtype, n)
    low = list(range(max(1, n - 2)))
    with capi.State(n, dtype) as s, capi.State(n, dtype) as r:
        for qubits, count, start in ((low, 1, None), (low, 30, None), (list(range(n)), 2, a), (list(range(n)), 40, a)):
            gs = _some_gates(rng, qubits, count)
            for x in (s, r):
                x.reset()
                if start is not None:
                    x.write(start)
            s.apply_gates(gs)
            for g in gs:
                r.apply_gate(g)
            assert np.array_equal(s.read(), r.read())


@pytest.mark.gpu
def test_gate_list_stops_at_the_gate_that_fails():
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    gs = [Gate("H", (q,)) for q in range(5)] + [Gate("I", (2,)), Gate("X", (1,), (1,)), Gate("H", (0,))]
    with capi.State(6) as s, capi.State(6) as r:
        for bad in (gs, gs[:6] + [Gate("X", (6,))] + gs[:3]):
            s.reset()
            r.reset()
            r.apply_gates(gs[:5])
            before = capi.counters()["gates"]
            with pytest.raises(capi.HsvError) as e:
                s.apply_gates(bad)
            assert e.value.code == -1
            assert capi.counters()["gates"] == before + 6
            assert np.array_equal(s.read(), r.read())


@pytest.mark.gpu
@pytest.mark.parametrize("circuit,n,k,reps", [("layered", 13, 12, 1), ("layered", 16, 13, 1), ("layered", 20, 14, 1),
                                              ("qft", 14, 13, 1), ("qft", 18, 12, 2), ("one", 14, 13, 3),
                                              ("one", 14, 13, 6), ("one", 14, 13, 12)])
def test_device_step_groups_equal_the_hosts(circuit, n, k, reps):
    """The chain, whose parts' steps are searched on the device, against its
    no-allocation form, whose steps the host searches: the same steps give the
    same bits. Parts of a few gates, of more than 64, of 128 and more (left to
    the host), layout changes between parts."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate, qft, random_layered
    rng = np.random.default_rng(n)
    if circuit == "layered":
        gs = random_layered(n, 5, n)
    elif circuit == "qft":
        gs = [Gate("U3", (q,), (), (0.3 + q, 0.2, 0.9)) for q in range(n)] + qft(n) * reps
    else:  # one part on 13 of the qubits
        gs = _some_gates(rng, list(range(13)), 9 * reps) + [Gate("RZZ", (0, q), (), (0.1 * q,)) for q in range(1, 13)]
    if circuit == "one":
        parts, lows = [gs], [list(range(5))]
    else:
        parts, lows = capi.chain_parts(gs, k, 5, 13, beam=(4, 4))
    a = _stored(n, "complex128", 2)
    with capi.State(n) as s, capi.State(n) as r:
        for start in (None, a):
            for x in (s, r):
                x.reset()
                if start is not None:
                    x.write(start)
            try:
                r.apply_fused_chain(parts, lows, "bf16split", noalloc=True)
            except capi.HsvError as e:      # more than 28 steps: not for that form's scratch
                assert e.code == -5
                s.apply_fused_chain(parts, lows, "bf16split")
                continue
            s.apply_fused_chain(parts, lows, "bf16split")
            assert np.array_equal(s.read(), r.read())


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["bf16split", "bf16x3"])
@pytest.mark.parametrize("count,bad", [(1, None), (16, None), (17, None), (33, None), (33, 0), (33, 20)])
def test_chain_parts_checked_ahead_equal_the_hosts(mode, count, bad):
    """Parts prepared several at a time on the device against the no-allocation
    form, whose parts are prepared one by one on the host: the same bits, also
    of what ran before a part with a matrix that is not unitary."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    n, rng = 16, np.random.default_rng(count)
    parts, lows = [], [list(range(5))]
    for p in range(count):
        qs = sorted(set(lows[p]) | set(int(q) for q in rng.permutation(n)[:6]))
        part = _some_gates(rng, qs, 12) + [Gate("H", (q,), (), ()) for q in qs]
        if p == bad:
            part.append(Gate("C2", (qs[0], qs[1]), (), tuple(complex(x) for x in rng.standard_normal(16))))
        parts.append(part)
        lows.append(sorted(int(q) for q in rng.permutation(qs)[:5]))
    a = _stored(n, "complex128", 2)
    with capi.State(n) as s, capi.State(n) as r:
        codes = []
        for x, noalloc in ((s, False), (r, True)):
            x.write(a)
            try:
                x.apply_fused_chain(parts, lows[:count], mode, noalloc=noalloc)
                codes.append(0)
            except capi.HsvError as e:
                codes.append((e.code, str(e).split(" (max")[0]))
        assert codes[0] == codes[1]
        assert codes[0] == 0 if bad is None else codes[0][0] == -6
        assert np.array_equal(s.read(), r.read())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 9, 10, 11, 12, 17])
def test_reset_fills_every_amplitude(n, dtype):
    """States below, at and above one run of the fill."""
    from hisvsim_amd import capi
    with capi.State(n, dtype) as s:
        s.write(_stored(n, dtype, 3))
        s.reset()
        a = s.read()
    assert a[0] == 1 and not a[1:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["bf16split", "bf16x3"])
@pytest.mark.parametrize("n,k", [(13, 9), (16, 12), (24, 12)])
def test_wide_parts_prepared_on_an_idle_stream(mode, n, k):
    """A wide part prepared on the device (nothing queued before it) and on
    the host (behind earlier work): the same bits; a matrix that is not unitary
    is refused either way."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    rng = np.random.default_rng(n)
    parts = [_some_gates(rng, sorted({int(q) for q in rng.permutation(n)[:k - 3]} | {0, 1, 2}), 3 * k) for _ in range(3)]
    bad = parts[0] + [Gate("C2", (0, 1), (), tuple(complex(x) for x in rng.standard_normal(16)))]
    a = _stored(n, "complex128", 2)
    with capi.State(n) as s, capi.State(n) as r:
        s.write(a)
        r.write(a)
        for p in parts:
            s.synchronize()
            s.apply_fused(p, mode)
        for _ in range(20):  # work to queue behind
            r.apply_gate(Gate("X", (n - 1,)))
        for p in parts:
            r.apply_fused(p, mode)
        assert np.array_equal(s.read(), r.read())
        for _ in range(2):
            with pytest.raises(capi.HsvError) as e:
                s.apply_fused(bad, mode)
            assert e.value.code == -6
            s.apply_gate(Gate("X", (0,)))


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["gates", "part", "reg", "lds", "f64", "f64dense", "f32split", "bf16split", "bf16col",
                                  "bf16wide", "bf16x3", "chain", "chain3"])
def test_matrices_that_are_not_finite_reach_the_whole_state(path):
    """A gate with a NaN entry on a state whose other qubits are still |0>:
    its products with those zeros are NaN, so the NaNs are where the same call
    leaves them on a state that was written (nothing known to be zero); and so
    after one more gate on an untouched qubit."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    n, nan = 15, float("nan")
    first = [Gate("H", (1,)), Gate("X", (6,), (1,))]
    bad = [Gate("H", (2,)), Gate("C1", (5,), (), (1, 0, 0, nan)), Gate("RZZ", (2, 5), (), (0.3,)), Gate("H", (8,))]
    if path == "f64dense":
        bad.append(Gate("X", (0,), (1, 2, 3, 4)))
    if path in ("bf16wide", "bf16x3", "chain", "chain3"):
        bad += [Gate("H", (q,)) for q in (0, 1, 3, 4, 7, 9)]
    with capi.State(n) as a, capi.State(n) as b:
        for s in (a, b):
            s.apply_gates(first)
        b.write(b.read())
        for s in (a, b):
            s.tune("part_kernel", {"reg": 1, "lds": 0}.get(path, 2))
            if path == "bf16col":
                s.tune("fused_variant", 1)
            if path == "gates":
                s.apply_gates(bad)
            elif path in ("part", "reg", "lds"):
                s.apply_part(bad, 0)
            elif path in ("chain", "chain3"):
                s.apply_fused_chain([bad, [Gate("H", (10,))]], [list(range(5))] * 2,
                                    "bf16x3" if path == "chain3" else "bf16split")
            else:
                s.apply_fused(bad, {"f64dense": "f64", "bf16col": "bf16split", "bf16wide": "bf16split"}.get(path, path))
            s.apply_gate(Gate("H", (13,)))
        x, y = a.read(), b.read()
    assert np.isnan(y).any()
    assert np.array_equal(np.isnan(x.real), np.isnan(y.real)) and np.array_equal(np.isnan(x.imag), np.isnan(y.imag))
    ok = ~np.isnan(y.real) & ~np.isnan(y.imag)
    assert np.abs(x[ok] - y[ok]).max(initial=0.0) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_pauli_sums_that_are_not_finite_have_no_zero_part(value, dtype):
    """<P> of a state with a NaN or an infinity: neither part is a number;
    the imaginary part of a finite state's is 0."""
    import ctypes
    from hisvsim_amd import capi
    n = 13
    a = _stored(n, dtype, 3)
    out = (ctypes.c_double * 2)()
    with capi.State(n, dtype) as s:
        for state, finite in ((a, True), (np.where(np.arange(2 ** n) == 1234, value, a), False)):
            s.write(state)
            for x, z in ((0, 3), (1, 0), (1, 1), (1 << (n - 1), 5), (6, 6)):
                capi._check(capi.lib().hsv_expect_pauli(s.handle, x, z, out))
                assert np.isfinite(out[0]) == finite
                assert out[1] == 0 if finite else np.isnan(out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n", [("complex128", 21), ("complex64", 22)])
def test_read_outs_keep_what_each_workgroup_adds(dtype, n):
    """One amplitude with all but 1.8e-13 of the mass, the rest spread over the
    workgroups in pieces below half an ulp of 1: a sum of the workgroups'
    partials one after another drops them all. At most 2 roundings per level of
    the sums (a thread's items, lanes, waves, workgroups: 32 levels) of 2^-53."""
    from hisvsim_amd import capi
    a = np.zeros(2 ** n, complex)
    a[0] = 1.0
    a[256:2 ** 19:256] = np.sqrt(0.9e-16)
    a = a if dtype == "complex128" else a.astype(np.complex64).astype(complex)
    p = np.abs(a) ** 2
    rest = p[1:].sum()
    tol = 32 * 2.0 ** -53
    top = 1 << (n - 1)
    with capi.State(n, dtype) as s:
        s.write(a)
        assert abs((s.norm2() - 1.0) - rest) <= tol
        assert abs((s.probability(n - 1, 0) - 1.0) - rest) <= tol
        assert abs((s.expectation((0, top)) - 1.0) - rest) <= tol


def test_gate_records_leave_the_module_path_alone():
    """Building gate records neither adds the package's folder to sys.path
    (its module names would hide a program's own) nor takes another module of
    the pybind module's name for it."""
    import subprocess
    import sys
    code = """
import sys, types
path = list(sys.path)
if {other}:
    sys.modules["svsimulator_py_wrapper"] = types.ModuleType("svsimulator_py_wrapper")
from hisvsim_amd import capi
from hisvsim_amd.circuit import Gate
arr = capi.gate_array([Gate("H", (3,))])
assert bytes(arr[0]) == bytes(capi.to_hsv_gate(Gate("H", (3,))))
assert sys.path == path, sys.path
import hisvsim_amd
if not {other}:
    assert hisvsim_amd.load_module()._fill_gates
"""
    for other in (False, True):
        subprocess.run([sys.executable, "-c", code.format(other=other)], check=True, timeout=300,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.gpu
def test_chain_behind_queued_work_does_not_wait_for_it():
    """A chain on a handle with 100 sweeps over 2 GB queued (some 70 ms) is
    queued behind them: the call returns in less than half of the time that
    all of it takes, with the same bits as on an idle handle."""
    import time

    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate, random_layered
    n = 27
    parts, lows = capi.chain_parts(random_layered(n, 2, 5), 13, 5, 13)
    sweeps = [Gate("H", (q % n,)) for q in range(100)]
    with capi.State(n) as s, capi.State(n) as r:
        for x in (s, r):
            x.write(np.array([0.6, 0.8j, 0, 0]))
            x.apply_fused_chain(parts, lows)   # code objects and scratch
            x.synchronize()
        for x in (s, r):
            t0 = time.perf_counter()
            x.apply_gates(sweeps)
            if x is r:
                x.synchronize()
            x.apply_fused_chain(parts, lows)
            called = time.perf_counter() - t0
            x.synchronize()
            total = time.perf_counter() - t0
            if x is s:
                assert called < 0.5 * total, (called, total)
        assert s.max_abs_diff(r) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 11, 13, 14, 15, 24, 25])
def test_few_shots_walk_the_serial_sum(n, dtype):
    """One shot and three, walked on the host: in the state fetched whole (up to
    14 qubits), in a chunk fetched (up to 24) or found on the device: the
    outcomes of the reference's walk, which passes the other chunks by their
    masses (a uniform in the middle of an amplitude's share, so that the
    masses' own rounding does not matter)."""
    from hisvsim_amd import capi
    a = _stored(n, dtype, n)
    p = a.real * a.real + a.imag * a.imag
    cum = np.cumsum(p)
    rng = np.random.default_rng(n)
    with capi.State(n, dtype) as s:
        s.write(a)
        for shots in (1, 3):
            at = np.sort(rng.choice(np.flatnonzero(p > 0.3 * 2.0 ** -n), shots))
            got = s.measure(list(range(n)), cum[at] - p[at] / 2) @ (1 << np.arange(n))
            assert np.array_equal(got, at)


@pytest.mark.gpu
@pytest.mark.parametrize("n,dtype", [(21, "complex128"), (22, "complex128"), (23, "complex128"), (22, "complex64"),
                                     (23, "complex64"), (24, "complex64")])
def test_read_outs_where_the_groups_grow(n, dtype):
    """States around the sizes from which a thread sums eight items at a time
    instead of four: norm, P(0) and strings with X on the lowest, a middle and
    the highest qubit against numpy; 2^-53 per level of the sums, 40 of them,
    and as much again in numpy's."""
    from hisvsim_amd import capi
    from oracle.oracle import pauli_expectation
    a = _stored(n, dtype, n)
    p = np.abs(a) ** 2
    with capi.State(n, dtype) as s:
        s.write(a)
        assert abs(s.norm2() - p.sum()) <= 1e-14
        for q in (0, 1, n // 2, n - 1):
            assert abs(s.probability(q, 0) - p.reshape(-1, 2, 2 ** q)[:, 0].sum()) <= 1e-14
        for x, z in ((0, 5), (1, 0), (1 << (n // 2), 3), (1 << (n - 1), 1 << (n - 1)), (3, 2 ** n - 1)):
            assert abs(s.expectation((x, z)) - pauli_expectation(a, x, z).real) <= 1e-14, (x, z)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(12, 128), (10, 128), (13, 256), (12, 256), (13, 512)])
def test_qaoa_high_chunks_of_every_width(shape):
    """High chunks from one high qubit to as many as leave the fewest low ones,
    narrower than, as wide as and wider than 16 amplitudes a thread: one layer
    against the closed form, at the bar of the batch's tests."""
    from hisvsim_amd.qaoa import Instance, QAOABatch, expectation_p1, random_3regular
    bits, threads = shape
    rng = np.random.default_rng(bits + threads)
    insts = [Instance(n, random_3regular(n, rng), [float(rng.uniform(0, np.pi))], [float(rng.uniform(0, np.pi))])
             for n in range(bits, min(bits + 10, 22) + 1)]
    with QAOABatch(insts) as b:
        b.tune("chunk_bits", bits)
        b.tune("threads", threads)
        got = b.run()
    for i, inst in enumerate(insts):
        want = expectation_p1(inst.n, inst.edges, inst.gammas[0], inst.betas[0])
        assert abs(got[i] - want) <= 1e-5 * max(1.0, abs(want)), inst.n


def _busy_part(rng, qubits, steps):
    """Random gates on the qubits, more than `steps` steps of 4 qubits."""
    from hisvsim_amd import capi
    gs = []
    while len(capi.part_steps(gs, 4, 16)) <= steps if gs else True:
        gs += _some_gates(rng, qubits, 6)
    return gs


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n,k,why", [(8, 4, "small"), (9, 5, "small"), (10, 6, "small"), (11, 7, "small"),
                                     (12, 5, "five"), (14, 6, "five"), (16, 7, "five"),
                                     (13, 5, "steps"), (15, 6, "steps"), (17, 7, "steps")])
def test_fused_f32split_dense_product(n, k, why, dtype):
    """The FP32-split product where the FP64 steps do not take the part (a
    state below a tile, a gate on five qubits, more steps than are worth it:
    1.5 * 2^(k - 4), at most 8), from a written state and from |0...0> with a
    few qubits touched, against the gates one by one. Each real product is
    accumulated in FP32 over 3 * 2^k terms of at most the state's norm: error
    below 1e-6, and on a complex128 state above 1e-12, where FP64 steps would
    be."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    rng = np.random.default_rng(100 * n + k)
    limit = min(8, (3 << (k - 4)) >> 1)
    with capi.State(n, dtype) as s, capi.State(n) as r:
        for start in (None, _stored(n, dtype, n)):
            for _ in range(3):
                qubits = [int(q) for q in rng.permutation(n)[:k]]
                if why == "steps":
                    gs = _busy_part(rng, qubits, limit)
                else:
                    gs = [Gate("H", (q,)) for q in qubits] + _some_gates(rng, qubits, 6)
                if why == "five":
                    gs.append(Gate("RX", (qubits[0],), tuple(qubits[1:5]), (0.7,)))
                for x in (s, r):
                    x.reset()
                    if start is not None:
                        x.write(start)
                    x.apply_gates([Gate("H", (1,)), Gate("RY", (n - 1,), (1,), (0.8,))])
                s.apply_fused(gs, "f32split")
                r.apply_gates(gs)
                err = np.abs(s.read() - r.read()).max()
                assert err <= 1e-6
                if dtype == "complex128":
                    assert err >= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("seed", range(10))
def test_every_kernel_skips_only_what_is_zero(seed, dtype):
    """Gates, parts on each kernel, fused parts of each precision as steps and
    as one product, both forms of small BF16 parts, wide BF16 parts and chains
    of several parts, one after another from |0...0>: the same numbers as on a
    state that is written before each call, where nothing is known to be zero.
    The tiles that are not skipped run the same arithmetic, but for the
    three-piece split, whose column signs are hashed from a tile's number in
    the launch: there to its bar, 1e-6 (and on from the same amplitudes)."""
    from hisvsim_amd import capi
    n, rng = 17, np.random.default_rng([seed, 5])
    ops = ["gates", "part", "reg", "lds", "f64", "f32split", "f64dense", "f32dense", "bf16tile", "bf16col", "bf16rows",
           "bf16wide", "bf16x3", "chain", "chain3", "permute", "reset"]
    weight = np.array([2, 2, 1, 1, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 1, 1.5])
    with capi.State(n, dtype) as a, capi.State(n, dtype) as b:
        for _ in range(16):
            b.write(b.read())        # forgets what b knows
            op = str(rng.choice(ops, p=weight / weight.sum()))
            wide = op in ("bf16wide", "bf16x3")
            k = int(rng.integers(8, 12)) if wide else int(rng.integers(5, 8))
            pick = [int(x) for x in rng.permutation(n)[:k]]
            if wide:
                pick = sorted(set(pick) | set(range(5)))[:12]
            if op in ("gates", "part", "reg", "lds"):
                pick = pick[:int(rng.integers(1, 6))]
            if op in ("f64dense", "f32dense"):
                gs = _busy_part(rng, pick, min(8, (3 << (k - 4)) >> 1))
            elif op in ("chain", "chain3"):
                gs = [g for _ in range(3) for g in _some_gates(rng, [int(x) for x in rng.permutation(n)[:6]], 5)]
                parts, lows = capi.chain_parts(gs, 12, 5, 7)
            else:
                gs = _some_gates(rng, pick, int(rng.integers(1, 4)))
            perm = [int(x) for x in rng.permutation(n)]
            for s in (a, b):
                s.tune("part_kernel", {"reg": 1, "lds": 0}.get(op, 2))
                s.tune("fused_variant", {"bf16col": 1, "bf16rows": 0}.get(op, 2))
                if op == "gates":
                    s.apply_gates(gs)
                elif op in ("part", "reg", "lds"):
                    s.apply_part(gs, 0)
                elif op in ("chain", "chain3"):
                    s.apply_fused_chain(parts, lows, "bf16x3" if op == "chain3" else "bf16split")
                elif op == "permute":
                    s.permute_qubits(perm)
                elif op == "reset":
                    s.reset()
                else:
                    mode = {"f64dense": "f64", "f32dense": "f32split"}.get(op, op)
                    s.apply_fused(gs, mode if mode in ("f64", "f32split", "bf16x3") else "bf16split")
            x, y = a.read(), b.read()
            if op in ("bf16x3", "chain3"):
                assert np.abs(x - y).max() <= 1e-6, op
                b.write(x)
            else:
                assert np.array_equal(x, y), op


@pytest.mark.gpu
@pytest.mark.parametrize("n", [11, 12, 16])
def test_fused_steps_says_which_arithmetic_runs(n):
    """capi.fused_steps, which the benchmark and the cost model price fused
    parts by, against what ran: an FP32-split part leaves an error of FP32's
    size exactly where the rule says that it is one dense product."""
    from hisvsim_amd import capi
    from hisvsim_amd.circuit import Gate
    rng = np.random.default_rng(n)
    a = _stored(n, "complex128", 3)
    seen = set()
    with capi.State(n) as s, capi.State(n) as r:
        for k in (2, 4, 5, 6, 7):
            for count in (1, 3, 8, 20):
                qubits = [int(q) for q in rng.permutation(n)[:k]]
                gs = _some_gates(rng, qubits, count) + [Gate("H", (q,)) for q in qubits] + [Gate("I", (qubits[0],))]
                for x in (s, r):
                    x.write(a)
                s.apply_fused(gs, "f32split")
                r.apply_gates(gs)
                dense = capi.fused_steps(gs, n, True) is None
                seen.add(dense)
                assert (np.abs(s.read() - r.read()).max() >= 1e-12) == dense, (k, count)
    assert seen == ({True} if n < 12 else {True, False})
