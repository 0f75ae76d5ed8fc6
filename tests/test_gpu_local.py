"""Per-shot persistent runs of small states, their tableau in LDS.

Programs with flagged H/S/CX/CZ, and second runs that start from what the first
left, have X/Z and pivots of their own in every shot.  Sizes: one and two
qubits, the edges of a 64-row word, the last size that fits and the first that
does not; staging windows that cut a program; few and many measurements, in
runs and alone."""
import sys

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ps():
    import plaquette_simulator as ps
    import plaquette_simulator_bindings as b
    if b.device_count() < 1:
        pytest.skip("no GPU")
    return ps


def conditional_ops(n, nops, seed, meas):
    """Every op: gates, flags from records and random flags on all of them,
    noise, measurements into new and existing records."""
    from plaquette_simulator import workloads as W
    rng = np.random.default_rng(seed)
    b = W.OpList()
    one = [W.OP_H, W.OP_S, W.OP_X, W.OP_Y, W.OP_Z]
    two = [W.OP_CX, W.OP_CZ] if n > 1 else []
    b.gate(W.OP_H, 0)
    for _ in range(nops):
        q = int(rng.integers(0, n))
        t = (q + 1 + int(rng.integers(0, max(1, n - 1)))) % n
        code = int(rng.choice(one + two + two))
        q1 = t if code in two else 0
        u = rng.random()
        if u < meas:
            again = b.nrec > 3 and rng.random() < 0.2
            b.measure(q, float(rng.choice([0.5, 0.5, 0.2])),
                      int(rng.integers(0, b.nrec)) if again else None)
        elif u < meas + 0.1:
            b.with_prob(code, q, float(rng.choice([0.1, 0.5])), q1)
        elif u < meas + 0.2 and b.nrec:
            b.flagged(W.FLAGGED[code], q, int(rng.integers(0, b.nrec)), q1)
        elif u < meas + 0.25:
            b.noise(q, 0.05, 0.03, 0.04)
        else:
            b.gate(code, q, q1)
    return b.array()


@pytest.mark.parametrize("n,B,nops,meas", [
    (1, 64, 40, 0.3), (2, 65, 80, 0.2), (3, 1, 60, 0.6), (31, 130, 400, 0.1),
    (32, 64, 300, 0.5), (33, 200, 900, 0.05), (41, 321, 800, 0.05), (63, 70, 1200, 0.1),
    (64, 129, 1500, 0.1), (64, 64, 200, 0.9), (65, 70, 400, 0.1)])
@pytest.mark.parametrize("form", ["persistent", "graph"])
def test_local_equals_oracle(ps, n, B, nops, meas, form):
    seed = 31 * n + B
    sys.stderr.write(f"n={n} B={B} nops={nops} meas={meas} {form}\n")
    sys.stderr.flush()
    ops = conditional_ops(n, nops, seed, meas)
    orc = O.OracleState(n, B, seed)
    st = ps.CliffordState(n, B, seed, True)
    prog = ps.Program(st, ops)
    for run in range(2):  # from |0...0>, then from what that left
        orc.run_program(ops.astype(np.int32))
        prog.run(st, form)
        st.sync_records()
        x, z, r = st.device_to_host_numpy()
        assert np.array_equal(x, orc.x), f"run {run}: x differs"
        assert np.array_equal(z, orc.z), f"run {run}: z differs"
        assert np.array_equal(r, orc.r), f"run {run}: r differs"
        for i, (res, det) in enumerate(orc.records):
            gres, gdet = st.get_record(i)
            assert np.array_equal(gdet, det), f"run {run}: record {i} determined differ"
            assert np.array_equal(gres, res), f"run {run}: record {i} results differ"
    st.reset_clifford_state()  # X/Z pending: the run writes them itself
    prog.run(st, form)
    x, _, _ = st.device_to_host_numpy()
    other = ps.CliffordState(n, B, seed, True)
    prog2 = ps.Program(other, ops)
    prog2.set_slices(1)  # keeps the kernel that works in memory
    prog2.run(other, "persistent")
    for _ in range(2):
        other.reset_clifford_state()
        prog2.run(other, "persistent")
    assert np.array_equal(x, other.device_to_host_numpy()[0])
