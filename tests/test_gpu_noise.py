"""The mask generator of the persistent, frame and batch forms.

A lane draws for one noise op and 64, 32 or 16 shots of a word group, by the
number of (word group, op) pairs; a draw is decided by the upper half of its
mix function alone where no threshold of the wave is above 2^31.  Sizes: one
op, the edges of a wave's 64 pairs, and both sides of each change of the shots
per lane; probabilities: 0, 1, small ones, and both sides of 1/2."""
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


def noisy_ops(n, nk, seed, most):
    """nk noise ops and random flags between gates, measurements at the end."""
    from plaquette_simulator import workloads as W
    rng = np.random.default_rng(seed)
    probs = [p for p in (0.0, 0.001, 0.3, 0.5, 0.5000001, 0.8, 1.0) if p <= most]
    b = W.OpList()
    for i in range(nk):
        q = int(rng.integers(0, n))
        b.gate(int(rng.choice([W.OP_H, W.OP_S])), q)
        b.gate(W.OP_CX, q, (q + 1) % n)
        p = float(rng.choice(probs))
        if i % 3 == 2:
            b.with_prob(int(rng.choice([W.OP_X, W.OP_Y, W.OP_Z])), q, p)
        else:
            s = rng.dirichlet((1, 1, 1)) * p
            b.noise(q, float(s[0]), float(s[1]), float(s[2]))
    for q in range(n):
        b.measure(q)
    return b.array()


@pytest.mark.parametrize("nk,B", [(1, 1), (1, 4100), (63, 70), (64, 64), (65, 130),
                                  (200, 64 * 327), (200, 64 * 328), (200, 64 * 655),
                                  (200, 64 * 656), (331, 64 * 400 + 3)])
@pytest.mark.parametrize("most", [0.5, 1.0])
def test_masks_are_the_oracles(ps, nk, B, most):
    n, seed = 5, 1000 + nk
    sys.stderr.write(f"nk={nk} B={B} most={most}\n")
    sys.stderr.flush()
    ops = noisy_ops(n, nk, seed, most)
    orc = O.OracleState(n, B, seed)
    orc.run_program(ops.astype(np.int32))
    batch, states = ps.Batch(), []
    for form in ("persistent", "frame", "batch"):
        st = ps.CliffordState(n, B, seed, True)
        prog = ps.Program(st, ops)
        if form == "batch":
            other = ps.CliffordState(2, 64, 1, True)
            oprog = ps.Program(other, noisy_ops(2, 3, 7, 0.5))
            batch.add(other, oprog)
            batch.add(st, prog)
            batch.run("graph")
        else:
            prog.run(st, form)
        states.append((form, st, prog))
    for form, st, _ in states:
        st.sync_records()
        x, z, r = st.device_to_host_numpy()
        assert np.array_equal(x, orc.x) and np.array_equal(z, orc.z), form
        assert np.array_equal(r, orc.r), f"{form}: signs differ"
        for i, (res, det) in enumerate(orc.records):
            gres, gdet = st.get_record(i)
            assert np.array_equal(gres, res) and np.array_equal(gdet, det), f"{form}: record {i}"
