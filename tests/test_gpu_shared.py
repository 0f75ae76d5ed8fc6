"""Programs run on the packed tableau that all shots share.

A program without flagged H/S/CX/CZ on the |0...0> tableau runs in the
shared-X/Z kernel; a program whose slice count was set keeps the per-shot
kernel.  Both must leave the oracle's words and records.  Sizes: one and two
qubits, the edges of a 64-row word, the last size whose packed columns fit the
LDS and the first that keeps them in the tableau, and the largest size taken
with the first refused."""
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


def say(msg):
    sys.stderr.write(msg + "\n")
    sys.stderr.flush()


def mixed_ops(n, nops, seed, meas, two=True):
    """Every op the shared form takes: gates, Paulis, noise, flags from records
    and random flags on Paulis, measurements into new and existing records."""
    from plaquette_simulator import workloads as W
    rng = np.random.default_rng(seed)
    b = W.OpList()
    for _ in range(nops):
        q = int(rng.integers(0, n))
        t = (q + 1 + int(rng.integers(0, max(1, n - 1)))) % n
        u = rng.random()
        if u < meas:
            again = b.nrec > 3 and rng.random() < 0.2
            b.measure(q, 0.5, int(rng.integers(0, b.nrec)) if again else None)
        elif u < meas + 0.1:
            b.noise(q, 0.05, 0.03, 0.04)
        elif u < meas + 0.15 and b.nrec:
            b.flagged(int(rng.choice([W.OP_X_FLAG, W.OP_Y_FLAG, W.OP_Z_FLAG])), q,
                      int(rng.integers(0, b.nrec)))
        elif u < meas + 0.2:
            b.with_prob(int(rng.choice([W.OP_X, W.OP_Y, W.OP_Z])), q, 0.3)
        else:
            codes = [W.OP_H, W.OP_S, W.OP_X, W.OP_Y, W.OP_Z]
            if n > 1:
                codes += [W.OP_CX, W.OP_CX, W.OP_CZ]
            code = int(rng.choice(codes))
            b.gate(code, q, t if code in (W.OP_CX, W.OP_CZ) else 0)
    return b.array()


def check(st, orc):
    st.sync_records()
    x, z, r = st.device_to_host_numpy()
    assert np.array_equal(x, orc.x), "x differs"
    assert np.array_equal(z, orc.z), "z differs"
    assert np.array_equal(r, orc.r), "r differs"
    assert st.num_records == len(orc.records)
    for i, (res, det) in enumerate(orc.records):
        gres, gdet = st.get_record(i)
        assert np.array_equal(gres, res), f"record {i} results differ"
        assert np.array_equal(gdet, det), f"record {i} determined differ"


@pytest.mark.parametrize("n,B,nops,meas", [
    (1, 130, 60, 0.2), (2, 64, 80, 0.2), (3, 1, 80, 0.3),
    (63, 65, 900, 0.1), (64, 65, 900, 0.1), (65, 65, 900, 0.1),
    (128, 64, 1500, 0.05), (129, 70, 1500, 0.05),
    (464, 3, 1600, 0.05), (465, 3, 1600, 0.05), (513, 3, 1600, 0.04),
    (700, 3, 1500, 0.03), (2048, 1, 2400, 0.01), (2049, 1, 2400, 0.01),
    # two and four word groups per workgroup, the last one short
    (20, 8193, 300, 0.1), (20, 16385, 300, 0.1), (500, 323, 900, 0.03),
])
def test_shared_equals_oracle(ps, n, B, nops, meas):
    ops = mixed_ops(n, nops, 10 * n + B, meas)
    say(f"[case] n={n} B={B} ops={len(ops)}")
    orc = O.OracleState(n, B, 17)
    orc.run_program(ops.astype(np.int32))
    st = ps.CliffordState(n, B, 17, True)
    ps.Program(st, ops).run(st, "persistent")
    check(st, orc)


@pytest.mark.parametrize("n", [30, 500])
def test_scratch_row_of_mixed_runs(ps, n):
    """The scratch row keeps the last determined measurement of a run, also where
    random ones follow it."""
    from plaquette_simulator import workloads as W
    b = W.OpList()
    for r in range(4):
        for q in range(n):
            b.cx(q, (q + 1 + r) % n)
        b.h(5 + r)
        b.cx(5 + r, 9 + r)
        for q in (0, 1 + r, 9 + r, 3, 5 + r, 9 + r, 12 + r)[:4 + r]:
            b.measure(q)
    ops = b.array()
    say(f"[case] n={n} determined before random")
    for cut in (len(ops), len(ops) - 2):
        orc = O.OracleState(n, 3, 5)
        orc.run_program(ops[:cut].astype(np.int32))
        st = ps.CliffordState(n, 3, 5, True)
        ps.Program(st, ops[:cut]).run(st, "persistent")
        check(st, orc)


@pytest.mark.parametrize("n", [487, 488])
def test_programs_without_masks(ps, n):
    # no noise, no flags: no mask area in LDS, so the packed columns fit longer
    from plaquette_simulator import workloads as W
    ops = W.random_clifford(n, 1500, n, meas_prob=0.05)
    say(f"[case] n={n} without masks")
    orc = O.OracleState(n, 3, 5)
    orc.run_program(ops.astype(np.int32))
    st = ps.CliffordState(n, 3, 5, True)
    ps.Program(st, ops).run(st, "persistent")
    check(st, orc)


@pytest.mark.parametrize("n,B", [(65, 200), (500, 70)])
def test_per_shot_kernel_is_still_reached(ps, n, B):
    # the same program in both kernels, and each again from the state it left
    ops = mixed_ops(n, 3 * n, 5, 0.05)
    a, b = (ps.CliffordState(n, B, 3, True) for _ in range(2))
    pa, pb = ps.Program(a, ops), ps.Program(b, ops)
    pb.set_slices(1)
    for i in range(2):
        say(f"[case] n={n} B={B} run {i}")
        pa.run(a, "persistent")
        pb.run(b, "persistent")
        assert a.compare(b) == (0, 0)


def test_graph_replays_from_any_state(ps):
    n, B = 40, 150
    ops = mixed_ops(n, 500, 8, 0.1)
    st, ref = (ps.CliffordState(n, B, 9, True) for _ in range(2))
    prog, pref = ps.Program(st, ops), ps.Program(ref, ops)
    pref.set_slices(1)
    for i, reset in enumerate([False, False, True, False, True]):
        say(f"[case] graph replay {i} reset={reset}")
        if reset:
            st.reset_clifford_state()
            ref.reset_clifford_state()
        prog.run(st, "graph")
        pref.run(ref, "persistent")
        assert st.compare(ref) == (0, 0)


_RAW_POINTER = """
import sys
import torch  # first: its HIP runtime must be the one the process loads
assert torch.cuda.is_available()
sys.path[:0] = sys.argv[1:]
import plaquette_simulator as ps
from test_gpu_shared import mixed_ops
# the check inside the kernel, and as a launch of its own (columns in LDS, in
# the tableau)
for n, B, where in ((70, 200, "none"), (70, 200, "first"), (70, 200, "last"),
                    (70, 14000, "first"), (70, 14000, "last"),
                    (500, 300, "none"), (500, 300, "first"), (500, 300, "last")):
    ops = mixed_ops(n, 600, 4, 0.1)
    got = []
    for per_shot in (False, True):
        st = ps.CliffordState(n, B, 21, True)
        planes = torch.from_dlpack(st.planes_dlpack()).view(torch.int64)
        st.reset_clifford_state()
        st.synchronize()
        if where == "first":    # H on qubit 0 of the first 64 shots
            planes[0, [0, n]] = planes[0, [n, 0]]
        elif where == "last":   # z of the last row, in two shots
            planes[-1, 2 * n - 1, 2 * n - 1] = 5
        torch.cuda.synchronize()
        prog = ps.Program(st, ops)
        if per_shot:
            prog.set_slices(1)
        prog.run(st, "persistent")
        st.synchronize()
        got.append((st, planes))
    assert got[0][0].compare(got[1][0]) == (0, 0), (n, B, where)
    del got, planes, st
print("raw pointer ok")
"""


def test_words_changed_through_the_raw_pointer(ps):
    """The holder of the planes may change words between the reset and the run:
    those word groups run per shot, the others packed.  (In a child process
    that imports torch before the engine: each carries its own HIP runtime.)"""
    pytest.importorskip("torch")
    import os
    import subprocess
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    say("[case] words changed through the raw pointer (child process)")
    r = subprocess.run([sys.executable, "-c", _RAW_POINTER,
                        os.path.join(root, "plaquette-simulator_amd"),
                        os.path.join(root, "tests"), os.path.join(root, "oracle")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "raw pointer ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.parametrize("form", ["persistent", "graph"])
def test_batch_members_in_both_kernels(ps, form):
    """A batch of members with packed columns in LDS and in the tableau, one with
    a flagged H (per shot), run from |0...0>, then from the states that left, then
    with one member reset: every member equals its standalone per-shot run."""
    from plaquette_simulator import workloads as W
    specs = [(40, 200, mixed_ops(40, 300, 1, 0.1)), (500, 130, mixed_ops(500, 700, 2, 0.03)),
             (9, 65, mixed_ops(9, 200, 3, 0.2))]
    b = W.OpList()
    for q in range(12):
        b.h(q)
        b.with_prob(W.OP_H, q, 0.4)
        b.cx(q, (q + 1) % 12)
    for q in range(12):
        b.measure(q)
    specs.append((12, 100, b.array()))
    batch, got, ref = ps.Batch(), [], []
    for i, (n, B, ops) in enumerate(specs):
        st, rs = (ps.CliffordState(n, B, 50 + i, True) for _ in range(2))
        prog, rp = ps.Program(st, ops), ps.Program(rs, ops)
        rp.set_slices(1)
        batch.add(st, prog)
        got.append((st, prog))
        ref.append((rs, rp))
    batch.set_word_tile(2)
    for step in range(3):
        say(f"[case] batch {form} step {step}")
        if step == 2:
            got[0][0].reset_clifford_state()
            ref[0][0].reset_clifford_state()
        batch.run(form)
        batch.wait()
        for (st, _), (rs, rp) in zip(got, ref):
            rp.run(rs, "persistent")
            assert st.compare(rs) == (0, 0)


@pytest.mark.parametrize("n,B,width,runs", [
    (100, 130, 100, 30),   # 130 ops a round: a layer behind measurements spans ops 390..490
    (161, 64, 161, 17), (33, 70, 33, 31), (64, 16385, 64, 20),
    # columns in the tableau
    (500, 70, 300, 13), (520, 323, 200, 9)])
def test_windows_that_end_between_measurements_and_a_layer(ps, n, B, width, runs):
    """Ops are staged 448 at a time, and a layer that does not fit opens the next
    window.  Rounds of one layer and one run of measurements, so that windows end
    right behind measurements, with the next layer's first op read already."""
    from plaquette_simulator import workloads as W
    rng = np.random.default_rng(n)
    b = W.OpList()
    for r in range(9):
        for q in range(width):
            code = int(rng.choice([W.OP_H, W.OP_S, W.OP_X, W.OP_H]))
            b.gate(code, q)
            if rng.random() < 0.05:
                b.noise(q, 0.1, 0.1, 0.1)
        for _ in range(runs):
            b.measure(int(rng.integers(0, n)))
        for q in range(r % 2, n - 1, 2):
            b.cx(q, q + 1)
        for _ in range(runs):
            b.measure(int(rng.integers(0, n)))
    ops = b.array()
    say(f"[case] windows n={n} B={B} ops={len(ops)}")
    orc = O.OracleState(n, B, 23)
    orc.run_program(ops.astype(np.int32))
    st = ps.CliffordState(n, B, 23, True)
    ps.Program(st, ops).run(st, "persistent")
    check(st, orc)


_COPIES = """
import sys
import torch  # first: its HIP runtime must be the one the process loads
assert torch.cuda.is_available()
sys.path[:0] = sys.argv[1:]
import plaquette_simulator as ps
from test_gpu_shared import mixed_ops

def edited(n, B):
    st = ps.CliffordState(n, B, 21, True)
    planes = torch.from_dlpack(st.planes_dlpack()).view(torch.int64)
    st.reset_clifford_state()
    st.synchronize()
    planes[0, [0, n]] = planes[0, [n, 0]]  # H on qubit 0 of the first 64 shots
    torch.cuda.synchronize()
    return st, planes

def copy_of(st, how, n, B):
    if how == "copy":
        return st.copy()
    if how == "copy of a copy":
        return st.copy().copy()
    dst = ps.CliffordState(n, B, 21, True)
    if how == "into a reset state":
        dst.reset_clifford_state()
    dst.device_to_device(st)
    return dst

for n, B in ((70, 200), (70, 14000), (500, 300)):
    ops = mixed_ops(n, 600, 4, 0.1)
    for how in ("copy", "copy of a copy", "into a state", "into a reset state"):
        for form in ("persistent", "graph", "batch"):
            st, planes = edited(n, B)
            got, ref = copy_of(st, how, n, B), copy_of(st, how, n, B)
            assert got.compare(st) == (0, 0)
            pg, pr = ps.Program(got, ops), ps.Program(ref, ops)
            pr.set_slices(1)  # keeps the per-shot kernel, which reads the words
            if form == "batch":
                batch = ps.Batch()
                batch.add(got, pg)
                batch.run("persistent")
                batch.wait()
            else:
                pg.run(got, form)
            pr.run(ref, "persistent")
            got.synchronize()
            ref.synchronize()
            assert got.compare(ref) == (0, 0), (n, B, how, form)
            # a reset determines the words again
            got.reset_clifford_state()
            ref.reset_clifford_state()
            pg.run(got, "persistent")
            pr.run(ref, "persistent")
            assert got.compare(ref) == (0, 0), (n, B, how, form, "reset")
            del got, ref, pg, pr, planes, st
    # a copy of an exposed |0...0> state still takes the frame form
    st = ps.CliffordState(n, B, 21, True)
    planes = torch.from_dlpack(st.planes_dlpack())
    a, b = st.copy(), st.copy()
    pa, pb = ps.Program(a, ops), ps.Program(b, ops)
    pa.run(a, "frame")
    pb.run(b, "persistent")
    assert a.compare(b) == (0, 0), (n, B, "frame")
print("copies ok")
"""


def test_copies_of_a_state_changed_through_the_raw_pointer(ps):
    """A copy holds the words that the raw pointer's holder wrote, whatever the
    calls on its source say: it runs from those words.  (In a child process that
    imports torch before the engine.)"""
    pytest.importorskip("torch")
    import os
    import subprocess
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    say("[case] copies of a state changed through the raw pointer (child process)")
    r = subprocess.run([sys.executable, "-c", _COPIES,
                        os.path.join(root, "plaquette-simulator_amd"),
                        os.path.join(root, "tests"), os.path.join(root, "oracle")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "copies ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.parametrize("n,B", [(2, 64), (40, 150), (70, 200), (161, 2700), (500, 70)])
def test_graph_replays_follow_their_state(ps, n, B):
    """One program replayed from states that take different kernels: |0...0> after
    a reset or behind a frame run that ends there, what the last replay left, one
    from the host, one whose planes were handed out; then another state."""
    from plaquette_simulator import workloads as W
    ops = mixed_ops(n, 3 * n + 60, n, 0.1)
    flips = W.OpList()  # X/Z end as they start
    for q in range(n):
        flips.gate(W.OP_X, q)
        flips.noise(q, 0.2, 0.1, 0.1)
    st, ref = (ps.CliffordState(n, B, 9, True) for _ in range(2))
    prog, pref = ps.Program(st, ops), ps.Program(ref, ops)
    fst, fref = ps.Program(st, flips.array()), ps.Program(ref, flips.array())
    pref.set_slices(1)  # the per-shot kernel
    held = []
    for i, step in enumerate(["", "", "reset", "", "reset", "frame", "host", "reset", "", "expose",
                              "reset", "", "frame", ""]):
        say(f"[case] n={n} B={B} graph replay {i} {step}")
        for s, f in ((st, fst), (ref, fref)):
            if step in ("reset", "frame"):
                s.reset_clifford_state()
            if step == "frame":
                f.run(s, "frame")
            if step == "host" and n <= 70:  # (int lists: small states only)
                x, z, r = s.device_to_host_numpy()
                s.host_to_device(x.ravel(), z.ravel(), r.ravel())
        if step == "expose":
            held.append(st.planes_dlpack())
        prog.run(st, "graph")
        pref.run(ref, "persistent")
        assert st.compare(ref) == (0, 0)
    other, oref = (ps.CliffordState(n, B, 10, True) for _ in range(2))
    for _ in range(2):
        prog.run(other, "graph")
        pref.run(oref, "persistent")
        assert other.compare(oref) == (0, 0)
    st.reset_clifford_state()
    ref.reset_clifford_state()
    prog.run(st, "graph")
    pref.run(ref, "persistent")
    assert st.compare(ref) == (0, 0)


def test_graph_of_a_state_that_is_gone(ps):
    """A program outlives the states that it ran on: a later state may have the
    address of one that is gone, and does not replay its captured launch."""
    n, B = 60, 200
    ops = mixed_ops(n, 300, 3, 0.1)
    home = ps.CliffordState(n, B, 1, True)
    prog = ps.Program(home, ops)
    kept = []
    for i in range(6):
        say(f"[case] graph on state {i}")
        st, ref = (ps.CliffordState(n, B, 30 + i, True) for _ in range(2))
        prog.run(st, "graph")
        ps.Program(ref, ops).run(ref, "persistent")
        assert st.compare(ref) == (0, 0)
        if i % 2:
            kept.append(ref)  # takes the memory of the one before
        del st, ref


_SMALL = """
import sys
import torch  # first: its HIP runtime must be the one the process loads
assert torch.cuda.is_available()
sys.path[:0] = sys.argv[1:]
import plaquette_simulator as ps
from test_gpu_shared import mixed_ops
# both sides of the line between the packed and the LDS-resident kernel: 33 and
# 64 qubits with few ops and many, groups that wait for compute units
for n, B, nops in ((2, 64, 30), (2, 17000, 40), (2, 17000, 70), (32, 130, 900), (33, 60, 5200),
                   (64, 64, 100), (64, 64, 260), (64, 16385, 110), (64, 16385, 200)):
    ops = mixed_ops(n, nops, 4, 0.1)
    for edit in (False, True):
        for form in ("persistent", "graph"):
            got = []
            for per_shot in (False, True):
                st = ps.CliffordState(n, B, 21, True)
                planes = torch.from_dlpack(st.planes_dlpack()).view(torch.int64)
                st.reset_clifford_state()
                st.synchronize()
                if edit:  # z of the last row, in two shots of the last group
                    planes[-1, 2 * n - 1, 2 * n - 1] = 5
                torch.cuda.synchronize()
                prog = ps.Program(st, ops)
                if per_shot:
                    prog.set_slices(1)
                prog.run(st, "persistent" if per_shot else form)
                st.synchronize()
                got.append((st, planes))
            assert got[0][0].compare(got[1][0]) == (0, 0), (n, B, nops, edit, form)
            del got, planes, st
print("small ok")
"""


def test_small_states_with_the_raw_pointer_out(ps):
    """Small states whose words have to be looked at take the packed kernel, with
    the check and the LDS-resident one behind it, or the latter alone."""
    pytest.importorskip("torch")
    import os
    import subprocess
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    say("[case] small states with the raw pointer out (child process)")
    r = subprocess.run([sys.executable, "-c", _SMALL,
                        os.path.join(root, "plaquette-simulator_amd"),
                        os.path.join(root, "tests"), os.path.join(root, "oracle")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "small ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
