"""What a user of this framework has it do, as cases to be timed.

Each case goes through the public Python API.  Sizes are those of the
repository's own workloads (``plaquette_simulator.workloads``, ``bench.py``):
the n=64 and n=1024 random Clifford circuits, surface-code memory experiments
from d=3 to d=17 up to the serving stream's shot counts, the mixed batch and
the server.  Every result is a bit (a measurement outcome, a tableau entry), so
there is no value "in 64 bits" to come near to: results are equal or wrong.

Kinds:
  gates     the reference's own way of working: one API call per gate, two
            measurements into existing records
  random    one random Clifford circuit run as a compiled program; with
            ``flags`` a tenth of its gates are applied per shot with
            probability 1/2, so X/Z differ between shots
  memory    one surface-code memory experiment, persistent form; its records, and
            with ``tableau`` the state that it leaves
  frame     the same in the frame form
  batch     many memory experiments of different sizes in one launch (``graph``: the
            tableaux come back too)
  serve     requests submitted to a server, waited for and collected
  readout   device_to_host of a whole tableau
"""
import math
import os
import sys

import numpy as np
import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "plaquette-simulator_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import plaquette_simulator as ps  # noqa: E402
from plaquette_simulator import workloads as wl  # noqa: E402


def listed():
    return [
        # interactive use of the reference's API: latency of single calls
        {"name": "gates_n64_b1024", "kind": "gates", "n": 64, "shots": 1024, "ops": 48},
        # the n=64 random Clifford circuit, 2000 gates and 20 measurements
        {"name": "random_n64_b1024", "kind": "random", "n": 64, "shots": 1024, "ops": 2000,
         "every": 100, "flags": False},
        # a circuit with gates applied per shot: every shot has its own X/Z and pivots
        {"name": "conditional_n41_b5000", "kind": "random", "n": 41, "shots": 5000, "ops": 800,
         "every": 20, "flags": True},
        # the n=1024 random Clifford circuit (a fifth of its ops): the largest state
        {"name": "random_n1024_b4096", "kind": "random", "n": 1024, "shots": 4096,
         "ops": 20000, "every": 10, "flags": False},
        # the smallest memory experiment: four word groups on an empty GPU
        {"name": "memory_d3_b256", "kind": "memory", "d": 3, "rounds": 3, "shots": 256,
         "p": 0.001, "tableau": False},
        # the headline: d=9, 9 rounds, 16384 shots, with the tableau that it leaves
        {"name": "memory_d9_b16384", "kind": "memory", "d": 9, "rounds": 9, "shots": 16384,
         "p": 0.001, "tableau": True},
        # a larger code at an odd shot count (449 qubits, segments cut into windows)
        {"name": "memory_d15_b3001", "kind": "memory", "d": 15, "rounds": 15, "shots": 3001,
         "p": 0.002, "tableau": True},
        # the headline circuit in the frame form: sampling at one word group per CU
        {"name": "frame_d9_b16384", "kind": "frame", "d": 9, "rounds": 9, "shots": 16384,
         "p": 0.001, "tableau": False},
        # a large sampling run
        {"name": "frame_d17_b32768", "kind": "frame", "d": 17, "rounds": 17, "shots": 32768,
         "p": 0.003, "tableau": False},
        # the mixed batch: 24 circuits d=3..11 in one launch
        {"name": "batch_24", "kind": "batch", "count": 24, "dmax": 11, "smax": 4096,
         "form": "graph", "p": 0.001},
        # a burst of sampling requests at a server
        {"name": "serve_16", "kind": "serve", "count": 16, "dmax": 9, "smax": 8192,
         "form": "frame"},
        # the whole tableau on the host in the reference's layout
        {"name": "readout_n64_b1024", "kind": "readout", "n": 64, "shots": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gates", "random", "random", "memory", "memory", "frame", "frame",
                       "batch", "serve", "readout"])
    if kind == "gates":
        return {"kind": kind, "n": _log_int(rng, 8, 128), "shots": _log_int(rng, 64, 16384),
                "ops": rng.randint(16, 96)}
    if kind == "random":
        n, shots = _log_int(rng, 16, 1024), _log_int(rng, 64, 8192)
        # no more than the n=1024 circuit's rows x word groups x ops
        most = 20000 * 64 * 2049 / ((2 * n + 1) * ((shots + 63) // 64))
        flags = n <= 192 and rng.random() < 0.4
        # shots with pivots of their own make measurements up to 64 times longer
        ops = _log_int(rng, 200, max(201, min(2000 if flags else 20000, most)))
        return {"kind": kind, "n": n, "shots": shots, "ops": ops,
                "every": _log_int(rng, 10, 100), "flags": flags}
    if kind in ("memory", "frame"):
        d = rng.choice([3, 5, 7, 9, 11, 13, 15, 17])
        rounds = rng.randint(2, d)
        # no more than the listed d=17 frame run, or d=15 persistent run, moves
        most = (577 * 17 * 32768 / (2 * d * d * rounds) if kind == "frame" else
                4.5e8 * 15 * 3001 / ((2 * d * d) ** 2 * 2 * rounds))
        return {"kind": kind, "d": d, "rounds": rounds,
                "shots": _log_int(rng, 64, min(65536 if kind == "frame" else 16384, most)),
                "p": round(rng.uniform(5e-4, 5e-3), 5), "tableau": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 24), "dmax": rng.choice([5, 7, 9, 11]),
                "smax": _log_int(rng, 256, 4096), "form": rng.choice(["graph", "frame"]),
                "p": round(rng.uniform(5e-4, 5e-3), 5)}
    if kind == "serve":
        return {"kind": kind, "count": rng.randint(4, 16), "dmax": rng.choice([5, 7, 9]),
                "smax": _log_int(rng, 512, 8192), "form": rng.choice(["frame", "persistent"])}
    return {"kind": kind, "n": _log_int(rng, 8, 128), "shots": _log_int(rng, 64, 1024)}


def _seed(seed):
    return int(seed) % (1 << 31)


def _random_ops(case, seed):
    """Uniform H/S/CX, a measurement after every ``every``-th."""
    if not case["flags"]:
        return wl.random_clifford(case["n"], case["ops"], seed, meas_every=case["every"])
    rng = np.random.default_rng(seed)
    n, b = case["n"], wl.OpList()
    for i in range(case["ops"]):
        code = (wl.OP_H, wl.OP_S, wl.OP_CX)[int(rng.integers(0, 3))]
        q = int(rng.integers(0, n))
        t = (q + 1 + int(rng.integers(0, n - 1))) % n if code == wl.OP_CX else 0
        if rng.random() < 0.1:
            b.with_prob(code, q, 0.5, t)
        else:
            b.gate(code, q, t)
        if (i + 1) % case["every"] == 0:
            b.measure(int(rng.integers(0, n)))
    return b.array()


def _mixed(case):
    """``count`` memory experiments: (d, shots), d over odd 3..dmax, shots log-uniform.

    The same for every seed: a seed is another stream of coins and noise."""
    rng = np.random.default_rng(case["count"])
    out = []
    for _ in range(case["count"]):
        d = int(rng.choice(list(range(3, case["dmax"] + 1, 2))))
        out.append((d, int(round(math.exp(rng.uniform(math.log(64), math.log(case["smax"])))))))
    return out


def _records(st):
    """The state's record arena [record][results, determined][word], on the device."""
    return torch.from_dlpack(st.records_dlpack()).view(torch.int64)


def _planes(st):
    """The state's tableau [word][column][row], on the device."""
    return torch.from_dlpack(st.planes_dlpack()).view(torch.int64)


def prepare(case, seed):
    kind, seed = case["kind"], _seed(seed)
    if kind in ("gates", "readout"):
        n, shots = case["n"], case["shots"]
        st = ps.CliffordState(n, shots, seed, True)
        # a state as a circuit leaves it, not |0...0>
        st.run_program(wl.random_clifford(n, 8 * n, seed), "persistent")
        if kind == "readout":
            return {"case": case, "st": st}
        ids = [st.measure_qubit(n // 3, 0.5, None), st.measure_qubit(n // 2, 0.5, None)]
        rng = np.random.default_rng(seed)
        calls = []
        for i in range(case["ops"]):
            q = int(rng.integers(0, n))
            t = (q + 1 + int(rng.integers(0, n - 1))) % n
            calls.append((int(rng.integers(0, 6)), q, t))
        return {"case": case, "st": st, "calls": calls, "ids": ids,
                "out": (_planes(st), _records(st))}
    if kind == "random":
        st = ps.CliffordState(case["n"], case["shots"], seed, True)
        prog = ps.Program(st, _random_ops(case, seed))
        prog.run(st, "persistent")  # makes the records that later runs write again
        return {"case": case, "st": st, "prog": prog, "out": (_planes(st), _records(st))}
    if kind in ("memory", "frame"):
        ops, n = wl.surface_code_memory_z(case["d"], case["rounds"], case["p"])
        st = ps.CliffordState(n, case["shots"], seed, True)
        prog = ps.Program(st, ops)
        prog.run(st, "frame" if kind == "frame" else "persistent")
        out = (_records(st), _planes(st)) if case["tableau"] else _records(st)
        return {"case": case, "st": st, "prog": prog, "out": out}
    if kind == "batch":
        batch, states, progs = ps.Batch(), [], []
        for i, (d, shots) in enumerate(_mixed(case)):
            ops, n = wl.surface_code_memory_z(d, d, case["p"])
            st = ps.CliffordState(n, shots, (seed + i) % (1 << 31), True)
            prog = ps.Program(st, ops)
            batch.add(st, prog)
            states.append(st)
            progs.append(prog)
        batch.run(case["form"])
        return {"case": case, "batch": batch, "states": states, "progs": progs,
                "out": [_records(st) for st in states] +
                       ([_planes(st) for st in states] if case["form"] == "graph" else [])}
    if kind == "serve":
        sv = ps.Server(64 << 30)
        sv.set_form(case["form"])
        rng = np.random.default_rng(seed)
        reqs = []
        for i, (d, shots) in enumerate(_mixed(case)):
            ops, n = wl.surface_code_memory_z(d, d, float(rng.uniform(5e-4, 5e-3)))
            reqs.append((n, shots, (seed + i) % (1 << 31), ops))
        return {"case": case, "server": sv, "reqs": reqs}
    raise ValueError(kind)


def run(state):
    kind = state["case"]["kind"]
    if kind == "gates":
        st, ids = state["st"], state["ids"]
        calls = state["calls"]
        for i, (code, q, t) in enumerate(calls):
            if code == 0:
                st.apply_hadamard_gate(q)
            elif code == 1:
                st.apply_phase_gate(q)
            elif code == 2:
                st.apply_pauli_x_gate(q)
            elif code == 3:
                st.apply_control_phase_gate(q, t)
            else:
                st.apply_control_not_gate(q, t)
            if i == len(calls) // 2:
                st.measure_qubit(q, 0.5, ids[0])
        st.measure_qubit(calls[0][1], 0.5, ids[1])
        return state["out"]
    if kind == "random":
        state["st"].reset_clifford_state()
        state["prog"].run(state["st"], "persistent")
        return state["out"]
    if kind in ("memory", "frame"):
        state["st"].reset_clifford_state()
        state["prog"].run(state["st"], "frame" if kind == "frame" else "persistent")
        return state["out"]
    if kind == "batch":
        for st in state["states"]:
            st.reset_clifford_state()
        state["batch"].run(state["case"]["form"])
        return state["out"]
    if kind == "serve":
        sv = state["server"]
        tickets = [sv.submit(n, shots, seed, ops) for n, shots, seed, ops in state["reqs"]]
        sv.drain()
        out = []
        for t in tickets:
            out.append(sv.result(t).view(np.int64))
            sv.release(t)
        return out
    x, z, r = state["st"].device_to_host_numpy()
    return x, z, r


def _groups(shots):
    return (shots + 63) // 64


def _memory_records(d, rounds):
    return rounds * (d * d - 1) + d * d


def work(case):
    """Bytes of one pass: the results written once, what it starts from read once.

    A program starts from |0...0>, which nothing has to read.  The work is
    bit logic, so there are no floating-point operations to count."""
    kind = case["kind"]
    if kind == "gates":
        # one call per gate: it reads and writes its columns (CX, CZ: 4 read,
        # 2 and r written; the others fewer), about 6 words a row and call
        R, W = 2 * case["n"] + 1, _groups(case["shots"])
        return {"bytes": 48.0 * R * W * case["ops"], "flops": 0}
    if kind == "random":
        R, W = 2 * case["n"] + 1, _groups(case["shots"])
        return {"bytes": 8.0 * W * (R * R + 2 * (case["ops"] // case["every"])), "flops": 0}
    if kind in ("memory", "frame"):
        R, W = 2 * (2 * case["d"] ** 2 - 1) + 1, _groups(case["shots"])
        rows = R * R if kind == "memory" or case["tableau"] else R
        return {"bytes": 8.0 * W * (rows + 2 * _memory_records(case["d"], case["rounds"])),
                "flops": 0}
    if kind in ("batch", "serve"):
        total = 0
        for d, shots in _mixed(case):
            R = 2 * (2 * d * d - 1) + 1
            rows = R if case["form"] == "frame" else R * R
            total += 8.0 * _groups(shots) * (rows + 2 * _memory_records(d, d))
        return {"bytes": total, "flops": 0}
    R = 2 * case["n"] + 1
    # bits read, int32 entries written
    return {"bytes": R * (2 * case["n"] + 1) * case["shots"] * (1 / 8 + 4), "flops": 0}
