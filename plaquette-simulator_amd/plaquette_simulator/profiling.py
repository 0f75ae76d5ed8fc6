"""Profiling helpers for the engine (run under rocprofv3).

  python profiling.py probe
      One persistent run of the d=9 surface-code workload (16384 shots),
      preceded by a warm-up run and by a device-to-device copy of the whole
      tableau (W*(2n+1)^2*8 bytes) that serves as the counter calibration
      dispatch.  Run it under `rocprofv3 --pmc FETCH_SIZE` and again under
      `--pmc WRITE_SIZE`.

  python profiling.py kernels <rocprof csv dir> <out.md>
      Summarise a `--kernel-trace --stats --output-format csv` run.

  python profiling.py traffic <fetch csv dir> <write csv dir> <out.json> <out.md>
      HBM traffic of the run's kernels, each counter scaled by what the
      same counter reads for the calibration copy of known size.

  python profiling.py sizes <read-size csv dir> <write-size csv dir> <out.json> <out.md>
      HBM traffic of the run's kernels from the request counters by size, no
      calibration: reads 32 x RDREQ_32B + 64 x RDREQ_64B + 128 x RDREQ_128B,
      writes 64 x WRREQ_64B + 32 x (WRREQ - WRREQ_64B) (TCC_EA0_*, summed
      over channels), beside the same for the calibration copy.

  python profiling.py probe-n1024 [slices ...]
      The n=1024 random circuit (4096 shots, 100000 ops): a device-to-device
      copy of the whole tableau (calibration), then one persistent run, or
      one run of the per-shot kernel per workgroups-per-word-group count.

  python profiling.py probe-conditional
      A random circuit of 41 qubits, 5000 shots, 800 ops of which a tenth are
      applied per shot with probability 1/2, 40 measurements: calibration copy, then
      one persistent run (the LDS-resident kernel).

  python profiling.py dispatches <out.md> <csv dir> [<csv dir> ...]
      Every counter of every `--pmc` pass for each of the run's kernels and the
      calibration copy, side by side, by kernel and grid.

  python profiling.py pmc <out.md> <csv dir> [<csv dir> ...]
      Every counter of every `--pmc` pass, for each kernel of the run and
      the calibration copy, side by side.

The run's kernels are those between the events that time it: k_program (or
k_program_shared and k_shared_expand, with k_shared_verify where it checks),
dispatched after the calibration copy; its noise and parameters come before.
"""
import csv
import glob
import json
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def _state_and_program(shots=16384):
    sys.path.insert(0, os.path.dirname(HERE))
    import plaquette_simulator as ps
    from plaquette_simulator import workloads as W
    w = W.config_surface_d9(shots=shots)
    st = ps.CliffordState(w.num_qubits, w.batch_size, w.seed, True)
    prog = ps.Program(st, w.ops)
    return ps, w, st, prog


def probe(shots=16384):
    ps, w, st, prog = _state_and_program(shots)
    prog.run(st, "persistent")              # warm-up (also creates records)
    st.synchronize()
    other = ps.CliffordState(w.num_qubits, w.batch_size, w.seed, False)
    other.synchronize()
    other.device_to_device(st)              # calibration copy
    other.synchronize()
    st.reset_clifford_state()
    prog.run(st, "persistent")              # measured dispatch
    st.synchronize()
    n = w.num_qubits
    words = (w.batch_size + 63) // 64
    copy_bytes = words * (2 * n + 1) ** 2 * 8
    print(json.dumps({"workload": w.name, "copy_bytes": copy_bytes}))


def probe_conditional():
    """A circuit with gates applied per shot, after a calibration copy."""
    import numpy as np
    sys.path.insert(0, os.path.dirname(HERE))
    import plaquette_simulator as ps
    from plaquette_simulator import workloads as W
    n, B, rng, b = 41, 5000, np.random.default_rng(5), W.OpList()
    for i in range(800):
        code = (W.OP_H, W.OP_S, W.OP_CX)[int(rng.integers(0, 3))]
        q = int(rng.integers(0, n))
        t = (q + 1 + int(rng.integers(0, n - 1))) % n if code == W.OP_CX else 0
        if rng.random() < 0.1:
            b.with_prob(code, q, 0.5, t)
        else:
            b.gate(code, q, t)
        if i % 20 == 19:
            b.measure(int(rng.integers(0, n)))
    st = ps.CliffordState(n, B, 5, True)
    other = ps.CliffordState(n, B, 5, False)
    prog = ps.Program(st, b.array())
    prog.run(st, "persistent")
    st.synchronize()
    other.device_to_device(st)              # calibration copy
    other.synchronize()
    st.reset_clifford_state()
    prog.run(st, "persistent")
    st.synchronize()
    words = (B + 63) // 64
    print(json.dumps({"probe": "done", "copy_bytes": words * (2 * n + 1) ** 2 * 8}), flush=True)


def probe_n1024(slices=(None,)):
    """The n=1024 random circuit (4096 shots, 100000 ops), one persistent run
    (None), or one of the per-shot kernel per workgroups-per-word-group count in
    `slices`, after a device-to-device copy of the whole 2.15 GB tableau (the
    calibration dispatch)."""
    sys.path.insert(0, os.path.dirname(HERE))
    import plaquette_simulator as ps
    from plaquette_simulator import workloads as W
    w = W.config_random_n1024()
    n, B = w.num_qubits, w.batch_size
    st = ps.CliffordState(n, B, w.seed, True)
    other = ps.CliffordState(n, B, w.seed, False)
    other.synchronize()
    other.device_to_device(st)              # calibration copy
    other.synchronize()
    del other
    prog = ps.Program(st, w.ops)
    for s in slices:
        if s is not None:
            prog.set_slices(s)
        st.reset_clifford_state()
        prog.run(st, "persistent")
        st.synchronize()
        used, failed = prog.slice_status(st)
        print(json.dumps({"workload": w.name, "slices": used, "barrier_failures": failed}),
              flush=True)
    words = (B + 63) // 64
    print(json.dumps({"probe": "done", "copy_bytes": words * (2 * n + 1) ** 2 * 8}), flush=True)


def dispatches(out, *dirs):
    """Every counter of every `--pmc` pass for each of the run's kernels (name
    and grid size) and the calibration copy."""
    table = {}
    order = []
    for d in dirs:
        rs = _counter_rows(d)
        copy = max((int(r["Dispatch_Id"]) for r in rs if "copyBuffer" in r["Kernel_Name"]),
                   default=0)
        for r in rs:
            k = r["Kernel_Name"]
            if int(r["Dispatch_Id"]) < copy:  # warm-up
                continue
            if not _of_run(k) and "copyBuffer" not in k:
                continue
            who = ("calibration copy" if "copyBuffer" in k else
                   "%s grid %s" % (_short(k), r["Grid_Size"]))
            if who not in table:
                table[who] = {}
                order.append(who)
            table[who][r["Counter_Name"]] = table[who].get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
    names = sorted({c for v in table.values() for c in v})
    md = ["| counter | " + " | ".join(order) + " |", "|---" * (len(order) + 1) + "|"]
    for c in names:
        md.append("| %s | " % c + " | ".join("%.6g" % table[w].get(c, float("nan")) for w in order) + " |")
    with open(out, "w") as f:
        f.write("\n".join(md) + "\n")
    print("\n".join(md))


def _find(d, pattern):
    hits = glob.glob(os.path.join(d, "**", pattern), recursive=True)
    if not hits:
        raise FileNotFoundError(f"{pattern} under {d}")
    return hits[0]


def kernels(d, out):
    path = _find(d, "*kernel_stats.csv")
    rows = list(csv.DictReader(open(path)))
    lines = ["| kernel | calls | total ms | avg us | min us | max us | % |", "|---|---|---|---|---|---|---|"]
    for r in rows:
        name = r["Name"].replace("(anonymous namespace)::", "").replace("pq::", "")
        name = name.split("(")[0]
        lines.append("| %s | %s | %.3f | %.2f | %.2f | %.2f | %.2f |" % (
            name[:60], r["Calls"], float(r["TotalDurationNs"]) / 1e6,
            float(r["AverageNs"]) / 1e3, float(r["MinNs"]) / 1e3,
            float(r["MaxNs"]) / 1e3, float(r["Percentage"])))
    # per-launch durations of the persistent kernel, in launch order
    try:
        trace = list(csv.DictReader(open(_find(d, "*kernel_trace.csv"))))
    except (FileNotFoundError, StopIteration, IndexError):
        trace = []
    for kname in ("k_program", "k_frame"):
        durs = [(int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3
                for r in sorted(trace, key=lambda r: int(r["Start_Timestamp"]))
                if kname + "_t" in r["Kernel_Name"] or kname + "(" in r["Kernel_Name"]]
        if durs:
            srt = sorted(durs)
            lines += ["", "%s launches in order (us): " % kname + ", ".join("%.1f" % v for v in durs),
                      "%s median: %.1f us over %d launches" % (kname, srt[len(srt) // 2], len(srt))]
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


def _counter_rows(d):
    path = _find(d, "*counter_collection.csv")
    return list(csv.DictReader(open(path)))


def _per_dispatch(rows, counter):
    out = {}
    for r in rows:
        if r.get("Counter_Name") != counter:
            continue
        key = (int(r["Dispatch_Id"]), r["Kernel_Name"])
        out[key] = out.get(key, 0.0) + float(r["Counter_Value"])
    return out


def _of_run(kernel):
    return ("k_program" in kernel or "k_shared_" in kernel) and "noise" not in kernel


def _short(kernel):
    name = kernel.replace("(anonymous namespace)::", "").replace("pq::", "").split("(")[0]
    return name[5:] if name.startswith("void ") else name


def _run_kernels(disp):
    """Kernel name -> counter of the run behind the last calibration copy, and the
    copy's counter."""
    copies = [i for (i, k) in disp if "copyBuffer" in k]
    if not copies:
        raise RuntimeError("calibration copy missing")
    copy = max(copies)
    run = {}
    for (i, k), v in sorted(disp.items()):
        if i > copy and _of_run(k):
            run[_short(k)] = run.get(_short(k), 0.0) + v
    if not run:
        raise RuntimeError("no kernel of the run behind the calibration copy")
    return run, next(v for (i, k), v in disp.items() if i == copy)


def traffic(fetch_dir, write_dir, out_json, out_md, copy_bytes=None):
    if copy_bytes is None:
        n, words = 161, 256
        copy_bytes = words * (2 * n + 1) ** 2 * 8
    res = {"copy_bytes": copy_bytes}
    for label, d, counter in (("fetch", fetch_dir, "FETCH_SIZE"), ("write", write_dir, "WRITE_SIZE")):
        run, kib_copy = _run_kernels(_per_dispatch(_counter_rows(d), counter))
        kib_run = sum(run.values())
        scale = copy_bytes / (kib_copy * 1024.0)
        res[label] = {"counter_kib_kernels": run, "counter_kib_copy": kib_copy,
                      "scale": scale, "bytes": kib_run * 1024.0 * scale}
    res["bytes_per_launch"] = res["fetch"]["bytes"] + res["write"]["bytes"]
    with open(out_json, "w") as f:
        json.dump(res, f, indent=1)
    md = [
        "| counter | kernels of the run (KiB) | calibration copy (KiB) | scale (copy bytes / counter bytes) | run's bytes |",
        "|---|---|---|---|---|",
    ]
    for label, counter in (("fetch", "FETCH_SIZE"), ("write", "WRITE_SIZE")):
        r = res[label]
        md.append("| %s | %s | %.0f | %.4f | %.4g |" % (
            counter, ", ".join("%s %.0f" % kv for kv in r["counter_kib_kernels"].items()),
            r["counter_kib_copy"], r["scale"], r["bytes"]))
    md.append("")
    md.append("traffic per run: %.4g bytes (calibration copy: %d bytes each way)"
              % (res["bytes_per_launch"], copy_bytes))
    with open(out_md, "w") as f:
        f.write("\n".join(md) + "\n")
    print("\n".join(md))
    return res


def sizes(rd_dir, wr_dir, out_json, out_md):
    def counter(d, name):
        return _run_kernels(_per_dispatch(_counter_rows(d), name))
    rd = {b: counter(rd_dir, "TCC_EA0_RDREQ_%sB_sum" % b) for b in (32, 64, 128)}
    wr = counter(wr_dir, "TCC_EA0_WRREQ_sum")
    wr64 = counter(wr_dir, "TCC_EA0_WRREQ_64B_sum")
    res = {}
    for who in list(wr[0]) + ["calibration_copy"]:
        def of(c):
            return c[1] if who == "calibration_copy" else c[0].get(who, 0.0)
        read = sum(b * of(rd[b]) for b in rd)
        write = 64 * of(wr64) + 32 * (of(wr) - of(wr64))
        res[who] = {"rdreq_32b": of(rd[32]), "rdreq_64b": of(rd[64]), "rdreq_128b": of(rd[128]),
                    "wrreq": of(wr), "wrreq_64b": of(wr64), "read_bytes": read,
                    "write_bytes": write, "bytes": read + write}
    with open(out_json, "w") as f:
        json.dump(res, f, indent=1)
    md = ["| dispatch | RDREQ 32B | RDREQ 64B | RDREQ 128B | WRREQ | WRREQ 64B | read bytes | write bytes | total |",
          "|---|---|---|---|---|---|---|---|---|"]
    for who, r in res.items():
        md.append("| %s | %.6g | %.6g | %.6g | %.6g | %.6g | %.4g | %.4g | %.4g |" % (
            who, r["rdreq_32b"], r["rdreq_64b"], r["rdreq_128b"], r["wrreq"], r["wrreq_64b"],
            r["read_bytes"], r["write_bytes"], r["bytes"]))
    with open(out_md, "w") as f:
        f.write("\n".join(md) + "\n")
    print("\n".join(md))


def pmc(out, *dirs):
    names, rows = [], []
    for d in dirs:
        rs = _counter_rows(d)
        for counter in sorted({r["Counter_Name"] for r in rs}):
            run, copy = _run_kernels(_per_dispatch(rs, counter))
            names += [k for k in run if k not in names]
            rows.append((counter, run, copy))
    md = ["| counter | " + " | ".join(names) + " | calibration copy |", "|---" * (len(names) + 2) + "|"]
    md += ["| %s | " % c + " | ".join("%.6g" % run.get(k, float("nan")) for k in names) +
           " | %.6g |" % copy for c, run, copy in rows]
    with open(out, "w") as f:
        f.write("\n".join(md) + "\n")
    print("\n".join(md))


if __name__ == "__main__":
    cmd = sys.argv[1] if len(sys.argv) > 1 else "probe"
    if cmd == "probe":
        probe()
    elif cmd == "kernels":
        kernels(sys.argv[2], sys.argv[3])
    elif cmd == "traffic":
        traffic(*sys.argv[2:6])
    elif cmd == "sizes":
        sizes(*sys.argv[2:6])
    elif cmd == "pmc":
        pmc(sys.argv[2], *sys.argv[3:])
    elif cmd == "probe-n1024":
        probe_n1024(tuple(int(a) for a in sys.argv[2:]) or (None,))
    elif cmd == "probe-conditional":
        probe_conditional()
    elif cmd == "dispatches":
        dispatches(sys.argv[2], *sys.argv[3:])
    else:
        raise SystemExit(__doc__)
