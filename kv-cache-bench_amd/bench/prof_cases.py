#!/usr/bin/env python3
"""One pass form of a case of perf/cases.py for a profiler (--case NAME), the list of them (--list), or the
summary of what profile_cases.sh wrote (OUT): per case, each kernel's time and HBM traffic."""
import csv
import importlib.util
import os
import re
import statistics
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
WARM, TIMED = 3, 10


def cases():
    os.chdir(ROOT)
    sys.path.insert(0, ROOT)
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(ROOT, "perf", "cases.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def one(name):
    m = cases()
    state = m.prepare(next(c for c in m.listed() if c["name"] == name), 1)
    for _ in range(WARM + TIMED):
        m.run(state)
    m.kvb.synchronize()


def rows(path, value):
    """{kernel: [value per dispatch, in order]} of the library's kernels but the fills."""
    out = {}
    with open(path) as f:
        for r in csv.DictReader(f):
            name = r["Kernel_Name"]
            if "kvbk::" in name and "fill_kernel" not in name:
                out.setdefault(name, []).append(value(r))
    return out


def timed(values):
    """The last TIMED passes' dispatches (a pass may launch a kernel more than once), and how many a pass."""
    per = len(values) // (WARM + TIMED)
    return values[-per * TIMED:], per


def short(name):
    name = re.sub(r"\(anonymous namespace\)::", "", name).replace("void ", "").replace("kvbk::", "")
    return name.split("(")[0]


def summary(out):
    m = cases()
    print("# The kernels of perf/cases.py's listed cases — MI355X\n\n```\n"
          "bash kv-cache-bench_amd/bench/profile_cases.sh OUT\n```\n")
    print(f"rocprofv3 kernel trace and counters (a run each) over the last {TIMED} of {WARM + TIMED} passes on the same "
          "buffers: medians per dispatch. FETCH_SIZE reports half of the bytes read (a 1 GiB read as 0.5 GiB, in "
          "every traffic record beside this file) and is doubled here; both counters count what leaves L2, so also "
          "what the memory-side cache serves.\n")
    print("| case | kernel | a pass | median us | min us | read MiB | written MiB | case's bytes, MiB |\n"
          "|---|---|---|---|---|---|---|---|")
    for c in m.listed():
        d = os.path.join(out, c["name"])
        times = rows(os.path.join(d, "trace", "run_kernel_trace.csv"),
                     lambda r: (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3)
        read, written = (rows(os.path.join(d, k, "run_counter_collection.csv"),
                              lambda r: float(r["Counter_Value"]) * scale / 1024)  # KiB
                         for k, scale in (("fetch", 2), ("write", 1)))
        for name, v in times.items():
            t, per = timed(v)
            print(f"| `{c['name']}` | `{short(name)}` | {per} | {statistics.median(t):.1f} | {min(t):.1f} | "
                  f"{statistics.median(timed(read[name])[0]):.1f} | {statistics.median(timed(written[name])[0]):.1f} | "
                  f"{m.work(c)['bytes'] / 2**20:.1f} |")


if __name__ == "__main__":
    if sys.argv[1] == "--list":
        print(" ".join(c["name"] for c in cases().listed()))
    elif sys.argv[1] == "--case":
        one(sys.argv[2])
    else:
        summary(sys.argv[1])
