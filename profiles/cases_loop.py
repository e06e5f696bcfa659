"""The listed cases of perf/cases.py as a profiler sees them.

    rocprofv3 --kernel-trace --output-format csv -d OUT -o run -- python3 profiles/cases_loop.py
    python3 profiles/cases_loop.py OUT/.../run_kernel_trace.csv

The first command runs every case CALLS times on the same inputs, one library kernel a call, and prints the
time per call of the second half, by events; the second one prints the kernels' times of the same half (the
first half warms the case up) and the averages of the first and last fifty launches.
"""
import csv
import re
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
CALLS = 400
_KERNEL = re.compile(r"(?:lava::|4lava\d+)(\w*?_kernel)")   # the names come demangled or not


def run():
    import torch
    from perf import cases
    for case in cases.listed():
        state = cases.prepare(case, 1)
        torch.cuda.synchronize()
        e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        for i in range(CALLS):
            if i == CALLS // 2:
                e0.record()
            cases.run(state)
        e1.record()
        e1.synchronize()
        print(f"{case['name']:26s} {e0.elapsed_time(e1) * 2e3 / CALLS:8.2f} us a call", flush=True)


def table(path):
    from perf import cases
    rows = sorted((int(r["Start_Timestamp"]), int(r["End_Timestamp"]), r["Kernel_Name"])
                  for r in csv.DictReader(open(path)) if _KERNEL.search(r["Kernel_Name"]))
    names = [c["name"] for c in cases.listed()]
    assert len(rows) == CALLS * len(names), f"{len(rows)} launches of the library, {CALLS * len(names)} expected"
    for i, name in enumerate(names):
        part = rows[i * CALLS:(i + 1) * CALLS]
        us = [(end - start) / 1e3 for start, end, _ in part]
        late = us[CALLS // 2:]
        kernel = _KERNEL.search(part[0][2]).group(1)
        print(f"| {name} | `{kernel}` | {sum(late) / len(late):.2f} | {min(late):.2f} | {max(late):.2f} | "
              f"{sum(us[:50]) / 50:.2f} | {sum(us[-50:]) / 50:.2f} |")


if __name__ == "__main__":
    table(sys.argv[1]) if len(sys.argv) > 1 else run()
