"""Turns two rocprofv3 counter passes of `bench.py --calibration-copy` into the memory-traffic
summary that `bench.py` reads its `roofline.traffic` figure from.

    python bench_traffic_summary.py FETCH_DIR WRITE_DIR > summary.txt

FETCH_DIR / WRITE_DIR: output folders of
    rocprofv3 --pmc FETCH_SIZE --output-format csv -d FETCH_DIR -o run -- \
        python3 bench.py --steps 3 --warmup 1 --no-cpu-baseline --calibration-copy
and the same with WRITE_SIZE.  The calibration dispatches (plain elementwise copies of the
input tensor, bytes known) give the bytes one count stands for; every other kernel's average
count per dispatch is scaled by it.  Lines that start with '@' are the machine-readable part:
the hashes of the kernel sources the run was made with, and per timed C-ABI call the kernel that
did its work with the bytes it read and wrote per launch.
"""
import collections
import csv
import glob
import hashlib
import os
import re
import sys

ROOT = os.path.dirname(os.path.abspath(__file__))
# The headline's kernels and what they include
KERNEL_SOURCES = ["mappedconvolutions_amd/csrc/" + name for name in
                  ("mcx_conv_mfma.hip", "mcx_conv_split.hip", "mcx_conv_split.h", "mcx_conv_runs.hip",
                   "mcx_conv_runs.h", "mcx_mfma_common.h", "mcx_taps.h", "mcx_device.h")]
COPY_BYTES = 8 * 64 * 256 * 512 * 4  # one calibration dispatch reads and writes the input once


def source_lines():
    """A line '@source sha256=... file=...' per kernel source."""
    lines = []
    for name in KERNEL_SOURCES:
        with open(os.path.join(ROOT, name), "rb") as f:
            lines.append("@source sha256=%s file=%s" % (hashlib.sha256(f.read()).hexdigest(), name))
    return lines


def short_name(name):
    name = name.replace("(anonymous namespace)::", "").replace("void mcx::", "")
    name = re.sub(r"\(.*", "", name)
    return name.replace(", ", ",")


def per_kernel(folder, counter):
    """{kernel: [count per dispatch]} and the list of calibration counts."""
    files = glob.glob(os.path.join(folder, "**", "*counter_collection.csv"), recursive=True)
    if not files:
        sys.exit("no counter_collection.csv under " + folder)
    counts, copies = collections.defaultdict(list), []
    for row in csv.DictReader(open(files[0])):
        if row["Counter_Name"] != counter:
            continue
        value = float(row["Counter_Value"])
        name = row["Kernel_Name"]
        if "elementwise_kernel" in name:
            if int(row["Grid_Size"]) * 4 >= COPY_BYTES // 16:  # the whole-tensor copies only
                copies.append(value)
            continue
        if "mcx::" in name:
            counts[short_name(name)].append(value)
    return counts, copies


def label_of(kernel):
    """The timed C-ABI calls whose work this kernel does (none: a helper kernel)."""
    if kernel.startswith(("weight_grad_runs_kernel<", "weight_grad_mfma_kernel<")):
        return ["conv_backward_weight"]
    if kernel.startswith("gather_product_split_kernel<"):
        return ["conv_forward", "conv_backward_input"]  # (one kernel: the average of both calls)
    m = re.match(r"gather_product_mfma_kernel<\w+,(\d+),(\d+),", kernel)
    if m:  # the forward resolves the four bilinear corners itself; the input gradient reads a
        # packed transposed map of one pair per slot
        return ["conv_forward" if m.group(1) == "4" else "conv_backward_input"]
    return []


def main(argv):
    if len(argv) != 2:
        sys.exit(__doc__)
    fetch, fcopies = per_kernel(argv[0], "FETCH_SIZE")
    write, wcopies = per_kernel(argv[1], "WRITE_SIZE")
    if not fcopies or not wcopies:
        sys.exit("no calibration dispatch found: run bench.py with --calibration-copy")
    fscale = COPY_BYTES / (sum(fcopies) / len(fcopies))
    wscale = COPY_BYTES / (sum(wcopies) / len(wcopies))
    print("Calibration: %d + %d copy dispatches of %d bytes each way;" %
          (len(fcopies), len(wcopies), COPY_BYTES))
    print("  one FETCH_SIZE count = %.1f bytes, one WRITE_SIZE count = %.1f bytes" %
          (fscale, wscale))
    print()
    print("%-58s %8s %12s %12s %10s %10s" % ("kernel (average per dispatch)", "launches",
                                             "FETCH_SIZE", "WRITE_SIZE", "read MB", "written MB"))
    rows = []
    for k in sorted(set(fetch) | set(write)):
        f = sum(fetch.get(k, [0])) / max(len(fetch.get(k, [])), 1)
        w = sum(write.get(k, [0])) / max(len(write.get(k, [])), 1)
        rows.append((k, len(fetch.get(k, [])), f, w, f * fscale, w * wscale))
    rows.sort(key=lambda r: -(r[4] + r[5]))
    for k, n, f, w, rb, wb in rows:
        print("%-58s %8d %12.0f %12.0f %10.1f %10.1f" % (k[:58], n, f, w, rb / 1e6, wb / 1e6))
    print()
    print("\n".join(source_lines()))
    best = {}
    for k, n, f, w, rb, wb in rows:
        for lab in label_of(k):
            if lab not in best or rb + wb > best[lab][1] + best[lab][2]:
                best[lab] = (k, rb, wb)  # of two launched variants, the one that did the work
    for lab, (k, rb, wb) in sorted(best.items()):
        print('@traffic label=%s kernel="%s" read_bytes=%d written_bytes=%d' % (lab, k, rb, wb))


if __name__ == "__main__":
    main(sys.argv[1:])
