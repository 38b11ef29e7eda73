#!/usr/bin/env python3
"""Build step: the register and scratch use of every compiled kernel instance.

hipcc compiles the kernel translation units with
-Rpass-analysis=kernel-resource-usage, and the Makefile keeps each unit's
remarks in a `.res` file beside its object. This script reads them and writes
a C++ initializer list, one line per kernel function:

    {"<kernel family>", {<template arguments>}, vgprs, agprs, sgprs, scratch},

which csrc/plan/instances.cpp includes (`instance_resources.inc`), so the
plan knows, for each instance it can bind, how many registers it holds and
how many bytes per lane it spills to scratch, as the compiler reported them.

Kernel families and their template arguments (Itanium-mangled names):
  gemm_kernel      BM BN BK WGM WGN OUT STAGES SPREAD EPI
  gemm_kernel_pw   BM BN BK WGM WGN STAGES
  gemm_mfma16      EPI
  gemm_mfma16_f32  OUT EPI
  gemm_mfma16g     BM BN BK WGM WGN STAGES OUT EPI
  gemm_mfma16g_split  BM BN BK WGM WGN STAGES OUT

Usage: resource_table.py OUT.inc RES_FILE...
"""
from __future__ import annotations

import re
import sys

FAMILIES = ("gemm_kernel", "gemm_kernel_pw", "gemm_mfma16", "gemm_mfma16_f32",
            "gemm_mfma16g", "gemm_mfma16g_split")
NAME = re.compile(r"remark: Function Name: (\S+)")
FIELD = re.compile(r"remark:\s+(TotalSGPRs|VGPRs|AGPRs|ScratchSize \[bytes/lane\]): (\d+)")
MANGLED = re.compile(r"^_ZN3tbk(\d+)(\w+)$")
TARG = re.compile(r"L([ib])(n?)(\d+)E")


def parse_name(mangled: str):
    """(family, [template args]) of a tbk kernel, or None for other functions."""
    m = MANGLED.match(mangled)
    if not m:
        return None
    n = int(m.group(1))
    rest = m.group(2)
    family, tail = rest[:n], rest[n:]
    if family not in FAMILIES or not tail.startswith("I"):
        return None
    end = tail.index("EEv") if "EEv" in tail else len(tail)
    args = [(-1 if neg else 1) * int(v) for _, neg, v in TARG.findall(tail[1:end + 1])]
    return family, tuple(args)


def read(paths):
    rows = {}
    for path in paths:
        cur = None
        with open(path) as f:
            for line in f:
                m = NAME.search(line)
                if m:
                    cur = parse_name(m.group(1))
                    if cur:
                        rows[cur] = {}
                    continue
                m = FIELD.search(line)
                if m and cur:
                    rows[cur][m.group(1)] = int(m.group(2))
    return rows


def main() -> int:
    out, paths = sys.argv[1], sys.argv[2:]
    rows = read(paths)
    if not rows:
        print("resource_table.py: no kernel resource remarks found", file=sys.stderr)
        return 1
    lines = ["// generated by csrc/tools/resource_table.py from the compiler's",
             "// -Rpass-analysis=kernel-resource-usage remarks; do not edit"]
    for (family, args), r in sorted(rows.items()):
        missing = {"VGPRs", "AGPRs", "TotalSGPRs", "ScratchSize [bytes/lane]"} - set(r)
        if missing:
            print(f"resource_table.py: {family}{args}: no {sorted(missing)} remark",
                  file=sys.stderr)
            return 1
        lines.append('{"%s", {%s}, %d, %d, %d, %d},' % (
            family, ", ".join(str(a) for a in args), r["VGPRs"], r["AGPRs"],
            r["TotalSGPRs"], r["ScratchSize [bytes/lane]"]))
    text = "\n".join(lines) + "\n"
    with open(out, "w") as f:
        f.write(text)
    return 0


if __name__ == "__main__":
    sys.exit(main())
