"""The FFT pass kernels libcsipm launches, and the translation units that
instantiate them.

The pass kernels (csipm_kernels.hpp) are templates over the precision, the
workgroup size and the steps of a pass; every combination the host code launches is listed here.
`write(outdir, nunits)` writes

  fft_extern.inc      explicit instantiation declarations, included by
                      csipm.hip so that its own compilation skips them, and
                      the combinations as X-macros for its dispatch, and
  fft_inst_<k>.hip    nunits translation units holding the definitions,

so that the kernels compile in parallel.  A combination missing from the
table is still instantiated implicitly by csipm.hip (it only compiles more
slowly); one listed but never launched costs only compile time.
"""
from __future__ import annotations

import os

# the steps (load, middle, store) of the passes: of the batched chains, on the
# spectrum order, and of the entry points besides
CHAIN_SHORT = [
    "LD_LINES_U2 MID_NONE ST_LINES_BUF_INV", "LD_LINES_U3 MID_NONE ST_LINES_BUF_INV",
    "LD_LINES_BUF_INV MID_NONE ST_LINES_BUF_INV", "LD_LINES_BUF_FWD MID_NONE ST_LINES_BUF_FWD",
    "LD_LINES_BUF_FWD MID_NONE ST_LINES_U2", "LD_LINES_BUF_FWD MID_NONE ST_LINES_U3",
    "LD_COL_FIRST_U MID_NONE ST_COL_BUF_INV", "LD_COL_FIRST_U MID_NONE ST_COL_BUF_FWD",
    "LD_COL_REAL MID_NONE ST_COL_BUF_FWD", "LD_COL_BUF_INV MID_COL ST_COL_BUF_FWD",
    "LD_COL_BUF_FWD MID_NONE ST_COL_U", "LD_COL_BUF_INV MID_NONE ST_COL_U",
    "LD_ROW_INV MID_ROW_MASK ST_ROW_FWD", "LD_ROW_REAL MID_NONE ST_ROW_FWD",
    "LD_ROW_FWD MID_ROW_CONV_INV ST_ROW_INV", "LD_ROW_FWD MID_ROW_CONV_FWD ST_ROW_INV",
]
CHAIN_DIM1 = [
    "LD_DIM1_U MID_DIM1_MASK ST_DIM1_U", "LD_DIM1_BUF MID_DIM1_MASK ST_DIM1_BUF",
    "LD_DIM1_REAL MID_NONE ST_DIM1_U", "LD_DIM1_REAL MID_NONE ST_DIM1_BUF",
]
ENTRY_SHORT = [
    "LD_LINES_BETA2 MID_NONE ST_LINES_BUF_INV", "LD_LINES_BETA3 MID_NONE ST_LINES_BUF_INV",
    "LD_LINES_BUF_FWD MID_NONE ST_LINES_BETA2", "LD_LINES_BUF_FWD MID_NONE ST_LINES_BETA3",
    "LD_COL_FIRST_BETA MID_NONE ST_COL_BUF_INV", "LD_COL_FIRST_BETA MID_NONE ST_COL_BUF_FWD",
    "LD_COL_BUF_INV MID_NONE ST_COL_REAL", "LD_COL_BUF_FWD MID_NONE ST_COL_BETA",
    "LD_COL_BUF_INV MID_NONE ST_COL_BETA", "LD_ROW_INV MID_NONE ST_ROW_REAL",
]
ENTRY_DIM1 = [
    "LD_DIM1_BETA MID_DIM1_MASK ST_DIM1_BETA", "LD_DIM1_BETA MID_NONE ST_DIM1_REAL",
    "LD_DIM1_BUF MID_NONE ST_DIM1_REAL", "LD_DIM1_REAL MID_NONE ST_DIM1_BETA",
]
# workgroup sizes with the elements per thread: of tiles up to 4096 elements,
# and of longer lines (dimension 1 only)
NT_SHORT = ["128 8", "256 8", "512 8"]
NT_LONG = ["1024 8", "1024 16"]
# FP32 tiles of the 2D / 3D passes in which a thread holds 16 elements
NT_WIDE = ["256 16"]
MIXED = "-1 -1 -1"
# of these, the passes of 2D / 3D axes: in the dense form (256 threads)
DENSE_CHAIN = [s for s in CHAIN_SHORT if "LINES" in s] + CHAIN_DIM1[1:2] + CHAIN_DIM1[3:]
DENSE_ENTRY = [s for s in ENTRY_SHORT if "LINES" in s] + ENTRY_DIM1[2:3]


def instances():
    def rows(nts, steps, form="FORM_FFT"):
        return [f"{n} {s} {form}" for n in nts for s in steps]
    dense = NT_SHORT[1:2]
    table = {
        "k_pass": rows(NT_SHORT + NT_LONG, CHAIN_DIM1 + ENTRY_DIM1) +
        rows(NT_SHORT, CHAIN_SHORT + ENTRY_SHORT) +
        rows(dense, DENSE_CHAIN + DENSE_ENTRY, "FORM_DENSE"),
        "kb_pass": rows(NT_SHORT + NT_LONG, CHAIN_DIM1) + rows(NT_SHORT, CHAIN_SHORT) +
        rows(dense, DENSE_CHAIN, "FORM_DENSE") +
        rows(NT_SHORT[1:] + NT_LONG, [MIXED], "FORM_ANY"),
    }
    out = []
    for t in ("float", "double"):
        wide = {"k_pass": DENSE_CHAIN + DENSE_ENTRY, "kb_pass": DENSE_CHAIN}
        for k, rs in table.items():
            if t == "float":
                rs = rs + rows(NT_WIDE, wide[k])
            p = f"PassArgs<{t}>" if k == "k_pass" else f"const PassArgs<{t}>*, const BlockMap*"
            out += [f"void {k}<{', '.join([t] + r.split())}>({p})" for r in rs]
    return out


def write(outdir, nunits):
    os.makedirs(outdir, exist_ok=True)
    inst = instances()
    ext = ["// generated by fft_instances.py"]
    # the steps as X-macros, for the host's dispatch
    for name, steps in (("CHAIN_SHORT", CHAIN_SHORT), ("CHAIN_DIM1", CHAIN_DIM1),
                        ("ENTRY_SHORT", ENTRY_SHORT), ("ENTRY_DIM1", ENTRY_DIM1),
                        ("DENSE_CHAIN", DENSE_CHAIN), ("DENSE_ENTRY", DENSE_ENTRY)):
        ext += [f"#define CSIPM_{name}(X) " +
                " ".join("X(" + ", ".join(s.split()) + ")" for s in steps)]
    ext += ["namespace csipm {"]
    ext += [f"extern template __global__ {s};" for s in inst]
    ext += ["}  // namespace csipm", ""]
    _put(os.path.join(outdir, "fft_extern.inc"), "\n".join(ext))
    files = []
    for u in range(nunits):
        body = ["// generated by fft_instances.py", '#include "csipm_kernels.hpp"',
                "namespace csipm {"]
        body += [f"template __global__ {s};" for s in inst[u::nunits]]
        body += ["}  // namespace csipm", ""]
        p = os.path.join(outdir, f"fft_inst_{u}.hip")
        _put(p, "\n".join(body))
        files.append(p)
    return files


def _put(path, text):
    # rewrite only on change, so unchanged units keep their objects
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, "w") as f:
        f.write(text)
