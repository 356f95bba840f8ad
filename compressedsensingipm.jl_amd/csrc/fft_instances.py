"""The FFT pass kernels libcsipm launches, and the translation units that
instantiate them.

The pass kernels (csipm_kernels.hpp) are templates over the precision, the
workgroup size, the spectrum dimensionality and the source / destination /
mode of a pass; every combination the host code launches is listed here.
`write(outdir, nunits)` writes

  fft_extern.inc      explicit instantiation declarations, included by
                      csipm.hip so that its own compilation skips them, and
  fft_inst_<k>.hip    nunits translation units holding the definitions,

so that the kernels compile in parallel.  A combination missing from the
table is still instantiated implicitly by csipm.hip (it only compiles more
slowly); one listed but never launched costs only compile time.
"""
from __future__ import annotations

import os

# kernel -> template arguments after the precision
_LINES = ["2 0 3 true", "2 3 0 false", "3 0 0 false", "3 0 0 true", "3 0 3 true", "3 3 0 false"]
_LINES_BETA = ["2 0 1 true", "2 1 0 false", "3 0 1 true", "3 1 0 false"]
_COL = ["0 0 2", "0 3 3", "2 0 1", "3 0 0"]
_COL_BETA = ["0 1 3", "0 2 4", "1 0 0"]
_ROW = ["0", "2", "3", "4"]
_DIM1 = ["1 2 3 2", "1 3 3 0", "2 0 0 0", "2 2 0 2", "3 0 0 0", "3 2 0 2"]
_DIM1_BETA = ["1 1 1 0", "1 1 2 1", "1 2 1 2", "2 0 2 1", "3 0 2 1"]
# workgroup sizes with the elements per thread: of tiles up to 4096 elements,
# and of the dimension-1 passes with longer lines
_NT = ["256 8", "512 8"]
_NT_DIM1 = _NT + ["1024 8", "1024 16"]


def _rows(nts, rows):
    return [f"{nt} {r}" for nt in nts for r in rows]


TABLE = {
    "k_col": _rows(_NT, _COL + _COL_BETA),
    "k_row": _rows(_NT, _ROW + ["1"]),
    "k_lines": _rows(_NT, _LINES + _LINES_BETA),
    "k_dim1": _rows(_NT_DIM1, _DIM1[1:] + _DIM1_BETA),
    "kb_col": _rows(_NT, _COL),
    "kb_row": _rows(_NT, _ROW),
    "kb_lines": _rows(_NT, _LINES),
    "kb_dim1": _rows(_NT_DIM1, _DIM1),
}


def _params(kernel, t):
    return f"const PassArgs<{t}>*, BSeg" if kernel.startswith("kb_") else f"PassArgs<{t}>"


def instances():
    out = []
    for t in ("float", "double"):
        for k, rows in TABLE.items():
            for r in rows:
                args = ", ".join([t] + r.split())
                out.append(f"void {k}<{args}>({_params(k, t)})")
    return out


def write(outdir, nunits):
    os.makedirs(outdir, exist_ok=True)
    inst = instances()
    ext = ["// generated by fft_instances.py", "namespace csipm {"]
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
