"""Rules of the CG vector kernels that no run shows reliably, read off their source."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "compressedsensingipm.jl_amd", "csrc", "csipm_batch.hpp")


def _block(text, at):
    """The braces' contents from the first '{' at or after `at`, and its end."""
    a = text.index("{", at)
    depth = 0
    for i in range(a, len(text)):
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        if depth == 0:
            return text[a + 1:i], i + 1
    raise ValueError("unbalanced braces")


def _kernels():
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    out = {}
    for m in re.finditer(r"__global__[^{;]*?void\s+(bk_cg_\w+)\s*\(", text):
        out[m.group(1)] = _block(text, m.end())[0]
    return out


def _split(body):
    """(statements of the first workgroup's first thread, the rest)."""
    one, rest = "", ""
    while True:
        m = re.search(r"if\s*\(lb == 0 && threadIdx\.x == 0\)", body)
        if not m:
            return one, rest + body
        rest += body[:m.start()]
        if body[m.end():].lstrip().startswith("{"):
            inner, end = _block(body, m.end())
        else:
            end = body.index(";", m.end()) + 1
            inner = body[m.end():end]
        one += inner
        body = body[end:]


def _instances(body):
    """The body for SUM = true and for SUM = false."""
    m = re.search(r"if constexpr \(SUM\)", body)
    if not m:
        return [body]
    yes, end = _block(body, m.end())
    no = ""
    if body[end:].lstrip().startswith("else"):
        no, end = _block(body, end)
    return [v for keep, which in ((yes, 0), (no, 1))
            for v in [(_instances(body[:m.start()] + keep + body[end:]) * 2)[which]]]


WRITE = r"\bst\.(\w+)\s*(?:\+|-|\*)?=(?!=)"


@pytest.mark.parametrize("name", sorted(_kernels()))
def test_no_field_read_that_the_launch_writes(name):
    """Several workgroups of one instance (BSEG_BEGIN) do not read a CgState
    field that one thread of the same launch writes: waves that see different
    values part before a workgroup's sum."""
    body = _kernels()[name]
    if "BSEG_BEGIN" not in body:
        return
    helper = re.sub(r"//[^\n]*", "", open(SRC).read())
    for inst in _instances(body):
        _check(inst, helper)


def _check(body, helper):
    one, rest = _split(body)
    written = set(re.findall(WRITE, one))
    for call in re.findall(r"\b(\w+)\(st\)", one):      # helpers that get the state
        at = re.search(r"void\s+%s\s*\(" % call, helper).end()
        written |= set(re.findall(WRITE, _block(helper, at)[0]))
    assert not re.findall(WRITE, rest), "a field is written by every workgroup"
    read = set(re.findall(r"(?:\bst|cg\[inst\])\.(\w+)", rest))
    assert not (read & written), read & written
