"""The conjugate gradient's scalars, by its source: a kernel of several
workgroups must not write a scalar it returns on.  (Waves of one launch would
read it before or after that write, and those of a workgroup part ways at its
barriers.  The outcome depends on timing, so that no run shows it reliably.)"""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _kernels(text):
    """{name: body} of the __global__ functions with scal among their parameters."""
    out = {}
    for m in re.finditer(r"__global__ void\s+(?:__launch_bounds__\([^)]*\)\s*)?(k_\w+)\(", text):
        open_ = text.index("{", m.end())
        depth, end = 1, open_ + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        if re.search(r"\bscal\b", text[m.end():open_]):
            out[m.group(1)] = text[open_:end]
    return out


def test_no_kernel_writes_what_it_returns_on():
    with open(os.path.join(ROOT, "mongeampere_amd", "csrc", "engine.hip")) as f:
        text = f.read()
    kernels = _kernels(text)
    assert {"k_cg_begin", "k_cg_spmv", "k_cg_update", "k_cg_end"} <= set(kernels)
    checked = 0
    for name, body in kernels.items():
        launches = re.findall(r"hipLaunchKernelGGL\(\(?%s\b[^,]*,\s*([^,]+)," % name, text)
        assert launches, name
        if all(x.strip() == "dim3(1)" for x in launches):
            continue  # one workgroup: its barriers order the write
        returns = set(re.findall(r"if \(scal\[(\d)\] != 0\.0\)\s*(?:return;|\{[^}]*return;)", body))
        writes = set()
        for targets in re.findall(r"((?:scal\[\d\]\s*=\s*)+)", body):
            writes |= set(re.findall(r"\d", targets))
        writes |= set(re.findall(r"scal\[(\d)\]\s*[-+*/]=", body))
        assert not (returns & writes), f"{name}: scal{sorted(returns & writes)}"
        checked += bool(returns)
    assert checked >= 2
