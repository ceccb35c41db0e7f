"""What the built kernels occupy, read from the code objects' metadata in
libgi_hip.so (built from this source tree): the traversal kernels have no
static LDS, which their stacks' addresses rely on."""
import os
import re
import shutil
import subprocess

import pytest

import globillum_amd

LIB = os.path.join(os.path.dirname(globillum_amd.__file__), "libgi_hip.so")


def _kernels(tmp_path):
    readelf = next((c for c in ("/opt/rocm/llvm/bin/llvm-readelf", shutil.which("llvm-readelf"))
                    if c and os.path.exists(c)), None)
    if readelf is None or not os.path.exists(LIB):
        pytest.skip("llvm-readelf or the library is missing")
    blob = open(LIB, "rb").read()
    found = {}
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    assert at >= 0
    for k, m in enumerate(re.finditer(b"\x7fELF", blob[at:])):
        part = str(tmp_path / f"{k}.co")
        with open(part, "wb") as f:
            f.write(blob[at + m.start():])
        notes = subprocess.run([readelf, "--notes", part], capture_output=True, text=True, timeout=120).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel[kernel.index(".max_flat_workgroup_size"):]).group(1)
            found[name] = int(re.search(r"\.group_segment_fixed_size:\s+(\d+)", kernel).group(1))
    return found


def test_traversal_kernels_have_no_static_lds(tmp_path):
    lds = _kernels(tmp_path)
    trace = {n: b for n, b in lds.items() if "k_trace_closest" in n or "k_trace_any" in n}
    assert len(trace) >= 24, sorted(lds)[:10]
    assert {n: b for n, b in trace.items() if b} == {}
    assert any(b for n, b in lds.items() if "k_shade" in n)  # the static LDS of others is seen
