"""Registration of the xgen_amd operators: every schema has a Meta and a CUDA-key kernel in this process, the
latter the native one; a package imported before its native operators are built (or over a library that does
not load) imports, says on a call what is missing, and takes them once they are there."""
import json
import shutil
import subprocess
import sys

import pytest
import torch

from xgen_amd import _native as N
from xgen_amd import ops


@pytest.mark.parametrize("name", sorted(ops.SCHEMAS))
def test_every_operator_has_both_kernels(built_library, name):
    for key in ("Meta", "CUDA"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"{ops.NAMESPACE}::{name}", key), key


DUMP = r"""
import json, sys
sys.path.insert(0, sys.argv[1])
import torch
from xgen_amd import ops
print(json.dumps({name: torch._C._dispatch_dump(f"{ops.NAMESPACE}::{name}") for name in ops.SCHEMAS}))
"""


def test_cuda_kernels_are_the_native_ones(built_library):
    """In a process of its own: the CUDA-key kernels come from torch_ops.cpp (the SwiGLU's from ops.py), and no
    stand-in lies below them."""
    proc = subprocess.run([sys.executable, "-c", DUMP, str(N.Path(ops.__file__).parents[1])], stdout=subprocess.PIPE,
                          text=True, timeout=120, check=True)
    for name, dump in json.loads(proc.stdout.splitlines()[-1]).items():
        assert "CompositeExplicitAutograd" not in dump, dump
        cuda = [line for line in dump.splitlines() if line.startswith("CUDA")]
        assert len(cuda) == 1 and ("ops.py" if name == "swiglu_quant" else "torch_ops.cpp") in cuda[0], dump


LATE = r"""
import shutil, sys
import torch
sys.path.insert(0, sys.argv[1])
import xgen_amd
from xgen_amd import _native as N, ops
assert str(N.operators_path()).startswith(sys.argv[1])
cuda = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
x = torch.ones(4, 16, dtype=torch.bfloat16)
call = lambda: torch.ops.xgen_amd.abs_peak.default.redispatch(cuda, x)
def error(fn):
    try:
        fn()
    except Exception as e:
        return type(e).__name__, str(e)
assert torch.ops.xgen_amd.abs_peak(x.to("meta")).shape == ()
for _ in range(2):
    kind, text = error(call)
    assert kind == "RuntimeError" and sys.argv[3] in text and "libxgen_amd_ops.so" in text and "build" in text, (kind, text)
N.operators_path().unlink(missing_ok=True)
shutil.copy(sys.argv[2], N.operators_path())
error(call)
kind, text = error(call)  # the native kernel's own check
assert kind == "RuntimeError" and "require tensors on a HIP (cuda) device" in text, (kind, text)
kind, text = error(lambda: torch.ops.xgen_amd.abs_peak(x))
assert kind == "NotImplementedError" and "CPU" in text, (kind, text)
print("ok")
"""


@pytest.mark.parametrize("state,says", [("absent", "not found"), ("unloadable", "do not load")])
def test_operators_built_after_the_import(built_library, tmp_path, state, says):
    package = tmp_path / "xgen_amd"
    shutil.copytree(N.Path(ops.__file__).parent, package, ignore=shutil.ignore_patterns("_lib", "__pycache__", "csrc"))
    (package / "_lib").mkdir()
    if state == "unloadable":
        (package / "_lib" / N.operators_path().name).write_bytes(b"not a library")
    proc = subprocess.run([sys.executable, "-c", LATE, str(tmp_path), str(N.operators_path()), says], cwd=tmp_path,
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert proc.returncode == 0 and proc.stdout.strip().endswith("ok"), proc.stdout
    assert "Overriding a previously registered kernel" not in proc.stdout
