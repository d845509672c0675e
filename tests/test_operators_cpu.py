"""Registration of the xgen_amd operators: every schema has a Meta and a CUDA-key kernel in this process,
and an operator whose native library is not built raises with the way to build it."""
import pytest
import torch

from xgen_amd import _native as N
from xgen_amd import ops


@pytest.mark.parametrize("name", sorted(ops.SCHEMAS))
def test_every_operator_has_both_kernels(built_library, name):
    for key in ("Meta", "CUDA"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"{ops.NAMESPACE}::{name}", key), key


def test_operators_not_built_say_so():
    with pytest.raises(RuntimeError, match="native operators not found at .*libxgen_amd_ops.so.*build"):
        ops._not_built("quantize_rows", N.operators_path())(None)
