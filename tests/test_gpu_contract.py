"""The operators' two statements of their contract (the Meta functions of xgen_amd/ops.py and the checks of
csrc/torch_ops.cpp) accept and refuse the same calls: each call below on meta tensors and on the device
gives the same shapes, strides and dtypes, or the same RuntimeError."""
import pytest
import torch

import xgen_amd  # noqa: F401

pytestmark = pytest.mark.gpu
xops = torch.ops.xgen_amd
BF, HF, F32, F8, I8, I64 = (torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn, torch.int8, torch.int64)


class Make:
    def __init__(self, device):
        self.device = device

    def __call__(self, *shape, dtype=BF, of=None):
        """zeros of `shape`; of: the larger shape whose leading corner it is (strided)."""
        t = torch.zeros(of or shape, dtype=torch.uint8 if dtype == F8 else dtype, device=self.device)
        t = t.view(F8) if dtype == F8 else t
        return t[tuple(slice(0, n) for n in shape)] if of else t

    def cols(self, *shape, dtype=BF):
        """`shape` with a last stride that is not 1."""
        return self(*shape[:-2], shape[-1], shape[-2], dtype=dtype).transpose(-1, -2)


def rows(x, out=F8, act=0):
    return lambda t: xops.quantize_rows(x(t), out, act)


def norm(x=lambda t: t(2, 6, 64), weight=lambda t: t(64), scale=lambda t: t(3, 64), shift=lambda t: t(3, 64),
         indices=lambda t: t(6, dtype=I64), eps=1e-5, kind=1, out=I8, normed=False):
    return lambda t: xops.norm_affine_quant(x(t), weight(t), scale(t), shift(t), indices(t), eps, kind, out, normed)


def mm(a=lambda t: t(5, 32, dtype=F8), w=lambda t: t(48, 32, dtype=F8), sa=lambda t: t(5, dtype=F32),
       sw=lambda t: t(48, dtype=F32), bias=lambda t: t(48), out=BF, act=0, acc=False, exact=False):
    return lambda t: xops.scaled_mm(a(t), w(t), sa(t), sw(t), bias(t), out, act, acc, exact)


def mm_gate(a=lambda t: t(6, 32, dtype=F8), w=lambda t: t(48, 32, dtype=F8), sa=lambda t: t(6, dtype=F32),
            res=lambda t: t(6, 48), gate=lambda t: t(3, 48), idx=lambda t: t(2, dtype=I64)):
    return lambda t: xops.scaled_mm_gate_residual(a(t), w(t), sa(t), t(48, dtype=F32), None, res(t), gate(t), idx(t))


def gate(res=lambda t: t(2, 6, 64), branch=lambda t: t(2, 6, 64), table=lambda t: t(3, 64), idx=lambda t: t(6, dtype=I64)):
    return lambda t: xops.gate_residual(res(t), branch(t), table(t), idx(t))


def modulate(x=lambda t: t(2, 6, 64), scale=lambda t: t(3, 64), shift=lambda t: t(3, 64), idx=lambda t: t(6, dtype=I64), one=False):
    return lambda t: xops.indexed_modulate(x(t), scale(t), shift(t), idx(t), one)


def merge(x, out=F8):
    return lambda t: xops.merge_quant(x(t), out)


ACCEPTED = {
    "rows": rows(lambda t: t(3, 5, 64)), "rows f16 gelu int8": rows(lambda t: t(4, 24, dtype=HF), I8, 1),
    "rows 1-D": rows(lambda t: t(17)), "rows none": rows(lambda t: t(0, 8)), "rows strided": rows(lambda t: t(3, 16, of=(3, 40))),
    "rows by columns": rows(lambda t: t.cols(8, 16)),
    "peak": lambda t: xops.abs_peak(t(3, 7)), "scale": lambda t: xops.fp8_tensor_scale(t(7, dtype=HF)),
    "pack": lambda t: xops.fp8_pack(t(3, 9), t(1, dtype=F32)), "pack 0-dim scale": lambda t: xops.fp8_pack(t(5), t(dtype=F32)),
    "pack none": lambda t: xops.fp8_pack(t(0, 4), t(1, dtype=F32)), "quantize tensor": lambda t: xops.fp8_quantize_tensor(t.cols(4, 6)),
    "norm": norm(), "norm no weight, f32 weight": norm(weight=lambda t: None), "norm f32 weight": norm(weight=lambda t: t(64, dtype=F32)),
    "norm layer, prepared, normed": norm(kind=0x100, out=F8, normed=True), "norm no rows": norm(x=lambda t: t(0, 6, 64)),
    "norm strided": norm(x=lambda t: t(2, 6, 64, of=(2, 8, 72)), scale=lambda t: t(3, 64, of=(3, 68)), shift=lambda t: t(3, 64, of=(4, 64))),
    "norm widest": norm(x=lambda t: t(1, 1, 8192), weight=lambda t: t(8192), scale=lambda t: t(1, 8192),
                        shift=lambda t: t(1, 8192), indices=lambda t: t(1, dtype=I64)),
    "mm": mm(), "mm int8 acc": mm(a=lambda t: t(5, 32, dtype=I8), w=lambda t: t(48, 32, dtype=I8), acc=True),
    "mm f16 f32 bias gelu exact": mm(bias=lambda t: t(48, dtype=F32), out=HF, act=1, acc=True, exact=True),
    "mm scalars no bias": mm(sa=lambda t: t(dtype=F32), sw=lambda t: t(1, dtype=F32), bias=lambda t: None),
    "mm [N, 1] scale": mm(sw=lambda t: t(48, 1, dtype=F32)), "mm no rows": mm(a=lambda t: t(0, 32, dtype=F8), sa=lambda t: t(0, dtype=F32)),
    "mm strided": mm(a=lambda t: t(5, 32, dtype=F8, of=(5, 40)), w=lambda t: t.cols(48, 32, dtype=F8)),
    "gated": mm_gate(), "gated strided": mm_gate(res=lambda t: t(6, 48, of=(6, 50)), gate=lambda t: t(3, 48, of=(3, 64))),
    "gated no rows": mm_gate(a=lambda t: t(0, 32, dtype=F8), sa=lambda t: t(0, dtype=F32), res=lambda t: t(0, 48)),
    "gate": gate(), "gate no batch": gate(res=lambda t: t(0, 6, 64), branch=lambda t: t(0, 6, 64)), "gate strided": gate(table=lambda t: t.cols(3, 64)),
    "modulate": modulate(), "modulate one": modulate(one=True), "modulate strided": modulate(x=lambda t: t.cols(2, 6, 64)),
    "merge": merge(lambda t: t(2, 3, 5, 1, 16)), "merge int8": merge(lambda t: t(1, 1, 4, 2, 8), I8),
    "merge widest": merge(lambda t: t(2, 8, 1, 1, 1024)), "merge none": merge(lambda t: t(2, 3, 0, 1, 8)),
}

REFUSED = {
    "rows f32": rows(lambda t: t(3, 5, dtype=F32)), "rows activation": rows(lambda t: t(3, 5), F8, 2), "rows out": rows(lambda t: t(3, 5), BF),
    "rows no columns": rows(lambda t: t(3, 0)), "rows 0-dim": rows(lambda t: t()),
    "peak f32": lambda t: xops.abs_peak(t(3, dtype=F32)), "scale int8": lambda t: xops.fp8_tensor_scale(t(3, dtype=I8)),
    "quantize tensor f32": lambda t: xops.fp8_quantize_tensor(t(3, dtype=F32)),
    "pack f32": lambda t: xops.fp8_pack(t(3, dtype=F32), t(1, dtype=F32)), "pack scales": lambda t: xops.fp8_pack(t(3), t(2, dtype=F32)),
    "pack bf16 scale": lambda t: xops.fp8_pack(t(3), t(1)),
    "norm 2-D": norm(x=lambda t: t(6, 64)), "norm f16": norm(x=lambda t: t(2, 6, 64, dtype=HF)), "norm x columns": norm(x=lambda t: t.cols(2, 6, 64)),
    "norm no width": norm(x=lambda t: t(2, 6, 0)),
    "norm width": norm(x=lambda t: t(1, 6, 8193), weight=lambda t: None, scale=lambda t: t(3, 8193), shift=lambda t: t(3, 8193)),
    "norm weight size": norm(weight=lambda t: t(63)), "norm weight f16": norm(weight=lambda t: t(64, dtype=HF)),
    "norm weight 2-D": norm(weight=lambda t: t(1, 64)), "norm weight strided": norm(weight=lambda t: t(64, 2)[:, 0]),
    "norm table width": norm(scale=lambda t: t(3, 63)), "norm tables differ": norm(shift=lambda t: t(2, 64)),
    "norm no table": norm(scale=lambda t: t(0, 64), shift=lambda t: t(0, 64)), "norm table f32": norm(scale=lambda t: t(3, 64, dtype=F32)),
    "norm shift f32": norm(shift=lambda t: t(3, 64, dtype=F32)), "norm table columns": norm(scale=lambda t: t.cols(3, 64)),
    "norm shift columns": norm(shift=lambda t: t.cols(3, 64)), "norm indices": norm(indices=lambda t: t(5, dtype=I64)),
    "norm int32 indices": norm(indices=lambda t: t(6, dtype=torch.int32)), "norm strided indices": norm(indices=lambda t: t(6, 2, dtype=I64)[:, 0]),
    "norm 2-D indices": norm(indices=lambda t: t(6, 1, dtype=I64)), "norm eps 0": norm(eps=0.0), "norm eps 1": norm(eps=1.0),
    "norm eps nan": norm(eps=float("nan")), "norm kind": norm(kind=2), "norm kind bits": norm(kind=0x201), "norm negative kind": norm(kind=-1),
    "norm out": norm(out=HF),
    "mm f16 operand": mm(a=lambda t: t(5, 32, dtype=HF)), "mm mixed": mm(w=lambda t: t(48, 32, dtype=I8)), "mm 3-D": mm(a=lambda t: t(1, 5, 32, dtype=F8)),
    "mm K": mm(w=lambda t: t(48, 48, dtype=F8)), "mm scale count": mm(sa=lambda t: t(4, dtype=F32)), "mm scale f16": mm(sa=lambda t: t(5, dtype=HF)),
    "mm w scale count": mm(sw=lambda t: t(5, dtype=F32)), "mm w scale f64": mm(sw=lambda t: t(48, dtype=torch.float64)),
    "mm bias size": mm(bias=lambda t: t(47)), "mm bias 2-D": mm(bias=lambda t: t(1, 48)), "mm bias int8": mm(bias=lambda t: t(48, dtype=I8)),
    "mm out f32": mm(out=F32), "mm activation": mm(act=-1), "mm K 24": mm(a=lambda t: t(5, 24, dtype=F8), w=lambda t: t(48, 24, dtype=F8)),
    "mm N 40": mm(w=lambda t: t(40, 32, dtype=F8), sw=lambda t: t(40, dtype=F32), bias=lambda t: None),
    "mm exact int8": mm(a=lambda t: t(5, 32, dtype=I8), w=lambda t: t(48, 32, dtype=I8), exact=True),
    "gated residual shape": mm_gate(res=lambda t: t(5, 48)), "gated residual f16": mm_gate(res=lambda t: t(6, 48, dtype=HF)),
    "gated residual 3-D": mm_gate(res=lambda t: t(1, 6, 48)), "gated table width": mm_gate(gate=lambda t: t(3, 32)),
    "gated no table": mm_gate(gate=lambda t: t(0, 48)), "gated table f32": mm_gate(gate=lambda t: t(3, 48, dtype=F32)),
    "gated seq": mm_gate(idx=lambda t: t(4, dtype=I64)), "gated no indices": mm_gate(idx=lambda t: t(0, dtype=I64)),
    "gated int32 indices": mm_gate(idx=lambda t: t(2, dtype=torch.int32)),
    "gate 2-D": gate(res=lambda t: t(6, 64)), "gate branch": gate(branch=lambda t: t(2, 6, 32)), "gate no width": gate(res=lambda t: t(2, 6, 0), branch=lambda t: t(2, 6, 0)),
    "gate table": gate(table=lambda t: t(3, 32)), "gate no table": gate(table=lambda t: t(0, 64)), "gate indices": gate(idx=lambda t: t(5, dtype=I64)),
    "gate f16": gate(branch=lambda t: t(2, 6, 64, dtype=HF)), "gate table f32": gate(table=lambda t: t(3, 64, dtype=F32)),
    "modulate 2-D": modulate(x=lambda t: t(6, 64)), "modulate table": modulate(scale=lambda t: t(3, 32)), "modulate tables": modulate(shift=lambda t: t(2, 64)),
    "modulate no table": modulate(scale=lambda t: t(0, 64), shift=lambda t: t(0, 64)), "modulate indices": modulate(idx=lambda t: t(6, 1, dtype=I64)),
    "modulate f32": modulate(x=lambda t: t(2, 6, 64, dtype=F32)), "modulate shift f16": modulate(shift=lambda t: t(3, 64, dtype=HF)),
    "merge 4-D": merge(lambda t: t(2, 3, 5, 16)), "merge f16": merge(lambda t: t(2, 3, 5, 1, 16, dtype=HF)), "merge chunk": merge(lambda t: t(2, 3, 5, 1, 12)),
    "merge no owners": merge(lambda t: t(2, 0, 5, 1, 16)), "merge width": merge(lambda t: t(2, 8, 1, 1, 1032)), "merge out": merge(lambda t: t(2, 3, 5, 1, 16), BF),
}


def outcome(call, device):
    try:
        out = call(Make(device))
    except RuntimeError as error:
        return "refused", str(error).splitlines()[0]
    return "accepted", [(tuple(o.shape), o.stride(), o.dtype) for o in (out if isinstance(out, (tuple, list)) else (out,))]


@pytest.mark.parametrize("name", sorted(ACCEPTED))
def test_accepted_alike(cuda, name):
    meta, device = outcome(ACCEPTED[name], "meta"), outcome(ACCEPTED[name], cuda)
    assert meta[0] == "accepted" and device == meta


@pytest.mark.parametrize("name", sorted(REFUSED))
def test_refused_alike(cuda, name):
    meta, device = outcome(REFUSED[name], "meta"), outcome(REFUSED[name], cuda)
    assert meta[0] == "refused" and device == meta
